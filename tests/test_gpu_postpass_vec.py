"""The post-pass on 16-byte vectors (k_postpass_vec): both sides in one wave per
row, and one side alone (a frozen tower), against rows that are not 16-byte
vectors (k_postpass: the same features at an odd row stride), around the row
lengths where its registers double (1024) and where it ends (2048), and with
split contractions.  The same arithmetic with the feature sum <x^, h> in
another order, on contractions whose tiles the row stride does not change:
2e-6 of the largest gradient for fp32 (the register-staged tiles of an odd row
stride sum in another order too), one unit in the last place (and fp16's
smallest step, 2^-24) for the 16-bit types."""
import pytest
import torch

from helpers import max_rel, randn_pair
from memoryefficientclip_amd.clip_loss import MemoryEfficientCLIPLoss

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}


@pytest.mark.parametrize("parts", [1, 2])
@pytest.mark.parametrize("normed", [False, True], ids=["normalize", "raw"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("d", [8, 20, 1024, 1032, 2048, 2056])
def test_vectors_match_single_values(monkeypatch, d, dtype, normed, parts):
    n = 190
    monkeypatch.setenv("MEC_KEEP_EXP", "0")
    monkeypatch.setenv("MEC_CONTRACT_PARTS", str(parts))
    a, b = randn_pair(n, d, seed=d)
    if normed:
        a, b = torch.nn.functional.normalize(a, dim=1), torch.nn.functional.normalize(b, dim=1)
    a, b = a.to(dtype), b.to(dtype)
    print(f"postpass d={d} {dtype} normed={normed} parts={parts}", flush=True)

    def run(gx, gy, pad=0):
        w = torch.zeros(n, d + pad, dtype=dtype), torch.zeros(n, d + pad, dtype=dtype)
        w[0][:, pad:], w[1][:, pad:] = a, b
        x, y = (t.to(DEV)[:, pad:].requires_grad_(g) for t, g in zip(w, (gx, gy)))
        (MemoryEfficientCLIPLoss(0.07, normed)(x, y) * 64.0).backward()
        return x.grad, y.grad

    both, odd = run(True, True), run(True, True, pad=1)
    one = run(True, False)[0], run(False, True)[1]
    for got in (both, one):
        for u, v in zip(got, odd):
            u, v = u.float().cpu(), v.float().cpu()
            if dtype == torch.float32:
                assert max_rel(u, v) <= 2e-6
            else:
                floor = max(float(v.abs().max()) * 2.0 ** -14, 2.0 ** -24 if dtype == torch.float16 else 0.0)
                assert ((u - v).abs() <= ULP[dtype] * v.abs() + floor).all()
