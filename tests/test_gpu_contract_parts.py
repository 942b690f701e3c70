"""Contractions split over k (mec_backward_scratch_bytes): forced numbers of
parts (MEC_CONTRACT_PARTS) against the unsplit contractions of the same
problem, in every 16-bit kernel family, both tile widths and the narrow tiles,
several blocks with a short last one (parts past its end), and one side alone.

The same products are summed in another order: fp32 gradients (pairs, and bf16
products on fp32 data) may differ by the rounding of fp32 sums (2e-6 of the
largest), 16-bit ones by a unit in the last place where a value sits at a
rounding boundary (2^-7 of a value for bf16, 2^-10 for fp16 and never less than fp16's
smallest step 2^-24: gradients of 1e-5 are fp16 subnormals)."""
import pytest
import torch

from helpers import matmul_precision, max_rel, randn_pair
from memoryefficientclip_amd import _lib
from memoryefficientclip_amd.clip_loss import MemoryEfficientCLIPLoss
from memoryefficientclip_amd.lit_loss import MemoryEfficientLiTLoss

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}


def grads(a, b, lit, gx, gy, normed):
    x, y = a.to(DEV).requires_grad_(gx), b.to(DEV).requires_grad_(gy and not lit)
    (MemoryEfficientLiTLoss if lit else MemoryEfficientCLIPLoss)(0.07, normed)(x, y).backward()
    torch.cuda.synchronize()
    return [t.grad.cpu().float() for t in (x, y) if t.grad is not None]


# dtype, n, d, parts, mode, sides, block rows / 256 (0: default), env
CASES = [
    ("bf16", 1000, 96, 2, "clip", 3, 0, {}),
    ("bf16", 1024, 512, 8, "clip", 3, 0, {}),
    ("f16", 2050, 264, 3, "lit", 1, 0, {}),
    ("bf16", 2300, 384, 3, "clip", 3, 2, {}),  # 512-row blocks, the last of 252 rows
    ("f16", 1300, 72, 2, "clip", 2, 1, {}),
    ("bf16", 2304, 300, 4, "clip", 3, 0, {"MEC_NARROW_CONTRACT": "1"}),
    ("bf16", 2304, 768, 4, "clip", 3, 0, {"MEC_WIDE_CONTRACT": "1"}),
    ("bf16", 2304, 768, 4, "clip", 3, 4, {"MEC_WIDE_CONTRACT": "0"}),
    ("pairs", 1000, 96, 2, "clip", 3, 0, {}),
    ("pairs", 2300, 300, 3, "clip", 3, 2, {}),
    ("pairs", 2100, 520, 7, "lit", 1, 0, {}),
    ("medium", 1500, 200, 4, "clip", 1, 0, {}),
]


@pytest.mark.parametrize("kind,n,d,parts,mode,sides,tb,env", CASES, ids=lambda v: str(v) if not isinstance(v, dict) else
                         "-".join(v))
def test_parts_match_the_unsplit_contractions(monkeypatch, kind, n, d, parts, mode, sides, tb, env):
    lit = mode == "lit"
    dt = {"bf16": torch.bfloat16, "f16": torch.float16}.get(kind, torch.float32)
    code = {"bf16": 1, "f16": 2, "pairs": _lib.DTYPE_F32_PAIRS, "medium": _lib.DTYPE_F32_BF16}[kind]
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    if kind == "pairs":
        monkeypatch.setenv("MEC_F32_PAIRS", "1")
    if tb:
        monkeypatch.setenv("MEC_GRAD_BLOCK_TILES", str(tb))
    a, b = randn_pair(n, d, seed=n + d)
    a, b = a.to(dt), b.to(dt)
    lib = _lib.load()
    m = int(lit)
    base = lib.mec_grad_scratch_bytes_for(n, d, code, m, sides)
    out = []
    print(f"parts {kind} n={n} d={d} parts={parts} {mode} sides={sides} blocks={tb} {env}", flush=True)
    with matmul_precision("medium" if kind == "medium" else "highest"):
        for p in (1, parts):
            monkeypatch.setenv("MEC_CONTRACT_PARTS", str(p))
            want = base if p == 1 else (base + 255) // 256 * 256 + (p - 1) * n * d * 4 * bin(sides).count("1")
            assert lib.mec_backward_scratch_bytes(n, d, code, m, sides) == want
            out.append(grads(a, b, lit, bool(sides & 1), bool(sides & 2), False))
    assert len(out[0]) == len(out[1]) == (1 if lit else bin(sides).count("1"))
    for u, v in zip(*out):
        if dt == torch.float32:
            assert max_rel(v, u) <= 2e-6
        else:
            # (the smallest values sit next to cancelling terms: floor at 2^-14 of the largest)
            floor = max(float(u.abs().max()) * 2.0 ** -14, 2.0 ** -24 if dt == torch.float16 else 0.0)
            assert ((u - v).abs() <= ULP[dt] * u.abs() + floor).all()
            assert (u != v).float().mean() < 0.05
    # and the same bits again
    with matmul_precision("medium" if kind == "medium" else "highest"):
        torch.use_deterministic_algorithms(True)
        try:
            r = [grads(a, b, lit, bool(sides & 1), bool(sides & 2), False) for _ in range(2)]
        finally:
            torch.use_deterministic_algorithms(False)
    assert all(torch.equal(u, v) for u, v in zip(*r))


def test_the_scratch_is_sized_on_the_tensors_device(monkeypatch):
    """The parts follow the compute units of the current device: with another one
    current, the size is asked for after the switch and the switch undone."""
    x, y = (torch.randn(300, 64, device=DEV, dtype=torch.bfloat16, requires_grad=True) for _ in range(2))
    loss = MemoryEfficientCLIPLoss(0.07)(x, y)
    lib, seen = _lib.load(), []
    size = lib.mec_backward_scratch_bytes
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    monkeypatch.setattr(torch.cuda, "set_device", lambda i: seen.append(i))
    monkeypatch.setattr(lib, "mec_backward_scratch_bytes", lambda *a: (seen.append("size"), size(*a))[1])
    loss.backward()
    assert seen == [0, "size", 1]
    assert x.grad is not None and y.grad is not None
