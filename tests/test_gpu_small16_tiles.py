"""128 x 128 tiles of the 16-bit kernels (small16_n), forced on and off
(MEC_16BIT_SMALL_TILES), around their edges: tiles, 32-value groups of the pairs,
blocks of 256 rows, contractions split over k, inputs normalized here or not,
rows that are not 16-byte vectors (the contractions alone change), one side
alone.  Against the fp64 oracle at each type's tolerance (16-bit 1e-2, fp32
pairs 4e-6: four times what the fp32 kernels show), and bitwise repeatable in
deterministic mode."""
import pytest
import torch

import oracle
from helpers import TOL, max_rel, randn_pair, rel_err
from memoryefficientclip_amd import _lib
from memoryefficientclip_amd.clip_loss import MemoryEfficientCLIPLoss
from memoryefficientclip_amd.lit_loss import MemoryEfficientLiTLoss

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# kind, n, d, mode, normalized inputs, row padding, blocks of 256 rows (0: default), parts (0: default), frozen y
CASES = [
    ("bf16", 1, 8, "clip", False, 0, 0, 0, False),
    ("bf16", 127, 64, "clip", False, 0, 0, 0, False),
    ("f16", 128, 120, "lit", True, 0, 0, 0, False),
    ("bf16", 129, 136, "clip", True, 0, 0, 0, False),
    ("bf16", 700, 37, "clip", False, 0, 0, 2, False),
    ("f16", 1300, 200, "clip", True, 0, 2, 2, False),
    ("bf16", 1300, 72, "lit", False, 8, 1, 0, False),
    ("bf16", 2050, 264, "clip", False, 0, 0, 0, True),
    ("bf16", 3000, 128, "clip", True, 0, 0, 0, False),
    ("medium", 900, 130, "clip", False, 0, 0, 3, False),
    ("pairs", 31, 33, "clip", False, 0, 0, 0, False),
    ("pairs", 129, 100, "lit", True, 3, 0, 0, False),
    ("pairs", 1300, 130, "clip", False, 0, 2, 3, False),
    ("pairs", 2600, 257, "clip", True, 0, 0, 0, False),
]


@pytest.mark.parametrize("small", ["1", "0"], ids=["128", "256"])
@pytest.mark.parametrize("kind,n,d,mode,normed,pad,tb,parts,frozen", CASES, ids=[f"{c[0]}-{c[1]}x{c[2]}" for c in CASES])
def test_small_tiles_against_the_oracle(monkeypatch, kind, n, d, mode, normed, pad, tb, parts, frozen, small):
    lit = mode == "lit"
    dt = {"bf16": torch.bfloat16, "f16": torch.float16}.get(kind, torch.float32)
    monkeypatch.setenv("MEC_16BIT_SMALL_TILES", small)
    if kind == "pairs":
        monkeypatch.setenv("MEC_F32_PAIRS", "1")
    if tb:
        monkeypatch.setenv("MEC_GRAD_BLOCK_TILES", str(tb))
    if parts:
        monkeypatch.setenv("MEC_CONTRACT_PARTS", str(parts))
    code = {"bf16": 1, "f16": 2, "pairs": _lib.DTYPE_F32_PAIRS, "medium": _lib.DTYPE_F32_BF16}[kind]
    want = 128 if small == "1" else 256
    assert _lib.backward_plan(n, d, code, int(lit), 1 if lit or frozen else 3, 256).contract_tile_rows == want
    a, b = randn_pair(n, d, seed=n + d)
    if normed:
        a, b = torch.nn.functional.normalize(a, dim=1), torch.nn.functional.normalize(b, dim=1)
    wa, wb = torch.zeros(n, d + pad, dtype=dt), torch.zeros(n, d + pad, dtype=dt)
    wa[:, pad:], wb[:, pad:] = a, b
    a, b = wa[:, pad:].contiguous(), wb[:, pad:].contiguous()
    print(f"small16 {kind} n={n} d={d} {mode} normed={normed} pad={pad} blocks={tb} parts={parts} small={small}", flush=True)

    def run():
        x = wa.to(DEV)[:, pad:].requires_grad_(True)
        y = wb.to(DEV)[:, pad:].requires_grad_(not lit and not frozen)
        loss = (MemoryEfficientLiTLoss if lit else MemoryEfficientCLIPLoss)(0.07, normed)(x, y)
        (loss * 8.0).backward()
        torch.cuda.synchronize()
        return [loss.detach().cpu()] + [t.grad.cpu() for t in (x, y) if t.grad is not None]

    old = torch.get_float32_matmul_precision()
    torch.set_float32_matmul_precision("medium" if kind == "medium" else "highest")
    torch.use_deterministic_algorithms(True)
    try:
        got, again = run(), run()
    finally:
        torch.use_deterministic_algorithms(False)
        torch.set_float32_matmul_precision(old)
    assert all(torch.equal(u, v) for u, v in zip(got, again))
    if lit:
        ref = oracle.lit_loss_and_grads(a.float(), b.float(), 0.07, normalized_inputs=normed, grad_output=8.0)
    else:
        ref = oracle.clip_loss_and_grads(a.float(), b.float(), 0.07, normalized_inputs=normed, grad_output=8.0)
    tol = 4e-6 if kind == "pairs" else TOL[torch.bfloat16]["grad"]
    assert rel_err(got[0], ref[0]) <= tol or abs(float(got[0]) - float(ref[0])) < 1e-6
    for g, r in zip(got[1:], ref[1:]):
        assert max_rel(g, r) <= tol
