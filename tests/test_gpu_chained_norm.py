"""The chained 16-bit kernels on inputs that they normalize (raw rows with norms
that differ): the forward's block walk with its scales loaded a tile ahead, and
the chained gradient-matrix tiles, at 128 x 128 and 256 x 256 tiles: one tile,
several per workgroup with uneven blocks, two-tile blocks (17 tiles a side), a
single k-chunk (D <= 64), ragged n.  Loss and gradients against the fp64
oracle at the 16-bit tolerance, the loss (sums in fp32 of exact products)
against 2e-6, and bitwise repeatable."""
import pytest
import torch

import oracle
from helpers import TOL, max_rel, randn_pair, rel_err
from memoryefficientclip_amd.clip_loss import MemoryEfficientCLIPLoss
from memoryefficientclip_amd.lit_loss import MemoryEfficientLiTLoss

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("n,d,lit,small", [(5, 8, False, "0"), (257, 64, False, "0"), (700, 72, True, "1"),
                                           (2900, 40, False, "1"), (4352, 72, False, "0"), (4700, 136, True, "0"),
                                           (6150, 64, False, "0")])
def test_raw_rows(monkeypatch, n, d, lit, small, dtype):
    monkeypatch.setenv("MEC_16BIT_SMALL_TILES", small)
    a, b = randn_pair(n, d, seed=n + d)
    g = torch.Generator().manual_seed(n)
    a = (a * torch.exp(torch.randn(n, 1, generator=g))).to(dtype)
    b = (b * torch.exp(torch.randn(n, 1, generator=g))).to(dtype)
    print(f"chained norm {dtype} n={n} d={d} lit={lit} small={small}", flush=True)
    outs = []
    for _ in range(2):
        x, y = a.to(DEV).requires_grad_(True), b.to(DEV).requires_grad_(not lit)
        loss = (MemoryEfficientLiTLoss if lit else MemoryEfficientCLIPLoss)(0.07)(x, y)
        (loss * 16.0).backward()
        torch.cuda.synchronize()
        outs.append([loss.detach().cpu()] + [t.grad.cpu() for t in (x, y) if t.grad is not None])
    assert all(torch.equal(u, v) for u, v in zip(*outs))
    fn = oracle.lit_loss_and_grads if lit else oracle.clip_loss_and_grads
    ref = fn(a.float(), b.float(), 0.07, grad_output=16.0)
    assert rel_err(outs[0][0], ref[0]) <= 2e-6
    for u, r in zip(outs[0][1:], ref[1:]):
        assert max_rel(u, r) <= TOL[dtype]["grad"]
