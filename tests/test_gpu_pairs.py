"""fp32 data as fp16 pairs (MEC_DTYPE_F32_PAIRS): the larger fp32 problems, and
fp32 data under matmul precision "high".

* The pairs that mec_prepass writes are checked bit for bit against a numpy
  restatement (scale by a power of two, hi = fp16(v), lo = fp16(v - hi)).
* Loss and gradients against the fp64 oracle at the edges of the tiles (256),
  of the 32-value groups and of the backward's blocks, in both modes, with rows
  that are normalized here and rows of any scale that come as they are.  Bar:
  every value that is left out is below 2^-22 of a product or 2^-39 of the
  largest value, and an fp32 sum rounds by 2^-24 a term; 4e-6 of the largest
  gradient is four times the most that the fp32 kernels show on these shapes.
* Against the fp32 kernels, the distance to the 64-bit gradients' off-diagonal
  part (what the pairs compute) is no larger.
"""
import os

import numpy as np
import pytest
import torch

import oracle
from helpers import max_rel, randn_pair, rel_err
from memoryefficientclip_amd import _lib
from memoryefficientclip_amd.clip_loss import MemoryEfficientCLIPLoss
from memoryefficientclip_amd.lit_loss import MemoryEfficientLiTLoss

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BAR = 4e-6


def say(*a):
    print(*a, flush=True)


@pytest.fixture
def pairs(monkeypatch):
    monkeypatch.setenv("MEC_F32_PAIRS", "1")
    return monkeypatch


def scale_of(v):
    """The power of two that puts the largest finite magnitude into [2^14, 2^15)."""
    m = np.abs(v[np.isfinite(v)]).max(initial=0.0)
    return np.float32(2.0 ** min(14 - np.floor(np.log2(m)), 126)) if m > 0 else np.float32(1)


def pair_rows(v):
    """Rows of pairs: every 32 values as 32 hi and then 32 lo, zero-padded."""
    n, d = v.shape
    dp = (d + 31) // 32 * 32
    w = np.zeros((n, dp), np.float32)
    w[:, :d] = v
    hi = w.astype(np.float16)
    with np.errstate(invalid="ignore"):
        lo = np.where(np.isinf(hi), np.float32(0), w - hi.astype(np.float32)).astype(np.float16)
    out = np.stack([hi.reshape(n, -1, 32), lo.reshape(n, -1, 32)], axis=2)
    return out.reshape(n, 2 * dp).view(np.uint16)


@pytest.mark.parametrize("norm", [1, 0], ids=["normalize", "raw"])
@pytest.mark.parametrize("n,d,ld", [(300, 96, 96), (77, 3, 5), (1001, 130, 136), (5, 2100, 2100)])
def test_pairs_are_exact(n, d, ld, norm):
    g = torch.Generator().manual_seed(n + d)
    xw = torch.randn(n, ld, generator=g) * torch.exp(3 * torch.randn(n, ld, generator=g))
    yw = torch.randn(n, ld, generator=g) * 1e-6
    xw[1] = 0.0
    if not norm:
        yw[2, 1] = float("inf")  # (an infinite value does not set the scale)
    x, y = xw.to(DEV), yw.to(DEV)
    lib, dt = _lib.load(), _lib.DTYPE_F32_PAIRS
    nf = lib.mec_workspace_floats_for(n, d, dt)
    ws = torch.zeros(nf, dtype=torch.float32, device=DEV)
    say(f"pairs n={n} d={d} ld={ld} normalize={norm}")
    _lib.call("mec_prepass", x.data_ptr(), ld, y.data_ptr(), ld, n, d, dt, norm, ws.data_ptr(),
              torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    dp = (d + 31) // 32 * 32
    off = (lib.mec_workspace_floats(n) + 63) // 64 * 64
    assert nf == off + 64 + 2 * n * dp
    scl = ws[off:off + 4].cpu().numpy()
    raw = ws[off + 64:].cpu().numpy().view(np.uint16).reshape(2, n, 2 * dp)
    rx, ry = ws[:n].cpu().numpy()[:, None], ws[n:2 * n].cpu().numpy()[:, None]
    vx, vy = xw[:, :d].numpy(), yw[:, :d].numpy()
    sx, sy = (np.float32(16384), np.float32(16384)) if norm else (scale_of(vx), scale_of(vy))
    assert list(scl) == [sx, sy, 1 / sx, 1 / sy]
    np.testing.assert_array_equal(raw[0], pair_rows(vx * rx * sx))
    np.testing.assert_array_equal(raw[1], pair_rows(vy * ry * sy))


CASES = [
    # (mode, n, d, normalized_inputs, temperature, row stride - d, blocks of 256 rows (0: the default))
    ("clip", 1, 1, False, 0.07, 0, 0),
    ("clip", 2, 33, False, 0.1, 0, 0),
    ("lit", 31, 31, False, 0.07, 3, 0),
    ("clip", 255, 32, True, 0.07, 0, 0),
    ("clip", 256, 64, False, 0.05, 0, 0),
    ("clip", 257, 257, False, 0.07, 1, 0),
    ("lit", 513, 255, True, 0.07, 0, 1),
    ("clip", 1300, 130, False, 0.07, 0, 2),
    ("clip", 2049, 320, True, 0.1, 5, 3),
    ("clip", 2600, 512, False, 0.07, 0, 0),
]


@pytest.mark.parametrize("mode,n,d,normed,t,pad,tb", CASES, ids=[f"{c[0]}-{c[1]}x{c[2]}-{c[6]}" for c in CASES])
def test_parity_against_the_oracle(pairs, mode, n, d, normed, t, pad, tb):
    lit = mode == "lit"
    if tb:
        pairs.setenv("MEC_GRAD_BLOCK_TILES", str(tb))
    a, b = randn_pair(n, d, seed=n + 3 * d)
    sa, sb = 1.0, 1.0
    if normed:
        # any scale whose products are those of unit rows
        sa, sb = 3000.0, 1.0 / 3000.0
        a, b = torch.nn.functional.normalize(a, dim=1), torch.nn.functional.normalize(b, dim=1)
    wa, wb = torch.zeros(n, d + pad), torch.zeros(n, d + pad)
    wa[:, pad:], wb[:, pad:] = a * sa, b * sb
    a, b = wa[:, pad:].contiguous(), wb[:, pad:].contiguous()
    ga = wa.to(DEV)[:, pad:].requires_grad_(True)
    gb = wb.to(DEV)[:, pad:].requires_grad_(not lit)
    say(f"pairs {mode} n={n} d={d} normed={normed} T={t} pad={pad} blocks={tb}")
    loss = (MemoryEfficientLiTLoss if lit else MemoryEfficientCLIPLoss)(t, normed)(ga, gb)
    assert loss.grad_fn.mec[4] == _lib.DTYPE_F32_PAIRS
    (loss * -2.0).backward()
    torch.cuda.synchronize()
    if lit:
        rl, rda = oracle.lit_loss_and_grads(a, b, t, normalized_inputs=normed, grad_output=-2.0)
        grads = [(ga.grad, rda)]
    else:
        rl, rda, rdb = oracle.clip_loss_and_grads(a, b, t, normalized_inputs=normed, grad_output=-2.0)
        grads = [(ga.grad, rda), (gb.grad, rdb)]
    le = rel_err(loss.detach().cpu(), rl) if float(rl) != 0.0 else abs(float(loss.detach()))
    ge = [max_rel(g, r) for g, r in grads]
    say(f"  loss rel {le:.2e}, grads {['%.2e' % e for e in ge]}")
    assert le <= BAR or abs(float(loss.detach()) - float(rl)) < 1e-6
    assert all(e <= BAR for e in ge)


# noise 0.3 and 0.5: pairs that match well, whose off-diagonal entries are 1e-8
# and less (stored under a scale that follows the rows' off-diagonal shares)
@pytest.mark.parametrize("n,d,t,noise", [(300, 64, 0.05, 3), (2100, 640, 0.07, 3), (4097, 192, 0.1, 3),
                                         (2100, 640, 0.05, 0.5), (1500, 256, 0.03, 0.3)])
def test_off_diagonal_sums_are_as_exact_as_in_fp32(n, d, t, noise):
    """acc_x, acc_y of mec_grad (the sums over j != i of G'_ij y^_j and their
    transpose) with both dtypes, against 64 bits."""
    lib = _lib.load()
    g = torch.Generator().manual_seed(n)
    x = torch.nn.functional.normalize(torch.randn(n, d, generator=g), dim=1)
    y = torch.nn.functional.normalize(x + noise * torch.nn.functional.normalize(torch.randn(n, d, generator=g), dim=1),
                                      dim=1)
    xh, yh = x.double(), y.double()
    e = torch.exp((xh @ yh.T - 1.0) / t)
    gm = e / e.sum(1, keepdim=True) + e / e.sum(0, keepdim=True)
    gm.fill_diagonal_(0.0)
    ref = gm @ yh, gm.T @ xh
    st = torch.cuda.current_stream().cuda_stream
    x, y = x.to(DEV), y.to(DEV)
    err = {}
    for dt in (_lib.DTYPE_F32, _lib.DTYPE_F32_PAIRS):
        ws = torch.empty(lib.mec_workspace_floats_for(n, d, dt), device=DEV)
        loss = torch.empty((), device=DEV)
        nbytes = lib.mec_grad_scratch_bytes(n, d, dt)
        scratch = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
        acc = torch.empty(n, d, device=DEV), torch.empty(n, d, device=DEV)
        _lib.call("mec_forward", x.data_ptr(), d, y.data_ptr(), d, n, d, dt, _lib.MODE_CLIP, 0, t, ws.data_ptr(),
                  loss.data_ptr(), st)
        _lib.call("mec_grad", x.data_ptr(), d, y.data_ptr(), d, n, d, dt, _lib.MODE_CLIP, 0, t, ws.data_ptr(),
                  scratch.data_ptr(), nbytes, acc[0].data_ptr(), acc[1].data_ptr(), st)
        torch.cuda.synchronize()
        err[dt] = [((a.cpu().double() - r).norm() / r.norm()).item() for a, r in zip(acc, ref)]
    say(f"off-diagonal sums n={n} d={d} T={t}: fp32 {err[0]}, pairs {err[_lib.DTYPE_F32_PAIRS]}")
    for p, f in zip(err[_lib.DTYPE_F32_PAIRS], err[_lib.DTYPE_F32]):
        assert p <= 1.1 * f


def stages(x, y, t, dt, mode):
    """acc_x, acc_y of mec_forward + mec_grad on normalized x, y."""
    lib, (n, d) = _lib.load(), x.shape
    st = torch.cuda.current_stream().cuda_stream
    ws = torch.empty(lib.mec_workspace_floats_for(n, d, dt), device=DEV)
    loss = torch.empty((), device=DEV)
    nbytes = lib.mec_grad_scratch_bytes(n, d, dt)
    scratch = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    acc = torch.empty(n, d, device=DEV), torch.empty(n, d, device=DEV)
    _lib.call("mec_forward", x.data_ptr(), d, y.data_ptr(), d, n, d, dt, mode, 0, t, ws.data_ptr(), loss.data_ptr(), st)
    _lib.call("mec_grad", x.data_ptr(), d, y.data_ptr(), d, n, d, dt, mode, 0, t, ws.data_ptr(), scratch.data_ptr(),
              nbytes, acc[0].data_ptr(), acc[1].data_ptr(), st)
    torch.cuda.synchronize()
    return acc if mode == _lib.MODE_CLIP else acc[:1]


def dense_sums(x, y, t, mode):
    """The off-diagonal sums of stages() by definition, in 64 bits, and the
    diagonal coefficient kappa."""
    xh, yh = x.double(), y.double()
    e = torch.exp((xh @ yh.T - 1.0) / t)
    gm = e / e.sum(1, keepdim=True)
    if mode == _lib.MODE_CLIP:
        gm += e / e.sum(0, keepdim=True)
    # kappa from the off-diagonal shares (as 1 - p_ii it would cancel)
    r, c = e.sum(1), e.sum(0)
    e.fill_diagonal_(0.0)
    kappa = -e.sum(1) / r - (e.sum(0) / c if mode == _lib.MODE_CLIP else 0.0)
    gm.fill_diagonal_(0.0)
    if mode == _lib.MODE_CLIP:
        return (gm @ yh, gm.T.contiguous() @ xh), kappa
    return (gm @ yh,), kappa


def features(kind, n, d):
    """Unit rows x and y, a pair's cosine about 0.3: of either sign, positive,
    or at least 0 with half the values 0 (what follows a ReLU)."""
    g = torch.Generator(device=DEV).manual_seed(n + d)
    f = {"normal": lambda v: v, "positive": torch.abs, "relu": torch.relu}[kind]
    x, z = (torch.nn.functional.normalize(f(torch.randn(n, d, generator=g, device=DEV)), dim=1) for _ in range(2))
    return x, torch.nn.functional.normalize(x + 3.0 * z, dim=1)


# (4200 and 8192 rows: one block of pairs, three and two blocks of the fp32
# kernels; 4999 with its contractions split over k; 2300 in 128 x 128 tiles; 30000
# where the fp32 kernels' blocks are shorter than the pieces of the pairs' sums)
@pytest.mark.parametrize("mode", ["clip", "lit"])
@pytest.mark.parametrize("kind,n,d", [("positive", 4200, 512), ("relu", 4200, 512), ("normal", 4200, 512),
                                      ("positive", 8192, 256), ("positive", 4999, 640), ("positive", 2300, 128),
                                      ("normal", 30000, 256)])
def test_no_further_from_64_bits_than_fp32(kind, n, d, mode):
    """Sums that grow with every term round the most, and the more the longer
    they are: those of the pairs, in pieces of the fp32 kernels' blocks, end no
    further from 64 bits than the fp32 kernels' (one sum per block of pairs:
    1.9 times as far)."""
    m = _lib.MODE_CLIP if mode == "clip" else _lib.MODE_LIT
    x, y = features(kind, n, d)
    ref, _ = dense_sums(x, y, 0.07, m)
    f, p = ([((a.double() - r).norm() / r.norm()).item() for a, r in zip(stages(x, y, 0.07, dt, m), ref)]
            for dt in (_lib.DTYPE_F32, _lib.DTYPE_F32_PAIRS))
    say(f"{kind} {mode} n={n} d={d}: fp32 {f}, pairs {p}")
    assert all(a <= b for a, b in zip(p, f))


def held_wide(ws, n):
    """The rule of pair_grad_scale on what the forward left in its workspace:
    the largest |kappa| and the smallest off-diagonal share."""
    off = (_lib.load().mec_workspace_floats(n) + 63) // 64 * 64
    kmax, smin = ws[off + 4:off + 6].cpu().numpy().astype(np.float64)
    e = 0 if kmax >= 0.5 else np.frexp(max(kmax, 2.0 ** -26))[1]
    return not 2.0 ** (14 - e) * smin >= np.sqrt(n)


def matching(kind, n, d, seed=1):
    """Unit rows whose pairs match well: all of them, all but two that are
    swapped, or all but one that has nothing to do with any other."""
    g = torch.Generator(device=DEV).manual_seed(seed)

    def unit(v):
        return torch.nn.functional.normalize(v, dim=1)

    x, z = (unit(torch.randn(n, d, generator=g, device=DEV)) for _ in range(2))
    y = unit(x + 0.4 * z)
    if kind == "swapped":
        y[[0, n // 2]] = y[[n // 2, 0]]
    elif kind == "stray":
        y[n // 3] = unit(torch.randn(1, d, generator=g, device=DEV))[0]
    return x, y


def row_errors(a, ref):
    return ((a.double() - ref).norm(dim=1) / ref.norm(dim=1)).cpu()


@pytest.mark.parametrize("mode", ["clip", "lit"])
@pytest.mark.parametrize("kind,n,d,t", [("swapped", 4097, 768, 0.03), ("swapped", 4097, 768, 0.02),
                                        ("stray", 4200, 512, 0.03), ("matching", 4200, 512, 0.02),
                                        ("swapped", 2300, 200, 0.03), ("swapped", 8192, 320, 0.04)])
def test_every_row_is_as_exact_as_in_fp32(kind, n, d, t, mode):
    """Batches whose rows' off-diagonal shares lie far apart, or are all tiny:
    under one scale the small rows' entries fell below fp16's range (4097 x 768,
    T = 0.03: nothing was left of most rows' sums).  Every row's sum on its own,
    against 64 bits."""
    m = _lib.MODE_CLIP if mode == "clip" else _lib.MODE_LIT
    x, y = matching(kind, n, d)
    ref, _ = dense_sums(x, y, t, m)
    for side in range(len(ref)):
        f, p = (row_errors(stages(x, y, t, dt, m)[side], ref[side]) for dt in (_lib.DTYPE_F32, _lib.DTYPE_F32_PAIRS))
        say(f"{kind} {mode} n={n} d={d} T={t} side {side}: rows' errors, median and largest: "
            f"fp32 {f.median():.2e} {f.max():.2e}, pairs {p.median():.2e} {p.max():.2e}")
        # (the largest of n rows: two draws of the same rounding differ)
        assert p.median() <= f.median() and p.max() <= 1.5 * f.max()


# as CASES, with the parts of the contractions (0: the default)
WIDE = [("clip", 2, 33, False, 0, 0, 0), ("clip", 31, 31, False, 3, 0, 0), ("lit", 255, 32, True, 0, 0, 0),
        ("clip", 257, 130, False, 1, 0, 0), ("lit", 513, 255, True, 0, 1, 3), ("clip", 1300, 257, False, 0, 2, 0),
        ("clip", 2049, 320, True, 5, 3, 2), ("clip", 2600, 512, False, 0, 0, 4), ("clip", 3001, 100, False, 0, 4, 8),
        ("lit", 4097, 600, False, 0, 0, 0)]


@pytest.mark.parametrize("mode,n,d,normed,pad,tb,parts", WIDE, ids=[f"{c[0]}-{c[1]}x{c[2]}" for c in WIDE])
def test_wide_matrix_against_the_definition(pairs, mode, n, d, normed, pad, tb, parts):
    """Gradient matrices that are held wide, at the edges of tiles, chunks, blocks
    and parts.  Bar, row by row: S of unit rows, sums that stay below 1, is off by
    about 2 x 2^-24 and the exponent (S - 1) / T by 2^-24 of itself (S > -0.5), an
    entry of G' by twice their sum (its E and its R), and a row that matches well
    loses up to 2 / |x^ - y^| (about 5 here) to the normalisation backward."""
    lit = mode == "lit"
    t = 0.03
    if tb:
        pairs.setenv("MEC_GRAD_BLOCK_TILES", str(tb))
    if parts:
        pairs.setenv("MEC_CONTRACT_PARTS", str(parts))
    x, y = matching("swapped" if n > 2 else "matching", n, d)
    if not normed:
        g = torch.Generator(device=DEV).manual_seed(7)
        x, y = (v * torch.exp(torch.randn(n, 1, generator=g, device=DEV)) for v in (x, y))
    wx, wy = torch.zeros(n, d + pad, device=DEV), torch.zeros(n, d + pad, device=DEV)
    wx[:, pad:], wy[:, pad:] = x, y
    gx, gy = wx[:, pad:].requires_grad_(True), wy[:, pad:].requires_grad_(not lit)
    say(f"wide {mode} n={n} d={d} normed={normed} pad={pad} blocks={tb} parts={parts}")
    loss = (MemoryEfficientLiTLoss if lit else MemoryEfficientCLIPLoss)(t, normed)(gx, gy)
    assert loss.grad_fn.mec[4] == _lib.DTYPE_F32_PAIRS
    assert held_wide(loss.grad_fn.saved_tensors[2], n)
    loss.backward()
    norms = [torch.ones(n, 1, device=DEV).double() if normed else v.double().norm(dim=1, keepdim=True) for v in (x, y)]
    xh, yh = x.double() / norms[0], y.double() / norms[1]
    sums, kappa = dense_sums(xh, yh, t, _lib.MODE_LIT if lit else _lib.MODE_CLIP)
    bar = 5 * 2 * (2 + 1.5) * 2.0 ** -24 / t
    for a, own, oth, nrm, acc in zip([gx.grad, gy.grad], [xh, yh], [yh, xh], norms, sums):
        r = (acc + kappa[:, None] * oth) / (n * t * (1 if lit else 2))
        if not normed:
            r = (r - own * (own * r).sum(1, keepdim=True)) / nrm
        e = row_errors(a, r)
        say(f"  rows' errors: median {e.median():.2e}, largest {e.max():.2e} (bar {bar:.2e})")
        assert e.max() <= bar


@pytest.mark.parametrize("ex,ey", [(118, -118), (-118, 118), (119, 119), (-100, -100)])
@pytest.mark.parametrize("mode", ["clip", "lit"])
def test_scales_at_the_ends_of_fp32(pairs, mode, ex, ey):
    """Rows that come as they are, 2^ex and 2^ey times unit rows: with the exponents
    opposed the products are those of unit rows; with both large, rows of x and y
    without a common feature (S = 0); with both small, S = 0 to fp32 too.  The
    gradients of 2^e x scale as 2^-e times those of x."""
    n, d, t = 300, 64, 0.1
    lit = mode == "lit"
    a, b = (torch.nn.functional.normalize(v, dim=1) for v in randn_pair(n, d, seed=3))
    if ex == ey:
        a[:, d // 2:] = 0
        b[:, :d // 2] = 0
    x, y = (a * 2.0 ** ex).to(DEV).requires_grad_(True), (b * 2.0 ** ey).to(DEV).requires_grad_(not lit)
    say(f"scales {mode} 2^{ex} 2^{ey}")
    loss = (MemoryEfficientLiTLoss if lit else MemoryEfficientCLIPLoss)(t, True)(x, y)
    assert loss.grad_fn.mec[4] == _lib.DTYPE_F32_PAIRS
    loss.backward()
    f = oracle.lit_loss_and_grads if lit else oracle.clip_loss_and_grads
    ref = f(a, b, t, normalized_inputs=True)
    assert rel_err(loss.detach().cpu(), ref[0]) <= BAR
    # (d loss / d x_i is a sum of rows of y)
    for g, r, e in [(x.grad, ref[1], ey)] + ([] if lit else [(y.grad, ref[2], ex)]):
        assert max_rel(g.double() * 2.0 ** -e, r) <= BAR


def test_noalloc_and_one_side(pairs):
    """mec_backward_noalloc and a frozen tower, bitwise as mec_backward with both
    sides (unsplit: each chooses its own split of the contractions)."""
    pairs.setenv("MEC_CONTRACT_PARTS", "1")
    n, d, t = 1100, 72, 0.07
    a, b = randn_pair(n, d, seed=5)
    ga, gb = a.to(DEV).requires_grad_(True), b.to(DEV).requires_grad_(True)
    loss = MemoryEfficientCLIPLoss(t)(ga, gb)
    ws = loss.grad_fn.saved_tensors[2]
    x, y = ga.detach(), gb.detach()
    dx, dy = torch.empty(n, d, device=DEV), torch.empty(n, d, device=DEV)
    _lib.call("mec_backward_noalloc", x.data_ptr(), d, y.data_ptr(), d, n, d, _lib.DTYPE_F32_PAIRS, _lib.MODE_CLIP, 1,
              t, 1.0 / t, ws.data_ptr(), None, dx.data_ptr(), dy.data_ptr(), dx.data_ptr(), dy.data_ptr(),
              torch.cuda.current_stream().cuda_stream)
    loss.backward()
    assert torch.equal(dx, ga.grad) and torch.equal(dy, gb.grad)
    for fx, fy in ((True, False), (False, True)):
        px, py = a.to(DEV).requires_grad_(fx), b.to(DEV).requires_grad_(fy)
        MemoryEfficientCLIPLoss(t)(px, py).backward()
        assert torch.equal(px.grad if fx else py.grad, ga.grad if fx else gb.grad)


def test_rule_reaches_the_module():
    os.environ.pop("MEC_F32_PAIRS", None)
    for n, d, want in [(2048, 512, _lib.DTYPE_F32), (2049, 64, _lib.DTYPE_F32), (4097, 64, _lib.DTYPE_F32_PAIRS), (4999, 640, _lib.DTYPE_F32_PAIRS)]:
        x = torch.randn(n, d, device=DEV).requires_grad_(True)
        loss = MemoryEfficientCLIPLoss()(x, torch.randn(n, d, device=DEV))
        assert loss.grad_fn.mec[4] == want, (n, d)
