"""The medium-problem GEMM kernel (csrc/gemm_mid.hip) at the edges of its tiles.

Bound per output: the bf16 rounding of the result (8 significant bits: 2^-8 |y|) and the
fp32 accumulation, at most K 2^-23 sum_k |x_k w_k| (one rounding per term, any order)."""
import numpy as np
import pytest
import torch

from gpu_util import best_times

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def dsk():
    import ds_kernels
    return ds_kernels


def _check(out, x, w, scale=None):
    xd, wd = x.double(), w.double()
    ref, room = xd @ wd.t(), xd.abs() @ wd.abs().t()
    if scale is not None:
        ref, room = ref * scale, room * scale
    err = (out.double() - ref).abs()
    assert bool((err <= 2.0 ** -8 * ref.abs() + x.shape[1] * 2.0 ** -23 * room).all()), float(err.max())


# 64 x 128, 64 x 256 and 128 x 256 tiles (by the rule: few tiles, more than a CU each, large),
# one row past a tile, one short of it, widths of one block and of a partial tile, odd
# numbers of 64-K stages
@pytest.mark.parametrize("M,N,K", [
    (65, 32, 64), (127, 96, 192), (128, 160, 128), (129, 2048, 2048), (200, 3648, 64),
    (777, 3648, 2048), (1000, 4096, 512), (1111, 3648, 2048), (2049, 2080, 1408),
    (4097, 4096, 512)])
def test_dense(dsk, M, N, K):
    g = torch.Generator().manual_seed(M + N)
    x = torch.randn(M, K + 64, generator=g).to(torch.bfloat16).to(DEV)[:, :K]   # strided rows
    w = (torch.randn(N, K, generator=g) * 0.05).to(torch.bfloat16).to(DEV)
    tiled = dsk.linear(x, dsk.tile_weights(w[None])[0])
    _check(tiled, x, w)
    assert torch.equal(tiled, dsk.linear(x, w))          # row-major weight: the same sums
    guard = torch.full((M + 2, N + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    dsk.linear(x, dsk.tile_weights(w[None])[0], out=guard[1:M + 1, :N])
    assert torch.equal(guard[1:M + 1, :N], tiled)
    assert bool((guard[0] == 7).all() and (guard[M + 1] == 7).all() and (guard[:, N:] == 7).all())


# several launches of 2^20 rows; in one, rows times blocks would pass 2^31 from 2.1 million
# rows in 64-row tiles (N = 128), from 3.0 in 128-row ones
@pytest.mark.parametrize("M,N", [((1 << 20) + 1, 128), (2200003, 128), (3100003, 256)])
def test_dense_millions_of_rows(dsk, M, N):
    g = torch.Generator(device=DEV).manual_seed(N)
    x = torch.randn(M, 64, generator=g, device=DEV, dtype=torch.bfloat16)
    w = torch.randn(N, 64, generator=g, device=DEV).mul_(0.05).to(torch.bfloat16)
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    dsk.linear(x, dsk.tile_weights(w[None])[0], out=out)
    for r in range(0, M, 400000):
        _check(out[r:r + 400000], x[r:r + 400000], w)


@pytest.mark.parametrize("M", [1, 33, 64, 200, 777, 1111, 4100])
def test_row_statistics(dsk, M):
    """linear_rowsq / linear_rowscale on 64- and 128-row tiles."""
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, 256, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(800, 256, generator=g) * 0.05).to(torch.bfloat16).to(DEV)
    wt = dsk.tile_weights(w[None])[0]
    y, ss = dsk.linear_rowsq(x, wt, 256, 768)
    _check(y, x, w)
    ref = y[:, 256:768].double().square().view(M, 2, 256).sum(-1).t()
    assert bool(((ss.double() - ref).abs() <= 256 * 2.0 ** -23 * ref).all())
    z = dsk.linear_rowscale(x, wt, ss, 512, 1e-6)
    r = torch.rsqrt(ss.double().sum(0) / 512 + 1e-6)[:, None]
    _check(z, x, w, r * (1 + 2.0 ** -20))


def test_row_statistics_of_millions_of_rows(dsk):
    """The sums of squares and the row scales of every launch's rows."""
    M = (1 << 20) + 77
    g = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randn(M, 128, generator=g, device=DEV, dtype=torch.bfloat16)
    w = torch.randn(256, 128, generator=g, device=DEV).mul_(0.05).to(torch.bfloat16)
    wt = dsk.tile_weights(w[None])[0]
    y, ss = dsk.linear_rowsq(x, wt, 0, 256)
    z = dsk.linear_rowscale(x, wt, ss, 256, 1e-6)
    for r in (slice(0, 5000), slice(M - 5000, M)):
        _check(y[r], x[r], w)
        ref = y[r].double().square().sum(-1)
        assert bool(((ss[0, r].double() - ref).abs() <= 256 * 2.0 ** -23 * ref).all())
        s = torch.rsqrt(ss[0, r].double() / 256 + 1e-6)[:, None]
        _check(z[r], x[r], w, s * (1 + 2.0 ** -20))


@pytest.mark.parametrize("T,bias", [(65, 0.0), (150, 3.0), (600, 0.0), (600, 6.0), (1400, 3.0),
                                    (3000, 0.0)])
def test_fused_layer_groups(dsk, T, bias):
    """The grouped forms in the fused layer: equal and very unequal groups (some empty, some
    of nearly T rows) against per-expert products of the routing it returns."""
    _fused_layer_groups(dsk, T, bias, 16, 4, 256, 192, 2)


@pytest.mark.parametrize("T,bias", [(500, 0.0), (700, 0.0), (700, 3.0), (1070, 0.0), (1300, 0.0),
                                    (1500, 0.0), (1500, 4.0), (2130, 0.0), (2140, 0.0)])
def test_fused_layer_groups_without_always_on(dsk, T, bias):
    """64 experts and none always on, on both sides of the row counts where whole 128-row tiles
    and the 256 x 256 kernels are taken (50, 80, 100, 128 and 200 rows per group)."""
    _fused_layer_groups(dsk, T, bias, 64, 6, 1024, 512, 0)


def test_time_of_groups_past_64_rows(dsk):
    """A layer of 800 tokens on 64 routed experts (75 rows each) in no more time than of 1000:
    GEMM1 + GEMM2 222 and 229 us; 239 and 230 when the groups took two 64-row tiles."""
    E, K, H, I = 64, 6, 2048, 1408
    g = torch.Generator().manual_seed(0)
    w1, w2 = (dsk.tile_weights((torch.randn(*s, device=DEV) * 0.02).to(torch.bfloat16))
              for s in ((E, 2 * I, H), (E, H, I)))
    x = torch.randn(1000, H, generator=g).to(torch.bfloat16).to(DEV)
    logits = torch.randn(1000, E, generator=g).to(DEV)
    few, many = best_times(*(
        lambda T=T: dsk.moe_fused_forward_logits(logits[:T], x[:T], w1, w2, K, 0, E)
        for T in (800, 1000)))
    assert few < 1.01 * many, (few, many)


def _fused_layer_groups(dsk, T, bias, E, K, H, I, nsh):
    g = torch.Generator().manual_seed(T)
    rnd = lambda *s, std=0.08: (torch.randn(*s, generator=g) * std).to(torch.bfloat16).to(DEV)  # noqa: E731
    x, wg = rnd(T, H, std=1.0), rnd(E, H)
    w1, w2 = rnd(E + nsh, 2 * I, H), rnd(E + nsh, H, I)
    logits = (x.float() @ wg.float().t()
              - bias * torch.log(torch.arange(1.0, E + 1)).to(DEV)).contiguous()
    out, (idx, wt, off) = dsk.moe_fused_forward_logits(
        logits, x, dsk.tile_weights(w1), dsk.tile_weights(w2), K, nsh, E, return_routing=True)
    ref = torch.zeros(T, H, dtype=torch.float64, device=DEV)
    for e in range(E + nsh):
        t, k = (idx == e).nonzero(as_tuple=True) if e < E else (torch.arange(T, device=DEV), None)
        h = x[t].double() @ w1[e].double().t()
        h = torch.nn.functional.silu(h[:, :I]) * h[:, I:]
        y = h @ w2[e].double().t()
        ref.index_add_(0, t, y if k is None else y * wt[t, k].double()[:, None])
    counts = (off[1:] - off[:-1]).cpu().numpy()
    np.testing.assert_array_equal(counts, np.bincount(idx.cpu().numpy().ravel(), minlength=E))
    # bf16 h, y and out: three roundings of 2^-8 on sums that add in quadrature
    err = (out.double() - ref).norm() / ref.norm()
    assert float(err) <= 2.0 ** -7, float(err)
    assert torch.equal(out, dsk.moe_fused_forward_logits(
        logits, x, dsk.tile_weights(w1), dsk.tile_weights(w2), K, nsh, E))


@pytest.mark.parametrize("counts", [[65], [64, 0, 1, 33, 31], [40] * 8, [127, 128, 129, 0, 65],
                                    [300, 2, 0, 70], [500, 20, 20, 20]])
@pytest.mark.parametrize("I,K", [(96, 64), (192, 192)])
def test_row_major_groups(dsk, counts, I, K):
    """The ops on row-major weights: 64- and 128-row tiles, SwiGLU from the halves of a block,
    uncovered rows zero (3 before the first group, 2 after the last)."""
    E, S = len(counts), sum(counts) + 5
    g = torch.Generator().manual_seed(S + I)
    rnd = lambda *s: (torch.randn(*s, generator=g) * 0.3).to(torch.bfloat16).to(DEV)  # noqa: E731
    x, w1, w2 = rnd(S, K), rnd(E, 2 * I, K), rnd(E, K, I)
    off = torch.tensor(np.concatenate([[3], 3 + np.cumsum(counts)]), dtype=torch.int32, device=DEV)
    torch.full((S, 2 * I), float("nan"), dtype=torch.bfloat16, device=DEV)   # stale memory
    gu = dsk.moe_gemm1(x, w1, off)
    h = dsk.moe_gemm1_swiglu(x, w1, off)
    y = dsk.moe_gemm2(h, w2, off) if I % 64 == 0 else None
    ends = off.cpu().tolist()
    for e in range(E):
        r = slice(ends[e], ends[e + 1])
        if ends[e] == ends[e + 1]:
            continue
        _check(gu[r], x[r], w1[e])
        if y is not None:
            _check(y[r], h[r], w2[e])
        a = x[r].double() @ w1[e].double().t()
        ref = torch.nn.functional.silu(a[:, :I]) * a[:, I:]
        assert float((h[r].double() - ref).norm() / ref.norm()) <= 2.0 ** -8
    for t in (gu, h) + (() if y is None else (y,)):
        assert bool((t[:3] == 0).all() and (t[S - 2:] == 0).all())


def test_row_major_overlapping_offsets(dsk):
    """Offsets that decrease: a group's rows are [off[g], max(off[g], off[g + 1])), a row of
    two groups may come from either, and rows outside [off[0], off[G]) that some group
    covers are not zeroed."""
    off = torch.tensor([5, 130, 90, 300, 290], dtype=torch.int32, device=DEV)
    g = torch.Generator().manual_seed(0)
    x = torch.randn(320, 128, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(4, 64, 128, generator=g) * 0.1).to(torch.bfloat16).to(DEV)
    out = dsk.moe_gemm1(x, w, off)
    _check(out[5:90], x[5:90], w[0])
    _check(out[130:300], x[130:300], w[2])
    assert bool((out[:5] == 0).all() and (out[300:] == 0).all())


@pytest.mark.parametrize("G,M", [(8, 1000), (16, 1000), (30, 1900)])
def test_row_major_offsets_that_overlap_whole_groups(dsk, G, M):
    """Offsets 0, M, 0, M, ...: every other group is all M rows, so the tiles are several times
    the grid and a workgroup runs tile after tile, the staging of one against the DMA of the
    next. All groups have the same weights, so each row has one right value."""
    off = torch.tensor(([0, M] * G)[:G + 1], dtype=torch.int32, device=DEV)
    g = torch.Generator().manual_seed(G)
    rnd = lambda *s: (torch.randn(*s, generator=g) * 0.2).to(torch.bfloat16).to(DEV)  # noqa: E731
    w1, w2 = rnd(384, 192).expand(G, 384, 192).contiguous(), rnd(256, 192).expand(G, 256, 192).contiguous()
    x = rnd(M, 192)
    rows = 64 if M // G <= 70 else 128
    tiles = (G // 2) * -(-M // rows)
    assert tiles > -(-M // rows) + G + 8      # more than the grid, rounded up to the XCDs
    for _ in range(3):
        gu = dsk.moe_gemm1(x, w1, off)
        _check(gu, x, w1[0])
        a = x.double() @ w1[0].double().t()
        ref = torch.nn.functional.silu(a[:, :192]) * a[:, 192:]
        h = dsk.moe_gemm1_swiglu(x, w1, off)
        # rounding of h (2^-8), the hardware exp and reciprocal and K fp32 roundings: per element
        room = a[:, :192].abs() * a[:, 192:].abs()
        assert bool(((h.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -12 * (room + 1)).all())
        y = dsk.moe_gemm2(h, w2, off)
        _check(y, h, w2[0])


@pytest.mark.parametrize("counts", [[131, 160, 192, 224, 256, 300], [257, 385, 512, 97, 33]])
@pytest.mark.parametrize("I,K", [(96, 64), (192, 320)])
def test_row_major_large_groups(dsk, counts, I, K):
    """Row-major groups past the medium-problem kernel: the 8-wave kernel with one to eight
    row blocks in a tile, and odd numbers of 64-K stages."""
    E, S = len(counts), sum(counts)
    g = torch.Generator().manual_seed(S + I)
    rnd = lambda *s: (torch.randn(*s, generator=g) * 0.3).to(torch.bfloat16).to(DEV)  # noqa: E731
    x, w1 = rnd(S, K), rnd(E, 2 * I, K)
    off = torch.tensor(np.concatenate([[0], np.cumsum(counts)]), dtype=torch.int32, device=DEV)
    gu, h = dsk.moe_gemm1(x, w1, off), dsk.moe_gemm1_swiglu(x, w1, off)
    ends = off.cpu().tolist()
    for e in range(E):
        r = slice(ends[e], ends[e + 1])
        _check(gu[r], x[r], w1[e])
        a = x[r].double() @ w1[e].double().t()
        ref = torch.nn.functional.silu(a[:, :I]) * a[:, I:]
        assert float((h[r].double() - ref).norm() / ref.norm()) <= 2.0 ** -8


def test_row_major_partial_tiles_time(dsk):
    """64 groups of 375 rows (6 of 8 row blocks a tile) in less time than of 512 (full tiles):
    335 and 380 us; 413 and 391 when the partial tile's loop reloaded spilled registers."""
    w = (torch.randn(64, 2816, 2048, device=DEV) * 0.02).to(torch.bfloat16)
    x = torch.randn(64 * 512, 2048, device=DEV).to(torch.bfloat16)
    offs = [(torch.arange(65, device=DEV) * rows).int() for rows in (375, 512)]
    part, full = best_times(*(lambda o=o, r=r: dsk.moe_gemm1(x[:64 * r], w, o)
                              for o, r in zip(offs, (375, 512))))
    assert part < 0.98 * full, (part, full)
