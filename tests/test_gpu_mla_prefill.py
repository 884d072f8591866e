"""mla_prefill_attention against 64-bit attention of the same bf16 operands.

Bound per output element: bf16 keeps 8 significant bits, so rounding to nearest is off
by at most 2^-8 of the value. The probabilities are rounded to bf16 (at most 2^-8
sum_j p_j |v_j|) and the result once more (2^-8 |o|), together below 2^-7 sum_j p_j
|v_j|; the fp32 scores and sums add less than 1e-3 of that."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
SCALE = 0.1147


@pytest.fixture(scope="module")
def dsk():
    import ds_kernels
    return ds_kernels


def _operands(b, n, L, heads, seed, ld_extra=64):
    from ds_kernels.mla import yarn_cos_sin
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)  # noqa: E731
    q = rnd(b, n, heads * 192 + ld_extra)[..., :heads * 192]     # strided rows
    kv = rnd(b, L, heads * 256)
    kr = rnd(b, L, 192)[..., 64:128]                              # a view of cache rows
    cos, sin = (t.to(torch.bfloat16).to(DEV) for t in yarn_cos_sin(L))
    return q, kv, kr, cos, sin


def _reference(q, kv, kr, cos, sin, heads, causal, mask):
    """(output, sum_j p_j |v_j|) in fp64, q_pe rotated by the RoPE kernel."""
    from ds_kernels import ops
    b, n, _ = q.shape
    L = kv.shape[1]
    q4 = q.reshape(b, n, heads, 192).transpose(1, 2)
    tab = [(t if t.dim() == 3 else t[None])[:, L - n:L].expand(b, n, 64)[:, None].contiguous()
           for t in (cos, sin)]
    q_rot = ops.rope_single(q4[..., 128:], *tab).double()
    kv4 = kv.view(b, L, heads, 256).transpose(1, 2).double()
    kn, v = kv4[..., :128], kv4[..., 128:]
    s = q4[..., :128].double() @ kn.transpose(-1, -2)
    s = (s + q_rot @ kr.double()[:, None].transpose(-1, -2)) * SCALE
    if mask is not None:
        s = s + mask.double()
    if causal:
        hide = torch.ones(n, L, dtype=torch.bool, device=DEV).triu_(L - n + 1)
        s = s.masked_fill(hide, float("-inf"))
    p = torch.softmax(s, -1)
    back = lambda t: t.transpose(1, 2).reshape(b, n, heads * 128)  # noqa: E731
    return back(p @ v), back(p @ v.abs())


def _check(out, ref, room):
    nan = torch.isnan(ref)
    assert torch.equal(torch.isnan(out), nan)
    err = (out.double() - ref).abs()[~nan]
    assert bool((err <= (2.0 ** -7 * 1.001) * room[~nan] + 1e-6).all()), float(err.max())


# tile and block edges of the 128-query kernel, and (b * heads * blocks >= 256) the
# 256-query one; one query, odd lengths, queries after a cached prefix
@pytest.mark.parametrize("b,n,L,heads", [
    (1, 1, 1, 2), (2, 31, 31, 3), (1, 63, 64, 2), (1, 65, 65, 2), (2, 128, 128, 1),
    (1, 129, 200, 2), (3, 257, 257, 2), (1, 300, 1111, 4), (1, 1, 513, 2),
    (16, 70, 70, 16), (16, 257, 259, 8), (8, 256, 320, 32)])
def test_causal(dsk, b, n, L, heads):
    ops_in = _operands(b, n, L, heads, n + L)
    out = dsk.mla_prefill_attention(*ops_in, SCALE, heads=heads)
    _check(out, *_reference(*ops_in, heads, True, None))
    assert torch.equal(out, dsk.mla_prefill_attention(*ops_in, SCALE, heads=heads))


def test_sequence_of_more_than_4_gib(dsk):
    """Key rows 16 KB apart: 270000 of them span 4.4 GB."""
    n, L, heads = 40, 270000, 2
    q, _, kr, cos, sin = _operands(1, n, L, heads, 11)
    kv = torch.empty(1, L, 8192, dtype=torch.bfloat16, device=DEV)[..., :heads * 256]
    kv.copy_(torch.randn(1, L, heads * 256, device=DEV))
    out = dsk.mla_prefill_attention(q, kv, kr, cos, sin, SCALE, heads=heads)
    _check(out, *_reference(q, kv, kr, cos, sin, heads, True, None))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", ["b1qk", "bhqk", "11qk", "k", "bhqk_strided"])
@pytest.mark.parametrize("b,n,L", [(2, 70, 77), (16, 130, 131)])
def test_additive_mask(dsk, dtype, shape, b, n, L):
    heads = 2 if b == 2 else 16
    g = torch.Generator().manual_seed(b + L)
    dims = {"b1qk": (b, 1, n, L), "bhqk": (b, heads, n, L), "11qk": (1, 1, n, L), "k": (L,),
            "bhqk_strided": (b, heads, L, n)}[shape]
    mask = torch.randn(*dims, generator=g)
    mask[torch.rand(*dims, generator=g) < 0.3] = float("-inf")
    if shape == "b1qk":
        mask[0, 0, 3] = float("-inf")                        # no key at all: NaN rows
        mask[1, 0, 5] = torch.finfo(dtype).min               # all at the lowest: uniform
        mask[1, 0, 6] = torch.finfo(dtype).min               # one key beside the lowest
        mask[1, 0, 6, L - 1] = 0.5
    mask = mask.to(dtype).to(DEV)
    if shape == "bhqk_strided":
        mask = mask.transpose(-1, -2)
    ops_in = _operands(b, n, L, heads, 7)
    out = dsk.mla_prefill_attention(*ops_in, SCALE, heads=heads, causal=False, mask=mask)
    if shape == "b1qk":   # 64 bits would still tell lowest + score apart: fp32 does not
        lowest = mask[1, 0, 5, 0].double()
        m64 = mask.double()
        m64[1, 0, 5] = 0
        ref, room = _reference(*ops_in, heads, False, m64)
        v = ops_in[1].view(b, L, heads, 256)[1, :, :, 128:].double().mean(0).flatten()
        assert lowest < -1e38
        assert bool(((out[1, 5].double() - v).abs() <= 2.0 ** -7).all())
        keep = torch.ones(b, n, dtype=torch.bool, device=DEV)
        keep[1, 5] = False
        _check(out[keep], ref[keep], room[keep])
    else:
        _check(out, *_reference(*ops_in, heads, False, mask))


def test_tables_per_batch_entry_and_causal_with_mask(dsk):
    b, n, L, heads = 2, 40, 90, 2
    q, kv, kr, cos, sin = _operands(b, n, L, heads, 3)
    perm = torch.stack([torch.randperm(L) for _ in range(b)]).to(DEV)
    cos, sin = cos[perm], sin[perm]
    mask = torch.zeros(b, 1, 1, L, device=DEV)
    mask[1, ..., :5] = float("-inf")
    out = dsk.mla_prefill_attention(q, kv, kr, cos, sin, SCALE, heads=heads, mask=mask)
    _check(out, *_reference(q, kv, kr, cos, sin, heads, True, mask))


def test_non_finite_scores(dsk):
    """A NaN or infinite key makes the rows that see it NaN and leaves the others."""
    q, kv, kr, cos, sin = _operands(1, 96, 96, 1, 5)
    for bad in (float("nan"), float("inf")):
        kv2 = kv.clone()
        kv2[0, 50, 3] = bad
        out = dsk.mla_prefill_attention(q, kv2, kr, cos, sin, SCALE, heads=1)
        ref, room = _reference(q, kv2, kr, cos, sin, 1, True, None)
        finite = ~torch.isnan(ref)
        assert torch.equal(torch.isnan(out[0, :50]), torch.zeros_like(out[0, :50]).bool())
        err = (out.double() - ref).abs()[finite]
        assert bool((err <= (2.0 ** -7 * 1.001) * room[finite] + 1e-6).all())
        assert bool(torch.isnan(out)[~finite].all())
