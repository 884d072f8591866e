"""The one-call forms of the MLA module against the same kernels issued op by op: bitwise."""
import dataclasses

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def setup():
    import ds_kernels as dsk
    from ds_kernels import mla as dm
    from ds_kernels import synthetic as syn
    w = syn.mla_weights()
    w["kva_norm"] = 1 + 0.1 * torch.randn(512, generator=torch.Generator().manual_seed(1))
    W = dm.MLAWeights.from_tensors(w, torch.device(DEV, 0))
    cos, sin = (t.to(torch.bfloat16).to(DEV) for t in dm.yarn_cos_sin(700))
    return dsk, dm, W, dsk.AbsorbedMLAWeights.from_mla(W), cos, sin


def _x(*shape, seed=0):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g).to(torch.bfloat16).to(DEV)


@pytest.mark.parametrize("b,s,masked,ids", [(1, 1, False, False), (2, 77, False, False),
                                            (3, 130, True, False), (2, 60, False, True)])
def test_forward(setup, b, s, masked, ids):
    dsk, dm, W, _, cos, sin = setup
    x = _x(b, s, 2048, seed=b + s)
    mask = pid = None
    if masked:
        mask = torch.zeros(b, 1, s, s, device=DEV, dtype=torch.bfloat16)
        mask[:, :, :, s - 9:] = float("-inf")
    if ids:
        pid = torch.stack([torch.randperm(s) for _ in range(b)]).to(DEV)
    out = dm.mla_forward(x, W, cos, sin, attention_mask=mask, position_ids=pid)
    q, kv, kva, _ = dm._projection_rows(x, W, 1e-6, with_latent=False)
    cs, sn = dm.rope_tables_for(cos, sin, s, pid)
    ct, st = ((t if t.dim() == 3 else t[None])[:, None].expand(b, 1, s, 64) for t in (cs, sn))
    k_rot = dsk.ops.rope_single(kva[:, None, :, 512:], ct, st)[:, 0]
    o = dsk.mla_prefill_attention(q, kv, k_rot, cs, sn, W.softmax_scale, causal=mask is None,
                                  mask=mask)
    assert torch.equal(out, dsk.linear(o, W.o))
    # strided activations, and weights whose o is not tiled (the op-by-op path)
    wide = torch.zeros(b, s, 2048 + 64, dtype=torch.bfloat16, device=DEV)
    wide[..., :2048] = x
    assert torch.equal(out, dm.mla_forward(wide[..., :2048], W, cos, sin, attention_mask=mask,
                                           position_ids=pid))
    W_rm = dataclasses.replace(W, o=dsk.untile_weights(W.o[None])[0])
    ref = dm.mla_forward(x, W_rm, cos, sin, attention_mask=mask, position_ids=pid)
    assert float((out.double() - ref.double()).norm() / ref.double().norm()) <= 2.0 ** -8


@pytest.mark.parametrize("b,n", [(1, 1), (1, 3), (4, 1), (5, 1), (1, 64), (64, 1), (33, 1)])
def test_decode_step(setup, b, n):
    dsk, dm, W, A, cos, sin = setup
    prefix = 150
    caches = [dsk.LatentKVCache.for_inference(b, max_seq=prefix + 2 * n) for _ in range(2)]
    for c in caches:
        dsk.mla_decode_forward(_x(b, prefix, 2048, seed=3), W, c, cos, sin, A)
    for step in range(2):
        x = _x(b, n, 2048, seed=10 + step)
        out = dsk.mla_decode_forward(x, W, caches[0], cos, sin, A)
        # op by op on the other cache
        c, T = caches[1], b * n
        rows = c.append_slots(n)
        L = c.current_len
        q = torch.empty(T, 3072, dtype=torch.bfloat16, device=DEV)
        dst = rows[0] if b == 1 else rows[:, 0]
        few = T <= 4
        if few:
            dsk.linear_rows(x.view(T, 2048), W.q_kva, out=q, out1=dst, n_split=3072)
        else:
            dsk.linear_split(x.view(T, 2048), W.q_kva, q, dst)
        q4 = q.view(T, 16, 192)
        batched = dsk.linear_rows if few else dsk.linear_batched
        q_abs = batched(q4[..., :128].transpose(0, 1), A.uk_tiled)
        lat, kpe = c.get(L)
        o_lat = dsk.mla_decode_attention(q_abs.transpose(0, 1), q4[..., 128:], lat, kpe, cos, sin,
                                         W.softmax_scale, k_rope=c.k_rope[:, :L],
                                         rope_len=c.rope_len)
        c._rope_len = L
        o = torch.empty(T, 2048, dtype=torch.bfloat16, device=DEV)
        batched(o_lat.transpose(0, 1), A.uv_tiled, out=o.view(T, 16, 128).transpose(0, 1))
        ref = (dsk.linear_rows if few else dsk.linear)(o, W.o).view(b, n, 2048)
        assert torch.equal(out, ref)
        assert torch.equal(caches[0].rows, caches[1].rows)
        assert caches[0].rope_len == caches[1].rope_len == L


@pytest.mark.parametrize("dims", [(128, 128), (128, 64), (64, 64)])
@pytest.mark.parametrize("b,n,launches", [(1, 1, 4), (3, 1, 4), (1, 7, 1), (33, 1, 1)])
def test_decode_step_op_by_op(monkeypatch, dims, b, n, launches):
    """Steps that the C call does not take (other head dims; an o_proj that is not tiled) keep
    the decode kernels: all projections on the row kernel up to 4 tokens where the weights are
    tiled, q and kv_a in one launch up to 64. Against mla_forward on the whole sequence: bf16
    roundings of the latent, of the absorbed weights and of four intermediates, 2e-2 as for
    the other decode steps."""
    import ds_kernels as dsk
    from ds_kernels import mla as dm
    from ds_kernels import ops
    from ds_kernels import synthetic as syn
    nope, vd = dims
    w = syn.mla_weights(H=512, nope=nope, v_dim=vd)
    W = dataclasses.replace(dm.MLAWeights.from_tensors(w, torch.device(DEV, 0)), nope=nope, v_dim=vd)
    A = dsk.AbsorbedMLAWeights.from_mla(W)
    if dims == (128, 128):
        W = dataclasses.replace(W, o=dsk.untile_weights(W.o[None])[0])
    if dims != (128, 64):     # the row kernel takes tiled weights with inner sizes of 128
        launches = 1
    cos, sin = (t.to(torch.bfloat16).to(DEV) for t in dm.yarn_cos_sin(64))
    calls = []
    for name in ("linear_rows", "linear_split"):
        real = getattr(ops, name)
        monkeypatch.setattr(ops, name,
                            lambda *a, _f=real, _n=name, **k: (calls.append(_n), _f(*a, **k))[1])
    x = _x(b, 20 + n, 512, seed=b + n)
    cache = dsk.LatentKVCache.for_inference(b, max_seq=20 + n)
    dsk.mla_decode_forward(x[:, :20], W, cache, cos, sin, A)
    calls.clear()
    out = dsk.mla_decode_forward(x[:, 20:].contiguous(), W, cache, cos, sin, A)
    assert calls == (["linear_rows"] * 4 if launches == 4 else ["linear_split"])
    ref = dm.mla_forward(x, W, cos, sin)[:, 20:].double()
    assert float((out.double() - ref).abs().max() / ref.abs().max()) <= 2e-2
