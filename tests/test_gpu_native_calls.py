"""The native forms of the per-layer calls against their Python forms: the same
kernels on the same operands, so every output, gradient and cache row is equal
bit for bit; forms that the native calls do not take (another layout, batch,
gate or seed type; transforms) and errors are the Python forms' own."""
import importlib

import pytest
import torch
import torch.utils.checkpoint
from torch.autograd import forward_ad

from gpu_helpers import chunk_layout, qkv

rope = importlib.import_module("mtp-glora_amd.rope")

DTYPES = [torch.bfloat16, torch.float16, torch.float32]


def both(mga, monkeypatch, run):
    """run() through the native calls and through the Python forms; returns (name, taken) of the native calls."""
    taken = []
    native = mga._lib.native

    def spy(name, *args):
        r = native(name, *args)
        taken.append((name, r is not None))
        return r

    with monkeypatch.context() as m:
        m.setattr(mga._lib, "native", spy)
        a = run()
    with monkeypatch.context() as m:
        m.setattr(mga._lib, "native", lambda *args: None)
        b = run()
    assert len(a) == len(b)
    for i, (x, y) in enumerate(zip(a, b)):
        assert (x is None) == (y is None), i
        if x is not None:
            assert x.shape == y.shape and x.stride() == y.stride() and x.dtype == y.dtype, i
            assert torch.equal(torch.nan_to_num(x.float()), torch.nan_to_num(y.float())), i
            assert x.requires_grad == y.requires_grad, i
    return taken


def grads(outs, ins, douts):
    return list(torch.autograd.grad(outs, ins, douts, allow_unused=True))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("form", ["staged", "keys", "query_only", "no_grad", "strided", "expanded_grad",
                                  "one_row_grad", "far_rows_grad"])
def test_attention_and_cache(mga, dev, monkeypatch, dtype, form):
    P, Hq, Hkv, D = 37, 4, 2, 64
    seq = chunk_layout(65, 5, 3, P, seed=1, pad=2)
    S = len(seq.gate)
    q, k, v, kp, vp, do = qkv(S, P, Hq, Hkv, D, dtype, dev, seed=1, std=1.0)
    mask = mga.build_mtp_block_mask(torch.tensor(seq.gate, device=dev)[None], P)

    def run():
        if form == "strided":   # a layout that both forms copy, and the one that the model's projections have
            qq = q.transpose(2, 3).contiguous().transpose(2, 3).detach().requires_grad_()
        else:
            qq = q.transpose(1, 2).contiguous().transpose(1, 2).detach().requires_grad_(form != "no_grad")
        kk, vv = (t.detach().clone().requires_grad_(form not in ("no_grad", "query_only")) for t in (k, v))
        cache = mga.StreamingKVCache(capacity=P + S, num_layers=1, num_kv_heads=Hkv, head_dim=D, dtype=dtype, device=dev)
        cache.append_prefix([kp], [vp])
        if form == "keys":
            kf, vf = torch.cat([kp, kk], 2), torch.cat([vp, vv], 2)
        else:
            kf, vf = cache.update(kk, vv, 0)
        version = cache.key_buffer(0)._version
        o, lse = mga.attention.mtp_attention(qq, kf, vf, mask)
        out = [o, lse, kf, vf, torch.tensor(version)]
        if form == "no_grad":
            return out
        d = torch.ones((), device=dev, dtype=dtype).expand(o.shape) if form == "expanded_grad" else do
        if form == "one_row_grad":    # as the gradient of o.sum(1)
            d = do[:, :1].expand(o.shape)
        if form == "far_rows_grad":
            d = torch.empty(S << 23, device=dev, dtype=dtype).as_strided(o.shape, (S << 23, 1 << 23, D, 1)).copy_(do)
        ins = [t for t in (qq, kk, vv) if t.requires_grad]
        if form.endswith("_grad"):
            dense = torch.autograd.grad(o, ins, do.new_empty(o.shape).copy_(d), retain_graph=True)
            assert all(torch.equal(a, b) for a, b in zip(dense, torch.autograd.grad(o, ins, d, retain_graph=True)))
        return [t.detach() if t.dim() else t for t in out] + grads(o, ins, d) + list(grads(kf, [kk], kf.detach())
                                                                                      if kf.requires_grad else [])

    taken = both(mga, monkeypatch, run)
    assert ("attention", form != "strided") in taken
    assert form == "keys" or ("update_kv", True) in taken


@pytest.mark.gpu
def test_attention_errors_and_hooks(mga, dev, monkeypatch):
    P, Hq, Hkv, D = 0, 2, 1, 64
    seq = chunk_layout(40, 3, 3, P, seed=1, pad=0)
    S = len(seq.gate)
    q, k, v, _, _, do = qkv(S, P, Hq, Hkv, D, torch.bfloat16, dev, seed=1, std=1.0)
    mask = mga.build_mtp_block_mask(torch.tensor(seq.gate, device=dev)[None], P)
    attend = mga.attention.mtp_attention
    qq = q.detach().requires_grad_()
    with pytest.raises(RuntimeError, match="functorch"):
        torch.vmap(lambda t: attend(t, k, v, mask)[0])(q[None])
    assert mga._lib.native("soft_ce", q[0, :1], q[0, :1]) is not None   # a transform that has ended changes nothing
    o, lse = attend(qq, k, v, mask)
    with pytest.raises(NotImplementedError, match="LSE"):
        lse.sum().backward()
    o, _ = attend(qq, k, v, mask)
    o.backward(do)
    with pytest.raises(RuntimeError, match="second time"):
        o.backward(do)
    kk = k.clone()
    o, _ = attend(qq, kk, v, mask)
    kk.add_(1)
    with pytest.raises(RuntimeError, match="inplace"):
        o.backward(do)
    # saved tensors pass through the hooks, and a checkpointed call stops its recomputation early
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t, lambda t: t):
        attend(qq, k, v, mask)
    assert len(packed) == 5
    qq.grad = None
    attend(qq, k, v, mask)[0].backward(do)
    want, qq.grad = qq.grad, None
    torch.utils.checkpoint.checkpoint(lambda t: attend(t, k, v, mask)[0], qq, use_reentrant=False).backward(do)
    assert torch.equal(qq.grad, want)
    with forward_ad.dual_level(), pytest.raises(Exception, match="jvp"):
        attend(forward_ad.make_dual(q, q), k, v, mask)
    with pytest.raises(RuntimeError, match="GPU tensor"):
        attend(q.cpu(), k.cpu(), v.cpu(), mask)
    cache = mga.StreamingKVCache(capacity=S - 1, num_layers=1, num_kv_heads=Hkv, head_dim=D, dtype=q.dtype, device=dev)
    with pytest.raises(mga._lib.CapacityError):
        cache.update(k, v, 0)
    # an error of the library inside a native backward is the package's own exception
    x, w, a, b = (torch.zeros(n, m, device=dev, dtype=q.dtype) for n, m in ((8, 128), (96, 128), (16, 128), (96, 16)))

    def misaligned(t):
        return torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)

    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, misaligned):
        y = mga.gated_lora_linear(x, w, a.requires_grad_(), b, None, 1.0, 0.5)
        with pytest.raises(mga._lib.MGAError, match="not 16-byte aligned"):
            y.sum().backward()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("S,Hq,Hkv,D", [(1, 1, 1, 64), (33, 6, 2, 128)])
def test_norm_rope_stage(mga, dev, monkeypatch, dtype, S, Hq, Hkv, D):
    g = torch.Generator(dev).manual_seed(2)
    qkv_ = torch.randn(1, S, (Hq + 2 * Hkv) * D, device=dev, generator=g).to(dtype)
    qw, kw = (torch.randn(D, device=dev, generator=g).to(dtype) for _ in range(2))
    cos, sin = (torch.randn(1, S, D, device=dev, generator=g).to(dtype) for _ in range(2))
    gq, gk, gv = (torch.randn(1, h, S, D, device=dev, generator=g).to(dtype) for h in (Hq, Hkv, Hkv))
    idx = torch.arange(0, S, 2, device=dev, dtype=torch.int32)

    def run():
        x = qkv_.detach().clone().requires_grad_()
        q, k, v = (t.unflatten(2, (-1, D)) for t in x.split([Hq * D, Hkv * D, Hkv * D], 2))
        cache = mga.StreamingKVCache(capacity=2 * S + 3, num_layers=1, num_kv_heads=Hkv, head_dim=D, dtype=dtype, device=dev)
        cache.key_buffer(0).zero_(), cache.value_buffer(0).zero_()
        cache.prefix_len = 3
        qe, ke, ve = rope.qk_norm_rope_stage(q, k, v, qw, kw, cos, sin, 1e-6, cache, 0)
        kf, vf = cache.update(ke, ve, 0)
        outs = [t.detach().clone() for t in (qe, ke, ve, kf, vf)]
        dx = grads([qe, ke, ve], [x], [gq, gk, gv])
        dx += grads([rope.qk_norm_rope_stage(q, k, v, qw, kw, cos, sin, 1e-6, cache, 0)[2]], [v], [gv])
        cache.commit_regular(idx, idx.numel())
        return outs + dx + [cache.key_buffer(0).clone(), cache.value_buffer(0).clone()]

    taken = both(mga, monkeypatch, run)
    assert ("norm_rope_stage", True) in taken and ("update_kv", True) in taken


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("x_form", ["3d", "rows", "transposed", "misaligned"])
@pytest.mark.parametrize("gate_form", [None, "int64", "float", "host"])
def test_gated_lora(mga, dev, monkeypatch, dtype, x_form, gate_form):
    S, K, N, r = 37, 256, 96, 16
    g = torch.Generator(dev).manual_seed(3)
    w, a, b = (torch.randn(*s, device=dev, generator=g).to(dtype) * 0.1 for s in ((N, K), (r, K), (N, r)))
    x0 = torch.randn(S, K + 16, device=dev, generator=g).to(dtype)
    gate = (torch.arange(S, device=dev) % 3 == 0).to(torch.float32 if gate_form == "float" else torch.int64)[None]
    gate = None if gate_form is None else gate.cpu() if gate_form == "host" else gate
    dy = torch.randn(S, N, device=dev, generator=g).to(dtype)

    def run():
        x = x0.detach().clone().requires_grad_()
        aa, bb = a.clone().requires_grad_(), b.clone().requires_grad_()
        xx = {"3d": x[:, :K].contiguous()[None], "rows": x[:, :K], "misaligned": x[:, 1:K + 1],
              "transposed": x[:, :K].t().contiguous().t()}[x_form]
        y = mga.gated_lora_linear(xx, w, aa, bb, gate, 2.0, 0.1, seed=-5)
        return [y.detach()] + grads(y, [x, aa, bb], dy.view(y.shape)) + grads(
            mga.gated_lora_linear(xx.detach(), w, aa, b, gate, 2.0, 0.0), [aa],
            torch.ones((), device=dev, dtype=dtype).expand(y.shape))

    taken = both(mga, monkeypatch, run)
    assert set(taken) == {("gated_lora", x_form in ("3d", "rows") and gate_form != "host")}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("form", ["plain", "strided", "batch", "columns"])
def test_soft_ce(mga, dev, monkeypatch, dtype, form):
    g = torch.Generator(dev).manual_seed(4)
    x0, t0 = (torch.randn(2, 6, 1003, device=dev, generator=g).to(dtype) for _ in range(2))

    def run():
        x, t = x0.clone().requires_grad_(), t0
        xx, tt = {"plain": (x[:1], t[:1]), "strided": (x[:1, 1:5:2], t[:1, 1:5:2]), "batch": (x, t),
                  "columns": (x[:1, :, ::2], t[:1, :, ::2])}[form]
        loss = mga.StableSoftCrossEntropy.apply(xx, tt)
        return [loss.detach()] + grads(loss * 3, [x], None)

    taken = both(mga, monkeypatch, run)
    assert taken == [("soft_ce", form in ("plain", "strided"))]
    with pytest.raises(ValueError):
        mga.StableSoftCrossEntropy.apply(x0[:1], t0[:1, :, :5])
