"""HIP / hipBLASLt gated LoRA layer (mga_gated_lora_*) against the float64
oracle (oracle/gated_lora.py, pinned by tests/test_oracle_gated_lora.py) on the
same bf16 inputs, the mask included.

Tolerances follow the bf16 roundings on each path (u = 2^-8 covers two
roundings of 2^-9):
* y: the rank-r term (whose activations t are rounded) is rounded, the base
  product accumulated onto it and the sum rounded:
  |y - y*| <= u (|y*| + |x W^T| + s g |h A^T| |B|^T) + 1e-5 max|y*|,
  plus, with dropout, the rounding of the dropout output h = T(x / (1 - p))
  carried through both products without cancellation: u/2 s g (|h| |A|^T) |B|^T
  (at rank 8 a few terms carry it and it alone exceeds the first bound);
* dX: the LoRA term goes through three roundings (u = dY B, d_a A, the
  dropout scaling), the base gradient dY W is accumulated onto it and the sum
  is rounded:
  |dX - dX*| <= u (|dX*| + |dY W| + 2 |d_a| |A| / (1 - p)) + 1e-5 max|dX*|;
* dA = d_a^T h and dB = dY^T t (sums over the S rows of rounded factors):
  |d - d*| <= u (|d*| + |a|^T |b|) with |a|^T |b| the sum of absolute products;
* the dropout output h equals the oracle's keep mask times T(x / (1 - p)) bit
  for bit.
The full Qwen3-8B qkv shape (S = 5120) is compared with an fp32 torch
reference on the GPU under the same bounds.

fp16 and fp32 layers (the reference's other model dtypes, args.py:15) run the
general path (hipBLASLt products in the layer's dtype, HIP dropout and row
scaling): the same bounds with u = 2^-10 for fp16; for fp32, u = 2^-18 and
the same u on the sums of absolute products, which covers fp32 accumulation
over K = 4096 terms.
"""
import importlib

import numpy as np
import pytest
import torch

from oracle import gated_lora as gl

pytestmark = pytest.mark.gpu
U = 2.0 ** -8
# rounding unit per dtype; ACC: the bound's factor on sums of absolute
# products (fp32 accumulation error), 0 where the roundings dominate
UNIT = {torch.bfloat16: (2.0 ** -8, 0.0), torch.float16: (2.0 ** -10, 0.0), torch.float32: (2.0 ** -18, 2.0 ** -18)}


def lora_mod():
    return importlib.import_module("mtp-glora_amd.lora")


def make(S, K, N, r, dev, seed=0, gate="mixed", dtype=torch.bfloat16):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(S, K, generator=g, device=dev).to(dtype)
    W = (torch.randn(N, K, generator=g, device=dev) / K ** 0.5).to(dtype)
    A = (torch.randn(r, K, generator=g, device=dev) / K ** 0.5).to(dtype)
    B = (torch.randn(N, r, generator=g, device=dev) * (0.5 / r ** 0.5)).to(dtype)
    gt = None if gate is None else (torch.rand(S, generator=g, device=dev) < 0.7).float()
    return x, W, A, B, gt


def f64(t):
    return None if t is None else t.detach().double().cpu().numpy()


def check(name, got, ref, bound):
    err = np.abs(got - ref)
    worst = (err / bound).max()
    print(f"  {name}: max-abs {err.max():.3e}, worst err/bound {worst:.3f}", flush=True)
    assert worst <= 1.0, name


def run_case(dev, S, K, N, r, p, gate="mixed", seed=0, scaling=2.0, dtype=torch.bfloat16):
    """The layer's own path (bf16: no dropout output kept when K is a multiple
    of 128, grad_A draws the mask again from x), checked against the oracle;
    with dropout on, also the path that keeps h: h bit for bit, the same y,
    and a grad_A over h that meets the same bound."""
    lm = lora_mod()
    U, ACC = UNIT[dtype]
    x, W, A, B, gt = make(S, K, N, r, dev, seed, gate, dtype)
    sd = 1234567 + seed
    y, t, h = lm.gated_lora_forward(x, W, A, B, gt, scaling, p, sd)
    assert h is None or K % 128 or p == 0 or dtype != torch.bfloat16
    assert (h is not None) == (p > 0) or dtype == torch.bfloat16
    dy = torch.randn(S, N, generator=torch.Generator(device=dev).manual_seed(seed + 7), device=dev).to(dtype)
    gx, ga, gb = lm.gated_lora_backward(dy, x, h, t, W, A, B, gt, scaling, p, sd, True, True, True)
    if p > 0:
        yk, tk, hk = lm.gated_lora_forward(x, W, A, B, gt, scaling, p, sd, keep_h=True)
        _, gak, _ = lm.gated_lora_backward(dy, x, hk, tk, W, A, B, gt, scaling, p, sd, False, True, False)
    torch.cuda.synchronize()
    X, Wn, An, Bn, G, DY = f64(x), f64(W), f64(A), f64(B), f64(gt), f64(dy)
    keep = gl.keep_mask(sd, S, K, p) if p > 0 else None
    if p > 0:   # the kernel's dropout output, bit for bit, and the same forward with or without it
        want = (keep * f64(x.float().mul(1.0 / (1.0 - p)).to(dtype)))
        np.testing.assert_array_equal(f64(hk), want)
        assert torch.equal(yk, y) and torch.equal(tk, t)
    Gv = np.ones(S) if G is None else G
    H = X if keep is None else X * keep / (1 - p)
    ks = 1.0 if p == 0 else 1.0 / (1 - p)
    y_ref = gl.forward(X, Wn, An, Bn, G, scaling, keep, p)
    lora_abs = scaling * Gv[:, None] * (np.abs(H @ An.T) @ np.abs(Bn).T)
    lora_sum = scaling * Gv[:, None] * ((np.abs(H) @ np.abs(An).T) @ np.abs(Bn).T)
    h_round = 0.0 if p == 0 else (U / 2) * lora_sum
    acc_y = ACC * (np.abs(X) @ np.abs(Wn).T + lora_sum)
    check("y", f64(y), y_ref,
          U * (np.abs(y_ref) + np.abs(X @ Wn.T) + lora_abs) + h_round + acc_y + 1e-5 * np.abs(y_ref).max())
    dx_ref, dA_ref, dB_ref = gl.backward(DY, X, Wn, An, Bn, G, scaling, keep, p)
    d_a = scaling * Gv[:, None] * (DY @ Bn)
    acc_x = ACC * (np.abs(DY) @ np.abs(Wn) + 2 * ks * ((Gv[:, None] * scaling * (np.abs(DY) @ np.abs(Bn))) @ np.abs(An)))
    bx = U * (np.abs(dx_ref) + np.abs(DY @ Wn) + 2 * ks * (np.abs(d_a) @ np.abs(An))) + acc_x \
        + 1e-5 * np.abs(dx_ref).max()
    check("dX", f64(gx), dx_ref, bx)
    check("dA", f64(ga), dA_ref, U * (np.abs(dA_ref) + np.abs(d_a).T @ np.abs(H)) + 1e-30)
    if p > 0:
        check("dA (kept h)", f64(gak), dA_ref, U * (np.abs(dA_ref) + np.abs(d_a).T @ np.abs(H)) + 1e-30)
    T = scaling * Gv[:, None] * (H @ An.T)
    check("dB", f64(gb), dB_ref, U * (np.abs(dB_ref) + np.abs(DY).T @ np.abs(T)) + 1e-30)
    return y, t, h


@pytest.mark.parametrize("p", [0.0, 0.05])
def test_qwen3_qkv_shape(dev, p):
    """Qwen3-8B fused qkv_proj with the reference's training ranks (3 x 32)."""
    run_case(dev, S=512, K=4096, N=6144, r=96, p=p)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("S,K,N,r,p,gate", [
    (512, 4096, 6144, 96, 0.05, "mixed"),   # Qwen3-8B qkv_proj, dropout on
    (512, 4096, 6144, 96, 0.0, "mixed"),
    (333, 4096, 4096, 32, 0.05, None),      # o_proj-like, ragged rows, no gate
    (40, 1024, 200, 64, 0.5, "mixed"),      # heavy dropout, odd N
    (31, 128, 64, 1, 0.0, "mixed"),         # rank 1
    (50, 272, 100, 24, 0.05, "mixed"),      # in_features not a multiple of 128
])
def test_fp16_fp32_layers(dev, dtype, S, K, N, r, p, gate):
    """fp16 and fp32 layers through the general path against the float64
    oracle, the dropout mask identical to the bf16 path's."""
    print(f"case {dtype} S={S} K={K} N={N} r={r} p={p}", flush=True)
    run_case(dev, S, K, N, r, p, gate=gate, seed=S + 1, dtype=dtype)


@pytest.mark.parametrize("S,K,N,r,p,gate", [
    (333, 4096, 4096, 32, 0.05, None),      # o_proj-like, ragged rows, no gate
    (100, 256, 256, 8, 0.0, "mixed"),       # config-1 sizes
    (64, 512, 384, 160, 0.1, "mixed"),      # rank above 96: chunked down-projection
    (40, 1024, 200, 64, 0.5, "mixed"),      # gate_up-like rank, heavy dropout, odd N
    (31, 128, 64, 1, 0.0, "mixed"),         # rank 1, one partial row block
    (50, 272, 100, 24, 0.05, "mixed"),      # in_features not a multiple of 128 (direct-load kernel)
    (70, 320, 512, 16, 0.0, "mixed"),       # ragged rows, in_features 320
    (256, 512, 192, 40, 0.0, None),         # rank 40 (not a multiple of 32), N = 192
    (300, 256, 64, 8, 0.05, "mixed"),       # rank 8 with dropout (the y bound's h-rounding term), N = 64
])
def test_shapes(dev, S, K, N, r, p, gate):
    run_case(dev, S, K, N, r, p, gate=gate, seed=S)


def test_full_qkv_forward_against_fp32(dev):
    """S = 5120 (config 2's chunk): forward against torch fp32 on the GPU."""
    lm = lora_mod()
    S, K, N, r, p, s = 5120, 4096, 6144, 96, 0.05, 2.0
    x, W, A, B, gt = make(S, K, N, r, dev, seed=3)
    y, t, h = lm.gated_lora_forward(x, W, A, B, gt, s, p, 99, keep_h=True)
    hf, xf, Wf, Af, Bf = h.float(), x.float(), W.float(), A.float(), B.float()
    base = xf @ Wf.T
    lora = s * gt[:, None] * ((hf @ Af.T) @ Bf.T)
    ref = base + lora
    lora_abs = s * gt[:, None] * ((hf @ Af.T).abs() @ Bf.abs().T)
    bound = U * (ref.abs() + base.abs() + lora_abs) + 1e-5 * ref.abs().max()
    worst = ((y.float() - ref).abs() / bound).max().item()
    kept = (h != 0).float().mean().item()
    print(f"  S=5120: worst err/bound {worst:.3f}, kept fraction {kept:.4f}", flush=True)
    assert worst <= 1.0
    assert abs(kept - (1 - gl.drop_threshold(p) / 65536)) < 1e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_module_forward_backward(dev, dtype):
    """GatedLoRALinear (the mirror) in train mode through autograd: x, lora_A
    and lora_B get gradients, the base weight none, and the result equals the
    functional entry points with the same seed."""
    lm = lora_mod()
    torch.manual_seed(0)
    base = torch.nn.Linear(256, 384, bias=False).to(dev, dtype)
    layer = lm.GatedLoRALinear(base, rank=16, alpha=32, dropout=0.05, lora_bias=False, use_rslora=False)
    base.weight.requires_grad_(False)
    with torch.no_grad():
        layer.lora_B.weight.normal_(0, 0.05)
    x = torch.randn(1, 100, 256, device=dev).to(dtype).requires_grad_()
    gate = (torch.rand(1, 100, 1, device=dev) < 0.5).long()
    torch.manual_seed(5)
    y = layer(x, gate)
    y.float().square().sum().backward()
    assert y.shape == (1, 100, 384) and y.dtype == dtype
    assert x.grad is not None and layer.lora_A.weight.grad is not None and layer.lora_B.weight.grad is not None
    assert base.weight.grad is None
    torch.manual_seed(5)
    seed = int(torch.randint(0, 2 ** 62, (), dtype=torch.int64).item())
    y2, _, _ = lm.gated_lora_forward(x.detach()[0], base.weight, layer.lora_A.weight, layer.lora_B.weight,
                                     gate.reshape(-1).float(), 2.0, 0.05, seed)
    assert torch.equal(y.detach()[0], y2)
    layer.eval()
    y3 = layer(x.detach(), gate)
    y4, _, _ = lm.gated_lora_forward(x.detach()[0], base.weight, layer.lora_A.weight, layer.lora_B.weight,
                                     gate.reshape(-1).float(), 2.0, 0.0, 0)
    assert torch.equal(y3[0], y4)


def test_argument_errors(dev):
    lm = lora_mod()
    x, W, A, B, gt = make(8, 64, 32, 4, dev)
    with pytest.raises(TypeError):
        lm.gated_lora_linear(x.float(), W, A, B, gt, 2.0)
    with pytest.raises(NotImplementedError):
        lm.gated_lora_linear(x, W.clone().requires_grad_(), A, B, gt, 2.0)
    with pytest.raises(ValueError):
        lm.gated_lora_linear(x, W, A, B, gt[:5], 2.0)
    x2, W2, A2, B2, g2 = make(8, 40, 32, 4, dev)
    with pytest.raises(Exception, match="multiple of 16"):
        lm.gated_lora_linear(x2, W2, A2, B2, g2, 2.0)
    with pytest.raises(RuntimeError):
        lm.gated_lora_linear(x.cpu(), W.cpu(), A.cpu(), B.cpu(), None, 2.0)


def test_dx_row_stride_multiple_of_4(dev):
    """grad_x rows 8-byte aligned only (row stride K + 4): the in-place dropout
    update takes its 8-byte path and still matches the oracle."""
    lm = lora_mod()
    lib = importlib.import_module("mtp-glora_amd._lib")
    S, K, N, r, p, s = 96, 512, 384, 32, 0.1, 2.0
    x, W, A, B, gt = make(S, K, N, r, dev, seed=11)
    sd = 4242
    y, t, h = lm.gated_lora_forward(x, W, A, B, gt, s, p, sd)
    dy = torch.randn(S, N, generator=torch.Generator(device=dev).manual_seed(12), device=dev).bfloat16()
    buf = torch.zeros(S, K + 4, device=dev, dtype=torch.bfloat16)
    gx = buf[:, :K]
    ws = lm._workspace(S, K, N, r, dev)
    lib.call("mga_gated_lora_bwd", dy.data_ptr(), dy.stride(0), x.data_ptr(), x.stride(0), None,
             0, W.data_ptr(), W.stride(0), A.data_ptr(), A.stride(0), B.data_ptr(), B.stride(0),
             t.data_ptr(), t.stride(0), gt.data_ptr(), s, p, sd, S, K, N, r, gx.data_ptr(), gx.stride(0),
             None, 0, None, 0, ws.data_ptr(), ws.numel(), lib.DTYPE_BF16,
             torch.cuda.current_stream(dev).cuda_stream)
    torch.cuda.synchronize()
    assert torch.count_nonzero(buf[:, K:]).item() == 0   # the 4 pad columns are untouched
    X, Wn, An, Bn, G, DY = f64(x), f64(W), f64(A), f64(B), f64(gt), f64(dy)
    keep = gl.keep_mask(sd, S, K, p)
    dx_ref, _, _ = gl.backward(DY, X, Wn, An, Bn, G, s, keep, p)
    d_a = s * G[:, None] * (DY @ Bn)
    bx = U * (np.abs(dx_ref) + np.abs(DY @ Wn) + 2 / (1 - p) * (np.abs(d_a) @ np.abs(An))) + 1e-5 * np.abs(dx_ref).max()
    check("dX (stride K + 4)", f64(gx), dx_ref, bx)


def test_repeated_calls_equal_bit_for_bit(dev):
    # Every reduction runs in a fixed order, so the layer's own kernels give the
    # same bits every time (dX passes through the base GEMM, whose library
    # kernel may sum in another order, and is left out). A streaming buffer
    # refilled while a slow wave still reads it shows here as a rare mismatch.
    lm = lora_mod()
    x, W, A, B, gate = make(5120, 4096, 6144, 96, dev)
    gy = torch.randn(5120, 6144, device=dev, generator=torch.Generator(device=dev).manual_seed(1)).bfloat16()
    first = None
    for _ in range(40):
        y, t, h = lm.gated_lora_forward(x, W, A, B, gate, 2.0, 0.05, 11)
        _, ga, gb = lm.gated_lora_backward(gy, x, h, t, W, A, B, gate, 2.0, 0.05, 11, True, True, True)
        out = (t, ga, gb)
        if first is None:
            first = [v.clone() for v in out]
        else:
            for name, a, b in zip(("t", "grad_A", "grad_B"), first, out):
                assert torch.equal(a, b), name


@pytest.mark.parametrize("S,K,N,r", [(1303, 4096, 24576, 64), (97, 4096, 24576, 32), (2500, 12288, 4096, 16)])
def test_long_reductions(dev, S, K, N, r):
    """Qwen3-8B gate_up- and down-projections: dX sums over up to 24 576
    columns, where the GEMM library's first choice of algorithm can need more
    workspace than the layer has. Against float64 on the GPU, with the bf16
    unit roundoff 2^-8 for each rounding: y rounds t (carried by |t| |B|^T), the
    LoRA term and the sum; dX rounds d_a (by |d_a| |A|), d_a A and the sum."""
    lm = lora_mod()
    x, W, A, B, gt = make(S, K, N, r, dev, seed=S)
    dy = torch.randn(S, N, generator=torch.Generator(device=dev).manual_seed(S + 7), device=dev).bfloat16()
    y, t, h = lm.gated_lora_forward(x, W, A, B, gt, 2.0, 0.0, 0)
    gx, _, _ = lm.gated_lora_backward(dy, x, h, t, W, A, B, gt, 2.0, 0.0, 0, True, False, False)
    X, Wd, Ad, Bd, DY, G = (v.double() for v in (x, W, A, B, dy, gt[:, None]))
    lora = 2.0 * G * ((X @ Ad.t()) @ Bd.t())
    ref = X @ Wd.t() + lora
    lora_abs = 2.0 * G * ((X @ Ad.t()).abs() @ Bd.abs().t())
    bound = U * (ref.abs() + lora.abs() + lora_abs) + 1e-5 * ref.abs().max()
    assert bool(((y.double() - ref).abs() <= bound).all())
    d_a = 2.0 * G * (DY @ Bd)
    base = DY @ Wd
    ref = base + d_a @ Ad
    bound = U * (ref.abs() + (ref - base).abs() + d_a.abs() @ Ad.abs()) + 1e-5 * ref.abs().max()
    assert bool(((gx.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("S,K,N,r,p,gate", [
    (129, 144, 136, 128, 0.3, "mixed"),     # one line past a block, a column tail in every product, the largest rank block
    (65, 208, 72, 100, 0.05, "mixed"),      # ranks past 96 that are not a multiple of 32; 16-column tails
    (1, 16, 8, 3, 0.5, None),               # a single row, the smallest columns (p = 1/2 scales exactly: h is not rounded,
                                            # as the dA and dB bounds, which have no term for it, need at one row)
    (700, 4096, 256, 33, 0.9375, "mixed"),  # nearly everything dropped (again an exact scale); more splits than line blocks
    (260, 1168, 520, 130, 0.1, "mixed"),    # ranks in two launches, one of two ranks
    (320, 128, 32768, 128, 0.05, "mixed"),  # the wide write of y by ten waves a workgroup, the largest LDS of both forms
    (320, 32768, 64, 128, 0.05, "mixed"),   # and of dX
])
def test_streaming_edges(dev, S, K, N, r, p, gate):
    """The streaming products and the wide writes at the edges of their 128-line
    blocks, 64-wide chunks and rank blocks."""
    run_case(dev, S, K, N, r, p, gate=gate, seed=S + r)


def test_unaligned_rows_take_the_library_products(dev):
    """N = 4: lora_B's products and the up-projection cannot use 16-byte rows."""
    run_case(dev, 70, 256, 4, 12, 0.1, seed=3)


@pytest.mark.parametrize("S,K,r,p,x_rs,a_rs", [
    (100, 256, 33, 0.1, 1 << 23, 256),               # x: the first stride past the 32-bit lane offsets
    (65, 144, 8, 0.5, (1 << 23) + 8, 144),           # dropout output written, a 16-column tail
    (3, 128, 96, 0.1, (1 << 26) + 16, 128),
    (200, 640, 64, 0.0, 640, 1 << 23),               # lora_A
    (70, 384, 128, 0.2, (1 << 22) + 8, (1 << 23) + 64),
    (40, 256, 130, 0.1, 1 << 23, 1 << 23),           # both, ranks in two launches
])
def test_wide_row_strides(dev, S, K, r, p, x_rs, a_rs):
    """x and lora_A as rows of far wider buffers: the streaming products are
    those of dense rows bit for bit; y and dX, which pass through the library's
    base product, within its fp32 order (1e-5) and the roundings of two results."""
    print(f"case S={S} K={K} r={r} p={p} strides {x_rs} {a_rs}", flush=True)
    lm = lora_mod()
    x, W, A, B, gt = make(S, K, 96, r, dev, seed=S)
    dy = torch.randn(S, 96, generator=torch.Generator(device=dev).manual_seed(S + 7), device=dev).bfloat16()

    def wide(t, rs):
        if rs == t.shape[1]:
            return t
        w = torch.empty((t.shape[0] - 1) * rs + t.shape[1], dtype=t.dtype, device=dev).as_strided(t.shape, (rs, 1))
        return w.copy_(t)

    def layer(x, A):
        y, t, h = lm.gated_lora_forward(x, W, A, B, gt, 2.0, p, 77)
        gx, ga, gb = lm.gated_lora_backward(dy, x, h, t, W, A, B, gt, 2.0, p, 77, True, p > 0, True)
        return (y, gx), (t, h, ga, gb)

    xw = wide(x, x_rs)
    y = lm.gated_lora_linear(xw, W, A, B, gt, 2.0, p, seed=77)   # the public call reads the rows where they are
    rounded, exact = layer(x, A)
    assert bool(((y.float() - rounded[0].float()).abs() <= 2 * U * y.float().abs() + 1e-5 * y.float().abs().max()).all())
    rounded_wide, exact_wide = layer(xw, wide(A, a_rs))
    for a, b in zip(exact, exact_wide):
        assert (a is None and b is None) or torch.equal(a, b)
    for a, b in zip(rounded, rounded_wide):
        assert bool(((a.float() - b.float()).abs() <= 2 * U * a.float().abs() + 1e-5 * a.float().abs().max()).all())
