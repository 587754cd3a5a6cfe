"""HIP stable soft cross-entropy (mga_soft_ce_*) against the float64 oracle
(oracle/soft_ce.py, pinned by tests/test_oracle_soft_ce.py).

* The reference's own test (mtp_glora/core/loss.py:335-385): fp32 logits
  [4, 4, 4096] and [8, 2, 151936], loss sum and student gradient within its
  tolerances (rtol = atol = 2e-4, and 3e-4 at V = 151936).
* bf16 logits (the model dtype) at the sampler's shape, V = 151936: the oracle
  runs on the same bf16 values; loss within rtol 1e-4, gradient (bf16) within
  one bf16 rounding of the oracle's value (rtol 2^-7) plus atol 1e-7.
* fp16 logits at the same shape: loss within rtol 1e-4, gradient (fp16)
  within 2^-10 of the oracle's value plus 3e-8 (half the spacing of fp16's
  subnormals, where most of the gradient's elements lie).
* A strided teacher (the reference's call site passes a strided view,
  core/mtp.py:124), widths that are not multiples of the vector width, a
  misaligned row stride (element-load path), a single column, and rows whose
  maxima differ by hundreds of units (stable rescaling).
"""
import numpy as np
import pytest
import torch

from oracle import soft_ce as sc

pytestmark = pytest.mark.gpu


def _run(mga, x, t, go=1.0):
    xg = x.detach().clone().requires_grad_()
    loss = mga.StableSoftCrossEntropy.apply(xg, t)
    loss.backward(torch.tensor(go, device=x.device))
    torch.cuda.synchronize()
    return loss.item(), xg.grad


def _f64(t):
    return t.detach().double().cpu().numpy()


@pytest.mark.parametrize("shape,tol", [((4, 4, 4096), 2e-4), ((8, 2, 151936), 3e-4)])
def test_reference_test_shapes_fp32(mga, dev, shape, tol):
    g = torch.Generator(device=dev).manual_seed(0)
    x = torch.randn(*shape, generator=g, device=dev)
    t = torch.randn(*shape, generator=g, device=dev)
    loss, grad = _run(mga, x, t)
    ref = sc.soft_ce_loss(_f64(x), _f64(t))
    ref_g = sc.soft_ce_grad(_f64(x), _f64(t))
    print(f"  loss {loss:.6f} ref {ref:.6f}", flush=True)
    assert abs(loss - ref) <= tol + tol * abs(ref)
    assert grad.dtype == torch.float32
    np.testing.assert_allclose(_f64(grad), ref_g, rtol=tol, atol=tol)


@pytest.mark.parametrize("rows", [1, 255, 512])
def test_bf16_sampler_shape(mga, dev, rows):
    g = torch.Generator(device=dev).manual_seed(rows)
    V = 151936
    x = (torch.randn(1, rows, V, generator=g, device=dev) * 3).bfloat16()
    t = (torch.randn(1, rows, V, generator=g, device=dev) * 3).bfloat16()
    loss, grad = _run(mga, x, t, go=0.5)
    ref = sc.soft_ce_loss(_f64(x), _f64(t))
    ref_g = 0.5 * sc.soft_ce_grad(_f64(x), _f64(t))
    assert abs(loss - ref) <= 1e-4 * abs(ref)
    assert grad.dtype == torch.bfloat16
    err = np.abs(_f64(grad) - ref_g)
    print(f"  rows {rows}: loss {loss:.4f} ref {ref:.4f} grad max-abs {err.max():.3e}", flush=True)
    assert (err <= 2.0 ** -7 * np.abs(ref_g) + 1e-7).all()


@pytest.mark.parametrize("rows", [1, 300])
def test_fp16_sampler_shape(mga, dev, rows):
    g = torch.Generator(device=dev).manual_seed(rows + 7)
    V = 151936
    x = (torch.randn(1, rows, V, generator=g, device=dev) * 3).half()
    t = (torch.randn(1, rows, V, generator=g, device=dev) * 3).half()
    loss, grad = _run(mga, x, t, go=0.5)
    ref = sc.soft_ce_loss(_f64(x), _f64(t))
    ref_g = 0.5 * sc.soft_ce_grad(_f64(x), _f64(t))
    assert abs(loss - ref) <= 1e-4 * abs(ref)
    assert grad.dtype == torch.float16
    err = np.abs(_f64(grad) - ref_g)
    print(f"  rows {rows}: loss {loss:.4f} ref {ref:.4f} grad max-abs {err.max():.3e}", flush=True)
    assert (err <= 2.0 ** -10 * np.abs(ref_g) + 3e-8).all()


def test_strided_teacher_and_odd_widths(mga, dev):
    g = torch.Generator(device=dev).manual_seed(3)
    # teacher as a strided row view of a larger logits tensor (every 5th row)
    base = torch.randn(1, 60, 1000, generator=g, device=dev).bfloat16()
    t = base[:, 3::5, :]
    x = torch.randn(1, t.shape[1], 1000, generator=g, device=dev).bfloat16()
    loss, grad = _run(mga, x, t)
    assert abs(loss - sc.soft_ce_loss(_f64(x), _f64(t))) <= 1e-4 * abs(loss)
    np.testing.assert_allclose(_f64(grad), sc.soft_ce_grad(_f64(x), _f64(t)), rtol=2.0 ** -7, atol=1e-6)
    for V in (1, 7, 4099, 20011):   # tails and the element-load path (odd row strides)
        x = torch.randn(2, 3, V, generator=g, device=dev)
        t = torch.randn(2, 3, V, generator=g, device=dev)
        loss, grad = _run(mga, x, t)
        ref = sc.soft_ce_loss(_f64(x), _f64(t))
        assert abs(loss - ref) <= 1e-4 * (1 + abs(ref)), V
        np.testing.assert_allclose(_f64(grad), sc.soft_ce_grad(_f64(x), _f64(t)), rtol=1e-4, atol=1e-6)


def test_large_offsets_and_identical_rows(mga, dev):
    g = torch.Generator(device=dev).manual_seed(4)
    x = torch.randn(1, 6, 70000, generator=g, device=dev)
    x += torch.tensor([0.0, 300.0, -300.0, 80.0, -80.0, 0.0], device=dev)[None, :, None]
    t = x.clone()
    t[0, 5] = torch.randn(70000, generator=g, device=dev) * 20
    loss, grad = _run(mga, x, t)
    ref = sc.soft_ce_loss(_f64(x), _f64(t))
    assert abs(loss - ref) <= 1e-4 * abs(ref)
    ref_g = sc.soft_ce_grad(_f64(x), _f64(t))
    np.testing.assert_allclose(_f64(grad), ref_g, rtol=1e-4, atol=1e-7)
    assert np.abs(_f64(grad)[0, :5]).max() < 1e-6   # identical rows: zero gradient


def test_argument_errors(mga, dev):
    x = torch.randn(1, 2, 64, device=dev)
    with pytest.raises(ValueError):
        mga.StableSoftCrossEntropy.apply(x, torch.randn(1, 2, 65, device=dev))
    with pytest.raises(TypeError):
        mga.StableSoftCrossEntropy.apply(x, x.bfloat16())
    with pytest.raises(RuntimeError):
        mga.StableSoftCrossEntropy.apply(x.cpu(), x.cpu())


@pytest.mark.parametrize("rows,V,dtype", [(1, 600008, torch.bfloat16),    # more splits than lanes of a wave
                                          (52, 151936, torch.bfloat16), (3, 8191, torch.float32),
                                          (1025, 4104, torch.float16),    # a row past the workgroup's first pass
                                          (7, 2049, torch.bfloat16)])
def test_splits_and_row_sum(mga, dev, rows, V, dtype):
    """Row splits and the row sum at the edges of their loops, against float64
    on the GPU: fp32 sums of V terms, so 1e-5 relative; a leading run of
    masked (-inf) teacher logits longer than a turn of the workgroup (4096 of
    the 16-bit types) and, where there are splits, than a whole split."""
    from importlib import import_module
    lossmod = import_module("mtp-glora_amd.loss")
    g = torch.Generator(device=dev).manual_seed(V)
    x = (torch.randn(1, rows, V, generator=g, device=dev) * 3).to(dtype)
    t = (torch.randn(1, rows, V, generator=g, device=dev) * 3).to(dtype)
    t[:, :, :{600008: 9000, 151936: 9000, 8191: 4200, 4104: 4100, 2049: 2000}[V]] = float("-inf")
    want = -(torch.softmax(t.double(), -1) * torch.log_softmax(x.double(), -1)).sum(-1)[0]
    loss, _ = lossmod.soft_ce_forward(x, t)
    assert bool(((loss.double() - want).abs() <= 1e-5 * want.abs()).all())
    total = mga.StableSoftCrossEntropy.apply(x, t)
    assert total.shape == () and abs(float(total) - float(want.sum())) <= 1e-5 * float(want.sum())


@pytest.mark.gpu
@pytest.mark.parametrize("rows,V,dtype", [(1, 4088, torch.bfloat16),      # vectors, no whole turn
                                          (1030, 4096, torch.bfloat16),   # one turn
                                          (1030, 8195, torch.bfloat16),   # rows not 16-byte aligned
                                          (1030, 14384, torch.bfloat16),  # three turns and a part of one
                                          (40, 9004, torch.float32),      # splits, a short last one
                                          (1030, 6148, torch.float32)])   # three turns and one vector
def test_gradient_turns(mga, dev, rows, V, dtype):
    """The gradient at the edges of its column walk, against float64 on the
    GPU: two fp32 probabilities p and q, each within 1e-5 (sums of V terms), and
    the output's rounding, |g - g'| <= u |g'| + 1e-5 (p + q)."""
    print(f"case {rows} {V} {dtype}", flush=True)
    gen = torch.Generator(device=dev).manual_seed(V)
    x, t = ((torch.randn(1, rows, V, generator=gen, device=dev) * 3).to(dtype) for _ in range(2))
    _, grad = _run(mga, x, t)
    p, q = x.double().softmax(-1), t.double().softmax(-1)
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    assert bool(((grad.double() - (p - q)).abs() <= u * (p - q).abs() + 1e-5 * (p + q) + 1e-30).all())


@pytest.mark.gpu
@pytest.mark.parametrize("rows,V", [(3072, 96), (3073, 96),      # the last size of one workgroup, one pass more
                                    (9 * 1024 + 5, 33),          # the sum's second turn
                                    (1000, 10240)])              # several lanes a row
def test_many_rows(mga, dev, rows, V):
    """Row losses and their sum where one workgroup ends and one a pass begins,
    against float64 on the GPU (1e-5, sums of V terms); without a sum asked for
    the rows are the same bit for bit."""
    from importlib import import_module
    lossmod = import_module("mtp-glora_amd.loss")
    gen = torch.Generator(device=dev).manual_seed(rows)
    x, t = (torch.randn(1, rows, V, generator=gen, device=dev) * 3 for _ in range(2))
    want = -(torch.softmax(t.double(), -1) * torch.log_softmax(x.double(), -1)).sum(-1)[0]
    loss, total, stats = lossmod._forward(x, t)
    assert bool(((loss.double() - want).abs() <= 1e-5 * want.abs()).all())
    assert abs(float(total) - float(want.sum())) <= 1e-5 * float(want.sum())
    again, stats2 = torch.empty_like(loss), torch.empty_like(stats)
    ws = torch.empty(int(mga.load_library().mga_soft_ce_workspace_floats(rows, V)), device=dev)
    mga._lib.call("mga_soft_ce_fwd", x.data_ptr(), V, t.data_ptr(), V, rows, V, mga.ops.dtype_code(x.dtype),
                  again.data_ptr(), stats2.data_ptr(), ws.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert torch.equal(again, loss) and torch.equal(stats2, stats)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,V,dtype", [(9000, 4088, torch.bfloat16),    # vectors, no whole turn
                                          (9000, 4096, torch.float16),     # one turn
                                          (5000, 14384, torch.bfloat16),   # three turns and a part of one
                                          (3000, 6148, torch.float32)])    # three turns and one vector
def test_gradient_past_the_cache(mga, dev, rows, V, dtype):
    """More bytes than the last-level cache holds: written past it, the gradient
    of a row is what it is among fewer rows, bit for bit (one split either way)."""
    print(f"case {rows} {V} {dtype}", flush=True)
    gen = torch.Generator(device=dev).manual_seed(V)
    x, t = ((torch.randn(1, rows, V, generator=gen, device=dev) * 3).to(dtype) for _ in range(2))
    few = 1100
    assert 3 * x.nbytes > 210 << 20 > 3 * x[:, :few].nbytes
    _, grad = _run(mga, x, t)
    for i in (0, rows - few):
        assert torch.equal(grad[:, i:i + few], _run(mga, x[:, i:i + few], t[:, i:i + few])[1])
