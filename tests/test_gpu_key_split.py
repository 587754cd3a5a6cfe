"""Attention launches whose last work items are split over their keys
(mga_attn_fwd_ws / mga_attn_bwd_ws with a workspace) against the same calls
without one, at chunk sizes around the plan's edges: fewer items than slots,
one item past a round, rows and keys past the last tile, an item whose tile
list is shorter than its parts.

Bounds, u the operand type's unit roundoff (2^-8 bf16, 2^-11 fp16: half a
unit in the last place of a value at the bottom of its binade, so two
roundings of nearly the same value lie up to 2 u apart):
* o: the parts round their probabilities at another running offset, so each
  of the two outputs is off by at most u sum p |v| before its own rounding (the
  sum is the forward of |v|): |o - o'| <= 2 u (sum p |v| + |o|);
* lse: fp32 sums in another order, |lse - lse'| <= 1e-5;
* dQ: dS is formed from the same lse, so only the fp32 sum's order (bounded by
  1e-5 max|dq|) and the output's rounding differ:
  |dq - dq'| <= 2 u |dq| + 1e-5 max|dq|;
* dK, dV, whose pass splits its query lists: the same P and dS, so again the
  fp32 sum's order and the output's rounding only, the bound of dQ;
* fp32 operands: every output within 1e-5 of its largest entry (fp32 sums in
  another order).
Repeated calls are equal bit for bit."""
import pytest
import torch

from gpu_helpers import attn_fwd_unsplit, chunk_layout, qkv

UNIT = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}

CASES = [
    dict(n_reg=371, n_anchor=33, P=4491, Hq=32, Hkv=8, D=128, pad=5),     # 8 items an XCD
    dict(n_reg=2049, n_anchor=8, P=1500, Hq=32, Hkv=8, D=128, pad=0),     # one 64-row item past a round
    dict(n_reg=1201, n_anchor=75, P=4099, Hq=32, Hkv=8, D=128, pad=35),   # 24 items: a long and a short part each
    dict(n_reg=129, n_anchor=3, P=8197, Hq=28, Hkv=4, D=128, pad=1),      # G = 7: 4-wave workgroups
    dict(n_reg=65, n_anchor=5, P=2500, Hq=8, Hkv=8, D=64, pad=0),         # G = 1
    dict(n_reg=500, n_anchor=40, P=1500, Hq=12, Hkv=2, D=64, pad=70),     # G = 6, 16 items on 8 XCDs, pad tiles
    dict(n_reg=1500, n_anchor=75, P=0, Hq=16, Hkv=8, D=128, pad=0),      # no prefix: lists shorter than the longest
    dict(n_reg=1999, n_anchor=131, P=4093, Hq=32, Hkv=8, D=128, pad=6),  # dK/dV: more than a round of items in parts
]


CASES_F32 = [
    dict(n_reg=256, n_anchor=16, P=768, Hq=4, Hkv=2, D=64, pad=3),        # 12 items on 8 XCDs
    dict(n_reg=33, n_anchor=2, P=1000, Hq=8, Hkv=8, D=128, pad=0),        # two row blocks, a key tile of 41 keys
    dict(n_reg=700, n_anchor=60, P=0, Hq=6, Hkv=2, D=64, pad=90),         # G = 3, no prefix
    dict(n_reg=2100, n_anchor=100, P=300, Hq=16, Hkv=8, D=128, pad=0),    # more than a round of items
]


@pytest.mark.gpu
@pytest.mark.parametrize("c,dtype", [(c, t) for c in CASES for t in (torch.bfloat16, torch.float16)]
                         + [(c, torch.float32) for c in CASES_F32])
def test_split_equals_unsplit(mga, dev, c, dtype):
    print(f"case {c} {dtype}", flush=True)
    ops, lib = mga.ops, mga._lib
    P, D, scale, u = c["P"], c["D"], c["D"] ** -0.5, UNIT[dtype]
    seq = chunk_layout(c["n_reg"], c["n_anchor"], 4, P, seed=5, pad=c["pad"])
    S = len(seq.gate)
    q, k, v, kp, vp, do = qkv(S, P, c["Hq"], c["Hkv"], D, dtype, dev, seed=5, std=1.0)
    kf, vf = torch.cat([kp, k], 2), torch.cat([vp, v], 2)
    mask = mga.build_mtp_block_mask(torch.tensor(seq.gate, device=dev)[None], P)
    bm, code = mask.kernel_tensors(), mask.mtp_code
    size = (S, P + S, c["Hq"], c["Hkv"], D, ops.dtype_code(dtype))
    assert lib.load().mga_attn_workspace_bytes(*size, 0, 0) > 0 and lib.load().mga_attn_workspace_bytes(*size, 1, P) > 0

    o, lse = ops.attn_fwd(q, kf, vf, code, bm, P, scale)
    o1, lse1 = attn_fwd_unsplit(mga, q, kf, vf, mask, scale)
    pv = attn_fwd_unsplit(mga, q, kf, vf.abs(), mask, scale)[0].float()
    assert torch.equal(torch.isneginf(lse), torch.isneginf(lse1))
    seen = torch.isfinite(lse1)
    assert float((lse - lse1)[seen].abs().max()) <= 1e-5
    d = (o.float() - o1.float()).abs()
    eps = 1e-5 * float(o1.float().abs().max()) if dtype == torch.float32 else 0.0
    assert bool((d <= eps + 2 * u * (pv + o1.float().abs())).all())

    args = (q, kf, vf, o1, lse1, do, code, bm, P, scale, P)
    dq, dk, dv = ops.attn_bwd(*args, key_split=True)
    dq1, dk1, dv1 = ops.attn_bwd(*args)
    for a, b in ((dq, dq1), (dk, dk1), (dv, dv1)):
        d = (a.float() - b.float()).abs()
        assert bool((d <= 2 * u * b.float().abs() + 1e-5 * float(b.float().abs().max())).all())

    again, _ = ops.attn_fwd(q, kf, vf, code, bm, P, scale)
    assert torch.equal(o, again)
    for a, b in zip((dq, dk, dv), ops.attn_bwd(*args, key_split=True)):
        assert torch.equal(a, b)


def test_workspace_plan(mga):
    """Whole rounds and short key lists need no workspace; the split ones stay
    within four rounds of parts (a part: 8 waves of a 32-row O^T with its offsets
    and sums) at the largest sizes; a smaller workspace is refused before any
    device work."""
    lib = mga.load_library()
    assert lib.mga_attn_workspace_bytes(2048, 30720, 32, 8, 128, 0, 0, 0) == 0     # 32 items an XCD
    assert lib.mga_attn_workspace_bytes(320, 320, 32, 8, 128, 0, 0, 0) == 0        # three tiles of keys
    assert lib.mga_attn_workspace_bytes(508, 20999, 32, 8, 96, 0, 0, 0) == 0       # not a supported head_dim
    most = 4 * 32 * 8 * 8 * (128 * 32 + 128) * 4   # rounds, slots an XCD, XCDs, waves, fp32 words of a wave
    for S in range(33, 6200, 97):
        for P in (0, 1000, 30000, 131072):
            for back in (0, 1):
                assert 0 <= lib.mga_attn_workspace_bytes(S, P + S, 32, 8, 128, 0, back, P) <= most
    p = 16
    base = [p, 128, 4096, p, 128 * 64, 128, p, 128 * 64, 128, p, 128, 4096, p, p, p, p, p, p]
    rc = lib.mga_attn_fwd_ws(*base, 508, 20999, 20491, 32, 8, 128, 0, 0.1, p, 64, None)
    assert rc == mga._lib.MGA_ERR_INVALID and b"workspace" in lib.mga_last_error()


@pytest.mark.parametrize("S,P,D", [(872, 1500, 128), (872, 1500, 64), (872, 6000, 64), (1000, 2500, 128),
                                   (3248, 1500, 128), (3624, 2500, 128), (3624, 5000, 128), (724, 2489, 64)])
def test_whole_items_where_they_end_first(mga, S, P, D):
    """Chunks whose own keys are a large share of their lists (32 / 8 heads): the
    slots that end early level the whole items, and the split launches timed 3
    to 15% slower, so neither the forward nor the dQ pass is split."""
    lib = mga.load_library()
    assert lib.mga_attn_workspace_bytes(S, P + S, 32, 8, D, 0, 0, 0) == 0
    assert lib.mga_attn_workspace_bytes(S, P + S, 32, 8, D, 0, 1, P + S) == 0   # no key gradients: dQ alone
    assert lib.mga_attn_workspace_bytes(508, 20491 + 508, 32, 8, D, 0, 0, 0) > 0


@pytest.mark.parametrize("S,Hq,Hkv,D", [(2872, 32, 8, 128), (3062, 32, 8, 128), (3248, 32, 8, 64), (2000, 16, 8, 64)])
def test_key_tiles_whole_where_they_end_first(mga, S, Hq, Hkv, D):
    """Chunks whose key tiles level the CUs whole (the pass timed 2 to 10% slower
    in parts): the backward's workspace is the dQ pass's alone."""
    lib = mga.load_library()
    for P in (0, 800):
        dq = lib.mga_attn_workspace_bytes(S, P + S, Hq, Hkv, D, 0, 1, P + S)
        assert lib.mga_attn_workspace_bytes(S, P + S, Hq, Hkv, D, 0, 1, P) == dq
    assert lib.mga_attn_workspace_bytes(872, 872, 32, 8, D, 0, 1, 0) > 0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("c", [dict(n_reg=520, n_anchor=18, P=200, Hq=32, Hkv=8, D=128, pad=8),
                               dict(n_reg=500, n_anchor=25, P=500, Hq=28, Hkv=4, D=128, pad=0),
                               dict(n_reg=401, n_anchor=24, P=199, Hq=12, Hkv=2, D=64, pad=3)])
@pytest.mark.parametrize("from_first", [True, False])
def test_prefix_keys_in_parts(mga, dev, c, dtype, from_first):
    """dK and dV of prefix keys too (plain key tensors), all of them or from a row
    inside a key tile on, with the pass's query lists in parts: the bound of
    split and whole above, the combined rows of the first and the last tile among
    them."""
    ops, lib = mga.ops, mga._lib.load()
    P, D, scale, u = c["P"], c["D"], c["D"] ** -0.5, UNIT[dtype]
    start = 0 if from_first else 71
    seq = chunk_layout(c["n_reg"], c["n_anchor"], 4, P, seed=6, pad=c["pad"])
    S = len(seq.gate)
    size = (S, P + S, c["Hq"], c["Hkv"], D, ops.dtype_code(dtype), 1)
    print(f"case {c} {dtype} from {start}", flush=True)
    assert lib.mga_attn_workspace_bytes(*size, start) > lib.mga_attn_workspace_bytes(*size, P + S)   # beyond dQ's
    q, k, v, kp, vp, do = qkv(S, P, c["Hq"], c["Hkv"], D, dtype, dev, seed=6, std=1.0)
    kf, vf = torch.cat([kp, k], 2), torch.cat([vp, v], 2)
    mask = mga.build_mtp_block_mask(torch.tensor(seq.gate, device=dev)[None], P)
    o, lse = attn_fwd_unsplit(mga, q, kf, vf, mask, scale)
    args = (q, kf, vf, o, lse, do, mask.mtp_code, mask.kernel_tensors(), P, scale, start)
    for a, b in zip(ops.attn_bwd(*args, key_split=True), ops.attn_bwd(*args)):
        d = (a.float() - b.float()).abs()
        assert a.shape[2] in (S, P + S - start)
        assert bool((d <= 2 * u * b.float().abs() + 1e-5 * float(b.float().abs().max())).all())
