"""Causal attention (flash-style forward + recompute backward, MFMA) on the GPU
against the oracle restatement of dtrain's causal_attention.

Bar: float64 normwise relative error <= 1e-12; float32 <= 1e-5 (dtrain itself
computes the float32 case in float64 under NumPy 2; the oracle reproduces that).
"""
import numpy as np
import pytest

from helpers import bits_equal, rel_err
from oracle import ops

pytestmark = pytest.mark.gpu

TOL = {np.float64: 1e-12, np.float32: 1e-5}


def _dev():
    from dtmi import device as D, kernels as K
    return D, K


def _check(D, K, q, k, v, g, dt):
    o_ref, p, scale = ops.attention_fwd(q, k, v)
    gq, gk, gv = ops.attention_bwd(g, q, k, v, p, scale)
    m_ref, l_ref = ops.row_stats(q, k)
    dq_, dk_, dv_ = D.from_numpy(q), D.from_numpy(k), D.from_numpy(v)
    o, rmax, rsum = K.attn_fwd(dq_, dk_, dv_)
    assert rel_err(o.numpy(), o_ref) <= TOL[dt]
    # the kernels keep the row max in base-2 units (log2(e) * max), for exp2
    assert rel_err(rmax.numpy(), m_ref * np.log2(np.e)) <= TOL[dt]
    assert rel_err(rsum.numpy(), l_ref) <= TOL[dt]
    gq_d, gk_d, gv_d = K.attn_bwd(dq_, dk_, dv_, o, D.from_numpy(g), rmax, rsum)
    assert rel_err(gq_d.numpy(), gq) <= TOL[dt]
    assert rel_err(gk_d.numpy(), gk) <= TOL[dt]
    assert rel_err(gv_d.numpy(), gv) <= TOL[dt]


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [(1, 2, 4, 3), (1, 2, 8, 4), (2, 2, 5, 4), (8, 4, 32, 16), (2, 3, 100, 64),
                                   (1, 1, 257, 33), (16, 12, 256, 64), (2, 3, 32, 64), (1, 2, 64, 64),
                                   (2, 2, 96, 64)])
def test_attention_forward_backward(dev, dt, shape):
    D, K = _dev()
    rng = np.random.default_rng(sum(shape))
    q, k, v, g = (rng.standard_normal(shape).astype(dt) for _ in range(4))
    _check(D, K, q, k, v, g, dt)


@pytest.mark.parametrize("shape", [(1, 2, 16, 64), (2, 3, 208, 64), (3, 2, 512, 64), (1, 2, 2048, 64)])
def test_float64_backward_at_head_dim_64(dev, shape):
    """float64, D = 64 on the aligned path (64-key blocks of 16 per wave, dS
    stored at wave-uniform row offsets and read back through a buffer
    resource by the dQ pass; one tile, T not a multiple of 32 or of 64, and
    T 2048, where a (batch, head)'s dS spans 32 MB), against the oracle at
    1e-12."""
    D, K = _dev()
    rng = np.random.default_rng(sum(shape) + 64)
    q, k, v, g = (rng.standard_normal(shape) for _ in range(4))
    _check(D, K, q, k, v, g, np.float64)


@pytest.mark.parametrize("T", [512, 640, 768, 896, 1024, 2048])
def test_forward_over_many_key_tiles(dev, T):
    """T of 512 to 2048 on the aligned float32 path (the paired-range
    forward, 33 to 129 key tiles of 16 per query tile pair), where the forward's
    reference max moves only when a score exceeds it by 2^8: oracle parity of
    the output, of the row statistics (the true max) and of the backward that
    reads them; identical bits over repeated calls."""
    D, K = _dev()
    rng = np.random.default_rng(T)
    q, k, v, g = (rng.standard_normal((2, 3, T, 64)).astype(np.float32) for _ in range(4))
    _check(D, K, q, k, v, g, np.float32)
    dq_, dk_, dv_ = D.from_numpy(q), D.from_numpy(k), D.from_numpy(v)
    runs = [tuple(x.numpy() for x in K.attn_fwd(dq_, dk_, dv_)) for _ in range(3)]
    for r in runs[1:]:
        for x, y in zip(runs[0], r):
            assert bits_equal(x, y)


@pytest.mark.parametrize("T", [4096, 8192])
def test_float32_attention_at_long_sequences(dev, T):
    """The float32 kernels accumulate in float32 where dtrain (NumPy 2)
    promotes to float64: at T = 4096 and 8192 (one batch element and head, so
    the oracle's T x T arrays stay within a few GB) the outputs, the row
    statistics and dQ, dK, dV stay within 1e-5 of the float64-promoted
    oracle."""
    D, K = _dev()
    rng = np.random.default_rng(T + 1)
    q, k, v, g = (rng.standard_normal((1, 1, T, 64)).astype(np.float32) for _ in range(4))
    _check(D, K, q, k, v, g, np.float32)


@pytest.mark.parametrize("T", [32, 64, 96, 160, 288, 352])
def test_backward_paired_ranges_at_every_pair_count(dev, T):
    """The float32 paired-range backward (16 x 16 tiles, key tile j with its
    mirror, dQ-pass blocks of query-tile pairs) at T / 32 = 1, 2, 3, 5,
    9 and 11 pairs: blocks whose last waves have no pair, one and two key
    tiles per dQ step, a single pair; dQ, dK and dV against the oracle, and
    identical bits over repeated calls."""
    D, K = _dev()
    rng = np.random.default_rng(T + 7)
    q, k, v, g = (rng.standard_normal((2, 3, T, 64)).astype(np.float32) for _ in range(4))
    _check(D, K, q, k, v, g, np.float32)
    dq_, dk_, dv_, dg_ = D.from_numpy(q), D.from_numpy(k), D.from_numpy(v), D.from_numpy(g)
    o, rmax, rsum = K.attn_fwd(dq_, dk_, dv_)
    runs = [tuple(x.numpy() for x in K.attn_bwd(dq_, dk_, dv_, o, dg_, rmax, rsum)) for _ in range(3)]
    for r in runs[1:]:
        for x, y in zip(runs[0], r):
            assert bits_equal(x, y)


@pytest.mark.parametrize("B,H,T,D_", [(40, 8, 256, 64), (36, 4, 352, 64), (40, 8, 512, 64), (40, 8, 345, 64),
                                      (33, 13, 345, 64), (64, 8, 345, 64), (33, 13, 345, 48), (40, 8, 345, 96),
                                      (40, 8, 345, 128)])
def test_paired_grid_shapes_agree_bit_for_bit(dev, B, H, T, D_):
    """The float32 paired-range passes pick their grids by size: the dQ pass
    takes four query-tile pairs per block when there are at least two such
    blocks per CU, else two pairs with each query tile's d-tiles split over two
    waves; the key pass and the forward take several tile pairs per block when
    one pair per block would need more than one round of resident blocks (at
    T 352 the key pass's 11 pairs do not divide evenly over the blocks; at
    T 512 the forward takes two pairs per block). At lengths that are no
    multiple of 32 the forward up to D = 64 also deals its blocks in another
    order, whole heads to an XCD (429 heads: not a multiple of 8; 512 heads at
    T 345: several groups per XCD), and above it the key pass's and the
    forward's four waves reuse their LDS from pair to pair. Each order of
    additions is the same either way, so a (batch, head) gets the same bits:
    the full batch against its first two batch elements alone (split d-tiles,
    one pair per block), and those against the oracle."""
    D, K = _dev()
    rng = np.random.default_rng(B + T)
    q, k, v, g = (rng.standard_normal((B, H, T, D_)).astype(np.float32) for _ in range(4))

    def bwd(sl):
        x = [D.from_numpy(np.ascontiguousarray(t[sl])) for t in (q, k, v, g)]
        o, rmax, rsum = K.attn_fwd(x[0], x[1], x[2])
        return [t.numpy() for t in K.attn_bwd(x[0], x[1], x[2], o, x[3], rmax, rsum) + (o, rmax, rsum)]
    full, part = bwd(slice(0, B)), bwd(slice(0, 2))
    assert bits_equal(full[3][:2], part[3])  # the forward's output
    assert bits_equal(full[4][:2], part[4]) and bits_equal(full[5][:2], part[5])  # its row statistics
    full, part = full[:3], part[:3]
    for a, b in zip(full, part):
        assert bits_equal(a[:2], b)
    o_ref, p, scale = ops.attention_fwd(q[:2], k[:2], v[:2])
    for a, ref in zip(part, ops.attention_bwd(g[:2], q[:2], k[:2], v[:2], p, scale)):
        assert rel_err(a, ref) <= TOL[np.float32]


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_attention_golden_from_dtrain(dev, golden, dt):
    D, K = _dev()
    G = golden("dtrain_attention.npz")
    key = np.dtype(dt).name
    q, k, v, g = (G[f"{key}/{s}"] for s in "qkvg")
    o, rmax, rsum = K.attn_fwd(D.from_numpy(q), D.from_numpy(k), D.from_numpy(v))
    assert rel_err(o.numpy(), G[f"{key}/o"]) <= TOL[dt]
    gq, gk, gv = K.attn_bwd(D.from_numpy(q), D.from_numpy(k), D.from_numpy(v), o, D.from_numpy(g), rmax, rsum)
    assert rel_err(gq.numpy(), G[f"{key}/gq"]) <= TOL[dt]
    assert rel_err(gk.numpy(), G[f"{key}/gk"]) <= TOL[dt]
    assert rel_err(gv.numpy(), G[f"{key}/gv"]) <= TOL[dt]


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_attention_on_fused_qkv_layout(dev, dt):
    """q, k, v as strided views of a [B, T, 3, H, D] projection output (the
    reshape/transpose/split of dtrain/nn.py:100-103), outputs written into
    [B, T, H, D] and [B, T, 3, H, D] buffers."""
    D, K = _dev()
    B, T, H, Dh = 2, 96, 3, 16
    rng = np.random.default_rng(4)
    qkv = rng.standard_normal((B, T, 3, H, Dh)).astype(dt)
    g = rng.standard_normal((B, T, H, Dh)).astype(dt)
    q, k, v = (np.ascontiguousarray(qkv[:, :, i].transpose(0, 2, 1, 3)) for i in range(3))
    gh = np.ascontiguousarray(g.transpose(0, 2, 1, 3))
    o_ref, p, scale = ops.attention_fwd(q, k, v)
    gq, gk, gv = ops.attention_bwd(gh, q, k, v, p, scale)

    dqkv = D.from_numpy(qkv)
    t5 = dqkv.transpose(2, 0, 3, 1, 4)  # [3, B, H, T, D] view
    qd, kd, vd = t5[0], t5[1], t5[2]
    assert not qd.is_contiguous
    obuf = D.empty((B, T, H, Dh), dt)
    o, rmax, rsum = K.attn_fwd(qd, kd, vd, out=obuf.transpose(0, 2, 1, 3))
    assert rel_err(obuf.numpy().transpose(0, 2, 1, 3), o_ref) <= TOL[dt]
    gbuf = D.from_numpy(g)
    dbuf = D.full((B, T, 3, H, Dh), 7.0, dt)
    d5 = dbuf.transpose(2, 0, 3, 1, 4)
    K.attn_bwd(qd, kd, vd, obuf.transpose(0, 2, 1, 3), gbuf.transpose(0, 2, 1, 3), rmax, rsum,
               dq=d5[0], dk=d5[1], dv=d5[2])
    got = dbuf.numpy()
    assert rel_err(got[:, :, 0].transpose(0, 2, 1, 3), gq) <= TOL[dt]
    assert rel_err(got[:, :, 1].transpose(0, 2, 1, 3), gk) <= TOL[dt]
    assert rel_err(got[:, :, 2].transpose(0, 2, 1, 3), gv) <= TOL[dt]


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [(1, 2, 4, 3), (2, 2, 5, 4), (2, 3, 100, 64), (1, 1, 257, 33), (16, 12, 256, 64),
                                   (1, 2, 384, 64), (2, 2, 100, 80), (1, 3, 77, 96), (2, 2, 130, 128)])
def test_recompute_dq_path_matches_oracle(dev, dt, shape):
    """With the dS workspace bound set to 0 the dQ pass recomputes S, P and
    dP from q, k, v, dO and the row statistics (the path taken above 4 GiB of
    dS), or above D = 64 the scores are materialised: forward and backward
    against the oracle at the same bar."""
    D, K = _dev()
    rng = np.random.default_rng(sum(shape) + 7)
    q, k, v, g = (rng.standard_normal(shape).astype(dt) for _ in range(4))
    prev = K.attn_set_ds_limit(0)
    try:
        _check(D, K, q, k, v, g, dt)
    finally:
        K.attn_set_ds_limit(prev)
    assert prev == 4 << 30


def test_backward_without_the_ds_workspace_matches_with_it(dev):
    """A causal dS of 2.4 GB under a bound of 2 GiB: the dQ pass recomputes dS
    instead of reading it from a workspace. Splitting the heads in two keeps
    each half under the bound (dS path); the two paths must agree to the float32
    bar (their key passes add dK and dV over 6144 queries in different orders),
    and not to the bit."""
    D, K = _dev()
    B, H, T, Dh = 1, 32, 6144, 64
    rng = np.random.default_rng(21)
    hq, hk, hv, hg = (rng.standard_normal((B, H, T, Dh)).astype(np.float32) for _ in range(4))
    q, k, v, g = (D.from_numpy(x) for x in (hq, hk, hv, hg))
    o, rmax, rsum = K.attn_fwd(q, k, v)
    prev = K.attn_set_ds_limit(2 << 30)
    try:
        dq, dk, dv = K.attn_bwd(q, k, v, o, g, rmax, rsum)  # recompute path
    finally:
        K.attn_set_ds_limit(prev)
    ho, hm, hs = o.numpy(), rmax.numpy(), rsum.numpy()
    halves = []
    for lo in (0, H // 2):
        sl = slice(lo, lo + H // 2)
        sub = [D.from_numpy(np.ascontiguousarray(x[:, sl])) for x in (hq, hk, hv, ho, hg)]
        stats = [D.from_numpy(np.ascontiguousarray(x[:, sl])) for x in (hm, hs)]
        halves.append([t.numpy() for t in K.attn_bwd(*sub, *stats)])  # 1.2 GB each: dS path
    for i, full in enumerate((dq, dk, dv)):
        ref = np.concatenate([halves[0][i], halves[1][i]], axis=1)
        assert rel_err(full.numpy(), ref) <= 1e-5 and not bits_equal(full.numpy(), ref)


def test_ragged_backward_without_memory_for_the_ds_workspace(dev):
    """dS of the whole batch (576 batch elements of T 16384: 309 GB) cannot be
    allocated: the backward takes as many batch elements at a time as can. The
    batch elements share their inputs (stride 0), so each one's gradients are
    those of a batch of one, to the bit."""
    D, K = _dev()
    B, T, Dh = 576, 16384, 72
    rng = np.random.default_rng(72)
    q1, k1, v1, g1 = (D.from_numpy(rng.standard_normal((1, 1, T, Dh)).astype(np.float32)) for _ in range(4))
    o1, m1, l1 = K.attn_fwd(q1, k1, v1)

    def batch(x):
        return D.DeviceArray(x.block, (B, 1, T, Dh), x.dtype, x.offset, (0, T * Dh, Dh, 1))
    stats = [D.from_numpy(np.ascontiguousarray(np.broadcast_to(x.numpy(), (B, 1, T)))) for x in (m1, l1)]
    one = K.attn_bwd(q1, k1, v1, o1, g1, m1, l1)
    prev = K.attn_set_ds_limit(1 << 50)
    try:
        got = K.attn_bwd(*(batch(x) for x in (q1, k1, v1, o1, g1)), *stats)
    finally:
        K.attn_set_ds_limit(prev)
    for x, r in zip(got, one):
        for b in (0, 100, B - 1):
            assert bits_equal(x[b].numpy(), r[0].numpy())


@pytest.mark.parametrize("shape", [(5, 3, 100, 64), (5, 3, 77, 80), (2, 3, 130, 128)])
@pytest.mark.parametrize("heads", [1, 2, 3, 4, 7])
def test_ragged_backward_in_parts_of_the_batch(dev, shape, heads):
    """A dS bound of a few (batch, head)s: parts of heads of one batch element,
    of whole batch elements, and a smaller last part, to the bit as at once."""
    D, K = _dev()
    B, H, T, _ = shape
    rng = np.random.default_rng(sum(shape))
    # q, k, v and the gradients' buffers as views of a [B, T, 3, H, D] projection
    qkv = D.from_numpy(rng.standard_normal((B, T, 3, H, shape[3])).astype(np.float32)).transpose(2, 0, 3, 1, 4)
    g = D.from_numpy(rng.standard_normal((B, T, H, shape[3])).astype(np.float32)).transpose(0, 2, 1, 3)
    o, rmax, rsum = K.attn_fwd(qkv[0], qkv[1], qkv[2])

    def bwd():
        buf = D.full((B, T, 3, H, shape[3]), 7.0, np.float32)
        d5 = buf.transpose(2, 0, 3, 1, 4)
        K.attn_bwd(qkv[0], qkv[1], qkv[2], o, g, rmax, rsum, dq=d5[0], dk=d5[1], dv=d5[2])
        return buf.numpy()
    whole = bwd()
    nt = 2 * -(-T // 32)
    prev = K.attn_set_ds_limit(heads * nt * (nt + 1) // 2 * 1024)
    try:
        assert bits_equal(bwd(), whole)
    finally:
        K.attn_set_ds_limit(prev)


@pytest.mark.parametrize("T,D_", [(47, 48), (63, 64), (65, 72), (100, 128)])
@pytest.mark.parametrize("route", ["aligned", "unaligned dO", "expanded dO", "no dS"])
def test_backward_probabilities_sum_to_one_by_every_route(dev, T, D_, route):
    """With dO[r, d] = 1 for d = r the sum of dV's column r is the sum of row r of
    the probabilities that the backward recomputed. At scores of up to a few
    hundred, rounded to 1e-5, it is 1 to a float32 sum's error (T terms of at most
    1, each off by a few units in the last place) only if the statistics are of
    scores added in the backward's own order; so whatever route the backward
    takes, they have to be. "expanded": dO's rows overlap in memory."""
    D, K = _dev()
    rng = np.random.default_rng(T)
    q, k, v = (D.from_numpy((3 * rng.standard_normal((1, 2, T, D_))).astype(np.float32)) for _ in range(3))
    o, rmax, rsum = K.attn_fwd(q, k, v, scale=1.0)
    eye = np.broadcast_to(np.eye(T, D_, dtype=np.float32), (1, 2, T, D_))
    if route == "unaligned dO":
        g = D.empty((2 * T * D_ + 1,), np.float32)[1:].reshape(1, 2, T, D_)
        g.assign(eye)
    elif route == "expanded dO":  # row r starts one element before row r - 1
        line = np.zeros(T + D_, np.float32)
        line[T] = 1
        buf = D.from_numpy(line)
        g = D.DeviceArray(buf.block, (1, 2, T, D_), np.float32, 4 * T, (0, 0, -1, 1))
    else:
        g = D.from_numpy(np.ascontiguousarray(eye))
    if route == "expanded dO" and D_ > 64:  # the batched products have never taken such rows
        with pytest.raises(Exception, match="too small"):
            K.attn_bwd(q, k, v, o, g, rmax, rsum, scale=1.0)
        return
    prev = K.attn_set_ds_limit(0 if route == "no dS" else 4 << 30)
    try:
        dv = K.attn_bwd(q, k, v, o, g, rmax, rsum, scale=1.0)[2].numpy()
    finally:
        K.attn_set_ds_limit(prev)
    sums = dv.astype(np.float64).sum(axis=2)[..., :min(T, D_)]
    assert np.max(np.abs(sums - 1)) <= 8 * np.finfo(np.float32).eps


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [(2, 2, 64, 128), (1, 3, 100, 80), (2, 1, 33, 256)])
def test_head_dimensions_beyond_64(dev, dt, shape):
    """D > 64 (e.g. dtrain's --dim 256 --heads 2): float64, and float32 above D =
    128, with scores materialised per batch element and the products as batched
    GEMMs, float32 up to D = 128 on the paired-range kernels; against the oracle."""
    D, K = _dev()
    rng = np.random.default_rng(sum(shape) + 1)
    q, k, v, g = (rng.standard_normal(shape).astype(dt) for _ in range(4))
    _check(D, K, q, k, v, g, dt)


@pytest.mark.parametrize("B,T,H,N", [(2, 64, 2, 96), (4, 1024, 12, 768)])
def test_rowsum_formed_by_the_projection_gradient(dev, B, T, H, N):
    """dtmi_linear_bwd_dx_rowdot (the projection that reads the attention
    output O: dO = dY W^T, plus rowsum(dO * O) per 64-wide head, in the split-K
    pass at the GPT-2-small shape and in a pass over dO at the small one) then
    dtmi_attn_bwd_rowsum: dO bit-equal to dtmi_linear_bwd_dx's, the row sums
    within float32 rounding of a float64 sum, and dq, dk, dv bit-equal to
    dtmi_attn_bwd computing the row sums itself (dtrain/autograd.py:242,
    nn.py:103-104)."""
    D, K = _dev()
    dt = np.float32
    C = H * 64
    rng = np.random.default_rng(B + T)
    qkv = rng.standard_normal((B, T, 3, H, 64)).astype(dt)
    w = (rng.standard_normal((C, N)) * 0.05).astype(dt)
    dy = rng.standard_normal((B * T, N)).astype(dt)
    dqkv = D.from_numpy(qkv)
    t5 = dqkv.transpose(2, 0, 3, 1, 4)
    obuf = D.empty((B, T, H, 64), dt)
    _, rmax, rsum = K.attn_fwd(t5[0], t5[1], t5[2], out=obuf.transpose(0, 2, 1, 3))
    x2 = obuf.reshape(B * T, C)
    dw_ = D.from_numpy(w)
    rs = D.empty((B * H * T,), dt)
    do_fused, _, _ = K.linear_bwd(x2, dw_, D.from_numpy(dy), need_db=False, rowdot=rs, rowdot_t=T)
    do_plain, _, _ = K.linear_bwd(x2, dw_, D.from_numpy(dy), need_db=False)
    assert np.array_equal(do_fused.numpy().view(np.uint32), do_plain.numpy().view(np.uint32))
    o64 = obuf.numpy().astype(np.float64).reshape(B, T, H, 64)
    g64 = do_plain.numpy().astype(np.float64).reshape(B, T, H, 64)
    ref = np.einsum("bthd,bthd->bht", o64, g64)
    assert rel_err(rs.numpy().reshape(B, H, T), ref) <= 1e-6
    g4 = do_plain.reshape(B, T, H, 64).transpose(0, 2, 1, 3)
    o4 = obuf.transpose(0, 2, 1, 3)
    a = [D.full((B, T, 3, H, 64), 3.0, dt) for _ in range(2)]
    for buf, drow in zip(a, (None, rs)):
        d5 = buf.transpose(2, 0, 3, 1, 4)
        K.attn_bwd(t5[0], t5[1], t5[2], o4, g4, rmax, rsum, dq=d5[0], dk=d5[1], dv=d5[2], drow=drow)
    assert np.array_equal(a[0].numpy().view(np.uint32), a[1].numpy().view(np.uint32))


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [(2, 3, 256, 64), (1, 2, 128, 32), (2, 3, 100, 64), (1, 2, 77, 48), (2, 3, 77, 80),
                                   (1, 2, 130, 128)])
def test_results_written_through_unaligned_views(dev, dt, shape):
    """O, dQ, dK and dV written into views one element past a 16-byte
    boundary take the element-wise stores; aligned outputs take 16-byte
    stores. Both must give the same bits, and the values the oracle's. dO read
    from such a view is packed first on the ragged paired-range path (the same
    bits) and takes the general kernels elsewhere."""
    D, K = _dev()
    rng = np.random.default_rng(sum(shape))
    hq, hk, hv, hg = (rng.standard_normal(shape).astype(dt) for _ in range(4))
    q, k, v, g = (D.from_numpy(x) for x in (hq, hk, hv, hg))
    n = int(np.prod(shape))

    def shifted():
        return D.empty((n + 1,), dt)[1:].reshape(*shape)

    o, rmax, rsum = K.attn_fwd(q, k, v)
    o2, rmax2, rsum2 = K.attn_fwd(q, k, v, out=shifted())
    assert o2.ptr % 16 != 0
    for a, b in ((o, o2), (rmax, rmax2), (rsum, rsum2)):
        assert bits_equal(a.numpy(), b.numpy())
    grads = K.attn_bwd(q, k, v, o, g, rmax, rsum)
    grads2 = K.attn_bwd(q, k, v, o, g, rmax, rsum, dq=shifted(), dk=shifted(), dv=shifted())
    for a, b in zip(grads, grads2):
        assert bits_equal(a.numpy(), b.numpy())
    o_ref, p, scale = ops.attention_fwd(hq, hk, hv)
    ref = ops.attention_bwd(hg, hq, hk, hv, p, scale)
    assert rel_err(o2.numpy(), o_ref) <= TOL[dt]
    for a, r in zip(grads2, ref):
        assert rel_err(a.numpy(), r) <= TOL[dt]
    g2 = shifted()
    g2.assign(hg)
    for a, r, b in zip(K.attn_bwd(q, k, v, o, g2, rmax, rsum), ref, grads):
        assert rel_err(a.numpy(), r) <= TOL[dt]
        if dt == np.float32 and 32 < shape[3] <= 128 and (shape[3] != 64 or shape[2] % 32):
            assert bits_equal(a.numpy(), b.numpy())


@pytest.mark.parametrize("D_", [36, 64, 80, 96, 100, 128])
@pytest.mark.parametrize("T", [1, 15, 17, 33, 49, 97, 130, 257])
def test_paired_ranges_at_ragged_lengths_and_other_head_dimensions(dev, T, D_):
    """The paired-range kernels where T is no multiple of 32 and D is not 64
    (a last query tile that is partly or wholly past T, columns past D, padded
    widths 64, 96 and 128), on strided q, k and v of a [B, T, 3, H, D]
    projection. Batch element 1 is NaN throughout, so a row or column read
    past the end of batch element 0 shows in its results; what lies between
    and after the written gradients keeps its value. Oracle and bar as above."""
    D, K = _dev()
    H = 3
    rng = np.random.default_rng(T * 131 + D_)
    qkv = np.full((2, T, 3, H, D_), np.nan, np.float32)
    qkv[0] = rng.standard_normal((T, 3, H, D_))
    g = np.full((2, T, H, D_), np.nan, np.float32)
    g[0] = rng.standard_normal((T, H, D_))
    q, k, v = (np.ascontiguousarray(qkv[:1, :, i].transpose(0, 2, 1, 3)) for i in range(3))
    gh = np.ascontiguousarray(g[:1].transpose(0, 2, 1, 3))
    o_ref, p, scale = ops.attention_fwd(q, k, v)
    refs = ops.attention_bwd(gh, q, k, v, p, scale)
    t5 = D.from_numpy(qkv).transpose(2, 0, 3, 1, 4)
    obuf = D.full((T + 1, 2, H, D_), 7.0, np.float32)
    ov = obuf[:T].transpose(1, 2, 0, 3)
    _, rmax, rsum = K.attn_fwd(t5[0], t5[1], t5[2], out=ov)
    dbuf = D.full((T + 1, 2, 3, H, D_), 7.0, np.float32)
    d5 = dbuf[:T].transpose(2, 1, 3, 0, 4)
    K.attn_bwd(t5[0], t5[1], t5[2], ov, D.from_numpy(g).transpose(0, 2, 1, 3), rmax, rsum,
               dq=d5[0], dk=d5[1], dv=d5[2])
    go, gd = obuf.numpy(), dbuf.numpy()
    tol = TOL[np.float32]
    assert rel_err(go[:T, :1].transpose(1, 2, 0, 3), o_ref) <= tol
    m_ref, l_ref = ops.row_stats(q, k)
    assert rel_err(rmax.numpy()[:1], m_ref * np.log2(np.e)) <= tol
    assert rel_err(rsum.numpy()[:1], l_ref) <= tol
    for i, ref in enumerate(refs):
        if T == 1 and i < 2:  # one key: dQ and dK are 0, what is left is rounding of dP - rowsum(dO * O)
            assert np.max(np.abs(gd[:T, 0, i])) <= tol
        else:
            assert rel_err(gd[:T, :1, i].transpose(1, 2, 0, 3), ref) <= tol
    assert np.all(go[T:] == 7.0) and np.all(gd[T:] == 7.0)


@pytest.mark.parametrize("T,D_", [(100, 36), (100, 64), (96, 64), (100, 80), (100, 96), (100, 128)])
def test_scores_of_minus_infinity(dev, T, D_):
    """Scores that overflow to -inf have probability 0, wherever they lie: the
    first keys that a query sees, the whole of a 16-key tile, or the one key
    that is unmasked in the first tile of one of a block's waves (key 16 w
    for query 16 w). A product q[i, d] k[j, d] of -9e40 in one of the first
    four dimensions makes them; in the oracle's float64 the score is finite
    and its probability 0 all the same. dQ and dK have entries of up to 3e20
    in those four dimensions, so each dimension is held against its own
    largest entry."""
    D, K = _dev()
    rng = np.random.default_rng(T + D_)
    q, k, v, g = (rng.standard_normal((1, 2, T, D_)).astype(np.float32) for _ in range(4))
    pairs = [((16,), (16,)), ((32,), (32,)), ((48,), (48,)), ((90, 91, 95), range(48))]
    q[..., :4] = k[..., :4] = 0
    for d, (qs, ks) in enumerate(pairs):
        q[:, :, list(qs), d] = 3e20
        k[:, :, list(ks), d] = -3e20
    o_ref, p, scale = ops.attention_fwd(q, k, v)
    refs = ops.attention_bwd(g, q, k, v, p, scale)
    m_ref, l_ref = ops.row_stats(q, k)
    dq_, dk_, dv_ = D.from_numpy(q), D.from_numpy(k), D.from_numpy(v)
    o, rmax, rsum = K.attn_fwd(dq_, dk_, dv_)
    tol = TOL[np.float32]
    assert rel_err(o.numpy(), o_ref) <= tol
    assert rel_err(rmax.numpy(), m_ref * np.log2(np.e)) <= tol
    assert rel_err(rsum.numpy(), l_ref) <= tol
    for got, ref in zip(K.attn_bwd(dq_, dk_, dv_, o, D.from_numpy(g), rmax, rsum), refs):
        for d in range(4):
            assert rel_err(got.numpy()[..., d], ref[..., d]) <= tol
        assert rel_err(got.numpy()[..., 4:], ref[..., 4:]) <= tol


@pytest.mark.parametrize("T,D_", [(100, 36), (100, 64), (96, 64), (100, 80), (130, 128)])
def test_keys_masked_by_an_infinite_feature(dev, T, D_):
    """A mask carried by a feature: 1 in every query, -inf in the masked keys and
    0 in the others. The masked keys' dK and dV are 0 and everything else is as
    without them (dQ's own entry of that feature is 0 * inf), also where the
    last query tile has rows past T, whose zeros times -inf are no numbers."""
    D, K = _dev()
    rng = np.random.default_rng(T + D_)
    q, k, v, g = (rng.standard_normal((1, 2, T, D_)).astype(np.float32) for _ in range(4))
    off = [3, 16, 17, 40, T - 1]
    q[..., 0], k[..., 0] = 1, 0
    k[:, :, off, 0] = -np.inf
    o_ref, p, scale = ops.attention_fwd(q, k, v)
    gq, gk, gv = ops.attention_bwd(g, q, k, v, p, scale)
    dq_, dk_, dv_ = D.from_numpy(q), D.from_numpy(k), D.from_numpy(v)
    o, rmax, rsum = K.attn_fwd(dq_, dk_, dv_)
    tol = TOL[np.float32]
    assert rel_err(o.numpy(), o_ref) <= tol
    dq, dk, dv = (x.numpy() for x in K.attn_bwd(dq_, dk_, dv_, o, D.from_numpy(g), rmax, rsum))
    assert rel_err(dq[..., 1:], gq[..., 1:]) <= tol
    assert rel_err(dk, gk) <= tol and rel_err(dv, gv) <= tol
    assert np.all(dk[:, :, off] == 0) and np.all(dv[:, :, off] == 0)


@pytest.mark.parametrize("D_", [80, 128])
def test_results_with_overlapping_rows_are_refused_above_64(dev, D_):
    """Output rows less than D apart: refused above D = 64 in the forward and the
    backward, in float32 as in float64."""
    D, K = _dev()
    T = 40
    for dt in (np.float32, np.float64):
        q, k, v, g = (D.full((1, 1, T, D_), 0.5, dt) for _ in range(4))
        bad = D.DeviceArray(D.full((T * D_,), 0.0, dt).block, (1, 1, T, D_), dt, 0, (0, 0, D_ - 16, 1))
        with pytest.raises(Exception, match="ldc"):
            K.attn_fwd(q, k, v, out=bad)
        o, rmax, rsum = K.attn_fwd(q, k, v)
        for i in range(3):
            with pytest.raises(Exception, match="ldc"):
                K.attn_bwd(q, k, v, o, g, rmax, rsum, **{("dq", "dk", "dv")[i]: bad})
