"""GPU parity of RMSNorm and one-token attention against the oracle, through
the C ABI.

Bar: bit-exact.  RMSNorm sums the squares in order (src/ops/norm.rs:25-28);
attention keeps the reference's in-order score sums, softmax_in_place and
the position-ordered context (src/model/attention.rs:31-86), so every
output of every position equals the oracle's bits.  The accumulation-order
tolerance (rel-L2 <= 1e-5) is asserted as well.
"""
import numpy as np
import pytest

import hale_moe as H
import oracle as O

pytestmark = pytest.mark.gpu

REL_L2 = 1e-5


def same_bits(a, b):
    a = np.ascontiguousarray(a, dtype=np.float32)
    b = np.ascontiguousarray(b, dtype=np.float32)
    return a.shape == b.shape and bool((a.view(np.uint32) == b.view(np.uint32)).all())


def rel_l2(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


@pytest.mark.parametrize("n", [1, 7, 64, 2048, 4096, 8192])
@pytest.mark.parametrize("eps", [1e-6, 0.0])
def test_rms_norm_bit_exact(ctx, n, eps):
    x = O.normal(n + 1, n, 0.0, 3.0)
    w = O.normal(n + 2, n, 1.0, 0.1)
    got = H.rms_norm(ctx, x, w, eps)
    want = O.rms_norm(x, w, eps)
    assert same_bits(got, want)


def test_rms_norm_reference_case_and_zero_row(ctx):
    x = np.array([3.0, -4.0, 0.0, 5.0], np.float32)
    got = H.rms_norm(ctx, x, np.ones(4, np.float32), 0.0)
    assert same_bits(got, O.rms_norm(x, np.ones(4, np.float32), 0.0))
    z = H.rms_norm(ctx, np.zeros(64, np.float32), np.ones(64, np.float32), 1e-6)
    assert same_bits(z, O.rms_norm(np.zeros(64, np.float32), np.ones(64, np.float32), 1e-6))
    with pytest.raises(ValueError):
        H.rms_norm(ctx, np.zeros(8193, np.float32), np.ones(8193, np.float32), 1e-6)


def squares_case(kind, n):
    """Rows whose sum of squares meets the cases of the lanes' ordered sum:
    every square half-way between two results (ties to even), values of all
    binades, a first square of an exact power of two above all the rest,
    zeros, a sum that becomes infinite, a NaN."""
    g = np.random.default_rng(n * 31 + len(kind))
    if kind == "normal":
        return g.standard_normal(n).astype(np.float32)
    if kind == "ties":
        return (g.integers(0, 4, n) * np.where(g.random(n) < 0.1, 4096.0, 1.0)).astype(np.float32)
    if kind == "binades":
        return np.exp(g.uniform(-45, 40, n)).astype(np.float32)
    if kind == "growing":
        return np.exp(np.linspace(-43, 43, n)).astype(np.float32)
    if kind == "sink":
        x = (g.random(n) * 1e-3).astype(np.float32)
        x[0] = 1.0
        return x
    if kind == "zeros":
        return np.where(g.random(n) < 0.02, g.standard_normal(n), 0.0).astype(np.float32)
    x = g.standard_normal(n).astype(np.float32)
    x[n // 2] = 1e20 if kind == "inf" else np.nan
    return x


@pytest.mark.parametrize("kind", ["normal", "ties", "binades", "growing", "sink", "zeros", "inf", "nan"])
def test_rms_norm_ordered_sum_edges(ctx, kind):
    for n in (1, 3, 64, 65, 255, 256, 257, 1000, 1024, 1025, 2047, 2048, 2049, 3001, 4096, 4097, 5120, 8191, 8192):
        x = squares_case(kind, n)
        w = O.normal(n + 2, n, 1.0, 0.1)
        got, want = H.rms_norm(ctx, x, w, 1e-6), O.rms_norm(x, w, 1e-6)
        assert (np.isnan(got) == np.isnan(want)).all(), n
        ok = ~np.isnan(want)
        assert same_bits(got[ok], want[ok]), n


def test_residual_rms_norm_rows_on_device(ctx):
    rows, n = 5, 2048
    x = O.normal(31, rows * n)
    d = O.normal(32, rows * n)
    w = O.normal(33, n, 1.0, 0.1)
    bx, bd, bw, bo = ctx.malloc(x.nbytes), ctx.malloc(d.nbytes), ctx.malloc(w.nbytes), ctx.malloc(x.nbytes)
    bx.upload(x)
    bd.upload(d)
    bw.upload(w)
    ctx.check(H.lib().hale_rms_norm_device(ctx.handle, H._vp(bx.address), H._vp(bd.address),
                                           H._vp(bw.address), rows, n, np.float32(1e-6),
                                           H._vp(bo.address)), "rms_norm")
    xs = bx.download(np.float32, rows * n).reshape(rows, n)
    got = bo.download(np.float32, rows * n).reshape(rows, n)
    want_x = (x + d).reshape(rows, n)  # add_in_place, one rounding per element
    assert same_bits(xs, want_x)
    for r in range(rows):
        assert same_bits(got[r], O.rms_norm(want_x[r], w, 1e-6))
    for b in (bx, bd, bw, bo):
        b.free()


def build(ctx, dtype, Hd, nh, nkv, hd, seed, qk_norm, max_len):
    mats, gm = [], []
    for j, (r, c) in enumerate(((nh * hd, Hd), (nkv * hd, Hd), (nkv * hd, Hd), (Hd, nh * hd))):
        m = O.encode_matrix(dtype, O.normal(seed + j, r * c, 0.0, 0.05).reshape(r, c))
        mats.append(m)
        gm.append(H.WeightMatrix.new(ctx, r, c, dtype, m))
    qn = kn = None
    if qk_norm:
        qn, kn = O.normal(seed + 10, hd, 1.0, 0.1), O.normal(seed + 11, hd, 1.0, 0.1)
    if qk_norm == "q":
        kn = None
    if qk_norm == "k":
        qn = None
    ref = O.OracleAttention(dtype, Hd, nh, nkv, hd, 1e-6, *mats, q_norm=qn, k_norm=kn, max_len=max_len)
    att = H.Attention(ctx, *gm, qn, kn, nh, nkv, hd, 1e-6, max_len=max_len)
    return ref, att


@pytest.mark.parametrize("dtype,Hd,nh,nkv,hd,qk,steps", [
    (O.F32, 64, 4, 2, 16, True, 40),            # small, GQA group 2
    (O.BF16, 2048, 32, 4, 128, True, 24),       # Qwen3-30B-A3B attention shape
    (O.Q8_0, 2048, 32, 4, 128, True, 12),
    (O.Q4_0, 4096, 32, 8, 128, False, 10),      # Mixtral shape, no QK-norm
])
def test_attention_decode_bit_exact(ctx, dtype, Hd, nh, nkv, hd, qk, steps):
    ref, att = build(ctx, dtype, Hd, nh, nkv, hd, seed=Hd + nh, qk_norm=qk, max_len=64)
    for pos in range(steps):
        x = O.normal(1000 + pos, Hd)
        c, s = O.rope_angles(hd, 1e6, pos)
        got = att.forward(x, pos, c, s)
        want = ref.forward(x, c, s)
        assert rel_l2(got, want) <= REL_L2
        assert same_bits(got, want), (dtype, pos)
    assert len(att) == steps
    att.close()


@pytest.mark.parametrize("dtype,Hd,nh,nkv,hd", [
    (O.Q8_0, 1024, 6, 2, 80),    # 480 and 160 rows: padded to 512 and 192, three matrices in one launch
    (O.Q4_0, 1056, 4, 2, 48),    # 33-block rows, 96-row key and value matrices
    (O.Q8_0, 4096, 32, 8, 128),  # 6144 rows: 32-row work-groups for all three
    (O.Q4_0, 512, 4, 2, 64),     # 16-block rows: one launch each
    (O.F16, 260, 3, 1, 80),      # rows that no 16-byte piece divides
    (O.F32, 64, 5, 5, 16),       # 80 rows each: ten work-groups per matrix
])
def test_attention_projections_together(ctx, dtype, Hd, nh, nkv, hd):
    ref, att = build(ctx, dtype, Hd, nh, nkv, hd, seed=Hd + hd, qk_norm=False, max_len=4)
    for pos in range(4):
        x = O.normal(700 + pos, Hd)
        c, s = O.rope_angles(hd, 1e6, pos)
        assert same_bits(att.forward(x, pos, c, s), ref.forward(x, c, s)), pos
    att.close()


@pytest.mark.parametrize("norms", ["q", "k", ""])
@pytest.mark.parametrize("hd", [128, 144])
def test_attention_one_sided_norms(ctx, norms, hd):
    # only the queries normed, only the keys, or neither (then no wave sums
    # squares), in the one launch for short rows and in the score kernel for
    # longer ones; heads of one register pass and with a remainder of 16
    ref, att = build(ctx, O.F32, 64, 3, 1, hd, seed=hd, qk_norm=norms, max_len=1030)
    for pos in range(1030):
        x = O.normal(7000 + pos, 64, 0.0, 3.0)
        c, s = O.rope_angles(hd, 1e6, pos)
        got = att.forward(x, pos, c, s)
        want = ref.forward(x, c, s)
        if pos < 4 or pos % 200 == 0 or pos >= 1022:
            assert same_bits(got, want), pos
    att.close()


@pytest.mark.parametrize("nh,nkv,hd", [(8, 2, 32), (16, 2, 16), (16, 1, 16), (6, 2, 16), (4, 4, 16)])
def test_attention_long_context(ctx, nh, nkv, hd):
    # 1100 positions with GQA groups of 4, 8, 16, 3 and 1: rows of one launch,
    # then 18 score blocks of 64 positions and context passes over nine
    # 128-position tiles, so every register stage of the value stream is
    # refilled and the three LDS buffers alternate; group 16 takes two score
    # work-groups, groups 3 and 1 leave a score wave with one query head
    ref, att = build(ctx, O.BF16, 256, nh, nkv, hd, seed=77, qk_norm=True, max_len=1100)
    for pos in range(1100):
        x = O.normal(5000 + pos, 256)
        c, s = O.rope_angles(hd, 1e6, pos)
        got = att.forward(x, pos, c, s)
        want = ref.forward(x, c, s)
        if pos % 100 == 99 or pos == 1099:
            assert same_bits(got, want), pos
    att.close()


@pytest.mark.parametrize("nh,nkv,hd,qk,steps", [
    (8, 1, 128, True, 1100),   # one launch to 768 positions, then two key chunks per score wave
    (8, 1, 128, False, 520),   # one launch to 512
    (3, 1, 272, True, 1100),   # one launch to 512, then both key register sets refilled
    (5, 5, 144, True, 800),
    (8, 2, 1024, True, 520),   # 256 work-groups
    (9, 1, 1024, True, 140),   # 288: scores and context in two launches from the first position
    (16, 2, 528, False, 70),   # 272, heads whose last column block is half full
])
def test_attention_one_or_two_launches(ctx, nh, nkv, hd, qk, steps):
    ref, att = build(ctx, O.F32, 64, nh, nkv, hd, seed=nh + hd, qk_norm=qk, max_len=steps)
    edges = {n - 1 for c in (1, 64, 128, 512, 768, 1024, 1088) for n in (c, c + 1, c + 2)}
    for pos in range(steps):
        x = O.normal(3000 + pos, 64, 0.0, 3.0)
        c, s = O.rope_angles(hd, 1e6, pos)
        got = att.forward(x, pos, c, s)
        want = ref.forward(x, c, s)
        if pos in edges or pos == steps - 1:
            assert same_bits(got, want), pos
    att.close()


@pytest.mark.parametrize("nh,nkv,hd,steps", [(2, 1, 80, 2060), (3, 1, 272, 600), (2, 2, 16, 4100)])
def test_attention_softmax_context_edges(ctx, nh, nkv, hd, steps):
    # both sides of the row lengths that pick the values per lane of the
    # ordered sum, of the 128-position tiles and of their 64-position batches,
    # and of the rows that one launch takes (512, 768), with head sizes whose last
    # column block is half full and whose keys fill several chunks of 64
    ref, att = build(ctx, O.F32, 64, nh, nkv, hd, seed=hd, qk_norm=True, max_len=steps)
    edges = {n - 1 for c in (1, 32, 64, 128, 192, 256, 384, 512, 1024, 2048, 4096) for n in (c, c + 1, c + 2)}
    for pos in range(steps):
        x = O.normal(9000 + pos, 64, 0.0, 3.0)
        c, s = O.rope_angles(hd, 1e6, pos)
        got = att.forward(x, pos, c, s)
        want = ref.forward(x, c, s)
        if pos in edges or pos == steps - 1:
            assert same_bits(got, want), pos
    att.close()


def test_attention_softmax_past_one_lds_chunk(ctx):
    # rows up to 8192 positions run softmax and context in one kernel, longer
    # ones in two; a score row longer than the softmax keeps in LDS (12288)
    # goes through global memory in chunks: positions on both sides of both
    # limits
    ref, att = build(ctx, O.F32, 64, 4, 2, 16, seed=91, qk_norm=False, max_len=12300)
    for pos in range(12300):
        x = O.normal(100 + pos, 64)
        c, s = O.rope_angles(16, 1e6, pos)
        got = att.forward(x, pos, c, s)
        want = ref.forward(x, c, s)
        if pos in (8190, 8191, 8192, 12286, 12287, 12288, 12299):
            assert same_bits(got, want), pos
    att.close()


def test_attention_position_rules(ctx):
    ref, att = build(ctx, O.F32, 64, 4, 2, 16, seed=3, qk_norm=False, max_len=2)
    c, s = O.rope_angles(16, 1e6, 0)
    x = O.normal(1, 64)
    with pytest.raises(ValueError, match="cache holds 0"):
        att.forward(x, 1, c, s)                 # position must equal the cache length
    att.forward(x, 0, c, s)
    att.forward(x, 1, c, s)
    with pytest.raises(ValueError, match="context overflow"):
        att.forward(x, 2, c, s)
    att.reset()
    assert len(att) == 0
    assert same_bits(att.forward(x, 0, c, s), ref.forward(x, c, s))
    att.close()
