"""GPU parity of the attention kernels against the CPU oracle."""
import ctypes as C

import numpy as np
import pytest

from conftest import TOL, compute_units

pytestmark = pytest.mark.gpu


def _qkv(O, H, Lq, Lk, D, seed=0):
    return (O.fill_normal_f16((H, Lq, D), seed, 0, 1.0), O.fill_normal_f16((H, Lk, D), seed, 1, 1.0),
            O.fill_normal_f16((H, Lk, D), seed, 2, 1.0))


# config 3 decode: 32 heads x 64, kv = 1024; plus short / ragged lengths and the 2048 limit
@pytest.mark.parametrize("kv", [1, 2, 7, 8, 9, 63, 100, 1024, 2047, 2048])
def test_single_masked_sdpa(moon, O, ctx, kv):
    q, k, v = _qkv(O, 32, 1, kv, 64)
    mask = np.ones((1, 1, kv), dtype=bool)
    out = moon.attention.single_masked_sdpa(q, k, v, mask, ctx=ctx)
    assert O.rel_frobenius(out, O.sdpa_single(q, k, v, mask)) <= TOL


def test_single_masked_sdpa_with_holes_and_limit(moon, O, ctx):
    q, k, v = _qkv(O, 32, 1, 300, 64)
    mask = np.ones((1, 1, 300), dtype=bool)
    mask[0, 0, 10:200:3] = False
    out = moon.attention.single_masked_sdpa(q, k, v, mask, ctx=ctx)
    assert O.rel_frobenius(out, O.sdpa_single(q, k, v, mask)) <= TOL
    q, k, v = _qkv(O, 32, 1, 2049, 64)
    with pytest.raises(moon.SequenceTooLong):  # attention.zig:769
        moon.attention.single_masked_sdpa(q, k, v, np.ones((1, 1, 2049), dtype=bool), ctx=ctx)


# config 3 prefill: causal 768; continuation (pos > 0); tiny and ragged cases
@pytest.mark.parametrize("H,S,pos,D", [(32, 768, 0, 64), (32, 39, 729, 64), (4, 5, 0, 64), (2, 130, 3, 64), (3, 17, 0, 32)])
def test_multi_masked_sdpa_causal(moon, O, ctx, H, S, pos, D):
    q, k, v = _qkv(O, H, S, pos + S, D)
    mask = moon.attention.create_attention_mask(pos, S)
    assert np.array_equal(mask, O.attention_mask(pos, S))
    out = moon.attention.multi_masked_sdpa(q, k, v, mask, H, D, ctx=ctx)
    assert O.rel_frobenius(out, O.sdpa_multi(q, k, v, mask)) <= TOL


def test_multi_masked_sdpa_arbitrary_mask(moon, O, ctx):
    H, S, D = 4, 70, 64
    q, k, v = _qkv(O, H, S, S, D)
    rng = np.random.default_rng(0)
    mask = rng.random((1, S, S)) < 0.7
    mask[0, np.arange(S), np.arange(S)] = True  # no fully masked row
    out = moon.attention.multi_masked_sdpa(q, k, v, mask, H, D, ctx=ctx)
    assert O.rel_frobenius(out, O.sdpa_multi(q, k, v, mask)) <= TOL


# config 4 attention: 16 heads x 72, 729 tokens (and the reference's duplicated-crop 1458)
@pytest.mark.parametrize("H,L,D", [(16, 729, 72), (16, 1458, 72), (2, 50, 72), (1, 1, 72), (3, 65, 64)])
def test_multi_maskless_sdpa(moon, O, ctx, H, L, D):
    q, k, v = _qkv(O, H, L, L, D)
    out = moon.attention.multi_maskless_sdpa(H, D, q, k, v, ctx=ctx)
    assert O.rel_frobenius(out, O.sdpa_multi(q, k, v, None)) <= TOL


def test_duplicated_keys_leave_output_unchanged(moon, O, ctx):
    # the reference encodes the same crop twice and attends jointly over 2x729 tokens (vision_model.zig:36-38,308-310)
    q, k, v = _qkv(O, 16, 100, 100, 72)
    one = moon.attention.multi_maskless_sdpa(16, 72, q, k, v, ctx=ctx)
    two = moon.attention.multi_maskless_sdpa(16, 72, q, np.concatenate([k, k], 1), np.concatenate([v, v], 1), ctx=ctx)
    assert O.rel_frobenius(two, one) <= TOL


@pytest.mark.parametrize("pos", [0, 1, 8, 100, 1023, 2047])
def test_fused_decode_attention_step(moon, O, ctx, pos):
    """rope(q,k) + cache append + attention over pos+1 keys, on a cache in the reference layout."""
    H, D, rot, S = 32, 64, 32, 2048
    qkv = O.fill_normal_f16((3 * H * D,), 0, 0, 1.0)
    ck = np.zeros((H, S, D), dtype=np.float16)
    cv = np.zeros((H, S, D), dtype=np.float16)
    ck[:, :pos] = O.fill_normal_f16((H, pos, D), 0, 1, 1.0)
    cv[:, :pos] = O.fill_normal_f16((H, pos, D), 0, 2, 1.0)
    table = O.rope_table(rot, S, 10000.0)
    # oracle: text_model.zig:198-286
    q, k, v = (O.split_heads(qkv.reshape(1, -1), i, H, D) for i in range(3))
    pid = np.array([pos])
    qr, kr = O.rope_apply(q, table, pid, rot), O.rope_apply(k, table, pid, rot)
    ck_ref, cv_ref = ck.copy(), cv.copy()
    ck_ref[:, pos] = kr[:, 0]
    cv_ref[:, pos] = v[:, 0]
    want = O.merge_heads(O.sdpa_single(qr, np.ascontiguousarray(ck_ref[:, :pos + 1]), np.ascontiguousarray(cv_ref[:, :pos + 1]),
                                       np.ones((1, 1, pos + 1), bool)))
    d_qkv, d_ck, d_cv, d_tab = ctx.to_device(qkv), ctx.to_device(ck), ctx.to_device(cv), ctx.to_device(table)
    d_out = ctx.alloc(H * D * 2)
    ctx.check(ctx.lib.moon_dev_decode_attention(ctx.handle, d_qkv.ptr, d_ck.ptr, d_cv.ptr, d_tab.ptr, d_out.ptr, H, D, rot, S, pos))
    ctx.sync()
    got = d_out.to_host((1, H * D))
    assert O.rel_frobenius(got, want) <= TOL
    # the append wrote exactly k' and v at position pos and nothing else
    assert O.rel_frobenius(d_ck.to_host((H, S, D))[:, pos], ck_ref[:, pos]) <= TOL
    assert np.array_equal(d_cv.to_host((H, S, D)), cv_ref)
    got_ck = d_ck.to_host((H, S, D))
    got_ck[:, pos] = 0
    ck[:, pos] = 0
    assert np.array_equal(got_ck, ck)


@pytest.mark.parametrize("H,S,pos,D", [(2, 16, 0, 64), (2, 33, 31, 64), (1, 64, 0, 64), (3, 65, 1, 64), (2, 257, 300, 64),
                                       (2, 96, 64, 72), (1, 31, 0, 72), (2, 200, 0, 72)])
def test_matrix_core_attention_edge_shapes_causal(moon, O, ctx, H, S, pos, D):
    """Query blocks of 32 and key tiles of 64 with ragged ends, causal with and without a cached prefix."""
    q, k, v = _qkv(O, H, S, pos + S, D)
    mask = moon.attention.create_attention_mask(pos, S)
    out = moon.attention.multi_masked_sdpa(q, k, v, mask, H, D, ctx=ctx)
    err = O.rel_frobenius(out, O.sdpa_multi(q, k, v, mask))
    print(f"causal H={H} S={S} pos={pos} D={D}: rel-Frobenius {err:.2e}")
    assert err <= TOL


@pytest.mark.parametrize("H,Lq,Lkv,D", [(2, 16, 1, 64), (2, 40, 63, 64), (2, 40, 64, 64), (2, 40, 65, 64), (1, 100, 257, 72), (2, 729, 300, 72)])
def test_matrix_core_attention_rectangular_maskless(moon, O, ctx, H, Lq, Lkv, D):
    q = O.fill_normal_f16((H, Lq, D), 0, 1, 1.0)
    k = O.fill_normal_f16((H, Lkv, D), 0, 2, 1.0)
    v = O.fill_normal_f16((H, Lkv, D), 0, 3, 1.0)
    out = moon.attention.multi_maskless_sdpa(H, D, q, k, v, ctx=ctx)
    err = O.rel_frobenius(out, O.sdpa_multi(q, k, v, None))
    print(f"maskless H={H} Lq={Lq} Lkv={Lkv} D={D}: rel-Frobenius {err:.2e}")
    assert err <= TOL


def test_matrix_core_attention_peaked_softmax(moon, O, ctx):
    """Large score spread (one key dominates most rows): the running maximum has to rescale correctly."""
    H, L, D = 2, 300, 64
    q = O.fill_normal_f16((H, L, D), 0, 1, 4.0)
    k = O.fill_normal_f16((H, L, D), 0, 2, 4.0)
    v = O.fill_normal_f16((H, L, D), 0, 3, 1.0)
    out = moon.attention.multi_maskless_sdpa(H, D, q, k, v, ctx=ctx)
    assert np.isfinite(out.astype(np.float32)).all()
    assert O.rel_frobenius(out, O.sdpa_multi(q, k, v, None)) <= TOL


def test_matrix_core_attention_over_seeded_random_shapes(moon, O, ctx):
    """The matrix-core kernel over shapes no other test names: head counts 1..32 (multiples of 8 take the die-wise work
    mapping), 16..300 rows, head_dim 64 (causal with a past, and maskless) and 72, keys not a multiple of the 64-key tile."""
    rng = np.random.default_rng(1)
    worst = 0.0
    for it in range(48):
        D = 72 if it % 2 else 64
        H = int(rng.integers(1, 9)) if it % 5 else 8 * int(rng.integers(1, 5))
        S = int(rng.integers(16, 300))
        q = O.fill_normal_f16((H, S, D), it, 0, 1.0)
        if D == 64 and it % 3 == 0:
            pos = int(rng.integers(0, 200))
            k, v = O.fill_normal_f16((H, pos + S, D), it, 1, 1.0), O.fill_normal_f16((H, pos + S, D), it, 2, 1.0)
            mask = moon.attention.create_attention_mask(pos, S)
            out, want = moon.attention.multi_masked_sdpa(q, k, v, mask, H, D, ctx=ctx), O.sdpa_multi(q, k, v, mask)
        else:
            k, v = O.fill_normal_f16((H, S, D), it, 1, 1.0), O.fill_normal_f16((H, S, D), it, 2, 1.0)
            out, want = moon.attention.multi_maskless_sdpa(H, D, q, k, v, ctx=ctx), O.sdpa_multi(q, k, v, None)
        err = O.rel_frobenius(out, want)
        assert err <= TOL, (it, D, H, S, err)
        worst = max(worst, err)
    print(f"\nworst rel-Frobenius over 48 shapes: {worst:.2e}")


def form(H, rows, D, causal):
    """The kernel that a call of many rows takes."""
    cus = compute_units()
    if not (H * rows >= 112 * cus if causal else H * rows > (96 if D == 64 else 64) * cus):
        return f"flash_attn_kernel<{D}>"
    return f"flash_attn{96 if D == 72 and not causal and H * -(-rows // 96) <= cus else 64}_kernel<{D}>"


# 64 rows per workgroup where all heads together have more than 64 rows for each compute unit (heads of 64: 96; causal: at least 112),
# 32 below (on 256 units 32 heads cross the line behind 512, 768 and 895 rows); the last block of 64 with 1, 32, 33 and 64 rows.
# Heads of 72 take 96 rows as long as there is a compute unit for every 96 (32 heads: up to 768 rows).
@pytest.mark.parametrize("S,D,pos", [(511, 72, None), (512, 72, None), (513, 72, None), (544, 64, None), (545, 72, None), (767, 64, 62), (768, 64, 0),
                                     (769, 64, 62), (800, 64, 1), (801, 64, 62), (544, 72, None), (576, 72, None), (768, 64, None), (769, 64, None), (800, 64, None),
                                     (832, 64, None), (895, 64, 62), (896, 64, 0), (897, 64, 62), (928, 64, 1), (929, 64, 62), (960, 64, 0),
                                     (768, 72, None), (769, 72, None), (800, 72, None), (801, 72, None), (832, 72, None)])
def test_both_row_blocks_of_the_matrix_core_attention(moon, O, ctx, S, D, pos):
    """Scores that grow along the keys, from far below one to tens: every tile raises the maximum of its rows."""
    H, L = 32, S + (pos or 0)
    q, k, v = _qkv(O, H, S, L, D)
    k = (k.astype(np.float32) * np.linspace(0.02, 5.0, L, dtype=np.float32)[:, None]).astype(np.float16)
    if pos is None:
        out, want = moon.attention.multi_maskless_sdpa(H, D, q, k, v, ctx=ctx), O.sdpa_multi(q, k, v, None)
    else:
        mask = moon.attention.create_attention_mask(pos, S)
        out, want = moon.attention.multi_masked_sdpa(q, k, v, mask, H, D, ctx=ctx), O.sdpa_multi(q, k, v, mask)
    assert O.rel_frobenius(out, want) <= TOL
    assert ctx.last_kernel().split(" ")[0] == form(H, S, D, pos is not None)


@pytest.mark.parametrize("D,causal", [(64, False), (64, True), (72, False)])
def test_values_that_are_not_finite_meet_the_same_rows_in_both_row_blocks(moon, O, ctx, D, causal):
    """Infinities and NaN among queries, keys and values: calls of 64 rows (32 per workgroup) against one of all rows (64), bit for bit."""
    H, L = 32, 1041  # (the last part has 17 rows, enough for the matrix-core kernels)
    q, k, v = _qkv(O, H, L, L, D)
    q[:, 17], q[:, 77, 5], k[:, 300, 0] = np.nan, np.inf, np.inf
    v[:8, 200, 3], v[:8, 700, 5], v[8:16, 1040, 1] = np.inf, np.nan, -np.inf

    def rows(lo, hi):
        if not causal:
            return moon.attention.multi_maskless_sdpa(H, D, np.ascontiguousarray(q[:, lo:hi]), k, v, ctx=ctx)
        cut = [np.ascontiguousarray(a) for a in (q[:, lo:hi], k[:, :hi], v[:, :hi])]
        return moon.attention.multi_masked_sdpa(*cut, moon.attention.create_attention_mask(lo, hi - lo), H, D, ctx=ctx)

    whole = rows(0, L)
    assert ctx.last_kernel().split(" ")[0] == f"flash_attn64_kernel<{D}>"
    parts = []
    for lo in range(0, L, 64):
        parts.append(rows(lo, min(lo + 64, L)))
        assert ctx.last_kernel().startswith("flash_attn_kernel")
    parts = np.concatenate(parts, axis=1)
    assert 0.2 < np.isfinite(whole).mean() < 0.999
    assert np.array_equal(whole, parts, equal_nan=True)


# 96 rows per workgroup where they fit one round and 64 are more than 32 rows fit; the last block with 1, 32, 33, 64, 65 and 96 rows
@pytest.mark.parametrize("H,Lq,Lkv", [(16, 1025, 1025), (16, 1056, 63), (16, 1057, 64), (16, 1440, 65), (16, 1441, 300), (16, 1458, 1458), (16, 1536, 256), (32, 513, 700),
                                      (32, 768, 1), (8, 2112, 129), (5, 3300, 100)])
def test_row_blocks_that_share_tiles_give_the_same_bits(moon, ctx, H, Lq, Lkv):
    """Scores that grow along the keys, some values that are not finite: one call of all rows against calls of 64 (32 per workgroup)."""
    rng = np.random.default_rng(Lq)
    q, k, v = (rng.standard_normal((H, n, 72), dtype=np.float32) for n in (Lq, Lkv, Lkv))
    k *= np.linspace(0.02, 5.0, Lkv, dtype=np.float32)[:, None]
    q, k, v = (a.astype(np.float16) for a in (q, k, v))
    q[0, 17], v[1, Lkv // 2, 3], v[2, Lkv - 1, 5] = np.nan, np.inf, np.nan
    whole = moon.attention.multi_maskless_sdpa(H, 72, q, k, v, ctx=ctx)
    if compute_units() == 256:
        assert ctx.last_kernel().startswith("flash_attn96_kernel<72> ")
    parts = []
    for lo in range(0, Lq, 64):
        lo = min(lo, Lq - 16)  # (fewer rows take another kernel)
        parts.append((lo, moon.attention.multi_maskless_sdpa(H, 72, np.ascontiguousarray(q[:, lo:lo + 64]), k, v, ctx=ctx)))
        assert ctx.last_kernel().startswith("flash_attn_kernel")
    for lo, part in parts:
        assert np.array_equal(whole[:, lo:lo + 64], part, equal_nan=True)


@pytest.mark.parametrize("D", [64, 72])
def test_the_last_tile_reads_nothing_that_an_earlier_call_left(moon, O, ctx, D):
    """The 64-row kernel's last tile is cut off in memory; what lies behind the keys in LDS has weight 0 and must be a number."""
    H, L = 32, 1030
    q, k, v = _qkv(O, H, L, L, D)
    bad = np.full_like(v, np.nan)
    moon.attention.multi_maskless_sdpa(H, D, q, bad, bad, ctx=ctx)
    out = moon.attention.multi_maskless_sdpa(H, D, q, k, v, ctx=ctx)
    assert ctx.last_kernel().split(" ")[0] == f"flash_attn64_kernel<{D}>"
    assert O.rel_frobenius(out, O.sdpa_multi(q, k, v, None)) <= TOL


@pytest.mark.parametrize("D", [64, 72])
@pytest.mark.parametrize("rows", [64, 16384, 16416, 24608])  # on 256 units 32 rows per workgroup up to 16,384, then heads of 72 take 96, and behind 24,576 rows all take 64
@pytest.mark.parametrize("units", [1.45, 0.49])  # a probability, in steps of f16 below its normal range: rounded, it would count as one of them or none
def test_matrix_core_attention_sums_probabilities_in_f32(moon, ctx, rows, D, units):
    """One key whose value is 1 and many faint ones of value 0: the result is the reciprocal of the softmax denominator, 1 + keys x p.
    Limit: half a step of the f16 result (2^-12 below 1) and 1 % of the faint keys' share for the exponent's f32 rounding."""
    keys = 1 << 15
    faint = np.float16(np.log(units * 2.0**-24) * D**0.5)
    p = np.exp(float(faint) * D**-0.5)
    assert abs(p * 2**24 / units - 1) < 0.02  # (the score is a step of f16 away at most)
    q, k, v = [np.zeros((1, n, D), np.float16) for n in (rows, keys, keys)]
    q[..., 0] = 1.0
    k[:, 1:, 0] = faint
    v[:, 0] = 1.0
    out = moon.attention.multi_maskless_sdpa(1, D, q, k, v, ctx=ctx)
    assert ctx.last_kernel().split(" ")[0] == form(1, rows, D, False)
    want = 1.0 / (1.0 + (keys - 1) * p)
    assert np.abs(out.astype(np.float64) - want).max() <= 2.0**-12 + 0.01 * (1.0 - want)


def test_decode_attention_after_cleanup_starts_from_fresh_counters(moon, O, ctx):
    """moon_cleanup frees the workspace that holds the per-head counters of the one-launch decode attention
    (cleanupThreadPool, attention.zig:814).  The next call gets new memory, whatever it holds, at whatever address, and must
    give the same bits as before: counters that were believed to be still cleared would make the merge run early or never."""
    H, D, rot, S, pos = 32, 64, 32, 2048, 300
    qkv = O.fill_normal_f16((3 * H * D,), 0, 10, 1.0)
    ck = np.zeros((H, S, D), dtype=np.float16)
    cv = np.zeros((H, S, D), dtype=np.float16)
    ck[:, :pos] = O.fill_normal_f16((H, pos, D), 0, 11, 1.0)
    cv[:, :pos] = O.fill_normal_f16((H, pos, D), 0, 12, 1.0)
    d_qkv, d_tab = ctx.to_device(qkv), ctx.to_device(O.rope_table(rot, S, 10000.0))
    d_out = ctx.alloc(H * D * 2)

    def step():
        d_ck, d_cv = ctx.to_device(ck), ctx.to_device(cv)
        ctx.check(ctx.lib.moon_dev_decode_attention(ctx.handle, d_qkv.ptr, d_ck.ptr, d_cv.ptr, d_tab.ptr, d_out.ptr, H, D, rot, S, pos))
        ctx.sync()
        return d_out.to_host((1, H * D))

    first = step()
    assert np.array_equal(step(), first)  # the counters count on from launch to launch
    for nbytes in (1 << 16, 1 << 18, 1 << 20, 1 << 22):
        ctx.cleanup()
        junk = [ctx.to_device(np.full(nbytes, 0xFF, dtype=np.uint8)) for _ in range(4)]  # what freed memory may come back as
        del junk
        assert np.array_equal(step(), first)
        assert np.array_equal(step(), first)
