"""GPU parity of the wide (192 / 256 x 256) and thin (128 x 64) f16 product tiles against the CPU oracle: by themselves where they are
named, and where a decoder's prompt takes them (q, k, v with their rotation beside fc1; out_proj beside fc2)."""
import numpy as np
import pytest

from conftest import TOL

pytestmark = pytest.mark.gpu


# The tiles' edges in rows and columns (a lone row and the last of a tile, one more), columns that are no whole pieces of 64 or 256, and
# one to seven k-tiles (the thin kernel's ring holds six).  TOL is the bar of every f16 product here: one rounding of f32 sums.
@pytest.mark.parametrize("kernel", ["b192", "b256", "thin"])
@pytest.mark.parametrize("M,N,K,epi", [(2, 8, 64, "none"), (63, 64, 128, "bias"), (127, 72, 448, "bias_gelu"), (128, 256, 384, "bias"), (129, 264, 64, "bias_gelu"),
                                       (191, 248, 192, "none"), (192, 520, 320, "bias"), (193, 512, 128, "bias_gelu"), (255, 200, 192, "bias"),
                                       (256, 256, 256, "none"), (257, 328, 64, "bias"), (385, 1032, 448, "bias_gelu"), (513, 136, 128, "none")])
def test_named_tiles_at_their_edges(moon, O, ctx, kernel, M, N, K, epi):
    L = moon._lib
    a = O.fill_normal_f16((M, K), 0, 0, 1.0)
    w = O.fill_normal_f16((N, K), 0, 1, 0.05)
    b = O.fill_normal_f16((N,), 0, 2, 0.1)
    code = {"none": L.EPI_NONE, "bias": L.EPI_BIAS, "bias_gelu": L.EPI_BIAS_GELU}[epi]
    got = np.empty((M, N), dtype=np.float16)
    ctx.set_gemm_kernel(kernel)
    try:
        ctx.check(ctx.lib.moon_linear(ctx.handle, a.ctypes.data, M, K, w.ctypes.data, N, L.B_NK, b.ctypes.data if epi != "none" else None, code, got.ctypes.data))
        took = ctx.last_kernel()
    finally:
        ctx.set_gemm_kernel("")
    assert ("thin" if kernel == "thin" else "block") in took
    ref = O.hgemm_trans(a, w)
    if epi != "none":
        ref = O.bias_add(ref, b)
    if epi == "bias_gelu":
        ref = O.gelu(ref)
    assert O.rel_frobenius(got, ref) <= TOL
    # No row or column drowns in the norm of all: sums in another order move each of at most three roundings (product, bias, GELU, whose
    # slope stays below 1.13) by one step of f16 at the largest value, 2^-10 of it.
    far = np.abs(got.astype(np.float32) - ref.astype(np.float32)).max()
    assert far <= 4 * 2.0**-10 * np.abs(ref.astype(np.float32)).max()


# Prompts in pieces, each behind the ones before it, at the tiles' edges: two rows, a row short of a thin tile, a whole one, one and two
# rows more, the last size of thin pairs (191) and the first of tall ones, a feed-forward whose width is no whole k-tile (its product
# is not paired, and its last columns are no whole tile), at width 2048 the pair in 192 x 256 tiles, and heads of which other parts than the
# first half turn (the projection is written, the rotation a launch of its own).
@pytest.mark.parametrize("dim,hidden,heads,rot,pieces", [(512, 2048, 8, 32, (2, 127, 128, 129, 65)), (512, 2048, 8, 32, (191, 192, 193, 257)), (192, 776, 3, 32, (130, 37, 385)),
                                                         (192, 832, 3, 32, (64, 129, 513)), (2048, 8192, 32, 32, (1025, 37)), (512, 2048, 8, 64, (37, 128, 700)),
                                                         (192, 776, 3, 6, (129, 193)), (2048, 8192, 32, 16, (769,))])
def test_prompts_at_the_edges_of_the_tiles(moon, O, ctx, dim, hidden, heads, rot, pieces):
    cfg = dict(O.TEXT_CFG, vocab=1024, dim=dim, hidden_dim=hidden, n_layers=2, n_heads=heads, head_dim=64, rot_dim=rot, max_seq=1088)
    weights = O.synth_text_weights(cfg, 9)
    ref = O.TextModel(weights, cfg)
    mcfg = moon.text_model.make_config(vocab=cfg["vocab"], dim=dim, hidden_dim=hidden, n_layers=2, n_heads=heads, rot_dim=rot, max_seq=cfg["max_seq"])
    dev = moon.text_model.TextModel(mcfg, weights=weights, ctx=ctx)
    cache = ref.new_cache()
    for i, rows in enumerate(pieces):
        ids = O.fill_uniform_u32(rows, i, 57, cfg["vocab"])
        h_ref = ref.text_decoder(ref.text_encoder(ids), cache)
        dev.forward(ids)
        assert O.rel_frobenius(dev.hidden(rows), h_ref) <= TOL, (i, rows)
        assert O.rel_frobenius(dev.logits().reshape(1, -1), ref.lm_head(h_ref).reshape(1, -1)) <= TOL, (i, rows)
    dev.close()


# The same prompts with the projection, its rotation and fc1 in one launch and in three: of widths below 1024 neither product alone is taken in ranges
# of k, so the bits are the same, in thin tiles (width 512) and wide ones of both heights (960; the first piece is thin there too), behind other pieces, and where
# the rotation is a launch of its own either way (64 turning).  Which form a piece takes is asked of the choice itself (tests/cxx/gemm_choice_check.cpp); that out_proj and fc2 shared
# a launch, and its tiles, of the last launch.
@pytest.mark.parametrize("dim,hidden,heads,rot,pieces", [(512, 2048, 8, 32, (37, 129, 191, 385)), (512, 2048, 8, 64, (37, 129, 191, 385)), (960, 3840, 15, 32, (129, 897)),
                                                         (960, 3840, 15, 32, (130, 1729))])
def test_one_launch_gives_the_bits_of_three(moon, O, ctx, monkeypatch, dim, hidden, heads, rot, pieces):
    cfg = moon.text_model.make_config(vocab=1024, dim=dim, hidden_dim=hidden, n_layers=2, n_heads=heads, rot_dim=rot, max_seq=2048)
    dev = moon.text_model.TextModel(cfg, seed=6, std=0.03, ctx=ctx)
    out = []
    for apart in (False, True):
        if apart:
            monkeypatch.setenv("MOON_GEMM_NO_ROPE", "1")
        dev.reset()
        got = []
        for i, rows in enumerate(pieces):
            dev.forward(O.fill_uniform_u32(rows, i, 58, 1024))
            assert ctx.last_kernel().startswith("gemm_nt_thin_pair_kernel" if rows < 192 else "gemm_nt_dma192_pair_kernel"), rows
            got += [dev.hidden(rows).copy(), dev.logits().copy()]
        got.append(np.asarray(dev.greedy(5)).astype(np.uint32).view(np.uint16))
        out.append(got)
    monkeypatch.delenv("MOON_GEMM_NO_ROPE")
    dev.close()
    for x, y in zip(*out):
        assert np.array_equal(x.view(np.uint16), y.view(np.uint16))


# 256 x 256 tiles enough for every compute unit: whole k-tiles take the wide tiles, a K without them (80) the kernel with 128 x 128 accumulators
# a wavefront; the [K, N] operand and its [N, K] copy give the same bits.
@pytest.mark.parametrize("M,N,K,kernel", [(4097, 4088, 64, "gemm_nt_block_kernel"), (3841, 4104, 192, "gemm_nt_block_kernel"), (4000, 4096, 80, "gemm_nt_wide_kernel")])
def test_products_of_many_wide_tiles(moon, O, ctx, M, N, K, kernel):
    a = O.fill_normal_f16((M, K), 0, 0, 1.0)
    w = O.fill_normal_f16((N, K), 0, 1, 0.05)
    got = moon.hgemm_trans.matmul(a, w, ctx=ctx)
    assert kernel in ctx.last_kernel()
    assert np.array_equal(moon.hgemm.matmul(a, np.ascontiguousarray(w.T), ctx=ctx), got)
    assert kernel in ctx.last_kernel()
    ref = O.hgemm_trans(a, w)
    assert O.rel_frobenius(got, ref) <= TOL
    assert np.abs(got.astype(np.float32) - ref.astype(np.float32)).max() <= 2 * 2.0**-10 * np.abs(ref.astype(np.float32)).max()
