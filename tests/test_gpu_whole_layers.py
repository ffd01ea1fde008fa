"""One token through a whole layer of a list decoder in one launch (layer_whole.hip): sizes at the edges of what it takes."""
import generax_models as GM
import generax_oracle as G
import numpy as np
import pytest
import rikanex_models as RM
import rikanex_oracle as R
from conftest import compute_units
from decoder_checks import feed, opened, rows_close, run

pytestmark = pytest.mark.gpu
# of the lists' other tests: an f32 sum's result rounded to bf16 (2^-9 at most, 2^-10.8 on average) some dozens of times on the way to a logit
LIMIT = 3e-2
ROT = GM.rotation(64, 1e4)


def took_one_launch(ctx, splits=None):
    if compute_units() == 256:
        note = ctx.last_kernel()
        assert note.startswith("decode_whole_kernel") and (splits is None or f" {splits} splits" in note), note


def assert_close(got, want):
    ok, text = rows_close(got, want, LIMIT)
    assert ok, text


# (heads of 63 and 61 are padded to 64.)  One, two, four and eight heads a workgroup, and two workgroups for a key head; widths that end inside a piece of 64 elements,
# below and above 1024; rows that do not fill the last output workgroup; odd feed-forwards, the largest, none
RIKANEX = {
    "smallest": (64, 1, 1, 8, 5), "odd": (516, 6, 6, 70, 40), "pairs": (1020, 14, 7, 333, 17), "fours": (1024, 16, 4, 1728, 33), "eights": (1084, 10, 2, 1121, 64),
    "two workgroups": (256, 12, 1, 129, 20), "no feed-forward": (320, 4, 2, None, 9),
}


@pytest.mark.parametrize("name", sorted(RIKANEX))
def test_rikanex(moon, ctx, tmp_path, name):
    width, heads, kv_heads, ff, window = RIKANEX[name]
    mlp = RM.dense(ff) if ff else None
    cfg = RM.config(90, width, [RM.layer(RM.attention(heads, kv_heads, 63, 61, window, 0.13, mix), mlp) for mix in (False, True, True)], embed_scale=2.0)
    w, ids = RM.weights(cfg, 3), RM.tokens(75, 90)
    m = opened(moon, ctx, RM.write_folder(tmp_path / "m", cfg, w), "bfloat16")
    got = []
    for at in range(len(ids)):
        m.forward(ids[at:at + 1])
        took_one_launch(ctx, min(2, -(-min(at + 1, window) // 32)))
        got.append(m.logits_f32())
    m.close()
    want = R.forward(cfg, w, ids)[0]
    assert_close(np.array(got), want)
    assert_close(run(moon, ctx, tmp_path, cfg, w, ids, "bfloat16", [40, 1, 1, 3, 1]), want)


@pytest.mark.parametrize("width,heads,kv_heads,ff,delta_heads", [(64, 1, 1, 8, 1), (516, 6, 3, 70, 5), (1024, 16, 4, 1728, 16), (1084, 10, 2, 321, 4), (320, 4, 1, None, 2)])
def test_generax(moon, ctx, tmp_path, width, heads, kv_heads, ff, delta_heads):
    """Joined layers behind each other, in front of a plain one and as the last; borrowed keys; blocks before the window."""
    joined = GM.parallel(GM.softmax_mixer(heads, kv_heads, 64, 64, 9, 0.13, 4), GM.delta(delta_heads, 1, 64, 64, 4), ff)
    turned = GM.attention(heads, kv_heads, 64, 64, 20, 0.13, ROT)
    cfg = GM.config(90, width, [joined, joined, GM.plain(turned, ff), GM.plain(dict(turned, kv_from=2), ff), joined])
    w, ids = GM.weights(cfg, 3), RM.tokens(75, 90)
    got = run(moon, ctx, tmp_path, cfg, w, ids, "bfloat16", [1])
    want = G.forward(cfg, w, ids)[0]
    assert_close(got, want)
    assert_close(run(moon, ctx, tmp_path, cfg, w, ids, "bfloat16", [40, 1, 1, 3, 1]), want)


LARGE = [RM.config(128, 2048, [RM.layer(RM.attention(32, kv, 64, 64, window, 0.125, True), RM.dense(ff) if ff else None) for _ in range(3)], embed_scale=2.0)
         for kv, window, ff in ((32, 1024, 6144), (8, 1024, 5504), (8, 512, 6208), (1, 512, 10240), (4, 512, 1024), (8, 64, None))]
LARGE += [GM.config(128, width, [GM.parallel(GM.softmax_mixer(width // 64, kv, 64, 64, 512, 0.125, 16), GM.delta(width // 64, width // 64, 64, 64, 4), ff),
                                 GM.plain(GM.attention(width // 64, kv, 64, 64, 1024, 0.125, ROT), ff)] * 2) for width, kv, ff in ((2048, 8, 5632), (2048, 8, 6464), (1024, 16, 9856), (2048, 32, 3712), (1024, 4, 1728))]


@pytest.mark.parametrize("which", range(len(LARGE)))
def test_largest_sizes_beside_f32(moon, ctx, which):
    """Against an f32 session, which takes other kernels, behind few and many cached keys: the splits' numbers from one to the largest."""
    out = []
    ids = RM.tokens(1100, 128)
    for dtype in ("bfloat16", "float32"):
        m = moon.text_model.TextModel.open_synthetic(LARGE[which], dtype, 2048, seed=5, std=0.02, ctx=ctx)
        rows = []
        for prompt in (1, 31, 300, 1090):
            m.reset()
            rows.append(feed(m, ids[:prompt], [prompt])[-1:])
            for i in range(3):
                m.forward(ids[prompt + i:prompt + i + 1])
                if dtype == "bfloat16":
                    took_one_launch(ctx)
                rows.append(m.logits_f32()[None])
        out.append(np.concatenate(rows))
        m.close()
    assert_close(*out)


def config_of(name):
    """Configurations of the tests above and layers without a window, at every number of loads that a row takes: -> (configuration, made from weights of its own?)"""
    if name in RIKANEX:
        width, heads, kv_heads, ff, window = RIKANEX[name]
        return RM.config(90, width, [RM.layer(RM.attention(heads, kv_heads, 63, 61, window, 0.13, mix), RM.dense(ff) if ff else None) for mix in (False, True, True)], embed_scale=2.0), True
    if name.startswith("large"):
        return LARGE[int(name[5:])], False
    kind, width, heads, ff = name.split()
    width, heads, ff = int(width), int(heads), int(ff) or None
    whole = dict(window=10**6, scale=0.125)
    if kind == "plain":
        return RM.config(128, width, [RM.layer(RM.attention(heads, heads, 64, 64, v_mix=mix, **whole), RM.dense(ff) if ff else None) for mix in (False, True)], embed_scale=2.0), False
    if kind == "joined":
        return GM.config(128, width, [GM.parallel(GM.softmax_mixer(heads, heads, 64, 64, **whole), GM.delta(heads // 2, heads // 2, 64, 64, 4), ff)] * 2), False
    if kind == "odd":
        joined = GM.parallel(GM.softmax_mixer(heads, heads, 64, 64, 9, 0.13, 4), GM.delta(heads + 1, 1, 64, 64, 4), ff)
        return GM.config(128, width, [joined, GM.plain(GM.attention(heads, 1, 60, 62, 20, 0.13, GM.rotation(32, 1e4)), ff), joined]), True
    return GM.config(128, width, [GM.plain(GM.attention(heads, heads, 64, 64, rot=ROT, **whole), ff)] * 2), False


SAME = [*sorted(RIKANEX), *(f"large{i}" for i in range(len(LARGE))), "plain 2048 32 5504", "plain 2048 32 10240", "plain 2048 32 0", "plain 1024 16 2816", "plain 512 8 192", "joined 2048 32 6464",
        "turned 2048 32 320", "joined 1024 16 1728", "turned 1024 16 7168", "joined 512 8 64", "odd 516 5 70", "odd 1084 9 321", "odd 320 2 0", "odd 1020 15 2050"]


@pytest.mark.parametrize("name", SAME)
def test_one_launch_and_three_give_the_same_bits(moon, ctx, tmp_path, name):
    cfg, own = config_of(name)
    if own:
        weights = (RM if cfg["architecture"] == "Rikanex" else GM).weights(cfg, 3)
        m = opened(moon, ctx, RM.write_folder(tmp_path / "m", cfg, weights), "bfloat16")
    else:
        m = moon.text_model.TextModel.open_synthetic(cfg, "bfloat16", 512, seed=5, std=0.02, ctx=ctx)
    rows, tokens, ids = {}, {}, RM.tokens(400, 90)
    for mode in (0, 2):
        m.set_decode_mode(mode)
        rows[mode] = []
        for prompt in (2, 31, 150, 390):
            m.reset()
            m.forward(ids[:prompt])
            for i in range(3):
                m.forward(ids[prompt + i:prompt + i + 1])
                if mode == 0:
                    took_one_launch(ctx)
                else:
                    assert not ctx.last_kernel().startswith("decode_whole") # (the prompt's products have left their own note)
                rows[mode].append(m.logits_f32())
        tokens[mode] = m.greedy(20).tolist()
        rows[mode].append(m.logits_f32())
    m.close()
    assert np.isfinite(rows[0]).all() and np.array_equal(*(np.array(rows[mode]).view(np.uint32) for mode in (0, 2)))
    assert tokens[0] == tokens[2]


def test_few_producers_take_three_launches(moon, ctx):
    """Without a window the splits' workgroups take the producers' places: behind 20,000 keys of 32 heads 128 are left, behind 22,000 64, whose wavefronts would have 56 pairs of rows each."""
    cfg = RM.config(128, 2048, [RM.layer(RM.attention(32, 32, 64, 64, 10**6, 0.125), RM.dense(10240))], embed_scale=2.0)
    m = moon.text_model.TextModel.open_synthetic(cfg, "bfloat16", 23000, seed=5, std=0.02, ctx=ctx)
    ids = RM.tokens(22100, 128)
    at = 0
    for keys, whole in ((20000, True), (22000, False)):
        m.forward(ids[at:keys])
        rows = []
        for i, mode in enumerate((0, 2)):
            m.set_decode_mode(mode)
            m.forward(ids[keys + 4 * i:keys + 4 * i + 3]) # (its own note)
            m.forward(ids[keys + 4 * i + 3:keys + 4 * i + 4])
            if compute_units() == 256:
                assert ctx.last_kernel().startswith("decode_whole") == (whole and mode == 0)
            rows.append(m.logits_f32())
        at = keys + 8
        assert np.isfinite(rows).all()
    m.close()


def test_modes_of_list_decoders(moon, ctx):
    """0 and 2 where a layer runs in one launch; none where no launch waits."""
    dense, experts = (RM.config(128, 512, [RM.layer(RM.attention(8, 8, 64, 64, 40, 0.125), mlp)]) for mlp in (RM.dense(128), RM.moe(64, 8, 64)))
    for cfg, dtype, modes in ((dense, "bfloat16", (0, 2)), (dense, "float32", ()), (experts, "bfloat16", ())):
        m = moon.text_model.TextModel.open_synthetic(cfg, dtype, 64, seed=5, std=0.02, ctx=ctx)
        for mode in range(-1, 5):
            if mode in modes:
                m.set_decode_mode(mode)
            else:
                with pytest.raises(moon.MoonError):
                    m.set_decode_mode(mode)
        m.close()


@pytest.mark.parametrize("name", ["plain 1024 16 2816", "joined 2048 32 6464"])
def test_failed_wait_and_recovery(moon, ctx, name):
    """The error word of the waits raised from the host (every kernel still runs to its end): the call fails, the position stays, work is refused until reset, and behind it
    the session has the bits of a fresh one."""
    cfg, _ = config_of(name)
    ids = RM.tokens(60, 128)

    def session():
        return moon.text_model.TextModel.open_synthetic(cfg, "bfloat16", 256, seed=5, std=0.02, ctx=ctx)

    def work(m):
        m.forward(ids[:40])
        m.forward(ids[40:41])
        row = m.logits_f32()
        return m.greedy(6).tolist(), row.view(np.uint32).tolist(), m.logits_f32().view(np.uint32).tolist()

    m = session()
    want = work(m)
    m.close()
    m = session()
    for call in (lambda: m.forward(ids[40:41]), lambda: m.greedy(3), lambda: m.generate(9, 1), lambda: m.forward_logits(ids[40:41], [0])):
        m.forward(ids[:40])
        ctx.check(ctx.lib.moon_text_debug_raise_wait_error(m.handle))
        with pytest.raises(moon.context.HipError):
            call()
        assert m.position == 40
        for refused in (lambda: m.forward(ids[:1]), lambda: m.forward(ids[:5]), lambda: m.greedy(1)):
            with pytest.raises(moon.context.HipError):
                refused()
        m.reset()
        assert m.position == 0 and work(m) == want
        m.reset()
    m.close()
    m = moon.text_model.TextModel.open_synthetic(cfg, "float32", 64, seed=5, std=0.02, ctx=ctx)
    with pytest.raises(moon.MoonError):
        ctx.check(ctx.lib.moon_text_debug_raise_wait_error(m.handle))
    m.close()


@pytest.mark.parametrize("change", [dict(width=2112), dict(ff=10304), dict(dim=128), dict(experts=True)])
def test_other_sizes_take_three_launches(moon, ctx, change):
    width, dim = change.get("width", 1024), change.get("dim", 64)
    mlp = RM.moe(64, 64, 64) if "experts" in change else RM.dense(change.get("ff", 128))
    cfg = RM.config(128, width, [RM.layer(RM.attention(4, 2, dim, dim, 40, 0.125, True), mlp)], embed_scale=2.0)
    out = []
    ids = RM.tokens(40, 128)
    for dtype in ("bfloat16", "float32"):
        m = moon.text_model.TextModel.open_synthetic(cfg, dtype, 256, seed=5, std=0.02, ctx=ctx)
        m.forward(ids[:30])
        m.forward(ids[30:31])
        assert not ctx.last_kernel().startswith("decode_whole")
        out.append(np.concatenate([m.logits_f32()[None], feed(m, ids[31:], [1])]))
        m.close()
    assert_close(*out)


def test_sessions_of_two_contexts_at_once(moon, ctx):
    """Two threads decode: whichever call finds no places for its waiting workgroups takes three launches, with the same tokens up to rounding."""
    import threading
    cfg = LARGE[1]
    ids = RM.tokens(64, 128)
    sessions = [moon.text_model.TextModel.open_synthetic(cfg, "bfloat16", 256, seed=5, std=0.02, ctx=c) for c in (ctx, moon.Context(), moon.Context())]
    alone = feed(sessions[0], ids, [40] + [1] * 24)
    sessions[0].reset()
    out = [None] * len(sessions)

    def work(i):
        out[i] = feed(sessions[i], ids, [40] + [1] * 24)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sessions))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for m, got in zip(sessions, out):
        assert got is not None
        assert_close(got, alone)
        m.close()


def test_sessions_of_three_contexts_at_once(moon, ctx):
    """Three threads decode with waiting workgroups that all find places (40 of 128 a die each): the bits of a session alone."""
    import threading
    cfg = LARGE[1]
    ids = RM.tokens(64, 128)
    sessions = [moon.text_model.TextModel.open_synthetic(cfg, "bfloat16", 256, seed=5, std=0.02, ctx=c) for c in (ctx, moon.Context(), moon.Context())]
    alone = feed(sessions[0], ids, [40] + [1] * 24)
    sessions[0].reset()
    out = [None] * len(sessions)

    def work(i):
        out[i] = feed(sessions[i], ids, [40] + [1] * 24)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sessions))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for m, got in zip(sessions, out):
        assert got is not None
        assert np.array_equal(got.view(np.uint32), alone.view(np.uint32))
        m.close()


def test_a_call_without_places_takes_three_launches(moon, ctx):
    """While another context's call holds the places of 736 waiting workgroups (92 of 128 a die: 32 heads with room for 15,000 keys), a call with 320 of its own finds none: it takes
    three launches, with the same bits, and one launch again when the other call is over."""
    import threading
    import time
    if compute_units() != 256:
        pytest.skip("counted for 256 units")
    other = moon.Context()
    large = moon.text_model.TextModel.open_synthetic(RM.config(128, 2048, [RM.layer(RM.attention(32, 32, 64, 64, 10**6, 0.125), RM.dense(64))]), "bfloat16", 15000, seed=5, std=0.02, ctx=other)
    m = moon.text_model.TextModel.open_synthetic(LARGE[1], "bfloat16", 256, seed=5, std=0.02, ctx=ctx)
    ids = RM.tokens(64, 128)

    def token():
        m.reset()
        m.forward(ids[:40]) # (its products leave their own note)
        m.forward(ids[40:41])
        return ctx.last_kernel().startswith("decode_whole_kernel"), m.logits_f32().view(np.uint32)

    one, alone = token()
    assert one
    large.forward(ids[:8])
    done = []
    thread = threading.Thread(target=lambda: done.append(large.greedy(4000)))
    thread.start()
    time.sleep(0.02) # (it takes its places before this context's calls do; it runs some 300 ms)
    seen = []
    while thread.is_alive():
        one, bits = token()
        seen.append(one)
        assert np.array_equal(bits, alone)
    thread.join()
    assert len(done) == 1 and seen.count(False) > 10, (len(done), seen)
    one, bits = token()
    assert one and np.array_equal(bits, alone)
    large.close()
    m.close()
