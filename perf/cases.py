"""What a user of this framework has it do, as cases that can be timed and checked.

A case is a dict of plain values; `kind` says which entry points it calls:

  product    one matrix product on device buffers (moon_dev_linear), the operator that a host binds
  attention  one attention on device buffers (moon_dev_sdpa)
  image      VisionModel.encode_image_u8: a resized picture in host memory to its features in host memory
  encoder    VisionModel.encode: rows in host memory through the encoder blocks
  decoder    the f16 text decoder: a prompt, its logits, then tokens fed one by one by a host that keeps its own loop, and the logits
             behind the last of them
  reply      the f16 text decoder: a prompt, then the device's own sampled generation loop
  list       a decoder described as a list of layers (Rikanex, Generax): as `decoder`

Sizes are those of the shipped configurations, the tests and bench.py, or generic.  Sessions hold random weights made from the seed.
exact() computes the same in float64 with plain torch; it makes the sessions' random weights from their published definition.
"""
import importlib
import math

import numpy as np
import torch

VOCAB = 51200
PATCHES, PATCH_DIM, VISION_WIDTH, VISION_HIDDEN, VISION_LAYERS, VISION_HEADS = 729, 588, 1152, 4304, 27, 16
EPS_F16 = 1.00135803e-5  # 1e-5 as f16
GELU_C, GELU_A = 0.7978515625, 0.044708251953125  # the constants of the tanh form, as f16
STD = 0.02


def moon():
    return importlib.import_module("moondream-zig_amd")


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: one token's row through one weight matrix, launch and latency beside 34 MB of weights
        dict(name="product_row", kind="product", m=1, k=2048, n=8192, layout="nk", epilogue=2),
        # the picture encoder's hidden layer as the reference states it, with the operand in its [K, N] layout and ragged rows
        dict(name="product_patches", kind="product", m=729, k=1152, n=4304, layout="kn", epilogue=2),
        # attention over one crop's patches
        dict(name="attention_patches", kind="attention", heads=16, queries=729, past=0, head=72, causal=False),
        # a picture is shown: both crops through patch embedding, 27 blocks and projection
        dict(name="image", kind="image"),
        # picture features and question together make a prompt of about this length
        dict(name="decoder_prompt", kind="decoder", width=2048, layers=24, prompt=768, steps=0),
        # a short question, answered token by token by a host that keeps its loop
        dict(name="decoder_steps", kind="decoder", width=2048, layers=24, prompt=37, steps=24),
        # the smaller decoder generates on the device with the command line's default sampler
        dict(name="reply_small", kind="reply", width=1024, layers=24, prompt=53, steps=48),
        # a long document before the window has passed over it, grouped keys and values
        dict(name="rikanex_prompt", kind="list", design="Rikanex", width=2048, layers=24, kv_heads=8, window=1024, ff=5504, experts=0, prompt=1920, steps=0),
        # the same decoder token by token
        dict(name="rikanex_steps", kind="list", design="Rikanex", width=2048, layers=24, kv_heads=8, window=1024, ff=5504, experts=0, prompt=61, steps=24),
        # routed experts, prompt and tokens
        dict(name="rikanex_experts", kind="list", design="Rikanex", width=2048, layers=12, kv_heads=8, window=1024, ff=704, experts=64, prompt=768, steps=8),
        # joined mixers, rotated and borrowed layers; long enough that blocks before the window count; an odd length
        dict(name="generax_prompt", kind="list", design="Generax", width=2048, layers=24, kv_heads=8, window=1024, ff=3712, experts=0, prompt=1301, steps=0),
        # the smaller one token by token
        dict(name="generax_steps", kind="list", design="Generax", width=1024, layers=24, kv_heads=4, window=512, ff=1728, experts=0, prompt=45, steps=24),
    ]


def draw(rng):
    def spread(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["product", "product", "attention", "image rows", "decoder", "reply", "list", "list", "list"])
    if kind == "product":
        if rng.random() < 0.3:
            return dict(kind="product", m=1, k=8 * spread(32, 1024), n=spread(256, 8192), layout="nk", epilogue=rng.randrange(3))
        return dict(kind="product", m=spread(2, 1536), k=8 * spread(32, 1024), n=spread(256, 8192), layout=rng.choice(["nk", "kn"]), epilogue=rng.randrange(3))
    if kind == "attention":
        causal = rng.random() < 0.5
        return dict(kind="attention", heads=rng.choice([8, 16, 32]), queries=spread(16, 1458), past=rng.choice([0, spread(1, 500)]) if causal else 0,
                    head=64 if causal else 72, causal=causal)
    if kind == "image rows":
        return dict(kind="encoder", layers=rng.randrange(3, 28, 3), rows=spread(64, 1458))
    width, layers, prompt = rng.choice([1024, 2048]), rng.randrange(4, 25, 4), spread(2, 1536)
    steps = rng.choice([0, 0, rng.randrange(1, 17)])
    if kind == "decoder":
        return dict(kind="decoder", width=width, layers=layers, prompt=prompt, steps=steps)
    if kind == "reply":
        return dict(kind="reply", width=1024, layers=layers, prompt=prompt, steps=rng.randrange(4, 33))
    case = dict(kind="list", design=rng.choice(["Rikanex", "Rikanex", "Generax"]), width=width, layers=layers, kv_heads=rng.choice([4, 8, width // 64]),
                window=rng.choice([512, 1024, 1000]), ff=64 * rng.randrange(16, 88), experts=0, prompt=prompt, steps=steps)
    if case["design"] == "Rikanex" and rng.random() < 0.25:
        case.update(experts=64, ff=64 * rng.randrange(4, 12), layers=min(layers, 12), steps=min(steps, 8))
    return case


def late_ff(c):
    """Feed-forward size of the layers without a delta rule, which have weights to spare."""
    return c["ff"] * 7 // 256 * 64


def embedding_scale(c):
    """Routed experts: large beside the layers' results, for where a token's eighth and ninth expert are a rounding apart either may be taken."""
    return 512.0 if c["experts"] else 45.0


def list_config(c):
    """config.json of a case."""
    heads, layers = c["width"] // 64, []
    part = dict(heads=heads, kv_heads=c["kv_heads"], dim=64, vdim=64, scale=0.125)
    for i in range(c["layers"]):
        if c["design"] == "Rikanex":
            mlp = dict(kind="dense", ff=c["ff"]) if not c["experts"] else dict(kind="moe", router=dict(experts=c["experts"], top=8), expert=dict(ff=c["ff"]))
            layers.append(dict(type="attention", mixer=dict(part, mask=dict(size=c["window"]), v_mix=True), mlp=mlp))
            continue
        joined = dict(left=dict(part, mask=dict(size=c["window"], pool=16)), right=dict(heads=heads, kv_heads=heads, dim=64, vdim=64, conv=4))
        turned = dict(part, mask=dict(size=c["window"]), rot=dict(dims=64, base=10000.0))
        kind = i % 4
        layers.append(dict(type="parallel" if kind < 2 else "attention", mixer=joined if kind < 2 else turned if kind == 2 else dict(turned, kv_from=i - 1),
                           mlp=dict(kind="dense", ff=c["ff"] if kind < 2 else late_ff(c))))
    if c["design"] == "Rikanex":
        return dict(architecture="Rikanex", vocab=VOCAB, width=c["width"], embedding=dict(scale=embedding_scale(c)), norm=dict(eps=1e-5), layers=layers)
    return dict(architecture="Generax", vocab=VOCAB, width=c["width"], norm=dict(eps=1e-5), logit_softcap=30.0, layers=layers)


# ---------------------------------------------------------------- preparing and running
def generator(seed, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    return g


def normal(g, shape, std, dtype=torch.float16):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(dtype)


def product_inputs(c, seed):
    g = generator(seed)
    a = normal(g, (c["m"], c["k"]), 1.0)
    b = normal(g, (c["n"], c["k"]) if c["layout"] == "nk" else (c["k"], c["n"]), STD)
    return a, b, normal(g, (c["n"],), STD)


def attention_inputs(c, seed):
    g, h, d, past = generator(seed), c["heads"], c["head"], c["past"]
    return normal(g, (h, c["queries"], d), 1.0), normal(g, (h, past + c["queries"], d), 1.0), normal(g, (h, past + c["queries"], d), 1.0)


def picture(seed):
    return np.random.default_rng(seed).integers(0, 256, size=(378, 378, 3), dtype=np.uint8)


def encoder_rows(c, seed):
    return np.random.default_rng(seed).standard_normal((c["rows"], VISION_WIDTH), dtype=np.float32).astype(np.float16)


def token_ids(c, seed):
    return np.random.default_rng(seed).integers(0, VOCAB, size=c["prompt"] + c["steps"]).astype(np.uint32)


def reply_weights(c, seed):
    """A decoder that is as sure of its next token as a trained one: the LM head's row of a token's successor is the token's embedding,
    which the residual stream still holds at the end."""
    g, d, L = generator(seed), c["width"], c["layers"]
    successor = torch.randperm(VOCAB, generator=g, device="cuda")
    ones, zeros = (lambda *s: torch.ones(s, device="cuda", dtype=torch.float16)), (lambda *s: torch.zeros(s, device="cuda", dtype=torch.float16))
    w = dict(wte=normal(g, (VOCAB, d), 1.0), ln_w=ones(L, d), ln_b=zeros(L, d), Wqkv_w=normal(g, (L, 3 * d, d), STD), Wqkv_b=normal(g, (L, 3 * d), STD),
             out_proj_w=normal(g, (L, d, d), STD), out_proj_b=normal(g, (L, d), STD), fc1_w=normal(g, (L, 4 * d, d), STD), fc1_b=normal(g, (L, 4 * d), STD),
             fc2_w=normal(g, (L, d, 4 * d), STD), fc2_b=normal(g, (L, d), STD), linear_b=zeros(VOCAB), ln_out_w=ones(d), ln_out_b=zeros(d))
    w["linear_w"] = torch.empty_like(w["wte"])
    w["linear_w"][successor] = (w["wte"].float() * 0.05).half()
    return w, successor


def prepare(case, seed):
    m, kind = moon(), case["kind"]
    ctx = m.default_context()
    s = dict(case=case, ctx=ctx)
    if kind == "product":
        s["a"], s["b"], s["bias"] = product_inputs(case, seed)
        s["c"] = torch.empty((case["m"], case["n"]), device="cuda", dtype=torch.float16)
    elif kind == "attention":
        s["q"], s["k"], s["v"] = attention_inputs(case, seed)
        s["out"] = torch.empty_like(s["q"])
    elif kind == "image":
        v = m.vision_model
        s["model"] = v.VisionModel(v.default_config(), seed=seed, std=STD, ctx=ctx)
        s["model"].attach_io(seed=seed, std=STD)
        s["image"] = picture(seed)
    elif kind == "encoder":
        v = m.vision_model
        s["model"] = v.VisionModel(v.make_config(n_layers=case["layers"]), seed=seed, std=STD, ctx=ctx)
        s["x"] = encoder_rows(case, seed)
    elif kind in ("decoder", "reply"):
        t, d = m.text_model, case["width"]
        cfg = t.make_config(vocab=VOCAB, dim=d, hidden_dim=4 * d, n_layers=case["layers"], n_heads=d // 64)
        if kind == "decoder":
            s["model"], s["ids"] = t.TextModel(cfg, seed=seed, std=STD, ctx=ctx), token_ids(case, seed)
        else:
            weights = {k: w.cpu().numpy() for k, w in reply_weights(case, seed)[0].items()}
            s["model"], s["ids"] = t.TextModel(cfg, weights=weights, ctx=ctx), token_ids(case, seed)[:case["prompt"]]
            s["sampler"] = m.sampling.sampling_config("top_k")
            s["u"] = np.random.default_rng(seed).random(case["steps"], dtype=np.float32)
    else:
        s["model"] = m.text_model.TextModel.open_synthetic(list_config(case), "bfloat16", 2048, seed=seed, std=STD, ctx=ctx)
        s["ids"] = token_ids(case, seed)
    return s


def run(s):
    c, ctx = s["case"], s["ctx"]
    if c["kind"] == "product":
        ctx.check(ctx.lib.moon_dev_linear(ctx.handle, s["a"].data_ptr(), c["m"], c["k"], s["b"].data_ptr(), c["n"], 1 if c["layout"] == "nk" else 0,
                                          s["bias"].data_ptr() if c["epilogue"] else None, c["epilogue"], s["c"].data_ptr()))
        return s["c"]
    if c["kind"] == "attention":
        ctx.check(ctx.lib.moon_dev_sdpa(ctx.handle, s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["out"].data_ptr(), c["heads"], c["queries"],
                                        c["past"] + c["queries"], c["head"], c["past"] if c["causal"] else -1, None, 0))
        return s["out"]
    model = s["model"]
    if c["kind"] == "image":
        return model.encode_image_u8(s["image"])
    if c["kind"] == "encoder":
        return model.encode(s["x"])
    ids, n = s["ids"], c["prompt"]
    model.reset()
    if c["kind"] == "reply":
        model.forward(ids)
        tokens = model.sample(s["sampler"], s["u"])
        return dict(tokens=tokens.astype(np.int64), logits=model.logits())
    if c["kind"] == "decoder":
        model.forward(ids[:n])
        out = [model.logits()]
    else:
        out = [model.forward_logits(ids[:n], [n - 1])[0]]
    for i in range(c["steps"]):
        model.forward(ids[n + i:n + i + 1])
    if c["steps"]:
        out.append(model.logits() if c["kind"] == "decoder" else model.logits_f32())
    return out


# ---------------------------------------------------------------- what a pass cannot do without
def attended(n, past, window, causal=True):
    """Pairs of queries and keys."""
    if not causal:
        return n * (past + n)
    return sum(min(past + i + 1, window or past + n) for i in range(n))


def work(case):
    c, kind = case, case["kind"]
    if kind == "product":
        return dict(bytes=2 * (c["m"] * c["k"] + c["k"] * c["n"] + c["m"] * c["n"] + c["n"]), flops=2 * c["m"] * c["k"] * c["n"])
    if kind == "attention":
        kv = c["past"] + c["queries"]
        return dict(bytes=4 * c["heads"] * c["head"] * (c["queries"] + kv), flops=4 * c["heads"] * c["head"] * attended(c["queries"], c["past"], 0, c["causal"]))
    if kind in ("image", "encoder"):
        rows, layers, d, f = (2 * PATCHES, VISION_LAYERS, VISION_WIDTH, VISION_HIDDEN) if kind == "image" else (c["rows"], c["layers"], VISION_WIDTH, VISION_HIDDEN)
        weights = layers * (4 * d * d + 2 * d * f)
        flops = 2 * rows * weights + layers * 4 * rows * rows * d
        nbytes = 2 * weights + 4 * rows * d
        if kind == "image":
            ends = 2 * d * 8192 + 8192 * 2048
            flops += 2 * rows * PATCH_DIM * d + 2 * PATCHES * ends
            nbytes = 2 * (weights + PATCH_DIM * d + ends) + 378 * 378 * 3 + PATCHES * 2048 * 2
        return dict(bytes=nbytes, flops=flops)
    d, L, n, steps = c["width"], c["layers"], c["prompt"], c["steps"]
    if kind in ("decoder", "reply"):
        layer, kv_row, window = 12 * d * d, 2 * d, 0
        dense, routed = L * layer, 0
    else:
        window, kv_row = c["window"], 2 * 64 * c["kv_heads"]
        dense, routed = 0, 0
        for i in range(L):
            if c["design"] == "Rikanex":
                dense += 3 * d * d + d * kv_row
                if c["experts"]:
                    dense += c["experts"] * d
                    routed += 3 * d * c["ff"]
                else:
                    dense += 3 * d * c["ff"]
            else:
                ff = c["ff"] if i % 4 < 2 else late_ff(c)
                dense += 2 * d * d + (0 if i % 4 == 3 else d * kv_row) + 3 * d * ff
                if i % 4 < 2:
                    dense += 4 * d * d + (d // 64 + 128) * d + 2 * d * 64
    top = 8 if routed else 0
    head = VOCAB * d
    heads_out = 1 + (steps if kind == "reply" else 1 if steps else 0)
    nbytes = 2 * (dense + routed * min(c.get("experts", 0), top * n) + head * heads_out + steps * (dense + top * routed))
    nbytes += 2 * kv_row * L * (n + sum(min(n + i + 1, window or 1 << 30) for i in range(steps)))
    flops = 2 * (n + steps) * (dense + top * routed) + 2 * head * heads_out + 4 * d * L * attended(n + steps, 0, window)
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    # about four times the distance from exact(): 4e-4 for a product, 3e-4 for attention (one f16 rounding of an f32 sum is 2.8e-4), 1.9e-3 and 1.5e-3
    # where hundreds of such roundings add up in an encoder or the f16 decoder, 1e-2 in bf16
    return dict(rel={"product": 1.6e-3, "attention": 1.2e-3, "image": 8e-3, "encoder": 8e-3, "decoder": 6e-3, "reply": 6e-3, "list": 0.03}[case["kind"]])


# ---------------------------------------------------------------- the same in float64
MASK64 = (1 << 64) - 1


def _mix(z):
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & MASK64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & MASK64
    return z ^ (z >> 31)


def _signed(z):
    return z - (1 << 64) if z >> 63 else z


def _mix_t(z):
    for shift, factor in ((30, 0xBF58476D1CE4E5B9), (27, 0x94D049BB133111EB)):
        z = (z ^ ((z >> shift) & ((1 << (64 - shift)) - 1))) * _signed(factor)
    return z ^ ((z >> 31) & ((1 << 33) - 1))


def synthetic(shape, seed, stream, std, dtype=torch.float16):
    """The sessions' random weights: element i is the centred sum of the eight 16-bit fields of two splitmix64 words, scaled in f32."""
    golden = 0x9E3779B97F4A7C15
    key = _mix(_mix((seed + golden) & MASK64) ^ ((stream * 0xD1B54A32D192ED03 + 0x2545F4914F6CDD1D) & MASK64))
    scale = float(np.float32(std) * np.float32(1.0 / np.float32(53510.105)))
    n, parts = math.prod(shape), []
    for lo in range(0, n, 1 << 24):
        i = torch.arange(lo, min(n, lo + (1 << 24)), device="cuda", dtype=torch.int64)
        total = None
        for half in range(2):
            word = _mix_t((2 * i + half + 1) * _signed(golden) + _signed(key))
            for f in range(4):
                field = (word >> (16 * f)) & 0xFFFF
                total = field if total is None else total + field
        parts.append(((total - 262140).float() * scale).to(dtype))
    return torch.cat(parts).reshape(shape).double()


def layer_norm(x, eps):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def rms_norm(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def gelu(x):
    return 0.5 * x * (1 + torch.tanh(GELU_C * (x + GELU_A * x**3)))


def turn(x, pos, dims, base, sign=1.0):
    """x [T, heads, size]: pair m of the first dims dimensions is (m, m + dims / 2)."""
    half = dims // 2
    a = sign * pos[:, None, None] * base ** (-2.0 * torch.arange(half, device="cuda", dtype=torch.float64) / dims)
    u, v = x[..., :half], x[..., half:dims]
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin(), x[..., dims:]], -1)


def attend(q, k, v, scale, visible=None, sink=False):
    """q [T, H, d], k, v [S, G, d] -> [T, H d]; visible [T, S]."""
    per = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(per, 1).permute(1, 2, 0).contiguous(), v.repeat_interleave(per, 1).transpose(0, 1).contiguous()
    s = torch.matmul(q.transpose(0, 1).contiguous(), k) * scale
    if visible is not None:
        s = s.masked_fill(~visible, -math.inf)
    if sink:
        s = torch.cat([s, torch.zeros_like(s[..., :1])], -1)
    p = torch.softmax(s, -1)
    return torch.matmul(p[..., :v.shape[1]].contiguous(), v).transpose(0, 1).reshape(q.shape[0], -1)


def causal_mask(T, S=None, past=0, window=0):
    i = torch.arange(T, device="cuda")[:, None] + past
    j = torch.arange(S or T, device="cuda")[None]
    return (j <= i) & ((i - j < window) if window else True)


def exact_vision(x, layers, seed):
    d, f, L = VISION_WIDTH, VISION_HIDDEN, layers
    w = [synthetic(s, seed, 100 + i, STD) for i, s in ((0, (L, d, 3 * d)), (1, (L, 3 * d)), (2, (L, d, d)), (3, (L, d)), (4, (L, d, f)), (5, (L, f)),
                                                      (6, (L, f, d)), (7, (L, d)))]
    for i in range(L):
        h = layer_norm(x, EPS_F16)
        q, k, v = (h @ w[0][i] + w[1][i]).reshape(len(x), 3, VISION_HEADS, -1).unbind(1)
        x = x + attend(q, k, v, 72**-0.5) @ w[2][i] + w[3][i]
        h = layer_norm(x, EPS_F16)
        x = x + gelu(h @ w[4][i] + w[5][i]) @ w[6][i] + w[7][i]
    return layer_norm(x, EPS_F16)


def exact_image(seed):
    x = (torch.from_numpy(picture(seed)).cuda().double() / 255 - 0.5) / 0.5
    x = x.reshape(27, 14, 27, 14, 3).permute(0, 2, 4, 1, 3).reshape(PATCHES, PATCH_DIM)
    d = VISION_WIDTH
    x = x @ synthetic((PATCH_DIM, d), seed, 120, STD) + synthetic((d,), seed, 121, STD) + synthetic((PATCHES, d), seed, 122, STD)
    x = exact_vision(torch.cat([x, x]), VISION_LAYERS, seed)
    x = torch.cat([x[:PATCHES], x[PATCHES:]], 1)
    x = gelu(x @ synthetic((2 * d, 8192), seed, 123, STD) + synthetic((8192,), seed, 124, STD))
    return x @ synthetic((8192, 2048), seed, 125, STD) + synthetic((2048,), seed, 126, STD)


def exact_decoder(c, weight, ids, rows):
    """weight(name, layer or None) in float64; logits of the given rows."""
    x, T = weight("wte", None)[torch.from_numpy(ids.astype(np.int64)).cuda()], len(ids)
    pos, visible = torch.arange(T, device="cuda", dtype=torch.float64), causal_mask(T)
    for i in range(c["layers"]):
        h = layer_norm(x, EPS_F16)
        q, k, v = (h @ weight("Wqkv_w", i).T + weight("Wqkv_b", i)).reshape(T, 3, c["width"] // 64, 64).unbind(1)
        o = attend(turn(q, pos, 32, 1e4), turn(k, pos, 32, 1e4), v, 0.125, visible)
        x = x + (o @ weight("out_proj_w", i).T + weight("out_proj_b", i)) + (
            gelu(h @ weight("fc1_w", i).T + weight("fc1_b", i)) @ weight("fc2_w", i).T + weight("fc2_b", i))
    return layer_norm(x[rows], EPS_F16) @ weight("linear_w", None).T + weight("linear_b", None)


def synthetic_decoder_weights(c, seed):
    d, L = c["width"], c["layers"]
    shapes = dict(wte=(0, (VOCAB, d)), Wqkv_w=(3, (L, 3 * d, d)), Wqkv_b=(4, (L, 3 * d)), out_proj_w=(5, (L, d, d)), out_proj_b=(6, (L, d)), fc1_w=(7, (L, 4 * d, d)),
                  fc1_b=(8, (L, 4 * d)), fc2_w=(9, (L, d, 4 * d)), fc2_b=(10, (L, d)), linear_w=(11, (VOCAB, d)), linear_b=(12, (VOCAB,)))
    made = {}

    def weight(name, layer):
        if name not in made:
            stream, shape = shapes[name]
            made[name] = synthetic(shape, seed, stream, STD).half()
        return (made[name] if layer is None else made[name][layer]).double()

    return weight


def exact_delta(h, w1, o, p, d):
    """The gated delta rule with the sessions' random parameters: taps 0.5, decay rate 1, step bias -2, norms 1.  o: offsets of the rows of w1."""
    H, T = d // 64, len(h)
    x = torch.cat([torch.zeros(3, 3 * d, device="cuda", dtype=torch.float64), h @ w1[o["conv"]:o["conv"] + 3 * d].T])
    q, k, v = torch.nn.functional.silu(0.5 * sum(x[t:t + T] for t in range(4))).reshape(T, 3, H, 64).unbind(1)
    q, k = (y / torch.sqrt((y * y).sum(-1, keepdim=True) + 1e-6) for y in (q, k))
    q = q / 8
    inner = h @ w1[o["inner"]:o["inner"] + 128].T
    beta = torch.sigmoid(h @ w1[o["n16"]:o["n16"] + H].T)
    decay = torch.exp(-torch.nn.functional.softplus(inner[:, :64] @ p[d:, :64].T - 2.0)).reshape(T, H, 64)
    gate = torch.sigmoid(inner[:, 64:] @ p[:d, 64:].T).reshape(T, H, 64)
    S, out = torch.zeros(H, 64, 64, device="cuda", dtype=torch.float64), torch.empty(T, H, 64, device="cuda", dtype=torch.float64)
    for t in range(T):
        S = S * decay[t, :, :, None]
        u = beta[t, :, None] * (v[t] - (S * k[t, :, :, None]).sum(1))
        S = S + k[t, :, :, None] * u[:, None]
        out[t] = (S * q[t, :, :, None]).sum(1)
    return (rms_norm(out, 1e-5) * gate).reshape(T, -1)


def exact_list(c, seed, ids, rows):
    d, H, G, T, window = c["width"], c["width"] // 64, c["kv_heads"], len(ids), c["window"]
    generax, stream = c["design"] == "Generax", [0]

    def take(*shape):
        stream[0] += 1
        return synthetic(shape, seed, stream[0] - 1, STD, torch.bfloat16)

    norm = rms_norm if generax else layer_norm
    silu = torch.nn.functional.silu
    x = take(VOCAB, d)[torch.from_numpy(ids.astype(np.int64)).cuda()] * (1.0 if generax else embedding_scale(c))
    pos, visible = torch.arange(T, device="cuda", dtype=torch.float64), causal_mask(T, window=window)
    first = lent = None
    for i in range(c["layers"]):
        kind = i % 4 if generax else -1
        ff = 0 if c["experts"] else late_ff(c) if kind >= 2 else c["ff"]
        own = 0 if kind == 3 else G * 64
        o = dict(k=d, v=d + own, gate=d + 2 * own, conv=d + 2 * own)
        n16 = d + 2 * own + (0 if generax else d)
        if kind in (0, 1):
            o["inner"] = n16 + 3 * d
            n16 = o["inner"] + 128
        o["n16"] = n16
        n32 = n16 + (-(-H // 64) * 64 if kind in (0, 1) else c["experts"])
        w1 = take(n32 + 2 * ff, d)
        ka, kr = d, d if kind in (0, 1) else 0
        w2 = take(d, ka + kr + ff)
        p = take(2 * d, 128) if kr else None
        h = norm(x, 1e-5)
        q = h @ w1[:d].T
        if kind == 3:
            k, v = lent
        else:
            k, v = h @ w1[o["k"]:o["k"] + own].T, (h @ w1[o["v"]:o["v"] + own].T).reshape(T, G, 64)
        if not generax:
            q, k = rms_norm(q.reshape(T, H, 64), 1e-5), rms_norm(k.reshape(T, G, 64), 1e-5)
            first = v if first is None else first
            v = 0.5 * v + 0.5 * first
            a = attend(q, k, v, 0.125, visible, sink=True) * torch.sigmoid(h @ w1[o["gate"]:o["gate"] + d].T)
        else:
            q = rms_norm(q, 1e-5).reshape(T, H, 64)
            if kind != 3:
                k = rms_norm(k, 1e-5).reshape(T, G, 64)
            if kind < 2:
                n = T // 16
                kb, vb = (y[:16 * n].reshape(n, 16, G, 64).mean(1) for y in (k, v))
                blocks = torch.arange(n, device="cuda")[None] * 16 + 15 <= torch.arange(T, device="cuda")[:, None] - window
                a = attend(q, torch.cat([kb, k]), torch.cat([vb, v]), 0.125, torch.cat([blocks, visible], 1))
            else:
                if kind == 2:
                    k, v = turn(k, pos, 64, 1e4), turn(v, pos, 64, 1e4)
                    lent = k, v
                a = turn(attend(turn(q, pos, 64, 1e4), k, v, 0.125, visible).reshape(T, H, 64), pos, 64, 1e4, -1.0).reshape(T, d)
        if kr:
            out = 0.5 * (rms_norm(a @ w2[:, :ka].T, 1e-5) + rms_norm(exact_delta(h, w1, o, p, d) @ w2[:, ka:ka + kr].T, 1e-5))
        else:
            out = a @ w2[:, :ka].T
        if ff:
            pairs = (h @ w1[n32:].T).reshape(T, ff // 32, 2, 32)
            out = out + (silu(pairs[:, :, 0]) * pairs[:, :, 1]).reshape(T, ff) @ w2[:, ka + kr:].T
        if c["experts"]:
            s = torch.sigmoid(h @ w1[n16:n32].T)
            best = s.topk(8, -1).indices
            for e in range(c["experts"]):
                wgu, wd = take(2 * c["ff"], d), take(d, c["ff"])
                t = (best == e).any(-1).nonzero()[:, 0]
                pairs = (h[t] @ wgu.T).reshape(len(t), c["ff"] // 32, 2, 32)
                share = s[t, e] / (s[t].gather(1, best[t]).sum(-1) + 1e-20)
                out[t] += share[:, None] * ((silu(pairs[:, :, 0]) * pairs[:, :, 1]).reshape(len(t), c["ff"]) @ wd.T)
        x = x + out
    z = norm(x[rows], 1e-5) @ take(VOCAB, d).T
    return 30.0 * torch.tanh(z / 30.0) if generax else z


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "product":
        a, b, bias = (t.double() for t in product_inputs(c, seed))
        y = a @ (b.T if c["layout"] == "nk" else b)
        return y if not c["epilogue"] else y + bias if c["epilogue"] == 1 else gelu(y + bias)
    if kind == "attention":
        q, k, v = (t.double().transpose(0, 1) for t in attention_inputs(c, seed))
        o = attend(q, k, v, c["head"] ** -0.5, causal_mask(len(q), len(k), c["past"]) if c["causal"] else None)
        return o.reshape(len(q), c["heads"], -1).transpose(0, 1).contiguous()
    if kind == "image":
        return exact_image(seed)
    if kind == "encoder":
        return exact_vision(torch.from_numpy(encoder_rows(c, seed)).cuda().double(), c["layers"], seed)
    ids, n = token_ids(c, seed), c["prompt"]
    rows = [n - 1] + ([n + c["steps"] - 1] if c["steps"] else [])
    if kind == "list":
        return list(exact_list(c, seed, ids, rows))
    if kind == "decoder":
        return list(exact_decoder(c, synthetic_decoder_weights(c, seed), ids, rows))
    w, successor = reply_weights(c, seed)
    successor = successor.cpu().numpy()
    for i in range(n, n + c["steps"]):
        ids[i] = successor[ids[i - 1]]
    return dict(tokens=None, logits=exact_decoder(c, lambda name, i: (w[name] if i is None else w[name][i]).double(), ids, [n + c["steps"] - 1])[0])
