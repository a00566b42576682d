"""The inference work that a program using this framework has it do, as measurable cases.

Four kinds of case, each through the entry points that a program calls:

  forward      ``model(ids, pos, example_ids)``: a whole model over one prompt, logits at every
               position (scoring a prompt, test-time evaluation of one task).
  decode_call  one ``_decode_step`` of a whole model, launched from the host (sampling and the
               callers that drive their own loop): logits of the next token, K / V of this one.
  prompt       one layer of a batched prefill (``HipEngine.run_packed``: embedding, norm, qkv,
               RoPE, cache write, attention, out projection, SwiGLU MLP) over a left-padded batch:
               the residual stream and the layer's cache.
  decode       one layer of a batched decode step (``Generator.decode_layers``: embedding, the
               layer, LM head), replayed from a captured graph as the generation loop replays it:
               logits, residual stream, K / V of the new token.

Batches are left-padded ARC prompts (demo pairs of coloured grids, then the test input) of the
model presets' shapes; a model is bf16 or fp32 ("f32"), which selects the form of the path.
"""

import math

import numpy as np
import torch

import mdlarc_scale_amd as mdl
from mdlarc_scale_amd.engine import Scratch, engine_for, pack_prompt
from mdlarc_scale_amd.inference import Generator, StaticKVCache, _decode_step

# d_model, heads, d_ff and layers of the presets
PRESETS = {"tiny": (256, 4, 704, 4), "small": (768, 12, 2048, 4), "medium": (1024, 16, 2752, 8),
           "large": (1280, 20, 3392, 12)}
VOCAB, N_EXAMPLES, EPS, HEAD = 14, 1280, 1e-5, 64
AXES = ((32, 10), (32, 10), (8, 12))      # positions and rotation pairs of the x, y and z axes
KV_STD = 0.7                              # spread of the qkv projection's outputs at this init


def listed():
    return [
        # one prompt scored by the whole model: a single task, no batch to hide behind
        dict(name="forward_row", kind="forward", preset="small", dtype="bf16", batch=1, seq=523),
        # sampling one token for a chunk of 16 augmentations, launched from the host
        dict(name="decode_call", kind="decode_call", preset="small", dtype="bf16", batch=16,
             seq=743, spread=0.2, new=57),
        # greedy decode of one prompt: a step is launches and one pass over the weights
        dict(name="decode_row", kind="decode", preset="small", dtype="bf16", batch=1, seq=731,
             spread=0.0, new=101),
        # greedy decode of the 64 augmentations of one task
        dict(name="decode_task", kind="decode", preset="small", dtype="bf16", batch=64, seq=754,
             spread=0.1, new=333),
        # greedy decode of a full serving batch near the end of a 2,048-slot cache
        dict(name="decode_batch", kind="decode", preset="small", dtype="bf16", batch=256,
             seq=1763, spread=0.75, new=200),
        # greedy decode of an fp32 model (what the factories build unless it is converted)
        dict(name="decode_f32", kind="decode", preset="small", dtype="f32", batch=16, seq=811,
             spread=0.3, new=120),
        # prefill of a single prompt
        dict(name="prompt_row", kind="prompt", preset="small", dtype="bf16", batch=1, seq=731,
             spread=0.0),
        # prefill of a chunk of 16 augmentations
        dict(name="prompt_chunk", kind="prompt", preset="small", dtype="bf16", batch=16, seq=1203,
             spread=0.3),
        # prefill of the full serving batch: 32 tasks of very different lengths
        dict(name="prompt_batch", kind="prompt", preset="small", dtype="bf16", batch=256,
             seq=1763, spread=0.75),
        # prefill of long prompts by the widest preset
        dict(name="prompt_long", kind="prompt", preset="large", dtype="bf16", batch=8, seq=5203,
             spread=0.1),
        # prefill of a small batch by the smallest fp32 model
        dict(name="prompt_f32_tiny", kind="prompt", preset="tiny", dtype="f32", batch=8, seq=1001,
             spread=0.6),
        # prefill of a chunk of 16 by a wider fp32 model
        dict(name="prompt_f32", kind="prompt", preset="small", dtype="f32", batch=16, seq=811,
             spread=0.3),
    ]


MOST = {"flops": 3.5e12, "bytes": 3.0e9, "tokens": 300_000}   # a drawn case's largest


def draw(rng):
    while True:
        kind = rng.choice(["prompt", "prompt", "prompt", "decode", "decode", "decode", "forward",
                           "decode_call"])
        preset = rng.choice(["tiny", "small", "small", "medium", "large"])
        dtype = rng.choice(["bf16", "bf16", "f32"])
        longest = 5700 if preset == "large" else 3500 if preset == "medium" else 1800
        seq = round(math.exp(rng.uniform(math.log(90), math.log(longest))))
        batch = round(math.exp(rng.uniform(0.0, math.log(256))))
        case = dict(kind=kind, preset=preset, dtype=dtype, batch=batch, seq=seq)
        if kind == "forward":
            case["batch"] = min(batch, 16)
        else:
            case["spread"] = round(rng.uniform(0.0, 0.75), 2) if batch > 1 else 0.0
        if kind in ("decode", "decode_call"):
            case["new"] = rng.randint(1, 900)
        w = work(case)
        if (w["flops"] <= MOST["flops"] / (4 if dtype == "f32" else 1) and
                w["bytes"] <= MOST["bytes"] and batch * seq <= MOST["tokens"]):
            return case


# ---- sizes -------------------------------------------------------------------------------------

def layers_of(case):
    return PRESETS[case["preset"]][3] if case["kind"] in ("forward", "decode_call") else 1


def lengths(case):
    """Prompt length of each row: the first is the longest, the others lie at or below it."""
    seq, spread = case["seq"], case.get("spread", 0.0)
    return [max(1, seq - int(spread * seq * math.fmod(0.618034 * b, 1.0)))
            for b in range(case["batch"])]


def work(case):
    d, h, f, _ = PRESETS[case["preset"]]
    n_l, wide = layers_of(case), 4 if case["dtype"] == "f32" else 2
    lens, weights = lengths(case), 4 * d * d + 3 * d * f
    head = 2 * d * VOCAB
    if case["kind"] in ("forward", "prompt"):
        tokens, pairs = sum(lens), sum(n * (n + 1) / 2 for n in lens)
        out = (tokens * VOCAB * wide if case["kind"] == "forward"
               else tokens * (4 * d + 2 * d * wide))
        flops = n_l * (2 * tokens * weights + 4 * d * pairs)
        flops += tokens * head if case["kind"] == "forward" else 0
        return {"bytes": n_l * weights * wide + tokens * 32 + out, "flops": flops}
    slots = [n + case["new"] for n in lens]
    keys = sum(slots)
    return {"bytes": n_l * (weights * wide + keys * 2 * d * wide) + len(lens) * 4 * d,
            "flops": n_l * (2 * len(lens) * weights + 4 * d * keys) + len(lens) * head}


# Largest relative difference between two correct runs of the same precision: what another order
# of the sums gives, carried through the roundings to bf16 that follow (q, K, V, probabilities;
# none in the fp32 form, whose split weights and activations carry about 2^-17).  About four
# times the distance to exact(): 1.1e-3 to 2.0e-3 for a bf16 layer (3.4e-3 the logits of four),
# 4e-6 to 2.7e-5 in the fp32 form.
def tolerance(case):
    if case["dtype"] == "f32":
        return {"rel": 1e-4, "max": 1e-3}
    return {"rel": 1.2e-2 if case["kind"] in ("forward", "decode_call") else 7e-3, "max": 1e-1}


# ---- inputs ------------------------------------------------------------------------------------

def _prompt(rng, n):
    """The last n tokens of a sequence of demo pairs closed by IO_SEP: token ids and positions
    (column, row, layer of the sequence: start, input, separator, output, end)."""
    total, body, parts = 0, 1, []
    while total < n:
        h, w = rng.integers(3, 25, size=2)
        cells = np.where(rng.random((h, w)) < 0.5, 0, rng.integers(1, 10, size=(h, w)))
        cells = np.concatenate([cells, np.full((h, 1), 11)], axis=1).reshape(-1)
        xy = np.stack(np.meshgrid(np.arange(w + 1), np.arange(h)), -1).reshape(-1, 2)
        last, z = (12, 2) if body == 1 else (13, 4)
        first = [10] if body == 1 else []
        parts.append((np.concatenate([first, cells, [last]]).astype(np.int64),
                      np.concatenate([np.zeros((len(first), 3)),
                                      np.concatenate([xy, np.full((len(xy), 1), body)], 1),
                                      [[0, 0, z]]]).astype(np.int64)))
        total += len(parts[-1][0])
        body = 4 - body
    if parts[-1][0][-1] != 12:          # the test input closes with IO_SEP
        parts[-1][0][-1] = 12
        parts[-1][1][-1] = (0, 0, 2)
    ids = np.concatenate([p[0] for p in parts])[-n:]
    pos = np.concatenate([p[1] for p in parts])[-n:]
    return ids, pos


def _batch(case, seed):
    """Left-padded ids, positions and mask of the case's prompts, and the example ids (host)."""
    rng = np.random.default_rng(seed)
    lens = lengths(case)
    B, S = case["batch"], case["seq"]
    ids = np.full((B, S), 13, dtype=np.int64)
    pos = np.zeros((B, S, 3), dtype=np.int64)
    mask = np.zeros((B, S), dtype=bool)
    for b, n in enumerate(lens):        # 8 variants of one task, as the augmentations are
        if b % 8 == 0:
            base_ids, base_pos = _prompt(rng, S)
        perm = np.arange(14)
        perm[1:10] = 1 + rng.permutation(9)
        ids[b, S - n:], pos[b, S - n:] = perm[base_ids[S - n:]], base_pos[S - n:]
        mask[b, S - n:] = True
    ex = rng.integers(0, N_EXAMPLES, size=B)
    return [torch.from_numpy(a) for a in (ids, pos, mask, ex)]


def _weights(case, seed):
    """A state dict of the reference initialisation (xavier-uniform linears, N(0, 0.02)
    embeddings), norm gains and biases as after some training; values the model dtype holds."""
    d, h, f, _ = PRESETS[case["preset"]]
    dev = "cuda"
    g = torch.Generator(dev).manual_seed(seed)

    def xavier(n, k):
        a = math.sqrt(6.0 / (n + k))
        return (torch.rand(n, k, device=dev, generator=g) * 2 - 1) * a

    def normal(*s, std=0.02, mean=0.0):
        return torch.randn(*s, device=dev, generator=g) * std + mean

    w = {"token_embed.weight": normal(VOCAB, d), "example_embed.weight": normal(N_EXAMPLES, d)}
    for i in range(layers_of(case)):
        p = f"blocks.{i}."
        w[p + "ln1.weight"] = normal(d, std=0.1, mean=1.0)
        w[p + "attn.qkv_proj.weight"] = xavier(3 * d, d)
        w[p + "attn.out_proj.weight"] = xavier(d, d)
        w[p + "ln2.weight"] = normal(d, std=0.1, mean=1.0)
        for name, n, k in (("fc_gate", f, d), ("fc_up", f, d), ("fc_down", d, f)):
            w[p + f"ffn.{name}.weight"] = xavier(n, k)
            w[p + f"ffn.{name}.bias"] = normal(n)
    w["ln_f.weight"] = normal(d, std=0.1, mean=1.0)
    w["lm_head.weight"] = xavier(VOCAB, d)
    if case["dtype"] == "bf16":
        w = {k: v.to(torch.bfloat16) for k, v in w.items()}
    return w


def _cache_values(case, seed, shape):
    """K / V of the tokens before this one, as the projection leaves them."""
    g = torch.Generator("cuda").manual_seed(seed + 77)
    dtype = torch.float32 if case["dtype"] == "f32" else torch.bfloat16
    return (torch.randn(shape, device="cuda", generator=g, dtype=torch.float32) * KV_STD).to(dtype)


def _next_tokens(case, seed):
    """The decode step's input token and position of each row."""
    rng = np.random.default_rng(seed + 5)
    B, new = case["batch"], case["new"]
    tok = rng.integers(0, 10, size=B)
    pos = np.stack([rng.integers(0, 30, size=B), np.full(B, min(new // 12, 29)),
                    np.full(B, 3)], 1)
    return torch.from_numpy(tok), torch.from_numpy(pos)


def _model(case, seed):
    d, h, f, _ = PRESETS[case["preset"]]
    with torch.device("cuda"):
        m = mdl.create_model(d_model=d, n_heads=h, d_ff=f, n_layers=layers_of(case), dropout=0.0,
                             num_examples=N_EXAMPLES, max_seq_len=8192)
        if case["dtype"] == "bf16":
            m = m.to(torch.bfloat16)
    m.load_state_dict(_weights(case, seed))
    return m.eval()


# ---- the calls ---------------------------------------------------------------------------------

@torch.no_grad()
def prepare(case, seed):
    m = _model(case, seed)
    d, h, f, _ = PRESETS[case["preset"]]
    ids, pos, mask, ex = [t.cuda() for t in _batch(case, seed)]
    s = dict(kind=case["kind"], model=m, ids=ids, pos=pos, mask=mask, ex=ex)
    eng = engine_for(m)
    if case["kind"] == "forward":
        eng.packed(ids.device)
        return s
    B, S = ids.shape
    if case["kind"] == "decode_call":
        t = S + case["new"]
        c = StaticKVCache(B, t + 1, layers_of(case), h, HEAD, ids.device, _dtype(case))
        for i in range(layers_of(case)):
            for j in range(2):
                c.cache[i, j, :, :, :t] = _cache_values(case, seed + 10 * i + j, (B, h, t, HEAD))
        tok, tpos = _next_tokens(case, seed)
        eng.packed(ids.device)
        full = torch.cat([mask, torch.ones(B, t + 1 - S, dtype=torch.bool, device="cuda")], 1)
        s.update(cache=c, t=t, tok=tok.cuda()[:, None], tpos=tpos.cuda()[:, None], mask=full)
        return s
    gen = Generator(m)
    s.update(eng=eng, gen=gen, W=eng.packed(ids.device))
    if case["kind"] == "prompt":
        st = gen.prepare(ids, pos, ex, mask, S + 16)
        st.cache.cache.zero_()
        starts = torch.stack([st.kv_start, st.last_row]).cpu().numpy()
        pk = pack_prompt(starts[0], starts[1], B, S, ids.device)
        sc = Scratch.for_prompt(pk.n_tokens, m.config, ids.device, case["dtype"] == "f32")
        sc.x.zero_()                    # the rows that only fill up the last block of 16
        s.update(st=st, pk=pk, sc=sc)
        return s
    t = S + case["new"]
    st = gen.prepare(ids, pos, ex, mask, t + 1 + 100)
    for j in range(2):
        st.cache.cache[0, j] = _cache_values(case, seed + j, (B, h, t + 101, HEAD))
    tok, tpos = _next_tokens(case, seed)
    s["tok"] = tok.cuda()
    st.pos.copy_(tpos)
    st.counters.copy_(torch.tensor([t, t + 1], dtype=torch.int32))
    st.sc.x.zero_()
    s.update(st=st, t=t)

    def step():
        st.tok.copy_(s["tok"])
        gen.decode_layers(st, s["W"], True)

    step()                              # once from the host, then recorded
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        g.capture_begin()
        step()
        g.capture_end()
    torch.cuda.current_stream().wait_stream(side)
    s["graph"] = g
    return s


def _dtype(case):
    return torch.float32 if case["dtype"] == "f32" else torch.bfloat16


@torch.no_grad()
def run(s):
    if s["kind"] == "forward":
        return s["model"](s["ids"], s["pos"], s["ex"])
    if s["kind"] == "decode_call":
        c, t = s["cache"], s["t"]
        c.seq_len = t
        logits = _decode_step(s["model"], s["tok"], s["tpos"], s["ex"], c, s["mask"])
        return logits, c.cache[:, :, :, :, t]
    st = s["st"]
    if s["kind"] == "prompt":
        s["eng"].run_packed(s["W"], s["ids"], s["pos"], s["ex"], st.pmask, st.kv_start, s["pk"],
                            st.cache.layer, s["sc"], row_holes=st.holes)
        return s["sc"].x, st.cache.cache
    s["graph"].replay()
    return st.logits, st.sc.x, st.cache.cache[:, :, :, :, s["t"]]


# ---- the same in 64 bits, in plain torch -------------------------------------------------------

def _tile(x):
    """[rows, cols] in the residual stream's layout: 16 x 32 blocks, in each the elements 0..3 and
    4..7 of every run of 8 columns as [half][run][row][4]; rows filled up with zeros."""
    rows, cols = x.shape
    full = torch.zeros((rows + 15) // 16 * 16, cols, dtype=x.dtype, device=x.device)
    full[:rows] = x
    v = full.view(-1, 16, cols // 32, 4, 2, 4).permute(0, 2, 4, 3, 1, 5)
    return v.reshape(full.shape)


def _norm(x, gain):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gain


def _rope(v, pos):
    """v [n, heads, 64] rotated by the positions [n, 3]."""
    ang = []
    for axis, (n_pos, pairs) in enumerate(AXES):
        freq = 1.0 / (10000.0 ** (torch.arange(0, 2 * pairs, 2, device=v.device,
                                               dtype=torch.float64) / (2 * pairs)))
        ang.append(pos[:, axis].clamp(0, n_pos - 1).double()[:, None] * freq)
    ang = torch.cat(ang, 1)[:, None]
    a, b = v[..., 0::2], v[..., 1::2]
    return torch.stack((a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()),
                       -1).flatten(-2)


def _layer_qkv(w, p, x, pos, h):
    n, d = x.shape
    q, k, v = (_norm(x, w[p + "ln1.weight"]) @ w[p + "attn.qkv_proj.weight"].T).view(
        n, 3, h, HEAD).unbind(1)
    return _rope(q, pos), _rope(k, pos), v


def _mlp(w, p, x):
    y = _norm(x, w[p + "ln2.weight"])
    gate = y @ w[p + "ffn.fc_gate.weight"].T + w[p + "ffn.fc_gate.bias"]
    up = y @ w[p + "ffn.fc_up.weight"].T + w[p + "ffn.fc_up.bias"]
    return x + (torch.nn.functional.silu(gate) * up) @ w[p + "ffn.fc_down.weight"].T + \
        w[p + "ffn.fc_down.bias"]


def _prompt_layer(w, p, x, pos, h):
    """One row of a prompt through a layer: x after it, K and V."""
    n, d = x.shape
    q, k, v = _layer_qkv(w, p, x, pos, h)
    o = torch.empty_like(q)
    future = torch.ones(n, n, dtype=torch.bool, device=x.device).triu(1)
    for i in range(h):
        s = (q[:, i] @ k[:, i].T / 8.0).masked_fill_(future, float("-inf"))
        o[:, i] = s.softmax(-1) @ v[:, i]
    return _mlp(w, p, x + o.reshape(n, d) @ w[p + "attn.out_proj.weight"].T), k, v


def _exact_prompt(case, w, ids, pos, mask, ex):
    d, h, f, _ = PRESETS[case["preset"]]
    B, S = ids.shape
    lens = lengths(case)
    rows, extra = [], []
    cache = torch.zeros(1, 2, B, h, S + 16, HEAD, dtype=torch.float64, device="cuda")
    for b, n in enumerate(lens):
        x = w["token_embed.weight"][ids[b, S - n:]] + w["example_embed.weight"][ex[b]]
        x, k, v = _prompt_layer(w, "blocks.0.", x, pos[b, S - n:], h)
        rows.append(x)
        cache[0, 0, b, :, S - n:S], cache[0, 1, b, :, S - n:S] = k.transpose(0, 1), v.transpose(0, 1)
        if n - 1 < S - n:               # index length-1 is a padding token: no key, no attention
            x = w["token_embed.weight"][ids[b, n - 1]] + w["example_embed.weight"][ex[b]]
            extra.append(_mlp(w, "blocks.0.", x[None]))
    return _tile(torch.cat(rows + extra)), cache


def _exact_decode(case, seed, w, ex):
    d, h, f, _ = PRESETS[case["preset"]]
    lens, B, S = lengths(case), case["batch"], case["seq"]
    t = S + case["new"]
    tok, pos = [v.cuda() for v in _next_tokens(case, seed)]
    whole = case["kind"] == "decode_call"
    x = w["token_embed.weight"][tok] + w["example_embed.weight"][ex]
    new = []
    for i in range(layers_of(case)):
        p = f"blocks.{i}."
        past = [_cache_values(case, seed + (10 * i if whole else 0) + j,
                              (B, h, t if whole else t + 101, HEAD)) for j in range(2)]
        q, k, v = _layer_qkv(w, p, x, pos, h)
        new.append(torch.stack((k, v)))
        o = torch.empty_like(q)
        for b in range(B):
            K, V = (torch.cat([c[b, :, S - lens[b]:t].double(), u[b][:, None]], 1)
                    for c, u in zip(past, (k, v)))
            s = (K @ q[b][:, :, None])[..., 0] / 8.0
            o[b] = (s.softmax(-1)[:, None] @ V)[:, 0]
        x = _mlp(w, p, x + o.reshape(B, d) @ w[p + "attn.out_proj.weight"].T)
    logits = _norm(x, w["ln_f.weight"]) @ w["lm_head.weight"].T
    if whole:
        return logits[:, None], torch.stack(new)
    return logits, _tile(x), torch.stack(new)


@torch.no_grad()
def exact(case, seed):
    w = {k: v.double() for k, v in _weights(case, seed).items()}
    ids, pos, mask, ex = [t.cuda() for t in _batch(case, seed)]
    if case["kind"] == "prompt":
        return _exact_prompt(case, w, ids, pos, mask, ex)
    if case["kind"] in ("decode", "decode_call"):
        return _exact_decode(case, seed, w, ex)
    out = []
    for b in range(case["batch"]):
        x = w["token_embed.weight"][ids[b]] + w["example_embed.weight"][ex[b]]
        for i in range(layers_of(case)):
            x = _prompt_layer(w, f"blocks.{i}.", x, pos[b], PRESETS[case["preset"]][1])[0]
        out.append(_norm(x, w["ln_f.weight"]) @ w["lm_head.weight"].T)
    return torch.stack(out)
