"""Performance cases of the serving kernels: what a layer of each model design runs between its
matrix products, through the public entry points of `ops` and `ops.stream`, in the two forms a
serving engine calls them in -- a step of prompt chunks ("prompt") and a step of single rows of
running sequences ("decode") -- plus the routed experts of the mixture models.

A case is a dict:
  kind      gqa        Qwen3 / Llama attention: q / k norms, rotation, paged cache, attention
            sink       Bidetar attention: whole-projection norms, chunk mask, sinks, gates
            latent     Puputar / Venanex latent attention over one cached row per token
            talk       Sazepel attention whose heads mix their softmax weights
            pooled     Mudepel attention over a window and pooled blocks
            retention  Sazepel retention (decayed linear attention with a state)
            ssm        Mudepel state-space mixer: convolution, scan, gated group norm
            experts    router and expert feed-forward (softmax router over the top choices)
  phase     prompt | decode
  seqs, tokens, past, spread    sequences of the step; new tokens of the longest prompt chunk
            (1 for decode rows); cached tokens before it (prompt: of every sequence, decode: of
            the longest); how far the other sequences fall short of the longest (0: none do)
  dtype     bf16 | f32 (the designs' replay mode) | fp8 (bf16 rows over an e4m3 cache)
and the head / state / expert sizes of the layer.  The sizes are those of the registered models
and of `bench.py`: prompts of 512 to 2048 tokens in steps of up to 16384, decoding at contexts of
some hundred to some thousand tokens, pages of 32 tokens, models of 4096 positions."""
import math

import torch

from aws_k8s_ansible_provisioner_amd import ops
from aws_k8s_ansible_provisioner_amd.ops import stream as sops

PAGE = 32           # tokens per cache page
MAX_LEN = 4096      # positions of the served model
EPS = 1e-5
DEV = "cuda"

# layer sizes of the registered models, per kind
QWEN = dict(heads=16, kv_heads=8, dim=128, qk_norm=True)        # Qwen3-0.6B
LLAMA = dict(heads=32, kv_heads=8, dim=128, qk_norm=False)      # Llama-3-8B
SINK_2048 = dict(heads=16, kv_heads=4, dim=128, chunk=8192)     # bidetar-w2048
SINK_4096 = dict(heads=32, kv_heads=8, dim=128, chunk=8192)     # bidetar-w4096
SINK_D64 = dict(heads=24, kv_heads=8, dim=64, chunk=1024)       # bidetar-w1536-d64
LATENT_2048 = dict(heads=16, q_rank=768, kv_rank=512, rot=64, dim=128)     # puputar-w2048
LATENT_4096 = dict(heads=32, q_rank=1536, kv_rank=512, rot=64, dim=128)    # puputar-w4096
TALK_2048 = dict(heads=16, kv_heads=4, dim=128)                 # sazepel-w2048
TALK_4096 = dict(heads=32, kv_heads=8, dim=128)                 # sazepel-w4096
POOLED_2048 = dict(heads=16, kv_heads=4, dim=128, window=1024, pool=64)    # mudepel-w2048
POOLED_4096 = dict(heads=32, kv_heads=8, dim=128, window=1024, pool=64)    # mudepel-w4096
RET_2048 = dict(heads=8, dim=128, rot=64)                       # sazepel-w2048
RET_4096 = dict(heads=16, dim=128, rot=64)                      # sazepel-w4096
SSM_2048 = dict(heads=64, dim=64, state=128, groups=1, taps=4, norm_groups=1)    # mudepel-w2048
SSM_4096 = dict(heads=128, dim=64, state=128, groups=8, taps=4, norm_groups=8)   # mudepel-w4096
EXPERTS_2048 = dict(width=2048, ff=1408, experts=8, top=2)      # sazepel-w2048
EXPERTS_4096 = dict(width=4096, ff=3584, experts=8, top=2)      # sazepel-w4096
MIXTRAL = dict(width=4096, ff=14336, experts=8, top=2)          # Mixtral 8x7B


def _case(name, kind, phase, seqs, tokens, past, spread, dtype, sizes):
    return dict(name=name, kind=kind, phase=phase, seqs=seqs, tokens=tokens, past=past,
                spread=spread, dtype=dtype, **sizes)


def listed():
    return [
        # one user chatting: a single row of the headline model, where launches count
        _case("gqa decode, 1 row", "gqa", "decode", 1, 1, 900, 0.0, "bf16", QWEN),
        # the headline benchmark's prompt step: 512-token prompts, ragged as real ones are
        _case("gqa prompts, ragged", "gqa", "prompt", 37, 512, 0, 0.7, "bf16", QWEN),
        # the design benchmark's prompt step: 8 prompts of 2048 tokens
        _case("sink prompts", "sink", "prompt", 8, 2048, 0, 0.0, "bf16", SINK_2048),
        # a few long prompts of unequal, odd lengths
        _case("latent prompts, ragged", "latent", "prompt", 5, 2047, 0, 0.5, "bf16", LATENT_2048),
        # the design benchmark's decode step: 64 sequences at ~2100 cached tokens
        _case("latent decode, 64 rows", "latent", "decode", 64, 1, 2112, 0.1, "bf16",
              LATENT_2048),
        # second chunk of prompts that were cut by the step's token budget
        _case("talk prompts, continued", "talk", "prompt", 8, 1000, 1000, 0.2, "bf16",
              TALK_2048),
        _case("retention prompts", "retention", "prompt", 8, 2048, 0, 0.0, "bf16", RET_2048),
        # long documents: most keys are behind the window and seen as pooled blocks
        _case("pooled prompts, ragged", "pooled", "prompt", 5, 3001, 0, 0.3, "bf16",
              POOLED_2048),
        _case("ssm prompts", "ssm", "prompt", 8, 2048, 0, 0.0, "bf16", SSM_2048),
        _case("ssm decode, 64 rows", "ssm", "decode", 64, 1, 2112, 0.0, "bf16", SSM_2048),
        # a full prompt step through the routed experts (sizes of the 2048-wide models)
        _case("experts, prompt step", "experts", "prompt", 8, 2048, 0, 0.1, "bf16",
              EXPERTS_2048),
        # a decode step of the mixture model: the weights of every expert are read
        _case("experts, 48 rows", "experts", "decode", 48, 1, 0, 0.0, "bf16", MIXTRAL),
    ]


def _unnamed(*rest):
    case = _case(None, *rest)
    del case["name"]
    return case


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["gqa", "gqa", "sink", "latent", "talk", "pooled", "retention", "ssm",
                       "experts"])
    wide = rng.random() < 0.3
    phase = "decode" if rng.random() < 0.4 else "prompt"
    dtype = "bf16"
    if kind == "gqa":
        sizes = rng.choice([QWEN, LLAMA])
        wide = sizes is LLAMA
        if rng.random() < 0.2:
            dtype = "fp8"
    elif kind == "sink":
        sizes = SINK_4096 if wide else rng.choice([SINK_2048, SINK_2048, SINK_D64])
    elif kind == "experts":
        sizes = EXPERTS_4096 if wide else EXPERTS_2048
        if phase == "decode":
            sizes = MIXTRAL     # the other routed designs' decode rows run all experts densely
    else:
        small, big = {"latent": (LATENT_2048, LATENT_4096), "talk": (TALK_2048, TALK_4096),
                      "pooled": (POOLED_2048, POOLED_4096), "retention": (RET_2048, RET_4096),
                      "ssm": (SSM_2048, SSM_4096)}[kind]
        sizes = big if wide else small
        if kind in ("retention", "ssm") and rng.random() < 0.2:
            dtype = "f32"
    spread = round(rng.choice([0.0, rng.uniform(0.05, 0.9)]), 2)
    if phase == "decode":
        return _unnamed(kind, phase, _log(rng, 1, 96 if wide else 200), 1,
                        _log(rng, 40, 3000), spread, dtype, sizes)
    budget = _log(rng, 48, 6000 if wide else 12000)         # new tokens of the step
    if kind == "experts":
        budget = max(budget, 300)   # smaller steps of the routed designs run without the sort
    longest = min(_log(rng, 24, 2300), budget)
    seqs = max(1, min(64, budget // longest))
    past = rng.choice([0, 0, rng.randint(1, 1200)])
    return _unnamed(kind, phase, seqs, longest, past, spread, dtype, sizes)


# ---------------------------------------------------------------------------- the step's shape
def _lengths(n, longest, spread):
    """n lengths from `longest` down to (1 - spread) of it, in no particular order."""
    return [max(1, int(longest * (1.0 - spread * ((i * 0.6180339887) % 1.0)))) for i in range(n)]


def _shape(case):
    """[(cached tokens, new tokens)] of the step's sequences."""
    if case["phase"] == "decode":
        return [(n, 1) for n in _lengths(case["seqs"], case["past"], case["spread"])]
    return [(case["past"], n) for n in _lengths(case["seqs"], case["tokens"], case["spread"])]


def _rows(case):
    return sum(n for _, n in _shape(case))


class _Step:
    """The staged step as the engine hands it to the kernels: positions, cache slots, block
    tables, sequence starts and the tile map of prompt chunks (ascending work)."""

    def __init__(self, case, gen, group=1, tile_rows=128):
        shape = _shape(case)
        B = len(shape)
        pages = [-(-(p + n) // PAGE) for p, n in shape]
        self.num_blocks = sum(pages) + 2
        order = torch.randperm(self.num_blocks, generator=gen, device=DEV).cpu()
        tables = torch.zeros(B, MAX_LEN // PAGE, dtype=torch.int32)
        pos, slots, start, at, tiles = [], [], [0], 0, []
        for b, (p, n) in enumerate(shape):
            mine = order[at:at + pages[b]]
            at += pages[b]
            tables[b, :pages[b]] = mine.to(torch.int32)
            where = torch.arange(p, p + n)
            pos.append(where)
            slots.append(mine[where // PAGE] * PAGE + where % PAGE)
            start.append(start[-1] + n)
            for r in range(0, n * group, tile_rows):
                tiles.append((p + min(n, (r + tile_rows + group - 1) // group), b, r))
        tiles.sort(key=lambda t: t[0])
        self.shape, self.T, self.B = shape, start[-1], B
        self.positions = torch.cat(pos).to(DEV)
        self.slots = torch.cat(slots).to(DEV)
        self.tables = tables.to(DEV)
        self.seq_lens = torch.tensor([p + n for p, n in shape], dtype=torch.int32, device=DEV)
        self.q_start = torch.tensor(start, dtype=torch.int32, device=DEV)
        self.tile_seq = torch.tensor([t[1] for t in tiles], dtype=torch.int32, device=DEV)
        self.tile_row = torch.tensor([t[2] for t in tiles], dtype=torch.int32, device=DEV)
        self.tile_rows = tile_rows
        # one state slot per sequence, given per token row
        seq = torch.repeat_interleave(torch.arange(B), torch.tensor([n for _, n in shape]))
        self.seq_slot = (B - 1 - seq).to(torch.int32).to(DEV)
        self.prompt = case["phase"] == "prompt"


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 13)
    return g


def _normal(g, *shape, std=1.0, mean=0.0, dtype=torch.float32):
    return torch.empty(*shape, device=DEV).normal_(mean, std, generator=g).to(dtype)


def _angles(dims, base=500000.0):
    """fp32 [MAX_LEN, dims] = [cos | sin] of position times frequency."""
    f = torch.tensor(base, dtype=torch.float64) ** (-2.0 * torch.arange(dims // 2,
                                                                        dtype=torch.float64) / dims)
    a = torch.arange(MAX_LEN, dtype=torch.float64)[:, None] * f[None, :]
    return torch.cat([torch.cos(a), torch.sin(a)], dim=1).float().to(DEV)


def _dtype(case):
    return torch.float32 if case["dtype"] == "f32" else torch.bfloat16


# ---------------------------------------------------------------------------- prepare
def prepare(case, seed):
    g = _gen(seed)
    s = {"case": case}
    _PREPARE[case["kind"]](case, g, s)
    return s


def _prepare_gqa(c, g, s):
    H, G, D = c["heads"], c["kv_heads"], c["dim"]
    fp8 = c["dtype"] == "fp8"
    long = max(n for _, n in _shape(c)) * (H // G) > 1024
    st = s["step"] = _Step(c, g, H // G, 256 if long and not fp8 else 128)
    s["qkv"] = _normal(g, st.T, (H + 2 * G) * D, dtype=torch.bfloat16)
    k = _normal(g, st.num_blocks, G, PAGE, D)
    v = _normal(g, st.num_blocks, G, PAGE // 8, D, 8)
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    s["k"], s["v"] = (t.to(dt).view(torch.uint8) if fp8 else t.to(dt) for t in (k, v))
    s["cos_sin"] = _angles(D, 1e6)
    s["qw"], s["kw"] = [(_normal(g, D, std=0.1, mean=1.0, dtype=torch.bfloat16)
                         if c["qk_norm"] else None) for _ in range(2)]
    s["out"] = torch.empty(st.T, H, D, dtype=torch.bfloat16, device=DEV)
    s["q"] = torch.empty_like(s["out"])
    if not st.prompt:
        wgs = st.B * G
        parts = 1 if wgs >= 2048 else min(-(-2048 // wgs), MAX_LEN // 256)
        s["part_size"] = -(-(-(-MAX_LEN // parts)) // 128) * 128
        s["parts"] = -(-MAX_LEN // s["part_size"])
        s["ws"] = ops.decode_workspace(st.B, G, H // G, s["parts"], DEV)
        s["tail"] = s["tail_slot"] = None
        if not fp8:
            # the sequences' still-partial 8-token value groups, as earlier steps left them
            s["tail"] = torch.zeros(st.B, G, 8, D, dtype=torch.bfloat16, device=DEV)
            s["tail_slot"] = st.seq_slot
            page, off = st.slots // PAGE, st.slots % PAGE
            group = s["v"][page, :, off // 8].transpose(-1, -2)            # [B, G, 8, D]
            known = torch.arange(8, device=DEV)[None, :] < (off % 8)[:, None]
            s["tail"][st.seq_slot.long()] = group * known[:, None, :, None]


def _prepare_sink(c, g, s):
    H, G, D = c["heads"], c["kv_heads"], c["dim"]
    st, dt = _Step(c, g), _dtype(c)
    s["step"] = st
    s["proj"] = _normal(g, st.T, (H + G) * D + H, dtype=dt)
    s["k"] = _normal(g, st.num_blocks, G, PAGE, D, dtype=dt)
    s["v"] = _normal(g, st.num_blocks, G, PAGE // 8, D, 8, dtype=dt)
    s["cos_sin"] = _angles(D)
    s["qw"], s["kw"] = (_normal(g, n * D, std=0.1, mean=1.0) for n in (H, G))
    s["qb"], s["kb"] = (_normal(g, n * D, std=0.02, dtype=dt) for n in (H, G))
    s["sink"] = _normal(g, H)
    s["q"] = torch.empty(st.T, H, D, dtype=dt, device=DEV)
    s["out"] = torch.empty(st.T, H * D, dtype=dt, device=DEV)
    wgs = st.B * G
    span = -(-min(MAX_LEN, c["chunk"]) // sops.DECODE_PART)
    s["parts"] = 1 if wgs >= 1024 else min(span, 64, -(-1024 // wgs))
    s["ws"] = None
    if s["parts"] > 1 and not st.prompt:
        s["ws"] = sops.decode_workspace(st.B, H, D, s["parts"], DEV)


def _prepare_latent(c, g, s):
    H, R, r, D, Q = c["heads"], c["kv_rank"], c["rot"], c["dim"], c["q_rank"]
    st = s["step"] = _Step(c, g)
    bf = torch.bfloat16
    s["proj"] = _normal(g, st.T, Q + R + r, dtype=bf)
    s["rows"] = _normal(g, st.num_blocks, PAGE, R + r, dtype=bf)
    s["groups"] = s["rows"][:, :, :R].reshape(-1, PAGE // 8, 8, R).transpose(2, 3).contiguous()
    s["cos_sin"] = _angles(r)
    s["qw"], s["kvw"] = _normal(g, Q, std=0.1, mean=1.0), _normal(g, R, std=0.1, mean=1.0)
    s["cq"] = torch.empty(st.T, Q, dtype=bf, device=DEV)
    # the heads' queries: rotated part beside the part already multiplied into the latent space
    s["q"] = _normal(g, st.T, H, D + r, dtype=bf)
    s["q_lat"] = _normal(g, H, st.T, R, std=0.5, dtype=bf)
    s["out"] = torch.empty(H, st.T, R, dtype=bf, device=DEV)
    s["parts"] = min(MAX_LEN // 128, 64, max(1, -(-256 // (st.B * -(-H // 32)))))
    s["ws"] = None
    if s["parts"] > 1 and not st.prompt:
        s["ws"] = sops.latent_decode_workspace(st.B, H, R, s["parts"], DEV)


def _prepare_talk(c, g, s):
    H, G, D = c["heads"], c["kv_heads"], c["dim"]
    st = s["step"] = _Step(c, g)
    bf = torch.bfloat16
    s["proj"] = _normal(g, st.T, 2 * H * D + 2 * G * D, dtype=bf)
    # cached keys and values have been divided by their root mean square
    s["k"] = _normal(g, st.num_blocks, G, PAGE, D, dtype=bf)
    s["v"] = _normal(g, st.num_blocks, G, PAGE // 8, D, 8, dtype=bf)
    s["talk"] = torch.eye(H, device=DEV) + _normal(g, H, H, std=0.2)
    s["q"] = torch.empty(st.T, H, D, dtype=bf, device=DEV)
    s["out"] = torch.empty(st.T, H * D, dtype=bf, device=DEV)
    if not st.prompt:
        s["parts"] = sops.talking_attention_parts(st.T, G, MAX_LEN)
        s["ws"] = sops.talking_attention_workspace(st.T, H, G, D, s["parts"], DEV)


def _prepare_pooled(c, g, s):
    H, G, D = c["heads"], c["kv_heads"], c["dim"]
    st = s["step"] = _Step(c, g)
    bf = torch.bfloat16
    s["proj"] = _normal(g, st.T, (H + 2 * G) * D, dtype=bf)
    s["bias"] = _normal(g, (H + 2 * G) * D, std=0.1)
    s["k"] = _normal(g, st.num_blocks, G, PAGE, D, dtype=bf)
    s["v"] = _normal(g, st.num_blocks, G, PAGE // 8, D, 8, dtype=bf)
    n = sops.pool_slots(PAGE, c["pool"])
    s["kp"], s["vp"] = (_normal(g, st.num_blocks, G, n, D, std=c["pool"] ** -0.5)
                        for _ in range(2))
    s["cos_sin"] = _angles(D)
    s["q"] = torch.empty(st.T, H, D, dtype=bf, device=DEV)
    s["out"] = torch.empty(st.T, H * D, dtype=bf, device=DEV)


def _prepare_retention(c, g, s):
    H, D = c["heads"], c["dim"]
    st, dt = _Step(c, g), _dtype(c)
    s["step"] = st
    s["proj"] = _normal(g, st.T, 4 * H * D, dtype=dt)
    s["state"] = _normal(g, st.B, H, D, D)
    s["cos_sin"] = _angles(c["rot"])
    h = torch.arange(H, dtype=torch.float64)
    s["log2_decay"] = torch.log2(1.0 - 2.0 ** (-5.0 - 5.0 * h / max(1, H - 1))).float().to(DEV)
    s["out"] = torch.empty(st.T, H * D, dtype=dt, device=DEV)


def _prepare_ssm(c, g, s):
    H, V, N, G, taps = c["heads"], c["dim"], c["state"], c["groups"], c["taps"]
    st, dt = _Step(c, g), _dtype(c)
    s["step"] = st
    inner, C = H * V, H * V + 2 * G * N
    s["proj"] = _normal(g, st.T, inner + C + H, dtype=dt)
    s["conv_w"], s["conv_b"] = _normal(g, C, taps, std=0.3), _normal(g, C, std=0.1)
    s["dt_bias"] = _normal(g, H, std=0.5, mean=-1.0)
    s["a_log"] = _normal(g, H, std=0.5)
    s["d_skip"] = _normal(g, H, std=0.2, mean=1.0)
    s["gnorm"] = _normal(g, inner, std=0.1, mean=1.0)
    s["conv_state"] = _normal(g, st.B, taps - 1, C, dtype=dt)
    s["state"] = _normal(g, st.B, H, N, V, std=0.3)
    s["xbc"] = torch.empty(st.T, C, device=DEV)
    s["y"] = torch.empty(st.T, inner, device=DEV)
    s["out"] = torch.empty(st.T, inner, dtype=dt, device=DEV)


def _prepare_experts(c, g, s):
    d, F, E = c["width"], c["ff"], c["experts"]
    T, bf = _rows(c), torch.bfloat16
    s["h"] = _normal(g, T, d, dtype=bf)
    s["router"], s["router_b"] = _normal(g, E, d, std=0.03), _normal(g, E, std=0.1)
    s["w13"] = torch.empty(E, 2 * F, d, dtype=bf, device=DEV).normal_(0.0, 0.02, generator=g)
    s["w2"] = torch.empty(E, d, F, dtype=bf, device=DEV).normal_(0.0, 0.02, generator=g)


_PREPARE = {"gqa": _prepare_gqa, "sink": _prepare_sink, "latent": _prepare_latent,
            "talk": _prepare_talk, "pooled": _prepare_pooled, "retention": _prepare_retention,
            "ssm": _prepare_ssm, "experts": _prepare_experts}


# ---------------------------------------------------------------------------- run
def run(s):
    return _RUN[s["case"]["kind"]](s["case"], s)


def _run_gqa(c, s):
    H, G, D = c["heads"], c["kv_heads"], c["dim"]
    st, scale = s["step"], c["dim"] ** -0.5
    if st.prompt:
        ops.qk_norm_rope_cache(s["qkv"], s["q"], s["k"], s["v"], st.positions, st.slots,
                               s["cos_sin"], s["qw"], s["kw"], H, G, EPS, True, q_rows=0)
        ops.paged_attention_prefill(s["out"], s["q"], s["k"], s["v"], st.tables, st.seq_lens,
                                    st.q_start, st.tile_seq, st.tile_row, H // G, scale,
                                    tile_rows=st.tile_rows,
                                    qprep=(s["qkv"], st.positions, s["cos_sin"], s["qw"], EPS))
        return {"out": s["out"], "k": s["k"], "v": s["v"]}
    ops.paged_attention_decode_fused(s["out"], s["qkv"], s["k"], s["v"], st.tables, st.seq_lens,
                                     st.positions, st.slots, s["cos_sin"], s["qw"], s["kw"],
                                     H // G, scale, EPS, workspace=s["ws"], num_parts=s["parts"],
                                     part_size=s["part_size"], v_tail=s["tail"],
                                     tail_slot=s["tail_slot"])
    return {"out": s["out"], "k": s["k"], "v": s["v"], "tail": s["tail"]}


def _run_sink(c, s):
    H, G, D = c["heads"], c["kv_heads"], c["dim"]
    st, proj = s["step"], s["proj"]
    sops.proj_norm_rope_cache(proj, s["q"], s["k"], s["v"], st.positions, st.slots, s["cos_sin"],
                              s["qw"], s["kw"], H, G, D, 0, H * D, EPS, s["qb"], s["kb"])
    gate = proj[:, (H + G) * D:]
    if st.prompt:
        sops.sink_attention_prefill(s["out"], s["q"], s["k"], s["v"], st.tables, st.seq_lens,
                                    st.q_start, st.tile_seq, st.tile_row, st.tile_rows, gate,
                                    s["sink"], D ** -0.5, c["chunk"])
    else:
        sops.sink_attention_decode(s["out"], s["q"], s["k"], s["v"], st.tables, st.seq_lens,
                                   gate, s["sink"], D ** -0.5, c["chunk"], 0, s["ws"], s["parts"])
    return {"out": s["out"], "k": s["k"], "v": s["v"]}


def _run_latent(c, s):
    R, r, D, Q = c["kv_rank"], c["rot"], c["dim"], c["q_rank"]
    st, scale = s["step"], (c["dim"] + c["rot"]) ** -0.5
    sops.latent_prep(s["proj"], s["cq"], s["rows"], st.positions, st.slots, s["cos_sin"], s["qw"],
                     s["kvw"], Q, R, r, 0, Q, EPS, s["groups"])
    if st.prompt:
        sops.latent_attention_prefill(s["out"], s["q_lat"], s["q"], D, s["rows"], s["groups"],
                                      st.tables, st.seq_lens, st.q_start, st.positions,
                                      st.tile_seq, st.tile_row, st.tile_rows, scale)
    else:
        sops.latent_attention_decode(s["out"], s["q_lat"], s["q"], D, s["rows"], s["groups"],
                                     st.tables, st.seq_lens, st.positions, scale, s["ws"],
                                     s["parts"])
    return {"out": s["out"], "cq": s["cq"], "rows": s["rows"], "groups": s["groups"]}


def _run_talk(c, s):
    H, G, D = c["heads"], c["kv_heads"], c["dim"]
    st, proj, scale = s["step"], s["proj"], c["dim"] ** -0.5
    nq, nk = H * D, G * D
    sops.head_norm_cache(proj, s["q"], s["k"], s["v"], st.slots, H, G, D, D, 0, nq, nq + nk, EPS)
    gate = proj[:, nq + 2 * nk:]
    if st.prompt:
        sops.talking_attention_prefill(s["out"], s["q"], s["k"], s["v"], st.tables, st.seq_lens,
                                       st.q_start, st.positions, st.tile_seq, st.tile_row,
                                       st.tile_rows, s["talk"], gate, scale)
    else:
        sops.talking_attention_decode(s["out"], s["q"], s["k"], s["v"], st.tables, st.seq_lens,
                                      st.positions, s["talk"], gate, scale, s["ws"], s["parts"])
    return {"out": s["out"], "k": s["k"], "v": s["v"]}


def _run_pooled(c, s):
    H, G, D, W, P = c["heads"], c["kv_heads"], c["dim"], c["window"], c["pool"]
    st, scale = s["step"], c["dim"] ** -0.5
    sops.bias_rope_cache(s["proj"], s["q"], s["k"], s["v"], st.positions, st.slots, s["cos_sin"],
                         s["bias"], H, G, D, D, 0, H * D, (H + G) * D)
    sops.pool_cache_blocks(s["k"], s["v"], s["kp"], s["vp"], st.positions, st.slots, st.tables,
                           st.q_start if st.prompt else None, P)
    if st.prompt:
        sops.pooled_window_attention_prefill(s["out"], s["q"], s["k"], s["v"], s["kp"], s["vp"],
                                             st.tables, st.q_start, st.positions, st.slots,
                                             st.tile_seq, st.tile_row, st.tile_rows, scale, W, P,
                                             True)
    else:
        sops.pooled_window_attention_decode(s["out"], s["q"], s["k"], s["v"], s["kp"], s["vp"],
                                            st.tables, st.positions, st.slots, scale, W, P, True)
    return {"out": s["out"], "k": s["k"], "v": s["v"], "kp": s["kp"], "vp": s["vp"]}


def _run_retention(c, s):
    H, D = c["heads"], c["dim"]
    st = s["step"]
    sops.retention(s["out"], s["proj"], 0, H * D, 2 * H * D, 3 * H * D, s["state"], st.seq_slot,
                   st.positions, st.q_start if st.prompt else None, s["cos_sin"],
                   s["log2_decay"], H, D, D, EPS)
    return {"out": s["out"], "state": s["state"]}


def _run_ssm(c, s):
    H, V, N, G = c["heads"], c["dim"], c["state"], c["groups"]
    st, proj = s["step"], s["proj"]
    q_start = st.q_start if st.prompt else None
    inner, C = H * V, H * V + 2 * G * N
    sops.conv_silu(s["xbc"], proj, inner, s["conv_w"], s["conv_b"], s["conv_state"], st.seq_slot,
                   st.positions, q_start)
    sops.selective_scan(s["y"], s["xbc"], proj, inner + C, s["dt_bias"], s["a_log"], s["d_skip"],
                        s["state"], st.seq_slot, st.positions, q_start, H, V, N, G)
    sops.gate_group_norm(s["out"], s["y"], proj[:, :inner], s["gnorm"], c["norm_groups"], EPS)
    return {"out": s["out"], "y": s["y"], "state": s["state"], "conv_state": s["conv_state"]}


def _run_experts(c, s):
    ids, w = sops.route_topk(s["h"], s["router"], s["router_b"], c["top"])
    return {"out": ops.fused_moe(s["h"], s["w13"], s["w2"], w, ids), "ids": ids, "w": w}


_RUN = {"gqa": _run_gqa, "sink": _run_sink, "latent": _run_latent, "talk": _run_talk,
        "pooled": _run_pooled, "retention": _run_retention, "ssm": _run_ssm,
        "experts": _run_experts}


# ---------------------------------------------------------------------------- work
def _visible(case):
    """(sum over the new rows of the keys they see, distinct cached keys that are read)."""
    chunk, window, pool = case.get("chunk", 0), case.get("window", 0), case.get("pool", 0)
    seen = distinct = 0
    for p, n in _shape(case):
        first = 0
        for i in range(p, p + n):
            lo = i // chunk * chunk if chunk else 0
            if window:
                lo = max(lo, i - window + 1)
            seen += i - lo + 1 + (lo // pool if pool else 0)
            if i == p:
                first = lo
        distinct += p + n - first
    return seen, distinct


def work(case):
    c, T = case, _rows(case)
    kind, es = c["kind"], 4 if case["dtype"] == "f32" else 2
    if kind == "experts":
        d, F, E, top = c["width"], c["ff"], c["experts"], c["top"]
        used = min(E, T * top)
        return {"bytes": used * 3 * F * d * 2 + 2 * T * d * 2 + E * d * 4,
                "flops": T * top * 6 * F * d + 2 * T * E * d}
    H, D = c["heads"], c["dim"]
    if kind == "retention":
        # one row in, one out, the state in and out; per state entry a decay, an outer product
        # and a read-out
        return {"bytes": T * 5 * H * D * es + 2 * c["seqs"] * H * D * D * 4,
                "flops": T * H * D * D * 5}
    if kind == "ssm":
        N, G = c["state"], c["groups"]
        inner, C = H * D, H * D + 2 * G * N
        return {"bytes": T * ((inner + C + H) * es + inner * (4 + es))
                + 2 * c["seqs"] * (H * N * D * 4 + (c["taps"] - 1) * C * es),
                "flops": T * (H * N * D * 6 + 2 * C * c["taps"] + 8 * inner)}
    seen, distinct = _visible(c)
    if kind == "latent":
        R, r, Q = c["kv_rank"], c["rot"], c["q_rank"]
        row = R + r
        return {"bytes": 2 * (T * (Q + row) + T * Q + 2 * T * row + T * R
                              + T * H * (2 * R + r) + (distinct - T) * row),
                "flops": seen * H * 2 * (row + R)}
    G = c["kv_heads"]
    ks = 1 if c["dtype"] == "fp8" else es
    rows = T * (H + 2 * G) * D * es if kind != "sink" else T * (H + G) * D * es
    gates = T * H * D * es if kind == "talk" else 0
    mixing = 2 * T * H * H * D if kind == "talk" else 0
    # heads that mix need, per visible key, the weighted value sums of their own value head under
    # the mixed weights: scores, mixing of the weights, sums
    return {"bytes": rows + gates + T * H * D * es + 2 * distinct * G * D * ks
            + 2 * T * G * D * ks,
            "flops": seen * H * 4 * D + (seen * H * H * 2 - mixing if kind == "talk" else 0)
            + mixing}


# relative error that another correct implementation shows: about four times what the present
# one is measured to be off from 64 bits (bf16: 2 to 6e-3, where the softmax weights and the
# queries are rounded on the way; fp32: 0.1 to 2e-6)
def tolerance(case):
    if case["dtype"] == "f32":
        return {"rel": 2e-5, "max": 2e-3}
    # whole values: experts whose fp32 scores tie to the last bits may swap; e4m3 cache bytes
    # may round the other way
    rel = 2e-2 if case["kind"] in ("sink", "pooled") else 1.2e-2
    return {"rel": rel, "max": 0.2, "differ": 1e-3}


# ---------------------------------------------------------------------------- exact
def exact(case, seed):
    s = prepare(case, seed)
    return _EXACT[case["kind"]](case, s)


def _f(t):
    return t.double()


def _rms(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _half(x, cs):
    """x [T, heads, D] with its first cs.shape[1] entries turned, entry i with i + dims / 2."""
    n = cs.shape[1] // 2
    c, s = cs[:, None, :n], cs[:, None, n:]
    u, v = x[..., :n], x[..., n:2 * n]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * n:]], dim=-1)


def _pairs(x, cs):
    """x [T, heads, D] with neighbouring entries of its first cs.shape[1] turned."""
    n = cs.shape[1]
    c, s = cs[:, None, :n // 2], cs[:, None, n // 2:]
    u, v = x[..., 0:n:2], x[..., 1:n:2]
    y = torch.stack([u * c - v * s, v * c + u * s], dim=-1).flatten(-2)
    return torch.cat([y, x[..., n:]], dim=-1)


def _put(cache, st, rows):
    """Token-major cache [NB, G, PAGE, D] with `rows` [T, G, D] at the step's slots."""
    out = _f(cache).clone()
    out[st.slots // PAGE, :, st.slots % PAGE] = rows
    return out


def _put_groups(cache, st, rows):
    out = _f(cache).clone()
    at = st.slots % PAGE
    out[st.slots // PAGE, :, at // 8, :, at % 8] = rows
    return out


def _tokens(cache):
    """[NB, G, PAGE / 8, D, 8] as [NB, G, PAGE, D]."""
    return cache.transpose(3, 4).reshape(cache.shape[0], cache.shape[1], PAGE, cache.shape[3])


def _sequence(st, b, k, v):
    """Keys and values [G, length, D] of sequence b."""
    n = int(st.seq_lens[b])
    pages = st.tables[b, :-(-n // PAGE)].long()
    return [t[pages].transpose(0, 1).reshape(t.shape[1], -1, t.shape[3])[:, :n] for t in (k, v)]


def _attend(st, q, k, v, scale, c, sink=None, one=False, talk=None, extra=None):
    """q [T, H, D] over the sequences' keys: [T, H, Dv].  sink [H] or one: what the softmax's
    denominator has beside the keys; talk: the heads' mixing; extra: pooled blocks."""
    T, H, _ = q.shape
    G = k.shape[1]
    rep = H // G
    out = torch.zeros(T, H, v.shape[3], dtype=torch.float64, device=q.device)
    chunk, window, pool = c.get("chunk", 0), c.get("window", 0), c.get("pool", 0)
    for b, (p, n) in enumerate(st.shape):
        K, V = _sequence(st, b, k, v)
        j = torch.arange(K.shape[1], device=q.device)[None, :]
        r0 = int(st.q_start[b])
        if extra is not None:
            firsts = torch.arange(K.shape[1] // pool, device=q.device) * pool
            pages = st.tables[b][firsts // PAGE].long()
            KP, VP = (e[pages, :, (firsts % PAGE) // pool].transpose(0, 1) for e in extra)
        for a in range(0, n, 512):
            e = min(n, a + 512)
            i = torch.arange(p + a, p + e, device=q.device)[:, None]
            ok = j <= i
            if chunk:
                ok = ok & (j // chunk == i // chunk)
            if window:
                ok = ok & (j > i - window)
            rows = slice(r0 + a, r0 + e)
            kk, vv = K, V
            if extra is not None:
                ok = torch.cat([ok, (firsts + pool - 1)[None, :] <= i - window], dim=1)
                kk, vv = torch.cat([K, KP], 1), torch.cat([V, VP], 1)
            kk, vv = kk.repeat_interleave(rep, 0), vv.repeat_interleave(rep, 0)
            x = torch.matmul(q[rows].transpose(0, 1), kk.transpose(1, 2)) * scale
            x = x.masked_fill(~ok, float("-inf"))
            if sink is not None or one:
                z = sink.view(H, 1, 1) if sink is not None else torch.zeros(H, 1, 1).to(x)
                w = torch.softmax(torch.cat([x, z.expand(H, x.shape[1], 1)], 2), 2)[..., :-1]
            else:
                w = torch.softmax(x, 2)
            if talk is not None:
                w = torch.matmul(talk, w.flatten(1)).view_as(w)
            out[rows] = torch.matmul(w, vv).transpose(0, 1)
    return out


def _exact_gqa(c, s):
    H, G, D = c["heads"], c["kv_heads"], c["dim"]
    st = s["step"]
    x = _f(s["qkv"])
    q, k, v = (t.reshape(st.T, -1, D) for t in x.split([H * D, G * D, G * D], 1))
    if c["qk_norm"]:
        q, k = _rms(q) * _f(s["qw"]), _rms(k) * _f(s["kw"])
    cs = _f(s["cos_sin"])[st.positions]
    q, k = _half(q, cs), _half(k, cs)

    def values(t):
        return _f(t.view(torch.float8_e4m3fn).to(torch.bfloat16) if t.dtype == torch.uint8 else t)

    # the key cache keeps each 32-token chunk in matrix-operand order: token o at tile
    # (o >> 2) & 1, row (o >> 3) * 4 + (o & 3), dimensions in pieces of 32
    NB = st.num_blocks
    o = torch.arange(PAGE, device=DEV)
    kt = values(s["k"]).view(NB, G, 2, D // 32, 16, 32)[:, :, (o >> 2) & 1, :,
                                                         (o >> 3) * 4 + (o & 3), :]
    kt = kt.permute(1, 2, 0, 3, 4).reshape(NB, G, PAGE, D)     # indexed axis leads
    K, V = _put(kt, st, k), _put(_tokens(values(s["v"])), st, v)
    out = _attend(st, q, K, V, D ** -0.5, {})
    if st.prompt:
        return {"out": out, "k": None, "v": None}
    return {"out": out, "k": None, "v": None, "tail": None}


def _exact_sink(c, s):
    H, G, D = c["heads"], c["kv_heads"], c["dim"]
    st, x = s["step"], _f(s["proj"])
    q = x[:, :H * D] + _f(s["qb"])
    k = x[:, H * D:(H + G) * D] + _f(s["kb"])
    v = k.view(st.T, G, D)
    q, k = (_rms(q) * _f(s["qw"])).view(st.T, H, D), (_rms(k) * _f(s["kw"])).view(st.T, G, D)
    cs = _f(s["cos_sin"])[st.positions]
    q, k = _pairs(q, cs), _pairs(k, cs)
    K, V = _put(s["k"], st, k), _put_groups(s["v"], st, v)
    o = _attend(st, q, K, _tokens(V), D ** -0.5, c, sink=_f(s["sink"]))
    o = o * torch.sigmoid(x[:, (H + G) * D:])[:, :, None]
    return {"out": o.reshape(st.T, H * D), "k": K, "v": V}


def _exact_latent(c, s):
    H, R, r, D, Q = c["heads"], c["kv_rank"], c["rot"], c["dim"], c["q_rank"]
    st, x = s["step"], _f(s["proj"])
    cq = _rms(x[:, :Q]) * _f(s["qw"])
    lat = _rms(x[:, Q:Q + R]) * _f(s["kvw"])
    rot = _pairs(x[:, None, Q + R:], _f(s["cos_sin"])[st.positions])[:, 0]
    rows = _put(s["rows"][:, None], st, torch.cat([lat, rot], 1)[:, None])
    groups = _put_groups(s["groups"][:, None], st, lat[:, None])
    q = torch.cat([_f(s["q_lat"]).transpose(0, 1), _f(s["q"])[:, :, D:]], 2)
    o = _attend(st, q, rows, rows[..., :R], (D + r) ** -0.5, {})
    return {"out": o.transpose(0, 1), "cq": cq, "rows": rows[:, 0], "groups": groups[:, 0]}


def _exact_talk(c, s):
    H, G, D = c["heads"], c["kv_heads"], c["dim"]
    st, x = s["step"], _f(s["proj"])
    q, k, v, gate = x.split([H * D, G * D, G * D, H * D], 1)
    q, k, v = (_rms(t.reshape(st.T, -1, D)) for t in (q, k, v))
    K, V = _put(s["k"], st, k), _put_groups(s["v"], st, v)
    o = _attend(st, q, K, _tokens(V), D ** -0.5, {}, talk=_f(s["talk"])).reshape(st.T, H * D)
    return {"out": o * torch.sigmoid(gate), "k": K, "v": V}


def _exact_pooled(c, s):
    H, G, D, P = c["heads"], c["kv_heads"], c["dim"], c["pool"]
    st, x = s["step"], _f(s["proj"]) + _f(s["bias"])
    q, k, v = (t.reshape(st.T, -1, D) for t in x.split([H * D, G * D, G * D], 1))
    cs = _f(s["cos_sin"])[st.positions]
    q, k = _half(q, cs), _half(k, cs)
    K, V = _put(s["k"], st, k), _put_groups(s["v"], st, v)
    VT = _tokens(V)
    KP, VP = _f(s["kp"]).clone(), _f(s["vp"]).clone()
    for b, (p, n) in enumerate(st.shape):
        # the blocks whose last token came with this step
        first = torch.arange(p // P * P, (p + n) // P * P, P, device=DEV)
        if first.numel():
            kk, vv = _sequence(st, b, K, VT)
            page, idx = st.tables[b][first // PAGE].long(), (first % PAGE) // P
            for pool, t in ((KP, kk), (VP, vv)):
                a, e = int(first[0]), int(first[-1]) + P
                pool[page, :, idx] = t[:, a:e].view(G, -1, P, D).mean(2).transpose(0, 1)
    o = _attend(st, q, K, VT, D ** -0.5, c, one=True, extra=(KP, VP))
    return {"out": o.reshape(st.T, H * D), "k": K, "v": V, "kp": KP, "vp": VP}


def _sequences_padded(st, rows):
    """[B, longest, ...] of rows [T, ...], zeros behind a sequence's end."""
    n = max(n for _, n in st.shape)
    out = torch.zeros(st.B, n, *rows.shape[1:], dtype=rows.dtype, device=rows.device)
    for b, (_, m) in enumerate(st.shape):
        out[b, :m] = rows[int(st.q_start[b]):int(st.q_start[b]) + m]
    return out


def _sequences_joined(st, rows):
    return torch.cat([rows[b, :m] for b, (_, m) in enumerate(st.shape)])


def _exact_retention(c, s):
    H, D = c["heads"], c["dim"]
    st, x = s["step"], _f(s["proj"])
    q, k, v, gate = (t.reshape(st.T, H, D) for t in x.split([H * D] * 4, 1))
    cs = _f(s["cos_sin"])[st.positions]
    q, k = _half(q, cs), _half(k, cs) * D ** -0.5
    q, k, v = (_sequences_padded(st, t) for t in (q, k, v))
    decay = torch.exp2(_f(s["log2_decay"])).view(1, H, 1, 1)
    slots = st.seq_slot[st.q_start[:-1].long()].long()
    S = _f(s["state"])[slots].transpose(2, 3)                    # [B, H, D, V]
    fresh = torch.tensor([p == 0 for p, _ in st.shape], device=DEV)
    S = torch.where(fresh.view(-1, 1, 1, 1), torch.zeros_like(S), S)
    live = torch.tensor([n for _, n in st.shape], device=DEV)
    o = torch.zeros_like(v)
    for t in range(q.shape[1]):
        new = decay * S + k[:, t, :, :, None] * v[:, t, :, None, :]
        S = torch.where((t < live).view(-1, 1, 1, 1), new, S)
        o[:, t] = torch.matmul(q[:, t, :, None, :], S)[:, :, 0]
    o = _rms(_sequences_joined(st, o)) * torch.nn.functional.silu(gate)
    state = _f(s["state"]).clone()
    state[slots] = S.transpose(2, 3)
    return {"out": o.reshape(st.T, H * D), "state": state}


def _exact_ssm(c, s):
    H, V, N, G, taps = c["heads"], c["dim"], c["state"], c["groups"], c["taps"]
    st, p = s["step"], _f(s["proj"])
    inner, C = H * V, H * V + 2 * G * N
    slots = st.seq_slot[st.q_start[:-1].long()].long()
    fresh = torch.tensor([a == 0 for a, _ in st.shape], device=DEV).view(-1, 1, 1)
    old = _f(s["conv_state"])[slots]
    u = torch.cat([torch.where(fresh, torch.zeros_like(old), old),
                   _sequences_padded(st, p[:, inner:inner + C])], 1)
    n = u.shape[1] - (taps - 1)
    acc = _f(s["conv_b"]).view(1, 1, C)
    for j in range(taps):
        acc = acc + _f(s["conv_w"])[:, j] * u[:, j:j + n]
    xbc = torch.nn.functional.silu(acc)
    conv_state = _f(s["conv_state"]).clone()
    for b, (_, m) in enumerate(st.shape):
        conv_state[slots[b]] = u[b, m:m + taps - 1]
    x = xbc[..., :inner].reshape(st.B, n, H, V)
    Bm, Cm = (t.reshape(st.B, n, G, N).repeat_interleave(H // G, 2)
              for t in xbc[..., inner:].split([G * N, G * N], 2))
    dt = torch.nn.functional.softplus(p[:, inner + C:] + _f(s["dt_bias"]), threshold=1000.0)
    dt = _sequences_padded(st, dt)
    decay = torch.exp(-torch.exp(_f(s["a_log"])) * dt)
    S = _f(s["state"])[slots]
    S = torch.where(fresh[..., None], torch.zeros_like(S), S)
    live = torch.tensor([m for _, m in st.shape], device=DEV)
    y = torch.zeros_like(x)
    for t in range(n):
        new = decay[:, t, :, None, None] * S + \
            (dt[:, t, :, None] * Bm[:, t])[..., None] * x[:, t, :, None, :]
        S = torch.where((t < live).view(-1, 1, 1, 1), new, S)
        y[:, t] = torch.matmul(Cm[:, t, :, None, :], S)[:, :, 0]
    y = y + _f(s["d_skip"]).view(1, 1, H, 1) * x
    y = _sequences_joined(st, y).reshape(st.T, inner)
    state = _f(s["state"]).clone()
    state[slots] = S
    g = (y * torch.nn.functional.silu(p[:, :inner])).view(st.T, c["norm_groups"], -1)
    out = _rms(g).reshape(st.T, inner) * _f(s["gnorm"])
    return {"out": out, "y": y, "state": state, "conv_state": conv_state}


def _exact_experts(c, s):
    E, F, top = c["experts"], c["ff"], c["top"]
    h = _f(s["h"])
    val, ids = (h @ _f(s["router"]).T + _f(s["router_b"])).topk(top, 1)
    w = torch.softmax(val, 1)
    out = torch.zeros_like(h)
    for e in range(E):
        t, k = (ids == e).nonzero(as_tuple=True)
        gu = h[t] @ _f(s["w13"][e]).T
        y = (torch.nn.functional.silu(gu[:, :F]) * gu[:, F:]) @ _f(s["w2"][e]).T
        out.index_add_(0, t, y * w[t, k][:, None])
    return {"out": out, "ids": ids, "w": w}


_EXACT = {"gqa": _exact_gqa, "sink": _exact_sink, "latent": _exact_latent, "talk": _exact_talk,
          "pooled": _exact_pooled, "retention": _exact_retention, "ssm": _exact_ssm,
          "experts": _exact_experts}
