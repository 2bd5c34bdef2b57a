"""Timed cases: whole steps of the decoder stacks this package serves, through the model runner's two phases
(``execute_model``, ``sample_tokens``), as an engine loop calls them.

A case is one step of one stack:

  model   "talker"   the Qwen2.5-Omni-7B talker (28 layers), the stack the package exists for
          "moe"      the Qwen3-Omni talker with its sparse-MoE feed-forward (20 layers, 128 experts, 8 chosen)
          "pupopel"  channel-wise delta rule, biased sink attention beside decayed linear attention, routed experts (8 layer runs)
          "lifuzen"  state-space recurrence, attention whose values are its keys, all feed-forwards routed (8 layer runs)
  kind    "decode"   one token for each of ``batch`` requests whose contexts end at ``ctx`` tokens (``ragged``: the longest does, the
                     others are a quarter of it or more), outputs fetched one step behind, as the engine does;
          "prefill"  the rest of each prompt behind ``behind`` tokens that are in the cache already, tokens handed back at once
  sampled            temperature 0.9, top-k 40, top-p 0.8, repetition penalty 1.05 (what the talker stage runs with) instead of greedy

Sizes are those of the package's own configurations (``configs/*.json``), and of the stacks that ``bench.py`` measures.

Weights are random with one thing added that trained ones have and random ones lack: choices with a margin.  The first columns of
the stream carry the token (64 signs) and, where experts are routed, a level per expert; no sublayer adds to them, the output
head reads the signs and the routers the levels.  Tokens and experts are then the same at any rounding, different from token to
token and spread over all experts, and what is compared is arithmetic alone.
"""
import json
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PACKAGE = os.path.join(ROOT, "vllm-omni_amd")
if PACKAGE not in sys.path:
    sys.path.insert(0, PACKAGE)

BLOCK = 16          # tokens of a cache block
SIGNS = 64          # columns of the stream that carry the token
TAPS = 4
F64 = torch.float64


# ------------------------------------------------------------------------------------------------ the cases
def _case(model, kind, batch, ctx, behind=0, ragged=False, sampled=False, width=0):
    return {"model": model, "kind": kind, "batch": batch, "ctx": ctx, "behind": behind, "ragged": ragged, "sampled": sampled,
            "width": width}


def listed():
    return [
        # one caller, the start of an utterance: latency, every launch counts
        dict(_case("talker", "decode", 1, 150), name="talker decode 1 x 150"),
        # a small server's batch, contexts and batch of no particular size
        dict(_case("talker", "decode", 23, 1700, ragged=True, sampled=True), name="talker decode 23 ragged"),
        # the package's second named configuration
        dict(_case("talker", "decode", 64, 2048, sampled=True), name="talker decode 64 x 2048"),
        # the headline of bench.py: the largest
        dict(_case("talker", "decode", 256, 4096), name="talker decode 256 x 4096"),
        # a batch between them, many short contexts: the linears carry it
        dict(_case("talker", "decode", 120, 700, ragged=True), name="talker decode 120 ragged"),
        # several prompts of uneven length in one step
        dict(_case("talker", "prefill", 5, 1900, ragged=True), name="talker prefill 5 ragged"),
        # the Qwen3 talker at the batch its configuration names
        dict(_case("moe", "decode", 512, 4096), name="moe decode 512 x 4096"),
        # the last chunk of an 8k-token multimodal prompt
        dict(_case("moe", "prefill", 1, 8192, behind=6144), name="moe prefill chunk 2048"),
        # the text stacks, as bench.py runs them
        dict(_case("pupopel", "decode", 32, 4096, width=4096), name="pupopel decode 32 x 4096"),
        dict(_case("pupopel", "prefill", 1, 8192, width=4096), name="pupopel prefill 8192"),
        dict(_case("lifuzen", "decode", 200, 3001, ragged=True, width=4096), name="lifuzen decode 200 ragged"),
        dict(_case("lifuzen", "prefill", 4, 2048, ragged=True, width=4096), name="lifuzen prefill 4 ragged"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    model = rng.choice(["talker", "talker", "moe", "pupopel", "lifuzen"])
    width = rng.choice([2048, 4096]) if model in ("pupopel", "lifuzen") else 0
    sampled = rng.random() < 0.4
    if rng.random() < 0.55:
        batch = _log_uniform(rng, 1, 512 if model == "moe" else 256)
        ctx = _log_uniform(rng, 24, min(4096, 2_000_000 // batch))
        return _case(model, "decode", batch, ctx, ragged=batch > 1 and rng.random() < 0.6, sampled=sampled, width=width)
    batch = rng.choice([1, 1, 2, 3, 4, 7])
    ctx = _log_uniform(rng, 33, 8192 // batch)
    if model == "talker":
        ctx = min(ctx, 6000 // batch)
    behind = rng.randrange(ctx // 4, ctx - 16) if ctx > 600 and rng.random() < 0.3 else 0
    return _case(model, "prefill", batch, ctx, behind=behind, ragged=batch > 1 and rng.random() < 0.6, sampled=sampled, width=width)


def requests(case):
    """(tokens in the cache, tokens of this step) of every request"""
    n, ctx = case["batch"], case["ctx"]
    low = max(1 if case["kind"] == "decode" else case["behind"] + 1, ctx // 4)
    rng = random.Random(n * 100_003 + ctx)
    ends = [ctx] + [rng.randint(low, ctx) if case["ragged"] else ctx for _ in range(n - 1)]
    return [(e - 1, 1) if case["kind"] == "decode" else (case["behind"], e - case["behind"]) for e in ends]


# ------------------------------------------------------------------------------------------------ configurations
def config(case):
    """sizes of the stack as a plain dict"""
    m, w = case["model"], case["width"]
    if m in ("talker", "moe"):
        name = "qwen2_5_omni_talker" if m == "talker" else "qwen3_omni_talker"
        with open(os.path.join(PACKAGE, "vllm_omni_amd", "configs", name + ".json")) as f:
            c = json.load(f)
        # no column of the logits is masked: a value of -1e9 would hide every other
        c.update({k: None for k in c if k.startswith("tts_")})
        return c
    h, ff, dim = w // 128, 3 * w, 128
    c = {"architecture": m.capitalize(), "vocab": 15360, "width": w, "norm": {"eps": 1e-6}, "loop": {"start": 2, "stop": 4, "times": 2}}
    if m == "pupopel":
        delta = {"type": "channel_delta", "mixer": {"heads": h, "kv_heads": h // 2, "dim": dim, "vdim": dim, "conv": TAPS}}
        par = {"type": "parallel", "mixer": {
            "left": {"heads": h, "kv_heads": h // 4, "dim": dim, "vdim": dim, "scale": dim ** -0.5, "q_temp": {"coef": 0.1, "every": 8192}},
            "right": {"heads": h // 2, "dim": dim, "vdim": dim, "decay": [1 - 2.0 ** -(3 + 5 * i / h) for i in range(h // 2)]},
            "left_scale": 0.8, "right_scale": 0.5}}
        dense = {"kind": "dense", "ff": ff}
        moe = {"kind": "moe", "router": {"experts": 64, "top": 6}, "expert": {"ff": ff // 8}, "shared": {"ff": ff // 4}}
        c["layers"] = [dict(a, mlp=b) for a, b in ((delta, dense), (par, dense), (delta, moe), (par, moe), (delta, dense), (par, dense))]
        return c
    ssm = {"type": "mamba2", "mixer": {"heads": 2 * h, "groups": 8, "state": 128, "vdim": 64, "conv": TAPS, "norm_groups": 8}}
    attn = {"type": "attention", "mixer": {"heads": h, "kv_heads": h // 4, "dim": dim, "vdim": dim, "conv": TAPS, "scale": dim ** -0.5,
                                           "rot": {"base": 500000.0, "dims": dim // 2}}}
    moe = {"kind": "moe", "router": {"experts": 64, "top": 8}, "expert": {"ff": ff // 8}}
    return dict(c, residual_mult=0.5, logit_softcap=25.0, layers=[dict(a, mlp=moe) for a in (ssm, attn) * 3])


def runs(c):
    """(layer, pass of the loop that starts with it or None) in the order the layers run"""
    a, b, t = c["loop"]["start"], c["loop"]["stop"], c["loop"]["times"]
    looped = [(i, p if i == a else None) for p in range(t) for i in range(a, b)]
    return [(i, None) for i in range(a)] + looped + [(i, None) for i in range(b, len(c["layers"]))]


def num_experts(c):
    return c.get("num_experts", 0) if "layers" not in c else next(e["mlp"]["router"]["experts"] for e in c["layers"] if e["mlp"]["kind"] == "moe")


def kept(c):
    """columns of the stream that no sublayer adds to"""
    return SIGNS + num_experts(c)


# ------------------------------------------------------------------------------------------------ weights and caches, from the seed
class Draws:
    def __init__(self, seed, part):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed * 1009 + part)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
        return torch.empty(shape, dtype=dtype, device="cuda").normal_(mean, std, generator=self.gen)

    def matrix(self, n, k, gain=1.0, quiet=0):
        """[n, k] that keeps a row's scale; the first ``quiet`` outputs are zero"""
        w = self.normal(n, k, std=gain * k ** -0.5)
        w[:quiet] = 0
        return w

    def about(self, n, mean, std, quiet=0, quiet_value=0.0):
        w = self.normal(n, std=std, mean=mean)
        w[:quiet] = quiet_value
        return w

    def embedding(self, vocab, width, experts, scale, noise):
        e = self.normal(vocab, width, std=noise)
        e[:, :SIGNS] = (torch.rand(vocab, SIGNS, generator=self.gen, device="cuda") < 0.5).to(e.dtype) * (2 * scale) - scale
        if experts:
            order = torch.rand(vocab, experts, generator=self.gen, device="cuda").argsort(-1)
            e[:, SIGNS:SIGNS + experts] = (torch.linspace(-2, 2, experts, device="cuda") * scale)[order].to(e.dtype)
        return e

    def router(self, experts, width, gain):
        w = torch.zeros(experts, width, dtype=torch.bfloat16, device="cuda")
        at = torch.randperm(experts, generator=self.gen, device="cuda")
        w[torch.arange(experts, device="cuda"), SIGNS + at] = gain
        return w


def next_token_head(d, embed, keep):
    """the token behind token t is t + 1, whatever else the stream holds"""
    head = d.matrix(*embed.shape)
    head[:, :keep] = 0
    head[:, :SIGNS] = 0.8 * embed[:, :SIGNS].roll(1, 0)
    return head


def talker_outer(c, seed):
    d, w, keep = Draws(seed, 0), c["hidden_size"], kept(c)
    embed = d.embedding(c["vocab_size"], c["embedding_size"], num_experts(c), 1.0, 1.0)
    out = {"language_model.model.embed_tokens.weight": embed, "language_model.lm_head.weight": next_token_head(d, embed, keep),
           "language_model.model.norm.weight": d.about(w, 1.0, 0.1, keep, 1.0)}
    if c.get("input_projection", True):
        proj = d.matrix(w, c["embedding_size"], quiet=keep)
        proj[:keep, :keep] = torch.eye(keep, device="cuda", dtype=proj.dtype)
        out["thinker_to_talker_proj.weight"], out["thinker_to_talker_proj.bias"] = proj, d.about(w, 0.0, 0.1, keep)
    return out


def talker_layer(c, seed, i):
    d, w, keep = Draws(seed, 1 + i), c["hidden_size"], kept(c)
    nq, nkv, dim, inter = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"], c["intermediate_size"]
    rows = (nq + 2 * nkv) * dim
    out = {"self_attn.qkv_proj.weight": d.matrix(rows, w), "self_attn.o_proj.weight": d.matrix(w, nq * dim, quiet=keep),
           "input_layernorm.weight": d.about(w, 1.0, 0.1, keep, 1.0), "post_attention_layernorm.weight": d.about(w, 1.0, 0.1, keep, 1.0)}
    if c["attention_bias"]:
        out["self_attn.qkv_proj.bias"] = d.normal(rows, std=0.3)
    if c["qk_norm"]:
        out["self_attn.q_norm.weight"], out["self_attn.k_norm.weight"] = d.normal(dim, std=0.1, mean=1.0), d.normal(dim, std=0.1, mean=1.0)
    e = num_experts(c)
    if not e:
        return dict(out, **{"mlp.gate_up_proj.weight": d.matrix(2 * inter, w), "mlp.down_proj.weight": d.matrix(w, inter, 0.5, keep)})
    inter, shared = c["moe_intermediate_size"], c["shared_expert_intermediate_size"]
    down = d.matrix(e * w, inter).view(e, w, inter)
    down[:, :keep] = 0
    return dict(out, **{"mlp.gate.weight": d.router(e, w, 1.5), "mlp.experts.gate_up_proj": d.matrix(e * 2 * inter, w).view(e, 2 * inter, w),
                        "mlp.experts.down_proj": down, "mlp.shared_expert.gate_up_proj.weight": d.matrix(2 * shared, w),
                        "mlp.shared_expert.down_proj.weight": d.matrix(w, shared, 0.5, keep), "mlp.shared_expert_gate.weight": d.matrix(1, w)})


def text_outer(c, seed):
    d, w, v, keep = Draws(seed, 0), c["width"], c["vocab"], kept(c)
    if c["architecture"] == "Lifuzen":     # the table is the head as well: small values beside the signs
        out = {"embed": d.embedding(v, w, num_experts(c), 0.7, 0.02), "loop.step": d.normal(c["loop"]["times"], w, std=0.5)}
        out["loop.step"][:, :keep] = 0
    else:
        out = {"embed": d.embedding(v, w, num_experts(c), 1.0, 1.0), "loop.in": d.matrix(w, 2 * w, quiet=keep)}
        out["loop.in"][:keep, w:w + keep] = torch.eye(keep, device="cuda", dtype=torch.bfloat16)
        out["head"] = next_token_head(d, out["embed"], keep)
    return dict(out, **{"final.norm": d.about(w, 0.0, 0.1, keep)})


def text_layer(c, seed, i):
    d, w, keep = Draws(seed, 1 + i), c["width"], kept(c)
    entry = c["layers"][i]
    m, mlp = entry["mixer"], entry["mlp"]
    out = {"norm1": d.about(w, 0.0, 0.1, keep)}

    def glu(p, ff, gain):
        out.update({p + "gate": d.matrix(ff, w), p + "up": d.matrix(ff, w), p + "down": d.matrix(w, ff, gain, keep)})

    if entry["type"] == "channel_delta":
        kd, hd, hv, rank = m["kv_heads"] * m["dim"], m["heads"] * m["dim"], m["heads"] * m["vdim"], m["dim"]
        for n, ch in (("q", kd), ("k", kd), ("v", hv)):
            out["mix." + n], out[f"mix.{n}.conv"] = d.matrix(ch, w), d.normal(ch, m["conv"], std=0.6)
        for n, ch in (("a", hd), ("g", hv)):
            out[f"mix.{n}1"], out[f"mix.{n}2"] = d.matrix(rank, w), d.matrix(ch, rank)
        out.update({"mix.b": d.matrix(m["heads"], w), "mix.A_log": d.normal(m["heads"], std=0.9, mean=-1.5), "mix.dt_bias": d.normal(hd, std=0.8),
                    "mix.norm": d.normal(m["vdim"], std=0.2, mean=1.0), "mix.o": d.matrix(w, hv, 1.0, keep)})
    elif entry["type"] == "parallel":
        a, r = m["left"], m["right"]
        out.update({"mix.left.q": d.matrix(a["heads"] * a["dim"], w), "mix.left.k": d.matrix(a["kv_heads"] * a["dim"], w),
                    "mix.left.v": d.matrix(a["kv_heads"] * a["vdim"], w), "mix.left.q.norm": d.normal(a["dim"], std=0.2, mean=1.2),
                    "mix.left.k.norm": d.normal(a["dim"], std=0.2, mean=1.0), "mix.left.sink": d.normal(a["heads"], std=1.0, mean=0.5),
                    "mix.left.o": d.matrix(w, a["heads"] * a["vdim"], 1.0, keep)})
        hd, hv = r["heads"] * r["dim"], r["heads"] * r["vdim"]
        out.update({"mix.right." + n: d.matrix(ch, w) for n, ch in (("q", hd), ("k", hd), ("v", hv), ("g", hv))})
        out.update({"mix.right.norm": d.normal(hv, std=0.2, mean=1.0), "mix.right.o": d.matrix(w, hv, 1.0, keep)})
    elif entry["type"] == "mamba2":
        inner, ch = m["heads"] * m["vdim"], m["heads"] * m["vdim"] + 2 * m["groups"] * m["state"]
        out.update({"mix.in": d.matrix(inner + ch + m["heads"], w), "mix.conv": d.normal(ch, m["conv"], std=0.6), "mix.conv.b": d.normal(ch, std=0.3),
                    "mix.dt_bias": d.normal(m["heads"], std=1.0, mean=-2.0), "mix.A_log": d.normal(m["heads"], std=1.2, mean=-0.5),
                    "mix.D": d.normal(m["heads"], std=0.5, mean=1.0), "mix.norm": d.normal(inner, std=0.2, mean=1.0),
                    "mix.o": d.matrix(w, inner, 1.0, keep)})
    else:
        nq, nk = m["heads"] * m["dim"], m["kv_heads"] * m["dim"]
        out.update({"mix.q": d.matrix(nq, w), "mix.k": d.matrix(nk, w), "mix.q.conv": d.normal(nq, m["conv"], std=0.6),
                    "mix.k.conv": d.normal(nk, m["conv"], std=0.6), "mix.o": d.matrix(w, nq, 1.0, keep)})
    if mlp["kind"] == "dense":
        glu("mlp.", mlp["ff"], 0.7)
        return out
    gated = entry["type"] in ("channel_delta", "parallel")
    e, ff = mlp["router"]["experts"], mlp["expert"]["ff"]
    out["mlp.router"] = d.router(e, w, 1.5 if gated else 0.45)
    if gated:
        out["mlp.router.b"] = torch.zeros(e, device="cuda")
        glu("mlp.shared.", mlp["shared"]["ff"], 0.7)
    else:
        out["norm2"] = d.about(w, 0.0, 0.1, keep)
    for n, rows, cols in ((("gate", ff, w),) if gated else ()) + (("up", ff, w), ("down", w, ff)):
        block = d.matrix(e * rows, cols, 1.5).view(e, rows, cols)
        if n == "down":
            block[:, :keep] = 0
        out.update({f"mlp.e{j}.{n}": block[j] for j in range(e)})
    return out


def all_weights(case, c, seed):
    talker = case["model"] in ("talker", "moe")
    yield from (talker_outer if talker else text_outer)(c, seed).items()
    for i in range(c["num_hidden_layers"] if talker else len(c["layers"])):
        p = f"language_model.model.layers.{i}." if talker else f"l{i}."
        for name, t in (talker_layer if talker else text_layer)(c, seed, i).items():
            yield p + name, t


def cache_shapes(c):
    """[kv heads, dim] of every K/V cache, in the order of the layers"""
    if "layers" not in c:
        return [(c["num_key_value_heads"], c["head_dim"])] * c["num_hidden_layers"]
    kinds = [c["layers"][i] for i, _ in runs(c)]
    return [(a["kv_heads"], a["dim"]) for a in (e["mixer"].get("left", e["mixer"]) for e in kinds if e["type"] in ("parallel", "attention"))]


def cache_fill(seed, k, blocks, heads, dim):
    d = Draws(seed, 1000 + k)
    return d.normal(blocks, BLOCK, heads, dim), d.normal(blocks, BLOCK, heads, dim)


def state_shapes(c):
    """per layer run: (shape of a request's state, its type) of every state tensor"""
    out = []
    for e in [c["layers"][i] for i, _ in runs(c)] if "layers" in c else []:
        m = e["mixer"]
        if e["type"] == "channel_delta":
            ch = 2 * m["kv_heads"] * m["dim"] + m["heads"] * m["vdim"]
            out.append([((m["heads"], m["dim"], m["vdim"]), torch.float32), ((m["conv"], ch), torch.bfloat16)])
        elif e["type"] == "parallel":
            r = m["right"]
            out.append([((r["heads"], r["dim"], r["vdim"]), torch.float32)])
        elif e["type"] == "mamba2":
            ch = m["heads"] * m["vdim"] + 2 * m["groups"] * m["state"]
            out.append([((m["heads"], m["state"], m["vdim"]), torch.float32), ((m["conv"], ch), torch.bfloat16)])
        else:
            out.append([((m["conv"], (m["heads"] + m["kv_heads"]) * m["dim"]), torch.bfloat16)])
    return out


def state_fill(seed, r, j, n, shape, dtype):
    return Draws(seed, 2000 + 8 * r + j).normal(n, *shape, std=0.3 if dtype == torch.float32 else 1.0, dtype=dtype)


def block_tables(case, seed):
    """every request's blocks, scattered over the pool (block 0 belongs to nobody), and the pool's size"""
    need = [-(-(done + new) // BLOCK) for done, new in requests(case)]
    ids = np.random.default_rng(seed + 5).permutation(np.arange(1, sum(need) + 1))
    return [t.tolist() for t in np.split(ids, np.cumsum(need)[:-1])], sum(need) + 1


def tokens(case, c, seed):
    """every request's tokens up to the end of the step"""
    rng = np.random.default_rng(seed + 6)
    return [rng.integers(0, c.get("vocab") or c["vocab_size"], done + new) for done, new in requests(case)]


def prompt_rows(case, c, seed, embed):
    """what the stage in front hands over for every prompt: input rows"""
    d, keep = Draws(seed, 3000), kept(c)
    out = []
    for t in tokens(case, c, seed):
        rows = embed[torch.from_numpy(t).cuda()]
        noise = d.normal(*rows.shape, std=0.5)
        noise[:, :keep] = 0
        out.append(rows + noise)
    return out


# ------------------------------------------------------------------------------------------------ a step
@torch.inference_mode()
def prepare(case, seed):
    from vllm_omni_amd.model_runner import GPUARModelRunner
    from vllm_omni_amd.sched_output import NewRequestData, SamplingParams

    c, reqs = config(case), requests(case)
    talker = case["model"] in ("talker", "moe")
    if talker:
        from vllm_omni_amd.talker import TalkerConfig

        cfg = TalkerConfig(**{k: v for k, v in c.items() if k in TalkerConfig.__dataclass_fields__})
    else:
        from vllm_omni_amd.registry import config_from_hf

        cfg = config_from_hf(c)
    n, decode = len(reqs), case["kind"] == "decode"
    r = GPUARModelRunner(cfg, torch.device("cuda", 0), torch.bfloat16, max_num_reqs=n, max_model_len=case["ctx"] + BLOCK,
                         max_num_batched_tokens=sum(new for _, new in reqs), block_size=BLOCK, seed=0,
                         engine_output_type="latent" if talker else "text", copy_outputs=False)
    r.load_model()
    r.model.load_weights(all_weights(case, c, seed))
    tables, pool = block_tables(case, seed)
    r.initialize_kv_cache(pool)
    for k, ((heads, dim), (kc, vc)) in enumerate(zip(cache_shapes(c), r.kv_caches)):
        for dst, src in zip((kc, vc), cache_fill(seed, k, pool, heads, dim)):
            dst.copy_(src)
    states = []
    for k, specs in enumerate(state_shapes(c)):
        for j, (shape, dtype) in enumerate(specs):
            states.append(r.model.memory[k].states[j])
            states[-1][:n] = state_fill(seed, k, j, n, shape, dtype)
    params = SamplingParams(temperature=0.9, top_k=40, top_p=0.8, repetition_penalty=1.05) if case["sampled"] else SamplingParams()
    toks = tokens(case, c, seed)
    rows = prompt_rows(case, c, seed, r.model.language_model.model.embed_tokens) if talker and not decode else [None] * n
    new = [NewRequestData(f"r{i}", [] if x is not None else t.tolist(), params, (b,), done, prompt_embeds=x)
           for i, (t, b, (done, _), x) in enumerate(zip(toks, tables, reqs, rows))]
    if decode:
        r.capture_model([n])
    torch.cuda.synchronize()
    return {"runner": r, "new": new, "sched": [k for _, k in reqs], "done": [k for k, _ in reqs], "decode": decode, "passes": 0, "pending": None,
            "states": [s[:n] for s in states]}


def run(state):
    from vllm_omni_amd.sched_output import CachedRequestData, NewRequestData, SchedulerOutput

    r, n, p = state["runner"], len(state["new"]), state["passes"]
    state["passes"] += 1
    if state["decode"] and p:      # the same requests at the same place: bytes per step stay what they are
        ids = [x.req_id for x in state["new"]]
        so = SchedulerOutput(num_scheduled_tokens=dict(zip(ids, state["sched"])), total_num_scheduled_tokens=sum(state["sched"]),
                             scheduled_cached_reqs=CachedRequestData(req_ids=ids, new_token_ids=[], new_block_ids=[None] * n,
                                                                     num_computed_tokens=state["done"], num_output_tokens=[1] * n))
    else:                          # new requests; a prefill's of the pass before have finished
        new = [NewRequestData(f"{x.req_id}.{p}", list(x.prompt_token_ids), x.sampling_params, ([*x.block_ids[0]],), x.num_computed_tokens,
                              prompt_embeds=x.prompt_embeds) for x in state["new"]]
        gone = [x.req_id for x in state.get("live", [])]
        state["live"] = new
        if state["decode"]:
            state["new"] = new
        so = SchedulerOutput(scheduled_new_reqs=new, num_scheduled_tokens={x.req_id: k for x, k in zip(new, state["sched"])},
                             total_num_scheduled_tokens=sum(state["sched"]), finished_req_ids=gone)
    r.execute_model(so)
    st = r.execute_model_state
    out = {"logits": st.logits[:n], "hidden": st.hidden_states[:st.num_tokens], "tokens": st.sampled_ids[:n], "kv": [[x[1:] for x in kv] for kv in r.kv_caches],
           "states": state["states"]}
    if state["decode"]:            # outputs reach the host one step behind
        done = r.sample_tokens(async_output=True)
        if state["pending"] is not None:
            state["pending"].get_output()
        state["pending"] = done
    else:
        r.sample_tokens()
    return out


# ------------------------------------------------------------------------------------------------ what a step cannot do without
def _linear_sizes(case, c):
    """per layer run: (weights every row meets, weights of one expert, experts, chosen), and the output head's"""
    w = c.get("width") or c["hidden_size"]
    if "layers" not in c:
        d, e = c["head_dim"], num_experts(c)
        own = w * (2 * c["num_attention_heads"] + 2 * c["num_key_value_heads"]) * d
        own += 3 * w * (c["shared_expert_intermediate_size"] if e else c["intermediate_size"]) + w * e
        return [(own, 3 * w * c["moe_intermediate_size"] if e else 0, e, c.get("num_experts_per_tok", 0))] * c["num_hidden_layers"], w * c["vocab_size"]
    out = []
    for i, start in runs(c):
        m, mlp = c["layers"][i]["mixer"], c["layers"][i]["mlp"]
        own = 2 * w * w if start is not None and c["architecture"] == "Pupopel" else 0
        if "left" in m:
            a, r = m["left"], m["right"]
            own += w * (2 * a["heads"] + 2 * a["kv_heads"]) * a["dim"] + w * 5 * r["heads"] * r["dim"]
        elif "state" in m:
            inner = m["heads"] * m["vdim"]
            own += w * (3 * inner + 2 * m["groups"] * m["state"] + m["heads"])
        elif c["layers"][i]["type"] == "channel_delta":
            hd = m["heads"] * m["dim"]
            own += w * (2 * m["kv_heads"] * m["dim"] + 2 * hd + 2 * m["dim"] + m["heads"]) + 2 * hd * m["dim"]
        else:
            own += w * (2 * m["heads"] + m["kv_heads"]) * m["dim"]
        if mlp["kind"] == "dense":
            out.append((own + 3 * w * mlp["ff"], 0, 0, 0))
        else:
            shared = 3 * w * mlp["shared"]["ff"] if mlp.get("shared") else 0
            per = (3 if mlp.get("shared") else 2) * w * mlp["expert"]["ff"]
            out.append((own + shared + w * mlp["router"]["experts"], per, mlp["router"]["experts"], mlp["router"]["top"]))
    return out, w * c["vocab"]


def work(case):
    c, reqs = config(case), requests(case)
    rows = sum(new for _, new in reqs)
    layers, head = _linear_sizes(case, c)
    w = c.get("width") or c["hidden_size"]
    nbytes, flops = 2.0 * head, 2.0 * head * len(reqs)
    for own, expert, experts, top in layers:
        read = experts * (1 - (1 - top / experts) ** rows) if experts else 0
        nbytes += 2 * own + 2 * expert * read
        flops += 2.0 * rows * (own + expert * top)
    if c.get("input_projection", True) and "layers" not in c:
        nbytes, flops = nbytes + 2 * w * w, flops + 2.0 * rows * w * w
    pairs = sum(new * done + new * (new + 1) / 2 for done, new in reqs)
    heads = c.get("num_attention_heads") or w // 128
    for kvh, dim in cache_shapes(c):
        nbytes += 4.0 * kvh * dim * sum(done + new for done, new in reqs)
        flops += 4.0 * heads * dim * pairs
    for specs in state_shapes(c):
        for shape, dtype in specs:
            moved = 2 if case["kind"] == "decode" or case["behind"] else 1        # read and written; a prompt's start only writes
            nbytes += moved * len(reqs) * math.prod(shape) * (4 if dtype == torch.float32 else 2)
            if dtype == torch.float32:
                flops += 6.0 * rows * math.prod(shape)
    nbytes += 2.0 * rows * 2 * w + 2.0 * len(reqs) * (c.get("vocab") or c["vocab_size"])
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # bf16 activations, and in the talkers a bf16 stream through 20 to 28 layers: against 64 bits the talker's hidden rows were 0.019
    # off, the other stacks' outputs 0.004 to 0.012
    return {"rel": 0.03 if case["model"] == "talker" else 0.02, "max": 0.3}


# ------------------------------------------------------------------------------------------------ the same in 64 bits
def rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def silu(x):
    return x * torch.sigmoid(x)


def softplus(x):
    return torch.log1p(torch.exp(-x.abs())) + x.clamp(min=0)


def lin(x, w):
    return x @ w.to(F64).T


def rotated(x, pos, base, dims, pairs):
    """x [T, H, D]; neighbours (``pairs``) or halves of the first ``dims`` dimensions turn with the position"""
    a = pos.to(F64)[:, None, None] * base ** (-torch.arange(0, dims, 2, device=x.device, dtype=F64) / dims)
    u, v = (x[..., 0:dims:2], x[..., 1:dims:2]) if pairs else (x[..., :dims // 2], x[..., dims // 2:dims])
    u, v = u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()
    turned = torch.stack([u, v], -1).flatten(-2) if pairs else torch.cat([u, v], -1)
    return torch.cat([turned, x[..., dims:]], -1)


class Step:
    """the rows of a step, request after request, and what lies behind them in caches and states"""

    def __init__(self, case, c, seed):
        self.case, self.c, self.seed, self.reqs = case, c, seed, requests(case)
        self.tables, self.pool = block_tables(case, seed)
        self.tables = [torch.tensor(t, device="cuda") for t in self.tables]
        self.spans, at = [], 0
        for done, new in self.reqs:
            self.spans.append((at, at + new, done))
            at += new
        self.pos = torch.cat([torch.arange(done, done + new, device="cuda") for done, new in self.reqs])
        self.kv, self.states = [], []

    def attend(self, q, k, v, scale, slopes=None, sink=None):
        """q [T, H, D], k and v [T, G, D]: behind what the cache holds, causal; ``sink``: a score without a value"""
        kc, vc = cache_fill(self.seed, len(self.kv), self.pool, k.shape[1], k.shape[2])
        h, g, out = q.shape[1], k.shape[1], torch.empty_like(q)
        sink = torch.full((h,), -math.inf, device=q.device, dtype=F64) if sink is None else sink.to(F64)
        for (lo, hi, done), t in zip(self.spans, self.tables):
            keys, vals = (torch.cat([x[t].flatten(0, 1)[:done].to(F64), y[lo:hi]]) for x, y in ((kc, k), (vc, v)))
            dist = (torch.arange(done, done + hi - lo, device=q.device)[:, None] - torch.arange(done + hi - lo, device=q.device)[None]).to(F64)
            for j in range(g):
                of = slice(j * h // g, (j + 1) * h // g)
                s = (q[lo:hi, of].transpose(0, 1) @ keys[:, j].T) * scale
                if slopes is not None:
                    s -= slopes[of, None, None] * dist
                s.masked_fill_(dist < 0, -math.inf)
                top = torch.maximum(s.amax(-1), sink[of, None])[..., None]
                e = s.sub_(top).exp_()
                out[lo:hi, of] = ((e @ vals[:, j]) / (e.sum(-1, keepdim=True) + (sink[of, None, None] - top).exp())).transpose(0, 1)
        if self.case["kind"] == "prefill":
            for cache, rows in ((kc, k), (vc, v)):
                for (lo, hi, done), t in zip(self.spans, self.tables):
                    p = torch.arange(done, done + hi - lo, device=q.device)
                    cache[t[p // BLOCK], p % BLOCK] = rows[lo:hi].to(cache.dtype)
            self.kv.append([kc[1:].to(F64), vc[1:].to(F64)])
        else:
            self.kv.append([None, None])
        return out.flatten(1)

    def state(self, run, j):
        shape, dtype = state_shapes(self.c)[run][j]
        return state_fill(self.seed, run, j, len(self.reqs), shape, dtype).to(F64)

    def filtered(self, x, w, run, j):
        """each channel's taps over time; the rows in front come from the ring, where position p lies in place p % taps"""
        ring, taps, out, w = self.state(run, j), w.shape[1], torch.empty_like(x), w.to(F64)
        for i, (lo, hi, done) in enumerate(self.spans):
            past = torch.stack([ring[i, p % taps] if p >= 0 else torch.zeros_like(x[0]) for p in range(done - taps + 1, done)])
            full = torch.cat([past, x[lo:hi]])
            out[lo:hi] = sum(w[:, b] * full[b:b + hi - lo] for b in range(taps))
            for p in range(max(done, done + hi - lo - taps), done + hi - lo):
                ring[i, p % taps] = x[lo + p - done]
        self.states.append(ring)
        return out

    def recurrence(self, run, j, token):
        """``token(t, S)``: the state [N, ...] after rows ``t`` of N requests and what they read from it; one-token rows of all requests at once"""
        S = self.state(run, j)
        one = all(new == 1 for _, new in self.reqs)
        S *= torch.tensor([done > 0 for done, _ in self.reqs], device=S.device).view(-1, *[1] * (S.dim() - 1))
        if one:
            S, out = token(slice(0, len(self.reqs)), S)
            out = [out]
        else:
            out = []
            for i, (lo, hi, _) in enumerate(self.spans):
                s = S[i:i + 1]
                for t in range(lo, hi):
                    s, y = token(slice(t, t + 1), s)
                    out.append(y)
                S[i:i + 1] = s
        return S, torch.cat(out)


def exact_experts(h, score, top, expert, soft):
    """sum over each row's ``top`` experts; ``soft``: weights as a function of the chosen scores, None where ``expert`` takes them itself"""
    val, idx = score.sort(dim=-1, descending=True, stable=True)
    val, idx = val[:, :top], idx[:, :top]
    weight, y = (val if soft is None else soft(val)), torch.zeros_like(h)
    for e in range(score.shape[1]):
        t, j = (idx == e).nonzero(as_tuple=True)
        if t.numel():
            p = weight[t, j][:, None]
            y.index_add_(0, t, expert(e, h[t] * p) if soft is None else p * expert(e, h[t]))
    return y


def exact_talker(case, c, seed, step):
    outer, eps = talker_outer(c, seed), c["rms_norm_eps"]
    embed = outer["language_model.model.embed_tokens.weight"]
    if case["kind"] == "decode":
        x = embed[torch.tensor([int(t[-1]) for t in tokens(case, c, seed)], device="cuda")]
    else:
        x = torch.cat([r[done:] for r, (done, _) in zip(prompt_rows(case, c, seed, embed), step.reqs)])
    x = x.to(F64)
    if c.get("input_projection", True):
        x = lin(x, outer["thinker_to_talker_proj.weight"]) + outer["thinker_to_talker_proj.bias"].to(F64)
    nq, nkv, d, e = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"], num_experts(c)
    for i in range(c["num_hidden_layers"]):
        W = talker_layer(c, seed, i)
        h = rms(x, eps) * W["input_layernorm.weight"].to(F64)
        y = lin(h, W["self_attn.qkv_proj.weight"]) + (W["self_attn.qkv_proj.bias"].to(F64) if c["attention_bias"] else 0)
        q, k, v = (t.reshape(len(x), -1, d) for t in y.split([nq * d, nkv * d, nkv * d], -1))
        if c["qk_norm"]:
            q, k = rms(q, eps) * W["self_attn.q_norm.weight"].to(F64), rms(k, eps) * W["self_attn.k_norm.weight"].to(F64)
        q, k = (rotated(t, step.pos, c["rope_theta"], d, False) for t in (q, k))
        x = x + lin(step.attend(q, k, v, d ** -0.5), W["self_attn.o_proj.weight"])
        h = rms(x, eps) * W["post_attention_layernorm.weight"].to(F64)

        def glu(h, gate_up, down):
            g, u = lin(h, gate_up).chunk(2, -1)
            return lin(silu(g) * u, down)

        if not e:
            x = x + glu(h, W["mlp.gate_up_proj.weight"], W["mlp.down_proj.weight"])
            continue
        y = exact_experts(h, torch.softmax(lin(h, W["mlp.gate.weight"]), -1), c["num_experts_per_tok"],
                          lambda j, r: glu(r, W["mlp.experts.gate_up_proj"][j], W["mlp.experts.down_proj"][j]), lambda v: v)
        x = x + y + torch.sigmoid(lin(h, W["mlp.shared_expert_gate.weight"])) * glu(h, W["mlp.shared_expert.gate_up_proj.weight"],
                                                                                   W["mlp.shared_expert.down_proj.weight"])
    hidden = rms(x, eps) * outer["language_model.model.norm.weight"].to(F64)
    return hidden, outer["language_model.lm_head.weight"]


def exact_channel_delta(h, W, m, eps, step, run):
    H, K, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    x = torch.cat([lin(h, W["mix." + n]) for n in "qkv"], -1)
    state = len(step.states)
    x = silu(step.filtered(x, torch.cat([W[f"mix.{n}.conv"] for n in "qkv"]), run, 1))
    q, k, v = x.split([K * D, K * D, H * V], -1)
    q, k = (t.view(-1, K, D) * torch.rsqrt((t.view(-1, K, D) ** 2).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
    q, k = (t.repeat_interleave(H // K, 1) for t in (q / math.sqrt(D), k))
    low = lin(lin(h, W["mix.a1"]), W["mix.a2"]) + W["mix.dt_bias"].to(F64)
    keep = torch.exp(-W["mix.A_log"].to(F64).exp()[:, None] * softplus(low).view(-1, H, D))
    beta, v = torch.sigmoid(lin(h, W["mix.b"])), v.view(-1, H, V)

    def token(t, S):
        S = S * keep[t, :, :, None]
        u = beta[t, :, None] * (v[t] - (k[t, :, :, None] * S).sum(2))
        S = S + k[t, :, :, None] * u[:, :, None]
        return S, (q[t, :, :, None] * S).sum(2)

    S, o = step.recurrence(run, 0, token)
    step.states.insert(state, S)
    gate = torch.sigmoid(lin(lin(h, W["mix.g1"]), W["mix.g2"])).view(-1, H, V)
    return lin((rms(o, eps) * W["mix.norm"].to(F64) * gate).flatten(1), W["mix.o"])


def exact_parallel(h, W, m, eps, step, run):
    a, r = m["left"], m["right"]
    H, G, D = a["heads"], a["kv_heads"], a["dim"]
    q, k, v = (lin(h, W["mix.left." + n]).view(len(h), -1, D) for n in "qkv")
    q, k = rms(q, eps) * W["mix.left.q.norm"].to(F64), rms(k, eps) * W["mix.left.k.norm"].to(F64)
    temp = 1 + a["q_temp"]["coef"] * torch.log(torch.div(step.pos + 1, a["q_temp"]["every"], rounding_mode="floor").to(F64) + 1)
    slopes = 2.0 ** (-8 * torch.arange(1, H + 1, device=h.device, dtype=F64) / H)
    left = lin(step.attend(q * temp[:, None, None], k, v, a["scale"], slopes, W["mix.left.sink"]), W["mix.left.o"])
    H, D = r["heads"], r["dim"]
    q, k, v = (silu(lin(h, W["mix.right." + n])).view(len(h), H, -1) for n in "qkv")
    decay = torch.tensor(r["decay"], device=h.device, dtype=F64)[:, None, None]

    def token(t, S):
        S = S * decay + k[t, :, :, None] * v[t, :, None]
        return S, (q[t, :, :, None] * S).sum(2)

    S, o = step.recurrence(run, 0, token)
    step.states.append(S)
    right = lin(rms(o.flatten(1), eps) * W["mix.right.norm"].to(F64) * torch.sigmoid(lin(h, W["mix.right.g"])), W["mix.right.o"])
    return m["left_scale"] * left + m["right_scale"] * right


def exact_state_space(h, W, m, eps, step, run):
    H, V, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
    z, x, raw = lin(h, W["mix.in"]).split([H * V, H * V + 2 * G * N, H], -1)
    state = len(step.states)
    x = silu(step.filtered(x.contiguous(), W["mix.conv"], run, 1) + W["mix.conv.b"].to(F64))
    x, B, C = x.split([H * V, G * N, G * N], -1)
    x, B, C = x.reshape(-1, H, V), *(t.reshape(-1, G, N).repeat_interleave(H // G, 1) for t in (B, C))
    dt = softplus(raw + W["mix.dt_bias"].to(F64))
    keep, skip = torch.exp(-W["mix.A_log"].to(F64).exp() * dt), W["mix.D"].to(F64)[:, None]

    def token(t, S):
        S = S * keep[t, :, None, None] + (dt[t, :, None] * B[t])[..., None] * x[t, :, None]
        return S, (C[t, :, :, None] * S).sum(2) + skip * x[t]

    S, y = step.recurrence(run, 0, token)
    step.states.insert(state, S)
    g = y.flatten(1) * silu(z)
    return lin(rms(g.view(len(g), m["norm_groups"], -1), eps).flatten(1) * W["mix.norm"].to(F64), W["mix.o"])


def exact_key_value(h, W, m, eps, step, run):
    H, G, D = m["heads"], m["kv_heads"], m["dim"]
    x = torch.cat([lin(h, W["mix.q"]), lin(h, W["mix.k"])], -1)
    x = step.filtered(x, torch.cat([W["mix.q.conv"], W["mix.k.conv"]]), run, 0).view(len(h), H + G, D)
    q, k = (rms(rotated(t, step.pos, m["rot"]["base"], m["rot"]["dims"], True), eps) for t in (x[:, :H], x[:, H:]))
    return lin(step.attend(q, k, x[:, H:].contiguous(), m["scale"], sink=torch.zeros(H, device=h.device)), W["mix.o"])


MIXERS = {"channel_delta": exact_channel_delta, "parallel": exact_parallel, "mamba2": exact_state_space, "attention": exact_key_value}


def exact_text(case, c, seed, step):
    outer, eps, lifuzen = text_outer(c, seed), c["norm"]["eps"], c["architecture"] == "Lifuzen"
    ids = torch.cat([torch.from_numpy(t[done:]) for t, (done, _) in zip(tokens(case, c, seed), step.reqs)]).cuda()
    first = x = outer["embed"][ids].to(F64)

    def normed(x, w):
        return rms(x, eps) * (1 + w.to(F64))

    for r, (i, start) in enumerate(runs(c)):
        W, entry = text_layer(c, seed, i), c["layers"][i]
        if start is not None:
            x = x + (first if start else 0) + outer["loop.step"][start].to(F64) if lifuzen else lin(torch.cat([x, first], -1), outer["loop.in"])
        h, mlp = normed(x, W["norm1"]), entry["mlp"]
        y = MIXERS[entry["type"]](h, W, entry["mixer"], eps, step, r)
        if lifuzen:
            h = normed(x, W["norm2"])
            y = y + exact_experts(h, torch.sigmoid(lin(h, W["mlp.router"])), mlp["router"]["top"],
                                  lambda e, t: lin(lin(t, W[f"mlp.e{e}.up"]).clamp(min=0) ** 2, W[f"mlp.e{e}.down"]), None)
            x = x + c["residual_mult"] * y
            continue

        def glu(p, t, act):
            return lin(act(lin(t, W[p + "gate"])) * lin(t, W[p + "up"]), W[p + "down"])

        if mlp["kind"] == "dense":
            y = y + glu("mlp.", h, lambda t: torch.nn.functional.gelu(t, approximate="tanh"))
        else:
            y = y + glu("mlp.shared.", h, silu)
            y = y + exact_experts(h, lin(h, W["mlp.router"]), mlp["router"]["top"], lambda e, t: glu(f"mlp.e{e}.", t, silu), lambda v: torch.softmax(v, -1))
        x = x + y
    return normed(x, outer["final.norm"]), outer["embed" if lifuzen else "head"]


@torch.inference_mode()
def exact(case, seed):
    c = config(case)
    step = Step(case, c, seed)
    hidden, head = (exact_talker if case["model"] in ("talker", "moe") else exact_text)(case, c, seed, step)
    last = torch.tensor([hi - 1 for _, hi, _ in step.spans], device="cuda")
    logits = lin(hidden[last], head)
    if c.get("logit_softcap"):
        logits = c["logit_softcap"] * torch.tanh(logits / c["logit_softcap"])
    return {"logits": logits, "hidden": hidden, "tokens": None, "kv": step.kv, "states": step.states}
