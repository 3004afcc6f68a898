"""Performance cases of the serving path: what a user of the package has it do, step by step, through ModelRunner and the
layers it is made of.

Most cases are ONE forward step of a model over a batch that a scheduler would hand it (a ModelWorkerBatch: requests
with their slots and cached tokens), as a worker runs it: ForwardBatch.init_new -> ModelRunner.forward -> sample.

  decode   every request adds one token to the tokens it has cached (a captured graph where the family allows it)
  prefill  whole prompts, nothing cached
  extend   new tokens on top of a cached prefix: a chunk of a long prompt, or a prompt whose head the radix tree holds

Two cases are parts of such a step that models outside the listed ones share: a grouped mixture of experts behind its
router, and the non-greedy sampler.

Request lengths are ragged: request i of a case has between (1 - spread) and 1 times the case's length, by a rule that
depends on the case alone.  Inputs (weights, tokens, cached rows) come from the seed alone.  `exact` restates every path in
plain float64 torch on whole sequences, with none of the package's arithmetic."""
import math
import random

import torch

DEV = "cuda"


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # one user alone with a small model: a step is nothing but launches and latency
        dict(name="llama1b decode 1", kind="step", model="llama-3.2-1b", phase="decode", requests=1, length=131, spread=0.0),
        # the headline workload, as continuous batching meets it: 64 requests between 1024 and 1152 tokens
        dict(name="llama8b decode 64", kind="step", model="llama-3-8b", phase="decode", requests=64, length=1152, spread=0.11),
        # fp8 weights and fp8 cache, few long conversations of unequal length
        dict(name="llama8b fp8 decode 16", kind="step", model="llama-3-8b", phase="decode", requests=16, length=4000, spread=0.75, fp8=True),
        # a batch of fresh prompts that share one prefill
        dict(name="llama8b prefill", kind="step", model="llama-3-8b", phase="prefill", requests=5, length=1100, spread=0.5),
        # chunks of longer prompts, or prompts whose head is cached: new tokens over a prefix three times as long
        dict(name="llama8b extend", kind="step", model="llama-3-8b", phase="extend", requests=4, length=515, spread=0.3, prefix=1999),
        # latent attention (DeepSeek's dense layers): long contexts in a compressed cache
        dict(name="deepseek decode 64", kind="step", model="deepseek-w4096", phase="decode", requests=64, length=4096, spread=0.1),
        dict(name="deepseek prefill", kind="step", model="deepseek-w4096", phase="prefill", requests=4, length=2048, spread=0.2),
        # window + block attention, a state-space recurrence and a delta rule: prompts through the recurrent layers
        dict(name="fudonex prefill", kind="step", model="fudonex-fx2048", phase="prefill", requests=4, length=2048, spread=0.2),
        # latent attention over every earlier token on an fp32 stream
        dict(name="silatar prefill", kind="step", model="silatar-si2048", phase="prefill", requests=4, length=2048, spread=0.2),
        # capped and gated attention beside difference attention, one token at a time
        dict(name="lomazen decode 64", kind="step", model="lomazen-lz2048", phase="decode", requests=64, length=1024, spread=0.2),
        # the mixture feed-forward of a prefill: 32 experts of which a token takes 4
        dict(name="moe 3000", kind="moe", size="vz2048", tokens=3000),
        # a batch that does not decode greedily, over a large vocabulary
        dict(name="sample 64", kind="sample", requests=64, vocab=128256, top_k=50, top_p=0.9, min_p=0.0),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode"] * 5 + ["prefill"] * 5 + ["extend"] * 2 + ["moe"] * 2 + ["sample"])
    if kind == "moe":
        return dict(kind="moe", size=rng.choice(["vz2048", "vz4096"]), tokens=_log_uniform(rng, 16, 5000))
    if kind == "sample":
        return dict(kind="sample", requests=_log_uniform(rng, 1, 64), vocab=rng.choice([32768, 128256, 129280]), top_k=_log_uniform(rng, 2, 1000),
                    top_p=round(rng.uniform(0.5, 1.0), 3), min_p=rng.choice([0.0, 0.0, 0.05]))
    spread = round(rng.uniform(0.0, 0.6), 2)
    if kind == "extend":
        case = dict(kind="step", model=rng.choice(["llama-3.2-1b", "llama-3-8b"]), phase="extend", requests=rng.randint(1, 6),
                    length=_log_uniform(rng, 65, 500), spread=spread, prefix=_log_uniform(rng, 100, 3000))
    else:
        model = rng.choice(["llama-3.2-1b", "llama-3-8b", "llama-3-8b", "deepseek-w4096", "fudonex-fx2048", "silatar-si2048", "lomazen-lz2048"])
        if kind == "decode":
            n = _log_uniform(rng, 1, 64)
            case = dict(kind="step", model=model, phase="decode", requests=n, length=_log_uniform(rng, 64, min(4096, 66000 // n)), spread=spread)
        else:
            n = rng.randint(1, 6)
            most = {"llama-3-8b": 4000, "llama-3.2-1b": 6000}.get(model, 8000) // n
            case = dict(kind="step", model=model, phase="prefill", requests=n, length=_log_uniform(rng, 70, min(4000, most)), spread=spread)
    if case["model"] == "llama-3-8b" and rng.random() < 0.4:
        case["fp8"] = True
    return case


def _lengths(case):
    """(tokens cached, new tokens) of every request."""
    r = random.Random("%s %s %d %d" % (case["model"], case["phase"], case["requests"], case["length"]))
    whole = [max(2, int(case["length"] * (1.0 - case["spread"] * r.random()))) for _ in range(case["requests"])]
    if case["phase"] == "decode":
        return [n - 1 for n in whole], [1] * len(whole)
    if case["phase"] == "prefill":
        return [0] * len(whole), whole
    return [max(1, int(case["prefix"] * (1.0 - case["spread"] * r.random()))) for _ in whole], whole


# ------------------------------------------------------------------------------------------------ configurations and weights
def _family(case):
    return case["model"].split("-")[0]


def _config(case):
    from sglang_custom_amd import bench_designs as bd
    from sglang_custom_amd.model_loader.synthetic import hf_config_dict

    fam, size = _family(case), case["model"].split("-")[-1]
    if fam == "llama":
        return hf_config_dict(case["model"], "bfloat16")
    if fam == "deepseek":
        return bd.deepseek_config(bd.SIZES[size], "bfloat16")
    if fam == "fudonex":
        return bd.fudonex_config(bd.FUDONEX_SIZES[size])
    if fam == "silatar":
        return bd.silatar_config(bd.SILATAR_SIZES[size], "latent")
    return bd.lomazen_config(bd.LOMAZEN_SIZES[size], "dense")


def _transformer_shapes(c):
    """Llama's and the dense DeepSeek layers' checkpoint tensors."""
    D, H, ff, V = c["hidden_size"], c["num_attention_heads"], c["intermediate_size"], c["vocab_size"]
    s = {"model.embed_tokens.weight": (V, D), "model.norm.weight": (D,)}
    if not c["tie_word_embeddings"]:
        s["lm_head.weight"] = (V, D)
    for i in range(c["num_hidden_layers"]):
        p, a = "model.layers.%d." % i, "model.layers.%d.self_attn." % i
        s.update({p + "input_layernorm.weight": (D,), p + "post_attention_layernorm.weight": (D,), p + "mlp.gate_proj.weight": (ff, D),
                  p + "mlp.up_proj.weight": (ff, D), p + "mlp.down_proj.weight": (D, ff)})
        if "kv_lora_rank" in c:
            qr, kr, dn, dr, dv = c["q_lora_rank"], c["kv_lora_rank"], c["qk_nope_head_dim"], c["qk_rope_head_dim"], c["v_head_dim"]
            s.update({a + "q_a_proj.weight": (qr, D), a + "q_a_layernorm.weight": (qr,), a + "q_b_proj.weight": (H * (dn + dr), qr),
                      a + "kv_a_proj_with_mqa.weight": (kr + dr, D), a + "kv_a_layernorm.weight": (kr,),
                      a + "kv_b_proj.weight": (H * (dn + dv), kr), a + "o_proj.weight": (D, H * dv)})
        else:
            d, G = c["head_dim"], c["num_key_value_heads"]
            s.update({a + "q_proj.weight": (H * d, D), a + "k_proj.weight": (G * d, D), a + "v_proj.weight": (G * d, D), a + "o_proj.weight": (D, H * d)})
    return s


def _design_shapes(c):
    """Checkpoint tensors of the designs whose configuration lists its layers (Fudonex, Silatar, Lomazen)."""
    D, V, arch = c["width"], c["vocab"], c["architecture"]
    s = {"embed": (V, D), "final.norm": (D,)}
    if arch == "Silatar":
        s["head"] = (V, D)
    for i, spec in enumerate(c["layers"]):
        p, m, ff = "l%d." % i, spec["mixer"], spec["mlp"]["ff"]
        x, H = p + "mix.", spec["mixer"]["heads"]
        s.update({p + "norm1": (D,), p + "norm2": (D,), p + "mlp.up": (ff, D), p + "mlp.down": (D, ff)})
        if arch != "Silatar":
            s[p + "mlp.gate"] = (ff, D)
        s.update({p + "ls1": (D,), p + "ls2": (D,)} if arch == "Fudonex" else {p + "norm1b": (D,), p + "norm2b": (D,)})
        t = spec["type"]
        if t == "latent_attention":
            s.update({x + "q": (H * (m["dim"] + m["rot_dim"]), D), x + "dkv": (m["kv_rank"] + m["rot_dim"], D), x + "dkv.norm": (m["kv_rank"],),
                      x + "uk": (H * m["dim"], m["kv_rank"]), x + "uv": (H * m["vdim"], m["kv_rank"])})
        elif t == "mamba2":
            inner, gn = H * m["vdim"], m["groups"] * m["state"]
            s.update({x + "in": (2 * inner + 2 * gn + H, D), x + "conv": (inner + 2 * gn, m["conv"]), x + "conv.b": (inner + 2 * gn,),
                      x + "dt_bias": (H,), x + "A_log": (H,), x + "D": (H,), x + "norm": (inner,)})
        elif t == "delta":
            G, d, dv = m["kv_heads"], m["dim"], m["vdim"]
            s.update({x + "q": (G * d, D), x + "k": (G * d, D), x + "v": (H * dv, D), x + "g": (H * dv, D), x + "q.conv": (G * d, m["conv"]),
                      x + "k.conv": (G * d, m["conv"]), x + "v.conv": (H * dv, m["conv"]), x + "b": (H, D), x + "a": (H, D), x + "dt_bias": (H,),
                      x + "A_log": (H,), x + "norm": (dv,)})
        elif arch == "Fudonex":
            G, d, dv = m["kv_heads"], m["dim"], m["vdim"]
            s.update({x + "q": (H * d, D), x + "q.b": (H * d,), x + "q.norm": (d,), x + "g": (H, D), x + "sink": (H,)})
            if m.get("kv_from") is None:
                s.update({x + "k": (G * d, D), x + "k.b": (G * d,), x + "k.norm": (d,), x + "v": (G * dv, D), x + "v.b": (G * dv,)})
        else:
            G, d, dv, n = m["kv_heads"], m["dim"], m["vdim"], 2 if t == "attention_2" else 1
            s.update({x + "q": (n * H * d, D), x + "k": (n * G * d, D), x + "v": (G * dv, D), x + "g": (H if n == 2 else H * dv, D)})
            if n == 2:
                s.update({x + k: (d,) for k in ("lq1", "lk1", "lq2", "lk2")})
        s[x + "o"] = (D, H * m["vdim"])
    return s


def _weights(case, cfg, seed):
    """bf16 checkpoint of the configuration: projections N(0, 1 / fan-in), those that write a pre-norm stream smaller by the
    square root of how many do, norms around one (or zero, where they are stored so)."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    pre = _family(case) in ("llama", "deepseek")
    zero = cfg.get("architecture") == "Fudonex"
    out = {}
    for name, shape in (_transformer_shapes(cfg) if pre else _design_shapes(cfg)).items():
        w = torch.randn(shape, generator=g, device=DEV, dtype=torch.bfloat16)
        last = name.split(".")[-1]
        if len(shape) == 1 and (last.startswith("lq") or last.startswith("lk") or last in ("b", "dt_bias", "A_log", "sink")):
            w.mul_(0.1)
        elif len(shape) == 1 and zero and (last in ("norm1", "norm2") or name == "final.norm"):
            w.mul_(0.1)
        elif len(shape) == 1:
            w.mul_(0.1).add_(1.0)
        elif "embed" in name:
            pass
        else:
            std = shape[-1] ** -0.5
            if pre and ("o_proj" in name or "down_proj" in name):
                std *= (2 * cfg["num_hidden_layers"]) ** -0.5
            w.mul_(std)
        out[name] = w
    return out


def _tokens(case, vocab, seed):
    """Every request's tokens, cached ones first."""
    r = random.Random(seed)
    return [r.choices(range(vocab), k=a + b) for a, b in zip(*_lengths(case))]


def _cached(case, cfg, layer, seed):
    """What the cache holds of the cached tokens (all requests', in order) in one layer: normal rows."""
    g = torch.Generator(device=DEV).manual_seed(seed * 131 + layer)
    n, fam = sum(_lengths(case)[0]), _family(case)

    def rows(*shape):
        return torch.randn((n,) + shape, generator=g, device=DEV, dtype=torch.bfloat16)

    if fam == "llama":
        return rows(cfg["num_key_value_heads"], cfg["head_dim"]), rows(cfg["num_key_value_heads"], cfg["head_dim"])
    if fam == "deepseek":
        return (rows(cfg["kv_lora_rank"] + cfg["qk_rope_head_dim"]),)
    m = cfg["layers"][layer]["mixer"]
    if fam == "silatar":
        return (rows(m["kv_rank"] + m["rot_dim"]),)
    return rows(m["kv_heads"], m["dim"] * (2 if cfg["layers"][layer]["type"] == "attention_2" else 1)), rows(m["kv_heads"], m["vdim"])


def _shown(case, cfg):
    """The layers whose new cache rows are returned beside the logits."""
    n = cfg.get("num_hidden_layers") or len(cfg["layers"])
    return [0] if _family(case) == "fudonex" or case.get("fp8") else sorted({0, n // 2, n - 1})


# ------------------------------------------------------------------------------------------------ what a program has in hand
class _Step:
    """A model runner, and the batch that the scheduler gives it."""


def prepare(case, seed):
    if case["kind"] == "moe":
        return _prepare_moe(case, seed)
    if case["kind"] == "sample":
        return _prepare_sample(case, seed)
    from sglang_custom_amd.configs.model_config import ModelConfig
    from sglang_custom_amd.managers.schedule_batch import Req, ScheduleBatch
    from sglang_custom_amd.model_executor.forward_batch_info import ForwardBatch
    from sglang_custom_amd.model_executor.hip_graph_runner import get_batch_sizes_to_capture
    from sglang_custom_amd.model_executor.model_runner import ModelRunner
    from sglang_custom_amd.server_args import ServerArgs

    cfg, fam = _config(case), _family(case)
    had, new = _lengths(case)
    n, total, ctx = len(new), sum(had) + sum(new), max(a + b for a, b in zip(had, new)) + 16
    tokens = _tokens(case, cfg.get("vocab_size") or cfg["vocab"], seed)
    decode = case["phase"] == "decode"
    graph_bs = [b for b in get_batch_sizes_to_capture(64) if b >= n][:1]
    fp8 = bool(case.get("fp8"))
    args = ServerArgs(dtype="bfloat16", max_total_tokens=total + 64, max_running_requests=max(n, 64) + 8, context_length=ctx,
                      disable_cuda_graph=not decode, cuda_graph_bs=graph_bs, quantization="w8a8_fp8" if fp8 else None,
                      kv_cache_dtype="fp8_e4m3" if fp8 else "auto")
    s = _Step()
    s.runner = mr = ModelRunner(ModelConfig(cfg, dtype="bfloat16", context_length=ctx), args, weights=_weights(case, cfg, seed))
    pool, rows = mr.token_to_kv_pool, mr.req_to_token_pool.req_to_token
    layers = range(cfg.get("num_hidden_layers") or len(cfg["layers"]))

    def fill(slots):
        for l in layers:
            for buf, part in zip(pool.get_kv_buffer(l), _cached(case, cfg, l, seed)):
                part = part if part.dtype == buf.dtype else part.to(buf.dtype)
                if buf.dtype == torch.float8_e4m3fn:
                    buf, part = buf.view(torch.uint8), part.view(torch.uint8)
                buf[slots] = part.view((-1,) + tuple(buf.shape[1:]))

    def batch_of(reqs):
        b = ScheduleBatch.init_new(reqs, mr.req_to_token_pool, mr.token_to_kv_pool_allocator, None, mr.model_config)
        b.prepare_for_extend()
        return b

    with torch.no_grad():
        if decode:
            # most of the cached tokens came with the prompt (neighbouring slots), the last few one step at a time
            steps = 0 if fam == "fudonex" else min(16, min(had) - 1)
            batch = batch_of([Req(i, t[: a - steps]) for i, (t, a) in enumerate(zip(tokens, had))])
            if fam == "fudonex":      # recurrent state and averaged blocks: the prompts really run
                mr.forward(ForwardBatch.init_new(batch.get_model_worker_batch(), mr))
            for k in range(steps + 1):
                batch.output_ids = torch.tensor([t[a - steps + k] for t, a in zip(tokens, had)], device=DEV)
                batch.prepare_for_decode()
            if fam != "fudonex":
                fill(torch.cat([rows[i, :a] for i, a in zip(batch.req_pool_indices.tolist(), had)]).long())
        else:
            reqs = [Req(i, t) for i, t in enumerate(tokens)]
            if sum(had):
                slots = mr.token_to_kv_pool_allocator.alloc(sum(had))
                for r, part in zip(reqs, slots.split(had)):
                    r.init_next_round_input(part)
                fill(slots.long())
            batch = batch_of(reqs)
    s.batch = batch.get_model_worker_batch()
    loc = s.batch.out_cache_loc
    first = int(loc[0])
    assert bool((loc == torch.arange(first, first + loc.numel(), device=loc.device)).all())
    s.cache = [[b[first: first + loc.numel()] for b in ([pool.get_key_buffer(l)] if fam in ("deepseek", "silatar") else pool.get_kv_buffer(l))]
               for l in _shown(case, cfg)]
    state = mr.req_to_token_pool.state_pool
    # a decode step moves the state on, so repeated passes are steps of one conversation
    s.state = [] if state is None else [state.matrices[l][1: n + 1] for l in sorted(state.matrices)]
    s.init = ForwardBatch.init_new
    return s


def run(state):
    if not isinstance(state, _Step):
        return state.run()
    with torch.no_grad():
        forward_batch = state.init(state.batch, state.runner)
        out, _ = state.runner.forward(forward_batch)
        state.runner.sample(out, forward_batch)
    return dict(logits=out.next_token_logits, cache=state.cache, state=state.state)


class _Moe:
    """A Verozen layer's feed-forward: router on the fp32 stream, experts on its 16-bit copy, the sum of the chosen experts'
    outputs and the norm behind it."""

    def run(self):
        self.x.copy_(self.stream)      # the layer's mixer leaves a new stream on every step
        with torch.no_grad():
            y, rows, weights = self.moe(self.x, self.h)
            h = self.norm(self.x, y, rows=rows, coef=weights)
        return dict(x=self.x, h=h, weights=weights)


def _moe_parts(case, seed):
    from sglang_custom_amd import bench_designs as bd

    s = bd.VEROZEN_SIZES[case["size"]]
    g = torch.Generator(device=DEV).manual_seed(seed)
    E, D, ff = s["experts"], s["width"], s["ff"]

    def normal(*shape, std=1.0, dtype=torch.bfloat16):
        return torch.randn(shape, generator=g, device=DEV, dtype=dtype).mul_(std)

    return s, dict(x=normal(case["tokens"], D, dtype=torch.float32), router=normal(E, D, std=D ** -0.5, dtype=torch.float32),
                   correction=normal(E, std=0.1, dtype=torch.float32), up=normal(E, ff, D, std=D ** -0.5), down=normal(E, D, ff, std=ff ** -0.5),
                   norm=normal(D, std=0.1).add_(1.0))


def _prepare_moe(case, seed):
    from sglang_custom_amd.layers.post_norm import GroupRMSNorm
    from sglang_custom_amd.models.verozen import VerozenMoE

    size, p = _moe_parts(case, seed)
    s = _Moe()
    mlp = dict(expert=dict(ff=size["ff"]), router=dict(experts=size["experts"], top=size["top"], scale=1.0,
                                                       groups=dict(count=size["groups"], keep=size["keep"])))
    s.moe = VerozenMoE(size["width"], mlp, torch.bfloat16, DEV)
    s.norm = GroupRMSNorm(size["width"], size["norm_groups"], 1e-6, torch.bfloat16, DEV, residual_scale=2.0)
    for param, w in ((s.moe.router.weight, p["router"]), (s.moe.router.correction, p["correction"]), (s.moe.experts.w_up, p["up"]),
                     (s.moe.experts.w_down, p["down"]), (s.norm.weight, p["norm"])):
        param.data.copy_(w)
    s.stream, s.x, s.h = p["x"], torch.empty_like(p["x"]), p["x"].bfloat16()
    return s


class _Sample:
    def run(self):
        self.logits.copy_(self.fresh)      # the model's head writes new logits on every step; the sampler works in place
        with torch.no_grad():
            ids = self.sampler(self.out, self.info)
        return dict(ids=ids, probs=self.logits)


def _sample_parts(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    # a few likely tokens above a broad floor, as language models give
    z = torch.randn(case["requests"], case["vocab"], generator=g, device=DEV).mul_(2.5)
    r = random.Random(seed)
    return z, [round(r.uniform(0.6, 1.2), 3) for _ in range(case["requests"])]


def _prepare_sample(case, seed):
    from sglang_custom_amd.layers.logits_processor import LogitsProcessorOutput
    from sglang_custom_amd.layers.sampler import Sampler
    from sglang_custom_amd.managers.schedule_batch import Req
    from sglang_custom_amd.sampling.sampling_batch_info import SamplingBatchInfo
    from sglang_custom_amd.sampling.sampling_params import SamplingParams

    s = _Sample()
    s.fresh, temps = _sample_parts(case, seed)
    s.logits = torch.empty_like(s.fresh)
    s.out = LogitsProcessorOutput(next_token_logits=s.logits)
    reqs = [Req(i, [1], SamplingParams(temperature=t, top_p=case["top_p"], top_k=case["top_k"], min_p=case["min_p"])) for i, t in enumerate(temps)]
    s.info = SamplingBatchInfo.from_reqs(reqs, case["vocab"], DEV)
    s.sampler = Sampler(generator=torch.Generator(device=DEV).manual_seed(seed))
    return s


# ------------------------------------------------------------------------------------------------ bytes and operations
def work(case):
    if case["kind"] == "sample":
        n = case["requests"] * case["vocab"]
        return dict(bytes=3 * 4 * n, flops=4 * n)      # logits copied in, read, probabilities written
    if case["kind"] == "moe":
        from sglang_custom_amd import bench_designs as bd

        s, T = bd.VEROZEN_SIZES[case["size"]], case["tokens"]
        used = min(s["experts"], T * s["top"])
        return dict(bytes=used * 2 * s["width"] * s["ff"] * 2 + T * s["width"] * (4 + 4 + 2 + 2 + 4) + s["experts"] * s["width"] * 4,
                    flops=T * s["top"] * 4 * s["width"] * s["ff"] + 2 * T * s["experts"] * s["width"])
    cfg, fam = _config(case), _family(case)
    had, new = _lengths(case)
    T = sum(new)
    shapes = _transformer_shapes(cfg) if fam in ("llama", "deepseek") else _design_shapes(cfg)
    head = next(v for k, v in shapes.items() if k in ("lm_head.weight", "head")) if any(k in ("lm_head.weight", "head") for k in shapes) else \
        next(v for k, v in shapes.items() if "embed" in k)
    mats = sum(a * b for (k, v) in shapes.items() if len(v) == 2 and "embed" not in k and k not in ("lm_head.weight", "head") for a, b in [v])
    head = head[0] * head[1]
    fp8 = bool(case.get("fp8"))
    nbytes = mats * (1 if fp8 else 2) + head * 2 + len(new) * (head // (cfg.get("hidden_size") or cfg["width"])) * 4
    flops = 2.0 * mats * T + 2.0 * head * len(new)
    kvb = 1 if fp8 else 2

    def pairs(window=0, pool=0):
        got = 0
        for a, b in zip(had, new):
            for p in range(a, a + b):
                got += min(p + 1, window) + ((p - window + 1) // pool if pool and p >= window else 0) if window else p + 1
        return got

    everything = pairs()
    rows = sum(had) + T
    if fam == "llama":
        L, H, G, d = cfg["num_hidden_layers"], cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
        nbytes += L * rows * 2 * G * d * kvb
        flops += L * everything * H * 4 * d
    elif fam == "deepseek":
        L, H, R, r = cfg["num_hidden_layers"], cfg["num_attention_heads"], cfg["kv_lora_rank"], cfg["qk_rope_head_dim"]
        per = 2 * (2 * R + r) if case["phase"] == "decode" else 2 * (cfg["qk_nope_head_dim"] + r + cfg["v_head_dim"])
        nbytes += L * rows * (R + r) * 2
        flops += L * everything * H * per
    else:
        for spec in cfg["layers"]:
            m, t = spec["mixer"], spec["type"]
            if t == "latent_attention":
                per = 2 * (2 * m["kv_rank"] + m["rot_dim"]) if case["phase"] == "decode" else 2 * (m["dim"] + m["rot_dim"] + m["vdim"])
                nbytes += rows * (m["kv_rank"] + m["rot_dim"]) * 2
                flops += everything * m["heads"] * per
            elif t in ("mamba2", "delta"):
                k = m["state"] if t == "mamba2" else m["dim"]
                nbytes += len(new) * m["heads"] * k * m["vdim"] * 4 * (2 if case["phase"] == "decode" else 1)
                flops += T * m["heads"] * k * m["vdim"] * (6 if t == "mamba2" else 8)
            else:
                mask = m.get("mask") or {}
                see = pairs(mask["size"], mask["pool"]) if mask else everything
                n = 2 if t == "attention_2" else 1
                reach = rows if not mask or case["phase"] != "decode" else see
                nbytes += 0 if m.get("kv_from") is not None and case["phase"] != "decode" else reach * m["kv_heads"] * (n * m["dim"] + m["vdim"]) * 2
                flops += see * m["heads"] * 2 * n * (m["dim"] + m["vdim"])
    return dict(bytes=float(nbytes), flops=float(flops))


def tolerance(case):
    if case["kind"] == "sample":
        return dict(rel=1e-5, max=1e-4, differ=0.0)
    if case["kind"] == "moe":
        return dict(rel=7e-3)
    # measured against float64: 0.006 for the families that keep an fp32 stream or few layers, 0.008 .. 0.014 for the others
    return dict(rel=2e-2 if _family(case) in ("deepseek", "silatar") else 3e-2)


# ------------------------------------------------------------------------------------------------ the same in float64
def _lin(x, w):
    return x @ w.double().T


def _rms(x, eps, w=None):
    x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
    return x if w is None else x * w.double()


def _layer_norm(x, w, eps):
    x = x - x.mean(-1, keepdim=True)
    return _rms(x, eps, w)


def _silu(z):
    return z * torch.sigmoid(z)


def _blend(f, share, factor):
    """f where share is 1, f / factor where it is 0, linear in between."""
    share = share.clamp(0.0, 1.0)
    return share * f + (1.0 - share) * f / factor


def _freqs(dims, base):
    return float(base) ** (-2.0 * torch.arange(dims // 2, device=DEV, dtype=torch.float64) / dims)


def _freqs_by_turns(dims, base, sc, factor="factor", low="low", high="high", original="original"):
    """Pairs that turn often over the original length keep their frequency, those that seldom do are slowed."""
    f = _freqs(dims, base)
    return f if not sc else _blend(f, (sc[original] * f / (2 * math.pi) - sc[low]) / (sc[high] - sc[low]), sc[factor])


def _freqs_by_index(dims, base, sc):
    """The same over the pair's index, and the factor on cos and sin."""
    f = _freqs(dims, base)
    if not sc:
        return f, 1.0
    at = [dims * math.log(sc["original"] / (2 * math.pi * sc[k])) / (2 * math.log(base)) for k in ("fast", "slow")]
    lo, hi = max(math.floor(at[0]), 0), min(math.ceil(at[1]), dims - 1)
    i = torch.arange(dims // 2, device=DEV, dtype=torch.float64)
    return _blend(f, 1.0 - (i - lo) / max(hi - lo, 0.001), sc["factor"]), 0.1 * math.log(sc["factor"]) + 1.0


def _rotate(x, pos, f, neighbours, mag=1.0):
    """x [T, H, d]: pairs (2 i, 2 i + 1), or (i, i + n), turn by pos * f_i; the rest pass."""
    n = f.numel()
    a = pos.double()[:, None, None] * f
    c, s = mag * torch.cos(a), mag * torch.sin(a)
    out = x.clone()
    u, v = (x[..., 0: 2 * n: 2], x[..., 1: 2 * n: 2]) if neighbours else (x[..., :n], x[..., n: 2 * n])
    r1, r2 = u * c - v * s, v * c + u * s
    if neighbours:
        out[..., 0: 2 * n: 2], out[..., 1: 2 * n: 2] = r1, r2
    else:
        out[..., :n], out[..., n: 2 * n] = r1, r2
    return out


def _attend(q, k, v, scale, first, cap=None, window=0, pool=0, sink=None):
    """q [n, H, d] at positions first .. first + n - 1 over the keys k [m, G, d] and values v [m, G, dv] of positions 0 .. m - 1.
    window / pool: only the last `window` positions, and the mean of every block of `pool` that ends before them; sink [H]: a
    logit without a value."""
    n, H, m, G = q.shape[0], q.shape[1], k.shape[0], k.shape[1]
    per = H // G
    if pool:
        nb = m // pool
        k = torch.cat([k, k[: nb * pool].view(nb, pool, G, -1).mean(1)])
        v = torch.cat([v, v[: nb * pool].view(nb, pool, G, -1).mean(1)])
    out = torch.empty(n, H, v.shape[2], device=q.device, dtype=q.dtype)
    step = max(1, int(1.5e8) // (per * k.shape[0]))
    j = torch.arange(m, device=q.device)
    for a in range(0, n, step):
        i = torch.arange(first + a, first + min(n, a + step), device=q.device)
        seen = j[None] <= i[:, None]
        if window:
            seen &= i[:, None] - j[None] < window
        if pool:
            seen = torch.cat([seen, (torch.arange(nb, device=q.device)[None] + 1) * pool - 1 <= i[:, None] - window], 1)
        for g in range(G):
            s = torch.matmul(q[a: a + step, g * per: (g + 1) * per].transpose(0, 1).reshape(-1, q.shape[2]), k[:, g].T.contiguous())
            s = s.view(per, -1, k.shape[0]) * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            s = s.masked_fill(~seen, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[g * per: (g + 1) * per].double()[:, None, None].expand(per, s.shape[1], 1)], 2)
            p = torch.softmax(s, -1)
            if sink is not None:
                p = p[..., :-1]
            o = torch.matmul(p.reshape(-1, k.shape[0]), v[:, g].contiguous())
            out[a: a + step, g * per: (g + 1) * per] = o.view(per, -1, v.shape[2]).transpose(0, 1)
    return out


class _Restated:
    """The batch of a case on whole float64 rows: x [new tokens of all requests, width]."""

    def __init__(self, case, seed):
        self.case, self.cfg, self.seed = case, _config(case), seed
        self.had, self.new = _lengths(case)
        self.whole = _family(case) == "fudonex"       # no cached rows to start from: the cached tokens are run too
        if self.whole:
            self.had, self.new = [0] * len(self.new), [a + b for a, b in zip(self.had, self.new)]
        tokens = _tokens(case, self.cfg.get("vocab_size") or self.cfg["vocab"], seed)
        self.tokens = torch.tensor([x for t, a in zip(tokens, self.had) for x in t[a:]], device=DEV)
        self.pos = torch.cat([torch.arange(a, a + b, device=DEV) for a, b in zip(self.had, self.new)])
        self.last = torch.tensor(self.new, device=DEV).cumsum(0) - 1
        self.w = _weights(case, self.cfg, seed)
        self.cache, self.state = {}, []

    def attend(self, layer, q, new, scale, **opts):
        """new: the rows that the layer adds to the cache, (keys, values) or (one row,) whose first features are the values."""
        self.cache[layer] = new
        old = _cached(self.case, self.cfg, layer, self.seed) if not self.whole and sum(self.had) else None
        if old is not None and self.case.get("fp8"):
            old = [o.to(torch.float8_e4m3fn) for o in old]
        out, at, was = [], 0, 0
        width = opts.pop("vdim", None)
        split = opts.pop("maps", 1)
        for a, b in zip(self.had, self.new):
            rows = [n[at: at + b] for n in new]
            if old is not None:
                rows = [torch.cat([o[was: was + a].double().view((a,) + tuple(r.shape[1:])), r]) for o, r in zip(old, rows)]
            if width is not None:
                rows = [rows[0][:, None], rows[0][:, None, :width]]
            k, v, qs = rows[0], rows[1], q[at: at + b]
            if split == 1:
                out.append(_attend(qs, k, v, scale, a, **opts))
            else:
                d = qs.shape[-1]
                out.append(torch.stack([_attend(qs[:, :, i], k[..., i * d: (i + 1) * d], v, scale, a, **opts) for i in range(split)], 1))
            at, was = at + b, was + a
        return torch.cat(out)

    def answer(self, logits):
        return dict(logits=logits, cache=[list(self.cache[l]) if not self.case.get("fp8") else [None] * len(self.cache[l])
                                          for l in _shown(self.case, self.cfg)], state=self.state)

    # ---- the families
    def llama(self):
        c, w = self.cfg, self.w
        H, G, d, eps = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"], c["rms_norm_eps"]
        sc = c.get("rope_scaling")
        f = _freqs_by_turns(d, c["rope_theta"], sc, "factor", "low_freq_factor", "high_freq_factor", "original_max_position_embeddings")

        def weight(name):
            v = w[name + ".weight"]
            if not self.case.get("fp8"):
                return v
            s = v.float().abs().amax(1, keepdim=True) / 448.0      # per-channel e4m3 weights
            return (v.float() / s).to(torch.float8_e4m3fn).double() * s.double()

        x = w["model.embed_tokens.weight"][self.tokens].double()
        for i in range(c["num_hidden_layers"]):
            p = "model.layers.%d." % i
            h = _rms(x, eps, w[p + "input_layernorm.weight"])
            q, k, v = (_lin(h, weight(p + "self_attn.%s_proj" % n)).view(len(h), -1, d) for n in "qkv")
            o = self.attend(i, _rotate(q, self.pos, f, False), (_rotate(k, self.pos, f, False), v), d ** -0.5)
            x = x + _lin(o.reshape(len(h), H * d), weight(p + "self_attn.o_proj"))
            h = _rms(x, eps, w[p + "post_attention_layernorm.weight"])
            x = x + _lin(_silu(_lin(h, weight(p + "mlp.gate_proj"))) * _lin(h, weight(p + "mlp.up_proj")), weight(p + "mlp.down_proj"))
        return _lin(_rms(x[self.last], eps, w["model.norm.weight"]), w["model.embed_tokens.weight" if c["tie_word_embeddings"] else "lm_head.weight"])

    def deepseek(self):
        c, w = self.cfg, self.w
        H, R, dn, dr, dv, eps = (c["num_attention_heads"], c["kv_lora_rank"], c["qk_nope_head_dim"], c["qk_rope_head_dim"], c["v_head_dim"],
                                 c["rms_norm_eps"])
        f = _freqs(dr, c["rope_theta"])
        x = w["model.embed_tokens.weight"][self.tokens].double()
        T = len(x)
        for i in range(c["num_hidden_layers"]):
            p = "model.layers.%d." % i
            a = p + "self_attn."
            h = _rms(x, eps, w[p + "input_layernorm.weight"])
            q = _lin(_rms(_lin(h, w[a + "q_a_proj.weight"]), eps, w[a + "q_a_layernorm.weight"]), w[a + "q_b_proj.weight"]).view(T, H, dn + dr)
            y = _lin(h, w[a + "kv_a_proj_with_mqa.weight"])
            row = torch.cat([_rms(y[:, :R], eps, w[a + "kv_a_layernorm.weight"]), _rotate(y[:, None, R:], self.pos, f, True)[:, 0]], 1)
            kv = w[a + "kv_b_proj.weight"].double().view(H, dn + dv, R)
            o = self.latent(i, q, kv[:, :dn], kv[:, dn:], row, f, 1.0, (dn + dr) ** -0.5)
            x = x + _lin(o.reshape(T, H * dv), w[a + "o_proj.weight"])
            h = _rms(x, eps, w[p + "post_attention_layernorm.weight"])
            x = x + _lin(_silu(_lin(h, w[p + "mlp.gate_proj.weight"])) * _lin(h, w[p + "mlp.up_proj.weight"]), w[p + "mlp.down_proj.weight"])
        for l in list(self.cache):
            self.cache[l] = (self.cache[l][0][:, None],)
        return _lin(_rms(x[self.last], eps, w["model.norm.weight"]), w["lm_head.weight"])

    def latent(self, layer, q, uk, uv, row, f, mag, scale):
        """Attention over latent rows: the queries are taken to the latent space, the result back out of it."""
        H, dn, R = uk.shape
        qa = torch.matmul(q[..., :dn].transpose(0, 1).contiguous(), uk).transpose(0, 1)
        qq = torch.cat([qa, _rotate(q[..., dn:], self.pos, f, True, mag)], -1)
        o = self.attend(layer, qq, (row,), scale, vdim=R)
        return torch.matmul(o.transpose(0, 1).contiguous(), uv.transpose(1, 2).contiguous()).transpose(0, 1)

    def silatar(self):
        c, w, eps = self.cfg, self.w, self.cfg["norm"]["eps"]
        x = w["embed"][self.tokens].double()
        T = len(x)
        for i, spec in enumerate(c["layers"]):
            p, m = "l%d." % i, spec["mixer"]
            H, dn, dr, dv, R = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
            f, mag = _freqs_by_index(m["rot"]["dims"], m["rot"]["base"], m["rot"].get("scaling"))
            h = _layer_norm(x, w[p + "norm1"], eps)
            y = _lin(h, w[p + "mix.dkv"])
            row = torch.cat([_rms(y[:, :R], eps, w[p + "mix.dkv.norm"]), _rotate(y[:, None, R:], self.pos, f, True, mag)[:, 0]], 1)
            o = self.latent(i, _lin(h, w[p + "mix.q"]).view(T, H, dn + dr), w[p + "mix.uk"].double().view(H, dn, R),
                            w[p + "mix.uv"].double().view(H, dv, R), row, f, mag, m["scale"])
            x = x + _layer_norm(_lin(o.reshape(T, H * dv), w[p + "mix.o"]), w[p + "norm1b"], eps)
            h = _layer_norm(x, w[p + "norm2"], eps)
            z = _lin(h, w[p + "mlp.up"])
            x = x + _layer_norm(_lin(0.5 * z * (1.0 + torch.erf(z / math.sqrt(2.0))), w[p + "mlp.down"]), w[p + "norm2b"], eps)
        z = _lin(_layer_norm(x[self.last], w["final.norm"], eps), w["head"])
        return c["logit_softcap"] * torch.tanh(z / c["logit_softcap"])

    def lomazen(self):
        c, w, eps = self.cfg, self.w, self.cfg["norm"]["eps"]
        x = w["embed"][self.tokens].double()
        T = len(x)
        for i, spec in enumerate(c["layers"]):
            p, m = "l%d." % i, spec["mixer"]
            H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
            f = _freqs_by_turns(m["rot"]["dims"], m["rot"]["base"], m["rot"].get("scaling"))
            h = _rms(x, eps, w[p + "norm1"])
            q, k, v, g = (_lin(h, w[p + "mix." + n]) for n in "qkvg")
            v = v.view(T, G, dv)
            if spec["type"] == "attention":
                q, k = (_rms(_rotate(z.view(T, -1, d), self.pos, f, True), eps) for z in (q, k))
                o = self.attend(i, q, (k, v), m["scale"], cap=m["softcap"]).reshape(T, H * dv) * torch.sigmoid(g)
            else:
                q = _rotate(q.view(T, 2 * H, d), self.pos, f, False).view(T, H, 2, d)
                k = _rotate(k.view(T, 2 * G, d), self.pos, f, False).view(T, G, 2 * d)
                lam = (torch.exp((w[p + "mix.lq1"].double() * w[p + "mix.lk1"].double()).sum())
                       - torch.exp((w[p + "mix.lq2"].double() * w[p + "mix.lk2"].double()).sum()) + m["diff"])
                o = self.attend(i, q, (k, v), m["scale"], maps=2)
                o = (_rms(o[:, 0] - lam * o[:, 1], eps) * (1.0 - m["diff"]) * torch.sigmoid(g)[:, :, None]).reshape(T, H * dv)
            x = x + _rms(_lin(o, w[p + "mix.o"]), eps, w[p + "norm1b"])
            h = _rms(x, eps, w[p + "norm2"])
            z = _lin(h, w[p + "mlp.gate"])
            z = 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))
            x = x + _rms(_lin(z * _lin(h, w[p + "mlp.up"]), w[p + "mlp.down"]), eps, w[p + "norm2b"])
        return _lin(_rms(x[self.last], eps, w["final.norm"]), w["embed"]) * c["logit_scale"]

    def fudonex(self):
        c, w, eps = self.cfg, self.w, self.cfg["norm"]["eps"]
        x = w["embed"][self.tokens].double() * c["embedding"]["scale"]
        T = len(x)
        kv = {}
        for i, spec in enumerate(c["layers"]):
            p, m, t = "l%d." % i, spec["mixer"], spec["type"]
            n = p + "mix."
            H, dv = m["heads"], m["vdim"]
            if t == "attention":
                G, d, mask = m["kv_heads"], m["dim"], m["mask"]
                f, mag = _freqs_by_index(m["rot"]["dims"], m["rot"]["base"], m["rot"].get("scaling"))
                q = _rotate(_rms((_lin(x, w[n + "q"]) + w[n + "q.b"].double()).view(T, H, d), eps, w[n + "q.norm"]), self.pos, f, False, mag)
                src = m.get("kv_from")
                if src is None:
                    k = _rms((_lin(x, w[n + "k"]) + w[n + "k.b"].double()).view(T, G, d), eps, w[n + "k.norm"])
                    kv[i] = (_rotate(k, self.pos, f, False, mag), _rms((_lin(x, w[n + "v"]) + w[n + "v.b"].double()).view(T, G, dv), eps))
                o = self.attend(i, q, kv[i if src is None else src], m["scale"], window=mask["size"], pool=mask["pool"], sink=w[n + "sink"])
                y = (o * torch.sigmoid(_lin(x, w[n + "g"]))[:, :, None]).reshape(T, H * dv)
            elif t == "mamba2":
                inner, G, N = H * dv, m["groups"], m["state"]
                z = _lin(x, w[n + "in"])
                u = _silu(self.conv(z[:, inner: 2 * inner + 2 * G * N], w[n + "conv"]) + w[n + "conv.b"].double())
                dt = torch.nn.functional.softplus(z[:, 2 * inner + 2 * G * N:] + w[n + "dt_bias"].double())
                xs, B, C = u[:, :inner].view(T, H, dv), u[:, inner: inner + G * N].view(T, G, N), u[:, inner + G * N:].view(T, G, N)
                B, C = B.repeat_interleave(H // G, 1), C.repeat_interleave(H // G, 1)
                y = self.recur(torch.exp(-torch.exp(w[n + "A_log"].double()) * dt), B * dt[..., None], xs, C)
                y = (y + w[n + "D"].double()[:, None] * xs).reshape(T, inner) * _silu(z[:, :inner])
                parts = m["norm_groups"]
                y = _rms(y.view(T, parts, inner // parts), eps).reshape(T, inner) * w[n + "norm"].double()
            else:
                G, d = m["kv_heads"], m["dim"]
                q, k, v = (_silu(self.conv(_lin(x, w[n + a]), w[n + a + ".conv"])) for a in "qkv")
                q, k = (z.view(T, G, d) * torch.rsqrt((z.view(T, G, d) ** 2).sum(-1, keepdim=True) + 1e-6) for z in (q, k))
                q, k = (z.repeat_interleave(H // G, 1) for z in (q * d ** -0.5, k))
                keep = torch.exp(-torch.exp(w[n + "A_log"].double()) * torch.nn.functional.softplus(_lin(x, w[n + "a"]) + w[n + "dt_bias"].double()))
                y = self.recur(keep, k, v.view(T, H, dv), q, beta=torch.sigmoid(_lin(x, w[n + "b"])))
                y = (_rms(y, eps) * w[n + "norm"].double()).reshape(T, H * dv) * _silu(_lin(x, w[n + "g"]))
            mult = c["residual_mult"]
            x = x + mult * w[p + "ls1"].double() * _rms(_lin(y, w[n + "o"]), eps) * (1.0 + w[p + "norm1"].double())
            y = _lin(_silu(_lin(x, w[p + "mlp.gate"])) * _lin(x, w[p + "mlp.up"]), w[p + "mlp.down"])
            x = x + mult * w[p + "ls2"].double() * _rms(y, eps) * (1.0 + w[p + "norm2"].double())
        if self.case["phase"] == "decode":
            self.cache = {l: tuple(r[self.last] for r in rows) for l, rows in self.cache.items()}
        z = _lin(_rms(x[self.last], eps) * (1.0 + w["final.norm"].double()), w["embed"])
        return c["logit_softcap"] * torch.tanh(z / c["logit_softcap"])

    def conv(self, u, w):
        """The last tap multiplies the current token."""
        w, taps, out = w.double(), w.shape[1], []
        for part in u.split(self.new):
            part = torch.cat([part.new_zeros(taps - 1, part.shape[1]), part])
            out.append(sum(part[k: part.shape[0] - taps + 1 + k] * w[:, k] for k in range(taps)))
        return torch.cat(out)

    def recur(self, keep, k, v, q, beta=None):
        """S <- keep S + k v^T (with beta: k (beta (v - S^T k))^T after the decay), o = S^T q, per request and head, token by token."""
        B, longest = len(self.new), max(self.new)
        at = torch.full((B, longest), -1, device=DEV)
        for b, (end, n) in enumerate(zip(self.last.tolist(), self.new)):
            at[b, :n] = torch.arange(end - n + 1, end + 1, device=DEV)
        H, d, dv = k.shape[1], k.shape[2], v.shape[2]
        S = torch.zeros(B, H, d, dv, device=DEV, dtype=torch.float64)
        out = torch.zeros_like(v)
        for t in range(longest):
            live = (at[:, t] >= 0).nonzero()[:, 0] if min(self.new) <= t else slice(None)
            i = at[live, t]
            R = S[live] * keep[i][:, :, None, None]
            u = v[i]
            if beta is not None:
                u = beta[i][..., None] * (u - torch.matmul(k[i][:, :, None], R)[:, :, 0])
            R = R + k[i][..., None] * u[:, :, None]
            out[i] = torch.matmul(q[i][:, :, None], R)[:, :, 0]
            S[live] = R
        self.state.append(S)
        return out


def exact(case, seed):
    with torch.no_grad():
        if case["kind"] == "sample":
            z, temps = _sample_parts(case, seed)
            return dict(ids=None, probs=torch.softmax(z.double() / torch.tensor(temps, device=DEV, dtype=torch.float64)[:, None], -1))
        if case["kind"] == "moe":
            return _exact_moe(case, seed)
        r = _Restated(case, seed)
        return r.answer(getattr(r, _family(case))())


def _exact_moe(case, seed):
    s, p = _moe_parts(case, seed)
    x, h = p["x"].double(), p["x"].bfloat16().double()
    E, gc, top = s["experts"], s["groups"], s["top"]
    score = torch.sigmoid(_lin(x, p["router"]))
    choice = score + p["correction"].double()
    best = choice.view(-1, gc, E // gc).topk(2, -1).values.sum(-1).topk(s["keep"], -1).indices
    allowed = torch.zeros(len(x), gc, device=DEV, dtype=torch.bool).scatter_(1, best, True).repeat_interleave(E // gc, 1)
    ids = choice.masked_fill(~allowed, -math.inf).topk(top, -1).indices
    weights = score.gather(1, ids)
    weights = weights / (weights.sum(-1, keepdim=True) + 1e-20)
    y = torch.zeros_like(x)
    for e in range(E):
        t, j = (ids == e).nonzero(as_tuple=True)
        z = _lin(h[t], p["up"][e])
        y.index_add_(0, t, weights[t, j][:, None] * _lin(0.5 * z * (1.0 + torch.erf(z / math.sqrt(2.0))), p["down"][e]))
    g = s["norm_groups"]
    x = _rms((2.0 * x + y).view(len(x), g, -1), 1e-6).view(len(x), -1) * p["norm"].double()
    return dict(x=x, h=x, weights=weights)
