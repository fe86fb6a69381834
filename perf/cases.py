"""The work that this framework is measured on: steps of its models through the calls its engine makes, with random weights of real layer sizes.

A case is one step of one model.  Models: GLM-4-MoE at the sizes the decode metric is quoted on (width 4096, 96 query and 8 key/value heads
of 128, 64 experts of 1408 of which 8 are taken, a shared one, a dense first layer of 10944) and the four decoders that run step batches
(Dafolorn, Napadra, Gulozen, Loselix) at the two widths their benchmarks have.  A few layers of each kind stand for the whole stack.

Steps: "decode" (one token per sequence over a filled cache, replayed from a HIP graph, as the engine does), "prefill" (whole prompts,
eager) and "mixed" (prompts beside decoding sequences in one step).  Sequences of a step have different lengths.  Outputs are the logits of
every sequence's last token, the caches and the recurrent states, all as the step leaves them."""
import math
import os
import sys
import types
import zlib

import torch

_PACKAGE = os.path.join(os.getcwd(), "glm4_moe_nano-vllm_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

DEV, BF16, F64 = "cuda", torch.bfloat16, torch.float64
VOCAB, EPS, TAPS = 32768, 1e-5, 4
BLOCK = {"glm": 256}            # tokens per cache block; the others have 64
FAMILIES = ("dafolorn", "napadra", "gulozen", "loselix")


# ---- cases ------------------------------------------------------------------------------------------------------------------
def listed():
    c = lambda name, family, size, mode, batch, length, **kw: dict(name=name, family=family, size=size, mode=mode, batch=batch, length=length, **kw)  # noqa: E731
    return [
        # one user waiting for the next token: launches, latency, weights read for a single row
        c("glm_decode_b1_1k", "glm", "air", "decode", 1, 1024),
        # the headline: 32 sequences of 4096 tokens
        c("glm_decode_b32_4k", "glm", "air", "decode", 32, 4096),
        # quantised experts and long contexts
        c("glm_decode_b64_8k_fp8", "glm", "air", "decode", 64, 8192, experts="fp8"),
        # one short prompt: every weight is read for a few rows
        c("glm_prefill_1x211", "glm", "air", "prefill", 1, 211),
        # a full step of prompts
        c("glm_prefill_4x4096", "glm", "air", "prefill", 4, 4096),
        # many users at once on a small model: projections of 128 rows, windowed attention over latents
        c("dafolorn_decode_b128_4k", "dafolorn", "2k", "decode", 128, 4096),
        c("dafolorn_prefill_4x4096", "dafolorn", "2k", "prefill", 4, 4096),
        # new prompts beside running sequences, an odd number of both
        c("napadra_mixed_27_5x2500", "napadra", "2k", "mixed", 27, 2500, prompts=5),
        c("gulozen_decode_b100_3k", "gulozen", "2k", "decode", 100, 3000),
        c("gulozen_prefill_4x4096", "gulozen", "2k", "prefill", 4, 4096),
        c("loselix_decode_b1_4k", "loselix", "4k", "decode", 1, 4096),
        c("loselix_prefill_4x4096", "loselix", "2k", "prefill", 4, 4096),
    ]


def draw(rng):
    """A step within the listed ones' ranges: batches up to 128 (GLM: 64), contexts from 64 up to 4096 (GLM with quantised experts: 8192),
    prompts up to 16384 tokens together."""
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    family = rng.choice(("glm", "glm") + FAMILIES)
    mode = rng.choice(("decode", "decode", "prefill") + (() if family == "glm" else ("mixed",)))
    case = {"family": family, "size": "air" if family == "glm" else rng.choice(("2k", "4k")), "mode": mode}
    if mode == "decode":
        fp8 = family == "glm" and rng.random() < 0.3
        case.update(batch=log(1, 64 if family == "glm" else 128), length=log(64, 8192 if fp8 else 4096))
        if fp8:
            case["experts"] = "fp8"
    else:
        length = log(64, 4096)
        prompts = log(1, max(1, min(32, 16384 // length)))
        case.update(batch=prompts, length=length)
        if mode == "mixed":
            case.update(batch=log(1, 64), prompts=prompts)
    return case


def _lengths(case):
    """[(tokens in front of the step, tokens of the step)] per sequence: shorter and shorter by something odd, down to three quarters."""
    n = case["length"]
    ragged = [n - (b * 389) % max(1, n // 4) for b in range(max(case["batch"], case.get("prompts", 0)))]
    decode, prefill = [(m - 1, 1) for m in ragged], [(0, m) for m in ragged]
    if case["mode"] == "mixed":
        return decode[: case["batch"]] + prefill[: case["prompts"]]
    return (decode if case["mode"] == "decode" else prefill)[: case["batch"]]


# ---- sizes and weights --------------------------------------------------------------------------------------------------------
GLM_LAYERS = 4                  # the first one dense


def _glm_config(case):
    return types.SimpleNamespace(
        hidden_size=4096, num_attention_heads=96, num_key_value_heads=8, head_dim=128, attention_bias=True, use_qk_norm=False, partial_rotary_factor=0.5,
        rope_theta=1e6, rope_scaling=None, max_position_embeddings=16384, rms_norm_eps=EPS, n_routed_experts=64, num_experts_per_tok=8, n_group=1, topk_group=1,
        routed_scaling_factor=1.0, n_shared_experts=1, moe_intermediate_size=1408, intermediate_size=10944, first_k_dense_replace=1, hidden_act="silu",
        vocab_size=VOCAB, num_hidden_layers=GLM_LAYERS, num_layers_to_load=GLM_LAYERS, tie_word_embeddings=False, torch_dtype=BF16,
        expert_weight_dtype="fp8_e4m3" if case.get("experts") == "fp8" else None)


def _config(case):
    """The raw configuration of a step-batch model."""
    big = case["size"] == "4k"
    w, H, dim = (4096, 32, 128) if big else (2048, 16, 128)
    family = case["family"]
    if family == "dafolorn":    # three layers, the middle one twice
        one = {"type": "latent_attention", "mixer": {"heads": H, "dim": dim, "vdim": dim, "kv_rank": 512 if big else 256, "mask": {"size": 4096 if big else 1024},
               "scale": dim ** -0.5}, "mlp": {"kind": "dense", "ff": 3 * w}}
        return {"architecture": "Dafolorn", "width": w, "vocab": VOCAB, "canon": {"taps": TAPS}, "norm": {"eps": EPS}, "layers": [one] * 3,
                "loop": {"start": 1, "stop": 2, "times": 2}, "logit_softcap": 30.0}
    if family == "napadra":     # attention twice, once more over the second one's cache, a matrix memory
        mlp = {"kind": "dense", "ff": 2 * w, "limit": 7.0}
        att = {"heads": H, "kv_heads": H // 4, "dim": dim, "vdim": dim, "mask": {"size": 4096 if big else 1024}, "scale": dim ** -0.5}
        mem = {"heads": H // 2, "dim": 128, "vdim": 256, "gate_cap": 15.0}
        kinds = [("attention", att), ("attention", att), ("attention", dict(att, kv_from=1)), ("mlstm", mem)]
        return {"architecture": "Napadra", "width": w, "vocab": VOCAB, "streams": 2, "residual_mult": 0.5, "norm": {"eps": EPS},
                "layers": [{"type": t, "mixer": m, "mlp": mlp} for t, m in kinds]}
    if family == "gulozen":     # latent attention three times, linear attention, all with experts
        mlp = {"kind": "moe", "expert": {"ff": 1408 if big else 1024}, "router": {"experts": 64, "top": 8 if big else 6}}
        att = {"type": "latent_attention", "mlp": mlp, "mixer": {
            "heads": H, "dim": dim, "rot_dim": 64, "vdim": dim, "q_rank": 1536 if big else 768, "kv_rank": 512, "scale": 192 ** -0.5,
            "rot": {"base": 10000.0, "dims": 64, "scaling": {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}}
        lin = {"type": "lightning", "mlp": mlp, "mixer": {"heads": H, "dim": 128, "vdim": 128, "decay": [1 - 2.0 ** -(2 + 8 * h / H) for h in range(H)]}}
        return {"architecture": "Gulozen", "width": w, "vocab": VOCAB, "norm": {"eps": EPS, "groups": 4}, "canon": {"taps": TAPS}, "embedding": {"scale": 4.0},
                "layers": [att, att, att, lin]}
    base = {"heads": H, "kv_heads": H // 4, "dim": dim, "vdim": dim, "scale": dim ** -0.5}     # loselix: three kinds of attention, all of them twice
    kinds = [("attention", dict(base, dim=dim // 2, scale=(dim // 2) ** -0.5, rot={"base": 1e4, "dims": dim // 4}, diff=0.6, softcap=40.0)),
             ("attention_2", dict(base, rot={"base": 1e4, "dims": dim // 2})), ("attention_3", dict(base, q_temp={"coef": 0.3, "every": 1024}))]
    return {"architecture": "Loselix", "width": w, "vocab": VOCAB, "norm": {"eps": EPS}, "loop": {"start": 0, "stop": 3, "times": 2},
            "layers": [{"type": t, "mixer": m, "mlp": {"kind": "dense", "ff": 3 * w}} for t, m in kinds]}


FLAGS = 16      # columns of the residual that carry a token's signs to the routers
MARGIN = {"glm": 0.1, "gulozen": 0.05}


def _weights(case):
    """{name: (shape, standard deviation, mean, what its last FLAGS columns or rows are)} of every tensor of the model.

    Which expert is the last one taken is a jump that a rounding can decide, and then nothing more is to be compared in that row.  The last
    FLAGS columns of the residual are therefore signs that every token brings along ("signs"), that no sublayer changes ("rows", "zeros",
    "ones") and that the routers read above all ("columns"); tokens for which the choice is close are not drawn (_tokens).  Rows spread over
    the experts as they would otherwise."""
    t = {}

    def mat(name, n, k, std=None, flags=None):
        t[name] = ((n, k), k ** -0.5 if std is None else std, 0.0, flags)

    def vec(name, n, std, mean=0.0, flags=None):
        t[name] = (n if isinstance(n, tuple) else (n,), std, mean, flags)

    if case["family"] == "glm":
        c = _glm_config(case)
        w, hd = c.hidden_size, c.head_dim
        mat("model.embed_tokens.weight", VOCAB, w, 0.7, "signs"), mat("lm_head.weight", VOCAB, w, 0.02)
        vec("model.norm.weight", w, 0.02, 1.0)
        for i in range(GLM_LAYERS):
            p = f"model.layers.{i}."
            N = (c.num_attention_heads + 2 * c.num_key_value_heads) * hd
            mat(p + "self_attn.qkv_proj.weight", N, w, 0.02), vec(p + "self_attn.qkv_proj.bias", N, 0.02)
            mat(p + "self_attn.o_proj.weight", w, c.num_attention_heads * hd, 0.02, "rows")
            for q in ("input_layernorm", "post_attention_layernorm"):
                vec(p + q + ".weight", w, 0.02, 1.0, "ones")
            blocks = [("mlp.", c.intermediate_size)]
            if i >= c.first_k_dense_replace:
                mat(p + "mlp.gate.weight", c.n_routed_experts, w, 1e-4, "columns"), vec(p + "mlp.gate.e_score_correction_bias", c.n_routed_experts, 0.0)
                blocks = [(f"mlp.experts.{e}.", c.moe_intermediate_size) for e in range(c.n_routed_experts)] + [("mlp.shared_experts.", c.moe_intermediate_size)]
            for q, f in blocks:
                mat(p + q + "gate_up_proj.weight", 2 * f, w, 0.02), mat(p + q + "down_proj.weight", w, f, 0.02, "rows")
        return t
    raw, family = _config(case), case["family"]
    w = raw["width"]
    mat("embed", VOCAB, w, 0.25 if family == "gulozen" else 0.7, "signs" if family == "gulozen" else None)
    if family == "dafolorn":
        vec("final.norm", w, 0.1), mat("loop.in", w, 2 * w), vec("loop.step", (raw["loop"]["times"], w), 0.3)
    else:
        vec("final.norm", () if family == "napadra" else w, 0.1, 1.0), mat("head", VOCAB, w)
    for i, e in enumerate(raw["layers"]):
        p, s, kind = f"l{i}.", e["mixer"], e["type"]
        H, d, v, G = s["heads"], s["dim"], s["vdim"], s.get("kv_heads")
        m = 2 if "diff" in s else 1
        mat(p + "mix.o", w, H * v)
        if family == "dafolorn":
            for q in ("norm1", "norm1b", "norm2", "norm2b"):
                vec(p + q, w, 0.1)
            vec(p + "canon1", (w, TAPS), 0.3), vec(p + "canon2", (w, TAPS), 0.3), vec(p + "mlp.act", 2, 0.5)
            mat(p + "mlp.up", e["mlp"]["ff"], w), mat(p + "mlp.down", w, e["mlp"]["ff"])
            mat(p + "mix.q", H * d, w), mat(p + "mix.dkv", s["kv_rank"], w)
        elif family == "napadra":
            vec(p + "shift", w, 0.3)
            for q in (1, 2):
                vec(p + f"norm{q}", (), 0.1, 1.0), vec(p + f"ls{q}", w, 0.2, 1.0), vec(p + f"hc{q}.in", 2, 0.2, 0.5), vec(p + f"hc{q}.out", 2, 0.2, 1.0)
                vec(p + f"hc{q}.mix", (2, 2), 0.1)           # and the identity (_tensor)
            for q in ("gate", "up"):
                mat(p + "mlp." + q, e["mlp"]["ff"], w)
            mat(p + "mlp.down", w, e["mlp"]["ff"]), mat(p + "mix.q", H * d, w)
            if kind == "mlstm":
                mat(p + "mix.k", H * d, w), mat(p + "mix.v", H * v, w), mat(p + "mix.g", H * v, w), vec(p + "mix.norm", H * v, 0.1, 1.0)
                mat(p + "mix.i", H, w), vec(p + "mix.i.b", H, 1.0), mat(p + "mix.f", H, w), vec(p + "mix.f.b", H, 1.0, 4.0)
            else:
                vec(p + "mix.sink", H, 1.0)
                if "kv_from" not in s:
                    mat(p + "mix.k", G * d, w), mat(p + "mix.v", G * v, w)
        elif family == "gulozen":
            vec(p + "norm1", w, 0.1, 1.0, "zeros"), vec(p + "norm2", w, 0.1, 1.0, "zeros"), vec(p + "canon1", (w, TAPS), 0.3, 0.0, "rows"), vec(p + "dwa", i + 2, 0.2)
            E, f = e["mlp"]["router"]["experts"], e["mlp"]["expert"]["ff"]
            mat(p + "mix.g", H * v, w), mat(p + "mlp.router", E, w, 0.004 * w ** -0.5, "columns")
            for x in range(E):
                mat(p + f"mlp.e{x}.gate", f, w), mat(p + f"mlp.e{x}.up", f, w), mat(p + f"mlp.e{x}.down", w, f)
            if kind == "lightning":
                mat(p + "mix.q", H * d, w), mat(p + "mix.k", H * d, w), mat(p + "mix.v", H * v, w), vec(p + "mix.norm", H * v, 0.1, 1.0)
            else:
                r, rd, qr = s["kv_rank"], s["rot_dim"], s["q_rank"]
                mat(p + "mix.dq", qr, w), vec(p + "mix.dq.norm", qr, 0.1, 1.0), mat(p + "mix.uq", H * (d + rd), qr), mat(p + "mix.dkv", r + rd, w)
        else:
            vec(p + "norm1", w, 0.1, 1.0), mat(p + "mlp.up", e["mlp"]["ff"], w), mat(p + "mlp.down", w, e["mlp"]["ff"])
            mat(p + "mix.q", H * m * d, w), mat(p + "mix.k", G * m * d, w)
            if kind != "attention_3":
                mat(p + "mix.v", G * v, w)
            if kind == "attention":
                for q in ("lq1", "lk1", "lq2", "lk2"):
                    vec(p + "mix." + q, d, 0.1)
            elif kind == "attention_2":
                mat(p + "mix.g", H, w)
            else:
                vec(p + "mix.q.norm", H * d, 0.1, 1.0), vec(p + "mix.k.norm", G * d, 0.1, 1.0), vec(p + "mix.pb", H, 0.3, -7.0), mat(p + "mix.g", H * v, w)
        if "kv_rank" in s:
            r = s["kv_rank"]
            vec(p + "mix.dkv.norm", r, 0.1, 1.0), mat(p + "mix.uk", H * d, r), mat(p + "mix.uv", H * v, r), vec(p + "mix.sink", H, 1.0)
    return t


def _randn(seed, name, shape, std=1.0, mean=0.0, dtype=BF16):
    g = torch.Generator(device=DEV).manual_seed((seed * 1000003 + zlib.crc32(name.encode())) % (1 << 31))
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).mul_(std).add_(mean).to(dtype)


def _tensor(seed, name, spec):
    shape, std, mean, flags = spec
    t = _randn(seed, name, shape, std, mean, torch.float32 if name.endswith("correction_bias") else BF16)
    if flags == "signs":
        t[:, -FLAGS:] = torch.where(t[:, -FLAGS:] < 0, -1.0, 1.0) * (2.0 if std > 0.5 else 0.5)      # (Gulozen's embedding is scaled by 4)
    elif flags == "columns":
        t[:, -FLAGS:] = _randn(seed, name + "+", (shape[0], FLAGS), 0.2)
    elif flags:
        t[-FLAGS:] = 1.0 if flags == "ones" else 0.0
    if name.endswith(".dwa"):           # an average that keeps the first and above all the last layer
        t[0], t[-1] = 0.4, 0.7
    return t + torch.eye(2, device=DEV, dtype=BF16) if name.endswith(".mix") else t


# ---- one step: tokens, cache blocks, caches and states ---------------------------------------------------------------------------
def _tokens(case, seed):
    """Tokens of every sequence; where there are routers, of those whose experts do not hang on a rounding."""
    g, spec, usable = torch.Generator().manual_seed(seed), _weights(case), torch.arange(VOCAB)
    for name, v in spec.items():
        if v[3] == "signs":
            signs, top = _tensor(seed, name, v)[:, -FLAGS:].float().sign(), 8 if case["size"] != "2k" else 6
            ok = torch.ones(VOCAB, dtype=torch.bool, device=DEV)
            for gate, u in spec.items():
                if u[3] == "columns":
                    z = signs @ _tensor(seed, gate, u)[:, -FLAGS:].float().T
                    best = z.topk(top + 1, -1).values
                    ok &= best[:, top - 1] - best[:, top] > MARGIN[case["family"]] * z.std()
            usable = ok.nonzero().flatten().cpu()
    return [usable[torch.randint(0, usable.numel(), (n,), generator=g)].tolist() for _, n in _lengths(case)]


def _blocks(case, seed):
    """Cache blocks of every sequence, scattered over the pool."""
    bs = BLOCK.get(case["family"], 64)
    need = [-(-(start + n) // bs) for start, n in _lengths(case)]
    perm = iter(torch.randperm(sum(need), generator=torch.Generator().manual_seed(seed + 1)).tolist())
    return [[next(perm) for _ in range(k)] for k in need], sum(need), bs


def _fill(seed, named):
    """Caches and states as an earlier program left them: random values."""
    for name, t in named:
        t.copy_(_randn(seed, name, t.shape, dtype=t.dtype)) if not name.endswith("factors") else t.fill_(1.0)


def _buffers(model):
    """(name, tensor) of every cache and state of a step-batch model."""
    for i, layer in enumerate(model.layers):
        for k, c in enumerate(getattr(layer.mixer, "caches", ())):
            parts = c if isinstance(c, tuple) else (c,)
            for q, t in zip(("keys", "values", "factors"), parts):
                if t is not None and not (q == "values" and t is parts[0]):
                    yield f"{i}.{k}.{q}", t
        for q in ("entry1", "entry2"):
            for k, t in enumerate(getattr(getattr(layer, q, None), "state", None) or ()):
                yield f"{i}.{k}.{q}", t
        for q in ("sub1", "taps", "mixer"):
            s = getattr(getattr(layer, q, None), "state", None)
            for k, t in enumerate(s if isinstance(s, tuple) else (s,) if s is not None else ()):
                yield f"{i}.{k}.{q}.state", t


def _graph(fn):
    fn()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = fn()
    torch.cuda.synchronize()
    return g, out


@torch.inference_mode()
def prepare(case, seed):
    from nanovllm import hip_ops
    hip_ops.load_library()
    return (_prepare_glm if case["family"] == "glm" else _prepare_step)(case, seed)


def _prepare_glm(case, seed):
    from nanovllm.models.glm4_moe.model import Glm4MoeForCausalLM
    from nanovllm.utils.context import reset_context, set_context
    cfg, spec = _glm_config(case), _weights(case)
    old = torch.get_default_dtype()
    torch.set_default_dtype(BF16)
    try:
        with torch.device(DEV):
            m = Glm4MoeForCausalLM(cfg)
    finally:
        torch.set_default_dtype(old)
    for name, p in list(m.named_parameters()) + [b for b in m.named_buffers() if b[0] in spec]:
        p.data.copy_(_tensor(seed, name, spec[name]))
    blocks, total, bs = _blocks(case, seed)
    kv = [[torch.empty(total, bs, cfg.num_key_value_heads, cfg.head_dim, dtype=BF16, device=DEV) for _ in range(2)] for _ in range(GLM_LAYERS)]
    _fill(seed, [(f"{i}.{'kv'[q]}", kv[i][q]) for i in range(GLM_LAYERS) for q in range(2)])
    for layer, (k, v) in zip(m.model.layers, kv):
        layer.self_attn.attn.k_cache, layer.self_attn.attn.v_cache = k, v
    seqs, toks = _lengths(case), _tokens(case, seed)
    dev = lambda x, dt: torch.tensor(x, dtype=dt, device=DEV)  # noqa: E731
    pos = [p for start, n in seqs for p in range(start, start + n)]
    slots = [b[p // bs] * bs + p % bs for (start, n), b in zip(seqs, blocks) for p in range(start, start + n)]
    s = dict(model=m, kv=kv, ids=dev([t for row in toks for t in row], torch.int64), pos=dev(pos, torch.int64), slots=dev(slots, torch.int32), graph=None)
    if case["mode"] == "prefill":
        cu = [0]
        for _, n in seqs:
            cu.append(cu[-1] + n)
        s["cu"], s["longest"] = dev(cu, torch.int32), max(n for _, n in seqs)
        return s
    width = max(len(b) for b in blocks)
    s["lens"], s["tables"] = dev([a + n for a, n in seqs], torch.int32), dev([b + [-1] * (width - len(b)) for b in blocks], torch.int32)
    s["fixed"] = {k: s[k].clone() for k in ("ids", "pos", "slots", "lens", "tables")}
    f = s["fixed"]
    set_context(False, slot_mapping=f["slots"], context_lens=f["lens"], block_tables=f["tables"])
    s["graph"], s["hidden"] = _graph(lambda: m(f["ids"], f["pos"]))
    reset_context()
    return s


def _model(case):
    family = case["family"]
    if family == "dafolorn":
        from nanovllm.models.dafolorn.config import read_config
        from nanovllm.models.dafolorn.model import DafolornForCausalLM as Model
    elif family == "napadra":
        from nanovllm.models.napadra.config import read_config
        from nanovllm.models.napadra.model import NapadraForCausalLM as Model
    elif family == "gulozen":
        from nanovllm.models.gulozen.config import read_config
        from nanovllm.models.gulozen.model import GulozenForCausalLM as Model
    else:
        from nanovllm.models.loselix.config import read_config
        from nanovllm.models.loselix.model import LoselixForCausalLM as Model
    with torch.device(DEV):
        return Model(read_config(_config(case)))


def _prepare_step(case, seed):
    from nanovllm.engine.step_batch import Chunk, build_step
    spec = _weights(case)
    m = _model(case)
    with torch.device(DEV):
        m.load_from(lambda prefix: {k: _tensor(seed, k, v) for k, v in spec.items() if k == prefix or k.startswith(prefix + ".")})
    blocks, total, bs = _blocks(case, seed)
    seqs, toks = _lengths(case), _tokens(case, seed)
    m.allocate(total, bs, len(seqs), torch.device(DEV, 0))
    _fill(seed, _buffers(m))
    chunks = [Chunk(t, start, b, 2 * i, 2 * i + 1, [n - 1]) for i, ((start, n), t, b) in enumerate(zip(seqs, toks, blocks))]
    decode = case["mode"] == "decode"
    host, on_device, _ = build_step(chunks, m, bs, **(dict(pad_rows=len(seqs), table_width=max(map(len, blocks))) if decode else {}))
    s = dict(model=m, host=torch.from_numpy(host).pin_memory(), on_device=on_device, buffers=dict(_buffers(m)), graph=None)
    if decode:
        s["buf"] = s["host"].to(DEV)
        meta = on_device(s["buf"])
        s["graph"], s["logits"] = _graph(lambda: m(meta))
    return s


@torch.inference_mode()
def run(s):
    m = s["model"]
    if "kv" not in s:
        if s["graph"] is None:
            return {"logits": m(s["on_device"](s["host"].to(DEV, non_blocking=True))), **s["buffers"]}
        s["buf"].copy_(s["host"], non_blocking=True)
        s["graph"].replay()
        return {"logits": s["logits"].clone(), **s["buffers"]}
    from nanovllm.utils.context import reset_context, set_context
    if s["graph"] is None:
        set_context(True, s["cu"], s["cu"], s["longest"], s["longest"], s["slots"], None, None)
        logits = m.compute_logits(m(s["ids"], s["pos"]))
    else:
        f = s["fixed"]
        for k, t in f.items():
            t.copy_(s[k])
        set_context(False, slot_mapping=f["slots"], context_lens=f["lens"], block_tables=f["tables"])
        s["graph"].replay()
        logits = m.compute_logits(s["hidden"])
    reset_context()
    return {"logits": logits, "kv": s["kv"]}


# ---- what a step cannot do without ------------------------------------------------------------------------------------------------
def _pairs(seqs, window=0, chunk=0):
    """(query-key pairs, cached rows that are read) of one attention layer."""
    pairs = rows = 0
    for start, n in seqs:
        if n == 1:
            seen = start + 1 if not window else min(start + 1, window)
            seen = start % chunk + 1 if chunk else seen
            pairs, rows = pairs + seen, rows + seen - 1
        else:
            p = torch.arange(start, start + n)
            seen = p % chunk + 1 if chunk else p + 1
            pairs += int((seen.clamp(max=window) if window else seen).sum())
    return pairs, rows


def work(case):
    seqs, spec = _lengths(case), _weights(case)
    T, S = sum(n for _, n in seqs), len(seqs)
    nbytes, flops = 4.0 * S * VOCAB, 0.0
    size = lambda v: math.prod(v[0])  # noqa: E731
    runs = {}
    if case["family"] == "glm":
        c = _glm_config(case)
        layers, E, top = GLM_LAYERS, c.n_routed_experts, c.num_experts_per_tok
        expert_bytes = 1 if case.get("experts") == "fp8" else 2
        is_expert, looked_up = (lambda k: ".experts." in k), "model.embed_tokens.weight"
        pairs, rows = _pairs(seqs)
        flops += layers * 4 * pairs * c.num_attention_heads * c.head_dim
        nbytes += layers * (rows + T) * 4 * c.num_key_value_heads * c.head_dim
        head = "lm_head.weight"
    else:
        raw = _config(case)
        loop, L = raw.get("loop"), raw["layers"]
        E, top = (L[0]["mlp"]["router"]["experts"], L[0]["mlp"]["router"]["top"]) if case["family"] == "gulozen" else (1, 1)
        expert_bytes, is_expert, looked_up = 2, (lambda k: ".mlp.e" in k), "embed"
        head = "embed" if case["family"] == "dafolorn" else "head"
        for i, e in enumerate(L):
            s = e["mixer"]
            n = runs[f"l{i}"] = loop["times"] if loop and loop["start"] <= i < loop["stop"] else 1
            H, d, v = s["heads"], s["dim"], s["vdim"]
            if "kv_rank" in s:
                d += s.get("rot_dim", 0)
                pairs, rows = _pairs(seqs, s.get("mask", {}).get("size", 0))
                flops += n * 2 * pairs * H * (d + v)        # of the expanded form; the absorbed form's are more
                nbytes += n * 2 * (rows + T) * (s["kv_rank"] + s.get("rot_dim", 0))
            elif "kv_heads" in s:
                pairs, rows = _pairs(seqs, chunk=s.get("mask", {}).get("size", 0))
                m = 2 if "diff" in s else 1
                row = s["kv_heads"] * (m * d + (0 if e["type"] == "attention_3" else v))
                flops += n * 2 * pairs * H * m * (d + v)
                nbytes += n * 2 * (rows + (T if "kv_from" not in s else 0)) * row
            else:
                flops += 4 * T * H * d * v
                nbytes += 4 * H * d * v * (S + sum(start > 0 for start, _ in seqs))
    touched = E * (1 - (1 - top / E) ** T)
    for name, v in spec.items():
        if name == looked_up:
            nbytes += 2 * T * v[0][1]
        if name == head:
            nbytes, flops = nbytes + 2 * size(v), flops + 2.0 * S * size(v)
        elif is_expert(name):
            nbytes, flops = nbytes + expert_bytes * size(v) * touched / E, flops + 2.0 * T * size(v) * top / E
        elif name != looked_up:
            n = runs.get(name.split(".")[0], 1)             # (a layer that runs twice reads its weights twice)
            nbytes += 2 * n * size(v)
            flops += 2.0 * T * n * size(v) if len(v[0]) == 2 and min(v[0]) > TAPS else 0
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """bfloat16 activations through every projection.  Against 64 bits: GLM (bf16 residual) logits off by 1.1e-2 to 1.8e-2 and single values by up to
    0.077, the others (32-bit residual) by 3e-3 to 8e-3 and 0.049."""
    return {"rel": 3e-2, "max": 0.3} if case["family"] == "glm" else {"rel": 2e-2, "max": 0.2}


# ---- the same step in 64 bits ----------------------------------------------------------------------------------------------------
class _Exact:
    """Sequences of a step, weights, caches and states, all as 64-bit values."""

    def __init__(self, case, seed):
        self.case, self.seed, self.spec = case, seed, _weights(case)
        self.seqs, self.toks = _lengths(case), _tokens(case, seed)
        self.blocks, self.total, self.bs = _blocks(case, seed)
        self.rows, r = [], 0
        for _, n in self.seqs:
            self.rows.append(slice(r, r + n))
            r += n
        self.T = r
        self.ids = torch.tensor([t for row in self.toks for t in row], device=DEV)
        self.pos = torch.cat([torch.arange(a, a + n, device=DEV) for a, n in self.seqs])
        self.last = torch.tensor([s.stop - 1 for s in self.rows], device=DEV)
        self.out = {}

    def w(self, name):
        return _tensor(self.seed, name, self.spec[name]).double()

    def lin(self, x, name):
        return x @ self.w(name).T

    def buffer(self, name, shape, fill=None, dtype=BF16):
        """A cache or a state as it is before the step."""
        t = _randn(self.seed, name, shape, dtype=dtype).double() if fill is None else torch.full(shape, fill, dtype=F64, device=DEV)
        self.out[name] = t
        return t

    def slots(self, i, lo, hi):
        """Cache rows of the tokens lo .. hi-1 of sequence i."""
        p = torch.arange(lo, hi, device=DEV)
        return torch.tensor(self.blocks[i], device=DEV)[p // self.bs] * self.bs + p % self.bs

    def store(self, flat, new):
        """New rows into a cache [tokens, ...]; flat is a view of it."""
        for i, ((start, n), r) in enumerate(zip(self.seqs, self.rows)):
            flat[self.slots(i, start, start + n)] = new[r]

    def keys(self, flat, i, window=0, chunk=0):
        """(rows of the tokens that sequence i sees, visible [its rows, tokens], distances)"""
        start, n = self.seqs[i]
        lo = max(0, start - window + 1) if window else start // chunk * chunk if chunk and n == 1 else 0
        q, k = torch.arange(start, start + n, device=DEV)[:, None], torch.arange(lo, start + n, device=DEV)[None]
        seen = k <= q
        if window:
            seen &= q - k < window
        if chunk:
            seen &= torch.div(q, chunk, rounding_mode="floor") == torch.div(k, chunk, rounding_mode="floor")
        return flat[self.slots(i, lo, start + n)], seen, (q - k).double()

    def conv(self, x, w, state):
        """x + causal convolution; the last inputs go to the state.  state [rows, taps - 1, width], w [width, taps]"""
        out = torch.empty_like(x)
        for i, ((start, n), r) in enumerate(zip(self.seqs, self.rows)):
            front = state[2 * i] if start else torch.zeros_like(state[0])
            z = torch.cat([front, x[r]])
            out[r] = x[r] + sum(z[j: j + n] * w[:, j] for j in range(TAPS))
            state[2 * i + 1] = z[-(TAPS - 1):]
        return out


def _rms(x, eps=EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _softmax(s, seen, sink=None):
    s = s.masked_fill(~seen, -math.inf)
    m = s.amax(-1, keepdim=True)
    m = m if sink is None else torch.maximum(m, sink)
    e = torch.exp(s - m)
    return e / (e.sum(-1, keepdim=True) + (0 if sink is None else torch.exp(sink - m)))


def _rotate(x, pos, freq, half, scale=1.0):
    """Column pairs (i, i + half) or, with half 0, (2i, 2i + 1) turn with frequency i."""
    a = (pos.double()[:, None] * freq).view(-1, *(1,) * (x.dim() - 2), freq.numel())
    c, s, n, out = scale * torch.cos(a), scale * torch.sin(a), 2 * freq.numel(), x.clone()
    i, j = (slice(0, half), slice(half, n)) if half else (slice(0, n, 2), slice(1, n, 2))
    u, v = x[..., i], x[..., j]
    out[..., i], out[..., j] = u * c - v * s, v * c + u * s
    return out


def _freq(base, dims):
    return base ** (-2.0 * torch.arange(dims // 2, dtype=F64, device=DEV) / dims)


def _silu(z):
    return z * torch.sigmoid(z)


@torch.inference_mode()
def exact(case, seed):
    z = _Exact(case, seed)
    if case["family"] == "glm":
        return _exact_glm(z)
    logits = {"dafolorn": _exact_dafolorn, "napadra": _exact_napadra, "gulozen": _exact_gulozen, "loselix": _exact_loselix}[case["family"]](z, _config(case))
    return {"logits": logits, **z.out}


def _exact_glm(z):
    c = _glm_config(z.case)
    H, G, d, E = c.num_attention_heads, c.num_key_value_heads, c.head_dim, c.n_routed_experts
    fp8 = c.expert_weight_dtype is not None

    def stored(name):       # an expert's matrix as it is kept: e4m3 with a factor per row
        w = _tensor(z.seed, name, z.spec[name])
        if not fp8:
            return w.double()
        f = (w.abs().amax(-1, keepdim=True).float() / 448.0).clamp_min(1e-12)
        return (w.float() / f).clamp(-448, 448).to(torch.float8_e4m3fn).double() * f.double()

    def unit(x, p, get):
        g, u = (x @ get(p + "gate_up_proj.weight").T).chunk(2, -1)
        return (_silu(g) * u) @ get(p + "down_proj.weight").T

    x, freq, caches = z.w("model.embed_tokens.weight")[z.ids], _freq(c.rope_theta, d // 2), []
    y = torch.zeros_like(x)
    for i in range(GLM_LAYERS):
        p = f"model.layers.{i}."
        x = x + y
        h = _rms(x) * z.w(p + "input_layernorm.weight")
        q, k, v = (z.lin(h, p + "self_attn.qkv_proj.weight") + z.w(p + "self_attn.qkv_proj.bias")).split([H * d, G * d, G * d], -1)
        q, k, v = _rotate(q.view(-1, H, d), z.pos, freq, d // 4), _rotate(k.view(-1, G, d), z.pos, freq, d // 4), v.view(-1, G, d)
        kc, vc = (z.buffer(f"{i}.{n}", (z.total, z.bs, G, d)) for n in "kv")
        z.store(kc.view(-1, G, d), k), z.store(vc.view(-1, G, d), v)
        caches.append([kc, vc])
        o = torch.empty_like(q)
        for b, r in enumerate(z.rows):
            ks, seen, _ = z.keys(kc.view(-1, G, d), b)
            vs = z.keys(vc.view(-1, G, d), b)[0]
            for g in range(G):
                own = slice(g * H // G, (g + 1) * H // G)
                a = _softmax(q[r, own].transpose(0, 1) @ ks[:, g].T * d ** -0.5, seen)
                o[r, own] = (a @ vs[:, g]).transpose(0, 1)
        x = x + z.lin(o.reshape(-1, H * d), p + "self_attn.o_proj.weight")
        h = _rms(x) * z.w(p + "post_attention_layernorm.weight")
        if i < c.first_k_dense_replace:
            y = unit(h, p + "mlp.", z.w)
            continue
        s = torch.sigmoid(z.lin(h, p + "mlp.gate.weight"))
        best = (s + z.w(p + "mlp.gate.e_score_correction_bias")).topk(c.num_experts_per_tok, -1).indices
        wt = s.gather(-1, best)
        wt = wt / (wt.sum(-1, keepdim=True) + 1e-20) * c.routed_scaling_factor
        y = unit(h, p + "mlp.shared_experts.", stored)
        for e in range(E):
            row, at = (best == e).nonzero(as_tuple=True)
            if row.numel():
                y[row] += unit(h[row], p + f"mlp.experts.{e}.", stored) * wt[row, at, None]
    h = _rms(y) * z.w("model.norm.weight")       # (of the last layer's output alone, as the model has it)
    return {"logits": z.lin(h[z.last], "lm_head.weight"), "kv": caches}


def _exact_latent(z, h, p, s, cache, freq=None, scale=1.0):
    """Heads' outputs of latent attention."""
    H, d, v, r, rd = s["heads"], s["dim"], s["vdim"], s["kv_rank"], s.get("rot_dim", 0)
    q = z.lin(h, p + "q") if not rd else z.lin(_rms(z.lin(h, p + "dq")) * z.w(p + "dq.norm"), p + "uq")
    q = q.view(-1, H, d + rd)
    both = z.lin(h, p + "dkv")
    c = _rms(both[:, :r]) * z.w(p + "dkv.norm")
    if rd:
        q = torch.cat([q[..., :d], _rotate(q[..., d:], z.pos, freq, 0, scale)], -1)
        c = torch.cat([c, _rotate(both[:, r:], z.pos, freq, 0, scale)], -1)
    z.store(cache.view(-1, r + rd), c)
    uk, uv, sink, out = z.w(p + "uk").view(H, d, r), z.w(p + "uv").view(H, v, r), z.w(p + "sink"), torch.empty(z.T, H, v, dtype=F64, device=DEV)
    for b, rows in enumerate(z.rows):
        cs, seen, _ = z.keys(cache.view(-1, r + rd), b, s.get("mask", {}).get("size", 0))
        if rows.stop - rows.start == 1:     # keys stay latents
            qa = torch.cat([(q[rows].transpose(0, 1)[..., :d] @ uk), q[rows].transpose(0, 1)[..., d:]], -1)
            a = _softmax(qa @ cs.T * s["scale"], seen, sink[:, None, None])
            out[rows] = (a @ cs[:, :r] @ uv.transpose(1, 2)).transpose(0, 1)
            continue
        for i in range(H):
            k = torch.cat([cs[:, :r] @ uk[i].T, cs[:, r:]], -1)
            out[rows, i] = _softmax(q[rows, i] @ k.T * s["scale"], seen, sink[i]) @ (cs[:, :r] @ uv[i].T)
    return out.reshape(z.T, H * v)


def _exact_dafolorn(z, raw):
    w, L, loop = raw["width"], raw["layers"], raw["loop"]
    x = x0 = z.w("embed")[z.ids]
    n = 2 * len(z.seqs)

    def layer(i, x, k):
        p, s = f"l{i}.", L[i]["mixer"]
        for q in "12":
            h = z.conv(_rms(x) * (1 + z.w(p + "norm" + q)), z.w(p + "canon" + q), z.buffer(f"{i}.{k}.entry{q}", (n, TAPS - 1, w), dtype=torch.float32))
            if q == "1":
                y = z.lin(_exact_latent(z, h, p + "mix.", s, z.buffer(f"{i}.{k}.keys", (z.total, z.bs, s["kv_rank"]))), p + "mix.o")
            else:
                u, (a, b) = z.lin(h, p + "mlp.up"), torch.nn.functional.softplus(z.w(p + "mlp.act"))
                m = u.clamp(max=0)
                y = z.lin(torch.where(u > 0, a * u * u, (0.5 + b) * (torch.exp(m) - 1 - m)) + 0.5 * u, p + "mlp.down")
            x = x + _rms(y) * (1 + z.w(p + f"norm{q}b"))
        return x

    for i in range(loop["start"]):
        x = layer(i, x, 0)
    for t in range(loop["times"]):
        x = z.lin(torch.cat([x, x0], -1), "loop.in") + z.w("loop.step")[t]
        for i in range(loop["start"], loop["stop"]):
            x = layer(i, x, t)
    for i in range(loop["stop"], len(L)):
        x = layer(i, x, 0)
    y = z.lin((_rms(x) * (1 + z.w("final.norm")))[z.last], "embed")
    return raw["logit_softcap"] * torch.tanh(y / raw["logit_softcap"])


def _grouped(cache):
    """A cache [blocks, groups, tokens of a block, columns] as [tokens, groups, columns]."""
    return cache.transpose(1, 2).reshape(-1, cache.shape[1], cache.shape[3])


def _store_grouped(z, cache, new):
    flat = _grouped(cache)
    z.store(flat, new)
    cache.copy_(flat.view(cache.shape[0], cache.shape[2], cache.shape[1], cache.shape[3]).transpose(1, 2))
    return flat


def _exact_memory(z, h, p, s, i):
    """Heads' outputs of the gated matrix memory."""
    H, d, v, cap, n = s["heads"], s["dim"], s["vdim"], s["gate_cap"], 2 * len(z.seqs)
    S, N, M = (z.buffer(f"{i}.{k}.mixer.state", (n, H, *shape), dtype=torch.float32) for k, shape in enumerate(((d, v), (d,), ())))
    q, k, u = z.lin(h, p + "q").view(-1, H, d) * d ** -0.5, z.lin(h, p + "k").view(-1, H, d), z.lin(h, p + "v").view(-1, H, v)
    gi, gf = (cap * torch.tanh((z.lin(h, p + g) + z.w(p + g + ".b")) / cap) for g in "if")
    gf = torch.nn.functional.logsigmoid(gf)
    out = torch.empty(z.T, H, v, dtype=F64, device=DEV)
    for b, ((start, T), r) in enumerate(zip(z.seqs, z.rows)):
        F = gf[r].cumsum(0)
        zero = lambda t: t[2 * b] if start else torch.zeros_like(t[2 * b])  # noqa: E731
        S0, N0, M0 = zero(S), zero(N), zero(M)
        for a in range(H):
            D = (F[:, None, a] - F[None, :, a] + gi[r][None, :, a]).masked_fill(~torch.ones(T, T, dtype=torch.bool, device=DEV).tril(), -math.inf)
            front = F[:, a] + M0[a]
            m = torch.maximum(D.amax(-1), front)
            A, e = torch.exp(D - m[:, None]) * (q[r, a] @ k[r, a].T), torch.exp(front - m)
            num = A @ u[r, a] + e[:, None] * (q[r, a] @ S0[a])
            den = A.sum(-1) + e * (q[r, a] @ N0[a])
            out[r, a] = num / (torch.maximum(den.abs(), torch.exp(-m)) + 1e-6)[:, None]
            add = torch.exp(D[-1] - m[-1])
            S[2 * b + 1, a] = e[-1] * S0[a] + (k[r, a] * add[:, None]).T @ u[r, a]
            N[2 * b + 1, a], M[2 * b + 1, a] = e[-1] * N0[a] + add @ k[r, a], m[-1]
    return (_rms(out).reshape(z.T, -1) * z.w(p + "norm")) * torch.sigmoid(z.lin(h, p + "g"))


def _exact_napadra(z, raw):
    w, n, kv = raw["width"], 2 * len(z.seqs), {}
    j = torch.arange(w, device=DEV)
    a = z.pos.double()[:, None] * 10000.0 ** (-2.0 * torch.div(j, 2, rounding_mode="floor").double() / w)
    e = z.w("embed")[z.ids] + torch.where(j % 2 == 0, torch.sin(a), torch.cos(a))
    x = torch.stack([e, e], 1)
    for i, entry in enumerate(raw["layers"]):
        p, s = f"l{i}.", entry["mixer"]
        for q in "12":
            h = _rms((x * z.w(p + f"hc{q}.in")[:, None]).sum(1)) * z.w(p + "norm" + q)
            if q == "1":
                state, prev = z.buffer(f"{i}.0.sub1.state", (n, w), dtype=torch.float32), torch.zeros_like(h)
                for b, ((start, _), r) in enumerate(zip(z.seqs, z.rows)):
                    prev[r] = torch.cat([state[2 * b][None] if start else torch.zeros_like(h[:1]), h[r][:-1]])
                    state[2 * b + 1] = h[r][-1]
                h = h + (prev - h) * z.w(p + "shift")
                if entry["type"] == "mlstm":
                    y = _exact_memory(z, h, p + "mix.", s, i)
                else:
                    H, G, d, v = s["heads"], s["kv_heads"], s["dim"], s["vdim"]
                    if "kv_from" in s:
                        kv[i] = kv[s["kv_from"]]
                    else:
                        kv[i] = [_store_grouped(z, z.buffer(f"{i}.0.{t}", (z.total, G, z.bs, m)), z.lin(h, p + "mix." + t[0]).view(-1, G, m))
                                 for t, m in (("keys", d), ("values", v))]
                    qs, sink, y = z.lin(h, p + "mix.q").view(-1, H, d), z.w(p + "mix.sink"), torch.empty(z.T, H, v, dtype=F64, device=DEV)
                    slope = torch.tensor([2.0 ** (-8.0 * (t + 1) / H) for t in range(H)], dtype=F64, device=DEV)
                    for b, r in enumerate(z.rows):
                        ks, seen, dist = z.keys(kv[i][0], b, chunk=s["mask"]["size"])
                        vs = z.keys(kv[i][1], b, chunk=s["mask"]["size"])[0]
                        for g in range(G):
                            own = slice(g * H // G, (g + 1) * H // G)
                            sc = qs[r, own].transpose(0, 1) @ ks[:, g].T * s["scale"] - slope[own, None, None] * dist
                            y[r, own] = (_softmax(sc, seen, sink[own, None, None]) @ vs[:, g]).transpose(0, 1)
                    y = y.reshape(z.T, -1)
                y = z.lin(y, p + "mix.o")
            else:
                lim = entry["mlp"]["limit"]
                g, u = z.lin(h, p + "mlp.gate").clamp(max=lim), z.lin(h, p + "mlp.up").clamp(-lim, lim)
                y = z.lin(g * torch.sigmoid(1.702 * g) * (u + 1), p + "mlp.down")
            y = y * z.w(p + "ls" + q)
            x = torch.einsum("nsw,st->ntw", x, z.w(p + f"hc{q}.mix")) + raw["residual_mult"] * z.w(p + f"hc{q}.out")[:, None] * y[:, None]
    return z.lin((_rms(x.sum(1)) * z.w("final.norm"))[z.last], "head")


def _exact_gulozen(z, raw):
    w, groups, n = raw["width"], raw["norm"]["groups"], 2 * len(z.seqs)
    norm = lambda x, g: _rms(x.view(-1, groups, w // groups)).reshape(-1, w) * g  # noqa: E731
    rot = raw["layers"][0]["mixer"]["rot"]
    dims, sc, f = rot["dims"], rot["scaling"], _freq(rot["base"], rot["dims"])
    at = lambda t: dims * math.log(sc["original"] / (2 * math.pi * t)) / (2 * math.log(rot["base"]))  # noqa: E731
    lo, hi = max(math.floor(at(sc["fast"])), 0), min(math.ceil(at(sc["slow"])), dims - 1)
    ramp = ((torch.arange(dims // 2, dtype=F64, device=DEV) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    freq, scale = f / sc["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(sc["factor"]) + 1
    x = z.w("embed")[z.ids] * raw["embedding"]["scale"]
    X = [x]
    for i, entry in enumerate(raw["layers"]):
        p, s = f"l{i}.", entry["mixer"]
        H, v = s["heads"], s["vdim"]
        h = z.conv(x, z.w(p + "canon1"), z.buffer(f"{i}.0.taps.state", (n, TAPS - 1, w), dtype=torch.float32))
        if entry["type"] == "latent_attention":
            o = _exact_latent(z, h, p + "mix.", s, z.buffer(f"{i}.0.keys", (z.total, z.bs, s["kv_rank"] + s["rot_dim"])), freq, scale)
        else:
            S, d = z.buffer(f"{i}.0.mixer.state", (n, H, s["dim"], v), dtype=torch.float32), s["dim"]
            q, k, u = (_silu(z.lin(h, p + "mix." + t)).view(z.T, H, -1) for t in "qkv")
            o, decay = torch.empty(z.T, H, v, dtype=F64, device=DEV), torch.tensor(s["decay"], dtype=F64, device=DEV)
            for b, ((start, T), r) in enumerate(zip(z.seqs, z.rows)):
                t = torch.arange(T, device=DEV).double()
                for a in range(H):
                    S0 = S[2 * b, a] if start else torch.zeros(d, v, dtype=F64, device=DEV)
                    D = torch.where(t[:, None] >= t, decay[a] ** (t[:, None] - t).clamp(min=0), 0.0)
                    o[r, a] = (D * (q[r, a] @ k[r, a].T)) @ u[r, a] + (decay[a] ** (t + 1))[:, None] * (q[r, a] @ S0)
                    S[2 * b + 1, a] = decay[a] ** T * S0 + (k[r, a] * D[-1][:, None]).T @ u[r, a]
            o = _rms(o.reshape(z.T, -1)) * z.w(p + "mix.norm")
        x = x + norm(z.lin(o * torch.sigmoid(z.lin(h, p + "mix.g")), p + "mix.o"), z.w(p + "norm1"))
        E, top = entry["mlp"]["router"]["experts"], entry["mlp"]["router"]["top"]
        score = torch.softmax(z.lin(x, p + "mlp.router"), -1)
        best, y = score.topk(top, -1).indices, torch.zeros_like(x)
        for t in range(E):
            row = (best == t).any(-1).nonzero().flatten()
            if row.numel():
                q = f"{p}mlp.e{t}."
                y[row] += score[row, t, None] * z.lin(_silu(z.lin(x[row], q + "gate")) * z.lin(x[row], q + "up"), q + "down")
        X.append(x + norm(y, z.w(p + "norm2")))
        x = sum(a * b for a, b in zip(z.w(p + "dwa"), X))
    return z.lin(norm(x, z.w("final.norm"))[z.last], "head")


def _exact_loselix(z, raw):
    L, loop = raw["layers"], raw["loop"]
    e = z.w("embed")[z.ids]
    x = e
    for t in range(loop["times"]):
        x = x + e if t else x
        for i, entry in enumerate(L):
            p, s, kind = f"l{i}.mix.", entry["mixer"], entry["type"]
            H, G, d, v, m = s["heads"], s["kv_heads"], s["dim"], s["vdim"], 2 if "diff" in s else 1
            h = _rms(x) * z.w(f"l{i}.norm1")
            q, k = z.lin(h, p + "q").view(-1, H, m, d), z.lin(h, p + "k")
            cache = lambda name, c: z.buffer(f"{i}.{t}.{name}", (z.total, G, z.bs, c))  # noqa: E731
            if kind == "attention_3":
                raw_k = _store_grouped(z, cache("keys", d), k.view(-1, G, d))
                f = z.buffer(f"{i}.{t}.factors", (z.total, z.bs), fill=1.0)
                z.store(f.view(-1), 1 / torch.sqrt((k * k).mean(-1) + EPS))
                every = torch.div(z.pos + 1, s["q_temp"]["every"], rounding_mode="floor").double()
                q = (_rms(q.reshape(z.T, -1)) * z.w(p + "q.norm") * (1 + s["q_temp"]["coef"] * torch.log(every + 1))[:, None]).view(-1, H, 1, d)
                keys, vals = raw_k * f.view(-1, 1, 1) * z.w(p + "k.norm").view(G, d), raw_k
            else:
                dims = s["rot"]["dims"]
                freq = _freq(s["rot"]["base"], dims)
                q = _rotate(q, z.pos, freq, dims // 2)
                keys = _store_grouped(z, cache("keys", m * d), _rotate(k.view(-1, G, m, d), z.pos, freq, dims // 2).reshape(-1, G, m * d))
                vals = _store_grouped(z, cache("values", v), z.lin(h, p + "v").view(-1, G, v))
            o = torch.empty(z.T, H, v, dtype=F64, device=DEV)
            lam = 0.0 if m == 1 else torch.exp((z.w(p + "lq1") * z.w(p + "lk1")).sum()) - torch.exp((z.w(p + "lq2") * z.w(p + "lk2")).sum()) + s["diff"]
            for b, r in enumerate(z.rows):
                ks, seen, _ = z.keys(keys, b)
                vs = z.keys(vals, b)[0]
                for g in range(G):
                    own = slice(g * H // G, (g + 1) * H // G)
                    a = []
                    for c in range(m):
                        sc = q[r, own, c].transpose(0, 1) @ ks[:, g, c * d: (c + 1) * d].T * s["scale"]
                        if "softcap" in s:
                            sc = s["softcap"] * torch.tanh(sc / s["softcap"])
                        wt = torch.sigmoid(sc + z.w(p + "pb")[own, None, None]) * seen if kind == "attention_3" else _softmax(sc, seen)
                        a.append(wt @ vs[:, g])
                    y = a[0] if m == 1 else _rms(a[0] - lam * a[1]) * (1 - s["diff"])
                    o[r, own] = y.transpose(0, 1)
            if kind == "attention_2":
                o = o * torch.sigmoid(z.lin(h, p + "g"))[..., None]
            o = o.reshape(z.T, -1)
            if kind == "attention_3":
                o = o * torch.sigmoid(z.lin(h, p + "g"))
            x = x + z.lin(o, p + "o") + z.lin(z.lin(h, f"l{i}.mlp.up").clamp(min=0) ** 2, f"l{i}.mlp.down")
    return z.lin((_rms(x) * z.w("final.norm"))[z.last], "head")
