"""The work whose speed this repository answers for: prefill, decode and serving of its decoder designs on one GPU.

A case is one pass of the engine's step function with the sampler behind it (`ModelRunner.step`, `Sampler`), or of a
whole serving job through `Engine.generate`, on a model with random weights.  The designs' sizes are those that
`bench.py` measures (layers of the dense shapes; the other designs at a width of 2,048, vocabulary 32,768, four layers,
which hold every kind of layer in the proportions of a deeper model); `draw` varies width, lengths, batch and type.

Weights are drawn so that a model behaves as a trained one does where it matters for what runs: a token's own direction
stays visible in the residual (sublayers add a fraction of it each), logits have a clear best token, and routers, whose
rows lie along clusters of the token embeddings, choose experts by a clear margin with uneven loads.  (Weights without
any structure would choose experts and tokens by the last bit of a sum, and no two correct programs would agree.)

`exact` computes the same logits by whole sequences in float64 with plain torch.
"""

import math
import queue

import torch

from cwm_amd.cache import CacheManager, CacheStorage
from cwm_amd.config.registry import parse_config
from cwm_amd.engine import Engine, GenArgs, ModelRunner, Packet, Portion, parse_dtype
from cwm_amd.engine.loading import wants_stream_copies
from cwm_amd.models.model import Model
from cwm_amd.parts import PagedKVSpec, StateSpec
from cwm_amd.parts.base import Runtime
from cwm_amd.sampling import Sampler

DEVICE = "cuda:0"
PAGE = 256  # GenArgs.cache_block
MOST_PREFILL = 4096  # GenArgs.max_prefill: tokens of a prompt that one step takes
REWIND = 64  # a decode case's requests go back to their prompts after so many tokens, as if sampled again
CLUSTERS = 32


# ---- the cases ----------------------------------------------------------------------- #
def listed():
    return [
        # one user's chat with a small model: one request, launches and latency are all there is
        {"name": "dense_1b_decode_b1", "design": "dense", "shape": "1b", "layers": 16, "dtype": "bf16", "contexts": "913", "prompts": ""},
        # a burst of short questions to a small model through the whole engine: admission, mixed steps, decode bursts, sampling
        {"name": "dense_1b_engine_12", "design": "dense", "shape": "1b", "layers": 16, "dtype": "bf16", "contexts": "",
         "prompts": "37,512,129,700,64,333,20,801,256,95,410,181", "engine": True, "new": 24},
        # the headline: eight requests of very different lengths, the longest at 32,768 tokens, one period of window and global layers
        {"name": "dense_32b_decode_b8_long", "design": "dense", "shape": "32b", "layers": 4, "dtype": "bf16",
         "contexts": "32767,20011,12288,8193,6000,4097,2500,1023", "prompts": ""},
        # a long document read in portions of 4,096 tokens: the largest
        {"name": "dense_32b_prefill_16k", "design": "dense", "shape": "32b", "layers": 4, "dtype": "bf16", "contexts": "", "prompts": "16384"},
        # continuous batching: 23 requests decode while a new prompt comes in, in one step
        {"name": "dense_8b_mixed_step", "design": "dense", "shape": "8b", "layers": 4, "dtype": "bf16",
         "contexts": "310,2871,777,1500,64,1999,640,1023,2048,415,96,3001,1270,512,888,1713,230,2555,1100,350,1999,47,905", "prompts": "1017"},
        # the 32-bit path: two texts are scored in full precision, the logits of every token wanted
        {"name": "dense_8b_score_fp32", "design": "dense", "shape": "8b", "layers": 2, "dtype": "fp32", "contexts": "", "prompts": "613,130", "score": True},
        # the other designs, prompts and decode steps in turn
        {"name": "lapevik_prefill_2048", "design": "lapevik", "width": 2048, "layers": 4, "dtype": "bf16", "contexts": "", "prompts": "2048"},
        {"name": "segedra_decode_b8", "design": "segedra", "width": 2048, "layers": 4, "dtype": "bf16",
         "contexts": "4095,1300,3777,256,2048,911,3001,64", "prompts": ""},
        {"name": "dogotar_prefill_ragged", "design": "dogotar", "width": 2048, "layers": 4, "dtype": "bf16", "contexts": "", "prompts": "1531,700,65"},
        {"name": "digasun_prefill_1500", "design": "digasun", "width": 2048, "layers": 4, "dtype": "bf16", "contexts": "", "prompts": "1500"},
        {"name": "sunusun_decode_b24", "design": "sunusun", "width": 2048, "layers": 4, "dtype": "bf16",
         "contexts": "1800,650,1201,33,999,512,1440,260,700,1111,90,345,1650,205,801,1337,420,64,1024,577,888,1500,130,256", "prompts": ""},
        {"name": "sorovik_decode_b8", "design": "sorovik", "width": 2048, "layers": 4, "dtype": "bf16",
         "contexts": "4095,1300,3777,256,2048,911,3001,64", "prompts": ""},
    ]


def draw(rng):
    """Another design, width, batch, set of lengths, direction and type of the same ranges."""
    def spread(low, high):  # over the logarithm, odd sizes among them
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    design = rng.choice(["dense", "dense", "lapevik", "segedra", "dogotar", "digasun", "sunusun", "sorovik"])
    case = {"design": design, "dtype": "fp32" if rng.random() < 0.15 else "bf16"}
    if design == "dense":
        case["shape"] = rng.choice(["1b", "8b", "8b", "32b"])
        case["layers"] = {"1b": 16, "8b": 4, "32b": 4}[case["shape"]]
    else:
        case["width"], case["layers"] = rng.choice([1024, 1536, 2048, 3072]), 4
    most = 1024 if case["dtype"] == "fp32" else 4096
    lengths = lambda n, low, high: ",".join(str(spread(low, high)) for _ in range(n))  # noqa: E731
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "mixed"])
    case["contexts"], case["prompts"] = "", ""
    if kind != "prefill":
        case["contexts"] = lengths(spread(1, 16 if case["dtype"] == "fp32" else 48), 16, most // 2)
    if kind != "decode":
        n = spread(1, 6)
        case["prompts"] = lengths(n, 16, most // n)
        if sum(numbers(case["prompts"])) <= 1024 and rng.random() < 0.3:
            case["score"] = True  # the logits of every token of the prompts
    return case


def numbers(text):
    return [int(part) for part in text.split(",") if part]


# ---- configurations ------------------------------------------------------------------- #
DENSE = {
    "1b": dict(dim=2048, n_heads=32, head_dim=64, ffn_dim_multiplier=1.5, multiple_of=256, max_seq_len=131072),
    "8b": dict(dim=4096, n_heads=32, head_dim=128, ffn_dim_multiplier=1.3, multiple_of=1024, max_seq_len=8192),
    "32b": dict(dim=6144, n_heads=48, head_dim=128, ffn_dim_multiplier=1.3125, multiple_of=256, max_seq_len=131072, vocab_size=32768,
                pos_embed_impl="scaled_rope", rope_theta=1000000.0,
                scaled_rope={"scale_factor": 16, "old_context_len": 8192, "low_freq_factor": 1, "high_freq_factor": 4},
                window_attn={"window_pattern": 4, "local_window": 8192, "global_last_layer": True}),
}


def config_of(case):
    design, layers = case["design"], case["layers"]
    if design == "dense":
        config = dict(architecture="llama3_dense", n_layers=layers, n_kv_heads=8, vocab_size=128256, norm_eps=1e-5,
                      pos_embed_impl="rope", rope_theta=500000.0)
        config.update(DENSE[case["shape"]])
        if "window_attn" in config:
            config["layer_types"] = ["global" if i % 4 == 3 else "local" for i in range(layers)]
        return config
    width = case["width"]
    heads, experts = width // 128, 16 if width <= 2048 else 32
    kv_heads = 8 if heads % 8 == 0 else 4
    ff = width // 2
    attention = {"heads": heads, "kv_heads": kv_heads, "dim": 128, "vdim": 128, "scale": 128 ** -0.5}
    half, router = {"base": 10000.0, "dims": 64}, {"experts": experts, "top": 4}
    latent = {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 192, "scale": 192 ** -0.5, "rot": half}
    config = {"vocab": 32768, "width": width}
    if design == "lapevik":
        mlp = {"kind": "moe", "expert": {"ff": ff}, "router": router}
        space = {"heads": width // 32, "vdim": 64, "state": 128, "groups": 8, "norm_groups": 8, "conv": 4}
        kinds = [{"type": "mamba2", "mixer": space, "mlp": mlp}] * 3 + [{"type": "latent_attention", "mixer": dict(latent, q_rank=3 * width // 8), "mlp": mlp}]
        config.update(architecture="Lapevik", norm={"eps": 1e-5, "groups": 4})
    elif design == "segedra":
        mixer = dict(attention, mask={"size": 8192}, rot={"base": 500000.0, "dims": 128})
        moe = {"kind": "moe", "expert": {"ff": ff, "limit": 7.0}, "router": dict(router, scale=1.0)}
        kinds = [{"type": "attention", "mixer": mixer, "mlp": {"kind": "dense", "ff": 2 * width}}] + [{"type": "attention", "mixer": mixer, "mlp": moe}] * 3
        config.update(architecture="Segedra", norm={"eps": 1e-6}, embedding={"scale": 1.0}, streams=4)
    elif design == "dogotar":
        mlp = {"kind": "dense", "ff": 3 * width}
        around = dict(attention, softcap=30.0, mask={"size": 8192}, rot=dict(half, scaling={"factor": 4.0}), v_mix=True)
        beside = {"left": dict(attention, softcap=30.0, mask={"size": 2048}), "right": {"heads": heads, "dim": 128, "vdim": 128, "gate_cap": 15.0},
                  "left_scale": 1.0, "right_scale": 1.0}
        outer, inner = {"type": "attention", "mixer": around, "mlp": mlp}, {"type": "parallel", "mixer": beside, "mlp": mlp}
        kinds = [outer, inner, inner, outer]
        config.update(architecture="Dogotar", norm={"eps": 1e-5})
    elif design == "digasun":
        moe = {"kind": "moe", "expert": {"ff": ff}, "router": router, "shared": {"ff": ff}}
        dense = {"kind": "dense", "ff": 5 * width // 2, "limit": 7.0}
        mixer = dict(attention, mask={"size": 8192}, rot=half)
        kinds = [{"type": "attention", "mixer": mixer, "mlp": dense}, {"type": "attention", "mixer": dict(mixer, kv_from=0), "mlp": moe},
                 {"type": "gla", "mixer": {"heads": heads, "dim": 128, "vdim": 128, "tau": 8.0}, "mlp": moe}, {"type": "attention", "mixer": mixer, "mlp": moe}]
        config.update(architecture="Digasun", norm={"eps": 1e-6}, embedding={"scale": 1.0}, canon={"taps": 4}, token_side={"dim": 64})
    elif design == "sunusun":
        mlp = {"kind": "dense", "ff": 3 * width}
        beside = {"type": "parallel", "mixer": {"left": dict(attention, q_temp={"coef": 0.1, "every": 4096}), "right": {"width": width}}, "mlp": mlp}
        wkv = {"type": "wkv", "mixer": {"heads": width // 64, "dim": 64}, "mlp": mlp}
        kinds = [beside, wkv, wkv, beside]
        config.update(architecture="Sunusun", norm={"eps": 1e-5}, logit_scale=1.0)
    else:
        moe = {"kind": "moe", "expert": {"ff": ff}, "router": dict(router, groups={"count": experts // 4, "keep": experts // 8})}
        dense = {"kind": "dense", "ff": 2 * width}
        through = dict(latent, mask={"size": 8192})
        convolved = dict(attention, conv=3, mask={"size": 8192, "keep_first": 16}, rot=half)
        kinds = [{"type": "latent_attention", "mixer": through, "mlp": dense}, {"type": "latent_attention", "mixer": dict(through, kv_from=0), "mlp": moe},
                 {"type": "attention", "mixer": convolved, "mlp": moe}, {"type": "latent_attention", "mixer": through, "mlp": moe}]
        config.update(architecture="Sorovik", norm={"eps": 1e-6})
    config["layers"] = [kinds[i % 4] for i in range(layers)]
    return config


def vocab_of(config):
    return config["vocab_size"] if "vocab_size" in config else config["vocab"]


# ---- weights and tokens, from the seed alone -------------------------------------------- #
def draw_weights(config, specs, seed, act_dtype):
    """Tensors by name, as a loaded folder gives them: matrices in the model's type, what is stored in 32 bits in 32 bits."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    normal = lambda shape, std=1.0: torch.randn(shape, generator=gen, device=DEVICE) * std  # noqa: E731
    uniform = lambda shape, low, high: torch.rand(shape, generator=gen, device=DEVICE) * (high - low) + low  # noqa: E731
    design = config["architecture"]
    dense = design == "llama3_dense"
    width, vocab = config["dim"] if dense else config["width"], vocab_of(config)
    tied = "head" not in specs and not dense
    centres = normal((CLUSTERS, width))
    sharpness = 16.0 / (0.7 * width)  # the best token's logit is about 16
    if dense:
        table = normal((vocab, width))
    else:
        table = (centres[torch.randint(CLUSTERS, (vocab,), generator=gen, device=DEVICE)] + normal((vocab, width))) * 0.5 ** 0.5
    uniform_ranges = {"mix.dt_bias": (-2, 0), "mix.A_log": (-4, -1), "mix.left.r1": (0.2, 1), "mix.left.r2": (0.01, 0.3), "mix.right.z.b": (-4, 0),
                      "mix.w0": (-6, -1), "mix.a2.b": (0, 4), "mix.right.f.b": (1, 4), "shift": (0, 1), "mix.vmix": (0.3, 0.3)}
    stds = {"mix.conv": 0.5, "mix.conv.b": 0.2, "canon1": 0.1, "canon2": 0.1, "mix.q.conv": 0.6, "mix.k.conv": 0.6, "mix.sink": 1.0,
            "mlp.correction": 0.01, "mix.right.i.b": 1.0, "mix.right.x.b": 0.5, "mix.u": 0.5, "mlp.router.b": 0.1, "side.embed": 1.0}
    after = {"lapevik": ("norm1", "norm2"), "sorovik": ("norm1b", "norm2b"), "digasun": ("side.norm",), "sunusun": ("mix.left.out", "mix.right.out")}.get(design.lower(), ())
    choices = None
    out = {}
    for name, spec in specs.items():
        shape = spec.drawn_shape()
        local = name
        if name.startswith("layers."):
            local = name.split(".", 2)[2]
        elif name[0] == "l" and name.split(".")[0][1:].isdigit():
            local = name.split(".", 1)[1]
        last = local.rsplit(".", 1)[-1]
        if name in ("embed", "tok_embeddings.weight"):
            t = table
        elif name in ("head", "output.weight"):  # every token has one that follows it
            t = torch.empty_like(table)
            t[torch.randperm(vocab, generator=gen, device=DEVICE)] = table * sharpness
        elif name in ("final.norm", "norm.weight"):
            t = uniform(shape, 0.8, 1.2) * (sharpness if tied else 1.0) - (1.0 if design == "Segedra" else 0.0)
        elif name == "final.norm.b":
            t = normal(shape, 0.1 * (sharpness if tied else 1.0))
        elif local == "mlp.router":
            # a cluster's tokens choose four experts, two neighbours out of each of two groups of four: shares of 1 and more, the others' near 0
            n, top = shape[0], 4
            order = torch.rand((CLUSTERS, n // 4), generator=gen, device=DEVICE).argsort(-1)[:, :2]
            member = torch.rand((CLUSTERS, 2, 4), generator=gen, device=DEVICE).argsort(-1)[:, :, :2]
            chosen = (order[..., None] * 4 + member).reshape(CLUSTERS, top)
            choices = torch.zeros((CLUSTERS, n), device=DEVICE).scatter(1, chosen, 1.0 + 0.1 * torch.arange(top, device=DEVICE).expand(CLUSTERS, top))
            t = choices.T @ centres * (5.0 / width) + normal(shape, 0.02 * width ** -0.5)
        elif local in uniform_ranges:
            t = uniform(shape, *uniform_ranges[local])
        elif local in stds:
            t = normal(shape, stds[local])
        elif local == "mix.D":
            t = 1.0 + normal(shape, 0.5)
        elif local.startswith("mix.mu."):
            t = uniform(shape, 0, 1)
        elif local == "mix.talk":
            t = 0.8 * torch.eye(shape[0], device=DEVICE) + normal(shape, 0.1)
        elif local.startswith("hc"):
            t = (torch.eye(shape[0], device=DEVICE) if last == "mix" else torch.ones(shape, device=DEVICE) * (1.0 if last == "out" else 0.25)) + normal(shape, 0.05)
        elif design == "Segedra" and local in ("norm1", "norm2"):
            t = normal(shape, 0.1)
        elif spec.init == "norm":
            t = uniform(shape, 0.8, 1.2) * (0.35 if local in after else 1.0)
        elif len(shape) == 2:
            leaves = last in ("o", "down") or local.endswith(("wo.weight", "w2.weight"))
            t = normal(shape, shape[1] ** -0.5 * (0.5 if leaves else 1.0))
        else:
            t = normal(shape, 0.1)
        out[name] = t.to(act_dtype if spec.precision == "activation" else torch.float32)
    return out


def draw_tokens(case, seed):
    """(tokens cached of every decoding request and the one it runs now, the new prompts) as lists."""
    gen = torch.Generator().manual_seed(seed ^ 0x5EED)
    vocab = vocab_of(config_of(case))
    some = lambda n: torch.randint(vocab, (n,), generator=gen).tolist()  # noqa: E731
    return [some(n + 1) for n in numbers(case["contexts"])], [some(n) for n in numbers(case["prompts"])]


def model_of(case, seed):
    """(plan's model with nothing in it, its configuration, its tensors)."""
    config = config_of(case)
    arch, typed = parse_config(config)
    model = Model(arch.build_plan(typed))
    return model, config, draw_weights(config, model.tensor_specs(), seed, parse_dtype(case["dtype"]))


# ---- what a program has in hand, and a pass --------------------------------------------- #
@torch.inference_mode()
def prepare(case, seed):
    model, config, tensors = model_of(case, seed)
    device, act_dtype = torch.device(DEVICE), parse_dtype(case["dtype"])
    model.bind(tensors, Runtime(device=device, act_dtype=act_dtype, stream_copies=wants_stream_copies(model, act_dtype, device)))
    cached, prompts = draw_tokens(case, seed)
    state = {"case": case, "model": model, "prompts": prompts}
    if case.get("engine"):
        most = sum(len(p) + case["new"] + 2 * PAGE for p in prompts)
        state["engine"] = Engine(GenArgs(temperature=0.7, top_p=0.95, max_batch=len(prompts), max_seq=most), model)
        return state
    pages = sum((n + PAGE - 1) // PAGE + 1 for n in [len(t) + REWIND for t in cached] + [len(p) for p in prompts])
    manager = CacheManager(model.cache_specs, PAGE, pages, len(cached) + len(prompts))
    storage = CacheStorage(manager, device, act_dtype)
    runner = ModelRunner(model, manager, storage, num_graphs=16, graphs_where_host_bound=True)  # as the engine's defaults
    rids = [("cached", i) for i in range(len(cached))]
    for rid, tokens in zip(rids, cached):
        runner.admit(rid)
        if len(tokens) > 1:
            assert manager.extend(rid, len(tokens) - 1)
    for rid, tokens in zip(rids, cached):
        for at in range(0, len(tokens) - 1, MOST_PREFILL):
            runner.step([Portion(rid, tokens[at : min(at + MOST_PREFILL, len(tokens) - 1)])])
    n = len(cached) + (sum(len(p) for p in prompts) if case.get("score") else len(prompts))
    params = torch.zeros((3, n), dtype=torch.float32, device=device)
    params[0], params[1] = 0.7, 0.95
    params[2] = torch.rand(n, generator=torch.Generator().manual_seed(seed)) * 0.9
    state.update(
        runner=runner, manager=manager, sampler=Sampler(device), params=params, rids=rids, last=[t[-1] for t in cached], lengths=[len(t) - 1 for t in cached],
        decoded=0, tokens_device=torch.tensor([t[-1] for t in cached], dtype=torch.int32, device=device),
    )
    return state


def rewind(state):
    """The decoding requests go back to their prompts.  They get the pages they had: the same ones are free, lowest first."""
    manager, rids = state["manager"], state["rids"]
    for rid in reversed(rids):
        manager.release(rid)
    for rid, n in zip(rids, state["lengths"]):
        manager.admit(rid)
        assert manager.extend(rid, n)
    for rid, n in zip(rids, state["lengths"]):
        manager.advance(rid, n)
    state["decoded"] = 0


@torch.inference_mode()
def run(state):
    if "engine" in state:
        requests = queue.Queue()
        for i, prompt in enumerate(state["prompts"]):
            requests.put(Packet(thread_id=i, tokens=prompt, max_gen=state["case"]["new"]))
        requests.put(None)
        tokens = {packet.thread_id: packet.tokens for packet in state["engine"].generate(requests) if packet is not None}
        return {"tokens": [torch.tensor(tokens[i]) for i in range(len(tokens))]}
    runner, manager, rids = state["runner"], state["manager"], state["rids"]
    prompts, score = state["prompts"], state["case"].get("score")
    if rids and state["decoded"] == REWIND:
        rewind(state)
    state["decoded"] += 1
    for rid in rids:
        assert manager.extend(rid, 1)
    if not prompts:  # a decode step, fed from the device as in a burst of them
        logits = runner.step([Portion(rid, [0], [0]) for rid in rids], tokens_device=state["tokens_device"])
    else:
        new = [("new", i) for i in range(len(prompts))]
        ends = [0] * len(prompts)
        for rid in new:
            runner.admit(rid)
        portions = [Portion(rid, [token], [0]) for rid, token in zip(rids, state["last"])]
        while True:
            room = MOST_PREFILL
            for i, prompt in enumerate(prompts):
                take = min(room, len(prompt) - ends[i])
                if take > 0:
                    assert manager.extend(new[i], take)
                    ends[i] += take
                    room -= take
                    portions.append(Portion(new[i], prompt[ends[i] - take : ends[i]], list(range(take)) if score else [take - 1] if ends[i] == len(prompt) else []))
            logits = runner.step(portions)
            if all(end == len(prompt) for end, prompt in zip(ends, prompts)):
                break
            portions = []
        for rid in new:
            runner.release(rid)
    packed = state["sampler"].sample_packed(logits, state["params"][0], state["params"][1], state["params"][2])
    return {"logits": logits, "tokens": packed[0]}


# ---- what a pass cannot do without --------------------------------------------------------- #
def work(case):
    """Bytes: every weight that some token meets once (of routed experts the share that so many tokens choose), the rows of
    the embedding, cached keys and values that the new tokens read, those they write, states in and out, the logits.
    Operations: two for every matrix entry and token, and the attention's two products."""
    config = config_of(case)
    arch, typed = parse_config(config)
    model = Model(arch.build_plan(typed))
    size = 2 if case["dtype"] == "bf16" else 4
    cached, prompts = numbers(case["contexts"]), numbers(case["prompts"])
    steps = case["new"] if case.get("engine") else 1
    rows = [(n, 1) for n in cached] + [(0, n) for n in prompts]  # (tokens before, new tokens) of every request
    tokens = sum(n for _, n in rows)
    wanted = tokens if case.get("score") else len(rows)
    weights, active, head = 0.0, 0.0, 0
    layers = config.get("layers")
    for name, spec in model.tensor_specs().items():
        shape = spec.drawn_shape()
        count = math.prod(shape)
        if name in ("embed", "tok_embeddings.weight", "side.embed"):
            if name == "embed" and "head" not in model.tensor_specs():
                weights, head = weights + count * size, count
            continue
        parts = name.split(".")
        if layers is not None and len(parts) > 2 and parts[1] == "mlp" and parts[2][0] == "e" and parts[2][1:].isdigit():
            share = 4 / layers[int(parts[0][1:])]["mlp"]["router"]["experts"]
            weights += count * size * (1 - (1 - share) ** tokens)
            active += count * share
        else:
            weights += count * size
            if name in ("head", "output.weight"):
                head = count
            elif len(shape) == 2:
                active += count
    width = model.dim
    total_bytes = weights * steps + tokens * width * size + 4 * wanted * model.vocab_size
    total_flops = 2.0 * active * tokens + 2.0 * head * wanted
    for call, slots, writes in zip(model.run_order, model.cache_slots, model.writes_cache):
        for m, (mixer, slot) in enumerate(zip(model.blocks[call.layer].mixers(), slots)):
            spec = model.cache_specs[slot]
            writes_one = writes if isinstance(writes, bool) else writes[m]
            if isinstance(spec, PagedKVSpec):
                token = spec.bytes_per_token(size)
                span = spec.keys_kept(1)
                for before, n in rows:
                    here = lambda p: p + 1 if span is None else min(p + 1, span)  # noqa: E731
                    read = min(before, here(before + n - 1))
                    total_bytes += token * (read + (n if writes_one else 0))
                    keys = n * (here(before) + here(before + n - 1)) / 2
                    total_flops += 4.0 * keys * getattr(mixer, "n_heads", spec.n_kv_heads) * spec.head_dim
            elif isinstance(spec, StateSpec):
                one = math.prod(spec.shape) * torch.empty((), dtype=spec.dtype).element_size()
                total_bytes += one * (2 * len(cached) + len(prompts))
                total_flops += 4.0 * math.prod(spec.shape) * tokens
    if case.get("engine"):  # the tokens that it decodes, one step of all requests after the other
        total_flops += (steps - 1) * (2.0 * active + 2.0 * head) * len(rows)
    return {"bytes": int(total_bytes), "flops": int(total_flops)}


def tolerance(case):
    if case.get("engine"):
        return {"differ": 0.005}
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "differ": 0.005}
    # measured against `exact`: 0.005 for 16 dense layers, 0.003 for four, 0.001 for four of the other designs, whose
    # embeddings carry more of the residual
    return {"rel": 0.02 if case["layers"] > 4 else 0.012 if case["design"] == "dense" else 0.006, "differ": 0.005}


# ---- the same in float64, by whole sequences ------------------------------------------------- #
F = torch.float64


def unit(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def layer_norm(x, g, b, eps):
    x = x - x.mean(-1, keepdim=True)
    return unit(x, eps) * g + b


def group_unit(x, groups, eps):
    return unit(x.unflatten(-1, (groups, -1)), eps).flatten(-2)


def silu(x):
    return x * torch.sigmoid(x)


def gelu_tanh(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def before(x):
    """The token before each one's, zeros before the first."""
    return torch.nn.functional.pad(x, (0, 0, 1, 0))[:, :-1]


def causal_conv(x, w):
    """[B, T, C] with taps [C, n]: the newest input meets the last tap."""
    out = x * w[:, -1]
    for lag in range(1, w.shape[1]):
        x = before(x)
        out = out + x * w[:, w.shape[1] - 1 - lag]
    return out


def turn(x, angles, pairs):
    """[B, T, H, d]: the first 2 * angles' width elements of every head, paired by neighbours or by halves."""
    n = angles.shape[-1]
    c, s = torch.cos(angles)[None, :, None], torch.sin(angles)[None, :, None]
    if pairs == "neighbours":
        a, b = x[..., 0 : 2 * n : 2], x[..., 1 : 2 * n : 2]
        turned = torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)
    else:
        a, b = x[..., :n], x[..., n : 2 * n]
        turned = torch.cat([a * c - b * s, b * c + a * s], -1)
    return torch.cat([turned, x[..., 2 * n :]], -1)


def plain_angles(n, rot):
    half = rot["dims"] // 2
    freqs = rot["base"] ** (-2.0 * torch.arange(half, dtype=F, device=DEVICE) / rot["dims"]) / (rot.get("scaling") or {}).get("factor", 1.0)
    return torch.arange(n, dtype=F, device=DEVICE)[:, None] * freqs


def dense_angles(n, config):
    """This design's angles are float32 by definition: a float32 table of frequencies times the position."""
    d = config["head_dim"]
    freqs = 1.0 / (config["rope_theta"] ** (torch.arange(0, d, 2).float() / d))
    if config["pos_embed_impl"] == "scaled_rope":
        r = config["scaled_rope"]
        for i, f in enumerate(freqs.tolist()):
            length = 2 * math.pi / f
            if length > r["old_context_len"] / r["low_freq_factor"]:
                freqs[i] = f / r["scale_factor"]
            elif length >= r["old_context_len"] / r["high_freq_factor"]:
                x = (r["old_context_len"] / length - r["low_freq_factor"]) / (r["high_freq_factor"] - r["low_freq_factor"])
                freqs[i] = (1 - x) * f / r["scale_factor"] + x * f
    return (torch.arange(n, dtype=torch.float32, device=DEVICE)[:, None] * freqs.to(DEVICE)).to(F)


def attend(q, k, v, scale, size=None, keep=0, block=None, cap=None, sink=None, bias=None, talk=None):
    """q [B, T, H, d], k [B, T, G, d], v [B, T, G, e] -> [B, T, H, e]: query i reads keys j <= i within `size` (or among the
    first `keep`), or of its own block; the softmax's denominator has exp(sink) beside the keys; `talk` mixes heads' weights."""
    nb, n, heads, _ = q.shape
    groups = k.shape[2]
    per = heads // groups
    out = torch.empty(nb, n, heads, v.shape[-1], dtype=F, device=DEVICE)
    kt, vt = k.permute(0, 2, 3, 1).contiguous(), v.permute(0, 2, 1, 3).contiguous()  # [B, G, d, T], [B, G, T, e]
    chunk = max(16, min(n, int(6e7) // (nb * heads * n)))
    for i in range(0, n, chunk):
        j = min(n, i + chunk)
        low = 0 if size is None or keep else max(0, i - size + 1)
        at, key = torch.arange(i, j, device=DEVICE)[:, None], torch.arange(low, j, device=DEVICE)[None]
        seen = key <= at
        if size is not None:
            seen = seen & ((at - key < size) | (key < keep))
        if block is not None:
            seen = seen & (at // block == key // block)
        rows = q[:, i:j].reshape(nb, j - i, groups, per, -1).permute(0, 2, 3, 1, 4).reshape(nb, groups, per * (j - i), -1)
        s = (rows @ kt[..., low:j]).reshape(nb, heads, j - i, j - low) * scale
        if cap is not None:
            s = cap * torch.tanh(s / cap)
        if bias is not None:
            r1, r2 = (t[:, None, None] for t in bias)
            s = s - r1 * torch.log1p(r2 * (at - key).clamp(min=0).to(F))
        s = s.masked_fill(~seen, -math.inf)
        top = s.amax(-1, keepdim=True)
        if sink is not None:
            top = torch.maximum(top, sink[:, None, None])
        e = torch.exp(s - top)
        total = e.sum(-1, keepdim=True)
        if sink is not None:
            total = total + torch.exp(sink[:, None, None] - top)
        p = e / total
        if talk is not None:
            p = (talk @ p.flatten(2)).reshape(p.shape)
        mixed = p.reshape(nb, groups, per * (j - i), j - low) @ vt[:, :, low:j]
        out[:, i:j] = mixed.reshape(nb, groups, per, j - i, -1).permute(0, 3, 1, 2, 4).reshape(nb, j - i, heads, -1)
    return out


class Plain:
    """The decoder of a configuration on [B, T] tokens; what follows a sequence's end does not reach back."""

    def __init__(self, config, tensors):
        self.config, self.w = config, tensors
        self.design = config["architecture"].lower()

    def __call__(self, tokens, ends, score=None):
        """Logits [B, V] of the tokens before `ends`, or of all tokens between `score` and there."""
        x = getattr(self, self.design)(tokens, self.config)
        if score:
            x = torch.cat([x[i, first:end] for i, (first, end) in enumerate(zip(score, ends))])
        else:
            x = x[torch.arange(len(ends), device=DEVICE), torch.tensor(ends, device=DEVICE) - 1]
        return self.final(x)

    def t(self, name):
        return self.w[name].to(F)

    def mul(self, x, name):
        y = x @ self.t(name).T
        return y + self.t(name + ".b") if name + ".b" in self.w else y

    def heads(self, x, name, n):
        return self.mul(x, name).unflatten(-1, (n, -1))

    def final(self, x):
        d, eps = self.design, self.config["norm_eps"] if self.design == "llama3_dense" else self.config["norm"]["eps"]
        if d == "llama3_dense":
            return (unit(x, eps) * self.t("norm.weight")) @ self.t("output.weight").T
        g = self.t("final.norm")
        if d in ("dogotar", "digasun"):
            x = layer_norm(x, g, self.t("final.norm.b"), eps)
        elif d == "lapevik":
            x = group_unit(x, self.config["norm"]["groups"], eps) * g
        elif d == "segedra":
            x = unit(x, eps) * (1 + g)
        else:
            x = unit(x, eps) * g * self.config.get("logit_scale", 1.0)
        return x @ self.t("head" if "head" in self.w else "embed").T

    # -- feed-forwards
    def experts(self, h, p, chosen, share, act):
        """chosen, share [rows, top] for h [rows, D]."""
        out = torch.zeros_like(h)
        for e in range(int(chosen.max()) + 1):
            rows, place = torch.nonzero(chosen == e, as_tuple=True)
            if rows.numel():
                q = f"{p}e{e}."
                out[rows] += share[rows, place][:, None] * (act(self.mul(h[rows], q + "gate"), self.mul(h[rows], q + "up")) @ self.t(q + "down").T)
        return out

    def routed(self, x, p, mlp, rule, act):
        h = x.flatten(0, 1)
        chosen, share = rule(self.mul(h, p + "router"))
        return self.experts(h, p, chosen, share, act).reshape(x.shape)

    @staticmethod
    def top_softmax(top):
        def rule(z):
            best = torch.topk(z, top, -1)
            return best.indices, torch.softmax(best.values, -1)
        return rule

    # -- the designs
    def llama3_dense(self, tokens, c):
        x, n, eps = self.t("tok_embeddings.weight")[tokens], tokens.shape[1], c["norm_eps"]
        angles = dense_angles(n, c)
        for i in range(c["n_layers"]):
            p = f"layers.{i}."
            h = unit(x, eps) * self.t(p + "attention_norm.weight")
            q, k, v = (self.heads(h, p + f"attention.w{r}.weight", m) for r, m in (("q", c["n_heads"]), ("k", c["n_kv_heads"]), ("v", c["n_kv_heads"])))
            q, k = turn(q, angles, "neighbours"), turn(k, angles, "neighbours")
            size = c["window_attn"]["local_window"] if c.get("layer_types", ["global"] * c["n_layers"])[i] == "local" else None
            x = x + self.mul(attend(q, k, v, c["head_dim"] ** -0.5, size=size).flatten(-2), p + "attention.wo.weight")
            h = unit(x, eps) * self.t(p + "ffn_norm.weight")
            x = x + self.mul(silu(self.mul(h, p + "feed_forward.w1.weight")) * self.mul(h, p + "feed_forward.w3.weight"), p + "feed_forward.w2.weight")
        return x

    def lapevik(self, tokens, c):
        eps, groups = c["norm"]["eps"], c["norm"]["groups"]
        x = group_unit(self.t("embed")[tokens], groups, eps) * self.t("embed.norm")
        for i, layer in enumerate(c["layers"]):
            p, m = f"l{i}.", layer["mixer"]
            s = x + (before(x) - x) * self.t(p + "shift")
            y = self.state_space(s, p + "mix.", m, eps) if layer["type"] == "mamba2" else self.latent_gated(s, p + "mix.", m, eps)
            x = x + group_unit(y, groups, eps) * self.t(p + "norm1")
            y = self.routed(x, p + "mlp.", layer["mlp"], self.top_softmax(4), lambda g, u: silu(g) * u)
            x = x + group_unit(y, groups, eps) * self.t(p + "norm2")
        return x

    def state_space(self, s, p, m, eps):
        heads, vdim, state, groups = m["heads"], m["vdim"], m["state"], m["groups"]
        inner, gn = heads * vdim, groups * state
        z, xbc, dt = self.mul(s, p + "in").split([inner, inner + 2 * gn, heads], -1)
        xbc = silu(causal_conv(xbc, self.t(p + "conv")) + self.t(p + "conv.b"))
        xs, b, cc = xbc.split([inner, gn, gn], -1)
        xs = xs.unflatten(-1, (heads, vdim))
        b, cc = (t.unflatten(-1, (groups, state)).repeat_interleave(heads // groups, 2) for t in (b, cc))
        dt = torch.nn.functional.softplus(dt + self.t(p + "dt_bias"))
        decay = torch.exp(-torch.exp(self.t(p + "A_log")) * dt)
        y = linear_scan(cc, b * dt[..., None], xs, decay[..., None]) + self.t(p + "D")[:, None] * xs
        y = y.flatten(-2) * silu(z)
        return self.mul(group_unit(y, m["norm_groups"], eps) * self.t(p + "norm"), p + "o")

    def latent_gated(self, s, p, m, eps):
        n = s.shape[1]
        q = self.heads(unit(self.mul(s, p + "dq"), eps) * self.t(p + "dq.norm"), p + "uq", m["heads"])
        down = self.mul(s, p + "dkv")
        mixed = self.through_latent(q, unit(down[..., : m["kv_rank"]], eps) * self.t(p + "dkv.norm"),
                                    turn(down[:, :, None, m["kv_rank"] :], plain_angles(n, m["rot"]), "neighbours"), p, m, "neighbours")
        return self.mul(mixed * torch.sigmoid(self.mul(s, p + "g")), p + "o")

    def through_latent(self, q, latent, key_part, p, m, pairs, **more):
        n, heads, dim = q.shape[1], m["heads"], m["dim"]
        q = torch.cat([q[..., :dim], turn(q[..., dim:], plain_angles(n, m["rot"]), pairs)], -1)
        k = torch.cat([self.heads(latent, p + "uk", heads), key_part.expand(-1, -1, heads, -1)], -1)
        return attend(q, k, self.heads(latent, p + "uv", heads), m["scale"], **more).flatten(-2)

    def segedra(self, tokens, c):
        eps = c["norm"]["eps"]
        streams = self.t("embed")[tokens][None].repeat(c["streams"], 1, 1, 1) * c["embedding"]["scale"]

        def rule(z):
            scores = torch.softmax(z, -1)
            chosen = torch.topk(scores + self.t(p + "mlp.correction"), 4, -1).indices
            return chosen, torch.gather(scores, 1, chosen)

        for i, layer in enumerate(c["layers"]):
            p, m, limit = f"l{i}.", layer["mixer"], layer["mlp"].get("expert", {}).get("limit")
            for number in (1, 2):
                u = torch.einsum("s,sbnd->bnd", self.t(p + f"hc{number}.in"), streams)
                h = unit(u, eps) * (1 + self.t(p + f"norm{number}"))
                if number == 1:
                    a, n = p + "mix.", h.shape[1]
                    q, k = ((unit(self.mul(h, a + r), eps) * self.t(a + r + ".norm")).unflatten(-1, (m[w], -1)) for r, w in (("q", "heads"), ("k", "kv_heads")))
                    angles = plain_angles(n, m["rot"])
                    y = attend(turn(q, angles, "neighbours"), turn(k, angles, "neighbours"), self.heads(h, a + "v", m["kv_heads"]), m["scale"],
                               size=m["mask"]["size"], sink=self.t(a + "sink"))
                    y = self.mul(y.flatten(-2), a + "o")
                elif layer["mlp"]["kind"] == "dense":
                    y = self.mul(torch.relu(self.mul(h, p + "mlp.up")) ** 2, p + "mlp.down")
                else:
                    act = lambda g, u: g.clamp(max=limit) * torch.sigmoid(1.702 * g.clamp(max=limit)) * (u.clamp(-limit, limit) + 1)  # noqa: B023,E731
                    y = self.routed(h, p + "mlp.", layer["mlp"], rule, act)
                streams = torch.einsum("st,sbnd->tbnd", self.t(p + f"hc{number}.mix"), streams) + self.t(p + f"hc{number}.out")[:, None, None, None] * y
        return streams.sum(0)

    def dogotar(self, tokens, c):
        eps, x, n, first = c["norm"]["eps"], self.t("embed")[tokens], tokens.shape[1], None

        def attention(h, p, m, **more):
            nonlocal first
            q, k = (unit(self.heads(h, p + r, m[w]), eps) * self.t(p + r + ".norm") for r, w in (("q", "heads"), ("k", "kv_heads")))
            v = self.heads(h, p + "v", m["kv_heads"])
            if m.get("rot"):
                q, k = (turn(t, plain_angles(n, m["rot"]), "halves") for t in (q, k))
            if m.get("v_mix"):
                if first is not None:
                    v = (1 - self.t(p + "vmix")) * v + self.t(p + "vmix") * first
                first = v if first is None else first
            y = attend(q, k, v, m["scale"], cap=m["softcap"], **more).flatten(-2)
            if p + "g" in self.w:
                y = y * torch.sigmoid(self.mul(h, p + "g"))
            return self.mul(y, p + "o")

        for i, layer in enumerate(c["layers"]):
            p, m = f"l{i}.", layer["mixer"]
            h = layer_norm(x, self.t(p + "norm1"), self.t(p + "norm1.b"), eps)
            if layer["type"] == "attention":
                y = attention(h, p + "mix.", m, size=m["mask"]["size"])
            else:
                y = attention(h, p + "mix.left.", m["left"], block=m["left"]["mask"]["size"]) * m["left_scale"]
                y = y + m["right_scale"] * self.matrix_memory(h, p + "mix.right.", m["right"], eps)
            h = layer_norm(x, self.t(p + "norm2"), self.t(p + "norm2.b"), eps)
            x = x + y + self.mul(gelu_tanh(self.mul(h, p + "mlp.up")), p + "mlp.down")
        return x

    def matrix_memory(self, h, p, m, eps):
        heads, cap = m["heads"], m["gate_cap"]
        q, k, v = self.heads(h, p + "q", heads) * m["dim"] ** -0.5, self.heads(h, p + "k", heads), self.heads(h, p + "v", heads)
        gi = cap * torch.tanh(self.mul(h, p + "i") / cap)
        gf = torch.nn.functional.logsigmoid(cap * torch.tanh(self.mul(h, p + "f") / cap))
        # r_t = max(f_t + r_(t-1), i_t) from zero, by the running maximum of i - (sum of f)
        total = gf.cumsum(1)
        r = total + torch.cummax((gi - total), 1).values.clamp(min=0)
        keep = torch.exp(gf + torch.nn.functional.pad(r, (0, 0, 1, 0))[:, :-1] - r)[..., None]
        take = torch.exp(gi - r)[..., None]
        ones = torch.ones_like(v[..., :1])
        o = linear_scan(q, k * take, torch.cat([v, ones], -1), keep)
        o, norm = o[..., :-1], o[..., -1:]
        o = o / (torch.maximum(norm.abs(), torch.exp(-r)[..., None]) + 1e-6)
        y = unit(o, eps).flatten(-2) * self.t(p + "norm")
        return self.mul(y * torch.sigmoid(self.mul(h, p + "g")), p + "o")

    def digasun(self, tokens, c):
        eps, n = c["norm"]["eps"], tokens.shape[1]
        x, side, kept = self.t("embed")[tokens] * c["embedding"]["scale"], c["token_side"]["dim"], {}
        for i, layer in enumerate(c["layers"]):
            p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
            h = layer_norm(x, self.t(p + "norm1"), self.t(p + "norm1.b"), eps)
            a, b = h + causal_conv(h, self.t(p + "canon1")), h + causal_conv(h, self.t(p + "canon2"))
            mix = p + "mix."
            if layer["type"] == "attention":
                angles = plain_angles(n, m["rot"])
                if m.get("kv_from") is None:
                    kept[i] = turn(self.heads(a, mix + "k", m["kv_heads"]), angles, "halves"), self.heads(a, mix + "v", m["kv_heads"])
                k, v = kept[i if m.get("kv_from") is None else m["kv_from"]]
                y = attend(turn(self.heads(a, mix + "q", m["heads"]), angles, "halves"), k, v, m["scale"], size=m["mask"]["size"],
                           sink=self.t(mix + "sink"), talk=self.t(mix + "talk"))
                y = self.mul(y.flatten(-2), mix + "o")
            else:
                q, k, v = (self.heads(a, mix + r, m["heads"]) for r in "qkv")
                alpha = torch.sigmoid(self.mul(self.mul(a, mix + "a1"), mix + "a2")) ** (1 / m["tau"])
                o = linear_scan(q * m["dim"] ** -0.5, k, v, alpha.unflatten(-1, (m["heads"], -1)))
                y = self.mul((unit(o, eps) * self.t(mix + "norm")).flatten(-2) * silu(self.mul(a, mix + "g")), mix + "o")
            f = p + "mlp."
            if mlp["kind"] == "dense":
                g, u = self.mul(b, f + "gate").clamp(max=mlp["limit"]), self.mul(b, f + "up").clamp(-mlp["limit"], mlp["limit"])
                y = y + self.mul(g * torch.sigmoid(1.702 * g) * (u + 1), f + "down")
            else:
                y = y + self.routed(b, f, mlp, self.top_softmax(4), lambda g, u: silu(g) * u)
                s = f + "shared."
                y = y + torch.sigmoid(self.mul(b, s + "sg")) * self.mul(silu(self.mul(b, s + "gate")) * self.mul(b, s + "up"), s + "down")
            x = x + y
            rows = self.t("side.embed")[tokens][..., i * side : (i + 1) * side]
            y = self.mul(gelu_tanh(self.mul(x, p + "side.gate")) * rows, p + "side.proj")
            x = x + unit(y, eps) * self.t(p + "side.norm")
        return x

    def sunusun(self, tokens, c):
        eps, n, width = c["norm"]["eps"], tokens.shape[1], c["width"]
        at = torch.arange(n, dtype=F, device=DEVICE)[:, None]
        angles = at * 10000.0 ** (-2.0 * torch.arange(width // 2, dtype=F, device=DEVICE) / width)
        x = self.t("embed")[tokens] + torch.stack([torch.sin(angles), torch.cos(angles)], -1).flatten(-2)
        for i, layer in enumerate(c["layers"]):
            p, m = f"l{i}.", layer["mixer"]
            h, a = unit(x, eps) * self.t(p + "norm1"), p + "mix."
            if layer["type"] == "parallel":
                b, left = a + "left.", m["left"]
                q, k = (unit(self.heads(h, b + r, left[w]), eps) * self.t(b + r + ".norm") for r, w in (("q", "heads"), ("k", "kv_heads")))
                temp = left["q_temp"]
                q = q * (1 + temp["coef"] * torch.log(torch.floor((at + 1) / temp["every"]) + 1))[..., None]
                y = attend(q, k, self.heads(h, b + "v", left["kv_heads"]), left["scale"], sink=torch.zeros(left["heads"], dtype=F, device=DEVICE),
                           bias=(self.t(b + "r1"), self.t(b + "r2")))
                y = unit(self.mul(y.flatten(-2), b + "o"), eps) * self.t(b + "out")
                b = a + "right."
                z, u = torch.sigmoid(self.mul(h, b + "z")), self.mul(h, b + "x")
                u, carry, rows = z * torch.where(u >= 0, u + 0.5, torch.sigmoid(u)), torch.zeros_like(z[:, 0]), []
                for t in range(n):
                    carry = (1 - z[:, t]) * carry + u[:, t]
                    rows.append(carry)
                right = self.mul(torch.stack(rows, 1) * silu(self.mul(h, b + "g")), b + "o")
                x = x + 0.5 * (y + unit(right, eps) * self.t(b + "out"))
            else:
                step = before(h) - h
                r, k, v, g, s = (h + step * self.t(a + "mu." + name) for name in "rkvgw")
                r, k, v = (self.heads(t, a + name, m["heads"]) for t, name in ((r, "r"), (k, "k"), (v, "v")))
                low = torch.tanh(self.mul(s, a + "w1"))
                decay = torch.exp(-torch.exp(self.mul(low, a + "w2") + self.t(a + "w0"))).unflatten(-1, (m["heads"], -1))
                o = linear_scan(r, k, v, decay, after=True) + (r * self.t(a + "u") * k).sum(-1, keepdim=True) * v
                x = x + self.mul(unit(o, eps).flatten(-2) * self.t(a + "norm") * silu(self.mul(g, a + "g")), a + "o")
            h = unit(x, eps) * self.t(p + "norm2")
            h = self.mul(h, p + "mlp.up")
            x = x + self.mul(0.5 * h * (1 + torch.erf(h / math.sqrt(2))), p + "mlp.down")
        return x

    def sorovik(self, tokens, c):
        eps, n = c["norm"]["eps"], tokens.shape[1]
        norm = lambda x, name: unit(x, eps) * self.t(name)  # noqa: E731
        x, kept = norm(self.t("embed")[tokens], "embed.norm"), {}
        for i, layer in enumerate(c["layers"]):
            p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
            h, a = norm(x, p + "norm1"), p + "mix."
            if layer["type"] == "latent_attention":
                if m.get("kv_from") is None:
                    down = self.mul(h, a + "dkv")
                    kept[i] = norm(down[..., : m["kv_rank"]], a + "dkv.norm"), turn(down[:, :, None, m["kv_rank"] :], plain_angles(n, m["rot"]), "halves")
                latent, key_part = kept[i if m.get("kv_from") is None else m["kv_from"]]
                y = self.through_latent(self.heads(h, a + "q", m["heads"]), latent, key_part, a, m, "halves", size=m["mask"]["size"], sink=self.t(a + "sink"))
            else:
                q, k = (causal_conv(self.mul(h, a + r), self.t(a + r + ".conv")) for r in "qk")
                v = k.unflatten(-1, (m["kv_heads"], -1))
                angles = plain_angles(n, m["rot"])
                q, k = (turn(norm(t, a + r + ".norm").unflatten(-1, (m[w], -1)), angles, "halves") for t, r, w in ((q, "q", "heads"), (k, "k", "kv_heads")))
                y = attend(q, k, v, m["scale"], size=m["mask"]["size"], keep=m["mask"]["keep_first"], sink=torch.zeros(m["heads"], dtype=F, device=DEVICE))
                y = (y * torch.sigmoid(self.mul(h, a + "g"))[..., None]).flatten(-2)
            x = x + norm(self.mul(y, a + "o"), p + "norm1b")
            h, f = norm(x, p + "norm2"), p + "mlp."
            if mlp["kind"] == "dense":
                y = self.mul(gelu_tanh(self.mul(h, f + "gate")) * self.mul(h, f + "up"), f + "down")
            else:
                def rule(z, groups=mlp["router"]["groups"]):
                    s = torch.softmax(z, -1)
                    members = s.unflatten(-1, (groups["count"], -1))
                    best = torch.topk(members.amax(-1), groups["keep"], -1).indices
                    open_ = torch.zeros_like(members[..., 0], dtype=torch.bool).scatter(1, best, True)
                    chosen = torch.topk(members.masked_fill(~open_[..., None], -1.0).flatten(-2), 4, -1).indices
                    return chosen, torch.gather(s, 1, chosen)
                y = self.routed(h, f, mlp, rule, lambda g, u: silu(g) * u)
            x = x + norm(y, p + "norm2b")
        return x


def linear_scan(q, k, v, decay, after=False):
    """S_t = decay_t S_(t-1) + k_t v_t^T, o_t = S_t^T q_t (`after`: S_(t-1)); q, k, decay [B, T, H, d or 1], v [B, T, H, e]."""
    nb, n, heads, d = k.shape
    state = torch.zeros(nb, heads, d, v.shape[-1], dtype=F, device=DEVICE)
    out = torch.empty_like(v)
    for t in range(n):
        if after:
            out[:, t] = (q[:, t, :, None] @ state)[:, :, 0]
        state = state * decay[:, t, ..., None] + k[:, t, ..., None] * v[:, t, :, None]
        if not after:
            out[:, t] = (q[:, t, :, None] @ state)[:, :, 0]
    return out


@torch.inference_mode()
def exact(case, seed):
    if case.get("engine"):
        return None  # whole numbers only
    _model, config, tensors = model_of(case, seed)
    cached, prompts = draw_tokens(case, seed)
    sequences = cached + prompts
    plain = Plain(config, tensors)
    if case["design"] == "dense":
        together = [[s] for s in sequences]
    else:  # the recurrences walk over the tokens of all sequences at once
        together = [sequences]
    rows = []
    wanted = [len(s) - 1 for s in cached] + [0] * len(prompts)
    for some in together:
        ends = [len(s) for s in some]
        firsts, wanted = wanted[: len(some)], wanted[len(some) :]
        padded = torch.zeros((len(some), max(ends)), dtype=torch.long)
        for i, s in enumerate(some):
            padded[i, : len(s)] = torch.tensor(s)
        rows.append(plain(padded.to(DEVICE), ends, firsts if case.get("score") else None))
    return {"logits": torch.cat(rows), "tokens": None}
