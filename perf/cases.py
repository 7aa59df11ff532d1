"""The framework's calls as a serving program makes them, for timing and for comparing outputs.

A case is a dict of plain values; ``kind`` names what one pass calls:

* ``apply``   ``HipLoRABackend.apply_lora_multi`` over one segment table (with ``norm``,
              ``rmsnorm_apply_lora_multi``): a projection's LoRA in decode, prefill or a mixed batch.
              With ``captured`` the call is replayed from a HIP graph, as the decode step of a serving
              loop is; otherwise it is made directly, as prompts of ever-changing lengths are.
* ``layer``   the LoRA calls and norms of one decoder layer in decode, captured in one graph.
* ``step``    one captured decode step of the package's decoder (base weights included); returns logits.
* ``kernels`` ``sgemm_lora_a_fwd`` then ``sgemm_lora_b_fwd``, the two-call form.
* ``norm``    ``fused_add_rmsnorm`` (or ``rmsnorm_fwd``), the norm between two projections.
* ``upload``  ``scatter_stage``: staged adapters into their pool slots, every module key.

Segment lengths are texts such as ``"512*2,1*64"``.  A table uses ``adapters`` adapters, each at least
once, of ranks taken in turn from ``ranks``, in random slots of a pool of ``slots``; the other slots are
empty.  Stacks hold values past a slot's rank too, as reused slots do.
"""

import math
import random

import torch

from multi_lora_amd import AdapterWeights, HipLoRABackend, LoRAMemoryPool, MultiLoRAManager
from multi_lora_amd.batch_info import BatchLoRAInfo, empty_kernel_input_metadata, write_kernel_input_metadata
from multi_lora_amd.decoder import Decoder, DecoderConfig
from multi_lora_amd.graph_decode import DecodeStep, capture_graph
from multi_lora_amd.kernels import fused_add_rmsnorm, rmsnorm_fwd
from multi_lora_amd.kernels.lora_ops import sgemm_lora_a_fwd, sgemm_lora_b_fwd
from multi_lora_amd.kernels.scatter_bank import scatter_stage
from multi_lora_amd.layers import fuse_gate_up_projections, fuse_qkv_projections

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZES = {"bf16": 2, "fp16": 2, "fp32": 4}
EPS = 1e-5
SCALINGS = (2.0, 0.5, 1.0)


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # One sequence decoding one token with one adapter: the smallest call, all latency.
        dict(name="decode one token", kind="apply", lens="1", in_dim=1024, outs="1024", ranks="8", r_max=8,
             adapters=1, slots=4, dtype="fp16", norm=False, captured=False),
        # q_proj of a decode batch of 128 sequences over 32 rank-16 adapters, called directly.
        dict(name="decode q", kind="apply", lens="1*128", in_dim=4096, outs="4096", ranks="16", r_max=16,
             adapters=32, slots=64, dtype="bf16", norm=False, captured=False),
        # Input norm and fused q|k|v of a large decode batch over many adapters, in a captured step.
        dict(name="decode norm+qkv", kind="apply", lens="1*256", in_dim=4096, outs="4096,1024,1024", ranks="32",
             r_max=32, adapters=112, slots=256, dtype="bf16", norm=True, captured=True),
        # A whole layer in decode: ragged segments (some sequences verify a few tokens), mixed ranks, fp16.
        dict(name="decode layer", kind="layer", lens="1*51,2*7,3*4", hidden=4096, kv=1024, inter=14336,
             ranks="8,16,32,64", r_max=64, adapters=40, slots=64, dtype="fp16"),
        # A captured decode step of a small decoder, 32 sequences over 8 adapters.
        dict(name="decode step", kind="step", batch=32, hidden=2048, kv=512, inter=7168, layers=4, vocab=4096,
             rank=16, adapters=8, slots=16, start=200, dtype="fp16"),
        # One prompt of a new request: what a user waits for before the first token.
        dict(name="one prompt", kind="apply", lens="203", in_dim=4096, outs="4096", ranks="64", r_max=64, adapters=1,
             slots=8, dtype="bf16", norm=False, captured=False),
        # gate|up of a batch of prompts of very different lengths and ranks: the largest call.
        dict(name="prefill gate|up", kind="apply", lens="837,64,1024,391,702,133,498,426", in_dim=4096,
             outs="14336,14336", ranks="16,32,64", r_max=64, adapters=8, slots=8, dtype="bf16", norm=False,
             captured=False),
        # down of the same batch: the longest reduction.
        dict(name="prefill down", kind="apply", lens="837,64,1024,391,702,133,498,426", in_dim=14336, outs="4096",
             ranks="16,32,64", r_max=64, adapters=8, slots=8, dtype="bf16", norm=False, captured=False),
        # Continuous batching: two prompts and 64 decoding sequences in one batch, fused q|k|v.
        dict(name="mixed qkv", kind="apply", lens="512*2,1*64", in_dim=4096, outs="4096,1024,1024", ranks="16",
             r_max=16, adapters=35, slots=128, dtype="bf16", norm=False, captured=False),
        # Three short ragged segments in fp32 through the two-call form, as correctness runs use it.
        dict(name="fp32 segments", kind="kernels", lens="5,17,42", in_dim=1024, out=1024, ranks="8", r_max=8,
             adapters=3, slots=4, dtype="fp32"),
        # Residual add and norm between two projections of a mixed batch.
        dict(name="add norm", kind="norm", rows=1088, hidden=4096, add=True, dtype="bf16"),
        # Four missing adapters into their slots: two layers' keys.
        dict(name="upload", kind="upload", staged=4, layers=2, hidden=4096, kv=1024, inter=14336, rank=16, r_max=16,
             slots=8, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A projection width: mostly multiples of 64, some of 8, a few odd ones."""
    w = _log(rng, lo, hi)
    step = rng.choice((64, 64, 64, 64, 64, 8, 8, 1))
    return max(lo, w // step * step)


def _bytes_of(case):
    return work(case)["bytes"]


def draw(rng):
    limit = _bytes_of(next(c for c in listed() if c["name"] == "prefill gate|up"))
    while True:
        case = _draw(rng)
        if _bytes_of(case) <= limit:
            return case


def _draw(rng):
    what = rng.choice(("decode", "decode", "decode", "prefill", "prefill", "prefill", "mixed", "mixed", "kernels",
                       "norm", "layer", "upload"))
    dtype = rng.choice(("bf16", "bf16", "fp16"))
    r_max = rng.choice((8, 16, 16, 32, 64))
    ranks = str(r_max) if rng.random() < 0.5 else ",".join(str(r) for r in (8, 16, 32, 64) if r <= r_max)
    if what == "norm":
        return dict(kind="norm", rows=_log(rng, 1, 4500), hidden=rng.choice((128, 1000, 1024, 2560, 4096, 4096, 14336)),
                    add=rng.random() < 0.6, dtype=rng.choice(("bf16", "bf16", "fp16", "fp32")))
    if what == "upload":
        return dict(kind="upload", staged=rng.randint(1, 4), layers=rng.randint(1, 4), hidden=_width(rng, 256, 4096),
                    kv=_width(rng, 128, 1024), inter=_width(rng, 512, 14336), rank=rng.choice((8, 16, 16, 32)),
                    r_max=32, slots=8, dtype=dtype)
    if what == "kernels":
        n = rng.randint(1, 8)
        lens = ",".join(str(_log(rng, 1, 300)) for _ in range(n))
        return dict(kind="kernels", lens=lens, in_dim=_width(rng, 256, 4096), out=_width(rng, 256, 4096), ranks=ranks,
                    r_max=r_max, adapters=n, slots=n + 1, dtype=rng.choice(("fp32", "fp32", dtype)))
    n_dec = _log(rng, 1, 300)
    decode = "1*%d" % n_dec
    segs = n_dec
    if rng.random() < 0.3:
        more = [rng.randint(2, 16) for _ in range(rng.randint(1, 6))]
        decode += "," + ",".join(str(m) for m in more)
        segs += len(more)
    if what == "layer":
        used = rng.randint(1, min(segs, 48))
        return dict(kind="layer", lens=decode, hidden=rng.choice((2048, 2560, 4096)), kv=1024,
                    inter=rng.choice((7168, 14336)), ranks=ranks, r_max=r_max, adapters=used,
                    slots=max(used, rng.choice((16, 32, 64))), dtype=dtype)
    slices = rng.choice((1, 1, 2, 3))
    if slices == 1:
        outs = [_width(rng, 256, 14336)]
    elif slices == 2:
        outs = [_width(rng, 512, 14336)] * 2
    else:
        outs = [_width(rng, 512, 4096)] + [_width(rng, 128, 1024)] * 2
    in_dim = _width(rng, 256, 14336)
    if what == "decode":
        used = rng.randint(1, min(segs, 128))
        return dict(kind="apply", lens=decode, in_dim=in_dim, outs=",".join(map(str, outs)), ranks=ranks, r_max=r_max,
                    adapters=used, slots=max(used, rng.choice((8, 64, 256))), dtype=dtype, norm=rng.random() < 0.3,
                    captured=rng.random() < 0.6)
    n = rng.randint(1, 8)
    lens = ",".join(str(_log(rng, 17, 1024)) for _ in range(n))
    if what == "mixed":
        lens += ",1*%d" % rng.randint(1, 64)
        n += int(lens.rsplit("*", 1)[1])
    used = rng.randint(1, min(n, 40))
    return dict(kind="apply", lens=lens, in_dim=in_dim, outs=",".join(map(str, outs)), ranks=ranks, r_max=r_max,
                adapters=used, slots=max(used, 16), dtype=dtype, norm=False, captured=False)


# ---------------------------------------------------------------- inputs
def _lens(text):
    out = []
    for part in text.split(","):
        n, _, times = part.partition("*")
        out += [int(n)] * int(times or 1)
    return out


def _ints(text):
    return [int(v) for v in str(text).split(",")]


def _table(case, seed):
    """Slot of each segment, rank and scaling of each slot, as lists.  Segment ``i`` uses adapter
    ``i % adapters``; which slot an adapter sits in comes from the seed."""
    lens, ranks = _lens(case["lens"]), _ints(case["ranks"])
    slot_of = random.Random(seed).sample(range(case["slots"]), case["adapters"])
    slot_ranks, scalings = [0] * case["slots"], [0.0] * case["slots"]
    for j, s in enumerate(slot_of):
        slot_ranks[s], scalings[s] = ranks[j % len(ranks)], SCALINGS[j % len(SCALINGS)]
    return lens, [slot_of[i % case["adapters"]] for i in range(len(lens))], slot_ranks, scalings


def _gen(seed):
    return torch.Generator("cuda").manual_seed(int(seed))


def _randn(g, shape, dtype, std=1.0, mean=0.0):
    t = torch.empty(shape, dtype=dtype, device="cuda").normal_(mean, std, generator=g)
    return t


def _stacks(g, case, in_dim, outs, dtype):
    """The pool's slot tensors of one projection group: A [slots, r_max, in], B [slots, out, r_max]."""
    a = [_randn(g, (case["slots"], case["r_max"], in_dim), dtype, in_dim ** -0.5) for _ in outs]
    b = [_randn(g, (case["slots"], o, case["r_max"]), dtype, 0.05) for o in outs]
    return a, b


def _write_table(case, seed, dtype):
    lens, slots, ranks, scalings = _table(case, seed)
    return write_kernel_input_metadata(empty_kernel_input_metadata(device=torch.device("cuda"), dtype=dtype),
                                       BatchLoRAInfo(slots, ranks, scalings), device=torch.device("cuda"),
                                       dtype=dtype, seq_lens=lens)


def _cols(outs):
    return [sum(outs[:i]) for i in range(len(outs))]


def _apply_inputs(case, seed):
    dt, outs = DTYPES[case["dtype"]], _ints(case["outs"])
    g, rows = _gen(seed), sum(_lens(case["lens"]))
    a, b = _stacks(g, case, case["in_dim"], outs, dt)
    d = dict(x=_randn(g, (rows, case["in_dim"]), dt), a=a, b=b, out=_randn(g, (rows, sum(outs)), dt), cols=_cols(outs))
    if case["norm"]:
        d["w"] = _randn(g, (case["in_dim"],), dt, 0.1, 1.0)
    return d


def _layer_inputs(case, seed):
    dt, g, rows = DTYPES[case["dtype"]], _gen(seed), sum(_lens(case["lens"]))
    h, kv, inter = case["hidden"], case["kv"], case["inter"]
    d = {"qkv": _stacks(g, case, h, [h, kv, kv], dt), "o": _stacks(g, case, h, [h], dt),
         "gu": _stacks(g, case, h, [inter, inter], dt), "down": _stacks(g, case, inter, [h], dt)}
    for name, width in (("x", h), ("attn", h), ("proj", h), ("residual", h), ("act", inter), ("qkv_out", h + 2 * kv),
                        ("o_out", h), ("gu_out", 2 * inter), ("down_out", h)):
        d[name] = _randn(g, (rows, width), dt)
    d["w1"], d["w2"] = _randn(g, (h,), dt, 0.1, 1.0), _randn(g, (h,), dt, 0.1, 1.0)
    return d


def _captured(call, keep):
    """``call`` recorded in a graph after a run on the capture's stream; ``keep``: buffers that calls change."""
    kept = [t.clone() for t in keep]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = call()
    torch.cuda.current_stream().wait_stream(side)
    for t, k in zip(keep, kept):
        t.copy_(k)
    return graph, out


PROJECTIONS = (("self_attn.q_proj", "hidden", "hidden"), ("self_attn.k_proj", "hidden", "kv"),
               ("self_attn.v_proj", "hidden", "kv"), ("self_attn.o_proj", "hidden", "hidden"),
               ("mlp.gate_proj", "hidden", "inter"), ("mlp.up_proj", "hidden", "inter"),
               ("mlp.down_proj", "inter", "hidden"))
HEAD_DIM = 128


def _step_inputs(case, seed):
    """Weights, adapters, caches and token ids of the decoder step, by name."""
    dt, g = DTYPES[case["dtype"]], _gen(seed)
    h, r, batch = case["hidden"], case["rank"], case["batch"]
    d = {"embed_tokens.weight": _randn(g, (case["vocab"], h), dt), "norm.weight": _randn(g, (h,), dt, 0.1, 1.0),
         "lm_head.weight": _randn(g, (case["vocab"], h), dt, h ** -0.5)}
    for i in range(case["layers"]):
        for leaf, n_in, n_out in PROJECTIONS:
            key, ni, no = "layers.%d.%s" % (i, leaf), case[n_in], case[n_out]
            d[key + ".weight"] = _randn(g, (no, ni), dt, ni ** -0.5)
            d[key + ".a"] = _randn(g, (case["adapters"], r, ni), dt, ni ** -0.5)
            d[key + ".b"] = _randn(g, (case["adapters"], no, r), dt, 0.02)
        for norm in ("input_layernorm", "post_attention_layernorm"):
            d["layers.%d.%s.weight" % (i, norm)] = _randn(g, (h,), dt, 0.1, 1.0)
        kvh = case["kv"] // HEAD_DIM
        d["keys.%d" % i] = _randn(g, (batch, kvh, HEAD_DIM, case["start"]), dt)
        d["values.%d" % i] = _randn(g, (batch, kvh, case["start"], HEAD_DIM), dt)
    d["ids"] = torch.randint(0, case["vocab"], (batch, 1), device="cuda", generator=g)
    return d


def _step_config(case):
    return DecoderConfig(vocab_size=case["vocab"], hidden_size=case["hidden"], intermediate_size=case["inter"],
                         num_hidden_layers=case["layers"], num_attention_heads=case["hidden"] // HEAD_DIM,
                         num_key_value_heads=case["kv"] // HEAD_DIM, rms_norm_eps=EPS)


def _prepare_step(case, seed):
    d, dt = _step_inputs(case, seed), DTYPES[case["dtype"]]
    with torch.device("cuda"):
        model = Decoder(_step_config(case)).to(dt).eval()
    with torch.inference_mode():
        for name, p in model.named_parameters():
            p.copy_(d[name])
    adapters = {}
    for j in range(case["adapters"]):
        mods = {"layers.%d.%s" % (i, leaf): tuple(d["layers.%d.%s.%s" % (i, leaf, side)][j].cpu() for side in "ab")
                for i in range(case["layers"]) for leaf, _, _ in PROJECTIONS}
        adapters["a%d" % j] = AdapterWeights(rank=case["rank"], scaling=SCALINGS[j % len(SCALINGS)], modules=mods)
    mgr = MultiLoRAManager.from_adapters(model, adapters, max_loras_per_batch=case["slots"],
                                         max_lora_rank=case["rank"])
    fuse_qkv_projections(mgr.lora_wrappers)
    fuse_gate_up_projections(mgr.lora_wrappers)
    step = DecodeStep.new(mgr, case["batch"], case["start"], case["start"] + 8)
    for i in range(case["layers"]):
        step.kv.keys[i][..., : case["start"]] = d["keys.%d" % i]
        step.kv.values[i][:, :, : case["start"]] = d["values.%d" % i]
    step.input_ids.copy_(d["ids"])
    names = ["a%d" % (i % case["adapters"]) for i in range(case["batch"])]
    with torch.inference_mode():
        mgr._setup_forward_batch(names, seq_lens=[1] * case["batch"])
        graph, out = capture_graph(mgr, step)
    return dict(mgr=mgr, step=step, graph=graph, logits=out.logits)


def _upload_keys(case):
    return {"layers.%d.%s" % (i, leaf): (case[n_in], case[n_out]) for i in range(case["layers"])
            for leaf, n_in, n_out in PROJECTIONS}


def _apply_call(be, x, a, b, out, cols, norm, w=None):
    """The call as a function that holds the tensors, not the state that holds it (a graph in a reference
    cycle would be destroyed by the collector, perhaps during the capture of the next one)."""
    if norm:
        return lambda: [be.rmsnorm_apply_lora_multi(x, w, EPS, a, b, out, cols), out]
    return lambda: be.apply_lora_multi(x, a, b, out, cols)


def prepare(case, seed):
    kind = case["kind"]
    dt = DTYPES[case["dtype"]]
    if kind == "apply":
        d, be = _apply_inputs(case, seed), HipLoRABackend()
        be.set_kernel_input_metadata(_write_table(case, seed, dt))
        call = _apply_call(be, norm=case["norm"], **d)
        # The state keeps the backend: a graph's launches use its workspace and its segment table.
        d["backend"] = be
        if case["captured"]:
            d["graph"], d["result"] = _captured(call, [d["out"]])
        else:
            d["call"] = call
        return d
    if kind == "layer":
        d, be = _layer_inputs(case, seed), HipLoRABackend()
        be.set_kernel_input_metadata(_write_table(case, seed, dt))
        d["backend"] = be
        h, kv, inter = case["hidden"], case["kv"], case["inter"]

        def call():
            y1 = be.rmsnorm_apply_lora_multi(d["x"], d["w1"], EPS, *d["qkv"], d["qkv_out"], _cols([h, kv, kv]))
            be.apply_lora(d["attn"], d["o"][0][0], d["o"][1][0], d["o_out"])
            y2 = fused_add_rmsnorm(d["proj"], d["residual"], d["w2"], EPS)
            be.apply_lora_multi(y2, *d["gu"], d["gu_out"], [0, inter])
            be.apply_lora(d["act"], d["down"][0][0], d["down"][1][0], d["down_out"])
            return [y1, d["qkv_out"], d["o_out"], y2, d["residual"], d["gu_out"], d["down_out"]]

        d["graph"], d["result"] = _captured(call, [d[k] for k in ("qkv_out", "o_out", "residual", "gu_out", "down_out")])
        return d
    if kind == "step":
        return _prepare_step(case, seed)
    if kind == "kernels":
        g, rows = _gen(seed), sum(_lens(case["lens"]))
        a, b = _stacks(g, case, case["in_dim"], [case["out"]], dt)
        return dict(x=_randn(g, (rows, case["in_dim"]), dt), a=a[0], b=b[0], out=_randn(g, (rows, case["out"]), dt),
                    meta=_write_table(case, seed, dt), mid=torch.empty((rows, case["r_max"]), dtype=dt, device="cuda"))
    if kind == "norm":
        g, shape = _gen(seed), (case["rows"], case["hidden"])
        d = dict(x=_randn(g, shape, dt), w=_randn(g, shape[1:], dt, 0.1, 1.0))
        if case["add"]:
            d["residual"] = _randn(g, shape, dt, 2.0)
        return d
    g, dims = _gen(seed), _upload_keys(case)
    pool = LoRAMemoryPool(case["slots"], case["r_max"], torch.device("cuda"), dt)
    pool.ensure_buffers(AdapterWeights(rank=case["rank"], scaling=1.0, modules={
        k: (torch.empty(case["rank"], i, device="meta"), torch.empty(o, case["rank"], device="meta"))
        for k, (i, o) in dims.items()}))
    plan = pool.buffers.layout(case["rank"])
    slots = random.Random(seed).sample(range(case["slots"]), case["staged"])
    return dict(pool=pool, stage=_randn(g, (case["staged"], plan.total), dt), total=plan.total, h=case["staged"],
                rank=case["rank"], tables=plan.build_tables(pool.buffers, pool.device),
                slots=torch.tensor(slots, dtype=torch.int32, device="cuda"))


# ---------------------------------------------------------------- one pass
def run(state):
    if "step" in state:
        state["step"].rewind()
        state["graph"].replay()
        return state["logits"]
    if "graph" in state:
        state["graph"].replay()
        return state["result"]
    if "call" in state:
        return state["call"]()
    if "mid" in state:
        mid = sgemm_lora_a_fwd(state["x"], state["a"], state["meta"], state["mid"])
        return [mid, sgemm_lora_b_fwd(mid, state["b"], state["meta"], state["out"])]
    if "pool" in state:
        scatter_stage(state["stage"], state["slots"], state["tables"], state["total"], state["h"], state["rank"])
        buf = state["pool"].buffers
        return [buf.A, buf.B]
    if "residual" in state:
        return [fused_add_rmsnorm(state["x"], state["residual"], state["w"], EPS), state["residual"]]
    return rmsnorm_fwd(state["x"], state["w"], EPS)


# ---------------------------------------------------------------- work
def _lora_work(case, in_dim, outs):
    """Bytes and operations of one projection group: x and the adapters in use read once, the output
    read and written once."""
    lens, ranks, e = _lens(case["lens"]), _ints(case["ranks"]), SIZES[case["dtype"]]
    rank = [ranks[j % len(ranks)] for j in range(case["adapters"])]
    width = sum(in_dim + o for o in outs)
    return {"bytes": e * (sum(lens) * (in_dim + 2 * sum(outs)) + sum(rank) * width),
            "flops": 2 * sum(n * rank[i % len(rank)] for i, n in enumerate(lens)) * width}


def _sum(parts):
    return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}


def _norm_work(case, rows, hidden, add):
    return {"bytes": SIZES[case["dtype"]] * (rows * hidden * (4 if add else 2) + hidden), "flops": 4 * rows * hidden}


def work(case):
    kind, e = case["kind"], SIZES[case["dtype"]]
    if kind == "apply":
        parts = [_lora_work(case, case["in_dim"], _ints(case["outs"]))]
        if case["norm"]:  # x is read once for both; y is written
            n = _norm_work(case, sum(_lens(case["lens"])), case["in_dim"], False)
            n["bytes"] -= e * sum(_lens(case["lens"])) * case["in_dim"]
            parts.append(n)
        return _sum(parts)
    if kind == "layer":
        h, kv, inter, rows = case["hidden"], case["kv"], case["inter"], sum(_lens(case["lens"]))
        return _sum([_lora_work(case, h, [h, kv, kv]), _lora_work(case, h, [h]), _lora_work(case, h, [inter, inter]),
                     _lora_work(case, inter, [h]), _norm_work(case, rows, h, True),
                     {"bytes": e * rows * h, "flops": 4 * rows * h}])
    if kind == "step":
        b, h, kv, inter = case["batch"], case["hidden"], case["kv"], case["inter"]
        base = 2 * h * h + 2 * h * kv + 3 * h * inter
        lora = case["rank"] * (4 * h + 2 * (h + kv) + 3 * (h + inter))
        return {"bytes": e * (case["layers"] * (base + case["adapters"] * lora + 2 * b * kv * case["start"])
                              + case["vocab"] * h + b * (h + case["vocab"])),
                "flops": 2 * b * (case["layers"] * (base + lora + 2 * h * case["start"]) + case["vocab"] * h)}
    if kind == "kernels":
        w = _lora_work(case, case["in_dim"], [case["out"]])
        return {"bytes": w["bytes"] + e * sum(_lens(case["lens"])) * case["r_max"], "flops": w["flops"]}
    if kind == "norm":
        return _norm_work(case, case["rows"], case["hidden"], case["add"])
    return {"bytes": 2 * e * case["staged"] * case["rank"] * sum(i + o for i, o in _upload_keys(case).values()),
            "flops": 0}


def tolerance(case):
    """Rounding of the outputs to their type, and of the rank-r intermediate before the second product: about
    four times the errors against ``exact`` (bf16 1.7e-3..2.4e-3, fp16 2.0e-4..3.1e-4, fp32 up to 4.4e-7; fp16
    through the layers of the decode step 1.7e-3)."""
    if case["kind"] == "upload":
        return "exact"
    if case["kind"] == "step":
        return {"rel": 7e-3}
    return {"rel": {"bf16": 8e-3, "fp16": 1.2e-3, "fp32": 2e-6}[case["dtype"]]}


# ---------------------------------------------------------------- 64 bits
def _exact_lora(case, seed, x, a, b, out, cols):
    """out + scaling * (x A^T) B^T per segment, in 64 bits; also the intermediate of the first slice."""
    lens, slots, ranks, scalings = _table(case, seed)
    out, r0 = out.double(), 0
    mid = torch.zeros((x.shape[0], case["r_max"]), dtype=torch.float64, device=x.device)
    for n, s in zip(lens, slots):
        r = ranks[s]
        for i, c in enumerate(cols):
            m = x[r0:r0 + n].double() @ a[i][s, :r].double().t()
            if i == 0:
                mid[r0:r0 + n, :r] = m
            out[r0:r0 + n, c:c + b[i].shape[1]] += scalings[s] * (m @ b[i][s, :, :r].double().t())
        r0 += n
    return out, mid


def _exact_norm(x, w):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _exact_step(case, seed):
    d = {k: (v if k == "ids" else v.double()) for k, v in _step_inputs(case, seed).items()}
    b, h, kvh, heads = case["batch"], case["hidden"], case["kv"] // HEAD_DIM, case["hidden"] // HEAD_DIM
    inv = 1.0 / (_step_config(case).rope_theta ** (torch.arange(0, HEAD_DIM, 2, dtype=torch.float64, device="cuda")
                                                   / HEAD_DIM))
    ang = case["start"] * torch.cat((inv, inv))

    def rotate(t):
        half = HEAD_DIM // 2
        return t * ang.cos() + torch.cat((-t[..., half:], t[..., :half]), -1) * ang.sin()

    def linear(x, key):
        y = x @ d[key + ".weight"].t()
        for j in range(case["adapters"]):
            rows = slice(j, b, case["adapters"])
            y[rows] += SCALINGS[j % len(SCALINGS)] * (x[rows] @ d[key + ".a"][j].t()) @ d[key + ".b"][j].t()
        return y

    x = d["embed_tokens.weight"][d["ids"].reshape(-1)]
    for i in range(case["layers"]):
        p = "layers.%d." % i
        y = _exact_norm(x, d[p + "input_layernorm.weight"])
        q = rotate(linear(y, p + "self_attn.q_proj").view(b, kvh, heads // kvh, HEAD_DIM))
        k = rotate(linear(y, p + "self_attn.k_proj").view(b, kvh, HEAD_DIM))
        v = linear(y, p + "self_attn.v_proj").view(b, kvh, 1, HEAD_DIM)
        keys = torch.cat((d["keys.%d" % i], k[..., None]), -1)
        probs = torch.softmax(q @ keys / math.sqrt(HEAD_DIM), -1)
        attn = (probs @ torch.cat((d["values.%d" % i], v), 2)).reshape(b, h)
        x = x + linear(attn, p + "self_attn.o_proj")
        y = _exact_norm(x, d[p + "post_attention_layernorm.weight"])
        act = torch.nn.functional.silu(linear(y, p + "mlp.gate_proj")) * linear(y, p + "mlp.up_proj")
        x = x + linear(act, p + "mlp.down_proj")
    return (_exact_norm(x, d["norm.weight"]) @ d["lm_head.weight"].t())[:, None]


def exact(case, seed):
    kind, dt = case["kind"], DTYPES[case["dtype"]]
    if kind == "apply":
        d = _apply_inputs(case, seed)
        y = _exact_norm(d["x"], d["w"]) if case["norm"] else d["x"]
        out = _exact_lora(case, seed, y, d["a"], d["b"], d["out"], d["cols"])[0]
        return [y, out] if case["norm"] else out
    if kind == "layer":
        d, h, kv, inter = _layer_inputs(case, seed), case["hidden"], case["kv"], case["inter"]
        y1 = _exact_norm(d["x"], d["w1"])
        res = d["proj"].double() + d["residual"].double()
        y2 = _exact_norm(res, d["w2"])
        return [y1, _exact_lora(case, seed, y1, *d["qkv"], d["qkv_out"], _cols([h, kv, kv]))[0],
                _exact_lora(case, seed, d["attn"], *d["o"], d["o_out"], [0])[0], y2, res,
                _exact_lora(case, seed, y2, *d["gu"], d["gu_out"], [0, inter])[0],
                _exact_lora(case, seed, d["act"], *d["down"], d["down_out"], [0])[0]]
    if kind == "step":
        return _exact_step(case, seed)
    if kind == "kernels":
        g, rows = _gen(seed), sum(_lens(case["lens"]))
        a, b = _stacks(g, case, case["in_dim"], [case["out"]], dt)
        x, out = _randn(g, (rows, case["in_dim"]), dt), _randn(g, (rows, case["out"]), dt)
        out, mid = _exact_lora(case, seed, x, a, b, out, [0])
        return [mid, out]
    if kind == "norm":
        g, shape = _gen(seed), (case["rows"], case["hidden"])
        x, w = _randn(g, shape, dt), _randn(g, shape[1:], dt, 0.1, 1.0)
        if not case["add"]:
            return _exact_norm(x, w)
        res = x.double() + _randn(g, shape, dt, 2.0).double()
        return [_exact_norm(res, w), res]
    return None
