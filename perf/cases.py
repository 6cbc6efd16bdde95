"""Performance cases of the gfx950 decode backend: the work its users run.

Every case is a plan that a program prepares once (weights laid out, buffers
bound, launches captured by Runtime.sequence or by the batched decode
executor) and then replays; run() is one replay.  Shapes are those of the
benchmark (7B widths: hidden 4096, 32 heads x 128, intermediate 11008,
vocabulary 32000; paged GQA 32:8 at batch 16; the contiguous cache of
capacity 4096), of the tests (head dim 64, odd widths) and generic ones.

kinds:
  mlp     decode MLP block over `layers` weight sets: RMSNorm, gate/up with
          SiLU*Mul, down with the residual, in the form the decoder runs at
          that batch (row-major GEMVs at 1, packed weights above)
  linear  RMSNorm, then a row-major fp16 linear layer with fp32 output (the
          graph path and the contiguous-cache executor)
  paged   paged decode attention of a batch with ragged lengths
  contig  contiguous-cache decode attention
  pattn   causal attention of one prompt chunk over its paged cache
  prompt  one whole transformer layer over a prompt chunk
  step    one whole decode step of the batched executor, logits included
"""
from __future__ import annotations

import importlib
import math
import random

import torch

EPS = 1e-6
F16 = torch.float16
tmc = importlib.import_module("aicompiler-test_amd")

_shared = {}


def _runtime():
    """One runtime (one stream) for every plan of the process."""
    if "rt" not in _shared:
        _shared["rt"] = tmc.Runtime()
    return _shared["rt"]


def _host_runtime():
    if "host" not in _shared:
        _shared["host"] = tmc.host().HipRuntime()
    return _shared["host"]


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: one chat user's attention, a few hundred
        # positions, where launch latency and dependent round trips count
        dict(name="paged_b1_short", kind="paged", batch=1, heads=32, kv_heads=32, dim=128,
             page=16, max_pages=64, low=300, high=300, layers=1),
        # the MLP block of a single-user decode step (weight streaming)
        dict(name="mlp_b1", kind="mlp", batch=1, hidden=4096, inter=11008, layers=4),
        # the same block at the benchmark's batch
        dict(name="mlp_b16", kind="mlp", batch=16, hidden=4096, inter=11008, layers=4),
        # a busy server: more rows than one matrix-core pass, not a multiple of it
        dict(name="mlp_b50", kind="mlp", batch=50, hidden=4096, inter=11008, layers=2),
        # row-major linear layer of a small batch at odd widths
        dict(name="linear_b7", kind="linear", batch=7, inp=4104, out=5003, layers=4),
        # paged GQA attention of the benchmark: batch 16, up to 4096 positions
        dict(name="paged_gqa_b16", kind="paged", batch=16, heads=32, kv_heads=8, dim=128,
             page=16, max_pages=256, low=65, high=4096, layers=3),
        # head dim 64 grouped-query model, a mid-size batch
        dict(name="paged_d64_b24", kind="paged", batch=24, heads=32, kv_heads=8, dim=64,
             page=16, max_pages=128, low=100, high=2000, layers=3),
        # contiguous cache near its capacity
        dict(name="contig_4095", kind="contig", heads=32, kv_heads=32, dim=128, capacity=4096,
             length=4095, layers=4),
        # the last chunk of a long prompt, grouped-query
        dict(name="pattn_512_at_3584", kind="pattn", rows=512, start=3584, heads=32, kv_heads=8,
             dim=128, page=16, layers=1),
        # a short prompt of odd length through one layer
        dict(name="prompt_200", kind="prompt", rows=200, start=0, hidden=4096, heads=32,
             kv_heads=32, dim=128, inter=11008, page=16, layers=2),
        # a full-size chunk of a long prompt through one layer
        dict(name="prompt_2048", kind="prompt", rows=2048, start=0, hidden=4096, heads=32,
             kv_heads=32, dim=128, inter=11008, page=16, layers=2),
        # the whole decode step of the benchmark at batch 16
        dict(name="step_b16", kind="step", batch=16, layers=32, hidden=4096, heads=32,
             kv_heads=32, dim=128, inter=11008, vocab=32000, capacity=1024, page=16, low=96,
             high=576),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng: random.Random):
    """One more case of the ranges above (batches 1 to 64, contexts up to
    8192 positions, prompt chunks of 16 to 2048 rows)."""
    kind = rng.choice(["mlp", "mlp", "linear", "paged", "paged", "contig", "pattn", "prompt",
                       "prompt", "step"])
    if kind == "mlp":
        return dict(kind=kind, batch=_log(rng, 1, 64), hidden=128 * rng.randint(8, 40),
                    inter=8 * rng.randint(256, 1700), layers=rng.randint(1, 3))
    if kind == "linear":
        return dict(kind=kind, batch=_log(rng, 1, 32), inp=8 * rng.randint(64, 1400),
                    out=_log(rng, 500, 14000), layers=rng.randint(1, 3))
    if kind == "paged":
        group = rng.choice([1, 1, 2, 4, 8])
        batch = _log(rng, 1, 64)
        high = _log(rng, 64, 8192 if batch * 8 // group <= 128 else 2048)
        page = rng.choice([16, 16, 32, 64, 12])
        return dict(kind=kind, batch=batch, heads=32, kv_heads=32 // group,
                    dim=rng.choice([64, 128, 128]), page=page,
                    max_pages=-(-high // page) + rng.randint(0, 16), low=max(1, high // 8),
                    high=high, layers=rng.randint(1, 2))
    if kind == "contig":
        capacity = _log(rng, 128, 8192)
        return dict(kind=kind, heads=32, kv_heads=rng.choice([32, 32, 8]),
                    dim=rng.choice([64, 128, 128]), capacity=capacity,
                    length=rng.randint(capacity // 4, capacity), layers=rng.randint(1, 3))
    if kind == "pattn":
        rows = _log(rng, 16, 2048)
        return dict(kind=kind, rows=rows, start=rng.choice([0, rng.randint(1, 4096 - rows)]),
                    heads=32, kv_heads=rng.choice([32, 16, 8]), dim=rng.choice([64, 128, 128]),
                    page=rng.choice([16, 16, 32, 12]), layers=1)
    if kind == "prompt":
        dim, heads = rng.choice([(128, 32), (128, 16), (64, 32), (128, 20)])
        rows = _log(rng, 16, 2048)
        return dict(kind=kind, rows=rows, start=rng.choice([0, 0, rng.randint(1, 2048)]),
                    hidden=dim * heads, heads=heads, kv_heads=heads // rng.choice([1, 2, 4]),
                    dim=dim, inter=8 * rng.randint(300, 1600), page=16, layers=1)
    dim, heads = rng.choice([(128, 32), (128, 16), (64, 16)])
    high = _log(rng, 48, 1000)
    return dict(kind=kind, batch=_log(rng, 1, 64), layers=rng.randint(2, 8), hidden=dim * heads,
                heads=heads, kv_heads=heads // rng.choice([1, 2, 4]), dim=dim,
                inter=8 * rng.randint(128, 1376), vocab=rng.randint(2000, 32000), capacity=1024,
                page=16, low=max(1, high // 6), high=high)


# ---------------------------------------------------------------- inputs
class _Inputs:
    """Seeded tensors on the GPU: activations ~ N(0, 1), weights ~ N(0, 0.02),
    norm weights ~ U(0.5, 1.5)."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        t = torch.randn(shape, generator=self.g, device="cuda", dtype=F16)
        return t if std == 1.0 else t.mul_(std)

    def weight(self, *shape):
        return self.normal(*shape, std=0.02)

    def gamma(self, width):
        return (torch.rand(width, generator=self.g, device="cuda") + 0.5).to(F16)


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def _lengths(case, seed):
    """Context lengths of the batch: spread over [low, high], the longest at high."""
    rng = random.Random(seed * 7919 + 13)
    out = [rng.randint(case["low"], case["high"]) for _ in range(case["batch"])]
    out[rng.randrange(len(out))] = case["high"]
    return out


def _tables(seed, lengths, page, max_pages):
    """Block tables over a pool of exactly the pages needed, in random order."""
    need = [-(-n // page) for n in lengths]
    order = list(range(sum(need)))
    random.Random(seed * 104729 + 5).shuffle(order)
    rows, at = [], 0
    for n in need:
        rows.append(order[at:at + n] + [-1] * (max_pages - n))
        at += n
    return rows, sum(need)


def _rope_tables(positions, dim):
    p = torch.arange(positions, device="cuda", dtype=torch.float64)[:, None]
    f = 10000.0 ** (-torch.arange(0, dim, 2, device="cuda", dtype=torch.float64) / dim)
    return torch.cos(p * f).float(), torch.sin(p * f).float()


def _make(case, seed):
    """The tensors of one case, from the seed alone: one dict per layer."""
    r = _Inputs(seed)
    kind, out = case["kind"], []
    if kind == "mlp":
        b, h, i = case["batch"], case["hidden"], case["inter"]
        x, u = r.normal(b, h), r.normal(b, h)
        for _ in range(case["layers"]):
            out.append(dict(x=x, u=u, gamma=r.gamma(h), wg=r.weight(i, h), wu=r.weight(i, h),
                            wd=r.weight(h, i)))
    elif kind == "linear":
        x = r.normal(case["batch"], case["inp"])
        for _ in range(case["layers"]):
            out.append(dict(x=x, gamma=r.gamma(case["inp"]), w=r.weight(case["out"], case["inp"])))
    elif kind == "paged":
        lengths = _lengths(case, seed)
        for layer in range(case["layers"]):
            table, pages = _tables(seed + 31 * layer, lengths, case["page"], case["max_pages"])
            pool = (pages, case["kv_heads"], case["page"], case["dim"])
            out.append(dict(q=r.normal(case["batch"], case["heads"] * case["dim"]),
                            k=r.normal(*pool), v=r.normal(*pool), table=table, lengths=lengths))
    elif kind == "contig":
        cache = (1, case["kv_heads"], case["capacity"], case["dim"])
        for _ in range(case["layers"]):
            out.append(dict(q=r.normal(1, case["heads"] * case["dim"]), k=r.normal(*cache),
                            v=r.normal(*cache)))
    else:  # pattn, prompt
        rows, d, kvh = case["rows"], case["dim"], case["kv_heads"]
        end = case["start"] + rows
        for layer in range(case["layers"]):
            table, pages = _tables(seed + 31 * layer, [end], case["page"], -(-end // case["page"]))
            pool = (pages, kvh, case["page"], d)
            one = dict(table=table, k=r.normal(*pool), v=r.normal(*pool))
            if kind == "pattn":
                one["q"] = r.normal(rows, case["heads"] * d)
            else:
                h, i = case["hidden"], case["inter"]
                one.update(x=r.normal(rows, h), g1=r.gamma(h), g2=r.gamma(h),
                           wqkv=r.weight((case["heads"] + 2 * kvh) * d, h),
                           wo=r.weight(h, case["heads"] * d), wg=r.weight(i, h),
                           wu=r.weight(i, h), wd=r.weight(h, i))
            out.append(one)
    return out


# ---------------------------------------------------------------- prepare
class _Plan:
    """Kernels bound to tensors, then captured as one sequence."""

    def __init__(self):
        self.rt, self.steps, self.bound = _runtime(), [], {}

    def _wrap(self, t):
        if id(t) not in self.bound:
            self.bound[id(t)] = self.rt.wrap(t)
        return self.bound[id(t)]

    def add(self, key, inputs, outputs):
        self.steps.append(self.rt.prepare(self.rt.resolve(key), [self._wrap(t) for t in inputs],
                                          [self._wrap(t) for t in outputs]))

    def sequence(self):
        torch.cuda.synchronize()
        return self.rt.sequence(self.steps)


def _empty(*shape, dtype=F16):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def _plan_mlp(case, layers, plan, outputs):
    b, h, i = case["batch"], case["hidden"], case["inter"]
    for t in layers:
        if b == 1:
            s, g, y = _empty(1, h), _empty(1, i), _empty(1, h)
            plan.add(f"add_rmsnorm_gate_up_silu?in={h}&out={i}&eps={EPS}",
                     [t["x"], t["u"], t["gamma"], t["wg"], t["wu"]], [s, g])
            plan.add(f"gemv_residual?in={i}&out={h}", [g, t["wd"], s], [y])
            outputs.append([s, y])
        else:
            t["xp"] = tmc.pack_activations(t["x"])
            wg = tmc.pack_weights(t["wg"], gamma=t["gamma"])
            wu = tmc.pack_weights(t["wu"], gamma=t["gamma"])
            wd = tmc.pack_weights(t["wd"])
            g = _empty(tmc.packed_activation_elements(b, i))
            y = _empty(b, h)
            plan.add(f"gate_up_silu_packed?batch={b}&hidden={h}&inter={i}&norm=1&eps={EPS}"
                     "&x_layout=packed&y_layout=packed", [t["xp"], wg, wu], [g])
            plan.add(f"gemm_packed?batch={b}&in={i}&out={h}&residual=1&x_layout=packed",
                     [g, wd, t["x"]], [y])
            for name in ("wg", "wu", "wd"):  # the program keeps the packed copies
                del t[name]
            outputs.append([y])


def _plan_linear(case, layers, plan, outputs):
    b, k, n = case["batch"], case["inp"], case["out"]
    for t in layers:
        norm, y = _empty(b, k), _empty(b, n, dtype=torch.float32)
        plan.add(f"rmsnorm?rows={b}&width={k}&eps={EPS}&dtype=f16", [t["x"], t["gamma"]], [norm])
        plan.add(f"decode_gemv?batch={b}&in={k}&out={n}&out_dtype=f32", [norm, t["w"]], [y])
        outputs.append([y])


def _plan_paged(case, layers, plan, outputs):
    b, d = case["batch"], case["dim"]
    for t in layers:
        o = _empty(b, case["heads"] * d)
        plan.add(f"paged_attention?max_batch={b}&q_heads={case['heads']}"
                 f"&kv_heads={case['kv_heads']}&head_dim={d}&page_size={case['page']}"
                 f"&max_pages={case['max_pages']}",
                 [t["q"], t["k"], t["v"], _i32(t["lengths"]), _i32(t["table"]), _i32([b])], [o])
        outputs.append([o])


def _plan_contig(case, layers, plan, outputs):
    for t in layers:
        o = _empty(1, case["heads"] * case["dim"])
        plan.add(f"decode_attention?batch=1&q_heads={case['heads']}&kv_heads={case['kv_heads']}"
                 f"&head_dim={case['dim']}&capacity={case['capacity']}",
                 [t["q"], t["k"], t["v"], _i32([case["length"]])], [o])
        outputs.append([o])


def _prompt_geometry(case):
    return (f"rows={case['rows']}&q_heads={case['heads']}&kv_heads={case['kv_heads']}"
            f"&head_dim={case['dim']}&page_size={case['page']}")


def _plan_pattn(case, layers, plan, outputs):
    rows, start = case["rows"], case["start"]
    valid = _i32(list(range(start + 1, start + rows + 1)))
    for t in layers:
        o = _empty(rows, case["heads"] * case["dim"])
        plan.add(f"prefill_attention?{_prompt_geometry(case)}&max_pages={len(t['table'][0])}",
                 [t["q"], t["k"], t["v"], valid, _i32(t["table"][0]), _i32([rows])], [o])
        outputs.append([o])


def _plan_prompt(case, layers, plan, outputs):
    m, h, i, d = case["rows"], case["hidden"], case["inter"], case["dim"]
    qw, kw = case["heads"] * d, case["kv_heads"] * d
    start, geometry = case["start"], _prompt_geometry(case)
    valid, active = _i32(list(range(start + 1, start + m + 1))), _i32([m])
    workspace = torch.zeros(tmc.gemm_rows_workspace_bytes() // 4, dtype=torch.int32, device="cuda")
    capacity = len(layers[0]["table"][0]) * case["page"]
    cos, sin = _rope_tables(capacity, d)
    n, qkv, q, ctx, o = _empty(m, h), _empty(m, qw + 2 * kw), _empty(m, qw), _empty(m, qw), _empty(m, h)
    n2, gate, up, act = _empty(m, h), _empty(m, i), _empty(m, i), _empty(m, i)

    def linear(x, w, y):
        plan.add(f"gemm_rows?m={m}&in={w.shape[1]}&out={w.shape[0]}&workspace=1",
                 [x, w, workspace], [y])

    for t in layers:
        s, y = _empty(m, h), _empty(m, h)
        table = _i32(t["table"][0])
        plan.add(f"rmsnorm?rows={m}&width={h}&eps={EPS}&dtype=f16", [t["x"], t["g1"]], [n])
        linear(n, t["wqkv"], qkv)
        plan.add(f"prefill_rope_append?{geometry}&capacity={capacity}",
                 [qkv, cos, sin, valid, table, active], [q, t["k"], t["v"]])
        plan.add(f"prefill_attention?{geometry}&max_pages={table.numel()}",
                 [q, t["k"], t["v"], valid, table, active], [ctx])
        linear(ctx, t["wo"], o)
        plan.add(f"add_rmsnorm?rows={m}&width={h}&eps={EPS}&dtype=f16", [t["x"], o, t["g2"]],
                 [s, n2])
        linear(n2, t["wg"], gate)
        linear(n2, t["wu"], up)
        plan.add(f"silu_mul?count={m * i}&dtype=f16", [gate, up], [act])
        linear(act, t["wd"], y)
        outputs.append([s, y, t["k"], t["v"]])


class _Pool:
    """A framework-owned device buffer seen as a tensor (fp16)."""

    def __init__(self, pointer, count):
        self.__cuda_array_interface__ = dict(data=(pointer, False), shape=(count,),
                                             typestr="<f2", version=3)


def _prepare_step(case, seed):
    host, rt = tmc.host(), _host_runtime()
    plan, att = host.DecoderLLMPlan(), host.KVCachePlan()
    att.heads, att.head_dimension, att.capacity = case["heads"], case["dim"], case["capacity"]
    att.dtype = host.DType.Float16
    plan.attention = att
    plan.layer_count, plan.intermediate_size = case["layers"], case["inter"]
    plan.vocabulary_size, plan.rms_norm_epsilon = case["vocab"], EPS
    plan.key_value_heads = case["kv_heads"]
    model = host.create_synthetic_model_resources(rt, plan, seed * 1000 + 1)
    lengths, page = _lengths(case, seed), case["page"]
    r = _Inputs(seed)
    pools, tables, caches = [], [], []
    max_pages = -(-case["capacity"] // page)
    pages = max(sum(-(-n // page) for n in lengths), max_pages)
    # the order in which a server's requests take their pages
    turns = [b for b, n in enumerate(lengths) for _ in range(-(-n // page))]
    random.Random(seed * 104729 + 5).shuffle(turns)
    for _ in range(case["layers"]):
        pool = host.create_kv_page_pool(rt, plan.kv_plan(), page, pages)
        count = pages * pool.page_elements()
        for pointer in (pool.key_pointer(), pool.value_pointer()):
            torch.as_tensor(_Pool(pointer, count), device="cuda").copy_(r.normal(count))
        states = [host.create_kv_cache_state(rt, plan.kv_plan(), pool, False) for _ in lengths]
        held = [0] * len(lengths)
        for b in turns:
            held[b] = min(held[b] + page, lengths[b])
            error = states[b].stage_length(rt, held[b]) or states[b].commit_length(held[b])
            if error:
                raise RuntimeError(error)
        pools.append(pool)
        caches.append(states)
        tables.append([p for state in states
                       for p in state.page_table() + [-1] * (max_pages - len(state.page_table()))])
    rng = random.Random(seed)
    return dict(tokens=[rng.randrange(case["vocab"]) for _ in lengths], lengths=lengths,
                tables=tables, model=model, pools=pools, caches=caches,
                executor=host.create_batched_decode_executor(rt, model, pools, case["batch"]))


def prepare(case, seed):
    if case["kind"] == "step":
        return _prepare_step(case, seed)
    layers, plan, outputs = _make(case, seed), _Plan(), []
    {"mlp": _plan_mlp, "linear": _plan_linear, "paged": _plan_paged, "contig": _plan_contig,
     "pattn": _plan_pattn, "prompt": _plan_prompt}[case["kind"]](case, layers, plan, outputs)
    return dict(sequence=plan.sequence(), plan=plan, layers=layers, outputs=outputs)


def run(state):
    if "executor" in state:
        r = state["executor"].run(state["tokens"], state["lengths"], state["tables"], True, False)
        if not r["passed"]:
            raise RuntimeError(r["error"])
        return [r["logits"]]
    state["sequence"].launch()
    return state["outputs"]


# ---------------------------------------------------------------- bounds
def work(case):
    """Bytes read and written once and operations of one pass."""
    kind, layers = case["kind"], case["layers"]
    if kind == "mlp":
        b, h, i = case["batch"], case["hidden"], case["inter"]
        return dict(bytes=layers * (6 * h * i + 2 * h + b * h * (2 if b > 1 else 6) + 2 * b * h),
                    flops=layers * 6.0 * b * h * i)
    if kind == "linear":
        b, k, n = case["batch"], case["inp"], case["out"]
        return dict(bytes=layers * (2 * n * k + 2 * b * k + 2 * k + 4 * b * n),
                    flops=layers * 2.0 * b * n * k)
    d, qh, kvh = case["dim"], case["heads"], case["kv_heads"]
    if kind in ("paged", "step"):
        # the mean of the drawn lengths, of which one is the longest
        b = case["batch"]
        positions = (b - 1) * (case["low"] + case["high"]) / 2 + case["high"]
        kv, att = positions * kvh * d * 4, positions * qh * d * 4.0
        if kind == "paged":
            return dict(bytes=layers * (kv + 4 * b * qh * d), flops=layers * att)
        h, i, v = case["hidden"], case["inter"], case["vocab"]
        weights = layers * (h * (qh + 2 * kvh) * d + h * qh * d + 3 * h * i) + v * h
        return dict(bytes=2 * weights + layers * kv + 4 * b * v,
                    flops=2.0 * b * weights + layers * att)
    if kind == "contig":
        kv = case["length"] * kvh * d * 4
        return dict(bytes=layers * (kv + 4 * qh * d), flops=layers * 4.0 * case["length"] * qh * d)
    m, start = case["rows"], case["start"]
    attended = m * start + m * (m + 1) / 2
    att, kv = 4.0 * attended * qh * d, (start + m) * kvh * d * 4
    if kind == "pattn":
        return dict(bytes=layers * (kv + 4 * m * qh * d), flops=layers * att)
    h, i = case["hidden"], case["inter"]
    weights = h * (qh + 2 * kvh) * d + h * qh * d + 3 * h * i
    return dict(bytes=layers * (2 * weights + 2 * m * h * 3 + kv + m * kvh * d * 4),
                flops=layers * (2.0 * m * weights + att))


def tolerance(case):
    """Against another fp16-in, fp32-accumulate implementation.  Measured
    against 64-bit results of the same inputs, times about four: outputs
    rounded to fp16 after fp16 intermediates, fp32 sums behind an fp16 norm,
    and logits after every layer of a model."""
    return {"mlp": dict(rel=2.5e-3, max=1e-2), "linear": dict(rel=1e-3, max=1e-2),
            "paged": dict(rel=2e-3, max=2e-2), "contig": dict(rel=2e-3, max=2e-2),
            "pattn": dict(rel=2e-3, max=2e-2), "prompt": dict(rel=4e-3, max=3e-2),
            "step": dict(rel=2.5e-2, max=2e-1)}[case["kind"]]


# ---------------------------------------------------------------- 64 bits
def _norm64(x, gamma):
    x = x.double()
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * gamma.double()


def _silu64(g):
    return g / (1.0 + torch.exp(-g))


def _gather64(pool, table, length, page):
    """[length, kv_heads, dim] of one request's pages."""
    pages = torch.tensor(table[:-(-length // page)], device="cuda")
    t = pool[pages].double().permute(0, 2, 1, 3)  # pages, slots, heads, dim
    return t.reshape(-1, t.shape[2], t.shape[3])[:length]


def _attend64(q, k, v, offset):
    """q [rows, heads, dim] against k, v [positions, kv_heads, dim]; row r
    attends the first offset + r + 1 positions."""
    rows, heads, dim = q.shape
    group = heads // k.shape[1]
    out = torch.empty(rows, heads, dim, dtype=torch.float64, device="cuda")
    allowed = (torch.arange(k.shape[0], device="cuda")[None, :]
               <= offset + torch.arange(rows, device="cuda")[:, None])
    for head in range(heads):
        kh, vh = k[:, head // group].contiguous(), v[:, head // group].contiguous()
        s = q[:, head].contiguous() @ kh.t().contiguous() / math.sqrt(dim)
        out[:, head] = torch.softmax(s.masked_fill(~allowed, -math.inf), -1) @ vh
    return out


def _rope64(x, cos, sin):
    """Interleaved pairs of x [rows, heads, dim]."""
    c, s = cos.double()[:, None, :], sin.double()[:, None, :]
    even, odd = x[..., 0::2], x[..., 1::2]
    return torch.stack([even * c - odd * s, even * s + odd * c], -1).reshape(x.shape)


def _exact_prompt(case, t):
    m, d, qh, kvh = case["rows"], case["dim"], case["heads"], case["kv_heads"]
    start, page, end = case["start"], case["page"], case["start"] + case["rows"]
    mat = lambda x, w: x @ w.double().t().contiguous()  # noqa: E731
    cos, sin = _rope_tables(end, d)
    qkv = mat(_norm64(t["x"], t["g1"]), t["wqkv"])
    q, k, v = qkv.split([qh * d, kvh * d, kvh * d], -1)
    q = _rope64(q.reshape(m, qh, d), cos[start:], sin[start:])
    k = _rope64(k.reshape(m, kvh, d), cos[start:], sin[start:])
    v = v.reshape(m, kvh, d)
    pools = []
    position = torch.arange(start, end, device="cuda")
    pages = torch.tensor(t["table"][0], device="cuda")[position // page]
    for pool, new in ((t["k"], k), (t["v"], v)):
        pool = pool.double()
        pool[pages, :, position % page] = new
        pools.append(pool)
    ctx = _attend64(q, _gather64(pools[0], t["table"][0], end, page),
                    _gather64(pools[1], t["table"][0], end, page), start)
    s = t["x"].double() + mat(ctx.reshape(m, qh * d), t["wo"])
    n = _norm64(s, t["g2"])
    return [s, mat(_silu64(mat(n, t["wg"])) * mat(n, t["wu"]), t["wd"]), *pools]


def exact(case, seed):
    kind, out = case["kind"], []
    if kind == "step":
        return None
    for t in _make(case, seed):
        if kind == "mlp":
            s = t["x"].double() + (t["u"].double() if case["batch"] == 1 else 0.0)
            n = _norm64(s, t["gamma"])
            g = _silu64(n @ t["wg"].double().t()) * (n @ t["wu"].double().t())
            y = s + g @ t["wd"].double().t()
            out.append([s, y] if case["batch"] == 1 else [y])
        elif kind == "linear":
            out.append([_norm64(t["x"], t["gamma"]) @ t["w"].double().t()])
        elif kind == "paged":
            q = t["q"].double().reshape(case["batch"], case["heads"], case["dim"])
            rows = []
            for b, length in enumerate(t["lengths"]):
                kv = [_gather64(t[p], t["table"][b], length, case["page"]) for p in ("k", "v")]
                rows.append(_attend64(q[b:b + 1], *kv, length - 1))
            out.append([torch.cat(rows).reshape(case["batch"], -1)])
        elif kind == "contig":
            q = t["q"].double().reshape(1, case["heads"], case["dim"])
            k, v = (t[p][0, :, :case["length"]].double().permute(1, 0, 2) for p in ("k", "v"))
            out.append([_attend64(q, k, v, case["length"] - 1).reshape(1, -1)])
        elif kind == "pattn":
            q = t["q"].double().reshape(case["rows"], case["heads"], case["dim"])
            end = case["start"] + case["rows"]
            k, v = (_gather64(t[p], t["table"][0], end, case["page"]) for p in ("k", "v"))
            out.append([_attend64(q, k, v, case["start"]).reshape(case["rows"], -1)])
        else:
            out.append(_exact_prompt(case, t))
    return out
