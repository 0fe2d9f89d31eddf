"""Performance cases: the calls a serving program makes on one layer's state pool.

A case names its entry point in ``kind``: one decode step (``decode``: eager or
replayed from a HIP graph, fused or with the writer on a side stream, packed
or byte pages), a chunked prefill (``prefill``), a decode step on a
baseline-format pool (``format``), or a copy of prefix pages (``copy``).
K = V = 128 throughout; the page and batch sizes are those of the benchmark
workloads and the range around them.
"""
import math

import torch

from stepquant_amd.formats import FormatPlan, get_format
from stepquant_amd.kernels.format_pool import FormatStatePool
from stepquant_amd.kernels.pool import PackedStatePool
from stepquant_amd.quantization import QuantizationPlan

K = V = 128
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _decode(name, **kw):
    case = dict(name=name, kind="decode", arch="gdn", nominal=6, batch=1, heads=32, key_heads=16, dtype="bf16",
                storage="packed", writer=False, graph=False, layers=1)
    case.update(kw)
    return case


def _prefill(name, **kw):
    case = dict(name=name, kind="prefill", arch="gdn", nominal=6, batch=1, heads=32, key_heads=16, dtype="bf16",
                tokens=2048, ragged=False, checkpoints=1)
    case.update(kw)
    return case


def listed():
    return [
        # one user's chat: a single request's step, launched eagerly
        _decode("decode_gdn6_b1", batch=1),
        # a lightly loaded server: eight requests, four layers in one captured graph
        _decode("decode_gdn6_b8_graph", batch=8, layers=4, graph=True),
        # the headline workload: a full serving batch
        _decode("decode_gdn6_b256", batch=256),
        # the four-bit plan at the largest batch
        _decode("decode_gdn4_b512", nominal=4, batch=512),
        # Kimi-Linear style layers: per-row widths, FP16 pivot rows, per-channel decay
        _decode("decode_kda6_b256", arch="kda", batch=256, key_heads=32),
        # byte pages with the writer on its own stream (byte storage always has one)
        _decode("decode_gdn6_b128_byte", batch=128, storage="byte", writer=True),
        # the prefill workload: eight prompts, five prefix slots each
        _prefill("prefill_gdn6_b8_t2048", batch=8, tokens=2048, checkpoints=5),
        # one long prompt, its final state only
        _prefill("prefill_gdn6_b1_t8192", batch=1, tokens=8192),
        # a few KDA prompts of unequal, odd lengths
        _prefill("prefill_kda6_b3_ragged", arch="kda", batch=3, tokens=3001, key_heads=32, ragged=True, checkpoints=2),
        # many short prompts of unequal lengths in one extend call
        _prefill("prefill_gdn6_b24_ragged", batch=24, tokens=333, ragged=True),
        # the symmetric baseline that a format comparison runs beside the packed pool
        dict(name="format_sym_int6_b256", kind="format", arch="gdn", format="sym_int6_g128", batch=256, heads=32,
             key_heads=16, dtype="bf16"),
        # prefix-cache hits: cached pages copied into the requests' slots
        dict(name="copy_gdn6_n64", kind="copy", arch="gdn", nominal=6, pages=64, heads=32),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode"] * 5 + ["prefill"] * 4 + ["format"] * 2 + ["copy"])
    arch = rng.choice(["gdn", "gdn", "kda"])
    heads = rng.choice([8, 16, 32])
    key_heads = heads if arch == "kda" else rng.choice([heads // 2, heads // 2, heads])
    nominal = rng.choice([6, 6, 4])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
    if kind == "decode":
        case = _decode("", arch=arch, nominal=nominal, heads=heads, key_heads=key_heads, dtype=dtype)
        case["storage"] = rng.choice(["packed", "packed", "packed", "byte"])
        case["writer"] = case["storage"] == "byte" or rng.random() < .25
        case["graph"] = not case["writer"] and rng.random() < .4
        case["layers"] = rng.choice([2, 3, 4]) if case["graph"] else 1
        case["batch"] = _log(rng, 1, 256 if case["writer"] else 512 // case["layers"])
    elif kind == "prefill":
        case = _prefill("", arch=arch, nominal=6, heads=heads, key_heads=key_heads,
                        dtype="bf16" if dtype == "fp32" else dtype)
        case["batch"] = _log(rng, 1, 24)
        most = min(3001 if arch == "kda" else 8192, 16384 // case["batch"])
        case["tokens"] = _log(rng, 32, most)
        case["ragged"] = rng.random() < .6
        case["checkpoints"] = rng.choice([1, 1, 2, 5])
    elif kind == "format":
        case = dict(kind="format", arch=arch, heads=heads, key_heads=key_heads, dtype=dtype,
                    format=rng.choice(["fp32", "sym_int4_g128", "sym_int6_g128", "sym_int8_g128", "dsq_int4",
                                       "dsq_int6"]))
        case["batch"] = _log(rng, 1, 256)
    else:
        case = dict(kind="copy", arch=arch, nominal=nominal, heads=heads, pages=_log(rng, 1, 256))
    case.pop("name", None)
    return case


# ---------------------------------------------------------------- inputs
def _lengths(case):
    """Prompt lengths: all ``tokens``, or spread over [tokens / 6, tokens] with
    the longest ``tokens``."""
    if not case["ragged"]:
        return [case["tokens"]] * case["batch"]
    spread = case["tokens"] * 5 // 6
    return [max(1, case["tokens"] - int(spread * (i * .6180339887 % 1.))) for i in range(case["batch"])]


def _widths(arch, nominal, heads, rng):
    """Widths averaging ``nominal``: per head (GDN) or per key row with 1% FP16
    pivot rows (KDA)."""
    if arch == "gdn":
        if nominal == 6:
            w = [4] * (heads // 4) + [6] * (heads // 2) + [8] * (heads - heads // 4 - heads // 2)
        else:
            n = 3 * heads // 8
            n6 = (heads - 2 * n) // 2
            w = [2] * n + [4] * n + [6] * n6 + [8] * (heads - 2 * n - n6)
        w = torch.tensor(w)[torch.randperm(heads, generator=rng)]
        return w[:, None].expand(heads, K).contiguous()
    choice = torch.tensor([4, 6, 8] if nominal == 6 else [2, 2, 2, 4, 4, 4, 6, 8])
    w = choice[torch.randint(0, choice.numel(), (heads, K), generator=rng)]
    w[torch.rand(heads, K, generator=rng) < .01] = 16
    return w


def _plan(case, dev):
    """The layer's plan: part of the model, whatever its inputs."""
    rng = torch.Generator().manual_seed(0)
    if case["kind"] == "format":
        bits = torch.full((case["heads"], K), get_format(case["format"]).bits, dtype=torch.long)
        return FormatPlan(case["arch"], bits.to(dev), torch.ones(case["heads"], K, device=dev))
    bits = _widths(case["arch"], case["nominal"], case["heads"], rng)
    impact = torch.rand(case["heads"], K, generator=rng) + .5
    return QuantizationPlan(case["arch"], bits.to(dev), impact.to(dev))


def _states(n, case, dev, rng):
    """Recurrent states in use: N(0, 0.05^2), at four bits with log-normal
    key-row and value-column scales."""
    shape = (n, case["heads"], K, V)
    if case.get("nominal") != 4:
        return torch.randn(shape, device=dev, generator=rng) * .05
    r = torch.exp(torch.randn(*shape[:3], 1, device=dev, generator=rng) * .5)
    c = torch.exp(torch.randn(*shape[:2], 1, V, device=dev, generator=rng) * .5)
    return r * torch.randn(shape, device=dev, generator=rng) * c


def _projections(rows, case, dev, rng):
    """q, k, v as column views of one projection's output, raw gates, write
    logits, A_log and dt_bias."""
    h, hk, kda = case["heads"], case["key_heads"], case["arch"] == "kda"
    mixed = torch.randn(rows, 2 * hk * K + h * V, device=dev, generator=rng).to(DTYPES[case["dtype"]])
    q, k, v = mixed.split([hk * K, hk * K, h * V], -1)
    gate = torch.randn(rows, h, K, device=dev, generator=rng) * .5 if kda else \
        torch.randn(rows, h, device=dev, generator=rng)
    beta = torch.randn(rows, h, device=dev, generator=rng)
    a_log = torch.zeros(h, device=dev)
    dt_bias = torch.zeros(h * K if kda else h, device=dev)
    return q, k, v, gate, beta, a_log, dt_bias


def _fill(pool, case, slots, rng):
    for at in range(0, slots.numel(), 128):  # 128 dense states at a time: 268 MB at 32 heads
        part = slots[at:at + 128]
        pool.encode(_states(part.numel(), case, pool.device, rng), part)


def _prepare_decode(case, seed, dev, rng):
    batch, layers = case["batch"], case.get("layers", 1)
    plan = _plan(case, dev)
    if case["kind"] == "format":
        pools = [FormatStatePool(plan, batch + 1, V, get_format(case["format"]))]
    else:
        stream = torch.cuda.Stream() if case["writer"] else None
        pools = [PackedStatePool(plan, batch + 1, V, writeback_stream=stream, storage=case["storage"])
                 for _ in range(layers)]
    slots = (torch.randperm(batch, generator=torch.Generator().manual_seed(seed)) + 1).to(dev)
    for pool in pools:
        _fill(pool, case, slots, rng)
    inputs = [_projections(batch, case, dev, rng) for _ in pools]
    state = dict(kind=case["kind"], pools=pools, slots=slots, inputs=inputs, graph=None)
    if case.get("graph"):
        # a step before the capture, as a server runs one to warm up; its
        # pages are put back
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            pages = [pool.data.clone() for pool in pools]
            _steps(state)
            for pool, page in zip(pools, pages):
                pool.data.copy_(page)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outs = _steps(state)
        state.update(graph=graph, outs=outs)
    return state


def _prepare_prefill(case, seed, dev, rng):
    lengths, n = _lengths(case), case["checkpoints"]
    batch, total = case["batch"], sum(lengths)
    pool = PackedStatePool(_plan(case, dev), batch * (n + 1) + 1, V)
    init = torch.arange(1, batch + 1, device=dev)
    _fill(pool, case, init, rng)
    offsets = torch.tensor([0] + lengths, dtype=torch.int32).cumsum(0).to(torch.int32)  # on the host, as a
    marks = torch.tensor([[max(1, t * (c + 1) // n) for c in range(n)] for t in lengths],  # scheduler holds
                         dtype=torch.int32)                                                # them
    targets = torch.arange(batch + 1, batch + 1 + batch * n).reshape(batch, n)
    return dict(kind="prefill", pool=pool, inputs=_projections(total, case, dev, rng), init=init, offsets=offsets,
                marks=marks, targets=targets, lengths=lengths)


def prepare(case, seed):
    dev = torch.device("cuda:0")
    rng = torch.Generator(device=dev).manual_seed(seed)
    if case["kind"] in ("decode", "format"):
        return _prepare_decode(case, seed, dev, rng)
    if case["kind"] == "prefill":
        return _prepare_prefill(case, seed, dev, rng)
    n = case["pages"]
    pool = PackedStatePool(_plan(case, dev), 2 * n + 1, V)
    order = torch.randperm(2 * n, generator=torch.Generator().manual_seed(seed)).to(dev) + 1
    _fill(pool, case, order[:n].contiguous(), rng)
    return dict(kind="copy", pool=pool, source=order[:n].contiguous(), target=order[n:].contiguous())


# ---------------------------------------------------------------- one pass
def _steps(state):
    outs = []
    for pool, (q, k, v, gate, beta, a_log, dt_bias) in zip(state["pools"], state["inputs"]):
        outs.append(pool.step(q, k, v, gate, beta, state["slots"], normalize=True, scale=K ** -.5, a_log=a_log,
                              dt_bias=dt_bias))
    return outs


def _pages(pool):
    """The pool's pages: bytes, or the fp32 format's numbers."""
    return pool.float_data if getattr(pool, "floating", False) else pool.data


def run(state):
    """One pass; returns its outputs and the pool's pages."""
    if state["kind"] == "copy":
        state["pool"].copy(state["source"], state["target"])
        return {"pages": state["pool"].data}
    if state["kind"] == "prefill":
        q, k, v, gate, beta, a_log, dt_bias = state["inputs"]
        out = state["pool"].extend(q, k, v, gate, beta, state["init"], state["offsets"], checkpoints=state["marks"],
                                   checkpoint_slots=state["targets"], init_slots=state["init"], normalize=True,
                                   scale=K ** -.5, a_log=a_log, dt_bias=dt_bias)
        return {"out": out, "pages": state["pool"].data}
    if state["graph"] is not None:
        state["graph"].replay()
        outs = state["outs"]
    else:
        outs = _steps(state)
    for pool in state["pools"]:
        pool.wait()  # the next reader of the pages comes after their writer
    return {"out": outs, "pages": [_pages(pool) for pool in state["pools"]]}


# ---------------------------------------------------------------- cost
def _page_bytes(case):
    """Bytes of one page: codes and scales."""
    h = case["heads"]
    if case["kind"] == "format":
        spec = get_format(case["format"])
        meta = {"fp32": 0, "symmetric": 4 * K, "dsq": 2 * K + 4 * V}[spec.kind]
        return h * (K * V * spec.bits // 8 + meta)
    bits = 8 if case.get("storage") == "byte" else case["nominal"]
    return h * (K * V * bits // 8 + 2 * K + 2 * V)


def work(case):
    page, h = _page_bytes(case), case["heads"]
    if case["kind"] == "copy":
        return {"bytes": 2 * page * case["pages"], "flops": 0}
    hk, kda, n = case["key_heads"], case["arch"] == "kda", DTYPES[case["dtype"]].itemsize
    row = (2 * hk * K + 2 * h * V) * n + (h * K if kda else h) * 4 + h * 4  # q, k, v, out, gate, beta
    if case["kind"] != "prefill":
        tiles = case["batch"] * case.get("layers", 1)
        return {"bytes": tiles * (2 * page + row), "flops": tiles * h * 7 * K * V}
    lengths = _lengths(case)
    total, c = sum(lengths), 32 if kda else 64
    chunk = 6 * c * c * K + 4 * c * c * V + 6 * c * K * V + 2 * c ** 3 // 3
    return {"bytes": total * row + case["batch"] * (1 + case["checkpoints"]) * page,
            "flops": total * h * chunk / c}


def tolerance(case):
    """Outputs: values at a rounding boundary of the output type (measured
    against float64 rounded to it: 4e-5, fp16 1e-5, fp32 1.4e-7; prefill
    1.6e-4).  Pages: codes at a boundary and the column scales that follow
    them (measured 2e-5 of the bytes, prefill 5e-4)."""
    if case["kind"] == "copy":
        return "exact"
    if case["kind"] == "prefill":
        return {"rel": 6e-4, "max": .03, "differ": 2e-3}
    rel, most = {"bf16": (2e-4, .016), "fp16": (5e-5, .002), "fp32": (1e-6, 1e-5)}[case["dtype"]]
    return {"rel": rel, "max": most, "differ": 1e-4}


# ---------------------------------------------------------------- 64 bits
def _codes(pages, base, width, stride, tile):
    """Codes [n, rows, V] of rows that start ``base`` bytes into their page."""
    j = torch.arange(V, device=pages.device)
    bit = (j % tile) * width
    at = base[:, None] + (j // tile) * stride + bit // 8
    # a code spans two bytes at most; the last one may end its page
    low = pages[:, at].long()
    high = pages[:, (at + 1).clamp_max(pages.shape[1] - 1)].long()
    return (low + 256 * high >> bit % 8) & ((1 << width) - 1)


def _halves(pages, at):
    both = pages[:, torch.stack([at, at + 1], -1)].contiguous()
    return both.view(torch.float16)[..., 0].double()


def _dense(pool, slots, case):
    """Dense float64 states [n, heads, K, V] of the slots' pages."""
    pages = pool.data[slots]
    dev, h = pages.device, case["heads"]
    offsets, rows, columns = pool.offsets.long(), pool.rows.long(), pool.columns.long()
    bits, j = pool.bits.long(), torch.arange(V, device=dev)
    state = torch.zeros(slots.numel(), h, K, V, device=dev, dtype=torch.float64)
    for i in range(h):
        base, row = offsets[i * K:(i + 1) * K], rows[i * K:(i + 1) * K]
        if case["kind"] == "format":
            state[:, i] = _dense_format(pages, get_format(case["format"]), base, row, columns[i], j)
            continue
        kda, byte = case["arch"] == "kda", case.get("storage") == "byte"
        tail = offsets[h * K + i]
        for width in bits[i].unique().tolist():
            pick = (bits[i] == width).nonzero()[:, 0]
            if width == 16:
                step = 2 * j if byte else (j // 4 if kda else j // 16) * tail + 2 * (j % (4 if kda else 16))
                state[:, i, pick] = _halves(pages, base[pick][:, None] + step)
                continue
            if byte:
                z = pages[:, tail + pick[:, None] + j * K].view(torch.int8).double()
            else:
                code = _codes(pages, base[pick], width, tail, 4 if kda else 16).double()
                z = 2 * code - 3 if width == 2 and not kda else (code - (2 ** (width - 1) - 1)) * (
                    2 ** (8 - width) if kda else 1)
            group = 2 * (j // pool.plan.value_group_size) if width == 2 and not kda else 0 * j
            state[:, i, pick] = _halves(pages, row[pick][:, None] + group) * _halves(pages, columns[i] + 2 * j)[:, None] * z
    return state


def _dense_format(pages, spec, base, row, column, j):
    if spec.kind == "fp32":
        at = base[:, None, None] + 4 * j[:, None] + torch.arange(4, device=j.device)
        return pages[:, at].contiguous().view(torch.float32)[..., 0].double()
    code = _codes(pages, base, spec.bits, 16 * spec.bits // 8, 16).double()
    if spec.kind == "dsq":
        return _halves(pages, row)[..., None] * _halves(pages, column + 4 * j)[:, None] * (code - (2 ** (spec.bits - 1) - 1))
    return (code - _halves(pages, row + 2)[..., None]) * _halves(pages, row)[..., None]


def _prepared(inputs, case):
    """q, k, v, retention and write strength per value head, in float64."""
    q, k, v, gate, beta, a_log, dt_bias = (t.double() for t in inputs)
    n, h, hk = q.shape[0], case["heads"], case["key_heads"]
    q, k = (t.reshape(n, hk, K) for t in (q, k))
    q, k = (t / (t.square().sum(-1, keepdim=True) + 1e-6).sqrt() for t in (q, k))
    q, k = (t.repeat_interleave(h // hk, 1) for t in (q * K ** -.5, k))
    gate = gate.reshape(n, h, -1)
    keep = torch.exp(-a_log.exp()[:, None] * torch.nn.functional.softplus(gate + dt_bias.reshape(h, -1)))
    return q, k, v.reshape(n, h, V), keep, beta.sigmoid()


def _token(state, q, k, v, keep, beta):
    """One token of the gated delta rule on [n, h, K, V], in place."""
    state *= keep[..., None]
    delta = beta[..., None] * (v - torch.matmul(k.unsqueeze(-2), state).squeeze(-2))
    state += k[..., None] * delta[..., None, :]
    return torch.matmul(q.unsqueeze(-2), state).squeeze(-2)


def exact(case, seed):
    if case["kind"] == "copy":
        return None
    state = prepare(case, seed)
    if case["kind"] != "prefill":
        outs = [_token(_dense(pool, state["slots"], case), *_prepared(inputs, case))
                for pool, inputs in zip(state["pools"], state["inputs"])]
        return {"out": outs, "pages": None}
    lengths = torch.tensor(state["lengths"], device=state["init"].device)
    start = state["offsets"].to(lengths.device)[:-1].long()
    q, k, v, keep, beta = _prepared(state["inputs"], case)
    dense = _dense(state["pool"], state["init"], case)
    out = torch.zeros_like(v)
    order = torch.argsort(lengths, descending=True)  # the longest first: the sequences still running lead
    dense, start, running = dense[order], start[order], sorted(state["lengths"], reverse=True)
    live = len(running)
    for t in range(running[0]):
        while running[live - 1] <= t:
            live -= 1
        at = start[:live] + t
        out[at] = _token(dense[:live], q[at], k[at], v[at], keep[at], beta[at])
    return {"out": out, "pages": None}
