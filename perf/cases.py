"""The work that this framework's performance is measured on.

Every case goes through the package's public entry points, as a serving or
training program calls them.  Sizes are those of the repository's benchmark
configurations and tests (7 SDM layers, N = 256 slots, width 128, top-4
writes and top-16 reads, batch 1 to 64, several memory heads, tables of up
to 65,536 slots) and the ranges around them.

Kinds:

* ``step``        one decode step of one layer with its capacity proof
                  (``decode_sdm_layer``): the reference's per-layer call.
* ``trace``       consecutive steps of every layer whose routes are resident
                  (``DecodeTrace.run``): teacher-forced or replayed decode,
                  the benchmark's loop.
* ``graph``       one token through every layer, controller included, as one
                  captured replay (``ControllerDecodeGraph``).
* ``stack``       the same token through ``decode_faithful_sdm_stack``.
* ``prefill``     one layer over a prefix (``prefill_sdm_layer``).
* ``recurrence``  the training forward of one layer's memory: sparse routes
                  scattered to dense vectors (``dense_sparse_routes``), then
                  the recurrence with every token's memory kept for the
                  backward (``sdm_recurrence(return_states=True)``).
* ``turnover``    continuous batching: finished requests are released, the
                  batch compacted, a prefilled cohort packed and admitted.

Selections must not hang on the last bit of a 32-bit sum, or two correct
orders of summation give other rows and all that follows differs: tokens
whose routes are decided by less than ``MARGIN`` are drawn again.
"""

from __future__ import annotations

import math

import torch

import copy_on_write_sdm_amd as cow

MARGIN = 1e-5
DEVICE = "cuda"


# ------------------------------------------------------------------- cases


def listed():
    return [
        # the smallest call: one request, one layer, launch latency
        dict(name="step-b1", kind="step", batch=1, heads=1, slots=256, width=128, writes=4,
             reads=16, index="int64", floats="float32", filled=0.4),
        # a bfloat16 model's step: route weights, values and gates come in 16 bits
        dict(name="step-bf16", kind="step", batch=48, heads=2, slots=1024, width=64, writes=4,
             reads=16, index="int64", floats="bfloat16", filled=0.5),
        # more banks than one wave's first-touch table, a large table filling up
        dict(name="step-b512-n16k", kind="step", batch=128, heads=4, slots=16384, width=128,
             writes=4, reads=16, index="int32", floats="float32", filled=0.0),
        # the benchmark's run of 20 steps, 7 layers at batch 64, after a prefix
        dict(name="trace-20", kind="trace", layers=7, batch=64, slots=256, width=128, writes=4,
             reads=16, steps=20, recorded=400, index="int32", filled=0.98),
        # its long run, at the occupancy of a trained model
        dict(name="trace-512", kind="trace", layers=7, batch=64, slots=256, width=128, writes=4,
             reads=16, steps=512, recorded=512, index="int32", filled=0.37),
        # one token of 64 requests through 7 layers, captured
        dict(name="graph-b64", kind="graph", layers=7, batch=64, width=128, heads=1, slots=256,
             writes=4, reads=16, filled=0.6),
        # one token of 16 requests through 7 layers, launched call by call
        dict(name="stack-b16", kind="stack", layers=7, batch=16, width=128, heads=1, slots=256,
             writes=4, reads=16, filled=0.6),
        # the prefix of a small cohort being admitted
        dict(name="prefill-b4-t128", kind="prefill", batch=4, time=128, width=128, heads=1,
             slots=256, writes=4, reads=16),
        # the long prefix at full batch: the largest call
        dict(name="prefill-b64-t2048", kind="prefill", batch=64, time=2048, width=128, heads=1,
             slots=256, writes=4, reads=16),
        # several heads, a wider model, ragged sizes, the largest table of the recurrence
        dict(name="prefill-h4-n1024", kind="prefill", batch=7, time=333, width=400, heads=4,
             slots=1024, writes=6, reads=24),
        # the training forward, every token's memory kept
        dict(name="recurrence-states", kind="recurrence", batch=16, time=128, slots=256,
             width=128, writes=4, reads=16, states=True),
        # 16 of 64 requests finish and 16 prefilled ones take their place, 7 layers
        dict(name="turnover-16-of-64", kind="turnover", layers=7, batch=64, incoming=16,
             time=256, slots=256, width=128, writes=4, filled=0.5),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["step", "trace", "graph", "stack", "prefill", "prefill", "recurrence",
                       "turnover"])
    if kind == "step":
        heads = rng.choice([1, 2, 4])
        wide = rng.random() < 0.2          # beyond the usual route counts
        writes = rng.randint(5, 16) if wide else rng.randint(1, 4)
        slots = _log_int(rng, 64, 16384)
        return dict(kind=kind, batch=_log_int(rng, 1, 512 // heads), heads=heads, slots=slots,
                    width=rng.choice([32, 64, 100, 128, 128, 160, 256, 320]), writes=writes,
                    reads=min(slots, rng.randint(17, 64) if wide else rng.randint(4, 16)),
                    index=rng.choice(["int32", "int64"]),
                    floats=rng.choice(["float32", "float32", "bfloat16", "float16"]),
                    filled=0.0 if slots > 4096 else round(rng.uniform(0.1, 1.0), 2))
    if kind == "trace":
        steps = _log_int(rng, 8, 512)
        return dict(kind=kind, layers=rng.randint(1, 7), batch=_log_int(rng, 1, 64),
                    slots=_log_int(rng, 64, 4096), width=rng.choice([64, 100, 128, 128]),
                    writes=rng.randint(1, 4), reads=rng.randint(4, 16), steps=steps,
                    recorded=steps * max(1, min(8, 256 // steps)),
                    index=rng.choice(["int32", "int64"]), filled=round(rng.uniform(0.1, 1.0), 2))
    if kind in ("graph", "stack"):
        heads = rng.choice([1, 1, 2, 4])
        root = rng.randint(8, 32)
        return dict(kind=kind, layers=rng.randint(1, 7), batch=_log_int(rng, 1, 64),
                    width=heads * rng.choice([32, 48, 64, 100, 128]), heads=heads,
                    slots=root * root, writes=rng.randint(1, 4), reads=rng.randint(4, 16),
                    filled=round(rng.uniform(0.1, 1.0), 2))
    if kind == "prefill":
        heads = rng.choice([1, 1, 2, 4])
        width = heads * rng.choice([32, 50, 64, 96, 128])
        batch = _log_int(rng, 1, 64)
        root = rng.randint(8, 32)
        most = min(2048, 131072 * 128 // (batch * width))
        return dict(kind=kind, batch=batch, time=_log_int(rng, 16, most), width=width,
                    heads=heads, slots=root * root, writes=rng.randint(1, 8),
                    reads=rng.randint(4, 32))
    if kind == "recurrence":
        states = rng.random() < 0.6
        batch, slots = _log_int(rng, 1, 64), _log_int(rng, 32, 1024)
        width = rng.choice([32, 64, 100, 128, 256])
        most = (1 << (27 if states else 31)) // (batch * slots * width)
        return dict(kind=kind, batch=batch, time=_log_int(rng, 8, max(8, min(1024, most))),
                    slots=slots, width=width, writes=rng.randint(1, 8),
                    reads=rng.randint(4, 32), states=states)
    batch = _log_int(rng, 2, 64)
    return dict(kind=kind, layers=rng.randint(1, 7), batch=batch,
                incoming=rng.randint(1, max(1, batch // 2)), time=_log_int(rng, 16, 1024),
                slots=_log_int(rng, 64, 1024), width=rng.choice([64, 100, 128, 128]),
                writes=rng.randint(1, 4), filled=round(rng.uniform(0.1, 1.0), 2))


# ------------------------------------------------------------------ inputs


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed) * 1_000_003 + 17)
    return g


def _routes(g, rows, slots, k, dtype=torch.int64):
    """k distinct slots of each row, ascending, and softmax weights."""

    chunk = max(1, (1 << 27) // slots)
    parts = [torch.rand(min(chunk, rows - at), slots, generator=g, device=DEVICE)
             .topk(k, dim=1).indices.sort(dim=1).values for at in range(0, rows, chunk)]
    weights = torch.softmax(torch.randn(rows, k, generator=g, device=DEVICE), dim=1)
    return torch.cat(parts).to(dtype), weights


def _gates(g, *shape):
    """(input gate = sigmoid(N(0, 1)), forget log gate = -U(0, 1))"""

    return (torch.sigmoid(torch.randn(*shape, generator=g, device=DEVICE)),
            -torch.rand(*shape, generator=g, device=DEVICE))


def _memories(g, layers, heads, slots, width):
    return [0.02 * torch.randn(heads, slots, width, generator=g, device=DEVICE)
            for _ in range(layers)]


def _tables(g, m0s, batch, filled):
    """Per layer the dense tables a prefix leaves and the mask of the slots it wrote."""

    finals, masks = [], []
    for m0 in m0s:
        heads, slots, width = m0.shape
        mask = torch.rand(batch * heads, slots, generator=g, device=DEVICE) < filled
        final = m0.repeat(batch, 1, 1)
        final += (0.3 * torch.randn(final.shape, generator=g, device=DEVICE)
                  * mask.unsqueeze(-1))
        finals.append(final)
        masks.append(mask)
    return finals, masks


def _zero_free_rows(state):
    """No row of the slab or its headroom is left as the allocator found it."""

    free = int(state.free_count)
    state.values[state.free_rows[:free].long()] = 0
    if state.slab_buffers is not None:
        state.slab_buffers[0][state.capacity_rows:].zero_()


def _states(m0s, finals, masks, batch, writes):
    """The packed states after the handoff, growing four steps at a time, with room
    in the slab's buffers for the largest the decode can make them."""

    heads, slots, _ = m0s[0].shape
    banks = batch * heads
    quantum = max(16, banks * writes * 4)
    states = cow.PackedSDMCopyOnWriteState.from_dense_overlay_layers(
        m0s, finals, masks, growth_quantum_rows=quantum,
        template_indices=torch.arange(heads, device=DEVICE).repeat(batch))
    for state in states:
        state.reserve_rows(banks * slots + banks * writes + 2 * quantum)
        _zero_free_rows(state)
    return states


def _parameters(case, g):
    """One layer's controller parameters, distributed as after initialisation and a
    little training (no bias left at zero)."""

    width, heads, root = case["width"], case["heads"], math.isqrt(case["slots"])
    std = width ** -0.5

    def normal(*shape, scale):
        return scale * torch.randn(*shape, generator=g, device=DEVICE)

    def linear(out):
        return normal(out, width, scale=std), normal(out, scale=0.1)

    def norm(n, eps):
        return 1 + normal(n, scale=0.1), normal(n, scale=0.1), eps

    key = heads * 2 * root
    return dict(
        input_norm=norm(width, 1e-5), read_projection=linear(key), write_projection=linear(key),
        value_projection=linear(width), forget_projection=linear(heads),
        input_projection=linear(heads),
        a_log=torch.log(0.5 + 2 * torch.rand(heads, generator=g, device=DEVICE)),
        dt_bias=normal(heads, scale=0.5) - 3, output_gate=linear(width),
        output_projection=linear(width), readings_norm=norm(width // heads, 1e-6))


def _controller(case, parameters):
    return cow.SDMController.from_parts(
        width=case["width"], slots=case["slots"], reads=case["reads"], writes=case["writes"],
        memory_heads=case["heads"], device=DEVICE, **parameters)


# ----------------------------------------- the same arithmetic in 64 bits


def _norm64(x, norm):
    weight, bias, eps = norm
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), weight.double(), bias.double(), eps)


def _linear64(x, layer):
    return torch.nn.functional.linear(x, layer[0].double(), layer[1].double())


def _select64(keys, root, k):
    """Per row the top k pair sums' slots (ascending), softmax weights, and the gap
    between the last pair taken and the first one left."""

    k = min(k, min(k, root) ** 2)
    slots, weights, gaps = [], [], []
    for part in keys.split(max(1, (1 << 26) // (root * root))):
        sums = (part[:, :root, None] + part[:, None, root:]).flatten(1)
        top = sums.topk(min(k + 1, root * root), dim=1)
        order = top.indices[:, :k].sort(dim=1)
        slots.append(order.values)
        weights.append(torch.softmax(top.values[:, :k], dim=1).gather(1, order.indices))
        gaps.append(top.values[:, k - 1] - top.values[:, k] if top.values.shape[1] > k
                    else torch.full_like(top.values[:, 0], math.inf))
    return torch.cat(slots), torch.cat(weights), torch.cat(gaps)


def _prepare64(p, case, x):
    """The controller's outputs of tokens x [n, width], bank n * H + h."""

    n, heads, root = x.shape[0], case["heads"], math.isqrt(case["slots"])
    normalized = _norm64(x.double(), p["input_norm"])
    read = _select64(_linear64(normalized, p["read_projection"]).reshape(n * heads, 2 * root),
                     root, case["reads"])
    write = _select64(_linear64(normalized, p["write_projection"]).reshape(n * heads, 2 * root),
                      root, case["writes"])
    forget = -p["a_log"].double().exp() * torch.nn.functional.softplus(
        _linear64(normalized, p["forget_projection"]) + p["dt_bias"].double())
    gaps = torch.minimum(read[2], write[2]).reshape(n, heads).amin(dim=1)
    return dict(normalized=normalized, read_indices=read[0], read_weights=read[1],
                write_indices=write[0], write_weights=write[1],
                values=_linear64(normalized, p["value_projection"]).reshape(n * heads, -1),
                input_gate=torch.sigmoid(_linear64(normalized, p["input_projection"])).flatten(),
                forget_log_gate=forget.flatten()), gaps


def _finish64(p, normalized, reading):
    r = _norm64(reading, p["readings_norm"]).reshape(normalized.shape)
    return _linear64(torch.sigmoid(_linear64(normalized, p["output_gate"])) * r,
                     p["output_projection"])


def _update64(table, banks, x):
    """One step of every bank on float64 tables [B, N, D], in place; the readings."""

    write = x["write_indices"].long()
    weights = x["write_weights"].double().unsqueeze(-1)
    gate = x["input_gate"].double().unsqueeze(-1)
    rows = table[banks, write] * x["forget_log_gate"].double().exp()[:, None, None]
    delta = gate * (x["values"].double() - (weights * rows).sum(dim=1))
    table[banks, write] = rows + weights * delta.unsqueeze(1)
    return (x["read_weights"].double().unsqueeze(-1)
            * table[banks, x["read_indices"].long()]).sum(dim=1)


def _tokens64(case, parameters, finals, tokens, passes):
    """``passes`` times the same token of every request through every layer, the
    tables updated in between: the last pass's output and each request's smallest gap."""

    tables = [f.double() for f in finals]
    banks = torch.arange(tables[0].shape[0], device=DEVICE).unsqueeze(1)
    least = torch.full((tokens.shape[0],), math.inf, device=DEVICE, dtype=torch.float64)
    for _ in range(passes):
        x = tokens[:, 0].double()
        for p, table in zip(parameters, tables):
            step, gaps = _prepare64(p, case, x)
            least = torch.minimum(least, gaps)
            x = x + _finish64(p, step["normalized"], _update64(table, banks, step))
    return x.unsqueeze(1), least


# ----------------------------------------------------------------- prepare


def _step_inputs(case, g, steps):
    banks = case["batch"] * case["heads"]
    index, floats = getattr(torch, case["index"]), getattr(torch, case["floats"])
    out = []
    for _ in range(steps):
        wi, ww = _routes(g, banks, case["slots"], case["writes"], index)
        ri, rw = _routes(g, banks, case["slots"], case["reads"], index)
        gate, forget = _gates(g, banks)
        out.append(cow.SDMStepInputs(
            write_indices=wi, write_weights=ww.to(floats),
            values=torch.randn(banks, case["width"], generator=g, device=DEVICE).to(floats),
            input_gate=gate.to(floats), forget_log_gate=forget.to(floats), read_indices=ri,
            read_weights=rw.to(floats)))
    return out


def _prepare_step(case, g):
    m0 = _memories(g, 1, case["heads"], case["slots"], case["width"])
    if case["filled"]:
        finals, masks = _tables(g, m0, case["batch"], case["filled"])
    else:
        finals = masks = None
    steps = _step_inputs(case, g, 8)
    return m0, finals, masks, steps


def _prepare_trace(case, g):
    layers, batch, recorded = case["layers"], case["batch"], case["recorded"]
    m0s = _memories(g, layers, 1, case["slots"], case["width"])
    finals, masks = _tables(g, m0s, batch, case["filled"])
    shape = (recorded, layers, batch)
    rows = recorded * layers * batch
    index = getattr(torch, case["index"])
    wi, ww = _routes(g, rows, case["slots"], case["writes"], index)
    ri, rw = _routes(g, rows, case["slots"], case["reads"], index)
    gate, forget = _gates(g, *shape)
    inputs = dict(
        write_indices=wi.view(*shape, -1), write_weights=ww.view(*shape, -1),
        values=torch.randn(*shape, case["width"], generator=g, device=DEVICE),
        input_gate=gate, forget_log_gate=forget, read_indices=ri.view(*shape, -1),
        read_weights=rw.view(*shape, -1))
    return m0s, finals, masks, inputs


def _prepare_tokens(case, g):
    parameters = [_parameters(case, g) for _ in range(case["layers"])]
    m0s = _memories(g, case["layers"], case["heads"], case["slots"],
                    case["width"] // case["heads"])
    finals, masks = _tables(g, m0s, case["batch"], case["filled"])
    tokens = torch.randn(case["batch"], 1, case["width"], generator=g, device=DEVICE)
    for _ in range(8):
        close = _tokens64(case, parameters, finals, tokens, 2)[1] < MARGIN
        if not bool(close.any()):
            break
        tokens[close] = torch.randn(int(close.sum()), 1, case["width"], generator=g,
                                    device=DEVICE)
    return parameters, m0s, finals, masks, tokens


def _prepare_prefill(case, g):
    parameters = _parameters(case, g)
    m0 = _memories(g, 1, case["heads"], case["slots"], case["width"] // case["heads"])[0]
    tokens = torch.randn(case["batch"] * case["time"], case["width"], generator=g,
                         device=DEVICE)
    ask = torch.arange(tokens.shape[0], device=DEVICE)
    for _ in range(8):
        close = ask[_prepare64(parameters, case, tokens[ask])[1] < MARGIN]
        if not close.numel():
            break
        tokens[close] = torch.randn(close.numel(), case["width"], generator=g, device=DEVICE)
        ask = close
    return parameters, m0, tokens.reshape(case["batch"], case["time"], case["width"])


def _prepare_recurrence(case, g):
    batch, time, slots, width = (case[k] for k in ("batch", "time", "slots", "width"))
    wi, ww = _routes(g, batch * time, slots, min(case["writes"], slots))
    ri, rw = _routes(g, batch * time, slots, min(case["reads"], slots))
    gate, forget = _gates(g, batch, time)
    return dict(
        memory=0.02 * torch.randn(batch, slots, width, generator=g, device=DEVICE),
        write_indices=wi.view(batch, time, -1), write_weights=ww.view(batch, time, -1),
        read_indices=ri.view(batch, time, -1), read_weights=rw.view(batch, time, -1),
        values=torch.randn(batch, time, width, generator=g, device=DEVICE),
        input_gate=gate, forget_log_gate=forget)


def _decode_state(states, batch):
    return cow.FaithfulSDMDecodeState(
        layout="B" * len(states), position=0, capacity=1 << 30, activation_dtype=torch.float32,
        active_sequences=torch.ones(batch, dtype=torch.bool, device=DEVICE),
        sdm_layer_positions=tuple(range(len(states))), sdm_states=tuple(states))


def prepare(case, seed):
    g, kind = _generator(seed), case["kind"]
    if kind == "step":
        m0, finals, masks, steps = _prepare_step(case, g)
        if finals is not None:
            state = _states(m0, finals, masks, case["batch"], case["writes"])[0]
        else:
            banks = case["batch"] * case["heads"]
            quantum = max(16, banks * case["writes"] * 4)
            state = cow.PackedSDMCopyOnWriteState.allocate(
                m0[0], banks=banks, capacity_rows=quantum, growth_quantum_rows=quantum,
                template_indices=torch.arange(case["heads"], device=DEVICE).repeat(case["batch"]))
            state.reserve_rows(quantum * 8)
            _zero_free_rows(state)
        return dict(kind=kind, state=state, steps=steps, at=0)
    if kind == "trace":
        m0s, finals, masks, inputs = _prepare_trace(case, g)
        states = _states(m0s, finals, masks, case["batch"], case["writes"])
        outputs = torch.zeros(case["recorded"], case["layers"], case["batch"], case["width"],
                              device=DEVICE)
        trace = cow.DecodeTrace(states=states, outputs=outputs, **inputs)
        return dict(kind=kind, trace=trace, states=states, steps=case["steps"],
                    recorded=case["recorded"], at=0)
    if kind in ("graph", "stack"):
        parameters, m0s, finals, masks, tokens = _prepare_tokens(case, g)
        controllers = [_controller(case, p) for p in parameters]
        states = _states(m0s, finals, masks, case["batch"], case["writes"])
        if kind == "stack":
            return dict(kind=kind, controllers=controllers, tokens=tokens, states=states,
                        decode=_decode_state(states, case["batch"]))
        graph = cow.ControllerDecodeGraph(controllers, states, case["batch"])
        graph.reserve_tokens(1 << 20)
        graph.capture()
        return dict(kind=kind, graph=graph, tokens=tokens, states=states)
    if kind == "prefill":
        parameters, m0, tokens = _prepare_prefill(case, g)
        return dict(kind=kind, controller=_controller(case, parameters), m0=m0, tokens=tokens)
    if kind == "recurrence":
        return dict(kind=kind, slots=case["slots"], states=case["states"],
                    **_prepare_recurrence(case, g))
    m0s = _memories(g, case["layers"], 1, case["slots"], case["width"])
    finals, masks = _tables(g, m0s, case["batch"], case["filled"])
    states = _states(m0s, finals, masks, case["batch"], case["writes"])
    new, _ = _tables(g, m0s, case["incoming"], 1.0)
    routes = [_routes(g, case["incoming"] * case["time"], case["slots"], case["writes"])[0]
              .view(case["incoming"], case["time"], 1, case["writes"]) for _ in m0s]
    return dict(kind=kind, decode=_decode_state(states, case["batch"]), m0s=m0s, routes=routes,
                finals=[t.unsqueeze(1) for t in new], incoming=case["incoming"],
                quantum=max(16, case["incoming"] * case["writes"] * 4))


# --------------------------------------------------------------------- run


def _layer_outputs(states):
    # the slab with its headroom, whose size growth does not change
    return [[s.slab_buffers[0], s.logical_to_physical, s.free_count] for s in states]


def run(s):
    kind = s["kind"]
    if kind == "step":
        step = s["steps"][s["at"]]
        s["at"] = (s["at"] + 1) % len(s["steps"])
        reading = cow.decode_sdm_layer(s["state"], step)
        return [reading, _layer_outputs([s["state"]])]
    if kind == "trace":
        at = s["at"]
        if at + s["steps"] > s["recorded"]:
            at = 0
            s["trace"].set_step(0)
        s["trace"].run(s["steps"])
        s["at"] = at + s["steps"]
        return [s["trace"].outputs[at:at + s["steps"]], _layer_outputs(s["states"])]
    if kind == "graph":
        # the graph's output buffer is rewritten by the next token
        return [s["graph"](s["tokens"]), _layer_outputs(s["states"])]
    if kind == "stack":
        out = cow.decode_faithful_sdm_stack(s["decode"].layout, s["controllers"], s["tokens"],
                                            s["decode"])
        return [out, _layer_outputs(s["states"])]
    if kind == "prefill":
        p = cow.prefill_sdm_layer(s["controller"], s["m0"], s["tokens"])
        return [p.output, p.final_memory, p.values, p.input_gate, p.forget_log_gate,
                p.read_weights, p.write_weights, p.read_indices, p.write_indices]
    if kind == "recurrence":
        write = cow.dense_sparse_routes(s["write_weights"], s["write_indices"], s["slots"])
        read = cow.dense_sparse_routes(s["read_weights"], s["read_indices"], s["slots"])
        return list(cow.sdm_recurrence(s["memory"], write, s["values"], s["input_gate"],
                                       s["input_gate"], s["forget_log_gate"], read,
                                       return_states=s["states"]))
    decode = s["decode"]
    decode.release(list(range(s["incoming"])))
    cohort = cow.pack_prefill_layers(s["m0s"], s["finals"], s["routes"], capacity_rows=None,
                                     decode_capacity=decode.capacity,
                                     growth_quantum_rows=s["quantum"])
    decode.admit(_decode_state(cohort, s["incoming"]))
    return _layer_outputs(decode.sdm_states)


# ------------------------------------------------------- work and tolerance


def _step_work(banks, width, writes, reads, index_bytes, float_bytes):
    routes = writes + reads
    moved = banks * ((2 * writes + reads) * width * 4 + 2 * width * float_bytes
                     + routes * (index_bytes + float_bytes + 4) + 3 * float_bytes)
    return moved, banks * width * (6 * writes + 2 * reads)


def _controller_work(case, tokens):
    """(weight bytes, token bytes in and out, flops) of the controller around the memory"""

    width = case["width"]
    rows = 4 * case["heads"] * math.isqrt(case["slots"]) + width + 2 * case["heads"]
    weights = 4 * (width * (rows + 2 * width) + rows + 6 * width)
    return weights, 2 * tokens * width * 4, 2 * tokens * width * (rows + 2 * width)


def work(case):
    kind = case["kind"]
    if kind == "step":
        moved, flops = _step_work(case["batch"] * case["heads"], case["width"], case["writes"],
                                  case["reads"], 4 if case["index"] == "int32" else 8,
                                  4 if case["floats"] == "float32" else 2)
        return dict(bytes=moved, flops=flops)
    if kind == "trace":
        moved, flops = _step_work(case["layers"] * case["batch"], case["width"], case["writes"],
                                  case["reads"], 4 if case["index"] == "int32" else 8, 4)
        return dict(bytes=moved * case["steps"], flops=flops * case["steps"])
    if kind in ("graph", "stack"):
        banks, width = case["batch"] * case["heads"], case["width"] // case["heads"]
        rows = banks * (2 * case["writes"] + case["reads"]) * width * 4
        weights, tokens, flops = _controller_work(case, case["batch"])
        return dict(bytes=case["layers"] * (rows + weights) + tokens,
                    flops=case["layers"] * (flops + banks * width
                                            * (6 * case["writes"] + 2 * case["reads"])))
    if kind == "prefill":
        n, heads, width = case["batch"] * case["time"], case["heads"], case["width"]
        weights, tokens, flops = _controller_work(case, n)
        routes = n * heads * (case["writes"] + case["reads"]) * 12
        memory = (case["batch"] + 1) * case["slots"] * width * 4
        return dict(bytes=weights + tokens + routes + n * width * 4 + 2 * n * heads * 4 + memory,
                    flops=flops + n * width * (6 * case["writes"] + 2 * case["reads"]))
    if kind == "recurrence":
        n, table = case["batch"] * case["time"], case["slots"] * case["width"] * 4
        moved = (n * ((case["writes"] + case["reads"]) * 12 + 2 * case["width"] * 4 + 8)
                 + 2 * case["batch"] * table)
        return dict(bytes=moved + (n * table if case["states"] else 0),
                    flops=n * case["width"] * (6 * case["writes"] + 2 * case["reads"]))
    # released map rows; written slots marked; live rows packed, then appended
    rows = case["incoming"] * case["slots"]
    written = 1 - (1 - case["writes"] / case["slots"]) ** case["time"]
    maps = (case["incoming"] + 2 * case["batch"]) * case["slots"] * 4
    return dict(bytes=int(case["layers"] * (maps + rows * written * 4 * case["width"] * 4
                                            + case["incoming"] * case["time"]
                                            * case["writes"] * 8)), flops=0)


def tolerance(case):
    """About four times the distance from ``exact`` that the path shows: 1e-7 for the sums
    of a step, up to 5e-7 behind the controller's norms and projections, and the rounding
    of a reading to 16 bits."""

    kind = case["kind"]
    if kind == "turnover":
        return "exact"
    if kind == "step" and case["floats"] != "float32":
        return dict(rel=7e-3 if case["floats"] == "bfloat16" else 1e-3)
    return dict(rel=2e-6 if kind in ("graph", "stack", "prefill") else 6e-7)


def exact(case, seed):
    g, kind = _generator(seed), case["kind"]
    if kind == "step":
        m0, finals, _, steps = _prepare_step(case, g)
        x = {k: v for k, v in vars(steps[0]).items() if v is not None}
        banks = torch.arange(case["batch"] * case["heads"], device=DEVICE)
        if finals is not None:
            reading = _update64(finals[0].double(), banks.unsqueeze(1), x)
        else:       # the tables are the shared memory: only the routed rows are widened
            slots = torch.cat((x["write_indices"], x["read_indices"]), dim=1).long()
            rows = m0[0][banks.unsqueeze(1) % case["heads"], slots].double()
            writes = case["writes"]
            same = slots[:, writes:, None] == slots[:, None, :writes]
            x["write_indices"] = torch.arange(writes, device=DEVICE).expand(len(banks), -1)
            own = torch.arange(writes, slots.shape[1], device=DEVICE).expand(len(banks), -1)
            x["read_indices"] = torch.where(same.any(dim=2), same.int().argmax(dim=2), own)
            reading = _update64(rows, banks.unsqueeze(1), x)
        return [reading, [[None, None, None]]]
    if kind == "trace":
        _, finals, _, inputs = _prepare_trace(case, g)
        layers, batch = case["layers"], case["batch"]
        table = torch.stack([f.double() for f in finals]).flatten(0, 1)
        banks = torch.arange(layers * batch, device=DEVICE).unsqueeze(1)
        readings = [_update64(table, banks, {k: v[t].flatten(0, 1) for k, v in inputs.items()})
                    for t in range(case["steps"])]
        return [torch.stack(readings).view(case["steps"], layers, batch, -1),
                [[None, None, None] for _ in range(layers)]]
    if kind in ("graph", "stack"):
        parameters, _, finals, _, tokens = _prepare_tokens(case, g)
        out, _ = _tokens64(case, parameters, finals, tokens, 1)
        return [out, [[None, None, None] for _ in range(case["layers"])]]
    if kind == "prefill":
        p, m0, tokens = _prepare_prefill(case, g)
        batch, time, heads = case["batch"], case["time"], case["heads"]
        step, _ = _prepare64(p, case, tokens.flatten(0, 1))
        table = m0.double().repeat(batch, 1, 1)
        banks = torch.arange(batch * heads, device=DEVICE).unsqueeze(1)
        routed = {k: v.reshape(batch, time, heads, *v.shape[1:]) for k, v in step.items()
                  if k != "normalized"}
        readings = [_update64(table, banks, {k: v[:, t].flatten(0, 1)
                                             for k, v in routed.items()}) for t in range(time)]
        readings = torch.stack(readings).view(time, batch, heads, -1).transpose(0, 1)
        out = _finish64(p, step["normalized"], readings.reshape(batch * time * heads, -1))
        return [out.view(batch, time, -1),
                table.view(batch, heads, *table.shape[1:]), routed["values"],
                routed["input_gate"], routed["forget_log_gate"], routed["read_weights"],
                routed["write_weights"], None, None]
    if kind == "recurrence":
        x = _prepare_recurrence(case, g)
        table = x.pop("memory").double()
        banks = torch.arange(case["batch"], device=DEVICE).unsqueeze(1)
        readings, states = [], []
        for t in range(case["time"]):
            readings.append(_update64(table, banks, {k: v[:, t] for k, v in x.items()}))
            if case["states"]:
                states.append(table.clone())
        out = [torch.stack(readings, dim=1), table]
        return out + [torch.stack(states, dim=1)] if case["states"] else out
    return None
