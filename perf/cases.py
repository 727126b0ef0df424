"""Timed cases of the EXL3 mixture-of-experts path, through its public Python entry points.

Four kinds of work, as a serving engine has them done:

* ``moe``    one MoE layer call (routing, grouping, expert GEMMs, combine), decode and prefill;
* ``linear`` one or several EXL3 linears over the same rows (attention projections, output head);
* ``router`` the router's dense product, top-k routing and token grouping of a chunk;
* ``load``   a checkpoint-order weight brought into the library's layout.

Weights are uniform random trellis codes, suh random signs, svh random signs times U(0.5, 1.5)
divided by the square root of the input width (so a layer's outputs are of the size of its
inputs, as trained ones are); activations N(0, 1); router logits N(0, 1), with a Zipf-like
per-expert bias where the case says so.  Everything comes from the seed.
"""
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "crucible-strix-halo_amd"))
import exl3moe  # noqa: E402
from exl3moe import ops  # noqa: E402

DEV = "cuda"
MODES = {"auto": exl3moe.CX_MOE_AUTO, "decode": exl3moe.CX_MOE_DECODE, "prefill": exl3moe.CX_MOE_PREFILL}


def _moe(name, rows, E=512, H=2048, I=512, topk=10, bits=4.0, bits_down=4.0, codebook="mul1", x="f16", sessions=0,
         streams=0, zipf=0.0):
    return dict(name=name, kind="moe", rows=rows, E=E, H=H, I=I, topk=topk, bits=bits, bits_down=bits_down,
                codebook=codebook, x=x, sessions=sessions, streams=streams, zipf=zipf)


def _linear(name, rows, I, outs, bits=4.0, codebook="mul1", x="f16", y="f32", sessions=0):
    return dict(name=name, kind="linear", rows=rows, I=I, outs=outs, bits=bits, codebook=codebook, x=x, y=y,
                sessions=sessions)


def listed():
    return [
        # One user, one token at a time: the latency of a layer.
        _moe("moe_decode_1", 1),
        # Eight sessions with 1 to 5 draft rows each: batched decode, the serving case.
        _moe("moe_decode_23", 23, sessions=8),
        # A busier decode batch of a mixed-rate layer with the engine's fp32 activations, written
        # back into the four residual streams.
        _moe("moe_decode_61_residual", 61, bits=3.0, bits_down=5.0, x="f32", sessions=16, streams=4),
        # A short prompt, or the tail chunk of a longer one.
        _moe("moe_prefill_199", 199),
        # A 2048-token prompt chunk whose tokens favour some experts.
        _moe("moe_prefill_2048_skewed", 2048, zipf=1.1),
        # A long prompt chunk of a layer with mixed rates.
        _moe("moe_prefill_8192", 8192, bits=3.0, bits_down=5.0),
        # An attention projection in batched decode, and the same projection for a prompt chunk.
        _linear("linear_decode_24", 24, 2048, "4096", sessions=8),
        _linear("linear_prefill_2047", 2047, 2048, "4096", x="f32", y="f16"),
        # The query, key and value projections of a decode batch in one group.
        _linear("group_qkv_decode_24", 24, 2048, "4096,512,512", x="f32", sessions=8),
        # The output head for the last token of each of four sessions.
        _linear("head_4", 4, 2048, "151936", bits=6.0),
        # Router product, routing and grouping of a prompt chunk.
        dict(name="router_2048", kind="router", rows=2048, E=512, H=2048, topk=10, x="f32"),
        # Loading: a large projection's tiles into the library's layout.
        dict(name="load_2048x32768", kind="load", I=2048, O=32768, bits=4.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["moe_decode", "moe_prefill", "moe_prefill", "linear_decode", "linear_prefill", "router", "load"])
    codebook = rng.choice(["mul1", "mul1", "mul1", "mcg", "3inst"])
    bits = rng.choice([2.0, 2.5, 3.0, 3.5, 4.0, 4.0, 5.0, 6.0, 8.0])
    if bits != int(bits):
        codebook = "mul1"  # half rates exist in this codebook only
    if kind.startswith("moe"):
        H = 128 * rng.randint(6, 16)
        I = 128 * rng.randint(2, 5)
        E = rng.randint(32, 512)
        rows = _log_int(rng, 1, 64) if kind == "moe_decode" else _log_int(rng, 65, 6000)
        c = _moe("", rows, E=E, H=H, I=I, topk=rng.randint(2, 10), bits=bits, bits_down=min(8.0, math.ceil(bits + rng.choice([0, 0, 1, 2]))),
                 codebook=codebook, x=rng.choice(["f16", "f32"]), sessions=min(rows, rng.choice([0, 4, 8])) if kind == "moe_decode" else 0,
                 streams=rng.choice([0, 0, 4]), zipf=rng.choice([0.0, 1.1]))
    elif kind.startswith("linear"):
        rows = _log_int(rng, 1, 64) if kind == "linear_decode" else _log_int(rng, 65, 4096)
        outs = rng.choice([[rng.randint(4, 40)], [rng.randint(4, 32), 4, 4], [8 * rng.randint(8, 100)]])
        if kind == "linear_prefill":
            outs = [min(o, 48) for o in outs]
        c = _linear("", rows, 128 * rng.randint(4, 32), ",".join(str(128 * o) for o in outs), bits=bits, codebook=codebook,
                    x=rng.choice(["f16", "f32"]), y=rng.choice(["f16", "f32"]))
    elif kind == "router":
        c = dict(kind="router", rows=_log_int(rng, 1, 8192), E=rng.randint(32, 512), H=128 * rng.randint(6, 24),
                 topk=rng.randint(2, 10), x=rng.choice(["f16", "f32"]))
    else:
        c = dict(kind="load", I=128 * rng.randint(4, 32), O=128 * _log_int(rng, 4, 500), bits=bits)
    c.pop("name", None)
    return c


# ---- inputs ----------------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 12345)
    return g


def _sign(shape, g):
    return (torch.randint(0, 2, shape, device=DEV, generator=g) * 2 - 1).to(torch.float16)


def _weights(g, n, I, O, bits):
    """n matrices' trellis [n, I/16, O/16, 16 bits] int16, suh [n, I] and svh [n, O] fp16."""
    tr = torch.randint(-32768, 32768, (n, I // 16, O // 16, int(round(16 * bits))), dtype=torch.int16, device=DEV, generator=g)
    suh = _sign((n, I), g)
    svh = ((torch.rand((n, O), device=DEV, generator=g) + 0.5) * _sign((n, O), g).float() / math.sqrt(I)).to(torch.float16)
    return tr, suh, svh


def _offsets(rows, sessions):
    if not sessions:
        return None
    return [rows * s // sessions for s in range(sessions)] + [rows]


def _tensors(c, seed):
    """The case's inputs and weights in checkpoint form, from the seed alone."""
    g = _gen(seed)
    t = {}
    xt = torch.float32 if c.get("x") == "f32" else torch.float16
    if c["kind"] == "moe":
        E, H, I, M = c["E"], c["H"], c["I"], c["rows"]
        t["gate"] = _weights(g, E + 1, H, I, c["bits"])  # the last one: the shared expert
        t["up"] = _weights(g, E + 1, H, I, c["bits"])
        t["down"] = _weights(g, E + 1, I, H, c["bits_down"])
        t["x"] = torch.randn((M, H), device=DEV, generator=g).to(xt)
        logits = torch.randn((M, E + 1), device=DEV, generator=g)
        if c["zipf"]:
            w = (torch.randperm(E, device=DEV, generator=g) + 1).double() ** -c["zipf"]
            logits[:, :E] += (0.23 * torch.log(w / w.mean())).float()
        t["logits"] = logits
        if c["streams"]:
            t["post"] = torch.rand((M, c["streams"]), device=DEV, generator=g) + 0.5
            t["H"] = torch.randn((M, c["streams"], H), device=DEV, generator=g)
    elif c["kind"] == "linear":
        t["x"] = torch.randn((c["rows"], c["I"]), device=DEV, generator=g).to(xt)
        t["w"] = [_weights(g, 1, c["I"], int(o), c["bits"]) for o in c["outs"].split(",")]
    elif c["kind"] == "router":
        t["x"] = torch.randn((c["rows"], c["H"]), device=DEV, generator=g).to(xt)
        t["W"] = (torch.randn((c["E"] + 1, c["H"]), device=DEV, generator=g) / math.sqrt(c["H"])).to(torch.float16)
    else:
        t["w"] = _weights(g, 1, c["I"], c["O"], c["bits"])
    return t


def prepare(case, seed):
    c, t = case, _tensors(case, seed)
    s = {"case": c}
    if c["kind"] == "moe":
        def lins(key, bits):
            tr, suh, svh = t[key]
            return [ops.DeviceLinear.from_trellis(tr[e], suh[e], svh[e], bits, c["codebook"]) for e in range(c["E"] + 1)]
        gate, up, down = lins("gate", c["bits"]), lins("up", c["bits"]), lins("down", c["bits_down"])
        ex = [{"gate": a, "up": b, "down": d} for a, b, d in zip(gate, up, down)]
        s["plan"] = ops.MoePlan(c["H"], c["I"], ex[:-1], ex[-1], c["topk"])
        s["offsets"] = _offsets(c["rows"], c["sessions"])
        s["ws"] = torch.empty(s["plan"].workspace_size(c["rows"]), dtype=torch.uint8, device=DEV)
        s["sel"] = torch.empty((c["rows"], c["topk"]), dtype=torch.int32, device=DEV)
        s["wts"] = torch.empty((c["rows"], c["topk"] + 1), dtype=torch.float32, device=DEV)
        s["y"] = None if c["streams"] else torch.empty((c["rows"], c["H"]), dtype=torch.float32, device=DEV)
        s.update({k: t[k] for k in ("x", "logits", "post", "H") if k in t})
    elif c["kind"] == "linear":
        yt = torch.float32 if c["y"] == "f32" else torch.float16
        s["lins"] = [ops.DeviceLinear.from_trellis(tr[0], suh[0], svh[0], c["bits"], c["codebook"]) for tr, suh, svh in t["w"]]
        s["x"] = t["x"]
        s["ys"] = [torch.empty((c["rows"], lin.out_features), dtype=yt, device=DEV) for lin in s["lins"]]
        s["offsets"] = _offsets(c["rows"], c["sessions"])
        n = s["lins"][0].workspace_size(c["rows"]) if len(s["lins"]) == 1 else ops.group_workspace_size(s["lins"], c["rows"])
        s["ws"] = torch.empty(n, dtype=torch.uint8, device=DEV)
    elif c["kind"] == "router":
        s["x"], s["W"] = t["x"], t["W"]
        n = int(exl3moe.lib().cx_moe_group_workspace_size(c["rows"], c["E"], c["topk"]))
        s["ws"] = torch.empty(max(n, 1), dtype=torch.uint8, device=DEV)
    else:
        tr, suh, svh = t["w"]
        s["w"] = (tr[0], suh[0], svh[0])
    return s


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "moe":
        if c["streams"]:
            out = s["plan"].forward_hc(s["x"], s["logits"], s["post"], s["H"], row_offsets=s["offsets"], workspace=s["ws"],
                                       sel=s["sel"], wts=s["wts"])
        else:
            out = s["plan"](s["x"], s["logits"], row_offsets=s["offsets"], workspace=s["ws"], y=s["y"], sel=s["sel"],
                            wts=s["wts"])
        return {"out": out, "sel": s["sel"], "wts": s["wts"]}
    if c["kind"] == "linear":
        if len(s["lins"]) == 1:
            return [s["lins"][0].forward_into(s["x"], s["ys"][0], s["offsets"], s["ws"])]
        ops.linear_group([(lin, s["x"], y) for lin, y in zip(s["lins"], s["ys"])], s["offsets"], s["ws"])
        return s["ys"]
    if c["kind"] == "router":
        logits = ops.dense_linear(s["W"], s["x"])
        sel, wts = ops.route(logits, c["E"], c["topk"])
        counts, offsets, pairs, rows = ops.group(sel, c["E"], s["ws"])
        return {"logits": logits, "wts": wts, "counts": counts, "offsets": offsets, "sel": sel}
    tr, suh, svh = s["w"]
    return ops.DeviceLinear.from_trellis(tr, suh, svh, c["bits"]).tiles


# ---- what a pass cannot do without -------------------------------------------------------------


def _matrix_bytes(I, O, bits):
    return I * O * bits / 8 + 2 * I + 2 * O


def work(case):
    c = case
    xb = 4 if c.get("x") == "f32" else 2
    if c["kind"] == "moe":
        M, E, H, I, k = c["rows"], c["E"], c["H"], c["I"], c["topk"]
        distinct = E * (1 - (1 - k / E) ** M) + 1  # evenly routed tokens, and the shared expert
        ex = 2 * _matrix_bytes(H, I, c["bits"]) + _matrix_bytes(I, H, c["bits_down"])
        out = M * H * 4 if not c["streams"] else 2 * M * H * 4 * c["streams"] + M * c["streams"] * 4
        return {"bytes": distinct * ex + M * H * xb + M * (E + 1) * 4 + out + M * (2 * k + 1) * 4,
                "flops": 2.0 * (k + 1) * M * 3 * H * I}
    if c["kind"] == "linear":
        yb = 4 if c["y"] == "f32" else 2
        outs = [int(o) for o in c["outs"].split(",")]
        return {"bytes": sum(_matrix_bytes(c["I"], o, c["bits"]) + c["rows"] * o * yb for o in outs) + c["rows"] * c["I"] * xb,
                "flops": 2.0 * c["rows"] * c["I"] * sum(outs)}
    if c["kind"] == "router":
        M, E, k = c["rows"], c["E"], c["topk"]
        return {"bytes": (E + 1) * c["H"] * 2 + M * c["H"] * xb + M * (E + 1) * 4 + M * (4 * k + 1) * 4 + 8 * E,
                "flops": 2.0 * M * (E + 1) * c["H"]}
    return {"bytes": 2 * c["I"] * c["O"] * c["bits"] / 8, "flops": 0.0}


def tolerance(case):
    if case["kind"] == "load":
        return "exact"
    if case["kind"] == "router":
        # fp32 sums in another order: the logits move by about 1e-6 of their size, a weight (a
        # softmax of them) by as much.  The fp16 form of more than 8 rows is within 5e-4 of the
        # exact product; near-equal logits may change places.
        return {"rel": 2e-4, "max": 2e-2, "differ": 4e-3}
    if case["kind"] == "linear":
        # Against 64 bits 2.1e-4 to 2.9e-4 (the fp16 roundings of x and of the transformed inputs),
        # 4.6e-4 with an fp16 y.
        return {"rel": 1e-3, "max": 8e-3}
    # A layer has one more fp16 rounding (the down projection's input), a prefill one more again
    # (the down projection's output): 4e-4 to 5.5e-4 against 64 bits.
    return {"rel": 2e-3, "max": 1.2e-2}


# ---- the same in 64 bits -----------------------------------------------------------------------


def _codebook(codebook):
    """The 65,536 fp16 weight values of a codebook, as float64."""
    s = torch.arange(65536, device=DEV, dtype=torch.int64)

    def half(bits):
        return torch.where(bits >= 32768, bits - 65536, bits).to(torch.int16).view(torch.float16).double()

    if codebook == "mul1":
        p = (s * 0x83DCD12D) & 0xFFFFFFFF
        h = 1024 + (p & 255) + (p >> 8 & 255) + (p >> 16 & 255) + (p >> 24)
        k = half(torch.tensor([0x1EEE, 0xC931], device=DEV))
        v = h.double() * k[0] + k[1]  # exact: the product has 22 bits
    else:
        p = (s * (0xCBAC1FED if codebook == "mcg" else 89226354) + (0 if codebook == "mcg" else 64248484)) & 0xFFFFFFFF
        p = (p & 0x8FFF8FFF) ^ 0x3B603B60
        v = half(p & 0xFFFF) + half(p >> 16)  # exact
    return v.float().half().double()  # v is exact in float32: one rounding, to fp16


def _dense(tr, bits, table):
    """The weight matrix [I, O] (float64) of one trellis [I/16, O/16, 16 bits]."""
    A, B, n = tr.shape
    k2, T = int(round(2 * bits)), n // 2
    w = tr.to(torch.int64) & 0xFFFF
    d = w[..., 0::2] | (w[..., 1::2] << 16)
    i = torch.arange(256, device=DEV)
    width = (k2 >> 1) + (i & 1) * (k2 & 1)
    start = torch.cumsum(width, 0) - 16
    a, off = torch.div(start, 32, rounding_mode="floor"), torch.remainder(start, 32)
    lo, hi = d[..., torch.remainder(a, T)], d[..., torch.remainder(a + 1, T)]
    v = table[((lo << 32 | hi) >> (48 - off)) & 0xFFFF]  # the sign bit is shifted out or masked
    t, j = i // 8, i % 8
    row, col = 2 * (t % 4) + (j & 1) + 8 * (j >> 1 & 1), t // 4 + 8 * (j >> 2)
    tile = torch.empty((A, B, 256), dtype=torch.float64, device=DEV)
    tile[..., row * 16 + col] = v
    return tile.view(A, B, 16, 16).permute(0, 2, 1, 3).reshape(16 * A, 16 * B)


def _had(v):
    h = torch.ones((1, 1), dtype=torch.float64, device=DEV)
    for _ in range(7):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (v.reshape(-1, 128) @ h / math.sqrt(128)).reshape(v.shape)


def _apply(x, w, n, bits, table):
    """x through matrix n of the weights w, in 64 bits."""
    tr, suh, svh = w
    cols = 8192
    xh = _had(x * suh[n].double())
    y = torch.cat([xh @ _dense(tr[n][:, b:b + cols // 16], bits, table) for b in range(0, tr.shape[2], cols // 16)], 1)
    return _had(y) * svh[n].double()


def _topk(logits, E, k):
    l = logits[:, :E].double()
    v, sel = torch.sort(l, dim=1, descending=True, stable=True)
    return sel[:, :k], torch.cat([torch.softmax(v[:, :k], 1), torch.sigmoid(logits[:, E:E + 1].double())], 1)


def exact(case, seed):
    c, t = case, _tensors(case, seed)
    if c["kind"] == "load":
        return None
    if c["kind"] == "router":
        logits = t["x"].double() @ t["W"].double().t()
        # The weights follow the logits that the path itself computed: near-equal ones may change places.
        return {"logits": logits, "wts": None, "counts": None, "offsets": None, "sel": None}
    table = _codebook(c["codebook"])
    x = t["x"].double()
    if c["kind"] == "linear":
        return [_apply(x, w, 0, c["bits"], table) for w in t["w"]]
    E, k = c["E"], c["topk"]
    sel, wts = _topk(t["logits"], E, k)
    y = torch.zeros((c["rows"], c["H"]), dtype=torch.float64, device=DEV)
    for e in range(E + 1):
        if e < E:
            r, slot = torch.nonzero(sel == e, as_tuple=True)
            wt = wts[r, slot]
        else:
            r, wt = torch.arange(c["rows"], device=DEV), wts[:, k]
        if r.numel():
            g = _apply(x[r], t["gate"], e, c["bits"], table)
            u = _apply(x[r], t["up"], e, c["bits"], table)
            d = _apply(g * torch.sigmoid(g) * u, t["down"], e, c["bits_down"], table)
            y.index_add_(0, r, d * wt[:, None])
    out = t["H"].double() + t["post"].double()[:, :, None] * y[:, None, :] if c["streams"] else y
    return {"out": out, "sel": None, "wts": wts}
