"""Workloads of this package as a user's program calls them, for timing and comparison.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges, ``prepare(case,
seed)`` makes what a program holds before the call, ``run(state)`` is one pass through the
public entry points, ``work(case)`` the bytes and operations a pass cannot do without, and
``exact(case, seed)`` the same outputs in 64 bits from plain torch.

Kinds of case, and the ranges they stand for:

round    ``virtual_round`` of 2^10 .. 2^27 values: a small layer's activation up to the
         largest weight or gradient tensor, to nearest or stochastically, formats of 4 to 16
         bits and mantissa-only targets; odd lengths.
mx       ``virtual_mx_round`` of 2^12 .. 2^26 values in blocks of 16 to 64 along the rows.
pack     ``pack.encode`` then ``pack.decode`` of 2^12 .. 2^26 values, 4 to 11 bits each.
gemm     ``gemm`` / ``lof_gemm`` with 1 .. 4096 rows, columns and k, on pre-rounded or FP32
         operands, mantissa-only and binary16-shaped accumulators, chunks of 1, 8 and 32.
linear   ``LoF_Linear``: inference from one row up and training steps (forward, backward),
         per-tensor formats, FP32 formats (what ``lofloatify`` installs) and MX blocks.
conv     ``LoF_Conv2d`` inference: 1x1 to 7x7 filters, stride 1 and 2, 1 to 32 images.
grouped  a ``GroupedPlan`` of many small rounding, MX and GEMM jobs, run as one launch.
"""
import math

import torch

import lofloat_amd as lof

DEV = "cuda"

# name -> (total bits, mantissa bits, bias); signed, saturating
FORMATS = {"e2m1": (4, 1, 1), "e4m3": (8, 3, 7), "e5m2": (8, 2, 15), "8e7m": (16, 7, 127),
           "5e10m": (16, 10, 15), "fp32": (32, 23, 127)}
# codec formats: name -> (mantissa bits, bias, bits), and the factory that makes the format
PACKED = {"e2m1": (1, 1, 4), "e4m3fn": (3, 7, 8), "p3109_11p5": (4, 32, 11)}
SR_LEN = 8


def listed():
    return [
        # one small activation tensor, odd length: the cost is the call and the launch
        {"name": "round_small_e4m3", "kind": "round", "n": 5003, "to": "e4m3", "mode": "rne"},
        # a training step's gradient tensor, stochastic with the built-in generator
        {"name": "round_sr_e5m2", "kind": "round", "n": 33554435, "to": "e5m2", "mode": "sr"},
        # the headline MX block rounding of a weight matrix
        {"name": "mx_8192_e4m3", "kind": "mx", "rows": 8192, "cols": 8192, "block": 32,
         "to": "e4m3", "mode": "rne"},
        # a checkpoint tensor packed to 11 bits and read back, ragged length
        {"name": "pack_11p5", "kind": "pack", "n": 67108871, "to": "p3109_11p5"},
        # lof_gemm as the reference's own harness runs it: FP32 uniform operands, 10-bit
        # accumulator rounded after every multiply-add
        {"name": "gemm_4096_fp32u_m10", "kind": "gemm", "m": 4096, "n": 4096, "k": 4096,
         "inputs": "fp32u", "accum": "mant10", "chunk": 1},
        # bfloat16-like operands in a ragged product, binary16 accumulator every 8 products
        {"name": "gemm_ragged_8e7m_c8", "kind": "gemm", "m": 1537, "n": 3001, "k": 2047,
         "inputs": "8e7m", "accum": "5e10m", "chunk": 8},
        # token-by-token inference of one projection, 8 sequences, default accumulator
        {"name": "linear_decode_8", "kind": "linear", "rows": 8, "in": 4096, "out": 4096,
         "formats": "e4m3", "accum": "mant23", "chunk": 1, "step": False},
        # a training step of a layer as lofloatify leaves it: FP32 formats, 23-bit accumulator
        {"name": "linear_step_fp32_m23", "kind": "linear", "rows": 2048, "in": 1024,
         "out": 4096, "formats": "fp32", "accum": "mant23", "chunk": 1, "step": True},
        # the headline training step: MX e4m3 operands, binary16 accumulator every 32 products
        {"name": "linear_step_mx_c32", "kind": "linear", "rows": 8192, "in": 4096, "out": 4096,
         "formats": "mx_e4m3", "accum": "5e10m", "chunk": 32, "step": True},
        # a training step of a mid-sized layer, 10-bit accumulator after every multiply-add
        {"name": "linear_step_e4m3_m10", "kind": "linear", "rows": 1000, "in": 768, "out": 3072,
         "formats": "e4m3", "accum": "mant10", "chunk": 1, "step": True},
        # inference of a 3x3 convolution layer, 10-bit accumulator
        {"name": "conv_3x3_128", "kind": "conv", "batch": 32, "cin": 128, "cout": 128,
         "size": 28, "kernel": 3, "stride": 1, "formats": "e4m3", "accum": "mant10",
         "chunk": 1},
        # many small tensors and products in one launch
        {"name": "grouped_small", "kind": "grouped", "rounds": 36, "mx": 12, "gemms": 12,
         "lg": 16, "side": 256},
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["round", "mx", "pack", "gemm", "gemm", "linear", "linear", "conv",
                       "grouped"])
    accum, chunk = rng.choice(["mant10", "mant23", "mant23", "5e10m"]), rng.choice([1, 1, 8, 32])
    if kind == "round":
        return {"kind": kind, "n": _log(rng, 1 << 10, 1 << 27),
                "to": rng.choice(["e2m1", "e4m3", "e5m2", "5e10m", "mant7", "mant10"]),
                "mode": rng.choice(["rne", "rne", "rtz", "sr"])}
    if kind == "mx":
        block = rng.choice([16, 32, 64])
        cols = block * _log(rng, 1, 8192 // block)
        return {"kind": kind, "rows": _log(rng, max(1, 4096 // cols), (1 << 26) // cols),
                "cols": cols, "block": block, "to": rng.choice(["e2m1", "e4m3"]),
                "mode": rng.choice(["rne", "rne", "sr"])}
    if kind == "pack":
        return {"kind": kind, "n": _log(rng, 1 << 12, 1 << 26), "to": rng.choice(sorted(PACKED))}
    if kind == "gemm":
        m, n, k = (_log(rng, 1, 4096), _log(rng, 16, 4096), _log(rng, 16, 4096))
        while m * n * k > 1 << 33:
            m = max(1, m // 2)
        return {"kind": kind, "m": m, "n": n, "k": k,
                "inputs": rng.choice(["e4m3", "8e7m", "fp32u"]), "accum": accum, "chunk": chunk}
    if kind == "linear":
        rows, cin, cout = _log(rng, 1, 4096), 32 * _log(rng, 2, 128), _log(rng, 32, 4096)
        while rows * cin * cout > 1 << 32:
            rows = max(1, rows // 2)
        return {"kind": kind, "rows": rows, "in": cin, "out": cout,
                "formats": rng.choice(["e4m3", "e4m3", "fp32", "mx_e4m3"]), "accum": accum,
                "chunk": chunk, "step": rng.random() < 0.5}
    if kind == "conv":
        kernel, stride, size = rng.choice([1, 3, 3, 5, 7]), rng.choice([1, 1, 2]), _log(rng, 7, 112)
        batch, cin, cout = _log(rng, 1, 32), _log(rng, 3, 256), _log(rng, 16, 512)
        while batch * cin * cout * (size * kernel // stride) ** 2 > 1 << 32:
            batch, cin = max(1, batch // 2), max(3, cin // 2)
            size = max(7, size * 3 // 4)
        return {"kind": kind, "batch": batch, "cin": cin, "cout": cout, "size": size,
                "kernel": kernel, "stride": stride, "formats": rng.choice(["e4m3", "fp32"]),
                "accum": accum, "chunk": chunk}
    return {"kind": kind, "rounds": rng.randint(4, 40), "mx": rng.randint(2, 12),
            "gemms": rng.randint(1, 12), "lg": rng.randint(12, 18),
            "side": 64 * rng.randint(1, 6)}


# ------------------------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 2654435761 % (1 << 31) + 7)


def _spread(n, g):
    """N(0, 1) values spread over 24 binades, 1 % of them zeros."""
    x = torch.randn(n, device=DEV, generator=g)
    x *= torch.exp2(torch.rand(n, device=DEV, generator=g) * 24 - 12)
    return torch.where(torch.rand(n, device=DEV, generator=g) < 0.01, torch.zeros((), device=DEV), x)


def _rows(rows, cols, g):
    """A matrix whose rows have their own magnitude, as weight channels do."""
    return (torch.randn(rows, cols, device=DEV, generator=g) *
            torch.exp2(torch.rand(rows, 1, device=DEV, generator=g) * 16 - 8))


def _operand(rows, cols, inputs, g):
    """An FP32 GEMM operand before its rounding: uniform, or small normal values."""
    if inputs == "fp32u":
        return torch.rand(rows, cols, device=DEV, generator=g) * 2 - 1
    return torch.randn(rows, cols, device=DEV, generator=g) / 64


def _inputs(case, seed):
    """The raw FP32 tensors of a case, from its seed alone."""
    g, c = _gen(seed), case
    randn = lambda *s: torch.randn(*s, device=DEV, generator=g)   # noqa: E731
    if c["kind"] == "round":
        return {"x": _spread(c["n"], g)}
    if c["kind"] == "mx":
        return {"x": _rows(c["rows"], c["cols"], g)}
    if c["kind"] == "pack":
        return {"x": randn(c["n"])}
    if c["kind"] == "gemm":
        return {"a": _operand(c["m"], c["k"], c["inputs"], g),
                "b": _operand(c["k"], c["n"], c["inputs"], g)}
    if c["kind"] == "linear":
        d = {"x": randn(c["rows"], c["in"]), "w": randn(c["out"], c["in"]) / math.sqrt(c["in"]),
             "b": randn(c["out"]) * 0.1}
        if c["step"]:
            d["g"] = randn(c["rows"], c["out"])
        return d
    if c["kind"] == "conv":
        s, k = c["size"], c["kernel"]
        return {"x": randn(c["batch"], c["cin"], s, s),
                "w": randn(c["cout"], c["cin"], k, k) / math.sqrt(c["cin"] * k * k),
                "b": randn(c["cout"]) * 0.1}
    d, sizes = {}, _grouped_sizes(c)
    for i, n in enumerate(sizes["rounds"]):
        d["r%d" % i] = randn(n)
    for i, n in enumerate(sizes["mx"]):
        d["m%d" % i] = randn(n)
    for i, (m, n, k) in enumerate(sizes["gemms"]):
        d["a%d" % i], d["b%d" % i] = randn(m, k) / 64, randn(k, n) / 64
    return d


def _grouped_sizes(c):
    """Uneven job sizes of a grouped case: rounding jobs of up to 2^lg values, MX jobs of
    whole blocks of 32, products of up to ``side`` a side."""
    lo = c["lg"] - 6
    rounds = [int(2 ** (lo + 6.0 * ((7 * i) % 13) / 13)) + 13 * i for i in range(c["rounds"])]
    mx = [32 * (1 + (int(2 ** (lo + 6.0 * ((5 * i) % 11) / 11)) >> 5)) for i in range(c["mx"])]
    side = lambda i: max(64, c["side"] * (1 + i % 4) // 4)   # noqa: E731
    return {"rounds": rounds, "mx": mx,
            "gemms": [(side(i), side(i + 1), side(3 * i + 2)) for i in range(c["gemms"])]}


# A grouped case's rounding jobs go through these formats and modes in turn.
_JOB_FORMATS = ("e4m3", "e5m2", "5e10m", "e2m1")
_JOB_MODES = ("rne", "rtz", "sr")


# --------------------------------------------------------------------------- the package side
def _format(name):
    return lof.create_single_params() if name == "fp32" else lof.make_format(*FORMATS[name])


def _mode(name):
    return {"rne": lof.RoundingMode.RoundToNearestEven, "rtz": lof.RoundingMode.RoundTowardsZero,
            "sr": lof.RoundingMode.StochasticRoundingA}[name]


def _target(to):
    return int(to[4:]) if to.startswith("mant") else _format(to)


def _accum(case):
    if case["accum"] == "5e10m":
        return lof.AccumSpec(fmt=_format("5e10m"), chunk=case["chunk"])
    return lof.AccumSpec(mant_bits=int(case["accum"][4:]), chunk=case["chunk"])


def _layer_args(case):
    """Formats and accumulator of a LoF layer."""
    name = case["formats"].replace("mx_", "")
    args = dict(act_params=_format(name), weight_params=_format(name),
                accum_chunk=case["chunk"])
    if case["formats"] == "fp32":
        args["bias_params"] = _format("fp32")
    if case["formats"].startswith("mx_"):
        args.update(scaling="mx", mx_block_size=32)
    if case["accum"] == "5e10m":
        args["accum_format"] = _format("5e10m")
    else:
        args["accum_mant_bits"] = int(case["accum"][4:])
    return args


def _own(layer, d):
    with torch.no_grad():
        layer.weight.copy_(d["w"])
        layer.bias.copy_(d["b"])
    return layer


def prepare(case, seed):
    d, kind = _inputs(case, seed), case["kind"]
    state = {"kind": kind, "case": case}
    if kind in ("round", "mx"):
        state.update(x=d["x"], to=_target(case["to"]), mode=_mode(case["mode"]),
                     len=SR_LEN if case["mode"] == "sr" else 0, seed=int(seed) + 17,
                     scale=lof.create_e8m0_params())
    elif kind == "pack":
        make = {"e2m1": lof.create_ocp_e2m1_params, "e4m3fn": lof.create_ocp_e4m3fn_params,
                "p3109_11p5": lambda: lof.create_p3109_params(11, 5)}
        state.update(x=d["x"], to=make[case["to"]]())
    elif kind == "gemm":
        if case["inputs"] != "fp32u":
            d = {k: lof.virtual_round(v, _format(case["inputs"])) for k, v in d.items()}
        state.update(d, accum=_accum(case))
    elif kind == "linear":
        layer = lof.LoF_Linear(case["in"], case["out"],
                               grad_spec=lof.LinearGradSpec(seed=int(seed) + 29),
                               **_layer_args(case)).to(DEV)
        state.update(layer=_own(layer, d), x=d["x"].requires_grad_(case["step"]), g=d.get("g"))
    elif kind == "conv":
        layer = lof.LoF_Conv2d(case["cin"], case["cout"], case["kernel"], stride=case["stride"],
                               padding=case["kernel"] // 2, **_layer_args(case)).to(DEV)
        state.update(layer=_own(layer, d), x=d["x"])
    else:
        jobs, sizes = [], _grouped_sizes(case)
        for i in range(len(sizes["rounds"])):
            mode = _JOB_MODES[i % 3]
            jobs.append(lof.RoundJob(d["r%d" % i], _format(_JOB_FORMATS[i % 4]), _mode(mode),
                                     SR_LEN if mode == "sr" else 0, seed=int(seed) + i))
        for i in range(len(sizes["mx"])):
            jobs.append(lof.MXJob(d["m%d" % i], 32, _format("e4m3"), lof.create_e8m0_params()))
        for i in range(len(sizes["gemms"])):
            ab = [lof.virtual_round(d[k + str(i)], _format("e4m3")) for k in "ab"]
            jobs.append(lof.GemmJob(*ab, lof.AccumSpec(fmt=_format("5e10m"), chunk=32)))
        state.update(plan=lof.GroupedPlan(jobs))
    return state


def run(state):
    s, kind = state, state["kind"]
    if kind == "round":
        return lof.virtual_round(s["x"], s["to"], s["mode"], s["len"], seed=s["seed"])
    if kind == "mx":
        return lof.virtual_mx_round(s["x"], s["case"]["block"], s["to"], s["scale"], s["mode"],
                                    stoch_len=s["len"], seed=s["seed"])
    if kind == "pack":
        buf = lof.pack.encode(s["x"], s["to"])
        return {"packed": buf, "values": lof.pack.decode(buf, s["to"], s["x"].numel())}
    if kind == "gemm":
        if s["case"]["chunk"] == 1 and s["case"]["accum"].startswith("mant"):
            return lof.lof_gemm(s["a"], s["b"], s["accum"].mant_bits)
        return lof.gemm(s["a"], s["b"], s["accum"])
    if kind == "linear":
        layer, x = s["layer"], s["x"]
        if not s["case"]["step"]:
            with torch.no_grad():
                return layer(x)
        x.grad = layer.weight.grad = layer.bias.grad = None
        out = layer(x)
        out.backward(s["g"])
        return {"out": out, "dx": x.grad, "dw": layer.weight.grad, "db": layer.bias.grad}
    if kind == "conv":
        with torch.no_grad():
            return s["layer"](s["x"])
    s["plan"].run()
    return s["plan"].outputs


# --------------------------------------------------------------------------------------- work
def _conv_out(c):
    return (c["size"] + 2 * (c["kernel"] // 2) - c["kernel"]) // c["stride"] + 1


def work(case):
    c, kind = case, case["kind"]
    if kind == "round":
        return {"bytes": 8 * c["n"], "flops": 0}
    if kind == "mx":
        return {"bytes": 8 * c["rows"] * c["cols"], "flops": 0}
    if kind == "pack":
        return {"bytes": 2 * c["n"] * (4 + PACKED[c["to"]][2] / 8), "flops": 0}
    if kind == "gemm":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    if kind == "linear":
        r, i, o = c["rows"], c["in"], c["out"]
        if c["step"]:   # reads x, w, b, g; writes out, dx, dw, db
            return {"bytes": 4 * (2 * r * i + 2 * o * i + 2 * r * o + 2 * o),
                    "flops": 6 * r * i * o}
        return {"bytes": 4 * (r * i + o * i + r * o + o), "flops": 2 * r * i * o}
    if kind == "conv":
        p, taps = _conv_out(c), c["cin"] * c["kernel"] ** 2
        return {"bytes": 4 * (c["batch"] * c["cin"] * c["size"] ** 2 + c["cout"] * taps +
                              c["batch"] * c["cout"] * p * p),
                "flops": 2 * c["batch"] * c["cout"] * p * p * taps}
    s = _grouped_sizes(c)
    return {"bytes": 8 * (sum(s["rounds"]) + sum(s["mx"])) +
            4 * sum(m * k + k * n + m * n for m, n, k in s["gemms"]),
            "flops": 2 * sum(m * n * k for m, n, k in s["gemms"])}


# -------------------------------------------------------------------------------- 64-bit truth
def _lsr(z, n):
    """Logical right shift of 64-bit patterns held as int64."""
    return (z >> n) & ((1 << (64 - n)) - 1)


def _words(seed, n):
    """The first n 32-bit words of SplitMix64 (Steele, Lea, Flood 2014) from ``seed``."""
    s64 = lambda v: v - (1 << 64) if v >= 1 << 63 else v   # noqa: E731
    z = torch.arange(1, n + 1, device=DEV) * s64(0x9E3779B97F4A7C15) + int(seed)
    z = (z ^ _lsr(z, 30)) * s64(0xBF58476D1CE4E5B9)
    z = (z ^ _lsr(z, 27)) * s64(0x94D049BB133111EB)
    return _lsr(z ^ _lsr(z, 31), 32)


def _rounded(x, to, mode="rne", seed=None, limits=True):
    """x in 64 bits rounded to ``to``: (bits, mantissa bits, bias), or a number of mantissa
    bits.  A value past the largest passes through (a saturating format's rule here)."""
    x = x.double()
    mant = isinstance(to, int)
    m = to if mant else to[1]
    mag = x.abs()
    e = torch.frexp(mag).exponent.double() - 1
    if not mant:
        e = e.clamp(min=1 - to[2])
    q = torch.exp2(e - m)
    t = mag / q
    if mode == "rne":
        t = t.round()
    elif mode == "rtz":
        t = t.floor()
    else:
        r = (_words(seed, x.numel()) & ((1 << SR_LEN) - 1)).reshape(x.shape).double()
        up = (t + r / (1 << SR_LEN)).floor()
        t = up if mant else torch.where(t < 1, torch.zeros_like(t), up)
    y = torch.where(x < 0, -(t * q), t * q)
    if mant or not limits:
        return y
    top = 2.0 ** ((1 << (to[0] - 1 - to[1])) - 1 - to[2])
    return torch.where(y.abs() >= 2 * top, x, y)


def _mx_rounded(x, block, to, mode="rne", seed=None):
    """MX rounding in 64 bits: a power-of-two scale near amax / largest value per block."""
    v = x.double().reshape(-1, block)
    largest = (2.0 - 2.0 ** -to[1]) * 2.0 ** ((1 << (to[0] - 1 - to[1])) - 1 - to[2])
    f = torch.frexp(v.abs().amax(1, keepdim=True) / largest)
    e = f.exponent.double() - 1
    up = (f.mantissa > 0.75) | ((f.mantissa == 0.75) & (torch.remainder(e, 2) == 0))
    scale = torch.exp2(e + up.double())
    return (_rounded(v / scale, to, mode, seed) * scale).reshape(x.shape)


def _layer_operands(c, d):
    name = c["formats"].replace("mx_", "")
    if c["formats"].startswith("mx_"):
        return [_mx_rounded(d[k], 32, FORMATS[name]) for k in "xw"]
    if name == "fp32":
        return [d[k].double() for k in "xw"]
    return [_rounded(d[k], FORMATS[name]) for k in "xw"]


def exact(case, seed):
    c, kind, d = case, case["kind"], _inputs(case, seed)
    with torch.no_grad():
        if kind == "round":
            to = int(c["to"][4:]) if c["to"].startswith("mant") else FORMATS[c["to"]]
            return _rounded(d["x"], to, c["mode"], int(seed) + 17)
        if kind == "mx":
            return _mx_rounded(d["x"], c["block"], FORMATS[c["to"]], c["mode"], int(seed) + 17)
        if kind == "pack":
            m, bias, bits = PACKED[c["to"]]
            y = _rounded(d["x"], (bits, m, bias), limits=False)
            if c["to"] == "e2m1":   # 6 is its largest value; N(0, 1) data stays below
                y = y.clamp(-6, 6)
            return {"packed": None, "values": y}
        if kind == "gemm":
            if c["inputs"] == "fp32u":
                return d["a"].double() @ d["b"].double()
            a, b = (_rounded(d[k], FORMATS[c["inputs"]]) for k in "ab")
            return a @ b
        if kind == "linear":
            x, w = _layer_operands(c, d)
            out = x @ w.t() + d["b"].double()
            if not c["step"]:
                return out
            g = _rounded(d["g"], FORMATS["e5m2"], "sr", int(seed) + 29)
            return {"out": out, "dx": g @ w, "dw": g.t() @ x, "db": d["g"].double().sum(0)}
        if kind == "conv":
            x, w = _layer_operands(c, d)
            p, k = _conv_out(c), c["kernel"]
            cols = torch.nn.functional.unfold(x.cpu(), k, padding=k // 2, stride=c["stride"])
            y = w.reshape(c["cout"], -1) @ cols.to(DEV).contiguous()
            return y.reshape(c["batch"], c["cout"], p, p) + d["b"].double().view(1, -1, 1, 1)
        out, sizes = [], _grouped_sizes(c)
        for i in range(len(sizes["rounds"])):
            out.append(_rounded(d["r%d" % i], FORMATS[_JOB_FORMATS[i % 4]], _JOB_MODES[i % 3],
                                int(seed) + i))
        out += [_mx_rounded(d["m%d" % i], 32, FORMATS["e4m3"]) for i in range(len(sizes["mx"]))]
        for i in range(len(sizes["gemms"])):
            a, b = (_rounded(d[k + str(i)], FORMATS["e4m3"]) for k in "ab")
            out.append(a @ b)
        return out
