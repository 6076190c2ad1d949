"""The work this library is used for, as cases that can be timed and checked.

A case is one of these kinds of call:

* ``linear``: one quantized linear of a prompt, launched eagerly as a lowered
  graph calls it (``voyager_amd.lower``): the activation's quantize and the
  GEMM on the packed weight, in one of the four formats that are lowered.
* ``layer``: the seven linears of one decoder layer at decode batch sizes,
  each a lowered call, in a HIP graph that the program replays per token.
* ``outlier``: a converted graph's linear with an outlier stream, not lowered:
  ``quantize_mx_outlier`` and ``linear_mx`` with its CSR term.
* ``decode``: consecutive steps of two MX-int8 decoder layers over a 2-bit
  KIVI cache (``voyager_amd.decode``), in a HIP graph, the cache advancing.
* ``codec``: an elementwise quantize with one scale and the way back.
* ``mx``: a block-scaled quantize in the reference form and the way back
  (``quantize_mx`` / ``dequantize_mx``).
* ``affine``: a prompt's keys and values into the KIVI cache formats and the
  way back (``quantize_affine`` / ``dequantize``).

Sizes are the ones of ``bench.py`` and the tests, or generic.
"""

import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "voyager-compiler-2_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

BF16 = torch.bfloat16
BYTES_PER_WEIGHT = {"fp8": 1.0, "posit8": 2.0, "mxint8": 1.0 + 1 / 16, "mxnf4": 0.5 + 1 / 64}

# The block-scaled formats: element type, block, largest value, scale map
# (None: powers of two).
MX = {
    "mxint8": ("int8", 16, 127.0, None),
    "mxfp8": ("fp8_e4m3", 32, 448.0, None),
    "mxfp4": ("fp4_e2m1", 32, 6.0, None),
    "nvfp4": ("fp4_e2m1", 16, 6.0, "fp8_e4m3"),
    "mxnf4": ("lut4_to_int6", 64, 31.0, "fp8_e5m3"),
}
NF4_LEVELS = (-31., -22., -16., -12., -9., -6., -3., 0., 2., 5., 8., 10., 14., 17., 22., 31.)
OUTLIER, OUTLIER_SHARE = 5.0, 0.01
DECODE_STEPS = 4
EPS, THETA, HEAD = 1e-5, 5e5, 128


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: one token's activation, where launch and host time count
        {"name": "mx_one_token", "kind": "mx", "fmt": "mxint8", "rows": 1, "cols": 4096, "axis": -1},
        # a layer's linears for one token of a single user (bench.py's config 3 sizes)
        {"name": "layer_mxnf4_m1", "kind": "layer", "fmt": "mxnf4", "m": 1, "hidden": 4096, "kv": 1024, "inter": 14336},
        # the same for a batch of 16 users in the per-tensor FP8 format (config 2's weights)
        {"name": "layer_fp8_m16", "kind": "layer", "fmt": "fp8", "m": 16, "hidden": 4096, "kv": 1024, "inter": 14336},
        # ... and for a few users in MX-int8 (config 1's format)
        {"name": "layer_mxint8_m4", "kind": "layer", "fmt": "mxint8", "m": 4, "hidden": 4096, "kv": 1024,
         "inter": 14336},
        # a short prompt of odd length through the 4-bit format's up projection
        {"name": "linear_mxnf4_m201", "kind": "linear", "fmt": "mxnf4", "m": 201, "k": 4096, "n": 14336},
        # config 2's largest prefill projection
        {"name": "linear_fp8_m2048", "kind": "linear", "fmt": "fp8", "m": 2048, "k": 4096, "n": 14336},
        # a ragged prompt through the long-K projection in MX-int8
        {"name": "linear_mxint8_m1111", "kind": "linear", "fmt": "mxint8", "m": 1111, "k": 14336, "n": 4096},
        # config 1's linear with an outlier stream, as converted (not lowered)
        {"name": "outlier_m256", "kind": "outlier", "m": 256, "k": 4096, "n": 4096},
        # config 5: batch 8 over a context of 4096
        {"name": "decode_b8_4096", "kind": "decode", "batch": 8, "context": 4032, "hidden": 4096, "inter": 14336},
        # config 4: a 64M-element tensor to posit8 bytes and back
        {"name": "codec_posit8_64m", "kind": "codec", "fmt": "posit8_1", "packed": True, "n": 1 << 26},
        # a ragged prompt's MLP activation to MX FP8 and back
        {"name": "mx_fp8_1777", "kind": "mx", "fmt": "mxfp8", "rows": 1777, "cols": 14336, "axis": -1},
        # a prompt's keys and values into the KIVI cache formats and back (config 5's cache)
        {"name": "affine_kv_3968", "kind": "affine", "batch": 8, "heads": 8, "tokens": 3968},
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of ``step`` in [lo, hi], spread evenly over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, round(v / step) * step))


def draw(rng):
    kind = rng.choice(["linear", "linear", "layer", "layer", "outlier", "decode", "codec", "mx", "mx", "affine"])
    if kind == "linear":
        fmt = rng.choice(["fp8", "mxint8", "mxnf4", "posit8"])
        k, n = rng.choice([(4096, 4096), (4096, 1024), (4096, 14336), (14336, 4096), None]) or (
            _log(rng, 512, 14336, 64), _log(rng, 256, 14336, 16))
        most = 2048 * 4096 * 14336 // (k * n)
        return {"kind": kind, "fmt": fmt, "m": _log(rng, 17, min(2048, most)), "k": k, "n": n}
    if kind == "layer":
        hidden, kv, inter = rng.choice([(4096, 1024, 14336), (4096, 1024, 14336), (2048, 512, 8192), (3072, 1024, 8192),
                                        (1536, 256, 8960), (1024, 512, 2816)])
        return {"kind": kind, "fmt": rng.choice(["fp8", "mxint8", "mxnf4"]), "m": _log(rng, 1, 64), "hidden": hidden,
                "kv": kv, "inter": inter}
    if kind == "outlier":
        k, n = rng.choice([(4096, 4096), (4096, 1024), (2048, 2048)])
        return {"kind": kind, "m": _log(rng, 16, 1024), "k": k, "n": n}
    if kind == "decode":
        hidden, inter = rng.choice([(4096, 14336), (4096, 14336), (2048, 8192), (1024, 2816)])
        return {"kind": kind, "batch": _log(rng, 1, 16), "context": _log(rng, 40, 8000), "hidden": hidden,
                "inter": inter}
    if kind == "codec":
        return {"kind": kind, "fmt": rng.choice(["posit8_1", "fp8_e4m3", "int8"]), "packed": rng.random() < 0.5,
                "n": _log(rng, 1 << 12, 1 << 26)}
    if kind == "mx":
        return {"kind": kind, "fmt": rng.choice(sorted(MX)), "rows": _log(rng, 1, 2048),
                "cols": rng.choice([1024, 4096, 4096, 14336, _log(rng, 256, 14336, 64)]),
                "axis": rng.choice([-1, -1, -1, -2])}
    return {"kind": kind, "batch": _log(rng, 1, 8), "heads": rng.choice([1, 2, 8]), "tokens": _log(rng, 33, 4000)}


def _projections(case):
    """(name, K, N, input) of a decoder layer's seven linears."""
    h, kv, f = case["hidden"], case["kv"], case["inter"]
    return [("q", h, h, "h1"), ("k", h, kv, "h1"), ("v", h, kv, "h1"), ("o", h, h, "attn"), ("gate", h, f, "h2"),
            ("up", h, f, "h2"), ("down", f, h, "act")]


def _linears(case):
    """(name, M, K, N, input) of the linears of a ``linear`` or ``layer`` case."""
    if case["kind"] == "linear":
        return [("y", case["m"], case["k"], case["n"], "x")]
    return [(name, case["m"], k, n, x) for name, k, n, x in _projections(case)]


def work(case):
    kind = case["kind"]
    if kind in ("linear", "layer"):
        seen, b, f = set(), 0.0, 0.0
        for _, m, k, n, x in _linears(case):
            b += n * k * BYTES_PER_WEIGHT[case["fmt"]] + m * n * 2 + (0 if x in seen else m * k * 2)
            f += 2.0 * m * n * k
            seen.add(x)
        return {"bytes": b, "flops": f}
    if kind == "outlier":
        m, k, n = case["m"], case["k"], case["n"]
        # the weight's codes and scales as the converted graph holds them (bf16)
        return {"bytes": m * k * 2 + n * k * 2 + n * k // 16 * 2 + m * n * 2, "flops": 2.0 * m * n * k}
    if kind == "decode":
        b, h, f = case["batch"], case["hidden"], case["inter"]
        kv = h // 4
        weights = (h * (h + 2 * kv) + h * h + 3 * h * f) * 17 // 16
        main, res = _context(case)
        heads = kv // HEAD
        cache = b * heads * (main * 96 + (res + 1) * HEAD * 4)
        attn = 4.0 * b * (h // HEAD) * HEAD * (main + res + 1)
        n = 2 * DECODE_STEPS
        return {"bytes": n * (weights + cache + 4 * b * h), "flops": n * (2.0 * b * weights * 16 / 17 + attn)}
    if kind == "codec":
        # there (bf16 in, codes out) and back (codes in, bf16 out)
        return {"bytes": case["n"] * 2 * (2 + (1 if case["packed"] else 2)), "flops": 0}
    if kind == "mx":
        bs = MX[case["fmt"]][1]
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * (4 * n + 2 * n / bs), "flops": 0}
    n = case["batch"] * case["heads"] * case["tokens"] * HEAD
    return {"bytes": 2 * 2 * (4 * n + 4 * n / 32), "flops": 0}


def tolerance(case):
    # Codes, block scales and decoded values have one right answer.
    if case["kind"] in ("codec", "mx", "affine"):
        return "exact"
    # bf16 results of float32 sums, the FP8 ones rounded twice: measured 1.6e-3 to
    # 2.4e-3 from the 64-bit result.  A decode step quantizes four times on the
    # way, where one rounding moves whole codes: 6e-3 between two orders of its
    # sums, 1.7e-2 from 64 bits.
    return {"rel": 2.5e-2} if case["kind"] == "decode" else {"rel": 1e-2}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator("cuda").manual_seed(int(seed))


def _activation(g, *shape):
    """N(0, 1) with one value in a thousand twenty times as large (config 1)."""
    x = torch.randn(*shape, generator=g, device="cuda")
    return torch.where(torch.rand(*shape, generator=g, device="cuda") < 0.001, x * 20, x).to(BF16)


def _weight(g, n, k):
    return (torch.randn(n, k, generator=g, device="cuda") * 0.02).to(BF16)


def _amax_scale(t):
    """bf16(amax / 448), a calibrated per-tensor scale."""
    return (t.abs().amax().float() / 448.0).to(BF16)


def _linear_inputs(case, seed):
    """The activations by name, and each linear's weight, in bf16."""
    g = _gen(seed)
    xs, ws = {}, []
    for name, m, k, n, x in _linears(case):
        if x not in xs:
            xs[x] = _activation(g, m, k)
        ws.append((name, x, _weight(g, n, k)))
    return xs, ws


def _outlier_inputs(case, seed):
    g = _gen(seed)
    return _activation(g, case["m"], case["k"]), _weight(g, case["n"], case["k"])


def _context(case):
    """(main tokens, residual tokens) of the cache before the first step."""
    return case["context"] // 128 * 128, case["context"] % 128


def _decode_inputs(case, seed):
    """Two layers: weights, the cache's codes, scales and zero points, the
    residual window, and the step's input."""
    h, f, b = case["hidden"], case["inter"], case["batch"]
    kv, heads = h // 4, h // 4 // HEAD
    main, res = _context(case)
    layers = []
    for i in range(2):
        g = _gen(seed * 2 + i)

        def norm():
            return (1 + 0.1 * torch.randn(h, generator=g, device="cuda")).to(BF16)

        w = {"ln1": norm(), "wq": _weight(g, h, h), "wk": _weight(g, kv, h), "wv": _weight(g, kv, h),
             "wo": _weight(g, h, h), "ln2": norm(), "wg": _weight(g, f, h), "wu": _weight(g, f, h),
             "wd": _weight(g, h, f)}

        def affine(groups):
            """(scale, zero point, codes) as quantize_affine leaves N(0, 1) values."""
            codes = torch.randint(0, 4, (b, heads, main, HEAD), generator=g, device="cuda").to(BF16)
            scale = (1.2 + 0.2 * torch.randn(b, heads, *groups, generator=g, device="cuda")).clamp(0.5, 2).to(BF16)
            zero = (1.5 + 0.2 * torch.randn(b, heads, *groups, generator=g, device="cuda")).to(BF16)
            return scale, zero, codes

        kq, vq = affine((main // 32, HEAD)), affine((main, HEAD // 32))
        kr, vr = (torch.randn(b, heads, res, HEAD, generator=g, device="cuda").to(BF16) for _ in range(2))
        x = torch.randn(b, h, generator=g, device="cuda").to(BF16)
        layers.append((w, kq, vq, kr, vr, x))
    return layers


def _codec_input(case, seed):
    return (torch.randn(case["n"], generator=_gen(seed), device="cuda") * 2).to(BF16)


def _codec_scale(case, x):
    return torch.ones((), dtype=BF16, device="cuda") if case["fmt"].startswith("posit") else (
        x.abs().amax().float() / (448.0 if case["fmt"].startswith("fp8") else 127.0)).to(BF16)


def _affine_inputs(case, seed):
    g = _gen(seed)
    shape = (case["batch"], case["heads"], case["tokens"], HEAD)
    return tuple(torch.randn(*shape, generator=g, device="cuda").to(BF16) for _ in range(2))


# ------------------------------------------------------------------ prepare and run
_TABLES = {}


def _table(dtype):
    """A dtype's map, one per program as in a graph's buffers."""
    from voyager_amd import formats

    if dtype not in _TABLES:
        _TABLES[dtype] = (formats.codebook_tables(dtype, "cuda") if dtype.startswith("lut")
                          else formats.quantization_map(dtype, "cuda"))
    return _TABLES[dtype]


def _bake(fmt, x, w):
    """A lowered site's call on the activation ``x``, its weight packed once."""
    from voyager_amd import formats, gemm, lower, packed

    if fmt == "fp8":
        tab, sx, sw = _table("fp8_e4m3"), _amax_scale(x), _amax_scale(w)
        wq, s = packed.quantize_packed(w, sw, tab), sx * sw
        return lambda: lower.lowered_fp8_linear(x, sx, tab, wq, s)
    if fmt == "posit8":
        tab, one = _table("posit8_1"), torch.ones((), dtype=BF16, device="cuda")
        wq = torch.ops.quantized_ops.quantize(w, one, qmap=tab)
        return lambda: lower.lowered_posit8_linear(x, one, tab, wq)
    if fmt == "mxint8":
        tab = _table("int8")
        p = packed.quantize_mx_packed(w, tab, [-1], 16, 127.0, True)
        return lambda: lower.lowered_mxint8_linear(x, tab, p.codes, p.scale, p.bias, 16)
    index, entries, _ = _table("lut4_to_int6")
    stab = _table("fp8_e5m3")
    formats.classify(index)
    b = gemm.bake_nf4_weight(w, index, stab, entries)
    levels = tuple(b.levels)
    return lambda: lower.lowered_mxnf4_linear(x, index, stab, b.packed, b.scale, levels, b.N)


def _capture(fn):
    """A HIP graph of ``fn`` and what it returns, after two eager runs."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = fn()
    return g, out


def prepare(case, seed):
    import voyager_amd.library  # noqa: F401  (defines quantized_ops)
    from voyager_amd import decode, packed

    q = torch.ops.quantized_ops
    kind = case["kind"]
    if kind in ("linear", "layer"):
        xs, ws = _linear_inputs(case, seed)
        calls = [(name, _bake(case["fmt"], xs[x], w)) for name, x, w in ws]
        del ws
        if kind == "linear":
            return {"call": calls[0][1]}
        g, out = _capture(lambda: {name: call() for name, call in calls})
        return {"graph": g, "out": out, "keep": calls}
    if kind == "outlier":
        x, w = _outlier_inputs(case, seed)
        tab = _table("int8")
        ws, wc = q.quantize_mx(w, tab, [-1], 16, 127.0, True)

        def call():
            d, i, p, s, c = q.quantize_mx_outlier(x, tab, [-1], 16, 127.0, True, threshold=OUTLIER,
                                                  max_pct=OUTLIER_SHARE)
            return q.linear_mx(c, wc, input_scale=s, weight_scale=ws, block_size=16, A_data=d, A_indices=i,
                               A_indptr=p)

        return {"call": call}
    if kind == "decode":
        h = case["hidden"]
        heads, kv = h // HEAD, h // 4 // HEAD
        main, res = _context(case)
        capacity = main + 2 * decode.RES_CAP
        runs = []
        for w, kq, vq, kr, vr, x in _decode_inputs(case, seed):
            layer = decode.DecoderLayer(w, heads, kv, EPS, THETA, max_batch=case["batch"], max_pos=capacity)
            cache = decode.KiviCache(case["batch"], kv, capacity, torch.device("cuda"))
            cache.load_main(kq, vq)
            cache.load_residual(kr, vr)
            layer.stages(x, cache)  # sizes the attention workspace
            runs.append((layer, cache, x, cache.state.clone(), (cache.n_main, cache.n_res)))

        def steps():
            # from the same position each time, so that every pass is the same steps
            for _, cache, _, state, (cache.n_main, cache.n_res) in runs:
                cache.state.copy_(state)
            for _ in range(DECODE_STEPS):
                outs = [layer.step(x, cache) for layer, cache, x, _, _ in runs]
            return {"out": outs, "keys": [r[1].kr for r in runs], "values": [r[1].vr for r in runs]}

        g, out = _capture(steps)
        return {"graph": g, "out": out, "keep": runs}
    if kind == "codec":
        x, tab = _codec_input(case, seed), _table(case["fmt"])
        s = _codec_scale(case, x)
        if case["packed"]:
            def call():
                c = packed.quantize_packed(x, s, tab)
                return c, packed.unpack_codes(c, tab)
        else:
            def call():
                c = q.quantize(x, s, qmap=tab)
                return c, q.dequantize(c, s)
        return {"call": call}
    if kind == "mx":
        x = _activation(_gen(seed), case["rows"], case["cols"])
        dtype, bs, qmax, scale = MX[case["fmt"]]
        code = None
        if dtype.startswith("lut"):
            tab, code, mid = _table(dtype)
        else:
            tab, mid = _table(dtype), None
        stab = None if scale is None else _table(scale)

        axis = case["axis"]  # -2: blocks along the rows, as a product's second operand is quantized

        def call():
            s, c = q.quantize_mx(x, tab, [axis], bs, qmax, scale is None, stab, mid)
            return s, c, q.dequantize_mx(c, s, bs, code)

        return {"call": call}
    k, v = _affine_inputs(case, seed)
    tab, stab = _table("uint2"), _table("fp16_e5m10")

    def call():
        out = []
        for t, axis in ((k, -2), (v, -1)):
            s, z, c = q.quantize_affine(t, tab, [axis], 32, 0.0, 3.0, stab)
            out += [s, z, c, q.dequantize(c, s, z, [axis], 32)]
        return out

    return {"call": call}


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return state["call"]()


# ------------------------------------------------------------------ in 64 bits
def _exp2(e):
    """2**e of whole numbers, exactly."""
    return ((e.to(torch.int64) + 1023) << 52).view(torch.float64)


def _pot(v, qmax, bs):
    """The power-of-two block scale of each element's block along the last dim."""
    n = v.shape[-1]
    p = torch.nn.functional.pad(v.double(), (0, -n % bs)).unflatten(-1, (-1, bs))
    amax = p.abs().amax(-1)
    e = torch.frexp(torch.where(amax > 0, amax, 2.0 ** -126))[1] - 1 - math.floor(math.log2(qmax))
    return _exp2(e)


def _spread(s, bs, n):
    return s.repeat_interleave(bs, dim=-1)[..., :n]


def _int8_mx(v):
    """``v`` as MX-int8 (blocks of 16) holds it."""
    s = _spread(_pot(v, 127.0, 16), 16, v.shape[-1])
    return torch.clamp(torch.round(v.double() / s), -128, 127) * s


def _minifloat(v, emin, mbits, most):
    """Round half to even onto a minifloat's grid, saturating."""
    v = v.double()
    e = torch.clamp(torch.frexp(v)[1] - 1, min=emin)
    step = _exp2(e - mbits)
    return torch.clamp(torch.round(v / step) * step, -most, most)


def _posit8(v):
    """The nearest posit<8, 1> of each value by its bit string (a 9-bit
    posit's odd codes lie between), zero under 2**-13."""
    def value(code, n):
        body = [(code >> i) & 1 for i in range(n - 2, -1, -1)]
        run = 1
        while run < len(body) and body[run] == body[0]:
            run += 1
        k = run - 1 if body[0] else -run
        rest = body[run + 1:] + [0]
        e, frac = rest[0], rest[1:]
        return 2.0 ** (2 * k + e) * (1 + sum(b / 2.0 ** (i + 1) for i, b in enumerate(frac)))

    dev = v.device
    pos = torch.tensor([0.0] + [value(c, 8) for c in range(1, 128)], dtype=torch.float64, device=dev)
    mid = torch.tensor([2.0 ** -13] + [value(2 * c + 1, 9) for c in range(1, 127)], dtype=torch.float64, device=dev)
    # a tie goes to the even code: above the midpoint for even codes, from it on for odd ones
    odd = torch.arange(127, device=dev) % 2 == 1
    edge = torch.where(odd | (torch.arange(127, device=dev) == 0), mid, torch.nextafter(mid, torch.full_like(mid, 1e9)))
    d = v.double()
    return torch.sign(d) * pos[torch.bucketize(d.abs(), edge, right=True)]


def _nf4(v):
    """(scale per block, index) of MX-NF4's 64-element blocks."""
    n = v.shape[-1]
    amax = torch.nn.functional.pad(v, (0, -n % 64)).unflatten(-1, (-1, 64)).abs().amax(-1)
    s = _minifloat((amax.float() / 31.0).to(BF16), -14, 3, 61440.0).to(BF16)
    s = torch.where(s > 0, s, torch.ones_like(s))
    lv = torch.tensor(NF4_LEVELS, dtype=torch.float64, device=v.device)
    quot = (v.float() / _spread(s, 64, n).float()).to(BF16).double()
    return s, torch.bucketize(quot, (lv[:-1] + lv[1:]) / 2), lv


def _operand(fmt, v):
    """``v`` as the format's GEMM operand holds it, in 64 bits."""
    if fmt == "posit8":
        return _posit8(v)
    if fmt == "mxint8":
        return _int8_mx(v)
    s, i, lv = _nf4(v)
    return lv[i] * _spread(s, 64, v.shape[-1]).double()


def _fp8(v, s):
    return _minifloat((v.float() / s.float()).to(BF16), -6, 3, 448.0)


def _exact_decode(case, seed):
    main, res = _context(case)
    if res + DECODE_STEPS >= 128:
        return None  # the window folds into the quantized cache on the way
    b, h = case["batch"], case["hidden"]
    heads, kv = h // HEAD, h // 4 // HEAD
    outs, keys, values = [], [], []
    inv = 1.0 / (THETA ** (torch.arange(0, HEAD, 2, device="cuda").double() / HEAD))

    def norm(x, w):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()

    def turn(t, pos):
        a = torch.cat((pos * inv, pos * inv))
        half = torch.cat((-t[..., HEAD // 2:], t[..., :HEAD // 2]), dim=-1)
        return t * a.cos() + half * a.sin()

    for w, kq, vq, kr, vr, x in _decode_inputs(case, seed):
        x = x.double()
        wd = {n: _int8_mx(w[n]) for n in ("wq", "wk", "wv", "wo", "wg", "wu", "wd")}
        h1 = _int8_mx(norm(x, w["ln1"]))
        qh = (h1 @ wd["wq"].T).view(b, heads, HEAD)
        kh, vh = ((h1 @ wd[n].T).view(b, kv, HEAD) for n in ("wk", "wv"))
        ks, kz, kc = (t.double() for t in kq)
        vs, vz, vc = (t.double() for t in vq)
        km = (kc - kz.repeat_interleave(32, 2)) * ks.repeat_interleave(32, 2)
        vm = (vc - vz.repeat_interleave(32, 3)) * vs.repeat_interleave(32, 3)
        new_k = torch.stack([turn(kh, main + res + i) for i in range(DECODE_STEPS)], dim=2)
        new_v = vh[:, :, None].expand(-1, -1, DECODE_STEPS, -1)
        k_win, v_win = torch.cat((kr.double(), new_k), 2), torch.cat((vr.double(), new_v), 2)
        ka, va = torch.cat((km, k_win), 2), torch.cat((vm, v_win), 2)
        qg = turn(qh, main + res + DECODE_STEPS - 1).view(b, kv, heads // kv, HEAD)
        p = torch.softmax(torch.matmul(qg, ka.transpose(2, 3).contiguous()) * HEAD ** -0.5, -1)
        attn = torch.matmul(p, va.contiguous()).reshape(b, h)
        x1 = x + _int8_mx(attn) @ wd["wo"].T
        h2 = _int8_mx(norm(x1, w["ln2"]))
        gate, up = h2 @ wd["wg"].T, h2 @ wd["wu"].T
        outs.append(x1 + _int8_mx(gate * torch.sigmoid(gate) * up) @ wd["wd"].T)
        pad = (0, 0, 0, 128 - k_win.shape[2])
        keys.append(torch.nn.functional.pad(k_win, pad).reshape(b * kv, 128, HEAD))
        values.append(torch.nn.functional.pad(v_win, pad).reshape(b * kv, 128, HEAD))
    return {"out": outs, "keys": keys, "values": values}


def _exact_mx(case, seed):
    x = _activation(_gen(seed), case["rows"], case["cols"])
    dtype, bs, qmax, scale = MX[case["fmt"]]
    if case["axis"] == -2:
        x = x.T.contiguous()
    n = x.shape[-1]
    if case["fmt"] == "mxnf4":
        s, i, lv = _nf4(x)
        out = (s.double(), i.double(), lv[i] * _spread(s, bs, n).double())
    else:
        if scale is None:
            s = _pot(x, qmax, bs)
        else:
            amax = torch.nn.functional.pad(x, (0, -n % bs)).unflatten(-1, (-1, bs)).abs().amax(-1)
            s = _minifloat((amax.float() / qmax).to(BF16), -6, 3, 448.0)
            s = torch.where(s > 0, s, torch.ones_like(s))
        quot = (x.float() / _spread(s, bs, n).float()).to(BF16)
        if dtype == "int8":
            c = torch.clamp(torch.round(quot.double()), -128, 127)
        else:
            c = _minifloat(quot, -6, 3, 448.0) if dtype == "fp8_e4m3" else _minifloat(quot, 0, 1, 6.0)
        out = (s, c, c * _spread(s, bs, n))
    return tuple(t.T.contiguous() for t in out) if case["axis"] == -2 else out


def _exact_affine(case, seed):
    out = []
    for t, axis in zip(_affine_inputs(case, seed), (-2, -1)):
        v = t.mT if axis == -2 else t
        n = v.shape[-1]
        g = torch.nn.functional.pad(v, (0, -n % 32)).unflatten(-1, (-1, 32))
        hi, lo = g.amax(-1), g.amin(-1)
        half = lambda a: _minifloat(a, -14, 10, 65504.0).to(BF16)  # noqa: E731
        s = half(((hi - lo).float() / 3.0).to(BF16))
        z = half((-lo.float() / s.float()).to(BF16))
        sp, zp = _spread(s, 32, n), _spread(z, 32, n)
        quot = ((v.float() / sp.float()).to(BF16).float() + zp.float()).to(BF16)
        c = torch.clamp(torch.round(quot.double()), 0, 3)
        got = (s.double(), z.double(), c, (c - zp.double()) * sp.double())
        out += [a.mT.contiguous() if axis == -2 else a for a in got]
    return out


def exact(case, seed):
    kind, fmt = case["kind"], case.get("fmt")
    if kind in ("linear", "layer"):
        xs, ws = _linear_inputs(case, seed)
        out = {}
        for name, x, w in ws:
            if fmt == "fp8":
                sx, sw = _amax_scale(xs[x]), _amax_scale(w)
                out[name] = (_fp8(xs[x], sx) @ _fp8(w, sw).T) * (sx * sw).double()
            else:
                out[name] = _operand(fmt, xs[x]) @ _operand(fmt, w).T
        return out["y"] if kind == "linear" else out
    if kind == "outlier":
        x, w = _outlier_inputs(case, seed)
        big = x.abs() >= OUTLIER
        inliers = torch.where(big, torch.zeros_like(x), x)
        return (_int8_mx(inliers) + torch.where(big, x, torch.zeros_like(x)).double()) @ _int8_mx(w).T
    if kind == "decode":
        return _exact_decode(case, seed)
    if kind == "codec":
        x = _codec_input(case, seed)
        s = _codec_scale(case, x)
        if fmt.startswith("posit"):
            v = _posit8(x)
        elif fmt.startswith("fp8"):
            v = _fp8(x, s)
        else:
            v = torch.clamp(torch.round((x.float() / s.float()).to(BF16).double()), -128, 127)
        return (None, v) if case["packed"] else (v, v * s.double())
    if kind == "mx":
        return _exact_mx(case, seed)
    return _exact_affine(case, seed)
