"""The work whose time matters to a program that serves or packs models with this package.

Every case runs through the public entry points: the drop-in operators on one layer as the
layer packers return it ((K, N) codes), the packed Linear layers over a container's (N, K)
rows, whole-stream decode steps, and the two layer packers themselves.  The weights are what
the package's benchmark synthesises: a heavy-tailed base shared by the models plus a small
Gaussian difference per model, so codes, plug tables and group scales are distributed as in a
packed model.  Codes are made here, not by the package's packers, so that the inputs depend on
the seed alone.
"""
import math

import torch

from polar_pack_amd import polar_kernels as pk
from polar_pack_amd import quad_kernels as qk
from polar_pack_amd.container import DualPackDevice, QuadPackDevice
from polar_pack_amd.linear import DualPackedLinear, QuadPackedLinear
from polar_pack_amd.stream import DualStream, QuadStream

DEV = "cuda:0"
MU = 255.0
GROUP = 32
CHUNK = 50_000_000
STD = 0.02
# The Linear weights of one layer of the 3B-shaped model, (N, K) in stream order.
LAYER = [(2048, 2048), (256, 2048), (256, 2048), (2048, 2048), (11008, 2048), (11008, 2048), (2048, 11008)]


def listed():
    return [
        # the smallest call: one token through a key/value projection of a packed model
        {"name": "quad_rows_kv_m1", "kind": "quad_rows", "N": 256, "K": 2048, "M": 1},
        # a small serving batch through the widest projection of that model
        {"name": "quad_rows_gate_m16", "kind": "quad_rows", "N": 11008, "K": 2048, "M": 16},
        # the reference benchmark's layer as the layer packer returns it: one token ...
        {"name": "quad_kn_4096_m1", "kind": "quad_kn", "N": 4096, "K": 4096, "M": 1},
        # ... a batch of decodes or a short prompt ...
        {"name": "quad_kn_4096_m32", "kind": "quad_kn", "N": 4096, "K": 4096, "M": 32},
        # ... and prefill
        {"name": "quad_kn_4096_m1024", "kind": "quad_kn", "N": 4096, "K": 4096, "M": 1024},
        # the same layer for two models: a small batch, and prefill
        {"name": "dual_kn_4096_m8", "kind": "dual_kn", "N": 4096, "K": 4096, "M": 8},
        {"name": "dual_kn_4096_m512", "kind": "dual_kn", "N": 4096, "K": 4096, "M": 512},
        # a Linear of odd sizes in a two-model container: few tokens, ragged rows
        {"name": "dual_rows_ragged_m3", "kind": "dual_rows", "N": 1531, "K": 4104, "M": 3},
        # one decode step of a whole 3B-shaped model: four models from one stream ...
        {"name": "quad_stream_3b", "kind": "quad_stream", "layers": 36, "M": 1},
        # ... and two models of unequal length, the longer one's last weights as fp16 tails
        {"name": "dual_stream_3b", "kind": "dual_stream", "layers": 36, "M": 1},
        # packing a layer (the encoding direction), four models and two
        {"name": "quad_pack_4096", "kind": "quad_pack", "N": 4096, "K": 4096},
        {"name": "dual_pack_down", "kind": "dual_pack", "N": 2048, "K": 11008},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size over [lo, hi]: half of them multiples of 64, a quarter of 8, the rest any."""
    v = _log_int(rng, lo, hi)
    step = rng.choice((64, 64, 8, 1))
    return max(lo, v // step * step)


def draw(rng):
    kind = rng.choice(("quad_rows", "quad_kn", "dual_rows", "dual_kn", "quad_stream", "dual_stream", "quad_pack",
                       "dual_pack"))
    if kind.endswith("stream"):
        return {"kind": kind, "layers": _log_int(rng, 1, 36), "M": rng.choice((1, 1, 2, 4))}
    while True:
        N, K = _size(rng, 256, 11008), _size(rng, 256, 11008)
        if N * K <= 4096 * 4096:
            break
    if kind.endswith("pack"):
        return {"kind": kind, "N": N, "K": K}
    return {"kind": kind, "N": N, "K": K, "M": _log_int(rng, 1, 1024 if kind.endswith("kn") else 256)}


# ------------------------------------------------------------------------------ weights

def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _base(n, df, g):
    """Student-t(df) values of standard deviation STD."""
    z = torch.randn(n, generator=g, device=DEV)
    chi = torch.zeros_like(z)
    for _ in range(df):
        chi += torch.randn(n, generator=g, device=DEV).square_()
    return z.div_(chi.div_(df).sqrt_()).mul_(STD / math.sqrt(df / (df - 2.0)))


def _quad_models(n, g):
    base = _base(n, 5, g)
    return [(base + torch.randn(n, generator=g, device=DEV) * (0.1 * STD * (m + 1))).half() for m in range(4)]


def _quad_rms():
    return [STD * math.sqrt(1.0 + (0.1 * (m + 1)) ** 2) for m in range(4)]


def _dual_models(n, g):
    base = _base(n, 3, g)
    return base.half(), (base + torch.randn(n, generator=g, device=DEV) * (0.2 * STD)).half()


# -------------------------------------------------------------------------------- codes

def _threshold(values, share):
    """The value that about ``share`` of ``values`` exceed (from at most 2 million of them)."""
    flat = values[::max(1, values.numel() // 2_000_000)]
    return torch.sort(flat).values[min(flat.numel() - 1, int(flat.numel() * (1.0 - share)))]


def _quad_codes(models, r_max):
    """(code words as int32, tuple norms, normalised tuples) of four flat weight tensors."""
    a, b, c, d = (m.float() / s for m, s in zip(models, _quad_rms()))
    cd = c * c + d * d
    bcd = cd + b * b
    r = torch.sqrt(bcd + a * a)
    top = r_max if r_max is not None else float(r.max()) * 1.001
    nq = torch.round(torch.log1p(MU * r / top) / math.log1p(MU) * 255).clamp_(0, 255).int()
    q1 = torch.round(torch.atan2(bcd.sqrt(), a) * (255 / math.pi)).int()
    q2 = torch.round(torch.atan2(cd.sqrt(), b) * (255 / math.pi)).int()
    q3 = torch.round(torch.atan2(d, c).remainder(2 * math.pi) * (255 / (2 * math.pi))).int().clamp_(0, 255)
    return (nq << 24) | (q1 << 16) | (q2 << 8) | q3, r, (a, b, c, d), top


def _quad_pack(sizes, g, share=0.001):
    """A four-model stream of projections of ``sizes`` weights, the tuples of largest norm
    (``share`` of them) in the plug table."""
    n = sum(sizes)
    codes = torch.empty(n, dtype=torch.int32, device=DEV)
    idx, vals, pos, thr = [], [], 0, None
    r_max = None if len(sizes) == 1 else 128.0        # of the order a 3B stream's tail reaches
    for size in sizes:
        w, r, wn, top = _quad_codes(_quad_models(size, g), r_max)
        codes[pos:pos + size] = w
        thr = _threshold(r, share) if thr is None else thr
        hit = torch.nonzero(r > thr).flatten()
        idx.append(hit + pos)
        vals.append(torch.stack([x[hit] for x in wn], 1).half())
        pos += size
    idx = torch.cat(idx)
    idx = torch.where(idx >= 1 << 31, idx - (1 << 32), idx).int().view(torch.uint32)
    return QuadPackDevice(n=n, s=tuple(_quad_rms()), r_max=top, codes=codes.view(torch.uint32), plug_idx=idx,
                          plug_vals=torch.cat(vals), tails=[torch.zeros(0, dtype=torch.float16, device=DEV)] * 4)


def _dual_codes(w1, w2):
    """(16-bit codes as int32, fp16 group scales, amplitudes, amplitude errors) of two flat
    weight tensors, groups of GROUP pairs from the first."""
    w1, w2 = w1.float(), w2.float()
    amp = torch.sqrt(w1 * w1 + w2 * w2)
    phase = torch.round((torch.atan2(w2, w1) + math.pi) * (1024 / (2 * math.pi))).int() & 1023
    pad = (-amp.numel()) % GROUP
    grouped = torch.nn.functional.pad(amp, (0, pad)).view(-1, GROUP)
    top = grouped.amax(dim=1, keepdim=True)
    top = torch.where(top > 1e-10, top, torch.ones_like(top))
    level = torch.round(torch.log1p(MU * (grouped / top)) * (63 / math.log1p(MU))).clamp_(0, 63)
    err = (torch.expm1(level * (math.log1p(MU) / 63)) / MU * top - grouped).abs().flatten()[:amp.numel()]
    return (level.int().flatten()[:amp.numel()] << 10) | phase, top.flatten().half(), amp, err


def _dual_pack(n1, n2, g, share=0.01, tails=False):
    """A two-model container of n1 and n2 weights (tails: the longer one's rest in fp16)."""
    n = 8 * (min(n1, n2) // 8) if tails else n1
    m1 = torch.empty(n1, dtype=torch.float16, device=DEV)
    m2 = torch.empty(n2, dtype=torch.float16, device=DEV)
    for lo in range(0, n1, CHUNK):
        hi = min(lo + CHUNK, n1)
        a, b = _dual_models(hi - lo, g)
        m1[lo:hi] = a
        m2[lo:min(hi, n2)] = b[:max(0, min(hi, n2) - lo)]
    codes = torch.empty(n, dtype=torch.int16, device=DEV)
    scales, idx, vals = [], [], []
    for lo in range(0, n, CHUNK):
        hi = min(lo + CHUNK, n)
        c, sc, amp, err = _dual_codes(m1[lo:hi], m2[lo:hi])
        c = ((c & 0xFF) << 8) | (c >> 8)                                     # the file's big-endian words
        codes[lo:hi] = torch.where(c >= 0x8000, c - 0x10000, c).short()
        hit = torch.nonzero(err > _threshold(err, share)).flatten()
        scales.append(sc)
        idx.append(hit + lo)
        vals.append(amp[hit].half())
    idx = torch.cat(idx)
    idx = torch.where(idx >= 1 << 31, idx - (1 << 32), idx).int().view(torch.uint32)
    return DualPackDevice(n_codes=n, n1=n1, n2=n2, codes=codes, layout="u16be", scales=torch.cat(scales),
                          plug_idx=idx, plug_val=torch.cat(vals), group_size=GROUP, chunk_size=CHUNK,
                          tails=[m1[n:].clone(), m2[n:].clone()] if tails else [])


def _quad_layer_luts(r_max):
    return [t.half() for t in qk.header_luts(r_max, device=DEV)]


# --------------------------------------------------------------------------------- cases

def _shapes(case):
    return LAYER * case["layers"]


def _x(M, K, g):
    return torch.randn((M, K), generator=g, device=DEV).half()


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind in ("quad_stream", "dual_stream"):
        shapes, M = _shapes(case), case["M"]
        if kind == "quad_stream":
            pack = _quad_pack([n * k for n, k in shapes], g)
            st = QuadStream(pack, shapes, M=M)
        else:
            n1 = sum(n * k for n, k in shapes)
            pack = _dual_pack(n1, int(0.95 * n1), g, tails=True)
            st = DualStream(pack, shapes, M=M)
        xs = [_x(M, K, g) for _, K in shapes]
        # every projection's outputs as column slices of one buffer a model
        outs = [torch.empty((M, sum(N for N, _ in shapes)), dtype=torch.float16, device=DEV)
                for _ in range(4 if kind == "quad_stream" else 2)]
        st.bind(xs, [list(t) for t in zip(*(o.split([N for N, _ in shapes], 1) for o in outs))])
        return {"kind": kind, "stream": st, "xs": xs, "outs": outs}
    N, K = case["N"], case["K"]
    if kind == "quad_pack":
        return {"kind": kind, "ws": [w.view(K, N) for w in _quad_models(K * N, g)]}
    if kind == "dual_pack":
        return {"kind": kind, "ws": [w.view(K, N) for w in _dual_models(K * N, g)]}
    x = _x(case["M"], K, g)
    if kind == "quad_rows":
        return {"kind": kind, "x": x, "layer": QuadPackedLinear(_quad_pack([N * K], g), N, K, 0)}
    if kind == "dual_rows":
        return {"kind": kind, "x": x, "layer": DualPackedLinear(_dual_pack(N * K, N * K, g), N, K, 0)}
    if kind == "quad_kn":
        codes, _, _, top = _quad_codes(_quad_models(K * N, g), None)
        return {"kind": kind, "x": x, "codes": codes.view(torch.uint32).view(K, N), "luts": _quad_layer_luts(top),
                "scales": _quad_rms()}
    codes, scales, _, _ = _dual_codes(*_dual_models(K * N, g))
    luts = [t.half() for t in pk.header_luts(device=DEV)]
    return {"kind": kind, "x": x, "codes": (codes - 32768).short().view(K, N), "scales": scales, "luts": luts}


def run(state):
    kind = state["kind"]
    if kind in ("quad_stream", "dual_stream"):
        state["stream"]()
        return state["outs"]
    if kind in ("quad_rows", "dual_rows"):
        return state["layer"](state["x"])
    if kind == "quad_kn":
        return qk.quad_bitpacked(state["x"], state["codes"], state["luts"], state["scales"])
    if kind == "dual_kn":
        return pk.polar_dual_bitpacked(state["x"], state["codes"], state["scales"], *state["luts"])
    if kind == "quad_pack":
        codes, luts, scales = qk.pack_quad_layer(*state["ws"])
        return codes.view(torch.int32), luts, scales
    return pk.quantize_polar_bitpacked(*state["ws"])


def work(case):
    kind = case["kind"]
    models = 4 if kind.startswith("quad") else 2
    if kind == "quad_pack":
        n = case["N"] * case["K"]
        return {"bytes": 12 * n, "flops": 0}
    if kind == "dual_pack":
        n = case["N"] * case["K"]
        return {"bytes": 6 * n + 2 * (n // GROUP), "flops": 0}
    shapes = _shapes(case) if kind.endswith("stream") else [(case["N"], case["K"])]
    M = case["M"]
    n = sum(N * K for N, K in shapes)
    act = sum(2 * M * K + 2 * models * M * N for N, K in shapes)
    if models == 4:
        code = 4 * n + (0 if kind == "quad_kn" else 12 * int(0.001 * n))
    else:
        coded = int(0.95 * n) if kind == "dual_stream" else n
        code = 2 * coded + 2 * (coded // GROUP) + (0 if kind == "dual_kn" else 6 * int(0.01 * coded)) + 2 * (n - coded)
    return {"bytes": code + act, "flops": 2 * models * M * n}


def tolerance(case):
    kind = case["kind"]
    if kind.endswith("pack"):
        return "exact"
    # One token: float32 weights and sums, fp16 outputs (2.1e-4 of the norm measured).  More
    # tokens: the weights are rounded to fp16 as well, as the reference's kernels do (2.9e-4).
    if kind.endswith("stream") or case["M"] == 1:
        return {"rel": 8e-4}
    return {"rel": 1.2e-3}


# ---------------------------------------------------------------------------- 64-bit values

def _quad_rows_f64(words, luts):
    """The four normalised weights of int32 code words, decoded in 64 bits."""
    norm, c1, s1, c2, s2, c3, s3 = luts
    r = norm[(words >> 24) & 255]
    q1, q2, q3 = (words >> 16) & 255, (words >> 8) & 255, words & 255
    out = [r * c1[q1]]
    r = r * s1[q1]
    out.append(r * c2[q2])
    r = r * s2[q2]
    return out + [r * c3[q3], r * s3[q3]]


def _header_quad_luts(r_max):
    i = torch.arange(256, dtype=torch.float64, device=DEV) / 255
    half, full = i * math.pi, i * 2 * math.pi
    return [torch.expm1(i * math.log1p(MU)) * r_max / MU, half.cos(), half.sin(), half.cos(), half.sin(), full.cos(),
            full.sin()]


def _header_dual_luts():
    i = torch.arange(64, dtype=torch.float64, device=DEV) / 63
    ang = torch.arange(1024, dtype=torch.float64, device=DEV) / 1024 * 2 * math.pi - math.pi
    return [torch.expm1(i * math.log1p(MU)) / MU, ang.cos(), ang.sin()]


def _positions(idx):
    return idx.view(torch.int32).long() & 0xFFFFFFFF


def _quad_linear_f64(pack, luts, pos0, N, K, x):
    """The four outputs (M, N) of the (N, K) rows at stream position ``pos0``, 64-bit."""
    xd = x.double()
    pos = _positions(pack.plug_idx)
    step = max(1, (1 << 24) // K)
    outs = [[] for _ in range(4)]
    for lo in range(0, N, step):
        hi = min(N, lo + step)
        a, b = pos0 + lo * K, pos0 + hi * K
        w = _quad_rows_f64(pack.codes.view(torch.int32)[a:b], luts)
        p0, p1 = (int(v) for v in torch.searchsorted(pos, torch.tensor([a, b], device=DEV)))
        for m in range(4):
            w[m][pos[p0:p1] - a] = pack.plug_vals[p0:p1, m].double()
            outs[m].append(xd @ (w[m].view(hi - lo, K).t() * pack.s[m]))
    return [torch.cat(o, 1) for o in outs]


def _dual_linear_f64(pack, luts, pos0, N, K, x):
    """The two outputs (M, N) of the (N, K) rows at stream position ``pos0``, 64-bit."""
    amp_lut, cos, sin = luts
    xd = x.double()
    pos = _positions(pack.plug_idx)
    per_chunk = -(-pack.chunk_size // GROUP)
    step = max(1, (1 << 24) // K)
    outs = [[], []]
    for lo in range(0, N, step):
        hi = min(N, lo + step)
        a, b = pos0 + lo * K, pos0 + hi * K
        c = max(a, min(b, pack.n_codes))                      # coded up to here, tails above
        v = pack.codes[a:c].int() & 0xFFFF
        v = ((v & 0xFF) << 8) | (v >> 8)
        at = torch.arange(a, c, device=DEV)
        group = at // pack.chunk_size * per_chunk + at % pack.chunk_size // GROUP
        amp = amp_lut[v >> 10] * pack.scales[group].double()
        p0, p1 = (int(q) for q in torch.searchsorted(pos, torch.tensor([a, c], device=DEV)))
        amp[pos[p0:p1] - a] = pack.plug_val[p0:p1].double()
        for m, lut in enumerate((cos, sin)):
            w = torch.zeros(b - a, dtype=torch.float64, device=DEV)
            w[:c - a] = amp * lut[v & 1023]
            if b > c and m < len(pack.tails):
                tail = pack.tails[m][c - pack.n_codes:b - pack.n_codes].double()
                w[c - a:c - a + tail.numel()] = tail
            outs[m].append(xd @ w.view(hi - lo, K).t())
    return [torch.cat(o, 1) for o in outs]


def exact(case, seed):
    state = prepare(case, seed)
    kind = state["kind"]
    if kind.endswith("pack"):
        return _pack_f64(kind, state["ws"])
    if kind.endswith("stream"):
        st = state["stream"]
        xs = state["xs"]
        luts = _header_quad_luts(st.pack.r_max) if kind == "quad_stream" else _header_dual_luts()
        linear = _quad_linear_f64 if kind == "quad_stream" else _dual_linear_f64
        outs, pos = [], 0
        for (N, K), x in zip(st.shapes, xs):
            outs.append(linear(st.pack, luts, pos, N, K, x))
            pos += N * K
        return [torch.cat(o, 1) for o in zip(*outs)]
    if kind == "quad_rows":
        pack = state["layer"].pack
        return tuple(_quad_linear_f64(pack, _header_quad_luts(pack.r_max), 0, case["N"], case["K"], state["x"]))
    if kind == "dual_rows":
        return tuple(_dual_linear_f64(state["layer"].pack, _header_dual_luts(), 0, case["N"], case["K"], state["x"]))
    xd = state["x"].double()
    luts = [t.double() for t in state["luts"]]
    if kind == "quad_kn":
        w = _quad_rows_f64(state["codes"].view(torch.int32), luts)
        return [xd @ (w[m] * state["scales"][m]) for m in range(4)]
    v = state["codes"].int() + 32768
    n = torch.arange(v.numel(), device=DEV).view(v.shape)
    amp = luts[0][v >> 10] * state["scales"].double()[n // GROUP]
    return tuple(xd @ (amp * lut[v & 1023]) for lut in luts[1:])


def _pack_f64(kind, ws):
    """The packers' tables and scales in 64 bits.  The codes are rounded to the nearest step
    of 32-bit (quad) or 16-bit (dual) values, so they have no 64-bit counterpart."""
    if kind == "quad_pack":
        scales = [float(w.double().square().mean().sqrt()) for w in ws]
        r = sum((w.double() / s).square() for w, s in zip(ws, scales)).sqrt()
        return None, _header_quad_luts(float(r.max()) * 1.001), scales
    return (None, None, *_header_dual_luts())
