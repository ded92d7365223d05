"""The layer packers' device passes (pack.hip) against the tensor expressions they replace, which
still pack host tensors and whatever the kernels do not read: every code, scale and LUT entry bit
for bit, at sizes around the threads' 4- and 8-element runs and a wavefront's 512 pairs, for heavy
tails, zeros, subnormals, infinities and NaN."""
import pytest
import torch

from polar_pack_amd import _native as nat
from polar_pack_amd import polar_kernels as pk
from polar_pack_amd import quad_kernels as qk

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def weights(count, shape, dtype, kind, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    base = torch.randn(shape, generator=g, device=DEV)
    if kind == "heavy":
        base = base / torch.rand(shape, generator=g, device=DEV).clamp_min(1e-3)
    ws = []
    for m in range(count):
        w = (0.02 * (base + 0.1 * (m + 1) * torch.randn(shape, generator=g, device=DEV))).to(dtype)
        if kind == "zeros":
            w[torch.rand(shape, generator=g, device=DEV) < 0.5] = 0
        elif kind == "axes":                          # one model zero, another negative: angles 0 and pi
            w = torch.zeros_like(w) if m == count - 1 else -w.abs() if m == 0 else w
        elif kind == "tiny":
            w = (w.float() * 1e-5).to(dtype)          # fp16 subnormals
        elif kind in ("inf", "nan"):
            w.view(-1)[m::97] = float(kind)
        ws.append(w)
    return ws


def tensors(result):
    return [t for r in result for t in (r if isinstance(r, list) else [r])]


def assert_same(got, want):
    got, want = tensors(got), tensors(want)
    assert len(got) == len(want)
    for i, (a, b) in enumerate(zip(got, want)):
        if isinstance(a, float):
            assert a == b or (a != a and b != b), (i, a, b)
            continue
        assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride(), i
        if a.dtype.is_floating_point:                 # NaN payloads aside
            assert torch.equal(a.isnan(), b.isnan()), i
            a, b = a.nan_to_num(0.0), b.nan_to_num(0.0)
        bits = {2: torch.int16, 4: torch.int32}[a.element_size()]
        bad = (a.view(bits) != b.view(bits)).sum()
        assert int(bad) == 0, f"output {i}: {int(bad)} of {a.numel()} differ"


def both(monkeypatch, fn, *args, **kw):
    took = []
    monkeypatch.setattr(nat, "upload", lambda *a, _f=nat.upload: took.append(1) or _f(*a))
    got = fn(*args, **kw)
    assert took, "the device passes did not run"
    monkeypatch.setattr(nat, "packable", lambda ws: False)
    return got, fn(*args, **kw)


KINDS = ("normal", "heavy", "zeros", "axes", "tiny")
SHAPES = [(1, 1), (3, 5), (64, 96), (1000, 777), (2048, 4100)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("kind", KINDS + ("inf", "nan"))
@pytest.mark.parametrize("shape", SHAPES)
def test_quad_pack_is_the_tensor_expressions(monkeypatch, shape, kind, dtype):
    ws = weights(4, shape, dtype, kind, 3)
    got, want = both(monkeypatch, qk.pack_quad_layer, *ws)
    assert_same(got, want)


@pytest.mark.parametrize("shape", [(1, 1), (3, 5), (2, 8), (1000, 777)])
def test_quad_pack_of_weights_whose_squares_underflow(monkeypatch, shape):
    """float32 weights of ~1e-25: a scale of 0, so norms of infinity, which the reads past an element
    count that is no multiple of 4 must not turn into NaN."""
    ws = [w * 1e-23 for w in weights(4, shape, torch.float32, "normal", 7)]
    assert all(bool((w != 0).all()) and float((w.float() ** 2).mean()) == 0 for w in ws)
    got, want = both(monkeypatch, qk.pack_quad_layer, *ws)
    assert bool(want[1][0][1:].isinf().all())
    assert_same(got, want)


def test_quad_pack_keeps_a_transposed_layout(monkeypatch):
    ws = [w.t() for w in weights(4, (130, 64), torch.float16, "normal", 4)]
    got, want = both(monkeypatch, qk.pack_quad_layer, *ws)
    assert_same(got, want)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("kind", KINDS + ("inf", "nan"))
@pytest.mark.parametrize("shape,kw", [(s, {}) for s in SHAPES] + [
    ((100, 77), {"group_size": 8}), ((100, 77), {"group_size": 512}), ((7, 73), {"group_size": 64}),
    ((64, 96), {"amp_bits": 4, "num_phases": 256, "mu": 127.5}), ((64, 96), {"num_phases": 1000})])
def test_dual_pack_is_the_tensor_expressions(monkeypatch, shape, kw, kind, dtype):
    ws = weights(2, shape, dtype, kind, 5)
    got, want = both(monkeypatch, pk.quantize_polar_bitpacked, *ws, **kw)
    assert_same(got, want)


def test_what_the_kernels_do_not_read_keeps_the_expressions(monkeypatch):
    """Other types, strides, groups, gradients and transforms: same results, no kernel."""
    def refuse(*a):
        raise AssertionError("the device passes ran")
    monkeypatch.setattr(nat, "upload", refuse)
    w = weights(4, (64, 96), torch.float32, "normal", 6)
    a = qk.pack_quad_layer(*[x[:, ::2] for x in w])
    assert a[0].shape == (64, 48)
    qk.pack_quad_layer(*[x.double() for x in w])
    qk.pack_quad_layer(w[0], w[1].half(), w[2], w[3])
    pk.quantize_polar_bitpacked(w[0].t(), w[1].t())
    pk.quantize_polar_bitpacked(w[0], w[1], group_size=24)
    pk.quantize_polar_bitpacked(w[0].bfloat16(), w[1].bfloat16())
    r = pk.quantize_polar_bitpacked(w[0].clone().requires_grad_(), w[1])
    assert r[1].requires_grad
    one = pk.quantize_polar_bitpacked(w[0], w[1], group_size=24)
    many = torch.func.vmap(lambda x, y: pk.quantize_polar_bitpacked(x, y, group_size=32)[0])(
        torch.stack(w[:2]), torch.stack(w[2:]))
    assert many.shape == (2, *one[0].shape)


def test_a_function_mode_sees_the_expressions():
    class Seen(torch.overrides.TorchFunctionMode):
        def __init__(self):
            super().__init__()
            self.names = set()

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.names.add(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    w = weights(4, (64, 96), torch.float32, "normal", 8)
    for fn, ws in ((qk.pack_quad_layer, w), (pk.quantize_polar_bitpacked, w[:2])):
        with Seen() as mode:
            got = fn(*ws)
        assert {"atan2", "log1p", "round"} <= mode.names, fn
        assert_same(got, fn(*ws))


def test_luts_are_tensors_of_their_own():
    """As the expressions' are: no two share storage or a version, so one can be changed in place,
    saved or released by itself."""
    w = weights(4, (64, 96), torch.float16, "normal", 9)
    for luts in (qk.pack_quad_layer(*w)[1], pk.quantize_polar_bitpacked(*w[:2])[2:]):
        assert len({t.untyped_storage().data_ptr() for t in luts}) == len(luts)
        for t in luts:
            assert not t._is_view() and t.untyped_storage().nbytes() == t.numel() * t.element_size()
        luts[0].zero_()
        assert [t._version for t in luts[1:]] == [luts[1]._version] * (len(luts) - 1) != [luts[0]._version]


def test_every_call_builds_its_own_tables(monkeypatch):
    """Nothing of a packed layer is kept for the next call: the LUTs are computed in each."""
    w = weights(4, (64, 96), torch.float16, "normal", 10)
    for mod, name, fn, ws in ((qk, "_lut_tables", qk.pack_quad_layer, w),
                              (pk, "_layer_luts", pk.quantize_polar_bitpacked, w[:2])):
        calls = []
        monkeypatch.setattr(mod, name, lambda *a, _f=getattr(mod, name): calls.append(1) or _f(*a))
        for i in range(3):
            fn(*ws)
            assert len(calls) == i + 1, name


@pytest.mark.parametrize("sizes", [(1,), (896,), (897, 0, 5), (3, 2000, 1, 1), (1,) * 20, (0, 0)])
def test_upload_of_several_tables(sizes):
    """Tables that end inside, at and past a launch's 896 words, and more of them than its 8 parts."""
    g = torch.Generator().manual_seed(sum(sizes))
    hosts = [torch.randint(-2 ** 31, 2 ** 31 - 1, (n,), generator=g, dtype=torch.int32) for n in sizes]
    outs = [torch.empty(n, dtype=torch.int32, device=DEV) for n in sizes]
    nat.upload(outs, [h.data_ptr() for h in hosts])
    one = torch.zeros_like(outs[0])
    nat.check(nat.lib().pp_upload(one.data_ptr(), hosts[0].data_ptr(), 4 * sizes[0], nat.raw_stream(DEV)), "pp_upload")
    for got, want in zip([*outs, one], [*hosts, hosts[0]]):
        assert torch.equal(got.cpu(), want)
