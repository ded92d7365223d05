"""The container-row decode of 1-4 tokens (dual_rows_kernel) against float64 sums over the
oracle's group rule: rows shorter than a lane's 8 pairs up to several 512-pair chunks, ragged row
groups, every split of K over a workgroup's waves and more than one round of tasks, padded rows,
groups restarting inside a row, and plug tables from empty to several windows a task."""
import numpy as np
import pytest
import torch

from oracle import dualpack as odp
from parity import assert_gemv_close
from polar_pack_amd import polar_kernels as pk

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")

# N, K, padding of a row, group size, chunk size, first position, share of plug entries
CASES = [(1, 8, 0, 32, 50_000_000, 0, 0.5), (7, 8, 8, 8, 24, 16, 0.0), (5, 504, 0, 32, 1000, 800, 0.3),
         (33, 520, 8, 16, 50_000_000, 4096, 0.02), (250, 2056, 0, 32, 5000, 2504, 0.01),
         (1531, 4104, 0, 32, 50_000_000, 0, 0.01), (300, 4680, 24, 64, 1 << 40, 1 << 20, 0.001),
         (2050, 1032, 0, 32, 8, 0, 0.0), (20_000, 72, 0, 32, 100_000, 8, 0.05)]


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


@pytest.mark.parametrize("layout", ["u16be", "i16"])
@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,K,pad,gs,chunk,base,share", CASES)
def test_container_rows(N, K, pad, gs, chunk, base, share, M, layout):
    rng = np.random.default_rng(N + K + M)
    ld, dtype = K + pad, torch.float32 if M % 2 else torch.float16
    codes = rng.integers(0, 1 << 16, (N, ld), dtype=np.uint16)
    pos = base + np.arange(N)[:, None] * ld + np.arange(K)[None]
    g = odp.group_index(pos, chunk, gs)
    scales = (0.01 + rng.random(int(g.max()) + 1)).astype(np.float16)
    luts = [t.to(dtype) for t in pk.header_luts(device=DEV)]
    amp_lut, cos, sin = (t.double().cpu().numpy() for t in luts)
    amp = amp_lut[codes[:, :K] >> 10] * scales[g].astype(np.float64)
    plug = None
    if share:
        # table entries also before, between (padding) and past the rows
        at = np.flatnonzero(rng.random(N * ld + 64) < share)
        vals = rng.random(at.size).astype(np.float16)
        row, k = at // ld, at % ld
        ok = (row < N) & (k < K)
        amp[row[ok], k[ok]] = vals[ok]
        at = np.concatenate([np.arange(0, min(base, 8)), at + base])
        vals = np.concatenate([np.full(at.size - vals.size, 9, np.float16), vals])
        plug = (dev(at.astype(np.uint32).view(np.int32)).view(torch.uint32), dev(vals))
    stored = codes.byteswap() if layout == "u16be" else codes ^ np.uint16(0x8000)
    view = dev(stored.view(np.int16))[:, :K].t()
    x = rng.standard_normal((M, K)).astype(np.float16)
    assert pk.dual_call_route(view, M, layout=layout, group_size=gs, chunk_size=chunk, elem_base=base,
                              plug_n=int(bool(plug)), fused=False) == "dual_rows"
    got = pk.polar_dual_bitpacked(dev(x), view, dev(scales), *luts, group_size=gs, plug=plug, elem_base=base,
                                  layout=layout, chunk_size=chunk, fused=False)
    for o, lut in zip(got, (cos, sin)):
        w = amp * lut[codes[:, :K] & 1023]
        # float32 weights and sums: a few ulps of the terms' sum beside the fp16 rounding
        bound = 2.0 ** -21 * (np.abs(x).astype(np.float64) @ np.abs(w).T)
        assert_gemv_close(o.float().cpu().numpy(), x.astype(np.float64) @ w.T, bound=bound)


@pytest.mark.parametrize("layout", ["u16be", "i16"])
@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,K,chunk,base", [(11, 1032, 50_000_000, 0), (3, 8, 1000, 80), (5, 4104, 1 << 27, 1 << 20)])
def test_rows_far_apart(N, K, chunk, base, M, layout):
    """Rows 2^26 + 8 pairs apart, past the 32-bit offsets of a task: a base a row.  Groups that restart
    between rows, every chunk inside them, and never; ragged tasks; entries in, between and past rows."""
    rng = np.random.default_rng(N + K + M)
    ld = (1 << 26) + 8
    codes = rng.integers(0, 1 << 16, (N, K), dtype=np.uint16)
    pos = base + np.arange(N, dtype=np.int64)[:, None] * ld + np.arange(K)[None]
    g = odp.group_index(pos, chunk, 32)
    scales = (0.01 + rng.random(int(g.max()) + 1)).astype(np.float16)
    luts = pk.header_luts(device=DEV)
    amp_lut, cos, sin = (t.double().cpu().numpy() for t in luts)
    amp = amp_lut[codes >> 10] * scales[g].astype(np.float64)
    row, k = np.nonzero(rng.random((N, K)) < 0.05)
    vals = rng.random(row.size).astype(np.float16)
    amp[row, k] = vals
    past = np.arange(N, dtype=np.int64) * ld + K + 5
    at = np.concatenate([pos[row, k], past + base])
    order = np.argsort(at)
    vals = np.concatenate([vals, np.full(N, 9, np.float16)])[order]
    plug = (dev(at[order].astype(np.uint32).view(np.int32)).view(torch.uint32), dev(vals))
    stored = codes.byteswap() if layout == "u16be" else codes ^ np.uint16(0x8000)
    store = torch.zeros((N - 1) * ld + K, dtype=torch.int16, device=DEV)
    rows = store.as_strided((N, K), (ld, 1))
    rows.copy_(dev(stored.view(np.int16)))
    x = rng.standard_normal((M, K)).astype(np.float16)
    view = rows.t()
    assert pk.dual_call_route(view, M, layout=layout, chunk_size=chunk, elem_base=base, plug_n=1) == "dual_rows"
    got = pk.polar_dual_bitpacked(dev(x), view, dev(scales), *luts, plug=plug, elem_base=base, layout=layout,
                                  chunk_size=chunk)
    for o, lut in zip(got, (cos, sin)):
        w = amp * lut[codes & 1023]
        bound = 2.0 ** -21 * (np.abs(x).astype(np.float64) @ np.abs(w).T)
        assert_gemv_close(o.float().cpu().numpy(), x.astype(np.float64) @ w.T, bound=bound)
