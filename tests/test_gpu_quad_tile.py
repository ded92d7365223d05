"""The tile kernel of (N,K) quad rows (pp_quad_tile, 1-32 tokens) against the float32-decoded,
fp16-rounded operands of the oracle: partial tiles, one tile and several a workgroup, runs that
start and end inside a tile, fewer steps than wavefronts, several slices of K, projections
mid-stream, plug tables from none to dense, and both table layouts."""
import numpy as np
import pytest
import torch

from oracle import layer as olay
from parity import assert_gemv_close, normwise
from polar_pack_amd import _native as nat
from polar_pack_amd import quad_kernels as qk
from test_gpu_big import fp16_luts, random_codes, u32
from test_gpu_mfma import DEV, check, oracle, packed

pytestmark = pytest.mark.gpu

# N, K: one row and one step; ragged rows; one step a wavefront; three slices; two tiles a workgroup
# (with a part of a group left); one tile of many steps
SHAPES = [(1, 32), (20, 96), (100, 1024), (256, 2048), (6000, 256), (4097, 64), (16, 11008)]


@pytest.mark.parametrize("M", [5, 16, 17, 32])
@pytest.mark.parametrize("N,K", SHAPES)
def test_matches_oracle(N, K, M):
    qp, pack = packed([(3, 40), (N, K), (2, 36)], 7, threshold=0.015)
    pos = 120
    assert nat.lib().pp_quad_tile_ok(K, K, int(pack.plug_idx.numel()), M, N, K)
    x = np.random.default_rng(N + M).standard_normal((M, K)).astype(np.float16)
    codes = pack.codes[pos:pos + N * K].reshape(N, K).t()
    luts = [t.to(DEV) for t in qk.header_luts(qp.r_max)]
    got = qk.quad_bitpacked(torch.from_numpy(x).to(DEV), codes, luts, list(qp.s), plug=(pack.plug_idx, pack.plug_vals),
                            elem_base=pos)
    check(got, oracle(qp, pos, N, K, x), f"{N}x{K} M={M}")


@pytest.mark.parametrize("M", [5, 16, 32])
@pytest.mark.parametrize("N,K", [(680, 2816), (1500, 4096)])
def test_several_slices_of_several_tiles(N, K, M):
    """Two and three tiles a workgroup, each in slices of K."""
    qp, pack = packed([(3, 40), (N, K), (2, 36)], 7, threshold=0.015)
    pos, tiles = 120, -(-N // 16)
    slices = nat.lib().pp_quad_tile_workspace_size(M, N, K) // (16 * M * 16 * tiles)
    assert slices > 1 and tiles > torch.cuda.get_device_properties(DEV).multi_processor_count // slices
    x = np.random.default_rng(N + M).standard_normal((M, K)).astype(np.float16)
    codes = pack.codes[pos:pos + N * K].reshape(N, K).t()
    luts = [t.to(DEV) for t in qk.header_luts(qp.r_max)]
    got = qk.quad_bitpacked(torch.from_numpy(x).to(DEV), codes, luts, list(qp.s), plug=(pack.plug_idx, pack.plug_vals),
                            elem_base=pos)
    check(got, oracle(qp, pos, N, K, x), f"{N}x{K} M={M}")


@pytest.mark.parametrize("M", [5, 17, 32])
def test_rows_past_eight_tiles_a_cu(M):
    """A head's row count stays on pp_quad_mfma (search, atomics, finish)."""
    N, K = 16 * 8 * torch.cuda.get_device_properties(DEV).multi_processor_count + 21, 64
    qp, pack = packed([(3, 40), (N, K), (2, 36)], 7, threshold=0.015)
    pos = 120
    assert not nat.lib().pp_quad_tile_ok(K, K, int(pack.plug_idx.numel()), M, N, K)
    codes = pack.codes[pos:pos + N * K].reshape(N, K).t()
    assert qk.quad_call_route(codes, M, 1) == "mfma"
    x = np.random.default_rng(N + M).standard_normal((M, K)).astype(np.float16)
    got = qk.quad_bitpacked(torch.from_numpy(x).to(DEV), codes, [t.to(DEV) for t in qk.header_luts(qp.r_max)],
                            list(qp.s), plug=(pack.plug_idx, pack.plug_vals), elem_base=pos)
    check(got, oracle(qp, pos, N, K, x), f"{N}x{K} M={M}")


@pytest.mark.parametrize("M,share", [(8, 0.0), (16, 0.3), (32, 0.3)])
@pytest.mark.parametrize("split", [False, True])
def test_dense_plugs_strided_rows_and_workspace(M, share, split):
    """Rows wider than K, windows refilled in every step, fp16 tables of either layout, any
    workspace contents, and outputs with rows wider than N."""
    N, K, ldc = 72, 4096, 4104
    wide = random_codes((N, ldc), M)
    luts, scales = fp16_luts(M, split=split)
    rng = np.random.default_rng(M)
    x = rng.standard_normal((M, K)).astype(np.float16)
    pos = np.flatnonzero(rng.random(N * ldc) < share)
    vals = rng.standard_normal((pos.size, 4)).astype(np.float16)
    L = nat.lib()
    dc, dx, dl = u32(wide).to(DEV), torch.from_numpy(x).to(DEV), [t.to(DEV) for t in luts]
    di, dv = torch.from_numpy(pos.astype(np.int32) + 11).to(DEV), torch.from_numpy(vals).to(DEV)
    n_ws = L.pp_quad_tile_workspace_size(M, N, K)
    assert n_ws > 0
    ws = torch.full((n_ws // 4,), float("nan"), device=DEV)
    outs = [torch.full((M, N + 8), 7.0, dtype=torch.float16, device=DEV) for _ in range(4)]
    ptrs, dt = qk._lut_args(dl)
    rc = L.pp_quad_tile(dc.data_ptr(), ldc, 11, dx.data_ptr(), K, ptrs, dt, nat.float_array(scales),
                        di.data_ptr() if pos.size else None, dv.data_ptr() if pos.size else None, pos.size,
                        nat.ptr_array([o.data_ptr() for o in outs]), N + 8, M, N, K, ws.data_ptr(), n_ws,
                        nat.raw_stream(DEV))
    nat.check(rc, "pp_quad_tile")
    torch.cuda.synchronize()
    # the plain decode of every tuple, then the plug values in their places
    wn = olay.quad_dequant(wide[:, :K], [t.numpy() for t in luts], dtype=np.float32)
    r, c = pos // ldc, pos % ldc
    keep = c < K
    for m in range(4):
        h = wn[m].astype(np.float16)
        h[r[keep], c[keep]] = vals[keep, m]
        w = h.astype(np.float64) * float(np.float32(scales[m]))
        xd = x.astype(np.float64)
        g = outs[m].float().cpu().numpy()
        assert_gemv_close(g[:, :N], xd @ w.T, f"model {m}", bound=2.0 ** -18 * (np.abs(xd) @ np.abs(w).T))
        assert normwise(g[:, :N], xd @ w.T) <= 1e-3
        assert (g[:, N:] == 7.0).all()


def test_refused_operands():
    ok = nat.lib().pp_quad_tile_ok
    assert ok(2048, 2048, 10, 16, 11008, 2048)
    for args in ((2048, 2048, 10, 33, 64, 2048), (2040, 2048, 10, 16, 64, 2048), (2050, 2048, 10, 16, 64, 2048),
                 (2064, 2064, 10, 16, 64, 2064), (2048, 2044, 10, 16, 64, 2048), (64, 64, 1 << 28, 16, 64, 64),
                 (64, 64, 0, 16, 16 * 8 * 256 + 1, 64)):
        assert not ok(*args), args
