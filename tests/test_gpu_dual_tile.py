"""The tile kernel of container (N,K) dual rows (pp_dual_tile, 1-32 tokens) against the float64
oracle: partial tiles, one tile and several a workgroup, runs that start and end inside a tile, fewer
steps than wavefronts, several slices of K, chunks that end inside rows, projections mid-stream,
plug tables from none to more entries than a wavefront's part of LDS holds, and both code layouts."""
import numpy as np
import pytest
import torch

from oracle import dualpack as odp
from polar_pack_amd import _native as nat
from polar_pack_amd import polar_kernels as pk
from test_gpu_dual import be_codes_tensor
from test_gpu_dual_nk import DEV, check, pack, run, u32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 5, 16, 17, 32])
@pytest.mark.parametrize("N,K,chunk,cap", [(1, 32, 4096, 0.0), (20, 96, 1000, 0.05), (256, 2048, 50_000_000, 0.01),
                                           (6000, 256, 4104, 0.01), (4097, 64, 32, 0.02), (16, 11008, 8000, 0.3)])
def test_matches_oracle(N, K, chunk, cap, M):
    pos = 56
    dp = pack(pos + N * K + 40, pos + N * K + 8, N + M, cap, chunk)
    assert nat.lib().pp_dual_tile_ok(K, pos, K, 32, chunk, int(dp.plug_idx.size), M, N, K)
    route, a, outs, ws = run(dp, pos, N, K, M, fused=True)
    assert route == "dual_nk_mfma"
    check(a, outs, ws, f"{N}x{K} M={M}")


@pytest.mark.parametrize("M", [2, 16, 32])
@pytest.mark.parametrize("N,K,chunk", [(680, 2816, 50_000_000), (1500, 4096, 9000)])
def test_several_slices_of_several_tiles(N, K, chunk, M):
    """Two and three tiles a workgroup, each in slices of K."""
    pos, tiles = 56, -(-N // 16)
    dp = pack(pos + N * K + 40, pos + N * K + 8, N, 0.01, chunk)
    slices = nat.lib().pp_dual_tile_workspace_size(M, N, K) // (8 * M * 16 * tiles)
    assert slices > 1 and tiles > torch.cuda.get_device_properties(DEV).multi_processor_count // slices
    route, a, outs, ws = run(dp, pos, N, K, M, fused=True)
    assert route == "dual_nk_mfma"
    check(a, outs, ws, f"{N}x{K} M={M}")


@pytest.mark.parametrize("M", [3, 17, 32])
def test_rows_past_eight_tiles_a_cu(M):
    """A head's row count stays on pp_dual_nk_mfma (search, atomics, finish)."""
    N, K, pos, chunk = 16 * 8 * torch.cuda.get_device_properties(DEV).multi_processor_count + 21, 64, 56, 4104
    dp = pack(pos + N * K + 40, pos + N * K + 8, N, 0.02, chunk)
    assert not nat.lib().pp_dual_tile_ok(K, pos, K, 32, chunk, int(dp.plug_idx.size), M, N, K)
    route, a, outs, ws = run(dp, pos, N, K, M, fused=True)
    assert route == "dual_nk_mfma"
    check(a, outs, ws, f"{N}x{K} M={M}")


@pytest.mark.parametrize("M", [3, 20])
def test_more_entries_than_lds_holds(M):
    N, K = 4100, 1024          # four steps of 16 x 32 pairs a wavefront, over half of them plugged
    dp = pack(N * K, N * K, 5, 0.6, 50_000_000)
    assert dp.plug_idx.size > 0.5 * N * K
    _, a, outs, ws = run(dp, 0, N, K, M, fused=True)
    check(a, outs, ws, f"M={M}")


@pytest.mark.parametrize("M", [2, 24])
def test_c_abi_layouts_strides_and_workspace(M):
    """Rows and outputs wider than K and N, the offset int16 layout, any workspace contents."""
    N, K, ldc, o_sm = 72, 4096, 4104, 76
    dp = pack(N * ldc, N * ldc, 9, 0.02, 50_000_000)
    wide = be_codes_tensor(dp)[:N * ldc]
    v = wide.view(torch.int16).int() & 0xFFFF
    code = ((v & 0xFF) << 8) | (v >> 8)
    offset = (code - 32768).short()
    L = nat.lib()
    n_ws = L.pp_dual_tile_workspace_size(M, N, K)
    assert n_ws > 0
    luts = pk.header_luts(mu=dp.mu, device=DEV)
    scales, idx, val = (torch.from_numpy(dp.scales).to(DEV), u32(dp.plug_idx).to(DEV),
                        torch.from_numpy(dp.plug_val).to(DEV))
    a = np.random.default_rng(M).standard_normal((M, K)).astype(np.float16)
    da = torch.from_numpy(a).to(DEV)
    ref = [w.reshape(N, ldc)[:, :K] for w in odp.decode_pairs_f64(dp, 0, N * ldc)]
    ws = torch.full((n_ws // 4,), float("nan"), device=DEV)
    for codes, lay in ((wide, nat.PP_DUAL_U16_BE), (offset, nat.PP_DUAL_I16_OFFSET)):
        outs = [torch.full((M, o_sm), 7.0, dtype=torch.float16, device=DEV) for _ in range(2)]
        nat.check(L.pp_dual_tile(codes.data_ptr(), lay, ldc, 0, da.data_ptr(), K, scales.data_ptr(), scales.numel(),
                                 dp.group_size, dp.chunk_size, luts[0].data_ptr(), luts[0].numel(),
                                 luts[1].data_ptr(), luts[2].data_ptr(), luts[1].numel(), nat.PP_F32, idx.data_ptr(),
                                 val.data_ptr(), idx.numel(), outs[0].data_ptr(), outs[1].data_ptr(), o_sm, M, N, K,
                                 ws.data_ptr(), n_ws, nat.raw_stream(DEV)), "pp_dual_tile")
        torch.cuda.synchronize()
        check(a, [o[:, :N] for o in outs], ref, f"layout {lay} M={M}")
        assert all(bool((o[:, N:] == 7.0).all()) for o in outs)


def test_refused_operands():
    ok = nat.lib().pp_dual_tile_ok
    assert ok(2048, 8, 2048, 32, 4096, 9, 16, 11008, 2048)
    for args in ((2048, 8, 2048, 32, 4096, 9, 33, 64, 2048), (2052, 8, 2048, 32, 4096, 9, 16, 64, 2048),
                 (2048, 4, 2048, 32, 4096, 9, 16, 64, 2048), (2048, 8, 2044, 32, 4096, 9, 16, 64, 2048),
                 (2048, 8, 2048, 4, 4096, 9, 16, 64, 2048), (2048, 8, 2048, 32, 24, 9, 16, 64, 2048),
                 (2064, 8, 2064, 32, 4096, 9, 16, 64, 2064), (64, 8, 64, 32, 4096, 1 << 29, 16, 64, 64),
                 (64, 8, 64, 32, 4096, 0, 16, 16 * 8 * 256 + 1, 64)):
        assert not ok(*args), args
