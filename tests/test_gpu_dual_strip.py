"""The strip kernel of int16 (K,N) dual codes (pp_dual_strip, 1-32 tokens) against the oracle's
float32-decoded, fp16-rounded operands: one partial strip, a part of a second one, more strips than
CUs, fewer steps than wavefronts, several slices of K, groups of 4 to a whole row, fp16 and float32
tables shorter than the codes allow, and rows wider than the codes."""
import numpy as np
import pytest
import torch

from polar_pack_amd import _native as nat
from polar_pack_amd import polar_kernels as pk
from test_gpu_dual_mfma import DEV, check, layer, to_dev

pytestmark = pytest.mark.gpu

SHAPES = [(32, 8, 8), (96, 72, 8), (2080, 192, 64), (64, 16_448, 32), (8192, 256, 256), (4096, 520, 8)]


@pytest.mark.parametrize("M", [2, 16, 17, 32])
@pytest.mark.parametrize("K,N,gs", SHAPES)
def test_matches_oracle(K, N, gs, M):
    arrs = layer(K, N, K + N + M, gs)
    a = np.random.default_rng(N + M).standard_normal((M, K)).astype(np.float16)
    da, dp, *rest = to_dev(a, *arrs)
    assert nat.lib().pp_dual_strip_ok(dp.data_ptr(), N, da.data_ptr(), K, gs, M, N, K)
    outs = pk.polar_dual_bitpacked(da, dp, *rest, group_size=gs, fused=True)
    check(outs, a, *arrs, gs, what=f"K={K} N={N} M={M}")


@pytest.mark.parametrize("M", [1, 2, 16, 17, 32])
@pytest.mark.parametrize("K,N,gs", [(32, 8, 8), (96, 72, 8), (2080, 192, 64), (64, 16_448, 32), (4128, 256, 256)])
def test_entries_no_code_names_do_not_matter(K, N, gs, M):
    """The entries that a stored 0 names infinite or NaN (amplitude 32, phase 0), no code naming them:
    rows that a wave's walk has no more of are left out, never decoded as zeros."""
    packed, bmax, *luts = layer(K, N, K + N + M, gs)
    code = packed.view(np.uint16) ^ np.uint16(0x8000)
    code = np.where(code >> 10 == 32, code ^ np.uint16(1 << 10), code) | np.uint16(1)
    packed = (code ^ np.uint16(0x8000)).astype(np.uint16).view(np.int16)
    a = np.random.default_rng(N + M).standard_normal((M, K)).astype(np.float16)
    da, dp, db, amp, cos, sin = to_dev(a, packed, bmax, *luts)
    want = pk.polar_dual_bitpacked(da, dp, db, amp, cos, sin, group_size=gs, fused=True)
    for bad in (float("inf"), float("nan")):
        amp[32] = cos[0] = sin[0] = bad
        got = pk.polar_dual_bitpacked(da, dp, db, amp, cos, sin, group_size=gs, fused=True)
        for o, w in zip(got, want):
            assert bool(w.isfinite().all()) and torch.equal(o, w), bad


@pytest.mark.parametrize("M", [1, 7, 20])
def test_c_abi_strided_rows_and_workspace(M):
    """4-pair groups, float32 tables, rows of codes and outputs wider than N, any workspace."""
    K, N, gs, ldk, o_sm = 4096, 100, 4, 108, 104
    packed, bmax, *luts = layer(K, N, M, gs)
    a = np.random.default_rng(M).standard_normal((M, K)).astype(np.float16)
    wide = np.full((K, ldk), -1, np.int16)
    wide[:, :N] = packed
    L = nat.lib()
    da, dp, db = to_dev(a, wide, bmax)
    dl = [t.float() for t in to_dev(*luts)]
    n_ws = L.pp_dual_strip_workspace_size(M, N, K)
    assert n_ws > 0
    ws = torch.full((n_ws // 4,), float("nan"), device=DEV)
    outs = [torch.full((M, o_sm), 7.0, dtype=torch.float16, device=DEV) for _ in range(2)]
    for _ in range(2):
        nat.check(L.pp_dual_strip(dp.data_ptr(), ldk, da.data_ptr(), K, db.data_ptr(), gs, dl[0].data_ptr(),
                                  dl[0].numel(), dl[1].data_ptr(), dl[2].data_ptr(), dl[1].numel(), nat.PP_F32,
                                  outs[0].data_ptr(), outs[1].data_ptr(), o_sm, M, N, K, ws.data_ptr(), n_ws,
                                  nat.raw_stream(DEV)), "pp_dual_strip")
        torch.cuda.synchronize()
        check([o[:, :N] for o in outs], a, packed, bmax, *luts, gs, what=f"M={M}")
        assert all(bool((o[:, N:] == 7.0).all()) for o in outs)


def test_refused_operands():
    ok = nat.lib().pp_dual_strip_ok
    assert ok(0, 4096, 0, 4096, 32, 32, 4096, 4096)
    for args in ((0, 4096, 0, 4096, 32, 33, 4096, 4096), (4, 4096, 0, 4096, 32, 8, 4096, 4096),
                 (0, 4098, 0, 4096, 32, 8, 4096, 4096), (0, 4096, 0, 4096, 32, 8, 4080, 4096),
                 (0, 4096, 0, 4080, 32, 8, 4096, 4080), (0, 4096, 0, 4092, 32, 8, 4096, 4096),
                 (0, 64, 8, 64, 32, 8, 64, 64), (0, 64, 0, 64, 2, 8, 64, 64), (0, 64, 0, 64, 48, 8, 48, 64)):
        assert not ok(*args), args
