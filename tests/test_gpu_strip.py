"""The strip kernels of (K,N) quad codes (pp_quad_strip, 1-32 tokens, fp16 tables) against float64
products: partial strips and row units, one and several slices of K, more than one round of items,
rows wider than the codes, tokens around a tile, tables whose q1 and q2 differ, and the counts left
zero."""
import numpy as np
import pytest
import torch

from parity import assert_gemv_close, normwise
from polar_pack_amd import _native as nat
from polar_pack_amd import quad_kernels as qk
from refs import check_mfma, kn_mfma_reference
from test_gpu_big import fp16_luts, random_codes, u32

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")

# K, N, row stride: below a strip, ragged, one slice of many rounds (20,000 columns), many slices
SHAPES = [(32, 4, 4), (256, 36, 40), (96, 300, 520), (2080, 1000, 1000), (64, 20_000, 20_000), (8192, 256, 256)]


def check(got, exact, what):
    """Against the exact decode.  A weight's rounding to fp16 moves it by at most 2^-11 of itself, so
    over random signs an output moves by a standard deviation of at most 2^-11 / sqrt(3) of the
    outputs' root mean square (that of sqrt(K) random terms): held to 8 of them."""
    for m in range(4):
        g = got[m].float().cpu().numpy()
        rms = np.sqrt((exact[m] ** 2).mean(axis=1, keepdims=True))       # ~ sqrt(K) x the rms term
        assert_gemv_close(g, exact[m], f"{what} model {m}", bound=8 * 2.0 ** -11 / np.sqrt(3) * rms)
        assert normwise(g, exact[m]) <= 1e-3, f"{what} model {m}"


@pytest.mark.parametrize("K,N,ldk", SHAPES + [(40, 68, 68), (4104, 132, 136)])
def test_one_token(K, N, ldk):
    wide = random_codes((K, ldk), K + N)
    luts, scales = fp16_luts(K + N, split=N % 8 == 0)
    a = np.random.default_rng(N).standard_normal((1, K)).astype(np.float16)
    view = u32(wide).to(DEV)[:, :N]
    dl = [t.to(DEV) for t in luts]
    assert nat.lib().pp_quad_strip_ok(view.data_ptr(), ldk, 0, K, nat.PP_F16, 1, N, K)
    assert qk.quad_call_route(view, 1) == "kn"
    exact = kn_mfma_reference(a, wide[:, :N], luts, scales)[0]
    for rep in range(2):
        got = qk.quad_bitpacked(torch.from_numpy(a).to(DEV), view, dl, scales)
        torch.cuda.synchronize()
        for m in range(4):                    # float32 weights: no fp16 rounding allowed for
            assert_gemv_close(got[m].float().cpu().numpy(), exact[m], f"model {m} call {rep}", rtol=5.1e-4)


@pytest.mark.parametrize("M", [2, 15, 16, 17, 32])
@pytest.mark.parametrize("K,N,ldk", SHAPES)
def test_matrix_core_tokens(K, N, ldk, M):
    wide = random_codes((K, ldk), K + N + M)
    luts, scales = fp16_luts(K + M, split=M % 2 == 0)
    a = np.random.default_rng(N + M).standard_normal((M, K)).astype(np.float16)
    view = u32(wide).to(DEV)[:, :N]
    assert nat.lib().pp_quad_strip_ok(view.data_ptr(), ldk, 0, K, nat.PP_F16, M, N, K)
    got = qk.quad_bitpacked(torch.from_numpy(a).to(DEV), view, [t.to(DEV) for t in luts], scales, fused=True)
    check(got, kn_mfma_reference(a, wide[:, :N], luts, scales)[0], f"M={M}")


@pytest.mark.parametrize("M", [1, 2, 16, 17, 32])
@pytest.mark.parametrize("K,N", [(32, 8), (96, 300), (2080, 1000), (4128, 132), (64, 20_000)])
def test_entries_no_code_names_do_not_matter(K, N, M):
    """First table entries that are infinite or NaN, with no code 0 among the words: rows that a wave's
    walk has no more of are left out, never decoded as zeros."""
    words = random_codes((K, N), K + N + M) | np.uint32(0x01010101)
    luts, scales = fp16_luts(K + M, split=M % 2 == 0)
    a = torch.randn(M, K, device=DEV).half()
    codes, dl = u32(words).to(DEV), [t.to(DEV) for t in luts]
    want = qk.quad_bitpacked(a, codes, dl, scales, fused=True if M > 1 else None)
    for bad in (float("inf"), float("nan")):
        for t in dl:
            t[0] = bad
        got = qk.quad_bitpacked(a, codes, dl, scales, fused=True if M > 1 else None)
        for m in range(4):
            assert bool(want[m].isfinite().all()) and torch.equal(got[m], want[m]), (bad, m)


@pytest.mark.parametrize("M,K,N", [(1, 2112, 8308), (16, 3648, 8308), (32, 5952, 4148)])
def test_several_slices_and_rounds(M, K, N):
    """More items of strips x slices than CUs: a workgroup's second item after a slice that was not its
    strip's last, the buffers and the count's flag used again.  64 columns and the ragged last strip."""
    cols = np.unique(np.concatenate([np.random.default_rng(M).choice(N, 48, replace=False), np.arange(N - 16, N)]))
    words = random_codes((K, N), K + N + M)
    luts, scales = fp16_luts(K + M)
    a = np.random.default_rng(N + M).standard_normal((M, K)).astype(np.float16)
    width, cus = 32 if M > 16 else 64, torch.cuda.get_device_properties(DEV).multi_processor_count
    strips = -(-N // width)
    slices, rest = divmod(nat.lib().pp_quad_strip_workspace_size(M, N, K), 16 * M * strips * width)
    assert slices > 1 and rest == 0 and strips * slices > cus
    da, dc, dl = torch.from_numpy(a).to(DEV), u32(words).to(DEV), [t.to(DEV) for t in luts]
    exact = kn_mfma_reference(a, words, luts, scales, cols=cols)[0]
    first = None
    for rep in range(3):
        got = qk.quad_bitpacked(da, dc, dl, scales, fused=True if M > 1 else None)
        torch.cuda.synchronize()
        first = first or got
        assert all(torch.equal(g, f) for g, f in zip(got, first)), rep
    check([g[:, torch.from_numpy(cols).to(DEV)] for g in first], exact, f"M={M}")


@pytest.mark.parametrize("K,N,strip", [(4096, 6396, True), (4096, 6400, False), (8192, 8192, False)])
def test_one_token_of_a_large_layer(K, N, strip):
    """From 25 Mi words on one token takes the row kernel, which is the faster one there; other tokens
    and the outputs do not depend on it (float32 weights and sums either way)."""
    ok = nat.lib().pp_quad_strip_ok
    assert bool(ok(0, N, 0, K, nat.PP_F16, 1, N, K)) == strip and ok(0, N, 0, K, nat.PP_F16, 16, N, K)
    if N > 6400:
        return
    g = torch.Generator(device=DEV).manual_seed(N)
    words = torch.randint(-2 ** 31, 2 ** 31 - 1, (K, N), generator=g, device=DEV, dtype=torch.int64).int()
    luts, scales = fp16_luts(N)
    a = np.random.default_rng(N).standard_normal((1, K)).astype(np.float16)
    got = qk.quad_bitpacked(torch.from_numpy(a).to(DEV), words.view(torch.uint32), [t.to(DEV) for t in luts], scales)
    exact = kn_mfma_reference(a, words[:, ::101].cpu().numpy().view(np.uint32), luts, scales)[0]
    for m in range(4):
        assert_gemv_close(got[m][:, ::101].float().cpu().numpy(), exact[m], f"model {m}", rtol=5.1e-4)


@pytest.mark.parametrize("M", [1, 2, 16, 17, 32])
@pytest.mark.parametrize("K,N", [(256, 72), (2080, 1000)])
def test_float32_tables_keep_the_other_kernels(K, N, M):
    """Tables that fp16 does not hold: quad_kn_kernel at one token, quad_big_kernel above."""
    words = random_codes((K, N), K + N + M)
    luts, scales = fp16_luts(K + M, split=M % 2 == 0)
    luts = [t.float() * (1 + 2.0 ** -14) for t in luts]
    a = np.random.default_rng(N + M).standard_normal((M, K)).astype(np.float16)
    codes = u32(words).to(DEV)
    assert not nat.lib().pp_quad_strip_ok(codes.data_ptr(), N, 0, K, nat.PP_F32, M, N, K)
    got = qk.quad_bitpacked(torch.from_numpy(a).to(DEV), codes, [t.to(DEV) for t in luts], scales,
                            fused=True if M > 1 else None)
    ref = kn_mfma_reference(a, words, luts, scales)
    if M > 1:
        check_mfma(got, ref, f"M={M}")
        return
    for m in range(4):
        assert_gemv_close(got[m].float().cpu().numpy(), ref[0][m], f"model {m}", rtol=5.1e-4)


@pytest.mark.parametrize("M", [1, 5, 20])
def test_c_abi_workspace_and_strided_outputs(M):
    """Any workspace contents, counts zero before and after, outputs with a column stride, and the
    columns between left alone."""
    K, N = 4096, 200
    codes = random_codes((K, N), 9)
    luts, scales = fp16_luts(9)
    a = np.random.default_rng(M).standard_normal((M, K)).astype(np.float16)
    L = nat.lib()
    dc, da, dl = u32(codes).to(DEV), torch.from_numpy(a).to(DEV), [t.to(DEV) for t in luts]
    ptrs, dt = qk._lut_args(dl)
    n_ws, n_counts = L.pp_quad_strip_workspace_size(M, N, K), L.pp_quad_strip_counts(M, N, K)
    assert n_ws > 0 and (n_counts > 0) == (M == 1)
    ws = torch.full((n_ws // 4,), float("nan"), device=DEV)
    counts = torch.zeros(max(n_counts // 4, 1), dtype=torch.int32, device=DEV)
    wide = [torch.full((M, 2 * N), 7.0, dtype=torch.float16, device=DEV) for _ in range(4)]
    ref = kn_mfma_reference(a, codes, luts, scales)[0]
    for rep in range(2):
        rc = L.pp_quad_strip(dc.data_ptr(), N, da.data_ptr(), K, ptrs, dt, nat.float_array(scales),
                             nat.ptr_array([w.data_ptr() for w in wide]), 2 * N, 2, M, N, K, ws.data_ptr(), n_ws,
                             counts.data_ptr(), n_counts, torch.cuda.current_stream(DEV).cuda_stream)
        nat.check(rc, "pp_quad_strip")
        torch.cuda.synchronize()
        assert int(torch.count_nonzero(counts)) == 0
        check([w[:, ::2] for w in wide], ref, f"call {rep}")
        assert all(bool((w[:, 1::2] == 7.0).all()) for w in wide)
    rc = L.pp_quad_strip(dc.data_ptr(), N, da.data_ptr(), K, ptrs, dt, nat.float_array(scales),
                         nat.ptr_array([w.data_ptr() for w in wide]), 2 * N, 2, M, N, K, ws.data_ptr(), n_ws - 4,
                         counts.data_ptr(), n_counts, torch.cuda.current_stream(DEV).cuda_stream)
    assert rc == nat.PP_EINVAL


def test_replayed_graph():
    """A captured call replayed beside eager calls gives the eager outputs each time."""
    K, N = 4096, 512
    codes = u32(random_codes((K, N), 1)).to(DEV)
    luts, scales = fp16_luts(1)
    luts = [t.to(DEV) for t in luts]
    for M in (1, 16):
        a = torch.randn(M, K, device=DEV).half()
        want = qk.quad_bitpacked(a, codes, luts, scales)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            got = qk.quad_bitpacked(a, codes, luts, scales)
        for rep in range(4):
            for t in got:
                t.fill_(float("nan"))
            g.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(x, y) for x, y in zip(got, want)), (M, rep)
            again = qk.quad_bitpacked(a, codes, luts, scales)
            assert all(torch.equal(x, y) for x, y in zip(again, want))
