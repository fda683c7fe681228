"""quantized_matmul (QLinear::forward, qwen3_next.rs:174-221) on the GPU
against the oracle (the exact f64 contraction rounded once). A floating-point
contraction accumulated in f32, so the bar is the stated tolerance, written
here: every bf16/f16 output within 1 ulp of the oracle, or within atol 1e-3
next to zero (rtol 1e-2, atol 1e-3); at least 99 % bit-identical. bf16
with group 64 runs on the matrix cores from 16 rows on, and from 2 with K 512,
1024, 2048 or 4096; the rest on the GEMV kernels."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import higgs_amd as H
import oracle as O
from bits import assert_close, exact_frac
from gpu_util import to_dev, to_host, words_dev

pytestmark = pytest.mark.gpu


def _case(key, M, N, K, group=64, dt=O.BF16, xs=1.0):
    x = O.from_f32(O.normal(key, (M, K)) * np.float32(xs), dt)
    w = O.u32(key + 1, (N, K // 8))
    s = O.from_f32(O.uniform(key + 2, (N, K // group), 0.005, 0.02), dt)
    b = O.from_f32(O.uniform(key + 3, (N, K // group), -0.1, 0.1), dt)
    return x, w, s, b


def _run(dev, x, w, s, b, dt, group=64):
    y = H.quantized_matmul(to_dev(x, dt, dev), words_dev(w, dev), to_dev(s, dt, dev),
                           to_dev(b, dt, dev), True, group, 4)
    return to_host(y)


def _check(got, ref, dt, what):
    ef = exact_frac(got, ref, dt)
    print(f"[qgemm] {what}: exact={ef:.5f}", flush=True)
    assert_close(got, ref, dt, max_ulp=1, what=what)
    assert ef >= 0.99, what


@pytest.mark.parametrize("M,N,K", [(16, 256, 512), (64, 2048, 2048), (33, 640, 1536),
                                   (48, 200, 576), (64, 256, 4096), (100, 384, 1024),
                                   (512, 1024, 2048), (777, 1000, 512), (1024, 512, 4096)],
                         ids=["M16", "decode64", "odd-chunks", "K576", "skinny-K4096", "ragged-M",
                              "M512", "ragged-MN", "K4096"])
def test_mfma_path_matches_oracle(dev, M, N, K):
    x, w, s, b = _case(3000 + M + N, M, N, K)
    got = _run(dev, x, w, s, b, O.BF16)
    ref = O.quantized_matmul(x, O.BF16, w, s, b, O.BF16)
    _check(got, ref, O.BF16, f"M={M} N={N} K={K}")


@pytest.mark.parametrize("M,N", [(64, 12288), (40, 12288), (64, 12400)],
                         ids=["in_proj_qkvz", "rows40", "ragged-tiles"])
def test_decode_wide_projection(dev, M, N):
    """The decode step of a batch through in_proj_qkvz (2048 -> 12288), the
    launch geometry bench.py times, plus a partly filled second row half and
    a column count that leaves the last column tile ragged."""
    K = 2048
    x, w, s, b = _case(3701 + M + N, M, N, K)
    got = _run(dev, x, w, s, b, O.BF16)
    ref = O.quantized_matmul(x, O.BF16, w, s, b, O.BF16)
    _check(got, ref, O.BF16, f"decode M={M} N={N} K={K}")


@pytest.mark.parametrize("M,N,K,ys", [(65, 64, 512, 0), (129, 200, 1024, 0), (301, 1001, 512, 0),
                                      (300, 512, 12288, 8), (1024, 2048, 512, 0),
                                      (640, 8200, 512, 3), (700, 12288, 512, 0),
                                      (2050, 6150, 1024, 0), (4100, 12288, 512, 0)],
                         ids=["first-rows", "ragged", "odd-N", "long-K", "full-chip",
                              "odd-y-stride", "64x128", "128x128", "256x256"])
def test_tile_sizes(dev, M, N, K, ys):
    """Rows past the decode kernel: every tile size the launch chooses from,
    ragged rows and columns, y rows that are not 16-byte aligned. Large shapes
    are checked on rows and columns around the tile edges. |y - ref| <= 1 bf16
    ulp, as for every contraction: all products are exact, the sums f32."""
    x, w, s, b = _case(3801 + M + N, M, N, K)
    buf = torch.zeros((M, N + ys), dtype=torch.bfloat16, device=dev)
    H.quantized_matmul(to_dev(x, O.BF16, dev), words_dev(w, dev), to_dev(s, O.BF16, dev),
                       to_dev(b, O.BF16, dev), out=buf[:, :N])
    got = to_host(buf)
    assert (O.to_f32(got[:, N:], O.BF16) == 0).all()
    rows = np.unique(np.clip(np.r_[0:3, 62:66, 126:130, 254:258, M // 2, M - 70, M - 3:M], 0, M - 1))
    cols = np.unique(np.clip(np.r_[0:70, 120:140, 250:260, N // 2:N // 2 + 8, N - 140:N], 0, N - 1))
    ref = O.quantized_matmul(x[rows], O.BF16, w[cols], s[cols], b[cols], O.BF16)
    _check(got[:, :N][np.ix_(rows, cols)], ref, O.BF16, f"M={M} N={N} K={K}")


@pytest.mark.parametrize("M,N,K", [(65, 130, 576), (500, 300, 1088), (513, 257, 192), (777, 1000, 576)],
                         ids=["two-row-blocks", "eight", "hi-lo", "hi-lo-ragged"])
def test_other_k_over_many_rows(dev, M, N, K):
    """K that is no multiple of 512: the exact-product kernel up to 512 rows, the
    hi/lo-plane kernel above (weights to 2^-17, well inside the bar)."""
    x, w, s, b = _case(4201 + M + N, M, N, K)
    got = _run(dev, x, w, s, b, O.BF16)
    ref = O.quantized_matmul(x, O.BF16, w, s, b, O.BF16)
    _check(got, ref, O.BF16, f"M={M} N={N} K={K}")


@pytest.mark.parametrize("M,N,K", [(1, 70, 3584), (9, 200, 2048), (64, 300, 2048), (100, 384, 512),
                                   (600, 200, 1024)],
                         ids=["one-row", "few-rows", "decode", "exact", "hi-lo"])
def test_scales_off_a_word_boundary(dev, M, N, K):
    """Scales and biases that start at an odd element: the kernels that load them
    4 or 16 bytes at a time leave the call to the others."""
    x, w, s, b = _case(4301 + M + N, M, N, K)

    def odd(a):
        t = torch.empty(a.size + 1, dtype=torch.bfloat16, device=dev)
        t[1:] = to_dev(a, O.BF16, dev).flatten()
        assert t[1:].data_ptr() % 4 == 2
        return t[1:].view(a.shape)

    got = to_host(H.quantized_matmul(to_dev(x, O.BF16, dev), words_dev(w, dev), odd(s), odd(b)))
    ref = O.quantized_matmul(x, O.BF16, w, s, b, O.BF16)
    _check(got, ref, O.BF16, f"odd scales M={M} N={N} K={K}")


@pytest.mark.parametrize("M,N,K", [(33, 512, 2048), (64, 4096, 2048), (40, 8200, 2048),
                                   (129, 200, 1024), (301, 1001, 512), (1024, 2048, 512),
                                   (700, 12288, 512), (4100, 12288, 512)],
                         ids=["33-rows", "split-K", "decode", "64x64", "64x128x2", "64x128",
                              "128x128", "256x256"])
def test_a_row_with_inf_or_nan_leaves_the_others(dev, M, N, K):
    """Rows of x do not meet: with an Inf or NaN in the first and last rows, in
    a row and in the row 16 after it, every other row keeps its bits."""
    x, w, s, b = _case(3851 + M + N, M, N, K)
    clean = _run(dev, x, w, s, b, O.BF16)
    bad = [0, 3, 20, M - 1]
    x = x.copy()
    for r, v in zip(bad, (0x7F80, 0x7FC0, 0xFF80, 0x7F80)):  # Inf, NaN, -Inf, Inf
        x[r, (37 * r + 5) % K] = v
    got = _run(dev, x, w, s, b, O.BF16)
    rest = np.setdiff1d(np.arange(M), bad)
    assert np.array_equal(got[rest], clean[rest])
    # an Inf meets weights of both signs and a few zeros: no output is finite
    assert ((got[bad] & 0x7F80) == 0x7F80).mean() > 0.99


@pytest.mark.parametrize("M,N,K", [(64, 300, 2048), (129, 200, 1024), (301, 1001, 512),
                                   (1024, 2048, 512), (700, 12288, 512), (4100, 12288, 512)],
                         ids=["split-K", "64x64", "64x128x2", "64x128", "128x128", "256x256"])
def test_tiles_keep_the_sign_of_an_inf(dev, M, N, K):
    """What the tiles' group form cannot hold comes out as the f32 sum has it: a
    row with one Inf gives Inf with the sign of its weight, a row with one value
    whose product with a code overflows gives that value's finite result, an Inf
    bias gives Inf with the sign of its group's sum of x. The rest keeps its
    bits."""
    x, w, s, b = _case(3871 + M + N, M, N, K)
    clean = _run(dev, x, w, s, b, O.BF16)
    x, b = x.copy(), b.copy()
    inf, big, k, col, g = 2, M - 1, 70, min(77, N - 1), 3
    x[inf, k] = 0x7F80
    x[big, k] = 0x7F60  # 2.98e38
    b[col, g] = 0xFF80
    got = _run(dev, x, w, s, b, O.BF16)
    rows, cols = np.setdiff1d(np.arange(M), [inf, big]), np.setdiff1d(np.arange(N), [col])
    assert np.array_equal(got[np.ix_(rows, cols)], clean[np.ix_(rows, cols)])
    q = (w[:, k // 8] >> np.uint32(4 * (k % 8))) & 15
    wk = (O.to_f32(s[:, k // 64], O.BF16) * q.astype(np.float32) + O.to_f32(b[:, k // 64], O.BF16))[cols]
    want = np.where(wk == 0, np.nan, np.copysign(np.inf, wk))
    assert np.array_equal(O.to_f32(got[inf, cols], O.BF16), want, equal_nan=True)
    large = O.from_f32((O.to_f32(x[big, k], O.BF16) * wk).astype(np.float32), O.BF16)
    _check(got[big, cols][wk != 0], large[wk != 0], O.BF16, "one large value")
    sx = O.to_f32(x[rows, 64 * g:64 * g + 64], O.BF16).sum(1)
    assert np.array_equal(O.to_f32(got[rows, col], O.BF16), np.copysign(np.inf, -sx))


def test_qwen3_next_prefill_projection(dev):
    """A 2048-token prefill through a 2048 -> 4096 projection (the attention
    q projection's shape class)."""
    M, N, K = 2048, 4096, 2048
    x, w, s, b = _case(3101, M, N, K)
    got = _run(dev, x, w, s, b, O.BF16)
    # the oracle on a sample of rows (the full f64 product takes minutes)
    rows = np.r_[0:64, 1000:1032, M - 64:M]
    ref = O.quantized_matmul(x[rows], O.BF16, w, s, b, O.BF16)
    _check(got[rows], ref, O.BF16, "prefill 2048x4096x2048 (sampled rows)")


@pytest.mark.parametrize("M", [1, 3, 15])
def test_few_rows(dev, M):
    x, w, s, b = _case(3200 + M, M, 512, 2048)
    got = _run(dev, x, w, s, b, O.BF16)
    ref = O.quantized_matmul(x, O.BF16, w, s, b, O.BF16)
    _check(got, ref, O.BF16, f"M={M}")


@pytest.mark.parametrize("M,N,K", [(33, 4096, 2048), (64, 100, 12288), (50, 33, 4096),
                                   (64, 4097, 2048)], ids=["33-rows", "long-K", "ragged", "wider"])
def test_decode_rows_over_few_columns(dev, M, N, K):
    """33 to 64 rows over at most 4096 columns (32 x 32 tiles, K split over 8
    waves), and one column more (the decode kernel again)."""
    x, w, s, b = _case(4001 + M + N, M, N, K)
    got = _run(dev, x, w, s, b, O.BF16)
    ref = O.quantized_matmul(x, O.BF16, w, s, b, O.BF16)
    _check(got, ref, O.BF16, f"M={M} N={N} K={K}")


@pytest.mark.parametrize("M,N,K", [(1, 17, 512), (1, 4096, 3584), (2, 1000, 2048), (1, 512, 12288),
                                   (15, 64, 8192), (7, 12289, 512), (2, 12288, 2048), (2, 12289, 2048),
                                   (5, 4000, 1024), (4, 5100, 1024), (8, 7500, 512), (7, 8600, 512)])
def test_few_rows_of_any_k(dev, M, N, K):
    """1 to 15 rows: column tiles that are partly filled, K beyond the GEMV's
    list, few and many column tiles, both sides of the rules for few rows."""
    x, w, s, b = _case(3901 + M + N, M, N, K)
    got = _run(dev, x, w, s, b, O.BF16)
    ref = O.quantized_matmul(x, O.BF16, w, s, b, O.BF16)
    _check(got, ref, O.BF16, f"M={M} N={N} K={K}")


@pytest.mark.parametrize("M,N,K", [(1, 300, 512), (1, 130, 4096), (1, 35, 1536), (2, 17, 2560),
                                   (3, 64, 3584), (4, 100, 8192), (5, 33, 1536), (15, 48, 12288),
                                   (9, 70, 576), (1, 40, 14336)])
def test_few_rows_have_the_per_pair_kernels_bits(dev, M, N, K):
    """One row, and 1 to 15 rows with K outside 512, 1024, 2048 and 4096, are the
    per-pair kernels' sums operation by operation: the bits of gather_qmm over
    one expert, also for rows with an Inf or NaN."""
    x, w, s, b = _case(4101 + M + N, M, N, K)
    for bad in (None, 0x7F80, 0x7FC0):
        if bad is not None:
            x = x.copy()
            x[M - 1, K - 70] = bad
        y = to_host(H.gather_qmm(to_dev(x, O.BF16, dev), words_dev(w, dev)[None],
                                 to_dev(s, O.BF16, dev)[None], to_dev(b, O.BF16, dev)[None],
                                 torch.zeros(M, dtype=torch.int32, device=dev)))
        got = _run(dev, x, w, s, b, O.BF16)
        nan = np.isnan(O.to_f32(y, O.BF16))
        assert np.array_equal(np.isnan(O.to_f32(got, O.BF16)), nan)
        assert np.array_equal(got[~nan], y[~nan])


def sum_error(y, x, w, s, b):
    """The f32 sums' error: the rms error of the outputs within 1e-4 of the rms of
    all (their bf16 rounding is below 1e-7 of it), over that rms."""
    sh = torch.arange(0, 32, 4, device=w.device, dtype=torch.int32)
    q = ((w.unsqueeze(-1) >> sh) & 15).flatten(-2).double()
    wd = q * s.double().repeat_interleave(64, -1) + b.double().repeat_interleave(64, -1)
    ref = x.double() @ wd.t()
    rms = ref.pow(2).mean().sqrt()
    near = ref.abs() < 1e-4 * rms
    assert int(near.sum()) >= 20
    return float(((y.double() - ref)[near] / rms).pow(2).mean().sqrt())


def random_projection(g, dev, N, K):
    """Codes, scales and biases of weights with a mean near zero."""
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K // 8), dtype=torch.int32, device=dev, generator=g)
    s = 0.005 + 0.01 * torch.rand((N, K // 64), device=dev, generator=g)
    b = s * (3 * torch.rand((N, K // 64), device=dev, generator=g) - 9)
    return w, s.bfloat16(), b.bfloat16()


@pytest.mark.parametrize("mean", [0.0, 1.0])
@pytest.mark.parametrize("M,K", [(15, 512), (15, 2048), (12, 4096), (15, 1536)])
def test_few_rows_sum_as_exactly_as_one(dev, M, K, mean):
    """Sharing the weights between rows costs no precision: the f32 sums of M
    rows in one call are no further from 64 bits than the per-pair kernels'."""
    g = torch.Generator(device=dev)
    g.manual_seed(K)
    x = (torch.randn((M, K), device=dev, generator=g) + mean).bfloat16()
    q = random_projection(g, dev, 32768, K)
    together = sum_error(H.quantized_matmul(x, *q), x, *q)
    single = sum_error(H.gather_qmm(x, *(t[None] for t in q),
                                    torch.zeros(M, dtype=torch.int32, device=dev)), x, *q)
    print(f"[qgemm] M={M} K={K} mean={mean}: {together:.2e}, one by one {single:.2e}", flush=True)
    # some 40 outputs: the two rms have a spread of about 1 / sqrt(80) each
    assert together <= 1.25 * single


@pytest.mark.parametrize("dt,group", [(O.F16, 64), (O.BF16, 32), (O.BF16, 128)])
def test_other_dtypes_and_groups(dev, dt, group):
    x, w, s, b = _case(3300 + group, 40, 256, 1024, group=group, dt=dt)
    got = _run(dev, x, w, s, b, dt, group=group)
    ref = O.quantized_matmul(x, dt, w, s, b, dt, group=group)
    _check(got, ref, dt, f"dt={dt} group={group}")


def test_equals_gather_qmm_per_pair(dev):
    """The reference's own gather-vs-quantized_matmul check (qwen3_next.rs:
    2152-2206): gather_qmm over pairs of one expert equals quantized_matmul
    with that expert's weights, here within the same 1-ulp bar (the two run
    different kernels, with different f32 summation orders)."""
    M, E, N, K = 48, 4, 256, 1024
    x, _, _, _ = _case(3401, M, N, K)
    w = O.u32(3402, (E, N, K // 8))
    s = O.from_f32(O.uniform(3403, (E, N, K // 64), 0.005, 0.02), O.BF16)
    b = O.from_f32(O.uniform(3404, (E, N, K // 64), -0.1, 0.1), O.BF16)
    e = 2
    qm = _run(dev, x, w[e], s[e], b[e], O.BF16)
    ga = to_host(H.gather_qmm(to_dev(x, O.BF16, dev), words_dev(w, dev), to_dev(s, O.BF16, dev),
                              to_dev(b, O.BF16, dev),
                              torch.full((M,), e, dtype=torch.int32, device=dev)))
    _check(qm, ga, O.BF16, "quantized_matmul vs gather_qmm")


def test_strided_rows_and_leading_dims(dev):
    """x as [B, L, K] with a padded row stride; y written with the leading dims."""
    B, L, N, K = 3, 20, 256, 512
    x, w, s, b = _case(3501, B * L, N, K)
    buf = torch.zeros((B * L, K + 64), dtype=torch.bfloat16, device=dev)
    buf[:, :K] = to_dev(x, O.BF16, dev)
    xv = buf[:, :K]
    assert xv.stride(0) == K + 64
    y = H.quantized_matmul(xv, words_dev(w, dev), to_dev(s, O.BF16, dev), to_dev(b, O.BF16, dev))
    ref = O.quantized_matmul(x, O.BF16, w, s, b, O.BF16)
    _check(to_host(y), ref, O.BF16, "strided x")
    y3 = H.quantized_matmul(to_dev(x, O.BF16, dev).view(B, L, K), words_dev(w, dev),
                            to_dev(s, O.BF16, dev), to_dev(b, O.BF16, dev))
    assert tuple(y3.shape) == (B, L, N)
    _check(to_host(y3).reshape(B * L, N), ref, O.BF16, "3-d x")


def test_f16_gemv_grid_beyond_two_to_the_32_work_items(dev):
    """f16 runs one wave per output element: M = 512 rows of a 151936-column
    projection (the Qwen3 vocabulary) is 4.98e9 work-items, more than one HIP
    launch holds; the kernel walks the outputs in a capped grid instead. The
    oracle checks the first and last rows."""
    M, N, K = 512, 151936, 64
    x, w, s, b = _case(3601, M, N, K, dt=O.F16)
    got = _run(dev, x, w, s, b, O.F16)
    for rows in (np.r_[0:4], np.r_[M - 4:M]):
        ref = O.quantized_matmul(x[rows], O.F16, w, s, b, O.F16)
        _check(got[rows], ref, O.F16, f"f16 M={M} N={N} rows {rows[0]}..{rows[-1]}")
