"""One f32 row quantised inside the decode GEMV (packed bytes through each
wave's LDS row), at lengths around its chunk and wave counts and with rows of
special values, in both quantiser modes; and the compact-stream GEMV at row
counts around its three activation slices.  Integer sums and two f32
roundings: everything is compared bit for bit."""
import numpy as np
import pytest
import torch

import oracle
import xtern

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def weights(rng, fmt, K, N, ws):
    t = rng.integers(-1, 2, (N, K)).astype(np.int8)
    if fmt in (xtern.XT_XORSPARSE, xtern.XT_XORSPARSE_STREAM):
        b = np.frombuffer(xtern.encode_sparse_tensor(t, K, N)[0], np.uint8)
    else:
        pack = xtern.pack_ternary4 if fmt == xtern.XT_PACK4 else xtern.pack_ternary5
        b = np.concatenate([pack(r) for r in t])
    return t, xtern.DeviceWeights(fmt, K, N, b, ws)


def product(t, q, inv, ws):
    acc = (q.astype(np.float64) @ t.astype(np.float64).T).astype(np.int64)
    return ((acc.astype(np.float32) * inv[:, None]).astype(np.float32) * ws[None, :]).astype(np.float32)


def rows(rng, K):
    x = rng.standard_normal(K).astype(np.float32)
    ties = rng.integers(-254, 255, K).astype(np.float32) / 2  # absmax 127: exact .5 ties
    ties[K // 2] = 127.0
    last = np.zeros(K, np.float32)
    last[-1] = -3.0
    nan = x.copy()
    nan[K // 3] = np.nan
    return [x, ties, last, np.zeros(K, np.float32), nan]


@pytest.mark.parametrize("mode", ["avx512", "scalar"])
@pytest.mark.parametrize("fmt", [xtern.XT_PACK4, xtern.XT_XORSPARSE, xtern.XT_PACK5],
                         ids=["pack4", "sparse", "pack5"])
def test_fused_row_exact(fmt, mode):
    rng = np.random.default_rng(23)
    ch = 320 if fmt == xtern.XT_PACK5 else 256
    m = xtern.XT_QUANT_AVX512 if mode == "avx512" else xtern.XT_QUANT_SCALAR
    for K, N in ((4, 16), (ch - 4, 17), (ch, 1), (ch + 4, 640), (4 * ch, 33), (4 * ch + 16, 48),
                 (8 * ch + 4, 100), (10 * ch, 6500), (10 * ch + 4, 40), (16 * ch, 16), (16 * ch + 4, 50),
                 (17 * ch + 60, 200), (27 * ch, 64), (28 * ch, 2560)):
        print(f"[case] fused row fmt={fmt} {mode} K={K} N={N}", flush=True)
        ws = rng.uniform(0.2, 2.0, N).astype(np.float32)
        t, w = weights(rng, fmt, K, N, ws)
        for x in rows(rng, K):
            q, inv = oracle.quantize(x, m)
            y = xtern.linear_f32(w, torch.from_numpy(x[None]).to(DEV), mode=m).cpu().numpy()
            ref = product(t, np.asarray(q).reshape(1, K), np.float32(inv).reshape(1), ws)
            assert np.array_equal(y.view(np.int32), ref.view(np.int32)), f"{int(np.sum(y != ref))} differ"


@pytest.mark.parametrize("fmt,K,N", [(xtern.XT_PACK4, 8196, 40), (xtern.XT_XORSPARSE, 8448, 640),
                                     (xtern.XT_PACK4, 9020, 100), (xtern.XT_PACK4, 9216, 320),
                                     (xtern.XT_XORSPARSE, 9216, 17), (xtern.XT_PACK4, 9220, 40),
                                     (xtern.XT_PACK5, 8964, 40)])
def test_longest_fused_rows_exact(fmt, K, N):
    """Rows around the longest that the GEMV quantises (36 chunks of 256, three
    per wave of the last instantiation; Pack5 28 of 320): 9220 and 8964 take
    the separate quantiser."""
    rng = np.random.default_rng(K)
    print(f"[case] longest fused row fmt={fmt} K={K} N={N}", flush=True)
    ws = rng.uniform(0.2, 2.0, N).astype(np.float32)
    t, w = weights(rng, fmt, K, N, ws)
    for m in (xtern.XT_QUANT_AVX512, xtern.XT_QUANT_SCALAR):
        for x in rows(rng, K):
            q, inv = oracle.quantize(x, m)
            y = xtern.linear_f32(w, torch.from_numpy(x[None]).to(DEV), mode=m).cpu().numpy()
            ref = product(t, np.asarray(q).reshape(1, K), np.float32(inv).reshape(1), ws)
            assert np.array_equal(y.view(np.int32), ref.view(np.int32)), f"{int(np.sum(y != ref))} differ"


@pytest.mark.parametrize("K,N", [(512, 80), (1000, 777), (4096, 640)])
def test_stream_row_counts(K, N):
    rng = np.random.default_rng(K + N)
    ws = rng.uniform(0.2, 2.0, N).astype(np.float32)
    t, w = weights(rng, xtern.XT_XORSPARSE_STREAM, K, N, ws)
    for M in (2, 4, 5, 8, 9, 12, 16, 17, 21):
        print(f"[case] stream rows M={M} K={K} N={N}", flush=True)
        q = rng.integers(-128, 128, (M, K)).astype(np.int8)
        inv = rng.uniform(1e-3, 0.1, M).astype(np.float32)
        y = xtern.linear_q(w, torch.from_numpy(q).to(DEV), torch.from_numpy(inv).to(DEV)).cpu().numpy()
        assert np.array_equal(y.view(np.int32), product(t, q, inv, ws).view(np.int32))
