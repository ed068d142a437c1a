"""RMSNorm, activation and the MLP's requantisation at the row lengths and row
counts where the middle kernel changes its width (256, 512 or 1024 threads per
row, one to nine pieces of four elements per thread, whole or single
elements), against the oracle bit for bit; and rows made to break the exact
sequential sum there: every element a tie, one binade per block, zeros,
subnormals, sums that overflow."""
import numpy as np
import pytest
import torch

import oracle
import xtern

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def bits(x):
    return np.asarray(x, np.float32).view(np.int32)


def rows(rng, M, n):
    x = rng.standard_normal((M, n)).astype(np.float32)
    x *= np.exp2(rng.integers(-12, 12, (M, 1))).astype(np.float32)
    k = min(M, 7)
    idx = np.arange(n, dtype=np.float32)
    special = [np.full(n, 1.0), np.where(idx == 0, 4096.0, np.sqrt(np.float32(2.0) ** -12)),
               np.exp2(np.minimum(idx, 60.0)), np.zeros(n), np.full(n, 1e-22), np.full(n, 1.5e19),
               np.where(idx < n - 1, 0.0, 3.0)]
    for i in range(k):
        x[M - 1 - i] = np.asarray(special[i], np.float32)
    return x


@pytest.mark.parametrize("M,n", [(8, 1), (8, 63), (8, 64), (9, 1023), (8, 1024), (8, 1028), (9, 2560), (8, 3072),
                                 (8, 3076), (8, 4096), (8, 4100), (8, 8192), (8, 8196), (8, 14336), (8, 16384),
                                 (9, 2049), (8, 8193), (520, 5120), (520, 5124), (514, 9216), (514, 9220)])
def test_rms_norm_widths(M, n):
    print(f"[case] norm M={M} n={n}", flush=True)
    rng = np.random.default_rng(n + M)
    x = rows(rng, M, n)
    w = rng.uniform(0.5, 1.5, n).astype(np.float32)
    y = xtern.rms_norm(torch.from_numpy(x).to(DEV), torch.from_numpy(w).to(DEV), 1e-5).cpu().numpy()
    pick = range(M) if M < 20 else list(range(6)) + list(range(M - 8, M))
    for m in pick:
        ref = oracle.rms_norm(x[m], w, 1e-5)[0]
        assert np.array_equal(bits(y[m]), bits(ref)), f"row {m}: {np.sum(bits(y[m]) != bits(ref))} differ"


@pytest.mark.parametrize("M,n", [(3, 1024), (300, 1024), (300, 1023), (3, 1025), (2, 4096), (2, 4100), (3, 8195),
                                 (515, 8200), (514, 10244), (2, 16384), (5, 1), (3, 17), (300, 64), (4100, 255),
                                 (3, 256), (3, 257), (512, 512), (513, 512), (513, 511), (2, 513), (256, 1003),
                                 (257, 1003)])
def test_activation_widths(M, n):
    print(f"[case] act M={M} n={n}", flush=True)
    rng = np.random.default_rng(n)
    g = (rng.standard_normal((M, n)) * 4).astype(np.float32)
    u = rng.standard_normal((M, n)).astype(np.float32)
    gd, ud = torch.from_numpy(g).to(DEV), torch.from_numpy(u).to(DEV)
    got = xtern.activation_mul(xtern.XT_ACT_RELU2_MUL, gd, ud).cpu().numpy()
    r = np.maximum(g, np.float32(0))
    assert np.array_equal(bits(got), bits((r * r).astype(np.float32) * u))
    wide = xtern.activation_mul(xtern.XT_ACT_SILU_INPLACE_SCALAR, gd, ud)
    for m in (0, M // 2, M - 1):  # (a row alone can take another width)
        one = xtern.activation_mul(xtern.XT_ACT_SILU_INPLACE_SCALAR, gd[m:m + 1], ud[m:m + 1])
        assert torch.equal(one[0].view(torch.int32), wide[m].view(torch.int32))
        ref = oracle.silu_inplace(g[m], u[m], True, avx512=False)
        assert np.array_equal(bits(wide[m].cpu().numpy()), bits(ref))


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("M,K,I", [(2, 64, 1024), (300, 64, 1020), (520, 64, 4608), (3, 64, 4613), (3, 64, 240),
                                   (4, 64, 333), (5, 64, 700)])
def test_mlp_rows_match_single_row(M, K, I, norm):
    """The MLP of many rows equals each row's (ReLU^2: one row takes the same
    function) and the oracle's, through the requantisation of every width."""
    print(f"[case] mlp M={M} K={K} I={I} norm={norm}", flush=True)
    rng = np.random.default_rng(I + M)

    def lin(k, n):
        t = rng.integers(-1, 2, (n, k)).astype(np.int8)
        b, ws = np.concatenate([xtern.pack_ternary4(r) for r in t]), np.full(n, 0.7, np.float32)
        return xtern.DeviceWeights(xtern.XT_PACK4, k, n, b, ws), (xtern.XT_PACK4, k, n, ws, dict(wbytes=b))

    (gate, go), (up, uo), (down, do) = lin(K, I), lin(K, I), lin(I, 48)
    w = torch.rand(I, device=DEV) + 0.5 if norm else None
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(DEV)
    y = xtern.mlp_f32(gate, up, down, x, norm_w=w)
    for m in (0, M // 2, M - 1):
        one = xtern.mlp_f32(gate, up, down, x[m:m + 1], norm_w=w)
        assert torch.equal(one[0].view(torch.int32), y[m].view(torch.int32))
        ref = oracle.mlp_forward(x[m:m + 1].cpu().numpy(), go, uo, do, w.cpu().numpy() if norm else None, 1e-5,
                                 False, fused=False)[0]
        assert np.array_equal(bits(y[m].cpu().numpy()), bits(ref[0]))
