"""The many-row GEMM (gemmw_kernel) in every compiled shape, and the 16-token
shapes (mm_kernel) that the same rule chooses from, forced one at a time: chunk counts around its buffer counts (2, 3, 4: whole rounds, every
remainder, fewer chunks than buffers), token and output-row remainders, ragged
K, projections that end inside a tile, i32 accumulators requested or not.
Integer sums and two f32 roundings: everything is compared bit for bit."""
import numpy as np
import pytest
import torch

import xtern

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
PACK4 = ["4,2,4", "2,2,4", "2,1,4", "1,1,4"]
PACK5 = ["4,1,8", "4,1,4", "2,1,4", "1,1,4"]


def weights(rng, fmt, K, N, ws):
    t = rng.integers(-1, 2, (N, K)).astype(np.int8)
    if fmt == xtern.XT_XORSPARSE:
        b = xtern.encode_sparse_tensor(t, K, N)[0]
    else:
        pack = xtern.pack_ternary4 if fmt == xtern.XT_PACK4 else xtern.pack_ternary5
        b = np.concatenate([pack(r) for r in t])
    return t, xtern.DeviceWeights(fmt, K, N, b, ws)


def reference(t, q, inv, ws):
    acc = (q.astype(np.float64) @ t.astype(np.float64).T).astype(np.int64)
    y = ((acc.astype(np.float32) * inv[:, None]).astype(np.float32) * ws[None, :]).astype(np.float32)
    return acc, y.view(np.int32)


@pytest.mark.parametrize("fmt,shape", [(xtern.XT_PACK4, s) for s in PACK4]
                         + [(xtern.XT_XORSPARSE, "2,2,4")] + [(xtern.XT_PACK5, s) for s in PACK5])
def test_forced_shapes_exact(fmt, shape, monkeypatch):
    monkeypatch.setenv("XTERN_CONFIG", "gw," + shape)
    rng = np.random.default_rng(11)
    ch = 320 if fmt == xtern.XT_PACK5 else 256
    for M, K, N in ((17, 20, 16), (32, ch, 128), (33, 2 * ch, 129), (127, 3 * ch - 1, 257),
                    (128, 4 * ch, 256), (129, 5 * ch, 31), (31, 6 * ch + 4, 640), (65, 7 * ch, 100),
                    (64, 9 * ch, 64), (260, 8 * ch, 48)):
        print(f"[case] gw,{shape} fmt={fmt} M={M} K={K} N={N}", flush=True)
        ws = rng.uniform(0.2, 2.0, N).astype(np.float32)
        t, w = weights(rng, fmt, K, N, ws)
        q = rng.integers(-128, 128, (M, K)).astype(np.int8)
        inv = rng.uniform(1e-3, 0.1, M).astype(np.float32)
        acc_ref, y_ref = reference(t, q, inv, ws)
        qd, invd = torch.from_numpy(q).to(DEV), torch.from_numpy(inv).to(DEV)
        guard = torch.full((M + 1, N), 7.0, device=DEV)  # (a row past the output stays untouched)
        y = xtern.linear_q(w, qd, invd, out=guard[:M])
        y2, acc = xtern.linear_q(w, qd, invd, acc=True)
        assert np.array_equal(acc.cpu().numpy(), acc_ref)
        assert np.array_equal(y.cpu().numpy().view(np.int32), y_ref)
        assert np.array_equal(y2.cpu().numpy().view(np.int32), y_ref)
        assert bool((guard[M] == 7.0).all())


@pytest.mark.parametrize("fmt,shape", [(xtern.XT_PACK4, s) for s in PACK4] + [(xtern.XT_PACK5, s) for s in PACK5])
def test_forced_shapes_several_projections(fmt, shape, monkeypatch):
    """Projections of one launch that end inside a tile of every shape, the first
    or second wide enough that a later one starts past several tiles."""
    monkeypatch.setenv("XTERN_CONFIG", "gw," + shape)
    rng = np.random.default_rng(12)
    ch = 320 if fmt == xtern.XT_PACK5 else 256
    for M, K, widths in ((33, 2 * ch, (700, 96, 33)), (150, 3 * ch, (33, 700, 96, 1)), (17, ch, (256, 257))):
        print(f"[case] gw,{shape} fmt={fmt} M={M} K={K} N={widths}", flush=True)
        q = rng.integers(-128, 128, (M, K)).astype(np.int8)
        inv = rng.uniform(1e-3, 0.1, M).astype(np.float32)
        scales = [rng.uniform(0.2, 2.0, N).astype(np.float32) for N in widths]
        made = [weights(rng, fmt, K, N, s) for N, s in zip(widths, scales)]
        ys = xtern.linear_multi_q([w for _, w in made], torch.from_numpy(q).to(DEV), torch.from_numpy(inv).to(DEV))
        for (t, _), s, y in zip(made, scales, ys):
            assert np.array_equal(y.cpu().numpy().view(np.int32), reference(t, q, inv, s)[1])


@pytest.mark.parametrize("fmt,shape", [(xtern.XT_PACK4, s) for s in ("1,2,4,4,1", "1,4,8,2,1", "1,5,8,2,1", "1,8,8,2,1")]
                         + [(xtern.XT_XORSPARSE, "1,2,4,4,1")]
                         + [(xtern.XT_PACK5, s) for s in ("1,2,4,4,1", "1,4,8,2,1", "1,5,8,2,1", "1,5,16,1,1")])
def test_sixteen_token_shapes_exact(fmt, shape, monkeypatch):
    """Rows multiplied as they are (whole chunks, aligned: the kernel sums them
    itself) and through the padded copy (ragged K, or rows off 16 bytes: their
    sums are given), fewer and more chunks than a round of the waves, one and
    several projections."""
    monkeypatch.setenv("XTERN_CONFIG", shape)
    rng = np.random.default_rng(13)
    ch = 320 if fmt == xtern.XT_PACK5 else 256
    for M, K, widths in ((17, ch, (16,)), (33, 4 * ch, (129, 31)), (160, 9 * ch, (700,)), (48, 17 * ch, (96, 33, 257)),
                         (40, 5 * ch - 4, (130,)), (65, 18 * ch + 20, (33, 640))):
        print(f"[case] {shape} fmt={fmt} M={M} K={K} N={widths}", flush=True)
        q = rng.integers(-128, 128, (M, K)).astype(np.int8)
        inv = rng.uniform(1e-3, 0.1, M).astype(np.float32)
        scales = [rng.uniform(0.2, 2.0, N).astype(np.float32) for N in widths]
        made = [weights(rng, fmt, K, N, s) for N, s in zip(widths, scales)]
        off = torch.empty(M * K + 4, dtype=torch.int8, device=DEV)[4:].view(M, K)
        off.copy_(torch.from_numpy(q))
        for qd in (torch.from_numpy(q).to(DEV), off):
            ys = xtern.linear_multi_q([w for _, w in made], qd, torch.from_numpy(inv).to(DEV))
            for (t, _), s, y in zip(made, scales, ys):
                assert np.array_equal(y.cpu().numpy().view(np.int32), reference(t, q, inv, s)[1])


@pytest.mark.parametrize("fmt", [xtern.XT_PACK4, xtern.XT_PACK5], ids=["pack4", "pack5"])
@pytest.mark.parametrize("M", [17, 64, 200, 600])
def test_chosen_shapes_match_single_projections(fmt, M):
    """Whatever shape the dispatch takes: the f32 forward of three projections
    in one launch (widths that end inside a tile) equals the exact product of
    the quantised rows, and a repeated call gives the same bits."""
    rng = np.random.default_rng(M)
    K = 1340
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(DEV)
    q, inv = xtern.quantize_i8(x)
    made = []
    for N in (700, 96, 33):
        ws = rng.uniform(0.2, 2.0, N).astype(np.float32)
        made.append(weights(rng, fmt, K, N, ws) + (ws,))
    ys = xtern.linear_multi_f32([w for _, w, _ in made], x)
    again = xtern.linear_multi_f32([w for _, w, _ in made], x)
    for (t, _, ws), y, y2 in zip(made, ys, again):
        ref = reference(t, q.cpu().numpy(), inv.cpu().numpy(), ws)[1]
        assert np.array_equal(y.cpu().numpy().view(np.int32), ref)
        assert torch.equal(y, y2)
