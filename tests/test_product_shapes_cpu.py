"""The shape rule of products with more than 16 rows (choose_config, a host
function of libxtern.so), evaluated on the CPU: every shape it picks can be
launched for the rows that a call may have."""
import ctypes

import pytest

import xtern

BLOCKS = 65535  # row blocks of a 16-token launch (its grid's y)


class MMConfig(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in ("mb", "nb", "waves", "pf", "splitk", "kind")]


def choose(fmt, M, groups, nch, rowsum=False):
    f = xtern._lib["_ZN2xt13choose_configEiiiib"]
    f.restype = MMConfig
    f.argtypes = [ctypes.c_int] * 4 + [ctypes.c_bool]
    return f(fmt, M, groups, nch, rowsum)


@pytest.mark.parametrize("fmt,most", [(xtern.XT_PACK4, 18), (xtern.XT_XORSPARSE, 18), (xtern.XT_PACK5, 8)],
                         ids=["pack4", "sparse", "pack5"])
def test_rows_of_a_call_fit_the_chosen_launch(fmt, most, monkeypatch):
    """Calls of up to 65535 x 32 rows are taken up to `most` chunks of K (up
    to 65535 x 16 beyond): a 16-token shape must not be chosen above 65535
    row blocks, whatever it is priced at."""
    monkeypatch.delenv("XTERN_CONFIG", raising=False)
    bad = []
    for nch in list(range(1, most + 1)) + [most + 1, 40, 300]:
        limit = BLOCKS * (32 if nch <= most else 16)
        for M in (17, 1000, BLOCKS * 16 - 1, BLOCKS * 16, BLOCKS * 16 + 1, 1500001, BLOCKS * 32 - 31, BLOCKS * 32):
            if M > limit:
                continue
            for groups in (1, 2, 3, 4, 5, 6, 8, 16, 432):
                c = choose(fmt, M, groups, nch)
                blocks = -(-M // (16 * c.mb))
                if c.kind not in (0, 4) or (c.kind == 0 and blocks > BLOCKS):
                    bad.append((M, groups, nch, c.kind, c.mb, c.nb))
    assert not bad, f"{len(bad)}: {bad[:8]}"


def test_narrow_pack5_of_a_million_rows():
    assert choose(xtern.XT_PACK5, BLOCKS * 16, 2, 8).kind == 0  # (as priced, one block inside the limit)
    assert choose(xtern.XT_PACK5, BLOCKS * 16 + 1, 2, 8).kind == 4
    assert choose(xtern.XT_PACK5, 2097120, 6, 1).kind == 4


@pytest.mark.parametrize("cfg", ["gw,3,1,4", "gw,4,1,8", "gw,0,0,0", "gw,1,1,-4"])
def test_a_forced_shape_is_taken_or_refused(cfg, monkeypatch):
    """A forced shape of the many-row GEMM that is not compiled for the format
    must not run as another kernel (kind -1: the call fails)."""
    monkeypatch.setenv("XTERN_CONFIG", cfg)
    assert choose(xtern.XT_PACK4, 64, 432, 10).kind == -1
    assert choose(xtern.XT_PACK4, 16, 432, 10).kind == 2  # (no shape of that GEMM below 17 rows)


def test_a_forced_shape_keeps_the_offset_limit(monkeypatch):
    """4 GiB of weight tiles: beyond the kernel's 32-bit offsets."""
    monkeypatch.setenv("XTERN_CONFIG", "gw,4,2,4")
    c = choose(xtern.XT_PACK4, 64, 65535, 64)
    assert (c.kind, c.mb, c.nb, c.waves) == (4, 8, 16, 4)
    assert choose(xtern.XT_PACK4, 64, 65536, 64).kind == -1
    assert choose(xtern.XT_PACK4, 64, 16, 1 << 16).kind == -1


@pytest.mark.parametrize("M,K,N,mb,nb", [
    # one workgroup per CU at most: the smallest tile starts first (16 x 32
    # against 16 x 64, us: 5.3 / 5.8, 4.1 / 4.6, 5.0 / 6.2)
    (17, 4096, 2560, 1, 2), (17, 2048, 1024, 1, 2), (128, 4096, 640, 1, 2),
    # 25 columns of 16 x 128 tiles over 8 XCDs: each reads all of the weights
    # (against 32 x 128: 10.9 / 8.2, 9.2 / 6.9, 7.0 / 5.6)
    (128, 4096, 3200, 2, 8), (160, 3072, 3200, 2, 8), (64, 2048, 6912, 2, 8),
    # columns that divide over the XCDs (8.6 / 10.0)
    (128, 5120, 4096, 1, 8),
    # large activations, read again by every column (15.4 / 13.3)
    (512, 14336, 256, 1, 4),
])
def test_pack4_shapes_measured_fastest(M, K, N, mb, nb, monkeypatch):
    monkeypatch.delenv("XTERN_CONFIG", raising=False)
    for fmt in (xtern.XT_PACK4, xtern.XT_XORSPARSE):
        c = choose(fmt, M, -(-N // 16), -(-K // 256))
        assert (c.mb, c.nb) == (mb, nb)
