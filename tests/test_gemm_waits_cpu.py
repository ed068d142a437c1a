"""The waits of the many-row GEMM count loads: s_waitcnt vmcnt(n) before a
chunk is read from LDS assumes that every chunk in flight behind it was
requested with all of its weight loads and then all of its copies.  The
compiler may leave out loads whose result nothing reads, so the count is
checked where it is true or not: in the gfx950 assembly of each shape."""
import os
import re
import shutil
import subprocess

import pytest

import build_lib

HIPCC = build_lib.hipcc()
KERNEL = re.compile(r"^_ZN2xt12gemmw_kernelILi(\d)ELi(\d)ELi(\d)ELi(\d)ELi(\d)EEE\S*:")


def kernels_of(asm):
    """The instructions of every shape (fmt, MW, NW, W, D)."""
    out, cur = {}, None
    for line in asm.splitlines():
        m = KERNEL.match(line)
        if m:
            cur = out.setdefault(tuple(map(int, m.groups())), [])
        elif line.startswith("_ZN") or ".amdhsa_kernel" in line:
            cur = None
        elif cur is not None:
            cur.append(line)
    return out


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if shutil.which(HIPCC) is None:
        pytest.skip("hipcc not available")
    asm = str(tmp_path_factory.mktemp("asm") / "gemm.s")
    flags = [f for f in build_lib.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    cmd = [HIPCC] + flags + ["--cuda-device-only", "-S", os.path.join(build_lib.CSRC, "xtern_gemm.hip"), "-o", asm]
    res = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert res.returncode == 0, res.stderr[-3000:]
    with open(asm) as f:
        found = kernels_of(f.read())
    assert len(found) == 8
    return found


def test_copies_come_with_the_loads_the_waits_count(kernels):
    for (fmt, mw, nw, w, d), lines in kernels.items():
        # w: weights to registers, a: 16-byte copies to LDS
        loads = "".join("a" if re.search(r"\blds\b", x) else "w" for x in lines if "buffer_load_dwordx4" in x)
        chunk_cols = 320 if fmt == 1 else 256
        copies = -(-(32 * mw * chunk_cols // 1024) // w)  # per wave and chunk
        chunk = "w" * (2 * nw) + "a" * copies
        # the first chunks, one round of the loop, and no more
        assert loads == chunk * (2 * d), f"gemmw_kernel<{fmt},{mw},{nw},{w},{d}>: {loads} is not {chunk} x {2 * d}"


def test_no_store_waits_for_memory(kernels):
    """Scales loaded after the K loop put a wait before every store of a tile
    that M or N cuts, and with it one for the store before: the scales are
    requested before the first weights, and no wait for memory stands in a
    block of stores."""
    for shape, lines in kernels.items():
        first = next(i for i, x in enumerate(lines) if "buffer_load_dwordx4" in x)
        assert not [x for x in lines[first:] if "global_load" in x], shape
        blocks, block = [], []
        for x in lines:
            if re.match(r"\.LBB", x) or "s_cbranch" in x or "s_branch" in x:
                blocks.append(block)
                block = []
            else:
                block.append(x)
        stores = [b for b in blocks + [block] if any("global_store" in x for x in b)]
        assert stores
        for b in stores:
            assert not [x for x in b if "vmcnt" in x], shape
