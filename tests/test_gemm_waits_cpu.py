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


def loads_by_kernel(asm):
    """Per shape (fmt, MW, NW, W, D) its buffer loads in order: w (weights to
    registers) and a (16-byte copies to LDS)."""
    out, cur = {}, None
    for line in asm.splitlines():
        m = KERNEL.match(line)
        if m:
            cur = out.setdefault(tuple(map(int, m.groups())), [])
        elif line.startswith("_ZN") or ".amdhsa_kernel" in line:
            cur = None
        elif cur is not None and "buffer_load_dwordx4" in line:
            cur.append("a" if re.search(r"\blds\b", line) else "w")
    return out


@pytest.mark.skipif(shutil.which(HIPCC) is None, reason="hipcc not available")
def test_copies_come_with_the_loads_the_waits_count(tmp_path):
    asm = str(tmp_path / "gemm.s")
    flags = [f for f in build_lib.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    cmd = [HIPCC] + flags + ["--cuda-device-only", "-S", os.path.join(build_lib.CSRC, "xtern_gemm.hip"), "-o", asm]
    res = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert res.returncode == 0, res.stderr[-3000:]
    with open(asm) as f:
        kernels = loads_by_kernel(f.read())
    assert len(kernels) == 8
    for (fmt, mw, nw, w, d), loads in kernels.items():
        chunk_cols = 320 if fmt == 1 else 256
        copies = -(-(32 * mw * chunk_cols // 1024) // w)  # per wave and chunk
        chunk = "w" * (2 * nw) + "a" * copies
        seq = "".join(loads)
        assert len(seq) % len(chunk) == 0 and seq == chunk * (len(seq) // len(chunk)), \
            f"gemmw_kernel<{fmt},{mw},{nw},{w},{d}>: {seq} is no sequence of {chunk}"
        assert seq.count(chunk) == 2 * d  # the first chunks, one round of the loop, and no more
