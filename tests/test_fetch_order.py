"""The fetch kernels raise a flag in host memory that the host takes as the
arrival of the whole result, so every wave's stores have to be out before the
barrier ahead of the flag: a barrier by itself waits for none of them. Whether
they are cannot be seen from results (a late store is a matter of luck), so
this looks at the device code built here from this repository's source."""
import os
import re
import struct
import subprocess

import pytest

from pas_cg_amd import build as B

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def _device_code(path):
    """The gfx950 code objects bundled in the library."""
    d = open(path, "rb").read()
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", d):
        at = m.start()
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", d, at + 24)[0]):
            off, size, name = struct.unpack_from("<QQQ", d, entry)
            target = d[entry + 24:entry + 24 + name]
            entry += 24 + name
            if b"gfx950" in target and size:
                yield d[at + off:at + off + size]


def _waits_before_barrier(lines):
    """Each store to memory has a wait for it between itself and the next
    barrier, in the order of the code."""
    open_stores = False
    for x in lines:
        if re.match(r"(global|flat|buffer)_store", x):
            open_stores = True
        elif x.startswith("s_waitcnt") and "vmcnt(0)" in x:
            open_stores = False
        elif x.startswith("s_barrier"):
            return not open_stores
    return False


def test_the_check_itself():
    late = ["global_store_dwordx2 v[6:7], v[4:5], off", "s_waitcnt lgkmcnt(0)", "s_barrier",
            "buffer_wbl2 sc0 sc1", "s_waitcnt vmcnt(0)", "global_store_dword v0, v1, s[2:3]"]
    assert not _waits_before_barrier(late)
    assert _waits_before_barrier(late[:1] + ["s_waitcnt vmcnt(0)"] + late[2:])


@pytest.mark.skipif(not (os.path.exists(B.LIB) and os.path.exists(OBJDUMP)),
                    reason="needs the built library and llvm-objdump")
def test_fetch_releases_every_wave(tmp_path):
    seen = 0
    for k, code in enumerate(_device_code(B.LIB)):
        if b"k_fetch" not in code:
            continue
        f = tmp_path / f"{k}.co"
        f.write_bytes(code)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], capture_output=True,
                              text=True, check=True).stdout
        for body in re.split(r"\n\n", text):
            if not re.search(r"<\w*k_fetch\w*>:", body.splitlines()[0] if body else ""):
                continue
            lines = [x.split("//")[0].strip() for x in body.splitlines()[1:]]
            assert any(x.startswith("buffer_wbl2") for x in lines)
            assert _waits_before_barrier(lines), body
            seen += 1
    assert seen == 2  # FP32 and FP64 columns
