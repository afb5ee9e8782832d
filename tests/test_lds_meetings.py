"""Kernels whose tiles are copied from memory straight into LDS: what the compiler made of their meetings.

A meeting frees the buffers that the waves have read, and copies into them follow.  A read that is issued
but has not come back when its wave meets may be overtaken by such a copy, and only the machine's timing
decides which of the two it sees, so it is the instructions that are looked at, not results."""
import re
import shutil
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
KERNELS = ("gemm_tile_direct_kernel", "attn_stream_kernel")


@pytest.fixture(scope="module")
def listings(tmp_path_factory):
    """Instructions of every form of the kernels, by its symbol."""
    from zse_amd.runtime import build
    if shutil.which(OBJDUMP) is None:
        pytest.skip("no llvm-objdump")
    if not build.is_current("kernels_bf16"):
        build.build("kernels_bf16")
    folder = tmp_path_factory.mktemp("code")
    shutil.copy(build.lib_path("kernels_bf16"), folder / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=folder, check=True, stdout=subprocess.DEVNULL)
    out = {}
    for obj in sorted(folder.glob("*gfx950")):
        if not any(name.encode() in obj.read_bytes() for name in KERNELS):
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(obj)], check=True, capture_output=True, text=True).stdout
        for part in re.split(r"^(?=(?:[0-9a-f]+ )?<\w+>:$)", text, flags=re.M):
            head = re.match(r"(?:[0-9a-f]+ )?<(\w+)>:", part)
            if head and any(name in head[1] for name in KERNELS):
                out[head[1]] = [line.split("//")[0].strip() for line in part.splitlines()[1:]]
    return out


@pytest.mark.parametrize("kernel", KERNELS)
def test_no_wave_meets_with_reads_in_flight(listings, kernel):
    forms = {s: code for s, code in listings.items() if kernel in s}
    assert forms
    for symbol, code in forms.items():
        assert any(c.startswith(("buffer_load", "global_load_lds")) and "lds" in c for c in code), symbol
        flying, meetings = 0, 0
        for c in code:
            if c.startswith("ds_read"):
                flying += 1
            elif c.startswith("s_waitcnt"):              # LDS answers a wave in order
                left = re.search(r"lgkmcnt\((\d+)\)", c)
                flying = min(flying, int(left[1])) if left else flying
            elif c.startswith("s_barrier"):
                meetings += 1
                assert flying == 0, f"{symbol}: {flying} reads in flight at meeting {meetings}"
        assert meetings >= 2
