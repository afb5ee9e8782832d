"""Kernels that keep what they work on in registers: that the compiler did so, in both libraries."""
import re
import shutil
import subprocess

import pytest

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module", params=["kernels_bf16", "kernels_f32"])
def scratch(request, tmp_path_factory):
    """Bytes of scratch memory a lane of every kernel of a library, by its symbol."""
    from zse_amd.runtime import build
    if shutil.which(READELF) is None or shutil.which(OBJDUMP) is None:
        pytest.skip("no llvm-readelf or llvm-objdump")
    if not build.is_current(request.param):
        build.build(request.param)
    folder = tmp_path_factory.mktemp("code")
    shutil.copy(build.lib_path(request.param), folder / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=folder, check=True, stdout=subprocess.DEVNULL)
    out = {}
    for obj in sorted(folder.glob("*gfx950")):
        notes = subprocess.run([READELF, "--notes", str(obj)], check=True, capture_output=True, text=True).stdout
        for part in notes.split("  - .agpr_count:")[1:]:
            out[re.search(r"\.name:\s+(\w+)", part)[1]] = int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", part)[1])
    return out


# a kernel, the number of its forms, those of them that may go through scratch memory
@pytest.mark.parametrize("kernel,forms,but", [("streams_row_kernel", 7, "ILi4ELi4ELi1024E"), ("conv_rows_kernel", 16, None),
                                              ("rope_cache_write_token_kernel", 3, None), ("mlstm_output_kernel", 6, None),
                                              ("mlstm_local_kernel", 6, None), ("attention_f32_kernel", 8, None),
                                              ("gemm_f32_kernelILi4ELi2E", 1, None), ("gemm_f32_kernelILi5ELi4E", 1, None),
                                              ("gemm_mid_norm_kernel", 18, None), ("gemm_skinny_kernel", 94, None), ("gemm_mid_kernel", 74, None)])
def test_no_scratch_memory(scratch, kernel, forms, but):
    found = {s: n for s, n in scratch.items() if kernel in s}
    if not found and kernel.startswith(("attention_f32", "gemm_")):
        pytest.skip("in the other library only")
    assert len(found) == forms
    assert {s: n for s, n in found.items() if n and not (but and but in s)} == {}


def test_arguments_that_a_kernel_reads(tmp_path):
    """Products without a norm or a rotation inside are not launched with the numbers of one: 64 bytes more on every product of up to 16 rows took 2 % of a
    step of few decoded tokens of a small model."""
    from zse_amd.runtime import build
    if shutil.which(READELF) is None or shutil.which(OBJDUMP) is None:
        pytest.skip("no llvm-readelf or llvm-objdump")
    shutil.copy(build.ensure("kernels_bf16"), tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    found = {}
    for obj in sorted(tmp_path.glob("*gfx950")):
        notes = subprocess.run([READELF, "--notes", str(obj)], check=True, capture_output=True, text=True).stdout
        for part in notes.split("  - .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\w+)", part)[1]
            if "gemm_skinny_kernel" in name or "gemm_mid_kernel" in name:
                own = [int(o) + int(n) for o, n, kind in re.findall(r"\.offset:\s+(\d+)\n\s+\.size:\s+(\d+)\n\s+\.value_kind:\s+(\w+)", part)
                       if not kind.startswith("hidden")]
                found[name] = max(own)
    # (their last argument says whether they have a norm, or rotate)
    plain = {n: size for n, size in found.items() if ("gemm_skinny" in n and "ELi0EEv" in n) or ("gemm_mid" in n and "ELb0EEv" in n)}
    others = {n: size for n, size in found.items() if n not in plain}
    assert plain and others
    assert max(plain.values()) <= 144 and min(others.values()) >= 136, (plain, others)
    assert max(size for n, size in plain.items() if "gemm_mid" in n) <= 80
