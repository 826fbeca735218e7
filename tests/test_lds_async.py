"""The direct-to-LDS loads of lds_async.h write m0 in inline asm. Compiled between two uses of the
compiler's own direct-to-LDS builtin with one LDS base, each load must follow a write of m0 of its
own: if the compiler did not know that the asm changes m0, it would keep the first write for
both builtins, and the second would put its tile at the asm's address."""
import shutil
import subprocess
from pathlib import Path

import pytest

from kvip_amd.runtime import build

SOURCE = r"""
#include "lds_async.h"
namespace kvip {
extern "C" __global__ void mixed(const uint8_t* src, float* out, uint32_t at) {
    __shared__ __align__(16) float s[4096];
    const uint8_t* mine = src + threadIdx.x * 16;
    __builtin_amdgcn_global_load_lds(mine, LDS_PTR(&s[2048]), 16, 0, 0);
    LOAD(mine, lds_addr(&s[0]) + at);
    __builtin_amdgcn_global_load_lds(mine + 4096, LDS_PTR(&s[2048]), 16, 0, 0);
    wait_vmcnt<0>();
    __syncthreads();
    out[threadIdx.x] = s[threadIdx.x] + s[2048 + threadIdx.x];
}
}  // namespace kvip
"""


@pytest.mark.skipif(shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists(), reason="needs hipcc")
@pytest.mark.parametrize("load", ["dma16", "dma4"])
def test_m0_is_set_again_after_an_asm_load(tmp_path, load):
    source, listing = tmp_path / "mixed.hip", tmp_path / "mixed.s"
    source.write_text(f"#define LOAD {load}\n" + SOURCE)
    subprocess.run([build.hipcc(), *build.HIPCC_FLAGS, f"-I{build.INCLUDE}", f"-I{build.SOURCES}", "--cuda-device-only",
                    "-S", str(source), "-o", str(listing)], check=True, capture_output=True)
    order = []
    for line in listing.read_text().splitlines():
        words = line.replace(",", " ").split()
        if len(words) > 1 and words[1] == "m0" and words[0].startswith("s_"):
            order.append("m0")
        elif words and words[0].startswith("global_load_lds"):
            order.append("load")
    assert order == ["m0", "load"] * 3
