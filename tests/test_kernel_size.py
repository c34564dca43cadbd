"""Code size of the DMA-fed GEMM's instantiations with every load path, from the symbol tables of the
built libsa3k.so. A short product spends its time fetching instructions: with the rare load paths' address
arithmetic inline at every use these kernels were 12-24 KB larger and their launches up to 1.2 times
slower (f32 128 x 32 tiles 52 KB and 11.0 us against 28 KB and 9.3). No GPU."""
import re
import shutil
import subprocess

import pytest

from conftest import sa3k
from test_isa_m0 import LLVM, MAGIC, TARGET

# template arguments of gemm_dma_kernel -> most bytes of code
MOST = {
    "128, 32, 4, 4, false, 4, false, 0, false, false, 0": 36 << 10,   # f32 rank products
    "32, 128, 1, 4, false, 4, false, 0, false, false, 0": 36 << 10,   # f32, a few rows
    "64, 128, 1, 3, false, 4, false, 0, false, false, 0": 54 << 10,   # f32, short K
    "128, 256, 2, 3, true, 16, false, 0, true, false, 0": 56 << 10,   # bf16 head preparation
}


@pytest.fixture(scope="module")
def sizes(tmp_path_factory):
    """template arguments -> bytes, of every gemm_dma_kernel in the library"""
    d = tmp_path_factory.mktemp("size")
    lib, fat = d / "lib.so", d / "fat.bin"
    shutil.copyfile(sa3k.LIB_PATH, lib)
    subprocess.run(["objcopy", "--dump-section", f".hip_fatbin={fat}", str(lib), str(d / "lib.out")], check=True)
    blob = fat.read_bytes()
    starts = [m.start() for m in re.finditer(re.escape(MAGIC), blob)]
    got = {}
    for k, s in enumerate(starts):
        part, co = d / f"b{k}.bundle", d / f"b{k}.co"
        part.write_bytes(blob[s:starts[k + 1] if k + 1 < len(starts) else len(blob)])
        subprocess.run([f"{LLVM}/clang-offload-bundler", "--type=o", "--unbundle", f"--input={part}", f"--output={co}",
                        f"--targets={TARGET}"], check=True)
        out = subprocess.run([f"{LLVM}/llvm-readelf", "-sW", "--demangle", str(co)], check=True, capture_output=True,
                             text=True).stdout
        for m in re.finditer(r"(\d+)\s+FUNC\s.*gemm_dma_kernel<([^>]*)>", out):
            got[m.group(2)] = int(m.group(1))
    return got


@pytest.mark.parametrize("args", sorted(MOST))
def test_general_instantiations_stay_small(sizes, args):
    assert sizes[args] <= MOST[args], f"{sizes[args]} bytes"
