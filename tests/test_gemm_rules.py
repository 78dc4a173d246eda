"""The dense maps' host rules (workgroup tile, parts of the head's K loop), compiled from the library's own header with
g++ (no GPU): a product of few stages of K takes neither the large tile nor the parts that pay in a long one."""

import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
CSRC = ROOT / "alpha-fly_amd" / "csrc"
HIP_INCLUDE = pathlib.Path("/opt/rocm/include")
HEAD, ENCODER = 4299, 17937

PROGRAM = r"""
#include "gemm_rules.hpp"
#include <cstdio>
int main() {
  long long rows, batch, stages;
  while (scanf("%lld %lld %lld", &rows, &batch, &stages) == 3) {
    const int shape = fly::gemm_shape(rows, batch, stages, 0);
    const long long tiles = fly::gemm_tiles(rows, batch, shape);
    printf("%d %lld %d\n", shape, tiles, fly::head_parts(tiles, stages));
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None or not (HIP_INCLUDE / "hip" / "hip_runtime.h").exists():
        pytest.skip("g++ or the HIP headers are not installed")
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(PROGRAM)
    subprocess.run([gxx, "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{HIP_INCLUDE}", f"-I{CSRC}",
                    f"-I{ROOT / 'include'}", str(d / "rules.cpp"), "-o", str(d / "rules")], check=True)

    def ask(rows, batch, stages):
        out = subprocess.run([str(d / "rules")], input=f"{rows} {batch} {stages}", check=True, capture_output=True, text=True)
        return tuple(int(v) for v in out.stdout.split())

    return ask


@pytest.mark.parametrize("batch,shape,parts", [(1, 22, 3), (64, 22, 3), (65, 22, 3), (128, 22, 3), (129, 22, 2), (192, 22, 2),
                                               (193, 22, 3), (320, 22, 3), (321, 22, 1), (448, 22, 1), (449, 22, 2),
                                               (576, 22, 2), (577, 22, 1), (1120, 25, 1), (1500, 44, 1), (2048, 44, 2)])
def test_the_full_size_head(rule, batch, shape, parts):
    got = rule(HEAD, batch, 37)
    assert (got[0], got[2]) == (shape, parts)


@pytest.mark.parametrize("stages,batch,parts", [(1, 1, 1), (2, 64, 1), (2, 128, 1), (3, 64, 1), (4, 64, 2), (4, 65, 1), (10, 1, 2),
                                                (10, 64, 2), (10, 128, 1), (10, 256, 1), (16, 64, 2), (16, 576, 1),
                                                (19, 128, 3), (19, 320, 3), (19, 500, 2)])
def test_a_head_over_few_outputs_takes_fewer_parts(rule, stages, batch, parts):
    assert rule(HEAD, batch, stages)[2] == parts


@pytest.mark.parametrize("rows,batch,stages,shape", [(HEAD, 3000, 1, 22), (HEAD, 3000, 5, 22), (HEAD, 2048, 10, 22), (HEAD, 1700, 10, 44),
                                                     (HEAD, 1500, 19, 44), (ENCODER, 384, 14, 44), (ENCODER, 500, 14, 22),
                                                     (ENCODER, 640, 14, 44), (ENCODER, 1120, 14, 44), (HEAD, 4096, 1, 44)])
def test_the_large_tile_needs_full_rounds_and_some_stages(rule, rows, batch, stages, shape):
    assert rule(rows, batch, stages)[0] == shape
