"""The tile order of the prefill GEMMs (csrc/gemm_map.hpp) on the CPU: the
workgroups of a launch take every tile exactly once, whatever the rows and
outputs, up to the largest operands that fit the card's memory."""
import ctypes
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / 'fpga-qwen_amd' / 'csrc'

SHIM = r'''
#include <vector>
#include "gemm_map.hpp"
using namespace qwen_hip;
// Tiles taken twice or never; -1 where a workgroup falls outside the order.
extern "C" long long wrong_tiles(int M, int N, int BM, int BN) {
    const GemmMap map(M, N, BM, BN, 1);
    std::vector<unsigned char> seen(size_t(map.mtiles) * map.ntiles, 0);
    for (unsigned w = 0; w < map.groups(); ++w) {
        const auto [mt, nt] = map_tile(w, map.f, map.per, map.magic);
        if (mt < 0 || nt < 0) return -1;
        if (mt < map.mtiles && nt < map.ntiles && seen[size_t(mt) * map.ntiles + nt] < 2)
            ++seen[size_t(mt) * map.ntiles + nt];
    }
    long long wrong = 0;
    for (const unsigned char s : seen) wrong += s != 1;
    return wrong;
}
'''


@pytest.fixture(scope='module')
def shim(tmp_path_factory):
    where = tmp_path_factory.mktemp('map')
    (where / 'shim.cpp').write_text(SHIM)
    subprocess.run(['g++', '-std=c++20', '-O2', '-Wall', '-Werror', '-shared', '-fPIC', f'-I{CSRC}',
                    str(where / 'shim.cpp'), '-o', str(where / 'shim.so')], check=True)
    lib = ctypes.CDLL(str(where / 'shim.so'))
    lib.wrong_tiles.restype = ctypes.c_longlong
    return lib


@pytest.mark.parametrize('bm,bn', [(16, 32), (32, 64), (48, 128), (64, 96), (96, 192), (128, 256)])
def test_every_tile_once(shim, bm, bn):
    for m in [*range(1, 400, 7), 512, 513, 1000, 1024, 1536, 2049, 3073, 4096, 70001, 1048577]:
        for n in (768, 1536, 3072, 6144):
            assert shim.wrong_tiles(m, n, bm, bn) == 0, (m, n)


@pytest.mark.parametrize('m,n,bm,bn', [(16777215, 2176, 128, 128), (16500000, 3968, 128, 128)])
def test_every_tile_once_of_the_largest(shim, m, n, bm, bn):
    """Rows up to the launch limit of the kernel that splits the operand (2^32
    threads of 256 per row), with outputs of 146 and 262 GB."""
    assert shim.wrong_tiles(m, n, bm, bn) == 0
