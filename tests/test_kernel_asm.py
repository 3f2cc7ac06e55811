"""What the compiler says about the kernels' inline assembly (CPU only: device
code is compiled for gfx950, nothing runs)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HIPCC = shutil.which('hipcc') or '/opt/rocm/bin/hipcc'


@pytest.mark.skipif(not Path(HIPCC).is_file(), reason='needs hipcc')
def test_direct_loads_keep_m0(tmp_path):
    """The direct-to-LDS loads set M0, which the compiler reserves: it may not be
    listed as clobbered (the compiler warns that this is undefined) and so has to
    be put back behind the last."""
    src = tmp_path / 'load.hip'
    src.write_text('#include "prefill_gemm.hpp"\n'
                   '__global__ void probe(const char* p, unsigned at) {\n'
                   '    const unsigned t = 16 * threadIdx.x, offsets[4] = {t, t + 4096, t + 8192, t + 12288};\n'
                   '    qwen_hip::load4_lds16_opaque<1024>(p, offsets, at);\n'
                   '    qwen_hip::wait_vmcnt<0>();\n}\n')
    out = tmp_path / 'load.s'
    done = subprocess.run([HIPCC, '--offload-arch=gfx950', '-O3', '-std=c++20', '--cuda-device-only', '-S', '-Werror',
                           '-Wno-unused-function', '-Wno-unused-command-line-argument', f'-I{ROOT / "include"}',
                           f'-I{ROOT / "fpga-qwen_amd" / "csrc"}', str(src), '-o', str(out)],
                          capture_output=True, text=True)
    assert done.returncode == 0, done.stderr
    body = [line.split(';')[0].split() for line in out.read_text().splitlines()]
    loads = [i for i, words in enumerate(body) if words[:1] == ['global_load_lds_dwordx4']]
    assert len(loads) == 4
    saved = next(words[1].rstrip(',') for words in body[:loads[0]] if words[:1] == ['s_mov_b32'] and words[-1] == 'm0')
    assert ['s_mov_b32', 'm0,', saved] in body[loads[-1]:]
