"""Rules of the kernels' launches that need no GPU: the sources' own functions, compiled for the host and called here."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def run(tmp_path, source):
    """The lines that a C++ program prints; it may include anything of rai_amd/csrc."""
    src, exe = tmp_path / "rule.cpp", tmp_path / "rule"
    src.write_text(source)
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O0", "-Wno-unused-result", f"-I{ROOT / 'rai_amd' / 'csrc'}", f"-I{ROOT / 'include'}",
                    str(src), "-o", str(exe), "-Wl,--unresolved-symbols=ignore-all"], check=True, capture_output=True, text=True, timeout=300)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout.splitlines()


@pytest.mark.parametrize("n1,n2", [(6, 0), (2, 0), (1001, 0), (16, 0), (0, 6), (0, 1000), (6, 7), (6464, 0), (3, 16384), (4112, 4112)])
def test_every_wave_of_a_row_step_reads_a_vector_that_is_there(tmp_path, n1, n2):
    """A step's Linears behind a norm: what any wave takes from LDS, waves without rows among them, ends before the partial sums."""
    lines = run(tmp_path, f"""
#include "latent_decode.hip"
using namespace rai;
int main() {{
  for (int K : {{64, 2048, 4096}}) {{
    LatentInArgs a;
    memset(&a, 0, sizeof(a));
    a.N1 = {n1}; a.N2 = {n2}; a.K = K; a.H = K; a.groups = 1;
    const size_t sums = kRowWaves * (1 + kRowGroups) * sizeof(float);
    for (int cus : {{16, 240, 256}})
      for (int at = 0; at < latent_in_blocks(a, cus) * kRowWaves; ++at) {{
        const bool second = latent_in_second(a, at);
        const size_t begin = second && a.N1 > 0 ? 2 * K : 0;
        if (begin + 2 * K > latent_in_lds(a) - sums) printf("K %d, %d CUs, wave %d\\n", K, cus, at);
        if (at < (a.N1 + 1) / 2 + (a.N2 + 1) / 2 && second != (at >= (a.N1 + 1) / 2)) printf("K %d, wave %d: another's vector\\n", K, at);
      }}
  }}
  puts("done");
}}""")
    assert lines == ["done"]


def test_offsets_of_tile_rows_fit_32_bits(tmp_path):
    """The 256 x 256 tiles of one block per CU: whatever row strides they take, a row's offset in 32 bits is the one in 64."""
    lines = run(tmp_path, """
#include "gemm_device.h"
using namespace rai;
int main() {
  LinearArgs a;
  memset(&a, 0, sizeof(a));
  const int64_t usual[4] = {64, 64, 64, 64};
  for (int which = 0; which < 4; ++which)
    for (int64_t ld = 64; ld < 1ll << 34; ld += ld < 4096 ? 8 : ld / 64 * 8) {
      int64_t l[4];
      for (int i = 0; i < 4; ++i) l[i] = i == which ? ld : usual[i];
      a.lda = l[0]; a.ldw = l[1]; a.ld1 = l[2]; a.ld2 = l[3];
      const bool fits = which < 2 ? 255 * 2 * ld + 7 * 16 < 1ll << 32 : 15 * ld + 7 * 8 < 1ll << 32;
      if (gemm_persist_serves(a) && !fits) { printf("stride %d of %lld\\n", which, (long long)ld); break; }
      if (ld <= 1 << 20 && !gemm_persist_serves(a)) printf("stride %d of %lld refused\\n", which, (long long)ld);
    }
  puts("done");
}""")
    assert lines == ["done"]
