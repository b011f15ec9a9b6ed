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


RULES = """
#include "gemm_mfma.hip"
namespace rai { int device_cu_count(int) { return 256; } }
using namespace rai;
static LinearArgs product(int m, int n, int k) {
  LinearArgs a = linear_args_default();
  a.M = m; a.N = n; a.K = k; a.dev = 0;
  a.lda = a.ldw = k; a.ld1 = n;
  a.splitk_ws = (void *)16; a.splitk_ws_bytes = 256 << 20;
  return a;
}
static const char *tile(int m, int n, int k) {
  const int t = tile_plan(product(m, n, k)).tile;
  for (const auto &x : kTileNames) if (x.tile == t) return x.name;
  return t == kTileStreamK ? "streamk64" : "?";
}
"""


def test_which_256_tiles_go_from_tile_to_tile(tmp_path):
    lines = run(tmp_path, RULES + """
int main() {
  LinearArgs a = product(4096, 4096, 4096);
  printf("%d ", persists(a));
  a.K = 4064; printf("%d ", persists(a));
  a.K = 4096; a.lda = 1 << 22; printf("%d ", persists(a));
  a.lda = 4096; a.ld1 = 1ll << 28; printf("%d ", persists(a));
  printf("%d %d %d ", persists(product(16384, 16384, 4096)), persists(product(16385, 16384, 4096)), persists(product(1 << 20, 1 << 20, 65536)));
  LinearArgs r = product(16385, 16384, 4096);   // a residual that is asked for ahead, whatever the operands' size
  r.residual = (void *)64; r.ldr = 16384; printf("%d ", persists(r));
  r.bias = (void *)64; printf("%d ", persists(r));
  r.bias = nullptr; r.ldr = 16383; printf("%d\\n", persists(r));
}""")
    assert lines == ["1 0 0 0 1 0 0 1 0 0"]


def test_which_shares_go_from_tile_to_tile(tmp_path):
    """From 192 MB of operands on shares that fewer than two whole rounds follow are blocks' again, unless a residual is asked for ahead."""
    lines = run(tmp_path, RULES + """
static int shares(LinearArgs a) { return 10 * persists(a) + persists(a, true); }
int main() {
  printf("%02d %02d %02d %02d ", shares(product(16384, 1536, 4608)), shares(product(16384, 1536, 5632)), shares(product(16384, 1536, 7168)), shares(product(16384, 1536, 8960)));
  printf("%02d %02d %02d ", shares(product(8192, 3072, 8192)), shares(product(8192, 3072, 10240)), shares(product(4096, 10240, 8192)));
  LinearArgs r = product(16384, 1536, 6144);
  r.residual = (void *)64; r.ldr = 1536; printf("%02d ", shares(r));
  r.K = 8960; printf("%02d\\n", shares(r));
}""")
    assert lines == ["11 10 10 00 11 10 11 11 11"]


@pytest.mark.parametrize("m,n,k,want", [
    # K an odd number of 32s: 256 x 256 tiles are a block's each and cost as much
    (4397, 19664, 288, "192x256"), (14470, 5768, 224, "192x256"), (16384, 8960, 1504, "256x256k64"),
    # a half-full last round: shares, whole 256 x 256 tiles, others
    (16384, 1536, 8960, "streamk64"), (16384, 1536, 6144, "streamk64"), (4096, 6144, 4096, "streamk64"), (2827, 24480, 2048, "256x256k64"), (16384, 17920, 1536, "256x256k64"),
    (1341, 16320, 3584, "192x256"), (5900, 3936, 3840, "192x256")])
def test_tile_of_a_product(tmp_path, m, n, k, want):
    assert run(tmp_path, RULES + f'int main() {{ puts(tile({m}, {n}, {k})); }}') == [want]
