"""The loops of csrc/host_utils.cpp are compiled for three instruction sets, and the processor picks one: the other tests see that
one only, against the oracle.  Here every variant the machine can run is compared with the plain one, byte for byte, over
lengths around each variant's vector and at odd addresses."""
import os
import subprocess

from mixed_gemv_amd import build

SOURCE = r"""
#include "host_utils.cpp"
#include <cstdio>

static uint32_t g_state = 12345u;
static uint8_t random_byte() { return (uint8_t)((g_state = g_state * 1664525u + 1013904223u) >> 24); }
static std::vector<uint8_t> random_bytes(size_t n) {
  std::vector<uint8_t> v(n);
  for (auto& b : v) b = random_byte();
  return v;
}

// call(run, out): runs the loop's variant into out; all outputs have to be the plain variant's
template <typename Call>
static int compare(const char* name, size_t n, size_t out_bytes, Call call) {
  std::vector<uint8_t> want(out_bytes, 0xa5);
  call(0, want.data());
  for (int variant = 1; variant <= vector_variant(); ++variant) {
    std::vector<uint8_t> got(out_bytes, 0xa5);
    call(variant, got.data());
    if (got != want) {
      std::printf("%s: variant %d differs at n = %zu\n", name, variant, n);
      return 1;
    }
  }
  return 0;
}
template <typename Loop, typename... Args>
static void run_variant(int variant, Args... args) {
  if (variant == 2) run_avx512<Loop, Args...>(args...);
  else if (variant == 1) run_avx2<Loop, Args...>(args...);
  else run_plain<Loop, Args...>(args...);
}

template <int BITS>
static int compare_tiles(size_t rows, size_t k) {
  const size_t ksteps = (size_t)mgemv::num_ksteps((int)k, BITS), row_bytes = k * BITS / 8, tile_bytes = ksteps * mgemv::kUnitBytes;
  std::vector<uint8_t> matrix = random_bytes(rows * row_bytes + 1), tile = random_bytes(tile_bytes + 1);
  int bad = compare("recode", k, tile_bytes + 1, [&](int v, uint8_t* out) {
    run_variant<RecodeTile<BITS, false>>(v, out + 1, matrix.data() + 1, rows, row_bytes, ksteps);
  });
  bad += compare("decode", k, rows * row_bytes + 1, [&](int v, uint8_t* out) {
    run_variant<RecodeTile<BITS, true>>(v, tile.data() + 1, out + 1, rows, row_bytes, ksteps);
  });
  return bad;
}

int main() {
  int bad = 0;
  for (size_t n : {1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 1000}) {
    const auto wide = random_bytes(4 * n + 1);
    const int8_t* const in = reinterpret_cast<const int8_t*>(wide.data() + 1);
    bad += compare("pack", n, n + 1, [&](int v, uint8_t* out) { run_variant<PackInt4>(v, out + 1, in, (size_t)0, n); });
    bad += compare("unpack", n, 2 * n + 1, [&](int v, uint8_t* out) {
      run_variant<UnpackInt4>(v, reinterpret_cast<int8_t*>(out + 1), wide.data() + 1, (size_t)0, n);
    });
    bad += compare("fold", n, 2 * n, [&](int v, uint8_t* out) {
      run_variant<FoldZeroPoints>(v, reinterpret_cast<uint16_t*>(out), reinterpret_cast<const uint16_t*>(wide.data()), in + 2 * n, (size_t)0, n);
    });
  }
  {  // every scale with a few zero points
    std::vector<uint16_t> scales(65536);
    std::vector<int8_t> zeros(65536);
    for (size_t i = 0; i < 65536; ++i) { scales[i] = (uint16_t)i; zeros[i] = (int8_t)(i * 37 >> 3); }
    bad += compare("fold", 65536, 131072, [&](int v, uint8_t* out) {
      run_variant<FoldZeroPoints>(v, reinterpret_cast<uint16_t*>(out), (const uint16_t*)scales.data(), (const int8_t*)zeros.data(), (size_t)0, (size_t)65536);
    });
  }
  for (size_t rows : {4, 16})
    for (size_t k : {8, 64, 120, 128, 136, 512, 520, 1032}) bad += compare_tiles<4>(rows, k) + compare_tiles<8>(rows, k);
  std::printf("variants %d, differences %d\n", vector_variant() + 1, bad);
  return bad != 0;
}
"""


def test_every_variant_gives_the_plain_bytes(tmp_path):
    source, binary = tmp_path / "variants.cpp", tmp_path / "variants"
    source.write_text(SOURCE)
    subprocess.run([build.hipcc(), "-x", "c++", "-O2", "-std=c++17", "-ffp-contract=off", "-fopenmp",
                    "-I", build.CSRC, "-I", os.path.join(build.REPO_DIR, "include"), str(source), "-o", str(binary)], check=True)
    r = subprocess.run([str(binary)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
