// Host-side check of the windows that the MFMA epilogues store wave tiles of D through (zluda_amd/csrc/kernels/
// store_window.hpp), for matrices of a few bytes to 64 GiB: every store of an element that exists is inside the window of its
// wave tile, every store of a lane past the end of P (offset kStoreNowhere) and of a column past the end of D is outside.
// usage: store_window_check   (prints the number of stores checked, exits non-zero on the first violation)
#include <algorithm>
#include <cstdio>
#include <cstdlib>

#include "../../zluda_amd/csrc/kernels/store_window.hpp"

using namespace zluda_amd;

static long checked = 0;

static void fail(const char *what, int64_t pitch, int NP, int NQ, int p, int q, int esz) {
  printf("D of %d columns of %d elements of %d bytes, pitch %lld, tile at (%d, %d): %s\n", NQ, NP, esz, (long long)pitch, p, q, what);
  exit(1);
}

// the wave tile of wt_p x wt_q elements at (pc, qc)
static void check_tile(int64_t pitch, int NP, int NQ, int pc, int qc, int wt_p, int wt_q, int esz) {
  const uint64_t window = tile_window_bytes(pitch, NP, NQ, (int64_t)qc * pitch + pc, esz);
  const int qs[] = {0, 1, wt_q / 2, wt_q - 1, NQ - 1 - qc, NQ - qc};
  const int ps[] = {0, wt_p / 2 - 1, wt_p - 1, NP - 1 - pc, NP - pc};
  for (int q : qs) {
    if (q < 0 || q >= wt_q) continue;
    const uint64_t soff = (uint64_t)q * pitch * esz;
    for (int p : ps) {
      if (p < 0 || p >= wt_p) continue;
      const bool exists = pc + p < NP && qc + q < NQ;
      const uint64_t at = pc + p < NP ? soff + (uint64_t)p * esz : soff + (uint32_t)kStoreNowhere;
      if (at + esz > 0xffffffffull) fail("offsets beyond 32 bits", pitch, NP, NQ, pc, qc, esz);
      if (exists && at + esz > window) fail("an element that exists is dropped", pitch, NP, NQ, pc, qc, esz);
      if (!exists && at < window) fail("an element that does not exist is stored", pitch, NP, NQ, pc, qc, esz);
      checked++;
    }
  }
}

int main() {
  const int extents[] = {1, 5, 64, 129, 1000, 4097, 32003, 50257, 128257, 2000001, (1 << 22) - 9};
  for (int NP : extents)
    for (int NQ : extents)
      for (int pad : {0, 1, 8})
        for (int esz : {1, 2, 4}) {
          const int64_t pitch = std::min<int64_t>(NP + pad, kNarrowPitch - 1);
          if (pitch * NQ * esz > 64ll << 30) continue;
          for (int wt : {32, 96, 128}) {
            const int last_p = (NP - 1) / wt * wt, last_q = (NQ - 1) / 128 * 128;
            // the corners of the matrix, and the places where 2 GiB and 4 GiB are left behind the corner
            const int64_t at2 = NQ - (0x80000000ll / esz) / pitch, at4 = NQ - (0x100000000ll / esz) / pitch;
            for (int64_t q : {(int64_t)0, (int64_t)last_q, at2 - 128, at2, at2 + 128, at4 - 128, at4, at4 + 128}) {
              if (q < 0 || q >= NQ) continue;
              const int qc = (int)(q / 128 * 128);
              for (int pc : {0, last_p, last_p + wt}) check_tile(pitch, NP, NQ, pc, qc, wt, 128, esz);
            }
          }
        }
  printf("%ld stores checked\n", checked);
  return 0;
}
