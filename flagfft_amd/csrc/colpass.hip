// colpass.hip — register-resident two-stage super-stages (gfx950): the
// standalone kernels and their catalogue.  The pass body (colpass_body.hpp)
// is shared with the persistent queue kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "colpass_body.hpp"
#include "kernels.hpp"

namespace flagfft {
namespace dev {

// WPE: waves per SIMD the register allocation must leave room for (two
// workgroups of C * RB threads per CU: C * RB / 128).
template <typename T, int C, int RA, int RB, int NCH, int WPE, int MODE>
__global__ __launch_bounds__(C * RB) __attribute__((amdgpu_waves_per_eu(WPE))) void k_col(const StageArgs a) {
  col_body<T, C, RA, RB, NCH, MODE>(a, remap_block(blockIdx.x, a.nblocks, a.xcd_remap));
}

// The convolution launch of a two-pass Bluestein chain (square instances).
template <typename T, int C, int RA, int NCH, int WPE>
__global__ __launch_bounds__(C * RA) __attribute__((amdgpu_waves_per_eu(WPE))) void k_col_conv(const StageArgs a) {
  col_conv_body<T, C, RA, NCH>(a, remap_block(blockIdx.x, a.nblocks, a.xcd_remap));
}

}  // namespace dev

namespace {

constexpr int kColGroups = 256;  // one workgroup per CU

struct ColEntry {
  int r, ra, rb, c, nch, wpe;
  bool dbl;
  const void *f;   // plain passes
  const void *fb;  // ends of Bluestein chains
  int pref;  // default instance for first passes (1), later passes (2); 4: narrower tile for launches of few units
  int qvar;  // the persistent queue kernel's variant of this instance (k_queue in kernels.hip), -1 if none
  const void *fp;  // the instance with the DC / Nyquist pair modes, nullptr if none
  const void *fc;  // the convolution launch of a Bluestein chain (square instances), nullptr if none
};

#define FLAGFFT_COL(T, C, RA, RB, NCH, WPE, PREF) \
  {RA * RB, RA, RB, C, NCH, WPE, sizeof(T) == 8, (const void *)dev::k_col<T, C, RA, RB, NCH, WPE, dev::kColPlain>, \
   (const void *)dev::k_col<T, C, RA, RB, NCH, WPE, dev::kColBluestein>, PREF, \
   -1, nullptr, nullptr}
#define FLAGFFT_COLP(T, C, RA, RB, NCH, WPE, PREF) \
  {RA * RB, RA, RB, C, NCH, WPE, sizeof(T) == 8, (const void *)dev::k_col<T, C, RA, RB, NCH, WPE, dev::kColPlain>, \
   (const void *)dev::k_col<T, C, RA, RB, NCH, WPE, dev::kColBluestein>, PREF, \
   -1, (const void *)dev::k_col<T, C, RA, RB, NCH, WPE, dev::kColPair>, \
   (const void *)dev::k_col_conv<T, C, RA, NCH, WPE>}
#define FLAGFFT_COLQ(T, C, RA, RB, NCH, WPE, PREF, QVAR) \
  {RA * RB, RA, RB, C, NCH, WPE, sizeof(T) == 8, (const void *)dev::k_col<T, C, RA, RB, NCH, WPE, dev::kColPlain>, \
   (const void *)dev::k_col<T, C, RA, RB, NCH, WPE, dev::kColBluestein>, PREF, \
   QVAR, nullptr, nullptr}

#define FLAGFFT_COLC(T, C, RA, NCH, WPE, PREF, QVAR) \
  {RA * RA, RA, RA, C, NCH, WPE, sizeof(T) == 8, (const void *)dev::k_col<T, C, RA, RA, NCH, WPE, dev::kColPlain>, \
   (const void *)dev::k_col<T, C, RA, RA, NCH, WPE, dev::kColBluestein>, PREF, \
   QVAR, nullptr, (const void *)dev::k_col_conv<T, C, RA, NCH, WPE>}

// Measured on MI355X (2^20 x 16 and 2^24 C2C FP32): for R = 4096 (64 x 64
// in registers, 198 VGPRs, one 512-thread workgroup per CU) 8 units per
// workgroup, which makes 2^24 two passes instead of three (150 against
// 185 us) and the 4096-point columns of a 4096^2 transform one pass instead
// of two (75 against 95 us); for R = 1024 the first
// pass (contiguous stores) runs best with 32 units per workgroup, later
// passes (C-element stores) with 16; for R = 256 the first pass with 16
// units (65-67 us per 2^24 pass against 72-73 with 64), later passes with 64
// units in two exchange chunks (55-59 us against 62-65 with 16).
//
// A launch of fewer workgroups than CUs leaves the rest idle, and these
// transforms (a few MB, in the caches) are bound by one workgroup's latency,
// not by the row-segment width: the tile narrows until 256 workgroups are in
// flight (entries with 4, in order of falling C).  1024 x 1024 C2C: 1024-point
// columns in 32 workgroups of 32 units 21.3 us for the transform, 64 of 16
// 16.5, 128 of 8 16.0, 256 of 4 15.5; 1024 x 4096: 31.5, 29.0, 29.4 (C = 8);
// 65536 x 1: second pass of 64 / 32 / 16 units 14.2 / 11.2 / 10.5 us;
// 2048 x 2048: 16 / 8 units 35.1 / 33.3.  Narrower 128-, 256- (first pass)
// and 512-point FP32 tiles gave under 2 %.
const ColEntry kColTable[] = {
    FLAGFFT_COLP(float, 8, 64, 64, 2, 2, 3),          // 4096: 64-byte runs, 135 KB LDS, 198 VGPRs
    FLAGFFT_COL(float, 16, 64, 32, 2, 2, 3),          // 2048: 128-byte runs, 135 KB LDS, 256 VGPRs
    FLAGFFT_COL(float, 8, 64, 32, 2, 2, 4),           // 2048: 64-byte runs, 68 KB LDS
    FLAGFFT_COLC(float, 16, 32, 2, 4, 6, -1),          // 1024: 128-byte runs, 68 KB LDS, two workgroups per CU
    FLAGFFT_COL(float, 32, 32, 32, 2, 4, 1),          // 1024: 256-byte runs, 136 KB LDS, 1024 threads
    FLAGFFT_COL(float, 16, 32, 32, 1, 2, 0),          // 1024: 132 KB LDS, one workgroup per CU
    FLAGFFT_COLC(float, 8, 32, 2, 4, 4, 0),       // 1024: 64-byte runs, 35 KB LDS, four workgroups per CU
    FLAGFFT_COL(float, 8, 32, 32, 1, 2, 0),           // 1024: 64-byte runs
    FLAGFFT_COLC(float, 4, 32, 1, 2, 4, -1),           // 1024: 32-byte runs, 128 threads
    FLAGFFT_COLC(float, 16, 16, 1, 2, 5, 2),      // 256: 128-byte runs, 33 KB LDS
    FLAGFFT_COL(float, 32, 16, 16, 1, 4, 0),          // 256: 256-byte runs, 66 KB LDS
    FLAGFFT_COL(float, 64, 16, 16, 2, 4, 2),          // 256: 512-byte runs, 66 KB LDS, 1024 threads
    FLAGFFT_COLQ(float, 16, 32, 16, 1, 2, 3, 1),      // 512: 128-byte runs
    FLAGFFT_COLQ(float, 32, 16, 8, 1, 2, 3, 3),       // 128
    FLAGFFT_COL(float, 64, 8, 8, 1, 4, 3),            // 64: 512-byte runs
    FLAGFFT_COLC(float, 32, 8, 1, 2, 4, 4),        // 64: 256-byte runs
    FLAGFFT_COL(float, 16, 8, 8, 1, 2, 4),            // 64: 128-byte runs
    FLAGFFT_COLQ(float, 64, 8, 4, 1, 2, 3, 5),        // 32: 512-byte runs
    FLAGFFT_COLQ(float, 64, 4, 4, 1, 2, 3, 6),        // 16: 512-byte runs
    FLAGFFT_COLC(double, 8, 32, 2, 2, 3, -1),          // 1024: 128-byte runs, 70 KB LDS, 219 VGPRs
    FLAGFFT_COL(double, 4, 32, 32, 1, 2, 4),          // 1024: 64-byte runs
    FLAGFFT_COL(double, 8, 32, 16, 1, 2, 3),          // 512: 128-byte runs
    FLAGFFT_COL(double, 4, 32, 16, 1, 2, 4),          // 512: 64-byte runs
    FLAGFFT_COLC(double, 16, 16, 1, 2, 3, 7),     // 256: 256-byte runs, 66 KB LDS
    FLAGFFT_COLC(double, 8, 16, 1, 2, 4, -1),          // 256: 128-byte runs
    FLAGFFT_COLC(double, 4, 16, 1, 2, 4, -1),          // 256: 64-byte runs
    FLAGFFT_COL(double, 16, 16, 8, 1, 2, 3),          // 128
    FLAGFFT_COLC(double, 32, 8, 1, 2, 3, 9),       // 64
};

}  // namespace

namespace {

// Passes fused with the split-spectrum pass of a real transform, per super-radix
// in order of falling tile: half a tile's row segment is its mirror units', so the
// tiles are twice as wide as the plain passes' where they fit.  The narrow ones
// serve launches that leave CUs idle otherwise.  Two workgroups per CU of the wide
// tiles hide the exchanges (WPE 4; the 512-point one spills 10 VGPRs so and is still
// faster: 2^20 x 16 R2C 68.3 us, 70.4 without).
//
// Times of whole R2C / C2R transforms, with a pass of its own -> fused: 2^20 x 16
// 78 -> 68 / 83 -> 60 us, 65536 x 512 R2C 157 -> 102, 2^20 x 1 27.5 -> 18.7 / 28.3 -> 19.1,
// 2^17 x 8 R2C 19.7 -> 11.5, 2^22 x 4 97 -> 74 / 89 -> 61, FP64 2^20 x 8 93 -> 66 / 86 -> 55.
// Odd row lengths h + 1 misalign the runs of R2C stores, so those cannot bypass the
// caches (non-temporal stores: 68 -> 78 us), and the next transform's first pass
// shares HBM with their write-back.
struct ColRealEntry {
  int r, ra, rb, c;
  bool dbl;
  const void *post, *pre;
};
#define FLAGFFT_COLR(T, C, RA, RB, NCH, WPE)                                              \
  {RA * RB, RA, RB, C, sizeof(T) == 8,                                                    \
   (const void *)dev::k_col<T, C, RA, RB, NCH, WPE, dev::kColRealPost>,                   \
   (const void *)dev::k_col<T, C, RA, RB, NCH, WPE, dev::kColRealPre>}
const ColRealEntry kColRealTable[] = {
    FLAGFFT_COLR(float, 16, 64, 32, 2, 2),   // 2048
    FLAGFFT_COLR(float, 32, 32, 32, 2, 4),   // 1024
    FLAGFFT_COLR(float, 8, 32, 32, 2, 4),
    FLAGFFT_COLR(float, 32, 32, 16, 2, 4),   // 512
    FLAGFFT_COLR(float, 8, 32, 16, 2, 2),
    FLAGFFT_COLR(float, 32, 16, 16, 1, 4),   // 256
    FLAGFFT_COLR(float, 8, 16, 16, 1, 4),
    FLAGFFT_COLR(float, 32, 16, 8, 1, 4),    // 128
    FLAGFFT_COLR(float, 64, 8, 8, 1, 4),     // 64
    FLAGFFT_COLR(double, 8, 32, 32, 2, 2),   // 1024
    FLAGFFT_COLR(double, 16, 32, 16, 2, 2),  // 512
    FLAGFFT_COLR(double, 16, 16, 16, 1, 4),  // 256
    FLAGFFT_COLR(double, 4, 16, 16, 1, 4),
    FLAGFFT_COLR(double, 16, 16, 8, 1, 4),   // 128
    FLAGFFT_COLR(double, 32, 8, 8, 1, 4),    // 64
};

}  // namespace

int col_real_kernel_id(int64_t r, bool dbl, int64_t tcnt, int64_t total_units) {
  int best = -1, bc = 0;
  for (int id = 0; id < static_cast<int>(sizeof(kColRealTable) / sizeof(kColRealTable[0])); ++id) {
    const ColRealEntry &e = kColRealTable[id];
    if (e.r != r || e.dbl != dbl || tcnt % e.c != 0) continue;
    if (best < 0 || total_units < static_cast<int64_t>(kColGroups) * bc) {
      best = id;
      bc = e.c;
    }
  }
  // 2048 points once CUs run dry (2^22 x 1 C2R: 45 us, 37 with the pass of its own)
  if (r == 2048 && total_units < static_cast<int64_t>(kColGroups) * bc) return -1;
  return best;
}

void col_real_kernel_shape(int id, int &units, int &threads, size_t &lds_bytes, int &elem_bytes) {
  const ColRealEntry &e = kColRealTable[id];
  units = e.c;
  threads = e.c * e.rb;
  elem_bytes = e.dbl ? 16 : 8;
  const int half = e.ra / 2 * e.rb * e.c;  // the mirror exchange; the two-chunk forms' exchange and block store
  int need = half + half / 32;
  if (e.ra == 32 && e.rb == 32) need = std::max(need, e.ra * ((e.ra / 2) * e.c + 8));
  const int nch = e.ra >= 32 ? 2 : 1;
  const int ex = e.ra / nch * e.rb * e.c;
  const int bl = e.r / nch;
  need = std::max({need, ex + (ex >> 5) + 1, e.c * ((bl + bl / 32 + 28) / 32 * 32 + 4)});
  lds_bytes = static_cast<size_t>(need) * static_cast<size_t>(elem_bytes);
}

const void *col_real_kernel(int id, bool post) { return post ? kColRealTable[id].post : kColRealTable[id].pre; }

std::string col_real_targs(int id, bool post) {
  const ColRealEntry &e = kColRealTable[id];
  return std::to_string(e.c) + "," + std::to_string(e.ra) + "," + std::to_string(e.rb) + (post ? ",post" : ",pre");
}

// units: 0 for the default instance of a first (first = true) or later
// pass, C for the first instance with C units per workgroup, 1000 NCH + C
// for the one with NCH exchange chunks as well.
int col_kernel_id(int64_t r, bool dbl, int units, bool first) {
  const int n = static_cast<int>(sizeof(kColTable) / sizeof(kColTable[0]));
  const int c = units % 1000, nch = units / 1000;
  const int want = first ? 1 : 2;
  for (int id = 0; id < n; ++id) {
    const ColEntry &e = kColTable[id];
    if (e.r != r || e.dbl != dbl) continue;
    if (units <= 0 ? (e.pref & want) != 0 : (e.c == c && (nch == 0 || e.nch == nch))) return id;
  }
  return -1;
}

int col_kernel_id(int64_t r, bool dbl, int units) { return col_kernel_id(r, dbl, units, false); }

int col_kernel_id_for(int64_t r, bool dbl, bool first, int64_t total_units, bool rows, bool complex_ends) {
  const int n = static_cast<int>(sizeof(kColTable) / sizeof(kColTable[0]));
  // first 256-point passes of long 1D batches read 512-byte runs as the later
  // ones do (65536 x 128 48.0 -> 45.3 us, x 256 95.5 -> 89.4, x 64 the same; 256^3
  // columns lose 3 %)
  if (rows && first && r == 256 && !dbl && total_units >= 32768) first = false;
  int best = col_kernel_id(r, dbl, 0, first);
  if (best < 0) return best;
  for (int id = 0; id < n; ++id) {
    const ColEntry &e = kColTable[id], &b = kColTable[best];
    if (e.r != r || e.dbl != dbl || (e.pref & 4) == 0) continue;
    // (FP64: while the narrower workgroups are one per CU at most.  256-point passes
    // of 65536 x 8 / 10 / 12 in 128 / 160 / 192 workgroups of 16 14.3 / 15.7 / 16.5 us,
    // in 256 / 320 / 384 of 8 13.2 / 17.5 / 18.0; 2^19 x 3 29.7, in 384 of 4 33.2)
    const bool fits = !dbl || total_units <= static_cast<int64_t>(kColGroups) * e.c;
    if (total_units < static_cast<int64_t>(kColGroups) * b.c && e.c < b.c && fits) best = id;
  }
  // 2048 points in 64 elements per thread are slower than the LDS
  // super-stage's 16 once CUs run dry (2^21 x 1: 36 against 33 us, 2048 x 1024
  // columns: 20 against 18); 4096 points are not (2^22 x 1: 40 against 44).  Real and
  // Hermitian ends of a convolution have no super-stage, only the run-time-radix pass
  // of a fourth launch (R2C 1000003 x 1: 77 us, here 54; 160001 x 8: 147 and 53)
  if (complex_ends && r == 2048 && total_units < static_cast<int64_t>(kColGroups) * kColTable[best].c) return -1;
  return best;
}

int col_run_bytes(int64_t r, bool dbl, bool first) {
  const int id = col_kernel_id(r, dbl, 0, first);
  return id < 0 ? 0 : kColTable[id].c * (dbl ? 16 : 8);
}

bool col_tiles_divide(int64_t r, bool dbl, int64_t tcnt, int min_units) {
  for (const ColEntry &e : kColTable)
    if (e.r == r && e.dbl == dbl && e.c >= min_units && tcnt % e.c == 0) return true;
  return false;
}

std::vector<int64_t> col_kernel_radices(bool dbl) {
  std::vector<int64_t> v;
  for (const ColEntry &e : kColTable)
    if (e.dbl == dbl) v.push_back(e.r);
  return v;
}

int col_kernel_radix(int id) { return kColTable[id].r; }

int col_queue_kernel_id(int64_t r, bool dbl) {
  const int n = static_cast<int>(sizeof(kColTable) / sizeof(kColTable[0]));
  for (int id = 0; id < n; ++id)
    if (kColTable[id].r == r && kColTable[id].dbl == dbl && kColTable[id].qvar >= 0) return id;
  return -1;
}

int col_queue_variant(int id) { return kColTable[id].qvar; }

void col_kernel_shape(int id, int &units, int &threads, size_t &lds_bytes, int &elem_bytes) {
  const ColEntry &e = kColTable[id];
  units = e.c;
  threads = e.c * e.rb;
  elem_bytes = e.dbl ? 16 : 8;
  int need = 0;
  if (e.nch == 2 && e.ra == e.rb) {
    need = e.ra * ((e.ra / 2) * e.c + 8);  // two-chunk square form: RA rows of (RA / 2) C + 8 entries
  } else {
    const int ex = (e.ra / e.nch) * e.rb * e.c;                 // exchange chunk entries (+ 1 per 32)
    const int bl = e.r / e.nch;
    const int blk = e.c * ((bl + bl / 32 + 28) / 32 * 32 + 4);  // block-store chunk entries
    need = std::max(ex + (ex >> 5) + 1, blk);
  }
  lds_bytes = static_cast<size_t>(need) * static_cast<size_t>(elem_bytes);
}

const void *col_conv_kernel(int id) { return kColTable[id].fc; }

int col_conv_kernel_id(int64_t r, bool dbl, int64_t total_units) {
  const int n = static_cast<int>(sizeof(kColTable) / sizeof(kColTable[0]));
  int best = -1;
  for (int id = 0; id < n; ++id) {
    const ColEntry &e = kColTable[id];
    if (e.r != r || e.dbl != dbl || e.fc == nullptr) continue;
    if (best < 0 || (total_units < static_cast<int64_t>(kColGroups) * kColTable[best].c && e.c < kColTable[best].c)) best = id;
  }
  return best;
}

const void *col_kernel(int id, bool bluestein) { return bluestein ? kColTable[id].fb : kColTable[id].f; }

const void *col_pair_kernel(int id) { return kColTable[id].fp; }

int col_pair_kernel_id(int64_t r, bool dbl) {
  const int id = col_kernel_id(r, dbl, 0, true);
  return id >= 0 && kColTable[id].fp != nullptr ? id : -1;
}

std::string col_conv_targs(int id) {
  const ColEntry &e = kColTable[id];
  return std::to_string(e.c) + "," + std::to_string(e.ra) + "," + std::to_string(e.nch) + "," + std::to_string(e.wpe);
}

std::string col_kernel_targs(int id, int mode) {
  const ColEntry &e = kColTable[id];
  return std::to_string(e.c) + "," + std::to_string(e.ra) + "," + std::to_string(e.rb) + "," + std::to_string(e.nch) +
         "," + std::to_string(e.wpe) + "," + std::to_string(mode);
}

}  // namespace flagfft
