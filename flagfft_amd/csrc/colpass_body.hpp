// colpass_body.hpp — register-resident two-stage super-stages (gfx950 device code).
//
// One launch is one pass of a multi-pass chain (the reference's four-step
// column / row passes, python/flagfft_codegen/kernels.py:710-742) for a
// super-radix R = RA x RB whose two stages both run in registers:
//   * C adjacent units per workgroup, lane -> (unit slot = tid % C, t = tid / C),
//     so every HBM access of a wavefront is C-element row segments (C x 8 bytes
//     in FP32: 128-512 byte runs, the width a strided HBM stream needs);
//   * stage A: thread t loads the RA elements t + RB j (j < RA), applies the
//     inter-pass twiddles, and transforms them in registers (radix RA);
//   * inner twiddles w_R^(t k1), then the RA x RB transpose within each unit
//     goes through LDS in NCH chunks of k1, so a workgroup needs 1 / NCH of
//     its tile in LDS and two workgroups share a CU;
//   * stage B: thread t' transforms the RB values of k1 = t' + RB m (radix RB)
//     and holds outputs k1 + RA k2;
//   * the first pass of contiguous rows stores each unit's R outputs as one
//     contiguous block (through LDS, NCH chunks of k2); later passes store
//     C-element runs directly.
// Same index map, twiddles and results as the LDS Stockham super-stage
// (stage.hip, mode kStagePass): unit i of sequence b reads x[i + e tcnt]
// (e < R), multiplies element e by w_n^(e kt twp_mult), transforms, and
// writes y[(i - k) R + k + e' p], k = i mod p.
//
// Included by colpass.hip (the standalone kernels) and kernels.hip (the
// persistent queue kernel runs the same bodies).
#pragma once

#include <hip/hip_runtime.h>

#include "codelets.hpp"
#include "dev_common.hpp"
#include "fft_args.hpp"

namespace flagfft {
namespace dev {

// LDS slot of exchange entry (kk, t, slot) of a chunk: slots fastest, so a
// wavefront's stores of one kk are 64 consecutive entries; one pad entry per 32.
template <int C, int RB>
__device__ __forceinline__ int xslot(int kk, int t, int sl) {
  const int idx = (kk * RB + t) * C + sl;
  return idx + (idx >> 5);
}

// Store to element `idx` of an array with a uniform base and a 32-bit lane
// offset (global_store with saddr), as ldt loads.
template <typename T>
__device__ __forceinline__ void stt(GlbC<T> *base, uint32_t idx, V2<T> v) {
  FLAGFFT_GLB char *b = reinterpret_cast<FLAGFFT_GLB char *>(base);
  stg(reinterpret_cast<GlbC<T> *>(b + idx * static_cast<uint32_t>(sizeof(V2<T>))), v);
}

template <typename T>
__device__ __forceinline__ void stt_nt(GlbC<T> *base, uint32_t idx, V2<T> v) {
  FLAGFFT_GLB char *b = reinterpret_cast<FLAGFFT_GLB char *>(base);
  stg_nt<T>(reinterpret_cast<GlbC<T> *>(b + idx * static_cast<uint32_t>(sizeof(V2<T>))), v);
}

// p[j] = w^j for j < N <= 8 (p[0] = 1), at most two products from w, w^2 and w^4,
// which get(b) gives (b = 0, 1, 2; EXACT), or from w alone.  Powers of one
// rounded w carry its error up to j times over: FP32 chains of 2^20 points have
// a relative L2 error of 2.75e-7 that way and 2.03e-7 with the three values,
// for 1 % of their time.  Passes of 16 elements per thread keep the one load
// (with three, twice the loads of their data: second pass of 65536 x 256 44.5 ->
// 46.7 us) unless they are an end of a Bluestein chain, where they stand in for the
// run-time-radix pass with its table of all powers.
template <int N, bool EXACT, typename T, typename Get>
__device__ __forceinline__ void powers(Get get, V2<T> *p) {
  p[0] = V2<T>{1, 0};
  if constexpr (N > 1) p[1] = get(0);
  if constexpr (N > 2) p[2] = EXACT ? get(1) : cmul(p[1], p[1]);
  if constexpr (N > 3) p[3] = cmul(p[2], p[1]);
  if constexpr (N > 4) p[4] = EXACT ? get(2) : cmul(p[2], p[2]);
  if constexpr (N > 5) p[5] = cmul(p[4], p[1]);
  if constexpr (N > 6) p[6] = EXACT ? cmul(p[4], p[2]) : cmul(p[3], p[3]);
  if constexpr (N > 7) p[7] = cmul(p[4], p[3]);
}

// What an instance runs besides plain passes: the DC / Nyquist pair of a 2D real
// column pass (StageArgs::dc_nyq_pair), or the ends of Bluestein chains (chirp
// source, pointwise and chirp sinks).  Instances of their own: the sinks' table
// values cost the 64 x 256-point pass its second workgroup per CU (42 -> 54 us of
// 65536 x 256).
//
// kColRealPost / kColRealPre: the last / first pass of the n/2-point chain of an
// even-length real transform, with the split-spectrum pass in it (real_partner):
// a tile holds C / 2 units and their mirror units.
enum ColMode : int { kColPlain = 0, kColPair = 1, kColBluestein = 2, kColRealPost = 3, kColRealPre = 4 };

// Unit slot `sl` of tile `blk`: its position i in sequence bq + dq, where bq
// is the sequence of the tile's first unit (uniform over the workgroup: the
// addresses stay a uniform base plus 32-bit lane offsets; the host checks that
// the sequences a tile touches span under 4 GiB).  A tile may run over the end
// of a sequence into the next ones, so a sequence's units need not be a
// multiple of C (129 half-spectrum columns of 256 slabs: 2064 whole tiles
// where whole-sequence tiles were impossible and the LDS super-stage took
// 38 us per 67 MB sweep); slots past the last unit repeat it and stay idle.
struct ColUnit {
  uint32_t bq, dq, i;
  bool active;  // the slot has a unit
  bool whole;   // every slot of the tile has one (uniform)
};
// Unit of slot sl of a real tile whose first pair is j0.
template <int C>
__device__ __forceinline__ uint32_t pair_unit(uint32_t j0, uint32_t tcnt, int sl) {
  const uint32_t j = j0 + static_cast<uint32_t>(sl % (C / 2));
  return sl < C / 2 ? j : j == 0 ? tcnt / 2 : tcnt - j;
}
template <int C, int MODE>
__device__ __forceinline__ ColUnit col_unit(const StageArgs &a, int blk, int sl) {
  const uint32_t u0 = static_cast<uint32_t>(blk) * C;
  if constexpr (MODE == kColRealPost || MODE == kColRealPre) {
    // whole tiles of one sequence: units j and tcnt - j (0 and tcnt / 2 are their
    // own mirror units and share the pair j = 0)
    ColUnit r;
    const uint32_t tcnt = static_cast<uint32_t>(a.tcnt);
    r.bq = fdiv(u0, a.fd_tcnt);
    r.dq = 0;
    r.i = pair_unit<C>((u0 - r.bq * tcnt) / 2, tcnt, sl);
    r.active = r.whole = true;
    return r;
  }
  const uint32_t units = static_cast<uint32_t>(a.units);
  const uint32_t u = min(u0 + static_cast<uint32_t>(sl), units - 1u);
  ColUnit r;
  r.bq = fdiv(u0, a.fd_tcnt);
  const uint32_t b = fdiv(u, a.fd_tcnt);
  r.dq = b - r.bq;
  r.i = u - b * static_cast<uint32_t>(a.tcnt);
  r.active = u0 + static_cast<uint32_t>(sl) < units;
  r.whole = u0 + C <= units;
  return r;
}

// Loads of tile `blk`: element e = t + RB j of the thread's unit (zero
// outside the units); a Bluestein chirp source comes with its chirp.
template <typename T, int C, int RA, int RB, int MODE>
__device__ __forceinline__ void col_load(const StageArgs &a, int blk, V2<T> (&x)[RA]) {
  const int tid = threadIdx.x;
  const int sl = tid % C;
  const int t = tid / C;
  const ColUnit un = col_unit<C, MODE>(a, blk, sl);
  const uint32_t i = un.i;
  const uint32_t tcnt = static_cast<uint32_t>(a.tcnt);
  const uint32_t lead = un.dq * static_cast<uint32_t>(a.bs_in);
  const uint32_t ia = i + lead;
  const GlbC<T> *src = gc<T>(a.in) + static_cast<int64_t>(un.bq) * a.bs_in;
  const bool chirp_in = MODE == kColBluestein && (a.src_mode & kSrcChirpFlag) != 0;
  const uint32_t nlog = static_cast<uint32_t>(a.nlog);
  if (MODE == kColPair && a.dc_nyq_pair == 2 && blk == 0 && sl == 0) {
    // unit 0 of an inverse 2D real column pass: Herm(A) + i Herm(B) for the
    // DC column A (column 0) and the Nyquist column B (column `units`)
    constexpr int R = RA * RB;
    const uint32_t cb = static_cast<uint32_t>(a.units);
    const T half = T(0.5);
#pragma unroll
    for (int j = 0; j < RA; ++j) {
      const uint32_t e = static_cast<uint32_t>(t + RB * j);
      const uint32_t em = e == 0 ? 0u : static_cast<uint32_t>(R) - e;
      const V2<T> va = ldt(src, e * tcnt), vam = ldt(src, em * tcnt);
      const V2<T> vb = ldt(src, cb + e * tcnt), vbm = ldt(src, cb + em * tcnt);
      const V2<T> ha{(va.x + vam.x) * half, (va.y - vam.y) * half};
      const V2<T> hb{(vb.x + vbm.x) * half, (vb.y - vbm.y) * half};
      x[j] = V2<T>{ha.x - hb.y, ha.y + hb.x};
    }
    return;
  }
  // First passes, and those of 64 elements per thread, load without branches.
  // (Later passes read a workspace that the caches hold: the masked loads' waves
  // drift apart, so that loads, arithmetic and stores of a CU's workgroups
  // overlap: 65536 x 16 12.9 us straight, 12.7 masked, R2C of 2^15 x 8 10.8 and 10.4, 155
  // chains, images and volumes 1.5 % in the mean.  Not the tile whose unit 0 is a pair: its lanes left above.)
  const bool straight = RA >= 64 || MODE == kColRealPre || (MODE != kColRealPost && a.p == a.ncol);
  if (straight && !chirp_in && un.whole && !(MODE == kColPair && a.dc_nyq_pair == 2 && blk == 0)) {
    auto load_tile = [&](auto ld) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < RA; ++j) {
        x[j] = ld(src, ia + static_cast<uint32_t>(t + RB * j) * tcnt);
        // 64 loads per thread, each of a row 64 rows further on (2 MB at a 32 KB
        // pitch): the waves keep in step every 16 loads (issue order only, no
        // wait for data), so a CU walks the pages together instead of each wave
        // through its own.  4096-point columns of 4096^2 C2C 73 -> 63 us, the two
        // passes of 2^24 104 + 73 -> 86 + 61 us.
        if constexpr (RA >= 64) {
          if (j % 16 == 15) {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
    };
    if (a.stream & kStreamIn)
      load_tile([](const GlbC<T> *p, uint32_t e) __attribute__((always_inline)) { return ldt_nt<T>(p, e); });
    else
      load_tile([](const GlbC<T> *p, uint32_t e) __attribute__((always_inline)) { return ldt(p, e); });
    return;
  }
  if (chirp_in) {
    // chirp[e] x[e] for e < nlog.  nlog <= M / 2 (M >= 2 nlog - 1 and even), so
    // the upper half of every unit's elements is zero.  Straight-line loads,
    // element 0 standing for those past the end: under a mask each element's
    // chirp was a round trip of its own (first pass of 1 000 003 x 4 40 us).
    const GlbC<T> *chirp = gc<T>(a.chirp);
    constexpr int HA = RA / 2;
    V2<T> ch[HA];
    const int bm = a.src_mode & 3;
#pragma unroll
    for (int j = 0; j < HA; ++j) {
      const uint32_t e = i + static_cast<uint32_t>(t + RB * j) * tcnt;
      ch[j] = ldt(chirp, e < nlog ? e : 0u);
    }
    if (bm == kSrcComplex) {
#pragma unroll
      for (int j = 0; j < HA; ++j) {
        const uint32_t e = i + static_cast<uint32_t>(t + RB * j) * tcnt;
        x[j] = ldt(src, lead + (e < nlog ? e : 0u));
      }
    } else if (bm == kSrcReal) {
      const GlbR<T> *rsrc = gr<T>(a.in) + static_cast<int64_t>(un.bq) * a.bs_in;
#pragma unroll
      for (int j = 0; j < HA; ++j) {
        const uint32_t e = i + static_cast<uint32_t>(t + RB * j) * tcnt;
        x[j] = V2<T>{rsrc[lead + (e < nlog ? e : 0u)], T(0)};
      }
    } else {
      // Hermitian: bins past nlog / 2 are the conjugates of their mirror images,
      // Im of the bins that are their own dropped
#pragma unroll
      for (int j = 0; j < HA; ++j) {
        const uint32_t e = i + static_cast<uint32_t>(t + RB * j) * tcnt;
        const uint32_t el = e < nlog ? e : 0u;
        const bool up = el > nlog / 2;
        V2<T> v = ldt(src, lead + (up ? nlog - el : el));
        v.y = (el == 0 || 2 * el == nlog) ? T(0) : up ? -v.y : v.y;
        x[j] = v;
      }
    }
    const T cs = a.conj_in ? T(-1) : T(1);
#pragma unroll
    for (int j = 0; j < HA; ++j) {
      const uint32_t e = i + static_cast<uint32_t>(t + RB * j) * tcnt;
      const V2<T> v = cmul(V2<T>{x[j].x, x[j].y * cs}, ch[j]);
      const bool in = un.active && e < nlog;
      x[j] = V2<T>{in ? v.x : T(0), in ? v.y : T(0)};
      x[HA + j] = V2<T>{0, 0};
    }
    return;
  }
  // a tile that ends partially: idle slots hold zeros
#pragma unroll
  for (int j = 0; j < RA; ++j) {
    const uint32_t e = ia + static_cast<uint32_t>(t + RB * j) * tcnt;
    x[j] = un.active ? ldt(src, e) : V2<T>{0, 0};
  }
}

// Inter-pass twiddles of the unit's elements: e = t + RB j times w^(e kmul) =
// w^((t + RB j0) kmul) w^(8 RB jh kmul), j = j0 + 8 jh, from the two-level table.
template <typename T, int RA, int RB, bool EXACT>
__device__ __forceinline__ void col_twiddle(const StageArgs &a, uint32_t kmul, int t, V2<T> (&x)[RA]) {
  const GlbC<T> *tw_lo = gc<T>(a.tw_lo);
  const GlbC<T> *tw_hi = gc<T>(a.tw_hi);
  const uint32_t tw_mask = (1u << a.tw_bits) - 1u;
  constexpr int L8 = RA < 8 ? RA : 8;
  constexpr int H8 = (RA + 7) / 8;
  auto tw2 = [&](uint32_t mm) __attribute__((always_inline)) {
    return cmul(ldg(tw_hi + (mm >> a.tw_bits)), ldg(tw_lo + (mm & tw_mask)));
  };
  V2<T> blo[8], shi[8];
  const V2<T> base = tw2(static_cast<uint32_t>(t) * kmul);
  powers<L8, EXACT, T>([&](int q) __attribute__((always_inline)) { return tw2(static_cast<uint32_t>(RB << q) * kmul); }, blo);
  powers<H8, EXACT, T>([&](int q) __attribute__((always_inline)) { return tw2(static_cast<uint32_t>((8 * RB) << q) * kmul); }, shi);
  blo[0] = base;
#pragma unroll
  for (int j = 1; j < L8; ++j) blo[j] = cmul(base, blo[j]);
#pragma unroll
  for (int j = 0; j < RA; ++j) {
    const V2<T> w = (j >= 8) ? cmul(blo[j & 7], shi[j >> 3]) : blo[j];
    x[j] = cmul(x[j], w);
  }
}

// Both stages of the units' R-point transforms and the transpose between
// them: x (elements t + RB j) -> y.  bs: y[0] holds k1 = tid % RA of slot tid / RA
// (two-chunk square instances only), else y[m] holds k1 = t + RB m of slot sl;
// y[m][k2] is output k1 + RA k2.  Earlier reads of the LDS buffer are done.
template <typename T, int C, int RA, int RB, int NCH, bool EXACT>
__device__ __forceinline__ void col_stages(const GlbC<T> *tws, int t, int sl, bool bs, V2<T> (&x)[RA],
                                           V2<T> (&y)[RA / RB][RB]) {
  constexpr int NM = RA / RB;   // stage-B transforms per thread
  constexpr int KC = RA / NCH;  // k1 values per exchange chunk
  static_assert(RA % RB == 0 && RA % NCH == 0 && RB % NCH == 0, "shape");
  constexpr int L8 = RA < 8 ? RA : 8;
  constexpr int H8 = (RA + 7) / 8;
  LdsC<T> *lds = lds_base<T>();
  const int tid = threadIdx.x;
  // ---- stage A (radix RA over j) and the inner twiddles ------------------------
  dft<RA>(x);
  // w_R^(t k1) = lo[k1 mod 8] hi[k1 / 8], straight from the length-R table
  // (t k1 < R): two roundings per twiddle
  V2<T> wlo[8], whi[8];
  powers<L8, EXACT, T>([&](int q) __attribute__((always_inline)) { return ldt(tws, static_cast<uint32_t>(t << q)); }, wlo);
  powers<H8, EXACT, T>([&](int q) __attribute__((always_inline)) { return ldt(tws, static_cast<uint32_t>((t * 8) << q)); }, whi);
#pragma unroll
  for (int j = 1; j < RA; ++j) {
    const V2<T> w = (j >= 8) ? ((j & 7) ? cmul(wlo[j & 7], whi[j >> 3]) : whi[j >> 3]) : wlo[j];
    x[j] = cmul(x[j], w);
  }

  // ---- RA x RB transpose within each unit and stage B (radix RB over t) -------
  if constexpr (NCH == 2 && RA == RB) {
    // Two chunks, each holding half of every unit: entry (k1, tt) travels in
    // chunk c = (tt mod 2) xor (k1 >= H).  Every thread writes H values and
    // reads H values per chunk (the values of its k1 = t of one tt parity),
    // so no thread holds more than RA values at a time; stage B is then
    // radix 2 over the even / odd tt transforms of length H.
    //
    // Stage B runs on (unit slot, k1) = (tid % C, tid / C) for passes that
    // store C-element runs, or (tid / RA, tid % RA) for the first pass of
    // contiguous rows: there 32 consecutive lanes hold consecutive outputs
    // k1 + RA k2 of one unit and store RA-element runs directly.  The row
    // pitch of the chunk buffer keeps either reader at two accesses per bank.
    constexpr int H = RA / 2;
    V2<T> ye[H], yo[H];
    const int pitch = bs ? H * C + 1 : H * C + 8;
    const int rsl = bs ? tid / RA : sl;  // unit slot of this thread's stage-B transform
    const int rk1 = bs ? tid % RA : t;   // and its k1
    const int hw = rk1 / H;
    // odd t write their upper k1 half in chunk 0: swap the halves in
    // registers first (constant indices: a runtime index into x would put the
    // array in scratch memory)
    if (t & 1) {
#pragma unroll
      for (int kk = 0; kk < H; ++kk) {
        const V2<T> tmp = x[kk];
        x[kk] = x[H + kk];
        x[H + kk] = tmp;
      }
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if (c > 0) __syncthreads();  // the previous chunk's reads are done
      const int h = (t & 1) ^ c;    // the k1 half this thread writes in chunk c
#pragma unroll
      for (int kk = 0; kk < H; ++kk) stc(lds + (h * H + kk) * pitch + (t >> 1) * C + sl, x[c * H + kk]);
      __syncthreads();
      const int par = hw ^ c;  // tt parity this thread reads in chunk c
#pragma unroll
      for (int q = 0; q < H; ++q) {
        const V2<T> v = ldc(lds + rk1 * pitch + q * C + rsl);
        if (par) yo[q] = v;
        else ye[q] = v;
      }
    }
    dft<H>(ye);
    dft<H>(yo);
    sfor<H>([&](auto K) __attribute__((always_inline)) {
      constexpr int k2 = decltype(K)::value;
      const V2<T> o = twiddle_ct<k2, RA>(yo[k2]);
      y[0][k2] = cadd(ye[k2], o);
      y[0][k2 + H] = csub(ye[k2], o);
    });
  } else {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      if (c > 0) __syncthreads();  // the previous chunk's reads are done
#pragma unroll
      for (int kk = 0; kk < KC; ++kk) stc(lds + xslot<C, RB>(kk, t, sl), x[c * KC + kk]);
      __syncthreads();
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        const int k1 = t + RB * m;
        if (k1 / KC == c) {
          const int kk = k1 - c * KC;
#pragma unroll
          for (int tt = 0; tt < RB; ++tt) y[m][tt] = ldc(lds + xslot<C, RB>(kk, tt, sl));
        }
      }
    }
#pragma unroll
    for (int m = 0; m < NM; ++m) dft<RB>(y[m]);
  }
}

// Split-spectrum pass of a real transform on the elements m = i + e np of a tile
// of unit pairs: thread t holds e = t + RB q in v[q]; the mirror bin h - m
// (h = np R) is element R - 1 - e of the mirror unit np - i, so v[RA - 1 - q] of thread
// RB - 1 - t in the other half of the tile (unit 0 mirrors e into R - e of itself,
// unit np / 2 into R - 1 - e of itself).  The values change places through LDS in two
// halves; v[q] becomes combine(q, v[q], mirror value, own): own where the bin is
// its own mirror (bins 0 and h / 2, whose mirror value given is v[q] itself).
//
// In a pass of its own the bins are read and written once more (67 MB each way of
// 2^20 x 16 R2C, 22-37 us of 75-93).
template <typename T, int C, int RA, int RB, typename F>
__device__ __forceinline__ void real_partner(uint32_t i, uint32_t np, int t, int sl, V2<T> (&v)[RA], F combine) {
  constexpr int HQ = RA / 2;
  static_assert(RB * C % 32 == 0, "padding");
  LdsC<T> *lds = lds_base<T>();
  const bool own_unit = i == 0 || 2 * i == np;
  const int pt = i != 0 ? RB - 1 - t : t == 0 ? 0 : RB - t;
  const int ps = own_unit ? sl : sl ^ (C / 2);
  const bool wrap = i == 0 && t == 0;  // q mirrors into RA - q
  const int b0 = pt * C + ps;
  const int b1 = wrap ? b0 + RB * C : b0;
  const LdsC<T> *r0 = lds + b0 + (b0 >> 5), *r1 = lds + b1 + (b1 >> 5);
  constexpr int row = RB * C + RB * C / 32;
  V2<T> up[HQ];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    __syncthreads();  // earlier reads of the buffer are done
#pragma unroll
    for (int qq = 0; qq < HQ; ++qq) stc(lds + xslot<C, RB>(qq, t, sl), v[c * HQ + qq]);
    __syncthreads();
    sfor<HQ>([&](auto Q) __attribute__((always_inline)) {
      constexpr int qq = decltype(Q)::value;
      // the first of a half wraps past the buffer: those bins are their own mirror
      const V2<T> m = ldc((qq == 0 ? r0 : r1) + (HQ - 1 - qq) * row);
      if (c == 0) {
        up[qq] = m;
      } else {
        const bool own = qq == 0 && wrap;
        v[qq] = combine(std::integral_constant<int, qq>{}, v[qq], own ? v[qq] : m, own);
        v[HQ + qq] = combine(std::integral_constant<int, HQ + qq>{}, v[HQ + qq], own ? v[HQ + qq] : up[qq], own);
      }
    });
  }
}

// w_n^(i + t np) of the first element of a thread; element t + RB q has
// w_2RA^q times that (n = 2 np RA RB).
template <typename T>
__device__ __forceinline__ V2<T> real_twiddle(const StageArgs &a, uint32_t i, uint32_t np, int t) {
  const uint32_t m = i + static_cast<uint32_t>(t) * np;
  return cmul(ldg(gc<T>(a.tw_rhi) + (m >> a.tw_rbits)), ldg(gc<T>(a.tw_rlo) + (m & ((1u << a.tw_rbits) - 1u))));
}

// Everything after the loads of tile `blk` (x: what col_load gave).
template <typename T, int C, int RA, int RB, int NCH, int MODE>
__device__ __forceinline__ void col_rest(const StageArgs &a, int blk, V2<T> (&x)[RA]) {
  constexpr int R = RA * RB;
  constexpr int NM = RA / RB;   // stage-B transforms per thread
  constexpr int KD = RB / NCH;  // k2 values per block-store chunk
  constexpr int BL = R / NCH;   // block-store chunk length per unit
  constexpr int NT = C * RB;
  static_assert((C & (C - 1)) == 0, "C must be a power of two");
  LdsC<T> *lds = lds_base<T>();
  const int tid = threadIdx.x;
  const int sl = tid % C;
  const int t = tid / C;
  const int64_t u0 = static_cast<int64_t>(blk) * C;
  const ColUnit un = col_unit<C, MODE>(a, blk, sl);
  const bool active = un.active;
  const uint32_t bq = un.bq, i = un.i;
  const bool first = a.p == a.ncol;
  const uint32_t k = i - fdiv(i, a.fd_p) * static_cast<uint32_t>(a.p);
  const uint32_t kt = first ? 0u : fdiv(k, a.fd_ncol);
  const uint32_t tcnt = static_cast<uint32_t>(a.tcnt);
  const uint32_t kmul = kt * static_cast<uint32_t>(a.twp_mult);
  const T scale = static_cast<T>(a.scale);
  const uint32_t j0 = (static_cast<uint32_t>(u0) - bq * tcnt) / 2;  // first pair of a real tile

  // Bluestein chains: the last passes write conj(X bhat) (forward chain) or
  // conj(X) chirp for e < n = nlog (inverse chain)
  const uint32_t nlog = static_cast<uint32_t>(a.nlog);
  const GlbC<T> *chirp = gc<T>(a.chirp);
  // (a product, not a branch, which would wait for the data before the
  // twiddles are on their way; a chirp source is conjugated already)
  const T cs = (a.conj_in && !(MODE == kColBluestein && (a.src_mode & kSrcChirpFlag))) ? T(-1) : T(1);
#pragma unroll
  for (int j = 0; j < RA; ++j) x[j].y *= cs;
  constexpr bool kExact = RA >= 32 || MODE == kColBluestein;
  if constexpr (MODE == kColRealPre) {
    // x[q] = X_m -> conj Z'_m, Z'_m = (X_m + conj X_{h-m}) + i conj(w_n^m) (X_m - conj X_{h-m})
    // (conjugated: the inverse runs as a forward transform); Im of X_0 and X_h dropped
    const V2<T> wb = real_twiddle<T>(a, i, tcnt, t);
    const bool dc = i == 0 && t == 0;
    V2<T> xn{0, 0};  // X_h, which no unit reads
    if (dc) {
      xn.x = ldt(gc<T>(a.in) + static_cast<int64_t>(bq) * a.bs_in, tcnt * static_cast<uint32_t>(R)).x;
      x[0].y = T(0);
    }
    real_partner<T, C, RA, RB>(i, tcnt, t, sl, x, [&](auto Q, V2<T> xk, V2<T> xh, bool own) __attribute__((always_inline)) {
      constexpr int q = decltype(Q)::value;
      if (q == 0 && own) xh = xn;
      const V2<T> c = cconj(xh);
      const V2<T> u = twiddle_ct<q, 2 * RA>(cmul(wb, cconj(csub(xk, c))));  // conj(conj(w) (X_m - c))
      return cconj(cadd(cadd(xk, c), cmul_pi(cconj(u))));
    });
    __syncthreads();  // its reads are done
  }
  if (!first) col_twiddle<T, RA, RB, kExact>(a, kmul, t, x);
  V2<T> y[NM][RB];
  const bool bs = a.block_store != 0;
  col_stages<T, C, RA, RB, NCH, kExact>(gc<T>(a.tw_small), t, sl, bs, x, y);
  if constexpr (NCH == 2 && RA == RB) {
    const int rsl = tid / RA, rk1 = tid % RA;
    if (bs) {
      // unit u0 + rsl owns outputs (u0 + rsl) R + e', e' = rk1 + RA k2
      if (u0 + rsl < a.units) {
        GlbC<T> *dst = gc<T>(a.out) + (MODE == kColRealPre ? static_cast<int64_t>(bq) * a.bs_out : u0 * R);
        const uint32_t us = MODE == kColRealPre ? pair_unit<C>(j0, tcnt, rsl) : static_cast<uint32_t>(rsl);
        const uint32_t o0 = us * static_cast<uint32_t>(R) + static_cast<uint32_t>(rk1);
#pragma unroll
        for (int q = 0; q < RB; ++q) {
          V2<T> v = y[0][q];
          if (a.conj_out) v.y = -v.y;
          if (scale != T(1)) {
            v.x *= scale;
            v.y *= scale;
          }
          stt(dst, o0 + static_cast<uint32_t>(RA * q), v);
        }
      }
      return;
    }
  }

  if constexpr (MODE == kColRealPost) {
    // outputs e = t + RB q (q = m + NM k2) of the chain, Z_m, m = i + e p:
    // X_m = E + w_n^m O, E = (Z_m + conj Z_{h-m}) / 2, O = -i (Z_m - conj Z_{h-m}) / 2
    const uint32_t np = static_cast<uint32_t>(a.p);
    const V2<T> wb = real_twiddle<T>(a, i, np, t);
    V2<T> v[RA];
#pragma unroll
    for (int q = 0; q < RA; ++q) v[q] = y[q % NM][q / NM];
    const V2<T> z0 = v[0];
    const T half = T(0.5);
    real_partner<T, C, RA, RB>(i, np, t, sl, v, [&](auto Q, V2<T> zk, V2<T> zh, bool) __attribute__((always_inline)) {
      constexpr int q = decltype(Q)::value;
      const V2<T> zc = cconj(zh);
      const V2<T> ev{(zk.x + zc.x) * half, (zk.y + zc.y) * half};
      const V2<T> od = cmul_mi(V2<T>{(zk.x - zc.x) * half, (zk.y - zc.y) * half});
      return cadd(ev, twiddle_ct<q, 2 * RA>(cmul(wb, od)));
    });
    GlbC<T> *dst = gc<T>(a.out) + static_cast<int64_t>(bq) * a.bs_out;
    const uint32_t o0 = i + static_cast<uint32_t>(t) * np;
#pragma unroll
    for (int q = 0; q < RA; ++q) stt(dst, o0 + static_cast<uint32_t>(RB * q) * np, v[q]);
    if (i == 0 && t == 0) stt(dst, np * static_cast<uint32_t>(R), V2<T>{z0.x - z0.y, T(0)});
    return;
  }

  auto finish = [&](V2<T> v) __attribute__((always_inline)) {
    if (a.conj_out) v.y = -v.y;
    if (scale != T(1)) {
      v.x *= scale;
      v.y *= scale;
    }
    return v;
  };

  if (a.block_store) {
    // the C units' outputs are one contiguous block of C R elements; each
    // chunk d carries outputs e' = k1 + RA k2 with k2 in [d KD, (d + 1) KD),
    // a contiguous range of BL elements per unit
    // row pitch = 4 (mod 32) entries: the 16 slots of a wavefront's store land
    // on distinct bank octets
    constexpr int LSB = (BL + BL / 32 + 28) / 32 * 32 + 4;
    // (a real tile's units are contiguous rows of their own)
    GlbC<T> *dst = gc<T>(a.out) + (MODE == kColRealPre ? static_cast<int64_t>(bq) * a.bs_out : u0 * R);
    const int64_t total = a.units * static_cast<int64_t>(R);
#pragma unroll
    for (int d = 0; d < NCH; ++d) {
      __syncthreads();  // the exchange (or previous chunk) reads are done
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        const int k1 = t + RB * m;
#pragma unroll
        for (int q = 0; q < KD; ++q) {
          const int e2 = k1 + RA * q;  // e' - d BL
          stc(lds + sl * LSB + e2 + (e2 >> 5), y[m][d * KD + q]);
        }
      }
      __syncthreads();
      constexpr int PER = (C * BL + NT - 1) / NT;
#pragma unroll
      for (int r = 0; r < PER; ++r) {
        const int f = tid + r * NT;
        if (f < C * BL) {
          const int s2 = f / BL, e2 = f - s2 * BL;
          const int64_t us = MODE == kColRealPre ? pair_unit<C>(j0, tcnt, s2) : s2;
          const int64_t g = us * R + d * BL + e2;
          if (MODE == kColRealPre || u0 * R + g < total) stg(dst + g, finish(ldc(lds + s2 * LSB + e2 + (e2 >> 5))));
        }
      }
    }
  } else {
    // forward 2D real column pass with the DC / Nyquist pair in unit 0: its
    // outputs go through LDS so that each thread sees Z_e and Z_-e
    // (workgroup 0 only, uniform over the workgroup)
    const bool unpack = MODE == kColPair && a.dc_nyq_pair == 1 && blk == 0;
    if (unpack) {
      __syncthreads();  // the exchange's reads are done
      if (sl == 0) {
#pragma unroll
        for (int m = 0; m < NM; ++m) {
#pragma unroll
          for (int q = 0; q < RB; ++q) stc(lds + (t + RB * m + RA * q), y[m][q]);
        }
      }
      __syncthreads();
    }
    if (active) {
      GlbC<T> *dst = gc<T>(a.out) + static_cast<int64_t>(bq) * a.bs_out;
      const uint32_t lead = un.dq * static_cast<uint32_t>(a.bs_out);
      const uint32_t o0 = (i - k) * static_cast<uint32_t>(R) + k;
      const uint32_t pp = static_cast<uint32_t>(a.p);
      const GlbC<T> *bhat = gc<T>(a.bhat);
      if (unpack && sl == 0) {
        // unit 0 is column 0 of the single pass (o0 = 0); B goes to column `units`
        const uint32_t cb = static_cast<uint32_t>(a.units);
        const T half = T(0.5);
#pragma unroll
        for (int m = 0; m < NM; ++m) {
#pragma unroll
          for (int q = 0; q < RB; ++q) {
            const int e = t + RB * m + RA * q;
            const V2<T> z = y[m][q];
            const V2<T> zm = ldc(lds + (e == 0 ? 0 : R - e));  // Z_-e (conjugated below)
            const V2<T> va{(z.x + zm.x) * half, (z.y - zm.y) * half};
            const V2<T> vb{(z.y + zm.y) * half, (zm.x - z.x) * half};
            stt(dst, static_cast<uint32_t>(e) * pp, finish(va));
            stt(dst, cb + static_cast<uint32_t>(e) * pp, finish(vb));
          }
        }
      } else {
        // output index of y[m][q] within its sequence, less the lane's o0
        auto rel = [&](int m, int q) __attribute__((always_inline)) {
          return static_cast<uint32_t>(t + RB * m + RA * q) * pp;
        };
        // (table loads ahead of the stores in groups: one by one each would
        // wait for its own round trip)
        constexpr int G = RB < 16 ? RB : 16;
        if (MODE == kColBluestein && (a.dst_mode & kDstPointwiseFlag)) {
#pragma unroll
          for (int m = 0; m < NM; ++m) {
#pragma unroll
            for (int q0 = 0; q0 < RB; q0 += G) {
              V2<T> w[G];
#pragma unroll
              for (int q = 0; q < G; ++q) w[q] = ldt(bhat, o0 + rel(m, q0 + q));
#pragma unroll
              for (int q = 0; q < G; ++q) stt(dst, o0 + rel(m, q0 + q) + lead, cconj(cmul(y[m][q0 + q], w[q])));
            }
          }
        } else if (MODE == kColBluestein && (a.dst_mode & kDstChirpFlag)) {
          // outputs from M / 2 on lie past the user length; a half sink keeps
          // the bins up to nlog / 2, a real one the real parts
          const bool real_out = (a.dst_mode & 3) == kDstReal;
          const uint32_t olim = (a.dst_mode & 3) == kDstHalf ? nlog / 2 + 1 : nlog;
          GlbR<T> *rdst = gr<T>(a.out) + static_cast<int64_t>(bq) * a.bs_out;
          constexpr int HB = RB / 2, GB = HB < G ? HB : G;
#pragma unroll
          for (int m = 0; m < NM; ++m) {
#pragma unroll
            for (int q0 = 0; q0 < HB; q0 += GB) {
              V2<T> w[GB];
#pragma unroll
              for (int q = 0; q < GB; ++q) w[q] = ldt(chirp, min(o0 + rel(m, q0 + q), nlog - 1u));
#pragma unroll
              for (int q = 0; q < GB; ++q) {
                const uint32_t o = o0 + rel(m, q0 + q);
                const V2<T> v = finish(cmul(cconj(y[m][q0 + q]), w[q]));
                if (real_out) {
                  if (o < nlog) rdst[o + lead] = v.x;
                } else if (o < olim) {
                  stt(dst, o + lead, v);
                }
              }
            }
          }
        } else {
          const uint32_t oa = o0 + lead;
          auto store_tile = [&](auto st) __attribute__((always_inline)) {
#pragma unroll
            for (int m = 0; m < NM; ++m) {
#pragma unroll
              for (int q = 0; q < RB; ++q) st(dst, oa + rel(m, q), finish(y[m][q]));
            }
          };
          if (a.stream & kStreamOut)
            store_tile([](GlbC<T> *p, uint32_t e, V2<T> v) __attribute__((always_inline)) { stt_nt<T>(p, e, v); });
          else
            store_tile([](GlbC<T> *p, uint32_t e, V2<T> v) __attribute__((always_inline)) { stt(p, e, v); });
        }
      }
    }
  }
}

// One tile of the middle launch of a two-pass Bluestein convolution M = R0 R
// (R = RA RA): the forward chain's second pass (p = tcnt = R0), conj(X bhat), and
// the inverse chain's first pass, which reads the same R elements i + e R0 and
// writes y[i R + e'].  A square instance leaves its outputs t + RA k2 in the
// thread that transforms the elements t + RA j next, so the product and the second
// transform follow in registers.
template <typename T, int C, int RA, int NCH>
__device__ __forceinline__ void col_conv_body(const StageArgs &a, int blk) {
  constexpr int R = RA * RA;
  const int tid = threadIdx.x;
  const int sl = tid % C;
  const int t = tid / C;
  const int64_t u0 = static_cast<int64_t>(blk) * C;
  const ColUnit un = col_unit<C, kColPlain>(a, blk, sl);
  const uint32_t i = un.i, p = static_cast<uint32_t>(a.p);
  const uint32_t k = i - fdiv(i, a.fd_p) * p;
  V2<T> x[RA], y[1][RA];
  col_load<T, C, RA, RA, kColPlain>(a, blk, x);
  col_twiddle<T, RA, RA, true>(a, k * static_cast<uint32_t>(a.twp_mult), t, x);
  const GlbC<T> *tws = gc<T>(a.tw_small);
  col_stages<T, C, RA, RA, NCH, true>(tws, t, sl, false, x, y);
  const GlbC<T> *bhat = gc<T>(a.bhat);
  constexpr int G = RA < 16 ? RA : 16;
#pragma unroll
  for (int q0 = 0; q0 < RA; q0 += G) {
    V2<T> w[G];
#pragma unroll
    for (int q = 0; q < G; ++q) w[q] = ldt(bhat, i + static_cast<uint32_t>(t + RA * (q0 + q)) * p);
#pragma unroll
    for (int q = 0; q < G; ++q) x[q0 + q] = cconj(cmul(y[0][q0 + q], w[q]));
  }
  __syncthreads();  // the exchange's reads are done
  constexpr bool direct = NCH == 2;  // RA-element runs straight from registers
  col_stages<T, C, RA, RA, NCH, true>(tws, t, sl, direct, x, y);
  // the tile's units own one contiguous block of C R outputs
  GlbC<T> *dst = gc<T>(a.out) + u0 * R;
  const int ns = static_cast<int>(min(static_cast<int64_t>(C), a.units - u0));  // slots with a unit
  if constexpr (direct) {
    const int rsl = tid / RA;
    if (rsl < ns) {
      const uint32_t o0 = static_cast<uint32_t>(rsl * R + tid % RA);
#pragma unroll
      for (int q = 0; q < RA; ++q) stt(dst, o0 + static_cast<uint32_t>(RA * q), y[0][q]);
    }
  } else {
    LdsC<T> *lds = lds_base<T>();
    constexpr int LSB = (R + R / 32 + 28) / 32 * 32 + 4;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RA; ++q) {
      const int e2 = t + RA * q;
      stc(lds + sl * LSB + e2 + (e2 >> 5), y[0][q]);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RA; ++r) {
      const int f = tid + r * (C * RA);
      const int s2 = f / R, e2 = f - s2 * R;
      if (s2 < ns) stt(dst, static_cast<uint32_t>(f), ldc(lds + s2 * LSB + e2 + (e2 >> 5)));
    }
  }
}

// One tile (workgroup `blk` of the launch) of a register-resident pass; every
// one of the C * RB threads of the workgroup must call it (it synchronises).
template <typename T, int C, int RA, int RB, int NCH, int MODE>
__device__ __forceinline__ void col_body(const StageArgs &a, int blk) {
  V2<T> x[RA];
  col_load<T, C, RA, RB, MODE>(a, blk, x);
  col_rest<T, C, RA, RB, NCH, MODE>(a, blk, x);
}

}  // namespace dev
}  // namespace flagfft
