// planner.cpp — decomposition choice (host only).
#include "planner.hpp"

#include "kernels.hpp"

#include <algorithm>
#include <functional>
#include <sstream>
#include <stdexcept>

namespace flagfft {

bool is_prime(int64_t n) {
  if (n < 2) return false;
  if (n % 2 == 0) return n == 2;
  for (int64_t d = 3; d * d <= n; d += 2)
    if (n % d == 0) return false;
  return true;
}

namespace {

int64_t modpow(int64_t b, int64_t e, int64_t m) {
  __int128 r = 1, x = b % m;
  while (e > 0) {
    if (e & 1) r = (r * x) % m;
    x = (x * x) % m;
    e >>= 1;
  }
  return static_cast<int64_t>(r);
}

std::vector<int64_t> prime_factors(int64_t n) {
  std::vector<int64_t> f;
  for (int64_t d = 2; d * d <= n; ++d)
    while (n % d == 0) {
      f.push_back(d);
      n /= d;
    }
  if (n > 1) f.push_back(n);
  return f;
}

std::string join(const std::vector<int> &v, const char *sep) {
  std::ostringstream o;
  for (size_t i = 0; i < v.size(); ++i) o << (i ? sep : "") << v[i];
  return o.str();
}

std::string join64(const std::vector<int64_t> &v, const char *sep) {
  std::ostringstream o;
  for (size_t i = 0; i < v.size(); ++i) o << (i ? sep : "") << v[i];
  return o.str();
}

}  // namespace

// Smallest primitive root, as src/plan/rader_utils.cpp:55-77 chooses it.
int64_t primitive_root(int64_t p) {
  if (!is_prime(p)) return -1;
  if (p == 2) return 1;
  std::vector<int64_t> f = prime_factors(p - 1);
  f.erase(std::unique(f.begin(), f.end()), f.end());
  for (int64_t g = 2; g < p; ++g) {
    bool ok = true;
    for (int64_t q : f)
      if (modpow(g, (p - 1) / q, p) == 1) {
        ok = false;
        break;
      }
    if (ok) return g;
  }
  return -1;
}

bool smooth13(int64_t n) {
  if (n < 1) return false;
  for (int64_t p : {2, 3, 5, 7, 11, 13})
    while (n % p == 0) n /= p;
  return n == 1;
}

// Lengths whose prime factors all have a radix codelet: 2, 3, 5, 7, 11, 13,
// 17, 19 (the reference's supported radices, src/utils/include/flagfft/base.hpp:47).
bool smooth19(int64_t n) {
  if (n < 1) return false;
  for (int64_t p : {2, 3, 5, 7, 11, 13, 17, 19})
    while (n % p == 0) n /= p;
  return n == 1;
}

// First-fit-decreasing packing of the prime factors into radices <= 16;
// the primes 17 and 19 are radices of their own.
bool radix_factor(int64_t n, std::vector<int> &out) {
  out.clear();
  if (n < 1) return false;
  if (n == 1) return true;
  std::vector<int64_t> f = prime_factors(n);
  for (int64_t p : f)
    if (p > 19) return false;
  std::sort(f.begin(), f.end(), std::greater<int64_t>());
  std::vector<int> bins;
  for (int64_t p : f) {
    bool placed = false;
    for (int &b : bins)
      if (b * p <= 16) {
        b *= static_cast<int>(p);
        placed = true;
        break;
      }
    if (!placed) bins.push_back(static_cast<int>(p));
  }
  std::sort(bins.begin(), bins.end(), std::greater<int>());
  out = bins;
  return true;
}

bool passes_specialised(const std::vector<int64_t> &passes, bool fast_only) {
  std::vector<int> rad;
  for (int64_t r : passes) {
    if (!radix_factor(r, rad)) return false;
    const int id = stage_kernel_id(rad);
    if (id < 0 || (fast_only && !stage_kernel_fast(id))) return false;
  }
  return true;
}

int64_t leaf_max(const PlanOptions &o, Prec p) { return p == Prec::F32 ? o.leaf_max_f32 : o.leaf_max_f64; }
int64_t pass_max(const PlanOptions &o, Prec p) { return p == Prec::F32 ? o.pass_max_f32 : o.pass_max_f64; }

namespace {

// All splits of n into k factors (non-increasing), each <= cap and radix-factorable.
void enum_splits(int64_t n, int k, int64_t cap, int64_t hi, std::vector<int64_t> &cur,
                 std::vector<std::vector<int64_t>> &out) {
  std::vector<int> tmp;
  if (k == 1) {
    if (n <= cap && n <= hi && n >= 2 && radix_factor(n, tmp)) {
      cur.push_back(n);
      out.push_back(cur);
      cur.pop_back();
    }
    return;
  }
  for (int64_t d = std::min(cap, hi); d >= 2; --d) {
    if (n % d != 0 || !radix_factor(d, tmp)) continue;
    cur.push_back(d);
    enum_splits(n / d, k - 1, cap, d, cur, out);
    cur.pop_back();
  }
}

// Split n into k passes.  Prefer splits whose every pass has a specialised
// kernel, then the one with the largest smallest factor (fewest HBM round
// trips per element are equal for a fixed k; balance keeps every pass's
// workgroups full).
bool split_passes(int64_t n, int k, int64_t cap, std::vector<int64_t> &best) {
  std::vector<std::vector<int64_t>> all;
  std::vector<int64_t> cur;
  enum_splits(n, k, cap, cap, cur, all);
  if (all.empty()) return false;
  auto score = [](const std::vector<int64_t> &v) {
    return std::make_pair(passes_specialised(v) ? 1 : 0, *std::min_element(v.begin(), v.end()));
  };
  const std::vector<int64_t> *b = &all[0];
  for (const auto &v : all)
    if (score(v) > score(*b)) b = &v;
  best = *b;
  return true;
}

// Row-segment bytes of the widest specialised column super-stage for a radix
// sequence (adjacent columns per workgroup x element bytes); 0 if none.
int column_segment_bytes(const std::vector<int> &rad, Prec p) {
  for (int units : {64, 32, 16, 8, 4, 2, 1})
    if (stage_kernel_id(rad, p == Prec::F64, units) >= 0) return units * elem_bytes(p);
  return 0;
}

// Relative time of one HBM sweep by a pass of super-radix r: the inverse of
// its measured rate on MI355X (TB/s of read + write bytes).  Register-resident
// two-stage passes run at 3.8 (first pass, from uncached input) to 4.6 with
// row segments of 128 bytes or more, 3.0 to 4.2 with 64;
// LDS super-stages at 2.2 to 3.5 by the row-segment bytes their tile reads;
// the run-time-radix pass at about 1.1.
// tcnt: units per sequence (n / r).  A register-resident pass whose tiles do
// not divide them runs all the same, its tiles crossing sequence ends, but is
// not priced as one: 5- and 10-smooth lengths keep their chains of 25- to
// 1000-point passes (250000 as [125, 125, 16] would take 28 us against 32 for
// [100, 100, 25]).  Three things depend on the size of the whole transform:
//   * the 4-unit FP64 tile counts up to 24 MiB (150528 x 6 as [588, 256] 31 us, [512,
//     294] 50; but 3763200, whose 14700 256-point units only it divides, as [588, 256,
//     25] 190, [160, 160, 147] 127);
//   * FP64 run-time-radix passes of 512 to 1023 points, whose tiles fill a CU's LDS
//     with one workgroup, are slower past 64 MiB (294912 x 28 as [576, 512] 265 us,
//     [1152, 256] 186; x 7, 33 MB, 56 and 69);
//   * FP32 ones over 2048 points, a workgroup per unit, once a CU has more than one, to
//     20 MiB (150528 x 4 / 5 / 13 as [2352, 64], 256 / 320 / 832 units, 22 / 36 / 66 us, as
//     [512, 294] 28 / 28 / 46; 291600 x 2 as [2160, 135], 270 units, 41, [2916, 100], 200,
//     25.5, [729, 400] 25.3; 602112 x 13, 63 MB, as [2352, 256] 178, [1024, 588] 241).
double pass_time(int64_t r, Prec p, bool first, const PlanOptions &o, int64_t tcnt) {
  std::vector<int> rad;
  if (o.generic_kernels) {
    // persistent-queue plans: register-resident queue instances, else the run-time-radix pass
    return (o.queue_form && col_queue_kernel_id(r, p == Prec::F64) >= 0) ? 1.0 / 4.0 : 1.0 / 1.1;
  }
  const bool dbl = p == Prec::F64;
  const int64_t bytes = r * tcnt * elem_bytes(p) * o.nseq;
  auto up_to = [&](int64_t mib) { return o.nseq > 0 && bytes <= mib << 20; };
  if (o.stage_form != 2 && col_kernel_id(r, dbl, 0) >= 0 && col_tiles_divide(r, dbl, tcnt, dbl && up_to(24) ? 4 : 8)) {
    // 64-byte segments (the 4096-point instance: 8 units of 32 KiB in one
    // workgroup) run at 3.0 / 4.2, the 2048-point FP32 instance (one workgroup
    // per CU, as that one) at 3.1 / 4.1
    if (col_run_bytes(r, p == Prec::F64, first) < 128) return first ? 1.0 / 3.0 : 1.0 / 4.2;
    if (r == 2048) return first ? 1.0 / 3.1 : 1.0 / 4.1;
    // the 512-point FP64 instance runs a little slower than its neighbours (2^18 points
    // x 1 / 8 / 32 as [1024, 256] 15.2 / 31.1 / 98 us, as [512, 512] 16.7 / 34.3 / 113; the
    // 2^19-point real rows that have them 16-25 % more)
    if (r == 512 && p == Prec::F64) return first ? 1.03 / 3.8 : 1.03 / 4.6;
    return first ? 1.0 / 3.8 : 1.0 / 4.6;
  }
  if (radix_factor(r, rad)) {
    const int seg = column_segment_bytes(rad, p);
    if (seg >= 128) return 1.0 / 3.5;
    if (seg >= 64) return 1.0 / 3.0;
    if (seg > 0) return 1.0 / 2.2;
  }
  if (dbl && !up_to(64) && r >= 512 && r < 1024) return 1.0 / 0.85;
  if (!dbl && tcnt * o.nseq > 256 && up_to(20) && r > 2048) return 1.0;
  return 1.0 / 1.1;
}

// The split of n into 2-4 passes with the least total pass time; near ties
// (2 %) go to fewer passes, then to the larger smallest factor.
bool cheapest_split(int64_t n, Prec p, const PlanOptions &o, std::vector<int64_t> &best) {
  // the super-radices that may take part, in falling order, each priced once
  // as a first and as a later pass
  struct Radix {
    int64_t r;
    double first, later;
  };
  std::vector<Radix> rs;
  std::vector<int> tmp;
  for (int64_t d = std::min(pass_max(o, p), n); d >= 2; --d)
    if (n % d == 0 && radix_factor(d, tmp)) rs.push_back({d, pass_time(d, p, true, o, n / d), pass_time(d, p, false, o, n / d)});
  double best_t = 0.0;
  bool have = false;
  std::vector<int64_t> cur;
  std::function<void(int64_t, int, size_t, double)> rec = [&](int64_t rest, int k, size_t from, double tt) {
    for (size_t i = from; i < rs.size(); ++i) {
      const Radix &x = rs[i];
      if (rest % x.r != 0 || (k == 1 && x.r != rest)) continue;
      const double t2 = tt + (cur.empty() ? x.first : x.later);
      cur.push_back(x.r);
      if (k > 1) {
        rec(rest / x.r, k - 1, i, t2);
      } else {
        const bool better = !have || t2 < best_t * 0.98 ||
                            (t2 <= best_t * 1.02 && cur.size() == best.size() &&
                             *std::min_element(cur.begin(), cur.end()) > *std::min_element(best.begin(), best.end()));
        if (better) {
          best = cur;
          best_t = t2;
          have = true;
        }
      }
      cur.pop_back();
    }
  };
  for (int k = 2; k <= 4; ++k) rec(n, k, 0, 0.0);
  return have;
}

void chain_core(int64_t n, const std::vector<int64_t> &passes, Core &c) {
  c.kind = CoreKind::MultiPass;
  c.n = n;
  c.passes = passes;
  c.pass_radices.clear();
  for (int64_t r : passes) {
    std::vector<int> rad;
    radix_factor(r, rad);
    c.pass_radices.push_back(rad);
  }
}

// Relative time per element of the convolution pass of super-radix r: its
// sweep and two transforms; 0 if no kernel.  Square register-resident
// instances run at about 3.3 TB/s (4096 points: 1.9), LDS super-stages at 2.2,
// their 5- and 10-smooth instances at 0.9.
double conv_time(int64_t r, Prec p, const PlanOptions &o) {
  if (o.stage_form != 2 && o.forced_units == 0 && col_conv_kernel_id(r, p == Prec::F64, 0) >= 0)
    return r >= 4096 ? 1.0 / 1.9 : 1.0 / 3.3;
  std::vector<int> rad;
  if (!radix_factor(r, rad)) return 0.0;
  const int id = stage_kernel_id(rad);
  return id < 0 ? 0.0 : stage_kernel_fast(id) ? 1.0 / 2.2 : 1.0 / 0.9;
}

// Two-pass Bluestein convolutions M = R0 R1 in three launches, over the
// super-radices with a compiled kernel, by the time of the launches (the outer
// ones read or write the user's n <= M / 2 elements on one side).
class ConvSplits {
 public:
  ConvSplits(Prec p, const PlanOptions &o) : eb_(elem_bytes(p)), o_(o) {
    const int64_t cap = pass_max(o, p);
    const bool col_ok = o.stage_form != 2 && o.forced_units == 0;
    std::vector<int64_t> all = stage_kernel_radices();
    for (int64_t r : col_kernel_radices(p == Prec::F64)) all.push_back(r);
    std::sort(all.begin(), all.end(), std::greater<int64_t>());
    all.erase(std::unique(all.begin(), all.end()), all.end());
    for (int64_t r : all) {
      std::vector<int> rad;
      if (r > cap || !radix_factor(r, rad)) continue;
      const int sid = stage_kernel_id(rad);
      Radix x{r, 0.0, conv_time(r, p, o), sid >= 0 && stage_kernel_fast(sid)};
      if (col_ok && col_kernel_id(r, p == Prec::F64, 0) >= 0)
        x.outer = pass_time(r, p, true, o, 0) + pass_time(r, p, false, o, 0);
      else if (sid >= 0)
        x.outer = 2.0 / (stage_kernel_fast(sid) ? 2.6 : 1.2);  // an LDS super-stage with the chirp at either end
      if (x.outer > 0.0 || x.conv > 0.0) rs_.push_back(x);
    }
  }
  // The split of the cheapest M = R0 R1 in [lo, hi] (false: none).  The chain has two
  // workspaces of M elements per sequence, and the cheapest M is up to half longer
  // than the shortest of fast super-radices (48197 points: 98415 = 729 x 135, 131072 =
  // 512 x 256).  Two plans take the workspace into account:
  //   * C2C plans that the scratch array of flagfftxExecC2CNoAlloc holds with the
  //     shortest M take one that fits (49133 points x 38: 98415, 60 MB of 67; 131072
  //     would need 80);
  //   * least_ws: none longer than the shortest.
  bool best(int64_t lo, int64_t hi, std::vector<int64_t> &split) const {
    int64_t shortest = hi;
    for (const Radix &a : rs_)
      for (const Radix &b : rs_)
        if (a.fast && b.fast && a.r * b.r >= lo) shortest = std::min(shortest, a.r * b.r);
    if (!cheapest(lo, o_.least_ws ? shortest : hi, split)) return false;
    // (workspaces lie at 256-byte steps of the array)
    const int64_t fit = o_.scratch_fit && o_.nseq > 0 ? kScratchBytes / 2 / 256 * 256 / eb_ / o_.nseq : 0;
    std::vector<int64_t> s;
    if (split[0] * split[1] > fit && shortest <= fit && cheapest(lo, fit, s)) split = s;
    return true;
  }

 private:
  bool cheapest(int64_t lo, int64_t hi, std::vector<int64_t> &split) const {
    double best_t = 0.0;
    for (const Radix &x1 : rs_) {
      if (x1.conv == 0.0) continue;
      for (const Radix &x0 : rs_) {
        const int64_t M = x0.r * x1.r;
        if (x0.outer == 0.0 || M < lo || M > hi) continue;
        const double tt = (0.75 * x0.outer + x1.conv) * static_cast<double>(M);
        if (best_t == 0.0 || tt < best_t * 0.98 ||
            (tt <= best_t * 1.02 && std::min(x0.r, x1.r) > std::min(split[0], split[1]))) {
          split = {x0.r, x1.r};
          best_t = tt;
        }
      }
    }
    return best_t > 0.0;
  }

  struct Radix {
    int64_t r;
    double outer, conv;  // time as R0 / as R1, 0: no kernel
    bool fast;           // stage_kernel_fast
  };
  std::vector<Radix> rs_;
  int eb_;
  PlanOptions o_;
};

bool multipass_core(int64_t n, Prec p, const PlanOptions &o, Core &c, bool by_cost = false) {
  std::vector<int64_t> passes;
  const int64_t cap = pass_max(o, p);
  bool ok = false;
  if (!o.forced_passes.empty()) {
    int64_t prod = 1;
    bool valid = true;
    std::vector<int> tmp;
    for (int64_t r : o.forced_passes) {
      prod *= r;
      valid = valid && r >= 2 && r <= leaf_max(o, p) && radix_factor(r, tmp);
    }
    if (valid && prod == n) {
      passes = o.forced_passes;
      ok = true;
    }
  }
  if (!ok && by_cost) ok = cheapest_split(n, p, o, passes);
  for (int k = 2; !ok && k <= 4; ++k) ok = split_passes(n, k, cap, passes);
  if (!ok) return false;
  chain_core(n, passes, c);
  return true;
}

int rader_lds_bytes(int64_t p, Prec prec) {
  const int64_t m = p - 1;
  return static_cast<int>((lds_pad(static_cast<int>(p)) + 1 + lds_pad(static_cast<int>(m)) + 1 + 1) *
                          elem_bytes(prec));
}

}  // namespace

bool conv_passes_compiled(int64_t r0, int64_t r1, Prec p, const PlanOptions &o) {
  std::vector<int> rad;
  if (!radix_factor(r0, rad)) return false;
  const bool col = o.stage_form != 2 && o.forced_units == 0 && col_kernel_id(r0, p == Prec::F64, 0) >= 0;
  return (col || stage_kernel_id(rad) >= 0) && conv_time(r1, p, o) > 0.0;
}

Core plan_core(int64_t n, Prec p, const PlanOptions &o) {
  if (n < 1) throw std::invalid_argument("transform length must be positive");
  Core c;
  c.n = n;
  std::vector<int> rad;
  const int64_t lmax = leaf_max(o, p);
  // an explicit super-radix split of exactly n overrides the single pass
  int64_t forced_prod = o.forced_passes.size() >= 2 ? 1 : 0;
  for (int64_t r : o.forced_passes) forced_prod *= r;
  bool leaf = n <= lmax && radix_factor(n, rad) && forced_prod != n;
  if (!leaf && !o.generic_kernels && o.forced_passes.empty() && n <= 32768 && radix_factor(n, rad) &&
      leaf_kernel_id(rad) >= 0 &&
      static_cast<int64_t>(lds_pad(static_cast<int>(n) - 1) + 2) * elem_bytes(p) <= o.lds_cap_bytes) {
    // a specialised instance holding the whole sequence in LDS: one HBM round
    // trip instead of two (one workgroup per sequence)
    leaf = true;
  }
  if (leaf) {
    c.kind = CoreKind::Leaf;
    if (!o.forced_radices.empty()) {
      int64_t prod = 1;
      for (int r : o.forced_radices) prod *= r;
      bool valid = prod == n;
      for (int r : o.forced_radices) valid = valid && r >= 2 && (r <= 17 || r == 19);
      if (valid) rad = o.forced_radices;
    }
    c.radices = rad;
    return c;
  }
  if (is_prime(n) && n > 16) {
    const int64_t m = n - 1;
    if (m <= lmax && radix_factor(m, rad) && rader_lds_bytes(n, p) <= o.lds_cap_bytes) {
      c.kind = CoreKind::Rader;
      c.m = m;
      c.root = primitive_root(n);
      c.radices = rad;
      return c;
    }
  }
  if (smooth19(n) && multipass_core(n, p, o, c, true)) return c;
  // Bluestein over a 13-smooth convolution length M >= 2n-1: the first that
  // fits one LDS pass (the whole convolution is one launch), else the two-pass M
  // up to twice the minimum with the cheapest three launches (ConvSplits).
  // Lengths past those, explicit splits and persistent-queue plans weigh every
  // M by its HBM sweeps: M x passes, x 2.5 when a pass has no fast specialised
  // kernel (the run-time-radix pass and the 5- / 10-smooth instances run
  // about that much slower than the power-of-two passes).
  Core best;
  double best_cost = 0.0;
  bool have = false;
  const int64_t m0 = 2 * n - 1;
  if (m0 > lmax && o.forced_passes.empty()) {
    // whole convolution in LDS by a specialised instance: one launch (the
    // two-halves instances hold M / 2 at a time)
    const BluesteinLdsShape *pick = nullptr;
    const std::vector<BluesteinLdsShape> cands = bluestein_lds_candidates(p == Prec::F64);
    for (const BluesteinLdsShape &sh : cands)
      if (sh.m >= m0 && sh.m <= 2 * m0 && (pick == nullptr || sh.m < pick->m)) pick = &sh;
    if (pick != nullptr) {
      c.kind = CoreKind::Bluestein;
      c.m = pick->m;
      c.radices = pick->radices;
      c.conv.reset();
      c.lds_conv = true;
      c.lds_halves = pick->halves;
      return c;
    }
  }
  std::vector<int64_t> split;
  if (m0 > lmax && o.forced_passes.empty() && !o.generic_kernels && ConvSplits(p, o).best(m0, 2 * m0 + 64, split)) {
    c.kind = CoreKind::Bluestein;
    c.m = split[0] * split[1];
    c.radices.clear();
    c.conv = std::make_shared<Core>();
    chain_core(c.m, split, *c.conv);
    return c;
  }
  for (int64_t M = m0;; ++M) {
    if (have && static_cast<double>(M) >= best_cost) break;
    if (M > 2 * m0 + 64) {
      if (have) break;
      if (M > 64 * n + 1024) throw std::runtime_error("no Bluestein convolution length found");
    }
    if (!smooth13(M)) continue;
    if (M <= lmax && radix_factor(M, rad)) {
      c.kind = CoreKind::Bluestein;
      c.m = M;
      c.radices = rad;
      c.conv.reset();
      return c;
    }
    Core sub;
    if (!multipass_core(M, p, o, sub, o.queue_form)) continue;
    if (!o.forced_passes.empty()) {
      best = sub;
      have = true;
      break;
    }
    const double cost = static_cast<double>(M) * static_cast<double>(sub.passes.size()) / 2.0 *
                        (passes_specialised(sub.passes, true) ? 1.0 : 2.5);
    if (!have || cost < best_cost) {
      best = sub;
      best_cost = cost;
      have = true;
    }
  }
  c.kind = CoreKind::Bluestein;
  c.m = best.n;
  c.radices.clear();
  c.conv = std::make_shared<Core>(best);
  return c;
}

std::string Core::describe(int indent) const {
  std::ostringstream o;
  std::string pad(static_cast<size_t>(indent), ' ');
  switch (kind) {
    case CoreKind::Leaf:
      o << pad << "Leaf(n=" << n << ", radices=[" << join(radices, ",") << "], passes=1)";
      break;
    case CoreKind::MultiPass:
      o << pad << "MultiPassStockham(n=" << n << ", super_radices=[" << join64(passes, ",") << "], passes="
        << passes.size() << ")";
      for (size_t i = 0; i < passes.size(); ++i)
        o << "\n" << pad << "  pass" << i << ": R=" << passes[i] << " radices=[" << join(pass_radices[i], ",") << "]";
      break;
    case CoreKind::Rader:
      o << pad << "Rader(p=" << n << ", root=" << root << ", conv_length=" << m << ", fused=1)\n"
        << pad << "  conv: Leaf(n=" << m << ", radices=[" << join(radices, ",") << "])";
      break;
    case CoreKind::MatrixCore:
      o << pad << "MatrixCoreSplit(n=" << n << ", factors=[" << join(radices, ",") << "], operands="
        << (compute == 2 ? "fp16" : "bf16") << " hi+lo, products=3, accumulate=fp32)";
      break;
    case CoreKind::Bluestein:
      o << pad << "Bluestein(n=" << n << ", conv_length=" << m << ", fused=" << (conv ? 0 : 1)
        << (lds_conv ? ", lds_resident=1" : "") << (lds_halves ? ", halves=1" : "") << ")\n";
      if (conv)
        o << conv->describe(indent + 2);
      else if (lds_halves)
        o << pad << "  conv: Leaf(n=" << m << ", radices=[2," << join(radices, ",") << "], in LDS: two halves of "
          << m / 2 << ")";
      else
        o << pad << "  conv: Leaf(n=" << m << ", radices=[" << join(radices, ",") << "])";
      break;
  }
  return o.str();
}

std::string Plan1D::describe(int indent) const {
  std::ostringstream o;
  std::string pad(static_cast<size_t>(indent), ' ');
  const char *form = "";
  switch (real_form) {
    case RealForm::None: form = "Complex"; break;
    case RealForm::EvenFused: form = "RealEvenFused"; break;
    case RealForm::EvenMulti: form = "RealEvenSplitPass"; break;
    case RealForm::Full: form = "RealPromoted"; break;
  }
  o << pad << form << "(n=" << n << (real_fwd ? ", R2C" : "") << (real_inv ? ", C2R" : "") << ")\n"
    << core.describe(indent + 2);
  return o.str();
}

namespace {

Plan1D plan_1d(int64_t n, bool real_fwd, bool real_inv, Prec p, const PlanOptions &o) {
  Plan1D pl;
  pl.n = n;
  pl.real_fwd = real_fwd;
  pl.real_inv = real_inv;
  if (!real_fwd && !real_inv) {
    pl.real_form = RealForm::None;
    pl.core = plan_core(n, p, o);
    return pl;
  }
  if (n % 2 == 0 && n >= 2) {
    // half-length complex core, pack / unpack fused (single pass) or as a
    // split-spectrum pass beside the core (any other core kind)
    Core half = plan_core(n / 2, p, o);
    pl.real_form = half.kind == CoreKind::Leaf ? RealForm::EvenFused : RealForm::EvenMulti;
    pl.core = half;
    return pl;
  }
  pl.real_form = RealForm::Full;
  pl.core = plan_core(n, p, o);
  return pl;
}

// A column super-stage reads row segments of (adjacent columns per
// workgroup) x (element bytes).  When the single pass's widest specialised
// tile gives segments under 64 B (a long column filling the LDS with few
// columns), two passes of wide tiles move the data twice at full segment
// width and win (4096-point FP32 columns: 66 us against 108 us per
// 2049 x 4096 half spectrum).
// ncol columns per transform, nseq transforms.
void widen_columns(Plan1D &cols, Prec prec, const PlanOptions &o, int64_t ncol, int64_t nseq) {
  const bool tuned = !o.forced_passes.empty() || !o.forced_radices.empty() || o.forced_units != 0 || o.generic_kernels;
  if (tuned || cols.core.kind != CoreKind::Leaf) return;
  // a register-resident instance of the whole column length reads 64-byte
  // segments or more in one pass (4096-point FP32 columns: 75 us against
  // 95 us for two 64-point passes), when its workgroups (one per CU) fill the
  // 256 CUs in whole rounds (2049 half-spectrum columns are 257 tiles: the
  // last one would run alone, 228 against 173 us for the 4096^2 R2C->C2R
  // step).  Tiles may cross the ends of transforms (16 x 4096 x 500 R2C, whose 251
  // columns 8 units do not divide: 310 us as two passes, 265 so)
  const int run = o.stage_form != 2 ? col_run_bytes(cols.n, prec == Prec::F64, false) : 0;
  if (run >= 64) {
    constexpr int64_t kCus = 256;
    const int64_t c = run / elem_bytes(prec);
    const int64_t tiles = (ncol * nseq + c - 1) / c;
    const int64_t rounds = (tiles + kCus - 1) / kCus;
    if (4 * tiles >= 3 * rounds * kCus) return;
  }
  // (no LDS super-stage instance for the whole column either: the
  // run-time-radix pass would read it one element per column)
  const int seg = column_segment_bytes(cols.core.radices, prec);
  Core mc;
  if (seg >= 64 || !split_passes(cols.n, 2, pass_max(o, prec), mc.passes)) return;
  for (int64_t r : mc.passes) {
    std::vector<int> rad;
    if (!radix_factor(r, rad) || column_segment_bytes(rad, prec) < 64) return;
    mc.pass_radices.push_back(rad);
  }
  mc.kind = CoreKind::MultiPass;
  mc.n = cols.n;
  cols.core = mc;
}

}  // namespace

PlanTree plan_tree(const PlanDesc &d, const PlanOptions &o) {
  PlanTree t;
  t.desc = d;
  if (d.compute != 0) {
    if (d.rank != 1 || d.real_fwd || d.real_inv || d.prec != Prec::F32 || d.n0 != 1024)
      throw std::invalid_argument("matrix-core compute modes cover C2C n=1024 only");
    t.rows.n = d.n0;
    t.rows.real_form = RealForm::None;
    t.rows.core.kind = CoreKind::MatrixCore;
    t.rows.core.n = d.n0;
    t.rows.core.radices = {32, 32};
    t.rows.core.compute = d.compute;
    return t;
  }
  auto of = [&](int64_t nseq) {
    PlanOptions a = o;
    a.nseq = nseq;
    a.scratch_fit = d.prec == Prec::F32 && !d.real_fwd && !d.real_inv;
    return a;
  };
  auto half_len = [&](int64_t n) { return d.real_fwd || d.real_inv ? n / 2 + 1 : n; };
  if (d.rank == 1) {
    t.rows = plan_1d(d.n0, d.real_fwd, d.real_inv, d.prec, of(d.batch));
  } else if (d.rank == 2) {
    t.rows = plan_1d(d.n1, d.real_fwd, d.real_inv, d.prec, of(d.batch * d.n0));
    t.cols = plan_1d(d.n0, false, false, d.prec, of(d.batch * half_len(d.n1)));
    const bool half = d.real_fwd || d.real_inv;
    // one real transform whose n1 / 2 + 1 half-spectrum columns take two
    // passes only because the last tile would run alone: the DC and Nyquist
    // columns (both real on the real side) share a unit of the single pass
    // (4096^2 R2C: one 41-43 us column pass instead of two of 24-25 us)
    if (half && d.batch == 1 && d.n1 % 2 == 0 && !o.generic_kernels && t.rows.real_form == RealForm::EvenFused &&
        leaf_kernel_id(t.rows.core.radices) >= 0 && t.cols.core.kind == CoreKind::Leaf &&
        col_pair_kernel_id(d.n0, d.prec == Prec::F64) >= 0) {
      Plan1D split = t.cols, single = t.cols;
      widen_columns(split, d.prec, o, d.n1 / 2 + 1, 1);
      widen_columns(single, d.prec, o, d.n1 / 2, 1);
      t.dc_nyq_pair = split.core.kind != CoreKind::Leaf && single.core.kind == CoreKind::Leaf;
    }
    if (!t.dc_nyq_pair) widen_columns(t.cols, d.prec, o, half ? d.n1 / 2 + 1 : d.n1, d.batch);
  } else {
    const int64_t n2c = half_len(d.n2);
    t.rows = plan_1d(d.n2, d.real_fwd, d.real_inv, d.prec, of(d.batch * d.n0 * d.n1));
    t.mid = plan_1d(d.n1, false, false, d.prec, of(d.batch * d.n0 * n2c));
    t.cols = plan_1d(d.n0, false, false, d.prec, of(d.batch * d.n1 * n2c));
    widen_columns(t.mid, d.prec, o, n2c, d.n0 * d.batch);
    widen_columns(t.cols, d.prec, o, d.n1 * n2c, d.batch);
  }
  return t;
}

std::string PlanTree::describe() const {
  std::ostringstream o;
  o << "=== FlagFFT Plan (gfx950) ===\n";
  o << "rank=" << desc.rank << " n=[" << desc.n0;
  if (desc.rank >= 2) o << "," << desc.n1;
  if (desc.rank == 3) o << "," << desc.n2;
  o << "] batch=" << desc.batch << " type=" << desc.type << " precision=" << (desc.prec == Prec::F32 ? "fp32" : "fp64")
    << "\n\n-- Plan tree --\n";
  if (desc.rank == 1) {
    o << rows.describe(0) << "\n";
  } else if (desc.rank == 2) {
    o << "TwoDim(n0=" << desc.n0 << ", n1=" << desc.n1 << ", order=rows-then-columns, column_pass=strided-tile"
      << (dc_nyq_pair ? ", dc_nyquist_pair" : "") << ")\n";
    o << "  rows (axis 1):\n" << rows.describe(4) << "\n";
    o << "  columns (axis 0):\n" << cols.describe(4) << "\n";
  } else {
    o << "ThreeDim(n0=" << desc.n0 << ", n1=" << desc.n1 << ", n2=" << desc.n2
      << ", order=rows-then-axis1-then-axis0, column_pass=strided-tile)\n";
    o << "  rows (axis 2):\n" << rows.describe(4) << "\n";
    o << "  columns (axis 1):\n" << mid.describe(4) << "\n";
    o << "  columns (axis 0):\n" << cols.describe(4) << "\n";
  }
  return o.str();
}

}  // namespace flagfft
