// MAS-preconditioned CG in one launch per solve with one exchange between
// workgroups per iteration (mas_cg_solver.cu:193-311; the MAS preconditioner
// of mas_preconditioner.cu:601-728).
//
// k_pcg_persistent needs two: the dot product p.q and the coarse sums before
// alpha, then z's halo, the coarse corrections and r.z before beta.  What
// the second one carries is linear in alpha, so here it travels with the
// first.  With M0 the level-0 (bank) part of the preconditioner and
// w = M0 q, known inside a workgroup as banks do not straddle workgroups,
//   z0 after the step  = M0 r - alpha w
//   r.z0 after the step = r.z0 - 2 alpha r.w + alpha^2 q.w
//   r.r after the step  = r.r - 2 alpha r.q + alpha^2 q.q
// A workgroup publishes M0 r and w of the slots its neighbours read, the
// level-1 sums of q and seven dot products; M0 r, r.z0 and r.r are formed
// from r itself in every iteration, so that no error accumulates in them.  What
// is carried from one iteration to the next is r itself, as in any CG, and the
// coarse members' residual sums (in double, below).  The coarse banks are
// solved by every workgroup for itself (four wavefronts of its own, one to
// kOneBanks banks each), which is what makes a second exchange unnecessary:
// the sums it needs are all in the one exchange.
//
// What bounds it: latency, not bytes.  An iteration is one exchange (a store,
// the slowest publisher and a polling load through the memory-side cache) and
// a chain of dependent steps inside a workgroup: totals, coarse solve, p,
// q = A p, w, dots.  At 80x80 quads (28 workgroups) 5.6 us, of which about 2.1
// are the exchange, 1.9 totals and coarse solve, 0.8 the product with A, 0.6 w
// and the dots; k_pcg_persistent takes 7.7 us.  Between the exchange and the
// coarse corrections the two wavefronts of a SIMD issue about 880 vector
// instructions of four cycles, which is what that part takes.
//
// Work split: eight wavefronts, two roles of four.  Slot wavefronts own eight
// 32-slot level-0 banks, one thread per slot (row of the bank inverse, r, dx,
// p in registers) and solve one coarse bank each; coarse wavefronts solve the
// other coarse banks (residual sums in double, inverses in registers), form p
// of the halo and the level-1 sums.  Both add half of each row of q = A p.
// All eight poll the exchange.
//
// Exchange words are those of k_pcg_persistent (epoch << 32 | payload,
// device-scope relaxed 64-bit atomics), in two buffers by the parity of the
// epoch: a workgroup publishes epoch e + 2 only after it has read everyone's
// dot products of epoch e + 1, which each workgroup publishes after it has
// read all it needs of epoch e, so no word is overwritten before it is read.
// The level-1 sums are doubles cut to 48 bits under a 16-bit epoch (a word is
// never more than a few epochs old, see one_last_epoch): the coarse residuals are carried by
// cr -= alpha * (sum of q), and with sums rounded to FP32 their errors, 6e-8
// of the largest r there has been, end the convergence about a decade earlier
// (40x40 quads reach 1e-7 in 51 iterations instead of never).
// Waits are bounded; a wait that gives up raises an abort flag and every
// workgroup leaves.
#include <algorithm>
#include <iterator>

#include "hip/device_common.hpp"
#include "hip/dpp_dot.hpp"
#include "hip/kernels.hpp"
#include "hip/pcg_exchange.hpp"
#include "hip/pcg_rules.hpp"

namespace silk::amd {

using namespace dev;

namespace {

constexpr int kOneThreads = 2 * kPcgThreads;  // slot wavefronts, then coarse ones
constexpr int kDots = 8;                      // doubles per workgroup (7 used)

// Indices of the dot products.
enum { kPq, kRw, kQw, kRz0, kRr, kRq, kQq };

// Barrier of all eight wavefronts; the two roles reach it from different
// code, each the same number of times.
__device__ __forceinline__ void wg_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

__device__ __forceinline__ void sts4v(float* base, int i, f3 v) {
  *reinterpret_cast<float4*>(base + 4 * i) = float4{v.x, v.y, v.z, 0.0f};
}

// Rows of 16 lanes 1 and 3 of `a` swap with rows 0 and 2 of `b`, or the upper
// half of `a` with the lower half of `b`.
__device__ __forceinline__ void swap16(double& a, double& b) {
  const unsigned long long x = static_cast<unsigned long long>(__double_as_longlong(a));
  const unsigned long long y = static_cast<unsigned long long>(__double_as_longlong(b));
  const auto lo = __builtin_amdgcn_permlane16_swap(static_cast<unsigned>(x),
                                                   static_cast<unsigned>(y), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(
      static_cast<unsigned>(x >> 32), static_cast<unsigned>(y >> 32), false, false);
  a = __longlong_as_double(static_cast<long long>(
      (static_cast<unsigned long long>(hi[0]) << 32) | lo[0]));
  b = __longlong_as_double(static_cast<long long>(
      (static_cast<unsigned long long>(hi[1]) << 32) | lo[1]));
}
__device__ __forceinline__ void swap32(double& a, double& b) {
  const unsigned long long x = static_cast<unsigned long long>(__double_as_longlong(a));
  const unsigned long long y = static_cast<unsigned long long>(__double_as_longlong(b));
  const auto lo = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(x),
                                                   static_cast<unsigned>(y), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(
      static_cast<unsigned>(x >> 32), static_cast<unsigned>(y >> 32), false, false);
  a = __longlong_as_double(static_cast<long long>(
      (static_cast<unsigned long long>(hi[0]) << 32) | lo[0]));
  b = __longlong_as_double(static_cast<long long>(
      (static_cast<unsigned long long>(hi[1]) << 32) | lo[1]));
}

// Wavefront sums of four doubles: lane 16 r holds the sum of v[r].  A swap
// that trades halves of two values adds both in one step.
__device__ __forceinline__ double sum64_x4(double (&v)[4]) {
  swap32(v[0], v[2]);
  swap32(v[1], v[3]);
  v[0] += v[2];  // lower half: value 0, upper half: value 2
  v[1] += v[3];
  swap16(v[0], v[1]);
  double a = v[0] + v[1];  // row r: value r
  a += dpp_d<kDppXor1>(a);
  a += dpp_d<kDppXor2>(a);
  a += dpp_d<kDppHalfMirror>(a);
  a += dpp_d<kDppMirror>(a);
  return a;
}

// Wavefront sums of two doubles: lanes 0-31 hold that of a, 32-63 that of b.
__device__ __forceinline__ double sum64_x2(double a, double b) {
  swap32(a, b);
  return sum32(a + b);
}

// n / d to about an ulp, without the scaling and fix-up of the IEEE sequence
// (d is not subnormal or infinite here), which is on the iteration's chain.
__device__ __forceinline__ double quick_inv(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = fma(fma(-d, r, 1.0), r, r);
  return fma(fma(-d, r, 1.0), r, r);
}

__device__ __forceinline__ d3 ldd3(const double* p, int i) {
  return {p[3 * i], p[3 * i + 1], p[3 * i + 2]};
}

// A double cut to 48 bits (relative 2^-37 to nearest) under the epoch's low 16.
__device__ __forceinline__ void put_d48(unsigned long long* w, unsigned epoch, double v) {
  const unsigned long long b =
      static_cast<unsigned long long>(__double_as_longlong(v)) + 0x8000ull;
  __hip_atomic_store(w, (static_cast<unsigned long long>(epoch & 0xffffu) << 48) | (b >> 16),
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ double read_lane_d(double v, int l) {
  const long long b = __double_as_longlong(v);
  const unsigned lo =
      static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(b), l));
  const unsigned hi =
      static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(b >> 32), l));
  return __longlong_as_double(static_cast<long long>(
      (static_cast<unsigned long long>(hi) << 32) | lo));
}

/// Value of lane l ^ 8 within each row of 16 (DPP row_ror:8).
constexpr int kDppRor8 = 0x128;

// A thread's words of the exchange: word t + kOneThreads * m of the
// workgroup's list, by its index in the exchange buffer.  The list is stored
// in LDS as it stands (the level-1 sums as doubles, the rest as floats), so
// the list index is also the place of the payload.
template <int kWords>
struct OneShare {
  int off[kWords];
  unsigned mask;
  unsigned sums;  // bit m: word m is a level-1 sum
};

// Waits until each of the thread's words carries `epoch` and stores the
// payloads: list entry i at sums[i] or rest[i]; false when the wait gave up.
template <int kWords>
__device__ __forceinline__ bool one_collect(const OneShare<kWords>& sh,
                                            const unsigned long long* buf, unsigned epoch,
                                            double* sums, float* rest, int* abort_flag) {
  unsigned pending = sh.mask;
  unsigned spins = 0;
  while (pending != 0) {
    // Up to five loads in flight per thread: more would only hold registers.
    constexpr int kBatch = kWords < 6 ? kWords : (kWords + 1) / 2;
#pragma unroll
    for (int m0 = 0; m0 < kWords; m0 += kBatch) {
      unsigned long long v[kBatch];
#pragma unroll
      for (int m = 0; m < kBatch; ++m) {
        v[m] = 0;
        if (m0 + m < kWords && (pending & (1u << (m0 + m))))
          v[m] = __hip_atomic_load(const_cast<unsigned long long*>(buf + sh.off[m0 + m]),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
#pragma unroll
      for (int m = 0; m < kBatch; ++m)
        if (m0 + m < kWords && (pending & (1u << (m0 + m)))) {
          const int i = static_cast<int>(threadIdx.x) + kOneThreads * (m0 + m);
          const unsigned tag = static_cast<unsigned>(v[m] >> 32);
          if ((sh.sums >> (m0 + m)) & 1u) {
            if ((tag >> 16) == (epoch & 0xffffu)) {
              sums[i] = __longlong_as_double(static_cast<long long>(v[m] << 16));
              pending &= ~(1u << (m0 + m));
            }
          } else if (tag == epoch) {
            rest[i] = __uint_as_float(static_cast<unsigned>(v[m]));
            pending &= ~(1u << (m0 + m));
          }
        }
    }
    if (pending == 0) break;
    if ((++spins & 255) == 0 &&
        (spins > kSpinLimit ||
         __hip_atomic_load(abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
      __hip_atomic_store(abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  return true;
}

// Words mapped when they are collected (the exchanges of the true-residual
// test, once or twice a solve).
template <class WordFn>
__device__ __forceinline__ bool one_collect_fn(int total, WordFn&& word, unsigned epoch,
                                               float* lds, int* abort_flag) {
  for (int i = static_cast<int>(threadIdx.x); i < total; i += kOneThreads) {
    const unsigned long long* addr = nullptr;
    int dest = 0;
    word(i, addr, dest);
    unsigned spins = 0;
    for (;;) {
      const unsigned long long v = __hip_atomic_load(
          const_cast<unsigned long long*>(addr), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (static_cast<unsigned>(v >> 32) == epoch) {
        lds[dest] = __uint_as_float(static_cast<unsigned>(v));
        break;
      }
      if ((++spins & 255) == 0 &&
          (spins > kSpinLimit ||
           __hip_atomic_load(abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
        __hip_atomic_store(abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return false;
      }
      __builtin_amdgcn_s_sleep(1);
    }
  }
  return true;
}

// The solve's scalars.  Every wavefront of every workgroup of a system forms
// them from the same doubles with the same operations, so all take the same
// decisions.
struct Scalars {
  double rz = 0.0;    // r.z of the current r (from r's own dot products)
  double inv_rz = 0.0;  // its inverse, formed while the coarse banks are solved
  double rzc = 0.0;   // its coarse part
  double rr = 0.0, rr0 = 0.0, ref2 = 0.0;
  double abs2 = 0.0, rel2 = 0.0;
  double true_ratio = -1.0;
  int iter = 0, status = -1, replaced = 0, unverified = 0;
  bool start = true;
  // The last r.r came out of a cancellation too deep to decide on; the next
  // exchange's, formed from r itself, is tested before its step is taken.
  bool untrusted = false;

  __device__ __forceinline__ int test(double v) const {
    if (v <= abs2) return 0;
    if (v <= rel2 * ref2) return 1;
    return -1;
  }
};

// Coarse banks whose inverse a wavefront keeps in registers (16 each); more
// would spill.
template <int kBanks>
constexpr int kRegBanks = kBanks < 3 ? kBanks : 3;
/// LDS floats of one further bank per coarse wavefront.
constexpr int kOneLdsBank = 16 * kWave * kPcgWaves;

// kN entries of a bank inverse, `stride` apart from entry e0 on, in the
// storage of the launch.
template <int kN>
__device__ __forceinline__ void load_inverse(const PersistDev& a, int bank, size_t e0,
                                             int stride, float (&w)[kN]) {
  if (a.mas_half == 0) {
#pragma unroll
    for (int m = 0; m < kN; ++m) w[m] = a.bank_inv[e0 + static_cast<size_t>(m) * stride];
  } else {
    const float sc = a.bank_scale[bank];
#pragma unroll
    for (int m = 0; m < kN; ++m)
      w[m] = sc * half_bits_to_float(a.bank_inv_h[e0 + static_cast<size_t>(m) * stride],
                                     a.mas_half);
  }
}

// kBanks: coarse banks of a coarse wavefront, kWords: exchange words a thread
// may hold.
template <int kBanks, int kWords>
__global__ void __launch_bounds__(kOneThreads, 2) k_pcg_one(PersistDev a, float rel_tol) {
  // Dynamic LDS (floats): [coarse corrections, 4 per node, one zero record and
  // one for what absent members write][p of own and halo slots, 4 each][both halves of q, 4 per slot
  // each][the exchange's list: level-1
  // sums, 3 doubles per node; dots, 8 doubles per workgroup; halo, M0 r and
  // w, 6 per slot][bank inverses not held in registers][level-1 nodes of the
  // deep coarse nodes, 16-bit].
  extern __shared__ __align__(16) float dyn[];
  __shared__ double red[kPcgWaves][kDots];
  __shared__ double red_c[2 * kPcgWaves];
  __shared__ int aborted;

  const int cw = static_cast<int>(blockIdx.x) + a.wg_base;
  if (a.ctl != nullptr && a.ctl->done != 0) return;
  const int sys = a.one_sys[cw];
  if (a.sys_done != nullptr && a.sys_done[sys] != 0) return;
  if (a.ctl != nullptr) rel_tol = a.ctl->rel_tol;
  const PcgSysDev S = a.sys[sys];
  const int j = cw - S.owg0;
  const int bx = S.wg0 + j;
  unsigned* epoch_ctr = a.bar + kPcgBarrierStride * sys;
  unsigned ep = __hip_atomic_load(epoch_ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int t = static_cast<int>(threadIdx.x);
  const int wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int lane = t % kWave;
  const bool slot_role = wave < kPcgWaves;
  const bool coarse = S.ncb > 0;
  const int h0 = a.halo_ptr[bx];
  const int nh = a.halo_ptr[bx + 1] - h0;

  float* czl = dyn;                                          // 4 x (ncn_max + 2)
  float* pl = czl + 4 * static_cast<size_t>(a.ncn_max + 2);  // 4 x (256 + nhalo_max)
  float* qh = pl + 4 * (static_cast<size_t>(kPcgThreads) + a.nhalo_max);
  double* qz = reinterpret_cast<double*>(qh + 8 * kPcgThreads);  // the zero sum
  double* qs = qz + 4;
  const int zrec = a.ncn_max;

  // ---- the exchange's words.  Buffer words of the system: 3 per level-1
  // node (padded to an even count), 2 kDots per workgroup, 6 per slot; the
  // workgroup's list is the first two and its halo's.
  unsigned long long* const tw = a.tw + S.tw0;
  const int nw1 = 3 * S.n1;
  const int dots_at = (nw1 + 1) & ~1;
  const int slots_at = dots_at + 2 * kDots * S.nwg;
  const int w1 = slots_at + 6 * nh;
  float* rest = reinterpret_cast<float*>(qs + dots_at) - dots_at;  // entry i at rest[i]
  float* parts = rest + dots_at;
  float* hz = rest + slots_at;
  // Bank inverses beyond the kRegBanks a coarse wavefront holds in registers,
  // 16 entries per lane each.
  float* wlds = reinterpret_cast<float*>(qs) + a.list_max;
  unsigned short* deep =
      reinterpret_cast<unsigned short*>(wlds + kOneLdsBank * (kBanks - kRegBanks<kBanks>));
  OneShare<kWords> sh;
  sh.mask = 0;
  sh.sums = 0;
#pragma unroll
  for (int m = 0; m < kWords; ++m) {
    const int i = t + kOneThreads * m;
    sh.off[m] = i;
    bool take = i < w1;
    if (i < nw1) sh.sums |= 1u << m;
    if (i >= nw1 && i < dots_at) take = false;  // padding
    if (i >= dots_at && i < slots_at && (i - dots_at) % (2 * kDots) >= 2 * (kDots - 1))
      take = false;  // the dot products' eighth
    if (i >= slots_at && i < w1) {
      const int hh = (i - slots_at) / 6, k = (i - slots_at) % 6;
      sh.off[m] = slots_at + 6 * (a.halo_slot[h0 + hh] - S.slot0) + k;
    }
    sh.mask |= take ? 1u << m : 0u;
  }
  auto buf = [&](unsigned e) { return tw + (e & 1u) * static_cast<size_t>(a.tw_stride); };

  // Descendant lists of the deep coarse nodes.
  const int deep0 = a.cn_ptr[S.cn0 + S.n1];
  const int ndeep = a.cn_ptr[S.cn0 + S.ncn] - deep0;
  for (int i = t; i < ndeep; i += kOneThreads)
    deep[i] = static_cast<unsigned short>(a.cn_list[deep0 + i]);
  if (t < 4) {
    czl[4 * zrec + t] = 0.0f;
    qz[t] = 0.0;
  }
  if (t == 0) aborted = 0;

  Scalars s;
  s.abs2 = static_cast<double>(a.abs_tol) * a.abs_tol;
  s.rel2 = static_cast<double>(rel_tol) * rel_tol;
  double bb = 0.0;
  if (a.criterion >= 1) {
    const int q0 = a.sys_blk0[sys], q1 = a.sys_blk0[sys + 1];
    double v = 0.0;
    for (int q = q0 + lane; q < q1; q += kWave) v += a.part2[2 * q + 1];
    bb = sum64(v);
  }

  // Collects the exchange of epoch ep (all wavefronts); false when it gave up.
  auto exchange = [&]() -> bool {
    // Another workgroup's words are not there yet: a poll now would come back
    // empty and hold the next one up by its round trip (0.1 to 0.2 us per
    // iteration; 8 to 20 times 64 clocks measure alike).
    if (S.nwg > 1) __builtin_amdgcn_s_sleep(12);
    if (!one_collect(sh, buf(ep), ep, qs, rest, a.abort_flag)) aborted = 1;
    wg_barrier();
    return aborted == 0;
  };

  // The seven totals over the workgroups (lane l adds dot l % 8 of
  // workgroups l / 8, l / 8 + 8, ..., four loads at a time; three steps join
  // the eight lanes).
  double D[kDots - 1];
  auto totals = [&]() {
    const double* d = reinterpret_cast<const double*>(parts) + lane % kDots;
    constexpr int kStep = kWave / kDots;
    double v = 0.0;
    for (int w0 = lane / kDots; w0 < S.nwg; w0 += 4 * kStep) {
      double u[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) u[k] = d[kDots * min(w0 + kStep * k, S.nwg - 1)];
#pragma unroll
      for (int k = 0; k < 4; ++k) v += w0 + kStep * k < S.nwg ? u[k] : 0.0;
    }
    v += dpp_d<kDppRor8>(v);
    v = add_xor32(add_xor16(v));
#pragma unroll
    for (int k = 0; k < kDots - 1; ++k) D[k] = read_lane_d(v, k);
  };

  // After the totals: alpha of the step (0 at a start), the r.r it leaves and
  // the stopping test.
  auto step_scalars = [&]() -> float {
    if (s.start) return 0.0f;
    if (s.untrusted) {
      s.untrusted = false;
      s.rr = D[kRr];
      const int st = s.iter >= a.max_iter ? 2 : s.test(D[kRr]);
      if (st >= 0) {
        s.status = st;
        return 0.0f;
      }
    }
    s.rz = D[kRz0] + s.rzc;
    const float alpha =
        static_cast<float>(fabs(D[kPq]) < 1e-20 ? 0.0 : s.rz * quick_inv(D[kPq]));
    const double al = alpha;
    s.inv_rz = fabs(s.rz) < 1e-20 ? 0.0 : quick_inv(s.rz);
    s.rr = fma(al, fma(al, D[kQq], -2.0 * D[kRq]), D[kRr]);
    ++s.iter;
    // The three terms cancel down to about 1e-16 of the old r.r; a value
    // within a factor 1e6 of that (it may be negative) is neither decided on
    // nor reported: the next exchange's is, at the iteration limit too.
    s.untrusted = s.rr < 1e-10 * D[kRr];
    if (!s.untrusted) s.status = s.iter >= a.max_iter ? 2 : s.test(s.rr);
    return alpha;
  };

  // After the coarse solve: beta of the new direction (0 at a start).
  auto next_scalars = [&](float alpha) -> float {
    const double rzc = ((red_c[0] + red_c[1]) + (red_c[2] + red_c[3])) +
                       ((red_c[4] + red_c[5]) + (red_c[6] + red_c[7]));
    const double al = alpha;
    s.rzc = rzc;
    if (s.start) {
      s.rz = D[kRz0] + rzc;
      s.rr = D[kRr];
      if (s.iter == 0 && s.replaced == 0) {
        s.rr0 = s.rr;
        s.ref2 = a.criterion >= 1 ? bb : s.rr0;
      }
      s.status = isfinite(s.rz) ? -1 : 3;
      // Right-hand-side criterion: a start that already meets it takes no
      // iteration.
      if (s.status < 0 && a.criterion >= 1) s.status = s.test(s.rr);
      s.start = false;
      return 0.0f;
    }
    if (s.status >= 0) return 0.0f;  // stopped: the direction is not used
    const double rz_new = fma(al, fma(al, D[kQw], -2.0 * D[kRw]), D[kRz0]) + rzc;
    const float beta = static_cast<float>(rz_new * s.inv_rz);
    s.rz = rz_new;
    return beta;
  };

  // ---- true-residual test: exchanges of dx (words 3 per slot) and of the
  // wavefronts' sums of the squared residual.
  auto dx_word = [&](int i, const unsigned long long*& addr, int& dest) {
    const int hh = i / 3, c = i % 3;
    addr = a.tdx + 3 * static_cast<size_t>(a.halo_slot[h0 + hh]) + c;
    dest = static_cast<int>(pl - dyn) + 4 * (kPcgThreads + hh) + c;
  };
  constexpr int kWaveWords = 2 * kPcgWaves;
  auto true_word = [&](int i, const unsigned long long*& addr, int& dest) {
    const int w = i / kWaveWords, k = i % kWaveWords;
    addr = a.tp + kPcgPartWords * static_cast<size_t>(S.wg0 + w) + 3 * kWaveWords + k;
    dest = static_cast<int>(parts - dyn) + kWaveWords * w + k;
  };
  auto collect_dx = [&]() -> bool {
    if (!one_collect_fn(3 * nh, dx_word, ep, dyn, a.abort_flag)) aborted = 1;
    wg_barrier();
    return aborted == 0;
  };
  // True: the solve goes on from the replaced residual.
  auto collect_true = [&](bool& again) -> bool {
    if (!one_collect_fn(kWaveWords * S.nwg, true_word, ep, dyn, a.abort_flag)) aborted = 1;
    wg_barrier();
    if (aborted != 0) return false;
    const double* d = reinterpret_cast<const double*>(parts);
    double v = 0.0;
    for (int w = lane; w < kPcgWaves * S.nwg; w += kWave) v += d[w];
    const double true2 = sum64(v);
    s.true_ratio = s.ref2 > 0.0 ? true2 / s.ref2 : 0.0;
    again = false;
    if (true2 <= fmax(s.abs2, s.rel2 * s.ref2)) return true;
    if (s.replaced >= a.max_replace) {
      s.unverified = 1;
      return true;
    }
    ++s.replaced;
    s.start = true;
    s.untrusted = false;
    s.status = -1;
    again = true;
    return true;
  };

  // ---- the workgroup's slots, one per thread of each role: wavefront w of
  // either role holds the same 64 slots.  The row's entries are shared between
  // the roles (even ones here, odd ones there), which halves the longest chain
  // of the iteration's product.
  const int th = t & (kPcgThreads - 1);
  const int nb0 = S.nslot / kBankSlots;
  const int b_lo = (j * nb0) / S.nwg, b_hi = ((j + 1) * nb0) / S.nwg;
  const int lb = b_lo + th / kBankSlots;
  const int s_in_bank = th & (kBankSlots - 1);
  const bool in_bank = lb < b_hi;
  const int slot = S.slot0 + kBankSlots * lb + s_in_bank;
  // (A thread past the last bank looks at the last slot and uses nothing of it.)
  const int slot_c = min(slot, S.slot0 + kBankSlots * b_hi - 1);
  const int row_c = a.slot_row[slot_c];
  const int e_off = a.sell_off[slot_c / kSlice];
  const int row = in_bank ? row_c : -1;
  const bool own = row >= 0;
  const int e_w = own ? a.sell_width[slot_c / kSlice] : 0;
  const int e_lane = slot_c % kSlice;
  const int row_l = max(row, 0);
  const float d_l = a.d[row_l];
  const float dd = own ? d_l : 0.0f;
  // Neighbours (indices into pl) and entries in registers; rows wider than
  // kPcgNbr are read from memory by the slot wavefronts alone.
  constexpr int kHalf = kPcgNbr / 2;
  const bool reg_ell = e_w <= kPcgNbr;
  int ncol[kHalf];
  float nval[kHalf];
#pragma unroll
  for (int k = 0; k < kHalf; ++k) {
    const int e = 2 * k + (slot_role ? 0 : 1);
    const bool v = reg_ell && e < e_w;
    const int at = sell_place(e_off, v ? e_w : 0, e, kSlice, e_lane);
    const int col = a.sell_lcol[at];
    const float val = a.sell_val[at];
    ncol[k] = v ? col : th;
    nval[k] = v ? val : 0.0f;
  }
  // Fours of entries a wavefront adds (the same for all its lanes).
  int units = reg_ell ? e_w / 8 : 0;
  for (int m = kWave / 2; m > 0; m >>= 1) units = max(units, __shfl_xor(units, m, kWave));
  units = __builtin_amdgcn_readfirstlane(units);
  int scn0 = -1;
  int scz[4] = {zrec, zrec, zrec, zrec};
  const int4 slot_nodes =
      *reinterpret_cast<const int4*>(a.slot_cn + 4 * static_cast<size_t>(slot_c));
  if (in_bank && coarse) {
    const int4 q = slot_nodes;
    scn0 = q.x;
    scz[0] = q.x >= 0 ? q.x : zrec;
    scz[1] = q.y >= 0 ? q.y : zrec;
    scz[2] = q.z >= 0 ? q.z : zrec;
    scz[3] = q.w >= 0 ? q.w : zrec;
  }
  // Level-1 nodes of a bank have consecutive ids: first and count per bank.
  int n1_first = scn0 >= 0 ? scn0 : 0x7fffffff;
  int n1_last = scn0;
  for (int m = kBankSlots / 2; m > 0; m >>= 1) {
    n1_first = min(n1_first, __shfl_xor(n1_first, m, kBankSlots));
    n1_last = max(n1_last, __shfl_xor(n1_last, m, kBankSlots));
  }
  const int n1_count = n1_last >= 0 ? n1_last - n1_first + 1 : 0;
  // This role's share of sum_j K_ij (p_j - p_i), in difference form.
  auto row_half = [&](f3 p) -> f3 {
    float ax = 0.0f, ay = 0.0f, az = 0.0f;
#pragma unroll
    for (int c0 = 0; c0 < kHalf; c0 += 4) {
      if (4 * units <= c0) break;
      f3 pn[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) pn[k] = lds4(pl, ncol[c0 + k]);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float v = nval[c0 + k];
        ax += v * (pn[k].x - p.x);
        ay += v * (pn[k].y - p.y);
        az += v * (pn[k].z - p.z);
      }
    }
    return {ax, ay, az};
  };
  // The same in FP64, for the true-residual test.
  auto row_half64 = [&](f3 p) -> d3 {
    d3 s64 = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < kHalf; ++k) {
      const f3 pn = lds4(pl, ncol[k]);
      // Opaque, so that the conversions are not hoisted out of the solve's loop
      // (32 registers for a test made once or twice a solve).
      float nv = nval[k];
      asm volatile("" : "+v"(nv));
      const double v = nv;
      s64.x += v * (static_cast<double>(pn.x) - static_cast<double>(p.x));
      s64.y += v * (static_cast<double>(pn.y) - static_cast<double>(p.y));
      s64.z += v * (static_cast<double>(pn.z) - static_cast<double>(p.z));
    }
    return s64;
  };
  // Sums of q over the level-1 nodes of this thread's bank (coarse role).
  auto publish_node_sums = [&](f3 v) {
    for (int k = 0; k < n1_count; ++k) {
      const int target = n1_first + k;
      const bool in = scn0 == target;
      const double x = sum32(static_cast<double>(in ? v.x : 0.0f));
      const double y = sum32(static_cast<double>(in ? v.y : 0.0f));
      const double z = sum32(static_cast<double>(in ? v.z : 0.0f));
      if (s_in_bank < 3)
        put_d48(buf(ep) + 3 * target + s_in_bank, ep,
                s_in_bank == 0 ? x : s_in_bank == 1 ? y : z);
    }
  };

  // ---- coarse banks.  Lane l keeps the residual sum of member l % 32 of a
  // bank and computes output member i_out = l % 16 + 16 * (l / 32) over the
  // inputs kh + [0, 16), kh = l & 16; lanes l and l ^ 16 join their halves.
  // Banks are dealt from the last on, so that the deep ones, whose sums take
  // longest, go to the coarse wavefronts' first place: ranks 0-3 there, 4-7 to
  // the slot wavefronts, the rest to the coarse wavefronts.  An absent bank
  // has zero entries and writes nothing.
  const int wave4 = wave & (kPcgWaves - 1);
  const int i_out = (lane & 15) + 16 * (lane >> 5);
  const int kh = lane & 16;
  // 1 where the lane also holds the sum of its output, else 0.
  const float pairs = (lane & 31) == i_out ? 1.0f : 0.0f;
  // Member `at` of the bank of rank k, -1 when there is none.
  auto bank_member = [&](int k, int at) -> int {
    const int cbk = S.ncb - 1 - k;
    const int m = coarse ? a.cb_member[kBankSlots * (S.cb0 + max(cbk, 0)) + at] : -1;
    return cbk >= 0 ? m : -1;
  };
  // The bank's inverse at inputs kh + [0, 16) (all loads unconditional, so that
  // they are in flight together).
  auto bank_entries = [&](int k, float (&w)[16]) {
    const int cbk = S.ncb - 1 - k;
    const int bank = coarse ? a.cb_bank[S.cb0 + max(cbk, 0)] : 0;
    const size_t e = static_cast<size_t>(bank) * 1024 + kh * kBankSlots + i_out;
    load_inverse<16>(a, bank, e, kBankSlots, w);
#pragma unroll
    for (int m = 0; m < 16; ++m) w[m] = cbk >= 0 ? w[m] : 0.0f;
  };
  // A member's residual sum, cs = sum at a start and cs - alpha * (sum of q)
  // after a step (am = 1 or -alpha), as FP32 input of the bank product.
  auto advance = [&](d3& cs, d3 cq, double am) -> f3 {
    cs = {fma(am, cq.x, cs.x), fma(am, cq.y, cs.y), fma(am, cq.z, cs.z)};
    return {static_cast<float>(cs.x), static_cast<float>(cs.y), static_cast<float>(cs.z)};
  };
  // Joins the halves of a product, writes the corrections (constant over a
  // node) and returns this lane's part of the bank's r.z_coarse.
  auto finish_bank = [&](f3 c, f3 zc, int mem_o) -> double {
    zc = {add_xor16(zc.x), add_xor16(zc.y), add_xor16(zc.z)};
    sts4v(czl, mem_o, zc);  // (lanes l and l ^ 16 write the same bits)
    return ddot3(pairs * c, zc);
  };

  if (!slot_role) {
    // ================================================== coarse wavefronts
    constexpr int kReg = kRegBanks<kBanks>;
    float winv[kReg][16];
    int mem_o[kBanks], node[kBanks];  // node: a level-1 member's sum
    d3 cs[kBanks];
#pragma unroll
    for (int u = 0; u < kBanks; ++u) {
      const int k = u == 0 ? wave4 : kPcgWaves * (u + 1) + wave4;
      cs[u] = {0.0, 0.0, 0.0};
      node[u] = bank_member(k, lane & 31);
      mem_o[u] = bank_member(k, i_out);
      float w[16];
      bank_entries(k, w);
#pragma unroll
      for (int m = 0; m < 16; ++m) {
        if (u < kReg) winv[u < kReg ? u : 0][m] = w[m];
        else wlds[kOneLdsBank * (u - kReg) + 16 * (t - kPcgThreads) + m] = w[m];
      }
    }
    // A deep bank (in the first place): the sum of each of its nm members over
    // the level-1 nodes below it, by groups of g lanes (as many as the members
    // leave), strided over the member's range [db, de) of the list; the first
    // four nodes' places are kept in registers.
    const int nm = __popcll(__ballot(lane < kBankSlots && node[0] >= 0));
    const bool is_deep = __ballot(node[0] >= S.n1) != 0;
    const int g = nm <= 1 ? 64 : nm <= 2 ? 32 : nm <= 4 ? 16 : nm <= 8 ? 8 : nm <= 16 ? 4 : 2;
    const int from = ((lane & 31) * g) & (kWave - 1);
    int db = 0, de = 0, dn[4] = {0, 0, 0, 0};
    wg_barrier();  // the lists are in LDS
    if (is_deep) {
      const int member = __shfl(node[0], (lane / g) & 31);
      if (lane / g < nm) {
        db = a.cn_ptr[S.cn0 + member] - deep0 + lane % g;
        de = a.cn_ptr[S.cn0 + member + 1] - deep0;
      }
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        if (db + g * q4 < de) dn[q4] = deep[db + g * q4];
    }
    // From here on absent members read the zero sum and write the spare record.
    const bool in0 = node[0] >= 0;
#pragma unroll
    for (int u = 0; u < kBanks; ++u) {
      if (u > 0 || !is_deep) node[u] = node[u] >= 0 ? 3 * node[u] : -4;
      mem_o[u] = mem_o[u] >= 0 ? mem_o[u] : zrec + 1;
    }
    // p of the halo: this thread's slots and their coarse nodes.
    int hsc[kPcgHaloPerThread][4];
    f3 hp[kPcgHaloPerThread];
#pragma unroll
    for (int m = 0; m < kPcgHaloPerThread; ++m) {
      const int hh = th + kPcgThreads * m;
      hp[m] = f3{0.0f, 0.0f, 0.0f};
      const int4 cn = *reinterpret_cast<const int4*>(
          a.slot_cn + 4 * static_cast<size_t>(a.halo_slot[nh > 0 ? h0 + min(hh, nh - 1) : 0]));
      const int q4[4] = {cn.x, cn.y, cn.z, cn.w};
#pragma unroll
      for (int l = 0; l < 4; ++l) hsc[m][l] = hh < nh && q4[l] >= 0 ? q4[l] : zrec;
    }
    // Sum over the nodes of this lane's member of the first bank, a deep one.
    auto deep_sum = [&]() -> d3 {
      d3 v = {0.0, 0.0, 0.0};
      d3 cv[4];
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) cv[q4] = ldd3(qs, dn[q4]);
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        if (db + g * q4 < de) v = {v.x + cv[q4].x, v.y + cv[q4].y, v.z + cv[q4].z};
      for (int e = db + 4 * g; e < de; e += g) {
        const d3 w = ldd3(qs, deep[e]);
        v = {v.x + w.x, v.y + w.y, v.z + w.z};
      }
      auto add = [&](auto&& other) {
        v = {v.x + other(v.x), v.y + other(v.y), v.z + other(v.z)};
      };
      if (g >= 2) add([](double x) { return dpp_d<kDppXor1>(x); });
      if (g >= 4) add([](double x) { return dpp_d<kDppXor2>(x); });
      if (g >= 8) add([](double x) { return dpp_d<kDppHalfMirror>(x); });
      if (g >= 16) add([](double x) { return dpp_d<kDppMirror>(x); });
      if (g >= 32) v = {add_xor16(v.x), add_xor16(v.y), add_xor16(v.z)};
      if (g >= 64) v = {add_xor32(v.x), add_xor32(v.y), add_xor32(v.z)};
      // Lane l takes its member's group sum.
      if (g < 64) v = {__shfl(v.x, from), __shfl(v.y, from), __shfl(v.z, from)};
      return in0 ? v : d3{0.0, 0.0, 0.0};
    };
    f3 q = own ? ld3(a.r0, row) : f3{0.0f, 0.0f, 0.0f};  // r at a start, else q
    double pq = 0.0, qq = 0.0;
    for (;;) {
      ++ep;
      if (coarse) publish_node_sums(q);
      {
        const double v = sum64_x2(pq, qq);
        if ((lane & 31) == 0) red[wave4][lane == 0 ? kPq : kQq] = v;
      }
      wg_barrier();  // the dots are in LDS
      if (!exchange()) return;
      totals();
      const bool was_start = s.start;
      const float alpha = step_scalars();
      // Members' residual sums, then the bank products, three at a time (they
      // fill the wavefront's issue slots).
      const double am = was_start ? 1.0 : -static_cast<double>(alpha);
      double rzc = 0.0;
#pragma unroll
      for (int u0 = 0; u0 < kBanks; u0 += 3) {
        constexpr int kG = kBanks < 3 ? kBanks : 3;
        f3 c[kG], zc[kG];
        if (u0 > 0) __builtin_amdgcn_sched_barrier(0);  // holds the registers down
#pragma unroll
        for (int i = 0; i < kG; ++i) {
          const int u = u0 + i;
          if (u >= kBanks) break;
          const d3 cq = u == 0 && is_deep
                            ? deep_sum()
                            : d3{qs[node[u]], qs[node[u] + 1], qs[node[u] + 2]};
          c[i] = advance(cs[u], cq, am);
        }
#pragma unroll
        for (int i = 0; i < kG; ++i) {
          const int u = u0 + i;
          if (u >= kBanks) break;
          zc[i] = {0.0f, 0.0f, 0.0f};
          if (u < kReg) {
            row_bcast_dot16x3(zc[i].x, zc[i].y, zc[i].z, c[i].x, c[i].y, c[i].z,
                              winv[u < kReg ? u : 0]);
          } else {
            float w[16];
            const float4* src = reinterpret_cast<const float4*>(
                wlds + kOneLdsBank * (u - kReg) + 16 * (t - kPcgThreads));
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const float4 v = src[k];
              w[4 * k] = v.x;
              w[4 * k + 1] = v.y;
              w[4 * k + 2] = v.z;
              w[4 * k + 3] = v.w;
            }
            row_bcast_dot16x3(zc[i].x, zc[i].y, zc[i].z, c[i].x, c[i].y, c[i].z, w);
          }
        }
#pragma unroll
        for (int i = 0; i < kG; ++i) {
          if (u0 + i >= kBanks) break;
          rzc += finish_bank(c[i], zc[i], mem_o[u0 + i]);
        }
      }
      rzc = sum64(rzc);
      if (lane == 0) red_c[wave4] = rzc;
      wg_barrier();  // corrections and r.z_coarse are in LDS
      const float beta = next_scalars(alpha);
#pragma unroll
      for (int m = 0; m < kPcgHaloPerThread; ++m) {
        if (kPcgThreads * m + kWave * wave4 >= nh) break;  // (the same in all lanes)
        const int hh = th + kPcgThreads * m;
        if (hh < nh) {
          f3 z = fma3(-alpha, ld3(hz, 2 * hh + 1), ld3(hz, 2 * hh));
          f3 cv[4];
#pragma unroll
          for (int l = 0; l < 4; ++l) cv[l] = lds4(czl, hsc[m][l]);
          z = z + ((cv[0] + cv[1]) + (cv[2] + cv[3]));
          hp[m] = was_start ? z : fma3(beta, hp[m], z);
          sts4v(pl, kPcgThreads + hh, hp[m]);
        }
      }
      wg_barrier();  // p is in LDS
      if (s.status < 0) {
        const f3 p = lds4(pl, th);
        const f3 h = row_half(p);
        sts4v(qh, kPcgThreads + th, h);
        wg_barrier();  // both halves of q are in LDS
        q = lds4(qh, th) + h;
        pq = ddot3(p, q);  // (padding slots hold zeros)
        qq = ddot3(q, q);
        continue;
      }
      if (a.r0d == nullptr || s.status > 1) return;
      ++ep;
      if (!collect_dx()) return;
      {
        const d3 h = row_half64(lds4(pl, th));
        double* q64 = reinterpret_cast<double*>(qh) + 3 * th;
        q64[0] = h.x;
        q64[1] = h.y;
        q64[2] = h.z;
        wg_barrier();  // this role's half of A dx is in LDS
      }
      ++ep;
      bool again;
      if (!collect_true(again)) return;
      if (!again) return;
#pragma unroll
      for (int u = 0; u < kBanks; ++u) cs[u] = {0.0, 0.0, 0.0};
      wg_barrier();  // the replaced r is in LDS, the parts are free
      q = lds4(pl, th);
      pq = 0.0;
      qq = 0.0;
    }
  }

  // ====================================================== slot wavefronts
  // A slot some other workgroup reads.
  const bool shared = a.slot_pub[slot_c] != 0 && own;
  // This slot's row of its bank inverse, starting with the entries of the
  // slots in its own row of 16 lanes: winv[k] is entry k ^ row16.
  const int row16 = s_in_bank & 16;
  float winv[kBankSlots];
  {
    const int bank = S.bank0 + min(lb, b_hi - 1);
    const size_t e = static_cast<size_t>(bank) * 1024 + s_in_bank;
    float lo[16], hi[16];
    load_inverse<16>(a, bank, e + row16 * kBankSlots, kBankSlots, lo);
    load_inverse<16>(a, bank, e + (row16 ^ 16) * kBankSlots, kBankSlots, hi);
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      winv[k] = in_bank ? lo[k] : 0.0f;
      winv[16 + k] = in_bank ? hi[k] : 0.0f;
    }
  }
  const f3 r_l = ld3(a.r0, row_l), x0 = ld3(a.x, row_l);
  f3 r = own ? r_l : f3{0.0f, 0.0f, 0.0f};
  f3 dx = {0.0f, 0.0f, 0.0f};
  f3 p = {0.0f, 0.0f, 0.0f};
  f3 q = {0.0f, 0.0f, 0.0f};
  // Level-0 part of z = M v: this slot's bank row times v of its bank (all
  // lanes active; lanes outside a bank give 0).
  auto mas_l0 = [&](f3 v) -> f3 {
    f3 z = {0.0f, 0.0f, 0.0f};
    row_bcast_dot16x3(z.x, z.y, z.z, v.x, v.y, v.z, winv);
    row_bcast_dot16x3(z.x, z.y, z.z, xor16_f(v.x), xor16_f(v.y), xor16_f(v.z), winv + 16);
    return z;
  };

  // This wavefront's coarse bank.
  int node = bank_member(kPcgWaves + wave4, lane & 31);
  node = node >= 0 ? 3 * node : -4;
  int mem_o = bank_member(kPcgWaves + wave4, i_out);
  mem_o = mem_o >= 0 ? mem_o : zrec + 1;
  float cinv[16];
  bank_entries(kPcgWaves + wave4, cinv);
  const bool has_bank = S.ncb > kPcgWaves + wave4;
  d3 cs = {0.0, 0.0, 0.0};

  f3 z0 = mas_l0(r);  // M0 r of the current r
  // r.z0 and r.r of the wavefront, ahead of the rest of their exchange.
  auto own_dots = [&]() {
    const double v = sum64_x2(ddot3(r, z0), ddot3(r, r));
    if ((lane & 31) == 0) red[wave4][lane == 0 ? kRz0 : kRr] = v;
  };
  own_dots();
  unsigned long long* const my_words = tw + slots_at + 6 * (slot - S.slot0);
  // M0 r goes out as soon as it is known, ahead of the rest of its exchange.
  auto publish_z0 = [&](unsigned e) {
    if (shared) put_f3(my_words + (e & 1u) * static_cast<size_t>(a.tw_stride), e, z0);
  };
  publish_z0(ep + 1);
  wg_barrier();  // the lists are in LDS
  for (;;) {
    ++ep;
    {
      const f3 w = s.start ? f3{0.0f, 0.0f, 0.0f} : mas_l0(q);
      if (shared)
        put_f3(my_words + (ep & 1u) * static_cast<size_t>(a.tw_stride) + 3, ep, w);
      double v[4] = {0.0, 0.0, 0.0, 0.0};
      if (!s.start) {
        v[0] = ddot3(r, w);
        v[1] = ddot3(q, w);
        v[2] = ddot3(r, q);
      }
      const double d = sum64_x4(v);
      if ((lane & 15) == 0 && lane < 48)
        red[wave4][lane == 0 ? kRw : lane == 16 ? kQw : kRq] = d;
      wg_barrier();  // the dots are in LDS
      if (t < 2 * (kDots - 1)) {
        const int k = t >> 1;
        const double d = ((red[0][k] + red[1][k]) + red[2][k]) + red[3][k];
        const unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(d));
        put_word(buf(ep) + dots_at + 2 * kDots * j + t, ep,
                 static_cast<unsigned>(b >> (32 * (t & 1))));
      }
      if (!exchange()) return;
      totals();
      const bool was_start = s.start;
      const float alpha = step_scalars();
      double rzc = 0.0;
      if (has_bank) {
        f3 zc = {0.0f, 0.0f, 0.0f};
        const f3 c = advance(cs, d3{qs[node], qs[node + 1], qs[node + 2]},
                             was_start ? 1.0 : -static_cast<double>(alpha));
        row_bcast_dot16x3(zc.x, zc.y, zc.z, c.x, c.y, c.z, cinv);
        rzc = sum64(finish_bank(c, zc, mem_o));
      }
      if (lane == 0) red_c[kPcgWaves + wave4] = rzc;
      dx = fma3(alpha, p, dx);
      r = fma3(-alpha, q, r);
      f3 z = fma3(-alpha, w, z0);
      z0 = mas_l0(r);
      publish_z0(ep + 1);
      own_dots();
      wg_barrier();  // corrections and r.z_coarse are in LDS
      const float beta = next_scalars(alpha);
      f3 cv[4];
#pragma unroll
      for (int l = 0; l < 4; ++l) cv[l] = lds4(czl, scz[l]);
      z = z + ((cv[0] + cv[1]) + (cv[2] + cv[3]));
      p = was_start ? z : fma3(beta, p, z);
      sts4v(pl, t, p);
      wg_barrier();  // p is in LDS
      if (s.status < 0) {
        // q = (K + D) p in difference form, this role's half first.
        f3 h = row_half(p);
        if (own && !reg_ell)
          for (int k = 0; k < e_w; ++k)
            h = fma3(a.sell_val[e_off + k * kSlice + e_lane],
                     lds4(pl, a.sell_lcol[e_off + k * kSlice + e_lane]) - p, h);
        h = fma3(dd, p, h);
        sts4v(qh, th, h);
        wg_barrier();  // both halves of q are in LDS
        q = h + lds4(qh, kPcgThreads + th);
        continue;
      }
    }
    // True-residual test of the iterate x0 + dx (r0d holds b - A x0 in FP64).
    if (a.r0d == nullptr || s.status > 1) break;
    ++ep;
    if (own) put_f3(a.tdx + 3 * static_cast<size_t>(slot), ep, dx);
    sts4v(pl, t, dx);
    double r64[3] = {0.0, 0.0, 0.0};
    const size_t i3 = own ? 3 * static_cast<size_t>(row) : 0;
    if (own)
      for (int k = 0; k < 3; ++k) r64[k] = a.r0d[i3 + k];
    if (!collect_dx()) return;
    f3 rt = {0.0f, 0.0f, 0.0f};
    double e2 = 0.0;
    d3 ax = row_half64(dx);
    if (own && !reg_ell)
      for (int k = 0; k < e_w; ++k) {
        const f3 dn = lds4(pl, a.sell_lcol[e_off + k * kSlice + e_lane]);
        const double v = a.sell_val[e_off + k * kSlice + e_lane];
        ax.x += v * (static_cast<double>(dn.x) - static_cast<double>(dx.x));
        ax.y += v * (static_cast<double>(dn.y) - static_cast<double>(dx.y));
        ax.z += v * (static_cast<double>(dn.z) - static_cast<double>(dx.z));
      }
    wg_barrier();  // the coarse wavefronts' half of A dx is in LDS
    if (own) {
      const double* q64 = reinterpret_cast<const double*>(qh) + 3 * th;
      const double ddd = dd;
      r64[0] -= ax.x + q64[0] + ddd * dx.x;
      r64[1] -= ax.y + q64[1] + ddd * dx.y;
      r64[2] -= ax.z + q64[2] + ddd * dx.z;
      e2 = r64[0] * r64[0] + r64[1] * r64[1] + r64[2] * r64[2];
      rt = {static_cast<float>(r64[0]), static_cast<float>(r64[1]),
            static_cast<float>(r64[2])};
    }
    ++ep;
    {
      const double v = sum64(e2);
      if (lane == 0)
        put_double(a.tp + kPcgPartWords * static_cast<size_t>(bx) + 3 * kWaveWords + 2 * wave,
                   ep, v);
    }
    bool again;
    if (!collect_true(again)) return;
    // The residual of x0 + dxc + dx: kept for the next replacement.
    if (own)
      for (int k = 0; k < 3; ++k) a.r0d[i3 + k] = r64[k];
    if (!again) break;
    // Residual replacement: r from the FP64 residual; dx moves into the FP64
    // committed correction and the search starts afresh.
    if (own) {
      r = rt;
      double* c = a.dxc + 3 * static_cast<size_t>(row);
      const double d3v[3] = {dx.x, dx.y, dx.z};
      for (int k = 0; k < 3; ++k) c[k] = (s.replaced == 1 ? 0.0 : c[k]) + d3v[k];
    }
    dx = {0.0f, 0.0f, 0.0f};
    cs = {0.0, 0.0, 0.0};
    z0 = mas_l0(r);
    publish_z0(ep + 1);
    own_dots();
    sts4v(pl, t, r);
    wg_barrier();  // the replaced r is in LDS
  }
  if (own) {
    if (s.replaced == 0) {
      st3(a.x, row, x0 + dx);
      if (a.dx_out != nullptr) st3(a.dx_out, row, dx);
    } else {
      // x0 + dxc + dx rounded once.
      const double* c = a.dxc + 3 * static_cast<size_t>(row);
      const double t0 = c[0] + dx.x, t1 = c[1] + dx.y, t2 = c[2] + dx.z;
      st3(a.x, row, f3{static_cast<float>(x0.x + t0), static_cast<float>(x0.y + t1),
                       static_cast<float>(x0.z + t2)});
      if (a.dx_out != nullptr)
        st3(a.dx_out, row,
            f3{static_cast<float>(t0), static_cast<float>(t1), static_cast<float>(t2)});
    }
  }
  if (j == 0 && t == 0) {
    const unsigned before =
        __hip_atomic_load(epoch_ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(epoch_ctr, one_last_epoch(before, ep), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    PcgState o;
    o.rz = s.rz;
    o.rr = s.rr;
    o.rr0 = s.rr0;
    o.bb = 0.0;
    o.iter = s.iter;
    o.done = 1;
    o.status = s.status;
    o.pad = 0;
    a.out[sys] = o;
    if (a.ctl != nullptr) {
      atomicAdd(&a.ctl->pcg_iters, s.iter);
      atomicMax(&a.ctl->pcg_max_solve, s.iter);
      if (s.status == 2) atomicAdd(&a.ctl->pcg_stalled, 1);
      if (s.replaced != 0) atomicAdd(&a.ctl->pcg_restarts, s.replaced);
      if (s.unverified != 0) atomicAdd(&a.ctl->pcg_unverified, 1);
      if (s.true_ratio >= 0.0)
        atomicMax(&a.ctl->max_true_bits,
                  static_cast<unsigned long long>(__double_as_longlong(s.true_ratio)));
      if (a.restart != 0) {
        atomicAdd(&a.ctl->pcg_restarts, 1);
      } else if (sys == 0) {
        atomicAdd(&a.ctl->pcg_solves, 1);
        a.ctl->last_rel = static_cast<float>(s.rr0 > 0.0 ? sqrt(s.rr / s.rr0) : 0.0);
      }
    }
  }
}

// Instances by the banks of a coarse wavefront: a bank costs 28 registers and
// about 0.25 us per iteration, so a scene takes the smallest that holds its
// systems.  All use the 256 registers that two wavefronts per SIMD leave; the
// compiler spills 0, 7 and 21 of them to scratch (0, 32 and 76 bytes per lane),
// and 152 to 186 scalars to vector lanes.
struct OneInstance {
  const void* fn;
  int banks, words;
};
const OneInstance g_one[] = {
    {reinterpret_cast<const void*>(k_pcg_one<1, 4>), 1, 4},
    {reinterpret_cast<const void*>(k_pcg_one<2, 6>), 2, 6},
    {reinterpret_cast<const void*>(k_pcg_one<4, 10>), 4, 10},
};

}  // namespace

int pcg_one_instance(int ncb, int words) {
  for (int k = 0; k < static_cast<int>(std::size(g_one)); ++k)
    if (ncb <= (g_one[k].banks + 1) * kPcgWaves && words <= g_one[k].words * kOneThreads) return k;
  return -1;
}

size_t pcg_one_lds(const PersistDev& a) {
  return sizeof(float) * (4 * static_cast<size_t>(a.ncn_max + 2) + 8 +
                          4 * (static_cast<size_t>(kPcgThreads) + a.nhalo_max) +
                          8 * static_cast<size_t>(kPcgThreads) +
                          static_cast<size_t>(a.list_max) +
                          static_cast<size_t>(kOneLdsBank) *
                              std::max(0, g_one[std::max(0, a.one_inst)].banks - 3)) +
         2 * ((static_cast<size_t>(a.ndeep_max) + 7) & ~size_t{7});
}

int pcg_one_resident(const PersistDev& a) {
  if (a.one_inst < 0) return 0;
  return pcg_resident(g_one[a.one_inst].fn, kOneThreads, pcg_one_lds(a));
}

hipError_t launch_pcg_one(hipStream_t s, const PersistDev& a, float rel_tol, bool cooperative,
                          int64_t* coop_launches) {
  PersistDev arg = a;
  void* args[] = {&arg, &rel_tol};
  return launch_resident(g_one[a.one_inst].fn, a.grid, kOneThreads, pcg_one_lds(a), args, s,
                         cooperative, coop_launches);
}

}  // namespace silk::amd
