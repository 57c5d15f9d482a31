// Device helpers shared by the operator, Krylov and eigen translation units.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace sucem {

template <typename R> struct C2;
template <> struct C2<float> { using T = float2; };
template <> struct C2<double> { using T = double2; };

__device__ __forceinline__ float2 mk(float a, float b) { return make_float2(a, b); }
__device__ __forceinline__ double2 mk(double a, double b) { return make_double2(a, b); }

template <typename T>
__device__ __forceinline__ T cmul(T a, T b) {
  return mk(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 to_d(float2 a) { return make_double2(a.x, a.y); }
__device__ __forceinline__ double2 to_d(double2 a) { return a; }

template <typename C>
__device__ __forceinline__ C from_d(double2 v);
template <> __device__ __forceinline__ float2 from_d<float2>(double2 v) {
  return make_float2((float)v.x, (float)v.y);
}
template <> __device__ __forceinline__ double2 from_d<double2>(double2 v) { return v; }

// a / b, or 0 when b == 0 (an exactly converged recursion then stops moving)
__device__ __forceinline__ double2 cdiv0(double2 a, double2 b) {
  double den = b.x * b.x + b.y * b.y;
  if (den == 0.0) return make_double2(0.0, 0.0);
  return make_double2((a.x * b.x + a.y * b.y) / den, (a.y * b.x - a.x * b.y) / den);
}
__device__ __forceinline__ double2 cmuld(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// Paired recursions: two real systems packed in one complex vector (system 0 in the real
// parts, system 1 in the imaginary parts) run as two independent real recursions over the
// same operator and preconditioner passes (linear with real coefficients, so the two parts
// never mix).  Their products are taken per part, (sum a.x b.x, sum a.y b.y), and their
// scalars (a, b) scale the parts separately.
template <typename T>
__device__ __forceinline__ T pmul(T a, T b) {
  return mk(a.x * b.x, a.y * b.y);
}
// per part a / b, 0 where b == 0
__device__ __forceinline__ double2 pdiv0(double2 a, double2 b) {
  return make_double2(b.x != 0.0 ? a.x / b.x : 0.0, b.y != 0.0 ? a.y / b.y : 0.0);
}
// a.b into d: the complex bilinear product, or per part when paired
__device__ __forceinline__ void dot_acc(double2& d, double2 a, double2 b, bool paired) {
  if (paired) {
    d.x += a.x * b.x;
    d.y += a.y * b.y;
  } else {
    d.x += a.x * b.x - a.y * b.y;
    d.y += a.x * b.y + a.y * b.x;
  }
}
// |a|^2 into d.x, or per part (d.x, d.y) when paired
__device__ __forceinline__ void sq_acc(double2& d, double2 a, bool paired) {
  if (paired) {
    d.x += a.x * a.x;
    d.y += a.y * a.y;
  } else {
    d.x += a.x * a.x + a.y * a.y;
  }
}

// x of lane ^ M for M = 1 ... 32 by DPP moves and (M = 16, 32) row swaps, in the vector ALU:
// a shuffle goes through the LDS crossbar and back, and six of them in a row were most of a
// small reduction kernel's time.  Every lane of the wave has to be active.
template <int CTRL>
__device__ __forceinline__ int dpp_move(int x) {
  return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, true);
}
template <int M>
__device__ __forceinline__ int lane_xor(int x) {
  static_assert(M == 1 || M == 2 || M == 4 || M == 8 || M == 16 || M == 32, "one bit");
  if constexpr (M == 1) return dpp_move<0xB1>(x);          // quad permutation [1, 0, 3, 2]
  if constexpr (M == 2) return dpp_move<0x4E>(x);          // quad permutation [2, 3, 0, 1]
  if constexpr (M == 4) return dpp_move<0x1B>(dpp_move<0x141>(x));   // 7 - i, then 3 - i in quads
  if constexpr (M == 8) return dpp_move<0x128>(x);         // row rotation by 8 of 16
  const bool high = (__lane_id() & M) != 0;
  if constexpr (M == 16) {
    // the odd rows of 16 of the one operand change places with the even rows of the other
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return high ? r[0] : r[1];
  }
  if constexpr (M == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return high ? r[0] : r[1];
  }
}
template <int M>
__device__ __forceinline__ float lane_xor(float x) {
  return __int_as_float(lane_xor<M>(__float_as_int(x)));
}
template <int M>
__device__ __forceinline__ double lane_xor(double x) {
  return __hiloint2double(lane_xor<M>(__double2hiint(x)), lane_xor<M>(__double2loint(x)));
}
// Sum over the lanes of aligned groups of L that are MIN apart, the same in all of them; the
// order of a butterfly from distance L / 2 down to MIN.
template <int L, int MIN = 1, typename R>
__device__ __forceinline__ R group_sum(R x) {
  if constexpr (L >= 64 && MIN <= 32) x += lane_xor<32>(x);
  if constexpr (L >= 32 && MIN <= 16) x += lane_xor<16>(x);
  if constexpr (L >= 16 && MIN <= 8) x += lane_xor<8>(x);
  if constexpr (L >= 8 && MIN <= 4) x += lane_xor<4>(x);
  if constexpr (L >= 4 && MIN <= 2) x += lane_xor<2>(x);
  if constexpr (L >= 2 && MIN <= 1) x += lane_xor<1>(x);
  return x;
}

// Wavefront-then-block sums of NV double2 at once (one pair of barriers); every thread of
// the block gets the results.  Deterministic: fixed reduction tree.
template <int TB, int NV>
__device__ __forceinline__ void block_sums(double2 (&v)[NV]) {
  __shared__ double2 red[TB / 64][NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    v[k].x = group_sum<64>(v[k].x);
    v[k].y = group_sum<64>(v[k].y);
  }
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) red[w][k] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    double2 s = red[0][k];
    for (int i = 1; i < TB / 64; ++i) { s.x += red[i][k].x; s.y += red[i][k].y; }
    v[k] = s;
  }
}
template <int TB>
__device__ __forceinline__ double2 block_sum(double2 v) {
  double2 a[1] = {v};
  block_sums<TB, 1>(a);
  return a[0];
}

// This thread's sum of the block partials part[tid], part[tid + NT], ..., in that order, four
// loads in flight (the partials were written by other XCDs, so each load is a long one).
template <int NT>
__device__ __forceinline__ double2 thread_parts(const double2* part, int G) {
  double2 s = make_double2(0, 0);
  for (int k0 = threadIdx.x; k0 < G; k0 += 4 * NT) {
    double2 t[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) t[q] = part[min(k0 + q * NT, G - 1)];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (k0 + q * NT < G) { s.x += t[q].x; s.y += t[q].y; }
  }
  return s;
}

// Logical block index that gives each XCD a contiguous share of the rows
// (blocks are dispatched round-robin over the 8 XCDs; G is a multiple of 8).
__device__ __forceinline__ int xcd_block(int G) {
  const int b = blockIdx.x;
  return (b & 7) * (G >> 3) + (b >> 3);
}

// Position of `target` in the ascending col[lo, hi) (one CSR row), or -1.  The midpoint
// is lo + (hi - lo) / 2: the row pointers of a pattern with more than 2^30 nonzeros (the
// 120 x 60 x 90-box order-2 cavity has 1,078,395,480) make lo + hi overflow 32 bits.
__device__ __forceinline__ int find_col(const int32_t* col, int lo, int hi, int target) {
  hi -= 1;
  while (lo <= hi) {
    const int mid = lo + ((hi - lo) >> 1);
    const int cm = col[mid];
    if (cm == target) return mid;
    if (cm < target) lo = mid + 1; else hi = mid - 1;
  }
  return -1;
}

// ---- device scalars of the Krylov recursions -------------------------------------------
enum ScalarSlot {
  S_RHO = 0,      // complex: current rho
  S_ALPHA = 2,    // complex
  S_BETA = 4,     // complex
  S_OMEGA = 6,    // complex (BiCGStab)
  S_RR = 8,       // |r|^2 of the recursion
  S_TRUE = 9,     // |b - A x|^2 (FP64)
  S_BNORM = 10,   // |b|^2 (paired recursions: the two systems' |b|^2 at 10 and 11)
  S_RHO_NEXT = 12,  // complex: rho for the next alpha (equal to S_RHO except between the
                    // fused p update and the next x/r update of patch-operator COCG)
  S_COUNT = 14
};

enum FinalizeMode {
  FIN_NONE = 0,
  FIN_COCG_ALPHA,   // s0 = p.q            -> alpha = rho / s0
  FIN_COCG_BETA,    // s0 = r.z, s1 = |r|^2 -> beta = s0/rho, rho = s0, hist
  FIN_RESID,        // s0 = |r|^2 (true), s1 = rho of the replaced residual
  FIN_NORM,         // s0 = |b|^2
  FIN_BICG_ALPHA,   // s0 = conj(rt).v      -> alpha = rho / s0
  FIN_BICG_OMEGA,   // s0 = conj(s).t, s1 = |t|^2 -> omega = conj(s0)/s1
  FIN_BICG_BETA,    // s0 = conj(rt).r, s1 = |r|^2 -> beta = (s0/rho)(alpha/omega), rho = s0
  FIN_SET_RHO,      // s0 = r.z, s1 = |r|^2     -> rho = s0 (start / restart)
  FIN_DEFER,        // partials only: the consuming kernel forms the scalars itself
};

// One reduction site: per-block partial sums and the scalar array they are finalised
// into (counter: unused, kept for layout).
struct RedSite {
  double2* part;      // 2*G entries
  unsigned* counter;  // one per site
  double* scal;       // S_COUNT doubles
  double* hist;       // residual history (nullable)
  int mode;
  int it;
  int paired = 0;     // two real systems packed as real and imaginary parts (see pmul)
  // where the host waits for the value this site ends with (|r|, or the true |b - A x|^2):
  // the value and behind it seq, in pinned memory (null: nobody waits)
  double* host = nullptr;
  unsigned long long seq = 0;
};

// A value for the waiting host (Context::wait_mail), by one thread.  It is there as soon as it
// is written; a copy behind the kernel would take a launch and its completion (about 15 us
// for every host check).
__device__ __forceinline__ void post(const RedSite& rs, double v) {
  if (!rs.host) return;
  __hip_atomic_store(rs.host, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(reinterpret_cast<unsigned long long*>(rs.host + 1), rs.seq, __ATOMIC_RELEASE,
                     __HIP_MEMORY_SCOPE_SYSTEM);
}

// Paired recursions: the larger of the two systems' squared residual norms s.x, s.y, each
// relative to its |b|^2 (a system with b = 0 counts as solved).
__device__ __forceinline__ double prel2(const double* sc, double2 s) {
  const double b0 = sc[S_BNORM], b1 = sc[S_BNORM + 1];
  return fmax(b0 > 0.0 ? s.x / b0 : 0.0, b1 > 0.0 ? s.y / b1 : 0.0);
}

__device__ __forceinline__ void finalize(const RedSite& rs, double2 s0, double2 s1) {
  double* sc = rs.scal;
  const double2 rho = make_double2(sc[S_RHO], sc[S_RHO + 1]);
  double2 out;
  switch (rs.mode) {
    case FIN_COCG_ALPHA:
    case FIN_BICG_ALPHA:
      out = cdiv0(rho, s0);
      sc[S_ALPHA] = out.x; sc[S_ALPHA + 1] = out.y;
      break;
    case FIN_COCG_BETA:
      out = cdiv0(s0, rho);
      sc[S_BETA] = out.x; sc[S_BETA + 1] = out.y;
      sc[S_RHO] = s0.x; sc[S_RHO + 1] = s0.y;
      sc[S_RHO_NEXT] = s0.x; sc[S_RHO_NEXT + 1] = s0.y;
      sc[S_RR] = s1.x;
      if (rs.hist) rs.hist[rs.it] = sqrt(s1.x);
      post(rs, sqrt(s1.x));
      break;
    case FIN_RESID:   // paired: S_TRUE holds the larger relative square (see prel2)
      sc[S_TRUE] = rs.paired ? prel2(sc, s0) : s0.x;
      sc[S_RHO] = s1.x; sc[S_RHO + 1] = s1.y;
      sc[S_RHO_NEXT] = s1.x; sc[S_RHO_NEXT + 1] = s1.y;
      post(rs, sc[S_TRUE]);
      break;
    case FIN_NORM:
      sc[S_BNORM] = s0.x;
      sc[S_BNORM + 1] = s0.y;   // paired: system 1 (0 otherwise)
      break;
    case FIN_SET_RHO:
      sc[S_RHO] = s0.x; sc[S_RHO + 1] = s0.y;
      sc[S_RHO_NEXT] = s0.x; sc[S_RHO_NEXT + 1] = s0.y;
      sc[S_RR] = s1.x;
      break;
    case FIN_BICG_OMEGA:
      out = s1.x == 0.0 ? make_double2(0.0, 0.0) : make_double2(s0.x / s1.x, -s0.y / s1.x);
      sc[S_OMEGA] = out.x; sc[S_OMEGA + 1] = out.y;
      break;
    case FIN_BICG_BETA: {
      const double2 al = make_double2(sc[S_ALPHA], sc[S_ALPHA + 1]);
      const double2 om = make_double2(sc[S_OMEGA], sc[S_OMEGA + 1]);
      out = cmuld(cdiv0(s0, rho), cdiv0(al, om));
      sc[S_BETA] = out.x; sc[S_BETA + 1] = out.y;
      sc[S_RHO] = s0.x; sc[S_RHO + 1] = s0.y;
      sc[S_RHO_NEXT] = s0.x; sc[S_RHO_NEXT + 1] = s0.y;
      sc[S_RR] = s1.x;
      if (rs.hist) rs.hist[rs.it] = sqrt(s1.x);
      post(rs, sqrt(s1.x));
      break;
    }
    default:
      break;
  }
}

// Block sums of (v0, v1) -> partials part[lb] and part[G + lb]; k_finalize, launched
// after the producing kernel (finish_reduction), sums them in block order
// (deterministic) and finalises the scalars.  Ordering between the two kernels comes
// from the stream, so no block needs a device-scope fence (on a multi-XCD part each
// such fence writes back the XCD's L2).  Must be called by every thread of every block.
template <int TB>
__device__ __forceinline__ void reduce_finalize(const RedSite& rs, int G, double2 v0, double2 v1) {
  double2 v[2] = {v0, v1};
  block_sums<TB, 2>(v);
  if (threadIdx.x == 0) {
    const int lb = xcd_block(G);
    rs.part[lb] = v[0];
    rs.part[G + lb] = v[1];
  }
}

__device__ __forceinline__ double2 scal2(const double* sc, int slot) {
  return make_double2(sc[slot], sc[slot + 1]);
}

}  // namespace sucem
