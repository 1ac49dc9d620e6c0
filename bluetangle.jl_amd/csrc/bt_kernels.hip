// Streaming HIP kernels for gfx950: in-place k-bit operators on a state
// vector (or on vec(rho)), FP64 reductions, probabilities and helpers.
//
// Every operator pass is one read and one write of the 2^K amplitudes a
// thread owns (64-wide wavefronts, consecutive lanes on consecutive groups so
// that the free low bits give coalesced addresses); reductions accumulate in
// FP64 and finish in a fixed order, so they are bit-reproducible.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "bt_internal.hpp"

namespace bt {

template <typename R, int K>
struct ApplyArgs {
  static constexpr int D = 1 << K;
  static constexpr int kInline = (K <= 3) ? D * D : 1;
  C<R>* s;
  uint64_t ngroups;
  uint64_t ctrl;
  uint64_t off[D];
  int nfixed;
  int fixed[kMaxFixed];
  R scale;
  const C<R>* mptr;  // K >= 4: device copy of the matrix (column-major)
  C<R> m[kInline];   // K <= 3: matrix inline in the kernel arguments
};

template <typename R, int K>
__global__ void __launch_bounds__(256) k_apply(ApplyArgs<R, K> a) {
  constexpr int D = 1 << K;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; g < a.ngroups; g += stride) {
    uint64_t base = g;
    for (int i = 0; i < a.nfixed; i++) base = insert0(base, a.fixed[i]);
    base |= a.ctrl;
    C<R> v[D];
#pragma unroll
    for (int l = 0; l < D; l++) v[l] = a.s[base + a.off[l]];
#pragma unroll
    for (int r = 0; r < D; r++) {
      C<R> acc = cmake<C<R>>(0, 0);
#pragma unroll
      for (int c = 0; c < D; c++) {
        const C<R> mrc = (K <= 3) ? a.m[r + c * D] : a.mptr[r + c * D];
        acc = cfma(acc, mrc, v[c]);
      }
      acc.x *= a.scale;
      acc.y *= a.scale;
      a.s[base + a.off[r]] = acc;
    }
  }
}

// One-qubit operator on a low target bit b <= 6 of a complex64 state: every
// lane takes two consecutive amplitudes with one 16-byte access, so a
// wavefront reads and writes 1 KiB contiguous per instruction whatever the
// target (the generic kernel above gives each lane one amplitude of the pair,
// 8 bytes every 2^(b+1) x 8 bytes, for low b).  b = 0: the pair is in the
// lane; b >= 1: the partner amplitudes are in lane ^ 2^(b-1) of the same
// wavefront, exchanged with cross-lane shuffles.
__global__ void __launch_bounds__(256) k_apply1_low(float4* __restrict__ s, uint64_t nvec, int b, float2 u00,
                                                    float2 u01, float2 u10, float2 u11, float scale) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  // every lane of a wavefront runs the same trips (nvec is a multiple of 64),
  // so the shuffles below always find their partner lane active
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nvec; i += stride) {
    const float4 v = s[i];
    const float2 x0 = make_float2(v.x, v.y), x1 = make_float2(v.z, v.w);
    float2 y0, y1;
    if (b == 0) {
      y0 = cfma(cmul(u00, x0), u01, x1);
      y1 = cfma(cmul(u10, x0), u11, x1);
    } else {
      const int m = 1 << (b - 1);
      const float2 p0 = make_float2(__shfl_xor(x0.x, m, 64), __shfl_xor(x0.y, m, 64));
      const float2 p1 = make_float2(__shfl_xor(x1.x, m, 64), __shfl_xor(x1.y, m, 64));
      // this lane holds the amplitudes with target bit = (i >> (b - 1)) & 1
      const bool hi = (i >> (b - 1)) & 1;
      const float2 cs = hi ? u11 : u00, co = hi ? u10 : u01;
      y0 = cfma(cmul(cs, x0), co, p0);
      y1 = cfma(cmul(cs, x1), co, p1);
    }
    s[i] = make_float4(y0.x * scale, y0.y * scale, y1.x * scale, y1.y * scale);
  }
}

// Uncontrolled two-qubit operator on low target bits (both <= 6) of a
// complex64 state: a wavefront reads 64 consecutive 16-byte pairs of
// amplitudes (a 128-amplitude segment that holds whole groups) into LDS,
// every lane forms its two outputs from the segment, and writes them back
// with one 16-byte access, so reads and writes stay 1 KiB contiguous per
// wavefront whatever the targets.  The workgroup walks 256-pair blocks in a
// uniform trip count (nvec is a multiple of 256).
__global__ void __launch_bounds__(256) k_apply2_low(float4* __restrict__ s, uint64_t nvec, ApplyArgs<float, 2> a) {
  __shared__ float2 seg[4][128];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint32_t mask = (uint32_t)a.off[3];
  for (uint64_t b0 = (uint64_t)blockIdx.x * 256; b0 < nvec; b0 += (uint64_t)gridDim.x * 256) {
    const float4 v = s[b0 + threadIdx.x];
    seg[w][2 * lane] = make_float2(v.x, v.y);
    seg[w][2 * lane + 1] = make_float2(v.z, v.w);
    __syncthreads();
    float2 y[2];
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const uint32_t i = 2u * (uint32_t)lane + (uint32_t)e;  // index in the segment
      const uint32_t rest = i & ~mask;
      int r = 0;
#pragma unroll
      for (int l = 1; l < 4; l++)
        if ((i & mask) == (uint32_t)a.off[l]) r = l;
      float2 acc = cmake<float2>(0, 0);
#pragma unroll
      for (int c = 0; c < 4; c++) acc = cfma(acc, a.m[r + c * 4], seg[w][rest | (uint32_t)a.off[c]]);
      y[e] = acc;
    }
    s[b0 + threadIdx.x] = make_float4(y[0].x * a.scale, y[0].y * a.scale, y[1].x * a.scale, y[1].y * a.scale);
    __syncthreads();  // the segment is rewritten on the next trip
  }
}

// Uncontrolled two-qubit operator on a complex64 state whose target bits
// are both >= 1: every lane takes the two groups that differ in amplitude
// bit 0 (consecutive amplitudes) with one 16-byte access per matrix index,
// so a wavefront moves 1 KiB contiguous per access instead of 512 B.  The
// launcher uses it where that measured faster (both targets in [9, 24]:
// 5.4-5.9 TB/s against 4.3-5.2 for one group per lane on a 2^30-amplitude
// state; below and above that range one group per lane is as fast or
// faster).
__global__ void __launch_bounds__(256) k_apply2_pair(ApplyArgs<float, 2> a) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t nh = a.ngroups / 2;
  for (uint64_t h = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; h < nh; h += stride) {
    uint64_t base = 2 * h;  // bit 0 stays clear: every inserted bit is >= 1
    for (int i = 0; i < a.nfixed; i++) base = insert0(base, a.fixed[i]);
    float2 x[4], y[4];
#pragma unroll
    for (int l = 0; l < 4; l++) {
      const float4 w = *(const float4*)(a.s + base + a.off[l]);
      x[l] = make_float2(w.x, w.y);
      y[l] = make_float2(w.z, w.w);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      float2 u = cmake<float2>(0, 0), v = cmake<float2>(0, 0);
#pragma unroll
      for (int c = 0; c < 4; c++) {
        u = cfma(u, a.m[r + c * 4], x[c]);
        v = cfma(v, a.m[r + c * 4], y[c]);
      }
      *(float4*)(a.s + base + a.off[r]) = make_float4(u.x * a.scale, u.y * a.scale, v.x * a.scale, v.y * a.scale);
    }
  }
}

// ---------------------------------------------------------------------------
// reductions
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Per-wavefront sums of M per-thread values (blockDim.x == 256: 4 waves).
template <int M>
__device__ __forceinline__ void block_sums(const double (&acc)[M], double (*red)[M]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < M; j++) {
    double v = wave_sum(acc[j]);
    if (lane == 0) red[wave][j] = v;
  }
  __syncthreads();
}

// Where a reduction's M sums go: per-workgroup partials (part[b * M + j]),
// then, by the last workgroup to finish, the totals.  part and count are
// the state's, out its pinned host buffer: a reduction is one launch and one
// wait, where a second launch for the totals and a copy of them cost another
// 10 us of every call.
struct ReduceOut {
  double* part;
  unsigned* count;  // kCountWords, see count_last
  double* out;
};

// Store this workgroup's sums (red: [4][M] of block_sums) and, in the last
// workgroup to finish, add up all workgroups' in a fixed order: 256 / M2
// threads per sum (M2: M rounded up to a power of two), each over a fixed
// stride of workgroups, then a fixed tree.  The partials cross the XCDs' L2
// caches: agent-scope stores, complete before the count is raised, and
// agent-scope loads after it.  Returns true in the last workgroup, with the
// totals in sh[0..M).
template <int M>
__device__ __forceinline__ bool reduce_finish(const double (*red)[M], const ReduceOut& o, double* sh) {
  __shared__ int last;
  constexpr int M2 = M <= 1 ? 1 : M <= 2 ? 2 : M <= 4 ? 4 : M <= 16 ? 16 : 64;
  constexpr unsigned G = 256 / M2;  // threads per sum
  const unsigned nb = gridDim.x;
  const int j = threadIdx.x & (M2 - 1);
  const unsigned q = threadIdx.x / M2;
  if (nb == 1) {
    if (q == 0 && j < M) sh[j] = red[0][j] + red[1][j] + red[2][j] + red[3][j];
    __syncthreads();
    return true;
  }
  if (q == 0 && j < M)
    __hip_atomic_store(o.part + (size_t)blockIdx.x * M + j, red[0][j] + red[1][j] + red[2][j] + red[3][j],
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's partials have reached the point of coherence
  __syncthreads();
  if (threadIdx.x == 0) last = count_last(o.count, blockIdx.x, nb);
  __syncthreads();
  if (!last) return false;
  double t = 0.0;
  if (j < M) {
    unsigned b = q;
    for (; b + 7 * G < nb; b += 8 * G) {  // eight loads in flight
      double x[8];
#pragma unroll
      for (int i = 0; i < 8; i++)
        x[i] = __hip_atomic_load(o.part + (size_t)(b + i * G) * M + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int i = 0; i < 8; i++) t += x[i];
    }
    for (; b < nb; b += G)
      t += __hip_atomic_load(o.part + (size_t)b * M + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  sh[threadIdx.x] = t;  // slot j + M2 q
  __syncthreads();
  for (unsigned w = G / 2; w > 0; w >>= 1) {
    if (q < w) sh[threadIdx.x] += sh[threadIdx.x + w * M2];
    __syncthreads();
  }
  return true;
}

// Finish a reduction of M sums per thread: the totals go to o.out[0..M).
template <int M>
__device__ __forceinline__ void reduce_out(const double (&acc)[M], const ReduceOut& o) {
  __shared__ double red[4][M];
  __shared__ double sh[256];
  block_sums<M>(acc, red);
  if (reduce_finish<M>(red, o, sh) && threadIdx.x < M) o.out[threadIdx.x] = sh[threadIdx.x];
}

template <typename R, int K>
struct ReduceArgs {
  static constexpr int D = 1 << K;
  const C<R>* s;
  uint64_t ngroups;
  uint64_t off[D];
  int nfixed;
  int fixed[kMaxFixed];
  ReduceOut out;
};

// Packed layout of a reduced rho (D*D reals): [0, D) diagonal, then for
// each a < b (row-major over a): Re, Im of rho[a, b] = sum v_a conj(v_b).
// Items per loop trip of the reductions: their loads are issued together
// (more bytes in flight per wave); an item past the end re-reads the trip's
// first item and contributes nothing.
template <int K>
constexpr int red_unroll() { return K == 0 ? 4 : K == 1 ? 2 : 1; }

// The work items [lo, hi) of this workgroup in a reduction over n items:
// one contiguous range per workgroup, a whole number of loop trips of
// U * blockDim.x items each (the last ranges may be short or empty).  A trip
// reads U * blockDim.x consecutive items, and the workgroups that run at
// once stream separate long runs of the state: 6.1-6.2 TB/s for one read of
// a 2^30-amplitude complex64 state, against 5.5-5.6 TB/s for the same loads
// strided over the whole grid.
__device__ __forceinline__ void red_range(uint64_t n, int U, uint64_t& lo, uint64_t& hi) {
  const uint64_t trip = (uint64_t)U * blockDim.x;
  const uint64_t per = ((n + gridDim.x - 1) / gridDim.x + trip - 1) / trip * trip;
  lo = std::min<uint64_t>(n, (uint64_t)blockIdx.x * per);
  hi = std::min<uint64_t>(n, lo + per);
}

template <typename R, int K>
__global__ void __launch_bounds__(256) k_reduce(ReduceArgs<R, K> a) {
  constexpr int D = 1 << K;
  constexpr int M = D * D;
  constexpr int U = red_unroll<K>();
  double acc[M];
#pragma unroll
  for (int j = 0; j < M; j++) acc[j] = 0.0;
  uint64_t lo, hi;
  red_range(a.ngroups, U, lo, hi);
  const uint64_t stride = blockDim.x;
  for (uint64_t g0 = lo + threadIdx.x; g0 < hi; g0 += U * stride) {
    C<R> v[U][D];
    bool live[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint64_t g = g0 + u * stride;
      live[u] = g < hi;
      uint64_t base = live[u] ? g : g0;
      for (int i = 0; i < a.nfixed; i++) base = insert0(base, a.fixed[i]);
#pragma unroll
      for (int l = 0; l < D; l++) v[u][l] = a.s[base + a.off[l]];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (!live[u]) continue;
      double vr[D], vi[D];
#pragma unroll
      for (int l = 0; l < D; l++) {
        vr[l] = (double)v[u][l].x;
        vi[l] = (double)v[u][l].y;
      }
      int p = D;
#pragma unroll
      for (int x = 0; x < D; x++) {
        acc[x] = fma(vr[x], vr[x], fma(vi[x], vi[x], acc[x]));
#pragma unroll
        for (int y = x + 1; y < D; y++) {
          // v_x conj(v_y)
          acc[p] += vr[x] * vr[y] + vi[x] * vi[y];
          acc[p + 1] += vi[x] * vr[y] - vr[x] * vi[y];
          p += 2;
        }
      }
    }
  }
  reduce_out<M>(acc, a.out);
}

// <a|b> = sum conj(a_i) b_i in FP64 (either precision on either side): (re, im)
template <typename RA, typename RB>
__global__ void __launch_bounds__(256) k_inner(const C<RA>* a, const C<RB>* b, uint64_t n, ReduceOut o) {
  constexpr int U = 4;
  double acc[2] = {0.0, 0.0};
  uint64_t lo, hi;
  red_range(n, U, lo, hi);
  const uint64_t stride = blockDim.x;
  for (uint64_t i0 = lo + threadIdx.x; i0 < hi; i0 += U * stride) {
    C<RA> x[U];
    C<RB> y[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint64_t i = i0 + u * stride < hi ? i0 + u * stride : i0;
      x[u] = a[i];
      y[u] = b[i];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (i0 + u * stride >= hi) continue;
      acc[0] = fma((double)x[u].x, (double)y[u].x, fma((double)x[u].y, (double)y[u].y, acc[0]));
      acc[1] = fma((double)x[u].x, (double)y[u].y, fma(-(double)x[u].y, (double)y[u].x, acc[1]));
    }
  }
  reduce_out<2>(acc, o);
}

// Expectation of O = P(x, z) G(B): P(x, z)[a, b] = (-1)^popcount(a & z) when
// b = a ^ x, G a dense 2^K x 2^K block on the bits B (disjoint from x and z),
// identity elsewhere.  Work item g enumerates the indices a0 with the B bits
// clear and sums over a = a0 | off(i), b = (a0 ^ x) | off(j):
//   SV: conj(psi_a) O[a, b] psi_b       DM: O[a, b] rho[b + a 2^n]
// On a state vector with x != 0, a0 also has the top bit of x clear and the
// item takes both a0 and a0 ^ x, so each amplitude is read once.
// FP64 sums (re, im).
template <typename R, int D>
__device__ __forceinline__ void expect_quad(const C<R> (&u)[D], const C<R> (&v)[D], const double* g, double& sr,
                                            double& si) {
#pragma unroll
  for (int i = 0; i < D; i++) {
    double tr = 0.0, ti = 0.0;  // (G v)_i
#pragma unroll
    for (int j = 0; j < D; j++) {
      const double gr = g[2 * (i + j * D)], gi = g[2 * (i + j * D) + 1];
      tr = fma(gr, (double)v[j].x, fma(-gi, (double)v[j].y, tr));
      ti = fma(gr, (double)v[j].y, fma(gi, (double)v[j].x, ti));
    }
    sr = fma((double)u[i].x, tr, fma((double)u[i].y, ti, sr));
    si = fma((double)u[i].x, ti, fma(-(double)u[i].y, tr, si));
  }
}

template <typename R, int K, bool DM>
__global__ void __launch_bounds__(256) k_expect(const C<R>* s, ExpectArgs a, ReduceOut o) {
  constexpr int D = 1 << K;
  constexpr int U = DM ? 1 : red_unroll<K>();
  double acc[2] = {0.0, 0.0};
  uint64_t lo, hi;
  red_range(a.ngroups, U, lo, hi);
  const uint64_t stride = blockDim.x;
  for (uint64_t g0 = lo + threadIdx.x; g0 < hi; g0 += U * stride) {
    if constexpr (!DM) {
      C<R> u[U][D], v[U][D];
      uint64_t a0[U];
#pragma unroll
      for (int t = 0; t < U; t++) {
        const uint64_t g = g0 + t * stride < hi ? g0 + t * stride : g0;
        a0[t] = g;
        for (int j = 0; j < a.nfixed; j++) a0[t] = insert0(a0[t], a.fixed[j]);
        const uint64_t b0 = a0[t] ^ a.xmask;
#pragma unroll
        for (int j = 0; j < D; j++) v[t][j] = s[b0 | a.off[j]];
        if (a.xmask) {
#pragma unroll
          for (int j = 0; j < D; j++) u[t][j] = s[a0[t] | a.off[j]];
        }
      }
#pragma unroll
      for (int t = 0; t < U; t++) {
        if (g0 + t * stride >= hi) continue;
        if (!a.xmask) {
#pragma unroll
          for (int j = 0; j < D; j++) u[t][j] = v[t][j];
        }
        double sr = 0.0, si = 0.0;
        expect_quad<R, D>(u[t], v[t], a.g, sr, si);
        const bool neg = __popcll(a0[t] & a.zmask) & 1;
        acc[0] += neg ? -sr : sr;
        acc[1] += neg ? -si : si;
        if (a.xmask) {  // the partner item a0 ^ x
          double tr = 0.0, ti = 0.0;
          expect_quad<R, D>(v[t], u[t], a.g, tr, ti);
          const bool negb = __popcll((a0[t] ^ a.xmask) & a.zmask) & 1;
          acc[0] += negb ? -tr : tr;
          acc[1] += negb ? -ti : ti;
        }
      }
    } else {
      uint64_t a0 = g0;
      for (int j = 0; j < a.nfixed; j++) a0 = insert0(a0, a.fixed[j]);
      const uint64_t b0 = a0 ^ a.xmask;
      double sr = 0.0, si = 0.0;
#pragma unroll
      for (int i = 0; i < D; i++) {
        const uint64_t col = (a0 | a.off[i]) << a.n;
#pragma unroll
        for (int j = 0; j < D; j++) {
          const C<R> r = s[(b0 | a.off[j]) + col];
          const double gr = a.g[2 * (i + j * D)], gi = a.g[2 * (i + j * D) + 1];
          sr = fma(gr, (double)r.x, fma(-gi, (double)r.y, sr));
          si = fma(gr, (double)r.y, fma(gi, (double)r.x, si));
        }
      }
      const bool neg = __popcll(a0 & a.zmask) & 1;
      acc[0] += neg ? -sr : sr;
      acc[1] += neg ? -si : si;
    }
  }
  reduce_out<2>(acc, o);
}

// A Z string of a state vector: sum of |a_i|^2 with the sign of zmask's
// parity, in 16-byte words (two complex64 amplitudes or one complex128).
// Bound by the bytes in flight: k_expect holds 32 bytes per lane (four 8-byte
// loads), here 128: 2^25 complex64 amplitudes 77 -> 61 us a call, 2^26
// 147 -> 115, 2^28 445 -> 380 (5.7 TB/s).
template <typename R>
__global__ void __launch_bounds__(256) k_expect_diag(const C<R>* s, uint64_t words, uint64_t zmask, ReduceOut o) {
  constexpr int U = 8, A = sizeof(R) == 4 ? 2 : 1;  // words per trip, amplitudes per word
  typedef R word __attribute__((ext_vector_type(2 * A)));
  const word* w = (const word*)s;
  double acc[2] = {0.0, 0.0};
  uint64_t lo, hi;
  red_range(words, U, lo, hi);
  for (uint64_t g0 = lo + threadIdx.x; g0 < hi; g0 += U * 256) {
    word v[U];
#pragma unroll
    for (int t = 0; t < U; t++) v[t] = w[g0 + t * 256 < hi ? g0 + t * 256 : g0];
#pragma unroll
    for (int t = 0; t < U; t++) {
      if (g0 + t * 256 >= hi) continue;
      double q = (double)v[t][0] * (double)v[t][0] + (double)v[t][1] * (double)v[t][1];
      if constexpr (A == 2) {
        const double r = (double)v[t][2] * (double)v[t][2] + (double)v[t][3] * (double)v[t][3];
        q += (zmask & 1) ? -r : r;
      }
      acc[0] += (__popcll((A * (g0 + t * 256)) & zmask) & 1) ? -q : q;
    }
  }
  acc[1] = 0.0 * acc[0];  // imaginary part: 0, or NaN with a non-finite sum
  reduce_out<2>(acc, o);
}

// ---------------------------------------------------------------------------
// <X_b>, <Y_b> or <Z_b> of every index bit b at once
// ---------------------------------------------------------------------------
// One read of the state gives <Z_b> for all bits (each amplitude's weight
// enters every sum with a sign), and a tile of 2^12 amplitudes gives <X_b> or
// <Y_b> for its 12 bits, where a reduction per bit reads the state once per
// bit: 25 bits of a 2^25-amplitude complex64 state are 1 read instead of 25
// for Z and 3 for X.
constexpr int kEachT = 12;  // tile: 256 threads x 16 amplitudes
constexpr int kEachJ = 14;  // most bits of the tile number inside a workgroup's range

// Rows of part / out: [0, 12) the tile's bits, [12, 12 + J) the tile
// number's low bits (its range within a workgroup), then the total, whose
// signed sums over workgroups give the bits above.
constexpr int kEachZRows = kEachT + kEachJ + 1;

template <typename R>
__global__ void __launch_bounds__(256) k_expect_z(const C<R>* s, int nbits, int J, ReduceOut o) {
  const uint64_t n = 1ull << nbits;
  double acc[kEachZRows];
#pragma unroll
  for (int j = 0; j < kEachZRows; j++) acc[j] = 0.0;
  const uint64_t t0 = (uint64_t)blockIdx.x << J;
  double tot = 0.0;
  for (uint32_t t = 0; t < (1u << J); t++) {
    const uint64_t base = (t0 + t) << kEachT;
    double w[16];
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const uint64_t i = base + 256u * r + threadIdx.x;
      C<R> v = cmake<C<R>>(0, 0);
      if (i < n) v = s[i];
      w[r] = (double)v.x * (double)v.x + (double)v.y * (double)v.y;
    }
    // the four register bits by halving: sums of pairs go on, differences are the signed sums
#pragma unroll
    for (int b = 0; b < 4; b++) {
#pragma unroll
      for (int r = 0; r < (8 >> b); r++) {
        acc[8 + b] += w[2 * r] - w[2 * r + 1];
        w[r] = w[2 * r] + w[2 * r + 1];
      }
    }
    tot += w[0];
#pragma unroll
    for (int j = 0; j < kEachJ; j++)
      if (j < J) acc[kEachT + j] += ((t >> j) & 1u) ? -w[0] : w[0];
  }
#pragma unroll
  for (int b = 0; b < 8; b++) acc[b] = ((threadIdx.x >> b) & 1u) ? -tot : tot;
  acc[kEachZRows - 1] = tot;
  __shared__ double red[4][kEachZRows];
  block_sums<kEachZRows>(acc, red);
  // every workgroup's sums, row-major, for k_each_finish
  if (threadIdx.x < kEachZRows) {
    const int j = threadIdx.x;
    o.part[(size_t)j * gridDim.x + blockIdx.x] = red[0][j] + red[1][j] + red[2][j] + red[3][j];
  }
}

// Tile bits 0..3 are index bits 0..3, tile bits 4..11 the index bits
// hi0..hi0 + 7 (hi0 >= 4); tile t's base is t deposited on the other bits.
// imag: <Y> (2 Im conj(psi_0) psi_1) instead of <X> (2 Re).
template <typename R>
__global__ void __launch_bounds__(256) k_expect_xy(const C<R>* s, int nbits, int hi0, int imag, uint64_t ntiles,
                                                   ReduceOut o) {
  __shared__ C<R> tile[1 << kEachT];
  const uint64_t n = 1ull << nbits;
  const uint32_t tid = threadIdx.x;
  double acc[kEachT];
#pragma unroll
  for (int j = 0; j < kEachT; j++) acc[j] = 0.0;
  // one slot per 16-byte bank group: XOR the low bits with the ones above them
  auto slot = [](uint32_t l) { return l ^ ((l >> 4) & 15u) ^ ((l >> 8) & 15u); };
  auto pairs = [&](const C<R>* v, double* a) {  // the four register bits
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
      for (int r = 0; r < 16; r++) {
        if ((r >> b) & 1) continue;
        const C<R> x = v[r], y = v[r | (1 << b)];
        if (imag) a[b] = fma((double)x.x, (double)y.y, fma(-(double)x.y, (double)y.x, a[b]));
        else a[b] = fma((double)x.x, (double)y.x, fma((double)x.y, (double)y.y, a[b]));
      }
  };
  const bool low = hi0 == 4;  // the first call also takes bits 0..3
  // thread t, register r: tile index r * 256 + t; index bits of t and r
  const uint64_t thr = (tid & 15u) | ((uint64_t)(tid >> 4) << hi0);
  const uint64_t per = (ntiles + gridDim.x - 1) / gridDim.x;
  const uint64_t t1 = std::min<uint64_t>(ntiles, ((uint64_t)blockIdx.x + 1) * per);
  for (uint64_t t = (uint64_t)blockIdx.x * per; t < t1; t++) {
    // bits 4..hi0-1 below the window, the rest above it
    const uint64_t lo = t & ((1ull << (hi0 - 4)) - 1ull), up = t >> (hi0 - 4);
    const uint64_t base = (lo << 4) | (up << (hi0 + 8)) | thr;
    C<R> v[16];
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const uint64_t i = base | ((uint64_t)r << (hi0 + 4));
      v[r] = cmake<C<R>>(0, 0);
      if (i < n) v[r] = s[i];
    }
    pairs(v, acc + 8);
    __syncthreads();  // the last tile's reads are done
#pragma unroll
    for (int r = 0; r < 16; r++) tile[slot(tid | (r << 8))] = v[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; r++) v[r] = tile[slot((tid & 15u) | (r << 4) | ((tid >> 4) << 8))];
    pairs(v, acc + 4);
    if (low) {
#pragma unroll
      for (int r = 0; r < 16; r++) v[r] = tile[slot((uint32_t)r | (tid << 4))];
      pairs(v, acc);
    }
  }
  __shared__ double red[4][kEachT];
  block_sums<kEachT>(acc, red);
  if (tid < kEachT) o.part[(size_t)tid * gridDim.x + blockIdx.x] = 2.0 * (red[0][tid] + red[1][tid] + red[2][tid] + red[3][tid]);
}

// out[b]: row b's sum over the nb workgroups; for b >= rows, the last row
// (total) signed by bit b - rows of the workgroup number.  One workgroup per
// output, fixed order.
__global__ void __launch_bounds__(256) k_each_finish(const double* part, int nb, int rows, int total, double* out) {
  __shared__ double sh[256];
  const int b = blockIdx.x;
  const double* p = part + (size_t)(b < rows ? b : total) * nb;
  double t = 0.0;
  for (int i = threadIdx.x; i < nb; i += 256) t += b < rows || !((i >> (b - rows)) & 1) ? p[i] : -p[i];
  sh[threadIdx.x] = t;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[b] = sh[0];
}

// sum over i of Re(s[i * step]) for i < count (trace of vec(rho): step = D+1)
template <typename R>
__global__ void __launch_bounds__(256) k_strided_re_sum(const C<R>* s, uint64_t count, uint64_t step, ReduceOut o) {
  double acc[1] = {0.0};
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride)
    acc[0] += (double)s[i * step].x;
  reduce_out<1>(acc, o);
}

template <typename R>
__global__ void k_probabilities(const C<R>* s, uint64_t count, uint64_t step, double* out) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) {
    C<R> v = s[i * step];
    out[i] = step == 1 ? (double)v.x * (double)v.x + (double)v.y * (double)v.y : (double)v.x;
  }
}

template <typename R>
__global__ void k_scale(C<R>* s, uint64_t n, R f) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    C<R> v = s[i];
    v.x *= f;
    v.y *= f;
    s[i] = v;
  }
}

template <typename R>
__global__ void k_fill_basis(C<R>* s, uint64_t n, uint64_t index) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    s[i] = cmake<C<R>>(i == index ? (R)1 : (R)0, (R)0);
}

template <typename R>
__global__ void k_gather(const C<R>* s, uint64_t len, const uint64_t* idx, uint64_t n, double* out) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    uint64_t j = idx[i];
    C<R> v = j < len ? s[j] : cmake<C<R>>(0, 0);
    out[2 * i] = (double)v.x;
    out[2 * i + 1] = (double)v.y;
  }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// Workgroups of a reduction with M partial values each over `work` items:
// 16384 for large states (each a contiguous range, see red_range: 6.2 TB/s
// against 6.1 at 4096 and 6.0 at 2048 for one read of 2^30 complex64
// amplitudes), 4096 below 2^28 items, kRedBlocks below 2^26, where the launch
// and the final sum of the partials dominate; always within the partial
// buffer of kRedBlocks * kRedMax values.
static uint64_t red_cap(int M, uint64_t work) {
  const uint64_t c = (uint64_t)kRedBlocks * kRedMax / (uint64_t)M;
  const uint64_t want = work >= (1ull << 28) ? 16384 : work >= (1ull << 26) ? 4096 : kRedBlocks;
  return c < want ? c : want;
}

static ReduceOut reduce_to(bt_state_s* s) { return ReduceOut{s->d_part, s->d_count, s->h_out}; }

static int reduce_wait(bt_state_s* s) {
  BT_HIP(hipGetLastError());
  BT_HIP(hipStreamSynchronize(s->stream));
  return BT_OK;
}

static unsigned grid_for(uint64_t work, unsigned block = 256, uint64_t cap = (1ull << 20)) {
  uint64_t g = (work + block - 1) / block;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (unsigned)g;
}

int make_placement(int nbits, int k, const int* bits, uint64_t ctrl_mask, Placement* p) {
  if (k < 0 || k > kMaxK) return fail(BT_ERR_ARG, "operator width k out of range");
  uint64_t used = 0;
  for (int i = 0; i < k; i++) {
    if (bits[i] < 0 || bits[i] >= nbits) return fail(BT_ERR_ARG, "bit position out of range");
    if (used & (1ull << bits[i])) return fail(BT_ERR_ARG, "repeated bit position");
    used |= 1ull << bits[i];
  }
  if (nbits < 64 && (ctrl_mask >> nbits)) return fail(BT_ERR_ARG, "control bit out of range");
  if (ctrl_mask & used) return fail(BT_ERR_ARG, "control bit equals a target bit");
  uint64_t all = used | ctrl_mask;
  p->nfixed = 0;
  for (int b = 0; b < nbits; b++)
    if (all & (1ull << b)) {
      if (p->nfixed >= kMaxFixed) return fail(BT_ERR_ARG, "too many target/control bits");
      p->fixed[p->nfixed++] = b;
    }
  p->ctrl = ctrl_mask;
  for (int l = 0; l < (1 << k); l++) {
    uint64_t o = 0;
    for (int i = 0; i < k; i++)
      if ((l >> (k - 1 - i)) & 1) o |= 1ull << bits[i];
    p->off[l] = o;
  }
  return BT_OK;
}

template <typename R, int K>
static int apply_t(bt_state_s* s, int nbits, const double* m, const Placement& p, double scale, bool conj_mat) {
  constexpr int D = 1 << K;
  ApplyArgs<R, K> a;
  memset(&a, 0, sizeof a);
  a.s = (C<R>*)s->d;
  a.ngroups = 1ull << (nbits - p.nfixed);
  a.ctrl = p.ctrl;
  for (int l = 0; l < D; l++) a.off[l] = p.off[l];
  a.nfixed = p.nfixed;
  for (int i = 0; i < p.nfixed; i++) a.fixed[i] = p.fixed[i];
  a.scale = (R)scale;
  const double sgn = conj_mat ? -1.0 : 1.0;
  if (K <= 3) {
    for (int i = 0; i < D * D; i++) a.m[i] = cmake<C<R>>((R)m[2 * i], (R)(sgn * m[2 * i + 1]));
    a.mptr = nullptr;
  } else {
    std::vector<C<R>> hm(D * D);
    for (int i = 0; i < D * D; i++) hm[i] = cmake<C<R>>((R)m[2 * i], (R)(sgn * m[2 * i + 1]));
    if (!s->d_mat) BT_HIP(hipMalloc(&s->d_mat, sizeof(C<double>) * 1024));
    // the matrix must not change while an earlier launch may still read it
    BT_HIP(hipStreamSynchronize(s->stream));
    BT_HIP(hipMemcpy(s->d_mat, hm.data(), sizeof(C<R>) * D * D, hipMemcpyHostToDevice));
    a.mptr = (const C<R>*)s->d_mat;
  }
  if constexpr (K == 1 && sizeof(R) == 4) {
    // uncontrolled one-qubit operator on a low bit: the coalesced kernel
    if (p.ctrl == 0 && p.nfixed == 1 && p.fixed[0] <= 6 && nbits >= 7) {
      const uint64_t nvec = 1ull << (nbits - 1);  // two amplitudes per lane
      hipLaunchKernelGGL(k_apply1_low, dim3(grid_for(nvec)), dim3(256), 0, s->stream, (float4*)s->d, nvec,
                         p.fixed[0], a.m[0], a.m[2], a.m[1], a.m[3], (float)scale);
      BT_HIP(hipGetLastError());
      return BT_OK;
    }
  }
  if constexpr (K == 2 && sizeof(R) == 4) {
    // uncontrolled, both targets low: staged through LDS per wavefront
    if (p.ctrl == 0 && p.nfixed == 2 && p.fixed[1] <= 6 && nbits >= 9) {
      const uint64_t nvec = 1ull << (nbits - 1);  // 16-byte pairs, a multiple of 256
      hipLaunchKernelGGL(k_apply2_low, dim3(grid_for(nvec)), dim3(256), 0, s->stream, (float4*)s->d, nvec, a);
      BT_HIP(hipGetLastError());
      return BT_OK;
    }
    // uncontrolled, both targets in the middle bit range: two groups per lane
    if (p.ctrl == 0 && p.nfixed == 2 && p.fixed[0] >= 9 && p.fixed[1] <= 24) {
      hipLaunchKernelGGL(k_apply2_pair, dim3(grid_for(a.ngroups / 2)), dim3(256), 0, s->stream, a);
      BT_HIP(hipGetLastError());
      return BT_OK;
    }
  }
  hipLaunchKernelGGL((k_apply<R, K>), dim3(grid_for(a.ngroups)), dim3(256), 0, s->stream, a);
  BT_HIP(hipGetLastError());
  return BT_OK;
}

int launch_apply(bt_state_s* s, int nbits, int k, const double* m, const Placement& p, double scale,
                 bool conj_mat) {
  if (nbits - p.nfixed < 0) return fail(BT_ERR_ARG, "placement wider than the state");
  const bool f = s->prec == BT_C64;
  switch (k) {
    case 1: return f ? apply_t<float, 1>(s, nbits, m, p, scale, conj_mat) : apply_t<double, 1>(s, nbits, m, p, scale, conj_mat);
    case 2: return f ? apply_t<float, 2>(s, nbits, m, p, scale, conj_mat) : apply_t<double, 2>(s, nbits, m, p, scale, conj_mat);
    case 3: return f ? apply_t<float, 3>(s, nbits, m, p, scale, conj_mat) : apply_t<double, 3>(s, nbits, m, p, scale, conj_mat);
    case 4: return f ? apply_t<float, 4>(s, nbits, m, p, scale, conj_mat) : apply_t<double, 4>(s, nbits, m, p, scale, conj_mat);
    case 5: return f ? apply_t<float, 5>(s, nbits, m, p, scale, conj_mat) : apply_t<double, 5>(s, nbits, m, p, scale, conj_mat);
    default: return fail(BT_ERR_ARG, "operator width k out of range");
  }
}

template <typename R, int K>
static int reduce_t(bt_state_s* s, const Placement& p) {
  constexpr int D = 1 << K;
  constexpr int M = D * D;
  ReduceArgs<R, K> a;
  memset(&a, 0, sizeof a);
  a.s = (const C<R>*)s->d;
  a.ngroups = 1ull << (s->nbits - p.nfixed);
  for (int l = 0; l < D; l++) a.off[l] = p.off[l];
  a.nfixed = p.nfixed;
  for (int i = 0; i < p.nfixed; i++) a.fixed[i] = p.fixed[i];
  a.out = reduce_to(s);
  const unsigned blocks = grid_for(a.ngroups, 256, red_cap(M, a.ngroups));
  hipLaunchKernelGGL((k_reduce<R, K>), dim3(blocks), dim3(256), 0, s->stream, a);
  return reduce_wait(s);
}

int launch_inner(bt_state_s* a, bt_state_s* b, double* re, double* im) {
  const uint64_t n = a->len;
  const unsigned blocks = grid_for(n, 256, red_cap(2, n));
  const bool fa = a->prec == BT_C64, fb = b->prec == BT_C64;
  if (fa && fb)
    hipLaunchKernelGGL((k_inner<float, float>), dim3(blocks), dim3(256), 0, a->stream, (const C<float>*)a->d,
                       (const C<float>*)b->d, n, reduce_to(a));
  else if (fa)
    hipLaunchKernelGGL((k_inner<float, double>), dim3(blocks), dim3(256), 0, a->stream, (const C<float>*)a->d,
                       (const C<double>*)b->d, n, reduce_to(a));
  else if (fb)
    hipLaunchKernelGGL((k_inner<double, float>), dim3(blocks), dim3(256), 0, a->stream, (const C<double>*)a->d,
                       (const C<float>*)b->d, n, reduce_to(a));
  else
    hipLaunchKernelGGL((k_inner<double, double>), dim3(blocks), dim3(256), 0, a->stream, (const C<double>*)a->d,
                       (const C<double>*)b->d, n, reduce_to(a));
  const int rc = reduce_wait(a);
  if (rc) return rc;
  *re = a->h_out[0];
  *im = a->h_out[1];
  return BT_OK;
}

int launch_reduce(bt_state_s* s, int k, const int* bits) {
  Placement p;
  int rc = make_placement(s->nbits, k, bits, 0, &p);
  if (rc) return rc;
  const bool f = s->prec == BT_C64;
  switch (k) {
    case 0: return f ? reduce_t<float, 0>(s, p) : reduce_t<double, 0>(s, p);
    case 1: return f ? reduce_t<float, 1>(s, p) : reduce_t<double, 1>(s, p);
    case 2: return f ? reduce_t<float, 2>(s, p) : reduce_t<double, 2>(s, p);
    case 3: return f ? reduce_t<float, 3>(s, p) : reduce_t<double, 3>(s, p);
    default: return fail(BT_ERR_ARG, "reduction width k out of range");
  }
}

void unpack_reduced(int k, const double* packed, double* rho) {
  const int D = 1 << k;
  for (int i = 0; i < 2 * D * D; i++) rho[i] = 0.0;
  for (int a = 0; a < D; a++) rho[2 * (a + a * D)] = packed[a];
  int p = D;
  for (int a = 0; a < D; a++)
    for (int b = a + 1; b < D; b++) {
      // rho[a, b] = re + i im ; rho[b, a] = conj
      rho[2 * (a + b * D)] = packed[p];
      rho[2 * (a + b * D) + 1] = packed[p + 1];
      rho[2 * (b + a * D)] = packed[p];
      rho[2 * (b + a * D) + 1] = -packed[p + 1];
      p += 2;
    }
}

int launch_norm2(bt_state_s* s, double* out) {
  int rc = launch_reduce(s, 0, nullptr);
  if (rc) return rc;
  *out = s->h_out[0];
  return BT_OK;
}

int launch_trace(bt_state_s* s, double* out) {
  const uint64_t D = 1ull << s->n;
  const unsigned blocks = grid_for(D, 256, kRedBlocks);
  if (s->prec == BT_C64)
    hipLaunchKernelGGL(k_strided_re_sum<float>, dim3(blocks), dim3(256), 0, s->stream, (const C<float>*)s->d, D, D + 1,
                       reduce_to(s));
  else
    hipLaunchKernelGGL(k_strided_re_sum<double>, dim3(blocks), dim3(256), 0, s->stream, (const C<double>*)s->d, D,
                       D + 1, reduce_to(s));
  const int rc = reduce_wait(s);
  if (rc) return rc;
  *out = s->h_out[0];
  return BT_OK;
}

int launch_probabilities(bt_state_s* s, double* d_out) {
  const uint64_t D = 1ull << s->n;
  const uint64_t step = s->kind == BT_DM ? D + 1 : 1;
  if (s->prec == BT_C64)
    hipLaunchKernelGGL(k_probabilities<float>, dim3(grid_for(D)), dim3(256), 0, s->stream, (const C<float>*)s->d, D,
                       step, d_out);
  else
    hipLaunchKernelGGL(k_probabilities<double>, dim3(grid_for(D)), dim3(256), 0, s->stream, (const C<double>*)s->d, D,
                       step, d_out);
  BT_HIP(hipGetLastError());
  return BT_OK;
}

int launch_scale(bt_state_s* s, double f) {
  if (s->prec == BT_C64)
    hipLaunchKernelGGL(k_scale<float>, dim3(grid_for(s->len)), dim3(256), 0, s->stream, (C<float>*)s->d, s->len,
                       (float)f);
  else
    hipLaunchKernelGGL(k_scale<double>, dim3(grid_for(s->len)), dim3(256), 0, s->stream, (C<double>*)s->d, s->len, f);
  BT_HIP(hipGetLastError());
  return BT_OK;
}

int launch_set_basis(bt_state_s* s, uint64_t index) {
  if (s->prec == BT_C64)
    hipLaunchKernelGGL(k_fill_basis<float>, dim3(grid_for(s->len)), dim3(256), 0, s->stream, (C<float>*)s->d, s->len,
                       index);
  else
    hipLaunchKernelGGL(k_fill_basis<double>, dim3(grid_for(s->len)), dim3(256), 0, s->stream, (C<double>*)s->d,
                       s->len, index);
  BT_HIP(hipGetLastError());
  return BT_OK;
}

int launch_gather(bt_state_s* s, const uint64_t* d_idx, uint64_t n, double* d_out) {
  if (s->prec == BT_C64)
    hipLaunchKernelGGL(k_gather<float>, dim3(grid_for(n)), dim3(256), 0, s->stream, (const C<float>*)s->d, s->len,
                       d_idx, n, d_out);
  else
    hipLaunchKernelGGL(k_gather<double>, dim3(grid_for(n)), dim3(256), 0, s->stream, (const C<double>*)s->d, s->len,
                       d_idx, n, d_out);
  BT_HIP(hipGetLastError());
  return BT_OK;
}

template <typename R, int K>
static void expect_t(bt_state_s* s, const ExpectArgs& a, unsigned blocks) {
  if (s->kind == BT_DM)
    hipLaunchKernelGGL((k_expect<R, K, true>), dim3(blocks), dim3(256), 0, s->stream, (const C<R>*)s->d, a,
                       reduce_to(s));
  else
    hipLaunchKernelGGL((k_expect<R, K, false>), dim3(blocks), dim3(256), 0, s->stream, (const C<R>*)s->d, a,
                       reduce_to(s));
}

int launch_expect(bt_state_s* s, int k, const double* mat, const int* bits, uint64_t xmask, uint64_t zmask,
                  double* re, double* im) {
  if (k < 0 || k > 3) return fail(BT_ERR_ARG, "expectation: dense block width k must be 0..3");
  const int n = s->n;
  const uint64_t all = n == 64 ? ~0ull : ((1ull << n) - 1ull);
  if ((xmask | zmask) & ~all) return fail(BT_ERR_ARG, "expectation: Pauli mask outside the register");
  ExpectArgs a;
  std::memset(&a, 0, sizeof(a));
  a.n = n;
  a.xmask = xmask;
  a.zmask = zmask;
  uint64_t used = 0;
  for (int i = 0; i < k; i++) {
    if (bits[i] < 0 || bits[i] >= n) return fail(BT_ERR_ARG, "expectation: bit out of range");
    if ((used >> bits[i]) & 1) return fail(BT_ERR_ARG, "expectation: repeated bit");
    used |= 1ull << bits[i];
  }
  if (used & (xmask | zmask)) return fail(BT_ERR_ARG, "expectation: dense bits overlap the Pauli masks");
  // inserted bits, ascending: the block bits, and on a state vector the top bit of x
  uint64_t ins = used;
  if (s->kind == BT_SV && xmask) ins |= 1ull << (63 - __builtin_clzll(xmask));
  int j = 0;
  for (int b = 0; b < 64; b++)
    if ((ins >> b) & 1) a.fixed[j++] = b;
  a.nfixed = j;
  const int D = 1 << k;
  for (int l = 0; l < D; l++) {
    uint64_t o = 0;
    for (int i = 0; i < k; i++)
      if ((l >> (k - 1 - i)) & 1) o |= 1ull << bits[i];
    a.off[l] = o;
  }
  if (k == 0) {
    a.g[0] = 1.0;
  } else {
    for (int i = 0; i < 2 * D * D; i++) a.g[i] = mat[i];
  }
  a.ngroups = 1ull << (n - a.nfixed);
  const unsigned blocks = grid_for(a.ngroups, 256, red_cap(2, a.ngroups));
  const bool f = s->prec == BT_C64;
  if (k == 0 && !xmask && s->kind == BT_SV && s->len >= 2) {
    const uint64_t words = s->len * s->elem() / 16;
    const unsigned db = grid_for(words, 256, red_cap(2, a.ngroups));
    if (f)
      hipLaunchKernelGGL((k_expect_diag<float>), dim3(db), dim3(256), 0, s->stream, (const C<float>*)s->d, words,
                         zmask, reduce_to(s));
    else
      hipLaunchKernelGGL((k_expect_diag<double>), dim3(db), dim3(256), 0, s->stream, (const C<double>*)s->d, words,
                         zmask, reduce_to(s));
  } else {
    switch (k) {
      case 0: f ? expect_t<float, 0>(s, a, blocks) : expect_t<double, 0>(s, a, blocks); break;
      case 1: f ? expect_t<float, 1>(s, a, blocks) : expect_t<double, 1>(s, a, blocks); break;
      case 2: f ? expect_t<float, 2>(s, a, blocks) : expect_t<double, 2>(s, a, blocks); break;
      default: f ? expect_t<float, 3>(s, a, blocks) : expect_t<double, 3>(s, a, blocks); break;
    }
  }
  const int rc = reduce_wait(s);
  if (rc) return rc;
  *re = s->h_out[0];
  *im = s->h_out[1];
  return BT_OK;
}

// <P_b> of every bit b of a state vector, P = X (1), Y (2) or Z (3).
template <typename R>
static int expect_each_t(bt_state_s* s, int pauli, double* out) {
  const int N = s->n;
  const uint64_t ntiles = N > kEachT ? 1ull << (N - kEachT) : 1;
  if (pauli == 3) {
    // at most 2048 workgroups of at most 2^kEachJ tiles (N <= 36: 2^24 tiles)
    const int tb = N > kEachT ? N - kEachT : 0, J = std::max(0, tb - 11);
    if (J > kEachJ) return fail(BT_ERR_ARG, "expectation of every qubit: state too large");
    const int nb = (int)(ntiles >> J);
    hipLaunchKernelGGL(k_expect_z<R>, dim3((unsigned)nb), dim3(256), 0, s->stream, (const C<R>*)s->d, N, J,
                       reduce_to(s));
    BT_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_each_finish, dim3((unsigned)N), dim3(256), 0, s->stream, (const double*)s->d_part, nb,
                       kEachT + J, kEachZRows - 1, s->h_out);
    const int rc = reduce_wait(s);
    if (rc) return rc;
    for (int b = 0; b < N; b++) out[b] = s->h_out[b];
    return BT_OK;
  }
  // windows of 8 bits above the low 4; the last one ends at the top bit
  const unsigned nb = (unsigned)std::min<uint64_t>(ntiles, 2048);
  for (int b = 4; b < std::max(N, 5); b += 8) {
    const int hi0 = b == 4 ? 4 : std::min(b, N - 8);
    hipLaunchKernelGGL(k_expect_xy<R>, dim3(nb), dim3(256), 0, s->stream, (const C<R>*)s->d, N, hi0, pauli == 2 ? 1 : 0,
                       ntiles, reduce_to(s));
    BT_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_each_finish, dim3(kEachT), dim3(256), 0, s->stream, (const double*)s->d_part, (int)nb, kEachT,
                       0, s->h_out);
    const int rc = reduce_wait(s);
    if (rc) return rc;
    for (int j = hi0 == 4 ? 0 : 4; j < kEachT; j++) {
      const int bit = j < 4 ? j : hi0 + j - 4;
      if (bit < N) out[bit] = s->h_out[j];
    }
  }
  return BT_OK;
}

int launch_expect_each(bt_state_s* s, int pauli, double* out) {
  return s->prec == BT_C64 ? expect_each_t<float>(s, pauli, out) : expect_each_t<double>(s, pauli, out);
}

}  // namespace bt
