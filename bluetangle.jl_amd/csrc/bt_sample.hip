// Shot sampling from a state vector's basis-state probabilities p_i = |psi_i|^2
// (the final sampling of measure / sample, ops.jl:46-60,599-646), with
// explicit uniforms in place of StatsBase's RNG.  Rule: shot s returns the
// smallest i with u_s T < C_i, where C_i is the FP64 cumulative sum in index
// order and T = C_{2^N - 1} (so the state need not be normalised).
//
// Three kernels on the caller's stream:
//   k_chunk_sums   FP64 sum of each chunk of 2048 probabilities;
//   k_chunk_scan   exclusive prefix of the chunk sums, one workgroup per 2048
//                  chunks, whose last one to finish adds up the workgroups;
//   k_sample_find  one wavefront per shot: binary search of the chunk prefix,
//                  then the chunk's rows in order (one 1 KiB row per load).
// Sums are formed in a different order than a sequential cumsum; a shot whose
// u_s T lies within 1e-12 T of a cumulative boundary is flagged.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "bt_internal.hpp"

namespace bt {

constexpr int kChunk = 2048;       // probabilities per chunk
constexpr int kScanRun = 2048;     // chunks per workgroup of the scan
constexpr double kBoundaryTol = 1e-12;

template <typename R>
__device__ __forceinline__ double weight(R x, R y) {
  return (double)x * (double)x + (double)y * (double)y;
}

// Entries of a row: the consecutive probabilities one wavefront load covers
// (16 bytes per lane: two complex64 or one complex128 amplitude).
template <typename R>
constexpr int kRowEntries = 64 * 16 / (2 * sizeof(R));

// The lane's probabilities of row r of the chunk at `base` (0 past n).
template <typename R, int E>
__device__ __forceinline__ void row_weights(const C<R>* s, uint64_t n, uint64_t base, int r, int lane, double (&p)[E]) {
  const uint64_t i = base + (uint64_t)r * kRowEntries<R> + (uint64_t)(E * lane);
  typedef R vec __attribute__((ext_vector_type(2 * E)));
  if (i + E <= n) {
    const vec v = *(const vec*)(s + i);
#pragma unroll
    for (int e = 0; e < E; e++) p[e] = weight<R>(v[2 * e], v[2 * e + 1]);
  } else {
#pragma unroll
    for (int e = 0; e < E; e++) p[e] = i + e < n ? weight<R>(s[i + e].x, s[i + e].y) : 0.0;
  }
}

// One wavefront per chunk (no workgroup barriers): the rows in order, then a
// fixed butterfly over the lanes.  Also clears the scan's counter.
template <typename R>
__global__ void __launch_bounds__(256) k_chunk_sums(const C<R>* s, uint64_t n, uint64_t nchunks, double* sums,
                                                    unsigned* count) {
  constexpr int E = kRowEntries<R> / 64, ROWS = kChunk / kRowEntries<R>;
  if (blockIdx.x == 0 && threadIdx.x == 0) *count = 0;
  const int lane = threadIdx.x & 63;
  const uint64_t nw = (uint64_t)gridDim.x * 4;
  for (uint64_t c = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6); c < nchunks; c += nw) {
    double t = 0.0;
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
      double p[E];
      row_weights<R, E>(s, n, c * kChunk, r, lane, p);
#pragma unroll
      for (int e = 0; e < E; e++) t += p[e];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
    if (lane == 0) sums[c] = t;
  }
}

// Exclusive scan of x over the workgroup's 256 threads in two serial levels of
// 16: *outer is the sum of the groups of 16 threads before this thread's,
// *inner that of the threads before it in its group; returns the total.  With
// serial sums, and prefixes added from the inside out (outer + (inner + own)),
// the prefix after an entry is that before the next one, bit for bit: prefixes
// never decrease, and an entry of 0 leaves them as they are.  A tree's prefixes
// do not: an empty chunk's start could lie an ulp below the next chunk's, and
// a target between the two found no probability in its chunk.  32 dependent
// additions instead of a tree's 9: 8192 shots of 2^24 complex64 amplitudes
// take 89.2 us a call (88.7 with the tree).
__device__ __forceinline__ double block_scan(double x, double* outer, double* inner) {
  __shared__ double v[16 * 17], g[16];
  const int grp = threadIdx.x >> 4, at = grp * 17 + (threadIdx.x & 15);  // 17: off the same banks
  __syncthreads();
  v[at] = x;
  __syncthreads();
  if (threadIdx.x < 16) {
    double t = 0.0;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const double y = v[threadIdx.x * 17 + i];
      v[threadIdx.x * 17 + i] = t;
      t += y;
    }
    g[threadIdx.x] = t;
  }
  __syncthreads();
  double total = 0.0, before = 0.0;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    if (i == grp) before = total;
    total += g[i];
  }
  *outer = before;
  *inner = v[at];
  return total;
}

// pre[k]: sum of this workgroup's chunks before k (in place of the sums);
// off[b]: sum of the workgroups before b, off[gridDim.x] = T.  The starts
// off + pre never decrease and are equal up to the next chunk that holds
// probability (see block_scan).  One workgroup over all chunks took 20 us at
// 8192 chunks and grew with them.
__global__ void __launch_bounds__(256) k_chunk_scan(double* pre, uint64_t nchunks, double* off, unsigned* count) {
  __shared__ int last;
  const uint64_t b0 = (uint64_t)blockIdx.x * kScanRun;
  constexpr int P = kScanRun / 256;  // consecutive chunks per thread
  double x[P], mine = 0.0, outer, inner;
#pragma unroll
  for (int i = 0; i < P; i++) {
    const uint64_t k = b0 + (uint64_t)threadIdx.x * P + i;
    x[i] = k < nchunks ? pre[k] : 0.0;
    mine += x[i];
  }
  const double total = block_scan(mine, &outer, &inner);
  double run = 0.0;
#pragma unroll
  for (int i = 0; i < P; i++) {
    const uint64_t k = b0 + (uint64_t)threadIdx.x * P + i;
    if (k < nchunks) pre[k] = outer + (inner + run);
    run += x[i];
  }
  if (threadIdx.x == 0) {
    // the totals cross the XCDs' caches: complete before the count is raised
    __hip_atomic_store(off + blockIdx.x, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    last = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
  }
  __syncthreads();
  if (!last) return;
  // the last workgroup scans the workgroups' totals the same way
  const unsigned per = (gridDim.x + 255) / 256, r0 = threadIdx.x * per;
  auto load = [&](unsigned k) {
    return k < gridDim.x ? __hip_atomic_load(off + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.0;
  };
  mine = 0.0;
  for (unsigned i = 0; i < per; i++) mine += load(r0 + i);
  const double T = block_scan(mine, &outer, &inner);
  run = 0.0;
  for (unsigned i = 0; i < per; i++) {
    const unsigned k = r0 + i;
    const double y = load(k);
    if (k < gridDim.x) off[k] = outer + (inner + run);
    run += y;
  }
  if (threadIdx.x == 0) off[gridDim.x] = T;
}

// Where a shot's uniform comes from: the caller's array, one value for all
// (u null), or the counter stream u(seed, traj, draw0 + shot).
struct Uniforms {
  const double* u;
  double u0;
  uint64_t seed, traj, draw0;
  int stream;
};

// One wavefront per shot.
template <typename R>
__global__ void __launch_bounds__(256) k_sample_find(const C<R>* s, uint64_t n, const double* pre, const double* off,
                                                     uint64_t nchunks, Uniforms un, int64_t shots, uint64_t* out,
                                                     uint8_t* flag) {
  constexpr int E = kRowEntries<R> / 64, ROWS = kChunk / kRowEntries<R>;
  const int lane = threadIdx.x & 63;
  const int64_t shot = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (shot >= shots) return;  // whole wavefronts leave together
  const uint64_t nrun = (nchunks + kScanRun - 1) / kScanRun;
  const double T = off[nrun];
  const double u = un.stream ? uniform(un.seed, un.traj, un.draw0 + (uint64_t)shot) : un.u ? un.u[shot] : un.u0;
  const double tgt = u * T;
  // largest run, then largest chunk in it, that starts at or below the target
  uint64_t lo = 0, hi = nrun;
  while (hi - lo > 1) {
    const uint64_t mid = lo + (hi - lo) / 2;
    if (off[mid] <= tgt) lo = mid;
    else hi = mid;
  }
  const double o0 = off[lo];
  lo *= kScanRun;
  hi = std::min<uint64_t>(lo + kScanRun, nchunks);
  while (hi - lo > 1) {
    const uint64_t mid = lo + (hi - lo) / 2;
    if (o0 + pre[mid] <= tgt) lo = mid;
    else hi = mid;
  }
  const uint64_t base = lo * kChunk;
  double p[ROWS][E];
#pragma unroll
  for (int r = 0; r < ROWS; r++) row_weights<R, E>(s, n, base, r, lane, p[r]);
  // the first row that ends past the target; if rounding leaves none, the
  // last entry holding probability
  double c = o0 + pre[lo], before = c;
  int row = -1, last_row = -1;
  double last_before = c;
#pragma unroll
  for (int r = 0; r < ROWS; r++) {
    if (row >= 0) continue;  // the same in every lane
    double q = p[r][0];
    if (E > 1) q += p[r][E - 1];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) q += __shfl_xor(q, o, 64);
    if (q > 0.0) {
      last_row = r;
      last_before = c;
    }
    if (q > 0.0 && c + q > tgt) {
      row = r;
      before = c;
    }
    c += q;
  }
  const bool past = row < 0;
  if (past) {
    row = last_row;
    before = last_before;
  }
  if (row < 0) {  // a chunk without probability (a state of zeros or NaN)
    if (lane == 0) {
      out[shot] = 0;
      flag[shot] = 1;
    }
    return;
  }
  double w[E];
#pragma unroll
  for (int e = 0; e < E; e++) w[e] = 0.0;
#pragma unroll
  for (int r = 0; r < ROWS; r++)
    if (r == row)
#pragma unroll
      for (int e = 0; e < E; e++) w[e] = p[r][e];
  double mine = w[0];
  if (E > 1) mine += w[E - 1];
  double incl = mine;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double v = __shfl_up(incl, o, 64);
    if (lane >= o) incl += v;
  }
  const uint64_t hit = past ? 0 : __ballot(before + incl > tgt && mine > 0.0);
  const uint64_t nz = __ballot(mine > 0.0);
  const int src = hit ? __builtin_ctzll(hit) : 63 - __builtin_clzll(nz);
  if (lane == src) {
    const double l0 = before + (incl - mine);
    int pick = -1, fall = 0;
    double run = l0, lo_c = l0, hi_c = l0, fall_lo = l0, fall_hi = l0;
#pragma unroll
    for (int e = 0; e < E; e++) {
      const double nxt = run + w[e];
      if (w[e] > 0.0) {
        fall = e;
        fall_lo = run;
        fall_hi = nxt;
        if (hit && pick < 0 && tgt < nxt) {
          pick = e;
          lo_c = run;
          hi_c = nxt;
        }
      }
      run = nxt;
    }
    if (pick < 0) {  // past the end by rounding: the last entry with probability
      pick = fall;
      lo_c = fall_lo;
      hi_c = fall_hi;
    }
    out[shot] = base + (uint64_t)row * kRowEntries<R> + (uint64_t)(E * lane + pick);
    flag[shot] = (tgt - lo_c < kBoundaryTol * T || hi_c - tgt < kBoundaryTol * T) ? 1 : 0;
  }
}

static uint64_t chunks_of(int nbits) { return ((1ull << nbits) + kChunk - 1) / kChunk; }
static uint64_t runs_of(uint64_t nchunks) { return (nchunks + kScanRun - 1) / kScanRun; }

// chunk sums / prefix, the runs' offsets and the total, the scan's counter
size_t sample_scratch_bytes(int nbits) {
  const uint64_t nchunks = chunks_of(nbits);
  return sizeof(double) * (nchunks + runs_of(nchunks) + 2);
}

template <typename R>
static void launch_sample_t(const void* state, int nbits, hipStream_t st, void* scratch, int64_t shots,
                            const Uniforms& un, uint64_t* d_out, uint8_t* d_flag) {
  const uint64_t n = 1ull << nbits, nchunks = chunks_of(nbits), nrun = runs_of(nchunks);
  double* pre = (double*)scratch;
  double* off = pre + nchunks;
  unsigned* count = (unsigned*)(off + nrun + 1);
  const unsigned g1 = (unsigned)std::min<uint64_t>((nchunks + 3) / 4, 1u << 16);
  hipLaunchKernelGGL(k_chunk_sums<R>, dim3(g1), dim3(256), 0, st, (const C<R>*)state, n, nchunks, pre, count);
  hipLaunchKernelGGL(k_chunk_scan, dim3((unsigned)nrun), dim3(256), 0, st, pre, nchunks, off, count);
  hipLaunchKernelGGL(k_sample_find<R>, dim3((unsigned)((shots + 3) / 4)), dim3(256), 0, st, (const C<R>*)state, n,
                     (const double*)pre, (const double*)off, nchunks, un, shots, d_out, d_flag);
}

static int launch_sample_u(const void* state, int prec, int nbits, hipStream_t st, void* scratch, int64_t shots,
                           const Uniforms& un, uint64_t* d_out, uint8_t* d_flag) {
  if (prec == BT_C64) launch_sample_t<float>(state, nbits, st, scratch, shots, un, d_out, d_flag);
  else launch_sample_t<double>(state, nbits, st, scratch, shots, un, d_out, d_flag);
  BT_HIP(hipGetLastError());
  return BT_OK;
}

int launch_sample(const void* state, int prec, int nbits, hipStream_t st, void* scratch, int64_t shots,
                  const double* d_u, double u0, uint64_t* d_out, uint8_t* d_flag) {
  return launch_sample_u(state, prec, nbits, st, scratch, shots, Uniforms{d_u, u0, 0, 0, 0, 0}, d_out, d_flag);
}

// What bt_sample keeps with a state: device scratch and a pinned buffer (the
// uniforms in, indices and flags out, read and written by the kernels in
// place), so that a call is three launches and one wait.  At most
// kSampleKeep bytes of each; a larger request allocates for itself.
constexpr size_t kSampleKeep = 32ull << 20;

struct SampleBuffers {
  void* dev = nullptr;
  void* host = nullptr;
  size_t dev_bytes = 0, host_bytes = 0;
};

static void free_buffers(SampleBuffers* b) {
  if (b->dev) (void)hipFree(b->dev);
  if (b->host) (void)hipHostFree(b->host);
  *b = SampleBuffers();
}

void free_sample_res(SampleBuffers* b) {
  if (!b) return;
  free_buffers(b);
  delete b;
}

static bool grow_buffers(SampleBuffers* b, size_t dev, size_t host) {
  if (dev > b->dev_bytes) {
    if (b->dev) (void)hipFree(b->dev);
    b->dev = nullptr;
    b->dev_bytes = 0;
    if (hipMalloc(&b->dev, dev) != hipSuccess) return false;
    b->dev_bytes = dev;
  }
  if (host > b->host_bytes) {
    if (b->host) (void)hipHostFree(b->host);
    b->host = nullptr;
    b->host_bytes = 0;
    if (hipHostMalloc(&b->host, host) != hipSuccess) return false;
    b->host_bytes = host;
  }
  return true;
}

// Shots of state s with uniforms u (or un's stream): indices and the number
// flagged as near a boundary.
static int sample_shots(bt_state_s* s, int64_t shots, const double* u, Uniforms un, uint64_t* out, int64_t* nboundary) {
  const size_t sc = sample_scratch_bytes(s->nbits);
  const size_t ub = u ? sizeof(double) * (size_t)shots : 0, ob = sizeof(uint64_t) * (size_t)shots;
  const size_t host = ub + ob + (size_t)shots;
  SampleBuffers own;
  SampleBuffers* b = &own;
  if (sc <= kSampleKeep && host <= kSampleKeep) {  // powers of two: a few sizes over a state's life
    if (!s->sample) s->sample = new SampleBuffers();
    b = s->sample;
  }
  auto up = [&](size_t x) {
    if (b == &own) return x;
    size_t p = 4096;
    while (p < x) p *= 2;
    return p;
  };
  if (!grow_buffers(b, up(sc), up(host))) {
    (void)hipGetLastError();
    free_buffers(&own);
    return fail(BT_ERR_NOMEM, "bt_sample: buffers");
  }
  if (u) {
    memcpy(b->host, u, ub);
    un.u = (const double*)b->host;
  }
  uint64_t* h_out = (uint64_t*)((char*)b->host + ub);
  uint8_t* h_flag = (uint8_t*)b->host + ub + ob;
  int rc = launch_sample_u(s->d, s->prec, s->nbits, s->stream, b->dev, shots, un, h_out, h_flag);
  if (hipStreamSynchronize(s->stream) != hipSuccess && rc == BT_OK) rc = fail(BT_ERR_HIP, "bt_sample: sync");
  if (rc == BT_OK) {
    memcpy(out, h_out, ob);
    int64_t nb = 0;
    for (int64_t i = 0; i < shots; i++) nb += h_flag[i];
    if (nboundary) *nboundary = nb;
  }
  free_buffers(&own);
  return rc;
}

// ---------------------------------------------------------------------------
// the no-allocation variant's scratch: one static device array per GPU
// ---------------------------------------------------------------------------
// Holds the chunks' prefixes (in place of their sums), the runs' offsets and
// the scan's counter, the shots' uniforms, indices and boundary flags, and the
// boundary count: 32 MiB covers a 2^30-amplitude state (4 MiB of prefixes) with
// about 1.7 million shots of 17 bytes.  In host code the array's
// name is not a device address: kernels and copies take the address that
// hipGetSymbolAddress returned for the current device (noalloc_setup).
constexpr size_t kNoAllocScratch = 32ull << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratch];
constexpr int kMaxDevices = 64;
static void* g_scratch_ptr[kMaxDevices] = {};

// Once per device, with that device current (the library's device set-up).
int noalloc_setup(int device) {
  if (device < 0 || device >= kMaxDevices) return fail(BT_ERR_ARG, "noalloc_setup: device index out of range");
  if (g_scratch_ptr[device]) return BT_OK;
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p)
    return fail(BT_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
  g_scratch_ptr[device] = p;
  return BT_OK;
}

// Number of flagged shots, written (not accumulated) to *cnt: one workgroup.
__global__ void __launch_bounds__(256) k_count_flags(const uint8_t* flag, int64_t shots, int64_t* cnt) {
  __shared__ int64_t red[256];
  int64_t t = 0;
  for (int64_t i = threadIdx.x; i < shots; i += 256) t += flag[i];
  red[threadIdx.x] = t;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *cnt = red[0];
}

}  // namespace bt

using namespace bt;

extern "C" int bt_sample_noalloc(bt_state s, int64_t shots, const double* u, uint64_t* out, int64_t* nboundary) {
  if (!s) return fail(BT_ERR_ARG, "null state");
  if (s->kind != BT_SV) return fail(BT_ERR_UNSUPPORTED, "bt_sample_noalloc: state vectors only");
  if (shots < 0 || (shots > 0 && (!u || !out))) return fail(BT_ERR_ARG, "bt_sample_noalloc: bad arguments");
  if (shots == 0) {
    if (nboundary) *nboundary = 0;
    return BT_OK;
  }
  for (int64_t i = 0; i < shots; i++)
    if (!(u[i] >= 0.0 && u[i] < 1.0)) return fail(BT_ERR_ARG, "bt_sample_noalloc: uniforms must lie in [0, 1)");
  const size_t sc = (sample_scratch_bytes(s->nbits) + 255) / 256 * 256;
  const size_t ub = sizeof(double) * (size_t)shots, ob = sizeof(uint64_t) * (size_t)shots, fb = (size_t)shots;
  const size_t need = sc + ub + ob + (fb + 7) / 8 * 8 + sizeof(int64_t);
  if (need > kNoAllocScratch)
    return fail(BT_ERR_ARG, "bt_sample_noalloc: state and shots need " + std::to_string(need) +
                                " bytes of scratch, more than its " + std::to_string(kNoAllocScratch) +
                                " (use bt_sample)");
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices || !g_scratch_ptr[dev])
    return fail(BT_ERR_STATE, "bt_sample_noalloc: the device's scratch is not set up (bt_init)");
  char* base = (char*)g_scratch_ptr[dev];
  double* d_u = (double*)(base + sc);
  uint64_t* d_out = (uint64_t*)(base + sc + ub);
  uint8_t* d_flag = (uint8_t*)(base + sc + ub + ob);
  int64_t* d_cnt = (int64_t*)(base + sc + ub + ob + (fb + 7) / 8 * 8);
  int64_t nb = 0;
  int rc = BT_OK;
  if (hipMemcpyAsync(d_u, u, ub, hipMemcpyHostToDevice, s->stream) != hipSuccess)
    rc = fail(BT_ERR_HIP, "bt_sample_noalloc: upload");
  if (rc == BT_OK) rc = launch_sample(s->d, s->prec, s->nbits, s->stream, base, shots, d_u, 0.0, d_out, d_flag);
  if (rc == BT_OK) {
    hipLaunchKernelGGL(k_count_flags, dim3(1), dim3(256), 0, s->stream, (const uint8_t*)d_flag, shots, d_cnt);
    if (hipGetLastError() != hipSuccess) rc = fail(BT_ERR_HIP, "bt_sample_noalloc: count launch");
  }
  if (rc == BT_OK && (hipMemcpyAsync(out, d_out, ob, hipMemcpyDeviceToHost, s->stream) != hipSuccess ||
                      hipMemcpyAsync(&nb, d_cnt, sizeof nb, hipMemcpyDeviceToHost, s->stream) != hipSuccess))
    rc = fail(BT_ERR_HIP, "bt_sample_noalloc: download");
  if (hipStreamSynchronize(s->stream) != hipSuccess && rc == BT_OK) rc = fail(BT_ERR_HIP, "bt_sample_noalloc: sync");
  if (rc) return rc;
  if (nboundary) *nboundary = nb;
  return BT_OK;
}

extern "C" int bt_sample(bt_state s, int64_t shots, const double* u, uint64_t* out, int64_t* nboundary) {
  if (!s) return fail(BT_ERR_ARG, "null state");
  if (s->kind != BT_SV) return fail(BT_ERR_UNSUPPORTED, "bt_sample: state vectors only (sample, ops.jl:46-60)");
  if (shots < 0 || (shots > 0 && (!u || !out))) return fail(BT_ERR_ARG, "bt_sample: bad arguments");
  if (shots == 0) {
    if (nboundary) *nboundary = 0;
    return BT_OK;
  }
  for (int64_t i = 0; i < shots; i++)
    if (!(u[i] >= 0.0 && u[i] < 1.0)) return fail(BT_ERR_ARG, "bt_sample: uniforms must lie in [0, 1)");
  return sample_shots(s, shots, u, Uniforms{nullptr, 0.0, 0, 0, 0, 0}, out, nboundary);
}

extern "C" int bt_sample_stream(bt_state s, int64_t shots, uint64_t seed, uint64_t traj, uint64_t draw0, uint64_t* out,
                                int64_t* nboundary) {
  if (!s) return fail(BT_ERR_ARG, "null state");
  if (s->kind != BT_SV) return fail(BT_ERR_UNSUPPORTED, "bt_sample_stream: state vectors only (sample, ops.jl:46-60)");
  if (shots < 0 || (shots > 0 && !out)) return fail(BT_ERR_ARG, "bt_sample_stream: bad arguments");
  if (shots == 0) {
    if (nboundary) *nboundary = 0;
    return BT_OK;
  }
  return sample_shots(s, shots, nullptr, Uniforms{nullptr, 0.0, seed, traj, draw0, 1}, out, nboundary);
}
