// The tile pass on the CPU, one thread's step at a time.  Reached by the host
// emulation of the executors only (tests/emu): it runs the passes that the
// planner and build_geom make, with their slot tables, relabelling and operator
// order, and so checks those.  The kernels have their own forms of these steps
// (tile_pass and what it calls, in bt_tile.hpp), which the GPU tests check.
#pragma once

#include "bt_tile.hpp"

namespace bt {

template <typename R, int MASK>
inline void apply_reg(C<R>* v, const C<R>* mats) {
  constexpr int K = __builtin_popcount(MASK);
  constexpr int D = 1 << K;
  constexpr int NR = 1 << TileCfg<R>::RB;
  int P[K > 0 ? K : 1];
  {
    int c = 0;
#pragma unroll
    for (int j = 0; j < kRB; j++)
      if ((MASK >> j) & 1) P[c++] = j;
  }
#pragma unroll
  for (int base = 0; base < NR; base++) {
    if (base & MASK) continue;
    C<R> x[D];
#pragma unroll
    for (int l = 0; l < D; l++) {
      int idx = base;
#pragma unroll
      for (int j = 0; j < K; j++)
        if ((l >> j) & 1) idx |= 1 << P[j];
      x[l] = v[idx];
    }
#pragma unroll
    for (int r = 0; r < D; r++) {
      C<R> acc = cmake<C<R>>(0, 0);
#pragma unroll
      for (int c = 0; c < D; c++) acc = cfma(acc, mats[r + c * D], x[c]);
      int idx = base;
#pragma unroll
      for (int j = 0; j < K; j++)
        if ((r >> j) & 1) idx |= 1 << P[j];
      v[idx] = acc;
    }
  }
}

template <typename R>
inline void apply_mask(int mask, C<R>* v, const C<R>* m) {
  switch (mask) {
#define BT_CASE(M) \
  case M: apply_reg<R, M>(v, m); break;
#define BT_CASE5(M)                                   \
  case M:                                             \
    if constexpr (TileCfg<R>::RB == 5) apply_reg<R, M>(v, m); \
    break;
    BT_CASE(1) BT_CASE(2) BT_CASE(4) BT_CASE(8) BT_CASE(3) BT_CASE(5) BT_CASE(6) BT_CASE(9) BT_CASE(10) BT_CASE(12)
    BT_CASE5(16) BT_CASE5(17) BT_CASE5(18) BT_CASE5(20) BT_CASE5(24)
#undef BT_CASE
#undef BT_CASE5
    default: break;
  }
}

// A matched phase template: the operators' register applications in order,
// straight-line (the masks are compile-time constants of each case).
template <typename R>
inline void apply_template(int tm, C<R>* v, const C<R>* mats, const ROp* ops) {
#define BT_A(M, I) apply_reg<R, M>(v, mats + ops[I].moff);
  switch (tm) {
    case 1:
      BT_A(0x0c, 0)
      BT_A(0x03, 1)
      BT_A(0x06, 2)
      break;
    case 2:
      BT_A(0x0c, 0)
      BT_A(0x03, 1)
      break;
    case 3:
      BT_A(0x03, 0)
      break;
    default:
      break;
  }
#undef BT_A
}

// reduced rho over register positions P0 < P1 (K = 1 or 2), packed as
// diagonal then (a < b) Re, Im of rho[a, b]; index bit j <-> P_j
template <typename R, int MASK>
inline void rho_reg(const C<R>* v, int nvalid_mask, double* racc) {
  constexpr int K = __builtin_popcount(MASK);
  constexpr int D = 1 << K;
  constexpr int NR = 1 << TileCfg<R>::RB;
  int P[K];
  {
    int c = 0;
#pragma unroll
    for (int j = 0; j < kRB; j++)
      if ((MASK >> j) & 1) P[c++] = j;
  }
#pragma unroll
  for (int base = 0; base < NR; base++) {
    if (base & MASK) continue;
    if (base & nvalid_mask) continue;  // phantom registers
    double vr[D], vi[D];
#pragma unroll
    for (int l = 0; l < D; l++) {
      int idx = base;
#pragma unroll
      for (int j = 0; j < K; j++)
        if ((l >> j) & 1) idx |= 1 << P[j];
      vr[l] = (double)v[idx].x;
      vi[l] = (double)v[idx].y;
    }
    int p = D;
#pragma unroll
    for (int a = 0; a < D; a++) {
      racc[a] += vr[a] * vr[a] + vi[a] * vi[a];
#pragma unroll
      for (int b = a + 1; b < D; b++) {
        racc[p] += vr[a] * vr[b] + vi[a] * vi[b];
        racc[p + 1] += vi[a] * vr[b] - vr[a] * vi[b];
        p += 2;
      }
    }
  }
}

template <typename R>
inline void rho_mask(int mask, const C<R>* v, int nvalid_mask, double* racc) {
  switch (mask) {
#define BT_CASE(M) \
  case M: rho_reg<R, M>(v, nvalid_mask, racc); break;
#define BT_CASE5(M)                                                \
  case M:                                                          \
    if constexpr (TileCfg<R>::RB == 5) rho_reg<R, M>(v, nvalid_mask, racc); \
    break;
    BT_CASE(1) BT_CASE(2) BT_CASE(4) BT_CASE(8) BT_CASE(3) BT_CASE(5) BT_CASE(6) BT_CASE(9) BT_CASE(10) BT_CASE(12)
    BT_CASE5(16) BT_CASE5(17) BT_CASE5(18) BT_CASE5(20) BT_CASE5(24)
#undef BT_CASE
#undef BT_CASE5
    default: break;
  }
}

// k >= 3 operator on the tile in LDS (swizzled), thread tid of the block
template <typename R, int K>
inline void apply_lds(C<R>* lds, int T, const ROp& op, const C<R>* mats, uint32_t tid) {
  constexpr int NT = TileCfg<R>::NT;
  constexpr int D = 1 << K;
  const uint32_t ng = 1u << (T - K);
  for (uint32_t g = tid; g < ng; g += NT) {
    uint32_t lb = g;
#pragma unroll
    for (int i = 0; i < K; i++) lb = ins0(lb, op.lsorted[i]);
    C<R> x[D];
#pragma unroll
    for (int l = 0; l < D; l++) x[l] = lds[swz<R>(lb + op.loff[l])];
#pragma unroll 1
    for (int r = 0; r < D; r++) {  // rows one at a time: the D*D entries stay in LDS
      C<R> acc = cmake<C<R>>(0, 0);
#pragma unroll
      for (int c = 0; c < D; c++) acc = cfma(acc, mats[r + c * D], x[c]);
      lds[swz<R>(lb + op.loff[r])] = acc;
    }
  }
}

// Reduced rho over three tile bits: thread tid takes packed entry e = tid / 4
// and the index groups tid % 4, tid % 4 + 4, ...; returns e (-1: no entry)
// and the thread's partial sums.
template <typename R>
inline int rho3_partial(const C<R>* lds, const PassGeom& g, uint32_t tid, double* xr,
                                                     double* xi) {
  const int e = (int)(tid >> 2);
  *xr = 0.0;
  *xi = 0.0;
  if (e >= 36) return -1;
  int a, b;
  rho3_pair(e, &a, &b);
  rho3_sum<R>(lds, g.T, g.red_loff[a], g.red_loff[b], g.red_ls, tid & 3, xr, xi);
  return e;
}

// Local index of thread t's register r under a layout: thread bits are the
// local bits not in registers, ascending, holding t's bits in order.
inline uint32_t thread_base(const int8_t* rb, int T, uint32_t t) {
  uint32_t regm = 0;
#pragma unroll
  for (int j = 0; j < kRB; j++)
    if (rb[j] >= 0) regm |= 1u << rb[j];
  uint32_t base = 0;
  int i = 0;
  for (int b = 0; b < T; b++)
    if (!((regm >> b) & 1)) {
      base |= ((t >> i) & 1u) << b;
      i++;
    }
  return base;
}

// Slot of thread tid's register 0 under a layout (XOR of its bits' slots).
inline uint32_t slot_base(const LSlots& s, uint32_t tid) {
  uint32_t b = 0;
#pragma unroll
  for (int i = 0; i < kTB; i++)
    if ((tid >> i) & 1) b ^= s.ts[i];
  return b;
}

// XOR of the register-position slots of register r (uniform across the workgroup)
inline uint32_t reg_slot(const LSlots& s, int r) {
  uint32_t u = 0;
#pragma unroll
  for (int j = 0; j < kRB; j++)
    if ((r >> j) & 1) u ^= s.rs[j];
  return u;
}

template <typename R>
inline void regs_to_lds(const C<R>* v, C<R>* lds, const LSlots& S, uint32_t tid,
                                                     bool active, int nvalid_mask) {
  constexpr int NR = 1 << TileCfg<R>::RB;
  const uint32_t s0 = slot_base(S, tid);
  if (active && nvalid_mask == 0) {
#pragma unroll
    for (int r = 0; r < NR; r++) lds[s0 ^ reg_slot(S, r)] = v[r];
  } else {
#pragma unroll
    for (int r = 0; r < NR; r++)
      if (active && !(r & nvalid_mask)) lds[s0 ^ reg_slot(S, r)] = v[r];
  }
}

// Reads are unconditional (straight-line, so they issue back to back):
// inactive threads pass a mirrored tid < 2^tb and phantom registers alias a
// valid one; such values are never stored or reduced.
template <typename R>
inline void lds_to_regs(C<R>* v, const C<R>* lds, const LSlots& S, uint32_t ltid) {
  constexpr int NR = 1 << TileCfg<R>::RB;
  const uint32_t s0 = slot_base(S, ltid);
#pragma unroll
  for (int r = 0; r < NR; r++) v[r] = lds[s0 ^ reg_slot(S, r)];
}

// Per-thread constants of a pass: offsets (in amplitudes, from the tile's
// first amplitude) of the load / store layouts.  O = uint32_t when every
// tile bit is below 32 (states of up to 2^32 amplitudes), else uint64_t.
// Threads >= 2^tb are inactive; their loads mirror thread tid mod 2^tb, so
// every address is inside the state.
template <typename O>
struct ThreadIO {
  O gin[kRB], gout[kRB];
  O gthr_in, gthr_out;
  uint32_t tid, ltid;
  bool active;
  int nvalid_mask;  // register bits beyond nrb are phantom
};

template <typename R, typename O>
inline void thread_io(const PassGeom& g, uint32_t tid, ThreadIO<O>& io) {
  constexpr int NR = 1 << TileCfg<R>::RB;
  io.tid = tid;
  io.active = tid < (1u << g.tb);
  io.ltid = tid & ((1u << g.tb) - 1u);
  io.nvalid_mask = (NR - 1) & ~((1 << g.nrb) - 1);
#pragma unroll
  for (int j = 0; j < kRB; j++) {
    io.gin[j] = g.io_in[j] >= 0 ? (O)1 << g.tile[g.io_in[j]] : 0;
    io.gout[j] = g.io_out[j] >= 0 ? (O)1 << g.tile[g.io_out[j]] : 0;
  }
  io.gthr_in = 0;
  io.gthr_out = 0;
  const uint32_t bi = thread_base(g.io_in, g.T, io.ltid), bo = thread_base(g.io_out, g.T, io.ltid);
  for (int b = 0; b < g.T; b++) {
    if ((bi >> b) & 1) io.gthr_in |= (O)1 << g.tile[b];
    if ((bo >> b) & 1) io.gthr_out |= (O)1 << g.tile[b];
  }
}

// global index of tile t's first amplitude
inline uint64_t tile_base(const PassGeom& g, uint64_t t) {
  uint64_t base = 0;
  for (int i = 0; i < g.nrun; i++) {
    const int len = g.run_len[i];
    base |= (t & ((1ull << len) - 1ull)) << g.run_dst[i];
    t >>= len;
  }
  return base;
}

// Issue the loads of a tile's registers (io_in layout) into raw[].  The
// loads are unconditional and straight-line (phantom registers alias a
// valid address) so they are all in flight at once; the device loop issues
// them for the next tile before it computes on the current one.
template <typename R, typename O>
inline void fetch_regs(C<R>* raw, const C<R>* __restrict__ state, const ThreadIO<O>& io,
                                                    uint64_t base) {
  constexpr int NR = 1 << TileCfg<R>::RB;
  const C<R>* __restrict__ tp = state + base;
#pragma unroll
  for (int r = 0; r < NR; r++) {
    O off = io.gthr_in;
#pragma unroll
    for (int j = 0; j < kRB; j++)
      if ((r >> j) & 1) off |= io.gin[j];
    raw[r] = tp[off];
  }
}

// Registers of a tile from its fetched values: scaled, and zero where the
// register is phantom or the thread inactive.  fresh != 0: the state is
// |0...0> and nothing was fetched.
template <typename R, typename O>
inline void take_regs(C<R>* v, const C<R>* raw, const ThreadIO<O>& io, uint64_t base,
                                                   R scale, int fresh) {
  constexpr int NR = 1 << TileCfg<R>::RB;
  if (!fresh && io.active && io.nvalid_mask == 0) {  // every register real: no masks
#pragma unroll
    for (int r = 0; r < NR; r++) {
      v[r].x = raw[r].x * scale;
      v[r].y = raw[r].y * scale;
    }
    return;
  }
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const bool ok = io.active && !(r & io.nvalid_mask);
    if (fresh) {
      O off = io.gthr_in;
#pragma unroll
      for (int j = 0; j < kRB; j++)
        if ((r >> j) & 1) off |= io.gin[j];
      v[r] = cmake<C<R>>(ok && base == 0 && off == 0 ? scale : (R)0, (R)0);
    } else {
      v[r].x = ok ? raw[r].x * scale : (R)0;
      v[r].y = ok ? raw[r].y * scale : (R)0;
    }
  }
}

// Store a tile's registers (io_out layout) and accumulate FP64 norm^2 into
// acc[0] and the histogram over g.red_bits into acc[1..2^red_k].
template <typename R, typename O>
inline void store_regs(const C<R>* v, C<R>* __restrict__ state, const PassGeom& g,
                                                    const ThreadIO<O>& io, uint64_t base, double* acc) {
  constexpr int NR = 1 << TileCfg<R>::RB;
  C<R>* __restrict__ tp = state + base;
  const bool slow_hist = g.red == bti::RED_HIST && !g.hist_fast;
  const bool write = g.write, need_norm = g.need_norm;
  double s = 0.0;
  if (io.active && io.nvalid_mask == 0 && !slow_hist) {  // every register real: no masks
    if (write) {
#pragma unroll
      for (int r = 0; r < NR; r++) {
        O off = io.gthr_out;
#pragma unroll
        for (int j = 0; j < kRB; j++)
          if ((r >> j) & 1) off |= io.gout[j];
        tp[off] = v[r];
      }
    }
    if (need_norm) {
#pragma unroll
      for (int r = 0; r < NR; r++) {
        const double w = (double)v[r].x * (double)v[r].x + (double)v[r].y * (double)v[r].y;
        s += w;
      }
    }
  } else {
#pragma unroll
  for (int r = 0; r < NR; r++) {
    O off = io.gthr_out;
#pragma unroll
    for (int j = 0; j < kRB; j++)
      if ((r >> j) & 1) off |= io.gout[j];
    if (io.active && !(r & io.nvalid_mask)) {
      if (g.write) tp[off] = v[r];
      if (g.need_norm) {
        const double w = (double)v[r].x * (double)v[r].x + (double)v[r].y * (double)v[r].y;
        s += w;
        if (slow_hist) {
          int bin = 0;
          const uint64_t gi = base | (uint64_t)off;
          for (int j = 0; j < g.red_k; j++) bin |= (int)((gi >> g.red_bits[j]) & 1ull) << j;
#pragma unroll
          for (int b = 0; b < 16; b++) acc[1 + b] += (bin == b) ? w : 0.0;
        }
      }
    }
  }
  }
  acc[0] += s;
  if (g.red == bti::RED_HIST && g.hist_fast) {  // one bin for all of this thread's amplitudes
    const uint64_t gi = base | (uint64_t)io.gthr_out;
    int bin = 0;
    for (int j = 0; j < g.red_k; j++) bin |= (int)((gi >> g.red_bits[j]) & 1ull) << j;
#pragma unroll
    for (int b = 0; b < 16; b++) acc[1 + b] += (bin == b) ? s : 0.0;
  }
}

inline int rho_reg_mask(const PassGeom& g) {
  return (1 << g.red_bits[0]) | (g.red_k > 1 ? 1 << g.red_bits[1] : 0);
}

}  // namespace bt
