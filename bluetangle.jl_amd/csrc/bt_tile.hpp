// Tile pass shared by the circuit executors.
//
// A pass streams the state through the chip in tiles of 2^T amplitudes whose
// T local bits are the pass's tile bits, one tile at a time per workgroup of
// NT threads.  Its operators are split into phases.  In a phase each thread
// holds 2^RB amplitudes (32 of complex64, 16 of complex128): RB "register bits"
// of the local index are inside the thread and the log2(NT) others select it,
// and the phase's operators act on register bits, complex64 on the FP32 matrix
// cores and complex128 by FMAs, with the register positions fixed at compile
// time (one instantiation per set of positions), so a pass with many fused
// operators costs matrix work, not memory traffic.  Between phases the tile is
// in its LDS image: each phase reads it in its own layout and writes the same slots back,
// and a CNOT or SWAP between two phases only changes which slots the later one
// uses.  Tables of slots and of the load and store layouts come with the pass,
// read through the scalar cache; the layouts that load and store the tile
// keep the low local bits on the threads, so each wavefront touches contiguous
// runs of 64 B or more.  Reductions (norm, histogram over up to 4 bits, reduced
// rho over up to 3 bits) run in FP64 and are added per tile in a fixed order.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstring>

#include "bt_internal.hpp"
#include "bt_interp.hpp"

using bti::Plan;
using bti::PassResult;
using bti::QOp;

namespace bt {

constexpr int kMatEntries = bti::Interp::kPassMatEntries;
// accumulators of a pass: [0] norm^2, then either the histogram (16 bins) or
// the packed reduced rho (diagonal, then Re/Im of rho[a, b] for a < b: 16
// doubles over 2 bits, 64 over 3)
constexpr int kAcc = 65;
constexpr int kRB = 5;     // register bits (most)
constexpr int kTB = 8;     // thread bits (most)
constexpr int kMaxPh = 28;

// 256 threads per workgroup; complex64 takes 32 amplitudes per thread in a
// phase (T = 13), complex128 16 (T = 12): 64 KiB tiles, registers <= 256 per
// lane, two workgroups per CU.  Measured at 2^22 amplitudes x 256 noisy
// trajectories (32 layers): this 320 ms; 512 threads x 16 amplitudes at 128
// registers 341 ms; 512 x 32 on 2^14-amplitude tiles (one workgroup per CU)
// 314 ms there but 22.0 ms against 19.6 on a 2^30-amplitude circuit.
template <typename R>
struct TileCfg;
// WAVES: waves per SIMD the kernels are compiled for (launch-bounds minimum).
template <>
struct TileCfg<float> {
  static constexpr int NT = 256;
  static constexpr int LOGNT = 8;
  static constexpr int RB = 5;
  static constexpr int WAVES = 2;
};
template <>
struct TileCfg<double> {
  static constexpr int NT = 256;
  static constexpr int LOGNT = 8;
  static constexpr int RB = 4;
  static constexpr int WAVES = 2;
};

// An operator of a pass.  k <= 2: applied in registers, `mask` = register
// positions, matrix index bit j <-> j-th lowest position.  k >= 3 (rare:
// 3-bit channels, doubly controlled gates, 2-qubit density-matrix
// superoperators): applied to the tile in LDS, matrix in operand order
// (operand 0 = MSB) at local offsets loff.
struct ROp {
  int32_t k;
  int32_t mask;
  int32_t moff;
  int32_t stage;       // offset in the workgroup's staged operators (complex entries)
  int32_t lsorted[4];  // k >= 3: ascending local bits
  uint32_t loff[16];   // k >= 3: local offset of each matrix index
  uint64_t gctrl;      // control bits outside the tile (global positions)
};

// LDS slots of a layout, precomputed per pass: the tile image is indexed by
// a swizzled local index and the swizzle is XOR-linear, so the slot of
// (thread base | register offset) is the XOR of the slots of its bits.
struct LSlots {
  uint16_t ts[kTB];  // slot of thread-index bit i (0 where the thread bit is unused)
  uint16_t rs[kRB];  // slot of register position j (0 for phantoms)
  uint16_t pad[3];
};

struct RPhase {
  int8_t rb[kRB];  // local tile bit held at register position j (-1: phantom)
  int8_t tmpl;     // > 0: the phase's operators match kPhaseTemplates[tmpl]
  int8_t pad[2];
  int32_t op0, nops;
};

// Register-mask sequences that start a phase and that the device applies as
// one straight-line block (no per-operator dispatch, whose branch chain
// copies the 2^RB live registers at every level); the phase's remaining
// operators follow one by one.  These are the openings layered brickworks
// produce most (two disjoint register pairs).  Phases with out-of-tile
// controls or LDS operators never match.
struct PhaseTemplate {
  int8_t n;
  int8_t mask[4];
};
constexpr PhaseTemplate kPhaseTemplates[] = {
    {0, {0, 0, 0, 0}},
    {3, {0x0c, 0x03, 0x06, 0}},
    {2, {0x0c, 0x03, 0, 0}},
    {1, {0x03, 0, 0, 0}},
};
constexpr int kNumPhaseTemplates = (int)(sizeof(kPhaseTemplates) / sizeof(kPhaseTemplates[0]));

// slot tables of the load / store layouts, and of the store layout in an
// image without relabelling
constexpr int kLayIn = kMaxPh, kLayOut = kMaxPh + 1, kLayEnd = kMaxPh + 2;

struct PassGeom {
  int32_t T, nrb, tb, ncomp, write, need_norm, red, red_k, red_swap, nph, nops, nmats, nstage;
  int32_t hist_fast;         // RED_HIST with no histogram bit in the store layout's registers
  int32_t tile[bti::kMaxT];  // local bit -> global bit
  int32_t comp[40];          // global bits outside the tile, ascending
  int32_t nrun;              // tile index -> global base: runs of consecutive outside bits
  int8_t run_dst[bti::kMaxT + 1], run_len[bti::kMaxT + 1];
  int32_t red_bits[4];       // RED_HIST: global bits; RED_RHO: register positions (last phase), ascending
  int8_t io_in[kRB], io_out[kRB];
  int8_t pad[6];
  // the load / store layouts in global bits: thread-index bit i (0 where
  // unused: that bit of the thread index is never set), register position j
  // (63 for a phantom: it shifts out of a byte offset)
  uint8_t thr_in[12], thr_out[12], reg_in[8], reg_out[8];
  int32_t in_direct, out_direct;  // first phase reads / last phase stores in its own layout
  int32_t top_thr;                // highest global bit on a thread in either layout
  int32_t relabel;                // the image ends the pass relabelled (kLayOut reads it)
  uint64_t outside;               // global bits outside the tile
  uint32_t red_loff[8];      // RED_RHO: local offset of each packed index
  int32_t red_ls[4];         // RED_RHO: the local bits, ascending; RED_HIST: local bit of bin bit j (-1: outside)
  LSlots lay[kMaxPh + 3];    // slot tables: phases, then kLayIn, kLayOut, kLayEnd
  double scale;
  RPhase ph[kMaxPh];
  ROp ops[bti::kPMax];  // last: a packed table holds only the used ones
};

// ---------------------------------------------------------------------------
// host/device: plan + queue slots -> register-tile geometry and matrices
// ---------------------------------------------------------------------------
__host__ __device__ inline int popc32(uint32_t x) { return __builtin_popcount(x); }

// Layout with register positions 0..nrb-1 holding the given local bits
// (ascending) and the rest phantom.
__host__ __device__ inline void set_layout(int8_t* rb, const int* bits, int n) {
  for (int j = 0; j < kRB; j++) rb[j] = j < n ? (int8_t)bits[j] : (int8_t)-1;
}

// LDS element swizzle of local index l: XOR the low W bits with higher bits
// so strided layouts spread over the banks (W = 5 for 8-byte, 4 for 16-byte
// elements).  Linear over XOR.
template <typename R>
__host__ __device__ __forceinline__ uint32_t swz(uint32_t l) {
  constexpr int W = sizeof(C<R>) == 8 ? 5 : 4;
  return l ^ (((l >> W) ^ (l >> (2 * W))) & ((1u << W) - 1u));
}

// at: where the image holds the unit index of each local bit (see LinMap).
template <typename R>
__host__ __device__ inline void make_slots(const int8_t* rb, int T, const uint32_t* at, LSlots* s) {
  uint32_t regm = 0;
  for (int j = 0; j < kRB; j++) {
    if (rb[j] >= 0) regm |= 1u << rb[j];
    s->rs[j] = rb[j] >= 0 ? (uint16_t)swz<R>(at[rb[j]]) : (uint16_t)0;
  }
  int i = 0;
  for (int b = 0; b < T && i < kTB; b++)
    if (!((regm >> b) & 1)) s->ts[i++] = (uint16_t)swz<R>(at[b]);
  for (; i < kTB; i++) s->ts[i] = 0;
  s->pad[0] = s->pad[1] = s->pad[2] = 0;
}

// Operators as the workgroup holds them in LDS: a complex64 operator of one or
// two bits in the lane order of the matrix cores (see op_lane: 16 or 64
// floats), k >= 3 as complex entries; complex128 reads its k <= 2 matrices
// from the pass table instead.  Entries are complex numbers of the pass's
// precision; the most a pass can need follows from its operator and matrix
// limits (kPMax operators, kMatEntries entries: 20 two-bit, one four-bit and
// three three-bit operators).
template <typename R>
__host__ __device__ constexpr int stage_entries(int k) {
  return k >= 3 ? 1 << (2 * k) : sizeof(R) == 4 ? 2 << (2 * k) : 0;
}
template <typename R>
constexpr int kStageEntries = sizeof(R) == 4 ? 1088 : kMatEntries;

// Fill the staged form of a pass's operators (entries t, t + step, ... by
// worker t of `step`).
template <typename R>
__host__ __device__ inline void stage_ops(const PassGeom& g, const C<R>* mats, C<R>* out, int t, int step) {
  for (int o = 0; o < g.nops; o++) {
    const ROp& op = g.ops[o];
    const int n = stage_entries<R>(op.k), D = 1 << op.k;
    for (int e = t; e < n; e += step) {
      C<R> x;
      if (op.k >= 3) {
        x = mats[op.moff + e];
      } else {
        // lane i holds, per 4-row slice h, the coefficients of (Re x_c, Im x_c)
        // in output row 2h + (i >> 1), real part if i is even
        const int i = e / (n / 4), h = (e % (n / 4)) / D, c = e % D;
        const C<R> m = mats[op.moff + 2 * h + (i >> 1) + c * D];
        x = (i & 1) ? cmake<C<R>>(m.y, m.x) : cmake<C<R>>(m.x, -m.y);
      }
      out[op.stage + e] = x;
    }
  }
}

// CNOT, SWAP and their products on two bits map basis states by a linear map
// of their index bits, |j> -> |A j> over GF(2).  The tile image is addressed
// by XORs of one slot per index bit, so such an operator between two phases
// is a change of the slots the later phase uses and costs nothing: the image
// holds the amplitude of local index i at M i, and the operator turns M into
// M A^-1.  The two halves of every CNOT on a density matrix were 4 of the 7
// operators of its phases, and the CNOTs that no rotation absorbs end every
// circuit: exact evolution of 8 qubits, 16 layers 478 -> 355 us, of 12
// qubits, 4 layers 1110 -> 889 us; a 30-qubit circuit of 2 layers 19.3 ->
// 16.7 ms.
// inv2: A^-1 of a two-bit operator given by its expanded column -> row map
// (operand order, operand 0 = bit 1); false if it is no such map.
__host__ __device__ inline bool linear_inverse(const QOp& q, int nc, int* inv2) {
  if (q.k + nc != 2) return false;
  const int D = 1 << q.k;
  int seen = 0;
  for (int c = 0; c < 4; c++) {
    const int cc = c >> q.k, tc = c & (D - 1);
    int row = -1;
    if (cc != (1 << nc) - 1) {
      row = c;
    } else {
      for (int r = 0; r < D; r++) {
        const double re = q.m[2 * (r + tc * D)], im = q.m[2 * (r + tc * D) + 1];
        if (re == 0.0 && im == 0.0) continue;
        if (re != 1.0 || im != 0.0 || row >= 0) return false;
        row = (cc << q.k) | r;
      }
    }
    if (row < 0) return false;
    seen |= 1 << row;
    inv2[row] = c;
  }
  return seen == 15 && inv2[0] == 0;  // a permutation that keeps 0 is linear on two bits
}

template <typename R>
__host__ __device__ __attribute__((noinline)) int build_geom(const Plan& plan, const QOp* slots, int nbits, PassGeom* g,
                                                             C<R>* mats) {
  const int T = plan.ntile;
  g->T = T;
  constexpr int RB = TileCfg<R>::RB;
  g->nrb = T < RB ? T : RB;
  g->tb = T - g->nrb;
  for (int i = 0; i < T; i++) g->tile[i] = plan.tile[i];
  uint64_t tmask = 0;
  for (int i = 0; i < T; i++) tmask |= 1ull << plan.tile[i];
  g->ncomp = 0;
  for (int b = 0; b < nbits; b++)
    if (!((tmask >> b) & 1)) g->comp[g->ncomp++] = b;
  g->nrun = 0;
  for (int i = 0; i < g->ncomp; i++) {
    if (i == 0 || g->comp[i] != g->comp[i - 1] + 1) {
      if (g->nrun > bti::kMaxT) return BT_ERR_UNSUPPORTED;
      g->run_dst[g->nrun] = (int8_t)g->comp[i];
      g->run_len[g->nrun] = 0;
      g->nrun++;
    }
    g->run_len[g->nrun - 1]++;
  }
  int rank[64];
  for (int b = 0; b < 64; b++) rank[b] = -1;
  for (int i = 0; i < T; i++) rank[plan.tile[i]] = i;
  g->write = plan.write;
  g->need_norm = (plan.aligned || plan.red != bti::RED_NONE) ? 1 : 0;
  g->scale = plan.scale;
  g->red = plan.red;
  g->red_k = plan.red_k;
  g->red_swap = 0;
  const int nrb = g->nrb;
  // 1. operators in local bits; in-tile controls become target bits
  int lbits[bti::kPMax][kRB];
  int lk[bti::kPMax];
  for (int o = 0; o < plan.nops; o++) {
    const QOp& q = slots[plan.qidx[o]];
    int nb = 0;
    for (int b = 0; b < nbits; b++)
      if (((q.ctrl >> b) & 1) && rank[b] >= 0) {
        if (nb >= kRB) return BT_ERR_UNSUPPORTED;
        lbits[o][nb++] = rank[b];
      }
    for (int i = 0; i < q.k; i++) {
      if (nb >= kRB) return BT_ERR_UNSUPPORTED;
      lbits[o][nb++] = rank[q.bits[i]];
    }
    if (nb > 4) return BT_ERR_UNSUPPORTED;
    lk[o] = nb;
  }
  // 2. phases: sets of operators whose register bits fit together.
  //    Operators on disjoint qubits commute, so a phase may take any
  //    operator whose predecessors (earlier operators sharing a qubit) are
  //    already placed.  Greedy: each phase is grown from the seed that lets
  //    it take the most operators; within a phase the original order holds.
  const int nops = plan.nops;
  uint32_t opm[bti::kPMax];   // register bits an operator needs (k <= 2)
  uint32_t pred[bti::kPMax];  // operators that must run first
  for (int o = 0; o < nops; o++) {
    opm[o] = 0;
    if (lk[o] <= 2)
      for (int i = 0; i < lk[o]; i++) opm[o] |= 1u << lbits[o][i];
    const QOp& q = slots[plan.qidx[o]];
    uint64_t to = q.ctrl;
    for (int i = 0; i < q.k; i++) to |= 1ull << q.bits[i];
    pred[o] = 0;
    for (int a = 0; a < o; a++) {
      const QOp& qa = slots[plan.qidx[a]];
      uint64_t ta = qa.ctrl;
      for (int i = 0; i < qa.k; i++) ta |= 1ull << qa.bits[i];
      if (ta & to) pred[o] |= 1u << a;
    }
  }
  // Operators that only relabel the tile image (host planning; a pass whose
  // reduction or wide operator reads the image by index keeps them all).
  uint32_t lin = 0;
  int inv2[bti::kPMax][4];
#if !defined(__HIP_DEVICE_COMPILE__)
  if (plan.red == bti::RED_NONE) {
    bool wide = false;
    for (int o = 0; o < nops; o++) {
      const QOp& q = slots[plan.qidx[o]];
      wide = wide || lk[o] >= 3;
      const bool outside = (q.ctrl & ~tmask) != 0;
      if (lk[o] == 2 && !outside && linear_inverse(q, lk[o] - q.k, inv2[o])) lin |= 1u << o;
    }
    if (wide) lin = 0;
  }
#endif
  int nph = 0;
  uint32_t cur = 0;  // register-bit mask of the last phase
  int ph_of[bti::kPMax];
  int exec[bti::kPMax];  // execution order
  int ne = 0;
  uint32_t ph_mask[kMaxPh];
  uint32_t lin_at[kMaxPh + 1];  // linear operators in front of each phase / behind the last
  const uint32_t all = nops >= 32 ? 0xffffffffu : (1u << nops) - 1u;
  auto split = [&](uint32_t lin) -> bool {
    uint32_t done = 0;
    nph = ne = 0;
    cur = 0;
    for (int p = 0; p <= kMaxPh; p++) lin_at[p] = 0;
    for (;;) {
      for (int o = 0; o < nops; o++)
        if (((lin & ~done) >> o) & 1 && !(pred[o] & ~done)) {
          done |= 1u << o;
          lin_at[nph] |= 1u << o;
        }
      if (done == all) return true;
      uint32_t best = 0, best_m = 0;
      int best_n = -1;
      for (int sd = 0; sd < nops; sd++) {
        if (((done | lin) >> sd) & 1 || (pred[sd] & ~done)) continue;
        uint32_t sel = 1u << sd, m = opm[sd];
        int n = 1;
        for (bool grew = true; grew;) {
          grew = false;
          for (int o = 0; o < nops; o++) {
            if (((done | lin | sel) >> o) & 1) continue;
            if (pred[o] & ~(done | sel)) continue;
            if (popc32(m | opm[o]) > nrb) continue;
            sel |= 1u << o;
            m |= opm[o];
            n++;
            grew = true;
          }
        }
        if (n > best_n) {
          best_n = n;
          best = sel;
          best_m = m;
        }
      }
      if (best_n <= 0 || nph >= kMaxPh) return false;
      for (int o = 0; o < nops; o++)
        if ((best >> o) & 1) {
          ph_of[o] = nph;
          exec[ne++] = o;
        }
      ph_mask[nph++] = best_m;
      cur = best_m;
      done |= best;
    }
  };
  bool ok = split(lin);
  if (lin) {
    // Relabelling ends a phase, so it can cost more than it saves.  A phase
    // (an image round trip and a barrier) is 1.5 straight-line operators, an
    // operator behind the phase's opening two (the dispatch moves the
    // registers).
    auto cost = [&]() {
      int c = 0;
      for (int p = 0; p < nph; p++) {
        int n = 0;
        uint32_t first = 0;
        for (int e = 0; e < ne; e++)
          if (ph_of[exec[e]] == p) {
            const bool open = n == 0 || (n == 1 && !(first & opm[exec[e]]));
            c += open ? 2 : 4;
            first |= opm[exec[e]];
            n++;
          }
        c += 3;
      }
      return c + (lin_at[nph] ? 2 : 0);
    };
    const int with = ok ? cost() : 1 << 30;
    if (split(0) && cost() <= with) lin = 0;
    else ok = split(lin);
    if (!lin) ok = true;
  }
  if (!ok) return BT_ERR_UNSUPPORTED;
  uint32_t redm = 0;
  if (plan.red == bti::RED_RHO && plan.red_k == 3) {
    // read from the tile image in LDS after the last phase: no register
    // positions needed, but the pass needs a phase to end
    if (nph == 0) ph_mask[nph++] = 0;
  } else if (plan.red == bti::RED_RHO) {
    for (int i = 0; i < plan.red_k; i++) redm |= 1u << rank[plan.red_bits[i]];
    if (nph == 0 || popc32(cur | redm) > nrb) {
      if (nph >= kMaxPh) return BT_ERR_UNSUPPORTED;
      ph_mask[nph] = 0;
      nph++;
      cur = 0;
    }
    cur |= redm;
    ph_mask[nph - 1] = cur;
  }
  // 3. fill every phase to nrb register bits with the highest free local bits
  //    (the low bits stay on the threads), positions = ascending local bits
  for (int p = 0; p < nph; p++) {
    uint32_t m = ph_mask[p];
    for (int b = T - 1; b >= 0 && popc32(m) < nrb; b--) m |= 1u << b;
    ph_mask[p] = m;
    int bits[kRB], n = 0;
    for (int b = 0; b < T; b++)
      if ((m >> b) & 1) bits[n++] = b;
    set_layout(g->ph[p].rb, bits, n);
    g->ph[p].op0 = 0;
    g->ph[p].nops = 0;
    // Register order: a phase with the same bits as the one before keeps its
    // order (no relayout between them).  Otherwise a relayout enters it
    // anyway, so the order is free: an opening pair of disjoint two-bit
    // operators goes to positions (2,3) then (0,1) and a lone opening pair to
    // (0,1): the straight-line templates.
    if (p > 0 && ph_mask[p] == ph_mask[p - 1] && !lin_at[p]) {
      for (int j = 0; j < kRB; j++) g->ph[p].rb[j] = g->ph[p - 1].rb[j];
      continue;
    }
    int first[2], nf = 0;
    for (int e = 0; e < ne && nf < 2; e++)
      if (ph_of[exec[e]] == p) first[nf++] = exec[e];
    auto pair = [&](int o) { return lk[o] == 2 && popc32(opm[o]) == 2; };
    if (n < 4 || nf == 0 || !pair(first[0])) continue;
    int order[kRB], cnt = 0;
    uint32_t used = 0;
    auto put = [&](uint32_t m) {
      for (int b = 0; b < T; b++)
        if (((m >> b) & 1) && !((used >> b) & 1)) {
          order[cnt++] = b;
          used |= 1u << b;
        }
    };
    if (nf == 2 && pair(first[1]) && !(opm[first[0]] & opm[first[1]])) {
      put(opm[first[1]]);  // positions 0, 1
      put(opm[first[0]]);  // positions 2, 3
    } else {
      put(opm[first[0]]);  // positions 0, 1
    }
    put(ph_mask[p]);  // the rest, ascending
    if (cnt == n) set_layout(g->ph[p].rb, order, n);
  }
  // A relabelling in front of a phase (or the store) needs the image even
  // between equal layouts: the register order says so to what skips the
  // image there (the load and store layouts below; between phases the host
  // emulation, the kernel goes through the image at every phase).
  auto differ = [&](int8_t* rb, const int8_t* from) {
    bool same = true;
    for (int j = 0; j < kRB; j++) same = same && rb[j] == from[j];
    if (same) {
      const int8_t t = rb[0];
      rb[0] = rb[1];
      rb[1] = t;
    }
  };
  for (int p = 1; p < nph; p++)
    if (lin_at[p]) differ(g->ph[p].rb, g->ph[p - 1].rb);
  g->nph = nph;
  // load/store layouts: the top local bits in registers, unless the first /
  // last phase's layout holds at most two of the lowest four local bits in
  // registers (the wavefront still reads whole 128 B lines within a few
  // instructions, and a relayout costs more than the extra requests)
  {
    int bits[kRB], n = 0;
    for (int b = T - nrb; b < T; b++) bits[n++] = b;
    set_layout(g->io_in, bits, n);
    set_layout(g->io_out, bits, n);
    const uint32_t low = (1u << (g->tb < 4 ? g->tb : 4)) - 1u;
    if (nph > 0 && popc32(ph_mask[0] & low) <= 2 && !lin_at[0])
      for (int j = 0; j < kRB; j++) g->io_in[j] = g->ph[0].rb[j];
    if (nph > 0 && popc32(ph_mask[nph - 1] & low) <= 2 && !lin_at[nph])
      for (int j = 0; j < kRB; j++) g->io_out[j] = g->ph[nph - 1].rb[j];
    if (nph > 0 && lin_at[0]) differ(g->io_in, g->ph[0].rb);
    if (lin_at[nph]) differ(g->io_out, nph > 0 ? g->ph[nph - 1].rb : g->io_in);
    // a histogram is cheapest when its bits stay off the store layout's
    // registers: each thread's 2^RB amplitudes then share one bin per tile
    g->hist_fast = 0;
    if (plan.red == bti::RED_HIST) {
      uint32_t lm = 0;
      for (int i = 0; i < plan.red_k; i++)
        if (rank[plan.red_bits[i]] >= 0) lm |= 1u << rank[plan.red_bits[i]];
      uint32_t om = 0;
      for (int j = 0; j < kRB; j++)
        if (g->io_out[j] >= 0) om |= 1u << g->io_out[j];
      if (om & lm) {
        int hb[kRB], m = 0;
        for (int b = T - 1; b >= 0 && m < nrb; b--)
          if (!((lm >> b) & 1)) hb[m++] = b;
        if (m == nrb) {
          for (int i = 0; i < m / 2; i++) {
            const int t = hb[i];
            hb[i] = hb[m - 1 - i];
            hb[m - 1 - i] = t;
          }
          set_layout(g->io_out, hb, m);
          om = 0;
          for (int j = 0; j < kRB; j++)
            if (g->io_out[j] >= 0) om |= 1u << g->io_out[j];
        }
      }
      g->hist_fast = (om & lm) ? 0 : 1;
    }
  }
  // 4. operators in execution order, in register positions, matrices
  //    permuted to the ascending position convention (index bit j <-> j-th
  //    lowest position)
  int moff = 0, nstage = 0;
  g->nops = ne;
  for (int e = 0; e < ne; e++) {
    const int o = exec[e];
    const QOp& q = slots[plan.qidx[o]];
    const RPhase& ph = g->ph[ph_of[o]];
    if (ph.nops == 0) g->ph[ph_of[o]].op0 = e;
    g->ph[ph_of[o]].nops++;
    ROp& r = g->ops[e];
    const int k2 = lk[o], D2 = 1 << k2;
    r.k = k2;
    int pos[kRB];  // register position of lbits[o][i] (k <= 2), else the operand order
    r.mask = 0;
    if (k2 <= 2) {
      for (int i = 0; i < k2; i++)
        for (int j = 0; j < kRB; j++)
          if (ph.rb[j] == lbits[o][i]) pos[i] = j;
      for (int i = 0; i < k2; i++) r.mask |= 1 << pos[i];
    } else {
      for (int i = 0; i < k2; i++) pos[i] = k2 - 1 - i;  // identity: operand order, operand 0 = MSB
      for (int i = 0; i < k2; i++) r.lsorted[i] = lbits[o][i];
      for (int i = 0; i < k2; i++)
        for (int j = i + 1; j < k2; j++)
          if (r.lsorted[j] < r.lsorted[i]) {
            int t = r.lsorted[i];
            r.lsorted[i] = r.lsorted[j];
            r.lsorted[j] = t;
          }
      for (int l = 0; l < D2; l++) {
        uint32_t off = 0;
        for (int i = 0; i < k2; i++)
          if ((l >> (k2 - 1 - i)) & 1) off |= 1u << lbits[o][i];
        r.loff[l] = off;
      }
    }
    r.gctrl = 0;
    for (int b = 0; b < nbits; b++)
      if (((q.ctrl >> b) & 1) && rank[b] < 0) r.gctrl |= 1ull << b;
    // rank of each operand bit among the ascending positions
    int asc[kRB];
    for (int i = 0; i < k2; i++) {
      int c = 0;
      for (int j = 0; j < k2; j++) c += pos[j] < pos[i];
      asc[i] = c;
    }
    const int nc = k2 - q.k;  // leading operand bits are in-tile controls
    const int D = 1 << q.k;
    if (moff + D2 * D2 > kMatEntries) return BT_ERR_UNSUPPORTED;
    r.moff = moff;
    r.stage = nstage;
    nstage += stage_entries<R>(k2);
    for (int nr = 0; nr < D2; nr++)
      for (int ncl = 0; ncl < D2; ncl++) {
        // operand-order indices (operand 0 = MSB) of the new indices
        int orr = 0, occ = 0;
        for (int i = 0; i < k2; i++) {
          orr |= ((nr >> asc[i]) & 1) << (k2 - 1 - i);
          occ |= ((ncl >> asc[i]) & 1) << (k2 - 1 - i);
        }
        const int cr = orr >> q.k, cc = occ >> q.k;
        const int tr = orr & (D - 1), tc = occ & (D - 1);
        double vr = 0, vi = 0;
        if (cr == cc) {
          if (cr == (1 << nc) - 1) {
            vr = q.m[2 * (tr + tc * D)];
            vi = q.m[2 * (tr + tc * D) + 1];
          } else if (tr == tc) {
            vr = 1.0;
          }
        }
        mats[moff + nr + ncl * D2].x = (R)vr;
        mats[moff + nr + ncl * D2].y = (R)vi;
      }
    moff += D2 * D2;
  }
  g->nmats = moff;
  g->nstage = nstage;
  // straight-line phase templates
  for (int p = 0; p < nph; p++) {
    RPhase& ph = g->ph[p];
    ph.tmpl = 0;
    bool plain = ph.nops > 0;
    for (int e = ph.op0; e < ph.op0 + ph.nops && plain; e++)
      plain = g->ops[e].k <= 2 && g->ops[e].gctrl == 0;
    if (!plain) continue;
    for (int t = 1; t < kNumPhaseTemplates; t++) {
      const PhaseTemplate& pt = kPhaseTemplates[t];
      bool ok = pt.n <= ph.nops;  // a template covers the phase's first pt.n operators
      for (int i = 0; i < pt.n && ok; i++) {
        ok = g->ops[ph.op0 + i].mask == pt.mask[i];
        if (TileCfg<R>::RB < 5) ok = ok && pt.mask[i] < 16;
      }
      if (ok) {
        ph.tmpl = (int8_t)t;
        break;
      }
    }
  }
  // the input scale rides on the first operator that every amplitude of
  // every tile goes through (no out-of-tile control), sparing the per-tile
  // multiply of each register
  for (int e = 0; e < ne && g->scale != 1.0; e++) {
    const ROp& r = g->ops[e];
    if (r.gctrl) continue;
    const int D2 = 1 << r.k;
    for (int i = 0; i < D2 * D2; i++) {
      mats[r.moff + i].x = (R)((double)mats[r.moff + i].x * g->scale);
      mats[r.moff + i].y = (R)((double)mats[r.moff + i].y * g->scale);
    }
    g->scale = 1.0;
  }
  auto io_bits = [&](const int8_t* rb, uint8_t* thr, uint8_t* reg) {
    uint32_t regm = 0;
    for (int j = 0; j < 8; j++) {
      const bool real = j < kRB && rb[j] >= 0;
      reg[j] = real ? (uint8_t)plan.tile[rb[j]] : (uint8_t)63;
      if (real) regm |= 1u << rb[j];
    }
    int i = 0;
    for (int b = 0; b < T && i < 12; b++)
      if (!((regm >> b) & 1)) thr[i++] = (uint8_t)plan.tile[b];
    for (; i < 12; i++) thr[i] = 0;
  };
  io_bits(g->io_in, g->thr_in, g->reg_in);
  io_bits(g->io_out, g->thr_out, g->reg_out);
  g->top_thr = 0;
  for (int i = 0; i < g->tb && i < 12; i++) {
    if (g->thr_in[i] > g->top_thr) g->top_thr = g->thr_in[i];
    if (g->thr_out[i] > g->top_thr) g->top_thr = g->thr_out[i];
  }
  g->in_direct = g->out_direct = 1;
  const int8_t* first_rb = nph > 0 ? g->ph[0].rb : g->io_in;
  const int8_t* last_rb = nph > 0 ? g->ph[nph - 1].rb : g->io_in;
  for (int j = 0; j < kRB; j++) {
    if (g->io_in[j] != first_rb[j]) g->in_direct = 0;
    if (g->io_out[j] != last_rb[j]) g->out_direct = 0;
  }
  g->outside = (nbits < 64 ? (1ull << nbits) - 1ull : ~0ull) & ~tmask;
  uint32_t at[bti::kMaxT];
  for (int b = 0; b < T; b++) at[b] = 1u << b;
  make_slots<R>(g->io_in, T, at, &g->lay[kLayIn]);
  make_slots<R>(g->io_out, T, at, &g->lay[kLayEnd]);
  for (int p = 0; p <= nph; p++) {
    for (int o = 0; o < nops; o++)
      if ((lin_at[p] >> o) & 1) {
        const int x = lbits[o][0], y = lbits[o][1];  // operand 0 = bit 1 of the operand index
        const uint32_t ax = at[x], ay = at[y];
        at[x] = (inv2[o][2] & 2 ? ax : 0) ^ (inv2[o][2] & 1 ? ay : 0);
        at[y] = (inv2[o][1] & 2 ? ax : 0) ^ (inv2[o][1] & 1 ? ay : 0);
      }
    if (p < nph) make_slots<R>(g->ph[p].rb, T, at, &g->lay[p]);
    else make_slots<R>(g->io_out, T, at, &g->lay[kLayOut]);
  }
  g->relabel = 0;
  for (int b = 0; b < T; b++)
    if (at[b] != 1u << b) g->relabel = 1;
  // 5. reductions
  if (plan.red == bti::RED_HIST) {
    for (int i = 0; i < plan.red_k; i++) g->red_bits[i] = plan.red_bits[i];
  } else if (plan.red == bti::RED_RHO && plan.red_k == 3) {
    for (int a = 0; a < 8; a++) {
      uint32_t off = 0;
      for (int i = 0; i < 3; i++)
        if ((a >> (2 - i)) & 1) off |= 1u << rank[plan.red_bits[i]];
      g->red_loff[a] = off;
    }
  } else if (plan.red == bti::RED_RHO) {
    const RPhase& ph = g->ph[nph - 1];
    int p[2] = {0, 0};
    for (int i = 0; i < plan.red_k; i++)
      for (int j = 0; j < kRB; j++)
        if (ph.rb[j] == rank[plan.red_bits[i]]) p[i] = j;
    if (plan.red_k == 1) {
      g->red_bits[0] = p[0];
    } else {
      g->red_bits[0] = p[0] < p[1] ? p[0] : p[1];
      g->red_bits[1] = p[0] < p[1] ? p[1] : p[0];
      // packed rho is in ascending-position index order (bit 0 = lower
      // position); the plan wants red_bits[0] as the MSB
      g->red_swap = p[0] < p[1] ? 1 : 0;
    }
    for (int a = 0; a < (1 << plan.red_k); a++) {
      uint32_t off = 0;
      for (int j = 0; j < plan.red_k; j++)
        if ((a >> j) & 1) off |= 1u << ph.rb[g->red_bits[j]];
      g->red_loff[a] = off;
    }
  }
  if (plan.red == bti::RED_RHO) {
    int n = 0;
    for (int b = 0; b < T; b++)
      for (int i = 0; i < plan.red_k; i++)
        if (rank[plan.red_bits[i]] == b) g->red_ls[n++] = b;
  } else if (plan.red == bti::RED_HIST) {  // local bits (-1: outside the tile)
    for (int i = 0; i < plan.red_k; i++) g->red_ls[i] = rank[plan.red_bits[i]];
  }
  return BT_OK;
}

// A pass's table as the launched executors read it: the geometry up to its
// last used operator, the staged operators, and in complex128 the matrices
// (complex64 needs them in staged form only).
inline size_t geom_bytes(int nops) { return (offsetof(PassGeom, ops) + (size_t)nops * sizeof(ROp) + 15) / 16 * 16; }
template <typename R>
constexpr size_t kTableMax =
    (sizeof(PassGeom) + 15) / 16 * 16 + sizeof(C<R>) * (kStageEntries<R> + (sizeof(R) == 8 ? kMatEntries : 0));

// Build a pass's table in `out` (kTableMax<R> bytes, 16-byte aligned);
// *bytes: its size.  *head (nullable): a copy of what the host needs of it.
struct TableHead {
  int32_t red_swap, top_thr, nph;
};
template <typename R>
inline int build_table(const Plan& plan, const QOp* slots, int nbits, unsigned char* out, size_t* bytes,
                       TableHead* head) {
  C<R> mats[kMatEntries];
  PassGeom* g = (PassGeom*)out;
  const int rc = build_geom<R>(plan, slots, nbits, g, mats);
  if (rc) return rc;
  size_t n = geom_bytes(g->nops);
  C<R> staged[kStageEntries<R>];
  stage_ops<R>(*g, mats, staged, 0, 1);
  memcpy(out + n, staged, sizeof(C<R>) * (size_t)g->nstage);
  n += sizeof(C<R>) * (size_t)g->nstage;
  if (sizeof(R) == 8) {
    memcpy(out + n, mats, sizeof(C<R>) * (size_t)g->nmats);
    n += sizeof(C<R>) * (size_t)g->nmats;
  }
  *bytes = n;
  if (head) *head = TableHead{g->red_swap, g->top_thr, g->nph};
  return BT_OK;
}

// Whether a pass's per-thread byte offsets fit 32 bits (then every access is a
// scalar base plus a 32-bit offset per lane), and whether every pass of a
// state of nbits index bits does.
template <typename R>
inline bool narrow_io(const TableHead& h) {
  return h.top_thr + (sizeof(C<R>) == 8 ? 3 : 4) < 32;
}
template <typename R>
inline bool narrow_state(int nbits) {
  return nbits + (sizeof(C<R>) == 8 ? 3 : 4) <= 32;
}

// ---------------------------------------------------------------------------
// device side
// ---------------------------------------------------------------------------
__host__ __device__ __forceinline__ uint32_t ins0(uint32_t x, int b) { return ((x >> b) << (b + 1)) | (x & ((1u << b) - 1u)); }

// Indices a <= b of packed entry e < 36 of a reduced rho over three bits: the 8
// diagonal entries, then the 28 pairs a < b in order (0,1), (0,2), ..., (6,7).
__host__ __device__ __forceinline__ void rho3_pair(int e, int* a, int* b) {
  *a = *b = e;
  if (e < 8) return;
  int p = e - 8, x = 0;
  while (p >= 7 - x) {
    p -= 7 - x;
    x++;
  }
  *a = x;
  *b = x + 1 + p;
}

// Sum over the index groups s, s + 4, ... of the tile image in LDS
// (swizzled): Re (xr) and Im (xi) of rho[a, b], oa / ob the local offsets of
// indices a and b, ls the three local bits, ascending.
template <typename R>
__host__ __device__ __forceinline__ void rho3_sum(const C<R>* lds, int T, uint32_t oa, uint32_t ob, const int* ls,
                                                  uint32_t s, double* xr, double* xi) {
  const uint32_t ng = 1u << (T - 3);
  double sr = 0.0, si = 0.0;
  for (uint32_t grp = s; grp < ng; grp += 4) {
    uint32_t lb = grp;
#pragma unroll
    for (int i = 0; i < 3; i++) lb = ins0(lb, ls[i]);
    const C<R> va = lds[swz<R>(lb + oa)], vb = lds[swz<R>(lb + ob)];
    sr += (double)va.x * (double)vb.x + (double)va.y * (double)vb.y;
    si += (double)va.y * (double)vb.x - (double)va.x * (double)vb.y;
  }
  *xr = sr;
  *xi = si;
}

// packed index of entry e's real part (its imaginary part follows for e >= 8)
__host__ __device__ __forceinline__ int rho3_slot(int e) { return e < 8 ? e : 8 + 2 * (e - 8); }

#if defined(__HIPCC__)
// A double moved across lanes by a DPP pattern (both 32-bit halves).
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  // every lane reads a valid source under these permutations (full row and
  // bank masks), so no "old" value has to be materialised first
  const int lo = __builtin_amdgcn_mov_dpp((int)(uint32_t)u, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}

__device__ __forceinline__ double readlane_f64(double x, int lane) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)u, lane);
  const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// Sum over the 64 lanes of a wavefront in a fixed order (xor-1 and xor-2
// within quads, then the half-row and row mirrors, then the four rows in
// order); the same value in every lane.
__device__ __forceinline__ double wave_sum(double x) {
  x += dpp_f64<0xb1>(x);   // quad_perm [1,0,3,2]
  x += dpp_f64<0x4e>(x);   // quad_perm [2,3,0,1]
  x += dpp_f64<0x141>(x);  // row_half_mirror
  x += dpp_f64<0x140>(x);  // row_mirror
  return (readlane_f64(x, 0) + readlane_f64(x, 16)) + (readlane_f64(x, 32) + readlane_f64(x, 48));
}

#endif

// Hide a value's origin from the optimiser (no instruction is emitted), so
// the per-register offsets built from it are recomputed per tile instead of
// being hoisted out of the tile loop as 64 live registers.
template <typename T>
__host__ __device__ __forceinline__ void opaque(T& x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(x));
#else
  (void)x;
#endif
}

// Wait until every vector-memory access this wave issued has completed
// (s_waitcnt vmcnt(0), the LDS and export counters left alone).
__host__ __device__ __forceinline__ void vm_wait_all() {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_s_waitcnt(0x0F70);
#endif
}

#if defined(__HIPCC__)
// A value the whole workgroup holds in common, moved to scalar registers.

__device__ __forceinline__ uint64_t uniform_u64(uint64_t x) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)x);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
  return ((uint64_t)hi << 32) | lo;
}

// Finish the reductions of one pass over one state in the pass's own launch:
// every workgroup stores its nacc sums (LDS) as partials, accumulator-major
// (part[j * nb + block]); the last of the state's nb workgroups adds them in
// a fixed order that depends on nb and nacc alone (P threads per
// accumulator, each over every P-th workgroup, then a fixed tree) and writes
// the totals to out (pinned host memory): no second launch and no copy.
// The partials cross the XCDs' L2 caches: agent-scope stores, complete before
// the state's count is raised, and agent-scope loads after it.  count:
// kCountWords, see count_last.  red: NT/64 doubles of LDS.  One noisy trajectory of 22
// qubits in 30 passes: 1.29 -> 1.25 ms against a totals launch and a copy.
template <int NT>
__device__ __forceinline__ void item_finish(const double* sums, double* red, double* part, uint32_t block,
                                            uint32_t nb, unsigned* count, double* out, int nacc) {
  __shared__ int last;
  const int tid = threadIdx.x;
  if (nb == 1) {
    if (tid < nacc) out[tid] = sums[tid];
    return;
  }
  if (tid < nacc)
    __hip_atomic_store(part + (uint64_t)tid * nb + block, sums[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's partials have reached the point of coherence
  __syncthreads();
  if (tid == 0) last = count_last(count, block, nb);
  __syncthreads();
  if (!last) return;
  // a power of two of threads per accumulator, 16 at least: a norm alone gets all
  const int P = nacc <= 1 ? NT : nacc <= 2 ? NT / 2 : nacc <= 5 ? NT / 8 : NT / 16;
  static_assert(NT == 256, "thread split of the totals");
  const int W = P < 64 ? P : 64;
  const int q = tid & (P - 1);
  for (int j0 = 0; j0 < nacc; j0 += NT / P) {
    const int j = j0 + tid / P;
    double t = 0.0;
    if (j < nacc) {
      const double* p = part + (uint64_t)j * nb;
      uint32_t b = (uint32_t)q;
      for (; b + 7u * P < nb; b += 8u * P) {  // eight loads in flight
        double x[8];
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] = __hip_atomic_load(p + b + i * P, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int i = 0; i < 8; i++) t += x[i];
      }
      for (; b < nb; b += P) t += __hip_atomic_load(p + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    for (int o = W / 2; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
    if (P > 64) {
      __syncthreads();
      if ((tid & 63) == 0) red[tid >> 6] = t;
      __syncthreads();
      t = 0.0;
      for (int w = 0; w < P / 64; w++) t += red[((tid - q) >> 6) + w];
    }
    if (q == 0 && j < nacc) out[j] = t;
  }
}

// ---------------------------------------------------------------------------
// device pass
// ---------------------------------------------------------------------------
// Where a pass's table (geometry, matrices) lives.  In the launched executors
// it is read-only global memory: every field is the same in all lanes, so it
// is read through the constant address space into scalar registers, costing
// neither vector instructions nor LDS.  The persistent executor builds its
// tables on the device, in LDS.
typedef const __attribute__((address_space(4))) uint32_t* const_words;

struct GeomConst {
  const_words g, m;
  const unsigned char* staged;  // the staged operators, 16-byte aligned
  // a packed table (build_table) of element size `elem`
  __device__ GeomConst(const unsigned char* tab, int elem) : g((const_words)(uintptr_t)tab) {
    const uint32_t nops = w(offsetof(PassGeom, nops)), nstage = w(offsetof(PassGeom, nstage));
    staged = tab + (offsetof(PassGeom, ops) + nops * sizeof(ROp) + 15) / 16 * 16;
    m = (const_words)(uintptr_t)(staged + nstage * (uint32_t)elem);
  }
  __device__ __forceinline__ uint32_t w(size_t byte) const { return g[byte / 4]; }
  // Touch every 64-byte line of what the pass reads through the scalar cache,
  // 16 loads in flight at a time, so that no phase waits for memory on its
  // first use of a line (a complex128 operator's matrix alone is 4 lines: a
  // one-tile circuit of 120 two-bit operators ran at 328 us without it,
  // 303 with it).
  template <typename R>
  __device__ __forceinline__ void warm() const {
    const uint32_t head = (uint32_t)(offsetof(PassGeom, ops) + w(offsetof(PassGeom, nops)) * sizeof(ROp));
    const uint32_t nmat = sizeof(R) == 8 ? w(offsetof(PassGeom, nmats)) * (uint32_t)sizeof(C<R>) : 0u;
    touch(g, head);
    touch(m, nmat);
  }
  static __device__ __forceinline__ void touch(const_words p, uint32_t bytes) {
    uint32_t at = 0;
    for (; at + 1024 <= bytes; at += 1024) {
      uint32_t x[16];
#pragma unroll
      for (int i = 0; i < 16; i++) x[i] = p[at / 4 + 16 * i];
#pragma unroll
      for (int i = 0; i < 16; i++) asm volatile("" ::"s"(x[i]));
    }
    if (at < bytes) {  // the rest: lines past the end repeat the first one
      uint32_t x[16];
#pragma unroll
      for (int i = 0; i < 16; i++) x[i] = p[at + 64 * i < bytes ? at / 4 + 16 * i : at / 4];
#pragma unroll
      for (int i = 0; i < 16; i++) asm volatile("" ::"s"(x[i]));
    }
  }
  __device__ __forceinline__ uint32_t lane_w(size_t byte) const { return g[byte / 4]; }  // a word of each lane's own
  // The same table through a pointer whose origin is hidden from the
  // optimiser: what is read through it is not hoisted out of a loop (dozens of
  // live scalar registers otherwise).
  __device__ __forceinline__ GeomConst again() const {
    GeomConst c = *this;
    uint64_t x = (uint64_t)(uintptr_t)c.g, y = (uint64_t)(uintptr_t)c.m;
    asm volatile("" : "+s"(x), "+s"(y));
    c.g = (const_words)(uintptr_t)x;
    c.m = (const_words)(uintptr_t)y;
    return c;
  }
  template <typename R>
  __device__ __forceinline__ C<R> mat(int i) const {
    const auto* p = (const __attribute__((address_space(4))) R*)m;
    return cmake<C<R>>(p[2 * i], p[2 * i + 1]);
  }
};

struct GeomLds {
  const uint32_t* g;
  const void* m;
  const unsigned char* staged = nullptr;  // the caller has filled the staged operators
  __device__ GeomLds(const PassGeom* geom, const void* mats) : g((const uint32_t*)geom), m(mats) {}
  __device__ __forceinline__ uint32_t w(size_t byte) const {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)g[byte / 4]);
  }
  __device__ __forceinline__ uint32_t lane_w(size_t byte) const { return g[byte / 4]; }
  __device__ __forceinline__ GeomLds again() const { return *this; }
  template <typename R>
  __device__ __forceinline__ void warm() const {}
  template <typename R>
  __device__ __forceinline__ C<R> mat(int i) const {
    return ((const C<R>*)m)[i];
  }
};

#define BT_G(field) ((int)geo.w(offsetof(PassGeom, field)))
#define BT_GOP(o, field) ((int)geo.w(offsetof(PassGeom, ops) + (size_t)(o) * sizeof(ROp) + offsetof(ROp, field)))

static_assert(sizeof(LSlots) == 32 && offsetof(PassGeom, lay) % 4 == 0 && offsetof(PassGeom, thr_in) % 4 == 0 &&
                  offsetof(PassGeom, ph) % 4 == 0 && offsetof(RPhase, op0) == 8 && sizeof(RPhase) == 16,
              "the pass reads its table in words");

// A lane-uniform value whose origin is hidden from the optimiser (what is
// computed from it stays where it is used).
__device__ __forceinline__ int hide(int x) {
  asm volatile("" : "+s"(x));
  return x;
}

// A layout's slots in bytes: thread base (per lane) and register positions.
template <typename R, typename G>
struct SlotRegs {
  uint32_t base;      // byte address of this thread's register 0 in the tile image
  uint32_t rs[TileCfg<R>::RB];
  __device__ __forceinline__ SlotRegs(const G& geo, int lay, uint32_t tid) {
    const size_t at = offsetof(PassGeom, lay) + (size_t)lay * sizeof(LSlots);
    uint32_t w[8];
#pragma unroll
    for (int i = 0; i < 8; i++) w[i] = geo.w(at + 4 * i);
    auto half = [&](int i) { return (w[i >> 1] >> (16 * (i & 1))) & 0xffffu; };
    uint32_t b = 0;
#pragma unroll
    for (int i = 0; i < TileCfg<R>::LOGNT; i++) b ^= (0u - ((tid >> i) & 1u)) & half(i);
    base = b * (uint32_t)sizeof(C<R>);
#pragma unroll
    for (int j = 0; j < TileCfg<R>::RB; j++) rs[j] = half(kTB + j) * (uint32_t)sizeof(C<R>);
  }
  __device__ __forceinline__ uint32_t at(int r) const {
    uint32_t u = 0;
#pragma unroll
    for (int j = 0; j < TileCfg<R>::RB; j++)
      if ((r >> j) & 1) u ^= rs[j];
    return base ^ u;
  }
};

template <typename R, typename G>
__device__ __forceinline__ void image_write(const C<R>* v, C<R>* lds, const G& geo, int lay, uint32_t tid, bool active,
                                            int nvalid_mask) {
  constexpr int NR = 1 << TileCfg<R>::RB;
  const SlotRegs<R, G> S(geo, lay, tid);
  if (nvalid_mask == 0) {  // every register real
    if (active) {
#pragma unroll
      for (int r = 0; r < NR; r++) *(C<R>*)((char*)lds + S.at(r)) = v[r];
    }
  } else {
    const int nm = hide(nvalid_mask);
#pragma unroll
    for (int r = 0; r < NR; r++)
      if (active && !(r & nm)) *(C<R>*)((char*)lds + S.at(r)) = v[r];
  }
}

template <typename R, typename G>
__device__ __forceinline__ void image_read(C<R>* v, const C<R>* lds, const G& geo, int lay, uint32_t ltid) {
  constexpr int NR = 1 << TileCfg<R>::RB;
  const SlotRegs<R, G> S(geo, lay, ltid);
#pragma unroll
  for (int r = 0; r < NR; r++) v[r] = *(const C<R>*)((const char*)lds + S.at(r));
}

// Offsets of a load / store layout: register positions (the same in every
// lane) and the thread's own part.  O = uint32_t: the thread's byte offset
// fits 32 bits (every thread bit of the tile below 2^32 bytes), and an access
// is a scalar base plus that offset.
template <typename R, typename O>
struct IoRegs {
  uint32_t reg[TileCfg<R>::RB];  // global bit of register position j
  O thr;                         // byte offset of this thread
  template <typename G>
  __device__ __forceinline__ IoRegs(const G& geo, size_t thr_at, size_t reg_at, uint32_t tid) {
    uint32_t w[3], r[2];
#pragma unroll
    for (int i = 0; i < 3; i++) w[i] = geo.w(thr_at + 4 * i);
#pragma unroll
    for (int i = 0; i < 2; i++) r[i] = geo.w(reg_at + 4 * i);
#pragma unroll
    for (int j = 0; j < TileCfg<R>::RB; j++) reg[j] = (r[j >> 2] >> (8 * (j & 3))) & 63u;
    thr = 0;
#pragma unroll
    for (int i = 0; i < TileCfg<R>::LOGNT; i++) {
      const uint32_t b = (w[i >> 2] >> (8 * (i & 3))) & 63u;
      thr |= (O)((tid >> i) & 1u) << (b + (sizeof(C<R>) == 8 ? 3 : 4));
    }
  }
  // keep the per-register offsets from being hoisted out of the tile loop
  __device__ __forceinline__ void again() {
#pragma unroll
    for (int j = 0; j < TileCfg<R>::RB; j++) asm volatile("" : "+s"(reg[j]));
    opaque(thr);
  }
  // byte offset of register r: 0 for a phantom position (its bit is 63, which
  // the shift to bytes drops)
  __device__ __forceinline__ uint64_t at(int r) const {
    uint64_t u = 0;
#pragma unroll
    for (int j = 0; j < TileCfg<R>::RB; j++)
      if ((r >> j) & 1) u |= (1ull << reg[j]) * sizeof(C<R>);
    return u;
  }
};

// Address of register r's element: a scalar base (state, tile, register) plus
// the thread's offset.  The scalar part is hidden from the optimiser, which
// would otherwise add the thread's offset first and keep a 64-bit vector
// address per register.
template <typename R, typename O>
__device__ __forceinline__ __attribute__((address_space(1))) char* io_addr(const C<R>* tile0, const IoRegs<R, O>& io,
                                                                          int r) {
  uint64_t b = (uint64_t)(uintptr_t)tile0 + io.at(r);
  asm volatile("" : "+s"(b));
  return (__attribute__((address_space(1))) char*)(uintptr_t)b + io.thr;
}

// Loads are unconditional and straight-line (phantom registers alias a valid
// address, inactive threads mirror an active one), so all are in flight at once.
template <typename R, typename O>
__device__ __forceinline__ void pass_fetch(C<R>* raw, const C<R>* __restrict__ state, const IoRegs<R, O>& io,
                                           uint64_t base) {
  constexpr int NR = 1 << TileCfg<R>::RB;
  typedef R v2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const v2 x = *(const __attribute__((address_space(1))) v2*)io_addr<R, O>(state + base, io, r);
    raw[r] = cmake<C<R>>(x.x, x.y);
  }
}

// Registers of a tile from its fetched values, zero where the register is
// phantom or the thread inactive.
template <typename R>
__device__ __forceinline__ void pass_take(C<R>* v, const C<R>* raw, bool active, int nvalid_mask) {
  constexpr int NR = 1 << TileCfg<R>::RB;
  const int nm = hide(nvalid_mask);
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const bool ok = active && !(r & nm);
    v[r] = cmake<C<R>>(ok ? raw[r].x : (R)0, ok ? raw[r].y : (R)0);
  }
}

template <typename R, typename O>
__device__ __forceinline__ void pass_store(const C<R>* v, C<R>* __restrict__ state, const IoRegs<R, O>& io,
                                           uint64_t base, bool active, int nvalid_mask) {
  constexpr int NR = 1 << TileCfg<R>::RB;
  typedef R v2 __attribute__((ext_vector_type(2)));
  auto put = [&](int r) {
    v2 x;
    x.x = v[r].x;
    x.y = v[r].y;
    *(__attribute__((address_space(1))) v2*)io_addr<R, O>(state + base, io, r) = x;
  };
  if (nvalid_mask == 0) {
    if (active) {
#pragma unroll
      for (int r = 0; r < NR; r++) put(r);
    }
  } else {
    const int nm = hide(nvalid_mask);
#pragma unroll
    for (int r = 0; r < NR; r++)
      if (active && !(r & nm)) put(r);
  }
}

// ---- operators ------------------------------------------------------------
// complex64: the FP32 matrix cores.  v_mfma_f32_4x4x1f32 is 16 blocks of
// 4 x 4 x 1 products: lane l (block b = l / 4) gets D[i] += A(lane 4b + i) *
// B(lane l), i = 0..3.  With B = one real input of lane l's own group and
// A(lane 4b + i) = the operator's real form at output row i of a 4-row slice,
// every lane computes 4 real outputs of its own group from its own inputs:
// nothing moves between lanes, and the 2^K x 2^K complex product (2^(K+1)
// real inputs) costs 2^(K+1) instructions per 4 outputs, at twice the FP32
// rate of the vector FMAs and beside them.  Output slice h holds rows 2h,
// 2h + 1 of the complex matrix as (Re y_2h, Im y_2h, Re y_2h+1, Im y_2h+1);
// the lane with l % 4 = i holds the slice's row 2h + (i >> 1), real part if i
// is even, else imaginary, against the inputs (Re x_c, Im x_c): (Mr, -Mi)
// for a real part, (Mi, Mr) for an imaginary one.  The operators are staged in
// LDS in that lane order (stage_ops), so a lane reads its 16 coefficients
// with four 16-byte LDS reads.
typedef float floatx4_t __attribute__((ext_vector_type(4)));

template <int MASK>
__device__ __forceinline__ void op_lane(C<float>* v, const C<float>* staged) {
  constexpr int K = __builtin_popcount(MASK);
  static_assert(K == 1 || K == 2, "matrix-core register operators cover one and two bits");
  constexpr int D = 1 << K, NS = D / 2;
  constexpr int NR = 1 << TileCfg<float>::RB;
  int P[K];
  {
    int c = 0;
#pragma unroll
    for (int j = 0; j < kRB; j++)
      if ((MASK >> j) & 1) P[c++] = j;
  }
  const float4* ap = (const float4*)(staged + 2 * D * NS / 2 * (threadIdx.x & 3));
  float a[NS][2 * D];
#pragma unroll
  for (int h = 0; h < NS; h++)
#pragma unroll
    for (int q = 0; q < D / 2; q++) {
      const float4 w = ap[2 * h + q];
      a[h][4 * q] = w.x;
      a[h][4 * q + 1] = w.y;
      a[h][4 * q + 2] = w.z;
      a[h][4 * q + 3] = w.w;
    }
#pragma unroll
  for (int base = 0; base < NR; base++) {
    if (base & MASK) continue;
    C<float> x[D];
    int idx[D];
#pragma unroll
    for (int l = 0; l < D; l++) {
      idx[l] = base;
#pragma unroll
      for (int j = 0; j < K; j++)
        if ((l >> j) & 1) idx[l] |= 1 << P[j];
      x[l] = v[idx[l]];
    }
#pragma unroll
    for (int h = 0; h < NS; h++) {
      floatx4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < D; c++) {
        d = __builtin_amdgcn_mfma_f32_4x4x1f32(a[h][2 * c], x[c].x, d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_4x4x1f32(a[h][2 * c + 1], x[c].y, d, 0, 0, 0);
      }
      v[idx[2 * h]] = cmake<C<float>>(d[0], d[1]);
      v[idx[2 * h + 1]] = cmake<C<float>>(d[2], d[3]);
    }
  }
}

// complex128: vector FMAs, the matrix entries from the pass table (scalar
// registers where the table is in the constant address space).
template <int MASK, typename G>
__device__ __forceinline__ void op_fma(C<double>* v, const G& geo, int moff) {
  constexpr int K = __builtin_popcount(MASK);
  constexpr int D = 1 << K;
  constexpr int NR = 1 << TileCfg<double>::RB;
  int P[K];
  {
    int c = 0;
#pragma unroll
    for (int j = 0; j < kRB; j++)
      if ((MASK >> j) & 1) P[c++] = j;
  }
  C<double> m[D * D];
#pragma unroll
  for (int i = 0; i < D * D; i++) m[i] = geo.template mat<double>(moff + i);
#pragma unroll
  for (int base = 0; base < NR; base++) {
    if (base & MASK) continue;
    C<double> x[D];
    int idx[D];
#pragma unroll
    for (int l = 0; l < D; l++) {
      idx[l] = base;
#pragma unroll
      for (int j = 0; j < K; j++)
        if ((l >> j) & 1) idx[l] |= 1 << P[j];
      x[l] = v[idx[l]];
    }
#pragma unroll
    for (int r = 0; r < D; r++) {
      C<double> acc = cmake<C<double>>(0, 0);
#pragma unroll
      for (int c = 0; c < D; c++) acc = cfma(acc, m[r + c * D], x[c]);
      v[idx[r]] = acc;
    }
  }
}

// Operator o of the pass on the register positions MASK.
template <typename R, int MASK, typename G>
__device__ __forceinline__ void op_reg(C<R>* v, const G& geo, int o, const C<R>* staged) {
  if constexpr (sizeof(R) == 4) {
    op_lane<MASK>(v, staged + BT_GOP(o, stage));
  } else {
    op_fma<MASK>(v, geo, BT_GOP(o, moff));
  }
}

template <typename R, typename G>
__device__ __forceinline__ void op_any(int mask, C<R>* v, const G& geo, int o, const C<R>* staged) {
  switch (mask) {
#define BT_CASE(M) \
  case M: op_reg<R, M>(v, geo, o, staged); break;
#define BT_CASE5(M)                                                               \
  case M:                                                                         \
    if constexpr (TileCfg<R>::RB == 5) op_reg<R, M>(v, geo, o, staged); \
    break;
    BT_CASE(1) BT_CASE(2) BT_CASE(4) BT_CASE(8) BT_CASE(3) BT_CASE(5) BT_CASE(6) BT_CASE(9) BT_CASE(10) BT_CASE(12)
    BT_CASE5(16) BT_CASE5(17) BT_CASE5(18) BT_CASE5(20) BT_CASE5(24)
#undef BT_CASE5
#undef BT_CASE
    default: break;
  }
}

// k >= 3 operator on the tile image, thread tid of the block.
template <typename R, int K, typename G>
__device__ __forceinline__ void op_image(C<R>* lds, int T, const G& geo, int o, const C<R>* staged, uint32_t tid) {
  constexpr int NT = TileCfg<R>::NT;
  constexpr int D = 1 << K;
  const uint32_t ng = 1u << (T - K);
  const C<R>* m = staged + BT_GOP(o, stage);
  uint32_t srt[K];
#pragma unroll
  for (int i = 0; i < K; i++) srt[i] = (uint32_t)BT_GOP(o, lsorted[i]);
  for (uint32_t g = tid; g < ng; g += NT) {
    uint32_t lb = g;
#pragma unroll
    for (int i = 0; i < K; i++) lb = ((lb >> srt[i]) << (srt[i] + 1)) | (lb & ((1u << srt[i]) - 1u));
    C<R> x[D];
#pragma unroll
    for (int l = 0; l < D; l++) x[l] = lds[swz<R>(lb + (uint32_t)BT_GOP(o, loff[l]))];
#pragma unroll 1
    for (int r = 0; r < D; r++) {  // rows one at a time
      C<R> acc = cmake<C<R>>(0, 0);
#pragma unroll
      for (int c = 0; c < D; c++) acc = cfma(acc, m[r + c * D], x[c]);
      lds[swz<R>(lb + (uint32_t)BT_GOP(o, loff[r]))] = acc;
    }
  }
}

// ---- reductions -----------------------------------------------------------
// Norm^2 of register r.
template <typename R>
__device__ __forceinline__ double reg_norm(const C<R>& v) {
  return (double)v.x * (double)v.x + (double)v.y * (double)v.y;
}

// Add one value per thread to slot j of this wavefront's accumulators.
__device__ __forceinline__ void wave_add(double x, double* wred, int j, bool lead) {
  const double t = wave_sum(x);
  if (lead) wred[j] += t;
}

// Reduced rho over K = 1 or 2 tile bits from the tile image: thread t takes
// the index groups t, t + NT, ... and all entries, packed as rho_reg packs
// them (the tile is in LDS at this point anyway, and its registers are free).
template <typename R, int K, typename G>
__device__ __forceinline__ void rho_add(const C<R>* lds, int T, const G& geo, double* wred, bool lead) {
  constexpr int D = 1 << K;
  uint32_t ls[K], off[D];
#pragma unroll
  for (int i = 0; i < K; i++) ls[i] = (uint32_t)BT_G(red_ls[i]);
#pragma unroll
  for (int a = 0; a < D; a++) off[a] = swz<R>((uint32_t)BT_G(red_loff[a]));  // the swizzle is linear over XOR
  double acc[D * D];
#pragma unroll
  for (int j = 0; j < D * D; j++) acc[j] = 0.0;
  const uint32_t ng = 1u << (T - K);
#pragma unroll 1
  for (uint32_t g = threadIdx.x; g < ng; g += TileCfg<R>::NT) {
    uint32_t lb = g;
#pragma unroll
    for (int i = 0; i < K; i++) lb = ((lb >> ls[i]) << (ls[i] + 1)) | (lb & ((1u << ls[i]) - 1u));
    const uint32_t sb = swz<R>(lb);
    double vr[D], vi[D];
#pragma unroll
    for (int a = 0; a < D; a++) {
      const C<R> x = lds[sb ^ off[a]];
      vr[a] = (double)x.x;
      vi[a] = (double)x.y;
    }
    int p = D;
#pragma unroll
    for (int a = 0; a < D; a++) {
      acc[a] += vr[a] * vr[a] + vi[a] * vi[a];
#pragma unroll
      for (int b = a + 1; b < D; b++) {
        acc[p] += vr[a] * vr[b] + vi[a] * vi[b];
        acc[p + 1] += vi[a] * vr[b] - vr[a] * vi[b];
        p += 2;
      }
    }
  }
#pragma unroll
  for (int j = 0; j < D * D; j++) wave_add(acc[j], wred, 1 + j, lead);
}

// The quad's four partials of a 3-bit reduced-rho entry, summed in a fixed
// order ((s0 + s1) + (s2 + s3)), added by the quad's first lane to its
// wavefront's packed-rho slots (LDS; each entry has one writer).
template <typename R, typename G>
__device__ __forceinline__ void rho3_add(const C<R>* lds, int T, const G& geo, double* wred) {
  const int e = (int)(threadIdx.x >> 2);
  double xr = 0.0, xi = 0.0;
  if (e < 36) {
    int a, b, ls[3];
    rho3_pair(e, &a, &b);
#pragma unroll
    for (int i = 0; i < 3; i++) ls[i] = BT_G(red_ls[i]);
    rho3_sum<R>(lds, T, geo.lane_w(offsetof(PassGeom, red_loff) + 4 * (size_t)a),
                geo.lane_w(offsetof(PassGeom, red_loff) + 4 * (size_t)b), ls, threadIdx.x & 3, &xr, &xi);
  }
  xr += dpp_f64<0xb1>(xr);
  xr += dpp_f64<0x4e>(xr);
  xi += dpp_f64<0xb1>(xi);
  xi += dpp_f64<0x4e>(xi);
  if (e < 36 && (threadIdx.x & 3) == 0) {
    const int sl = 1 + rho3_slot(e);
    wred[sl] += xr;
    if (e >= 8) wred[sl + 1] += xi;
  }
}

// Bits of t deposited on the set bits of m, ascending.
__device__ __forceinline__ uint64_t deposit(uint64_t t, uint64_t m) {
  uint64_t r = 0;
  while (m) {
    const int lo = __builtin_ctzll(m);
    const uint64_t up = ~(m >> lo);
    const int len = up ? __builtin_ctzll(up) : 64 - lo;
    const uint64_t ones = len < 64 ? (1ull << len) - 1ull : ~0ull;
    r |= (t & ones) << lo;
    t = len < 64 ? t >> len : 0;
    m &= ~(ones << lo);
  }
  return r;
}

// The operators of phase p on its registers v (layout p), for a tile at base.
template <typename R, typename G>
__device__ __forceinline__ void phase_ops(C<R>* v, const G& geo, int p, uint64_t base, int T, const C<R>* staged,
                                          C<R>* lds, uint32_t tid, uint32_t ltid, bool active, int nvalid_mask) {
  const size_t pa = offsetof(PassGeom, ph) + (size_t)p * sizeof(RPhase);
  const int op0 = (int)geo.w(pa + offsetof(RPhase, op0)), op1 = op0 + (int)geo.w(pa + offsetof(RPhase, nops));
  const int tm = (int)((geo.w(pa + 4) >> 8) & 0xffu);
  int o = op0;
  switch (tm) {  // the openings of kPhaseTemplates, straight-line
    case 1:
      op_reg<R, 0x0c>(v, geo, o, staged);
      op_reg<R, 0x03>(v, geo, o + 1, staged);
      op_reg<R, 0x06>(v, geo, o + 2, staged);
      o += 3;
      break;
    case 2:
      op_reg<R, 0x0c>(v, geo, o, staged);
      op_reg<R, 0x03>(v, geo, o + 1, staged);
      o += 2;
      break;
    case 3:
      op_reg<R, 0x03>(v, geo, o, staged);
      o += 1;
      break;
    default: break;
  }
  for (; o < op1; o++) {
    const uint64_t gctrl = ((uint64_t)geo.w(offsetof(PassGeom, ops) + (size_t)o * sizeof(ROp) + offsetof(ROp, gctrl) + 4) << 32) |
                           (uint32_t)BT_GOP(o, gctrl);
    if ((base & gctrl) != gctrl) continue;
    const int k = BT_GOP(o, k);
    if (k <= 2) {
      op_any<R>(BT_GOP(o, mask), v, geo, o, staged);
    } else {
      image_write<R>(v, lds, geo, p, tid, active, nvalid_mask);
      __syncthreads();
      if (k == 3) op_image<R, 3>(lds, T, geo, o, staged, tid);
      else op_image<R, 4>(lds, T, geo, o, staged, tid);
      __syncthreads();
      image_read<R>(v, lds, geo, p, ltid);
    }
  }
}

// One pass over tiles t = t0, t0 + tstep, ... < tend.  Reductions are added
// to sums[0..kAcc) (LDS, zeroed by the caller): [0] norm^2, [1..16]
// histogram, [17..32] packed rho; each wavefront accumulates its tiles in
// red[wave * kAcc + j] (LDS, NT/64 * kAcc doubles) and the waves are summed
// in order at the end.  lds holds 2^T elements; staged holds kStageEntries
// elements, filled from geo.staged (null: already filled).
// fresh != 0: the state is |0...0> and is not read (its first pass).
//
// Between phases the tile lives in its LDS image, not in registers: a phase
// reads its slots, applies its operators and writes the same slots back (no
// other thread owns them in this layout), so one barrier separates phases
// and no register array is live across the phase loop.
// What bounds it: with neither operators nor relayouts the same loads and
// stores move a 2^30-amplitude complex64 state at 4.8 TB/s (256 resident
// states of 2^22: 5.2 TB/s); operators and relayouts add a third to that,
// as dependency chains of two workgroups per CU.  With the tile held in
// registers across phases (two barriers per relayout, geometry in LDS) a
// 2^30 pass took 4.96 ms on average, this way 4.5 ms.
// The host emulation (tests/emu) follows the same phases.
template <typename R, typename O, typename G>
__device__ __forceinline__ void tile_pass(C<R>* __restrict__ state, const G& geo0, C<R>* staged, C<R>* lds,
                                          uint64_t t0, uint64_t tstep, uint64_t tend, double* red,
                                          double* sums, int fresh = 0) {
  constexpr int NT = TileCfg<R>::NT;
  constexpr int NR = 1 << TileCfg<R>::RB;
  const G& geo = geo0;
  const int T = BT_G(T), tb = BT_G(tb), nrb = BT_G(nrb), nph = BT_G(nph), redk = BT_G(red_k), redt = BT_G(red);
  const bool write = BT_G(write) != 0, need_norm = BT_G(need_norm) != 0;
  const bool in_direct = BT_G(in_direct) != 0, out_direct = BT_G(out_direct) != 0;
  const bool hist_fast = BT_G(hist_fast) != 0;
  const R scale = (R)__builtin_bit_cast(
      double, ((uint64_t)geo.w(offsetof(PassGeom, scale) + 4) << 32) | (uint64_t)geo.w(offsetof(PassGeom, scale)));
  const uint64_t M = ((uint64_t)geo.w(offsetof(PassGeom, outside) + 4) << 32) | geo.w(offsetof(PassGeom, outside));
  const uint32_t tid = threadIdx.x, ltid = tid & ((1u << tb) - 1u);
  const bool active = tid < (1u << tb), lead = (tid & 63) == 0;
  const int nvalid_mask = (NR - 1) & ~((1 << nrb) - 1);
  double* wred = red + (tid >> 6) * kAcc;
  IoRegs<R, O> in(geo, offsetof(PassGeom, thr_in), offsetof(PassGeom, reg_in), ltid);
  // tile t's base is t's bits deposited on the outside bits M (ascending), so
  // the next tile's base is a masked add: ((base | ~M) + deposit(tstep)) & M
  const uint64_t S = uniform_u64(deposit(tstep, M));
  uint64_t base = uniform_u64(deposit(t0, M));
  C<R> nx[NR];
  if (t0 < tend && !fresh) pass_fetch<R, O>(nx, state, in, base);
  geo.template warm<R>();
  for (int i = tid; i < (NT / 64) * kAcc; i += NT) red[i] = 0.0;
  if (geo.staged) {
    const int n = BT_G(nstage) * (int)sizeof(C<R>) / 16;
    for (int e = tid; e < n; e += NT) ((float4*)staged)[e] = ((const float4*)geo.staged)[e];
  }
  IoRegs<R, O> out(geo, offsetof(PassGeom, thr_out), offsetof(PassGeom, reg_out), ltid);
  __syncthreads();
  // Software pipeline over the tiles (disjoint): tile t's operators run while
  // the loads of tile t+1 and the stores of tile t-1 are in flight.  The wait
  // for tile t+1's loads is placed before tile t's stores are issued: the
  // vector-memory counter does not order loads against stores, so a wait for
  // loads issued before stores also waits for the stores; waiting first lets
  // tile t's stores complete under tile t+1's operators instead.
  const int np = nph > 0 ? nph : 1;
  for (uint64_t t = t0; t < tend; t += tstep) {
    const uint64_t nbase = ((base | ~M) + S) & M;
    const bool more = t + tstep < tend;
    for (int p = 0; p < np; p++) {
      const G geo = geo0.again();
      C<R> v[NR];
      const int lay = nph > 0 ? p : kLayIn;
      if (p == 0) {
        // here and not in a function with the one-tile form: as a call with an
        // early return the prefetched registers cost 8 % of a batch's passes
        // (512 trajectories of 22 qubits 630 instead of 583 ms)
        if (!fresh && active && nvalid_mask == 0) {
#pragma unroll
          for (int r = 0; r < NR; r++) v[r] = cmake<C<R>>(nx[r].x * scale, nx[r].y * scale);
        } else {
          const int nm = hide(nvalid_mask);
#pragma unroll
          for (int r = 0; r < NR; r++) {
            const bool ok = active && !(r & nm);
            if (fresh) {
              v[r] = cmake<C<R>>(ok && r == 0 && base == 0 && in.thr == 0 ? scale : (R)0, (R)0);
            } else {
              v[r] = cmake<C<R>>(ok ? nx[r].x * scale : (R)0, ok ? nx[r].y * scale : (R)0);
            }
          }
        }
        if (!fresh && more) {
          in.again();
          pass_fetch<R, O>(nx, state, in, nbase);
        }
        if (!in_direct) {
          image_write<R>(v, lds, geo, kLayIn, tid, active, nvalid_mask);
          __syncthreads();
        }
      }
      if (p > 0 || !in_direct) image_read<R>(v, lds, geo, lay, ltid);
      if (nph > 0) phase_ops<R>(v, geo, p, base, T, staged, lds, tid, ltid, active, nvalid_mask);
      if (p + 1 < np || !out_direct || redt == bti::RED_RHO) {
        image_write<R>(v, lds, geo, lay, tid, active, nvalid_mask);
        __syncthreads();
        if (p + 1 < np) continue;
        if (redt == bti::RED_RHO) {
          if (redk == 1) rho_add<R, 1>(lds, T, geo, wred, lead);
          else if (redk == 2) rho_add<R, 2>(lds, T, geo, wred, lead);
          else rho3_add<R>(lds, T, geo, wred);
        }
        image_read<R>(v, lds, geo, kLayOut, ltid);
      }
      // tile t+1's loads (and tile t-1's stores) are done before tile t's
      // stores are issued, on every path
#pragma unroll
      for (int r = 0; r < NR; r++) {
        opaque(nx[r].x);
        opaque(nx[r].y);
      }
      vm_wait_all();
      out.again();
      if (write) pass_store<R, O>(v, state, out, base, active, nvalid_mask);
      if (need_norm) {
        double s = 0.0;
        if (nvalid_mask == 0) {
#pragma unroll
          for (int r = 0; r < NR; r++) s += reg_norm<R>(v[r]);
        } else {
          const int nm = hide(nvalid_mask);
#pragma unroll
          for (int r = 0; r < NR; r++) s += (r & nm) ? 0.0 : reg_norm<R>(v[r]);
        }
        s = active ? s : 0.0;
        wave_add(s, wred, 0, lead);
        if (redt == bti::RED_HIST) {
          const int nb = 1 << redk;
          if (hist_fast) {  // one bin for all of this thread's amplitudes
            const uint64_t gi = base | (uint64_t)out.thr / sizeof(C<R>);
            int bin = 0;
#pragma unroll
            for (int j = 0; j < bti::kGroupMax; j++)
              if (j < redk) bin |= (int)((gi >> BT_G(red_bits[j])) & 1ull) << j;
#pragma unroll 1
            for (int b = 0; b < nb; b++) wave_add(bin == b ? s : 0.0, wred, 1 + b, lead);
          } else {  // tiles too small to keep every bin bit off the registers: from the image, bin by bin
            image_write<R>(v, lds, geo, kLayOut, tid, active, nvalid_mask);
            __syncthreads();
#pragma unroll 1
            for (int b = 0; b < nb; b++) {
              double x = 0.0;
              for (uint32_t e = tid; e < (1u << T); e += NT) {
                int bin = 0;
                for (int j = 0; j < redk; j++) {
                  const int lb = BT_G(red_ls[j]);
                  bin |= (int)(lb >= 0 ? (e >> lb) & 1u : (uint32_t)(base >> BT_G(red_bits[j])) & 1u) << j;
                }
                x += bin == b ? reg_norm<R>(lds[swz<R>(e)]) : 0.0;
              }
              wave_add(x, wred, 1 + b, lead);
            }
          }
        }
      }
    }
    // the next tile's first write to the image waits for this tile's last reads
    if (more) __syncthreads();
    base = nbase;
  }
  __syncthreads();
  if (threadIdx.x < kAcc) {
    double t = 0.0;
    for (int w = 0; w < NT / 64; w++) t += red[w * kAcc + threadIdx.x];
    sums[threadIdx.x] += t;
  }
  __syncthreads();
}

// Every pass of a state that is one tile, by one workgroup: the tile is read
// once, stays in its LDS image from pass to pass (every pass has the same
// tile bits, so local indices agree) and is stored once.  Passes without
// reductions or input scale only.  Table q is at tab + q * stride; staged
// holds two passes' operators: the next pass's are requested before this
// pass's phases run and written after them.
template <typename R>
__device__ __forceinline__ void one_tile_passes(C<R>* __restrict__ state, const unsigned char* tab, uint32_t stride,
                                                int npass, C<R>* staged, C<R>* lds) {
  constexpr int NT = TileCfg<R>::NT;
  constexpr int NR = 1 << TileCfg<R>::RB;
  constexpr int W = (int)((sizeof(C<R>) * kStageEntries<R> + 16 * NT - 1) / (16 * NT));  // 16-byte words per thread
  const uint32_t tid = threadIdx.x;
  auto request = [&](const GeomConst& g, float4* w) {
    const int n = (int)g.w(offsetof(PassGeom, nstage)) * (int)sizeof(C<R>) / 16;
#pragma unroll
    for (int i = 0; i < W; i++)
      if ((int)tid + i * NT < n) w[i] = ((const float4*)g.staged)[tid + i * NT];
  };
  auto put = [&](const GeomConst& g, const float4* w, C<R>* to) {
    const int n = (int)g.w(offsetof(PassGeom, nstage)) * (int)sizeof(C<R>) / 16;
#pragma unroll
    for (int i = 0; i < W; i++)
      if ((int)tid + i * NT < n) ((float4*)to)[tid + i * NT] = w[i];
  };
  float4 w[W];
  for (int q = 0; q < npass; q++) {
    const GeomConst geo0(tab + (size_t)q * stride, sizeof(C<R>));
    const GeomConst geo = geo0.again();
    const int T = BT_G(T), tb = BT_G(tb), nrb = BT_G(nrb), nph = BT_G(nph);
    const uint32_t ltid = tid & ((1u << tb) - 1u);
    const bool active = tid < (1u << tb);
    const int nvalid_mask = (NR - 1) & ~((1 << nrb) - 1);
    C<R>* ops = staged + (q & 1) * kStageEntries<R>;
    const bool last = q + 1 == npass;
    bool fetched = false;
    C<R> nx[NR];
    if (q == 0) {
      const IoRegs<R, uint32_t> in(geo, offsetof(PassGeom, thr_in), offsetof(PassGeom, reg_in), ltid);
      pass_fetch<R, uint32_t>(nx, state, in, 0);
      fetched = true;
      request(geo, w);
      put(geo, w, ops);
      geo.template warm<R>();
      __syncthreads();
    }
    const GeomConst gnext(tab + (size_t)(last ? q : q + 1) * stride, sizeof(C<R>));
    if (!last) request(gnext, w);
    for (int p = 0; p < nph; p++) {
      const GeomConst gp = geo0.again();
      C<R> v[NR];
      if (p == 0 && fetched) {
        pass_take<R>(v, nx, active, nvalid_mask);
        if (BT_G(in_direct) == 0) {
          image_write<R>(v, lds, gp, kLayIn, tid, active, nvalid_mask);
          __syncthreads();
          image_read<R>(v, lds, gp, p, ltid);
        }
      } else {
        image_read<R>(v, lds, gp, p, ltid);
      }
      phase_ops<R>(v, gp, p, 0, T, ops, lds, tid, ltid, active, nvalid_mask);
      image_write<R>(v, lds, gp, p, tid, active, nvalid_mask);
      if (p + 1 < nph || last) __syncthreads();
    }
    if (!last && BT_G(relabel)) {  // the next pass finds a plain image
      __syncthreads();
      C<R> v[NR];
      image_read<R>(v, lds, geo, kLayOut, ltid);
      __syncthreads();
      image_write<R>(v, lds, geo, kLayEnd, tid, active, nvalid_mask);
    }
    if (last) {
      C<R> v[NR];
      image_read<R>(v, lds, geo, kLayOut, ltid);
      const IoRegs<R, uint32_t> out(geo, offsetof(PassGeom, thr_out), offsetof(PassGeom, reg_out), ltid);
      pass_store<R, uint32_t>(v, state, out, 0, active, nvalid_mask);
    } else {
      put(gnext, w, staged + ((q + 1) & 1) * kStageEntries<R>);
      gnext.template warm<R>();
      __syncthreads();
    }
  }
}
#endif

// Packed reduced rho (diag, then a < b Re/Im) over k bits -> column-major
// complex; swap: the packed index's bit 0 is the rho's MSB.
__host__ __device__ inline void unpack_rho(int k, const double* packed, double* rho, int swap = 0) {
  const int D = 1 << k;
  for (int i = 0; i < 2 * D * D; i++) rho[i] = 0.0;
  auto mp = [&](int a) { return (swap && k == 2) ? (((a & 1) << 1) | (a >> 1)) : a; };
  for (int a = 0; a < D; a++) rho[2 * (mp(a) + mp(a) * D)] = packed[a];
  int p = D;
  for (int a = 0; a < D; a++)
    for (int b = a + 1; b < D; b++) {
      const int A = mp(a), B = mp(b);
      rho[2 * (A + B * D)] = packed[p];
      rho[2 * (A + B * D) + 1] = packed[p + 1];
      rho[2 * (B + A * D)] = packed[p];
      rho[2 * (B + A * D) + 1] = -packed[p + 1];
      p += 2;
    }
}

// How many of a pass's sums its result takes (to_result).
__host__ __device__ inline int acc_count(const Plan& plan) {
  return plan.red == bti::RED_HIST ? 1 + (1 << plan.red_k) : plan.red == bti::RED_RHO ? 1 + (1 << 2 * plan.red_k) : 1;
}

__host__ __device__ inline void to_result(const Plan& plan, int red_swap, const double* sum, PassResult* res) {
  res->norm2 = sum[0];
  for (int j = 0; j < 16; j++) res->hist[j] = plan.red == bti::RED_HIST && j < (1 << plan.red_k) ? sum[1 + j] : 0.0;
  for (int j = 0; j < 128; j++) res->rho[j] = 0.0;
  if (plan.red == bti::RED_RHO) unpack_rho(plan.red_k, sum + 1, res->rho, red_swap);
}

}  // namespace bt

#if !defined(__HIPCC__)
#include "bt_tile_host.hpp"
#endif
