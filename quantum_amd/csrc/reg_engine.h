// Register-resident gate engine for a 2^L-amplitude state tile held in LDS.
//
// A workgroup of 512 threads keeps the tile in VGPRs (13-qubit tiles of two states:
// 1024 threads): each thread holds 2^R amplitudes (R = L - 9, or 10 there; 3..5) whose
// indices differ only in R "register qubits"; the thread index fills the other L - R bits.  Ops whose targets
// are register qubits (and diagonal ops on any qubits, with controls on any
// qubits) are applied in registers with no LDS traffic and no barrier.  The
// host planner splits the op list into segments whose non-diagonal targets
// fit R qubits and starts each with a kOpRemap op; a remap writes the registers
// to LDS and reloads them in the new layout (two barriers).  Between remaps LDS
// holds the tile in a swizzled layout (x ^ ((x >> 4) & 15)) so that the strided
// register loads and stores of a wavefront are spread over the LDS banks; on
// entry and exit the layout is the natural one.
//
// The amplitudes of a thread are kept as MFMA result tuples (Regs): register
// index i is element i & 3 of tuple i >> 2, and each index bit ("slot") stands
// for one register qubit.  A two-qubit op reads its operands from any two slots
// and writes whole result tuples, whose two in-tuple slots are its targets: it
// permutes the slots instead of moving registers, and goes from one set of
// registers to another, so the op loop has two halves, one per set.  (In place,
// with fixed slots, every op ended in 64 register moves beside its 64 MFMAs.)
// Each ordered pair of slots has a code path of its own: the targets are always
// taken in the order of the op's matrix, so the rounding of a state (and of the
// draws from it) does not depend on the slots, and the matrix rows need no
// rearranging.  (One path per unordered pair, rows exchanged: 5% more for a
// two-state pass, 0.7% less for a batch of 4-16-qubit gradients, whose kernel
// holds every engine and feels the code size.)
// The planner knows the slots at every op and stores in each descriptor which
// code path it takes (AnnotateEngine), so the device decodes nothing.
//
// Bound by instruction issue: per tile of a 28-qubit pass (13 qubits, 8.4 two-qubit
// ops and 2.8 remaps) a wavefront issues 1173 VALU instructions, 535 of them MFMA,
// and 738 SALU (in place, and with slots and layouts decoded on the device: 2062 and
// 1954), and the pass takes 1.35 ms (1.83 ms); copying the state takes 0.89 ms.
//
// Op matrices are read from an LDS window over the plan's matrix array,
// refilled when an op's matrices fall outside it.  Parameterised ops (reverse
// sweep) accumulate their FP64 gradient partials per thread, reduce them across
// the wavefront and hand the sum to the caller's accumulator.
#pragma once

#include <type_traits>

#include "lds_ops.h"

namespace tfqx {
namespace {

static_assert(kThreads == (1 << kRegThreadBits), "RegBitsForTile assumes 512 threads");

// Register-resident complex amplitude.  A plain two-float struct (not the HIP
// vector type, whose union members turn register arrays into scratch memory).
struct cf {
  float x, y;
};
// a * b.  FIXED: with the rounding written out.  Which product an fma takes in is up to
// the compiler otherwise, and may differ from one place to the next, which draws from a
// forward run's state must not; a reverse sweep is 3% faster with its choice.
template <bool FIXED>
__device__ __forceinline__ cf cmulr(cf a, cf b) {
  if constexpr (FIXED)
    return cf{__builtin_fmaf(a.x, b.x, -(a.y * b.y)), __builtin_fmaf(a.x, b.y, a.y * b.x)};
  return cf{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
// acc + u * v as four FMAs.
__device__ __forceinline__ cf cmac(cf acc, cf u, cf v) {
  acc.x = __builtin_fmaf(u.x, v.x, acc.x);
  acc.x = __builtin_fmaf(-u.y, v.y, acc.x);
  acc.y = __builtin_fmaf(u.x, v.y, acc.y);
  acc.y = __builtin_fmaf(u.y, v.x, acc.y);
  return acc;
}
__device__ __forceinline__ cf cconj(cf a) { return cf{a.x, -a.y}; }
__device__ __forceinline__ cf ldm(const float2* __restrict__ M, int i) {
  const float* f = reinterpret_cast<const float*>(M);
  return cf{f[2 * i], f[2 * i + 1]};
}

__device__ __forceinline__ uint32_t swz(uint32_t x) { return x ^ ((x >> 4) & 15u); }

// ------------------------------------------------------------------ MFMA 4x4 products
// v_mfma_f32_4x4x1f32 runs 16 independent 4x4x1 blocks per wavefront, block b
// on lanes 4b..4b+3: D_b[i][j] += A_b[i] * B_b[j] with A_b[i] taken from lane
// 4b + i, B_b[j] from lane 4b + j, and D_b[i][j] returned in register i of
// lane 4b + j.  With A in lane l holding G[l & 3][k] and B holding each
// lane's own amplitude of gate index k, four steps (k = 0..3) leave in
// register r of every lane sum_k G[r][k] * v_k of that lane's amplitudes: a
// 4x4 gate applied in place to the registers, at twice the FP32 rate of VALU
// FMAs.  Complex products split into real ones: Re = Gr vr - Gi vi,
// Im = Gi vr + Gr vi.  MFMA ignores the EXEC mask, so these paths run only in
// wave-uniform control flow (ops without per-lane control predicates).
typedef float mf4 __attribute__((ext_vector_type(4)));

// A operands of a 4x4 complex matrix (or its adjoint): row (lane & 3).
struct MfmaRows {
  float gr[4], gi[4], ngi[4];
};
template <bool DAG>
__device__ __forceinline__ void mfma_rows(const float2* __restrict__ M, MfmaRows& r) {
  const int row = int(threadIdx.x & 3u);
  const float* f = reinterpret_cast<const float*>(M);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    // (G^dag)[row][k] = conj(G[k][row]).
    const int e = DAG ? k * 4 + row : row * 4 + k;
    r.gr[k] = f[2 * e];
    r.gi[k] = DAG ? -f[2 * e + 1] : f[2 * e + 1];
    r.ngi[k] = -r.gi[k];
  }
}
__device__ __forceinline__ mf4 mfma4(float a, float b, mf4 c) {
  return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 0, 0, 0);
}

__host__ __device__ constexpr int ins0(int g, int j) {
  return ((g >> j) << (j + 1)) | (g & ((1 << j) - 1));
}

// ------------------------------------------------------------------ registers
template <int R>
struct Regs {
  mf4 re[1 << (R - 2)], im[1 << (R - 2)];
  __device__ __forceinline__ cf get(int i) const { return cf{re[i >> 2][i & 3], im[i >> 2][i & 3]}; }
  __device__ __forceinline__ void set(int i, cf v) {
    re[i >> 2][i & 3] = v.x;
    im[i >> 2][i & 3] = v.y;
  }
};

// Tile bit of slot j in a packed slot map (kOpRemap; 4 bits per slot).
__device__ __forceinline__ uint32_t slot_bit(uint32_t slots, int j) {
  return 1u << ((slots >> (4 * j)) & 15u);
}

// This thread's bits on the non-register positions of an L-qubit tile: its
// index with zeros inserted at the register positions (slots of a fresh map
// ascend).  Wave mode: the lane; lanes past 2^(L - R) replicate a lane below.
template <int R, bool WAVE>
__device__ __forceinline__ uint32_t thread_base(uint32_t slots, int L) {
  uint32_t x = (WAVE ? (threadIdx.x & 63u) : threadIdx.x) & ((1u << (L - R)) - 1u);
  asm volatile("" : "+v"(x));  // not kept in registers from remap to remap
#pragma unroll
  for (int j = 0; j < R; ++j) x = insert_zero(x, (slots >> (4 * j)) & 15u);
  return x;
}

// A slot map's tile bits in ascending order.
template <int R>
__device__ __forceinline__ uint32_t ascending_slots(uint32_t slots) {
  uint32_t mask = 0, out = 0;
#pragma unroll
  for (int j = 0; j < R; ++j) mask |= slot_bit(slots, j);
#pragma unroll
  for (int j = 0; j < R; ++j) {
    out |= uint32_t(__builtin_ctz(mask)) << (4 * j);
    mask &= mask - 1u;
  }
  return out;
}

// Byte offsets in LDS of the 2^R registers: register i's index is tbase XOR
// the bits of its set slots, and the swizzle is XOR-linear, so each offset is
// one XOR from the one without its highest bit.
template <int R>
__device__ __forceinline__ void reg_offsets(uint32_t tbase, uint32_t slots, bool swizzled,
                                            uint32_t (&off)[1 << R]) {
  uint32_t sb[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const uint32_t b = slot_bit(slots, j);
    sb[j] = (swizzled ? swz(b) : b) << 3;
  }
  off[0] = (swizzled ? swz(tbase) : tbase) << 3;
#pragma unroll
  for (int i = 1; i < (1 << R); ++i) {
    const int h = 31 - __builtin_clz(uint32_t(i));
    off[i] = off[i ^ (1 << h)] ^ sb[h];
  }
}

template <int R>
__device__ __forceinline__ void reg_load(Regs<R>& a, const float2* __restrict__ S,
                                         const uint32_t (&off)[1 << R]) {
  const char* base = reinterpret_cast<const char*>(S);
#pragma unroll
  for (int i = 0; i < (1 << R); ++i) {
    const float2 v = *reinterpret_cast<const float2*>(base + off[i]);
    a.set(i, cf{v.x, v.y});
  }
}
template <int R>
__device__ __forceinline__ void reg_store(const Regs<R>& a, float2* __restrict__ S,
                                          const uint32_t (&off)[1 << R]) {
  char* base = reinterpret_cast<char*>(S);
#pragma unroll
  for (int i = 0; i < (1 << R); ++i) {
    const cf v = a.get(i);
    *reinterpret_cast<float2*>(base + off[i]) = make_float2(v.x, v.y);
  }
}

// ------------------------------------------------------------------ dense ops
// A operands of a two-qubit op's matrix (or its adjoint).
template <bool DAG>
__device__ __forceinline__ void engine_rows(const float2* __restrict__ M, MfmaRows& r) {
  uint32_t row = threadIdx.x & 3u;
  asm volatile("" : "+v"(row));  // not kept in registers from op to op
  const float2* base = M + (DAG ? row : row * 4u);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    // (G^dag)[row][k] = conj(G[k][row]).
    const cf v = ldm(base, DAG ? k * 4 : k);
    r.gr[k] = v.x;
    r.gi[k] = DAG ? -v.y : v.y;
    r.ngi[k] = -r.gi[k];
  }
}

// Group g of slots (SA, SB), the op's two targets in its own order: the register
// indices of its four amplitudes.
template <int SA, int SB>
__device__ __forceinline__ void group_idx(int g, int (&idx)[4]) {
  const int i0 = ins0(ins0(g, SA < SB ? SA : SB), SA < SB ? SB : SA);
#pragma unroll
  for (int s = 0; s < 4; ++s) idx[s] = i0 | ((s & 1) << SA) | ((s >> 1) << SB);
}
template <int R, int SA, int SB>
__device__ __forceinline__ void group_product(const Regs<R>& a, int g, const MfmaRows& m, mf4& dr,
                                              mf4& di) {
  int idx[4];
  group_idx<SA, SB>(g, idx);
  dr = mf4{0.f, 0.f, 0.f, 0.f};
  di = mf4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float x = a.get(idx[k]).x;
    dr = mfma4(m.gr[k], x, dr);
    di = mfma4(m.gi[k], x, di);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float y = a.get(idx[k]).y;
    dr = mfma4(m.ngi[k], y, dr);
    di = mfma4(m.gr[k], y, di);
  }
}

// Does register i (slots before the op) satisfy the op's controls?  ok: the
// thread's part.
__device__ __forceinline__ bool ctrl_ok(const DevOp& op, bool ok, int i) {
  return ok && (uint32_t(i) & op.q[2]) == op.q[3];
}

// out <- M in (or M^dagger in) on slots (SA, SB); out's slots are SA, SB, then the
// others in order.
template <int R, int SA, int SB>
__device__ __forceinline__ void reg_dense(const Regs<R>& in, Regs<R>& out, const MfmaRows& m,
                                          const DevOp& op, bool ok) {
#pragma unroll
  for (int g = 0; g < (1 << (R - 2)); ++g) group_product<R, SA, SB>(in, g, m, out.re[g], out.im[g]);
  if (op.cmask) {
#pragma unroll
    for (int g = 0; g < (1 << (R - 2)); ++g) {
      int idx[4];
      group_idx<SA, SB>(g, idx);
#pragma unroll
      for (int s = 0; s < 4; ++s)
        if (!ctrl_ok(op, ok, idx[s])) out.set(g * 4 + s, in.get(idx[s]));
    }
  }
}

// Derivative d of a parameterised op: this thread's <dG u | lam> with u after the
// op (out's slots) and lam before it (in's slots).  CTRL: the op has controls (a
// kernel-uniform test inside would become selects on every op).
template <int R, int SA, int SB, bool CTRL>
__device__ __forceinline__ void reg_deriv(const Regs<R>& u, const Regs<R>& lam, const MfmaRows& m,
                                          const DevOp& op, bool ok, float& part, float& part_im) {
  part = part_im = 0.f;
#pragma unroll
  for (int g = 0; g < (1 << (R - 2)); ++g) {
    mf4 dr, di;
    group_product<R, 0, 1>(u, g, m, dr, di);
    int idx[4];
    group_idx<SA, SB>(g, idx);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const cf l = lam.get(idx[s]);
      if (CTRL && !ctrl_ok(op, ok, idx[s])) dr[s] = di[s] = 0.f;
      part = __builtin_fmaf(dr[s], l.x, part);
      part = __builtin_fmaf(di[s], l.y, part);
      part_im = __builtin_fmaf(dr[s], l.y, part_im);
      part_im = __builtin_fmaf(-di[s], l.x, part_im);
    }
  }
}

// One-qubit op on slot S: the slots stay.  FMAs on pairs, as many cycles as MFMAs on
// groups with the identity on another slot, which would take zero times that slot's other
// amplitudes into each sum (NaN where they are not finite).
template <int R, int S, bool REV>
__device__ __forceinline__ void reg_dense1(const Regs<R>& in, Regs<R>& out, const cf (&m)[4],
                                           const DevOp& op, bool ok) {
#pragma unroll
  for (int g = 0; g < (1 << (R - 1)); ++g) {
    const int i0 = ins0(g, S), i1 = i0 | (1 << S);
    const cf x0 = in.get(i0), x1 = in.get(i1);
    out.set(i0, cmac(cmulr<!REV>(m[0], x0), m[1], x1));
    out.set(i1, cmac(cmulr<!REV>(m[2], x0), m[3], x1));
  }
  if (op.cmask) {
#pragma unroll
    for (int i = 0; i < (1 << R); ++i)
      if (!ctrl_ok(op, ok, i)) out.set(i, in.get(i));
  }
}
template <int R, int S, bool CTRL>
__device__ __forceinline__ void reg_deriv1(const Regs<R>& u, const Regs<R>& lam, const cf (&m)[4],
                                           const DevOp& op, bool ok, float& part, float& part_im) {
  part = part_im = 0.f;
#pragma unroll
  for (int g = 0; g < (1 << (R - 1)); ++g) {
    const int i0 = ins0(g, S), i1 = i0 | (1 << S);
    const cf u0 = u.get(i0), u1 = u.get(i1);
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      cf d = cmac(cmulr<false>(m[2 * r], u0), m[2 * r + 1], u1);
      const int i = r ? i1 : i0;
      const cf l = lam.get(i);
      if (CTRL && !ctrl_ok(op, ok, i)) d = cf{0.f, 0.f};
      part = __builtin_fmaf(d.x, l.x, part);
      part = __builtin_fmaf(d.y, l.y, part);
      part_im = __builtin_fmaf(d.x, l.y, part_im);
      part_im = __builtin_fmaf(-d.y, l.x, part_im);
    }
  }
}
template <bool DAG>
__device__ __forceinline__ void one_qubit_matrix(const float2* __restrict__ M, cf (&m)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    m[i] = ldm(M, DAG ? (i & 1) * 2 + (i >> 1) : i);
    if (DAG) m[i] = cconj(m[i]);
  }
}

// f(SA, SB as constants) for slot pair number `pair` ((0,1), (0,2), .. in order).
// The last one is not compared: a path on which nothing ran would keep the
// result registers' old values alive through the op.
template <int V>
using IntC = std::integral_constant<int, V>;
template <int R, int SA = 0, int SB = 1, typename F>
__device__ __forceinline__ void for_pair(int pair, F&& f) {
  constexpr int kThis = SA * (2 * R - SA - 1) / 2 + (SB - SA - 1);
  if constexpr (kThis == R * (R - 1) / 2 - 1) {
    f(IntC<SA>(), IntC<SB>());
  } else {
    if (pair == kThis) {
      f(IntC<SA>(), IntC<SB>());
    } else if constexpr (SB + 1 < R) {
      for_pair<R, SA, SB + 1>(pair, f);
    } else {
      for_pair<R, SA + 1, SA + 2>(pair, f);
    }
  }
}
// The same in the order of a two-qubit op's targets: its products are then summed in the
// order of its matrix whatever slots they are in.
template <int R, typename F>
__device__ __forceinline__ void for_ordered_pair(uint32_t code, F&& f) {
  const int pair = int(code & kCodePair);
  if (code & kCodeSwap) for_pair<R>(pair, [&](auto SA, auto SB) { f(SB, SA); });
  else for_pair<R>(pair, f);
}
template <int R, int S = 0, typename F>
__device__ __forceinline__ void for_slot(int slot, F&& f) {
  if constexpr (S + 1 == R) {
    f(IntC<S>());
  } else {
    if (slot == S) f(IntC<S>());
    else for_slot<R, S + 1>(slot, f);
  }
}

// ------------------------------------------------------------------ diagonal ops
// out = D in (and lam in the reverse sweep), slots unchanged.  The op's code says where
// its targets are: no register slot (one factor per thread), one (a factor per
// value of that slot), or two.
template <int R, bool BOTH>
__device__ __forceinline__ void scale_reg(const Regs<R>& a, const Regs<R>& b, Regs<R>& oa,
                                          Regs<R>& ob, int i, cf e) {
  oa.set(i, cmulr<!BOTH>(e, a.get(i)));
  if (BOTH) ob.set(i, cmulr<!BOTH>(e, b.get(i)));
}
__device__ __forceinline__ cf pick(bool c, cf x, cf y) { return cf{c ? x.x : y.x, c ? x.y : y.y}; }

template <int R, bool DAG, bool BOTH>
__device__ __forceinline__ void reg_diag(const Regs<R>& a, const Regs<R>& b, Regs<R>& oa,
                                         Regs<R>& ob, const DevOp& op,
                                         const float2* __restrict__ Dg, uint32_t tbase, bool ok) {
  const bool two = op.k == 2;
  cf d[4];
  d[0] = ldm(Dg, 0);
  d[1] = ldm(Dg, 1);
  d[2] = two ? ldm(Dg, 2) : d[0];
  d[3] = two ? ldm(Dg, 3) : d[1];
  if (DAG) {
#pragma unroll
    for (int k = 0; k < 4; ++k) d[k] = cconj(d[k]);
  }
  // Thread bits of the targets (a register slot's bit of tbase is zero).
  const bool t0 = (tbase >> op.q[0]) & 1u, t1 = two && ((tbase >> op.q[1]) & 1u);
  const uint32_t s0 = op.code & 7u, s1 = (op.code >> 3) & 7u;  // slots, or R: thread bit
  const bool r0 = s0 < uint32_t(R), r1 = two && s1 < uint32_t(R);
  if (op.cmask) {
#pragma unroll
    for (int i = 0; i < (1 << R); ++i) {
      const bool b0 = r0 ? ((uint32_t(i) >> s0) & 1u) != 0u : t0;
      const bool b1 = r1 ? ((uint32_t(i) >> s1) & 1u) != 0u : t1;
      const cf e = pick(b1, pick(b0, d[3], d[2]), pick(b0, d[1], d[0]));
      scale_reg<R, BOTH>(a, b, oa, ob, i, pick(ctrl_ok(op, ok, i), e, cf{1.f, 0.f}));
    }
  } else if (!r0 && !r1) {
    const cf e = pick(t1, pick(t0, d[3], d[2]), pick(t0, d[1], d[0]));
#pragma unroll
    for (int i = 0; i < (1 << R); ++i) scale_reg<R, BOTH>(a, b, oa, ob, i, e);
  } else if (r0 != r1) {
    // e[v]: the factor for value v of the register slot.
    cf e[2];
#pragma unroll
    for (int v = 0; v < 2; ++v) e[v] = r0 ? pick(t1, d[2 + v], d[v]) : pick(t0, d[2 * v + 1], d[2 * v]);
    for_slot<R>(int(r0 ? s0 : s1), [&](auto S) {
#pragma unroll
      for (int i = 0; i < (1 << R); ++i) scale_reg<R, BOTH>(a, b, oa, ob, i, e[(i >> S.value) & 1]);
    });
  } else {
    // Slots in ascending order; d's index bits follow.
    const bool sw = s0 > s1;
    const cf e1 = pick(sw, d[2], d[1]), e2 = pick(sw, d[1], d[2]);
    const int lo = int(sw ? s1 : s0), hi = int(sw ? s0 : s1);
    for_pair<R>(lo * (2 * R - lo - 1) / 2 + (hi - lo - 1), [&](auto SA, auto SB) {
#pragma unroll
      for (int i = 0; i < (1 << R); ++i) {
        const int c = ((i >> SA.value) & 1) | (((i >> SB.value) & 1) << 1);
        scale_reg<R, BOTH>(a, b, oa, ob, i, c == 0 ? d[0] : c == 1 ? e1 : c == 2 ? e2 : d[3]);
      }
    });
  }
}

// ------------------------------------------------------------------ noise channels
// Trajectory context of a noisy forward run, passed as the run's acc_fn:
// channel c of trajectory `traj` of output row `row` draws
// uniform(seed, shot = traj, stream = (row, c)).  In wave mode a wavefront
// holds 2^(6 - gbits) trajectories side by side, each on 2^gbits consecutive
// lanes, and traj is this lane's.
//
// The variates of a trajectory are drawn 2^gbits at a time: lane li of the
// trajectory's group computes the variate of channel base + li, and channel
// c (base <= c < base + 2^gbits) reads it from lane c - base of its group.
// Channel ordinals only grow along the op list and every lane of a wavefront
// meets the same channels, so `base` is wave-uniform.
struct NoiseDraw {
  unsigned long long seed;
  unsigned long long traj;
  uint32_t row;
  int gbits;
  int base = -1;
  double cached = 0.0;
  __device__ __forceinline__ double operator()(int ch) {
    const int width = 1 << gbits;
    if (base < 0 || ch < base || ch >= base + width) {
      base = ch;
      const uint32_t li = (threadIdx.x & 63u) & uint32_t(width - 1);
      cached = philox_uniform(seed, traj, row, uint32_t(ch) + li);
    }
    const int src = int((threadIdx.x & 63u) & ~uint32_t(width - 1)) + (ch - base);
    return __shfl(cached, src, 64);
  }
  // Gradient partials (reverse runs only; never called on a forward run).
  __device__ __forceinline__ void operator()(int, int, double, double) const {}
};
template <typename T>
struct IsNoise : std::false_type {};
template <>
struct IsNoise<NoiseDraw> : std::true_type {};

// Sums over the 2^gbits lanes of this lane's trajectory group (all of them
// end with the same bits: each butterfly step adds the same two values).
// The DPP steps pair each lane with one that holds the same partial as its
// butterfly partner (lane ^ 4, lane ^ 8), so the sums are the butterfly's.
template <int N>
__device__ __forceinline__ void group_sums(double (&v)[N], int gbits) {
  auto step = [&](auto f) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = f(v[i]);
  };
  if (gbits > 0) step([](double x) { return dpp_add<0xB1>(x); });
  if (gbits > 1) step([](double x) { return dpp_add<0x4E>(x); });
  if (gbits > 2) step([](double x) { return dpp_add<0x141>(x); });
  if (gbits > 3) step([](double x) { return dpp_add<0x140>(x); });
  if (gbits > 4) step([](double x) { return x + __shfl_xor(x, 16, 64); });
  if (gbits > 5) step([](double x) { return x + __shfl_xor(x, 32, 64); });
}
__device__ __forceinline__ double group_sum(double v, int gbits) {
  double s[1] = {v};
  group_sums(s, gbits);
  return s[0];
}

// The operator that a channel applies to this lane's trajectory, times scale.
struct ChannelPick {
  int k;
  float scale;
};

// This lane's part of |x0|^2 and |x1|^2 summed over register slot J's qubit.  Every
// product is added to a sum that starts from a value the compiler does not know: it
// would compute the sums of all slots before looking at the op, for every op (2.2x
// this kernel's FP32 instructions).  The rounding is written out: draws depend on it.
template <int R, int J>
__device__ __forceinline__ void reg_density(const Regs<R>& a, float (&d)[2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    d[i] = 0.f;
    asm volatile("" : "+v"(d[i]));
  }
#pragma unroll
  for (int g = 0; g < (1 << (R - 1)); ++g) {
    const int i0 = ins0(g, J);
    const cf x0 = a.get(i0), x1 = a.get(i0 | (1 << J));
    d[0] += __builtin_fmaf(x0.x, x0.x, x0.y * x0.y);
    d[1] += __builtin_fmaf(x1.x, x1.x, x1.y * x1.y);
  }
}
// The first k with u < p_0 + ... + p_k, the last k with p_k > 0 when none.
template <typename Prob>
__device__ __forceinline__ ChannelPick pick_kraus(int nk, double u, Prob&& prob) {
  double cum = 0.0, pp = 1.0;
  int last = 0, pick = -1;
  for (int k = 0; k < nk; ++k) {
    const double pk = prob(k);
    if (pk > 0.0) last = k;
    cum += pk;
    if (pick < 0 && u < cum) {
      pick = k;
      pp = pk;
    }
  }
  if (pick < 0) {
    pick = last;
    pp = prob(last);
  }
  return ChannelPick{pick, float(1.0 / sqrt(pp))};
}

// Unitary mixtures pick unitary k with the first u < cum[k]; other channels take
// p_k = <psi|K_k^dag K_k|psi> from the qubit's populations (K_k^dag K_k is diagonal
// for every channel kind: its K_k have at most one entry in a row and column), pick the
// first k with u < p_0 + ... + p_k (the last k with p_k > 0 when none) and apply
// K_k / sqrt(p_k).  Lanes of different trajectories may pick different operators.
template <int R>
__device__ __forceinline__ ChannelPick channel_pick(const Regs<R>& a, const DevOp& op,
                                                    const float2* __restrict__ mats,
                                                    NoiseDraw& nd) {
  const int nk = ChanKraus(op.cval);
  const double u = nd(op.col[0]);
  const float2* X = mats + op.dmat[0];
  if (op.cval & kChanMixture) {
    int pick = nk - 1;
    for (int k = nk - 2; k >= 0; --k)
      if (u < double(X[k].x)) pick = k;
    return ChannelPick{pick, 1.0f};
  }
  float s[2];
  for_slot<R>(int(op.code), [&](auto J) { reg_density<R, J.value>(a, s); });
  double d[2] = {double(s[0]), double(s[1])};
  group_sums(d, nd.gbits);
  return pick_kraus(nk, u, [&](int k) {
    return double(X[4 * k].x) * d[0] + double(X[4 * k + 3].x) * d[1];
  });
}

// out = the picked operator on register slot J of in; the matrix is read per lane.
// Bound by the number of VALU instructions: with real matrices half the products
// go (every channel that is no unitary mixture has them): 700 us (965 us) for 32 rows of
// 1000 8-qubit trajectories with 128 channels.
template <int R, int J, bool REAL>
__device__ __forceinline__ void reg_channel(const Regs<R>& in, Regs<R>& out,
                                            const float2* __restrict__ M, float sc) {
  const cf m00{M[0].x * sc, M[0].y * sc}, m01{M[1].x * sc, M[1].y * sc};
  const cf m10{M[2].x * sc, M[2].y * sc}, m11{M[3].x * sc, M[3].y * sc};
#pragma unroll
  for (int g = 0; g < (1 << (R - 1)); ++g) {
    const int i0 = ins0(g, J);
    const cf x0 = in.get(i0), x1 = in.get(i0 | (1 << J));
    if constexpr (REAL) {
      out.set(i0, cf{__builtin_fmaf(m01.x, x1.x, m00.x * x0.x),
                     __builtin_fmaf(m01.x, x1.y, m00.x * x0.y)});
      out.set(i0 | (1 << J), cf{__builtin_fmaf(m11.x, x1.x, m10.x * x0.x),
                                __builtin_fmaf(m11.x, x1.y, m10.x * x0.y)});
    } else {
      out.set(i0, cmac(cmulr<true>(m00, x0), m01, x1));
      out.set(i0 | (1 << J), cmac(cmulr<true>(m10, x0), m11, x1));
    }
  }
}

// ------------------------------------------------------------------ driver
// LDS window [lo, hi) of the plan's matrix array (global g).  All waves of a
// workgroup run the same op sequence, so a refill (two barriers) happens at
// the same op in every wave; windows stay valid for the whole launch because
// the matrices do not change while it runs.
struct MatCache {
  float2* lds;  // n entries
  const float2* g;
  uint32_t lo, hi;  // kNoWindow: nothing there yet
  uint32_t n;
};
constexpr uint32_t kNoWindow = 1u << 31;  // past every offset
__device__ __forceinline__ MatCache mat_cache(float2* lds, const float2* g,
                                              uint32_t n = kMatCache) {
  return MatCache{lds, g, kNoWindow, kNoWindow, n};
}
// Make entries [off, off + len) resident in the window (every plan pads its
// matrix array by at least its kernel's window, so a refill stays inside).
__device__ __forceinline__ void cache_span(MatCache& c, uint32_t off, uint32_t len) {
  if (off >= c.lo && off + len <= c.hi) return;
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < c.n; i += kThreads) c.lds[i] = c.g[off + i];
  __syncthreads();
  c.lo = off;
  c.hi = off + c.n;
}
// Matrix entries an op reads: its unitary (or diagonal) and derivatives,
// stored back to back.
__device__ __forceinline__ uint32_t op_mat_len(const DevOp& op) {
  const uint32_t D = 1u << op.k;
  const uint32_t DD = op.type == kOpDiag ? D : D * D;
  return DD * (1u + (op.type == kOpParam ? uint32_t(op.nderiv) : 0u));
}

// Matrices read straight from the plan's array (wave mode: waves run
// independent circuits, so no workgroup-wide refill is possible).
struct GlobalMats {
  const float2* g;
};
// Make an op's matrices readable and return the array its offsets index
// (offsets rebased to the LDS window when cached).
__device__ __forceinline__ const float2* mats_for(MatCache& c, DevOp& op) {
  // Room for the longest op (one compare against the window's start, where the
  // op's own length takes a dozen scalar instructions per op).
  constexpr uint32_t kLongest = 16u * (1u + kMaxDeriv);
  if (op.mat - c.lo > c.n - kLongest) cache_span(c, op.mat, c.n);
  op.mat -= c.lo;
  op.dmat[0] -= c.lo;
  op.dmat[1] -= c.lo;
  return c.lds;
}
__device__ __forceinline__ const float2* mats_for(GlobalMats& c, DevOp&) { return c.g; }

// Engine synchronisation: the workgroup (one tile per workgroup) or, in wave
// mode, the wavefront (one circuit per wavefront; its LDS traffic is ordered
// by the wavefront's own in-order LDS queue).
template <bool WAVE>
__device__ __forceinline__ void esync() {
  if constexpr (WAVE) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    __syncthreads();
  }
}

// Tile I/O of the engine.  LdsIO: the tile enters and leaves in LDS buffers A
// (and B) in the natural layout; the caller synchronises before the run and
// the engine synchronises before returning.  TileIO: the first remap loads the
// registers straight from memory with load(thread, slot, set_a, set_b) and the run ends with
// store(thread, slot, get_a, get_b): register r's amplitude has index thread + the
// sum of slot[j] over the set bits j of r, and goes through set_a(r, v) or get_a(r)
// (set_b, get_b: the second state of the reverse sweep).
// LDS is then used only by the remaps in between, and no barrier surrounds the run
// (a remap's own barriers order its LDS use).  `thread` is index(x) of this
// thread's own tile bits x, and slot[j], which is wave-uniform, index of slot j's
// bit; index must be OR-linear over disjoint bits (a tile's bits
// deposited into the global index).
struct LdsIO {};
struct IdentityIndex {
  __device__ __forceinline__ uint64_t operator()(uint32_t x) const { return x; }
};
__device__ __forceinline__ uint64_t uniform64(uint64_t x) {
  return uint64_t(uint32_t(uniform(int(uint32_t(x))))) |
         (uint64_t(uint32_t(uniform(int(uint32_t(x >> 32))))) << 32);
}
// Global index parts of this thread's tile bits and of each register slot.
template <int R>
struct TileIndex {
  uint64_t thread;
  uint64_t slot[R];
};
template <int R, bool WAVE, typename IndexFn>
__device__ __forceinline__ TileIndex<R> tile_index_of(uint32_t slots, int L, IndexFn&& index) {
  TileIndex<R> t;
  t.thread = index(thread_base<R, WAVE>(ascending_slots<R>(slots), L));
#pragma unroll
  for (int j = 0; j < R; ++j) t.slot[j] = uniform64(index(slot_bit(slots, j)));
  return t;
}
template <typename LoadFn, typename StoreFn, typename IndexFn = IdentityIndex>
struct TileIO {
  LoadFn load;
  StoreFn store;
  IndexFn index;
  template <int R, bool WAVE>
  __device__ __forceinline__ TileIndex<R> in(uint32_t slots, int L) const {
    return tile_index_of<R, WAVE>(slots, L, index);
  }
  template <int R, bool WAVE>
  __device__ __forceinline__ TileIndex<R> out(uint32_t slots, int L) const {
    return tile_index_of<R, WAVE>(slots, L, index);
  }
};
// The same with the index parts of the first and last layout worked out by the caller
// (they are those of every tile of a pass).
template <int N, typename LoadFn, typename StoreFn>
struct FixedTileIO {
  LoadFn load;
  StoreFn store;
  TileIndex<N> first, last;
  template <int R, bool WAVE>
  __device__ __forceinline__ TileIndex<R> in(uint32_t, int) const {
    return first;
  }
  template <int R, bool WAVE>
  __device__ __forceinline__ TileIndex<R> out(uint32_t, int) const {
    return last;
  }
};
template <typename LoadFn, typename StoreFn>
__device__ __forceinline__ TileIO<LoadFn, StoreFn> tile_io(LoadFn l, StoreFn s) {
  return TileIO<LoadFn, StoreFn>{l, s, IdentityIndex{}};
}
template <typename IndexFn, typename LoadFn, typename StoreFn>
__device__ __forceinline__ TileIO<LoadFn, StoreFn, IndexFn> tile_io_indexed(IndexFn i, LoadFn l,
                                                                            StoreFn s) {
  return TileIO<LoadFn, StoreFn, IndexFn>{l, s, i};
}
template <int R, typename LoadFn, typename StoreFn>
__device__ __forceinline__ FixedTileIO<R, LoadFn, StoreFn> tile_io_fixed(const TileIndex<R>& first,
                                                                         const TileIndex<R>& last,
                                                                         LoadFn l, StoreFn s) {
  return FixedTileIO<R, LoadFn, StoreFn>{l, s, first, last};
}
// f(r, x + register r's part) for every register; x: an index or a pointer.  Each is
// one add from the one without its highest slot (sums of the parts kept in scalar
// registers: two scalar instructions a register more, and 32 registers).
template <size_t R, typename T, typename F>
__device__ __forceinline__ void each_reg(const uint64_t (&slot)[R], T x, F&& f) {
  T p[1 << R];
  p[0] = x;
#pragma unroll
  for (int r = 1; r < (1 << R); ++r) {
    const int h = 31 - __builtin_clz(uint32_t(r));
    p[r] = p[r ^ (1 << h)] + slot[h];
  }
#pragma unroll
  for (int r = 0; r < (1 << R); ++r) f(r, p[r]);
}
template <typename IO>
struct IsLdsIO {
  static constexpr bool value = false;
};
template <>
struct IsLdsIO<LdsIO> {
  static constexpr bool value = true;
};

// The part of a run that the op loop carries besides the registers.
struct RunState {
  uint32_t tbase;  // this thread's tile bits
  uint32_t mask;   // register qubits (wave-uniform)
  int slot;        // derivative matrices of earlier parameterised ops
  bool first_store;
  // The thread's part of an op's controls.
  __device__ __forceinline__ bool ok(const DevOp& op) const {
    return ((tbase ^ op.cval) & op.cmask & ~mask) == 0u;
  }
};

template <typename AccFn>
struct HasChannels {
  static constexpr bool value = IsNoise<std::decay_t<AccFn>>::value;
};

// A remap that leaves the wavefront-index qubits where they are moves
// every amplitude within its own wavefront: wavefront w stores and
// reloads exactly the (swizzled) LDS entries it read at the previous
// remap, so it needs no workgroup barrier.  The first store of a run
// still waits for the whole workgroup (entries last read in another
// layout, or by other wavefronts on the previous tile).
template <int R, bool REV, bool WAVE>
__device__ __forceinline__ void run_remap(const Regs<R>& ra, const Regs<R>& rb, Regs<R>& oa,
                                          Regs<R>& ob, const DevOp& op, float2* __restrict__ A,
                                          float2* __restrict__ B, int L, RunState& st) {
  const bool local = !WAVE && !st.first_store && (op.code & kCodeLocal);
  uint32_t off[1 << R];
  reg_offsets<R>(st.tbase, op.cval, true, off);
  if (!local) esync<WAVE>();
  reg_store<R>(ra, A, off);
  if (REV) reg_store<R>(rb, B, off);
  st.first_store = false;
  if (local) esync<true>();
  else esync<WAVE>();
  st.mask = op.cmask;
  st.tbase = thread_base<R, WAVE>(op.dmat[0], L);
  reg_offsets<R>(st.tbase, op.dmat[0], true, off);
  reg_load<R>(oa, A, off);
  if (REV) reg_load<R>(ob, B, off);
}

// One op, from (ra, rb) to (oa, ob).
template <int R, bool REV, bool WAVE, typename MS, typename AccFn>
__device__ __forceinline__ void run_op(const Regs<R>& ra, const Regs<R>& rb, Regs<R>& oa,
                                       Regs<R>& ob, DevOp& op, float2* __restrict__ A,
                                       float2* __restrict__ B, int L, MS& mc, AccFn&& acc_fn,
                                       RunState& st, const ChannelPick& cp) {
  if (op.type == kOpRemap) {
    run_remap<R, REV, WAVE>(ra, rb, oa, ob, op, A, B, L, st);
    return;
  }
  const float2* mats = mats_for(mc, op);
  const bool ok = st.ok(op);
  if (op.type == kOpDiag) {
    reg_diag<R, REV, REV>(ra, rb, oa, ob, op, mats + op.mat, st.tbase, ok);
    return;
  }
  if constexpr (!REV && HasChannels<AccFn>::value) {
    if (op.type == kOpChannel) {
      const float2* M = mats + op.mat + 4 * cp.k;
      for_slot<R>(int(op.code), [&](auto J) {
        if (op.cval & kChanReal) reg_channel<R, J.value, true>(ra, oa, M, cp.scale);
        else reg_channel<R, J.value, false>(ra, oa, M, cp.scale);
      });
      return;
    }
  }
  const int nd = REV && op.type == kOpParam ? op.nderiv : 0;
  float part[2 * kMaxDeriv] = {0.f, 0.f, 0.f, 0.f};
  auto keep = [&](int d, float re, float im) {
    if (d == 0) {
      part[0] = re;
      part[kMaxDeriv] = im;
    } else {
      part[1] = re;
      part[kMaxDeriv + 1] = im;
    }
  };
  if (op.k == 1) {
    cf m[4];
    one_qubit_matrix<REV>(mats + op.mat, m);
    for_slot<R>(int(op.code), [&](auto S) {
      reg_dense1<R, S.value, REV>(ra, oa, m, op, ok);
      if (REV) {
        reg_dense1<R, S.value, REV>(rb, ob, m, op, ok);
#pragma unroll 1
        for (int d = 0; d < nd; ++d) {
          cf dm[4];
          one_qubit_matrix<false>(mats + (d == 0 ? op.dmat[0] : op.dmat[1]), dm);
          float re, im;
          if (op.cmask) reg_deriv1<R, S.value, true>(oa, rb, dm, op, ok, re, im);
          else reg_deriv1<R, S.value, false>(oa, rb, dm, op, ok, re, im);
          keep(d, re, im);
        }
      }
    });
  } else {
    MfmaRows m;
    engine_rows<REV>(mats + op.mat, m);
    for_ordered_pair<R>(op.code, [&](auto SA, auto SB) {
      reg_dense<R, SA.value, SB.value>(ra, oa, m, op, ok);
      if (REV) {
        reg_dense<R, SA.value, SB.value>(rb, ob, m, op, ok);
#pragma unroll 1
        for (int d = 0; d < nd; ++d) {
          MfmaRows dm;
          engine_rows<false>(mats + (d == 0 ? op.dmat[0] : op.dmat[1]), dm);
          float re, im;
          if (op.cmask) reg_deriv<R, SA.value, SB.value, true>(oa, rb, dm, op, ok, re, im);
          else reg_deriv<R, SA.value, SB.value, false>(oa, rb, dm, op, ok, re, im);
          keep(d, re, im);
        }
      }
    });
  }
  if (nd > 0) {
    // Wave mode: gradient partials count each amplitude once (replica lanes 0).
    if (WAVE && ((threadIdx.x & 63u) >> (L - R)) != 0u)
      part[0] = part[1] = part[2] = part[3] = 0.f;
    // The imaginary parts reach only the callers that use them (the
    // compiler drops them elsewhere).
    const double w0 = wave_sum(double(part[0])), v0 = wave_sum(double(part[kMaxDeriv]));
    if ((threadIdx.x & 63) == 0) acc_fn(st.slot, op.col[0], w0, v0);
    if (nd > 1) {
      const double w1 = wave_sum(double(part[1])), v1 = wave_sum(double(part[kMaxDeriv + 1]));
      if ((threadIdx.x & 63) == 0) acc_fn(st.slot + 1, op.col[1], w1, v1);
    }
    st.slot += nd;
  }
}

// Apply ops [b, e) to a tile of 2^L amplitudes (A, and B in the reverse sweep).
// REV = false: apply each op's matrix to A.  REV = true: un-apply (M^dagger)
// non-parameterised ops on A and B; parameterised ops run the adjoint step
// and call acc_fn(slot, column, re, im) from lane 0 of each wavefront with the
// wavefront's partial <dG psi | lambda>
// per derivative, slot counting the derivative matrices of earlier
// parameterised ops and column being the derivative's symbol column.
// Ops [b, e) must start with a kOpRemap.  A and B also serve as the remap
// buffers.
template <int R, bool REV, bool WAVE, typename MS, typename AccFn, typename IO>
__device__ __forceinline__ void reg_run(float2* __restrict__ A, float2* __restrict__ B, int L,
                        const DevOp* __restrict__ ops, int b, int e,
                        MS& mc, AccFn&& acc_fn, IO& io) {
  constexpr bool kLds = IsLdsIO<IO>::value;
  Regs<R> xa, xb, ya, yb;  // two register sets; the b's unused when !REV
  const DevOp first = load_op(ops + b);
  RunState st{thread_base<R, WAVE>(first.dmat[0], L), first.cmask, 0, true};
  if constexpr (kLds) {
    uint32_t off[1 << R];
    reg_offsets<R>(st.tbase, first.dmat[0], false, off);
    esync<WAVE>();
    reg_load<R>(xa, A, off);
    if (REV) reg_load<R>(xb, B, off);
  } else {
    const TileIndex<R> t = io.template in<R, WAVE>(first.dmat[0], L);
    io.load(t.thread, t.slot, [&](int r, cf v) { xa.set(r, v); },
            [&](int r, cf v) { xb.set(r, v); });
  }
  auto finish = [&](Regs<R>& ra, Regs<R>& rb) {
    if constexpr (kLds) {
      uint32_t off[1 << R];
      reg_offsets<R>(st.tbase, first.dmat[1], false, off);
      esync<WAVE>();
      reg_store<R>(ra, A, off);
      if (REV) reg_store<R>(rb, B, off);
      esync<WAVE>();
    } else {
      const TileIndex<R> t = io.template out<R, WAVE>(first.dmat[1], L);
      io.store(t.thread, t.slot, [&](int r) { return ra.get(r); },
               [&](int r) { return rb.get(r); });
    }
  };
  // The next op to run on registers r; false at the end.  Channels that leave every
  // lane's trajectory as it is (unitary 0, the identity) are passed over.
  int i = b + 1;
  DevOp op;
  ChannelPick cp{0, 1.0f};
  auto next = [&](const Regs<R>& r) -> bool {
    while (i < e) {
      op = load_op(ops + i);
      ++i;
      if constexpr (!REV && HasChannels<AccFn>::value) {
        if (op.type == kOpChannel) {
          DevOp ch = op;
          const float2* mats = mats_for(mc, ch);
          cp = channel_pick<R>(r, ch, mats, acc_fn);
          if ((ch.cval & kChanFirstIdentity) && __ballot(cp.k != 0) == 0) continue;
        }
      }
      return true;
    }
    return false;
  };
  // One half of the loop per register set; every op goes from one to the other, so
  // that only one is live between ops.
  while (true) {
    if (!next(xa)) {
      finish(xa, xb);
      return;
    }
    run_op<R, REV, WAVE>(xa, xb, ya, yb, op, A, B, L, mc, acc_fn, st, cp);
    if (!next(ya)) {
      finish(ya, yb);
      return;
    }
    run_op<R, REV, WAVE>(ya, yb, xa, xb, op, A, B, L, mc, acc_fn, st, cp);
  }
}

// Run ops [b, e) on a tile of L qubits with the register engine when the op
// list was planned for it (starts with a remap); returns false otherwise,
// before touching the tile.
// RMAX = 5 adds 14-qubit one-state tiles (32 registers per thread); only the
// streaming pass kernel's wide instantiation, whose plans use them, asks for it.
template <bool REV, int RMAX = 4, typename AccFn, typename IO>
__device__ __forceinline__ bool reg_run_any(float2* A, float2* B, int L, const DevOp* ops, int b,
                                            int e, MatCache& mc, AccFn&& acc_fn, IO& io) {
  if (b >= e) return false;
  if (uniform(int(ops[b].type)) != kOpRemap) return false;
  switch (RegBitsForTile(L, RMAX)) {
    case 3: reg_run<3, REV, false>(A, B, L, ops, b, e, mc, acc_fn, io); return true;
    case 4: reg_run<4, REV, false>(A, B, L, ops, b, e, mc, acc_fn, io); return true;
    case 5:
      if constexpr (RMAX >= 5 && !REV) {
        reg_run<5, REV, false>(A, B, L, ops, b, e, mc, acc_fn, io);
        return true;
      }
      return false;
    default: return false;
  }
}
template <bool REV, typename AccFn>
__device__ __forceinline__ bool reg_run_any(float2* A, float2* B, int L, const DevOp* ops, int b,
                                            int e, MatCache& mc, AccFn&& acc_fn) {
  LdsIO io;
  return reg_run_any<REV>(A, B, L, ops, b, e, mc, acc_fn, io);
}

// Wave mode: one wavefront runs a whole circuit of L = kWaveRegBits..
// kWaveMaxQubits qubits (ops planned with remaps for kWaveRegBits register
// qubits), A and B being the wavefront's own LDS buffers of 2^L amplitudes.
template <bool REV, typename AccFn, typename IO>
__device__ __forceinline__ void reg_run_wave(float2* A, float2* B, int L, const DevOp* ops, int b,
                                             int e, const float2* mats, AccFn&& acc_fn, IO& io) {
  if (b >= e) return;
  GlobalMats gm{mats};
  reg_run<kWaveRegBits, REV, true>(A, B, L, ops, b, e, gm, acc_fn, io);
}

}  // namespace
}  // namespace tfqx
