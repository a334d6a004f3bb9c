// Gate engine for circuits whose state stays in LDS (two qubits up to the LDS
// tile, fused ops of at most two qubits; the register engine takes the tiles of
// 12-13 qubits).
//
// A lane owns the four amplitudes of a two-qubit op's targets: it loads them from
// LDS, multiplies by the 4x4 matrix on v_mfma_f32_4x4x1f32 (reg_engine.h) and stores
// them; a barrier separates ops.  A one-qubit op takes a pair a lane, on FMAs.  Lanes
// whose control qubits do not match run along and store nothing.
//
// What bounds small circuits is the latency of one op, not work: a 10-qubit
// op is 256 groups.  Hence
//  - matrices reach the lanes as MFMA rows, 32 B per lane and matrix.  As FMA
//    operands every lane read the whole matrix, 128 B, and again for each use:
//    up to 2,000 LDS cycles per parameterised op;
//  - up to eight qubits the groups fit one wavefront, which runs the list alone
//    (its LDS accesses are in order) without a barrier per op;
//  - op descriptors come from an LDS window; the next one is read while an op
//    runs (a scalar load would share the wait counter of the op's LDS reads).
//  - gradient partials are reduced eight at a time (PartRing).
// Per op of a circuit that has the chip to itself (64 circuits, two-qubit ops
// with two derivatives in the reverse sweep): 8 qubits 0.54 us forward and 1.21
// reverse (FMA sweeps with a barrier each: 0.68 and 1.69), 10 qubits 0.60 and
// 1.46 (0.80 and 1.87), 11 qubits 0.76 and 1.84 (1.01 and 2.29).  What is left is
// the issue of a few hundred dependent instructions by one wavefront per SIMD.
// One-qubit ops as MFMA groups of two pairs, the other half of the matrix zero, took
// 657 us on 64 circuits of 10 qubits and 600 symbols (half of the symbols in one-qubit
// ops), with a pair a lane 607.
#pragma once

#include "reg_engine.h"

namespace tfqx {
namespace {

constexpr int kSoloMaxQubits = 8;  // 2^6 groups: one wavefront

// Op descriptors in LDS: kDescWindow at a time.
constexpr int kDescWords = sizeof(DevOp) / 4;
constexpr int kDescWindow = 144;

// Descriptor i of the window: each lane reads one word of it (issued early),
// and the words become wave-uniform when it is unpacked.
__device__ __forceinline__ uint32_t desc_word(const uint32_t* win, int i) {
  return win[i * kDescWords + min(int(threadIdx.x & 63u), kDescWords - 1)];
}
__device__ __forceinline__ DevOp desc_unpack(uint32_t word) {
  uint32_t w[kDescWords - 1];
#pragma unroll
  for (int j = 0; j < kDescWords - 1; ++j) w[j] = uint32_t(__builtin_amdgcn_readlane(int(word), j));
  DevOp o;
  o.type = uint8_t(w[0]);
  o.k = uint8_t(w[0] >> 8);
  o.nderiv = uint8_t(w[0] >> 16);
  o.code = uint8_t(w[0] >> 24);
  o.q[0] = uint8_t(w[1]);
  o.q[1] = uint8_t(w[1] >> 8);
  o.q[2] = uint8_t(w[1] >> 16);
  o.q[3] = uint8_t(w[1] >> 24);
  o.cmask = w[2];
  o.cval = w[3];
  o.mat = w[4];
  o.dmat[0] = w[5];
  o.dmat[1] = w[6];
  o.col[0] = int32_t(w[7]);
  o.col[1] = int32_t(w[8]);
  return o;
}

// A lane's part of an op's matrix (or its adjoint, DAG) and its product with v, the lane's
// 2^K amplitudes.  Two qubits: MFMA rows.  One qubit: the matrix, for FMAs on a pair; on
// MFMA a pair would need another one beside it, with zeros between the two: NaN in both
// where one of them is not finite.
template <int K, bool DAG>
struct LaneMatrix;

// The products of a two-qubit op are added in the order of apply_dense (lds_ops.h):
// column 0 as cmul contracts it (the product that is rounded by itself first; another one
// in the adjoint, where the imaginary part is a difference), the others as cmacf.  So
// amplitudes have the bits that the FMA path gives them, and a shot, drawn by comparing a
// prefix sum with a uniform, the same outcome.
template <bool DAG>
struct LaneMatrix<2, DAG> {
  MfmaRows m;
  __device__ __forceinline__ explicit LaneMatrix(const float2* __restrict__ M) {
    mfma_rows<DAG>(M, m);
  }
  __device__ __forceinline__ void apply(const float2 (&v)[4], float2 (&o)[4]) const {
    const mf4 zero{0.f, 0.f, 0.f, 0.f};
    mf4 dr = mfma4(m.ngi[0], v[0].y, zero);
    mf4 di = DAG ? mfma4(m.gi[0], v[0].x, zero) : mfma4(m.gr[0], v[0].y, zero);
    dr = mfma4(m.gr[0], v[0].x, dr);
    di = DAG ? mfma4(m.gr[0], v[0].y, di) : mfma4(m.gi[0], v[0].x, di);
#pragma unroll
    for (int k = 1; k < 4; ++k) {
      dr = mfma4(m.gr[k], v[k].x, dr);
      di = mfma4(m.gr[k], v[k].y, di);
      dr = mfma4(m.ngi[k], v[k].y, dr);
      di = mfma4(m.gi[k], v[k].x, di);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) o[s] = make_float2(dr[s], di[s]);
  }
};
template <bool DAG>
struct LaneMatrix<1, DAG> {
  float2 m[4];
  __device__ __forceinline__ explicit LaneMatrix(const float2* __restrict__ M) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      m[i] = M[DAG ? (i & 1) * 2 + (i >> 1) : i];
      if (DAG) m[i].y = -m[i].y;
    }
  }
  __device__ __forceinline__ void apply(const float2 (&v)[2], float2 (&o)[2]) const {
    o[0] = cmacf(cmul(m[0], v[0]), m[1], v[1]);
    o[1] = cmacf(cmul(m[2], v[0]), m[3], v[1]);
  }
};

// As cache_span, by one wavefront.
__device__ __forceinline__ void cache_span_solo(MatCache& c, uint32_t off, uint32_t len) {
  if (off >= c.lo && off + len <= c.hi) return;
  esync<true>();
#pragma unroll 8
  for (uint32_t i = threadIdx.x & 63u; i < c.n; i += 64u) c.lds[i] = c.g[off + i];
  esync<true>();
  c.lo = off;
  c.hi = off + c.n;
}

// Gradient partials of one wavefront.  A derivative leaves one float per lane;
// reduced one by one they cost as much as the op itself (four FP64 steps across
// the lanes and an atomic, all latency), so kPartDerivs of them are kept in LDS
// and reduced together: lane l sums an eighth of derivative l / 8 in FP64, three
// steps add the eighths, and one instruction adds the sums of all of them.
constexpr int kPartDerivs = 8;
template <bool CPLX>
struct PartRing {
  float part[kPartDerivs][64];
  float part_im[CPLX ? kPartDerivs : 1][CPLX ? 64 : 1];
  int col[kPartDerivs];
};
template <bool CPLX, typename AccFn>
__device__ __forceinline__ void flush_parts(const PartRing<CPLX>* r, int count, AccFn&& acc_fn) {
  const int lane = int(threadIdx.x & 63u), d = lane >> 3, s = lane & 7;
  auto eighth = [&](const float* p) {
    double v = 0.0;
#pragma unroll
    for (int i = 0; i < 8; ++i) v += double(p[i]);
    v = dpp_add<0xB1>(v);    // lane ^ 1
    v = dpp_add<0x4E>(v);    // lane ^ 2
    return dpp_add<0x141>(v);  // the other half of the eight
  };
  const double re = eighth(&r->part[d][8 * s]);
  const double im = CPLX ? eighth(&r->part_im[CPLX ? d : 0][CPLX ? 8 * s : 0]) : 0.0;
  if (s == 0 && d < count) acc_fn(r->col[d], re, im);
}

// One dense or parameterised op of K qubits on the states A and (REV) B: 2^K amplitudes
// a lane and round.  A derivative's partials are summed over a lane's 2^K amplitudes in
// FP32, over everything else in FP64.
template <int K, bool REV, bool SOLO, bool CPLX, typename AccFn>
__device__ __forceinline__ void lds_dense(float2* __restrict__ A, float2* __restrict__ B, int n,
                                          const DevOp& op, const float2* __restrict__ M,
                                          PartRing<CPLX>* ring, int& parts, AccFn&& acc_fn) {
  constexpr int D = 1 << K;
  constexpr uint32_t kStep = SOLO ? 64u : uint32_t(kThreads);
  const uint32_t lane = threadIdx.x & 63u, first = SOLO ? 0u : threadIdx.x & ~63u;
  const uint32_t count = 1u << (n - K);
  const int nd = REV && op.type == kOpParam ? op.nderiv : 0;
  uint32_t dep[D];
#pragma unroll
  for (int s = 0; s < D; ++s)
    dep[s] = (uint32_t(s & 1) << op.q[0]) | (K == 2 ? uint32_t(s >> 1) << op.q[1] : 0u);
  double acc[2 * kMaxDeriv] = {0.0, 0.0, 0.0, 0.0};
  if (ring && first < count) {
    // Room for this op's partials: one per derivative and round.
    const int need = nd * (count > kStep ? int(count / kStep) : 1);
    if (parts + need > kPartDerivs) {
      esync<true>();
      flush_parts<CPLX>(ring, parts, acc_fn);
      esync<true>();
      parts = 0;
    }
    if (lane < uint32_t(need)) ring->col[parts + int(lane)] = nd > 1 && (lane & 1u) ? op.col[1] : op.col[0];
  }
  const LaneMatrix<K, REV> G(M);
  // Every lane runs every round: MFMA takes its operands from all lanes.
  // Lanes past the last repeat one (and store the same values).
  for (uint32_t g0 = first; g0 < count; g0 += kStep) {
    const uint32_t g = g0 + lane;
    uint32_t x0 = insert_zero(g & (count - 1u), op.q[0]);
    if (K == 2) x0 = insert_zero(x0, op.q[1]);
    const bool ok = (x0 & op.cmask) == op.cval;
    float2 a[D], l[D], u[D], w[D];
#pragma unroll
    for (int s = 0; s < D; ++s) a[s] = A[x0 | dep[s]];
    if constexpr (REV) {
#pragma unroll
      for (int s = 0; s < D; ++s) l[s] = B[x0 | dep[s]];
    }
    // All loads are under way before the first product: in the kernels that are short of
    // registers the compiler loads one amplitude after the other (a 16-qubit state in
    // 14-qubit tiles: 1357 us, with the barrier 1216).
    __builtin_amdgcn_sched_barrier(0);
    G.apply(a, u);
    if constexpr (REV) G.apply(l, w);
    auto store = [&]() {
#pragma unroll
      for (int s = 0; s < D; ++s) A[x0 | dep[s]] = u[s];
      if constexpr (REV) {
#pragma unroll
        for (int s = 0; s < D; ++s) B[x0 | dep[s]] = w[s];
      }
    };
    if (op.cmask == 0u) store();
    else if (ok) store();
    if constexpr (REV) {
      if (nd > 0) {
#pragma unroll
        for (int d = 0; d < kMaxDeriv; ++d) {
          if (d >= nd) break;
          float2 t[D];
          LaneMatrix<K, false>(M + D * D * (1 + d)).apply(u, t);
          float part = 0.f, part_im = 0.f;
#pragma unroll
          for (int s = 0; s < D; ++s) {
            part = __builtin_fmaf(t[s].x, l[s].x, part);
            part = __builtin_fmaf(t[s].y, l[s].y, part);
            part_im = __builtin_fmaf(t[s].x, l[s].y, part_im);
            part_im = __builtin_fmaf(-t[s].y, l[s].x, part_im);
          }
          if (g >= count || !ok) part = part_im = 0.f;
          if (ring) {
            ring->part[parts + d][lane] = part;
            if constexpr (CPLX) ring->part_im[parts + d][lane] = part_im;
          } else {
            acc[d] += double(part);
            acc[kMaxDeriv + d] += double(part_im);
          }
        }
        if (ring) parts += nd;
      }
    }
  }
  if (REV && nd > 0 && !ring && first < count) {
    const double w0 = wave_sum(acc[0]), v0 = wave_sum(acc[kMaxDeriv]);
    const double w1 = wave_sum(acc[1]), v1 = wave_sum(acc[kMaxDeriv + 1]);
    if (lane == 0u) {
      acc_fn(op.col[0], w0, v0);
      if (nd > 1) acc_fn(op.col[1], w1, v1);
    }
  }
}

// Ops [b, e) on the states A and (REV) B of n >= 2 qubits; SOLO: by this
// wavefront alone.  acc_fn(column, re, im) gets a wavefront's <dG psi | lambda>
// partials, from one lane each.  ring: room for this wavefront's partials, or
// null (LDS is full, or the state takes more rounds than the ring has entries):
// every derivative is then reduced at once.
template <bool REV, int KMAX, bool SOLO, bool CPLX, typename AccFn>
__device__ __forceinline__ void lds_ops_run(float2* __restrict__ A, float2* __restrict__ B, int n,
                                            const DevOp* __restrict__ ops, int b, int e,
                                            MatCache& mc, uint32_t* win, PartRing<CPLX>* ring,
                                            AccFn&& acc_fn) {
  constexpr uint32_t kStep = SOLO ? 64u : uint32_t(kThreads);
  const uint32_t tid = SOLO ? (threadIdx.x & 63u) : threadIdx.x;
  const uint32_t N = 1u << n;
  int parts = 0;  // derivatives in the ring
  DevOp op;
  for (int i = b, at = 0; i < e; ++i, ++at) {
    if (at == kDescWindow) at = 0;
    if (at == 0) {
      // Descriptors [i, i + kDescWindow) into the window; the op before ended
      // with a synchronisation, so its reads are done.
      const uint32_t* src = reinterpret_cast<const uint32_t*>(ops + i);
      const int words = min(e - i, kDescWindow) * kDescWords;
      for (uint32_t j = tid; j < uint32_t(words); j += kStep) win[j] = src[j];
      if (SOLO) esync<true>();
      else __syncthreads();
      op = desc_unpack(desc_word(win, 0));
    }
    const bool more = at + 1 < kDescWindow && i + 1 < e;
    const uint32_t next = desc_word(win, more ? at + 1 : at);
    if (SOLO) cache_span_solo(mc, op.mat, op_mat_len(op));
    else cache_span(mc, op.mat, op_mat_len(op));
    const float2* M = mc.lds + (op.mat - mc.lo);
    if (op.type == kOpDiag) {
      for (uint32_t x = tid; x < N; x += kStep) {
        uint32_t m = (x >> op.q[0]) & 1u;
        if (op.k > 1) m |= ((x >> op.q[1]) & 1u) << 1;
        if (KMAX > 2 && op.k > 2) m |= ((x >> op.q[2]) & 1u) << 2;
        if (KMAX > 2 && op.k > 3) m |= ((x >> op.q[3]) & 1u) << 3;
        float2 d = M[m];
        if (REV) d.y = -d.y;
        if ((x & op.cmask) != op.cval) continue;
        A[x] = cmul(d, A[x]);
        if (REV) B[x] = cmul(d, B[x]);
      }
    } else if (KMAX > 2 && op.k > 2) {
      apply_op<REV, KMAX>(A, n, op, M);
      if (REV) apply_op<REV, KMAX>(B, n, op, M);
    } else if (op.k == 2) {
      lds_dense<2, REV, SOLO, CPLX>(A, B, n, op, M, ring, parts, acc_fn);
    } else {
      lds_dense<1, REV, SOLO, CPLX>(A, B, n, op, M, ring, parts, acc_fn);
    }
    op = desc_unpack(next);
    if (SOLO) esync<true>();
    else __syncthreads();
  }
  if (REV && parts > 0) flush_parts<CPLX>(ring, parts, acc_fn);
}

// Ops [b, e) on a state (and, REV, a second one) in LDS.  The caller has
// synchronised its writes to the states; on return the workgroup has.  win:
// kDescWindow descriptors' room in LDS; rings: a PartRing per wavefront, or null.
template <bool REV, int KMAX, bool CPLX, typename AccFn>
__device__ __forceinline__ void lds_run(float2* A, float2* B, int n, const DevOp* ops, int b, int e,
                                        MatCache& mc, uint32_t* win, PartRing<CPLX>* rings,
                                        AccFn&& acc_fn) {
  if (b >= e) return;
  __syncthreads();
  // At most two rounds, so that an op's partials fit the ring.
  PartRing<CPLX>* ring =
      REV && rings && (1u << n) <= 4u * kThreads ? rings + (threadIdx.x >> 6) : nullptr;
  if (KMAX <= 2 && n <= kSoloMaxQubits) {
    // All wavefronts fill the window once; then the first runs the list.
    const DevOp op0 = load_op(ops + b);
    cache_span(mc, op0.mat, op_mat_len(op0));
    if (threadIdx.x < 64u)
      lds_ops_run<REV, KMAX, true, CPLX>(A, B, n, ops, b, e, mc, win, ring, acc_fn);
    mc.lo = mc.hi = kNoWindow;  // the others do not know where the window is now
    __syncthreads();
    return;
  }
  lds_ops_run<REV, KMAX, false, CPLX>(A, B, n, ops, b, e, mc, win, ring, acc_fn);
}

}  // namespace
}  // namespace tfqx
