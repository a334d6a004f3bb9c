// rebind_kernel: a plan's symbolic matrices re-evaluated on the device for
// new symbol values (tables described in rebind_device.h).
//
// Every function here is the device counterpart of a host function that
// builds the same matrices when a plan is created or rebound on the host
// (circuit.cc: UnitaryOrDeriv, EigenEval, GateDerivative; plan.cc: ApplyLeft,
// BlockMatrix, ParamBlockMatrices, Embed, WriteMatrix, RebindRow), with the
// same operations in the same order.  Contraction is off so every double
// product and sum is rounded on its own, as in the host build.
//
// Sixteen lanes work on one op, four ops per wavefront.  What bounds the
// kernel is latency, of memory and of instruction fetch: a call has few ops
// (hundreds to some ten thousand), and each is a chain of loads, a sine and
// cosine per gate, and a product of the gates.  So the lanes take the chain's
// independent parts: first every gate (and every +-eps evaluation of a gradient
// gate) is one lane's, which computes its phases; then every matrix entry is one
// lane's; then every column of the op's product and of its derivative products
// is one lane's, which runs the gates in order.  All gate kinds share one
// sine/cosine site and one entry routine, so the code stays small.
//
// One lane per op (the former layout, with each kind unrolled: 325 KB of code
// fetched anew by each launch) took 137 us on 64 circuits of 10 qubits and 600
// symbols, 107 us on one 12-qubit ansatz of 144 symbols and 659 us on 2048 uneven
// circuits; this one takes 47, 12 and 312 us.  Six gates at a time keep the working
// set at 3.4 KB per op, so eleven wavefronts share a CU (twelve gates, seven
// wavefronts: 59, 13 and 428 us).
#include "rebind_device.h"
#include "tfqx_internal.h"

#pragma clang fp contract(off)

namespace tfqx {
namespace {

constexpr double kPi = 3.14159265358979323846;
constexpr float kGradEps = 5e-3f;  // adj_util.cc:32
constexpr int kRbThreads = 64;
constexpr int kGroup = 16;                        // lanes per op
constexpr int kGroups = kRbThreads / kGroup;      // ops per workgroup (one wavefront)
constexpr int kChunk = 6;                         // gates evaluated at a time
constexpr int kSlots = kChunk + 2 * kMaxDeriv;    // ... and the +-eps evaluations of two derivatives
static_assert(kSlots <= kGroup, "a lane per evaluation");

struct dc {
  double re, im;
};

__device__ inline dc Mul(dc a, dc b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ inline dc Scale(dc a, double s) { return {a.re * s, a.im * s}; }
__device__ inline dc Add(dc a, dc b) { return {a.re + b.re, a.im + b.im}; }
__device__ inline double Mul32(float a, float b) { return double(a * b); }

// One evaluated gate of a chunk.  pidx < 0: the unitary; otherwise the exact
// derivative with respect to argument pidx, whose scale is sc.
struct Slot {
  dc w[4];       // the gate's phases (see Phases)
  double sc;
  int kind, pidx;
  int nt;        // targets
  int pos;       // block position of target 0 | of target 1 << 8
  int cm, cv;    // controls inside the block
};
// Per-op working set in LDS.
struct Work {
  Slot slot[kSlots];
  dc U[kSlots][16];
};

// LDS traffic of one wavefront is in order; this keeps the compiler's order too.
__device__ inline void WaveSync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The phases e^{iy} a gate's entries are made of, for arguments p:
//   eigen gates   w[k] = e^{i pi t (lam_k + gs)} (times i pi (lam_k + gs): derivative)
//   PhasedX       those of X, w[2] = e^{-i pi phase}
//   FSim          w[0] = e^{i theta}, w[1] = e^{-i phi}
//   PhasedISwap   those of ISwap, w[3] = e^{2 i pi phase}
__device__ void Phases(const RbEigen* table, int kind, const float* p, int pidx, Slot* s) {
  const bool phased = kind == 13 || kind == 15;
  const double a = Mul32(p[0], p[1]), b = Mul32(p[2], p[3]);
  const double t = phased ? b : a;
  const double gs = kind == 13 ? double(p[4]) : kind == 15 ? 0.0 : double(p[2]);
  const bool deriv = phased ? pidx == 2 : pidx >= 0;
  const RbEigen& e = table[kind == 13 ? 3 : kind == 15 ? 12 : kind == 14 ? 0 : kind];
  const int count = kind == 14 ? 2 : kind < 2 ? 0 : int(e.count);
#pragma unroll 1
  for (int k = 0; k < 4; ++k) {
    double y;
    if (kind == 14) y = k == 0 ? a : -b;
    else if (k < count) y = kPi * t * (e.lam[k] + gs);
    else if (kind == 13 && k == 2) y = -kPi * a;
    else if (kind == 15 && k == 3) y = 2 * kPi * a;
    else continue;
    if (kind == 14 && k >= count) continue;
    dc w;
    sincos(y, &w.im, &w.re);
    if (deriv && kind != 14 && k < count) w = Mul(w, dc{0.0, kPi * (e.lam[k] + gs)});
    s->w[k] = w;
  }
  s->sc = double((phased || kind == 14) && pidx == 2 ? p[3] : p[1]);
}

// Entry i (row-major) of the slot's matrix.
__device__ dc Entry(const RbEigen* table, const Slot& s, int i) {
  const dc zero{0.0, 0.0}, negI{-0.0, -1.0};
  const int kind = s.kind, pidx = s.pidx;
  if (kind < 2) return pidx < 0 && i % (kind == 0 ? 3 : 5) == 0 ? dc{1.0, 0.0} : zero;
  if (kind == 14) {
    const double c = s.w[0].re, sn = s.w[0].im;
    const bool diag = i == 5 || i == 10, off = i == 6 || i == 9;
    if (pidx < 0)
      return i == 0 ? dc{1.0, 0.0} : diag ? dc{c, 0.0} : off ? Scale(negI, sn) : i == 15 ? s.w[1] : zero;
    if (pidx == 0)
      return diag ? dc{-sn * s.sc, 0.0} : off ? Scale(Scale(negI, c), s.sc) : zero;
    return i == 15 ? Scale(Mul(negI, s.w[1]), s.sc) : zero;
  }
  const RbEigen& e = table[kind == 13 ? 3 : kind == 15 ? 12 : kind];
  dc u = zero;
  const int count = int(e.count);
  dc P[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) P[k] = dc{e.P[k][2 * i], e.P[k][2 * i + 1]};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const dc x = Add(u, Mul(s.w[k], P[k]));
    if (k < count) u = x;
  }
  if (kind <= 12) return pidx >= 0 ? Scale(u, s.sc) : u;
  // PhasedX / PhasedISwap: the off-diagonal pair gains opposite phases.
  const int lo = kind == 13 ? 1 : 6, hi = kind == 13 ? 2 : 9;
  if (i == lo || i == hi) {
    // PhasedX: e^{-i pi phase} above the diagonal; PhasedISwap: e^{2 i pi phase}.
    dc ph = s.w[kind == 13 ? 2 : 3];
    if (i == hi) ph.im = -ph.im;
    u = Mul(u, ph);
    if (pidx == 0) {
      const double f = kind == 13 ? (i == lo ? -kPi : kPi) : (i == lo ? 2 * kPi : -2 * kPi);
      u = Mul(u, Scale(dc{0.0, f}, s.sc));
    }
  } else if (pidx == 0) {
    u = zero;
  }
  return pidx == 2 ? Scale(u, s.sc) : u;
}

// Evaluate gate `src` for the row's values v into slot s: its unitary (delta =
// 0, pidx < 0), the unitary with argument pidx shifted by delta, or (delta = 0)
// the exact derivative.  bits: the op's K qubits.
__device__ void EvalGate(const RebindArgs& a, const RbGate& src, const float* v, int pidx,
                         float delta, const int* bits, int k, bool controls, Slot* s) {
  const int nsym = src.nsym;
  const float v0 = nsym > 0 ? v[src.sym_col[0]] : 0.0f;
  const float v1 = nsym > 1 ? v[src.sym_col[1]] : 0.0f;
  float p[5];
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    p[j] = (nsym > 1 && src.sym_pidx[1] == j) ? v1
         : (nsym > 0 && src.sym_pidx[0] == j) ? v0 : src.params[j];
    if (delta != 0.0f && j == pidx) p[j] += delta;
  }
  s->kind = src.kind;
  s->pidx = delta != 0.0f ? -1 : pidx;
  s->nt = src.nt;
  int pos = 0, cm = 0, cv = 0;
  for (int m = 0; m < k; ++m) {
    if (bits[m] == src.bits[0]) pos |= m;
    if (src.nt > 1 && bits[m] == src.bits[1]) pos |= m << 8;
    if (controls && (src.cmask >> bits[m] & 1)) {
      cm |= 1 << m;
      if (src.cval >> bits[m] & 1) cv |= 1 << m;
    }
  }
  s->pos = pos;
  s->cm = cm;
  s->cv = cv;
  Phases(a.eigen, src.kind, p, s->pidx, s);
}

// TFQ's gradient gate (adj_util.cc:175-302) from the two shifted unitaries: the
// float32 central difference, as the host combines them.
__device__ inline dc FdEntry(dc up, dc um) {
  const float scale = float(0.5 / double(kGradEps));
  const float re = float(up.re) - float(um.re), im = float(up.im) - float(um.im);
  return {double(re * scale), double(im * scale)};
}

// One column of the block product: v <- (gate embedded in the block) v.  The
// column's 2^K entries are in registers for K <= 2.  D: the derivative's slots
// instead of the gate's unitary (fd: two shifted unitaries to combine).
__device__ inline dc MatEntry(const Work& wk, int t, int d, bool fd, int i) {
  if (d < 0) return wk.U[t][i];
  const dc up = wk.U[kChunk + 2 * d][i];
  return fd ? FdEntry(up, wk.U[kChunk + 2 * d + 1][i]) : up;
}

template <int DIM>
__device__ void ApplyColumn(const Work& wk, int t, int d, bool fd, dc* v) {
  const Slot& s = wk.slot[t];
  const int p0 = s.pos & 255, p1 = s.pos >> 8, cm = s.cm, cv = s.cv;
  if (s.nt == 1) {
    dc u[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = MatEntry(wk, t, d, fd, i);
    if constexpr (DIM <= 4) {
#pragma unroll
      for (int b = 0; b < (DIM > 2 ? 2 : 1); ++b) {
        if (b != p0) continue;
#pragma unroll
        for (int r0 = 0; r0 < DIM; ++r0) {
          if (r0 & (1 << b)) continue;
          if ((r0 & cm) != cv) continue;
          const dc x = v[r0], y = v[r0 | (1 << b)];
          v[r0] = Add(Add(dc{0.0, 0.0}, Mul(u[0], x)), Mul(u[1], y));
          v[r0 | (1 << b)] = Add(Add(dc{0.0, 0.0}, Mul(u[2], x)), Mul(u[3], y));
        }
      }
    } else {
      for (int r0 = 0; r0 < DIM; ++r0) {
        if ((r0 >> p0) & 1 || (r0 & cm) != cv) continue;
        const dc x = v[r0], y = v[r0 | (1 << p0)];
        v[r0] = Add(Add(dc{0.0, 0.0}, Mul(u[0], x)), Mul(u[1], y));
        v[r0 | (1 << p0)] = Add(Add(dc{0.0, 0.0}, Mul(u[2], x)), Mul(u[3], y));
      }
    }
    return;
  }
  if constexpr (DIM <= 4) {
    // Both block qubits are targets (no room for a control).  Block index r is
    // the gate's index with its two bits swapped when target 0 (the matrix's
    // most significant bit) sits at position 0.
    if constexpr (DIM == 4) {
      const bool swap = p0 == 0;
      dc x[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = v[r];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int e = swap ? ((r & 1) << 1 | r >> 1) : r;
        // Summed in the gate's index order, as the host does.
        dc sum{0.0, 0.0};
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const int c = (b & 1) << 1 | b >> 1;
          const dc xb = swap ? x[c] : x[b];
          sum = Add(sum, Mul(MatEntry(wk, t, d, fd, e * 4 + b), xb));
        }
        v[r] = sum;
      }
    }
  } else {
    const int gm = (1 << p0) | (1 << p1);
    for (int r0 = 0; r0 < DIM; ++r0) {
      if ((r0 & gm) || (r0 & cm) != cv) continue;
      dc x[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) x[b] = v[r0 | ((b >> 1) << p0) | ((b & 1) << p1)];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        dc sum{0.0, 0.0};
#pragma unroll
        for (int b = 0; b < 4; ++b) sum = Add(sum, Mul(MatEntry(wk, t, d, fd, e * 4 + b), x[b]));
        v[r0 | ((e >> 1) << p0) | ((e & 1) << p1)] = sum;
      }
    }
  }
}

// One op per kGroup lanes: per-row tables list every row's ops (op.row names the
// row); shared tables hold one program's ops for every row.  DIM: 4 when every
// op has at most two qubits (columns in registers), else 16 (columns in LDS;
// such ops are fused blocks without derivatives, one column per lane).
template <int DIM>
__global__ __launch_bounds__(kRbThreads) void rebind_kernel(RebindArgs a) {
  __shared__ Work work[kGroups];
  __shared__ dc cols[DIM > 4 ? kRbThreads * DIM : 1];
  const int g = int(threadIdx.x) / kGroup, lane = int(threadIdx.x) % kGroup;
  const long long i = (long long)blockIdx.x * kGroups + g;
  const long long items = a.shared ? (long long)a.num_ops * a.num_rows : a.num_ops;
  if (i >= items) return;
  Work& wk = work[g];
  const RbOp& op = a.ops[a.shared ? int(i % a.num_ops) : int(i)];
  const RbRow& row = a.rows[a.shared ? int(i / a.num_ops) : op.row];
  const float* vals = a.values + size_t(row.vrow) * a.num_symbols;
  float2* mats = a.mats + row.mat_base;
  const int k = op.k, kind = op.kind, nd = op.nderiv, ng = op.gate_end - op.gate_begin;
  const bool block = kind == 0 || kind == 3;  // else one gate, controls outside the matrix
  const int npass = kind == 0 ? 1 : 1 + nd, ngates = block ? ng : 1;
  const bool fd = a.tfq_fd != 0;
  int bits[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) bits[m] = op.bits[m];
  const int dim = 1 << k;
  // This lane's column: of derivative product `pass - 1`, or of the op's matrix.
  const int pass = DIM > 4 && dim > 4 ? 0 : lane >> 2;
  const int col = DIM > 4 && dim > 4 ? lane : lane & 3;
  const bool mine = pass < npass && col < dim;
  const int dgate = pass > 0 && mine ? (block ? op.dgate[pass - 1] : 0) : -1;
  dc reg[4];
  dc* v = reg;
  if constexpr (DIM > 4) v = cols + threadIdx.x * DIM;
#pragma unroll
  for (int r = 0; r < (DIM > 4 ? 16 : 4); ++r) v[r] = {r == col ? 1.0 : 0.0, 0.0};
#pragma unroll 1
  for (int t0 = 0; t0 < ngates; t0 += kChunk) {
    const int nt = min(kChunk, ngates - t0);
    // Phases: lane t a gate of the chunk, the last lanes the gradient gates in it.
    int gate = -1, pidx = -1;
    float delta = 0.0f;
    if (lane < kChunk) {
      if (lane < nt) gate = t0 + lane;
    } else if (lane < kSlots) {
      const int s = (lane - kChunk) >> 1, minus = (lane - kChunk) & 1;
      if (s < npass - 1 && (fd || !minus)) {
        const int dg = block ? op.dgate[s] : 0;
        if (dg >= t0 && dg < t0 + nt) {
          gate = dg;
          delta = !fd ? 0.0f : minus ? -kGradEps : kGradEps;
        }
      }
    }
    if (gate >= 0) {
      const RbGate& src = a.gates[row.gate_base + a.gidx[row.gidx_base + op.gate_begin + gate]];
      if (lane >= kChunk) {
        const int s = (lane - kChunk) >> 1;
        pidx = src.sym_pidx[block ? op.dsym[s] : s];
      }
      EvalGate(a, src, vals, pidx, delta, bits, k, block, &wk.slot[lane]);
    }
    // Which slots hold a gate, for every lane of the group.
    const unsigned long long live = __ballot(gate >= 0) >> (g * kGroup);
    WaveSync();
    // Four slots at a time, four entries of each (a two-qubit gate's 16 in four steps).
#pragma unroll 1
    for (int t4 = 0; t4 < kSlots; t4 += 4) {
      const int t = t4 + (lane >> 2);
      if (t >= kSlots || !((live >> t) & 1)) continue;
      const int ne = wk.slot[t].nt == 1 ? 4 : 16;
#pragma unroll 1
      for (int e = lane & 3; e < ne; e += 4) wk.U[t][e] = Entry(a.eigen, wk.slot[t], e);
    }
    WaveSync();
    if (mine)
#pragma unroll 1
      for (int t = 0; t < nt; ++t)
        ApplyColumn<DIM>(wk, t, t0 + t == dgate ? pass - 1 : -1, fd, v);
    WaveSync();
  }
  if (!mine) return;
  float2* dst = mats + (pass == 0 ? op.mat : op.dmat[pass - 1]);
  if (pass == 0 && kind != 3 && op.diag != 0) {
#pragma unroll
    for (int r = 0; r < DIM; ++r)
      if (r == col) dst[r] = make_float2(float(v[r].re), float(v[r].im));
  } else {
#pragma unroll
    for (int r = 0; r < DIM; ++r)
      if (r < dim) dst[r * dim + col] = make_float2(float(v[r].re), float(v[r].im));
  }
}

}  // namespace

hipError_t LaunchRebind(const RebindArgs& a, int kmax, hipStream_t stream) {
  const long long items = a.shared ? (long long)a.num_ops * a.num_rows : a.num_ops;
  if (items <= 0) return hipSuccess;
  const dim3 grid(unsigned((items + kGroups - 1) / kGroups)), block(kRbThreads);
  if (kmax <= 2)
    hipLaunchKernelGGL(rebind_kernel<4>, grid, block, 0, stream, a);
  else
    hipLaunchKernelGGL(rebind_kernel<16>, grid, block, 0, stream, a);
  return hipGetLastError();
}

}  // namespace tfqx
