// Kernels of the VMC particle-move engine.  Included once, by qmcx_capi.hip.
//
// Data layout in HBM (per batch of W walkers, n = orbitals = electrons per spin,
// N = 2n electrons, M ions, K = delay rank):
//   R       double [W][3][N]       positions, SoA
//   A       T      [W][2][n][n]    Slater rows phi_j(r_i) (row = electron)
//   Ainv    T      [W][2][n][n]    psiM = (A^-1)^T (DiracDeterminant::psiM)
//   dpsiM   T      [W][2][n][3][n] orbital gradients of each row, SoA per row
//   d2psiM  T      [W][2][n][n]    h_xx of each row (einspline_spo.hpp:220)
//   J2, J1  T      [W][5][N]       Uat,dUx,dUy,dUz,d2Uat  /  Vat,Gx,Gy,Gz,Lap
//   Vbuf    T      [W][K][n]       stale inverse rows of the delayed electrons
//   Binv    T      [W][K][K]       inverse of the delayed capacitance matrix
//   rows    int    [W][K]          delayed rows;  ndelay int [W]
//   logdet, phase double [W][2]; jlog double [W][3] (J1, J2, J3)
#pragma once
#include <limits.h>

#include "qmcx_device.hpp"
#include "qmcx_j3.hpp"
#include "qmcx_walk.hpp"

namespace qmcx {

template <typename T>
struct SysP {
  const Cell<T>* cell;        // device copy of the minimum-image cell
  const double* spoG;         // [9] inverse of the SPO lattice
  int ng[3];
  int N, n, M, nspecies;
  int npad;
  long long xs, ys, zs;
  const T* coefs;
  const double* ions;         // [3][M]
  const int* species;         // [M]
  const Functor<T>* fn;       // [kMaxSpecies] J1 then [2] J2
  const Functor<double>* fn64;  // the same functors in FP64 (FP64 arbitration of the FP32 form)
  const Cell<double>* cell64;   // the minimum-image cell in FP64
  // three-body Jastrow: functor of (ion species, spin pair) at [2 * species + pair] (L = 0 for a
  // species without one), or null; mw = 64-bit words of an electron's ion mask, ceil(M / 64)
  const Poly3<T>* j3;
  const Poly3<double>* j3_64;   // the same functors in FP64 (FP64 re-evaluation of the FP32 form)
  int mw;
};

template <typename T>
struct BatchP {
  int W, K;
  int nch;         // delayed-update state slots per walker and determinant (one per chunk)
  double* R;
  T* A;
  T* Ainv;
  T* dpsiM;
  T* d2psiM;
  T* J2;
  T* J1;
  // delayed-update state of chunk j of determinant det of walker w, slot (w*2 + det)*nch + j:
  // V rows Vbuf[slot][K][n], Binv[slot][K][K], rows[slot][K], ndelay[slot]
  T* Vbuf;
  double* Binv;    // capacitance-matrix inverse kept in FP64 in both precisions
  int* rows;
  int* ndelay;
  double* logdet;
  double* phase;
  double* jlog;
  unsigned long long* nacc;
  double* trace;   // [W][N][9] or null
  // device sweep counters: [0] the sweep the moves are in (advanced on the batch stream after
  // evaluateGL), [1] the first sweep of the current run, [2] the sweep of the proposals being
  // evaluated (advanced on the proposals stream), [3] the history slot of the latest evaluateGL
  int* sweep;
  // FP32 form only (null in FP64): the Slater rows summed in FP64 from the same coefficients,
  // A64 [W][2][n][n] and at the sweep's proposals spo64 [W][2][n][npad]
  double* A64;
  double* spo64;
  unsigned long long* narb;   // [W] Metropolis decisions settled by the FP64 re-evaluation
  // three-body Jastrow (with S.j3): sums J3 [W][5][N] (U, grad U xyz, lap U), ion masks j3mask
  // [W][N][mw] (bit I: the electron is within L_I of ion I), near-ion records of the current
  // positions j3near [W][N][kJ3Rec] and of the sweep's proposals j3prop [W][2][n][kJ3Rec]
  T* J3;
  unsigned long long* j3mask;
  T* j3near;
  T* j3prop;
  int* flags;      // [1] error bits set by kernels (kFlag*)
};

// kernel error bits in BatchP::flags
constexpr int kFlagJ3Near = 1;    // an electron position with more than kJ3Near ions inside the J3 cutoff
constexpr int kFlagJ3Pairs = 2;   // a wave's J3 pairs of one move phase beyond its slots

// Proposal record of one electron, [W][2][n][kProp] doubles written by k_spo_proposals:
// J1 at the proposal (sum u, sum (d2u + 2 du/r), gradient), the displacement, the
// acceptance uniform.
constexpr int kProp = 10;
constexpr int kPropJ1 = 0, kPropDispl = 5, kPropU = 8;

template <typename T>
__host__ __device__ inline size_t state_slot(const BatchP<T>& B, int w, int det, int j) {
  return ((size_t)w * 2 + det) * B.nch + j;
}

struct MoveArgs {
  int e_begin, e_end, det, mode, slices;
  // The launch moves electrons [e_begin, e_end) in nchunks chunks of chunk_len; chunk is the
  // index of its first chunk in the determinant's sweep.  inflush: the kernel applies each
  // chunk's delayed updates to the walker's whole inverse before the next chunk (1), and after
  // the last chunk too (2); 0: a flush launch follows each single-chunk launch.  The kernel's
  // flush takes the new Slater rows from LDS when at most flush_u moves of the chunk were
  // accepted, else from HBM.
  int chunk, chunk_len, nchunks, inflush, flush_u;
  // streamed delayed updates: the launch continues from the delayed rows pending in its state slot
  // (flex_* calls keep them pending until the delay rank is reached or completeUpdates)
  int resume;
  // FP64 recompute cadence (cadence > 0 accepted rows): a walker's moves of the determinant start
  // at its own position cad[w][det][0] and stop after the move that brings its accepted rows since
  // the last recompute (cad[w][det][1]) to cadence; it then sets cad_flag[w] for the recompute
  int cadence;
  int* cad;
  int* cad_flag;
  const int* decide;     // [W] caller accept decisions (flex_acceptrestoreMove) or null
  double* record;        // [W][9] the move's trace record for the flex calls (host memory), or null
  // FP32 form, Metropolis: a move whose uniform u lies within band * ratio^2 of ratio^2 is
  // decided on its FP64 ratio (0: off)
  double band;
  const void* spo;       // [W][2][n][5][npad] T: SPO rows at the proposals (k_spo_proposals)
  const double* prop;    // [W][2][n][kProp] proposal records (k_spo_proposals)
};

// ------------------------------------------------------------------ spline gather
// One workgroup evaluates NO outputs (1: v; 5: v, gx, gy, gz, hxx; 10: full VGH) of
// every orbital at one point.  Lane (q, s): q = 16-byte orbital group, s =
// stencil slice owning 16/S of the (i,j) columns of the 4x4x4 stencil; each
// lane issues 4*16/S coalesced 16-byte loads along the orbital axis.  Slice
// partials go to LDS `part` [S][NO][npad] and are summed by `spline_finish`.
// weight, first and second derivative of cubic B-spline knot i (0..3) at fraction t
template <typename T>
__device__ inline void knot_weight(int i, T t, T& w, T& dw, T& d2w) {
  const T s6 = T(1) / T(6);
  // w = ((p3 t + p2) t + p1) t + p0, dw = (q2 t + q1) t + q0, d2w = r1 t + r0
  const T p3 = i == 0 ? T(-1) : i == 1 ? T(3) : i == 2 ? T(-3) : T(1);
  const T p2 = i == 0 ? T(3) : i == 1 ? T(-6) : i == 2 ? T(3) : T(0);
  const T p1 = i == 0 ? T(-3) : i == 1 ? T(0) : i == 2 ? T(3) : T(0);
  const T p0 = i == 0 ? T(1) : i == 1 ? T(4) : i == 2 ? T(1) : T(0);
  w = (((p3 * t + p2) * t + p1) * t + p0) * s6;
  dw = ((T(3) * p3 * t + T(2) * p2) * t + p1) * s6;
  d2w = (T(6) * p3 * t + T(2) * p2) * s6;
}

// V64: the value is also summed in FP64 (weights from the FP64 fraction, the same loaded
// coefficients) into part64 [S][npad]: the FP64 Slater rows of the FP32 form.
// The partial sums of lane tid (orbital quad q, stencil slice s) in registers: acc[o][e] for
// orbital q*VW + e, and with V64 the FP64 values acc64.  False for the lanes past the slices.
// UNI (one slice only): the point is the same on every lane of the wave, so its grid cell moves
// to scalar registers and every load takes a scalar address plus the lane's orbital offset.
// KEEP: cached loads (the points are ordered by place, so neighbours want the same coefficients);
// else non-temporal ones.
template <typename T, int NO, int PER, bool V64, bool UNI = false, bool KEEP = false>
__device__ inline bool spline_gather_regs(const SysP<T>& S, const double* spoG, double x, double y, double z, int tid,
                                          T (&acc)[NO][V16<T>::n], double (&acc64)[V16<T>::n], int& q, int& s) {
  using VT = typename V16<T>::type;
  constexpr int VW = V16<T>::n;
  constexpr int SL = 16 / PER;
  // stencil columns with loads in flight per batch: up to four in FP32 (two when the FP64 values
  // are summed as well), two in FP64
  constexpr int G = (sizeof(T) == 8 || V64) ? (PER > 2 ? 2 : PER) : (PER > 4 ? 4 : PER);
  const int nq = S.npad / VW;
  q = tid % nq;
  s = tid / nq;
  if (s >= SL) return false;
  static_assert(!UNI || SL == 1, "a wave-uniform point with one slice only");
  if constexpr (UNI) s = 0;
  int ix[3];
  double tt[3];
  spline_locate(spoG, S.ng, x, y, z, ix, tt);
  if constexpr (UNI) {
#pragma unroll
    for (int j = 0; j < 3; ++j) ix[j] = __builtin_amdgcn_readfirstlane(ix[j]);
  }
  // base0 (the cell's first coefficient) is wave-uniform with UNI; the lane's quad is added at the load
  const T* base0 = S.coefs + (size_t)ix[0] * S.xs + (size_t)ix[1] * S.ys + (size_t)ix[2] * S.zs;
  const unsigned lane_off = (unsigned)q * VW;
  const size_t zs = S.zs;
  T c[4], dc[4], d2c[4];
  bspline_weights<T>((T)tt[2], c, dc, d2c);
  const T tx = (T)tt[0], ty = (T)tt[1];
#pragma unroll
  for (int o = 0; o < NO; ++o)
#pragma unroll
    for (int e = 0; e < VW; ++e) acc[o][e] = 0;
  double c64[4];
  if constexpr (V64) {
    double dc64[4], d2c64[4];
    bspline_weights<double>(tt[2], c64, dc64, d2c64);
#pragma unroll
    for (int e = 0; e < VW; ++e) acc64[e] = 0.0;
  }
#pragma unroll
  for (int g0 = 0; g0 < PER; g0 += G) {
  VT v4[G][4];
#pragma unroll
  for (int pp = 0; pp < G; ++pp) {
    const int p = s * PER + g0 + pp;
    const T* src = base0 + (size_t)(p >> 2) * S.xs + (size_t)(p & 3) * S.ys;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const VT* c4 = reinterpret_cast<const VT*>(src + k * zs + lane_off);
      if constexpr (KEEP)
        v4[pp][k] = *c4;
      else
        v4[pp][k] = __builtin_nontemporal_load(c4);
    }
  }
#pragma unroll
  for (int pp = 0; pp < G; ++pp) {
    const int p = s * PER + g0 + pp;
    T ai, dai, d2ai, bj, dbj, d2bj;
    knot_weight<T>(p >> 2, tx, ai, dai, d2ai);
    knot_weight<T>(p & 3, ty, bj, dbj, d2bj);
    const T w00 = ai * bj, w10 = dai * bj, w01 = ai * dbj, w20 = d2ai * bj;
    const T w11 = dai * dbj, w02 = ai * d2bj;
    double w00d = 0.0;
    if constexpr (V64) {
      double a64, da64, d2a64, b64, db64, d2b64;
      knot_weight<double>(p >> 2, tt[0], a64, da64, d2a64);
      knot_weight<double>(p & 3, tt[1], b64, db64, d2b64);
      w00d = a64 * b64;
    }
#pragma unroll
    for (int e = 0; e < VW; ++e) {
      const T q0 = v4[pp][0][e], q1 = v4[pp][1][e], q2 = v4[pp][2][e], q3 = v4[pp][3][e];
      const T s0 = c[0] * q0 + c[1] * q1 + c[2] * q2 + c[3] * q3;
      acc[0][e] += w00 * s0;
      if constexpr (V64)
        acc64[e] += w00d * (c64[0] * (double)q0 + c64[1] * (double)q1 + c64[2] * (double)q2 + c64[3] * (double)q3);
      if constexpr (NO >= 5) {
        const T s1 = dc[0] * q0 + dc[1] * q1 + dc[2] * q2 + dc[3] * q3;
        acc[1][e] += w10 * s0;
        acc[2][e] += w01 * s0;
        acc[3][e] += w00 * s1;
        acc[4][e] += w20 * s0;
        if constexpr (NO == 10) {
          const T s2 = d2c[0] * q0 + d2c[1] * q1 + d2c[2] * q2 + d2c[3] * q3;
          acc[5][e] += w11 * s0;
          acc[6][e] += w10 * s1;
          acc[7][e] += w02 * s0;
          acc[8][e] += w01 * s1;
          acc[9][e] += w00 * s2;
        }
      }
    }
  }
  }
  return true;
}

template <typename T, int NO, int PER, bool V64 = false>
__device__ inline void spline_gather(const SysP<T>& S, const double* spoG, double x, double y, double z, T* part,
                                     int tid, double* part64 = nullptr) {
  using VT = typename V16<T>::type;
  constexpr int VW = V16<T>::n;
  T acc[NO][VW];
  double acc64[VW];
  int q, s;
  if (!spline_gather_regs<T, NO, PER, V64>(S, spoG, x, y, z, tid, acc, acc64, q, s)) return;
  // one 16-byte LDS store per output (npad is a multiple of VW)
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    VT v;
#pragma unroll
    for (int e = 0; e < VW; ++e) v[e] = acc[o][e];
    *reinterpret_cast<VT*>(part + ((size_t)s * NO + o) * S.npad + q * VW) = v;
  }
  if constexpr (V64)
#pragma unroll
    for (int e = 0; e < VW; ++e) part64[(size_t)s * S.npad + q * VW + e] = acc64[e];
}

template <typename T, int NO, bool V64 = false>
__device__ inline void spline_gather_rt(const SysP<T>& S, double x, double y, double z, int slices, T* part,
                                        double* part64 = nullptr) {
  switch (slices) {
    case 16: spline_gather<T, NO, 1, V64>(S, S.spoG, x, y, z, part, threadIdx.x, part64); break;
    case 8: spline_gather<T, NO, 2, V64>(S, S.spoG, x, y, z, part, threadIdx.x, part64); break;
    case 4: spline_gather<T, NO, 4, V64>(S, S.spoG, x, y, z, part, threadIdx.x, part64); break;
    case 2: spline_gather<T, NO, 8, V64>(S, S.spoG, x, y, z, part, threadIdx.x, part64); break;
    default: spline_gather<T, NO, 16, V64>(S, S.spoG, x, y, z, part, threadIdx.x, part64); break;
  }
}

// the FP64 value row: slice partials summed in order, out[j] for j < norb
template <typename T>
__device__ inline void spline_finish64(const SysP<T>& S, int slices, const double* part64, double* out, int norb) {
  for (int j = threadIdx.x; j < norb; j += blockDim.x) {
    double sum = 0;
    for (int s = 0; s < slices; ++s) sum += part64[(size_t)s * S.npad + j];
    out[j] = sum;
  }
}

// delta_inv powers of output o: 1, gx, gy, gz, gx^2, gx gy, gx gz, gy^2, gy gz, gz^2
template <typename T>
__device__ inline T vgh_scale(int o, T gx, T gy, T gz) {
  const T f1 = (o == 1 || o == 4 || o == 5 || o == 6) ? gx : (o == 2 || o == 7 || o == 8) ? gy : (o == 3 || o == 9) ? gz : T(1);
  const T f2 = (o == 4) ? gx : (o == 5 || o == 7) ? gy : (o == 6 || o == 8 || o == 9) ? gz : T(1);
  return f1 * f2;
}

// Sum the slice partials and scale by the grid's delta_inv powers.
// out(o, j) for j < norb is written at out[o*ostride + j].
template <typename T, int NO, typename TO>
__device__ inline void spline_finish(const SysP<T>& S, int slices, const T* part, TO* out, int ostride, int norb) {
  const T gx = (T)S.ng[0], gy = (T)S.ng[1], gz = (T)S.ng[2];
  for (int idx = threadIdx.x; idx < NO * norb; idx += blockDim.x) {
    const int o = idx / norb, j = idx - o * norb;
    T sum = 0;
    for (int s = 0; s < slices; ++s) sum += part[((size_t)s * NO + o) * S.npad + j];
    out[(size_t)o * ostride + j] = (TO)(sum * vgh_scale<T>(o, gx, gy, gz));
  }
}

// One slice (each lane sums all 64 stencil points of its orbital quad): the scaled outputs go from
// registers to out[o*npad + j] with 16-byte stores, no LDS.  The padded orbitals (zero
// coefficients) are written too.  Equal to spline_gather + spline_finish with one slice.  The
// point must be the same on every lane of the workgroup.
// With V64 the FP64 values go to out64[j] as well.
template <typename T, int NO, bool V64 = false>
__device__ inline void spline_gather_direct(const SysP<T>& S, double x, double y, double z, T* out,
                                            double* out64 = nullptr) {
  using VT = typename V16<T>::type;
  constexpr int VW = V16<T>::n;
  T acc[NO][VW];
  double acc64[VW];
  int q, s;
  if (!spline_gather_regs<T, NO, 16, V64, true>(S, S.spoG, x, y, z, threadIdx.x, acc, acc64, q, s)) return;
  if constexpr (V64) {
#pragma unroll
    for (int e = 0; e < VW; e += 2) {
      f64x2 v;
      v[0] = 0.0 + acc64[e];
      v[1] = 0.0 + acc64[e + 1];
      *reinterpret_cast<f64x2*>(out64 + q * VW + e) = v;
    }
  }
  const T gx = (T)S.ng[0], gy = (T)S.ng[1], gz = (T)S.ng[2];
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    const T f = vgh_scale<T>(o, gx, gy, gz);
    VT v;
#pragma unroll
    for (int e = 0; e < VW; ++e) v[e] = (T(0) + acc[o][e]) * f;
    *reinterpret_cast<VT*>(out + (size_t)o * S.npad + q * VW) = v;
  }
}

}  // namespace qmcx

#include "qmcx_moves.hpp"

namespace qmcx {

// ------------------------------------------------------------------ delayed flush
// updateInvMat for K > 1 (DelayedUpdate.h:176-193), rows [m0, m0+FB) of one walker:
//   T  = Ainv U^T - E          (U rows = new Slater rows, E_{m,d} = [m == rows_d])
//   T' = T Binv
//   Ainv -= T' V               (V rows = stale inverse rows)
// A launch covers rows [lo, hi) and applies the slots holding at least thr delayed rows (thr > 1:
// the walkers whose pending rows reached the delay rank, DelayedUpdate.h:151-152).
struct FlushRows {
  int lo, hi;
  int thr = 1;
  __device__ bool writes(int m) const { return m < hi; }
};
constexpr int kFlushRows = 16;
// After a flush launch over state slot 0 of determinant det with threshold thr: the applied slots
// hold no delayed rows (a thread per walker).
template <typename T>
__global__ void k_reset_delay(BatchP<T> B, int det, int thr) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= B.W) return;
  int* nd = B.ndelay + state_slot(B, w, det, 0);
  const int c = *nd;
  if (c > 0 && c >= thr) *nd = 0;
}
// FP64 recompute cadence: a determinant's sweep starts every walker at its first electron
__global__ void k_cadence_begin(int* cad, int W, int det) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w < W) cad[((size_t)w * 2 + det) * 2] = 0;
}
// an FP64 inversion of determinant det of every walker: no accepted rows since (det < 0: both)
__global__ void k_cadence_reset(int* cad, int W, int det) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= W) return;
  for (int d = 0; d < 2; ++d)
    if (det < 0 || d == det) cad[((size_t)w * 2 + d) * 2 + 1] = 0;
}
__global__ void k_cadence_clear(int* p, int count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) p[i] = 0;
}
// one state slot j per launch
template <typename T>
__global__ __launch_bounds__(256) void k_flush_generic(SysP<T> S, BatchP<T> B, int det, int j, FlushRows FR) {
  const int w = blockIdx.y, m0 = FR.lo + blockIdx.x * kFlushRows;
  const size_t sl = state_slot(B, w, det, j);
  const int c = B.ndelay[sl];
  if (c == 0 || c < FR.thr) return;
  const int n = S.n, K = B.K, tid = threadIdx.x, nt = blockDim.x;
  extern __shared__ __align__(16) unsigned char smem[];
  T* sT = (T*)smem;                     // [FB][K]
  T* sT2 = sT + kFlushRows * K;         // [FB][K]
  int* sRows = (int*)(sT2 + kFlushRows * K);
  const size_t moff = ((size_t)w * 2 + det) * n * n;
  T* Ainv = B.Ainv + moff;
  const T* Amat = B.A + moff;
  const T* Vb = B.Vbuf + sl * K * n;
  const double* Bi = B.Binv + sl * K * K;
  for (int i = tid; i < c; i += nt) sRows[i] = B.rows[sl * K + i];
  __syncthreads();
  const int lane = tid & 63, wid = tid >> 6, nw = nt >> 6;
  for (int idx = wid; idx < kFlushRows * c; idx += nw) {
    const int m = idx / c, d = idx - m * c;
    T s = 0;
    if (m0 + m < FR.hi) {
      const T* ar = Ainv + (size_t)(m0 + m) * n;
      const T* ur = Amat + (size_t)sRows[d] * n;
      for (int j = lane; j < n; j += 64) s += ar[j] * ur[j];
    }
    s = wave_sum(s);
    if (lane == 0) sT[m * K + d] = s - ((m0 + m) == sRows[d] ? T(1) : T(0));
  }
  __syncthreads();
  for (int idx = tid; idx < kFlushRows * c; idx += nt) {
    const int m = idx / c, d = idx - m * c;
    double s = 0;
    for (int e = 0; e < c; ++e) s += (double)sT[m * K + e] * Bi[e * K + d];
    sT2[m * K + d] = (T)s;
  }
  __syncthreads();
  for (int j = tid; j < n; j += nt) {
    T acc[kFlushRows];
#pragma unroll
    for (int m = 0; m < kFlushRows; ++m) acc[m] = 0;
    for (int d = 0; d < c; ++d) {
      const T v = Vb[(size_t)d * n + j];
#pragma unroll
      for (int m = 0; m < kFlushRows; ++m) acc[m] += sT2[m * K + d] * v;
    }
#pragma unroll
    for (int m = 0; m < kFlushRows; ++m)
      if (FR.writes(m0 + m)) Ainv[(size_t)(m0 + m) * n + j] -= acc[m];
  }
}

// FP32 flush on the matrix cores (v_mfma_f32_16x16x4f32), 16 rows per wave, kFlushWaves
// waves per workgroup (one workgroup per CU covers a walker's rows in one or two launches'
// worth of workgroups).  16x16x4 operand layout: lane l supplies A[l%16][l/16] and
// B[l/16][l%16]; accumulator register r of lane l is D[4*(l/16)+r][l%16].
//
// A wave's 16 rows stay in registers between the two products, in the one layout both use:
// lane (i = l%16, g = l/16) holds row r0+i, columns 16ct + 4g .. 16ct + 4g + 3 of every
// 16-column tile ct (a float4 per tile; one HBM read of the rows, 64 contiguous bytes per
// row per load).  Both products are computed transposed:
//   GEMM 1:  T^T = U Ainv_rows^T     A = U (16 delayed rows x 4 orbitals), B = the rows
//            (orbital 16ct + 4g + r of MFMA r is the k index g), D[d][i] = T[i][d]
//   GEMM 2:  Ainv_rows^T += V^T T2^T  A = V^T (16 orbitals x 4 delayed rows), B = T2^T,
//            accumulators started from the rows themselves
// V (the stale inverse rows) and U (the new Slater rows) are staged in LDS per workgroup when
// the delay rank allows.
constexpr int kFlushWaves = 12;     // waves per workgroup, 16 rows each
constexpr int kFlushBM = 16 * kFlushWaves;   // rows per workgroup
constexpr int kFlushTiles = 24;     // 16-column tiles held in registers: n <= 384
constexpr int kFlushBinvLds = 64;   // Binv staged in LDS up to this delay rank
constexpr int kFlushVLds = 32;      // V and U staged in LDS up to this delay rank
__host__ __device__ inline bool flush_mfma_fits(int n) { return n % 16 == 0 && n <= 16 * kFlushTiles; }
__host__ __device__ inline int flush_v_stride(int n) { return n + 16; }   // LDS row stride of V
// LDS of k_flush_mfma: per wave T and T2 (16 x cp floats each; past kFlushBinvLds T2 is written
// over T), Binv (K x K doubles when K <= kFlushBinvLds), V and U (cp x (n + 16) floats each when
// K <= kFlushVLds), the row list
__host__ __device__ inline int flush_t_tiles(int K) { return K <= kFlushBinvLds ? 2 : 1; }
__host__ __device__ inline size_t flush_mfma_lds(int n, int K) {
  const int cp = (K + 15) & ~15;
  const size_t kb = K <= kFlushBinvLds ? (size_t)(K * K + 1) & ~(size_t)1 : 0;   // keeps V 16-byte aligned
  const size_t vb = K <= kFlushVLds ? (size_t)2 * cp * flush_v_stride(n) : 0;
  return sizeof(float) * kFlushWaves * flush_t_tiles(K) * 16 * cp + sizeof(double) * kb + sizeof(float) * vb +
         sizeof(int) * K;
}
// the largest delay rank whose T2 is held in registers while it is written over T
constexpr int kFlushT2Regs = 128;

// State slots [j0, j1) of determinant det are applied in order to the rows held in registers.
// OVER (delay ranks past kFlushBinvLds): T2 is written over T.
template <bool OVER>
__global__ __launch_bounds__(64 * kFlushWaves) void k_flush_mfma(SysP<float> S, BatchP<float> B, int det, int j0,
                                                                  int j1, FlushRows FR) {
  const int w = blockIdx.y;
  const int n = S.n, K = B.K, tid = threadIdx.x, nt = blockDim.x;
  const int lane = tid & 63, wid = tid >> 6, li = lane & 15, g = lane >> 4;
  const int nct = n / 16;                  // column tiles (n % 16 == 0, nct <= kFlushTiles)
  const int r0 = FR.lo + blockIdx.x * kFlushBM + wid * 16;   // this wave's first row
  const int KC = (K + 15) & ~15;           // LDS sizing uses the delay rank, not c
  // nothing to apply for this walker: no Ainv traffic
  bool any = false;
  for (int j = j0; j < j1; ++j) {
    const int cj = B.ndelay[state_slot(B, w, det, j)];
    any = any || (cj > 0 && cj >= FR.thr);
  }
  if (!any) return;
  extern __shared__ __align__(16) unsigned char smem[];
  const int tt = OVER ? 1 : 2;
  float* sT = (float*)smem + wid * tt * 16 * KC;      // [16][cp]   T = Ainv U^T - E
  float* sT2 = sT + (tt - 1) * 16 * KC;                // [16][cp]  -T Binv (over T when tt = 1)
  const bool binv_lds = K <= kFlushBinvLds;
  const bool v_lds = K <= kFlushVLds;
  double* sB = (double*)((float*)smem + kFlushWaves * tt * 16 * KC);       // [c][c]
  float* sV = (float*)(sB + (binv_lds ? (K * K + 1) & ~1 : 0));            // [cp][n + 16]
  float* sU = sV + (v_lds ? (size_t)KC * flush_v_stride(n) : 0);           // [cp][n + 16]
  int* sRows = (int*)(sU + (v_lds ? (size_t)KC * flush_v_stride(n) : 0));
  const size_t moff = ((size_t)w * 2 + det) * n * n;
  float* Ainv = B.Ainv + moff;
  const float* Amat = B.A + moff;
  const int vs = flush_v_stride(n);
  // this wave's rows into registers (row clamped into the range, zeroed after)
  const int row = r0 + li;
  const bool rok = row < FR.hi;
  const float* ar = Ainv + (size_t)(rok ? row : FR.lo) * n + 4 * g;
  f32x4_t a[kFlushTiles];
#pragma unroll
  for (int ct = 0; ct < kFlushTiles; ++ct)
    if (ct < nct) a[ct] = *reinterpret_cast<const f32x4_t*>(ar + ct * 16);
#pragma unroll
  for (int ct = 0; ct < kFlushTiles; ++ct)
    if (!rok) a[ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  bool changed = false;
  for (int j = j0; j < j1; ++j) {
    const size_t sl = state_slot(B, w, det, j);
    const int c = B.ndelay[sl];
    if (c == 0 || c < FR.thr) continue;
    changed = true;
    const int cp = (c + 15) & ~15;         // delayed rows padded to a 16-wide tile
    const float* Vb = B.Vbuf + sl * K * n;
    const double* Bi = B.Binv + sl * K * K;
    __syncthreads();                       // the previous slot's LDS reads are done
    for (int i = tid; i < c; i += nt) sRows[i] = B.rows[sl * K + i];
    if (binv_lds)
      for (int i = tid; i < c * c; i += nt) sB[i] = Bi[(i / c) * K + i % c];
    if (v_lds) {
      // V rows and the U rows they pair with, zero-padded to cp rows, float4 at a time; the
      // row list comes from HBM here too (it is being staged beside)
      const int q = n / 4;
      for (int i = tid; i < cp * q; i += nt) {
        const int d = i / q, jj = i - d * q;
        const int dc = d < c ? d : 0;
        f32x4_t v = *reinterpret_cast<const f32x4_t*>(Vb + (size_t)dc * n + 4 * jj);
        f32x4_t u = *reinterpret_cast<const f32x4_t*>(Amat + (size_t)B.rows[sl * K + dc] * n + 4 * jj);
        if (d >= c) {
          v = f32x4_t{0.f, 0.f, 0.f, 0.f};
          u = v;
        }
        *reinterpret_cast<f32x4_t*>(sV + (size_t)d * vs + 4 * jj) = v;
        *reinterpret_cast<f32x4_t*>(sU + (size_t)d * vs + 4 * jj) = u;
      }
    }
    __syncthreads();
    // ---- GEMM 1: T^T tile by tile of 16 delayed rows; two accumulators split the orbitals.
    // U rows from LDS (staged) or HBM, in separate loops so that each is its own kind of load.
    auto gemm1 = [&](const float* ur, int dt, int d) {
      f32x4_t acc0 = f32x4_t{0.f, 0.f, 0.f, 0.f}, acc1 = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ct = 0; ct < kFlushTiles; ++ct) {
        if (ct < nct) {
          f32x4_t u = *reinterpret_cast<const f32x4_t*>(ur + ct * 16);
          if (d >= c) u = f32x4_t{0.f, 0.f, 0.f, 0.f};
          f32x4_t& acc = (ct & 1) ? acc1 : acc0;
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(u[0], a[ct][0], acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(u[1], a[ct][1], acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(u[2], a[ct][2], acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(u[3], a[ct][3], acc, 0, 0, 0);
        }
      }
      // lane (i, g) register r: T[i][dt*16 + 4g + r]; minus E (row r0+i is delayed row dd)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int dd = dt * 16 + 4 * g + r;
        float v = acc0[r] + acc1[r];
        if (dd < c && sRows[dd] == r0 + li) v -= 1.f;
        sT[li * KC + dd] = dd < c ? v : 0.f;
      }
    };
    for (int dt = 0; dt < cp / 16; ++dt) {
      const int d = dt * 16 + li;
      if (v_lds) gemm1(sU + (size_t)d * vs + 4 * g, dt, d);
      else gemm1(Amat + (size_t)(d < c ? sRows[d] : sRows[0]) * n + 4 * g, dt, d);
    }
    wave_lds_fence();   // T and T2 are this wave's own
    // ---- T2 = -(T Binv), FP64 products of the small capacitance inverse
    if constexpr (OVER) {
      // over T: every lane's entries into registers first (cp <= kFlushT2Regs)
      float t2v[kFlushT2Regs / 4];
#pragma unroll
      for (int q = 0; q < kFlushT2Regs / 4; ++q) {
        const int idx = lane + 64 * q;
        double sum = 0;
        if (idx < 16 * cp) {
          const int i = idx / cp, dd = idx - i * cp;
          if (dd < c)
            for (int e = 0; e < c; ++e) sum += (double)sT[i * KC + e] * Bi[e * K + dd];
        }
        t2v[q] = (float)(-sum);
      }
      wave_lds_fence();
#pragma unroll
      for (int q = 0; q < kFlushT2Regs / 4; ++q) {
        const int idx = lane + 64 * q;
        if (idx < 16 * cp) {
          const int i = idx / cp, dd = idx - i * cp;
          sT[i * KC + dd] = t2v[q];
        }
      }
    } else
    for (int idx = lane; idx < 16 * cp; idx += 64) {
      const int i = idx / cp, dd = idx - i * cp;
      double sum = 0;
      if (dd < c) {
        if (binv_lds) {
          for (int e = 0; e < c; ++e) sum += (double)sT[i * KC + e] * sB[e * c + dd];
        } else {
#pragma unroll 8
          for (int e = 0; e < c; ++e) sum += (double)sT[i * KC + e] * Bi[e * K + dd];
        }
      }
      sT2[i * KC + dd] = (float)(-sum);
    }
    wave_lds_fence();
    // ---- GEMM 2: rows^T += V^T T2^T over the delayed rows, four at a time
    for (int d0 = 0; d0 < cp; d0 += 4) {
      const int dk = d0 + g;
      const float bv = sT2[li * KC + dk];
      const float* vr = v_lds ? sV + (size_t)dk * vs + li : Vb + (size_t)(dk < c ? dk : 0) * n + li;
#pragma unroll
      for (int ct = 0; ct < kFlushTiles; ++ct) {
        if (ct < nct) {
          float v = vr[ct * 16];
          if (!v_lds && dk >= c) v = 0.f;
          a[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(v, bv, a[ct], 0, 0, 0);
        }
      }
    }
  }
  if (changed && FR.writes(row)) {
    float* aw = Ainv + (size_t)row * n + 4 * g;
#pragma unroll
    for (int ct = 0; ct < kFlushTiles; ++ct)
      if (ct < nct) *reinterpret_cast<f32x4_t*>(aw + ct * 16) = a[ct];
  }
}

// ------------------------------------------------------------------ FP64 inverse (recompute)
// psiM = (A^T)^-1 = transpose of A^-1 with log|det A| and its phase, the work of
// DiracMatrix::invert_transpose (DiracMatrix.h:93-121: transpose, getrf, log det
// from the pivots, getri).  Here: an in-place blocked Gauss-Jordan inversion of X = A^T in
// FP64 with partial pivoting on X's rows.  Its pivots are the U diagonal of LU with partial
// pivoting, so log|det| and the sign come out the same way.  One workgroup per matrix.
//
// X is kept transposed, Y[c][i] = X[i][c], so the first pass reads A as it is (and converts it)
// and a panel of X's columns is a set of Y's rows.  No rows are exchanged: row i of X that was the
// pivot of step k stays in place (kof[i] = k, piv[k] = i), and the permutations are applied as
// psiM is written:  psiM[k][j] = Y[kof[j]][piv[k]].
//
// A panel is B columns of X: thread i holds row i's B entries in registers for the panel's
// elimination steps.  The other columns of X then get the panel's rank-B update, P[c][i] the
// finished panel in LDS,
//   Y[c][i] <- (i a pivot row of the panel ? 0 : Y[c][i]) + sum_t Y[c][p_t] P[t][i]
// on the FP64 matrix cores (v_mfma_f64_16x16x4f64).  A wave owns a 16-column tile of X from its
// pivot-row entries to its last row, so the update needs no barriers, and it loads row tiles ahead
// of the one it multiplies.
//
// Bound: latency of the pivot steps (about 1 us each: two barriers, the pivot search, one division)
// and of a wave's tile; with as many matrices as CUs at n = 384 the passes over X, whose working
// set (302 MB) exceeds the last-level cache.  n = 384: one matrix 1.19 ms, 128 at once 1.40, 256 at
// once 2.1 (the form that exchanged rows and streamed X in 64-column chunks through LDS between
// barriers: 2.32, 2.51 and 2.97); n = 192, 256 at once: 0.41 (0.66) ms.  Sub-panels of 16 columns
// with a rank-16 update between them take 1.10, 1.30 and 2.0 ms but round differently: an element of
// the FP32 inverse may then differ by one ulp, which a chain of FP32 moves without a refresh amplifies
// to 1e-3 in an ill-conditioned walker.
constexpr int kGJAhead = 4;    // row tiles in flight per wave (even)
// LDS row stride of the panel (doubles): an odd multiple of 16, so that the four 16-lane groups of
// a matrix operand read different banks
__host__ __device__ inline int gj_stride(int n) { return 16 * (((n + 15) / 16) | 1); }
struct GJLds {
  size_t oP, oPr, oDv, oRed, oRi, oPiv, oKof, total;
};
__host__ __device__ inline GJLds gj_lds_b(int n, int b) {
  GJLds L;
  size_t o = 0;
  auto take = [&](size_t bytes) { const size_t at = o; o += (bytes + 15) & ~(size_t)15; return at; };
  L.oP = take(sizeof(double) * (size_t)b * (gj_stride(n) + 1));   // the panel; on the way out rows of stride + 1
  L.oPr = take(sizeof(double) * 2 * (size_t)(b + 2));            // scaled pivot row of a step and 1 / pivot (two in turn)
  L.oDv = take(sizeof(double) * (size_t)n);                      // the pivots
  L.oRed = take(sizeof(double) * 2 * 16);                        // per wave: best pivot candidate (two in turn)
  L.oRi = take(sizeof(int) * 2 * 16);                            // and its row
  L.oPiv = take(sizeof(int) * (size_t)gj_stride(n));             // row of each step's pivot
  L.oKof = take(sizeof(int) * (size_t)gj_stride(n));             // step in which each row was the pivot
  L.total = o;
  return L;
}
// panel width: a thread per row (512 threads for 32 columns, 1024 for 16), the panel within the LDS
__host__ __device__ inline int gj_panel(int n) { return n <= 512 ? 32 : 16; }
__host__ __device__ inline GJLds gj_lds(int n) { return gj_lds_b(n, gj_panel(n)); }

// the rank-B update of the columns outside the panel [k0, k0 + bb); TS: TI for the first panel
// (src = the input matrix), double after
template <typename TS, int B>
__device__ __forceinline__ void gj_update(int n, int ns, int k0, int bb, const TS* src, double* Y, const double* P,
                                          const int* piv, const int* kof) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int lj = lane & 15, lg = lane >> 4;
  const int nt = (n + 15) >> 4, ptile = k0 >> 4, np = (bb + 15) >> 4;   // tiles; the panel's tiles
  const bool whole = (n & 15) == 0;
  for (int idx = wid; idx < nt - np; idx += nw) {
    const int ct = idx < ptile ? idx : idx + np;
    // A operand, lane (j, g): column 16 ct + j of pivot row p_t, t = 4 s + g
    double a[B / 4];
    const TS* ac = src + (size_t)min(16 * ct + lj, n - 1) * n;
#pragma unroll
    for (int s = 0; s < B / 4; ++s) {
      const int t = 4 * s + lg;
      const double v = (double)ac[piv[k0 + min(t, bb - 1)]];
      a[s] = t < bb ? v : 0.0;
    }
    // C/D register r of lane (j, g): column 16 ct + g + 4 r, row 16 it + j
    const int c0 = 16 * ct + lg;
    const TS* xr[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) xr[r] = src + (size_t)min(c0 + 4 * r, n - 1) * n;
    // X entries of the next kGJAhead row tiles and the B operand (and pivot steps) of the next one
    // are on their way while a tile is multiplied
    TS x[kGJAhead][4];
    double b[2][B / 4];
    int kk[2];
    auto load = [&](int it, TS (&v)[4]) {
      const int i = min(16 * it + lj, n - 1);
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = xr[r][i];
    };
    auto operand = [&](int it, double (&v)[B / 4], int& k) {
      const int i = min(16 * it + lj, ns - 1);
#pragma unroll
      for (int s = 0; s < B / 4; ++s) v[s] = P[(size_t)(4 * s + lg) * ns + i];
      k = kof[i];
    };
#pragma unroll
    for (int q = 0; q < kGJAhead; ++q) load(q, x[q]);
    operand(0, b[0], kk[0]);
    for (int it0 = 0; it0 < nt; it0 += kGJAhead) {
#pragma unroll
      for (int q = 0; q < kGJAhead; ++q) {
        const int it = it0 + q;
        if (it < nt) {
          f64x4 acc;
          const bool pivot = (unsigned)(kk[q & 1] - k0) < (unsigned)bb;
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[r] = pivot ? 0.0 : (double)x[q][r];
          load(it + kGJAhead, x[q]);
          operand(it + 1, b[(q + 1) & 1], kk[(q + 1) & 1]);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int s = 0; s < B / 4; ++s) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], b[q & 1][s], acc, 0, 0, 0);
          const int i = 16 * it + lj;
          double* yr = Y + (size_t)c0 * n + i;
          if (whole) {
#pragma unroll
            for (int r = 0; r < 4; ++r) yr[(size_t)(4 * r) * n] = acc[r];
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (i < n && c0 + 4 * r < n) yr[(size_t)(4 * r) * n] = acc[r];
          }
        }
      }
    }
  }
}

template <typename TI, typename TO, int B, int NT>
__global__ __launch_bounds__(NT) void k_gj_invert(int n, const TI* A, TO* psiM, double* ws, double* logdet,
                                                          double* phase, int ld_stride, int mat_stride, const int* only) {
  const int mat = blockIdx.x, tid = threadIdx.x;
  if (only != nullptr && only[mat] == 0) return;   // only the matrices whose flag is set
  constexpr int nw = NT / 64;
  const int lane = tid & 63, wid = tid >> 6;
  const int ns = gj_stride(n);
  const GJLds L = gj_lds_b(n, B);
  extern __shared__ __align__(16) unsigned char smem[];
  double* P = (double*)(smem + L.oP);
  double* prow = (double*)(smem + L.oPr);
  double* dv = (double*)(smem + L.oDv);
  double* rv = (double*)(smem + L.oRed);
  int* ri = (int*)(smem + L.oRi);
  int* piv = (int*)(smem + L.oPiv);
  int* kof = (int*)(smem + L.oKof);
  const size_t mo = (size_t)mat * mat_stride;   // matrix slot (every mat_stride-th matrix)
  double* Y = ws + mo * 2 * n * n;
  const TI* a = A + mo * n * n;
  const bool own = tid < n;
  bool used = false;   // this thread's row has been a pivot
  unsigned par = 0;    // parity of the wave's unused rows below each pivot (the permutation's inversions)
  for (int i = tid; i < ns; i += NT) {
    piv[i] = min(i, n - 1);
    kof[i] = INT_MAX;
  }
  __syncthreads();

  for (int k0 = 0; k0 < n; k0 += B) {
    const int bb = min(B, n - k0);
    // ---- the panel's columns (zeros past bb) and its elimination steps
    double pr[B];
#pragma unroll
    for (int c = 0; c < B; ++c) {
      const size_t at = (size_t)(k0 + min(c, bb - 1)) * n + (own ? tid : 0);
      pr[c] = k0 == 0 ? (double)a[at] : Y[at];
    }
#pragma unroll
    for (int c = 0; c < B; ++c) pr[c] = (own && c < bb) ? pr[c] : 0.0;
#pragma unroll
    for (int j = 0; j < B; ++j) {
      if (j < bb) {
        const int k = k0 + j;
        double* pw = prow + (B + 2) * (j & 1);
        double* rw = rv + 16 * (j & 1);
        int* iw = ri + 16 * (j & 1);
        const double prj = pr[j];
        // pivot: the largest |P[j][i]| of the rows not used yet, the lowest of them: the wave's
        // largest magnitude and its first lane, then the waves' candidates side by side in the
        // lanes of every wave.  Candidates and pivot rows alternate between two slots, so a step
        // needs no barrier between its reads and the next step's writes
        // (a NaN, which a maximum never takes, is the pivot once no other row is left)
        const double av = (own && !used) ? fmax(fabs(prj), -0.5) : -1.0;
        const double best = wave_max(av);
        const unsigned long long hit = __ballot(av == best);
        if (lane == 0) {
          rw[wid] = best;
          iw[wid] = min(wid * 64 + max(__ffsll((long long)hit) - 1, 0), n - 1);
        }
        lds_sync();
        const double cv = rw[lane & (nw - 1)];
        const int cr = iw[lane & (nw - 1)];
        double cb = cv;
        cb = dpp_max<0xB1, 0xf>(cb);
        cb = dpp_max<0x4E, 0xf>(cb);
        cb = dpp_max<0x141, 0xf>(cb);   // of eight lanes
        if constexpr (nw > 8) cb = dpp_max<0x140, 0xf>(cb);
        const int qb = max(__ffsll((long long)__ballot(cv == cb)) - 1, 0);
        const int p = __builtin_amdgcn_readlane(cr, qb);   // in [0, n)
        const bool isp = tid == p;
        par ^= (unsigned)__popcll(__ballot(own && !used && tid < p)) & 1u;
        const double rinv = 1.0 / cb;   // 1 / |pivot|
        if (isp) {
          // the scaled pivot row for the others; its own new entries are left to the update below
          double dinv = prj < 0.0 ? -rinv : rinv;
          if (prj != prj) dinv = prj;
#pragma unroll
          for (int c = 0; c < B; ++c) {
            pw[c] = pr[c] * dinv;
            pr[c] = 0.0;
          }
          pw[B] = dinv;
          dv[k] = prj;
          piv[k] = p;
          kof[p] = k;
          used = true;
        }
        lds_sync();
        // the pivot row becomes the scaled row (its entry in the pivot column 1 / d), every other
        // row loses its multiple of it (its entry there -f / d)
        const double f = isp ? -1.0 : prj;
#pragma unroll
        for (int c = 0; c < B; ++c)
          if (c != j) pr[c] -= f * pw[c];
        pr[j] = -f * pw[B];
      }
    }
    if (own) {
#pragma unroll
      for (int c = 0; c < B; ++c) P[(size_t)c * ns + tid] = pr[c];
      // zeros past bb (a zero pivot's scaled row is NaN there): the update multiplies all B columns
      for (int c = bb; c < B; ++c) P[(size_t)c * ns + tid] = 0.0;
    }
    __syncthreads();
    // ---- the other columns, then the panel itself, back to Y
    if (k0 == 0)
      gj_update<TI, B>(n, ns, k0, bb, a, Y, P, piv, kof);
    else
      gj_update<double, B>(n, ns, k0, bb, Y, Y, P, piv, kof);
    if (own)
      for (int c = 0; c < bb; ++c) Y[(size_t)(k0 + c) * n + tid] = P[(size_t)c * ns + tid];
    __syncthreads();
  }

  // ---- from the first NaN pivot on every entry is NaN and the rows left were taken in ascending order;
  // the sign is that of row exchanges: place k's row is the pivot.  Place k held row k first, and a step
  // t that took the row of place k put that of its own place t there
  const int knan = n - __syncthreads_count(own && dv[tid] != dv[tid]);
  if (knan < n) {
    used = own && kof[tid] < knan;
    if (own && !used) kof[tid] = INT_MAX;
    __syncthreads();
    for (int k = knan; k < n; ++k) {
      int p = k;
      for (int t = kof[p]; t < k; t = kof[p]) p = t;
      par ^= (unsigned)__popcll(__ballot(own && !used && tid < p)) & 1u;
      __syncthreads();
      if (tid == p) {
        kof[p] = k;
        used = true;
      }
      __syncthreads();
    }
  }
  // ---- log|det| and phase: the product of the pivots as mantissa and binary exponent, the parity
  // of the row permutation and of the negative pivots
  {
    double m = 1.0;
    int ex = 0;
    unsigned neg = lane == 0 ? par : 0u;
    for (int k = tid; k < n; k += NT) {
      int e;
      const double d = dv[k];
      m = frexp(m * fabs(d), &e);
      ex += e;
      neg ^= d < 0.0 ? 1u : 0u;
    }
#pragma unroll
    for (int q = 1; q < 64; q <<= 1) {
      int e;
      m = frexp(m * __shfl_xor(m, q), &e);
      ex += __shfl_xor(ex, q) + e;
      neg ^= __shfl_xor((int)neg, q);
    }
    if (lane == 0) {
      rv[wid] = m;
      ri[wid] = ex;
      ri[16 + wid] = (int)neg;
    }
    __syncthreads();
    if (tid == 0) {
      for (int q = 1; q < nw; ++q) {
        int e;
        m = frexp(m * rv[q], &e);
        ex += ri[q] + e;
        neg ^= (unsigned)ri[16 + q];
      }
      logdet[(size_t)mat * ld_stride] = log(m) + (double)ex * 0.69314718055994530942;
      phase[(size_t)mat * ld_stride] = neg ? M_PI : 0.0;
    }
  }
  // ---- psiM[k][j] = Y[kof[j]][piv[k]], B columns j at a time through LDS (row stride ns + 1, so
  // the lanes' rows fall in different banks)
  TO* out = psiM + mo * n * n;
  for (int j0 = 0; j0 < n; j0 += B) {
    const int jb = min(B, n - j0);
    {
      double v[B];
#pragma unroll
      for (int c = 0; c < B; ++c) {
        const int l = min((unsigned)kof[j0 + min(c, jb - 1)], (unsigned)(n - 1));
        v[c] = Y[(size_t)l * n + (own ? tid : 0)];
      }
      if (own)
#pragma unroll
        for (int c = 0; c < B; ++c) P[(size_t)c * (ns + 1) + tid] = v[c];
    }
    __syncthreads();
    for (int e = tid; e < n * B; e += NT) {
      const int k = e / B, c = e % B;
      if (c < jb) out[(size_t)k * n + j0 + c] = (TO)P[(size_t)c * (ns + 1) + piv[k]];
    }
    __syncthreads();
  }
}

// host side: the panel width is a template argument (the panel row lives in registers)
// nmat matrices at A, A + mat_stride n^2, ...; log|det| and phase of matrix m at [m * ld_stride]
template <typename TI, typename TO>
inline hipError_t launch_gj_invert(int n, int nmat, hipStream_t st, const TI* A, TO* psiM, double* ws,
                                   double* logdet, double* phase, int ld_stride, int mat_stride = 1,
                                   const int* only = nullptr) {
  // a thread per row: 512 threads with panels of 32 columns, 1024 with 16 past n = 512
  const size_t lds = gj_lds(n).total;
  if (gj_panel(n) == 32)
    hipLaunchKernelGGL((k_gj_invert<TI, TO, 32, 512>), dim3(nmat), dim3(512), lds, st, n, A, psiM, ws, logdet, phase,
                       ld_stride, mat_stride, only);
  else
    hipLaunchKernelGGL((k_gj_invert<TI, TO, 16, 1024>), dim3(nmat), dim3(1024), lds, st, n, A, psiM, ws, logdet,
                       phase, ld_stride, mat_stride, only);
  return hipGetLastError();
}

// ------------------------------------------------------------------ SPO rows (evaluateLog)
// Blocks of 2^shift grid cells per axis, nb blocks per axis: the key of a point is its block's index
struct GridBlocks {
  int shift, nb[3];
  __host__ __device__ int keys() const { return nb[0] * nb[1] * nb[2]; }
};
template <typename T>
__device__ inline int block_key(const SysP<T>& S, const GridBlocks& nb, double x, double y, double z) {
  int ix[3];
  double t[3];
  spline_locate(S.spoG, S.ng, x, y, z, ix, t);
  return ((ix[0] >> nb.shift) * nb.nb[1] + (ix[1] >> nb.shift)) * nb.nb[2] + (ix[2] >> nb.shift);
}
// keys of the electrons' positions (point w*N + e) and the per-key counts
template <typename T>
__global__ __launch_bounds__(256) void k_electron_keys(SysP<T> S, BatchP<T> B, GridBlocks nb, int* key, int* kcnt) {
  const int N = S.N, np = B.W * N;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < np; i = walk_next(i, gridDim.x * blockDim.x, np)) {
    const int w = i / N, e = i - w * N;
    const double* R = B.R + (size_t)w * 3 * N;
    const int k = block_key(S, nb, R[e], R[N + e], R[2 * N + e]);
    key[i] = k;
    atomicAdd(kcnt + k, 1);
  }
}

// SPO at every electron of every walker -> A, dpsiM, d2psiM
// (evaluate_notranspose, SPOSet.h:94; DiracDeterminant.cpp:264-280).
template <typename T>
__global__ __launch_bounds__(1024) void k_spo_rows(SysP<T> S, BatchP<T> B, int slices) {
  extern __shared__ __align__(16) unsigned char smem[];
  T* part = (T*)smem;
  T* out = part + (size_t)slices * 5 * S.npad;  // [5][n]
  double* part64 = (double*)(smem + (((sizeof(T) * ((size_t)slices * 5 * S.npad + 5 * (size_t)S.n)) + 15) & ~(size_t)15));
  const int e = blockIdx.x, w = blockIdx.y, N = S.N, n = S.n;
  const double* R = B.R + (size_t)w * 3 * N;
  const int det = e < n ? 0 : 1, row = e - det * n;
  const size_t moff = ((size_t)w * 2 + det) * n * n;
  if (B.A64 != nullptr) {
    spline_gather_rt<T, 5, true>(S, R[e], R[N + e], R[2 * N + e], slices, part, part64);
    __syncthreads();
    spline_finish64<T>(S, slices, part64, B.A64 + moff + (size_t)row * n, n);
  } else {
    spline_gather_rt<T, 5>(S, R[e], R[N + e], R[2 * N + e], slices, part);
    __syncthreads();
  }
  spline_finish<T, 5, T>(S, slices, part, out, n, n);
  __syncthreads();
  T* Arow = B.A + moff + (size_t)row * n;
  T* dp = B.dpsiM + ((size_t)w * 2 + det) * (size_t)n * 3 * n + (size_t)row * 3 * n;
  T* d2 = B.d2psiM + moff + (size_t)row * n;
  for (int j = threadIdx.x; j < n; j += blockDim.x) {
    Arow[j] = out[j];
    dp[j] = out[n + j];
    dp[n + j] = out[2 * n + j];
    dp[2 * n + j] = out[3 * n + j];
    d2[j] = out[4 * n + j];
  }
}

// The same for many electrons, which come ordered by the block of grid cells they are in, each XCD
// (workgroup b runs on XCD b % 8) over a contiguous eighth of them, so that electrons whose
// stencils overlap share an L2.  A workgroup takes an electron, a lane an orbital quad with all 64
// stencil points, stored from registers; the sums go slice by slice (16 / PER slices of PER columns
// each) in the order k_spo_rows adds them, so the rows are the same bit for bit.
// Bound: L2 bandwidth of the stencils.  NiO-64 FP32, 98k electrons: 0.95 ms; unordered, from HBM with
// eight slices reduced through LDS, 2.40 ms (4.0 TB/s); ordered in that form still 2.39.  The slice loop
// is kept rolled: unrolled it spills and takes 2.0 ms.
constexpr int kOrderedThreads = 256;
template <typename T, int PER>
__global__ __launch_bounds__(kOrderedThreads) void k_spo_rows_ordered(SysP<T> S, BatchP<T> B, const int* order) {
  using VT = typename V16<T>::type;
  constexpr int VW = V16<T>::n, SL = 16 / PER;
  const int N = S.N, n = S.n, nq = S.npad / VW;
  const int np = B.W * N, x = blockIdx.x & 7, lo = (int)((long long)np * x / 8), hi = (int)((long long)np * (x + 1) / 8);
  const int k = lo + (int)(blockIdx.x >> 3), qd = threadIdx.x;
  if (k >= hi || qd >= nq) return;   // the grid is rounded up per XCD
  const int at = order[k], w = at / N, e = at - w * N;
  const double* R = B.R + (size_t)w * 3 * N;
  const int det = e < n ? 0 : 1, row = e - det * n;
  const size_t moff = ((size_t)w * 2 + det) * n * n;
  const double px = R[e], py = R[N + e], pz = R[2 * N + e];
  T sum[5][VW], acc[5][VW];
  double acc64[VW];   // not used
#pragma unroll
  for (int v = 0; v < VW; ++v) {
#pragma unroll
    for (int o = 0; o < 5; ++o) sum[o][v] = T(0);
  }
#pragma unroll 1
  for (int sl = 0; sl < SL; ++sl) {
    int q, s;
    spline_gather_regs<T, 5, PER, false, false, true>(S, S.spoG, px, py, pz, qd + sl * nq, acc, acc64, q, s);
#pragma unroll
    for (int v = 0; v < VW; ++v) {
#pragma unroll
      for (int o = 0; o < 5; ++o) sum[o][v] += acc[o][v];
    }
  }
  const T gx = (T)S.ng[0], gy = (T)S.ng[1], gz = (T)S.ng[2];
  T* Arow = B.A + moff + (size_t)row * n;
  T* dp = B.dpsiM + ((size_t)w * 2 + det) * (size_t)n * 3 * n + (size_t)row * 3 * n;
  T* d2 = B.d2psiM + moff + (size_t)row * n;
  T* dst[5] = {Arow, dp, dp + n, dp + 2 * n, d2};
  const int j = qd * VW;
#pragma unroll
  for (int o = 0; o < 5; ++o) {
    const T f = vgh_scale<T>(o, gx, gy, gz);
    if (n % VW == 0) {
      VT v;
#pragma unroll
      for (int c = 0; c < VW; ++c) v[c] = sum[o][c] * f;
      if (j < n) *reinterpret_cast<VT*>(dst[o] + j) = v;
    } else {
#pragma unroll
      for (int c = 0; c < VW; ++c)
        if (j + c < n) dst[o][j + c] = sum[o][c] * f;
    }
  }
}

// SPO values (v, d/dx, d/dy, d/dz, d2/dx2; einspline_spo.hpp:204-223) at the proposals of
// electrons det*n + [e0, e0 + gridDim.x) of every walker, into spo[w][det][e][5][npad].  Within
// a sweep an electron's position changes only at its own move, so the sweep's proposals
// r_e + displacement are fixed before the first of them is accepted; evaluating them here takes
// the spline's HBM traffic out of the move kernel's accept chain.  The displacement is the
// move kernel's: sqrt(tau) times the walker's Philox normals of (sweep, electron), or the
// caller's (displ[w][3]).
// the gather of one point with the slice count fixed at compile time (SLC > 0) or chosen at run
// time (SLC == 0): a kernel that carries one variant allocates registers for that one alone
template <typename T, int NO, int SLC, bool V64 = false>
__device__ inline void spline_gather_sl(const SysP<T>& S, double x, double y, double z, int slices, T* part,
                                        double* part64 = nullptr) {
  if constexpr (SLC == 0)
    spline_gather_rt<T, NO, V64>(S, x, y, z, slices, part, part64);
  else
    spline_gather<T, NO, 16 / SLC, V64>(S, S.spoG, x, y, z, part, threadIdx.x, part64);
}

// SLC: slices fixed at compile time (0: the run-time argument); V64: the FP32 form's FP64 value
// rows are written as well (only while the batch keeps them, B.spo64 != nullptr)
template <typename T, int SLC, bool V64>
__device__ __forceinline__ void spo_proposals_body(const SysP<T>& S, const BatchP<T>& B, int det, int e0, int ne,
                                                   uint64_t seed, const int* sweep_ctr, double sqrt_tau, int walker0,
                                                   const double* displ, T* spo, double* prop, int slices, const int w) {
  extern __shared__ __align__(16) unsigned char smem[];
  T* part = (T*)smem;
  const int N = S.N, n = S.n;
  const int sweep = displ != nullptr ? 0 : sweep_ctr[2];   // the random streams' sweep counter
  // a workgroup takes electrons e0 + blockIdx.x, + gridDim.x, ... (fewer workgroups than
  // electrons bound the gather's share of HBM beside the move kernel)
  for (int el = e0 + blockIdx.x; el < e0 + ne; el += gridDim.x) {
  const int iel = det * n + el;
  const double* R = B.R + (size_t)w * 3 * N;
  double d[3], u = 0.0;   // a caller's displacement comes with its own accept decision
  if (displ != nullptr) {
    d[0] = displ[3 * w + 0];
    d[1] = displ[3 * w + 1];
    d[2] = displ[3 * w + 2];
  } else {
    double nr[3];
    move_randoms(seed, (uint64_t)(walker0 + w), (uint64_t)sweep, (uint64_t)iel, nr, u);
    d[0] = sqrt_tau * nr[0];
    d[1] = sqrt_tau * nr[1];
    d[2] = sqrt_tau * nr[2];
  }
  const double x = R[iel] + d[0], y = R[N + iel] + d[1], z = R[2 * N + iel] + d[2];
  if constexpr (SLC == 1) {
  } else if constexpr (V64) {
    double* part64 = (double*)(smem + ((sizeof(T) * (size_t)slices * 5 * S.npad + 15) & ~(size_t)15));
    spline_gather_sl<T, 5, SLC, true>(S, x, y, z, slices, part, part64);
    __syncthreads();
    spline_finish64<T>(S, slices, part64, B.spo64 + (((size_t)w * 2 + det) * n + el) * S.npad, n);
  } else {
    spline_gather_sl<T, 5, SLC>(S, x, y, z, slices, part);
    __syncthreads();
  }
  T* out = spo + (((size_t)w * 2 + det) * n + el) * 5 * S.npad;
  if constexpr (SLC == 1) {
    spline_gather_direct<T, 5, V64>(S, x, y, z, out,
                                    V64 ? B.spo64 + (((size_t)w * 2 + det) * n + el) * S.npad : nullptr);
  } else {
    spline_finish<T, 5, T>(S, slices, part, out, S.npad, n);
    __syncthreads();
  }
  // J1 at the proposal (OneBodyJastrow::ratioGrad, OneBodyJastrow.h:259-268): it depends on the
  // proposal and the ions only, so it is evaluated here with the SPO row
  const Cell<T> C = *S.cell;
  double acc[5] = {0, 0, 0, 0, 0};
  for (int ci = threadIdx.x; ci < S.M; ci += blockDim.x) {
    const Functor<T>& f = S.fn[S.species[ci]];
    if (f.ncoef > 0) {
      T dx, dy, dz;
      const T r = min_image(C, (T)(S.ions[ci] - x), (T)(S.ions[S.M + ci] - y), (T)(S.ions[2 * S.M + ci] - z), T(-1),
                            dx, dy, dz);
      if (r < f.rcut) {
        T u, du, d2u;
        functor_vgl(f, r, u, du, d2u);
        acc[0] += (double)u;
        acc[1] += (double)(d2u + T(2) * du);
        acc[2] += (double)(du * dx);
        acc[3] += (double)(du * dy);
        acc[4] += (double)(du * dz);
      }
    }
  }
  double* red = (double*)smem;   // [waves][5]
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
#pragma unroll
  for (int k = 0; k < 5; ++k) acc[k] = wave_sum(acc[k]);
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < 5; ++k) red[wid * 5 + k] = acc[k];
  __syncthreads();
  if (threadIdx.x < 5) {
    double t = 0;
    for (int q = 0; q < nw; ++q) t += red[q * 5 + threadIdx.x];
    prop[(((size_t)w * 2 + det) * n + el) * kProp + kPropJ1 + threadIdx.x] = t;
  } else if (threadIdx.x < 9) {
    const int k = threadIdx.x - 5;
    prop[(((size_t)w * 2 + det) * n + el) * kProp + kPropDispl + k] = k < 3 ? d[k] : u;
  }
  if (S.j3 != nullptr && wid == 0) {
    // the ions within their three-body cutoff of the proposal, in ion order (ballot compaction
    // over 64 ions at a time): count, then (ion, r, ion - proposal)
    T* rec = B.j3prop + (((size_t)w * 2 + det) * n + el) * kJ3Rec;
    int cnt = 0;
    for (int c0 = 0; c0 < S.M; c0 += 64) {
      const int ci = c0 + lane;
      bool in = false;
      T r = 0, dx = 0, dy = 0, dz = 0;
      if (ci < S.M) {
        r = min_image(C, (T)(S.ions[ci] - x), (T)(S.ions[S.M + ci] - y), (T)(S.ions[2 * S.M + ci] - z), T(-1), dx,
                      dy, dz);
        in = r < S.j3[2 * S.species[ci]].L;
      }
      const unsigned long long bal = __ballot(in);
      const int pos = cnt + __popcll(bal & ((1ull << lane) - 1ull));
      if (in && pos < kJ3Near) {
        T* e = rec + 1 + 5 * pos;
        e[0] = (T)ci;
        e[1] = r;
        e[2] = dx;
        e[3] = dy;
        e[4] = dz;
      }
      cnt += __popcll(bal);
    }
    if (lane == 0) {
      rec[0] = (T)cnt;
      if (cnt > kJ3Near) atomicOr(B.flags, kFlagJ3Near);
    }
  }
  __syncthreads();   // the next electron's gather reuses the LDS
  }
}

template <typename T, int SLC, bool V64>
__global__ __launch_bounds__(1024) void k_spo_proposals(SysP<T> S, BatchP<T> B, int det, int e0, int ne, uint64_t seed,
                                                         const int* sweep_ctr, double sqrt_tau, int walker0,
                                                         const double* displ, T* spo, double* prop, int slices) {
  spo_proposals_body<T, SLC, V64>(S, B, det, e0, ne, seed, sweep_ctr, sqrt_tau, walker0, displ, spo, prop, slices,
                                  blockIdx.y);
}

// The proposals of one determinant of every walker of several batches in one launch: batch g owns
// the grid rows [first[g], first[g+1]); the workgroup size and LDS are the largest any batch needs.
constexpr int kMaxPropGroups = 4;
template <typename T>
struct PropGroup {
  int ng;
  int first[kMaxPropGroups + 1];
  SysP<T> S[kMaxPropGroups];
  BatchP<T> B[kMaxPropGroups];
  T* spo[kMaxPropGroups];
  double* prop[kMaxPropGroups];
  int walker0[kMaxPropGroups], slices[kMaxPropGroups];
};

template <typename T, bool V64>
__global__ __launch_bounds__(1024) void k_spo_proposals_group(PropGroup<T> G, int det, uint64_t seed, double sqrt_tau) {
  int g = 0;
  while (g + 1 < G.ng && (int)blockIdx.y >= G.first[g + 1]) ++g;
  spo_proposals_body<T, 0, V64>(G.S[g], G.B[g], det, 0, G.S[g].n, seed, G.B[g].sweep, sqrt_tau, G.walker0[g],
                                nullptr, G.spo[g], G.prop[g], G.slices[g], (int)blockIdx.y - G.first[g]);
}

// stand-alone VGH at arbitrary points: out[p][10][norb] (FP64)
template <typename T>
__global__ __launch_bounds__(1024) void k_spline_vgh(SysP<T> S, const double* r, double* out, int norb, int slices) {
  extern __shared__ __align__(16) unsigned char smem[];
  T* part = (T*)smem;
  const int p = blockIdx.x;
  spline_gather_rt<T, 10>(S, r[3 * p], r[3 * p + 1], r[3 * p + 2], slices, part);
  __syncthreads();
  spline_finish<T, 10, double>(S, slices, part, out + (size_t)p * 10 * norb, norb, norb);
}

// ------------------------------------------------------------------ virtual-move ratios
// WaveFunction::evaluateRatios (WaveFunction.cpp:281-297) for electron iel of every walker at
// nvp virtual positions vpos[w][k][3], ratios[w][k]:
//   determinant: value-only SPO row at the point dotted with the electron's inverse row
//     (DiracDeterminant::evaluateRatios, DiracDeterminant.cpp:216-224; SPOSet::evaluateDetRatios,
//     SPOSet.h:72-83; MultiBspline::evaluate_v, MultiBspline.hpp:34-63);
//   J1: exp(Vat[iel] - sum over ions of u(|ion - point|))   (OneBodyJastrow.h:136-140);
//   J2: exp(Uat[iel] - sum over j != iel of u(|r_j - point|)) (TwoBodyJastrow.h:103-107);
//   J3 (with a three-body Jastrow): exp(U3[iel] - U3 at the point)   (ThreeBodyJastrow.h:262-273).
// One workgroup per (point, walker).  The inverse must carry no pending delayed rows, which
// holds between the batch's calls.
// Three-body Jastrow sum U of electron e of walker w placed at (x, y, z), the others at their
// current positions (ThreeBodyJastrow::evaluateRatios' computeU, ThreeBodyJastrow.h:262-273):
// over ions I with the point within L_I and electrons k != e within L_I of I (the batch's ion
// masks of the current positions), F(r_xk, r_xI, r_kI) with the functor of I's species and the
// (e, k) spin pair.  The lanes [tid, tid + nt, ...) take the electrons k; returns this lane's part.
template <typename T>
__device__ inline double j3_value_partial(const SysP<T>& S, const BatchP<T>& B, const Cell<T>& C, int w, int e,
                                          double x, double y, double z, int tid, int nt) {
  const int N = S.N, n = S.n, M = S.M, mw = S.mw;
  const double* R = B.R + (size_t)w * 3 * N;
  const unsigned long long* mk = B.j3mask + (size_t)w * N * mw;
  const bool up = e < n;
  double acc = 0.0;
  for (int I = 0; I < M; ++I) {
    const int sp = S.species[I];
    const T L = S.j3[2 * sp].L;
    if (!(L > T(0))) continue;   // the species has no three-body functor
    const double ix = S.ions[I], iy = S.ions[M + I], iz = S.ions[2 * M + I];
    T dx, dy, dz;
    const T rxI = min_image(C, (T)(ix - x), (T)(iy - y), (T)(iz - z), T(-1), dx, dy, dz);
    if (!(rxI < L)) continue;
    const unsigned long long bit = 1ull << (I & 63);
    const int wd = I >> 6;
    for (int k = tid; k < N; k += nt) {
      if (k == e || !(mk[(size_t)k * mw + wd] & bit)) continue;
      const double kx = R[k], ky = R[N + k], kz = R[2 * N + k];
      const T rkI = min_image(C, (T)(ix - kx), (T)(iy - ky), (T)(iz - kz), T(-1), dx, dy, dz);
      const T rxk = min_image(C, (T)(kx - x), (T)(ky - y), (T)(kz - z), T(-1), dx, dy, dz);
      acc += (double)poly3_v(S.j3[2 * sp + (((k < n) == up) ? 0 : 1)], rxk, rxI, rkI);
    }
  }
  return acc;
}

// Ratio at one point for walker w, electron iel; the workgroup's lanes share the work and
// every lane returns the ratio.  part: LDS [slices][npad] T; red: LDS 48 doubles.
template <typename T>
__device__ inline double virtual_ratio(const SysP<T>& S, const BatchP<T>& B, const Cell<T>& C, int w, int iel,
                                       double x, double y, double z, int slices, T* part, double* red) {
  const int N = S.N, n = S.n, M = S.M;
  spline_gather_rt<T, 1>(S, x, y, z, slices, part);
  __syncthreads();
  const int det = iel < n ? 0 : 1, row = iel - det * n;
  const T* arow = B.Ainv + ((size_t)w * 2 + det) * n * n + (size_t)row * n;
  double v[3] = {0.0, 0.0, 0.0};   // det ratio, J1 sum, J2 and J3 sum (both enter the exponent alike)
  for (int j = threadIdx.x; j < n; j += blockDim.x) {
    T s = 0;
    for (int sl = 0; sl < slices; ++sl) s += part[(size_t)sl * S.npad + j];
    v[0] += (double)s * (double)arow[j];
  }
  T dx, dy, dz;   // values only
  for (int ci = threadIdx.x; ci < M; ci += blockDim.x) {
    const Functor<T>& f = S.fn[S.species[ci]];
    if (f.ncoef == 0) continue;
    const T r = min_image(C, (T)(S.ions[ci] - x), (T)(S.ions[M + ci] - y), (T)(S.ions[2 * M + ci] - z), T(-1), dx,
                          dy, dz);
    if (r < f.rcut) v[1] += (double)functor_v(f, r);
  }
  const double* R = B.R + (size_t)w * 3 * N;
  const bool up = iel < n;
  for (int j = threadIdx.x; j < N; j += blockDim.x) {
    if (j == iel) continue;
    const Functor<T>& f = S.fn[kMaxSpecies + (((j < n) == up) ? 0 : 1)];
    const T r = min_image(C, (T)(R[j] - x), (T)(R[N + j] - y), (T)(R[2 * N + j] - z), T(-1), dx, dy, dz);
    if (r < f.rcut) v[2] += (double)functor_v(f, r);
  }
  if (S.j3 != nullptr) v[2] += j3_value_partial<T>(S, B, C, w, iel, x, y, z, threadIdx.x, blockDim.x);
  block_sum<double, 3>(v, red);   // ends with a barrier: part and red are free again
  const size_t o = (size_t)w * 5 * N + iel;
  const double u23 = (double)B.J2[o] + (S.j3 != nullptr ? (double)B.J3[o] : 0.0);
  return v[0] * exp(((double)B.J1[o] - v[1]) + (u23 - v[2]));
}

template <typename T>
__global__ __launch_bounds__(1024) void k_virtual_ratios(SysP<T> S, BatchP<T> B, int iel, int nvp, const double* vpos,
                                                         double* ratios, int slices) {
  extern __shared__ __align__(16) unsigned char smem[];
  T* part = (T*)smem;                                  // [slices][npad]
  double* red = (double*)(part + (size_t)slices * S.npad);
  const int k = blockIdx.x, w = blockIdx.y;
  const double* p = vpos + ((size_t)w * nvp + k) * 3;
  const Cell<T> C = *S.cell;
  const double r = virtual_ratio<T>(S, B, C, w, iel, p[0], p[1], p[2], slices, part, red);
  if (threadIdx.x == 0) ratios[(size_t)w * nvp + k] = r;
}

// NonLocalPP::evaluate (NonLocalPP.hpp:115-140) for every electron of every walker.
// k_nlpp_pairs: one lane per (walker, electron) finds the ions within rmax in ion order (minimum
// image, ion - electron as the BA table's displacement), counts them in npairs[w][e] (the full
// count, also beyond maxp) and lists the first maxp: near[item][4] = distance, displacement of item =
// (w*N + e)*maxp + p, items[pos] = item in the order of arrival (an electron's pairs from first[w][e] on),
// cnt[0] = listed pairs.  Knot k of a pair sits at dist * spheres[w][k] + displ + r_e (NonLocalPP.hpp:133;
// every walker has its own randomly rotated knots, one rotation per walker and evaluation as the reference's
// per-mover NonLocalPP::randomize, NonLocalPP.hpp:100-113, miniqmc.cpp:470).
// k_nlpp_keys, k_key_offsets and k_key_scatter order all the knots (unit = pos * 12 + knot) by the
// block of spline grid cells they fall in (left out when there are few, or the table is small).
// k_nlpp_jastrow: the Jastrow exponents of the listed pairs' knots into ratios[pos][12], walker by walker
// (its positions and the functors in LDS, a wave per pair, lanes over the electrons); the knots' keys,
// which lay there, are done with.
// k_nlpp_ratios walks the ordered knots, each XCD over a
// contiguous eighth of it: knots whose stencils overlap run at the same time on CUs that share an
// L2, so the orbital table is read from HBM about once instead of once per knot.  ratios[pos][12] =
// (value row . inverse row) exp(exponent), in the exponent's place.
constexpr int kNlppKnots = 12;

__global__ void k_zero_ints(int* p, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}

template <typename T>
__global__ __launch_bounds__(256) void k_nlpp_pairs(SysP<T> S, BatchP<T> B, double rmax, int maxp, double* near,
                                                    int* items, int* npairs, int* first, int* cnt) {
  const int at = blockIdx.x * blockDim.x + threadIdx.x, N = S.N;
  const bool live = at < B.W * N;
  const int idx = live ? at : 0, M = live ? S.M : 0;
  const int w = idx / N, e = idx - w * N;
  const Cell<T> C = *S.cell;
  const double* R = B.R + (size_t)w * 3 * N;
  const double x = R[e], y = R[N + e], z = R[2 * N + e];
  int c = 0;
  for (int ci = 0; ci < M; ++ci) {
    T dx, dy, dz;
    const T r = min_image(C, (T)(S.ions[ci] - x), (T)(S.ions[M + ci] - y), (T)(S.ions[2 * M + ci] - z), T(-1), dx, dy,
                          dz);
    if ((double)r < rmax) {
      if (c < maxp) {
        double* q = near + ((size_t)idx * maxp + c) * 4;
        q[0] = (double)r;
        q[1] = (double)dx;
        q[2] = (double)dy;
        q[3] = (double)dz;
      }
      ++c;
    }
  }
  if (live) npairs[idx] = c;
  // the workgroup's pairs take one run of the list
  const int m = live ? min(c, maxp) : 0, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int inc = m;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int t = __shfl_up(inc, d);
    if (lane >= d) inc += t;
  }
  __shared__ int tot[4], base;
  if (lane == 63) tot[wid] = inc;
  __syncthreads();
  if (threadIdx.x == 0) base = atomicAdd(cnt, tot[0] + tot[1] + tot[2] + tot[3]);
  __syncthreads();
  int pos = base + inc - m;
  for (int q = 0; q < wid; ++q) pos += tot[q];
  if (live) first[idx] = pos;
  for (int p = 0; p < m; ++p) items[pos + p] = idx * maxp + p;
}

// the point of unit u (pair u / 12, knot u % 12); w, e: the pair's walker and electron
template <typename T>
__device__ inline void nlpp_point(const SysP<T>& S, const BatchP<T>& B, const double* spheres, int maxp,
                                  const double* near, const int* items, int u, int& w, int& e, double p[3]) {
  const int pos = u / kNlppKnots, k = u - pos * kNlppKnots, N = S.N;
  const int item = items[pos], idx = item / maxp;
  w = idx / N;
  e = idx - w * N;
  const double* R = B.R + (size_t)w * 3 * N;
  const double* sp = spheres + ((size_t)w * kNlppKnots + k) * 3;
  const double* q = near + (size_t)item * 4;
  const double d = q[0];
  const double ox = R[e] + q[1], oy = R[N + e] + q[2], oz = R[2 * N + e] + q[3];
  p[0] = d * sp[0] + ox;
  p[1] = d * sp[1] + oy;
  p[2] = d * sp[2] + oz;
}
template <typename T>
__global__ __launch_bounds__(256) void k_nlpp_keys(SysP<T> S, BatchP<T> B, const double* spheres, int maxp,
                                                   const double* near, const int* items, const int* cnt,
                                                   GridBlocks nb, int* ukey, int* kcnt) {
  const int nu = cnt[0] * kNlppKnots;
  for (int u = blockIdx.x * blockDim.x + threadIdx.x; u < nu; u = walk_next(u, gridDim.x * blockDim.x, nu)) {
    int w, e;
    double p[3];
    nlpp_point(S, B, spheres, maxp, near, items, u, w, e, p);
    const int key = block_key(S, nb, p[0], p[1], p[2]);
    ukey[u] = key;
    atomicAdd(kcnt + key, 1);
  }
}

// Exclusive prefix of the per-key counts into the per-key cursors.  One workgroup of 1024 lanes:
// each lane sums a contiguous run of keys, the run sums are scanned, each lane writes its cursors.
__global__ __launch_bounds__(1024) void k_key_offsets(const int* kcnt, int* kcur, int nkeys) {
  __shared__ int run[16];
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6, per = (nkeys + 1023) / 1024, a = min(t * per, nkeys);
  const int b = min(a + per, nkeys);
  int s = 0;
  for (int c = a; c < b; ++c) s += kcnt[c];
  int x = s;   // inclusive scan of the wave's run sums
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(x, d);
    if (lane >= d) x += y;
  }
  if (lane == 63) run[wid] = x;
  __syncthreads();
  int o = x - s;
  for (int q = 0; q < wid; ++q) o += run[q];
  for (int c = a; c < b; ++c) {
    kcur[c] = o;
    o += kcnt[c];
  }
}

// points u (cnt[0] * per of them) to their places in the order of their keys
__global__ __launch_bounds__(256) void k_key_scatter(const int* cnt, int per, const int* ukey, int* kcur, int* units) {
  const int nu = (cnt != nullptr ? cnt[0] : 1) * per;
  for (int u = blockIdx.x * blockDim.x + threadIdx.x; u < nu; u = walk_next(u, gridDim.x * blockDim.x, nu))
    units[atomicAdd(kcur + ukey[u], 1)] = u;
}

// j3_value_partial of the lanes of one wave, with the walker's positions and the ions in LDS: the lanes look
// for the ions in reach of the point, then sum over the electrons ion by ion, in the same order.  NiO-16, 32
// walkers, FP32: 129 us the whole Jastrow kernel, 277 with every ion looked at by all lanes from memory.
template <typename T>
__device__ inline double j3_value_wave(const SysP<T>& S, const BatchP<T>& B, const Cell<T>& C, int w, int e, double x,
                                       double y, double z, const double* sR, const double* sI, int lane) {
  const int N = S.N, n = S.n, M = S.M, mw = S.mw;
  const unsigned long long* mk = B.j3mask + (size_t)w * N * mw;
  const bool up = e < n;
  T dx, dy, dz;
  double acc = 0.0;
  for (int I0 = 0; I0 < M; I0 += 64) {
    const int Il = min(I0 + lane, M - 1);
    const T Ll = S.j3[2 * S.species[Il]].L;
    const T rl = min_image(C, (T)(sI[Il] - x), (T)(sI[M + Il] - y), (T)(sI[2 * M + Il] - z), T(-1), dx, dy, dz);
    unsigned long long near = __ballot(I0 + lane < M && Ll > T(0) && rl < Ll);
    for (; near != 0; near &= near - 1) {
      const int I = I0 + __ffsll((long long)near) - 1, sp = S.species[I], wd = I >> 6;
      const unsigned long long bit = 1ull << (I & 63);
      const double ix = sI[I], iy = sI[M + I], iz = sI[2 * M + I];
      const T rxI = min_image(C, (T)(ix - x), (T)(iy - y), (T)(iz - z), T(-1), dx, dy, dz);
      for (int k = lane; k < N; k += 64) {
        if (k == e || !(mk[(size_t)k * mw + wd] & bit)) continue;
        const double kx = sR[k], ky = sR[N + k], kz = sR[2 * N + k];
        const T rkI = min_image(C, (T)(ix - kx), (T)(iy - ky), (T)(iz - kz), T(-1), dx, dy, dz);
        const T rxk = min_image(C, (T)(kx - x), (T)(ky - y), (T)(kz - z), T(-1), dx, dy, dz);
        acc += (double)poly3_v(S.j3[2 * sp + (((k < n) == up) ? 0 : 1)], rxk, rxI, rkI);
      }
    }
  }
  return acc;
}

// J1, J2 (and J3) exponents of every listed pair's knots: sums at the electron's position (kept by the
// moves) less those at the knot (OneBodyJastrow.h:136-140, TwoBodyJastrow.h:103-107,
// ThreeBodyJastrow.h:262-273).  grid (parts, W): a workgroup stages its walker's positions, functors, cell
// and (IL: when they fit) the ions in LDS and takes electrons part, part + parts, ...; a wave takes four of a
// pair's knots at a time, so a position is read once for the four, and the workgroup's waves deal these
// fours out among themselves, whatever electrons have the pairs.
// Bound: vector arithmetic, (N + M) image distances per knot; with few walkers the latency of a wave's
// fours (13 us each at NiO-64).  NiO-64 FP32, 128 walkers, 396k knots: 0.68 ms; one walker, 3k knots: 26 us
// (0.91 ms and 163 us with an electron's pairs on one wave and workgroups of 16 electrons).
constexpr int kNlppTake = 4;
template <typename T>
__host__ __device__ inline size_t nlpp_jastrow_lds(int N, int M) {
  return sizeof(double) * 3 * (size_t)(N + M) + sizeof(Functor<T>) * (kMaxSpecies + 2) + sizeof(Cell<T>) +
         sizeof(int) * (size_t)N + 64;
}
template <typename T, bool J3, bool IL>
__global__ __launch_bounds__(256) void k_nlpp_jastrow(SysP<T> S, BatchP<T> B, const double* spheres, int maxp,
                                                      const double* near, const int* npairs, const int* first,
                                                      double* ratios) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int w = blockIdx.y, N = S.N, n = S.n, M = S.M, tid = threadIdx.x, nt = blockDim.x;
  const int lane = tid & 63, wid = tid >> 6, nw = nt >> 6;
  double* sR = (double*)smem;
  double* sI = sR + 3 * N;
  Functor<T>* sFn = (Functor<T>*)(smem + ((sizeof(double) * 3 * (size_t)(N + (IL ? M : 0)) + 15) & ~(size_t)15));
  Cell<T>* sCell = (Cell<T>*)(sFn + kMaxSpecies + 2);
  int* sNp = (int*)(sCell + 1);   // listed pairs of the workgroup's electrons
  const int ne = (N - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
  bool any = false;
  for (int i = tid; i < ne; i += nt) {
    sNp[i] = min(npairs[(size_t)w * N + blockIdx.x + (size_t)i * gridDim.x], maxp);
    any = any || sNp[i] > 0;
  }
  if (!__syncthreads_or(any)) return;
  for (int i = tid; i < 3 * N; i += nt) sR[i] = B.R[(size_t)w * 3 * N + i];
  if constexpr (IL)
    for (int i = tid; i < 3 * M; i += nt) sI[i] = S.ions[i];
  for (int i = tid; i < (int)(sizeof(Functor<T>) * (kMaxSpecies + 2) / 4); i += nt) ((int*)sFn)[i] = ((const int*)S.fn)[i];
  for (int i = tid; i < (int)(sizeof(Cell<T>) / 4); i += nt) ((int*)sCell)[i] = ((const int*)S.cell)[i];
  __syncthreads();
  const Cell<T>& C = *sCell;
  const bool ortho = C.ortho != T(0);
  auto value = [&](const Functor<T>& f, T dx, T dy, T dz) -> double {
    T ox, oy, oz;
    const T r = ortho ? image_distance_ortho(C, -dx, -dy, -dz) : min_image(C, dx, dy, dz, T(-1), ox, oy, oz);
    const bool in = r < f.rcut;   // an interior radius keeps the lookup in range
    const T u = functor_v(f, in ? r : f.rcut * T(0.5));
    return in ? (double)u : 0.0;
  };
  constexpr int kFours = kNlppKnots / kNlppTake;
  int turn = __builtin_amdgcn_readfirstlane(wid);   // fours to the wave's next one
  for (int i = 0; i < ne; ++i) {
    const int nf = __builtin_amdgcn_readfirstlane(sNp[i]) * kFours;   // the same on every lane
    if (turn >= nf) {
      turn -= nf;
      continue;
    }
    const int e = blockIdx.x + i * gridDim.x;
    const size_t idx = (size_t)w * N + e;
    const size_t o = (size_t)w * 5 * N + e;
    const double j1o = (double)B.J1[o], j2o = (double)B.J2[o] + (J3 ? (double)B.J3[o] : 0.0);
    const bool up = e < n;
    for (; turn < nf; turn += nw) {
      const int p = turn / kFours, k0 = (turn - p * kFours) * kNlppTake;
      const double* q = near + (idx * maxp + p) * 4;
      const double d = q[0], ox = sR[e] + q[1], oy = sR[N + e] + q[2], oz = sR[2 * N + e] + q[3];
      const double* sp = spheres + ((size_t)w * kNlppKnots + k0) * 3;
      double px[kNlppTake], py[kNlppTake], pz[kNlppTake], v[2 * kNlppTake];
#pragma unroll
      for (int k = 0; k < kNlppTake; ++k) {
        px[k] = d * sp[3 * k] + ox;
        py[k] = d * sp[3 * k + 1] + oy;
        pz[k] = d * sp[3 * k + 2] + oz;
        v[k] = v[kNlppTake + k] = 0.0;
      }
      for (int ci = lane; ci < M; ci += 64) {
        const Functor<T>& f = sFn[S.species[ci]];
        if (f.ncoef == 0) continue;
        double x, y, z;
        if constexpr (IL) x = sI[ci], y = sI[M + ci], z = sI[2 * M + ci];
        else x = S.ions[ci], y = S.ions[M + ci], z = S.ions[2 * M + ci];
#pragma unroll
        for (int k = 0; k < kNlppTake; ++k) v[k] += value(f, (T)(x - px[k]), (T)(y - py[k]), (T)(z - pz[k]));
      }
      for (int j = lane; j < N; j += 64) {
        const Functor<T>& f = sFn[kMaxSpecies + (((j < n) == up) ? 0 : 1)];
        const double x = sR[j], y = sR[N + j], z = sR[2 * N + j];
        const bool self = j == e;
#pragma unroll
        for (int k = 0; k < kNlppTake; ++k) {
          const double u = value(f, (T)(x - px[k]), (T)(y - py[k]), (T)(z - pz[k]));
          v[kNlppTake + k] += self ? 0.0 : u;
        }
      }
      if constexpr (J3)
#pragma unroll
        for (int k = 0; k < kNlppTake; ++k)
          v[kNlppTake + k] += j3_value_wave<T>(S, B, C, w, e, px[k], py[k], pz[k], sR, sI, lane);
      wave_sums_rows<2 * kNlppTake>(v);
      // row r (lanes 16r ..) holds sums 2r and 2r + 1: the J1 sums of knots k in rows 0 and 1, the J2
      // sums in rows 2 and 3; lanes 0 and 16 take their knots' J2 sums from lanes 32 and 48
      const double b0 = __shfl(v[0], (lane & 31) + 32), b1 = __shfl(v[1], (lane & 31) + 32);
      if ((lane & 15) == 0 && lane < 32) {
        double* out = ratios + ((size_t)first[idx] + p) * kNlppKnots + k0 + (lane >> 4) * 2;
        out[0] = (j1o - v[0]) + (j2o - b0);
        out[1] = (j1o - v[1]) + (j2o - b1);
      }
    }
    turn -= nf;
  }
}

// Determinant part and the ratios, in the order of the knot list: LK lanes of a wave take a knot and
// hold all of its 64 stencil points' sums for Q 16-byte orbital groups each (no LDS, no barriers).
// A wave takes `take` runs of 64 / LK consecutive knots at a time (units null: in the order of the pairs).  The
// stencil rows come from L2 and the CU's cache (cached loads: neighbouring knots want them).
// Bound: L2 and L1 bandwidth of the stencils, 64 rows per knot.  NiO-64, 128 walkers, 396k knots:
// 1.52 ms in FP32 (26 TB/s of stencil bytes, 2.3 GB from HBM); the whole evaluation's kernels 2.4 ms against
// 7.4 for a workgroup per knot in the order of ions, whose stencils came from HBM (38 GB at 5.2 TB/s).
template <typename T, int LK, int Q>
__global__ __launch_bounds__(256) void k_nlpp_ratios(SysP<T> S, BatchP<T> B, const double* spheres, int maxp,
                                                     const double* near, const int* items, const int* units,
                                                     const int* cnt, int take, double* ratios) {
  using VT = typename V16<T>::type;
  constexpr int VW = V16<T>::n, KW = 64 / LK;
  const int N = S.N, n = S.n, nq = S.npad / VW;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int lk = lane & (LK - 1), slot = lane / LK;
  // workgroup b runs on XCD b % 8, and XCD x takes the x-th eighth of the list (gridDim.x % 8 == 0)
  const int nu = cnt[0] * kNlppKnots, run = KW * take, nruns = ceil_div(nu, run);
  const int xcd = blockIdx.x & 7, per = (gridDim.x >> 3) * nw;
  const int lo = (int)((long long)nruns * xcd / 8), hi = (int)((long long)nruns * (xcd + 1) / 8);
  for (int rn = lo + (int)(blockIdx.x >> 3) * nw + wid; rn < hi; rn = walk_next(rn, per, hi))
    for (int t = 0; t < take; ++t) {
      const unsigned at = (unsigned)(rn * run) + (unsigned)(t * KW + slot);   // past INT_MAX at a full list's end
      const int last = (int)min(at, (unsigned)nu - 1u);   // past the end: the last knot again, not stored
      const int u = units != nullptr ? units[last] : last;
      int w, e;
      double pt[3];
      nlpp_point(S, B, spheres, maxp, near, items, u, w, e, pt);
      const int det = e < n ? 0 : 1, row = e - det * n;
      const T* arow = B.Ainv + ((size_t)w * 2 + det) * n * n + (size_t)row * n;
      VT av[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int o = (lk + LK * q) * VW;
        if (n % VW == 0)
          av[q] = *reinterpret_cast<const VT*>(arow + (o < n ? o : 0));
        else
#pragma unroll
          for (int v = 0; v < VW; ++v) av[q][v] = arow[o + v < n ? o + v : 0];
#pragma unroll
        for (int v = 0; v < VW; ++v) av[q][v] = o + v < n ? av[q][v] : T(0);
      }
      int ix[3];
      double tt[3];
      spline_locate(S.spoG, S.ng, pt[0], pt[1], pt[2], ix, tt);
      const T* base = S.coefs + (size_t)ix[0] * S.xs + (size_t)ix[1] * S.ys + (size_t)ix[2] * S.zs;
      int off[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) off[q] = min(lk + LK * q, nq - 1) * VW;
      T a[4], b[4], c[4], d1[4], d2[4];
      bspline_weights<T>((T)tt[0], a, d1, d2);
      bspline_weights<T>((T)tt[1], b, d1, d2);
      bspline_weights<T>((T)tt[2], c, d1, d2);
      T acc[Q][VW];
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int v = 0; v < VW; ++v) acc[q][v] = T(0);
#pragma unroll
      for (int p = 0; p < 16; ++p) {
        const T* col = base + (size_t)(p >> 2) * S.xs + (size_t)(p & 3) * S.ys;
        VT x[Q][4];
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
          for (int k = 0; k < 4; ++k) x[q][k] = *reinterpret_cast<const VT*>(col + (size_t)k * S.zs + off[q]);
        const T wxy = a[p >> 2] * b[p & 3];
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
          for (int v = 0; v < VW; ++v)
            acc[q][v] += wxy * (c[0] * x[q][0][v] + c[1] * x[q][1][v] + c[2] * x[q][2][v] + c[3] * x[q][3][v]);
      }
      double s = 0.0;
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int v = 0; v < VW; ++v) {
          // the table's columns past n may hold anything: they enter as zeros, like av.  (The sum is pinned
          // first, or the compiler computes it, loads and all, in a branch of its own: twice the time)
          T x = acc[q][v];
          asm volatile("" : "+v"(x));
          x = (lk + LK * q) * VW + v < n ? x : T(0);
          s += (double)x * (double)av[q][v];
        }
      s = dpp_add<0xB1, 0xf>(s);   // the lane's row of 16
      s = dpp_add<0x4E, 0xf>(s);
      s = dpp_add<0x141, 0xf>(s);
      s = dpp_add<0x140, 0xf>(s);
      if constexpr (LK >= 32) {
        double x = s, y = s;
        swap_rows(x, y);
        s = x + y;
      }
      if constexpr (LK == 64) {
        double x = s, y = s;
        swap_halves(x, y);
        s = x + y;
      }
      if (lk == 0 && at < (unsigned)nu)
        ratios[u] = s * exp(ratios[u]);
    }
}

// stand-alone distance rows: lane per (source, target)
template <typename T>
__global__ void k_distance_rows(Cell<T> C, int npts, const double* src, const int* flip_ind, int nt,
                                const double* tgt, double* r, double* dr) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)npts * nt) return;
  const int p = (int)(idx / nt), t = (int)(idx - (size_t)p * nt);
  const T flip = t < flip_ind[p] ? T(1) : T(-1);
  T dx, dy, dz;
  const T rr = min_image(C, (T)(tgt[3 * t] - src[3 * p]), (T)(tgt[3 * t + 1] - src[3 * p + 1]),
                         (T)(tgt[3 * t + 2] - src[3 * p + 2]), flip, dx, dy, dz);
  r[idx] = (double)rr;
  dr[3 * (size_t)idx] = (double)dx;
  dr[3 * (size_t)idx + 1] = (double)dy;
  dr[3 * (size_t)idx + 2] = (double)dz;
}

// ------------------------------------------------------------------ Jastrow from scratch
// J1 per electron over the ions and J2 per electron over its full row; the
// sums equal the lower-triangle recompute of TwoBodyJastrow.h:356-400.  With a
// three-body Jastrow (ThreeBodyJastrow::recompute, ThreeBodyJastrow.h:363-401): every
// electron's near-ion record and ion mask, then every electron's sums over its pairs
// (each pair is evaluated by both of its electrons, so each writes only its own sums).
// LDS: positions [3N], reduction [48], functors, cell, then the ion masks [N][mw].
template <typename T>
__host__ __device__ inline size_t jastrow_init_lds(int N, int mw) {
  return sizeof(double) * (3 * (size_t)N + 48) + sizeof(Functor<T>) * (kMaxSpecies + 2) + sizeof(Cell<T>) + 16 +
         sizeof(unsigned long long) * (size_t)N * mw;
}
template <typename T>
__global__ __launch_bounds__(1024) void k_jastrow_init(SysP<T> S, BatchP<T> B) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int w = blockIdx.x, tid = threadIdx.x, nt = blockDim.x, N = S.N, n = S.n, M = S.M;
  const int i0 = blockIdx.y * nt;   // gridDim.y > 1 (no three-body Jastrow): nt electrons per workgroup
  double* sR = (double*)smem;
  double* sRed = sR + 3 * N;
  Functor<T>* sFn = (Functor<T>*)(sRed + 48);
  Cell<T>* sCell = (Cell<T>*)(sFn + kMaxSpecies + 2);
  unsigned long long* sMask =
      (unsigned long long*)(smem + ((sizeof(double) * (3 * (size_t)N + 48) + sizeof(Functor<T>) * (kMaxSpecies + 2) +
                                      sizeof(Cell<T>) + 15) & ~(size_t)15));
  const bool j3 = S.j3 != nullptr;
  const int mw = S.mw;
  if (tid == 0) *sCell = *S.cell;
  for (int i = tid; i < 3 * N; i += nt) sR[i] = B.R[(size_t)w * 3 * N + i];
  {
    const int words = (int)(sizeof(Functor<T>) * (kMaxSpecies + 2) / 4);
    for (int i = tid; i < words; i += nt) ((int*)sFn)[i] = ((const int*)S.fn)[i];
  }
  __syncthreads();
  T* J2 = B.J2 + (size_t)w * 5 * N;
  T* J1 = B.J1 + (size_t)w * 5 * N;
  double vsum = 0, usum = 0, tsum = 0;
  for (int i = i0 + tid; i < N; i += nt * gridDim.y) {
    const double x = sR[i], y = sR[N + i], z = sR[2 * N + i];
    T v = 0, gx = 0, gy = 0, gz = 0, lap = 0;
    T* rec = j3 ? B.j3near + ((size_t)w * N + i) * kJ3Rec : nullptr;
    unsigned long long mk[kJ3MaxIons / 64] = {0, 0, 0, 0};
    int cnt = 0;
    for (int ci = 0; ci < M; ++ci) {
      const Functor<T>& f = sFn[S.species[ci]];
      const T L3 = j3 ? S.j3[2 * S.species[ci]].L : T(0);
      if (f.ncoef == 0 && !(L3 > T(0))) continue;
      T dx, dy, dz;
      const T r = min_image(*sCell, (T)(S.ions[ci] - x), (T)(S.ions[M + ci] - y), (T)(S.ions[2 * M + ci] - z), T(-1),
                            dx, dy, dz);
      if (f.ncoef > 0 && r < f.rcut) {
        T u, du, d2u;
        functor_vgl(f, r, u, du, d2u);
        v += u;
        lap += d2u + T(2) * du;
        gx += du * dx;
        gy += du * dy;
        gz += du * dz;
      }
      if (r < L3) {
        if (cnt < kJ3Near) {
          T* e = rec + 1 + 5 * cnt;
          e[0] = (T)ci;
          e[1] = r;
          e[2] = dx;
          e[3] = dy;
          e[4] = dz;
        }
        ++cnt;
        mk[ci >> 6] |= 1ull << (ci & 63);
      }
    }
    if (j3) {
      rec[0] = (T)cnt;
      if (cnt > kJ3Near) atomicOr(B.flags, kFlagJ3Near);
      for (int q = 0; q < mw; ++q) {
        sMask[(size_t)i * mw + q] = mk[q];
        B.j3mask[((size_t)w * N + i) * mw + q] = mk[q];
      }
    }
    J1[i] = v;
    J1[N + i] = gx;
    J1[2 * N + i] = gy;
    J1[3 * N + i] = gz;
    J1[4 * N + i] = lap;
    vsum += (double)v;
    T U = 0, hx = 0, hy = 0, hz = 0, l2 = 0;
    const bool up = i < n;
    for (int j = 0; j < N; ++j) {
      if (j == i) continue;
      const Functor<T>& f = sFn[kMaxSpecies + (((j < n) == up) ? 0 : 1)];
      T dx, dy, dz;
      const T r = min_image(*sCell, (T)(sR[j] - x), (T)(sR[N + j] - y), (T)(sR[2 * N + j] - z),
                            j < i ? T(1) : T(-1), dx, dy, dz);
      if (r < f.rcut) {
        T u, du, d2u;
        functor_vgl(f, r, u, du, d2u);
        U += u;
        l2 += d2u + T(2) * du;
        hx += du * dx;
        hy += du * dy;
        hz += du * dz;
      }
    }
    J2[i] = U;
    J2[N + i] = hx;
    J2[2 * N + i] = hy;
    J2[3 * N + i] = hz;
    J2[4 * N + i] = -l2;
    usum += (double)U;
  }
  if (j3) {
    __syncthreads();   // every electron's mask and near-ion record are in place
    T* J3 = B.J3 + (size_t)w * 5 * N;
    for (int j = tid; j < N; j += nt) {
      const double x = sR[j], y = sR[N + j], z = sR[2 * N + j];
      const T* rec = B.j3near + ((size_t)w * N + j) * kJ3Rec;
      const int cnt = min((int)rec[0], kJ3Near);
      const bool jup = j < n;
      T acc[5] = {0, 0, 0, 0, 0};
      for (int q = 0; q < cnt; ++q) {
        const T* e = rec + 1 + 5 * q;
        const int I = (int)e[0];
        const T rjI = e[1], jI[3] = {e[2], e[3], e[4]};
        const unsigned long long bit = 1ull << (I & 63);
        const int wd = I >> 6, sp = S.species[I];
        for (int k = 0; k < N; ++k) {
          if (k == j || !(sMask[(size_t)k * mw + wd] & bit)) continue;
          T kI[3], jk[3];
          const T rkI = min_image(*sCell, (T)(S.ions[I] - sR[k]), (T)(S.ions[M + I] - sR[N + k]),
                                  (T)(S.ions[2 * M + I] - sR[2 * N + k]), T(-1), kI[0], kI[1], kI[2]);
          const T rjk = min_image(*sCell, (T)(sR[k] - x), (T)(sR[N + k] - y), (T)(sR[2 * N + k] - z),
                                  k < j ? T(1) : T(-1), jk[0], jk[1], jk[2]);
          T o[9], js[5], ks[5];
          poly3_vgl(S.j3[2 * sp + (((k < n) == jup) ? 0 : 1)], rjk, rjI, rkI, o);
          j3_pair_terms(o, jk, jI, kI, js, ks);
#pragma unroll
          for (int c = 0; c < 5; ++c) acc[c] += js[c];
        }
      }
#pragma unroll
      for (int c = 0; c < 5; ++c) J3[(size_t)c * N + j] = acc[c];
      tsum += (double)acc[0];
    }
  }
  if (gridDim.y > 1) return;   // the logs come with evaluateGL, which follows
  double red[3] = {vsum, usum, tsum};
  block_sum<double, 3>(red, sRed);
  if (tid == 0) {
    B.jlog[w * 3 + 0] = -red[0];
    B.jlog[w * 3 + 1] = -0.5 * red[1];
    B.jlog[w * 3 + 2] = -0.5 * red[2];
  }
}

// ------------------------------------------------------------------ evaluateGL
// determinant part, one wave per electron row (DiracDeterminant.cpp:158-187)
template <typename T>
__global__ __launch_bounds__(256) void k_det_gl(SysP<T> S, BatchP<T> B, double* G, double* Lp) {
  const int w = blockIdx.y, N = S.N, n = S.n;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int e = blockIdx.x * nw + wid;
  if (e >= N) return;
  const int det = e < n ? 0 : 1, row = e - det * n;
  const size_t moff = ((size_t)w * 2 + det) * n * n;
  const T* a = B.Ainv + moff + (size_t)row * n;
  const T* dp = B.dpsiM + ((size_t)w * 2 + det) * (size_t)n * 3 * n + (size_t)row * 3 * n;
  const T* d2 = B.d2psiM + moff + (size_t)row * n;
  T gx = 0, gy = 0, gz = 0, l = 0;
  for (int j = lane; j < n; j += 64) {
    const T v = a[j];
    gx += v * dp[j];
    gy += v * dp[n + j];
    gz += v * dp[2 * n + j];
    l += v * d2[j];
  }
  gx = wave_sum(gx);
  gy = wave_sum(gy);
  gz = wave_sum(gz);
  l = wave_sum(l);
  if (lane == 0) {
    const size_t o = (size_t)w * N + e;
    G[3 * o] = gx;
    G[3 * o + 1] = gy;
    G[3 * o + 2] = gz;
    Lp[o] = (double)l - ((double)gx * gx + (double)gy * gy + (double)gz * gz);
  }
}

// Jastrow part + LogValue (WaveFunction.cpp:261-279; J logs from the sums,
// TwoBodyJastrow.h:413-430, OneBodyJastrow.h:148-160)
template <typename T>
__global__ __launch_bounds__(256) void k_finish_gl(SysP<T> S, BatchP<T> B, double* G, double* Lp, double* logv,
                                                   double* hist, int hist_cap) {
  __shared__ double sRed[48];
  const int w = blockIdx.x, N = S.N;
  const T* J2 = B.J2 + (size_t)w * 5 * N;
  const T* J1 = B.J1 + (size_t)w * 5 * N;
  const T* J3 = S.j3 != nullptr ? B.J3 + (size_t)w * 5 * N : nullptr;
  double vs = 0, us = 0, ts = 0;
  for (int i = threadIdx.x; i < N; i += blockDim.x) {
    const size_t o = (size_t)w * N + i;
    G[3 * o] += (double)J1[N + i] + (double)J2[N + i];
    G[3 * o + 1] += (double)J1[2 * N + i] + (double)J2[2 * N + i];
    G[3 * o + 2] += (double)J1[3 * N + i] + (double)J2[3 * N + i];
    Lp[o] += -(double)J1[4 * N + i] + (double)J2[4 * N + i];
    vs += (double)J1[i];
    us += (double)J2[i];
    if (J3 != nullptr) {   // ThreeBodyJastrow::evaluateGL (ThreeBodyJastrow.h:627-645)
      G[3 * o] += (double)J3[N + i];
      G[3 * o + 1] += (double)J3[2 * N + i];
      G[3 * o + 2] += (double)J3[3 * N + i];
      Lp[o] += (double)J3[4 * N + i];
      ts += (double)J3[i];
    }
  }
  double red[3] = {vs, us, ts};
  block_sum<double, 3>(red, sRed);
  if (threadIdx.x == 0) {
    B.jlog[w * 3 + 0] = -red[0];
    B.jlog[w * 3 + 1] = -0.5 * red[1];
    B.jlog[w * 3 + 2] = -0.5 * red[2];
    const double v = B.logdet[w * 2] + B.logdet[w * 2 + 1] - red[0] - 0.5 * red[1] - 0.5 * red[2];
    logv[w] = v;
    if (hist != nullptr) {
      const int slot = B.sweep[0] - B.sweep[1];
      if (slot >= 0 && slot < hist_cap) hist[(size_t)slot * B.W + w] = v;
      if (w == 0) B.sweep[3] = slot;
    }
  }
}

// Holds its stream for `ticks` of the constant 100 MHz wall clock (one lane, a bounded wait that
// always ends).  Side-stream work released by the same event as a move launch waits behind it, so
// the move kernel's workgroups, which each need a whole CU, are placed before the side kernels'
// workgroups take a share of every CU.
__global__ void k_hold(unsigned long long ticks) {
  if (threadIdx.x == 0) {
    const unsigned long long t0 = wall_clock64();
    while (wall_clock64() - t0 < ticks) __builtin_amdgcn_s_sleep(8);
  }
}

// a run begins: its history starts at slot 0 and its first proposals belong to the current sweep
__global__ void k_begin_run(int* sweep) {
  if (threadIdx.x == 0 && blockIdx.x == 0) sweep[1] = sweep[2] = sweep[0];
}

__global__ void k_count(int* counter) {
  if (threadIdx.x == 0 && blockIdx.x == 0) counter[0] += 1;
}

// The second determinant's FP64 refresh lands after that sweep's evaluateGL (it runs beside
// the next sweep's first-determinant moves): swap in the fresh log|det| and phase and move the
// sweep's recorded log|Psi| by the same difference.
// The sweep's history slot is the one its evaluateGL wrote (sweep[3]): this kernel runs after
// that evaluateGL and before the next one.
__global__ void k_refresh_det(int W, int det, const double* ld_fresh, const double* ph_fresh, double* logdet,
                              double* phase, double* logv, double* hist, int hist_cap, const int* sweep) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= W) return;
  const double delta = ld_fresh[w] - logdet[w * 2 + det];
  logdet[w * 2 + det] = ld_fresh[w];
  phase[w * 2 + det] = ph_fresh[w];
  logv[w] += delta;
  const int slot = sweep[3];
  if (hist != nullptr && slot >= 0 && slot < hist_cap) hist[(size_t)slot * W + w] += delta;
}

}  // namespace qmcx

namespace qmcx {

// ------------------------------------------------------------------ stand-alone delayed-update engine
// One determinant, device-resident inverse (the DU_TYPE plug point of
// DiracDeterminant<DU_TYPE>, DiracDeterminant.cpp:339-341).  The flush reuses the
// batch flush kernels with one walker.
//
// getInvRow (DelayedUpdate.h:96-114): invRow = Ainv[row] - V^T Binv^T U Ainv[row];
// Binv^T U Ainv[row] is parked in row c of Binv, where acceptRow reads it.
template <typename T>
__global__ __launch_bounds__(256) void k_du_get_inv_row(BatchP<T> B, int n, int row, double* out) {
  __shared__ double sp[128];
  const int c = B.ndelay[0], K = B.K, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const T* ar = B.Ainv + (size_t)row * n;
  for (int d = wid; d < c; d += 4) {
    const T* u = B.A + (size_t)B.rows[d] * n;
    double s = 0;
    for (int j = lane; j < n; j += 64) s += (double)u[j] * (double)ar[j];
    s = wave_sum(s);
    if (lane == 0) sp[d] = s;
  }
  __syncthreads();
  for (int r = tid; r < c; r += 256) {
    double s = 0;
    for (int q = 0; q < c; ++q) s += B.Binv[q * K + r] * sp[q];
    B.Binv[c * K + r] = s;
  }
  __syncthreads();
  for (int j = tid; j < n; j += 256) {
    double v = (double)ar[j];
    for (int d = 0; d < c; ++d) v -= (double)B.Vbuf[(size_t)d * n + j] * B.Binv[c * K + d];
    out[j] = v;
  }
}

// acceptRow (DelayedUpdate.h:124-153): V_c = Ainv[row], U_c = psiV (kept as row `row` of A),
// the capacitance inverse grows by one row and column (FP64).
template <typename T>
__global__ __launch_bounds__(256) void k_du_accept_row(BatchP<T> B, int n, int row, const double* psiv) {
  __shared__ double sp[130];
  const int c = B.ndelay[0], K = B.K, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const T* ar = B.Ainv + (size_t)row * n;
  for (int d = wid; d <= c; d += 4) {
    const T* v = d == c ? ar : B.Vbuf + (size_t)d * n;
    double s = 0;
    for (int j = lane; j < n; j += 64) s += (double)v[j] * psiv[j];
    s = wave_sum(s);
    if (lane == 0) sp[d] = -s;
  }
  __syncthreads();
  for (int j = tid; j < n; j += 256) {
    B.Vbuf[(size_t)c * n + j] = ar[j];
    B.A[(size_t)row * n + j] = (T)psiv[j];
  }
  double y = -sp[c];
  for (int i = 0; i < c; ++i) y += B.Binv[c * K + i] * sp[i];
  const double yi = 1.0 / y;
  for (int s2 = tid; s2 < c; s2 += 256) {
    double t = 0;
    for (int r = 0; r < c; ++r) t += B.Binv[s2 * K + r] * sp[r];
    B.Binv[s2 * K + c] = yi * t;
  }
  __syncthreads();
  for (int idx = tid; idx < c * c; idx += 256) {
    const int s2 = idx / c, r = idx - s2 * c;
    B.Binv[s2 * K + r] -= B.Binv[c * K + r] * B.Binv[s2 * K + c];
  }
  __syncthreads();
  for (int i = tid; i < c; i += 256) B.Binv[c * K + i] *= -yi;
  if (tid == 0) {
    B.Binv[c * K + c] = yi;
    B.rows[c] = row;
    B.ndelay[0] = c + 1;
  }
}

__global__ void k_du_reset(int* ndelay) {
  if (threadIdx.x == 0) ndelay[0] = 0;
}

}  // namespace qmcx
