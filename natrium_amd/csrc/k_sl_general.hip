// Fused semi-Lagrangian stream + BGK collide for arbitrary (non-affine) lattice
// hex meshes.
//
// The assembled reference operator stores, per (DoF, direction), the shape values
// of the departure cell at the departure point, dropping |w| < 1e-10
// (advection/SemiLagrangian.cpp:457-503, SemiLagrangianTools.cpp:15-64). Here each
// (direction, DoF) keeps only its departure point (assembled in FP64 on the GPU);
// the (p+1)^D tensor-product Lagrange weights are re-evaluated in FP64 registers
// every step with the same cut-off. Records: FP64 storage keeps the cell and FP64
// unit coordinates (4 + 8D bytes); FP32 storage keeps the cell and nearest GLL node
// packed in one int32 and the offsets from that node in 2^-30 fixed point (4 + 4D
// bytes, one interleaved record), instead of (p+1)^D stored weights plus column indices
// per row.
#include "nat_collide.hpp"
#include "nat_fastdiv.hpp"

#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>


namespace nat {

// Workgroup index regrouped so that each XCD (workgroup i is dispatched to XCD i % 8)
// runs a contiguous range of the grid: the gathers of a block read rows of the blocks
// one lattice plane away, which then sit in the same L2 (C3: FP32 1.60 -> 1.78 GLUPS,
// FP64 0.84 -> 0.92).
__device__ __forceinline__ int64_t xcd_block_index() {
  const int64_t b = blockIdx.x, per = gridDim.x / 8;
  return b < per * 8 ? (b % 8) * per + b / 8 : b;
}

template <typename T>
struct GeneralArgs {
  const T* fin;
  T* fout;
  int64_t stride;
  int64_t n;          // FE_Q DoFs
  int nfe[3];         // FE_Q lattice nodes per axis
  int N[3];           // cells per axis
  FastDivU divN0, divN1;  // division by N[0], N[1]
  int64_t rows;       // lattice rows along x (n / nfe[0]); 0: threads take DoFs in order
  FastDivU divM;      // division by nfe[0] - 2, the x-interior DoFs of a row
  FastDivU divG;      // division by 64 nfe[0], the DoFs of a group of 64 rows
  const int* cell;    // FP64 storage: [(alpha-1) * n + i] departure cell (-1: identity row)
  const double* xi;   //   unit coordinates, D per record
  const int* rec;     // FP32 storage: D + 1 int32 per record: cell * (p+1)^D + anchor node
                      //   (-1: identity row), then the offsets from the anchor (2^-30 units)
  int dir_bytes;      // bytes of one direction's array (buffer-load range)
  const int* wall_idx;        // walls: wall entry per DoF or -1 (null: no walls)
  const unsigned* wall_flip;  //   per entry: bit alpha set when alpha reads the opposite direction
  const double* wall_bias;    //   per entry: Q values added after interpolation
  double gll[MAXP + 1];
  double inv_den[MAXP + 1];
  double dgl[MAXP + 1][MAXP + 1];  // x_a - x_k
};

// Launch shape. A block owns G groups of 64 DoFs and has W waves; the items (group, direction)
// are dealt to the waves direction by direction, each wave taking another group from one
// direction to the next, and the streamed populations meet in LDS before one wave per group
// collides it. Two things follow. Waves whose DoFs lie on the faces of the box spend several
// times as long on a direction (kept_wave), and the block shares that. And W may exceed G, so
// that a mesh of few blocks still has waves to hide its dependent loads behind: one HBM round
// trip (the record) and P + 1 L2 round trips (the source planes) per item.
//
// Two forms. WIDE: W = 16 (8 at p >= 5, for registers), for grids of few blocks. Otherwise
// W = 2 G; FP32 storage at 6 waves per SIMD (80 registers), FP64 with the registers one plane of
// rows in flight needs (more waves, or more rows, measured slower: they take the L1 and L2 lines
// of the others' source planes). Before, a thread took its DoF through all directions by itself.
// us per step, perturbed boxes, before / W = 2 G / wide (the rule's choice in [ ]):
//   D3Q19 p=3 FP32   6^3 cells  64.0/ 34.3/[24.4]   16^3  91.8/ 45.3/[44.5]   24^3 157/[100]/111   36^3 511/[364]
//             FP64   6^3        70.1/ 59.4/[25.7]   16^3  90.6/[63.9]/74.9    24^3 241/[179]/237   36^3 676/[602]
//   D3Q27 p=3 FP32  10^3        71.3/ 38.9/[29.5]   24^3   242/[127]/143      30^3 542/[281]
//             FP64  10^3        90.2/ 66.4/[31.9]   24^3   333/[259]/361      30^3 638/[504]
//   D3Q19 p=2 FP64  16^3        48.0/ 24.7/[20.3]   36^3   170/[135]/139
//   D2Q9  p=4 FP64  32^2 walls  20.8/    -/[ 9.5]   64^2  23.7/ 18.3/[14.7]   128^2 43.6/[31.9]/36.8
template <int D, int Q, int P, typename T, bool WIDE>
struct GeneralShape {
  static constexpr int G = sizeof(T) == 4 ? 4 : 2;
  static constexpr int W = WIDE ? (P >= 5 ? 8 : 16) : 2 * G;
  static constexpr int bs = G * 64;  // DoFs per block
  static constexpr int nt = W * 64;
  static constexpr int waves = WIDE ? (P >= 5 ? 2 : 4) : (sizeof(T) == 4 ? 6 : 2);  // per SIMD, at least
  // source rows of `zu` z-planes are loaded together, as their raw values fit 64 registers
  static constexpr int nz = D == 3 ? P + 1 : 1;
  static constexpr int plane_regs = (P + 1) * (P + 1) * (int)(sizeof(T) / 4);
  static constexpr int zfit = 64 / plane_regs < 1 ? 1 : (64 / plane_regs > nz ? nz : 64 / plane_regs);
  static constexpr int zu = WIDE ? zfit : 1;
  // the next item's record loaded before this item's gathers (at 6 waves: spills, 108 -> 123 us)
  static constexpr bool prefetch = waves < 6;
  // cut-off rows a wave sums together, at most 4, by the LDS that keeps the waves resident
  static constexpr int NL = D == 3 ? (P + 1) * (P + 1) * (P + 1) : (P + 1) * (P + 1);
  static constexpr int row_bytes = (NL + 3 * (P + 1)) * 8;
  static constexpr int spare = (WIDE ? 80 * 1024 : 160 * 1024 * W / (4 * waves) - 64) -
                               (Q - 1) * bs * (int)sizeof(T) - bs * 4 - (P + 1) * (P + 1) * 8;
  static constexpr int fit = spare / (W * row_bytes);
  static constexpr int R = fit < 0 ? 0 : (fit > 4 ? 4 : fit);
};

// Lagrange values at x_a + d (anchor a), in FP64: prod_{k != j} (x_a - x_k + d) / den_j.
// The differences come from an LDS copy of the table: the anchor differs from lane to lane, and
// from the kernel arguments its row is six gathers per direction, behind the record's load.
template <int P>
__device__ __forceinline__ void basis_at(const double* dgl, const double (&inv)[MAXP + 1], int a, double d,
                                         double (&v)[P + 1]) {
  double s[P + 1];
#pragma unroll
  for (int k = 0; k <= P; k++) s[k] = dgl[a * (P + 1) + k] + d;
#pragma unroll
  for (int j = 0; j <= P; j++) {
    double t = inv[j];
#pragma unroll
    for (int k = 0; k <= P; k++)
      if (k != j) t *= s[k];
    v[j] = t;
  }
}

template <int P>
__device__ __forceinline__ void basis_xi(const double (&x)[MAXP + 1], const double (&inv)[MAXP + 1], double xi,
                                         double (&v)[P + 1]) {
#pragma unroll
  for (int j = 0; j <= P; j++) {
    double t = inv[j];
#pragma unroll
    for (int m = 0; m <= P; m++)
      if (m != j) t *= (xi - x[m]);
    v[j] = t;
  }
}

// p+1 consecutive lattice values (one x row of a source cell) through raw buffer
// loads: byte offsets against a per-direction resource, in the fewest loads the row's
// length allows (16, 12, 8 and 4 bytes; buffer loads need dword alignment only): p = 2
// rows are one load in FP32 and two in FP64, p = 4 rows two and three.
template <int P, typename T>
__device__ __forceinline__ void load_row(__amdgpu_buffer_rsrc_t r, int off, double (&v)[P + 1]) {
  constexpr int W = (int)sizeof(T) / 4, ND = (P + 1) * W;  // dwords per value and per row
  unsigned q[ND];
  static_for<0, (ND + 3) / 4>([&](auto K) {
    constexpr int k = 4 * decltype(K)::value, n = ND - k < 4 ? ND - k : 4;
    if constexpr (n == 4) {
      const auto x = __builtin_amdgcn_raw_buffer_load_b128(r, off + 4 * k, 0, 0);
      static_for<0, 4>([&](auto J) { q[k + decltype(J)::value] = x[decltype(J)::value]; });
    } else if constexpr (n == 3) {
      const auto x = __builtin_amdgcn_raw_buffer_load_b96(r, off + 4 * k, 0, 0);
      static_for<0, 3>([&](auto J) { q[k + decltype(J)::value] = x[decltype(J)::value]; });
    } else if constexpr (n == 2) {
      const auto x = __builtin_amdgcn_raw_buffer_load_b64(r, off + 4 * k, 0, 0);
      static_for<0, 2>([&](auto J) { q[k + decltype(J)::value] = x[decltype(J)::value]; });
    } else {
      q[k] = __builtin_amdgcn_raw_buffer_load_b32(r, off + 4 * k, 0, 0);
    }
  });
#pragma unroll
  for (int m = 0; m <= P; m++) {
    if constexpr (W == 1)
      v[m] = (double)__builtin_bit_cast(float, q[m]);
    else
      v[m] = __builtin_bit_cast(double, ((unsigned long)q[2 * m + 1] << 32) | q[2 * m]);
  }
}

// min(|a|, |b|) in one instruction (fmin of fabs also quiets signalling NaNs, two more)
__device__ __forceinline__ double min_abs(double a, double b) {
  double r;
  asm("v_min_f64 %0, |%1|, |%2|" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// Weights, cut-off and arithmetic in FP64 for both storage precisions (FP32 weights
// rounded the same way at every step bias the FP32-shifted result).
//
// Velocity-neq bounce-back (SemiLagrangian.cpp:358-385, VelocityNeqBounceBack.cpp:
// 137-195): a DoF whose path met a wall reads the opposite direction's populations
// at the reflected departure point and adds 2 w (e . u_wall) / cs2 per hit. Such
// rows take the term-by-term path with per-lane source addresses. With FP32
// storage the shift w rho0 passes through, since opposite directions share w.
//
// The departure record of one (direction, DoF): FP64 storage the cell and FP64 unit
// coordinates, FP32 storage the packed cell/anchor code and fixed-point offsets.
template <int D, typename T>
struct DepRec {
  int c;
  double xi[D];
};
template <int D>
struct DepRec<D, float> {
  int c;
  int off[D];
};

template <int D, typename T>
__device__ __forceinline__ DepRec<D, T> load_rec(const GeneralArgs<T>& a, int64_t r) {
  DepRec<D, T> rec;
  if constexpr (sizeof(T) == 8) {
    rec.c = a.cell[r];
#pragma unroll
    for (int d = 0; d < D; d++) rec.xi[d] = a.xi[r * D + d];
  } else {
    if constexpr (D == 3) {  // one 16-byte load per record
      const int4 v = reinterpret_cast<const int4*>(a.rec)[r];
      rec.c = v.x;
      rec.off[0] = v.y;
      rec.off[1] = v.z;
      rec.off[2] = v.w;
    } else {
      rec.c = a.rec[r * 3];
      rec.off[0] = a.rec[r * 3 + 1];
      rec.off[1] = a.rec[r * 3 + 2];
    }
  }
  return rec;
}

// 1-D Lagrange weights of a departure record in FP64 and the lattice index of its cell's
// first node (records with rec.c >= 0 only).
template <int D, int P, typename T>
__device__ __forceinline__ int64_t dep_weights(const GeneralArgs<T>& a, const double* dgl, const DepRec<D, T>& rec,
                                               double (&lx)[P + 1], double (&ly)[P + 1], double (&lz)[P + 1]) {
  constexpr int NP = P + 1;
  constexpr int NL = (D == 3) ? NP * NP * NP : NP * NP;
  int c;
  if constexpr (sizeof(T) == 8) {
    c = rec.c;
    basis_xi<P>(a.gll, a.inv_den, rec.xi[0], lx);
    basis_xi<P>(a.gll, a.inv_den, rec.xi[1], ly);
    if constexpr (D == 3) basis_xi<P>(a.gll, a.inv_den, rec.xi[2], lz);
  } else {
    const int code = rec.c;
    c = code / NL;
    const int lin = code - c * NL;
    const int ax = lin % NP, ay = (lin / NP) % NP, az = (D == 3) ? lin / (NP * NP) : 0;
    constexpr double q = 1.0 / 1073741824.0;
    basis_at<P>(dgl, a.inv_den, ax, (double)rec.off[0] * q, lx);
    basis_at<P>(dgl, a.inv_den, ay, (double)rec.off[1] * q, ly);
    if constexpr (D == 3) basis_at<P>(dgl, a.inv_den, az, (double)rec.off[2] * q, lz);
  }
  const uint32_t q0 = a.divN0.div((uint32_t)c), q1 = a.divN1.div(q0);
  const int cx = c - (int)q0 * a.N[0];
  const int cy = (int)q0 - (int)q1 * a.N[1];
  const int cz = (D == 3) ? (int)q1 : 0;
  return (int64_t)cx * P + (int64_t)a.nfe[0] * ((int64_t)cy * P + (int64_t)a.nfe[1] * ((int64_t)cz * P));
}

// Buffer resource over one direction's population array (wave-uniform base).
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t dir_rsrc(const GeneralArgs<T>& a, const T* arr) {
  const uint64_t pb = (uint64_t)arr;
  const uint32_t phi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(pb >> 32));
  const uint32_t plo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)pb);
  return __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)phi << 32) | (uint64_t)plo), (short)0,
                                           __builtin_amdgcn_readfirstlane(a.dir_bytes), 0x00020000);
}

// The row of the assembled operator under the reference cut-off: every product weight
// (same factors, same order) is formed and the terms with |w| < 1e-10 dropped, the source
// rows read through buffer loads.
template <int D, int P, typename T>
__device__ __forceinline__ double kept_sum(__amdgpu_buffer_rsrc_t rs, int b0, int n0, int n1,
                                           const double (&lx)[P + 1], const double (&ly)[P + 1],
                                           const double (&lz)[P + 1]) {
  constexpr int NP = P + 1;
  constexpr int NZ = (D == 3) ? NP : 1;
  double kept = 0;
#pragma unroll 1
  for (int mz = 0; mz < NZ; mz++) {
    // a departure point on a node line has exactly one non-zero weight there: the other lines'
    // rows add nothing
    if (D == 3 && !__any(lz[mz] != 0.0)) continue;
    // a plane's rows together at p <= 3, one row at a time above (registers)
    constexpr int NV = P <= 3 ? NP : 1;
#pragma unroll 1
    for (int m0 = 0; m0 < NP; m0 += NV) {
      double v[NV][NP];
#pragma unroll
      for (int m = 0; m < NV; m++) load_row<P, T>(rs, b0 + (int)sizeof(T) * (n0 * (m0 + m + n1 * mz)), v[m]);
#pragma unroll
      for (int m = 0; m < NV; m++) {
        const int my = NV == NP ? m : m0;
        if (!__any(ly[my] != 0.0)) continue;
#pragma unroll
        for (int mx = 0; mx <= P; mx++) {
          const double w = (D == 3) ? lx[mx] * ly[my] * lz[mz] : lx[mx] * ly[my];
          kept += fabs(w) < 1e-10 ? 0.0 : w * v[m][mx];
        }
      }
    }
  }
  return kept;
}

// The cut-off rows of a wave, a few lanes' rows at a time and a term per lane: each lane with a
// cut-off row (cut) puts its weights into LDS, all lanes form one product each of that row (one
// gather for the whole (p+1)^D stencil), and the row's lane adds the products up in the order and
// with the roundings of kept_sum. Perturbed cells give almost every wave such a lane in the six
// directions along the axes (24^3 cells, p = 3: two of the three weight factors are then of the
// order of the distortion), and the serial sum costs the whole wave 16 row loads and
// about 900 VALU instructions each time (24^3 cells, p = 3, D3Q19 FP32: 150 -> 135 us per step).
// sc: the wave's R x (3 (P + 1) + NL) doubles of LDS. Waves with more than R such lanes keep the
// serial sum: a whole wave of them costs it no more than one.
template <int D, int P, typename T, int R>
__device__ __forceinline__ double kept_wave(__amdgpu_buffer_rsrc_t rs, bool cut, int b0, int n0, int n1,
                                            const double (&lx)[P + 1], const double (&ly)[P + 1],
                                            const double (&lz)[P + 1], double acc, double* sc) {
  constexpr int NP = P + 1, NL = (D == 3) ? NP * NP * NP : NP * NP, WS = D * NP;
  const unsigned long long m = __ballot(cut);
  const int count = __popcll(m);
  if (R == 0 || count > R) {
    if (cut) acc = kept_sum<D, P, T>(rs, b0, n0, n1, lx, ly, lz);
    return acc;
  }
  const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  const int slot = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
  double* const prod = sc + R * WS;
  if (cut) {
#pragma unroll
    for (int k = 0; k < NP; k++) {
      sc[slot * WS + k] = lx[k];
      sc[slot * WS + NP + k] = ly[k];
      if constexpr (D == 3) sc[slot * WS + 2 * NP + k] = lz[k];
    }
  }
  asm volatile("" ::: "memory");  // one wave's LDS operations complete in order; the compiler keeps it
#pragma unroll
  for (int c = 0; c < (NL + 63) / 64; c++) {
    const int t = c * 64 + lane;
    const int mx = t % NP, my = (t / NP) % NP, mz = D == 3 ? t / (NP * NP) : 0;
    const int off = (int)sizeof(T) * (mx + n0 * (my + n1 * mz));
    unsigned long long left = m;
    T v[R > 0 ? R : 1];
#pragma unroll
    for (int s = 0; s < R; s++) {
      const int b = __builtin_amdgcn_readlane(b0, left ? __builtin_ctzll(left) : 0);
      if (left && t < NL) {
        if constexpr (sizeof(T) == 4)
          v[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, b + off, 0, 0));
        else
          v[s] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, b + off, 0, 0));
      }
      left &= left - 1;
    }
#pragma unroll
    for (int s = 0; s < R; s++) {
      if (s < count && t < NL) {
        const double wxy = sc[s * WS + mx] * sc[s * WS + NP + my];
        const double w = (D == 3) ? wxy * sc[s * WS + 2 * NP + mz] : wxy;
        prod[s * NL + t] = fabs(w) < 1e-10 ? 0.0 : w * (double)v[s];
      }
    }
  }
  asm volatile("" ::: "memory");
  if (cut) {
    double kept = 0;
#pragma unroll 16
    for (int t = 0; t < NL; t++) kept += prod[slot * NL + t];
    acc = kept;
  }
  asm volatile("" ::: "memory");
  return acc;
}

// Returns the streamed population of direction al at DoF i from its departure record.
//
// Reference cut-off: product weights |w| < 1e-10 are dropped. When the product of the
// smallest 1-D magnitudes is >= 1e-10 no product can fall under it and the sum factorises
// row by row (rows through buffer loads). Otherwise (a departure point on or next to a node
// line of some axis) the kept terms are summed one product at a time (kept_wave). Lanes
// reflected at a wall (another direction's array) gather term by term. The fused
// multiply-adds of the factorised sum are written out, so all forms of the kernel agree
// bit for bit.
template <int D, int Q, int P, typename T, int ZU, int R>
__device__ __forceinline__ T gen_direction(const GeneralArgs<T>& a, const double* dgl, double* sc, int64_t i, int al,
                                           int widx, unsigned wmask, const DepRec<D, T>& rec) {
#pragma clang fp contract(off)
  constexpr int NP = P + 1;
  const int n0 = a.nfe[0], n1 = a.nfe[1];
  const T* own = a.fin + (int64_t)al * a.stride;
  const bool flip = (wmask >> al) & 1u;
  const double bias = widx >= 0 ? a.wall_bias[(int64_t)widx * Q + al] : 0.0;
  const __amdgpu_buffer_rsrc_t rs = dir_rsrc<T>(a, own);
  double lx[NP], ly[NP], lz[NP];
  double acc = 0;
  bool cut = false;
  int b0 = 0;
  if (rec.c < 0) {
    acc = (double)own[i];  // tracker life-time limit: identity row
  } else {
    const int64_t base = dep_weights<D, P, T>(a, dgl, rec, lx, ly, lz);
    constexpr int NZ = (D == 3) ? NP : 1;
    if (!flip) {
      double mx_ = min_abs(lx[0], lx[1]), my_ = min_abs(ly[0], ly[1]), mz_ = (D == 3) ? min_abs(lz[0], lz[1]) : 1.0;
#pragma unroll
      for (int m = 2; m <= P; m++) {
        mx_ = min_abs(mx_, lx[m]);
        my_ = min_abs(my_, ly[m]);
        if constexpr (D == 3) mz_ = min_abs(mz_, lz[m]);
      }
      cut = !(mx_ * my_ * mz_ >= 1e-10);
      b0 = (int)base * (int)sizeof(T);
      if (!cut)  // (waves of x-face DoFs: every lane is cut in the directions along the face)
#pragma unroll
      for (int mz0 = 0; mz0 < NZ; mz0 += ZU) {
#pragma unroll
        for (int dz = 0; dz < ZU; dz++) {
          const int mz = mz0 + dz;
          if (NZ % ZU != 0 && mz >= NZ) break;
          double accz = 0;
#pragma unroll
          for (int my = 0; my <= P; my++) {
            double v[NP];
            load_row<P, T>(rs, b0 + (int)sizeof(T) * (n0 * (my + n1 * mz)), v);
            double row = fma(lx[0], v[0], lx[1] * v[1]);
#pragma unroll
            for (int mx = 2; mx <= P; mx++) row = fma(lx[mx], v[mx], row);
            accz = fma(ly[my], row, accz);
          }
          acc = (D == 3) ? fma(lz[mz], accz, acc) : acc + accz;
        }
        // ZU planes of rows in flight: reading further ahead would cost registers, and waves
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      const T* src = a.fin + (int64_t)opposite<Q>(al) * a.stride;
#pragma unroll 1
      for (int mz = 0; mz < NZ; mz++)
#pragma unroll
        for (int my = 0; my <= P; my++)
#pragma unroll
          for (int mx = 0; mx <= P; mx++) {
            const double w = (D == 3) ? lx[mx] * ly[my] * lz[mz] : lx[mx] * ly[my];
            if (!(fabs(w) < 1e-10)) acc = fma(w, (double)src[base + mx + (int64_t)n0 * (my + (int64_t)n1 * mz)], acc);
          }
    }
  }
  if (__any(cut)) acc = kept_wave<D, P, T, R>(rs, cut, b0, n0, n1, lx, ly, lz, acc, sc);
  return (T)(acc + bias);
}

// DoF of thread g. Departure points of DoFs on the x faces of the box (x = 0 and x = L,
// unmoved vertices) sit on node lines for the directions along those faces, and such rows
// take the kernel's term-by-term cut-off path for the whole wave; in x-fastest order almost
// every 64-DoF wave holds one or two of them. Threads therefore take the lattice rows in
// groups of 64: first the x-interior DoFs of the group's rows (rows in order, DoFs in order:
// nfe[0] - 2 whole waves), then the group's 128 x-face DoFs (two waves), so that interior
// waves stay on the factorised path and the face waves sit beside their neighbours in the
// grid instead of forming a tail. Loads of an interior wave's own DoFs stay contiguous
// within each row.
template <typename T>
__device__ __forceinline__ int64_t dof_of(const GeneralArgs<T>& a, int64_t g) {
  if (a.rows == 0) return g;
  const int64_t nfe0 = a.nfe[0];
  const uint32_t m = (uint32_t)nfe0 - 2u;
  const uint32_t k = a.divG.div((uint32_t)g);
  const int64_t r0 = (int64_t)k * 64;
  const int64_t R = a.rows - r0 < 64 ? a.rows - r0 : 64;
  const uint32_t gg = (uint32_t)(g - r0 * nfe0);
  const uint32_t ni = (uint32_t)R * m;
  if (gg < ni) {
    const uint32_t q = a.divM.div(gg);
    return (r0 + q) * nfe0 + 1 + (int64_t)(gg - q * m);
  }
  const uint32_t h = gg - ni;
  return (r0 + (h >> 1)) * nfe0 + ((h & 1) ? nfe0 - 1 : 0);
}

template <int D, int Q, int P, typename T, bool WIDE>
__global__ __launch_bounds__((GeneralShape<D, Q, P, T, WIDE>::nt)) __attribute__((amdgpu_waves_per_eu(GeneralShape<D, Q, P, T, WIDE>::waves))) void k_sl_general(
    GeneralArgs<T> a, CollideArgs<T> ca, int write_macro) {
  using S = GeneralShape<D, Q, P, T, WIDE>;
  constexpr int G = S::G, W = S::W, bs = S::bs;
  __shared__ __align__(16) T col[Q - 1][bs];
  __shared__ double scr[S::R > 0 ? W * S::R * S::row_bytes / 8 : 1];
  __shared__ int dofs[bs];
  // FP32 records: differences of the GLL nodes, read with lane-dependent rows
  __shared__ double dgl[sizeof(T) == 4 ? (P + 1) * (P + 1) : 1];
  const int t = threadIdx.x;
  if constexpr (sizeof(T) == 4)
    if (t < (P + 1) * (P + 1)) dgl[t] = a.dgl[t / (P + 1)][t % (P + 1)];
  if (t < bs) {
    // threads beyond the mesh repeat its last DoF and store nothing
    const int64_t g = xcd_block_index() * bs + t;
    dofs[t] = (int)dof_of(a, g < a.n ? g : a.n - 1);
  }
  __syncthreads();
  const int w = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  double* const sc = scr + (S::R > 0 ? w * S::R * S::row_bytes / 8 : 0);
  // item k: direction 1 + k / G of group (k + k / G) mod G
  struct Item {
    int al, at;
    int64_t i;
    DepRec<D, T> rec;
    int widx;
  };
  const auto fetch = [&](int k) {
    Item it;
    it.al = 1 + k / G;
    it.at = ((k + k / G) % G) * 64 + lane;
    it.i = dofs[it.at];
    it.rec = load_rec<D, T>(a, (int64_t)(it.al - 1) * a.n + it.i);
    it.widx = a.wall_idx ? a.wall_idx[it.i] : -1;
    return it;
  };
  const auto stream = [&](const Item& it) {
    const unsigned wmask = it.widx >= 0 ? a.wall_flip[it.widx] : 0u;
    col[it.al - 1][it.at] = gen_direction<D, Q, P, T, S::zu, S::R>(a, dgl, sc, it.i, it.al, it.widx, wmask, it.rec);
  };
  constexpr int NI = G * (Q - 1);
  if constexpr (S::prefetch) {
    // the next item's record is loaded before this item's gathers, so its latency overlaps them
    Item it = fetch(w < NI ? w : 0);
#pragma unroll 1
    for (int k = w; k < NI; k += W) {
      Item next = it;
      if (k + W < NI) next = fetch(k + W);
      stream(it);
      it = next;
    }
  } else {
#pragma unroll 1
    for (int k = w; k < NI; k += W) stream(fetch(k));
  }
  __syncthreads();
  if (w >= G) return;
  // wave w collides group w
  const int64_t g = xcd_block_index() * bs + t;
  if (g >= a.n) return;
  const int64_t i = dofs[t];
  T fs[Q];
  fs[0] = a.fin[i];
#pragma unroll
  for (int al = 1; al < Q; al++) fs[al] = col[al - 1][t];
  if (write_macro & STEP_STREAM_ONLY) {  // the SL stream with its wall values (CFDSolver::stream)
#pragma unroll
    for (int q = 0; q < Q; q++) a.fout[(int64_t)q * a.stride + i] = fs[q];
    return;
  }
  bgk_collide_store_pairs<Q, T>(fs, ca, i, (write_macro & STEP_MACRO) != 0, a.fout, a.stride);
}

template <int D, int Q, int P, typename T, bool WIDE>
static int launch_general_shape(nat_ctx* ctx, const GeneralArgs<T>& a, const CollideArgs<T>& ca, int wm) {
  using S = GeneralShape<D, Q, P, T, WIDE>;
  hipLaunchKernelGGL((k_sl_general<D, Q, P, T, WIDE>), dim3((unsigned)((a.n + S::bs - 1) / S::bs)), dim3(S::nt), 0,
                     ctx->stream, a, ca, wm);
  NAT_HIP(hipGetLastError());
  return 0;
}

// The wide form when the caller chose it, or the autotuner (FP32 3D), or by default up to 5/2
// blocks per CU, where the other form leaves a SIMD with few waves (figures at GeneralShape; FP32
// 460 blocks: equal; 887: 73 us against 74; FP64 516 blocks: 11.4 against 9.5; 920: 41 against 44).
template <int D, int Q, int P, typename T>
static bool wide_form(const nat_ctx* ctx, int64_t n) {
  if (ctx->form_pref >= 0) return ctx->form_pref == 1;
  if (sizeof(T) == 4 && D == 3 && ctx->gen_pref >= 0) return ctx->gen_pref == 1;
  constexpr int bs = GeneralShape<D, Q, P, T, true>::bs;
  return 2 * ((n + bs - 1) / bs) <= 5 * (int64_t)ctx->n_cu;
}

template <int D, int Q, int P, typename T>
static int launch_general(nat_ctx* ctx, const GeneralArgs<T>& a, const CollideArgs<T>& ca, int wm) {
  if (wide_form<D, Q, P, T>(ctx, a.n)) return launch_general_shape<D, Q, P, T, true>(ctx, a, ca, wm);
  return launch_general_shape<D, Q, P, T, false>(ctx, a, ca, wm);
}

// Calls f(D, Q, P) (as integral constants) for the context's instantiation.
template <typename F>
static int dispatch_dqp(nat_ctx* ctx, F&& f) {
  const int Q = ctx->Q, P = ctx->p;
#define NAT_G(DD, QQ, PP) \
  if (Q == QQ && P == PP)   \
    return f(std::integral_constant<int, DD>{}, std::integral_constant<int, QQ>{}, std::integral_constant<int, PP>{});
  NAT_G(2, 9, 1)
  NAT_G(2, 9, 2)
  NAT_G(2, 9, 3)
  NAT_G(2, 9, 4)
  NAT_G(2, 9, 5)
  NAT_G(2, 9, 6)
  NAT_G(3, 19, 1)
  NAT_G(3, 19, 2)
  NAT_G(3, 19, 3)
  NAT_G(3, 19, 4)
  NAT_G(3, 19, 6)
  NAT_G(3, 27, 1)
  NAT_G(3, 27, 2)
  NAT_G(3, 27, 3)
  NAT_G(3, 27, 4)
  NAT_G(3, 27, 6)
#undef NAT_G
  ctx->err = "general SL kernel not instantiated for this (stencil, order)";
  return NAT_ERR_UNSUPPORTED;
}

template <typename T>
static int dispatch_general(nat_ctx* ctx, const GeneralArgs<T>& a, const CollideArgs<T>& ca, int wm) {
  return dispatch_dqp(ctx, [&](auto d, auto q, auto p) {
    return launch_general<decltype(d)::value, decltype(q)::value, decltype(p)::value, T>(ctx, a, ca, wm);
  });
}

template <typename T>
static void fill_general(nat_ctx* ctx, GeneralArgs<T>& a) {
  const int src = ctx->cur, dst = 1 - ctx->cur;
  a.fin = (const T*)ctx->f[src];
  a.fout = (T*)ctx->f[dst];
  a.stride = ctx->stride;
  a.n = ctx->n_dofs;
  for (int d = 0; d < 3; d++) {
    a.nfe[d] = ctx->nfe[d];
    a.N[d] = d < ctx->D ? ctx->desc.ncells[d] : 1;
  }
  a.divN0.set((uint32_t)a.N[0]);
  a.divN1.set((uint32_t)a.N[1]);
  a.rows = 0;
  if (a.nfe[0] >= 3 && a.n % a.nfe[0] == 0) {
    a.rows = a.n / a.nfe[0];
    a.divM.set((uint32_t)(a.nfe[0] - 2));
    a.divG.set((uint32_t)(64 * a.nfe[0]));
  }
  a.cell = ctx->dep_cell;
  a.xi = ctx->dep_xi64;
  a.rec = ctx->dep_rec32;
  a.dir_bytes = (int)(ctx->stride * (int64_t)sizeof(T));
  a.wall_idx = ctx->has_walls ? ctx->wall_idx : nullptr;
  a.wall_flip = ctx->wall_flip;
  a.wall_bias = ctx->wall_bias;
  double x[MAXP + 1], w[MAXP + 1];
  gll_points(ctx->p, x, w);
  for (int j = 0; j <= MAXP; j++) {
    a.gll[j] = j <= ctx->p ? x[j] : 0.0;
    double d = 1;
    for (int m = 0; m <= ctx->p; m++)
      if (m != j && j <= ctx->p) d *= (x[j] - x[m]);
    a.inv_den[j] = j <= ctx->p ? 1.0 / d : 0.0;
  }
  for (int j = 0; j <= MAXP; j++)
    for (int k = 0; k <= MAXP; k++) a.dgl[j][k] = (j <= ctx->p && k <= ctx->p) ? (x[j] - x[k]) : 0.0;
}

}  // namespace nat

namespace {

// One fused step from f[cur] into f[1 - cur], without advancing cur.
int general_launch(nat_ctx* ctx, int write_macro) {
  using namespace nat;
  if (ctx->stride * (int64_t)(ctx->fp32 ? 4 : 8) > INT32_MAX) {
    ctx->err = "general backend: one direction's array exceeds 2 GiB";
    return NAT_ERR_UNSUPPORTED;
  }
  if (ctx->fp32) {
    GeneralArgs<float> a;
    fill_general<float>(ctx, a);
    CollideArgs<float> ca;
    ca.omega = (float)(1.0 / ctx->tau);
    ca.omega64 = 1.0 / ctx->tau;
    ca.rho0 = (float)(ctx->desc.rho0 > 0 ? ctx->desc.rho0 : 1.0);
    ca.scaling = ctx->st.s;
    ca.rho = (float*)ctx->rho;
    ca.u = (float*)ctx->u;
    ca.mstride = ctx->n_store;
    ca.status = ctx->d_status;
    ca.stab = ctx->stab_on();
    return dispatch_general<float>(ctx, a, ca, write_macro);
  }
  GeneralArgs<double> a;
  fill_general<double>(ctx, a);
  CollideArgs<double> ca;
  ca.omega = 1.0 / ctx->tau;
  ca.omega64 = 1.0 / ctx->tau;
  ca.rho0 = 0.0;
  ca.scaling = ctx->st.s;
  ca.rho = (double*)ctx->rho;
  ca.u = (double*)ctx->u;
  ca.mstride = ctx->n_store;
  ca.status = ctx->d_status;
  ca.stab = ctx->stab_on();
  return dispatch_general<double>(ctx, a, ca, write_macro);
}

struct GenKey {
  int Q, p, walls;
  int64_t n;
  bool operator<(const GenKey& o) const {
    return std::tie(Q, p, walls, n) < std::tie(o.Q, o.p, o.walls, o.n);
  }
};
std::mutex g_gen_mutex;
std::map<GenKey, int> g_gen_cache;

}  // namespace

// Form of the step: 0 W = 2 G waves per block, 1 the wide form (-1: no kernel for the context).
int nat_general_form(nat_ctx* ctx) {
  int form = -1;
  nat::dispatch_dqp(ctx, [&](auto d, auto q, auto p) {
    constexpr int D = decltype(d)::value, Q = decltype(q)::value, P = decltype(p)::value;
    form = ctx->fp32 ? nat::wide_form<D, Q, P, float>(ctx, ctx->n_dofs) : nat::wide_form<D, Q, P, double>(ctx, ctx->n_dofs);
    return 0;
  });
  return form;
}

int nat_launch_sl_general(nat_ctx* ctx, int write_macro) {
  const int rc = general_launch(ctx, write_macro);
  if (rc == 0) ctx->cur = 1 - ctx->cur;
  return rc;
}

// Form of the general SL kernel picked by measurement. FP32 3D contexts have two (eight
// or sixteen waves per block): each is timed for nsteps steps on the context's own mesh,
// writing the idle ping-pong buffer (populations, fields and time stay as they were), and the
// faster is kept for this context and, process-wide, for later contexts of the same
// instantiation and DoF count. Both forms run the same arithmetic in the same order, so
// results do not depend on the choice. tile receives the chosen form's DoFs per block, waves
// per SIMD it is built for, and z-planes of source rows loaded together.
int nat_internal_autotune_general(nat_ctx* ctx, int nsteps, int* tile, double* best_us) {
  using namespace nat;
  if (!ctx->assembled) return NAT_ERR_STATE;
  if (best_us) *best_us = 0;
  if (ctx->fp32 && ctx->D == 3) {
    const GenKey key{ctx->Q, ctx->p, ctx->has_walls ? 1 : 0, ctx->n_dofs};
    int cached = -1;
    {
      std::lock_guard<std::mutex> lk(g_gen_mutex);
      auto it = g_gen_cache.find(key);
      if (it != g_gen_cache.end()) cached = it->second;
    }
    if (cached >= 0) {
      ctx->gen_pref = cached;
    } else {
      if (nsteps < 1) nsteps = 10;
      hipEvent_t e0 = nullptr, e1 = nullptr;
      NAT_HIP(hipEventCreate(&e0));
      if (hipEventCreate(&e1) != hipSuccess) {
        (void)hipEventDestroy(e0);
        ctx->err = "hipEventCreate failed";
        return NAT_ERR_HIP;
      }
      int best = -1, rc = 0;
      float best_ms = 0;
      for (int pref = 0; pref < 2 && !rc; pref++) {
        ctx->gen_pref = pref;
        for (int s = 0; s < 2 && !rc; s++) rc = general_launch(ctx, 0);
        if (rc) break;
        if (hipEventRecord(e0, ctx->stream) != hipSuccess) {
          ctx->err = "autotune timing events failed";
          rc = NAT_ERR_HIP;
          break;
        }
        for (int s = 0; s < nsteps && !rc; s++) rc = general_launch(ctx, 0);
        if (rc) break;
        float ms = 0;
        if (hipEventRecord(e1, ctx->stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
            hipEventElapsedTime(&ms, e0, e1) != hipSuccess) {
          ctx->err = "autotune timing events failed";
          rc = NAT_ERR_HIP;
          break;
        }
        if (best < 0 || ms < best_ms) {
          best = pref;
          best_ms = ms;
        }
      }
      (void)hipEventDestroy(e0);
      (void)hipEventDestroy(e1);
      if (rc) {
        ctx->gen_pref = -1;
        return rc;
      }
      ctx->gen_pref = best;
      if (best_us) *best_us = 1e3 * best_ms / nsteps;
      std::lock_guard<std::mutex> lk(g_gen_mutex);
      g_gen_cache[key] = best;
    }
  }
  return dispatch_dqp(ctx, [&](auto d, auto q, auto p) {
    constexpr int D = decltype(d)::value, Q = decltype(q)::value, P = decltype(p)::value;
    auto put = [&](auto shape) {
      using S = decltype(shape);
      tile[0] = S::bs;
      tile[1] = S::waves;
      tile[2] = S::zu;
    };
    if (ctx->fp32) {
      if (wide_form<D, Q, P, float>(ctx, ctx->n_dofs))
        put(GeneralShape<D, Q, P, float, true>{});
      else
        put(GeneralShape<D, Q, P, float, false>{});
    } else {
      if (wide_form<D, Q, P, double>(ctx, ctx->n_dofs))
        put(GeneralShape<D, Q, P, double, true>{});
      else
        put(GeneralShape<D, Q, P, double, false>{});
    }
    return 0;
  });
}
