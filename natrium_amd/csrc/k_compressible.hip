// Compressible populations (f, g) with the quartic Hermite equilibrium and FP64
// temperature: SL streaming of both sets with one set of weights, fused with the
// compressible BGK collision.
//
// Collision semantics (per node, FP64), following
// collision_advanced/CollisionOperator.h:113-224, CollisionSchemes.h:43-118 and
// AuxiliaryCollisionFunctions.h:290-307,421-431:
//   rho = sum f, u = sum e f / rho (unscaled e)
//   T   = 1/2 sum_i [ |e_i - u|^2 f_i / cs2 + g_i ] / (rho C_v),  C_v = 1/(gamma-1)
//   f_eq = quartic Hermite polynomial (Equilibria.h:120-267), g_eq = f_eq T (2 C_v - D)
//   tau_v = (tau - 1/2) S(T) / (T rho) + 1/2, S = (T/0.85)^0.7 with Sutherland's law
//   optional Prandtl number: f* = w Q:(e e e - 3 cs2 e I)/(6 cs2^3), g* = w F.e / T
//   f -= omega_v (f - f_eq) - (omega_v - omega_p) f*;  g likewise with g_eq, g*
//   Knudsen estimate sum |f - f_eq| / w / Q written as the shock-sensor field.
// The per-direction constants (unscaled e, w, |e|^2, the independent H3 and H4
// components) come from a small FP64 table read with uniform addresses.
//
// FP32 storage keeps f~ = f - w rho0 and g~ = g - w rho0 (2 C_v - D), the
// equilibria at rest with T = 1; the collision un-shifts in FP64.
#include "nat_collide.hpp"
#include "nat_fastdiv.hpp"
#include "nat_offsets.hpp"

int nat_comp_form(const nat_ctx* ctx, int form = -1);

namespace nat {

constexpr int CTAB = 16;  // doubles per direction in the constant table
enum { CT_E0 = 0, CT_E1 = 1, CT_W = 2, CT_EE = 3, CT_H3 = 4, CT_H4 = 8, CT_IW = 13 };

template <typename T>
struct CompArgs {
  const T* fin;
  const T* gin;
  T* fout;
  T* gout;
  int64_t stride;
  int64_t n;
  int nfe[3];
  int N[3];
  FastDivU divN0;  // division by N[0]
  const int* cell;    // [(alpha-1) * n + i] departure cell (-1: identity row)
  const double* xi;   // unit coordinates, 2 per record
  const int* wall_idx;        // walls: wall entry per DoF or -1 (null: no walls)
  const unsigned* wall_flip;  //   per entry: bit alpha set when alpha reads the opposite direction
  const double* wall_bias;    //   per entry: Q values added to f after interpolation
  int opp[MAXQ];              // opposite direction index
  double gll[MAXP + 1];
  double inv_den[MAXP + 1];
  double cs2;         // unscaled c_s^2
  double ics2;        // 1 / cs2
  double k3, k4;      // 1 / (6 cs2^3), 1 / (24 cs2^4)
  double cv;          // C_v = 1 / (gamma - 1)
  double tau;
  double gamma;
  double prandtl;
  int prandtl_set;
  int sutherland;
  double rho0;        // FP32 shift of f (0 for FP64)
  double gshift;      // FP32 shift factor of g: w rho0 (2 C_v - D)
  double scaling;
  T* rho;
  T* u;
  double* temp;
  double* mask;
  int64_t mstride;
  int* status;
  int stream_only;  // CompressibleCFDSolver::stream alone: store the streamed f and g, no collision
};

// Quartic equilibrium of direction q for the node scalars (2D). The node factors
// (powers of 1/cs2 and rho) are folded into the Hermite coefficients once per node,
// so a direction costs multiply-adds only (no divisions).
struct QuarticNode {
  double rho, us0, us1, uu_term, k2a, k2b;
  double b_xxx, b_xxy, b_xyy, b_yyy, b_xxxx, b_yyyy, b_xxxy, b_xyyy, b_xxyy;
  template <typename T>
  __device__ void init(double r, double x, double y, double T_, const CompArgs<T>& a) {
    const double cs2 = a.cs2, ics2 = a.ics2;
    rho = r;
    us0 = x * ics2;
    us1 = y * ics2;
    uu_term = -(x * x) * (0.5 * ics2) - (y * y) * (0.5 * ics2);
    const double Tm1 = T_ - 1;
    // rho w (Tm1 |e|^2 - 2 cs2 Tm1) / (2 cs2)
    k2a = r * Tm1 * (0.5 * ics2);
    k2b = r * Tm1;
    const double T1 = cs2 * (T_ - 1);
    const double r3 = r * a.k3, r4 = r * a.k4;
    b_xxx = r3 * (x * x * x + T1 * (x + x + x));
    b_xxy = 3.0 * r3 * (x * x * y + T1 * y);
    b_xyy = 3.0 * r3 * (x * y * y + T1 * x);
    b_yyy = r3 * (y * y * y + T1 * (y + y + y));
    b_xxxx = r4 * (x * x * x * x + T1 * x * x * 6.0 + T1 * T1 * 3.0);
    b_yyyy = r4 * (y * y * y * y + T1 * y * y * 6.0 + T1 * T1 * 3.0);
    b_xxxy = 4.0 * r4 * (x * x * x * y + T1 * (x * y * 3.0));
    b_xyyy = 4.0 * r4 * (x * y * y * y + T1 * (x * y * 3.0));
    b_xxyy = 6.0 * r4 * (x * x * y * y + T1 * (x * x + y * y) + T1 * T1);
  }
  __device__ double feq(const double* __restrict__ t) const {
    const double ue = us0 * t[CT_E0] + us1 * t[CT_E1];
    double f = rho * (1 + ue * (1 + 0.5 * ue) + uu_term);
    f += k2a * t[CT_EE] - k2b;
    f += b_xxx * t[CT_H3 + 0] + b_xxy * t[CT_H3 + 1] + b_xyy * t[CT_H3 + 2] + b_yyy * t[CT_H3 + 3];
    f += b_xxxx * t[CT_H4 + 0] + b_yyyy * t[CT_H4 + 1] + b_xxyy * t[CT_H4 + 2] + b_xyyy * t[CT_H4 + 3] +
         b_xxxy * t[CT_H4 + 4];
    return t[CT_W] * f;
  }
};

// Node state of the compressible collision: moments, temperature, equilibrium
// coefficients and relaxation rates.
struct CompNode {
  double rho, u0, u1, temp, itemp, gfac, om_v, om_diff;
  QuarticNode qn;
};

// Node state from complete sums: rho, u, and tf = sum |e - u|^2 f, tg = sum g.
template <typename T>
__device__ __forceinline__ CompNode comp_node_sums(double rho, double u0, double u1, double tf, double tg,
                                                   const CompArgs<T>& a) {
  constexpr int D = 2;
  const double C_v = a.cv;
  CompNode nd;
  const double temp = (tf * a.ics2 + tg) * 0.5 / (rho * C_v);
  nd.rho = rho;
  nd.u0 = u0;
  nd.u1 = u1;
  nd.temp = temp;
  nd.itemp = 1.0 / temp;
  nd.qn.init(rho, u0, u1, temp, a);
  nd.gfac = temp * (2.0 * C_v - D);
  double S = 1.0;
  if (a.sutherland) S = pow(temp / 0.85, 0.7);
  const double visc_tau = (a.tau - 0.5) * S / (temp * rho) + 0.5;
  const double prandtl_tau = (visc_tau - 0.5) / (a.prandtl_set ? a.prandtl : 1.0) + 0.5;
  nd.om_v = 1. / visc_tau;
  nd.om_diff = nd.om_v - 1. / prandtl_tau;
  return nd;
}

// Sums over directions of the non-equilibrium parts: the Knudsen estimate and, with
// a Prandtl number (PR), the third moments Q of f_neq and first moments F of g_neq
// about u.
struct CompNeq {
  double kn = 0;
  double Qt[2][2][2] = {{{0, 0}, {0, 0}}, {{0, 0}, {0, 0}}};
  double Fg[2] = {0, 0};
};

// Adds direction t's terms; returns its f_eq.
template <bool PR, typename T>
__device__ __forceinline__ double comp_neq_add(CompNeq& s, const CompNode& nd, const CompArgs<T>& a,
                                               const double* __restrict__ t, double fq, double gq) {
  const double fe = nd.qn.feq(t);
  const double fneq = fq - fe;
  s.kn += fabs(fneq) * t[CT_IW];
  if (PR && a.prandtl_set) {
    const double gneq = gq - fe * nd.gfac;
    const double d[2] = {t[CT_E0] - nd.u0, t[CT_E1] - nd.u1};
    for (int x = 0; x < 2; x++)
      for (int y = 0; y < 2; y++)
        for (int z = 0; z < 2; z++) s.Qt[x][y][z] += (d[x] * d[y] * d[z]) * fneq;
    s.Fg[0] += d[0] * gneq;
    s.Fg[1] += d[1] * gneq;
  }
  return fe;
}

// Relaxed f and g of direction t, given its f_eq and the complete sums s.
template <bool PR, typename T>
__device__ __forceinline__ void comp_relax(const CompNode& nd, const CompNeq& s, const CompArgs<T>& a,
                                           const double* __restrict__ t, double fe, double fq, double gq, double& fn,
                                           double& gn) {
  const double cs2 = a.cs2;
  const double ge = fe * nd.gfac;
  double fstar = 0, gstar = 0;
  if (PR && a.prandtl_set) {
    // w Q:(e e e - 3 cs2 e I) / (6 cs2^3) with 1 / (6 cs2^3) = k3
    const double e[2] = {t[CT_E0], t[CT_E1]};
    double acc = 0;
    for (int x = 0; x < 2; x++)
      for (int y = 0; y < 2; y++)
        for (int z = 0; z < 2; z++) acc += s.Qt[x][y][z] * (e[x] * e[y] * e[z] - 3 * cs2 * e[z] * (x == y ? 1.0 : 0.0));
    fstar = t[CT_W] * acc * a.k3;
    gstar = t[CT_W] * (s.Fg[0] * e[0] + s.Fg[1] * e[1]) * nd.itemp;
  }
  fn = fq - (nd.om_v * (fq - fe) - nd.om_diff * fstar);
  gn = gq - (nd.om_v * (gq - ge) - nd.om_diff * gstar);
}

template <typename T>
__device__ __forceinline__ void comp_write_macro(const CompArgs<T>& a, const CompNode& nd, double kn_sum, int Q,
                                                 int64_t node) {
  a.rho[node] = (T)nd.rho;
  a.u[node] = (T)(nd.u0 * a.scaling);
  a.u[a.mstride + node] = (T)(nd.u1 * a.scaling);
  a.temp[node] = nd.temp;
  a.mask[node] = kn_sum / Q;
}

template <int P>
__device__ __forceinline__ void lag_all(const double (&x)[MAXP + 1], const double (&inv)[MAXP + 1], double xi,
                                        double (&v)[P + 1]) {
#pragma unroll
  for (int j = 0; j <= P; j++) {
    double s = inv[j];
#pragma unroll
    for (int m = 0; m <= P; m++)
      if (m != j) s *= (xi - x[m]);
    v[j] = s;
  }
}

// A departure record: cell (-1: identity row) and unit coordinates.
struct CompRec {
  int c;
  double xi0, xi1;
};

template <typename T>
__device__ __forceinline__ CompRec comp_record(const CompArgs<T>& a, int al, int64_t i) {
  const int64_t r = (int64_t)(al - 1) * a.n + i;
  const double2 x = reinterpret_cast<const double2*>(a.xi)[r];
  return {a.cell[r], x.x, x.y};
}

// Buffer resource from a direction's array on, for 32-bit byte offsets (uniform base). The rows of
// a direction and of its opposite are read from the lower one's array on, which takes arrays of at
// most 4/3 GiB (pair_offsets_fit, opposite directions are two arrays apart; in FP64 178,956,970
// DoFs, 241 GB of context). The stores stay within one array, below 2 GiB on any mesh whose
// populations and records fit the device.
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t comp_rsrc(const T* p) {
  const uint64_t pb = (uint64_t)p;
  const uint32_t phi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(pb >> 32));
  const uint32_t plo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)pb);
  return __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)phi << 32) | (uint64_t)plo), (short)0,
                                           (int)0xffffffffu, 0x00020000);
}

// Store to p[i] (p uniform), written through to the device (sc1): a wave stores whole lines, and
// the output leaves the caches while the kernel runs instead of in the write-back at its end
// (us per step, FP32 and FP64: p=2 128^2 25.9 -> 24.9, 26.2 -> 26.0; 64^2 11.3 -> 11.1,
// 12.8 -> 11.7; p=3 64^2 18.2 -> 17.8, 22.5 -> 21.2; beyond the Infinity Cache, p=2 256^2,
// 60.9 -> 60.4, 89 -> 91.5).
template <typename T>
__device__ __forceinline__ void comp_store(T* p, int64_t i, T v) {
  const int off = (int)((unsigned)i * (unsigned)sizeof(T));
  if constexpr (sizeof(T) == 4)
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), comp_rsrc(p), off, 0, 16);
  else
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(unsigned __attribute__((ext_vector_type(2))), v),
                                          comp_rsrc(p), off, 0, 16);
}

// A row of P + 1 values in the fewest loads of 16, 12, 8 and 4 bytes.
template <int P, typename T>
__device__ __forceinline__ void comp_row(__amdgpu_buffer_rsrc_t r, int off, T (&v)[P + 1]) {
  constexpr int W = (int)sizeof(T) / 4, ND = (P + 1) * W;
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
      v[m] = __builtin_bit_cast(float, q[m]);
    else
      v[m] = __builtin_bit_cast(double, ((unsigned long)q[2 * m + 1] << 32) | q[2 * m]);
  }
}

__device__ __forceinline__ double comp_min_abs(double a, double b) {
  double r;
  asm("v_min_f64 %0, |%1|, |%2|" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// Streamed f and g of direction al at DoF i (al uniform across the wave), with the
// FP32 shift added back. One set of FP64 weights serves f and g. The stencil's rows are loaded
// whole; where a product weight is under the cut-off (on the Cartesian meshes every lane of the
// directions along an axis) the terms are dropped by selects, not by branches around their loads.
// Lanes whose path was reflected at a wall read the opposite direction's array.
// FAR: arrays beyond the 32-bit offsets, read through 64-bit addresses instead.
template <int Q, int P, typename T, bool FAR>
__device__ __forceinline__ void comp_stream_dir(const CompArgs<T>& a, const double* __restrict__ tab, int64_t i,
                                                int al, int widx, unsigned wmask, const CompRec& rec, double& fo,
                                                double& go) {
  const int n0 = a.nfe[0];
  const bool flip = (wmask >> al) & 1u;
  const double bias = widx >= 0 ? a.wall_bias[(int64_t)widx * Q + al] : 0.0;
  const int c = rec.c;
  double af, ag;
  if (c < 0) {
    af = (double)a.fin[(int64_t)al * a.stride + i];
    ag = (double)a.gin[(int64_t)al * a.stride + i];
  } else {
    double lx[P + 1], ly[P + 1];
    lag_all<P>(a.gll, a.inv_den, rec.xi0, lx);
    lag_all<P>(a.gll, a.inv_den, rec.xi1, ly);
    const int cy = (int)a.divN0.div((uint32_t)c), cx = c - cy * a.N[0];
    const int base = cx * P + n0 * (cy * P);
    af = 0;
    ag = 0;
    // one resource over the direction and its opposite: a reflected lane adds their distance
    const int sd = flip ? a.opp[al] : al, lo = al < a.opp[al] ? al : a.opp[al];
    const __amdgpu_buffer_rsrc_t rf = comp_rsrc(a.fin + (int64_t)lo * a.stride),
                                 rg = comp_rsrc(a.gin + (int64_t)lo * a.stride);
    const unsigned src = (unsigned)(sd - lo) * (unsigned)(a.stride * (int64_t)sizeof(T));
    double mnx = comp_min_abs(lx[0], lx[1]), mny = comp_min_abs(ly[0], ly[1]);
#pragma unroll
    for (int m = 2; m <= P; m++) {
      mnx = comp_min_abs(mnx, lx[m]);
      mny = comp_min_abs(mny, ly[m]);
    }
    const bool cut = __any(!(mnx * mny >= 1e-10));
    constexpr int R = P <= 3 ? P + 1 : 2;  // rows in flight at a time (p = 4, all 5: 208 VGPRs, 96^2 84 us, not 67)
    static_for<0, (P + R) / R>([&](auto G) {
      constexpr int y0 = decltype(G)::value * R, ny = P + 1 - y0 < R ? P + 1 - y0 : R;
      T vf[ny][P + 1], vg[ny][P + 1];
#pragma unroll
      for (int y = 0; y < ny; y++) {
        if constexpr (FAR) {
          const int64_t k = (int64_t)sd * a.stride + base + n0 * (y0 + y);
#pragma unroll
          for (int m = 0; m <= P; m++) {
            vf[y][m] = a.fin[k + m];
            vg[y][m] = a.gin[k + m];
          }
        } else {
          const int off = (int)(src + (unsigned)(base + n0 * (y0 + y)) * (unsigned)sizeof(T));
          comp_row<P, T>(rf, off, vf[y]);
          comp_row<P, T>(rg, off, vg[y]);
        }
      }
      if (!cut) {
        // no product weight reaches the cut-off: every term is taken
#pragma unroll
        for (int y = 0; y < ny; y++)
#pragma unroll
          for (int mx = 0; mx <= P; mx++) {
            const double w = lx[mx] * ly[y0 + y];
            af = fma(w, (double)vf[y][mx], af);
            ag = fma(w, (double)vg[y][mx], ag);
          }
      } else {
#pragma unroll
        for (int y = 0; y < ny; y++)
#pragma unroll
          for (int mx = 0; mx <= P; mx++) {
            const double w = lx[mx] * ly[y0 + y];
            const bool keep = !(fabs(w) < 1e-10);
            const double sf = fma(w, (double)vf[y][mx], af), sg = fma(w, (double)vg[y][mx], ag);
            af = keep ? sf : af;
            ag = keep ? sg : ag;
          }
      }
    });
  }
  af = af + bias;
  fo = af + tab[al * CTAB + CT_W] * a.rho0;
  go = ag + tab[al * CTAB + CT_W] * a.gshift;
}

// Fused SL stream of f and g + compressible collision. The work of a block is spread
// over its waves: 64 DoFs per block, CW waves, wave w streaming and relaxing the directions
// w, w + CW, ... of those DoFs and holding their values in registers throughout (one thread per
// DoF would give a 66k-DoF grid only four waves per CU to hide its gather latency). The moments
// are summed over classes of directions, q modulo CL; the partial sums meet in LDS and are added
// in class order, so neither a repeated run nor another CW changes a bit. Every wave forms the
// node state from them and relaxes its own directions. Without a Prandtl number the equilibrium
// of a direction serves both its Knudsen term and its relaxation; with one (PR) the third moments
// must be complete first, through one more LDS reduction. Its 11-value reduction buffer allows 4
// classes only (8 would leave room for one block per CU; 128^2 p=2 with Pr = 0.71: 0.97 -> 1.60
// GLUPS FP32).
// Bound by the latency of a wave's serial chain (record, rows, sums; a step moves about 57 MB at
// 128^2 p=2 FP32, 9 us at the cache's rate), so the record of the next direction is loaded ahead
// and the rows come in whole-row loads that no branch splits. Against single loads with the cut
// terms behind branches and the values kept in LDS, us per step (FP32, FP64; walls in y):
// p=2 16^2 11.3 -> 9.6, 12.1 -> 9.3; p=2 128^2 29.2 -> 24.9, 33.0 -> 26.0; p=3 64^2 32.2 -> 17.8,
// 34.9 -> 21.2; p=2 256^2 80.2 -> 60.4, 121 -> 91.5; Pr 0.71 128^2 40.5 -> 33.1, 44.0 -> 34.3. Also
// fetching the next direction's rows ahead (156 VGPRs) is faster on 128^2 FP32 without walls
// (25.1 -> 22.7) and slower elsewhere.
template <bool PR>
constexpr int comp_classes() {
  return PR ? 4 : 8;
}
// ST = false: no streaming, each DoF's own populations are collided in place (the
// initial collision of CFDSolver::run; fin and fout may be the same arrays, since every
// value is read before it is written and only this block touches its 64 DoFs).
template <int Q, int P, typename T, bool PR, bool ST = true, int CW = comp_classes<PR>(), bool FAR = false>
__global__ __launch_bounds__(CW * 64) void k_sl_comp_wide(CompArgs<T> a, const double* __restrict__ tab,
                                                          int write_macro) {
  constexpr int CL = comp_classes<PR>(), NC = CL / CW;  // a wave holds NC classes
  constexpr int NK = (Q + CW - 1) / CW;  // directions of a wave, the last of them of the first waves only
  constexpr int NV = PR ? 11 : 5;  // kn, Q (8), F (2); moments: rho, j (3) + tf, tg (2)
  __shared__ double red[CL][NV][64];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t i = (int64_t)blockIdx.x * 64 + lane;
  const bool live = i < a.n;
  int widx = -1;
  unsigned wmask = 0;
  if (ST && live && a.wall_idx) {
    widx = a.wall_idx[i];
    if (widx >= 0) wmask = a.wall_flip[widx];
  }
  // stream only (uniform over the grid): each wave stores the directions it streamed
  const bool so = ST && a.stream_only;
  double fv[NK], gv[NK];
  // calls f(k, q) for the wave's k-th direction q
  const auto each = [&](auto&& f) {
    static_for<0, NK>([&](auto K) {
      constexpr int k = decltype(K)::value;
      const int q = w + k * CW;
      if ((k + 1) * CW <= Q || q < Q) f(K, q);  // uniform
    });
  };
  if (live) {
    CompRec next{};
    if constexpr (ST) next = comp_record<T>(a, w > 0 ? w : CW, i);  // (direction 0 has no record)
    each([&](auto K, int q) {
      constexpr int k = decltype(K)::value;
      if (ST && q > 0) {
        const CompRec rec = next;  // the next direction's record is loaded ahead of this one's stencil
        if (q + CW < Q) next = comp_record<T>(a, q + CW, i);
        comp_stream_dir<Q, P, T, FAR>(a, tab, i, q, widx, wmask, rec, fv[k], gv[k]);
        if (so) {
          a.fout[(int64_t)q * a.stride + i] = (T)(fv[k] - tab[q * CTAB + CT_W] * a.rho0);
          a.gout[(int64_t)q * a.stride + i] = (T)(gv[k] - tab[q * CTAB + CT_W] * a.gshift);
        }
      } else {
        const T f = a.fin[(int64_t)q * a.stride + i], g = a.gin[(int64_t)q * a.stride + i];
        if (so) {
          a.fout[(int64_t)q * a.stride + i] = f;
          a.gout[(int64_t)q * a.stride + i] = g;
        }
        fv[k] = (double)f + tab[q * CTAB + CT_W] * a.rho0;
        gv[k] = (double)g + tab[q * CTAB + CT_W] * a.gshift;
      }
    });
  }
  if (so) return;
  // moments: each wave sums its own classes; partial sums meet in LDS, added in class order
  double m[NC][3] = {};
  if (live)
    each([&](auto K, int q) {
      constexpr int k = decltype(K)::value, c = k % NC;
      m[c][0] += fv[k];
      m[c][1] += tab[q * CTAB + CT_E0] * fv[k];
      m[c][2] += tab[q * CTAB + CT_E1] * fv[k];
    });
#pragma unroll
  for (int c = 0; c < NC; c++)
#pragma unroll
    for (int d = 0; d < 3; d++) red[w + c * CW][d][lane] = m[c][d];
  __syncthreads();
  double rho = red[0][0][lane], j0 = red[0][1][lane], j1 = red[0][2][lane];
  for (int v = 1; v < CL; v++) {
    rho += red[v][0][lane];
    j0 += red[v][1][lane];
    j1 += red[v][2][lane];
  }
  const double u0 = j0 * (1.0 / rho), u1 = j1 * (1.0 / rho);
  double mt[NC][2] = {};
  if (live)
    each([&](auto K, int q) {
      constexpr int k = decltype(K)::value, c = k % NC;
      const double d0 = tab[q * CTAB + CT_E0] - u0, d1 = tab[q * CTAB + CT_E1] - u1;
      mt[c][0] += (d0 * d0 + d1 * d1) * fv[k];
      mt[c][1] += gv[k];
    });
#pragma unroll
  for (int c = 0; c < NC; c++)
#pragma unroll
    for (int d = 0; d < 2; d++) red[w + c * CW][3 + d][lane] = mt[c][d];
  __syncthreads();
  double tf = red[0][3][lane], tg = red[0][4][lane];
  for (int v = 1; v < CL; v++) {
    tf += red[v][3][lane];
    tg += red[v][4][lane];
  }
  CompNode nd = {};
  if (live) nd = comp_node_sums<T>(rho, u0, u1, tf, tg, a);
  if (w == 0 && live && !(nd.rho >= 1e-10)) atomicOr(a.status, 1);
  auto store = [&](int q, double fn, double gn) {
    comp_store(a.fout + (int64_t)q * a.stride, i, (T)(fn - tab[q * CTAB + CT_W] * a.rho0));
    comp_store(a.gout + (int64_t)q * a.stride, i, (T)(gn - tab[q * CTAB + CT_W] * a.gshift));
  };
  CompNeq s;
  if constexpr (PR) {
    static_assert(NC == 1, "one class per wave");
    if (live)
      each([&](auto K, int q) {
        comp_neq_add<true, T>(s, nd, a, tab + q * CTAB, fv[decltype(K)::value], gv[decltype(K)::value]);
      });
    __syncthreads();  // every wave has read the moment sums
    red[w][0][lane] = s.kn;
#pragma unroll
    for (int k = 0; k < 8; k++) red[w][1 + k][lane] = s.Qt[k >> 2][(k >> 1) & 1][k & 1];
    red[w][9][lane] = s.Fg[0];
    red[w][10][lane] = s.Fg[1];
    __syncthreads();
    CompNeq t;
    t.kn = red[0][0][lane];
#pragma unroll
    for (int k = 0; k < 8; k++) t.Qt[k >> 2][(k >> 1) & 1][k & 1] = red[0][1 + k][lane];
    t.Fg[0] = red[0][9][lane];
    t.Fg[1] = red[0][10][lane];
    for (int v = 1; v < CL; v++) {
      t.kn += red[v][0][lane];
#pragma unroll
      for (int k = 0; k < 8; k++) t.Qt[k >> 2][(k >> 1) & 1][k & 1] += red[v][1 + k][lane];
      t.Fg[0] += red[v][9][lane];
      t.Fg[1] += red[v][10][lane];
    }
    if (live)
      each([&](auto K, int q) {
        const double* tq = tab + q * CTAB;
        double fn, gn;
        comp_relax<true, T>(nd, t, a, tq, nd.qn.feq(tq), fv[decltype(K)::value], gv[decltype(K)::value], fn, gn);
        store(q, fn, gn);
      });
    s.kn = t.kn;
  } else {
    CompNeq sc[NC];
    if (live)
      each([&](auto K, int q) {
        constexpr int k = decltype(K)::value;
        const double* tq = tab + q * CTAB;
        const double fe = comp_neq_add<false, T>(sc[k % NC], nd, a, tq, fv[k], gv[k]);
        double fn, gn;
        comp_relax<false, T>(nd, sc[k % NC], a, tq, fe, fv[k], gv[k], fn, gn);
        store(q, fn, gn);
      });
    if (write_macro) {  // uniform over the block
#pragma unroll
      for (int c = 0; c < NC; c++) red[w + c * CW][0][lane] = sc[c].kn;
      __syncthreads();
      s.kn = red[0][0][lane];
      for (int v = 1; v < CL; v++) s.kn += red[v][0][lane];
    }
  }
  if (write_macro && w == 0 && live) comp_write_macro<T>(a, nd, s.kn, Q, i);
}

static int opposite_of(const nat_ctx* ctx, int q) {
  for (int r = 0; r < ctx->Q; r++)
    if (ctx->st.dir[r][0] == -ctx->st.dir[q][0] && ctx->st.dir[r][1] == -ctx->st.dir[q][1] &&
        ctx->st.dir[r][2] == -ctx->st.dir[q][2])
      return r;
  return q;
}

template <typename T>
static void fill_comp(nat_ctx* ctx, CompArgs<T>& a, int src, int dst) {
  a.fin = (const T*)ctx->f[src];
  a.gin = (const T*)ctx->g[src];
  a.fout = (T*)ctx->f[dst];
  a.gout = (T*)ctx->g[dst];
  a.stride = ctx->stride;
  a.n = ctx->n_dofs;
  for (int d = 0; d < 3; d++) {
    a.nfe[d] = ctx->nfe[d];
    a.N[d] = d < ctx->D ? ctx->desc.ncells[d] : 1;
  }
  a.divN0.set((uint32_t)a.N[0]);
  a.cell = ctx->dep_cell;
  a.xi = ctx->dep_xi64;
  a.wall_idx = ctx->has_walls ? ctx->wall_idx : nullptr;
  a.wall_flip = ctx->wall_flip;
  a.wall_bias = ctx->wall_bias;
  for (int q = 0; q < MAXQ; q++) a.opp[q] = q < ctx->Q ? opposite_of(ctx, q) : q;
  double x[MAXP + 1], w[MAXP + 1];
  gll_points(ctx->p, x, w);
  for (int j = 0; j <= MAXP; j++) {
    a.gll[j] = j <= ctx->p ? x[j] : 0.0;
    double d = 1;
    for (int m = 0; m <= ctx->p; m++)
      if (m != j && j <= ctx->p) d *= (x[j] - x[m]);
    a.inv_den[j] = j <= ctx->p ? 1.0 / d : 0.0;
  }
  const double s = ctx->st.s;
  a.cs2 = ctx->st.cs2 / (s * s);
  a.ics2 = 1.0 / a.cs2;
  a.k3 = 1.0 / (6.0 * a.cs2 * a.cs2 * a.cs2);
  a.k4 = 1.0 / (24.0 * a.cs2 * a.cs2 * a.cs2 * a.cs2);
  a.cv = 1.0 / (ctx->desc.gamma - 1.0);
  a.tau = ctx->tau;
  a.gamma = ctx->desc.gamma;
  a.prandtl = ctx->desc.prandtl;
  a.prandtl_set = ctx->desc.prandtl > 0 ? 1 : 0;
  a.sutherland = ctx->desc.sutherland;
  const double C_v = 1. / (ctx->desc.gamma - 1.0);
  const double rho0 = ctx->fp32 ? (ctx->desc.rho0 > 0 ? ctx->desc.rho0 : 1.0) : 0.0;
  a.rho0 = rho0;
  a.gshift = rho0 * (2.0 * C_v - ctx->D);
  a.scaling = s;
  a.rho = (T*)ctx->rho;
  a.u = (T*)ctx->u;
  a.temp = ctx->T;
  a.mask = ctx->mask;
  a.mstride = ctx->n_store;
  a.status = ctx->d_status;
  a.stream_only = 0;
}

// Waves per block: 8 spread a DoF's directions over the CU while there is about a block for each
// of the 256 CUs, 4 need fewer blocks' worth of waves at the barriers when there are more. FP32
// (but for p = 3, whose registers leave one block of 8 waves per CU) gains from 8 a little longer.
// us per step with 8 / 4 waves, walls in y, FP32 and FP64:
//   p=2  66 blocks (32^2)   7.7/ 9.8   8.5/10.4      p=2 329 blocks (72^2)  11.4/11.8  14.3/13.4
//   p=2 261 blocks (64^2)  11.3/11.5  14.1/13.2      p=2 512 blocks (90^2)  13.4/13.0  16.3/15.6
//   p=3 263 blocks (43^2)  20.0/13.8  15.9/15.2      p=4 407 blocks (40^2)  16.9/17.9  21.0/20.6
//   p=3 582 blocks (64^2)  24.2/18.4  22.8/22.5      p=2 1030 blocks (128^2) 27.1/26.1 31.0/26.2
template <typename T>
constexpr unsigned comp_blocks8(int p) {
  return sizeof(T) == 4 && p != 3 ? 410 : 256;
}

template <typename T>
static int step_comp(nat_ctx* ctx, int mode) {
  CompArgs<T> a;
  const int src = ctx->cur, dst = 1 - ctx->cur;
  fill_comp<T>(ctx, a, src, dst);
  a.stream_only = (mode & STEP_STREAM_ONLY) ? 1 : 0;
  const int write_macro = (mode & STEP_MACRO) ? 1 : 0;
  const unsigned grid = (unsigned)((a.n + 63) / 64);
  const double* tab = ctx->comp_tab;
  const bool far = nat_comp_form(ctx) == 0;
  const auto launch = [&](auto PP, auto PR, auto CW, auto FAR) {
    hipLaunchKernelGGL((k_sl_comp_wide<25, decltype(PP)::value, T, decltype(PR)::value, true, decltype(CW)::value,
                                       decltype(FAR)::value>),
                       dim3(grid), dim3(decltype(CW)::value * 64), 0, ctx->stream, a, tab, write_macro);
  };
  const auto pick = [&](auto PP) {
    using std::integral_constant;
    using four = integral_constant<int, 4>;
    if (far)  // a mesh of millions of blocks (or the caller's choice)
      a.prandtl_set ? launch(PP, std::true_type{}, four{}, std::true_type{})
                    : launch(PP, std::false_type{}, four{}, std::true_type{});
    else if (a.prandtl_set)
      launch(PP, std::true_type{}, four{}, std::false_type{});
    else if (grid <= comp_blocks8<T>(decltype(PP)::value))
      launch(PP, std::false_type{}, integral_constant<int, 8>{}, std::false_type{});
    else
      launch(PP, std::false_type{}, four{}, std::false_type{});
  };
  switch (ctx->p) {
    case 1:
      pick(std::integral_constant<int, 1>{});
      break;
    case 2:
      pick(std::integral_constant<int, 2>{});
      break;
    case 3:
      pick(std::integral_constant<int, 3>{});
      break;
    case 4:
      pick(std::integral_constant<int, 4>{});
      break;
    default:
      ctx->err = "compressible SL kernel instantiated for p <= 4";
      return NAT_ERR_UNSUPPORTED;
  }
  NAT_HIP(hipGetLastError());
  ctx->cur = dst;
  return 0;
}

template <typename T>
static int collide_comp(nat_ctx* ctx) {
  CompArgs<T> a;
  fill_comp<T>(ctx, a, ctx->cur, ctx->cur);
  const unsigned grid = (unsigned)((a.n + 63) / 64);
  const double* tab = ctx->comp_tab;
  if (a.prandtl_set)
    hipLaunchKernelGGL((k_sl_comp_wide<25, 1, T, true, false>), dim3(grid), dim3(comp_classes<true>() * 64), 0,
                       ctx->stream, a, tab, 1);
  else
    hipLaunchKernelGGL((k_sl_comp_wide<25, 1, T, false, false>), dim3(grid), dim3(comp_classes<false>() * 64), 0,
                       ctx->stream, a, tab, 1);
  NAT_HIP(hipGetLastError());
  return 0;
}

}  // namespace nat

// Constant table: unscaled e, w, |e|^2 and the independent H3 / H4 components
// (AuxiliaryCollisionFunctions.h:519-566) per direction.
int nat_comp_setup(nat_ctx* ctx) {
  using namespace nat;
  if (ctx->D != 2 || ctx->Q != 25) {
    ctx->err = "compressible populations are implemented for the D2Q25H stencil";
    return NAT_ERR_UNSUPPORTED;
  }
  const double s = ctx->st.s;
  const double cs2 = ctx->st.cs2 / (s * s);
  std::vector<double> t((size_t)ctx->Q * CTAB, 0.0);
  for (int q = 0; q < ctx->Q; q++) {
    const double e[2] = {ctx->st.dir[q][0] / s, ctx->st.dir[q][1] / s};
    double* r = &t[(size_t)q * CTAB];
    r[CT_E0] = e[0];
    r[CT_E1] = e[1];
    r[CT_W] = ctx->st.w[q];
    r[CT_EE] = e[0] * e[0] + e[1] * e[1];
    auto eye = [](int a, int b) { return a == b ? 1.0 : 0.0; };
    auto H3 = [&](int a, int b, int c) {
      return e[a] * e[b] * e[c] - cs2 * (e[a] * eye(b, c) + e[b] * eye(a, c) + e[c] * eye(a, b));
    };
    auto H4 = [&](int a, int b, int c, int d) {
      const double p4 = e[a] * e[b] * e[c] * e[d];
      const double p2 = e[a] * e[b] * eye(c, d) + e[a] * e[c] * eye(b, d) + e[a] * e[d] * eye(b, c) +
                        e[b] * e[c] * eye(a, d) + e[b] * e[d] * eye(a, c) + e[c] * e[d] * eye(a, b);
      const double p0 = eye(a, b) * eye(c, d) + eye(a, c) * eye(b, d) + eye(a, d) * eye(b, c);
      return p4 - cs2 * p2 + cs2 * cs2 * p0;
    };
    r[CT_H3 + 0] = H3(0, 0, 0);
    r[CT_H3 + 1] = H3(0, 0, 1);
    r[CT_H3 + 2] = H3(0, 1, 1);
    r[CT_H3 + 3] = H3(1, 1, 1);
    r[CT_H4 + 0] = H4(0, 0, 0, 0);
    r[CT_H4 + 1] = H4(1, 1, 1, 1);
    r[CT_H4 + 2] = H4(0, 0, 1, 1);
    r[CT_H4 + 3] = H4(0, 1, 1, 1);
    r[CT_H4 + 4] = H4(0, 0, 0, 1);
    r[CT_IW] = 1.0 / ctx->st.w[q];
  }
  if (!ctx->comp_tab) NAT_HIP(hipMalloc(&ctx->comp_tab, t.size() * sizeof(double)));
  NAT_HIP(hipMemcpy(ctx->comp_tab, t.data(), t.size() * sizeof(double), hipMemcpyHostToDevice));
  return 0;
}

// Form of the compressible step: 1 with 32-bit offsets into a pair of opposite directions, 0 with
// 64-bit addresses, for arrays beyond them. form: -1 the context's choice, else whether it exists.
int nat_comp_form(const nat_ctx* ctx, int form) {
  int apart = 0;
  for (int q = 0; q < ctx->Q; q++) apart = std::max(apart, std::abs(nat::opposite_of(ctx, q) - q));
  const bool fit = nat::pair_offsets_fit(apart, ctx->stride, ctx->fp32 ? 4 : 8);
  if (form >= 0) return form == 0 || (form == 1 && fit);
  return fit && ctx->form_pref != 0 ? 1 : 0;
}

int nat_launch_sl_comp(nat_ctx* ctx, int write_macro) {
  return ctx->fp32 ? nat::step_comp<float>(ctx, write_macro) : nat::step_comp<double>(ctx, write_macro);
}

int nat_launch_collide_comp(nat_ctx* ctx) {
  return ctx->fp32 ? nat::collide_comp<float>(ctx) : nat::collide_comp<double>(ctx);
}
