// Upwind SEDG stage of the low-storage RK5 step, two opposite directions at a time (the scheme
// and its arithmetic are described in k_sedg.hip, whose kernel gives the same bits and serves the
// central flux and arrays beyond 32-bit offsets).
//
// A stage moves 16 B per value in FP32 and 32 B in FP64 (populations and RK registers in and
// out), and what bounded it was latency: a thread went from one direction to the next with the
// face gathers of a direction behind branches, asked for only when that direction began, at 3-4
// waves per SIMD. Here
//   - directions go in opposite pairs. The face factors of the two differ in sign only, so a face
//     node is upwind for exactly one of them: one gather per axis serves both, through one buffer
//     resource, the lanes adding the distance to the opposite direction's array where that one
//     is upwind. A wall face reads the other value of the pair, which the thread already has;
//   - what the next pair reads is loaded before this pair is summed, without a branch: a lane
//     with nothing to read has an offset out of range, which loads nothing and gives 0;
//   - both values of a pair meet in LDS as one double2, with one barrier and one read of the
//     derivative matrix for the two.
// us per step (5 stages), one direction at a time with branches -> pairs, periodic (before the face
// sums were selected for the upwind one, which costs 0-3%):
//   D3Q19 p=3 FP32   8^3 106 -> 38    24^3  600 -> 270   40^3 3331 -> 1482
//   D3Q19 p=3 FP64   8^3  88 -> 38    24^3  737 -> 557   40^3 3191 -> 2435
//   D3Q27 p=3        24^3 FP32 973 -> 454, FP64 1028 -> 801
//   D3Q19 p=2        24^3 FP32 292 -> 130, FP64  246 -> 189
//   D2Q9  p=2        16^2 FP32  59 -> 22.3, FP64 41 -> 22.4    64^2  63 -> 23.3, 46 -> 24.5
//   D2Q9  p=2       200^2 FP32  98 -> 61,   FP64 99 -> 87
// At 24^3 FP32 the 1.7 GB of a step take 250-340 us between the cache's rate (6.7 TB/s) and
// memory's (5.0); the small meshes are 5 launches of a serial chain each (vertices, inverse
// Jacobian, 4 or 9 pairs).
#include "nat_offsets.hpp"
#include "nat_sedg.hpp"
namespace nat {

// al of the k-th pair of opposite directions (al, op), al < op
template <int Q>
constexpr int pair_dir(int k) {
  for (int i = 1; i < Q; i++)
    if (opposite<Q>(i) > i && k-- == 0) return i;
  return -1;
}

// Buffer resource of `bytes` from p on (uniform; 0 bytes: loads give 0, stores are dropped).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t sedg_rsrc(const void* p, uint32_t bytes) {
  const uint64_t pb = (uint64_t)p;
  const uint32_t phi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(pb >> 32));
  const uint32_t plo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)pb);
  return __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)phi << 32) | (uint64_t)plo), (short)0,
                                           __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000);
}

template <typename T>
__device__ __forceinline__ T sedg_load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  if constexpr (sizeof(T) == 4)
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
  else
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
}

template <int AUX, typename T>
__device__ __forceinline__ void sedg_store(__amdgpu_buffer_rsrc_t r, uint32_t off, T v) {
  if constexpr (sizeof(T) == 4)
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, (int)off, 0, AUX);
  else
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(unsigned __attribute__((ext_vector_type(2))), v), r,
                                          (int)off, 0, AUX);
}

// COL: the last stage collides in registers. WALLS: a non-periodic axis (its terms cost
// registers). BIG: the mesh exceeds the Infinity Cache.
template <int D, int Q, int P, typename T, bool COL, bool WALLS, bool BIG>
__global__ __launch_bounds__((SedgShape<D, P>::NT)) void k_sedg_pair(SedgArgs<T> s, CollideArgs<T> ca,
                                                                      int write_macro) {
  using L = Lattice<Q>;
  using S = SedgShape<D, P>;
  constexpr int NP = S::NP, NL = S::NL, NT = S::NT, K = (Q - 1) / 2;
  // pairs loaded ahead (2D: 2 gain 1-2% up to 64^2; 3D: the registers of 2 cost 2%)
  constexpr int DP = D == 2 ? 2 : 1;
  // Cache policy of the stores where a wave stores whole lines (64-node cells). While everything
  // fits the Infinity Cache: written through to the device (sc1), 5-10% on 8^3 and 16^3. Beyond:
  // populations streamed past it (nt; 24^3 FP64 572 -> 557, 40^3 FP32 1514 -> 1482), which costs
  // the smaller ones up to 20%. Partial lines (p = 2) lose 5-10% with either.
  constexpr int FA = NL != 64 ? 0 : BIG ? 2 : 16, DA = NL != 64 || BIG ? 0 : 16;
  // the derivative rows of this node in registers (2% in 2D, 1-3% in FP64; where a stage streams
  // from memory or 3D FP32 would lose a wave per SIMD they stay in LDS)
  constexpr bool ROWS = !BIG && (D == 2 || sizeof(T) == 8);
  constexpr uint32_t b = sizeof(T), off_none = 0xffffffffu, range = 0xfffffff0u;
  __shared__ double2 buf[2][NT];
  __shared__ double dl[NP][NP];
  const int tid = threadIdx.x;
  for (int i = tid; i < NP * NP; i += NT) dl[i / NP][i % NP] = s.dl[i / NP][i % NP];

  unsigned bid = blockIdx.x;
  // neighbouring cells on the same XCD (workgroup i goes to XCD i % 8; the last nb % 8 keep their
  // index) while the mesh fits the Infinity Cache: 16^3 p=3 FP64 153 -> 136 us, 24^3 p=2 206 -> 189;
  // beyond, the 8 XCDs are better on neighbouring planes (40^3 FP64 2475 -> 2574 with it)
  if (!BIG) {
    const unsigned per = gridDim.x / 8;
    if (bid < per * 8) bid = (bid % 8) * per + bid / 8;
  }
  const int cl = tid / NL, l = tid % NL;
  const int64_t cell = (int64_t)bid * S::CPB + cl;
  const bool active = cell < s.ncell;
  const int64_t node = active ? cell * NL + l : 0;
  const int mi[3] = {l % NP, (l / NP) % NP, (D == 3) ? l / (NP * NP) : 0};
  const int lstr[3] = {1, NP, NP * NP};
  const uint32_t own = active ? (uint32_t)node * b : off_none;
  const int64_t sb = s.stride * (int64_t)b;  // bytes of a direction's array

  // what a pair (al, op) reads: own values and RK registers of both, and through each face the
  // neighbour's value of the one of the two for which the face is upwind
  struct Own {
    T va, vo, da, dO;
  } rown[DP + 1];
  T rnb[DP + 1][3];
  double rG[DP + 1][3];
  const uint32_t df_range = s.first ? 0u : range;
  auto load_own = [&](auto KK) {
    constexpr int k = decltype(KK)::value;
    if constexpr (k < K) {
      constexpr int al = pair_dir<Q>(k), op = opposite<Q>(al);
      Own& o = rown[k % (DP + 1)];
      o.va = sedg_load<T>(sedg_rsrc(s.fin + al * s.stride, range), own);
      o.vo = sedg_load<T>(sedg_rsrc(s.fin + op * s.stride, range), own);
      o.da = sedg_load<T>(sedg_rsrc(s.df + al * s.stride, df_range), own);
      o.dO = sedg_load<T>(sedg_rsrc(s.df + op * s.stride, df_range), own);
    }
  };
  static_for<0, DP>(load_own);

  // geometry of this node
  double Ji[3][3];
  uint32_t nbo[3] = {0, 0, 0};
  double fac[3] = {0, 0, 0};    // s_a / w_a(i) for the face through this node along axis a, else 0
  int wallf[3] = {-1, -1, -1};  // box face 2 a + side when that face is a wall
  {
    const int N0 = s.m.N[0], N1 = s.m.N[1];
    const int c[3] = {(int)(cell % N0), (int)((cell / N0) % N1), (D == 3) ? (int)(cell / ((int64_t)N0 * N1)) : 0};
    const double xi[3] = {s.gll[mi[0]], s.gll[mi[1]], (D == 3) ? s.gll[mi[2]] : 0.0};
    double J[3][3];
    if (active) {
      cell_jac<D>(s.m, c, xi, J);
    } else {
      for (int a = 0; a < 3; a++)
        for (int d = 0; d < 3; d++) J[a][d] = (a == d) ? 1.0 : 0.0;
    }
    inv_det(D, J, Ji);
#pragma unroll
    for (int a = 0; a < D; a++) {
      if (active && (mi[a] == 0 || mi[a] == P)) {
        const int up = (mi[a] == P) ? 1 : 0;
        int cn[3] = {c[0], c[1], c[2]};
        const int n = s.m.N[a];
        const bool edge = up ? (c[a] + 1 == n) : (c[a] == 0);
        if (WALLS && edge && !s.m.periodic[a]) {
          wallf[a] = 2 * a + up;
        } else {
          cn[a] = up ? (c[a] + 1 == n ? 0 : c[a] + 1) : (c[a] == 0 ? n - 1 : c[a] - 1);
          const int64_t nc = cn[0] + (int64_t)N0 * (cn[1] + (int64_t)N1 * cn[2]);
          nbo[a] = (uint32_t)(nc * NL + l + (up ? -P : P) * lstr[a]) * b;
        }
        fac[a] = (up ? 1.0 : -1.0) * s.inv_gw[mi[a]];
      }
    }
  }
  __syncthreads();

  const double dt = s.dt, ra = s.a, rb = s.b, sc = s.scaling;
  T fs[COL ? Q : 1];
  fs[0] = sedg_load<T>(sedg_rsrc(s.fin, range), own);
  if constexpr (!COL) sedg_store<FA>(sedg_rsrc(s.fout, range), own, fs[0]);
  double drow[ROWS ? 3 : 1][NP];
  if constexpr (ROWS)
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
      for (int j = 0; j < NP; j++) drow[d][j] = dl[mi[d]][j];

  auto load_faces = [&](auto KK) {
#pragma clang fp contract(off)
    constexpr int k = decltype(KK)::value;
    if constexpr (k < K) {
      constexpr int al = pair_dir<Q>(k), op = opposite<Q>(al), r = k % (DP + 1);
      constexpr int e0 = L::e[al][0], e1 = L::e[al][1], e2 = (D == 3) ? L::e[al][2] : 0;
      const __amdgpu_buffer_rsrc_t src = sedg_rsrc(s.fin + al * s.stride, range);
      // G_b = sum_k e_k (J^-1)_bk, scaled velocities
#pragma unroll
      for (int d = 0; d < D; d++) {
        double g = 0;
        if (e0 != 0) g += e0 > 0 ? Ji[d][0] : -Ji[d][0];
        if (e1 != 0) g += e1 > 0 ? Ji[d][1] : -Ji[d][1];
        if (e2 != 0) g += e2 > 0 ? Ji[d][2] : -Ji[d][2];
        rG[r][d] = g * sc;
      }
#pragma unroll
      for (int a = 0; a < D; a++) {
        const double c = fac[a] * rG[r][a];
        uint32_t o = nbo[a] + (c > 0.0 ? (uint32_t)((op - al) * sb) : 0u);
        o = c != 0.0 ? o : off_none;
        if constexpr (WALLS) o = wallf[a] < 0 ? o : off_none;
        rnb[r][a] = sedg_load<T>(src, o);
      }
    }
  };
  static_for<0, DP>(load_faces);
  static_for<0, K>([&](auto KK) {
    // fused multiply-adds are written out and no other contraction is allowed, so that the
    // stream-only and the collide-after instantiations round the same way
#pragma clang fp contract(off)
    constexpr int k = decltype(KK)::value, r = k % (DP + 1), al = pair_dir<Q>(k), op = opposite<Q>(al);
    constexpr int e0 = L::e[al][0], e1 = L::e[al][1], e2 = (D == 3) ? L::e[al][2] : 0;
    load_own(std::integral_constant<int, k + DP>{});
    load_faces(std::integral_constant<int, k + DP>{});
    __builtin_amdgcn_sched_barrier(0);
    const double va = (double)rown[r].va, vo = (double)rown[r].vo;
    buf[k & 1][tid] = make_double2(va, vo);
    sedg_barrier();
    double la = 0, lo = 0;
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int base = tid - mi[d] * lstr[d];
      double der_a = 0, der_o = 0;
#pragma unroll
      for (int j = 0; j < NP; j++) {
        const double2 x = buf[k & 1][base + j * lstr[d]];
        const double w = ROWS ? drow[ROWS ? d : 0][j] : dl[mi[d]][j];
        der_a = fma(w, x.x, der_a);
        der_o = fma(w, x.y, der_o);
      }
      la = fma(-rG[r][d], der_a, la);
      lo = fma(rG[r][d], der_o, lo);
    }
#pragma unroll
    for (int a = 0; a < D; a++) {
      const double c = fac[a] * rG[r][a];
      double na = (double)rnb[r][a], no = na, cwu = 0.0;
      if (WALLS && wallf[a] >= 0) {
        na = vo;
        no = va;
        // wall velocity term: c w (e.u_wall) / cs2 with e and cs2 scaled, cs2 = s^2 / 3 (equal
        // for the two directions: c and e both change sign)
        const double* uw = s.m.wall_u[wallf[a]];
        double eu = 0.0;
        if (e0 != 0) eu += e0 * uw[0];
        if (e1 != 0) eu += e1 * uw[1];
        if (e2 != 0) eu += e2 * uw[2];
        cwu = c * L::w[al] * (3.0 * eu / sc);
      }
      // the face belongs to the one of the two for which it is upwind: for the other na or no is its
      // partner's value, and a flux of zero times it would hand on infinities
      la = c < 0.0 ? fma(c, va - na, la) : la;
      lo = c > 0.0 ? fma(-c, vo - no, lo) : lo;
      if constexpr (WALLS) {
        if (c < 0.0) la -= 2.0 * cwu;
        if (c > 0.0) lo -= 2.0 * cwu;
      }
    }
    const auto rk = [&](int q, double v, double lf, T dfo) {
#pragma clang fp contract(off)
      double d = fma((double)dfo, ra, lf * dt);
      d *= rb;
      const double fnew = v + d;
      d *= s.binv;
      sedg_store<DA>(sedg_rsrc(s.df + q * s.stride, s.store_df ? range : 0u), own, (T)d);
      if constexpr (!COL) sedg_store<FA>(sedg_rsrc(s.fout + q * s.stride, range), own, (T)fnew);
      return (T)fnew;
    };
    const T fa = rk(al, va, la, rown[r].da), fo = rk(op, vo, lo, rown[r].dO);
    if constexpr (COL) {
      fs[al] = fa;
      fs[op] = fo;
    }
    __builtin_amdgcn_sched_barrier(0);
  });
  if constexpr (COL) {
    if (active) bgk_collide_store_pairs<Q, T>(fs, ca, node, write_macro != 0, s.fout, s.stride);
  }
}

template <int D, int Q, int P, typename T>
static void launch_pair(nat_ctx* ctx, const SedgArgs<T>& s, const CollideArgs<T>& ca, int collide, int wm) {
  using S = SedgShape<D, P>;
  const auto launch = [&](auto COL, auto WALLS, auto BIG) {
    constexpr bool col = decltype(COL)::value, walls = decltype(WALLS)::value, big = decltype(BIG)::value;
    hipLaunchKernelGGL((k_sedg_pair<D, Q, P, T, col, walls, big>),
                       dim3((unsigned)((s.ncell + S::CPB - 1) / S::CPB)), dim3(S::NT), 0, ctx->stream, s, ca,
                       col ? wm : 0);
  };
  const auto pick = [&](auto COL, auto WALLS) {
    // two population arrays and the RK registers against the 256 MiB Infinity Cache
    if (3 * Q * s.stride * (int64_t)sizeof(T) > (256 << 20))
      launch(COL, WALLS, std::true_type{});
    else
      launch(COL, WALLS, std::false_type{});
  };
  if (ctx->has_walls)
    collide ? pick(std::true_type{}, std::true_type{}) : pick(std::false_type{}, std::true_type{});
  else
    collide ? pick(std::true_type{}, std::false_type{}) : pick(std::false_type{}, std::false_type{});
}

template <typename T>
bool nat_sedg_pair_stage(nat_ctx* ctx, const SedgArgs<T>& s, const CollideArgs<T>& ca, int collide, int wm) {
  if (nat_sedg_form(ctx) == 0) return false;
  const int Q = ctx->Q, P = ctx->p;
#define NAT_SP(DD, QQ, PP)                              \
  if (Q == QQ && P == PP) {                             \
    launch_pair<DD, QQ, PP, T>(ctx, s, ca, collide, wm); \
    return true;                                        \
  }
  NAT_SP(2, 9, 1)
  NAT_SP(2, 9, 2)
  NAT_SP(2, 9, 3)
  NAT_SP(2, 9, 4)
  NAT_SP(2, 9, 5)
  NAT_SP(2, 9, 6)
  NAT_SP(3, 19, 1)
  NAT_SP(3, 19, 2)
  NAT_SP(3, 19, 3)
  NAT_SP(3, 19, 4)
  NAT_SP(3, 27, 1)
  NAT_SP(3, 27, 2)
  NAT_SP(3, 27, 3)
  NAT_SP(3, 27, 4)
#undef NAT_SP
  return false;
}

template bool nat_sedg_pair_stage<float>(nat_ctx*, const SedgArgs<float>&, const CollideArgs<float>&, int, int);
template bool nat_sedg_pair_stage<double>(nat_ctx*, const SedgArgs<double>&, const CollideArgs<double>&, int, int);

}  // namespace nat
