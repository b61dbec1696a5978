// Arguments and block shape of the SEDG stage kernels.
#pragma once
#include "nat_collide.hpp"
#include "nat_geom.hpp"

int nat_sedg_form(const nat_ctx* ctx, int form = -1);

namespace nat {

template <typename T>
struct SedgArgs {
  const T* fin;
  T* fout;
  T* df;
  int64_t stride;
  int64_t ncell;
  MeshDev m;
  double scaling;
  double dt;
  double a, b;       // RK5 coefficients of this stage
  double binv;       // 1 / b (the division of df /= b is a multiplication by 1/b)
  double rho0;       // FP32 shift (0 for FP64)
  int first;         // first stage: df not read
  int store_df;      // 0 on the last stage (df is dead afterwards)
  int central;       // central flux
  double gll[MAXP + 1];
  double inv_gw[MAXP + 1];           // 1 / GLL weight
  double dl[MAXP + 1][MAXP + 1];     // dl[i][j] = phi_j'(x_i)
};

template <int D, int P>
struct SedgShape {
  static constexpr int NP = P + 1;
  static constexpr int NL = (D == 3) ? NP * NP * NP : NP * NP;
  // cells per block: ~256 threads; a 64-node cell (3D, p = 3) runs alone as one wave, whose
  // per-direction barrier then waits for no other wave (C3 SEDG +4% FP32, +1% FP64)
  static constexpr int CPB = (NL == 64) ? 1 : ((256 / NL) > 0 ? 256 / NL : 1);
  static constexpr int NT = CPB * NL;
};

__device__ __forceinline__ void sedg_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// One RK5 stage of the upwind flux, two opposite directions at a time; false: the context's form is
// another (the central flux, or arrays too large for 32-bit offsets) and the caller takes the
// general stage kernel.
template <typename T>
bool nat_sedg_pair_stage(nat_ctx* ctx, const SedgArgs<T>& s, const CollideArgs<T>& ca, int collide, int wm);

}  // namespace nat
