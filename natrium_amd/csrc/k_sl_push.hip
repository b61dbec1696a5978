// Collide-then-stream steps on affine periodic Cartesian meshes: the form of the structured
// step that runs of several steps take.
//
// nat_step(n) is n x (stream; collide). Taken as stream, (n - 1) x (collide; stream), collide,
// the middle launches collide a node's populations before they are streamed, so a workgroup can
// collide the nodes of its own source cells once, keep them in LDS, and let one thread carry a
// (direction, source cell) through all the one-dimensional passes of the interpolation in
// registers: p+1 values per line in, p outputs per axis out (the outputs that depart from that
// cell: for a positive component its nodes 1..p, otherwise 0..p-1, every node of the mesh exactly
// once). Between the collision and the streaming there is one barrier, and the passes need no
// LDS traffic, index arithmetic or barriers of their own: the pass-by-pass form of k_sl_struct
// has 20 barriers and 1,287 VALU instructions per node-wave for D3Q27 p = 4. The price is that the
// nodes on the upper faces of a tile are collided by the neighbouring tiles too.
//
// Lanes. A wave's 64 lanes hold items (part of the outputs, direction, cell) of one class of
// directions (the non-zero components), so lanes differ in the signs of their components and, in
// the classes with one or two of them, in which axes they lie on. All lanes run one code: the
// weights are chosen per lane by the sign, W(+, j, m) or, with GLL nodes' mirror symmetry,
// W(-, j, m) = W(+, (p - j) mod p, p - m); LDS strides and output addresses are chosen by the axis.
//
// Rounding. The passes run in the order z, y, x over the non-zero components, each summing over the
// nodes of its line from the lower end with explicit FMAs in FP64, and streamed values are rounded
// to storage precision before they are collided: the same operations in the same order as
// k_sl_struct, so the two forms agree bit for bit.
#include "nat_collide.hpp"

namespace nat {

template <typename T>
struct PushArgs {
  const T* fin;
  T* fout;
  int64_t stride;
  int n[3];      // unique nodes per axis
  int tiles[3];  // tiles per axis
  int dir_bytes;     // bytes of one direction's array
  unsigned all_bytes;  // bytes of all directions (32-bit store offsets)
};

// Compile-time shape: CX x CY x CZ source cells per workgroup, NT threads; in 3D an item is one
// S-th of the outputs of its (direction, cell), split along z or along an axis without a pass.
template <int D, int Q, int P, int CX, int CY, int CZ_, int NT_, int S_>
struct PushShape {
  static constexpr int CZ = D == 3 ? CZ_ : 1;
  static constexpr int NC = CX * CY * CZ;
  static constexpr int NT = NT_, NW = NT_ / 64, S = D == 3 ? S_ : 1;
  static constexpr int EX = CX * P + 1, EY = CY * P + 1, EZ = D == 3 ? CZ * P + 1 : 1;
  static constexpr int NN = EX * EY * EZ;
  static constexpr int PY = EX, PZ = EX * EY;  // LDS pitches
  static constexpr int DS = NN | 1;            // LDS elements per direction (odd: bank spread)
  static constexpr int ROUNDS = (NN + NT - 1) / NT;
  // jobs (waves of 64 items) per class of directions
  static constexpr int chunks(int dirs) { return (dirs * NC * S + 63) / 64; }
  static constexpr int J3 = D == 3 && Q == 27 ? chunks(8) : 0;  // three components
  static constexpr int JYZ = D == 3 ? chunks(4) : 0;            // y and z
  static constexpr int JX2 = chunks(D == 3 ? 8 : 4);            // x and y, x and z
  static constexpr int JA = chunks(D == 3 ? 4 : 2);             // y; z
  static constexpr int JX = chunks(2);                          // x
  static constexpr int NJ = J3 + JYZ + JX2 + JA + JX;
};

// Index of the direction (x, y, z) in the stencil's table.
template <int Q>
constexpr int dir_of(int x, int y, int z) {
  for (int i = 0; i < Q; i++)
    if (Lattice<Q>::e[i][0] == x && Lattice<Q>::e[i][1] == y && Lattice<Q>::e[i][2] == z) return i;
  return 0;
}

// Directions of a class as bytes of a 64-bit constant, indexed by sign bits (bit set: negative).
enum { PUSH_XYZ, PUSH_YZ, PUSH_X2, PUSH_A, PUSH_X };
template <int D, int Q, int CLS>
constexpr unsigned long long push_dirs() {
  unsigned long long k = 0;
  for (int d = 0; d < 8; d++) {
    const int s0 = (d & 1) ? -1 : 1, s1 = (d & 2) ? -1 : 1, s2 = (d & 4) ? -1 : 1;
    const bool z = CLS == PUSH_X2 ? (d & 4) : (d & 2);  // the second axis of X2, the axis of A
    int al = 0;
    if (CLS == PUSH_XYZ) al = dir_of<Q>(s0, s1, s2);
    if (CLS == PUSH_YZ) al = d < 4 ? dir_of<Q>(0, s0, s1) : 0;
    if (CLS == PUSH_X2) al = z ? (D == 3 ? dir_of<Q>(s0, 0, s1) : 0) : dir_of<Q>(s0, s1, 0);
    if (CLS == PUSH_A) al = d < 4 ? (z ? (D == 3 ? dir_of<Q>(0, 0, s0) : 0) : dir_of<Q>(0, s0, 0)) : 0;
    if (CLS == PUSH_X) al = d < 2 ? dir_of<Q>(s0, 0, 0) : 0;
    k |= (unsigned long long)al << (8 * d);
  }
  return k;
}

// n / DV for 0 <= n < N as a multiply and a shift (checked at compile time).
template <unsigned DV, unsigned N>
struct PushDiv {
  static constexpr unsigned shift() {
    for (unsigned s = 8; s < 24; s++) {
      const unsigned long long m = ((1ull << s) + DV - 1) / DV;
      if (m >= (1u << 24)) break;
      bool ok = true;
      for (unsigned n = 0; n < N && ok; n++) ok = ((unsigned long long)n * m >> s) == n / DV;
      if (ok) return s;
    }
    return 0;
  }
  static constexpr unsigned S = shift();
  static constexpr unsigned M = (unsigned)(((1ull << S) + DV - 1) / DV);
  static_assert((DV & (DV - 1)) == 0 || S > 0, "no 24-bit reciprocal for this divisor");
  __device__ static __forceinline__ unsigned div(unsigned n) {
    if constexpr ((DV & (DV - 1)) == 0)
      return n / DV;
    else
      return __umul24(n, M) >> S;
  }
};

template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t push_rsrc(const T* p, unsigned bytes) {
  const uint64_t pb = (uint64_t)p;
  const uint32_t phi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(pb >> 32));
  const uint32_t plo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)pb);
  return __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)phi << 32) | (uint64_t)plo), (short)0,
                                           __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000);
}

// Where a lane's outputs go along one axis: output j (0..P-1) of a positive component is node
// lo + 1 + j of the mesh, otherwise node lo + j; node n wraps to 0 (the last output of a positive
// component only). Byte offsets.
struct PushAxis {
  int o, d, last;
  __device__ __forceinline__ int at(int j, int P) const { return j == P - 1 ? last : o + j * d; }
};
__device__ __forceinline__ PushAxis push_axis(int lo, int sgn, int P, int n, int bytes) {
  PushAxis a;
  const int first = sgn > 0 ? lo + 1 : lo, l = first + P - 1;
  a.d = bytes;
  a.o = first * bytes;
  a.last = (l == n ? 0 : l) * bytes;
  return a;
}

// Stores one x line of P outputs. WRAP: the tile holds the last cell along x, whose last positive
// output is node 0. Plain write-back stores: with the sc1 write-through policy of the other step
// kernels these short lines reach memory as partial writes (16^3 cells, p = 4, D3Q27 FP32: 28.5
// against 22.3 us per step in an 8 x 8 x 8 tile).
template <int P, bool WRAP, typename T>
__device__ __forceinline__ void push_row(__amdgpu_buffer_rsrc_t rs, unsigned off, const PushAxis& ax, const double* v) {
  constexpr int W = (int)sizeof(T) / 4;  // dwords per value
  unsigned q[P * W];
#pragma unroll
  for (int i = 0; i < P; i++) {
    const T r = (T)v[i];
    if constexpr (W == 1) {
      q[i] = __builtin_bit_cast(unsigned, r);
    } else {
      const unsigned long b = __builtin_bit_cast(unsigned long, r);
      q[2 * i] = (unsigned)b;
      q[2 * i + 1] = (unsigned)(b >> 32);
    }
  }
  using u2 = unsigned __attribute__((ext_vector_type(2)));
  using u3 = unsigned __attribute__((ext_vector_type(3)));
  using u4 = unsigned __attribute__((ext_vector_type(4)));
  auto put = [&](unsigned u, auto I, auto N) {  // dwords I .. I + N of the line at byte offset u
    constexpr int i = decltype(I)::value, n = decltype(N)::value;
    const int o = (int)u;
    if constexpr (n == 1) __builtin_amdgcn_raw_buffer_store_b32(q[i], rs, o, 0, 0);
    if constexpr (n == 2) __builtin_amdgcn_raw_buffer_store_b64(u2{q[i], q[i + 1]}, rs, o, 0, 0);
    if constexpr (n == 3) __builtin_amdgcn_raw_buffer_store_b96(u3{q[i], q[i + 1], q[i + 2]}, rs, o, 0, 0);
    if constexpr (n == 4)
      __builtin_amdgcn_raw_buffer_store_b128(u4{q[i], q[i + 1], q[i + 2], q[i + 3]}, rs, o, 0, 0);
  };
  constexpr int H = (WRAP ? P - 1 : P) * W;
  static_for<0, (H + 3) / 4>([&](auto K) {
    constexpr int i = 4 * decltype(K)::value, n = H - i < 4 ? H - i : 4;
    put(off + ax.o + 4 * i, std::integral_constant<int, i>{}, std::integral_constant<int, n>{});
  });
  if constexpr (WRAP) put(off + ax.last, std::integral_constant<int, H>{}, std::integral_constant<int, W>{});
}

// acc (+)= w v, the first term a product: the accumulation of every pass
__device__ __forceinline__ double push_mad(bool first, double w, double v, double acc) {
#pragma clang fp contract(off)
  return first ? w * v : fma(w, v, acc);
}

// COL: collide before streaming (false: the run's first launch, streaming only).
template <int D, int Q, int P, typename T, int CX, int CY, int CZ_, int NT, int S_, int WPE, bool COL>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(WPE))) void k_sl_push(
    PushArgs<T> a, const double* __restrict__ wtab /* positive shift, [MAXP][MAXP+1] */, CollideArgs<T> ca) {
  using H = PushShape<D, Q, P, CX, CY, CZ_, NT, S_>;
  constexpr int S = H::S;
  constexpr int EX = H::EX, EY = H::EY, EZ = H::EZ, NN = H::NN, PY = H::PY, PZ = H::PZ, DS = H::DS, NC = H::NC;
  constexpr int CZ = H::CZ, TX = CX * P, TY = CY * P, TZ = D == 3 ? CZ * P : 1;
  constexpr int b = (int)sizeof(T);
  __shared__ T buf[(Q - 1) * DS];
  const int tid = threadIdx.x;
  const int nx = a.n[0], ny = a.n[1], nz = a.n[2];
  int bid = blockIdx.x;
  // tiles that share faces run on the same XCD (workgroup i goes to XCD i % 8); the last nb % 8
  // workgroups keep their index
  const int per = (int)gridDim.x / 8;
  if (bid < per * 8) bid = (bid % 8) * per + bid / 8;
  const int x0 = (bid % a.tiles[0]) * TX, y0 = ((bid / a.tiles[0]) % a.tiles[1]) * TY,
            z0 = D == 3 ? (bid / (a.tiles[0] * a.tiles[1])) * TZ : 0;
  // extents of this tile in nodes (ragged at the upper faces)
  const int vx = nx - x0 < TX ? nx - x0 : TX, vy = ny - y0 < TY ? ny - y0 : TY,
            vz = D == 3 ? (nz - z0 < TZ ? nz - z0 : TZ) : 1;

  double W[P][P + 1];  // W[j][m]: output j (node j + 1) of the positive shift
#pragma unroll
  for (int j = 0; j < P; j++)
#pragma unroll
    for (int m = 0; m <= P; m++) W[j][m] = wtab[((j + 1) % P) * (MAXP + 1) + m];

  // ---- the populations of the source cells' nodes: collided (COL), into LDS
  // (loads of a round are issued before the previous round is collided)
  const __amdgpu_buffer_rsrc_t src = push_rsrc(a.fin, a.all_bytes);
  struct Place {
    bool live, own;
    int lx, ly, lz, node;
  };
  auto place = [&](int r) {
    Place p;
    const int idx = tid + r * NT;
    const unsigned q1 = PushDiv<EX, H::ROUNDS * NT>::div(idx), q2 = PushDiv<EY, H::ROUNDS * NT / EX + 1>::div(q1);
    p.lx = idx - (int)q1 * EX;
    p.ly = (int)q1 - (int)q2 * EY;
    p.lz = (int)q2;
    p.live = idx < NN && p.lx <= vx && p.ly <= vy && (D == 2 || p.lz <= vz);
    p.own = p.lx < vx && p.ly < vy && (D == 2 || p.lz < vz);
    const int gx = x0 + p.lx == nx ? 0 : x0 + p.lx, gy = y0 + p.ly == ny ? 0 : y0 + p.ly,
              gz = D == 3 ? (z0 + p.lz == nz ? 0 : z0 + p.lz) : 0;
    p.node = p.live ? gx + nx * (gy + ny * gz) : 0;
    return p;
  };
  T fn[Q];
  auto load = [&](const Place& p) {
#pragma unroll
    for (int q = 0; q < Q; q++) {
      if constexpr (b == 4)
        fn[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(src, p.node * b, (int)((unsigned)q * (unsigned)a.dir_bytes), 0));
      else
        fn[q] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(src, p.node * b, (int)((unsigned)q * (unsigned)a.dir_bytes), 0));
    }
  };
  Place pn = place(0);
  load(pn);
#pragma unroll 1
  for (int r = 0; r < H::ROUNDS; r++) {
    const Place pc = pn;
    T f[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) f[q] = fn[q];
    if (r + 1 < H::ROUNDS) {
      pn = place(r + 1);
      load(pn);
    }
    if (!pc.live) continue;
    const int lx = pc.lx, ly = pc.ly, lz = pc.lz, node = pc.node;
    const bool own = pc.own;
    const int at = lx + PY * ly + PZ * lz;
    auto put = [&](auto I, T v) {
      constexpr int i = decltype(I)::value;
      if constexpr (i == 0) {
        if (own) a.fout[node] = v;
      } else {
        buf[(i - 1) * DS + at] = v;
      }
    };
    if constexpr (COL) {
      bgk_collide_pairs<Q, T, false>(f, ca, node, false, [&](auto I, double v) { put(I, (T)v); });
    } else {
      static_for<0, Q>([&](auto I) { put(I, f[decltype(I)::value]); });
    }
  }
  __syncthreads();

  // ---- streaming: each wave takes jobs of 64 items of one class
  const __amdgpu_buffer_rsrc_t rs = push_rsrc(a.fout, a.all_bytes);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const bool wrap = x0 + TX >= nx;
  const unsigned dirb = (unsigned)(a.stride * b);  // byte distance of directions (offsets are taken modulo 2^32)

  auto job = [&](auto CLS, unsigned chunk) {
    constexpr int cls = decltype(CLS)::value;
    constexpr int ND = cls == PUSH_XYZ ? 8
                       : cls == PUSH_YZ ? 4
                       : cls == PUSH_X2 ? (D == 3 ? 8 : 4)
                       : cls == PUSH_A  ? (D == 3 ? 4 : 2)
                                        : 2;
    constexpr bool deep = cls == PUSH_XYZ || cls == PUSH_YZ;  // the item's part: z outputs
    constexpr int H1 = P / S;                                 // outputs of an item along the split axis
    // the lane's addresses are formed in its own job, not hoisted for all classes
    unsigned it = chunk * 64 + lane;
    asm volatile("" : "+v"(it));
    const unsigned rd = PushDiv<NC, S * ND * NC + 64>::div(it);
    const int c = (int)(it - rd * NC);
    const unsigned d = rd % ND;
    const int part = (int)(rd / ND);
    if (part >= S) return;
    const int al = (int)((push_dirs<D, Q, cls>() >> (8 * d)) & 255);
    // signs per axis of the direction (0: no component); A: the axis of y or z, onz: it is z
    const int s0 = d & 1 ? -1 : 1, s1 = d & 2 ? -1 : 1, s2 = d & 4 ? -1 : 1;
    const bool onz = D == 3 && (cls == PUSH_X2 ? (d & 4) != 0 : (cls == PUSH_A && (d & 2) != 0));
    const int sx = cls == PUSH_XYZ || cls == PUSH_X2 || cls == PUSH_X ? s0 : 0;
    const int sA = cls == PUSH_X2 ? s1 : s0;  // X2, A
    const int sy = cls == PUSH_XYZ ? s1 : (cls == PUSH_YZ ? s0 : (cls == PUSH_X || onz ? 0 : sA));
    const int sz = cls == PUSH_XYZ ? s2 : (cls == PUSH_YZ ? s1 : (cls == PUSH_X || !onz ? 0 : sA));
    const int c0 = c % CX, c1 = (c / CX) % CY, c2 = D == 3 ? c / (CX * CY) : 0;
    const int px = x0 + P * c0, py = y0 + P * c1, pz = z0 + P * c2;
    if (px >= nx || py >= ny || (D == 3 && pz >= nz)) return;  // cell beyond a ragged tile
    const PushAxis ox = push_axis(px, sx, P, nx, b);
    const PushAxis oy = push_axis(py, sy, P, ny, nx * b);
    const PushAxis oz = push_axis(pz, sz, P, nz, nx * ny * b);
    const unsigned out = (unsigned)al * dirb;
    const T* __restrict__ in = buf + (al - 1) * DS + P * (c0 + PY * c1 + PZ * c2);

    // weights of output j from the node m of the source cell's line, by the sign
    auto weight = [&](int sgn, int j, int m) { return sgn > 0 ? W[j][m] : W[(P - 1 - j) % P][P - m]; };
    auto weights = [&](int sgn, double (&w)[P][P + 1]) {
#pragma unroll
      for (int j = 0; j < P; j++)
#pragma unroll
        for (int m = 0; m <= P; m++) w[j][m] = weight(sgn, j, m);
    };
    double wx[P][P + 1], wA[P][P + 1];
    if constexpr (cls == PUSH_XYZ || cls == PUSH_X2 || cls == PUSH_X) weights(sx, wx);
    if constexpr (cls != PUSH_X) weights(deep ? sy : sA, wA);

    if constexpr (deep) {
      // per plane of constant x: the z pass along each line, then y; XYZ: then x over the planes
      double wz[H1][P + 1];
#pragma unroll
      for (int j = 0; j < H1; j++)
#pragma unroll
        for (int m = 0; m <= P; m++) {
          double w = weight(sz, j, m);
#pragma unroll
          for (int r = 1; r < S; r++) w = part == r ? weight(sz, r * H1 + j, m) : w;
          wz[j][m] = w;
        }
      constexpr int NX = cls == PUSH_XYZ ? P + 1 : P;
      constexpr bool ahead = sizeof(T) == 4;  // the next plane's LDS reads before this plane's sums
      T nxt[P + 1][P + 1];
      auto fetch = [&](int pl) {
#pragma unroll
        for (int r = 0; r <= P; r++)
#pragma unroll
          for (int m = 0; m <= P; m++) nxt[r][m] = in[pl + PY * r + PZ * m];
      };
      double acc[H1][P][P];
      if (ahead) fetch(0);
#pragma unroll
      for (int pl = 0; pl < NX; pl++) {
        if (!ahead) fetch(pl);
        T cur[P + 1][P + 1];
#pragma unroll
        for (int r = 0; r <= P; r++)
#pragma unroll
          for (int m = 0; m <= P; m++) cur[r][m] = nxt[r][m];
        if (ahead && pl + 1 < NX) fetch(pl + 1);
        double ty[H1][P];
#pragma unroll
        for (int my = 0; my <= P; my++) {
#pragma unroll
          for (int jz = 0; jz < H1; jz++) {
            double tz = 0;
#pragma unroll
            for (int m = 0; m <= P; m++) tz = push_mad(m == 0, wz[jz][m], (double)cur[my][m], tz);
#pragma unroll
            for (int jy = 0; jy < P; jy++) ty[jz][jy] = push_mad(my == 0, wA[jy][my], tz, ty[jz][jy]);
          }
          __builtin_amdgcn_sched_barrier(0);  // or the compiler reads and converts ahead, into spills
        }
#pragma unroll
        for (int jz = 0; jz < H1; jz++)
#pragma unroll
          for (int jy = 0; jy < P; jy++) {
            if constexpr (cls == PUSH_XYZ) {
#pragma unroll
              for (int jx = 0; jx < P; jx++) acc[jz][jy][jx] = push_mad(pl == 0, wx[jx][pl], ty[jz][jy], acc[jz][jy][jx]);
            } else {
              acc[jz][jy][pl] = ty[jz][jy];
            }
          }
        __builtin_amdgcn_sched_barrier(0);
      }
      auto rows = [&](auto WR) {
#pragma unroll
        for (int jz = 0; jz < H1; jz++) {
          const int z = jz == H1 - 1 && part == S - 1 ? oz.last : oz.o + (part * H1 + jz) * oz.d;
#pragma unroll
          for (int jy = 0; jy < P; jy++)
            push_row<P, decltype(WR)::value, T>(rs, out + oy.at(jy, P) + z, ox, acc[jz][jy]);
        }
      };
      if (cls == PUSH_XYZ && wrap)
        rows(std::true_type{});
      else
        rows(std::false_type{});
    } else {
      // per line index of the axis B without a component (3D): X2: pass along A, then x; A: along
      // A; X: along x for each line of y
      constexpr int NB = D == 3 ? H1 : 1, NR = cls == PUSH_X ? P : (cls == PUSH_X2 ? P + 1 : P);
      const int stA = cls == PUSH_X ? PY : (onz ? PZ : PY), stB = cls == PUSH_X ? PZ : (onz ? PY : PZ);
      const PushAxis oA = cls != PUSH_X && onz ? oz : oy, oB = cls != PUSH_X && onz ? oy : oz;
      const int b0 = part * H1;  // (no component along B: its offsets are linear)
      const T* line = in + (D == 3 ? b0 * stB : 0);
      unsigned base = out + (D == 3 ? oB.o + b0 * oB.d : 0);
#pragma unroll
      for (int jb = 0; jb < NB; jb++, line += stB, base += oB.d) {
        T cur[NR][P + 1];
#pragma unroll
        for (int m = 0; m <= (cls == PUSH_X ? P - 1 : P); m++) {
          const T* q = line + m * stA;
#pragma unroll
          for (int r = 0; r < (cls == PUSH_X ? P + 1 : NR); r++) {
            if constexpr (cls == PUSH_X)
              cur[m][r] = q[r];
            else
              cur[r][m] = q[r];
          }
        }
        double acc[P][P];  // [along A][along x]
        if constexpr (cls == PUSH_X2) {
#pragma unroll
          for (int mx = 0; mx <= P; mx++)
#pragma unroll
            for (int ja = 0; ja < P; ja++) {
              double ta = 0;
#pragma unroll
              for (int m = 0; m <= P; m++) ta = push_mad(m == 0, wA[ja][m], (double)cur[mx][m], ta);
#pragma unroll
              for (int jx = 0; jx < P; jx++) acc[ja][jx] = push_mad(mx == 0, wx[jx][mx], ta, acc[ja][jx]);
            }
        } else {
#pragma unroll
          for (int ja = 0; ja < P; ja++)
#pragma unroll
            for (int jx = 0; jx < P; jx++) {
              double t = 0;
#pragma unroll
              for (int m = 0; m <= P; m++)
                t = cls == PUSH_A ? push_mad(m == 0, wA[ja][m], (double)cur[jx][m], t)
                                  : push_mad(m == 0, wx[jx][m], (double)cur[ja][m], t);
              acc[ja][jx] = t;
            }
        }
        auto rows = [&](auto WR) {
#pragma unroll
          for (int ja = 0; ja < P; ja++)
            push_row<P, decltype(WR)::value, T>(rs, base + oA.at(ja, P), ox, acc[ja]);
        };
        if (cls != PUSH_A && wrap)
          rows(std::true_type{});
        else
          rows(std::false_type{});
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // dearest classes first; the second round runs through the waves backwards
#pragma unroll 1
  for (int k = 0; k < H::NJ; k += H::NW) {
    unsigned j = (unsigned)(k + ((k / H::NW) & 1 ? H::NW - 1 - wave : wave));
    if (j < (unsigned)H::J3) {
      if constexpr (H::J3 > 0) job(std::integral_constant<int, PUSH_XYZ>{}, j);
    } else if ((j -= H::J3) < (unsigned)H::JYZ) {
      if constexpr (H::JYZ > 0) job(std::integral_constant<int, PUSH_YZ>{}, j);
    } else if ((j -= H::JYZ) < (unsigned)H::JX2) {
      job(std::integral_constant<int, PUSH_X2>{}, j);
    } else if ((j -= H::JX2) < (unsigned)H::JA) {
      job(std::integral_constant<int, PUSH_A>{}, j);
    } else if ((j -= H::JA) < (unsigned)H::JX) {
      job(std::integral_constant<int, PUSH_X>{}, j);
    }
  }
}

template <int D, int Q, int P, typename T, int CX, int CY, int CZ, int NT, int S, int WPE>
static int launch_push(nat_ctx* ctx, PushArgs<T> a, const CollideArgs<T>& ca, bool col) {
  using H = PushShape<D, Q, P, CX, CY, CZ, NT, S>;
  static_assert((size_t)(Q - 1) * H::DS * sizeof(T) <= 160 * 1024, "tile beyond the LDS of a CU");
  static_assert(P % H::S == 0, "items are equal parts");
  a.tiles[0] = (a.n[0] + CX * P - 1) / (CX * P);
  a.tiles[1] = (a.n[1] + CY * P - 1) / (CY * P);
  a.tiles[2] = D == 3 ? (a.n[2] + CZ * P - 1) / (CZ * P) : 1;
  const int nb = a.tiles[0] * a.tiles[1] * a.tiles[2];
  if (col)
    hipLaunchKernelGGL((k_sl_push<D, Q, P, T, CX, CY, CZ, NT, S, WPE, true>), dim3(nb), dim3(NT), 0, ctx->stream, a,
                       (const double*)ctx->ax_w, ca);
  else
    hipLaunchKernelGGL((k_sl_push<D, Q, P, T, CX, CY, CZ, NT, S, WPE, false>), dim3(nb), dim3(NT), 0, ctx->stream, a,
                       (const double*)ctx->ax_w, ca);
  NAT_HIP(hipGetLastError());
  return 0;
}

// One instantiated tile.
template <int D_, int Q_, int P_, int CX_, int CY_, int CZ_, int NT_, int S_, int WPE_>
struct PushTile {
  static constexpr int D = D_, Q = Q_, P = P_, CX = CX_, CY = CY_, CZ = CZ_, NT = NT_, S = S_, WPE = WPE_;
};

// Calls f(PushTile) for tile 1 (the small one) or 2 (the large one) of a stencil and order;
// NAT_ERR_UNSUPPORTED: no such tile.
template <typename T, typename F>
static int push_dispatch(int tile, int Q, int P, F&& f) {
  // cells per workgroup, threads, parts per item, waves per SIMD the registers are held to
#define NAT_P(tl, DD, QQ, PP, ...) \
  if (tile == tl && Q == QQ && P == PP) return f(PushTile<DD, QQ, PP, __VA_ARGS__>{});
#define NAT_P3(tl, PP, ...)      \
  NAT_P(tl, 3, 19, PP, __VA_ARGS__) \
  NAT_P(tl, 3, 27, PP, __VA_ARGS__)
  NAT_P3(1, 4, 2, 2, 1, 256, 2, 2)
  NAT_P3(1, 3, 4, 2, 1, 256, 1, 2)
  NAT_P3(1, 2, 4, 2, 2, 256, 1, 4)
  NAT_P(1, 2, 9, 4, 4, 4, 1, 256, 1, 2)
  NAT_P(1, 2, 9, 3, 4, 4, 1, 256, 1, 3)
  NAT_P(1, 2, 9, 2, 4, 4, 1, 128, 1, 4)
  NAT_P(2, 2, 9, 2, 8, 8, 1, 256, 1, 4)
  if constexpr (sizeof(T) == 4) {
    NAT_P3(2, 4, 4, 2, 1, 256, 2, 2)
    NAT_P3(2, 3, 4, 2, 2, 256, 1, 2)
    NAT_P3(2, 2, 8, 4, 2, 256, 1, 4)
    NAT_P(2, 2, 9, 4, 8, 4, 1, 256, 1, 2)
  }
#undef NAT_P3
#undef NAT_P
  return NAT_ERR_UNSUPPORTED;
}

template <typename F>
static int push_dispatch(const nat_ctx* ctx, int tile, F&& f) {
  return ctx->fp32 ? push_dispatch<float>(tile, ctx->Q, ctx->p, f) : push_dispatch<double>(tile, ctx->Q, ctx->p, f);
}

// Cells of the workgroups that a tile takes for the mesh, those beyond a ragged one included.
static int64_t push_cells(const nat_ctx* ctx, int tile) {
  const int* N = ctx->desc.ncells;
  int64_t cells = 0;
  push_dispatch(ctx, tile, [&](auto tl) {
    using L = decltype(tl);
    const auto up = [](int n, int c) { return (int64_t)((n + c - 1) / c) * c; };
    cells = up(N[0], L::CX) * up(N[1], L::CY) * (L::D == 3 ? up(N[2], L::CZ) : 1);
    return 0;
  });
  return cells;
}

// Whether k_sl_struct's 16 x 8 x 8 tiles (3D, p = 2 and 4) fill one round of the CUs: more than
// 5/6 of it, and no second one.
static bool push_one_round(const nat_ctx* ctx) {
  if (ctx->p == 3) return false;
  const int64_t tiles = (int64_t)((ctx->nu[0] + 15) / 16) * ((ctx->nu[1] + 7) / 8) * ((ctx->nu[2] + 7) / 8);
  return tiles <= ctx->n_cu && 6 * ctx->n_store >= 5 * (int64_t)ctx->n_cu * 1024;
}

// Tile of a context: 1 the small one, 2 the large one, 0 where k_sl_struct is faster. While the
// small tiles leave CUs idle, a step lasts as long as one workgroup does, and less work per
// workgroup wins; past a few workgroups per CU the share of nodes collided twice (NN over the
// tile's nodes) and the length of the stored lines decide, and with them the cells that the tiles
// hold beyond a ragged mesh: boxes a few cells thin stay with the small tile (2 x 32 x 25 cells,
// D3Q27 p=4 FP32: 15.1 / 12.3 / 18.2). k_sl_struct pays whole rounds of a tile of 1024 nodes per
// CU, so it is at its best where a mesh fills one (p=4 16^3, p=2 32^3 cells; from 5/6 of it on the
// other form is 3-8% ahead or behind), and in FP64 its longer lines win at p=4, and beyond the
// Infinity Cache at p=2.
// Cubic boxes, us per step in k_sl_struct / small / large tile (runs of 32 to 100 steps on a warm
// card, one MI355X; -: no such tile):
//   D3Q27 p=4 FP32   8^3 cells 14.1/ 9.2/11.8   12^3 17.4/14.3/13.8   16^3 20.8/25.0/20.3   30^3 221/171/139
//             FP64   8^3       16.0/10.3/ -     11^3 21.3/20.0/ -     12^3 18.8/21.3/ -     16^3 28.4/40.7/ -
//   D3Q19 p=4 FP32   8^3        9.4/ 7.0/ 8.4   12^3 11.0/10.0/ 9.1   16^3 13.4/18.5/14.0   24^3 47.8/56.2/42.2
//             FP64   8^3       10.1/ 7.7/ -     11^3 14.3/11.8/ -     12^3 12.5/12.8/ -     16^3 18.5/24.3/ -
//   D3Q19 p=3 FP32  16^3       13.9/ 8.7/ 8.7   21^3 32.5/16.7/14.8   32^3 66.5/41.1/37.9
//             FP64  24^3       35.1/30.1/ -     28^3 57.5/39.9/ -     32^3 83.9/78.0/ -
//   D3Q27 p=2 FP32  16^3       15.1/ 6.2/11.7   30^3 22.4/18.1/20.0   32^3 20.3/23.1/19.5   48^3 75.8/78.3/64.6
//             FP64  16^3       16.3/ 6.6/ -     30^3 26.6/23.2/ -     32^3 26.6/29.1/ -     40^3 60.0/48.0/ -
//   D3Q19 p=2 FP32  24^3       12.4/ 8.6/ 9.6   30^3 15.6/13.3/14.6   32^3 14.1/16.1/14.1   48^3 50.8/49.2/44.4
//             FP64  30^3       17.9/16.2/ -     32^3 17.7/18.7/ -     40^3 39.0/32.6/ -     48^3 65.5/73.9/ -
//   D2Q9  p=4 FP32   32^2       5.8/ 4.2/ 4.9   100^2 8.9/ 6.5/ 6.9   128^2 7.5/ 8.3/ 7.3   256^2 26.1/23.5/19.8
//             FP64   32^2       6.2/ 4.3/ -     100^2 9.6/ 7.7/ -     128^2 9.5/10.5/ -
//   D2Q9  p=2 FP32   64^2       5.7/ 3.3/ 4.0   128^2 5.6/ 4.0/ 4.1   256^2 7.6/ 7.7/ 7.0
static int push_tile(const nat_ctx* ctx) {
  const int* N = ctx->desc.ncells;
  const int64_t cells = (int64_t)N[0] * N[1] * (ctx->D == 3 ? N[2] : 1);
  int tile;
  if (ctx->D == 2) {
    if (ctx->p == 4)
      tile = cells <= 10240 ? 1 : (ctx->fp32 ? 2 : 0);
    else
      tile = ctx->p == 3 || cells <= 16384 ? 1 : 2;
  } else if (ctx->p == 3) {
    tile = ctx->fp32 && cells > 8192 ? 2 : 1;
  } else if (ctx->p == 2) {
    if (ctx->fp32)
      tile = cells <= 28672 ? 1 : 2;
    else
      tile = cells < 65536 && !push_one_round(ctx) ? 1 : 0;
  } else {
    if (ctx->fp32)
      tile = cells <= 1024 ? 1 : (ctx->Q == 19 && push_one_round(ctx) ? 0 : 2);
    else
      tile = cells <= 1400 ? 1 : 0;
  }
  return tile == 2 && 4 * push_cells(ctx, 2) > 5 * push_cells(ctx, 1) ? 1 : tile;
}

// The shortest run that takes the form. A run adds a launch and, with its collision, one more pass
// over the populations: 2 us up to 3 MB of them, then about 0.3 us per MB (D3Q27 p=4 32^3 FP32,
// 226 MB: 80 us), which the steps have to earn. Steps until they do, over 444 meshes, by what a
// step gains (3D p=3: 20-60%; 2D p=4: 4-30%): up to 3 MB 2; 3D p=3 2.4, p=2 and 4 7; 2D p=2 and 3
// 5, p=4 15. Where k_sl_struct's tiles fill one round the gain is 5% at most, and the first
// hundred launches lose it (D3Q27 p=4 16^3 FP32, us per step in k_sl_struct / k_sl_push: runs of
// 16 steps 21.8/23.3, 64 20.5/20.8, 128 20.6/20.0, 1000 20.9/19.9).
static int push_min_steps(const nat_ctx* ctx) {
  if (ctx->D == 3 && push_one_round(ctx)) return 96;
  if (ctx->n_store * ctx->Q * (ctx->fp32 ? 4 : 8) <= 3000000) return 2;
  if (ctx->D == 3) return ctx->p == 3 ? 3 : 8;
  return ctx->p == 4 ? 16 : 6;
}

template <typename T>
static int push_typed(nat_ctx* ctx, int tile, bool col) {
  PushArgs<T> a{};
  a.fin = (const T*)ctx->f[ctx->cur];
  a.fout = (T*)ctx->f[1 - ctx->cur];
  a.stride = ctx->stride;
  for (int i = 0; i < 3; i++) a.n[i] = ctx->nu[i];
  a.dir_bytes = (int)(ctx->stride * (int64_t)sizeof(T));
  a.all_bytes = (unsigned)(ctx->stride * (int64_t)sizeof(T) * ctx->Q);
  CollideArgs<T> ca{};
  ca.omega = (T)(1.0 / ctx->tau);
  ca.omega64 = 1.0 / ctx->tau;
  ca.rho0 = (T)(ctx->fp32 ? (ctx->desc.rho0 > 0 ? ctx->desc.rho0 : 1.0) : 0.0);
  ca.scaling = ctx->st.s;
  ca.status = ctx->d_status;
  ca.stab = ctx->stab_on();
  return push_dispatch<T>(tile, ctx->Q, ctx->p, [&](auto tl) {
    using L = decltype(tl);
    return launch_push<L::D, L::Q, L::P, T, L::CX, L::CY, L::CZ, L::NT, L::S, L::WPE>(ctx, a, ca, col);
  });
}

}  // namespace nat

// The tile exists for this context: a structured SL context with symmetric one-dimensional tables,
// populations within 32-bit buffer offsets, and a tile of this (stencil, order, storage).
bool nat_push_has(const nat_ctx* ctx, int tile) {
  if (ctx->desc.scheme != NAT_SL || ctx->desc.compressible || ctx->backend != NAT_BACKEND_STRUCTURED || !ctx->ax_sym ||
      !ctx->ax_w || ctx->stride * (ctx->fp32 ? 4 : 8) * ctx->Q >= (int64_t)0xffffffffu)
    return false;
  return nat::push_dispatch(ctx, tile, [](auto) { return 0; }) == 0;
}

// Form of a run of nsteps steps: 0 k_sl_struct, else the tile of the collide-then-stream form.
int nat_push_form(const nat_ctx* ctx, int nsteps) {
  if (nsteps < 2 || !nat_push_has(ctx, 1)) return 0;
  if (ctx->form_pref >= 0) return ctx->form_pref;
  if (nsteps < nat::push_min_steps(ctx)) return 0;
  return ctx->push_pref >= 0 ? ctx->push_pref : nat::push_tile(ctx);
}

// The rule's form of a long run.
int nat_push_tile(const nat_ctx* ctx) { return nat_push_has(ctx, 1) ? nat::push_tile(ctx) : 0; }

// One launch from f[cur] into f[1 - cur]: collide (when col) and stream. advance: the written
// buffer becomes the current one.
int nat_launch_sl_push(nat_ctx* ctx, int tile, bool col, bool advance) {
  const int rc = ctx->fp32 ? nat::push_typed<float>(ctx, tile, col) : nat::push_typed<double>(ctx, tile, col);
  if (rc == 0 && advance) ctx->cur = 1 - ctx->cur;
  return rc;
}
