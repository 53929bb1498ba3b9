// z4c_fused.hpp -- the Z4c right-hand side of a brick of vertices in one
// kernel: finite differences and algebra, no derivative slots in memory.
//
// A workgroup takes a brick of 17 x 5 x 3 interior vertices, one per thread,
// and the 22 fields one after another.  A field's window (the brick +-4) is
// loaded straight into LDS while the field before it is worked on (two
// windows); every thread forms its stencils from the window, and, for the
// fields with second derivatives, from the derived planes Dx_y and Dx_z that
// the threads write to LDS in between (the mixed derivatives are the
// reference's nested Dx(a, Dx(b, u)), a < b).  The algebra takes each field's
// derivatives as they come, so that at most about 100 values of the vertex are
// live: 256 VGPRs without a vector spill, two waves per SIMD (87 scalars wait in
// lanes of vector registers).
//
// Against the two-pass form (stencil pass writing 106 values a vertex, algebra
// pass reading them back: 67 GB of HBM traffic per stage of 2048 blocks of
// 16^3 .. 32^3 cells, 17.0 ms) a stage moves 37 GB (25.4 read, 11.5 written:
// the windows' halos come mostly from L2) and takes 11.4 ms.  Of that, 5.5 ms
// are FP64 and integer issue (8000 instructions a wave, no FMA) and 4 to 5 ms
// LDS reads (55 a vertex and field with second derivatives), which the
// barriers between fields keep from overlapping fully.  One 32^3 block's
// right-hand side: 79 -> 40 us.
//
// What it takes to get there, each measured: no vector load and no spill
// reload between the window loads and the next field (the memory counter is
// in order, so either waits for the whole window: 82 and 62 ms a step); a
// lane's window offsets kept in LDS, not formed anew for every field (52.1 ->
// 51.1 ms a step); barriers that wait for LDS traffic only; every load of the
// update issued before its first store (68 -> 60 ms).
//
// The operation order is the two-pass form's throughout
// (z4c_rhs_point.hpp, z4c_stencil.hpp): results are equal bit for bit.
#pragma once

#include "z4c_device.hpp"
#include "z4c_rhs_point.hpp"
#include "z4c_stencil.hpp"

namespace z4c {

// Brick of at most BX x BY x BZ interior vertices, one per thread.
template <int BX_, int BY_, int BZ_, int TH>
struct FusedCfg {
  static constexpr int BX = BX_, BY = BY_, BZ = BZ_, THREADS = TH;
  static_assert(BX * BY * BZ <= TH, "one vertex per thread");
  static constexpr int WAVES = TH / 64;
  // field window: the brick +-4, rows padded to whole 16-byte pairs
  static constexpr int PX = (BX + 8 + 1) / 2 * 2, PY = BY + 8, PZ = BZ + 8;
  static constexpr int PLANE = PX * PY;
  // a window in 16-byte pairs, 64 a load instruction, dealt to the waves in turn
  static constexpr int PAIRS = PLANE * PZ / 2, NLD = (PAIRS + 63) / 64;
  static constexpr int ROUNDS = (NLD + WAVES - 1) / WAVES;
  static_assert(ROUNDS == 8, "the offsets of a lane are two 16-byte reads");
  static constexpr int WIN = PLANE * PZ;  // doubles
  // Dx_y on the brick +-3 in x; Dx_z on the brick +-3 in x and in y
  static constexpr int DX = BX + 6;
  static constexpr int DYP = DX * BY, DZP = DX * (BY + 6);
  static constexpr int NDY = DYP * BZ, NDZ = DZP * BZ;
  // halo values of the derived planes: Dx_y and Dx_z at x +-3, Dx_z at y +-3
  static constexpr int HX = 6 * BY * BZ, HY = BX * 6 * BZ;
  static constexpr int SX = (HX + 63) / 64, SY = (HY + 63) / 64;  // wave slots
  static constexpr int HROUNDS = (2 * SX + SY + WAVES - 1) / WAVES;
  static constexpr int LDS = (2 * WIN + NDY + NDZ) * 8 + (HROUNDS + 1 + ROUNDS) * TH * 4;
  static_assert(LDS <= 80 * 1024, "two workgroups per CU");
};
// 17 vertices along x are a row of the 16-cell blocks most runs are made of,
// and half of a 32-cell one.  Measured on 2048 blocks of 17^3 .. 33^3 vertices:
// one workgroup of 512 threads per CU on 17 x 6 x 5 bricks 62.1 ms a step, two
// of 256 on 17 x 5 x 3 51.1 (at a barrier or a load of one, the other runs).
using FuCfg = FusedCfg<17, 5, 3, 256>;

struct FusedTile {
  int block;
  int i0, j0, k0, ni, nj, nk;  // interior-relative origin and extents
};

struct FusedArgs {
  const DevBlock* blocks;
  const FusedTile* tiles;
  int ntiles;
  const double* u;    // state read; rhs and out lie apart from it (every brick reads its
                      // neighbours' vertices).  In two passes out may be u itself
  const double* mat;  // may be null
  RhsParams o;
  int cowling;        // zero right-hand side (two passes only)
  int sommerfeld;     // apply the Sommerfeld rows on flagged faces (two passes: always)
  double* rhs;        // right-hand side (null: stage update)
  // stage update
  const double* un;
  int un_int;
  double* acc;
  double* out;
  double* keep;
  double wa, wb;
  int stage;
  int alg;            // AlgConstr of the point at the end
  double eps_floor;
  int tf_force, force_reg;
  int ls;             // low-storage update
  double ls_w[4];
  int ls_last;
};

// Vertex of thread `tid` in its brick; threads past it take vertex 0 (they
// form the same values and store none) and return false.
template <class C>
__device__ __forceinline__ bool fused_vertex(const FusedTile& T, int tid, int& tx, int& ty,
                                             int& tz) {
  tx = tid % C::BX;
  ty = tid / C::BX % C::BY;
  tz = tid / (C::BX * C::BY);
  const bool in = tx < T.ni && ty < T.nj && tz < T.nk;
  if (!in) tx = ty = tz = 0;
  return in;
}

// A copy the compiler cannot tell from another value.
template <class T>
__device__ __forceinline__ T opaque(T v) {
  asm volatile("" : "+v"(v));
  return v;
}

// A wave-uniform double in scalar registers.
__device__ __forceinline__ double uniform(double v) {
  const long long b = __builtin_bit_cast(long long, v);
  const unsigned lo = __builtin_amdgcn_readfirstlane((int)b);
  const unsigned hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __builtin_bit_cast(double, (long long)(((unsigned long long)hi << 32) | lo));
}

typedef __attribute__((address_space(3))) void* lds_ptr;

// Barrier that waits for this wave's LDS reads and writes only: loads into
// LDS issued before it stay in flight (the compiler's fence would wait for
// them too).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// st_lx without a branch: the reference's right-biased sum is minus the
// left-biased one of the reversed points, so the points are selected instead
// of the sums (exact: only signs move).
__device__ __forceinline__ double fu_lx(const double* v, double lidx, double vx) {
  const bool l = vx < 0;
  double w[7];
#pragma unroll
  for (int m = 0; m < 7; ++m) w[m] = m == 4 ? v[4] : (l ? v[m] : v[8 - m]);
  double dl = w[0];
  dl += -8.0 * w[1];
  dl += 30.0 * w[2];
  dl += -80.0 * w[3];
  dl += 35.0 * w[4];
  dl += 24.0 * w[5];
  dl += -2.0 * w[6];
  return -fabs(vx) * dl * lidx;
}

// The kernel's arguments, read where they are used: get() is opaque to the
// compiler, which otherwise loads every argument at the start and spills the
// scalar registers that hold them.
template <class A>
struct KernArgs {
  typedef const __attribute__((address_space(4))) A* Ptr;
  __device__ __forceinline__ const __attribute__((address_space(4))) A& get() const {
    Ptr p = (Ptr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *p;
  }
};

// Keeps a value's evaluation at this place: without it the compiler moves the
// algebra behind the last barrier, next to its uses, and holds every
// derivative until there.
__device__ __forceinline__ void pin(double& v) { asm volatile("" : "+v"(v)); }
template <int M>
__device__ __forceinline__ void pin(double (&v)[M]) {
#pragma unroll
  for (int q = 0; q < M; ++q) pin(v[q]);
}
template <int M, int K>
__device__ __forceinline__ void pin(double (&v)[M][K]) {
#pragma unroll
  for (int q = 0; q < M; ++q) pin(v[q]);
}

// order in which the fields are taken: the curvature's first, the shift's
// last (its first derivatives enter the finished terms)
__host__ __device__ constexpr int fu_field(int q) {
  constexpr int o[NVAR] = {V_GAMX, V_GAMX + 1, V_GAMX + 2, V_GXX, V_GXX + 1, V_GXX + 2,
                           V_GXX + 3, V_GXX + 4, V_GXX + 5, V_CHI, V_ALPHA, V_KHAT, V_THETA,
                           V_AXX, V_AXX + 1, V_AXX + 2, V_AXX + 3, V_AXX + 4, V_AXX + 5,
                           V_BETAX, V_BETAX + 1, V_BETAX + 2};
  return o[q];
}
__host__ __device__ constexpr bool fu_mixed(int f) {
  return dkind(f) == DK_FULL || dkind(f) == DK_METRIC;
}

// fields whose LD term waits in the destination until the shift's derivatives
// are known
__host__ __device__ constexpr bool fu_stash(int f) {
  return f != V_KHAT && f != V_THETA && f < V_ALPHA;
}

template <class C>
struct FusedPoint {
  const double* ub;       // state of the block
  int N;                  // vertices of the block
  double c1[3], c2[3], cd[3];  // stencil scalings (wave-uniform)
  double* win[2];         // field windows
  double* der;            // derived planes: Dx_y, then Dx_z
  int wave, lane;
  const int4* offs;       // byte offsets of this lane's pairs, one a round (LDS); bit 31: no
                          // field needs the pair, bit 30: only fields with mixed
                          // derivatives (either is out of the field's range)
  int o;                     // this vertex in a window
  const int* halo;        // this thread's vertex in the derived planes (last entry:
                          // Dx_y's index | Dx_z's << 16) and its halo values (LDS, one a round): window index |
                          // derived-plane index << 16 (negative: none)
  unsigned p8;            // this vertex in a field, bytes (no vertex: out of range)
  double* dst;            // destination of the block: holds LD terms (fu_stash)
                          // until the end
  double pend;            // LD of the field before, stored past the next barrier
  double diss, bx, by, bz;

  __device__ __forceinline__ double stashed(int f) const {
    return bload(make_buf(dst + (long long)f * N, (long long)N * 8), p8, 0);
  }
  // field f at the vertex, from memory
  __device__ __forceinline__ double at(int f) const {
    return bload(make_buf(ub + (long long)f * N, (long long)N * 8), p8, 0);
  }

  // starts the loads of field F's window
  template <int F, int PAR>
  __device__ __forceinline__ void fetch() const {
    const Buf U = make_buf(ub + (long long)F * N, (long long)N * 8);
    const int4 a = offs[0], b = offs[C::THREADS];
    const int v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int r = 0; r < C::ROUNDS; ++r) {
      const int q = r * C::WAVES + wave;
      // every lane writes LDS, needed or not: none may past the window
      if ((r + 1) * C::WAVES * 64 <= C::PAIRS || q * 64 + lane < C::PAIRS)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(U.r, (lds_ptr)(win[PAR] + q * 128), 16,
                                                 fu_mixed(F) ? v[r] & ~(1 << 30) : v[r], 0, 0, 0);
    }
  }

  // field Q of the order: d first derivatives, dd second derivatives, the
  // advective sum L and the KO sum D; returns the field at the vertex
  template <int Q>
  __device__ __forceinline__ double field(double* d, double* dd, double& L, double& D) {
    constexpr int F = fu_field(Q);
    constexpr int PAR = Q & 1;
    constexpr bool mixed = fu_mixed(F);
    constexpr bool grad = dkind(F) != DK_ADV;
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's part of the window is in LDS
    lds_barrier();
    if (Q + 1 < NVAR) fetch<fu_field(Q + 1 < NVAR ? Q + 1 : 0), (Q + 1) & 1>();
    if (Q > 0 && fu_stash(fu_field(Q > 0 ? Q - 1 : 0)))
      bstore(make_buf(dst + (long long)fu_field(Q > 0 ? Q - 1 : 0) * N, (long long)N * 8), pend, p8,
             0);
    const double* c = win[PAR] + opaque(o);
    const int wyz = mixed ? halo[C::HROUNDS * C::THREADS] : 0;
    const int wy = wyz & 0xffff, wz = wyz >> 16;
    double v[9];
#pragma unroll
    for (int m = 0; m < 9; ++m) v[m] = c[m - 4];
    const double u0 = v[4];
    if (grad) d[0] = st_dx(v, c1[0]);
    if (mixed) dd[0] = st_dxx(v, c2[0]);
    L = fu_lx(v, c1[0], bx);
    D = st_diss(v, cd[0], diss);
#pragma unroll
    for (int m = 0; m < 9; ++m) v[m] = c[(m - 4) * C::PX];
    if (grad) d[1] = st_dx(v, c1[1]);
    if (mixed) dd[3] = st_dxx(v, c2[1]);
    L += fu_lx(v, c1[1], by);
    D += st_diss(v, cd[1], diss);
#pragma unroll
    for (int m = 0; m < 9; ++m) v[m] = c[(m - 4) * C::PLANE];
    if (grad) d[2] = st_dx(v, c1[2]);
    if (mixed) dd[5] = st_dxx(v, c2[2]);
    L += fu_lx(v, c1[2], bz);
    D += st_diss(v, cd[2], diss);
    if (mixed) {
      der[wy] = d[1];
      der[wz] = d[2];
#pragma unroll
      for (int r = 0; r < C::HROUNDS; ++r) {
        const int q = r * C::WAVES + wave;  // the wave's slot: Dx_y at first, then Dx_z
        if ((r + 1) * C::WAVES <= 2 * C::SX + C::SY || q < 2 * C::SX + C::SY) {
          const int hd = halo[r * C::THREADS];
          const double* h = win[PAR] + (hd & 0xffff);
          const int st = q < C::SX ? C::PX : C::PLANE;
#pragma unroll
          for (int m = 0; m < 7; ++m)
            if (m != 3) v[m + 1] = h[(m - 3) * st];
          const double x = st_dx(v, q < C::SX ? c1[1] : c1[2]);
          if (hd >= 0) der[hd >> 16] = x;
        }
      }
      lds_barrier();
#pragma unroll
      for (int m = 1; m < 8; ++m)
        if (m != 4) v[m] = der[wy + (m - 4)];
      dd[1] = st_dx(v, c1[0]);  // d_x(d_y u)
#pragma unroll
      for (int m = 1; m < 8; ++m)
        if (m != 4) v[m] = der[wz + (m - 4)];
      dd[2] = st_dx(v, c1[0]);  // d_x(d_z u)
#pragma unroll
      for (int m = 1; m < 8; ++m)
        if (m != 4) v[m] = der[wz + (m - 4) * C::DX];
      dd[4] = st_dx(v, c1[1]);  // d_y(d_z u)
    }
    __builtin_amdgcn_sched_barrier(0);
    return u0;
  }
};

// The right-hand side of one vertex into k: fields in fu_field's order, each
// term in the reference's operation order (z4c_rhs_point.hpp's).
template <class C>
__device__ __forceinline__ void fused_rhs(FusedPoint<C>& P, const KernArgs<FusedArgs>& ka,
                                          const double* mat, double (&k)[NVAR]) {
  double &kchi = k[V_CHI], &kK = k[V_KHAT], &kT = k[V_THETA], &kal = k[V_ALPHA];
  double *kg = k + V_GXX, *kA = k + V_AXX, *kG = k + V_GAMX, *kb = k + V_BETAX;
  auto m = [&](int f) {
    return bload(make_buf(mat + (long long)f * P.N, (long long)P.N * 8), P.p8, 0);
  };
  double d[3], dd[6], L, D;

  double gdd[6], guu[6];
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) gdd[ab] = P.at(V_GXX + ab);
  {
    const double detg = det3(gdd);
    inv3(1.0 / detg, gdd, guu);
  }
  // ------------------------------------------------------------- Gamma~
  double dGam[3][3];  // [component][direction]
#define Z4C_GAM(c)                                     \
  P.template field<c>(dGam[c], dd, L, D);              \
  pin(dGam[c]);                                        \
  P.pend = L + D;                                      \
  pin(P.pend);
  Z4C_GAM(0) Z4C_GAM(1) Z4C_GAM(2)
#undef Z4C_GAM
  // -------------------------------------------------------------- metric
  double dg[6][3], Pab[6];
#define Z4C_MET(ab)                                                               \
  P.template field<3 + ab>(dg[ab], dd, L, D);                                     \
  P.pend = L + D;                                                                 \
  {                                                                               \
    double t = 0.0;                                                               \
    _Pragma("unroll") for (int c = 0; c < 3; ++c)                                 \
      _Pragma("unroll") for (int e = c; e < 3; ++e)                               \
        t += ((c == e) ? 0.5 : 1.0) * guu[sym(c, e)] * dd[sym(c, e)];             \
    Pab[ab] = t;                                                                  \
  }                                                                               \
  pin(dg[ab]);                                                                    \
  pin(Pab[ab]);                                                                   \
  pin(P.pend);
  Z4C_MET(0) Z4C_MET(1) Z4C_MET(2) Z4C_MET(3) Z4C_MET(4) Z4C_MET(5)
#undef Z4C_MET
  double Gudd[3][6], Gu[3], RR[6];
  {
    double Gddd[3][6];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = a; b < 3; ++b)
          Gddd[c][sym(a, b)] = 0.5 * (dg[sym(b, c)][a] + dg[sym(a, c)][b] - dg[sym(a, b)][c]);
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int ab = 0; ab < 6; ++ab) {
        double t = 0.0;
#pragma unroll
        for (int e = 0; e < 3; ++e) t += guu[sym(c, e)] * Gddd[e][ab];
        Gudd[c][ab] = t;
      }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      double t = 0.0;
#pragma unroll
      for (int b = 0; b < 3; ++b)
#pragma unroll
        for (int c = b; c < 3; ++c)
          t += ((b == c) ? 1.0 : 2.0) * guu[sym(b, c)] * Gudd[a][sym(b, c)];
      Gu[a] = t;
    }
    __builtin_amdgcn_sched_barrier(0);
    // conformal Ricci (calculate_z4c_rhs.cpp:357-396); the linear terms of all
    // components first, which frees dGam and Pab
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = a; b < 3; ++b) {
        double r = 0.0;
#pragma unroll
        for (int c = 0; c < 3; ++c)
          r += 0.5 * (gdd[sym(c, a)] * dGam[c][b] + gdd[sym(c, b)] * dGam[c][a] +
                      Gu[c] * (Gddd[a][sym(b, c)] + Gddd[b][sym(a, c)]));
        r -= Pab[sym(a, b)];
        RR[sym(a, b)] = r;
      }
    pin(RR);
    pin(Gddd);
    pin(Gudd);
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = a; b < 3; ++b) {
        double r = RR[sym(a, b)];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int e = 0; e < 3; ++e)
#pragma unroll
            for (int f = 0; f < 3; ++f)
              r += guu[sym(c, e)] * (Gudd[f][sym(c, a)] * Gddd[b][sym(f, e)] +
                                     Gudd[f][sym(c, b)] * Gddd[a][sym(f, e)] +
                                     Gudd[f][sym(a, e)] * Gddd[f][sym(c, b)]);
        RR[sym(a, b)] = r;
        pin(RR[sym(a, b)]);
        __builtin_amdgcn_sched_barrier(0);
      }
  }
  pin(Gudd);
  pin(Gu);
  pin(RR);
  // ----------------------------------------- conformal factor (:402-458)
  double dchi[3], dphi[3];
  const double chi = P.template field<9>(dchi, dd, L, D);
  P.pend = L + D;
  pin(P.pend);
  double oochi;
  {
  const auto& o = ka.get().o;
  const double pw = o.chi_psi_power;
  const double oochi_psi_power = 1.0 / pw;
  oochi = 1.0 / dmax(chi, o.chi_div_floor);
#pragma unroll
  for (int a = 0; a < 3; ++a) dphi[a] = dchi[a] * oochi * oochi_psi_power;
  {
    double Ddphi[6];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = a; b < 3; ++b) {
        double t = dd[sym(a, b)] * oochi * oochi_psi_power - pw * dphi[a] * dphi[b];
#pragma unroll
        for (int c = 0; c < 3; ++c) t -= Gudd[c][sym(a, b)] * dphi[c];
        Ddphi[sym(a, b)] = t;
      }
    double trphi = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int e = c; e < 3; ++e)
        trphi += ((c == e) ? 1.0 : 2.0) * guu[sym(c, e)] *
                 (Ddphi[sym(c, e)] + 2. * dphi[c] * dphi[e]);
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = a; b < 3; ++b)
        RR[sym(a, b)] = RR[sym(a, b)] + (4. * dphi[a] * dphi[b] - 2. * Ddphi[sym(a, b)] -
                                         2. * gdd[sym(a, b)] * trphi);
  }
  }
  pin(RR);
  pin(dchi);
  pin(dphi);
  pin(oochi);
  // ------------------------------------------------ D_a D_b alpha (:484-532)
  double dalpha[3], tA[6];
  const double lapse = P.template field<10>(dalpha, dd, L, D);
  double LDal, Ddalpha = 0.0, R = 0.0;
  {
    const auto& o = ka.get().o;
    const double pw = o.chi_psi_power;
    const double chi_guarded = dmax(chi, o.chi_div_floor);
    const double oopsi4 = (pw == -4.) ? chi_guarded : pow(chi_guarded, -4. / pw);
    const double alpha = lapse;
    LDal = o.lapse_advect * L + D;
    double DDa[6];
    double Dda = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int e = 0; e < 3; ++e) Dda += guu[sym(c, e)] * dphi[c] * dalpha[e];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = a; b < 3; ++b) {
        double t = dd[sym(a, b)] - 2. * (dphi[a] * dalpha[b] + dphi[b] * dalpha[a]) +
                   2. * gdd[sym(a, b)] * Dda;
#pragma unroll
        for (int c = 0; c < 3; ++c) t -= Gudd[c][sym(a, b)] * dalpha[c];
        DDa[sym(a, b)] = t;
      }
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = a; b < 3; ++b) {
        Ddalpha += ((a == b) ? 1.0 : 2.0) * oopsi4 * guu[sym(a, b)] * DDa[sym(a, b)];
        R += ((a == b) ? 1.0 : 2.0) * oopsi4 * guu[sym(a, b)] * RR[sym(a, b)];
      }
#pragma unroll
    for (int ab = 0; ab < 6; ++ab) {
      double t = oopsi4 * (-DDa[ab] + alpha * RR[ab]);
      t -= (1. / 3.) * gdd[ab] * (-Ddalpha + alpha * R);
      tA[ab] = t;
    }
  }
  pin(tA);
  pin(dalpha);
  pin(LDal);
  pin(Ddalpha);
  pin(R);
  // -------------------------------------------- Khat, Theta and A~ (:536-711)
  double dK[3], dT[3], LDK, LDT;
  const double Khat = P.template field<11>(dK, dd, L, D);
  LDK = L + D;
  pin(dK);
  pin(LDK);
  const double Theta = P.template field<12>(dT, dd, L, D);
  LDT = L + D;
  pin(LDT);
#pragma unroll
  for (int b = 0; b < 3; ++b) dK[b] = 2. * dK[b] + dT[b];
  pin(dK);
  double Add[6];
#define Z4C_AXX(ab)                                    \
  Add[ab] = P.template field<13 + ab>(d, dd, L, D);    \
  pin(Add[ab]);                                        \
  P.pend = L + D;                                      \
  pin(P.pend);
  Z4C_AXX(0) Z4C_AXX(1) Z4C_AXX(2) Z4C_AXX(3) Z4C_AXX(4) Z4C_AXX(5)
#undef Z4C_AXX
  double Auu[6], DA[3];
  {
    const auto& o = ka.get().o;
    const double k1 = o.damp_kappa1, k2 = o.damp_kappa2;
    const double chi_pow_DA_u = -6.0 / o.chi_psi_power;
    const double alpha = lapse;
    double Aud[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        double t = 0.0;
#pragma unroll
        for (int e = 0; e < 3; ++e) t += guu[sym(c, e)] * Add[sym(e, b)];
        Aud[c][b] = t;
      }
    double AA[6];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = a; b < 3; ++b) {
        double t = 0.0;
#pragma unroll
        for (int c = 0; c < 3; ++c) t += Add[sym(a, c)] * Aud[c][b];
        AA[sym(a, b)] = t;
      }
    double trAA = 0.0;
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = a; b < 3; ++b)
        trAA += ((a == b) ? 1.0 : 2.0) * guu[sym(a, b)] * AA[sym(a, b)];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = a; b < 3; ++b) {
        double t = 0.0;
#pragma unroll
        for (int c = 0; c < 3; ++c) t += guu[sym(b, c)] * Aud[a][c];
        Auu[sym(a, b)] = t;
      }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      double t = 0.0;
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        t -= chi_pow_DA_u * Auu[sym(a, b)] * dchi[b] * oochi;
        t -= (1. / 3.) * guu[sym(a, b)] * dK[b];
      }
#pragma unroll
      for (int b = 0; b < 3; ++b)
#pragma unroll
        for (int c = b; c < 3; ++c)
          t += ((b == c) ? 1.0 : 2.0) * Gudd[a][sym(b, c)] * Auu[sym(b, c)];
      DA[a] = t;
    }
    const double K = Khat + 2. * Theta;
    const double Ht = R + (2. / 3.) * (K * K) - trAA;
    kK = -Ddalpha + alpha * (trAA + (1. / 3.) * (K * K)) + LDK + k1 * (1 - k2) * alpha * Theta;
    kT = LDT + alpha * (0.5 * Ht - (2. + k2) * k1 * Theta);
    const double f = o.lapse_oplog * o.lapse_harmonicf + o.lapse_harmonic * alpha;
    kal = (LDal - f * alpha * (Khat + 2 * o.lapse_K * Theta));
#pragma unroll
    for (int ab = 0; ab < 6; ++ab) tA[ab] += alpha * (K * Add[ab] - 2. * AA[ab]);
  }
  pin(tA);
  pin(Auu);
  pin(DA);
  pin(kK);
  pin(kT);
  pin(kal);
  // -------------------------------------------------------------- shift
  double dbeta[3][3];     // [direction][component]
  double ddb[3][6];
#define Z4C_BETA(a)                                       \
  P.template field<19 + a>(d, ddb[a], L, D);              \
  kb[a] = ka.get().o.shift_advect * L + D;                         \
  dbeta[0][a] = d[0];                                     \
  dbeta[1][a] = d[1];                                     \
  dbeta[2][a] = d[2];                                     \
  pin(ddb[a]);                                            \
  pin(kb[a]);                                             \
  pin(dbeta[0][a]);                                       \
  pin(dbeta[1][a]);                                       \
  pin(dbeta[2][a]);
  Z4C_BETA(0) Z4C_BETA(1) Z4C_BETA(2)
#undef Z4C_BETA
  double dbeta_div = 0.0;
#pragma unroll
  for (int a = 0; a < 3; ++a) dbeta_div += dbeta[a][a];
  // the fields at the vertex again (not held through the shift's stencils)
  const auto& o = ka.get().o;
  const double pw = o.chi_psi_power, k1 = o.damp_kappa1;
  const double alpha = P.at(V_ALPHA);
  const double chi_guarded = dmax(P.at(V_CHI), o.chi_div_floor);
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) gdd[ab] = P.at(V_GXX + ab);
  {
    const double detg = det3(gdd);
    inv3(1.0 / detg, gdd, guu);
  }
  {
    const double K = P.at(V_KHAT) + 2. * P.at(V_THETA);
    double Lchi = P.stashed(V_CHI);
    Lchi += (1. / 6.) * pw * chi_guarded * dbeta_div;
    kchi = Lchi - (1. / 6.) * pw * chi_guarded * alpha * K;
  }
  const double oopsi4 = (pw == -4.) ? chi_guarded : pow(chi_guarded, -4. / pw);
  double Str = 0.0;
  if (mat) {
    const double rho = m(M_RHO);
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = a; b < 3; ++b)
        Str += ((a == b) ? 1.0 : 2.0) * oopsi4 * guu[sym(a, b)] * m(M_SXX + sym(a, b));
    kK += 4 * M_PI * alpha * (Str + rho);
    kT -= 8. * M_PI * alpha * rho;
  }
  __builtin_amdgcn_sched_barrier(0);
  // -------------------------------------------------- Gamma~ (:640-729)
  {
    double ddbeta_d[3];  // (1/3) sum_b d_a d_b beta^b
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      double t = 0.0;
#pragma unroll
      for (int b = 0; b < 3; ++b) t += (1. / 3.) * ddb[b][sym(a, b)];
      ddbeta_d[a] = t;
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      double LGam = P.stashed(V_GAMX + a);
      LGam += (2. / 3.) * Gu[a] * dbeta_div;
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        LGam += guu[sym(a, b)] * ddbeta_d[b] - Gu[b] * dbeta[b][a];
#pragma unroll
        for (int c = b; c < 3; ++c)
          LGam += ((b == c) ? 1.0 : 2.0) * guu[sym(b, c)] * ddb[a][sym(b, c)];
      }
      double t = 2. * alpha * DA[a] + LGam;
      t -= 2. * alpha * k1 * (P.at(V_GAMX + a) - Gu[a]);
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        t -= 2. * Auu[sym(a, b)] * dalpha[b];
        if (mat) t -= 16. * M_PI * alpha * guu[sym(a, b)] * m(M_SX + b);
      }
      kG[a] = t;
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // ------------------------------------------- g~ and A~ (:671-754)
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) Add[ab] = P.at(V_AXX + ab);
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = a; b < 3; ++b) {
      const int ab = sym(a, b);
      double Lg = P.stashed(V_GXX + ab);
      double LA = P.stashed(V_AXX + ab);
      Lg -= (2. / 3.) * gdd[ab] * dbeta_div;
      LA -= (2. / 3.) * Add[ab] * dbeta_div;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        Lg += dbeta[a][c] * gdd[sym(b, c)];
        LA += dbeta[b][c] * Add[sym(a, c)];
        Lg += dbeta[b][c] * gdd[sym(a, c)];
        LA += dbeta[a][c] * Add[sym(b, c)];
      }
      double t = tA[ab];
      t += LA;
      if (mat)
        t -= 8. * M_PI * alpha * (oopsi4 * m(M_SXX + ab) - (1. / 3.) * Str * gdd[ab]);
      kg[ab] = -2. * alpha * Add[ab] + Lg;
      kA[ab] = t;
    }
  __builtin_amdgcn_sched_barrier(0);
  // ------------------------------------------------------ shift (:774-902)
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double Gam_a = P.at(V_GAMX + a);
    double r = o.shift_Gamma * Gam_a + kb[a];
    if (fabs(o.shift_alpha2Gamma) > 0.0) r += o.shift_alpha2Gamma * (alpha * alpha) * Gam_a;
    if (fabs(o.shift_H) > 0.0) {
#pragma unroll
      for (int b = 0; b < 3; ++b)
        r += o.shift_H * alpha * chi_guarded * (0.5 * alpha * dchi[b] - dalpha[b]) *
             guu[sym(a, b)];
    }
    r -= o.shift_eta * P.at(V_BETAX + a);
    kb[a] = r;
  }
}

}  // namespace z4c
