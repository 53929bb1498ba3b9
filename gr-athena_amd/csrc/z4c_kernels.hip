// z4c_kernels.hip -- gfx950 kernels and the C-ABI of the batched Z4c hot path.
//
// Data layout (HBM): a buffer of `nvar` fields holds the registered blocks
// back to back; block b with point offset off_b (= sum of npts of earlier
// blocks) stores field n at element (off_b*nvar + n*npts_b + p), p the
// AthenaArray flat index i + nn1*(j + nn2*k).  One launch covers every
// block: a host-built tile table maps 256-thread workgroups to (block,
// first point) pairs of a per-block box (interior, derivative-prep region,
// or whole padded block).  Workgroup IDs are remapped so that the tiles one
// XCD receives are contiguous in the table, keeping a block's halo in one
// L2 (workgroups are dealt to the 8 XCDs round robin).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <limits>
#include <map>
#include <unordered_map>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "z4c_adjoint.hpp"
#include "z4c_device.hpp"
#include "z4c_fused.hpp"
#include "z4c_mesh.hpp"
#include "z4c_mi355x.h"
#include "z4c_refine.hpp"
#include "z4c_rhs_point.hpp"
#include "z4c_stencil.hpp"

using namespace z4c;

namespace {

thread_local std::string g_err;

// Device address of `scratch` on each GPU (z4c_history_noalloc), resolved
// once per device by z4c_ctx_create with that device current.
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
double* g_scratch_dev[MAX_DEVICES] = {};

int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

#define HIPCALL(expr)                                                        \
  do {                                                                       \
    hipError_t e_ = (expr);                                                  \
    if (e_ != hipSuccess)                                                    \
      return fail(Z4C_EHIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

// ---------------------------------------------------------------------------
// Tile decode: XCD-contiguous remap of the workgroup id, then tile -> point.
// ---------------------------------------------------------------------------
struct Launch {
  const Tile* tiles;
  const Box* boxes;
  int ntiles;
};

__device__ __forceinline__ bool tile_point(const Launch& L, int& blk, int& i,
                                           int& j, int& k) {
  const int G = gridDim.x;  // multiple of 8
  const int w = blockIdx.x;
  const int t = (w & 7) * (G >> 3) + (w >> 3);
  if (t >= L.ntiles) return false;
  const Tile T = L.tiles[t];
  blk = T.block;
  const Box bx = L.boxes[T.box];
  const int q = T.start + (int)threadIdx.x;
  const int n01 = bx.n[0] * bx.n[1];
  if (q >= n01 * bx.n[2]) return false;
  const int kk = q / n01;
  const int r = q - kk * n01;
  const int jj = r / bx.n[0];
  i = bx.lo[0] + (r - jj * bx.n[0]);
  j = bx.lo[1] + jj;
  k = bx.lo[2] + kk;
  return true;
}

__device__ __forceinline__ int flat(const DevBlock& B, int i, int j, int k) {
  return i + B.nn1 * (j + B.nn2 * k);
}

// ---------------------------------------------------------------------------
// PrepareZ4cDerivatives (src/z4c/adm_z4c.cpp:977-1013, aux fill :1044-1119)
// ---------------------------------------------------------------------------
struct PrepArgs {
  const DevBlock* blocks;
  Launch L;
  const double* u;
  double* d1;
  double* aux;  // may be null
  double chi_psi_power, chi_div_floor;
};

__global__ void __launch_bounds__(TILE) k_prep(PrepArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  const int N = B.npts;
  const double* u = a.u + B.off * NVAR;
  double* d1 = a.d1 + B.off * ND1;
  const int p = flat(B, i, j, k);
  const Buf U = make_buf(u, (long long)NVAR * N * 8);
  const Pt P = make_pt(p, B.nn1, B.nn2, N);
  const bool in_i = (i >= B.il && i <= B.iu), in_j = (j >= B.jl && j <= B.ju),
             in_k = (k >= B.kl && k <= B.ku);
  const bool inside[3] = {in_i, in_j, in_k};
#pragma unroll
  for (int dir = 0; dir < 3; ++dir) {
    if (!inside[dir]) continue;  // along `dir` only the interior is needed
    const double c = B.cidx1[dir];
    double* o = d1 + dir * 11 * N + p;
    o[F_ALPHA * N] = fd_dx(U, P, V_ALPHA, dir, c);
    o[F_CHI * N] = fd_dx(U, P, V_CHI, dir, c);
#pragma unroll
    for (int m = 0; m < 3; ++m) o[(F_BETA + m) * N] = fd_dx(U, P, V_BETAX + m, dir, c);
#pragma unroll
    for (int m = 0; m < 6; ++m) o[(F_G + m) * N] = fd_dx(U, P, V_GXX + m, dir, c);
  }
  if (a.aux == nullptr || !(in_i && in_j && in_k)) return;
  // storage.aux: physical derivatives by the chain rule (interior only)
  double* aux = a.aux + B.off * 30;
  const double pw = a.chi_psi_power;
  const double chi_g = dmax(u[V_CHI * N + p], a.chi_div_floor);
  const double oochi = 1.0 / chi_g;
  const double fac = 4.0 / pw;
  const double chi_pow = (pw == -4.) ? 0.0 : pow(chi_g, fac);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double dchi_c = d1[(c * 11 + F_CHI) * N + p];
#pragma unroll
    for (int ab = 0; ab < 6; ++ab) {
      const double dg = d1[(c * 11 + F_G + ab) * N + p];
      const double gab = u[(V_GXX + ab) * N + p];
      const double v = (pw == -4.) ? oochi * (dg - oochi * gab * dchi_c)
                                   : chi_pow * (dg + fac * oochi * gab * dchi_c);
      aux[(12 + c * 6 + ab) * N + p] = v;
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) aux[(3 + c * 3 + m) * N + p] = d1[(c * 11 + F_BETA + m) * N + p];
    aux[c * N + p] = d1[(c * 11 + F_ALPHA) * N + p];
  }
}

// ---------------------------------------------------------------------------
// Z4cRHS (+ optional fused Sommerfeld faces)
// ---------------------------------------------------------------------------
struct RhsArgs {
  const DevBlock* blocks;
  Launch L;
  const double* u;
  const double* dv;   // derivative slots from the stencil pass
  const double* mat;  // may be null
  double* rhs;
  RhsParams o;
};

template <class Out>
__device__ __forceinline__ void sommerfeld_point(const DevBlock& B, const Buf& U, const Pt& P,
                                                 const double* __restrict__ u, int i, int j,
                                                 int k, int N, Out&& out) {
  const int p = flat(B, i, j, k);
  const double sq2 = sqrt(2.);
  const double x1 = B.x0[0] + i * B.dx[0];
  const double x2 = B.x0[1] + j * B.dx[1];
  const double x3 = B.x0[2] + k * B.dx[2];
  const double r = sqrt(x1 * x1 + x2 * x2 + x3 * x3);
  const double su[3] = {x1 / r, x2 / r, x3 / r};
  double th = -u[V_THETA * N + p] / r;
  double kh = -sq2 * u[V_KHAT * N + p] / r;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    th -= su[a] * fd_ds(U, P, V_THETA, a, B.cidx1lo[a]);
    kh -= sq2 * su[a] * fd_ds(U, P, V_KHAT, a, B.cidx1lo[a]);
  }
  out(V_THETA, th);
  out(V_KHAT, kh);
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    double t = -u[(V_GAMX + a) * N + p] / r;
#pragma unroll
    for (int b = 0; b < 3; ++b) t -= su[b] * fd_ds(U, P, V_GAMX + a, b, B.cidx1lo[b]);
    out(V_GAMX + a, t);
  }
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) {
    double t = -u[(V_AXX + ab) * N + p] / r;
#pragma unroll
    for (int c = 0; c < 3; ++c) t -= su[c] * fd_ds(U, P, V_AXX + ab, c, B.cidx1lo[c]);
    out(V_AXX + ab, t);
  }
}

__device__ __forceinline__ bool on_sommerfeld_face(const DevBlock& B, int i,
                                                   int j, int k) {
  const int f = B.faces;
  return ((f & 1) && i == B.il) || ((f & 2) && i == B.iu) ||
         ((f & 4) && j == B.jl) || ((f & 8) && j == B.ju) ||
         ((f & 16) && k == B.kl) || ((f & 32) && k == B.ku);
}

// Stencil pass: one workgroup per (tile, field), z-marching over the tile.
// The field index varies fastest and each XCD takes a contiguous range of
// (tile, field) pairs, so the 22 fields of a tile stream through the same
// L2 together: the shift planes every field reads, and the halo rows of
// neighbouring tiles, come from HBM once.
template <class Cfg>
__global__ void __launch_bounds__(Cfg::THREADS) k_stencil(StencilArgs a) {
  __shared__ double sm[2 * Cfg::BUF];
  const int G = gridDim.x;  // multiple of 8: XCD-contiguous ranges
  const int w = blockIdx.x;
  const int t = (w & 7) * (G >> 3) + (w >> 3);
  if (t >= a.ntiles * NVAR) return;
  const int tile = t / NVAR;
  const int f = t - tile * NVAR;
  const PlaneTile T = a.tiles[tile];
  switch (dkind(f)) {
    case DK_METRIC: stencil_tile<Cfg, DK_METRIC>(a, T, f, sm); break;
    case DK_FULL: stencil_tile<Cfg, DK_FULL>(a, T, f, sm); break;
    case DK_GRAD: stencil_tile<Cfg, DK_GRAD>(a, T, f, sm); break;
    default: stencil_tile<Cfg, DK_ADV>(a, T, f, sm); break;
  }
}

// The linearisation the adjoint reads (first and second derivatives, the
// selected lop-sided derivatives; the adjoint's slot layout, stride nint),
// formed by the stencil pass's z-march with its stencils, 256-thread tiles.
__global__ void __launch_bounds__(StCfg256::THREADS) k_stencil_lin(StencilArgs a) {
  __shared__ double sm[2 * StCfg256::BUF];
  const int G = gridDim.x;  // multiple of 8: XCD-contiguous ranges
  const int w = blockIdx.x;
  const int t = (w & 7) * (G >> 3) + (w >> 3);
  if (t >= a.ntiles * NVAR) return;
  const int tile = t / NVAR;
  const int f = t - tile * NVAR;
  const PlaneTile T = a.tiles[tile];
  switch (dkind(f)) {
    case DK_METRIC:
    case DK_FULL: stencil_tile<StCfg256, DK_FULL, true>(a, T, f, sm); break;
    case DK_GRAD: stencil_tile<StCfg256, DK_GRAD, true>(a, T, f, sm); break;
    default: stencil_tile<StCfg256, DK_ADV, true>(a, T, f, sm); break;
  }
}

__device__ __forceinline__ PointIO point_io(const RhsArgs& a, const DevBlock& B, int p,
                                            int qi) {
  PointIO X;
  const int N = B.npts;
  X.U = make_buf(a.u + B.off * NVAR, (long long)NVAR * N * 8);
  X.DV = make_buf(a.dv + B.doff, (long long)NDV * B.nis * 8);
  X.has_mat = a.mat != nullptr;
  X.MT = X.has_mat ? make_buf(a.mat + B.off * NMAT, (long long)NMAT * N * 8) : X.U;
  X.vu = (unsigned)p * 8u;
  X.vd = (unsigned)qi * 8u;
  X.fu = N * 8;
  X.fd = B.nis * 8;
  return X;
}

// Algebra pass of Z4cRHS: one thread per interior vertex.  The curvature
// part (Ricci, D_aD_b alpha; 12 values) is formed first and kept in a
// per-thread LDS column, then the assembly reads it from there; the 22
// right-hand-side values are staged in LDS and stored at the end, so that no
// global store sits among the derivative loads.
template <bool WITH_SOMMERFELD>
__global__ void __launch_bounds__(TILE) k_rhs_alg(RhsArgs a) {
  __shared__ double ko[NVAR * TILE];
  __shared__ double cvs[12 * TILE];
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const int t = threadIdx.x;
  const DevBlock B = a.blocks[b];
  const int N = B.npts;
  const int p = flat(B, i, j, k);
  const int qi = (i - B.il) + B.ni * ((j - B.jl) + B.nj * (k - B.kl));
  const PointIO X = point_io(a, B, p, qi);
  rhs_curvature_point(a.o, X, [&](int n, double v) { cvs[n * TILE + t] = v; });
  rhs_assembly_point(a.o, X, [&](int n) { return cvs[n * TILE + t]; },
                     [&](int n, double v) { ko[n * TILE + t] = v; });
  if (WITH_SOMMERFELD && B.faces && on_sommerfeld_face(B, i, j, k)) {
    const Pt P = make_pt(p, B.nn1, B.nn2, N);
    sommerfeld_point(B, X.U, P, a.u + B.off * NVAR, i, j, k, N,
                     [&](int n, double v) { ko[n * TILE + t] = v; });
  }
  double* rhs = a.rhs + B.off * NVAR;
#pragma unroll
  for (int n = 0; n < NVAR; ++n) rhs[n * N + p] = ko[n * TILE + t];
}

__global__ void __launch_bounds__(TILE) k_sommerfeld(RhsArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  if (!B.faces || !on_sommerfeld_face(B, i, j, k)) return;
  const int N = B.npts;
  const double* u = a.u + B.off * NVAR;
  const Buf U = make_buf(u, (long long)NVAR * N * 8);
  const Pt P = make_pt(flat(B, i, j, k), B.nn1, B.nn2, N);
  double* rhs = a.rhs + B.off * NVAR;
  const int p = flat(B, i, j, k);
  sommerfeld_point(B, U, P, u, i, j, k, N, [&](int n, double v) { rhs[n * N + p] = v; });
}

// ---------------------------------------------------------------------------
// AlgConstr (src/z4c/z4c.cpp:677-991)
// ---------------------------------------------------------------------------
struct AlgArgs {
  const DevBlock* blocks;
  Launch L;
  double* u;
  double eps_floor;
  int tf_force, force_reg;
  int range[6];  // il,iu,jl,ju,kl,ku (ranged form) or all -1 = whole block
  int skip_physical;
};

// AlgConstr of one point's values (z4c.cpp:677-799); `chi` and `alpha` are
// changed only with force_reg.
__device__ __forceinline__ void algconstr_vals(double* g, double* A, double& chi, double& alpha,
                                               double eps_floor, int tf_force, int force_reg) {
  double detg = det3(g);
  bool project = true;
  if (tf_force)
    detg = detg > 0. ? detg : 1.;
  else
    project = detg > eps_floor;
  if (project) {
    const double oopsi4 = regularize_nth_root(detg, 1.0, eps_floor, -3.0);
#pragma unroll
    for (int ab = 0; ab < 6; ++ab) g[ab] *= oopsi4;
    const double tr = trace_rank2(1.0, g, A);
#pragma unroll
    for (int ab = 0; ab < 6; ++ab) A[ab] -= (1.0 / 3.0) * tr * g[ab];
  }
  if (force_reg) {
    chi = dmax(chi, eps_floor);
    alpha = regularize_near_zero(alpha, eps_floor);
  }
}

__device__ __forceinline__ void algconstr_point(double* __restrict__ u, int N,
                                                int p, double eps_floor,
                                                int tf_force, int force_reg) {
  double g[6], A[6];
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) {
    g[ab] = u[(V_GXX + ab) * N + p];
    A[ab] = u[(V_AXX + ab) * N + p];
  }
  double chi = u[V_CHI * N + p], alpha = u[V_ALPHA * N + p];
  algconstr_vals(g, A, chi, alpha, eps_floor, tf_force, force_reg);
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) {
    u[(V_GXX + ab) * N + p] = g[ab];
    u[(V_AXX + ab) * N + p] = A[ab];
  }
  if (force_reg) {
    u[V_CHI * N + p] = chi;
    u[V_ALPHA * N + p] = alpha;
  }
}

__global__ void __launch_bounds__(TILE) k_algconstr(AlgArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  if (a.range[0] >= 0) {
    if (i < a.range[0] || i > a.range[1] || j < a.range[2] || j > a.range[3] ||
        k < a.range[4] || k > a.range[5])
      return;
    if (a.skip_physical && i >= B.il && i <= B.iu && j >= B.jl && j <= B.ju &&
        k >= B.kl && k <= B.ku)
      return;
  }
  algconstr_point(a.u + B.off * NVAR, B.npts, flat(B, i, j, k), a.eps_floor,
                  a.tf_force, a.force_reg);
}

// The stage kernel's state stores are streaming (non-temporal): the next
// pass reads them back from HBM in any case.
__device__ __forceinline__ void st_state(double* p, double v) { __builtin_nontemporal_store(v, p); }

// Stage update of the vertex p (interior index qi) with right-hand side kv(n),
// then AlgConstr of the point.  The reference runs CalculateZ4cRHS, IntegrateZ4c
// (SumBT over the registers) and EnforceAlgConstr as separate tasks
// (src/task_list/gr/task_list_gr_z4c.cpp:46-64); the update is pointwise, so
// every variable's follows its right-hand side, with the same sums in the same
// order:
//   u_{s+1} = u_n + (A[s+1][s] dt) k_s          (the one nonzero of bt_rk4's row)
//   acc_1 = u_n + (b_1 dt) k_1,  acc_s = acc_{s-1} + (b_s dt) k_s
//   u_{n+1} = acc_3 + (b_4 dt) k_4 = ((u_n + b_1 dt k_1) + b_2 dt k_2) + ...
// followed by AlgConstr of the point (src/z4c/z4c.cpp:677-991).  ls: the
// low-storage 2S stage (task_list_gr_z4c.cpp:176-193) with WeightedAve_'s case
// split (weighted_ave.cpp:21-132):
//   u1 = WeightedAve(u1, u, -, {1, delta, 0})   (u1 = 0 before stage 1)
//   u  = WeightedAve(u, u1, -, {gamma_1, gamma_2, 0}) + (beta dt) rhs
// The running sum, the kept u_n and u1 are interior-indexed (whole 128-byte
// lines of interior points).
template <class A, class K>
__device__ __forceinline__ void stage_update(const A& a, bool alg, bool ls, const DevBlock& B, int p,
                                             int qi, K&& kv) {
  const int N = B.npts;
  const long long ibase = B.ioff * NVAR + qi;
  const int NI = B.nint;
  const long long base = B.off * NVAR;
  const double* u = a.u + base + p;
  double* out = a.out + base + p;
  double* acc = a.acc + ibase;
  const int stage = a.stage;
  // every load before the first store: one wait instead of one per field
  double s[NVAR], x[NVAR];
  if (ls) {
    double* u1 = acc;
    const double dl = a.ls_w[0], g1 = a.ls_w[1], g2 = a.ls_w[2], bdt = a.ls_w[3];
#pragma unroll
    for (int n = 0; n < NVAR; ++n) s[n] = u[(long long)n * N];
#pragma unroll
    for (int n = 0; n < NVAR; ++n) x[n] = (stage == 1) ? 0.0 : u1[(long long)n * NI];
#pragma unroll
    for (int n = 0; n < NVAR; ++n) {
      const double u0 = s[n];
      double v1 = x[n];
      if (dl != 0.0) v1 += dl * u0;
      if (!a.ls_last) st_state(u1 + (long long)n * NI, v1);
      double v;
      if (g1 == 1.0)
        v = (g2 != 0.0) ? u0 + g2 * v1 : u0;
      else if (g1 == 0.0)
        v = (g2 == 1.0) ? v1 : g2 * v1;
      else
        v = (g2 != 0.0) ? g1 * u0 + g2 * v1 : u0 * g1;
      s[n] = v + bdt * kv(n);
    }
  } else {
    const double wa = a.wa, wb = a.wb;
    const double* un = a.un_int ? a.un + ibase : a.un + base + p;
    const long long un_st = a.un_int ? NI : N;
    double* keep = a.keep ? a.keep + ibase : nullptr;
    if (stage < 4) {
#pragma unroll
      for (int n = 0; n < NVAR; ++n) s[n] = un[n * un_st];
    }
    if (stage > 1) {
#pragma unroll
      for (int n = 0; n < NVAR; ++n) x[n] = acc[(long long)n * NI];
    }
#pragma unroll
    for (int n = 0; n < NVAR; ++n) {
      const double v = kv(n);
      if (stage == 1) {
        if (keep) st_state(keep + (long long)n * NI, s[n]);
        st_state(acc + (long long)n * NI, s[n] + wb * v);
        s[n] = s[n] + wa * v;
      } else if (stage < 4) {
        st_state(acc + (long long)n * NI, x[n] + wb * v);
        s[n] = s[n] + wa * v;
      } else {
        s[n] = x[n] + wb * v;
      }
    }
  }
  if (alg)
    algconstr_vals(s + V_GXX, s + V_AXX, s[V_CHI], s[V_ALPHA], a.eps_floor, a.tf_force,
                   a.force_reg);
#pragma unroll
  for (int n = 0; n < NVAR; ++n) st_state(out + (long long)n * N, s[n]);
}

// Right-hand side of a brick (z4c_fused.hpp), stored as such or taken into the
// stage update.
template <class C>
__global__ void __launch_bounds__(C::THREADS) __attribute__((amdgpu_waves_per_eu(2)))
k_fused(FusedArgs args) {
  __shared__ __align__(16) double winA[C::WIN];
  __shared__ __align__(16) double winB[C::WIN];
  __shared__ double der[C::NDY + C::NDZ];
  __shared__ int4 offs[2 * C::THREADS];
  __shared__ int halo[(C::HROUNDS + 1) * C::THREADS];
  const KernArgs<FusedArgs> ka;
  const int G = gridDim.x;  // multiple of 8: XCD-contiguous ranges
  const int t = (blockIdx.x & 7) * (G >> 3) + (blockIdx.x >> 3);
  if (t >= args.ntiles) return;
  const int tid = threadIdx.x;
  double kv[NVAR] = {};
  {
    const auto& a = args;
    const FusedTile T = a.tiles[t];
    const DevBlock& B = a.blocks[T.block];
    const int N = B.npts;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tx, ty, tz;
    const bool in = fused_vertex<C>(T, tid, tx, ty, tz);
    const double* u = a.u + B.off * NVAR;
    FusedPoint<C> P;
    P.ub = u;
    P.N = __builtin_amdgcn_readfirstlane(N);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      // lidx equals cidx1
      P.c1[d] = uniform(B.cidx1[d]);
      P.c2[d] = uniform(B.cidx2[d]);
      P.cd[d] = uniform(B.cidxd[d]);
    }
    P.win[0] = winA;
    P.win[1] = winB;
    P.der = der;
    P.halo = halo + tid;
    P.wave = wave;
    P.lane = lane;
    {
      int v[C::ROUNDS];
#pragma unroll
      for (int r = 0; r < C::ROUNDS; ++r) {
        const int e = (r * C::WAVES + wave) * 64 + lane;
        const int row = e / (C::PX / 2), c0 = 2 * (e - row * (C::PX / 2));
        const int kk = row / C::PY, jj = row - kk * C::PY;
        // the pair's distances from the brick: a field needs the vertices that
        // lie off it along one axis (by up to 4) and, with mixed derivatives,
        // along two (by up to 3)
        const int dx = c0 + 1 < 4 ? 3 - c0 : max(0, c0 - T.ni - 3);
        const int dy = jj < 4 ? 4 - jj : max(0, jj - T.nj - 3);
        const int dz = kk < 4 ? 4 - kk : max(0, kk - T.nk - 3);
        const int off = (dx > 0) + (dy > 0) + (dz > 0);
        const int far = max(dx, max(dy, dz));
        const bool star = off <= 1 && far <= 4;
        const bool need = star || (off == 2 && far <= 3);
        v[r] = 8 * ((B.il + T.i0 - 4 + c0) +
                    B.nn1 * ((B.jl + T.j0 - 4 + jj) + B.nn2 * (B.kl + T.k0 - 4 + kk)));
        if (!need || e >= C::PAIRS) v[r] = (int)DV_DROP;
        else if (!star) v[r] |= 1 << 30;
      }
      offs[tid] = int4{v[0], v[1], v[2], v[3]};
      offs[C::THREADS + tid] = int4{v[4], v[5], v[6], v[7]};
      P.offs = offs + tid;
    }
    P.o = (tx + 4) + C::PX * (ty + 4) + C::PLANE * (tz + 4);
    halo[C::HROUNDS * C::THREADS + tid] =
        ((tx + 3) + C::DX * (ty + C::BY * tz)) |
        ((C::NDY + (tx + 3) + C::DX * (ty + 3) + C::DZP * tz) << 16);
#pragma unroll
    for (int r = 0; r < C::HROUNDS; ++r) {
      const int s = r * C::WAVES + wave;
      int x, y, z;
      bool ok;
      if (s < 2 * C::SX) {
        const int e = (s < C::SX ? s : s - C::SX) * 64 + lane;
        const int hx = e % 6;
        x = hx < 3 ? hx - 3 : T.ni + hx - 3;
        y = e / 6 % C::BY;
        z = e / (6 * C::BY);
        ok = e < C::HX;
      } else {
        const int e = (s - 2 * C::SX) * 64 + lane;
        const int hy = e / C::BX % 6;
        x = e % C::BX;
        y = hy < 3 ? hy - 3 : T.nj + hy - 3;
        z = e / (6 * C::BX);
        ok = e < C::HY;
      }
      const int src = ok ? (x + 4) + C::PX * (y + 4) + C::PLANE * (z + 4) : P.o;
      const int dst = !ok ? -1
                          : (s < C::SX ? (x + 3) + C::DX * (y + C::BY * z)
                                       : C::NDY + (x + 3) + C::DX * (y + 3) + C::DZP * z);
      halo[r * C::THREADS + tid] = src | (dst * 65536);
    }
    P.p8 = in ? 8u * (unsigned)flat(B, B.il + T.i0 + tx, B.jl + T.j0 + ty, B.kl + T.k0 + tz)
              : DV_DROP;
    P.dst = (a.rhs ? a.rhs : a.out) + B.off * NVAR;
    P.diss = a.o.diss;
    P.bx = P.at(V_BETAX);
    P.by = P.at(V_BETAX + 1);
    P.bz = P.at(V_BETAX + 2);
    P.template fetch<fu_field(0), 0>();
    fused_rhs<C>(P, ka, a.mat ? a.mat + B.off * NMAT : nullptr, kv);
  }
  // the tile again (nothing of it is held through the fields)
  const auto& a = ka.get();
  int t2 = t;
  asm volatile("" : "+v"(t2));
  const FusedTile T = a.tiles[__builtin_amdgcn_readfirstlane(t2)];
  const DevBlock& B = a.blocks[T.block];
  int tx, ty, tz;
  if (!fused_vertex<C>(T, tid, tx, ty, tz)) return;
  const int N = B.npts;
  const int i = B.il + T.i0 + tx, j = B.jl + T.j0 + ty, k = B.kl + T.k0 + tz;
  const int p = flat(B, i, j, k);
  const long long base = B.off * NVAR;
  if (a.sommerfeld && B.faces && on_sommerfeld_face(B, i, j, k)) {
    const Pt P = make_pt(p, B.nn1, B.nn2, N);
    sommerfeld_point(B, make_buf(a.u + base, (long long)NVAR * N * 8), P, a.u + base, i, j, k, N,
                     [&](int n, double v) { kv[n] = v; });
  }
  if (a.rhs) {
    double* rhs = a.rhs + base + p;
#pragma unroll
    for (int n = 0; n < NVAR; ++n) rhs[(long long)n * N] = kv[n];
    return;
  }
  const int qi = (i - B.il) + B.ni * ((j - B.jl) + B.nj * (k - B.kl));
  stage_update(a, a.alg, a.ls, B, p, qi, [&](int n) { return kv[n]; });
}

// The stage in two passes: after the stencil pass, the algebra of one vertex
// per thread and its update.  Curvature part and right-hand side wait in LDS
// columns as in k_rhs_alg.  The stage reads its input at its own vertex only
// (but for Sommerfeld rows), so without flagged faces out may be u itself.
// A zero right-hand side (cowling) takes this kernel without the stencil pass.
struct StageArgs {
  FusedArgs f;  // f.tiles unused
  Launch L;
  const double* dv;
};

template <bool ALG, bool LS>
__global__ void __launch_bounds__(TILE) __attribute__((amdgpu_waves_per_eu(2)))
k_rk4_stage(StageArgs a) {
  __shared__ double ko[NVAR * TILE];  // this point's k_s, staged (see k_rhs_alg)
  __shared__ double cvs[12 * TILE];   // this point's curvature part
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const int t = threadIdx.x;
  const DevBlock B = a.f.blocks[b];
  const int N = B.npts;
  const int p = flat(B, i, j, k);
  const int qi = (i - B.il) + B.ni * ((j - B.jl) + B.nj * (k - B.kl));
  if (a.f.cowling) {
    for (int n = 0; n < NVAR; ++n) ko[n * TILE + t] = 0.0;
  } else {
    const RhsArgs r{a.f.blocks, a.L, a.f.u, a.dv, a.f.mat, nullptr, a.f.o};
    const PointIO X = point_io(r, B, p, qi);
    rhs_curvature_point(a.f.o, X, [&](int n, double v) { cvs[n * TILE + t] = v; });
    rhs_assembly_point(a.f.o, X, [&](int n) { return cvs[n * TILE + t]; },
                       [&](int n, double v) { ko[n * TILE + t] = v; });
    if (B.faces && on_sommerfeld_face(B, i, j, k)) {
      const Pt P = make_pt(p, B.nn1, B.nn2, N);
      sommerfeld_point(B, X.U, P, a.f.u + B.off * NVAR, i, j, k, N,
                       [&](int n, double v) { ko[n * TILE + t] = v; });
    }
  }
  stage_update(a.f, ALG, LS, B, p, qi, [&](int n) { return ko[n * TILE + t]; });
}

// Ghost vertices of a fused step with ghosts held at u_n: what the unfused
// sequence leaves there after every stage is AlgConstr(u_n + 0), so the step
// applies AlgConstr to the state's ghosts once (after the first stage has
// read them), and copies them into the work register that the stages alternate
// with.  The 30.3 M ghost vertices of 2048 blocks of 16^3 .. 32^3 cells: 18.8 GB
// (8.9 read, 9.9 written; ghost rows of 32 bytes) in 5.4 ms a step, against 2.0 ms
// for AlgConstr in place (k_rk4_ghosts_inplace: steps in two passes), which is what
// the one kernel pays for its second buffer.
struct GhostArgs {
  const DevBlock* blocks;
  Launch L;
  double* u;
  double* w0;
  double eps_floor;
  int tf_force, force_reg;
};

// Copies the ghost vertices of all fields from a.u into a.w0.
__global__ void __launch_bounds__(TILE) k_ghost_copy(GhostArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  const int N = B.npts;
  const long long e = B.off * NVAR + flat(B, i, j, k);
#pragma unroll
  for (int n = 0; n < NVAR; ++n) a.w0[e + (long long)n * N] = a.u[e + (long long)n * N];
}

__global__ void __launch_bounds__(TILE) k_rk4_ghosts_inplace(GhostArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  algconstr_point(a.u + B.off * NVAR, B.npts, flat(B, i, j, k), a.eps_floor, a.tf_force,
                  a.force_reg);
}

// Held ghosts of a low-storage stage: AlgConstr of a.u's into a.w0.  Fields that
// AlgConstr leaves alone are the same in both states from the second stage on.
template <bool ALL>
__global__ void __launch_bounds__(TILE) k_ls_ghosts(GhostArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  const int N = B.npts;
  const long long e = B.off * NVAR + flat(B, i, j, k);
  const double* u = a.u + e;
  double* w = a.w0 + e;
  const bool reg = ALL || a.force_reg;  // chi and alpha change with force_reg only
  double s[NVAR];
#pragma unroll
  for (int n = 0; n < NVAR; ++n) {
    const bool alg = (n >= V_GXX && n < V_GXX + 6) || (n >= V_AXX && n < V_AXX + 6);
    s[n] = ALL || alg || n == V_CHI || n == V_ALPHA ? u[(long long)n * N] : 0.0;
  }
  algconstr_vals(s + V_GXX, s + V_AXX, s[V_CHI], s[V_ALPHA], a.eps_floor, a.tf_force,
                 a.force_reg);
#pragma unroll
  for (int n = 0; n < NVAR; ++n) {
    const bool alg = (n >= V_GXX && n < V_GXX + 6) || (n >= V_AXX && n < V_AXX + 6);
    if (ALL || alg || (reg && (n == V_CHI || n == V_ALPHA))) w[(long long)n * N] = s[n];
  }
}

// Interior vertices of all fields from one state into another.
struct CopyArgs {
  const DevBlock* blocks;
  Launch L;
  const double* from;
  double* to;
};

__global__ void __launch_bounds__(TILE) k_copy_interior(CopyArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  const int N = B.npts;
  const long long e = B.off * NVAR + flat(B, i, j, k);
  double v[NVAR];
#pragma unroll
  for (int n = 0; n < NVAR; ++n) v[n] = a.from[e + (long long)n * N];
#pragma unroll
  for (int n = 0; n < NVAR; ++n) a.to[e + (long long)n * N] = v[n];
}

__global__ void __launch_bounds__(TILE) k_rk4_ghosts(GhostArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  const int N = B.npts;
  const int p = flat(B, i, j, k);
  const long long base = B.off * NVAR;
  double* u = a.u + base;
  // every field is loaded once; AlgConstr works on the registers
  double s[NVAR];
#pragma unroll
  for (int n = 0; n < NVAR; ++n) s[n] = u[n * N + p];
  algconstr_vals(s + V_GXX, s + V_AXX, s[V_CHI], s[V_ALPHA], a.eps_floor, a.tf_force,
                 a.force_reg);
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) {
    u[(V_GXX + ab) * N + p] = s[V_GXX + ab];
    u[(V_AXX + ab) * N + p] = s[V_AXX + ab];
  }
  if (a.force_reg) {
    u[V_CHI * N + p] = s[V_CHI];
    u[V_ALPHA * N + p] = s[V_ALPHA];
  }
  double* w0 = a.w0 + base;
#pragma unroll
  for (int n = 0; n < NVAR; ++n) w0[n * N + p] = s[n];
}

// ---------------------------------------------------------------------------
// History sums of the Z4c constraints (src/outputs/history.cpp:178-205): over
// the reference's cell-index loop is..ie (vertices il..iu-1 per axis), with
// cell volume dx*dy*dz and the r_max_con cut on the cell-centre radius.
// One partial sum per tile; the host adds the partials in tile order.
// ---------------------------------------------------------------------------
constexpr int NHST = 8;
struct HstArgs {
  const DevBlock* blocks;
  Launch L;
  const double* u;
  const double* con;
  double r2max;
  double* partial;  // NHST per tile
};

__global__ void __launch_bounds__(TILE) k_history(HstArgs a) {
  __shared__ double red[NHST][TILE / 64];
  double v[NHST];
#pragma unroll
  for (int q = 0; q < NHST; ++q) v[q] = 0.0;
  int b, i, j, k;
  const int G = gridDim.x;
  const int t = (blockIdx.x & 7) * (G >> 3) + (blockIdx.x >> 3);
  if (tile_point(a.L, b, i, j, k)) {
    const DevBlock B = a.blocks[b];
    if (i < B.iu && j < B.ju && k < B.ku) {
      const double x1 = B.x0[0] + (i + 0.5) * B.dx[0];
      const double x2 = B.x0[1] + (j + 0.5) * B.dx[1];
      const double x3 = B.x0[2] + (k + 0.5) * B.dx[2];
      const double R2 = x1 * x1 + x2 * x2 + x3 * x3;
      if (R2 <= a.r2max) {
        const int N = B.npts;
        const int p = flat(B, i, j, k);
        const double* c = a.con + B.off * NCON;
        const double vol = B.dx[0] * B.dx[1] * B.dx[2];
        const double H = fabs(c[C_H * N + p]);
        const double Mx = fabs(c[(C_MX + 0) * N + p]);
        const double My = fabs(c[(C_MX + 1) * N + p]);
        const double Mz = fabs(c[(C_MX + 2) * N + p]);
        const double th = fabs(a.u[B.off * NVAR + V_THETA * N + p]);
        v[0] = vol * (H * H);
        v[1] = vol * fabs(c[C_M * N + p]);
        v[2] = vol * (Mx * Mx);
        v[3] = vol * (My * My);
        v[4] = vol * (Mz * Mz);
        v[5] = vol * fabs(c[C_Z * N + p]);
        v[6] = vol * (th * th);
        v[7] = vol * fabs(c[C_C * N + p]);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < NHST; ++q) {
    double x = v[q];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
    if ((threadIdx.x & 63) == 0) red[q][threadIdx.x >> 6] = x;
  }
  __syncthreads();
  if (threadIdx.x < NHST && t < a.L.ntiles) {
    double x = 0.0;
    for (int w = 0; w < TILE / 64; ++w) x += red[threadIdx.x][w];
    a.partial[(long long)t * NHST + threadIdx.x] = x;
  }
}

// Partials of z4c_history_noalloc: NHST doubles per tile in a file-scope
// device array instead of a context allocation, for callers that cannot
// allocate (HIP graph capture, serving loops).  Each GPU holds one copy until
// the process ends; host code reaches it only through the address
// hipGetSymbolAddress returns on that device (g_scratch_dev).  Every tile of a
// call writes its partials before k_history_sum reads them, so nothing needs
// clearing; calls that overlap on one GPU share the array and race.
constexpr int HIST_NOALLOC_MAX_TILES = 1 << 17;  // 8 MiB: 33.5 M interior vertices
static __device__ __align__(256) double scratch[(size_t)HIST_NOALLOC_MAX_TILES * NHST];

// out[q] = sum of the tiles' partials in tile order, one lane per column: the
// order (and so every rounding) of z4c_history's host loop.  The chain of
// additions is what cannot be shortened; the partials come to it through LDS,
// a chunk of 256 tiles loaded by the whole workgroup while the chunk before it
// is summed (one lane loading its own took 152 ns a tile, 2.47 ms for 16200
// tiles; now 0.12 ms).
constexpr int HSUM_TILES = 256;
__global__ void __launch_bounds__(512) k_history_sum(const double* partial, int ntiles,
                                                     double* out) {
  constexpr int CH = HSUM_TILES * NHST, PER = CH / 512;
  __shared__ double buf[2][CH];
  const int tid = threadIdx.x;
  const long long n = (long long)ntiles * NHST;
  double r[PER];
  auto load = [&](long long c) {
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const long long i = c * CH + e * 512 + tid;
      r[e] = i < n ? partial[i] : 0.0;
    }
  };
  const int nch = (ntiles + HSUM_TILES - 1) / HSUM_TILES;
  load(0);
  double x = 0.0;
  for (int c = 0; c < nch; ++c) {
    double* b = buf[c & 1];
#pragma unroll
    for (int e = 0; e < PER; ++e) b[e * 512 + tid] = r[e];
    __syncthreads();  // chunk c is whole; every lane is done with chunk c - 2
    if (c + 1 < nch) load(c + 1);
    if (tid < NHST) {
      const int m = min(HSUM_TILES, ntiles - c * HSUM_TILES);
      int t = 0;
      for (; t + 16 <= m; t += 16) {
        double v[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = b[(t + e) * NHST + tid];
#pragma unroll
        for (int e = 0; e < 16; ++e) x += v[e];
      }
      for (; t < m; ++t) x += b[t * NHST + tid];
    }
  }
  if (tid < NHST) out[tid] = x;
}

// ---------------------------------------------------------------------------
// ADMToZ4c (src/z4c/adm_z4c.cpp:46-192), Z4cToADM (:200-260),
// PrepareAuxExtended (:1139-1231)
// ---------------------------------------------------------------------------
struct AdmArgs {
  const DevBlock* blocks;
  Launch L;
  const double* adm_in;
  double* u;
  double* adm_out;
  double* aux_ext;
  double chi_psi_power, chi_div_floor;
};

__device__ __forceinline__ void aux_ext_point(double pw, double floor,
                                              const double* __restrict__ u,
                                              const double* __restrict__ adm,
                                              double* __restrict__ ax, int N,
                                              int p) {
  const double chi = fabs(u[V_CHI * N + p]);
  const double chi_g = dmax(chi, floor);
  const double sdg = (pw == -4.) ? 1.0 / (chi_g * sqrt(chi_g))
                                 : pow(chi_g, (12.0 / pw) / 2.0);
  ax[p] = sdg;
  double g[6], gi[6];
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) g[ab] = adm[(A_GXX + ab) * N + p];
  inv3(1.0 / (sdg * sdg), g, gi);
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) ax[(1 + ab) * N + p] = gi[ab];
}

__global__ void __launch_bounds__(TILE) k_adm2z4c_point(AdmArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  const int N = B.npts;
  const int p = flat(B, i, j, k);
  const double* adm = a.adm_in + B.off * NADM;
  double* u = a.u + B.off * NVAR;
  const double pw = a.chi_psi_power;
  u[V_ALPHA * N + p] = adm[A_ALPHA * N + p];
#pragma unroll
  for (int m = 0; m < 3; ++m) u[(V_BETAX + m) * N + p] = adm[(A_BETAX + m) * N + p];
  double G[6], gt[6], Kt[6];
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) G[ab] = adm[(A_GXX + ab) * N + p];
  double detg = det3(G);
  double oopsi4;
  if (pw == -4.) {
    oopsi4 = cbrt(1.0 / detg);
    u[V_CHI * N + p] = oopsi4;
  } else {
    oopsi4 = pow(detg, -1. / 3.);
    u[V_CHI * N + p] = pow(detg, 1. / 12. * pw);
  }
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) {
    gt[ab] = oopsi4 * G[ab];
    Kt[ab] = oopsi4 * adm[(A_KXX + ab) * N + p];
    u[(V_GXX + ab) * N + p] = gt[ab];
  }
  detg = det3(gt);
  const double Khat = trace_rank2(1.0 / detg, gt, Kt);
  u[V_KHAT * N + p] = Khat;
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) u[(V_AXX + ab) * N + p] = Kt[ab] - (1. / 3.) * Khat * gt[ab];
}

// Gamma~^a = -sum_b Dx_b g~^{ba} on the interior (zero in ghosts), Theta = 0.
__global__ void __launch_bounds__(TILE) k_adm2z4c_gamma(AdmArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  const int N = B.npts;
  const int p = flat(B, i, j, k);
  double* u = a.u + B.off * NVAR;
  // Only the Gamma and Theta slots are written here and they are not read,
  // so neighbouring threads see a stable g~.
  const double* ug = u;
  const bool interior = i >= B.il && i <= B.iu && j >= B.jl && j <= B.ju &&
                        k >= B.kl && k <= B.ku;
  double gam[3] = {0.0, 0.0, 0.0};
  if (interior) {
    const Buf U = make_buf(ug, (long long)NVAR * N * 8);
    const Pt P = make_pt(p, B.nn1, B.nn2, N);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        // g~^{dc} at the points -3..3 along d, then the 6th-order Dx
        double v[7];
#pragma unroll
        for (int m = 0; m < 7; ++m) {
          if (m == 3) { v[m] = 0.0; continue; }
          double g[6], gi[6];
#pragma unroll
          for (int ab = 0; ab < 6; ++ab) g[ab] = ldm(U, P, V_GXX + ab, d, m - 3);
          inv3(1.0 / det3(g), g, gi);
          v[m] = gi[sym(d, c)];
        }
        double out = 0.0;
        out += -1.0 * (v[0] - v[6]);
        out += 9.0 * (v[1] - v[5]);
        out += -45.0 * (v[2] - v[4]);
        gam[c] -= out * B.cidx1[d];
      }
    }
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) u[(V_GAMX + c) * N + p] = gam[c];
  u[V_THETA * N + p] = 0.0;
}

__global__ void __launch_bounds__(TILE) k_aux_ext(AdmArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  aux_ext_point(a.chi_psi_power, a.chi_div_floor, a.u + B.off * NVAR,
                a.adm_in + B.off * NADM, a.aux_ext + B.off * 7, B.npts,
                flat(B, i, j, k));
}

__global__ void __launch_bounds__(TILE) k_z4c2adm(AdmArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  const int N = B.npts;
  const int p = flat(B, i, j, k);
  const double* u = a.u + B.off * NVAR;
  double* adm = a.adm_out + B.off * NADM;
  adm[A_ALPHA * N + p] = u[V_ALPHA * N + p];
#pragma unroll
  for (int m = 0; m < 3; ++m) adm[(A_BETAX + m) * N + p] = u[(V_BETAX + m) * N + p];
  const double chi = u[V_CHI * N + p];
  const double psi4 = (a.chi_psi_power == -4.) ? 1.0 / chi : pow(chi, 4. / a.chi_psi_power);
  adm[A_PSI4 * N + p] = psi4;
  const double th = u[V_THETA * N + p], kh = u[V_KHAT * N + p];
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) {
    const double G = psi4 * u[(V_GXX + ab) * N + p];
    adm[(A_GXX + ab) * N + p] = G;
    adm[(A_KXX + ab) * N + p] = psi4 * u[(V_AXX + ab) * N + p] + (1. / 3.) * (kh + 2. * th) * G;
  }
  if (a.aux_ext)
    aux_ext_point(a.chi_psi_power, a.chi_div_floor, u, adm, a.aux_ext + B.off * 7, N, p);
}

// ---------------------------------------------------------------------------
// ADMConstraints (src/z4c/adm_z4c.cpp:382-930), p = -4 and general branch
// ---------------------------------------------------------------------------
struct ConArgs {
  const DevBlock* blocks;
  Launch L;
  const double* u;
  const double* adm;
  const double* mat;
  const double* d1;
  double* con;
  double chi_psi_power, chi_div_floor, r_max_con;
};

// WAVES 2: two waves a SIMD although 67 registers spill (324 unbounded, one
// wave); z4c_adm_constraints says when.
template <int WAVES>
__global__ void __launch_bounds__(TILE) __attribute__((amdgpu_waves_per_eu(WAVES)))
k_constraints(ConArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  const int N = B.npts;
  const int p = flat(B, i, j, k);
  const double* u = a.u + B.off * NVAR;
  const double* adm = a.adm + B.off * NADM;
  const double* d1 = a.d1 + B.off * ND1;
  double* con = a.con + B.off * NCON;
#define DP(bb, f) (d1 + ((bb) * 11 + (f)) * N + p)
  const Buf U = make_buf(u, (long long)NVAR * N * 8);
  const Buf D = make_buf(d1, (long long)ND1 * N * 8);
  const Buf AD = make_buf(adm, (long long)NADM * N * 8);
  const Pt P = make_pt(p, B.nn1, B.nn2, N);
  const double pw = a.chi_psi_power;
  double gt[6], G[6], Kdd[6];
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) {
    gt[ab] = u[(V_GXX + ab) * N + p];
    G[ab] = adm[(A_GXX + ab) * N + p];
    Kdd[ab] = adm[(A_KXX + ab) * N + p];
  }
  double rho = 0.0, Sd[3] = {0, 0, 0};
  if (a.mat) {
    const double* mat = a.mat + B.off * NMAT;
    rho = mat[M_RHO * N + p];
#pragma unroll
    for (int m = 0; m < 3; ++m) Sd[m] = mat[(M_SX + m) * N + p];
  }
  const double chi_g = dmax(u[V_CHI * N + p], a.chi_div_floor);
  const double oochi = 1.0 / chi_g;
  const bool p4 = (pw == -4.);
  const double fac = 4.0 / pw, fac2 = fac - 1.0;
  const double psi4 = p4 ? 0.0 : pow(chi_g, fac);
  double dchi[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) dchi[c] = *DP(c, F_CHI);
  double dg[3][6];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int ab = 0; ab < 6; ++ab)
      dg[c][ab] = p4 ? oochi * (*DP(c, F_G + ab) - oochi * gt[ab] * dchi[c])
                     : psi4 * (*DP(c, F_G + ab) + fac * oochi * gt[ab] * dchi[c]);
  double ddchi[6];
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = x; y < 3; ++y)
      ddchi[sym(x, y)] = (x == y) ? fd_dxx(U, P, V_CHI, x, B.cidx2[x])
                                  : fd_dx(D, P, d1f(y, F_CHI), x, B.cidx1[x]);
  double ddg[6][6];
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = x; y < 3; ++y)
#pragma unroll
      for (int cd = 0; cd < 6; ++cd) {
        const double dchi_a = dchi[x];
        const double gtil = gt[cd];
        double v;
        if (x == y) {
          const double ddg_conf = fd_dxx(U, P, V_GXX + cd, x, B.cidx2[x]);
          v = p4 ? oochi * (ddg_conf -
                            oochi * (2.0 * dchi_a * *DP(x, F_G + cd) + ddchi[sym(x, x)] * gtil) +
                            2.0 * oochi * oochi * dchi_a * dchi_a * gtil)
                 : psi4 * (ddg_conf +
                           fac * oochi * (2.0 * dchi_a * *DP(x, F_G + cd) + ddchi[sym(x, x)] * gtil) +
                           fac * fac2 * oochi * oochi * dchi_a * dchi_a * gtil);
        } else {
          const double dchi_b = dchi[y];
          const double ddg_conf = fd_dx(D, P, d1f(y, F_G + cd), x, B.cidx1[x]);
          v = p4 ? oochi * (ddg_conf -
                            oochi * (dchi_a * *DP(y, F_G + cd) + dchi_b * *DP(x, F_G + cd) +
                                     ddchi[sym(x, y)] * gtil) +
                            2.0 * oochi * oochi * dchi_a * dchi_b * gtil)
                 : psi4 * (ddg_conf +
                           fac * oochi * (dchi_a * *DP(y, F_G + cd) + dchi_b * *DP(x, F_G + cd) +
                                          ddchi[sym(x, y)] * gtil) +
                           fac * fac2 * oochi * oochi * dchi_a * dchi_b * gtil);
        }
        ddg[sym(x, y)][cd] = v;
      }
  double guu[6];
  inv3(1. / det3(G), G, guu);
  double Gddd[3][6], Gudd[3][6];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int y = x; y < 3; ++y)
        Gddd[c][sym(x, y)] = 0.5 * (dg[x][sym(y, c)] + dg[y][sym(x, c)] - dg[c][sym(x, y)]);
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int ab = 0; ab < 6; ++ab) {
      double t = 0.0;
#pragma unroll
      for (int d = 0; d < 3; ++d) t += guu[sym(c, d)] * Gddd[d][ab];
      Gudd[c][ab] = t;
    }
  double R = 0.0;
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = x; y < 3; ++y) {
      double r = 0.0;
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
          for (int e = 0; e < 3; ++e)
            r += guu[sym(d, e)] * (Gudd[c][sym(x, e)] * Gddd[c][sym(y, d)] -
                                   Gudd[c][sym(x, y)] * Gddd[c][sym(e, d)]);
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int d = 0; d < 3; ++d)
          r += 0.5 * guu[sym(c, d)] *
               (-ddg[sym(y, x)][sym(c, d)] + ddg[sym(d, x)][sym(y, c)] +
                ddg[sym(d, y)][sym(x, c)] - ddg[sym(d, c)][sym(x, y)]);
      R += ((x == y) ? 1.0 : 2.0) * guu[sym(x, y)] * r;
    }
  double Kud[3][3], K = 0.0;
#pragma unroll
  for (int x = 0; x < 3; ++x) {
#pragma unroll
    for (int y = 0; y < 3; ++y) {
      double t = 0.0;
#pragma unroll
      for (int c = 0; c < 3; ++c) t += guu[sym(x, c)] * Kdd[sym(c, y)];
      Kud[x][y] = t;
    }
    K += Kud[x][x];
  }
  double KK = 0.0;
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = 0; y < 3; ++y) KK += Kud[x][y] * Kud[y][x];
  double DKudd[3][6];
  {
    double DKddd[3][6];
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int y = 0; y < 3; ++y)
#pragma unroll
        for (int c = y; c < 3; ++c) {
          double t = fd_dx(AD, P, A_KXX + sym(y, c), x, B.cidx1[x]);
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            t -= Gudd[d][sym(x, y)] * Kdd[sym(d, c)];
            t -= Gudd[d][sym(x, c)] * Kdd[sym(y, d)];
          }
          DKddd[x][sym(y, c)] = t;
        }
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int bc = 0; bc < 6; ++bc) {
        double t = 0.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) t += guu[sym(x, d)] * DKddd[d][bc];
        DKudd[x][bc] = t;
      }
  }
  const double H = R + (K * K) - KK - 16 * M_PI * rho;
  double Mu[3] = {0, 0, 0};
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = 0; y < 3; ++y) {
      Mu[x] -= 8 * M_PI * guu[sym(x, y)] * Sd[y];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        Mu[x] += guu[sym(x, y)] * DKudd[c][sym(y, c)];
        Mu[x] -= guu[sym(y, c)] * DKudd[x][sym(y, c)];
      }
    }
  double Md[3];
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    double t = 0;
#pragma unroll
    for (int y = 0; y < 3; ++y) t += G[sym(x, y)] * Mu[y];
    Md[x] = t;
  }
  double M = 0.;
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = x; y < 3; ++y)
      M += ((x == y) ? 1.0 : 2.0) * G[sym(x, y)] * Mu[x] * Mu[y];
  // conformal contracted Christoffel from the prepared conformal derivatives
  double cguu[6];
  inv3(1. / det3(gt), gt, cguu);
  double cGu[3];
  {
    double cGddd[3][6];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int x = 0; x < 3; ++x)
#pragma unroll
        for (int y = x; y < 3; ++y)
          cGddd[c][sym(x, y)] = 0.5 * (*DP(x, F_G + sym(y, c)) + *DP(y, F_G + sym(x, c)) -
                                       *DP(c, F_G + sym(x, y)));
    double cGudd[3][6];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int ab = 0; ab < 6; ++ab) {
        double t = 0.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) t += cguu[sym(c, d)] * cGddd[d][ab];
        cGudd[c][ab] = t;
      }
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      double t = 0.0;
#pragma unroll
      for (int y = 0; y < 3; ++y)
#pragma unroll
        for (int c = y; c < 3; ++c)
          t += ((y == c) ? 1.0 : 2.0) * cguu[sym(y, c)] * cGudd[x][sym(y, c)];
      cGu[x] = t;
    }
  }
  double Zc = 0.;
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = x; y < 3; ++y)
      Zc += ((x == y) ? 0.25 : 0.5) * G[sym(x, y)] * (u[(V_GAMX + x) * N + p] - cGu[x]) *
            (u[(V_GAMX + y) * N + p] - cGu[y]);
  const double x1 = B.x0[0] + i * B.dx[0];
  const double x2 = B.x0[1] + j * B.dx[1];
  const double x3 = B.x0[2] + k * B.dx[2];
  const double R2 = x1 * x1 + x2 * x2 + x3 * x3;
  const double th = u[V_THETA * N + p];
  const bool cut = R2 > a.r_max_con * a.r_max_con;
  con[C_H * N + p] = cut ? 0.0 : H;
  con[C_M * N + p] = cut ? 0.0 : M;
  con[C_Z * N + p] = cut ? 0.0 : Zc;
#pragma unroll
  for (int x = 0; x < 3; ++x) con[(C_MX + x) * N + p] = cut ? 0.0 : Md[x];
  con[C_C * N + p] = cut ? 0.0 : (H * H) + M + (th * th) + 4.0 * Zc;
#undef DP
}

// ---------------------------------------------------------------------------
// Elementwise kernels
// ---------------------------------------------------------------------------
constexpr int MAXK = 8;
struct BtArgs {
  double* out;
  const double* u0;
  const double* k[MAXK];
  double w[MAXK];  // already multiplied by dt; zero weights removed
  int nk;
  long long n;
};

__global__ void __launch_bounds__(256) k_bt_sum(BtArgs a) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < a.n; e += stride) {
    double v = a.u0[e];
    for (int s = 0; s < a.nk; ++s) v += a.w[s] * a.k[s][e];
    a.out[e] = v;
  }
}

__global__ void __launch_bounds__(256) k_fill(double* p, double v, long long n) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += stride) p[e] = v;
}

__global__ void __launch_bounds__(256) k_copy(double* dst, const double* src, long long n) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += stride) dst[e] = src[e];
}

struct WaveArgs {
  const DevBlock* blocks;
  Launch L;
  int nvar;
  double* out;
  const double* in1;
  const double* in2;
  double w[3];
  int mode;  // 0 WeightedAve, 1 AddRHS (w[0] = weight, in1 = rhs)
};

// MeshBlock::WeightedAveVC / WeightedAve_ (src/mesh/weighted_ave.cpp:21-132)
// and Z4c::AddZ4cRHS (src/z4c/add_z4c_rhs.cpp:24-34), interior vertices.
__global__ void __launch_bounds__(TILE) k_wave(WaveArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  const int N = B.npts;
  const long long base = B.off * a.nvar;
  const int p = flat(B, i, j, k);
  const double w0 = a.w[0], w1 = a.w[1], w2 = a.w[2];
  for (int n = 0; n < a.nvar; ++n) {
    const long long e = base + (long long)n * N + p;
    double* o = a.out + e;
    if (a.mode == 1) {
      *o += w0 * a.in1[e];
      continue;
    }
    if (w0 == 1.0) {
      if (w2 != 0.0) *o += w1 * a.in1[e] + w2 * a.in2[e];
      else if (w1 != 0.0) *o += w1 * a.in1[e];
    } else if (w0 == 0.0) {
      if (w2 != 0.0) *o = w1 * a.in1[e] + w2 * a.in2[e];
      else if (w1 == 1.0) *o = a.in1[e];
      else *o = w1 * a.in1[e];
    } else {
      if (w2 != 0.0) *o = w0 * *o + w1 * a.in1[e] + w2 * a.in2[e];
      else if (w1 != 0.0) *o = w0 * *o + w1 * a.in1[e];
      else *o *= w0;
    }
  }
}

// Periodic VC self-exchange: ghosts take the periodic image, shared
// boundary vertices the mean of their images.  In place, in two launches with
// a field per grid row: the ghosts, which read interior vertices only, then
// the shared vertices, each set of images (2, 4 or 8) read and written by one
// thread.  Against a snapshot of the whole state and one thread per vertex for
// all fields: a 65^3 block 69 -> 34 us.  A block of 2 or 3 cells along an axis
// has ghosts whose image is a ghost; such batches keep the snapshot.
struct PerArgs {
  const DevBlock* blocks;
  Launch L;
  int nvar;
  double* u;
  const double* snap;
};

__device__ __forceinline__ int images(int i, int lo, int hi, int* s) {
  const int n = hi - lo;
  if (i < lo) { s[0] = i + n; return 1; }
  if (i > hi) { s[0] = i - n; return 1; }
  if (i == lo) { s[0] = lo; s[1] = hi; return 2; }
  if (i == hi) { s[0] = hi; s[1] = lo; return 2; }
  s[0] = i;
  return 1;
}

__global__ void __launch_bounds__(TILE) k_periodic(PerArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  int si[2], sj[2], sk[2];
  const int ni = images(i, B.il, B.iu, si);
  const int nj = images(j, B.jl, B.ju, sj);
  const int nk = images(k, B.kl, B.ku, sk);
  if (ni * nj * nk == 1 && si[0] == i && sj[0] == j && sk[0] == k) return;
  const int N = B.npts;
  const long long base = B.off * a.nvar;
  for (int n = 0; n < a.nvar; ++n) {
    const double* s = a.snap + base + (long long)n * N;
    double acc = 0.0;
    for (int x = 0; x < nk; ++x)
      for (int y = 0; y < nj; ++y)
        for (int z = 0; z < ni; ++z) acc += s[si[z] + B.nn1 * (sj[y] + B.nn2 * sk[x])];
    a.u[base + (long long)n * N + flat(B, i, j, k)] = acc / (double)(ni * nj * nk);
  }
}


__global__ void __launch_bounds__(TILE) k_periodic_ghosts(PerArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  int si[2], sj[2], sk[2];
  const int ni = images(i, B.il, B.iu, si);
  const int nj = images(j, B.jl, B.ju, sj);
  const int nk = images(k, B.kl, B.ku, sk);
  double* u = a.u + B.off * a.nvar + (long long)blockIdx.y * B.npts;
  double acc = 0.0;
  for (int x = 0; x < nk; ++x)
    for (int y = 0; y < nj; ++y)
      for (int z = 0; z < ni; ++z) acc += u[si[z] + B.nn1 * (sj[y] + B.nn2 * sk[x])];
  u[flat(B, i, j, k)] = acc / (double)(ni * nj * nk);
}

// One thread per set of images (its vertex on the lower faces).  Every image
// is the mean summed from itself on, as it would be formed at that vertex.
__global__ void __launch_bounds__(TILE) k_periodic_faces(PerArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  int si[2], sj[2], sk[2];
  const int ni = images(i, B.il, B.iu, si);
  const int nj = images(j, B.jl, B.ju, sj);
  const int nk = images(k, B.kl, B.ku, sk);
  double* u = a.u + B.off * a.nvar + (long long)blockIdx.y * B.npts;
  double v[2][2][2] = {};
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int z = 0; z < 2; ++z)
        if (x < nk && y < nj && z < ni) v[x][y][z] = u[si[z] + B.nn1 * (sj[y] + B.nn2 * sk[x])];
#pragma unroll
  for (int ox = 0; ox < 2; ++ox)
#pragma unroll
    for (int oy = 0; oy < 2; ++oy)
#pragma unroll
      for (int oz = 0; oz < 2; ++oz) {
        if (ox >= nk || oy >= nj || oz >= ni) continue;
        double acc = 0.0;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int z = 0; z < 2; ++z)
              if (x < nk && y < nj && z < ni) acc += v[x ^ ox][y ^ oy][z ^ oz];
        u[si[oz] + B.nn1 * (sj[oy] + B.nn2 * sk[ox])] = acc / (double)(ni * nj * nk);
      }
}

// Physical ghost fill of vertex-centred data (src/comm/physical_bcs.cpp:
// 187-290 ExtrapolateOutflowBC, ranges :506-676): one thread per ghost line
// (a field and two transverse coordinates), filling the four ghost layers
// outward in order, each from the five vertices inside it, with the weights
// of InterpolateLagrangeUniformBiasR<5>.  One launch per axis.
struct PhysLine {
  int block;
  int lo0, n0, lo1, n1;  // transverse ranges (fast, slow)
  long long start;       // first line of this entry
};
struct PhysArgs {
  const DevBlock* blocks;
  const PhysLine* lines;
  int nent;
  long long nlines1;  // lines per field
  long long nlines;   // nlines1 * nvar
  int axis;
  int nvar;
  double* u;
};

__global__ void __launch_bounds__(256) k_physical(PhysArgs a) {
  const long long Lg = (long long)blockIdx.x * 256 + threadIdx.x;
  if (Lg >= a.nlines) return;
  const int n = (int)(Lg / a.nlines1);  // field
  const long long L = Lg - (long long)n * a.nlines1;
  int lo = 0, hi = a.nent - 1;  // last entry with start <= L
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.lines[mid].start <= L) lo = mid; else hi = mid - 1;
  }
  const PhysLine E = a.lines[lo];
  const DevBlock B = a.blocks[E.block];
  const int r = (int)(L - E.start);
  const int t1 = E.lo1 + r / E.n0, t0 = E.lo0 + r % E.n0;
  const long long str[3] = {1, B.nn1, (long long)B.nn1 * B.nn2};
  const int ax = a.axis;
  // position of the line's axis-0 point and the other two coordinates
  const int o0 = ax == 0 ? 1 : 0, o1 = ax == 2 ? 1 : 2;  // axes of t0, t1
  double* v = a.u + B.off * a.nvar + (long long)n * B.npts + t0 * str[o0] + t1 * str[o1];
  const long long s = str[ax];
  const int lo_v = ax == 0 ? B.il : (ax == 1 ? B.jl : B.kl);
  const int ie = (ax == 0 ? B.iu : (ax == 1 ? B.ju : B.ku)) - 1;  // cell-centred end
  const double c[5] = {5., -10., 10., -5., 1.};
  if (B.pfaces & (1 << (2 * ax))) {
    for (int i = lo_v - 1; i >= lo_v - NG; --i) {
      double x = 0.0;
#pragma unroll
      for (int p = 0; p < 5; ++p) x += c[p] * v[(i + p + 1) * s];
      v[i * s] = x;
    }
  }
  if (B.pfaces & (2 << (2 * ax))) {
    for (int i = ie + 1; i <= ie + NG; ++i) {
      double x = 0.0;
#pragma unroll
      for (int p = 0; p < 5; ++p) x += c[p] * v[(i - p - 1) * s];
      v[i * s] = x;
    }
  }
}

// Same-level VC exchange between blocks (src/comm/comm_channel.cpp:1277-1330
// additive unpack, src/comm/node_multiplicity.cpp:349-420 division): each
// destination vertex takes the sum of its owners' values (interior vertices
// of any block at the same lattice point, in block and k, j, i order) from a
// snapshot, times 1/multiplicity.  One thread per destination.
struct ExArgs {
  const DevBlock* blocks;
  const int* dst;      // 2 ints per destination: block, point
  const int* src_off;  // CSR offsets into src
  const int* src;      // 2 ints per source: block, point
  int ndst;
  int nvar;
  double* u;
  double* tmp;         // nvar * ndst: the new values, field-major
};

// Phase 1: every destination's new value from the state as it stands (no
// destination is written yet, so shared vertices read their old values).
__global__ void __launch_bounds__(256) k_exchange_gather(ExArgs a) {
  const int d = blockIdx.x * 256 + threadIdx.x;
  if (d >= a.ndst) return;
  const int s0 = a.src_off[d], s1 = a.src_off[d + 1];
  const int cnt = s1 - s0;
  const double inv = 1.0 / (double)cnt;
  for (int n = 0; n < a.nvar; ++n) {
    double acc = 0.0;
    for (int e = s0; e < s1; ++e) {
      const DevBlock& S = a.blocks[a.src[2 * e]];
      acc += a.u[S.off * a.nvar + (long long)n * S.npts + a.src[2 * e + 1]];
    }
    a.tmp[(long long)n * a.ndst + d] = cnt > 1 ? acc * inv : acc;
  }
}

// Phase 2: the new values into the state.
__global__ void __launch_bounds__(256) k_exchange_scatter(ExArgs a) {
  const int d = blockIdx.x * 256 + threadIdx.x;
  if (d >= a.ndst) return;
  const DevBlock B = a.blocks[a.dst[2 * d]];
  const int p = a.dst[2 * d + 1];
  for (int n = 0; n < a.nvar; ++n)
    a.u[B.off * a.nvar + (long long)n * B.npts + p] = a.tmp[(long long)n * a.ndst + d];
}

// Transpose of the same-level exchange on a cotangent u-bar (z4c_exchange_vjp):
// the exchange sets destination d to w_d * (sum of its sources), w_d = 1/cnt
// (1 for a single source), and leaves every other vertex alone.  So a
// source vertex v receives sum_{d reading v} w_d ubar_d, plus its own ubar
// unless v is itself a destination; a destination that is no source (a
// ghost) receives zero.  Gather into a scratch, then scatter, so every
// value read is a pre-transpose value; the sums run in destination order.
struct ExTArgs {
  const DevBlock* blocks;
  const int* dst;      // the exchange's destinations (2 ints each)
  const int* src_off;  // the exchange's CSR offsets (source counts)
  const int* v;        // source vertices (2 ints each)
  const int* flag;     // 1 if the source vertex is also a destination
  const int* voff;     // CSR offsets into vd
  const int* vd;       // destinations reading each source vertex
  const int* z;        // destinations that are no source
  int nv, nz, nvar;
  double* ubar;
  double* tmp;         // nvar * nv
};

// NV > 0: nvar == NV with the accumulators in registers; NV == 0: any
// nvar, one field at a time (the same order of sums per field)
template <int NV>
__global__ void __launch_bounds__(256) k_exchange_vjp_gather(ExTArgs a) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= a.nv) return;
  const DevBlock& V = a.blocks[a.v[2 * t]];
  const int pv = a.v[2 * t + 1];
  const int e0 = a.voff[t], e1 = a.voff[t + 1];
  if constexpr (NV > 0) {
    double acc[NV];
    const bool self = !a.flag[t];
    const double* vp = a.ubar + V.off * a.nvar + pv;
#pragma unroll
    for (int n = 0; n < NV; ++n) acc[n] = self ? vp[(long long)n * V.npts] : 0.0;
    for (int e = e0; e < e1; ++e) {
      const int d = a.vd[e];
      const int cnt = a.src_off[d + 1] - a.src_off[d];
      const DevBlock& D = a.blocks[a.dst[2 * d]];
      const double* dp = a.ubar + D.off * a.nvar + a.dst[2 * d + 1];
      const double w = 1.0 / (double)cnt;
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        const double ud = dp[(long long)n * D.npts];
        acc[n] += cnt > 1 ? ud * w : ud;
      }
    }
#pragma unroll
    for (int n = 0; n < NV; ++n) a.tmp[(long long)n * a.nv + t] = acc[n];
    return;
  }
  for (int n = 0; n < a.nvar; ++n) {
    double acc = a.flag[t] ? 0.0 : a.ubar[V.off * a.nvar + (long long)n * V.npts + pv];
    for (int e = e0; e < e1; ++e) {
      const int d = a.vd[e];
      const int cnt = a.src_off[d + 1] - a.src_off[d];
      const DevBlock& D = a.blocks[a.dst[2 * d]];
      const double ud = a.ubar[D.off * a.nvar + (long long)n * D.npts + a.dst[2 * d + 1]];
      acc += cnt > 1 ? ud * (1.0 / (double)cnt) : ud;
    }
    a.tmp[(long long)n * a.nv + t] = acc;
  }
}

__global__ void __launch_bounds__(256) k_exchange_vjp_scatter(ExTArgs a) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t < a.nv) {
    const DevBlock& V = a.blocks[a.v[2 * t]];
    const int pv = a.v[2 * t + 1];
    for (int n = 0; n < a.nvar; ++n)
      a.ubar[V.off * a.nvar + (long long)n * V.npts + pv] = a.tmp[(long long)n * a.nv + t];
  } else if (t < a.nv + a.nz) {
    const int d = a.z[t - a.nv];
    const DevBlock& D = a.blocks[a.dst[2 * d]];
    for (int n = 0; n < a.nvar; ++n)
      a.ubar[D.off * a.nvar + (long long)n * D.npts + a.dst[2 * d + 1]] = 0.0;
  }
}


// ---------------------------------------------------------------------------
// Vertex-centred restriction and prolongation between levels
// (src/mesh/mesh_refinement_vc.cpp; the index algebra and the per-vertex
// operator are in z4c_refine.hpp).  The restriction takes a host-built chunk
// table (workgroup w handles coarse vertices start .. start+255 of block ent,
// one thread per vertex, all fields); the prolongation takes groups of boxes
// whose coarse reads are staged in LDS (PrGroup below).
// ---------------------------------------------------------------------------
struct RfBlock {
  long long coff;     // point offset of the block's coarse buffer
  int cn1, cn2, cn3;  // coarse vertex counts per axis (nx/2 + 9)
  int cnpts;          // cn1*cn2*cn3
  int cni, cnj, cnk;  // coarse interior vertex counts (nx/2 + 1)
};

struct RfChunk {
  int ent;
  int start;
};

struct RestrictArgs {
  const DevBlock* blocks;
  const RfBlock* cb;
  const RfChunk* chunks;
  int nvar;
  const double* u;
  double* coarse;
};

// RestrictInterior (src/comm/refinement_ops.cpp:178-205) ->
// RestrictVertexCenteredValues (src/mesh/mesh_refinement_vc.cpp:56-100):
// injection of the fine vertex at each coarse interior vertex.
__global__ void __launch_bounds__(256) k_restrict_vc(RestrictArgs a) {
  const RfChunk ch = a.chunks[blockIdx.x];
  const RfBlock R = a.cb[ch.ent];
  const int t = ch.start + (int)threadIdx.x;
  if (t >= R.cni * R.cnj * R.cnk) return;
  const DevBlock& B = a.blocks[ch.ent];
  const int ci = RF_NCG + t % R.cni, cj = RF_NCG + (t / R.cni) % R.cnj,
            ck = RF_NCG + t / (R.cni * R.cnj);
  const int i = rf_fine_of(ci, RF_NCG, RF_NCG + R.cni - 1, B.il, B.iu);
  const int j = rf_fine_of(cj, RF_NCG, RF_NCG + R.cnj - 1, B.jl, B.ju);
  const int k = rf_fine_of(ck, RF_NCG, RF_NCG + R.cnk - 1, B.kl, B.ku);
  const long long p = i + (long long)B.nn1 * (j + (long long)B.nn2 * k);
  const long long cp = ci + (long long)R.cn1 * (cj + (long long)R.cn2 * ck);
  const double* src = a.u + B.off * a.nvar + p;
  double* dst = a.coarse + R.coff * a.nvar + cp;
  for (int n = 0; n < a.nvar; ++n) dst[(long long)n * R.cnpts] = src[(long long)n * B.npts];
}

// A workgroup of the prolongation: entries [e0, e0 + ne) of one block, all
// of whose coarse reads lie in the box r0 + [0, rn) of the block's coarse
// buffer, which the workgroup stages in LDS (one field per workgroup).
struct PrGroup {
  int blk;
  int e0, ne;
  int r0[3], rn[3];
};
constexpr int PR_LDS = 8192;  // largest staged box, doubles (64 KiB)

struct ProlongArgs {
  const DevBlock* blocks;
  const RfBlock* cb;
  const RfEntry* ent;
  const PrGroup* groups;
  const double* coarse;
  double* u;
  int nvar;
};

// ProlongateVertexCenteredValues (src/mesh/mesh_refinement_vc.cpp:283-772):
// grid (groups, fields).  The coarse box is copied to LDS once, then each
// entry's vertices are taken one case at a time (the parities of the three
// fine indices), so a wave runs one case's stencil; the arithmetic is
// rf_prolong_point's.  A fine vertex's value depends only on the coarse
// buffer and its (coarse index, case), so entries whose boxes overlap store
// the same value there.
__global__ void __launch_bounds__(256) k_prolong_vc(ProlongArgs a) {
  extern __shared__ double cl[];
  const PrGroup G = a.groups[blockIdx.x];
  const int f = blockIdx.y;
  const DevBlock& B = a.blocks[G.blk];
  const RfBlock& R = a.cb[G.blk];
  const int s2 = G.rn[0], s3 = G.rn[0] * G.rn[1], nv = s3 * G.rn[2];
  {
    const double* C = a.coarse + R.coff * a.nvar + (long long)f * R.cnpts;
    for (int t = threadIdx.x; t < nv; t += 256) {
      const int k = t / s3, r = t - k * s3, j = r / s2, i = r - j * s2;
      cl[t] = C[(G.r0[0] + i) + (long long)R.cn1 * ((G.r0[1] + j) + (long long)R.cn2 * (G.r0[2] + k))];
    }
  }
  __syncthreads();
  const int nn1 = B.nn1, nn2 = B.nn2;
  double* dst = a.u + B.off * a.nvar + (long long)f * B.npts;
  for (int q = G.e0; q < G.e0 + G.ne; ++q) {
    const RfEntry E = a.ent[q];
    // both x parities of a coarse index per thread: the two cases differ
    // only in their x stencil, and the thread writes the adjacent fine
    // vertices 2 (ci - RF_H) and 2 (ci - RF_H) + 1 (coalesced stores)
    int x0[2], xn[2];
    rf_case_range(E, 0, 0, x0[0], xn[0]);
    rf_case_range(E, 0, 1, x0[1], xn[1]);
    int xlo = INT_MAX, xhi = INT_MIN;
    for (int h = 0; h < 2; ++h)
      if (xn[h] > 0) {
        xlo = min(xlo, x0[h]);
        xhi = max(xhi, x0[h] + xn[h]);
      }
    if (xlo >= xhi) continue;
    const int nx = xhi - xlo;
    for (int m2 = 0; m2 < 4; ++m2) {
      const int pj = m2 & 1, pk = m2 >> 1;
      int cy0, ny, cz0, nz;
      rf_case_range(E, 1, pj, cy0, ny);
      rf_case_range(E, 2, pk, cz0, nz);
      if (ny <= 0 || nz <= 0) continue;
      const int mb = (pj << 1) | (pk << 2);
      const int nxy = nx * ny, np = nxy * nz;
      for (int t = threadIdx.x; t < np; t += 256) {
        const int tk = t / nxy, r = t - tk * nxy, tj = r / nx, ti = r - tj * nx;
        const int ci = xlo + ti, cj = cy0 + tj, ck = cz0 + tk;
        const int li = ci - G.r0[0], lj = cj - G.r0[1], lk = ck - G.r0[2];
        const int fj = 2 * (cj - RF_H) + pj, fk = 2 * (ck - RF_H) + pk;
        double* row = dst + (long long)nn1 * (fj + (long long)nn2 * fk) + 2 * (ci - RF_H);
        if (ci >= x0[0] && ci < x0[0] + xn[0]) row[0] = rf_prolong_point(cl, s2, s3, li, lj, lk, mb);
        if (ci >= x0[1] && ci < x0[1] + xn[1])
          row[1] = rf_prolong_point(cl, s2, s3, li, lj, lk, mb | 1);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Ghost update across refinement levels (the plan of z4c_mesh.hpp): every
// destination vertex (fine array or coarse buffer) is its ordered source
// list summed from zero, times 1/multiplicity, all fields.  Sources are
// interior vertices, read before any of them is written: ghost destinations
// (never sources) are written at once, interior destinations (the first
// nint; shared boundary vertices, also sources) go through a scratch and a
// second launch, as the reference packs every message before the receivers
// unpack.  A reference 2*b + A addresses block b's fine array (A = 0) or
// coarse buffer (A = 1).
// ---------------------------------------------------------------------------
struct MlxArgs {
  const DevBlock* blocks;
  const RfBlock* cb;
  const int* dst;
  const long long* off;
  const int* src;
  const double* inv;
  int ndst;
  int nint;
  int nvar;
  double* u;
  double* coarse;
  double* tmp;  // nvar * nint, field-major
};

// base pointer and field stride of a vertex reference
__device__ __forceinline__ double* mlx_ptr(const MlxArgs& a, int blkarr, int p, long long& fs) {
  const int b = blkarr >> 1;
  if (blkarr & 1) {
    const RfBlock& R = a.cb[b];
    fs = R.cnpts;
    return a.coarse + R.coff * a.nvar + p;
  }
  const DevBlock& B = a.blocks[b];
  fs = B.npts;
  return a.u + B.off * a.nvar + p;
}

// NV > 0: exactly NV fields, sources outer (each resolved once) and the
// fields' sums in registers; NV = 0: any nvar, fields outer.  Every field's
// sum adds the sources in list order either way.
template <int NV>
__global__ void __launch_bounds__(256) k_mlx_gather(MlxArgs a) {
  const int d = blockIdx.x * 256 + threadIdx.x;
  if (d >= a.ndst) return;
  const long long s0 = a.off[d], s1 = a.off[d + 1];
  const double inv = a.inv[d];
  long long dfs;
  double* const dp = mlx_ptr(a, a.dst[2 * d], a.dst[2 * d + 1], dfs);
  if constexpr (NV > 0) {
    double acc[NV];
#pragma unroll
    for (int n = 0; n < NV; ++n) acc[n] = 0.0;
    for (long long e = s0; e < s1; ++e) {
      long long fs;
      const double* sp = mlx_ptr(a, a.src[2 * e], a.src[2 * e + 1], fs);
#pragma unroll
      for (int n = 0; n < NV; ++n) acc[n] += sp[n * fs];
    }
    if (d < a.nint) {
#pragma unroll
      for (int n = 0; n < NV; ++n) a.tmp[(long long)n * a.nint + d] = acc[n] * inv;
    } else {
#pragma unroll
      for (int n = 0; n < NV; ++n) dp[n * dfs] = acc[n] * inv;
    }
  } else {
    for (int n = 0; n < a.nvar; ++n) {
      double acc = 0.0;
      for (long long e = s0; e < s1; ++e) {
        long long fs;
        const double* sp = mlx_ptr(a, a.src[2 * e], a.src[2 * e + 1], fs);
        acc += sp[n * fs];
      }
      if (d < a.nint)
        a.tmp[(long long)n * a.nint + d] = acc * inv;
      else
        dp[n * dfs] = acc * inv;
    }
  }
}

__global__ void __launch_bounds__(256) k_mlx_scatter(MlxArgs a) {
  const int d = blockIdx.x * 256 + threadIdx.x;
  if (d >= a.nint) return;
  long long fs;
  double* const dp = mlx_ptr(a, a.dst[2 * d], a.dst[2 * d + 1], fs);
  for (int n = 0; n < a.nvar; ++n) dp[n * fs] = a.tmp[(long long)n * a.nint + d];
}

// ApplyPhysicalBCsOnCoarseLevel (src/comm/physical_bcs.cpp:687-876) for a
// block that prolongates: the fine level's face fill (k_physical) on the
// block's coarse buffer with the vertex-centred coarse ranges civs..cive
// that Z4c passes (src/z4c/z4c.cpp:48-58), so a face fills the 4 coarse
// ghosts beyond civs / cive by the 5-point extrapolation and keeps the
// boundary vertex; one thread per (field, line), faces in order x1, x2, x3.
struct PhysCArgs {
  const DevBlock* blocks;
  const RfBlock* cb;
  const PhysLine* lines;
  int nent;
  long long nlines1;
  long long nlines;
  int axis;
  int nvar;
  double* coarse;
};

__global__ void __launch_bounds__(256) k_physical_coarse(PhysCArgs a) {
  const long long Lg = (long long)blockIdx.x * 256 + threadIdx.x;
  if (Lg >= a.nlines) return;
  const int n = (int)(Lg / a.nlines1);
  const long long L = Lg - (long long)n * a.nlines1;
  int lo = 0, hi = a.nent - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.lines[mid].start <= L) lo = mid; else hi = mid - 1;
  }
  const PhysLine E = a.lines[lo];
  const RfBlock R = a.cb[E.block];
  const int pf = a.blocks[E.block].pfaces;
  const int r = (int)(L - E.start);
  const int t1 = E.lo1 + r / E.n0, t0 = E.lo0 + r % E.n0;
  const long long str[3] = {1, R.cn1, (long long)R.cn1 * R.cn2};
  const int ax = a.axis;
  const int o0 = ax == 0 ? 1 : 0, o1 = ax == 2 ? 1 : 2;
  double* v = a.coarse + R.coff * a.nvar + (long long)n * R.cnpts + t0 * str[o0] + t1 * str[o1];
  const long long s = str[ax];
  const int cni = ax == 0 ? R.cni : (ax == 1 ? R.cnj : R.cnk);
  const int vs = RF_NCG, ve = RF_NCG + cni - 1;
  const double c[5] = {5., -10., 10., -5., 1.};
  if (pf & (1 << (2 * ax))) {
    for (int i = vs - 1; i >= vs - RF_NCG; --i) {
      double x = 0.0;
#pragma unroll
      for (int p = 0; p < 5; ++p) x += c[p] * v[(i + p + 1) * s];
      v[i * s] = x;
    }
  }
  if (pf & (2 << (2 * ax))) {
    for (int i = ve + 1; i <= ve + RF_NCG; ++i) {
      double x = 0.0;
#pragma unroll
      for (int p = 0; p < 5; ++p) x += c[p] * v[(i - p - 1) * s];
      v[i * s] = x;
    }
  }
}

// ---------------------------------------------------------------------------
// Transpose of the ghost update across levels (z4c_exchange_vjp on several
// spacings).  The update is linear in the fine state: u' = P Phi_c E_g R u
// (restriction into the coarse buffers, the gather, the coarse level's
// physical fill, prolongation; vertices none of them writes pass through),
// so its transpose runs P^T, Phi_c^T, E_g^T, R^T on (u-bar, c-bar) with
// c-bar = 0 to start.  Every step is a fixed-order gather (deterministic).
// ---------------------------------------------------------------------------

// P^T: each coarse vertex c the prolongation reads gathers w * u-bar_f over
// the fine vertices f the prolongation writes (the mask: each counted once,
// however many boxes overlap there) whose stencil holds it.  Per axis a
// fine vertex either injects coarse index c (even f = 2 (c - RF_H), weight
// 1) or interpolates around base i (odd f = 2 (i - RF_H) + 1, reading
// i - 2 .. i + 3 with the 6-point midpoint weights), and its weight is the
// product over the axes, so P^T is three 1-D transposes of at most 7 terms
// (z, then y, then x).  One workgroup per tile (a block's coarse rows
// [cy0, cy0 + ncy) x [cz0, cz0 + ncz) over its coarse x range) and field:
// the masked fine cotangents the tile reads are staged in LDS, the z and y
// transposes go through two LDS intermediates, and every coarse vertex of
// the tile is written once (zero where nothing reads it).  The fine
// cotangents written are then zeroed.
struct PrTTile {
  int blk;
  int cx0, ncx, cy0, ncy, cz0, ncz;  // coarse vertices written
  int fx0, nfx, fy0, nfy, fz0, nfz;  // fine vertices staged
};
struct PrTArgs {
  const DevBlock* blocks;
  const RfBlock* cb;
  const PrTTile* tiles;
  const int* fl;   // fine vertices the prolongation writes (block, point)
  int nfl;
  const unsigned char* fmask;
  int nvar;
  double* ubar;
  double* cbar;
};

// sum over the fine candidates of coarse index c on one axis: get(k) reads
// the staged value at fine offset k = f - f0 (0 <= k < nf)
template <class Get>
__device__ __forceinline__ double prt_axis_sum(int c, int f0, int nf, Get get) {
  double acc = 0.0;
  const int fe = 2 * (c - RF_H) - f0;
  if (fe >= 0 && fe < nf) acc += get(fe);
#pragma unroll
  for (int o = -2; o <= 3; ++o) {
    const int fo = fe - 2 * o + 1;  // odd vertex around base c - o
    if (fo >= 0 && fo < nf) acc += rf_lag(o >= 1 ? 3 - o : 2 + o) * get(fo);
  }
  return acc;
}

constexpr int PRT_THREADS = 512;

__global__ void __launch_bounds__(PRT_THREADS) k_prolong_vjp(PrTArgs a) {
  extern __shared__ double lds[];
  const PrTTile T = a.tiles[blockIdx.x];
  const int n = blockIdx.y;
  const DevBlock& B = a.blocks[T.blk];
  const RfBlock& R = a.cb[T.blk];
  const int nfx = T.nfx, nfy = T.nfy, nfz = T.nfz;
  double* F = lds;                        // [z][y][x] staged fine cotangents
  double* T1 = F + nfx * nfy * nfz;       // [kz][y][x] after the z transpose
  double* T2 = T1 + nfx * nfy * T.ncz;    // [kz][ky][x] after the y transpose
  const double* ub = a.ubar + B.off * a.nvar + (long long)n * B.npts;
  const unsigned char* mk = a.fmask + B.off;
  const int nF = nfx * nfy * nfz;
  // both loads unconditional (every staged vertex lies in the block), so
  // the iterations' loads overlap
#pragma unroll 4
  for (int q = threadIdx.x; q < nF; q += PRT_THREADS) {
    const int x = q % nfx, r = q / nfx, y = r % nfy, z = r / nfy;
    const long long p = (T.fx0 + x) + (long long)B.nn1 * ((T.fy0 + y) + (long long)B.nn2 * (T.fz0 + z));
    const double v = ub[p];
    F[q] = mk[p] ? v : 0.0;
  }
  __syncthreads();
  const int n1 = nfx * nfy * T.ncz;
  for (int q = threadIdx.x; q < n1; q += PRT_THREADS) {
    const int xy = q % (nfx * nfy), kz = q / (nfx * nfy);
    T1[q] = prt_axis_sum(T.cz0 + kz, T.fz0, nfz,
                         [&](int k) { return F[xy + nfx * nfy * k]; });
  }
  __syncthreads();
  const int n2 = nfx * T.ncy * T.ncz;
  for (int q = threadIdx.x; q < n2; q += PRT_THREADS) {
    const int x = q % nfx, r = q / nfx, ky = r % T.ncy, kz = r / T.ncy;
    const double* t1 = T1 + x + nfx * nfy * kz;
    T2[q] = prt_axis_sum(T.cy0 + ky, T.fy0, nfy, [&](int k) { return t1[nfx * k]; });
  }
  __syncthreads();
  const int n3 = T.ncx * T.ncy * T.ncz;
  double* cbo = a.cbar + R.coff * a.nvar + (long long)n * R.cnpts;
  for (int q = threadIdx.x; q < n3; q += PRT_THREADS) {
    const int kx = q % T.ncx, r = q / T.ncx, ky = r % T.ncy, kz = r / T.ncy;
    const double* t2 = T2 + nfx * (ky + T.ncy * kz);
    const double v = prt_axis_sum(T.cx0 + kx, T.fx0, nfx, [&](int k) { return t2[k]; });
    cbo[(T.cx0 + kx) + R.cn1 * ((T.cy0 + ky) + R.cn2 * (T.cz0 + kz))] = v;
  }
}

__global__ void __launch_bounds__(256) k_prolong_vjp_zero(PrTArgs a) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= a.nfl) return;
  const DevBlock& B = a.blocks[a.fl[2 * t]];
  double* u = a.ubar + B.off * a.nvar + a.fl[2 * t + 1];
  for (int n = 0; n < a.nvar; ++n) u[(long long)n * B.npts] = 0.0;
}

// Transpose of one 5-point extrapolation line (the physical fill, fine or
// coarse): the forward fills the lower face's ghosts outward, then the upper
// face's (from the last cell-centred interior vertex on); the transpose runs
// those assignments in reverse order, each v[g] = sum c_p v[g -+ (p + 1)]
// becoming v-bar[g -+ (p + 1)] += c_p v-bar[g], then v-bar[g] = 0.
__device__ __forceinline__ void phys_line_vjp(double* v, long long s, bool lower, bool upper,
                                              int lo_v, int ie, int ng) {
  const double c[5] = {5., -10., 10., -5., 1.};
  if (upper) {
    for (int i = ie + ng; i >= ie + 1; --i) {
      const double g = v[i * s];
      v[i * s] = 0.0;
#pragma unroll
      for (int p = 0; p < 5; ++p) v[(i - p - 1) * s] += c[p] * g;
    }
  }
  if (lower) {
    for (int i = lo_v - ng; i <= lo_v - 1; ++i) {
      const double g = v[i * s];
      v[i * s] = 0.0;
#pragma unroll
      for (int p = 0; p < 5; ++p) v[(i + p + 1) * s] += c[p] * g;
    }
  }
}

__global__ void __launch_bounds__(256) k_physical_vjp(PhysArgs a) {
  const long long Lg = (long long)blockIdx.x * 256 + threadIdx.x;
  if (Lg >= a.nlines) return;
  const int n = (int)(Lg / a.nlines1);
  const long long L = Lg - (long long)n * a.nlines1;
  int lo = 0, hi = a.nent - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.lines[mid].start <= L) lo = mid; else hi = mid - 1;
  }
  const PhysLine E = a.lines[lo];
  const DevBlock B = a.blocks[E.block];
  const int r = (int)(L - E.start);
  const int t1 = E.lo1 + r / E.n0, t0 = E.lo0 + r % E.n0;
  const long long str[3] = {1, B.nn1, (long long)B.nn1 * B.nn2};
  const int ax = a.axis;
  const int o0 = ax == 0 ? 1 : 0, o1 = ax == 2 ? 1 : 2;
  double* v = a.u + B.off * a.nvar + (long long)n * B.npts + t0 * str[o0] + t1 * str[o1];
  const int lo_v = ax == 0 ? B.il : (ax == 1 ? B.jl : B.kl);
  const int ie = (ax == 0 ? B.iu : (ax == 1 ? B.ju : B.ku)) - 1;
  phys_line_vjp(v, str[ax], B.pfaces & (1 << (2 * ax)), B.pfaces & (2 << (2 * ax)), lo_v, ie, NG);
}

__global__ void __launch_bounds__(256) k_physical_coarse_vjp(PhysCArgs a) {
  const long long Lg = (long long)blockIdx.x * 256 + threadIdx.x;
  if (Lg >= a.nlines) return;
  const int n = (int)(Lg / a.nlines1);
  const long long L = Lg - (long long)n * a.nlines1;
  int lo = 0, hi = a.nent - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.lines[mid].start <= L) lo = mid; else hi = mid - 1;
  }
  const PhysLine E = a.lines[lo];
  const RfBlock R = a.cb[E.block];
  const int pf = a.blocks[E.block].pfaces;
  const int r = (int)(L - E.start);
  const int t1 = E.lo1 + r / E.n0, t0 = E.lo0 + r % E.n0;
  const long long str[3] = {1, R.cn1, (long long)R.cn1 * R.cn2};
  const int ax = a.axis;
  const int o0 = ax == 0 ? 1 : 0, o1 = ax == 2 ? 1 : 2;
  double* v = a.coarse + R.coff * a.nvar + (long long)n * R.cnpts + t0 * str[o0] + t1 * str[o1];
  const int cni = ax == 0 ? R.cni : (ax == 1 ? R.cnj : R.cnk);
  phys_line_vjp(v, str[ax], pf & (1 << (2 * ax)), pf & (2 << (2 * ax)), RF_NCG,
                RF_NCG + cni - 1, RF_NCG);
}

// E_g^T over fine and coarse references (a reference 2 b + A: block b's fine
// array, A = 0, or coarse buffer, A = 1): a source receives sum inv_d
// ubar_d over the destinations reading it, plus its own unless it is a
// destination; a destination that is no source receives zero.
struct MltArgs {
  const DevBlock* blocks;
  const RfBlock* cb;
  const int* dst;
  const double* inv;
  const int* v;
  const int* flag;
  const int* voff;
  const int* vd;
  const int* z;
  int nv, nz, nvar;
  double* ubar;
  double* cbar;
  double* tmp;  // nvar * nv
};

__device__ __forceinline__ double* mlt_ptr(const MltArgs& a, int blkarr, int p, long long& fs) {
  const int b = blkarr >> 1;
  if (blkarr & 1) {
    const RfBlock& R = a.cb[b];
    fs = R.cnpts;
    return a.cbar + R.coff * a.nvar + p;
  }
  const DevBlock& B = a.blocks[b];
  fs = B.npts;
  return a.ubar + B.off * a.nvar + p;
}

// NV > 0: nvar == NV, the accumulators in registers and each destination
// resolved once; NV == 0: any nvar, one field at a time.  Both sum each
// field in the same order.
template <int NV>
__global__ void __launch_bounds__(256) k_mlx_vjp_gather(MltArgs a) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= a.nv) return;
  long long fs;
  const double* vp = mlt_ptr(a, a.v[2 * t], a.v[2 * t + 1], fs);
  const int e0 = a.voff[t], e1 = a.voff[t + 1];
  if constexpr (NV > 0) {
    double acc[NV];
    const bool self = !a.flag[t];
#pragma unroll
    for (int n = 0; n < NV; ++n) acc[n] = self ? vp[n * fs] : 0.0;
    for (int e = e0; e < e1; ++e) {
      const int d = a.vd[e];
      long long dfs;
      const double* dp = mlt_ptr(a, a.dst[2 * d], a.dst[2 * d + 1], dfs);
      const double w = a.inv[d];
#pragma unroll
      for (int n = 0; n < NV; ++n) acc[n] += w * dp[n * dfs];
    }
#pragma unroll
    for (int n = 0; n < NV; ++n) a.tmp[(long long)n * a.nv + t] = acc[n];
    return;
  }
  for (int n = 0; n < a.nvar; ++n) {
    double acc = a.flag[t] ? 0.0 : vp[n * fs];
    for (int e = e0; e < e1; ++e) {
      const int d = a.vd[e];
      long long dfs;
      const double* dp = mlt_ptr(a, a.dst[2 * d], a.dst[2 * d + 1], dfs);
      acc += a.inv[d] * dp[n * dfs];
    }
    a.tmp[(long long)n * a.nv + t] = acc;
  }
}

__global__ void __launch_bounds__(256) k_mlx_vjp_scatter(MltArgs a) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  long long fs;
  if (t < a.nv) {
    double* vp = mlt_ptr(a, a.v[2 * t], a.v[2 * t + 1], fs);
    for (int n = 0; n < a.nvar; ++n) vp[n * fs] = a.tmp[(long long)n * a.nv + t];
  } else if (t < a.nv + a.nz) {
    const int d = a.z[t - a.nv];
    double* dp = mlt_ptr(a, a.dst[2 * d], a.dst[2 * d + 1], fs);
    for (int n = 0; n < a.nvar; ++n) dp[n * fs] = 0.0;
  }
}

// R^T: the restriction injects the fine vertex coincident with each coarse
// interior vertex, so that fine vertex receives the coarse cotangent.
struct RestrictTArgs {
  const DevBlock* blocks;
  const RfBlock* cb;
  const RfChunk* chunks;
  int nvar;
  double* ubar;
  const double* cbar;
};

__global__ void __launch_bounds__(256) k_restrict_vjp(RestrictTArgs a) {
  const RfChunk ch = a.chunks[blockIdx.x];
  const RfBlock R = a.cb[ch.ent];
  const int t = ch.start + (int)threadIdx.x;
  if (t >= R.cni * R.cnj * R.cnk) return;
  const DevBlock& B = a.blocks[ch.ent];
  const int ci = RF_NCG + t % R.cni, cj = RF_NCG + (t / R.cni) % R.cnj,
            ck = RF_NCG + t / (R.cni * R.cnj);
  const int i = rf_fine_of(ci, RF_NCG, RF_NCG + R.cni - 1, B.il, B.iu);
  const int j = rf_fine_of(cj, RF_NCG, RF_NCG + R.cnj - 1, B.jl, B.ju);
  const int k = rf_fine_of(ck, RF_NCG, RF_NCG + R.cnk - 1, B.kl, B.ku);
  const long long p = i + (long long)B.nn1 * (j + (long long)B.nn2 * k);
  const long long cp = ci + (long long)R.cn1 * (cj + (long long)R.cn2 * ck);
  double* ub = a.ubar + B.off * a.nvar + p;
  const double* cb = a.cbar + R.coff * a.nvar + cp;
  for (int n = 0; n < a.nvar; ++n) ub[(long long)n * B.npts] += cb[(long long)n * R.cnpts];
}

// ---------------------------------------------------------------------------
// Z4c::Z4cWeyl (src/z4c/calculate_weyl_scalars.cpp:44-628): Re / Im psi4 at
// interior vertices, one thread per vertex, in the reference's operation
// order: physical metric derivatives by the chain rule from the prepared
// conformal derivatives (:136-262; the mixed second derivatives are Dx_a of
// the prepared d_b g~, the mixed d_a d_b chi Dx_a of the prepared d_b chi, as
// PrepareZ4cDerivatives forms them), Christoffels and Ricci of the physical
// metric (:264-347), K traces and D_a K_bc (:349-390), the coordinate tetrad
// orthonormalised with gamma (:392-512) and the Gauss / Codazzi projection
// onto it (:514-628).
// ---------------------------------------------------------------------------
struct WeylArgs {
  const DevBlock* blocks;
  Launch L;
  const double* u;
  const double* adm;
  const double* d1;  // prepared first derivatives (k_prep)
  double* out;       // 2 fields per block
  double chi_psi_power, chi_div_floor;
};

__global__ void __launch_bounds__(TILE) k_weyl(WeylArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  const int N = B.npts;
  const int p = flat(B, i, j, k);
  const Buf U = make_buf(a.u + B.off * NVAR, (long long)NVAR * N * 8);
  const Buf AD = make_buf(a.adm + B.off * NADM, (long long)NADM * N * 8);
  const Buf D1 = make_buf(a.d1 + B.off * ND1, (long long)ND1 * N * 8);
  const Pt P = make_pt(p, B.nn1, B.nn2, N);
  const double pw = a.chi_psi_power;
  const double FR4 = 0.25;
  const double chi_g = dmax(ldc(U, P, V_CHI), a.chi_div_floor);
  double dchi[3], ddc[6], gt[6];
#pragma unroll
  for (int c = 0; c < 3; ++c) dchi[c] = ldc(D1, P, c * 11 + F_CHI);
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) gt[ab] = ldc(U, P, V_GXX + ab);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    ddc[sym(c, c)] = fd_dxx(U, P, V_CHI, c, B.cidx2[c]);
#pragma unroll
    for (int d = c + 1; d < 3; ++d) ddc[sym(c, d)] = fd_dx(D1, P, d * 11 + F_CHI, c, B.cidx1[c]);
  }
  double dg[3][6], dK[3][6];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int ab = 0; ab < 6; ++ab) {
      const double dg3 = ldc(D1, P, c * 11 + F_G + ab);
      if (pw == -4.) {
        const double oochi = 1.0 / chi_g;
        dg[c][ab] = oochi * (dg3 - oochi * gt[ab] * dchi[c]);
      } else {
        const double fac = 4.0 / pw;
        const double psi4 = pow(chi_g, fac);
        const double oochi = 1.0 / chi_g;
        dg[c][ab] = psi4 * (dg3 + fac * oochi * gt[ab] * dchi[c]);
      }
      dK[c][ab] = fd_dx(AD, P, A_KXX + ab, c, B.cidx1[c]);
    }
  double ddg[6][6];  // [sym(a,b)][sym(c,d)] = d_a d_b gamma_cd
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int d = c; d < 3; ++d)
#pragma unroll
      for (int x = 0; x < 3; ++x)
#pragma unroll
        for (int y = x; y < 3; ++y) {
          const int cd = sym(c, d);
          const double gtil = gt[cd];
          const double dgx = ldc(D1, P, x * 11 + F_G + cd), dgy = ldc(D1, P, y * 11 + F_G + cd);
          double v;
          if (pw == -4.) {
            const double oochi = 1.0 / chi_g;
            if (x == y) {
              const double conf = fd_dxx(U, P, V_GXX + cd, x, B.cidx2[x]);
              v = oochi * (conf - oochi * (2.0 * dchi[x] * dgx + ddc[sym(x, x)] * gtil) +
                           2.0 * oochi * oochi * dchi[x] * dchi[x] * gtil);
            } else {
              const double conf = fd_dx(D1, P, y * 11 + F_G + cd, x, B.cidx1[x]);
              v = oochi * (conf - oochi * (dchi[x] * dgy + dchi[y] * dgx + ddc[sym(x, y)] * gtil) +
                           2.0 * oochi * oochi * dchi[x] * dchi[y] * gtil);
            }
          } else {
            const double fac = 4.0 / pw, fac2 = fac - 1.0;
            const double psi4 = pow(chi_g, fac);
            const double oochi = 1.0 / chi_g;
            if (x == y) {
              const double conf = fd_dxx(U, P, V_GXX + cd, x, B.cidx2[x]);
              v = psi4 * (conf + fac * oochi * (2.0 * dchi[x] * dgx + ddc[sym(x, x)] * gtil) +
                          fac * fac2 * oochi * oochi * dchi[x] * dchi[x] * gtil);
            } else {
              const double conf = fd_dx(D1, P, y * 11 + F_G + cd, x, B.cidx1[x]);
              v = psi4 * (conf +
                          fac * oochi * (dchi[x] * dgy + dchi[y] * dgx + ddc[sym(x, y)] * gtil) +
                          fac * fac2 * oochi * oochi * dchi[x] * dchi[y] * gtil);
            }
          }
          ddg[sym(x, y)][cd] = v;
        }
  double gd[6], Kd[6], gu[6];
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) {
    gd[ab] = ldc(AD, P, A_GXX + ab);
    Kd[ab] = ldc(AD, P, A_KXX + ab);
  }
  inv3(1. / det3(gd), gd, gu);
  double Gd[3][6], Gu[3][6];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int y = x; y < 3; ++y)
        Gd[c][sym(x, y)] = 0.5 * (dg[x][sym(y, c)] + dg[y][sym(x, c)] - dg[c][sym(x, y)]);
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int ab = 0; ab < 6; ++ab) {
      double t = 0.0;
#pragma unroll
      for (int d = 0; d < 3; ++d) t += gu[sym(c, d)] * Gd[d][ab];
      Gu[c][ab] = t;
    }
  double Rd[6], R = 0.0;
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = x; y < 3; ++y) {
      double r = 0.0;
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
#pragma unroll
          for (int e = 0; e < 3; ++e) {
            r += gu[sym(c, d)] * Gu[e][sym(x, c)] * Gd[e][sym(y, d)];
            r -= gu[sym(c, d)] * Gu[e][sym(x, y)] * Gd[e][sym(c, d)];
          }
          r += 0.5 * gu[sym(c, d)] *
               (-ddg[sym(c, d)][sym(x, y)] - ddg[sym(x, y)][sym(c, d)] +
                ddg[sym(x, c)][sym(y, d)] + ddg[sym(y, c)][sym(x, d)]);
        }
      Rd[sym(x, y)] = r;
      R += ((x == y) ? 1.0 : 2.0) * gu[sym(x, y)] * r;
    }
  double K = 0.0;
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    double t = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c) t += gu[sym(x, c)] * Kd[sym(c, x)];
    K += t;
  }
  double DK[3][6];  // the last write of each symmetric pair, as the reference's loop leaves it
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = 0; y < 3; ++y)
#pragma unroll
      for (int z = 0; z < 3; ++z) {
        double t = dK[x][sym(y, z)];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          t -= Gu[d][sym(x, y)] * Kd[sym(d, z)];
          t -= Gu[d][sym(x, z)] * Kd[sym(y, d)];
        }
        DK[x][sym(y, z)] = t;
      }
  // tetrad
  const double xc = B.x0[0] + i * B.dx[0], yc = B.x0[1] + j * B.dx[1], zc = B.x0[2] + k * B.dx[2];
  double xx = xc;
  if (xc * xc + yc * yc < 1e-10) xx = xx + 1e-8;
  double uv[3] = {xx, yc, zc}, vv[3] = {xx * zc, yc * zc, -(xx * xx) - yc * yc},
         wv[3] = {yc * -1.0, xx, 0.0};
  auto dot = [&](const double* q, const double* r) {
    double t = 0.0;
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int y = 0; y < 3; ++y) t += gd[sym(x, y)] * q[x] * r[y];
    return t;
  };
  {
    const double dp = dot(wv, wv);
#pragma unroll
    for (int x = 0; x < 3; ++x) wv[x] = wv[x] / sqrt(dp);
  }
  {
    const double dp = dot(wv, uv);
#pragma unroll
    for (int x = 0; x < 3; ++x) uv[x] -= dp * wv[x];
  }
  {
    const double dp = dot(uv, uv);
#pragma unroll
    for (int x = 0; x < 3; ++x) uv[x] = uv[x] / sqrt(dp);
  }
  {
    const double dp1 = dot(wv, vv), dp2 = dot(uv, vv);
#pragma unroll
    for (int x = 0; x < 3; ++x) vv[x] -= dp1 * wv[x] + dp2 * uv[x];
  }
  {
    const double dp = dot(vv, vv);
#pragma unroll
    for (int x = 0; x < 3; ++x) vv[x] = vv[x] / sqrt(dp);
  }
  double rp = 0.0, ip = 0.0;
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = 0; y < 3; ++y) {
      double R4 = Rd[sym(x, y)] + K * Kd[sym(x, y)];
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int d = 0; d < 3; ++d) R4 -= gu[sym(c, d)] * Kd[sym(x, c)] * Kd[sym(d, y)];
      const double Tr = vv[x] * vv[y] - wv[x] * wv[y];
      const double Ti = -vv[x] * wv[y] - wv[x] * vv[y];
      rp += -FR4 * R4 * Tr;
      ip += -FR4 * R4 * Ti;
    }
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = 0; y < 3; ++y)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double R4 = -(DK[y][sym(x, c)] - DK[c][sym(x, y)]);
        const double Tr = vv[x] * vv[y] - wv[x] * wv[y];
        const double Ti = -vv[x] * wv[y] - wv[x] * vv[y];
        rp += 0.5 * R4 * uv[c] * Tr;
        ip += 0.5 * R4 * uv[c] * Ti;
      }
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = 0; y < 3; ++y)
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const double R4 = gd[sym(d, c)] * Rd[sym(x, y)] + gd[sym(x, y)] * Rd[sym(d, c)] -
                            gd[sym(d, y)] * Rd[sym(x, c)] - gd[sym(x, c)] * Rd[sym(d, y)] -
                            0.5 * R * (gd[sym(d, c)] * gd[sym(x, y)] - gd[sym(d, y)] * gd[sym(x, c)]) +
                            Kd[sym(d, c)] * Kd[sym(x, y)] - Kd[sym(d, y)] * Kd[sym(x, c)];
          const double Tr = vv[x] * vv[y] - wv[x] * wv[y];
          const double Ti = -vv[x] * wv[y] - wv[x] * vv[y];
          rp += -FR4 * R4 * uv[d] * uv[c] * Tr;
          ip += -FR4 * R4 * uv[d] * uv[c] * Ti;
        }
  double* o = a.out + B.off * 2;
  o[p] = rp;
  o[N + p] = ip;
}

// ---------------------------------------------------------------------------
// Adjoint of the right-hand side (no counterpart in the reference, which has
// no derivative code): linearisation, pointwise reverse mode, transposed
// stencils, parameter-gradient reduction.  Cotangent c of nw is blockIdx.y
// (times NVAR fields in the stencil kernel).
// ---------------------------------------------------------------------------
struct AdjArgs {
  const DevBlock* blocks;
  Launch L;
  RhsParams o;
  const double* u;   // state the right-hand side is linearised at
  double* lin;       // NLINF per interior vertex
  const double* w;   // nw cotangent registers (NVAR * total_pts each)
  double* ubar;      // nw output registers
  double* sb;        // nw derivative-cotangent sets (NADJ * total_int each)
  double* part;      // nw * gridDim.x * NPBAR workgroup partial sums
  long long reg;     // NVAR * total_pts
  long long sreg;    // NADJ * total_int
  int hseed;         // 1: seed = d/du of sum vol Ht^2 (w unused, may be null)
  double* carry;     // nw sets of NCARRY + 18 values per interior vertex
  long long creg;    // (NCARRY + 18) * total_int
};

// Two waves a SIMD, no spill (336 registers and one wave unbounded): 0.74 ->
// 0.56 ms for 320 blocks of 16^3.
__global__ void __launch_bounds__(TILE) __attribute__((amdgpu_waves_per_eu(2)))
k_adj_fwd(AdjArgs a) {
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  adj_lin_fwd_at(a.o, B, a.u + B.off * NVAR, a.lin + B.ioff * NLINF, i, j, k);
}

// Buffer accessors of the pointwise adjoint: one 32-bit lane offset per
// buffer, the slot / field offsets uniform (SGPR), so the hundreds of slot
// addresses cost no vector registers.
struct AdjXBuf {
  Buf U, L;
  unsigned vp, vq;  // p*8, q*8
  int fu, fl;       // npts*8, nint*8
  __device__ double u(int n) const { return bload(U, vp, n * fu); }
  __device__ double d1(int n, int a) const { return bload(L, vq, l_d1(n, a) * fl); }
  __device__ double d2(int n, int ab) const { return bload(L, vq, l_d2(n, ab) * fl); }
  __device__ double ls(int n, int a) const { return bload(L, vq, l_ls(n, a) * fl); }
};
struct AdjFBuf {
  Buf L;
  unsigned vq;
  int fl;
  __device__ double operator()(int s) const { return bload(L, vq, (NLIN + s) * fl); }
};
struct AdjSBuf {
  Buf S;
  unsigned vq;
  int fl;
  __device__ void d1(int n, int a, double v) const { bstore(S, v, vq, l_d1(n, a) * fl); }
  __device__ void d2(int n, int ab, double v) const { bstore(S, v, vq, l_d2(n, ab) * fl); }
};

// The pointwise adjoint in two kernels (the reverse sweep split before the
// Ricci adjoint, each phase with its own register budget).  Phase a: the
// cotangent w, every term down to D_aD_b alpha, the parameter partials
// (one sum per workgroup), the Gudd adjoints in registers; it stores the
// accumulators live across the split and the Gudd adjoints, slot-major.
constexpr int NCARRY_ALL = NCARRY + 18;

__global__ void __launch_bounds__(TILE) k_adj_point_a(AdjArgs a) {
  __shared__ double red[NPBAR][TILE / 64];
  const long long c = blockIdx.y;
  double pb[NPBAR] = {0.0, 0.0, 0.0};
  int b, i, j, k;
  if (tile_point(a.L, b, i, j, k)) {
    const DevBlock B = a.blocks[b];
    const long long N = B.npts, nint = B.nint;
    const unsigned vp = (unsigned)flat(B, i, j, k) * 8u, vq = (unsigned)iidx(B, i, j, k) * 8u;
    const AdjXBuf X{make_buf(a.u + B.off * NVAR, NVAR * N * 8),
                    make_buf(a.lin + B.ioff * NLINF, NLINF * nint * 8), vp, vq, (int)(N * 8),
                    (int)(nint * 8)};
    const AdjFBuf F{X.L, vq, (int)(nint * 8)};
    const AdjSBuf S{make_buf(a.sb + c * a.sreg + B.ioff * NADJ, NADJ * nint * 8), vq,
                    (int)(nint * 8)};
    double wp[NVAR];
    double wH = 0.0;
    if (a.hseed) {
#pragma unroll
      for (int n = 0; n < NVAR; ++n) wp[n] = 0.0;
      if (in_cell_loop(B, i, j, k))
        wH = 2.0 * (B.dx[0] * B.dx[1] * B.dx[2]) *
             ham_from_fwd(F(F_R), F(F_TRAA), X.u(V_KHAT), X.u(V_THETA));
    } else {
      const Buf W = make_buf(a.w + c * a.reg + B.off * NVAR, NVAR * N * 8);
#pragma unroll
      for (int n = 0; n < NVAR; ++n) wp[n] = bload(W, vp, n * X.fu);
    }
    const Buf UB = make_buf(a.ubar + c * a.reg + B.off * NVAR, NVAR * N * 8);
    const int fu = X.fu;
    double bG[42];
    AdjCarry cy;
    rhs_vjp_point_a(a.o, X, F, wp, [&](int n, double v) { bstore(UB, v, vp, n * fu); }, S, pb, bG,
                    1, wH, cy);
    const Buf CB = make_buf(a.carry + c * a.creg + B.ioff * NCARRY_ALL, NCARRY_ALL * nint * 8);
    const int fs = (int)(nint * 8);
#pragma unroll
    for (int e = 0; e < NCARRY; ++e) bstore(CB, carry_at(cy, e), vq, e * fs);
#pragma unroll
    for (int e = 0; e < 18; ++e) bstore(CB, bG[e], vq, (NCARRY + e) * fs);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int t = 0; t < NPBAR; ++t) {
    double v = pb[t];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if (lane == 0) red[t][wave] = v;
  }
  __syncthreads();
  if (threadIdx.x < NPBAR) {
    double v = 0.0;
    for (int q = 0; q < TILE / 64; ++q) v += red[threadIdx.x][q];
    a.part[(c * gridDim.x + blockIdx.x) * NPBAR + threadIdx.x] = v;
  }
}

// Phase b: the Ricci adjoint onward, the Christoffel adjoints in a per-thread
// LDS column (42 doubles) seeded from phase a.
__global__ void __launch_bounds__(TILE) k_adj_point_b(AdjArgs a) {
  __shared__ double shG[42 * TILE];
  const long long c = blockIdx.y;
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  const long long N = B.npts, nint = B.nint;
  const unsigned vp = (unsigned)flat(B, i, j, k) * 8u, vq = (unsigned)iidx(B, i, j, k) * 8u;
  const AdjXBuf X{make_buf(a.u + B.off * NVAR, NVAR * N * 8),
                  make_buf(a.lin + B.ioff * NLINF, NLINF * nint * 8), vp, vq, (int)(N * 8),
                  (int)(nint * 8)};
  const AdjFBuf F{X.L, vq, (int)(nint * 8)};
  const AdjSBuf S{make_buf(a.sb + c * a.sreg + B.ioff * NADJ, NADJ * nint * 8), vq,
                  (int)(nint * 8)};
  const Buf CB = make_buf(a.carry + c * a.creg + B.ioff * NCARRY_ALL, NCARRY_ALL * nint * 8);
  const int fs = (int)(nint * 8);
  AdjCarry cy;
#pragma unroll
  for (int e = 0; e < NCARRY; ++e) carry_at(cy, e) = bload(CB, vq, e * fs);
  double* bG = shG + threadIdx.x;
#pragma unroll
  for (int e = 0; e < 18; ++e) bG[e * TILE] = bload(CB, vq, (NCARRY + e) * fs);
#pragma unroll
  for (int e = 18; e < 42; ++e) bG[e * TILE] = 0.0;
  const Buf UB = make_buf(a.ubar + c * a.reg + B.off * NVAR, NVAR * N * 8);
  const int fu = X.fu;
  rhs_vjp_point_b(a.o, X, F, [&](int n, double v) { bstore(UB, v, vp, n * fu); }, S, bG, TILE, cy);
}

// blockIdx.y = 2 c + h: cotangent c, fields [0, 7) (h = 0: chi and g~, the
// second-derivative-heavy half) or [7, 22) (h = 1)
__global__ void __launch_bounds__(TILE) k_adj_stencil(AdjArgs a) {
  const long long c = blockIdx.y >> 1;
  const int half = blockIdx.y & 1;
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  const long long N = B.npts, nint = B.nint;
  const int fu = (int)(N * 8), fs = (int)(nint * 8);
  const Buf SB = make_buf(a.sb + c * a.sreg + B.ioff * NADJ, NADJ * nint * 8);
  const Buf UB = make_buf(a.u + B.off * NVAR, NVAR * N * 8);
  const Buf WB = make_buf(a.hseed ? a.u : a.w + c * a.reg + B.off * NVAR, NVAR * N * 8);
  const Buf OB = make_buf(a.ubar + c * a.reg + B.off * NVAR, NVAR * N * 8);
  auto S = [&](int slot, int q) { return bload(SB, (unsigned)q * 8u, slot * fs); };
  auto W = [&](int n, int p) { return bload(WB, (unsigned)p * 8u, n * fu); };
  auto Bx = [&](int d, int p) { return bload(UB, (unsigned)p * 8u, (V_BETAX + d) * fu); };
  const unsigned vp = (unsigned)flat(B, i, j, k) * 8u;
  const bool interior = is_interior(B, i, j, k);
  auto out = [&](int n, double v) {
    const double pt = interior ? bload(OB, vp, n * fu) : 0.0;
    bstore(OB, pt + v, vp, n * fu);
  };
  if (half == 0)
    adj_stencil_at<0, 7>(a.o, B, S, a.hseed ? nullptr : &W, Bx, i, j, k, out);
  else
    adj_stencil_at<7, NVAR>(a.o, B, S, a.hseed ? nullptr : &W, Bx, i, j, k, out);
}

// pbar[c*NPBAR + t] (+)= sum of the partials of cotangent c: one workgroup
// per (c, t), strided partial sums then a fixed-order tree (deterministic)
__global__ void __launch_bounds__(256) k_adj_pbar(const double* part, int G, int nw, double* pbar,
                                                  int accumulate) {
  __shared__ double red[256];
  const int e = blockIdx.x;
  const int c = e / NPBAR, t = e % NPBAR;
  double v = 0.0;
  for (int g = threadIdx.x; g < G; g += 256) v += part[((long long)c * G + g) * NPBAR + t];
  red[threadIdx.x] = v;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) pbar[e] = accumulate ? pbar[e] + red[0] : red[0];
}

// Partial sums of vol * Ht^2 over the cell loop, one per workgroup
__global__ void __launch_bounds__(TILE) k_hnorm(AdjArgs a) {
  __shared__ double red[TILE / 64];
  double v = 0.0;
  int b, i, j, k;
  if (tile_point(a.L, b, i, j, k)) {
    const DevBlock B = a.blocks[b];
    if (in_cell_loop(B, i, j, k)) {
      const long long N = B.npts, nint = B.nint;
      const double* un = a.u + B.off * NVAR + flat(B, i, j, k);
      const double* fw = a.lin + B.ioff * NLINF + (long long)NLIN * nint + iidx(B, i, j, k);
      const double H = ham_from_fwd(fw[F_R * nint], fw[F_TRAA * nint], un[V_KHAT * N],
                                    un[V_THETA * N]);
      v = (B.dx[0] * B.dx[1] * B.dx[2]) * (H * H);
    }
  }
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int q = 0; q < TILE / 64; ++q) t += red[q];
    a.part[blockIdx.x] = t;
  }
}

// ---------------------------------------------------------------------------
// Adjoint of one bt_rk4 step with ghosts held at u_n and AlgConstr after
// every stage (the fused step's semantics):
//   u_1 = u_n, u_s = AlgConstr(u_n + a_s dt k_{s-1}) (s = 2..4),
//   k_s = rhs(u_s), u_{n+1} = AlgConstr(u_n + dt sum_s b_s k_s),
// with k_s = 0 at ghosts (so ghosts of u_s and u_{n+1} are AlgConstr(u_n)).
// ---------------------------------------------------------------------------
struct AdjStepArgs {
  const DevBlock* blocks;
  Launch L;              // BOX_WHOLE
  const double* un;      // u_n
  const double* k[4];    // stage right-hand sides (zero at ghosts)
  const double* bar;     // final: cotangent of u_{n+1}; stage: cotangent of u_s
  double* ubar_in;       // cotangent of u_n (accumulated)
  double* ybar;          // AlgConstr cotangent at the final sum (interior)
  double* kbar;          // cotangent of k_{s-1} (interior), the next stage's w
  long long reg;
  double dt;
  int stage;             // 5 = final sum, 4..1 = stage input u_s
  double eps_floor;
  int tf_force, force_reg;
  // exchange mode (k_adj_step_ex): the stage cotangent, transformed in
  // place, and AlgConstr's input E(y_s)
  double* ybar_stage;
  const double* pre;
};

// un and the stage registers a.k[] share the state layout: both are read at
// the block's offset boff = B.off * NVAR
__device__ __forceinline__ void adj_alg_point(const AdjStepArgs& a, long long boff, long long p,
                                              long long N, bool interior, double wk, int kreg,
                                              double* bar) {
  const double* un = a.un + boff;
  double g[6], A[6], bg[6], bA[6];
  double chi = un[V_CHI * N + p], alpha = un[V_ALPHA * N + p];
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) {
    g[ab] = un[(V_GXX + ab) * N + p];
    A[ab] = un[(V_AXX + ab) * N + p];
  }
  if (interior) {
    // the forward state entering AlgConstr: u_n + w k (one register) or the
    // final sum ((u_n + b1 dt k1) + b2 dt k2 + b3 dt k3) + b4 dt k4
    if (kreg >= 0) {
      const double* kk = a.k[kreg] + boff;
      chi = chi + wk * kk[V_CHI * N + p];
      alpha = alpha + wk * kk[V_ALPHA * N + p];
#pragma unroll
      for (int ab = 0; ab < 6; ++ab) {
        g[ab] = g[ab] + wk * kk[(V_GXX + ab) * N + p];
        A[ab] = A[ab] + wk * kk[(V_AXX + ab) * N + p];
      }
    } else {
      const double bw[4] = {1. / 6., 1. / 3., 1. / 3., 1. / 6.};
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const double ws = bw[s] * a.dt;
        const double* kk = a.k[s] + boff;
        chi = chi + ws * kk[V_CHI * N + p];
        alpha = alpha + ws * kk[V_ALPHA * N + p];
#pragma unroll
        for (int ab = 0; ab < 6; ++ab) {
          g[ab] = g[ab] + ws * kk[(V_GXX + ab) * N + p];
          A[ab] = A[ab] + ws * kk[(V_AXX + ab) * N + p];
        }
      }
    }
  }
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) {
    bg[ab] = bar[V_GXX + ab];
    bA[ab] = bar[V_AXX + ab];
  }
  algconstr_vjp(g, A, chi, alpha, bg, bA, bar[V_CHI], bar[V_ALPHA], a.eps_floor, a.tf_force,
                a.force_reg);
#pragma unroll
  for (int ab = 0; ab < 6; ++ab) {
    bar[V_GXX + ab] = bg[ab];
    bar[V_AXX + ab] = bA[ab];
  }
}

__global__ void __launch_bounds__(TILE) k_adj_step(AdjStepArgs a) {
  const long long c = blockIdx.y;
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  const long long N = B.npts, p = flat(B, i, j, k);
  const bool interior = is_interior(B, i, j, k);
  const long long boff = B.off * NVAR;
  const long long cb = c * a.reg + boff;
  double bar[NVAR];
#pragma unroll
  for (int n = 0; n < NVAR; ++n) bar[n] = a.bar[cb + n * N + p];
  const double bw[4] = {1. / 6., 1. / 3., 1. / 3., 1. / 6.};
  const double aw[5] = {0., 0., 0.5, 0.5, 1.0};  // a_s of stage s
  if (a.stage == 5) {
    adj_alg_point(a, boff, p, N, interior, 0.0, -1, bar);
#pragma unroll
    for (int n = 0; n < NVAR; ++n) {
      a.ubar_in[cb + n * N + p] = bar[n];
      if (interior) {
        a.ybar[cb + n * N + p] = bar[n];
        a.kbar[cb + n * N + p] = (bw[3] * a.dt) * bar[n];
      }
    }
    return;
  }
  const int s = a.stage;
  if (s >= 2) adj_alg_point(a, boff, p, N, interior, aw[s] * a.dt, s - 2, bar);
#pragma unroll
  for (int n = 0; n < NVAR; ++n) {
    a.ubar_in[cb + n * N + p] += bar[n];
    if (s >= 2 && interior)
      a.kbar[cb + n * N + p] = (bw[s - 2] * a.dt) * a.ybar[cb + n * N + p] + (aw[s] * a.dt) * bar[n];
  }
}

// The step adjoint with the ghost update after every stage (exchange mode):
// u_s = AlgConstr(E(y_s)) with y_s the stage's sum and E the exchange, so
// the stage cotangent goes through AlgConstr's adjoint at E(y_s) (PHASE 1,
// in place; E(y_s) kept by the forward sweep in a.pre), then through E's
// transpose (launch_exchange_vjp), then splits into the cotangents of u_n
// and of the k's (PHASE 2), as k_adj_step does.
template <int PHASE>
__global__ void __launch_bounds__(TILE) k_adj_step_ex(AdjStepArgs a) {
  const long long c = blockIdx.y;
  int b, i, j, k;
  if (!tile_point(a.L, b, i, j, k)) return;
  const DevBlock B = a.blocks[b];
  const long long N = B.npts, p = flat(B, i, j, k);
  const bool interior = is_interior(B, i, j, k);
  const long long boff = B.off * NVAR;
  const long long cb = c * a.reg + boff;
  double* bar = a.ybar_stage + cb;
  if (PHASE == 1) {
    const double* y = a.pre + boff;
    double g[6], A[6], bg[6], bA[6];
#pragma unroll
    for (int ab = 0; ab < 6; ++ab) {
      g[ab] = y[(V_GXX + ab) * N + p];
      A[ab] = y[(V_AXX + ab) * N + p];
      bg[ab] = bar[(V_GXX + ab) * N + p];
      bA[ab] = bar[(V_AXX + ab) * N + p];
    }
    double bchi = bar[V_CHI * N + p], balpha = bar[V_ALPHA * N + p];
    algconstr_vjp(g, A, y[V_CHI * N + p], y[V_ALPHA * N + p], bg, bA, bchi, balpha, a.eps_floor,
                  a.tf_force, a.force_reg);
#pragma unroll
    for (int ab = 0; ab < 6; ++ab) {
      bar[(V_GXX + ab) * N + p] = bg[ab];
      bar[(V_AXX + ab) * N + p] = bA[ab];
    }
    bar[V_CHI * N + p] = bchi;
    bar[V_ALPHA * N + p] = balpha;
    return;
  }
  const double bw[4] = {1. / 6., 1. / 3., 1. / 3., 1. / 6.};
  const double aw[5] = {0., 0., 0.5, 0.5, 1.0};  // a_s of stage s
  const int s = a.stage;
#pragma unroll
  for (int n = 0; n < NVAR; ++n) {
    const double v = bar[n * N + p];
    if (s == 5) {
      a.ubar_in[cb + n * N + p] = v;
      if (interior) {
        a.ybar[cb + n * N + p] = v;
        a.kbar[cb + n * N + p] = (bw[3] * a.dt) * v;
      }
    } else {
      a.ubar_in[cb + n * N + p] += v;
      if (s >= 2 && interior)
        a.kbar[cb + n * N + p] = (bw[s - 2] * a.dt) * a.ybar[cb + n * N + p] + (aw[s] * a.dt) * v;
    }
  }
}
}  // namespace

// ===========================================================================
// Context
// ===========================================================================
struct z4c_ctx {
  int device = 0;
  int nblocks = 0;
  long long total_pts = 0;
  std::vector<z4c_block> hblocks;
  DevBlock* d_blocks = nullptr;
  Tile* d_tiles[NBOX] = {};
  Box* d_boxes[NBOX] = {};
  int ntiles[NBOX] = {};
  double* d1 = nullptr;     // prepared first derivatives (PrepareZ4cDerivatives)
  double* dv = nullptr;     // derivative slots of the RHS stencil pass
  // stencil plan: the workgroup configuration of every block, and per
  // configuration the plane tiles of its blocks
  std::vector<int> blk_cfg;
  std::vector<DevBlock> hdev;  // host copy of the device block table
  PlaneTile* st_tiles[NSTCFG] = {};
  PlaneTile* lin_tiles = nullptr;  // 256-thread tiles of every block (the adjoint's linearisation)
  int lin_ntiles = 0;
  int st_ntiles[NSTCFG] = {};
  long long total_int = 0;  // interior points
  long long total_dv = 0;   // doubles of the derivative slots (dv, allocated on first use)
  FusedTile* fu_tiles = nullptr;  // bricks of the one-kernel right-hand side
  int fu_ntiles = 0;
  double t_one = 0, t_two = 0;  // estimated right-hand side in one kernel, in two passes (us)
  int form = Z4C_FORM_AUTO; // z4c_set_rhs_form
  bool faces = false;       // some block has a Sommerfeld face
  bool per_snap = false;    // the periodic fill reads a snapshot (a block under 4 cells)
  double* snap = nullptr;  // periodic-fill snapshot / exchange scratch (lazy)
  long long snap_elems = 0;
  double* hst = nullptr;   // history partial sums (lazy)
  PhysLine* ph_lines[3] = {};  // physical-fill line tables per axis
  int ph_nent[3] = {};
  long long ph_nlines1[3] = {};  // lines per field
  int* ex_dst = nullptr;   // exchange map (z4c_set_exchange)
  int* ex_off = nullptr;
  int* ex_src = nullptr;
  int ex_ndst = 0;
  // its transpose (z4c_exchange_vjp): the source vertices (2 ints each),
  // whether each is itself a destination, CSR of the destinations that read
  // it, the destinations that are no source (ghosts), and a scratch of
  // NVAR values per source vertex
  int* ext_v = nullptr;
  int* ext_flag = nullptr;
  int* ext_off = nullptr;
  int* ext_d = nullptr;
  int* ext_z = nullptr;
  int ext_nv = 0, ext_nz = 0;
  double* ext_tmp = nullptr;
  void drop_ext() {
    int** q[5] = {&ext_v, &ext_flag, &ext_off, &ext_d, &ext_z};
    for (int** x : q) {
      hipFree(*x);
      *x = nullptr;
    }
    hipFree(ext_tmp);
    ext_tmp = nullptr;
    ext_nv = ext_nz = 0;
  }
  // ghost update across refinement levels (z4c_set_exchange on blocks of
  // several spacings): gather lists, the context's coarse buffers, the
  // gathered values, and the prolongation entries of the coarser neighbours
  bool ml = false;
  int* ml_dst = nullptr;        // 2 ints per destination: 2*block + array, point
  long long* ml_off = nullptr;  // CSR offsets into ml_src
  int* ml_src = nullptr;        // 2 ints per source
  double* ml_inv = nullptr;     // 1/multiplicity per destination
  int ml_ndst = 0;
  int ml_nint = 0;              // interior destinations (listed first)
  double* ml_coarse = nullptr;  // NVAR fields of every block's coarse buffer
  double* ml_tmp = nullptr;     // NVAR * ml_ndst
  RfEntry* ml_pent = nullptr;
  PrGroup* ml_pgroups = nullptr;
  int ml_npgroups = 0;
  int ml_prlds = 0;             // largest staged coarse box, doubles
  int ml_nent = 0;              // prolongation entries (ml_pent)
  PhysLine* mlp_lines[3] = {};  // the coarse level's physical fill, per axis
  int mlp_nent[3] = {};
  long long mlp_nlines1[3] = {};
  std::vector<std::vector<z4c_mesh::Nbr>> ml_nbrs;  // per block, for inspection
  std::vector<int> ml_level;

  // transpose of the update across levels (built on its first use)
  bool mlt_built = false;
  int* mlt_v = nullptr;      // source references (2 ints each)
  int* mlt_flag = nullptr;   // 1 if the source is also a destination
  int* mlt_off = nullptr;    // CSR offsets into mlt_d
  int* mlt_d = nullptr;      // destinations reading each source
  int* mlt_z = nullptr;      // destinations that are no source
  int mlt_nv = 0, mlt_nz = 0;
  double* mlt_tmp = nullptr;            // NVAR * mlt_nv
  unsigned char* ml_fmask = nullptr;    // fine vertices the prolongation writes (per point)
  int* ml_fl = nullptr;                 // those vertices (block, point)
  int ml_nfl = 0;
  PrTTile* ml_ptiles = nullptr;         // tiles of the prolongation's transpose
  int ml_nptiles = 0;
  int ml_ptlds = 0;                     // LDS doubles of the largest tile
  double* ml_cbar = nullptr;            // coarse cotangents, NVAR * rf_total
  void drop_mlt() {
    int** q[6] = {&mlt_v, &mlt_flag, &mlt_off, &mlt_d, &mlt_z, &ml_fl};
    for (int** x : q) {
      hipFree(*x);
      *x = nullptr;
    }
    hipFree(mlt_tmp);
    hipFree(ml_fmask);
    hipFree(ml_cbar);
    hipFree(ml_ptiles);
    mlt_tmp = nullptr;
    ml_fmask = nullptr;
    ml_cbar = nullptr;
    ml_ptiles = nullptr;
    mlt_nv = mlt_nz = ml_nfl = ml_nptiles = ml_ptlds = 0;
    mlt_built = false;
  }
  void drop_ml() {
    if (graph_exec) hipGraphExecDestroy(graph_exec);
    graph_exec = nullptr;
    hipFree(ml_dst);
    hipFree(ml_off);
    hipFree(ml_src);
    hipFree(ml_inv);
    hipFree(ml_coarse);
    hipFree(ml_tmp);
    hipFree(ml_pent);
    hipFree(ml_pgroups);
    for (int ax = 0; ax < 3; ++ax) {
      hipFree(mlp_lines[ax]);
      mlp_lines[ax] = nullptr;
      mlp_nent[ax] = 0;
      mlp_nlines1[ax] = 0;
    }
    ml_dst = ml_src = nullptr;
    ml_off = nullptr;
    ml_inv = ml_coarse = ml_tmp = nullptr;
    ml_pent = nullptr;
    ml_pgroups = nullptr;
    ml_ndst = ml_nint = ml_npgroups = ml_prlds = ml_nent = 0;
    drop_mlt();
    ml = false;
    ml_nbrs.clear();
    ml_level.clear();
  }
  // refinement (lazy): coarse-buffer table and restriction chunks, and the
  // prolongation entries set by z4c_set_prolongation with their groups
  std::vector<RfBlock> hrf;
  long long rf_total = 0;
  RfBlock* d_rf = nullptr;
  RfChunk* d_rchunks = nullptr;
  int n_rchunks = 0;
  RfEntry* d_pent = nullptr;
  PrGroup* d_pgroups = nullptr;
  int n_pgroups = 0;
  int pr_lds = 0;
  std::vector<double> hst_host;
  int n_cu = 256;
  // captured fused step (z4c_rk4_step_graph) and what it was captured for
  hipStream_t cap_stream = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  const double* g_u = nullptr;
  const double* g_work = nullptr;
  double g_dt = 0.0;
  int g_ghosts = 0;
  z4c_params g_params{};
  // per-pass kernel timing (events recorded on the launch stream)
  struct TimedLaunch {
    int pass;
    hipEvent_t a, b;
    double part;  // share of the launch's time that counts for the pass
  };
  bool timing = false;
  std::vector<TimedLaunch> tev;
  // adjoint scratch (lazy): linearisation, derivative cotangents, partial
  // sums, the step's stage right-hand sides and stage state, and three
  // per-cotangent registers (ybar, kbar, stage cotangent)
  double* adj_lin = nullptr;
  double* adj_sb = nullptr;
  double* adj_part = nullptr;
  double* adj_carry = nullptr;  // the pointwise adjoint's values between its two kernels
  long long adj_carry_n = 0;
  double* adj_k = nullptr;
  double* adj_stage = nullptr;
  double* adj_reg = nullptr;
  double* adj_pre = nullptr;  // step VJP with the exchange: the exchanged sums entering AlgConstr
  long long adj_pre_n = 0;
  bool adj_k_zero = false;  // adj_k's ghosts hold zeros (set by the first step VJP)
  long long adj_lin_n = 0, adj_sb_n = 0, adj_part_n = 0, adj_k_n = 0, adj_stage_n = 0,
            adj_reg_n = 0;

  void drop_timing() {
    for (auto& t : tev) {
      hipEventDestroy(t.a);
      hipEventDestroy(t.b);
    }
    tev.clear();
  }

  void drop_prolongation() {
    hipFree(d_pent);
    hipFree(d_pgroups);
    d_pent = nullptr;
    d_pgroups = nullptr;
    n_pgroups = pr_lds = 0;
  }

  void drop_refine() {
    drop_prolongation();
    hipFree(d_rf);
    hipFree(d_rchunks);
    d_rf = nullptr;
    d_rchunks = nullptr;
    n_rchunks = 0;
    hrf.clear();
    rf_total = 0;
  }

  // the captured step holds device pointers of the block table and plans
  void invalidate_graph() {
    if (graph_exec) hipGraphExecDestroy(graph_exec);
    graph_exec = nullptr;
  }

  void release() {
    invalidate_graph();
    hipFree(d_blocks);
    for (int b = 0; b < NBOX; ++b) {
      hipFree(d_tiles[b]);
      hipFree(d_boxes[b]);
      d_tiles[b] = nullptr;
      d_boxes[b] = nullptr;
      ntiles[b] = 0;
    }
    hipFree(d1);
    hipFree(dv);
    for (int q = 0; q < NSTCFG; ++q) {
      hipFree(st_tiles[q]);
      st_tiles[q] = nullptr;
      st_ntiles[q] = 0;
    }
    hipFree(lin_tiles);
    lin_tiles = nullptr;
    lin_ntiles = 0;
    hipFree(fu_tiles);
    fu_tiles = nullptr;
    fu_ntiles = 0;
    t_one = t_two = 0;
    faces = false;
    form = Z4C_FORM_AUTO;
    hipFree(snap);
    hipFree(hst);
    hst = nullptr;
    for (int q = 0; q < 3; ++q) {
      hipFree(ph_lines[q]);
      ph_lines[q] = nullptr;
      ph_nent[q] = 0;
      ph_nlines1[q] = 0;
    }
    hipFree(ex_dst);
    hipFree(ex_off);
    hipFree(ex_src);
    ex_dst = ex_off = ex_src = nullptr;
    ex_ndst = 0;
    drop_ext();
    drop_ml();
    drop_refine();
    hst_host.clear();
    double** adj[6] = {&adj_lin, &adj_sb, &adj_part, &adj_k, &adj_stage, &adj_reg};
    for (double** q : adj) {
      hipFree(*q);
      *q = nullptr;
    }
    adj_lin_n = adj_sb_n = adj_part_n = adj_k_n = adj_stage_n = adj_reg_n = 0;
    hipFree(adj_carry);
    adj_carry = nullptr;
    adj_carry_n = 0;
    hipFree(adj_pre);
    adj_pre = nullptr;
    adj_pre_n = 0;
    adj_k_zero = false;
    d_blocks = nullptr;
    d1 = nullptr;
    dv = nullptr;
    blk_cfg.clear();
    snap = nullptr;
    snap_elems = 0;
  }
};

namespace {

// Brackets the launches of one pass with events when timing is on.
struct PassTimer {
  z4c_ctx* c;
  int pass;
  hipStream_t s;
  hipEvent_t a = nullptr;
  double part;
  PassTimer(z4c_ctx* c_, int pass_, hipStream_t s_, double part_ = 1.0)
      : c(c_), pass(pass_), s(s_), part(part_) {
    if (c->timing && hipEventCreate(&a) == hipSuccess) hipEventRecord(a, s);
  }
  ~PassTimer() {
    if (!a) return;
    hipEvent_t b = nullptr;
    if (hipEventCreate(&b) != hipSuccess) {
      hipEventDestroy(a);
      return;
    }
    hipEventRecord(b, s);
    c->tev.push_back({pass, a, b, part});
  }
};

int grid_for(int ntiles) { return std::max(8, (ntiles + 7) / 8 * 8); }

Launch launch_of(const z4c_ctx* c, int kind) {
  return Launch{c->d_tiles[kind], c->d_boxes[kind], c->ntiles[kind]};
}

int check_ctx(const z4c_ctx* c) {
  if (!c) return fail(Z4C_EINVAL, "null context");
  if (c->nblocks <= 0) return fail(Z4C_ESTATE, "no blocks registered (call z4c_set_blocks)");
  return Z4C_OK;
}

RhsParams rhs_params(const z4c_params* p) {
  RhsParams o;
  o.chi_psi_power = p->chi_psi_power;
  o.chi_div_floor = p->chi_div_floor;
  o.diss = p->diss;
  o.damp_kappa1 = p->damp_kappa1;
  o.damp_kappa2 = p->damp_kappa2;
  o.lapse_oplog = p->lapse_oplog;
  o.lapse_harmonicf = p->lapse_harmonicf;
  o.lapse_harmonic = p->lapse_harmonic;
  o.lapse_advect = p->lapse_advect;
  o.lapse_K = p->lapse_K;
  o.shift_Gamma = p->shift_Gamma;
  o.shift_alpha2Gamma = p->shift_alpha2Gamma;
  o.shift_H = p->shift_H;
  o.shift_advect = p->shift_advect;
  o.shift_eta = p->shift_eta;
  return o;
}

int elementwise_grid(long long n) {
  long long g = (n + 255) / 256;
  return (int)std::min<long long>(g, 256LL * 64);
}

int fill(z4c_ctx* c, double* p, double v, long long n, hipStream_t s) {
  hipLaunchKernelGGL(k_fill, dim3(elementwise_grid(n)), dim3(256), 0, s, p, v, n);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

int launch_prep(z4c_ctx* c, const z4c_params* p, const double* u, double* aux,
                hipStream_t s) {
  PrepArgs a{c->d_blocks, launch_of(c, BOX_PREP), u, c->d1, aux, p->chi_psi_power,
             p->chi_div_floor};
  PassTimer t(c, Z4C_PASS_PREPARE, s);
  hipLaunchKernelGGL(k_prep, dim3(grid_for(a.L.ntiles)), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

// ---------------------------------------------------------------------------
// Stencil-pass plan
// ---------------------------------------------------------------------------
constexpr int ST_THREADS_OF[NSTCFG] = {StCfg256::THREADS, StCfg320::THREADS,
                                       StCfg192::THREADS, StCfg384::THREADS,
                                       StCfg640::THREADS, StCfg576::THREADS};

bool cfg_fits(int cfg, int ni, int nj) {
  switch (cfg) {
    case 0: return StCfg256::fits(ni, nj);
    case 1: return StCfg320::fits(ni, nj);
    case 2: return StCfg192::fits(ni, nj);
    case 3: return StCfg384::fits(ni, nj);
    case 4: return StCfg640::fits(ni, nj);
    default: return StCfg576::fits(ni, nj);
  }
}

// The fewest x-y tiles of an ni x nj plane that fit configuration `cfg`,
// preferring the widest x extent (coalescing); false if none fits.
bool plane_tiles(int cfg, int b, int ni, int nj, std::vector<PlaneTile>* out) {
  int best_tx = 0, best_ty = 0, best_n = 0;
  for (int ntx = 1; ntx <= ni; ++ntx) {
    const int tx = (ni + ntx - 1) / ntx;
    int nty = 1, ty = nj;
    while (nty <= nj && !cfg_fits(cfg, tx, ty)) {
      ++nty;
      ty = (nj + nty - 1) / nty;
    }
    if (!cfg_fits(cfg, tx, ty)) continue;
    if (best_n == 0 || ntx * nty < best_n) {
      best_n = ntx * nty;
      best_tx = tx;
      best_ty = ty;
    }
  }
  if (best_n == 0) return false;
  if (out)
    for (int j0 = 0; j0 < nj; j0 += best_ty)
      for (int i0 = 0; i0 < ni; i0 += best_tx)
        out->push_back(PlaneTile{b, i0, j0, std::min(best_tx, ni - i0), std::min(best_ty, nj - j0)});
  return true;
}

// Thread slots (tiles x threads) of a block under `cfg`, or -1.
long long cfg_slots(int cfg, int ni, int nj) {
  std::vector<PlaneTile> t;
  if (!plane_tiles(cfg, 0, ni, nj, &t)) return -1;
  return (long long)t.size() * ST_THREADS_OF[cfg];
}

// Uploads the tile lists of the blocks' configurations.
int build_stencil_plan(z4c_ctx* c, const std::vector<DevBlock>& hb) {
  c->invalidate_graph();
  std::vector<PlaneTile> lists[NSTCFG];
  for (int b = 0; b < (int)hb.size(); ++b)
    if (!plane_tiles(c->blk_cfg[b], b, hb[b].ni, hb[b].nj, &lists[c->blk_cfg[b]]))
      return fail(Z4C_EINVAL, "stencil plan: no tile fits block " + std::to_string(b));
  for (int q = 0; q < NSTCFG; ++q) {
    hipFree(c->st_tiles[q]);
    c->st_tiles[q] = nullptr;
    c->st_ntiles[q] = 0;
    if (lists[q].empty()) continue;
    if (hipMalloc(&c->st_tiles[q], sizeof(PlaneTile) * lists[q].size()) != hipSuccess)
      return fail(Z4C_ENOMEM, "stencil plan: allocation failed");
    HIPCALL(hipMemcpy(c->st_tiles[q], lists[q].data(), sizeof(PlaneTile) * lists[q].size(),
                      hipMemcpyHostToDevice));
    c->st_ntiles[q] = (int)lists[q].size();
  }
  std::vector<PlaneTile> lin;
  for (int b = 0; b < (int)hb.size(); ++b)
    if (!plane_tiles(0, b, hb[b].ni, hb[b].nj, &lin))
      return fail(Z4C_EINVAL, "stencil plan: no tile fits block " + std::to_string(b));
  hipFree(c->lin_tiles);
  c->lin_tiles = nullptr;
  c->lin_ntiles = 0;
  if (hipMalloc(&c->lin_tiles, sizeof(PlaneTile) * lin.size()) != hipSuccess)
    return fail(Z4C_ENOMEM, "stencil plan: allocation failed");
  HIPCALL(hipMemcpy(c->lin_tiles, lin.data(), sizeof(PlaneTile) * lin.size(), hipMemcpyHostToDevice));
  c->lin_ntiles = (int)lin.size();
  return Z4C_OK;
}

void launch_stencil_cfg(int cfg, const StencilArgs& sa, hipStream_t s) {
  const dim3 g(grid_for(sa.ntiles * NVAR));
  switch (cfg) {
    case 0: hipLaunchKernelGGL(k_stencil<StCfg256>, g, dim3(StCfg256::THREADS), 0, s, sa); break;
    case 1: hipLaunchKernelGGL(k_stencil<StCfg320>, g, dim3(StCfg320::THREADS), 0, s, sa); break;
    case 2: hipLaunchKernelGGL(k_stencil<StCfg192>, g, dim3(StCfg192::THREADS), 0, s, sa); break;
    case 3: hipLaunchKernelGGL(k_stencil<StCfg384>, g, dim3(StCfg384::THREADS), 0, s, sa); break;
    case 4: hipLaunchKernelGGL(k_stencil<StCfg640>, g, dim3(StCfg640::THREADS), 0, s, sa); break;
    default: hipLaunchKernelGGL(k_stencil<StCfg576>, g, dim3(StCfg576::THREADS), 0, s, sa); break;
  }
}

// Whether z4c_rhs runs in two passes (3 % in doubt: the one kernel, which needs no
// slots), and the stages of a step: a stage in one kernel pays for the second
// buffer that its state goes to, about 5 % of a right-hand side, and `extra` us.
bool rhs_two(const z4c_ctx* c) {
  return c->form ? c->form == Z4C_FORM_TWO_PASSES : c->t_one >= 1.03 * c->t_two;
}
bool step_two(const z4c_ctx* c, double extra = 0.0) {
  return c->form ? c->form == Z4C_FORM_TWO_PASSES : c->t_one + extra >= 0.95 * c->t_two;
}

// The derivative slots, allocated by the first two-pass right-hand side.
int ensure_slots(z4c_ctx* c) {
  if (c->dv) return Z4C_OK;
  // also while the caller captures a graph: the allocation is no part of it
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  HIPCALL(hipThreadExchangeStreamCaptureMode(&mode));
  const hipError_t e = hipMalloc(&c->dv, sizeof(double) * c->total_dv);
  HIPCALL(hipThreadExchangeStreamCaptureMode(&mode));
  if (e != hipSuccess) {
    c->dv = nullptr;
    return fail(Z4C_ENOMEM, "derivative-slot allocation failed");
  }
  return Z4C_OK;
}

// Whether to run in two passes where the estimate (`two`) or z4c_set_rhs_form says
// so: only a form that the caller fixed fails for want of memory, the estimate's
// falls back to the one kernel, which needs no slots, for good.
bool with_slots(z4c_ctx* c, bool two) {
  if (!two || c->form || ensure_slots(c) == Z4C_OK) return two;
  (void)hipGetLastError();
  c->t_two = std::numeric_limits<double>::infinity();
  return false;
}

// Bricks of the one-kernel right-hand side, cut as equal as they divide, and the
// time of both forms.
//
// One kernel: a brick takes 35 to 37 us however few there are (its 22 fields in
// turn), 53 us with a second one on its CU, 84 us when a third round begins, and
// from there 0.093 us a brick.  Two passes: a workgroup of the stencil pass
// marches the planes of a tile, 1.75 us each on top of 20 us (16 us once there
// are enough for the fields of a tile to meet on one XCD); a full chip takes
// 0.003 us a workgroup and 0.003 us a plane, the algebra 0.1 us per 256 vertices.
// Tiles that split a block's rows take half as long again a plane.  Against 132
// batches measured in both forms (2 to 64 cells a side; cubes, rods, plates and
// mixtures; 1 to 2048 blocks) the first estimate is within 6 % (rms) and the
// second within 9 % (7 % where the two are close).  z4c_rhs in the form that
// rhs_two takes from them loses 0.12 % to the better one on average and 4 % at most
// (18 blocks of 15 x 24 x 3 cells, 39.7 against 38.1 us), an rk4 step 0.11 % and 4 %;
// always one kernel loses 4.4 % on average and up to 58 % (16 blocks of 2^3: 34.0
// against 21.5 us; 64 of 4 x 64 x 4: 160 against 105).
int build_fused_tiles(z4c_ctx* c, const std::vector<DevBlock>& hb) {
  constexpr int M[3] = {FuCfg::BX, FuCfg::BY, FuCfg::BZ};
  std::vector<FusedTile> t;
  double planes = 0, march = 0, wgs = 0, alg = 0;
  std::vector<PlaneTile> pt;
  for (int b = 0; b < (int)hb.size(); ++b) {
    const int n[3] = {hb[b].ni, hb[b].nj, hb[b].nk};
    int s[3];
    for (int d = 0; d < 3; ++d) {
      const int q = (n[d] + M[d] - 1) / M[d];
      s[d] = (n[d] + q - 1) / q;
    }
    for (int k0 = 0; k0 < n[2]; k0 += s[2])
      for (int j0 = 0; j0 < n[1]; j0 += s[1])
        for (int i0 = 0; i0 < n[0]; i0 += s[0])
          t.push_back(FusedTile{b, i0, j0, k0, std::min(s[0], n[0] - i0), std::min(s[1], n[1] - j0),
                                std::min(s[2], n[2] - k0)});
    pt.clear();
    plane_tiles(c->blk_cfg[b], b, n[0], n[1], &pt);
    const double w = (double)pt.size() * NVAR;
    wgs += w;
    march += w * n[2] * (pt[0].ni < n[0] ? 1.5 : 1.0);
    planes = std::max(planes, (double)n[2]);
    alg += (hb[b].nint + TILE - 1) / TILE;
  }
  if (hipMalloc(&c->fu_tiles, sizeof(FusedTile) * t.size()) != hipSuccess)
    return fail(Z4C_ENOMEM, "set_blocks: brick table allocation failed");
  HIPCALL(hipMemcpy(c->fu_tiles, t.data(), sizeof(FusedTile) * t.size(), hipMemcpyHostToDevice));
  c->fu_ntiles = (int)t.size();
  const double nt = (double)t.size(), cu = c->n_cu;
  c->t_one = std::max(nt > 2 * cu ? 84.0 : nt > cu ? 53.0 : 37.0, 0.093 * nt + 8.0);
  const double lat = 20.0 + 1.75 * planes - (wgs >= 8 * NVAR ? 4.0 : 0.0);
  const double thr = 12.0 + 0.003 * wgs + 0.003 * march + 0.1 * alg;
  c->t_two = std::sqrt(std::sqrt(lat * lat * lat * lat + thr * thr * thr * thr));
  with_slots(c, rhs_two(c) || step_two(c));
  return Z4C_OK;
}

// The launch does the work of the stencil and the assembly passes: the kernel
// timer divides its time between them by their arithmetic (4435 and 3374
// operations per vertex).
int launch_fused(z4c_ctx* c, FusedArgs a, hipStream_t s) {
  a.blocks = c->d_blocks;
  a.tiles = c->fu_tiles;
  a.ntiles = c->fu_ntiles;
  PassTimer t1(c, Z4C_PASS_STENCIL, s, 0.57);
  PassTimer t2(c, Z4C_PASS_ASSEMBLY, s, 0.43);
  hipLaunchKernelGGL(k_fused<FuCfg>, dim3(grid_for(a.ntiles)), dim3(FuCfg::THREADS), 0, s, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

// The stencil pass over all blocks: one launch per configuration in use.
int launch_stencil(z4c_ctx* c, const double* u, const z4c_params* p, hipStream_t s) {
  const int rc = ensure_slots(c);
  if (rc) return rc;
  PassTimer t(c, Z4C_PASS_STENCIL, s);
  for (int q = 0; q < NSTCFG; ++q) {
    if (!c->st_ntiles[q]) continue;
    StencilArgs sa{c->d_blocks, c->st_tiles[q], c->st_ntiles[q], u, c->dv, p->diss,
                   p->lapse_advect, p->shift_advect};
    launch_stencil_cfg(q, sa, s);
    HIPCALL(hipGetLastError());
  }
  return Z4C_OK;
}

// One stage of a step: right-hand side of a.u, update and AlgConstr into a.out,
// in one kernel or in two passes.  A zero right-hand side (cowling) always takes
// the second pass alone.
int launch_stage(z4c_ctx* c, const z4c_params* p, bool two, FusedArgs a, hipStream_t s) {
  if (!two) return launch_fused(c, a, s);
  if (!a.cowling) {
    const int rc = launch_stencil(c, a.u, p, s);
    if (rc) return rc;
  }
  a.blocks = c->d_blocks;
  const StageArgs sa{a, launch_of(c, BOX_INTERIOR), c->dv};
  PassTimer t(c, Z4C_PASS_ASSEMBLY, s);
  auto* k = a.ls ? (a.alg ? k_rk4_stage<true, true> : k_rk4_stage<false, true>)
                 : (a.alg ? k_rk4_stage<true, false> : k_rk4_stage<false, false>);
  hipLaunchKernelGGL(k, dim3(grid_for(sa.L.ntiles)), dim3(TILE), 0, s, sa);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

int launch_rhs(z4c_ctx* c, const z4c_params* p, const double* u,
               const double* mat, double* rhs, bool sommerfeld, hipStream_t s) {
  if (p->cowling) return fill(c, rhs, 0.0, c->total_pts * NVAR, s);
  // one kernel, unless the batch is better off in two passes or the right-hand
  // side is written over its own input (every brick reads its neighbours' vertices)
  const long long nn = c->total_pts * NVAR;
  const bool apart = (uintptr_t)rhs + 8 * nn <= (uintptr_t)u || (uintptr_t)u + 8 * nn <= (uintptr_t)rhs;
  if (apart && !with_slots(c, rhs_two(c))) {
    FusedArgs a{};
    a.u = u;
    a.mat = mat;
    a.o = rhs_params(p);
    a.sommerfeld = sommerfeld;
    a.rhs = rhs;
    return launch_fused(c, a, s);
  }
  int rc = launch_stencil(c, u, p, s);
  if (rc) return rc;
  RhsArgs a{c->d_blocks, launch_of(c, BOX_INTERIOR), u, c->dv, mat, rhs, rhs_params(p)};
  const int g = grid_for(a.L.ntiles);
  {
    PassTimer t(c, Z4C_PASS_ASSEMBLY, s);
    if (sommerfeld)
      hipLaunchKernelGGL(k_rhs_alg<true>, dim3(g), dim3(TILE), 0, s, a);
    else
      hipLaunchKernelGGL(k_rhs_alg<false>, dim3(g), dim3(TILE), 0, s, a);
  }
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

int launch_alg(z4c_ctx* c, const z4c_params* p, double* u, const int* range,
               int skip, hipStream_t s) {
  AlgArgs a{};
  a.blocks = c->d_blocks;
  a.L = launch_of(c, BOX_WHOLE);
  a.u = u;
  a.eps_floor = p->eps_floor;
  a.tf_force = p->tf_force_regularization;
  a.force_reg = p->force_regularization;
  for (int q = 0; q < 6; ++q) a.range[q] = range ? range[q] : -1;
  a.skip_physical = skip;
  PassTimer t(c, Z4C_PASS_ALGCONSTR, s);
  hipLaunchKernelGGL(k_algconstr, dim3(grid_for(a.L.ntiles)), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

int launch_bt(z4c_ctx* c, int nvar, double* out, const double* u0, int nk,
              const double* const* k, const double* w, double dt, hipStream_t s) {
  if (nk < 0 || nk > MAXK) return fail(Z4C_EINVAL, "bt_sum: nk must be in [0, 8]");
  BtArgs a{};
  a.out = out;
  a.u0 = u0;
  a.n = c->total_pts * nvar;
  int m = 0;
  for (int j = 0; j < nk; ++j) {
    if (w[j] != 0) {
      if (!k[j]) return fail(Z4C_EINVAL, "bt_sum: null k pointer with nonzero weight");
      a.k[m] = k[j];
      a.w[m] = w[j] * dt;
      ++m;
    }
  }
  a.nk = m;
  PassTimer t(c, Z4C_PASS_BT_SUM, s);
  hipLaunchKernelGGL(k_bt_sum, dim3(elementwise_grid(a.n)), dim3(256), 0, s, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

int ensure_snapshot(z4c_ctx* c, long long n) {
  if (c->snap_elems >= n) return Z4C_OK;
  c->invalidate_graph();  // a captured step may hold the old scratch
  hipFree(c->snap);
  c->snap = nullptr;
  c->snap_elems = 0;
  if (hipMalloc(&c->snap, sizeof(double) * n) != hipSuccess)
    return fail(Z4C_ENOMEM, "snapshot allocation failed");
  c->snap_elems = n;
  return Z4C_OK;
}

int launch_periodic(z4c_ctx* c, int nvar, double* u, hipStream_t s) {
  if (!c->per_snap && nvar <= 65535) {
    PerArgs a{c->d_blocks, launch_of(c, BOX_GHOST), nvar, u, nullptr};
    hipLaunchKernelGGL(k_periodic_ghosts, dim3(grid_for(a.L.ntiles), nvar), dim3(TILE), 0, s, a);
    HIPCALL(hipGetLastError());
    a.L = launch_of(c, BOX_FACE);
    hipLaunchKernelGGL(k_periodic_faces, dim3(grid_for(a.L.ntiles), nvar), dim3(TILE), 0, s, a);
    HIPCALL(hipGetLastError());
    return Z4C_OK;
  }
  const long long n = c->total_pts * nvar;
  const int rc = ensure_snapshot(c, n);
  if (rc) return rc;
  hipLaunchKernelGGL(k_copy, dim3(elementwise_grid(n)), dim3(256), 0, s, c->snap, (const double*)u, n);
  HIPCALL(hipGetLastError());
  PerArgs a{c->d_blocks, launch_of(c, BOX_WHOLE), nvar, u, c->snap};
  hipLaunchKernelGGL(k_periodic, dim3(grid_for(a.L.ntiles)), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

// Line tables of the physical fill (per field; scaled by nvar at launch).
int build_physical_tables(z4c_ctx* c, const std::vector<DevBlock>& hb) {
  for (int ax = 0; ax < 3; ++ax) {
    std::vector<PhysLine> t;
    long long start = 0;
    for (int b = 0; b < (int)hb.size(); ++b) {
      const DevBlock& B = hb[b];
      if (!(B.pfaces & (3 << (2 * ax)))) continue;
      const int is = B.il, ie = B.iu - 1, js = B.jl, je = B.ju - 1, ks = B.kl, ke = B.ku - 1;
      const int bis = is - NG, bie = ie + NG;
      const int bjs = (B.pfaces & 4) ? js : js - NG, bje = (B.pfaces & 8) ? je : je + NG;
      const int bks = (B.pfaces & 16) ? ks : ks - NG, bke = (B.pfaces & 32) ? ke : ke + NG;
      PhysLine e{};
      e.block = b;
      if (ax == 0) { e.lo0 = bjs; e.n0 = bje - bjs + 1; e.lo1 = bks; e.n1 = bke - bks + 1; }
      else if (ax == 1) { e.lo0 = bis; e.n0 = bie - bis + 1; e.lo1 = bks; e.n1 = bke - bks + 1; }
      else { e.lo0 = bis; e.n0 = bie - bis + 1; e.lo1 = js - NG; e.n1 = je - js + 1 + 2 * NG; }
      e.start = start;
      start += (long long)e.n0 * e.n1;
      t.push_back(e);
    }
    hipFree(c->ph_lines[ax]);
    c->ph_lines[ax] = nullptr;
    c->ph_nent[ax] = (int)t.size();
    c->ph_nlines1[ax] = start;
    if (t.empty()) continue;
    if (hipMalloc(&c->ph_lines[ax], sizeof(PhysLine) * t.size()) != hipSuccess)
      return fail(Z4C_ENOMEM, "physical fill: allocation failed");
    HIPCALL(hipMemcpy(c->ph_lines[ax], t.data(), sizeof(PhysLine) * t.size(), hipMemcpyHostToDevice));
  }
  return Z4C_OK;
}

int launch_physical(z4c_ctx* c, int nvar, double* u, hipStream_t s) {
  for (int ax = 0; ax < 3; ++ax) {
    if (!c->ph_nent[ax]) continue;
    // the table holds one field's lines; the field is the slowest index
    PhysArgs a{c->d_blocks, c->ph_lines[ax], c->ph_nent[ax], c->ph_nlines1[ax],
               c->ph_nlines1[ax] * nvar, ax, nvar, u};
    hipLaunchKernelGGL(k_physical, dim3((unsigned)((a.nlines + 255) / 256)), dim3(256), 0, s, a);
    HIPCALL(hipGetLastError());
  }
  return Z4C_OK;
}

int launch_ml_exchange(z4c_ctx* c, int nvar, double* u, hipStream_t s) {
  if (nvar > NVAR) return fail(Z4C_EINVAL, "exchange: at most 22 fields across levels");
  // every block restricts its interior into its coarse buffer
  RestrictArgs ra{c->d_blocks, c->d_rf, c->d_rchunks, nvar, u, c->ml_coarse};
  hipLaunchKernelGGL(k_restrict_vc, dim3(c->n_rchunks), dim3(256), 0, s, ra);
  HIPCALL(hipGetLastError());
  if (c->ml_ndst) {
    MlxArgs a{c->d_blocks, c->d_rf, c->ml_dst, c->ml_off, c->ml_src, c->ml_inv,
              c->ml_ndst, c->ml_nint, nvar, u, c->ml_coarse, c->ml_tmp};
    const dim3 g((c->ml_ndst + 255) / 256);
    if (nvar == NVAR)
      hipLaunchKernelGGL(k_mlx_gather<NVAR>, g, dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL(k_mlx_gather<0>, g, dim3(256), 0, s, a);
    HIPCALL(hipGetLastError());
    if (c->ml_nint) {
      hipLaunchKernelGGL(k_mlx_scatter, dim3((c->ml_nint + 255) / 256), dim3(256), 0, s, a);
      HIPCALL(hipGetLastError());
    }
  }
  for (int ax = 0; ax < 3; ++ax) {
    if (!c->mlp_nent[ax]) continue;
    PhysCArgs pc{c->d_blocks, c->d_rf, c->mlp_lines[ax], c->mlp_nent[ax], c->mlp_nlines1[ax],
                 c->mlp_nlines1[ax] * nvar, ax, nvar, c->ml_coarse};
    hipLaunchKernelGGL(k_physical_coarse, dim3((unsigned)((pc.nlines + 255) / 256)), dim3(256), 0,
                       s, pc);
    HIPCALL(hipGetLastError());
  }
  if (c->ml_npgroups) {
    ProlongArgs pa{c->d_blocks, c->d_rf, c->ml_pent, c->ml_pgroups, c->ml_coarse, u, nvar};
    hipLaunchKernelGGL(k_prolong_vc, dim3(c->ml_npgroups, nvar), dim3(256),
                       sizeof(double) * c->ml_prlds, s, pa);
    HIPCALL(hipGetLastError());
  }
  return Z4C_OK;
}

int launch_exchange(z4c_ctx* c, int nvar, double* u, hipStream_t s) {
  if (c->ml) return launch_ml_exchange(c, nvar, u, s);
  if (!c->ex_ndst) return Z4C_OK;
  // the destinations' new values go through a scratch array of nvar * ndst
  // doubles (gather, then scatter), not through a copy of the whole state
  int rc = ensure_snapshot(c, (long long)c->ex_ndst * nvar);
  if (rc) return rc;
  ExArgs a{c->d_blocks, c->ex_dst, c->ex_off, c->ex_src, c->ex_ndst, nvar, u, c->snap};
  const dim3 g((c->ex_ndst + 255) / 256);
  hipLaunchKernelGGL(k_exchange_gather, g, dim3(256), 0, s, a);
  HIPCALL(hipGetLastError());
  hipLaunchKernelGGL(k_exchange_scatter, g, dim3(256), 0, s, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

bool rf_read_range(const RfEntry& E, int a, int& lo, int& hi);

// The transpose data of the update across levels, built on first use from
// the device plan: the transposed gather lists (sources in first-use order,
// each with its destinations in destination order), the fine vertices the
// prolongation writes (mask and list) and the coarse vertices it reads.
int build_ml_transpose(z4c_ctx* c) {
  if (c->mlt_built) return Z4C_OK;
  const int nd = c->ml_ndst;
  std::vector<long long> off(nd + 1, 0);
  std::vector<int> dst(2 * (size_t)nd);
  if (nd) {
    HIPCALL(hipMemcpy(off.data(), c->ml_off, sizeof(long long) * (nd + 1), hipMemcpyDeviceToHost));
    HIPCALL(hipMemcpy(dst.data(), c->ml_dst, sizeof(int) * 2 * nd, hipMemcpyDeviceToHost));
  }
  const long long ns = off[nd];
  if (ns >= (long long)std::numeric_limits<int>::max())
    return fail(Z4C_EINVAL, "exchange_vjp: plan too large");
  std::vector<int> src(2 * ns);
  if (ns) HIPCALL(hipMemcpy(src.data(), c->ml_src, sizeof(int) * 2 * ns, hipMemcpyDeviceToHost));
  std::vector<RfEntry> ent(c->ml_nent);
  if (c->ml_nent)
    HIPCALL(hipMemcpy(ent.data(), c->ml_pent, sizeof(RfEntry) * ent.size(), hipMemcpyDeviceToHost));
  const long long nf = c->total_pts, ncp = c->rf_total;
  auto slot = [&](int blkarr, int p) -> long long {
    const int b = blkarr >> 1;
    return (blkarr & 1) ? nf + c->hrf[b].coff + p : c->hdev[b].off + p;
  };
  // the sources in memory order (coalesced scatter), each numbered once
  std::vector<int> id(nf + ncp, -1), tv;
  std::vector<std::pair<long long, long long>> first;  // (slot, entry)
  for (long long e = 0; e < ns; ++e) {
    const long long k = slot(src[2 * e], src[2 * e + 1]);
    if (id[k] == -1) {
      id[k] = -2;
      first.emplace_back(k, e);
    }
  }
  std::sort(first.begin(), first.end());
  const int nv = (int)first.size();
  for (int q = 0; q < nv; ++q) {
    id[first[q].first] = q;
    tv.push_back(src[2 * first[q].second]);
    tv.push_back(src[2 * first[q].second + 1]);
  }
  std::vector<int> cnt(nv, 0);
  for (long long e = 0; e < ns; ++e) ++cnt[id[slot(src[2 * e], src[2 * e + 1])]];
  std::vector<int> toff(nv + 1, 0);
  for (int q = 0; q < nv; ++q) toff[q + 1] = toff[q] + cnt[q];
  std::vector<int> td(ns), pos(toff.begin(), toff.end() - 1);
  for (int d = 0; d < nd; ++d)
    for (long long e = off[d]; e < off[d + 1]; ++e) td[pos[id[slot(src[2 * e], src[2 * e + 1])]]++] = d;
  std::vector<int> tflag(nv, 0), tz;
  for (int d = 0; d < nd; ++d) {
    const int q = id[slot(dst[2 * d], dst[2 * d + 1])];
    if (q < 0)
      tz.push_back(d);
    else
      tflag[q] = 1;
  }
  std::vector<unsigned char> mask(nf, 0);
  std::vector<int> fl;
  // per block, the bounding box of the coarse vertices the prolongation reads
  const int nb = (int)c->hdev.size();
  std::vector<std::array<int, 6>> cbox(nb, {INT_MAX, INT_MIN, INT_MAX, INT_MIN, INT_MAX, INT_MIN});
  for (const RfEntry& E : ent) {
    const DevBlock& B = c->hdev[E.blk];
    const RfBlock& R = c->hrf[E.blk];
    for (int m = 0; m < 8; ++m) {
      int c0[3], n[3];
      for (int d = 0; d < 3; ++d) rf_case_range(E, d, (m >> d) & 1, c0[d], n[d]);
      if (n[0] <= 0 || n[1] <= 0 || n[2] <= 0) continue;
      for (int ck = c0[2]; ck < c0[2] + n[2]; ++ck)
        for (int cj = c0[1]; cj < c0[1] + n[1]; ++cj)
          for (int ci = c0[0]; ci < c0[0] + n[0]; ++ci) {
            const int fi = 2 * (ci - RF_H) + (m & 1), fj = 2 * (cj - RF_H) + ((m >> 1) & 1),
                      fk = 2 * (ck - RF_H) + (m >> 2);
            const int p = fi + B.nn1 * (fj + B.nn2 * fk);
            if (!mask[B.off + p]) {
              mask[B.off + p] = 1;
              fl.push_back(E.blk);
              fl.push_back(p);
            }
          }
    }
    int lo[3], hi[3];
    bool any = true;
    for (int d = 0; d < 3; ++d) any = any && rf_read_range(E, d, lo[d], hi[d]);
    if (!any) continue;
    auto& bx = cbox[E.blk];
    for (int d = 0; d < 3; ++d) {
      bx[2 * d] = std::min(bx[2 * d], lo[d]);
      bx[2 * d + 1] = std::max(bx[2 * d + 1], hi[d]);
    }
    (void)R;
  }
  // tiles of ty x tz coarse rows over each box, one (ty, tz) for the launch:
  // the fewest staged fine values whose largest tile fits in LDS
  auto fine_range = [](int c_lo, int c_hi, int nn, int& f0, int& nfv) {
    f0 = std::max(0, 2 * (c_lo - RF_H) - 5);
    nfv = std::min(nn - 1, 2 * (c_hi - RF_H) + 5) - f0 + 1;
  };
  auto make_tiles = [&](int ty, int tz, std::vector<PrTTile>* out, long long& staged,
                        int& lds) {
    staged = 0;
    lds = 0;
    for (int b = 0; b < nb; ++b) {
      const auto& bx = cbox[b];
      if (bx[0] > bx[1]) continue;
      const DevBlock& B = c->hdev[b];
      int fx0, nfx;
      fine_range(bx[0], bx[1], B.nn1, fx0, nfx);
      for (int cz = bx[4]; cz <= bx[5]; cz += tz)
        for (int cy = bx[2]; cy <= bx[3]; cy += ty) {
          PrTTile t{};
          t.blk = b;
          t.cx0 = bx[0];
          t.ncx = bx[1] - bx[0] + 1;
          t.cy0 = cy;
          t.ncy = std::min(ty, bx[3] - cy + 1);
          t.cz0 = cz;
          t.ncz = std::min(tz, bx[5] - cz + 1);
          t.fx0 = fx0;
          t.nfx = nfx;
          fine_range(cy, cy + t.ncy - 1, B.nn2, t.fy0, t.nfy);
          fine_range(cz, cz + t.ncz - 1, B.nn3, t.fz0, t.nfz);
          staged += (long long)t.nfx * t.nfy * t.nfz;
          lds = std::max(lds, t.nfx * t.nfy * t.nfz + t.nfx * t.nfy * t.ncz + t.nfx * t.ncy * t.ncz);
          if (out) out->push_back(t);
        }
    }
  };
  int smem = 0;
  HIPCALL(hipDeviceGetAttribute(&smem, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device));
  // within 76 KiB (two workgroups per CU), else within the device's LDS
  // (large blocks: the x extent of a tile is the block's coarse x range)
  const int lds_cap[2] = {std::min(9728, smem / (int)sizeof(double)),
                          smem / (int)sizeof(double)};
  int best_ty = 0, best_tz = 0;
  long long best = LLONG_MAX;
  int ymax = 1, zmax = 1;
  for (const auto& bx : cbox)
    if (bx[0] <= bx[1]) {
      ymax = std::max(ymax, bx[3] - bx[2] + 1);
      zmax = std::max(zmax, bx[5] - bx[4] + 1);
    }
  for (int pass = 0; pass < 2 && !best_ty; ++pass)
    for (int tz = 1; tz <= std::min(zmax, 8); ++tz)
      for (int ty = 1; ty <= ymax; ++ty) {
        long long staged;
        int lds;
        make_tiles(ty, tz, nullptr, staged, lds);
        if (lds <= lds_cap[pass] && staged < best) {
          best = staged;
          best_ty = ty;
          best_tz = tz;
        }
      }
  std::vector<PrTTile> tiles;
  if (!ent.empty()) {
    if (!best_ty) return fail(Z4C_EINVAL, "exchange_vjp: blocks too large for the prolongation's transpose");
    long long staged;
    make_tiles(best_ty, best_tz, &tiles, staged, c->ml_ptlds);
  }
  auto up = [&](auto*& d, const auto& h) {
    using T = std::remove_pointer_t<std::remove_reference_t<decltype(d)>>;
    if (h.empty()) return true;
    if (hipMalloc(&d, sizeof(T) * h.size()) != hipSuccess) return false;
    return hipMemcpy(d, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice) == hipSuccess;
  };
  bool ok = up(c->mlt_v, tv) && up(c->mlt_flag, tflag) && up(c->mlt_off, toff) &&
            up(c->mlt_d, td) && up(c->mlt_z, tz) && up(c->ml_fmask, mask) && up(c->ml_fl, fl) &&
            up(c->ml_ptiles, tiles);
  ok = ok && (nv == 0 || hipMalloc(&c->mlt_tmp, sizeof(double) * NVAR * (size_t)nv) == hipSuccess);
  ok = ok && hipMalloc(&c->ml_cbar, sizeof(double) * NVAR * (size_t)ncp) == hipSuccess;
  if (!ok) {
    c->drop_mlt();
    return fail(Z4C_ENOMEM, "exchange_vjp: allocation failed");
  }
  c->mlt_nv = nv;
  c->mlt_nz = (int)tz.size();
  c->ml_nfl = (int)(fl.size() / 2);
  c->ml_nptiles = (int)tiles.size();
  c->mlt_built = true;
  return Z4C_OK;
}

// u-bar <- (the update across levels)^T u-bar, nvar fields: P^T, Phi_c^T,
// E_g^T, R^T on (u-bar, c-bar), c-bar = 0 to start
int launch_ml_exchange_vjp(z4c_ctx* c, int nvar, double* ubar, hipStream_t s) {
  int rc = build_ml_transpose(c);
  if (rc) return rc;
  rc = fill(c, c->ml_cbar, 0.0, (long long)nvar * c->rf_total, s);
  if (rc) return rc;
  PrTArgs pa{c->d_blocks, c->d_rf, c->ml_ptiles, c->ml_fl, c->ml_nfl, c->ml_fmask,
             nvar, ubar, c->ml_cbar};
  if (c->ml_nptiles) {
    hipLaunchKernelGGL(k_prolong_vjp, dim3(c->ml_nptiles, nvar), dim3(PRT_THREADS),
                       sizeof(double) * c->ml_ptlds, s, pa);
    HIPCALL(hipGetLastError());
  }
  if (c->ml_nfl) {
    hipLaunchKernelGGL(k_prolong_vjp_zero, dim3((c->ml_nfl + 255) / 256), dim3(256), 0, s, pa);
    HIPCALL(hipGetLastError());
  }
  for (int ax = 2; ax >= 0; --ax) {
    if (!c->mlp_nent[ax]) continue;
    PhysCArgs pc{c->d_blocks, c->d_rf, c->mlp_lines[ax], c->mlp_nent[ax], c->mlp_nlines1[ax],
                 c->mlp_nlines1[ax] * nvar, ax, nvar, c->ml_cbar};
    hipLaunchKernelGGL(k_physical_coarse_vjp, dim3((unsigned)((pc.nlines + 255) / 256)), dim3(256),
                       0, s, pc);
    HIPCALL(hipGetLastError());
  }
  MltArgs ma{c->d_blocks, c->d_rf, c->ml_dst, c->ml_inv, c->mlt_v, c->mlt_flag, c->mlt_off,
             c->mlt_d, c->mlt_z, c->mlt_nv, c->mlt_nz, nvar, ubar, c->ml_cbar, c->mlt_tmp};
  if (c->mlt_nv) {
    if (nvar == NVAR)
      hipLaunchKernelGGL(k_mlx_vjp_gather<NVAR>, dim3((c->mlt_nv + 255) / 256), dim3(256), 0, s, ma);
    else
      hipLaunchKernelGGL(k_mlx_vjp_gather<0>, dim3((c->mlt_nv + 255) / 256), dim3(256), 0, s, ma);
    HIPCALL(hipGetLastError());
  }
  if (c->mlt_nv + c->mlt_nz) {
    hipLaunchKernelGGL(k_mlx_vjp_scatter, dim3((c->mlt_nv + c->mlt_nz + 255) / 256), dim3(256), 0,
                       s, ma);
    HIPCALL(hipGetLastError());
  }
  RestrictTArgs ra{c->d_blocks, c->d_rf, c->d_rchunks, nvar, ubar, c->ml_cbar};
  hipLaunchKernelGGL(k_restrict_vjp, dim3(c->n_rchunks), dim3(256), 0, s, ra);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

// u-bar <- (the exchange set by z4c_set_exchange)^T u-bar, nvar fields
int launch_exchange_vjp(z4c_ctx* c, int nvar, double* ubar, hipStream_t s) {
  if (nvar > NVAR) return fail(Z4C_EINVAL, "exchange_vjp: at most 22 fields");
  if (c->ml) return launch_ml_exchange_vjp(c, nvar, ubar, s);
  if (!c->ext_nv && !c->ext_nz) return Z4C_OK;
  ExTArgs a{c->d_blocks, c->ex_dst, c->ex_off, c->ext_v, c->ext_flag, c->ext_off, c->ext_d,
            c->ext_z, c->ext_nv, c->ext_nz, nvar, ubar, c->ext_tmp};
  if (c->ext_nv) {
    if (nvar == NVAR)
      hipLaunchKernelGGL(k_exchange_vjp_gather<NVAR>, dim3((c->ext_nv + 255) / 256), dim3(256), 0, s,
                         a);
    else
      hipLaunchKernelGGL(k_exchange_vjp_gather<0>, dim3((c->ext_nv + 255) / 256), dim3(256), 0, s, a);
    HIPCALL(hipGetLastError());
  }
  hipLaunchKernelGGL(k_exchange_vjp_scatter, dim3((c->ext_nv + c->ext_nz + 255) / 256), dim3(256),
                     0, s, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

// u-bar <- (the physical fill)^T u-bar: the axes in reverse order
int launch_physical_vjp(z4c_ctx* c, int nvar, double* ubar, hipStream_t s) {
  for (int ax = 2; ax >= 0; --ax) {
    if (!c->ph_nent[ax]) continue;
    PhysArgs a{c->d_blocks, c->ph_lines[ax], c->ph_nent[ax], c->ph_nlines1[ax],
               c->ph_nlines1[ax] * nvar, ax, nvar, ubar};
    hipLaunchKernelGGL(k_physical_vjp, dim3((unsigned)((a.nlines + 255) / 256)), dim3(256), 0, s,
                       a);
    HIPCALL(hipGetLastError());
  }
  return Z4C_OK;
}

int ensure_buf(double*& p, long long& have, long long need, const char* what) {
  if (have >= need) return Z4C_OK;
  hipFree(p);
  p = nullptr;
  have = 0;
  if (hipMalloc(&p, sizeof(double) * (size_t)need) != hipSuccess)
    return fail(Z4C_ENOMEM, std::string(what) + ": scratch allocation failed");
  have = need;
  return Z4C_OK;
}

constexpr int MAX_NW = Z4C_MAX_NW;  // grid.y / grid.x limits of the adjoint kernels
static_assert(MAX_NW * NPBAR <= 65535 && Z4C_NPBAR == NPBAR, "cotangent limit");
static_assert(2 * MAX_NW <= 65535, "k_adj_stencil's grid.y holds two field halves per cotangent");

int check_vjp_args(const z4c_ctx* c, const z4c_params* p, int nw, const char* what) {
  if (nw < 1 || nw > MAX_NW)
    return fail(Z4C_EINVAL, std::string(what) + ": nw must be in [1, " + std::to_string(MAX_NW) + "]");
  for (const DevBlock& B : c->hdev)
    if ((long long)NLINF * B.nint * 8 > 0x7fffffffLL || (long long)NVAR * B.npts * 8 > 0x7fffffffLL)
      return fail(Z4C_EINVAL, std::string(what) + ": block too large for the adjoint's 32-bit buffer offsets");
  if (p->cowling) return fail(Z4C_EINVAL, std::string(what) + ": the Cowling right-hand side has no adjoint here");
  return Z4C_OK;
}

// The derivative part of the adjoint's linearisation of state u (into
// adj_lin, which the caller has sized).
int launch_lin(z4c_ctx* c, const z4c_params* p, const double* u, hipStream_t s) {
  StencilArgs sa{c->d_blocks, c->lin_tiles, c->lin_ntiles, u, c->adj_lin, p->diss,
                 p->lapse_advect, p->shift_advect, NLINF};
  hipLaunchKernelGGL(k_stencil_lin, dim3(grid_for(sa.ntiles * NVAR)), dim3(StCfg256::THREADS), 0,
                     s, sa);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

// ubar_c = (d rhs / d u)^T w_c for the nw cotangents; pbar (+)= parameter gradients
int launch_rhs_vjp(z4c_ctx* c, const z4c_params* p, const double* u, int nw, const double* w,
                   double* ubar, double* pbar, int accumulate, hipStream_t s) {
  const long long reg = c->total_pts * NVAR, sreg = c->total_int * NADJ;
  const int Gi = grid_for(c->ntiles[BOX_INTERIOR]);
  int rc = ensure_buf(c->adj_lin, c->adj_lin_n, c->total_int * NLINF, "rhs_vjp");
  if (!rc) rc = ensure_buf(c->adj_sb, c->adj_sb_n, (long long)nw * sreg, "rhs_vjp");
  if (!rc) rc = ensure_buf(c->adj_part, c->adj_part_n, (long long)nw * Gi * NPBAR, "rhs_vjp");
  if (!rc)
    rc = ensure_buf(c->adj_carry, c->adj_carry_n, (long long)nw * c->total_int * NCARRY_ALL,
                    "rhs_vjp");
  if (rc) return rc;
  AdjArgs a{c->d_blocks, launch_of(c, BOX_INTERIOR), rhs_params(p), u, c->adj_lin, w, ubar,
            c->adj_sb, c->adj_part, reg, sreg, w ? 0 : 1, c->adj_carry,
            c->total_int * NCARRY_ALL};
  rc = launch_lin(c, p, u, s);
  if (rc) return rc;
  hipLaunchKernelGGL(k_adj_fwd, dim3(Gi), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  hipLaunchKernelGGL(k_adj_point_a, dim3(Gi, nw), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  hipLaunchKernelGGL(k_adj_point_b, dim3(Gi, nw), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  a.L = launch_of(c, BOX_WHOLE);
  hipLaunchKernelGGL(k_adj_stencil, dim3(grid_for(a.L.ntiles), 2 * nw), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  hipLaunchKernelGGL(k_adj_pbar, dim3(nw * NPBAR), dim3(256), 0, s,
                     (const double*)c->adj_part, Gi, nw, pbar, accumulate);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

// J = sum over blocks and the cell loop of dx dy dz Ht^2 (host result)
int launch_hnorm(z4c_ctx* c, const z4c_params* p, const double* u, double* J, hipStream_t s) {
  const int Gi = grid_for(c->ntiles[BOX_INTERIOR]);
  int rc = ensure_buf(c->adj_lin, c->adj_lin_n, c->total_int * NLINF, "hamiltonian_norm");
  if (!rc) rc = ensure_buf(c->adj_part, c->adj_part_n, (long long)Gi * NPBAR, "hamiltonian_norm");
  if (rc) return rc;
  AdjArgs a{c->d_blocks, launch_of(c, BOX_INTERIOR), rhs_params(p), u, c->adj_lin, nullptr,
            nullptr, nullptr, c->adj_part, 0, 0, 1, nullptr, 0};
  rc = launch_lin(c, p, u, s);
  if (rc) return rc;
  hipLaunchKernelGGL(k_adj_fwd, dim3(Gi), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  hipLaunchKernelGGL(k_hnorm, dim3(Gi), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  std::vector<double> part(Gi);
  HIPCALL(hipMemcpyAsync(part.data(), c->adj_part, sizeof(double) * Gi, hipMemcpyDeviceToHost, s));
  HIPCALL(hipStreamSynchronize(s));
  double t = 0.0;
  for (double v : part) t += v;
  *J = t;
  return Z4C_OK;
}

// Adjoint of the fused bt_rk4 step: a forward sweep forms the stage states
// u_2..u_4 once (u_s = AlgConstr(u_n + a_s dt k_{s-1})) and keeps them with
// k_1..k_4 (stage checkpointing: four right-hand sides and three states per
// step, nothing per cotangent); the reverse sweep then runs stage by stage
// from those kept states.
int launch_rk4_step_vjp(z4c_ctx* c, const z4c_params* p, double dt, const double* u, int nw,
                        const double* ubar_out, double* ubar_in, double* pbar, hipStream_t s) {
  const long long reg = c->total_pts * NVAR;
  const long long k_n_before = c->adj_k_n;
  int rc = ensure_buf(c->adj_k, c->adj_k_n, 4 * reg, "rk4_step_vjp");
  if (c->adj_k_n != k_n_before) c->adj_k_zero = false;  // new allocation
  if (!rc) rc = ensure_buf(c->adj_stage, c->adj_stage_n, 3 * reg, "rk4_step_vjp");
  if (!rc) rc = ensure_buf(c->adj_reg, c->adj_reg_n, 3LL * nw * reg, "rk4_step_vjp");
  if (rc) return rc;
  double* K[4] = {c->adj_k, c->adj_k + reg, c->adj_k + 2 * reg, c->adj_k + 3 * reg};
  double* ybar = c->adj_reg;
  double* kbar = c->adj_reg + (long long)nw * reg;
  double* usbar = c->adj_reg + 2LL * nw * reg;
  const double aw[5] = {0., 0., 0.5, 0.5, 1.0};
  // the right-hand side leaves ghosts untouched: they must read zero.  Only
  // launch_rhs writes these registers, and it writes interior vertices only
  // on every path that reaches this point (Cowling, whose right-hand side
  // fills whole blocks, and Sommerfeld faces, whose boundary update is not
  // part of this adjoint, are rejected by z4c_rk4_step_vjp before the
  // sweep), so one zero fill per allocation keeps their ghosts zero.  A
  // path that lets launch_rhs write ghosts must clear adj_k_zero.
  if (!c->adj_k_zero) {
    rc = fill(c, c->adj_k, 0.0, c->adj_k_n, s);
    if (rc) return rc;
    c->adj_k_zero = true;
  }
  // stage states u_2..u_4, formed once in the forward sweep and kept for the
  // reverse sweep
  auto stage_buf = [&](int st) -> double* { return c->adj_stage + (long long)(st - 2) * reg; };
  auto stage_state = [&](int st) -> const double* {  // u_s
    if (st == 1) return u;
    const double* kk[1] = {K[st - 2]};
    const double wa[1] = {aw[st]};
    if (launch_bt(c, NVAR, stage_buf(st), u, 1, kk, wa, dt, s)) return nullptr;
    if (launch_alg(c, p, stage_buf(st), nullptr, 0, s)) return nullptr;
    return stage_buf(st);
  };
  for (int st = 1; st <= 4; ++st) {
    const double* in = stage_state(st);
    if (!in) return Z4C_EHIP;
    rc = launch_rhs(c, p, in, nullptr, K[st - 1], false, s);
    if (rc) return rc;
  }
  AdjStepArgs a{};
  a.blocks = c->d_blocks;
  a.L = launch_of(c, BOX_WHOLE);
  a.un = u;
  for (int q = 0; q < 4; ++q) a.k[q] = K[q];
  a.ubar_in = ubar_in;
  a.ybar = ybar;
  a.kbar = kbar;
  a.reg = reg;
  a.dt = dt;
  a.eps_floor = p->eps_floor;
  a.tf_force = p->tf_force_regularization;
  a.force_reg = p->force_regularization;
  const dim3 g(grid_for(a.L.ntiles), nw);
  a.bar = ubar_out;
  a.stage = 5;
  hipLaunchKernelGGL(k_adj_step, g, dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  for (int st = 4; st >= 1; --st) {
    const double* in = st == 1 ? u : stage_buf(st);
    rc = launch_rhs_vjp(c, p, in, nw, kbar, usbar, pbar, st == 4 ? 0 : 1, s);
    if (rc) return rc;
    a.bar = usbar;
    a.stage = st;
    hipLaunchKernelGGL(k_adj_step, g, dim3(TILE), 0, s, a);
    HIPCALL(hipGetLastError());
  }
  return Z4C_OK;
}

// Adjoint of z4c_rk4_step_ghosts with the exchange after every stage
// (ghosts = 2, + 4 for the physical fill): the forward sweep forms
// y_s = u_n + a_s dt k_{s-1} (ghosts at u_n), its update G(y_s) (the
// exchange, on several spacings the update across levels, then the fill;
// kept as AlgConstr's linearisation point) and u_s = AlgConstr(G(y_s)), with
// k_s = rhs(u_s); the reverse sweep carries each stage cotangent through
// AlgConstr's adjoint, G's transpose and the stage sums.
int launch_rk4_step_ghosts_vjp(z4c_ctx* c, const z4c_params* p, double dt, const double* u,
                               int nw, const double* ubar_out, double* ubar_in, double* pbar,
                               int ghosts, hipStream_t s) {
  const long long reg = c->total_pts * NVAR;
  const long long k_n_before = c->adj_k_n;
  int rc = ensure_buf(c->adj_k, c->adj_k_n, 4 * reg, "rk4_step_ghosts_vjp");
  if (c->adj_k_n != k_n_before) c->adj_k_zero = false;
  if (!rc) rc = ensure_buf(c->adj_stage, c->adj_stage_n, 3 * reg, "rk4_step_ghosts_vjp");
  if (!rc) rc = ensure_buf(c->adj_pre, c->adj_pre_n, 4 * reg, "rk4_step_ghosts_vjp");
  if (!rc) rc = ensure_buf(c->adj_reg, c->adj_reg_n, 3LL * nw * reg, "rk4_step_ghosts_vjp");
  if (rc) return rc;
  double* K[4] = {c->adj_k, c->adj_k + reg, c->adj_k + 2 * reg, c->adj_k + 3 * reg};
  double* ybar = c->adj_reg;
  double* kbar = c->adj_reg + (long long)nw * reg;
  double* usbar = c->adj_reg + 2LL * nw * reg;
  const double aw[5] = {0., 0., 0.5, 0.5, 1.0};
  const double bw[4] = {1. / 6., 1. / 3., 1. / 3., 1. / 6.};
  // the right-hand side writes interior vertices only (see launch_rk4_step_vjp)
  if (!c->adj_k_zero) {
    rc = fill(c, c->adj_k, 0.0, c->adj_k_n, s);
    if (rc) return rc;
    c->adj_k_zero = true;
  }
  auto pre = [&](int st) -> double* { return c->adj_pre + (long long)(st - 2) * reg; };  // 2..5
  auto stage_buf = [&](int st) -> double* { return c->adj_stage + (long long)(st - 2) * reg; };
  for (int st = 1; st <= 4; ++st) {
    const double* in = u;
    if (st >= 2) {
      const double* kk[1] = {K[st - 2]};
      const double wa[1] = {aw[st]};
      rc = launch_bt(c, NVAR, pre(st), u, 1, kk, wa, dt, s);
      if (!rc) rc = launch_exchange(c, NVAR, pre(st), s);
      if (!rc && (ghosts & 4)) rc = launch_physical(c, NVAR, pre(st), s);
      if (rc) return rc;
      HIPCALL(hipMemcpyAsync(stage_buf(st), pre(st), sizeof(double) * reg, hipMemcpyDeviceToDevice, s));
      rc = launch_alg(c, p, stage_buf(st), nullptr, 0, s);
      if (rc) return rc;
      in = stage_buf(st);
    }
    rc = launch_rhs(c, p, in, nullptr, K[st - 1], false, s);
    if (rc) return rc;
  }
  {
    const double* kk[4] = {K[0], K[1], K[2], K[3]};
    rc = launch_bt(c, NVAR, pre(5), u, 4, kk, bw, dt, s);
    if (!rc) rc = launch_exchange(c, NVAR, pre(5), s);
    if (!rc && (ghosts & 4)) rc = launch_physical(c, NVAR, pre(5), s);
    if (rc) return rc;
  }
  AdjStepArgs a{};
  a.blocks = c->d_blocks;
  a.L = launch_of(c, BOX_WHOLE);
  a.un = u;
  for (int q = 0; q < 4; ++q) a.k[q] = K[q];
  a.ubar_in = ubar_in;
  a.ybar = ybar;
  a.kbar = kbar;
  a.reg = reg;
  a.dt = dt;
  a.eps_floor = p->eps_floor;
  a.tf_force = p->tf_force_regularization;
  a.force_reg = p->force_regularization;
  a.ybar_stage = usbar;
  const dim3 g(grid_for(a.L.ntiles), nw);
  // cotangent of the exchanged, filled, constrained sums: AlgConstr's
  // adjoint, then the physical fill's and the exchange's transposes
  auto through_update = [&](int st) -> int {
    a.pre = pre(st);
    hipLaunchKernelGGL(k_adj_step_ex<1>, g, dim3(TILE), 0, s, a);
    HIPCALL(hipGetLastError());
    for (int q = 0; q < nw; ++q) {
      double* ub = usbar + (long long)q * reg;
      int r = (ghosts & 4) ? launch_physical_vjp(c, NVAR, ub, s) : Z4C_OK;
      if (!r) r = launch_exchange_vjp(c, NVAR, ub, s);
      if (r) return r;
    }
    return Z4C_OK;
  };
  HIPCALL(hipMemcpyAsync(usbar, ubar_out, sizeof(double) * reg * nw, hipMemcpyDeviceToDevice, s));
  a.stage = 5;
  rc = through_update(5);
  if (rc) return rc;
  hipLaunchKernelGGL(k_adj_step_ex<2>, g, dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  for (int st = 4; st >= 1; --st) {
    const double* in = st == 1 ? u : stage_buf(st);
    rc = launch_rhs_vjp(c, p, in, nw, kbar, usbar, pbar, st == 4 ? 0 : 1, s);
    if (rc) return rc;
    a.stage = st;
    if (st >= 2) {
      rc = through_update(st);
      if (rc) return rc;
    }
    hipLaunchKernelGGL(k_adj_step_ex<2>, g, dim3(TILE), 0, s, a);
    HIPCALL(hipGetLastError());
  }
  return Z4C_OK;
}

}  // namespace

// ===========================================================================
// C-ABI
// ===========================================================================
extern "C" {

const char* z4c_last_error(void) { return g_err.c_str(); }
int z4c_abi_version(void) { return Z4C_ABI_VERSION; }

int z4c_ctx_create(z4c_ctx** out, int device) {
  if (!out) return fail(Z4C_EINVAL, "null output pointer");
  *out = nullptr;
  int ndev = 0;
  HIPCALL(hipGetDeviceCount(&ndev));
  if (device < 0 || device >= ndev) return fail(Z4C_EINVAL, "device index out of range");
  HIPCALL(hipSetDevice(device));
  if (device >= MAX_DEVICES) return fail(Z4C_EINVAL, "device index beyond 63");
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_dev[device]) {
      void* ptr = nullptr;
      const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
      if (e != hipSuccess || !ptr)
        return fail(Z4C_EHIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
      g_scratch_dev[device] = static_cast<double*>(ptr);
    }
  }
  z4c_ctx* c = new z4c_ctx();
  c->device = device;
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) == hipSuccess) c->n_cu = prop.multiProcessorCount;
  *out = c;
  return Z4C_OK;
}

int z4c_ctx_destroy(z4c_ctx* c) {
  if (!c) return Z4C_OK;
  hipSetDevice(c->device);
  c->release();
  c->drop_timing();
  if (c->cap_stream) hipStreamDestroy(c->cap_stream);
  delete c;
  return Z4C_OK;
}

int z4c_set_blocks(z4c_ctx* c, const z4c_block* blocks, int nblocks,
                   long long* elems_per_var) {
  if (!c || !blocks || nblocks <= 0) return fail(Z4C_EINVAL, "set_blocks: bad arguments");
  HIPCALL(hipSetDevice(c->device));
  std::vector<DevBlock> hb(nblocks);
  std::vector<Box> boxes[NBOX];
  std::vector<Tile> tiles[NBOX];
  long long off = 0, ioff = 0, doff = 0;
  std::vector<int> blk_cfg;
  bool per_snap = false, faces = false;
  const double diss_scaling = std::pow(2.0, -2 * NG) * (NG % 2 == 0 ? -1 : 1);
  for (int b = 0; b < nblocks; ++b) {
    const z4c_block& in = blocks[b];
    if (in.offset != off)
      return fail(Z4C_EINVAL, "set_blocks: block " + std::to_string(b) +
                                  " offset must equal the sum of npts of earlier blocks");
    const int nn[3] = {in.nn1, in.nn2, in.nn3};
    const int lo[3] = {in.il, in.jl, in.kl}, hi[3] = {in.iu, in.ju, in.ku};
    for (int d = 0; d < 3; ++d) {
      if (lo[d] != NG || hi[d] != nn[d] - 1 - NG || hi[d] - lo[d] < 2)
        return fail(Z4C_EINVAL, "set_blocks: block " + std::to_string(b) +
                                    " must be vertex-centred with 4 ghosts and >= 3 interior vertices per axis");
      if (!(in.dx[d] > 0.0)) return fail(Z4C_EINVAL, "set_blocks: dx must be positive");
    }
    DevBlock& B = hb[b];
    B.off = off;
    B.ioff = ioff;
    B.doff = doff;
    B.nn1 = in.nn1; B.nn2 = in.nn2; B.nn3 = in.nn3;
    B.il = in.il; B.iu = in.iu; B.jl = in.jl; B.ju = in.ju; B.kl = in.kl; B.ku = in.ku;
    const long long npts = (long long)in.nn1 * in.nn2 * in.nn3;
    if (npts * ND1 > std::numeric_limits<int>::max())
      return fail(Z4C_EINVAL, "set_blocks: block too large");
    B.npts = (int)npts;
    B.ni = in.iu - in.il + 1;
    B.nj = in.ju - in.jl + 1;
    B.nk = in.ku - in.kl + 1;
    B.nint = B.ni * B.nj * B.nk;
    B.nis = (B.nint + DV_PAD + 15) / 16 * 16;
    if ((long long)B.nis * NDV * 8 >= (long long)DV_DROP)
      return fail(Z4C_EINVAL, "set_blocks: block too large");
    B.faces = in.sommerfeld_faces & 63;
    faces = faces || B.faces;
    B.pfaces = (in.sommerfeld_faces | in.outflow_faces) & 63;
    // stencil configuration until tuned: 256 threads (the fastest on 17^2,
    // 25^2 and 33^2 planes when measured), or 192 when the whole plane fits
    // one 192-thread tile (fewer idle lanes)
    {
      int best = StCfg192::fits(B.ni, B.nj) ? 2 : 0;
      if (cfg_slots(best, B.ni, B.nj) <= 0)
        return fail(Z4C_EINVAL, "set_blocks: no stencil tile fits block " + std::to_string(b));
      blk_cfg.push_back(best);
    }
    for (int d = 0; d < 3; ++d) {
      const double dx = in.dx[d];
      const double t = 1.0 / dx;
      B.dx[d] = dx;
      B.x0[d] = in.x0[d];
      B.cidx1[d] = 1.0 / (dx * 60.0);
      B.cidx2[d] = (t * t) / 180.0;
      B.cidx1lo[d] = 1.0 / (dx * 2.0);
      B.cidxd[d] = diss_scaling / (dx * 1.0);
      B.lidx[d] = 1.0 / (dx * 60.0);
    }
    Box bi, bp, bw;
    for (int d = 0; d < 3; ++d) {
      bi.lo[d] = lo[d]; bi.n[d] = hi[d] - lo[d] + 1;
      bp.lo[d] = lo[d] - (NG - 1); bp.n[d] = hi[d] - lo[d] + 1 + 2 * (NG - 1);
      bw.lo[d] = 0; bw.n[d] = nn[d];
    }
    const Box bx[3] = {bi, bp, bw};
    for (int kind = 0; kind < 3; ++kind) {
      const int id = (int)boxes[kind].size();
      boxes[kind].push_back(bx[kind]);
      const int np = bx[kind].n[0] * bx[kind].n[1] * bx[kind].n[2];
      for (int s = 0; s < np; s += TILE) tiles[kind].push_back(Tile{b, id, s});
    }
    {
      // ghost slabs: below/above in z, then in y, then in x
      const int nj = bi.n[1], nk = bi.n[2];
      const Box gb[6] = {
          {{0, 0, 0}, {nn[0], nn[1], lo[2]}},
          {{0, 0, hi[2] + 1}, {nn[0], nn[1], nn[2] - hi[2] - 1}},
          {{0, 0, lo[2]}, {nn[0], lo[1], nk}},
          {{0, hi[1] + 1, lo[2]}, {nn[0], nn[1] - hi[1] - 1, nk}},
          {{0, lo[1], lo[2]}, {lo[0], nj, nk}},
          {{hi[0] + 1, lo[1], lo[2]}, {nn[0] - hi[0] - 1, nj, nk}}};
      for (int q = 0; q < 6; ++q) {
        const int id = (int)boxes[BOX_GHOST].size();
        boxes[BOX_GHOST].push_back(gb[q]);
        const int np = gb[q].n[0] * gb[q].n[1] * gb[q].n[2];
        for (int s = 0; s < np; s += TILE) tiles[BOX_GHOST].push_back(Tile{b, id, s});
      }
    }
    {
      // one vertex of every set of periodic images: the lower z, y, x faces
      // without the upper edges
      const int mi = bi.n[0] - 1, mj = bi.n[1] - 1, mk = bi.n[2] - 1;
      const Box fb[3] = {{{lo[0], lo[1], lo[2]}, {mi, mj, 1}},
                         {{lo[0], lo[1], lo[2] + 1}, {mi, 1, mk - 1}},
                         {{lo[0], lo[1] + 1, lo[2] + 1}, {1, mj - 1, mk - 1}}};
      for (int q = 0; q < 3; ++q) {
        const int id = (int)boxes[BOX_FACE].size();
        boxes[BOX_FACE].push_back(fb[q]);
        const int np = fb[q].n[0] * fb[q].n[1] * fb[q].n[2];
        for (int s = 0; s < np; s += TILE) tiles[BOX_FACE].push_back(Tile{b, id, s});
      }
      if (mi < NG || mj < NG || mk < NG) per_snap = true;
    }
    off += npts;
    ioff += B.nint;
    doff += (long long)NDV * B.nis;
  }
  c->release();
  c->nblocks = 0;
  if (hipMalloc(&c->d_blocks, sizeof(DevBlock) * nblocks) != hipSuccess)
    return fail(Z4C_ENOMEM, "set_blocks: allocation failed");
  HIPCALL(hipMemcpy(c->d_blocks, hb.data(), sizeof(DevBlock) * nblocks, hipMemcpyHostToDevice));
  for (int kind = 0; kind < NBOX; ++kind) {
    if (hipMalloc(&c->d_tiles[kind], sizeof(Tile) * tiles[kind].size()) != hipSuccess ||
        hipMalloc(&c->d_boxes[kind], sizeof(Box) * boxes[kind].size()) != hipSuccess)
      return fail(Z4C_ENOMEM, "set_blocks: allocation failed");
    HIPCALL(hipMemcpy(c->d_tiles[kind], tiles[kind].data(), sizeof(Tile) * tiles[kind].size(),
                      hipMemcpyHostToDevice));
    HIPCALL(hipMemcpy(c->d_boxes[kind], boxes[kind].data(), sizeof(Box) * boxes[kind].size(),
                      hipMemcpyHostToDevice));
    c->ntiles[kind] = (int)tiles[kind].size();
  }
  if (hipMalloc(&c->d1, sizeof(double) * off * ND1) != hipSuccess)
    return fail(Z4C_ENOMEM, "set_blocks: derivative storage allocation failed");
  // prepared derivatives start at zero (the reference zero-initialises them)
  HIPCALL(hipMemset(c->d1, 0, sizeof(double) * off * ND1));
  c->total_dv = doff;
  c->per_snap = per_snap;
  c->faces = faces;
  c->blk_cfg = blk_cfg;
  c->hdev = hb;
  {
    int rc = build_stencil_plan(c, hb);
    if (rc) return rc;
    rc = build_fused_tiles(c, hb);
    if (rc) return rc;
    rc = build_physical_tables(c, hb);
    if (rc) return rc;
  }
  c->hblocks.assign(blocks, blocks + nblocks);
  c->nblocks = nblocks;
  c->total_pts = off;
  c->total_int = ioff;
  if (elems_per_var) *elems_per_var = off;
  return Z4C_OK;
}

int z4c_prepare_derivatives(z4c_ctx* c, const z4c_params* p, const double* u,
                            double* aux, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u) return fail(Z4C_EINVAL, "prepare_derivatives: null argument");
  return launch_prep(c, p, u, aux, (hipStream_t)stream);
}

int z4c_rhs(z4c_ctx* c, const z4c_params* p, const double* u, const double* mat,
            double* rhs, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !rhs) return fail(Z4C_EINVAL, "rhs: null argument");
  return launch_rhs(c, p, u, mat, rhs, false, (hipStream_t)stream);
}

int z4c_boundary_rhs(z4c_ctx* c, const z4c_params* p, const double* u,
                     double* rhs, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !rhs) return fail(Z4C_EINVAL, "boundary_rhs: null argument");
  RhsArgs a{c->d_blocks, launch_of(c, BOX_INTERIOR), u, nullptr, nullptr, rhs, rhs_params(p)};
  hipLaunchKernelGGL(k_sommerfeld, dim3(grid_for(a.L.ntiles)), dim3(TILE), 0,
                     (hipStream_t)stream, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

int z4c_algconstr(z4c_ctx* c, const z4c_params* p, double* u, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u) return fail(Z4C_EINVAL, "algconstr: null argument");
  return launch_alg(c, p, u, nullptr, 0, (hipStream_t)stream);
}

int z4c_algconstr_range(z4c_ctx* c, const z4c_params* p, double* u, int il,
                        int iu, int jl, int ju, int kl, int ku,
                        int skip_physical, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u) return fail(Z4C_EINVAL, "algconstr_range: null argument");
  if (il < 0 || jl < 0 || kl < 0) return fail(Z4C_EINVAL, "algconstr_range: negative bound");
  const int r[6] = {il, iu, jl, ju, kl, ku};
  return launch_alg(c, p, u, r, skip_physical, (hipStream_t)stream);
}

int z4c_adm_to_z4c(z4c_ctx* c, const z4c_params* p, const double* adm, double* u,
                   double* aux_ext, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !adm || !u) return fail(Z4C_EINVAL, "adm_to_z4c: null argument");
  hipStream_t s = (hipStream_t)stream;
  AdmArgs a{c->d_blocks, launch_of(c, BOX_WHOLE), adm, u, nullptr, aux_ext,
            p->chi_psi_power, p->chi_div_floor};
  const int g = grid_for(a.L.ntiles);
  hipLaunchKernelGGL(k_adm2z4c_point, dim3(g), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  hipLaunchKernelGGL(k_adm2z4c_gamma, dim3(g), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  rc = launch_alg(c, p, u, nullptr, 0, s);
  if (rc) return rc;
  if (aux_ext) {
    hipLaunchKernelGGL(k_aux_ext, dim3(g), dim3(TILE), 0, s, a);
    HIPCALL(hipGetLastError());
  }
  return Z4C_OK;
}

int z4c_z4c_to_adm(z4c_ctx* c, const z4c_params* p, const double* u, double* adm,
                   double* aux_ext, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !adm || !u) return fail(Z4C_EINVAL, "z4c_to_adm: null argument");
  AdmArgs a{c->d_blocks, launch_of(c, BOX_WHOLE), nullptr, const_cast<double*>(u), adm,
            aux_ext, p->chi_psi_power, p->chi_div_floor};
  hipLaunchKernelGGL(k_z4c2adm, dim3(grid_for(a.L.ntiles)), dim3(TILE), 0,
                     (hipStream_t)stream, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

int z4c_adm_constraints(z4c_ctx* c, const z4c_params* p, const double* u,
                        const double* adm, const double* mat, double* con,
                        void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !adm || !con) return fail(Z4C_EINVAL, "adm_constraints: null argument");
  hipStream_t s = (hipStream_t)stream;
  rc = launch_prep(c, p, u, nullptr, s);
  if (rc) return rc;
  rc = fill(c, con, 0.0, c->total_pts * NCON, s);
  if (rc) return rc;
  ConArgs a{c->d_blocks, launch_of(c, BOX_INTERIOR), u, adm, mat, c->d1, con,
            p->chi_psi_power, p->chi_div_floor, p->r_max_con};
  // Two waves a SIMD hide the loads' latency of a full chip (2.03 -> 1.92 ms for
  // 400 uneven blocks, whole call 1531 -> 1458 us for 320 of 16^3) and of workgroups
  // just over one a CU (16 of 16^3: 79 -> 75 us); a single round pays the spills
  // for nothing (one 8^3 or 32^3 block: 34.7 -> 38.2, 41.4 -> 47.4 us), and between
  // two and six rounds neither is better throughout (64 of 16^3: 297 -> 304 us, a
  // 64^3 block: 173 -> 167).
  const int n = a.L.ntiles, cu = c->n_cu;
  const bool two = n >= 6 * cu || (n > cu && n <= cu + cu / 3);
  hipLaunchKernelGGL(two ? k_constraints<2> : k_constraints<1>, dim3(grid_for(n)), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

int z4c_bt_sum(z4c_ctx* c, int nvar, double* u_out, const double* u0, int nk,
               const double* const* k, const double* w, double dt, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!u_out || !u0 || (nk > 0 && (!k || !w)) || nvar <= 0)
    return fail(Z4C_EINVAL, "bt_sum: bad argument");
  return launch_bt(c, nvar, u_out, u0, nk, k, w, dt, (hipStream_t)stream);
}

int z4c_weighted_ave(z4c_ctx* c, int nvar, double* u_out, const double* u_in1,
                     const double* u_in2, const double* wght3, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!u_out || !wght3 || nvar <= 0) return fail(Z4C_EINVAL, "weighted_ave: bad argument");
  if ((wght3[1] != 0.0 && !u_in1) || (wght3[2] != 0.0 && !u_in2))
    return fail(Z4C_EINVAL, "weighted_ave: null input with nonzero weight");
  WaveArgs a{c->d_blocks, launch_of(c, BOX_INTERIOR), nvar, u_out, u_in1, u_in2,
             {wght3[0], wght3[1], wght3[2]}, 0};
  hipLaunchKernelGGL(k_wave, dim3(grid_for(a.L.ntiles)), dim3(TILE), 0, (hipStream_t)stream, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

int z4c_add_rhs(z4c_ctx* c, int nvar, const double* rhs, double wght, double* u_out,
                void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!u_out || !rhs || nvar <= 0) return fail(Z4C_EINVAL, "add_rhs: bad argument");
  WaveArgs a{c->d_blocks, launch_of(c, BOX_INTERIOR), nvar, u_out, rhs, nullptr,
             {wght, 0.0, 0.0}, 1};
  hipLaunchKernelGGL(k_wave, dim3(grid_for(a.L.ntiles)), dim3(TILE), 0, (hipStream_t)stream, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

int z4c_new_dt(z4c_ctx* c, double cfl, double* dt_out) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!dt_out) return fail(Z4C_EINVAL, "new_dt: null output");
  double m = std::numeric_limits<double>::infinity();
  for (const z4c_block& b : c->hblocks) {
    double md = (double)std::numeric_limits<float>::max();
    for (int d = 0; d < 3; ++d) md = std::min(md, b.dx[d]);
    m = std::min(m, md * cfl);
  }
  *dt_out = m;
  return Z4C_OK;
}

int z4c_periodic_fill(z4c_ctx* c, int nvar, double* u, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!u || nvar <= 0) return fail(Z4C_EINVAL, "periodic_fill: bad argument");
  return launch_periodic(c, nvar, u, (hipStream_t)stream);
}

int z4c_history(z4c_ctx* c, const z4c_params* p, const double* u, const double* con,
                double* out, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !con || !out) return fail(Z4C_EINVAL, "history: null argument");
  hipStream_t s = (hipStream_t)stream;
  const Launch L = launch_of(c, BOX_INTERIOR);
  if (!c->hst) {
    if (hipMalloc(&c->hst, sizeof(double) * NHST * (size_t)L.ntiles) != hipSuccess)
      return fail(Z4C_ENOMEM, "history: allocation failed");
    c->hst_host.assign((size_t)NHST * L.ntiles, 0.0);
  }
  const double r = p->r_max_con;
  HstArgs a{c->d_blocks, L, u, con, r * r, c->hst};
  hipLaunchKernelGGL(k_history, dim3(grid_for(L.ntiles)), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  HIPCALL(hipMemcpyAsync(c->hst_host.data(), c->hst, sizeof(double) * NHST * (size_t)L.ntiles,
                         hipMemcpyDeviceToHost, s));
  HIPCALL(hipStreamSynchronize(s));
  for (int q = 0; q < NHST; ++q) out[q] = 0.0;
  for (int t = 0; t < L.ntiles; ++t)
    for (int q = 0; q < NHST; ++q) out[q] += c->hst_host[(size_t)t * NHST + q];
  return Z4C_OK;
}

int z4c_history_noalloc(z4c_ctx* c, const z4c_params* p, const double* u, const double* con,
                        double* out, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !con || !out) return fail(Z4C_EINVAL, "history_noalloc: null argument");
  const Launch L = launch_of(c, BOX_INTERIOR);
  if (L.ntiles > HIST_NOALLOC_MAX_TILES)
    return fail(Z4C_EINVAL, "history_noalloc: the blocks need " + std::to_string(L.ntiles) +
                                " interior tiles, more than the " +
                                std::to_string(HIST_NOALLOC_MAX_TILES) +
                                " its fixed scratch holds; use z4c_history");
  double* part = g_scratch_dev[c->device];
  if (!part) return fail(Z4C_ESTATE, "history_noalloc: scratch not resolved on this device");
  hipStream_t s = (hipStream_t)stream;
  const double r = p->r_max_con;
  HstArgs a{c->d_blocks, L, u, con, r * r, part};
  hipLaunchKernelGGL(k_history, dim3(grid_for(L.ntiles)), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  hipLaunchKernelGGL(k_history_sum, dim3(1), dim3(512), 0, s, (const double*)part, L.ntiles, out);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

namespace {
int build_ml_exchange(z4c_ctx* c, const double* lo, const double* hi, const int* periodic);
}  // namespace

int z4c_set_exchange(z4c_ctx* c, const double* lo, const double* hi, const int* periodic) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!lo || !hi || !periodic) return fail(Z4C_EINVAL, "set_exchange: null argument");
  for (int d = 0; d < 3; ++d)
    if (!(hi[d] > lo[d])) return fail(Z4C_EINVAL, "set_exchange: empty domain");
  c->invalidate_graph();  // a captured step holds the old map
  bool levels = false;
  for (const z4c_block& B : c->hblocks)
    for (int d = 0; d < 3; ++d) levels = levels || B.dx[d] != c->hblocks[0].dx[d];
  if (levels) {
    hipFree(c->ex_dst);
    hipFree(c->ex_off);
    hipFree(c->ex_src);
    c->ex_dst = c->ex_off = c->ex_src = nullptr;
    c->ex_ndst = 0;
    c->drop_ext();
    return build_ml_exchange(c, lo, hi, periodic);
  }
  c->drop_ml();
  const double* h = c->hblocks[0].dx;
  long long Nd[3];
  for (int d = 0; d < 3; ++d) {
    if (!(hi[d] > lo[d])) return fail(Z4C_EINVAL, "set_exchange: empty domain");
    Nd[d] = std::llround((hi[d] - lo[d]) / h[d]);
    if (Nd[d] <= 0 || Nd[d] >= (1LL << 20) ||
        std::fabs((hi[d] - lo[d]) / h[d] - (double)Nd[d]) > 1e-6)
      return fail(Z4C_EINVAL, "set_exchange: domain is not a whole number of cells");
  }
  // lattice origin of every block's interior; one spacing for all blocks
  const int nb = c->nblocks;
  std::vector<std::array<long long, 3>> Lo(nb);
  for (int b = 0; b < nb; ++b) {
    const z4c_block& B = c->hblocks[b];
    const int il[3] = {B.il, B.jl, B.kl};
    for (int d = 0; d < 3; ++d) {
      if (B.dx[d] != h[d])
        return fail(Z4C_EINVAL, "set_exchange: blocks of different spacing: the same-level map "
                                "needs one spacing (levels go through z4c_restrict / "
                                "z4c_prolongate)");
      const double L = (B.x0[d] + il[d] * h[d] - lo[d]) / h[d];
      Lo[b][d] = std::llround(L);
      if (std::fabs(L - (double)Lo[b][d]) > 1e-6)
        return fail(Z4C_EINVAL, "set_exchange: block not aligned with the lattice");
    }
  }
  auto wrap = [&](long long w, int d) {
    return periodic[d] ? ((w % Nd[d]) + Nd[d]) % Nd[d] : w;
  };
  auto key = [&](long long I, long long J, long long K) -> long long {
    const long long off = 1LL << 20;  // non-periodic coordinates may be negative
    return ((I + off) << 42) | ((J + off) << 21) | (K + off);
  };
  // owners: (key, global point id, block, point), sorted by key then id
  struct Own {
    long long key, gid;
    int blk, p;
  };
  std::vector<Own> own;
  for (int b = 0; b < nb; ++b) {
    const z4c_block& B = c->hblocks[b];
    for (int k = B.kl; k <= B.ku; ++k)
      for (int j = B.jl; j <= B.ju; ++j)
        for (int i = B.il; i <= B.iu; ++i) {
          const long long I = wrap(Lo[b][0] + (i - B.il), 0), J = wrap(Lo[b][1] + (j - B.jl), 1),
                          K = wrap(Lo[b][2] + (k - B.kl), 2);
          const int p = i + B.nn1 * (j + B.nn2 * k);
          own.push_back({key(I, J, K), B.offset + p, b, p});
        }
  }
  std::sort(own.begin(), own.end(), [](const Own& x, const Own& y) {
    return x.key != y.key ? x.key < y.key : x.gid < y.gid;
  });
  std::vector<int> dst, off{0}, src;
  for (int b = 0; b < nb; ++b) {
    const z4c_block& B = c->hblocks[b];
    for (int k = 0; k < B.nn3; ++k)
      for (int j = 0; j < B.nn2; ++j)
        for (int i = 0; i < B.nn1; ++i) {
          const long long I = wrap(Lo[b][0] + (i - B.il), 0), J = wrap(Lo[b][1] + (j - B.jl), 1),
                          K = wrap(Lo[b][2] + (k - B.kl), 2);
          const long long kk = key(I, J, K);
          auto lo_it = std::lower_bound(own.begin(), own.end(), kk,
                                        [](const Own& x, long long v) { return x.key < v; });
          auto hi_it = lo_it;
          while (hi_it != own.end() && hi_it->key == kk) ++hi_it;
          const long cnt = hi_it - lo_it;
          const bool interior = i >= B.il && i <= B.iu && j >= B.jl && j <= B.ju &&
                                k >= B.kl && k <= B.ku;
          if (cnt == 0 || (interior && cnt == 1)) continue;
          dst.push_back(b);
          dst.push_back(i + B.nn1 * (j + B.nn2 * k));
          for (auto it = lo_it; it != hi_it; ++it) {
            src.push_back(it->blk);
            src.push_back(it->p);
          }
          if (src.size() / 2 > (size_t)std::numeric_limits<int>::max())
            return fail(Z4C_EINVAL, "set_exchange: map too large");
          off.push_back((int)(src.size() / 2));
        }
  }
  hipFree(c->ex_dst);
  hipFree(c->ex_off);
  hipFree(c->ex_src);
  c->ex_dst = c->ex_off = c->ex_src = nullptr;
  c->ex_ndst = 0;
  c->drop_ext();
  if (dst.empty()) return Z4C_OK;
  if (hipMalloc(&c->ex_dst, sizeof(int) * dst.size()) != hipSuccess ||
      hipMalloc(&c->ex_off, sizeof(int) * off.size()) != hipSuccess ||
      hipMalloc(&c->ex_src, sizeof(int) * src.size()) != hipSuccess)
    return fail(Z4C_ENOMEM, "set_exchange: allocation failed");
  HIPCALL(hipMemcpy(c->ex_dst, dst.data(), sizeof(int) * dst.size(), hipMemcpyHostToDevice));
  HIPCALL(hipMemcpy(c->ex_off, off.data(), sizeof(int) * off.size(), hipMemcpyHostToDevice));
  HIPCALL(hipMemcpy(c->ex_src, src.data(), sizeof(int) * src.size(), hipMemcpyHostToDevice));
  c->ex_ndst = (int)(dst.size() / 2);
  {
    // the transpose: every source vertex with the destinations that read
    // it (in destination order), and the destinations no list reads
    const size_t nd = dst.size() / 2;
    auto vkey = [](int b, int p) { return ((long long)b << 32) | (unsigned)p; };
    std::unordered_map<long long, int> vid;
    std::vector<int> tv;
    std::vector<std::vector<int>> tl;
    for (size_t d = 0; d < nd; ++d)
      for (int e = off[d]; e < off[d + 1]; ++e) {
        const long long k = vkey(src[2 * e], src[2 * e + 1]);
        auto it = vid.find(k);
        int id;
        if (it == vid.end()) {
          id = (int)tl.size();
          vid.emplace(k, id);
          tv.push_back(src[2 * e]);
          tv.push_back(src[2 * e + 1]);
          tl.emplace_back();
        } else {
          id = it->second;
        }
        tl[id].push_back((int)d);
      }
    {
      // renumber the sources in memory order (coalesced scatter)
      const size_t nv = tl.size();
      std::vector<int> order(nv), rank(nv);
      for (size_t q = 0; q < nv; ++q) order[q] = (int)q;
      auto addr = [&](int q) { return c->hdev[tv[2 * q]].off + tv[2 * q + 1]; };
      std::sort(order.begin(), order.end(), [&](int x, int y) { return addr(x) < addr(y); });
      std::vector<int> tv2(2 * nv);
      std::vector<std::vector<int>> tl2(nv);
      for (size_t q = 0; q < nv; ++q) {
        rank[order[q]] = (int)q;
        tv2[2 * q] = tv[2 * order[q]];
        tv2[2 * q + 1] = tv[2 * order[q] + 1];
        tl2[q] = std::move(tl[order[q]]);
      }
      for (auto& kv : vid) kv.second = rank[kv.second];
      tv = std::move(tv2);
      tl = std::move(tl2);
    }
    std::vector<int> tflag(tl.size(), 0), toff{0}, td, tz;
    for (size_t d = 0; d < nd; ++d) {
      auto it = vid.find(vkey(dst[2 * d], dst[2 * d + 1]));
      if (it == vid.end())
        tz.push_back((int)d);
      else
        tflag[it->second] = 1;
    }
    for (auto& l : tl) {
      td.insert(td.end(), l.begin(), l.end());
      toff.push_back((int)td.size());
    }
    auto up = [&](int*& dptr, const std::vector<int>& h) {
      if (h.empty()) return true;
      if (hipMalloc(&dptr, sizeof(int) * h.size()) != hipSuccess) return false;
      return hipMemcpy(dptr, h.data(), sizeof(int) * h.size(), hipMemcpyHostToDevice) == hipSuccess;
    };
    bool ok = up(c->ext_v, tv) && up(c->ext_flag, tflag) && up(c->ext_off, toff) &&
              up(c->ext_d, td) && up(c->ext_z, tz);
    ok = ok && (tl.empty() ||
                hipMalloc(&c->ext_tmp, sizeof(double) * NVAR * tl.size()) == hipSuccess);
    if (!ok) {
      c->drop_ext();
      return fail(Z4C_ENOMEM, "set_exchange: allocation failed");
    }
    c->ext_nv = (int)tl.size();
    c->ext_nz = (int)tz.size();
  }
  // the gather scratch for up to NVAR fields now, so that z4c_exchange
  // allocates nothing (and a step with the exchange can be captured)
  return ensure_snapshot(c, (long long)c->ex_ndst * NVAR);
}

int z4c_exchange(z4c_ctx* c, int nvar, double* u, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!u || nvar <= 0) return fail(Z4C_EINVAL, "exchange: bad argument");
  return launch_exchange(c, nvar, u, (hipStream_t)stream);
}

namespace {

// Coarse-buffer table of the registered blocks (built on first use).
int ensure_coarse(z4c_ctx* c) {
  if (c->d_rf) return Z4C_OK;
  std::vector<RfBlock> hr(c->nblocks);
  std::vector<RfChunk> ch;
  long long off = 0;
  for (int b = 0; b < c->nblocks; ++b) {
    const z4c_block& in = c->hblocks[b];
    const int nx[3] = {in.iu - in.il, in.ju - in.jl, in.ku - in.kl};
    int cn[3], ni[3];
    for (int d = 0; d < 3; ++d) {
      if (nx[d] % 2 != 0)
        return fail(Z4C_EINVAL, "refinement: block " + std::to_string(b) +
                                    " needs an even number of cells per axis");
      cn[d] = nx[d] / 2 + 2 * RF_NCG + 1;
      ni[d] = nx[d] / 2 + 1;
    }
    RfBlock& R = hr[b];
    R.coff = off;
    R.cn1 = cn[0];
    R.cn2 = cn[1];
    R.cn3 = cn[2];
    R.cnpts = cn[0] * cn[1] * cn[2];
    R.cni = ni[0];
    R.cnj = ni[1];
    R.cnk = ni[2];
    off += R.cnpts;
    const int np = ni[0] * ni[1] * ni[2];
    for (int s0 = 0; s0 < np; s0 += 256) ch.push_back(RfChunk{b, s0});
  }
  if (hipMalloc(&c->d_rf, sizeof(RfBlock) * hr.size()) != hipSuccess ||
      hipMalloc(&c->d_rchunks, sizeof(RfChunk) * ch.size()) != hipSuccess) {
    c->drop_refine();
    return fail(Z4C_ENOMEM, "refinement: allocation failed");
  }
  HIPCALL(hipMemcpy(c->d_rf, hr.data(), sizeof(RfBlock) * hr.size(), hipMemcpyHostToDevice));
  HIPCALL(hipMemcpy(c->d_rchunks, ch.data(), sizeof(RfChunk) * ch.size(), hipMemcpyHostToDevice));
  c->n_rchunks = (int)ch.size();
  c->hrf = hr;
  c->rf_total = off;
  return Z4C_OK;
}

// Coarse vertices entry E reads on axis a (injected c, prolongated c - RF_H
// .. c + RF_HSZ); false when the entry writes nothing on that axis.
bool rf_read_range(const RfEntry& E, int a, int& lo, int& hi) {
  lo = std::numeric_limits<int>::max();
  hi = std::numeric_limits<int>::min();
  if (E.s[a] <= E.e[a]) {
    lo = E.s[a];
    hi = E.e[a];
  }
  if (E.sp[a] < E.ep[a]) {
    lo = std::min(lo, E.sp[a] - RF_H);
    hi = std::max(hi, E.ep[a] - 1 + RF_HSZ);
  }
  return lo <= hi;
}

// The prolongation's workgroups: entries split (halving their coarse range
// along the axis of the widest read) until each one's read box fits the
// LDS bound, then packed per block, in order, into groups whose union box
// fits it.  `ent` is reordered to the groups' order; returns the largest box.
int prolong_groups(std::vector<RfEntry>& ent, std::vector<PrGroup>& grp) {
  std::vector<RfEntry> work(ent.rbegin(), ent.rend()), out;
  while (!work.empty()) {
    RfEntry E = work.back();
    work.pop_back();
    int lo[3], hi[3];
    bool any = true;
    for (int d = 0; d < 3; ++d) any = any && rf_read_range(E, d, lo[d], hi[d]);
    if (!any) continue;
    if ((long long)(hi[0] - lo[0] + 1) * (hi[1] - lo[1] + 1) * (hi[2] - lo[2] + 1) <= PR_LDS) {
      out.push_back(E);
      continue;
    }
    int ax = -1, wid = 0;
    for (int d = 0; d < 3; ++d) {
      const int c0 = std::min(E.s[d], E.sp[d]), c1 = std::max(E.e[d], E.ep[d] - 1);
      if (c1 > c0 && hi[d] - lo[d] > wid) {
        ax = d;
        wid = hi[d] - lo[d];
      }
    }
    // a single coarse index per axis reads at most 6^3 vertices, so some
    // axis has a range to halve
    if (ax < 0) return -1;
    const int c0 = std::min(E.s[ax], E.sp[ax]), c1 = std::max(E.e[ax], E.ep[ax] - 1);
    const int cm = (c0 + c1 + 1) / 2;
    RfEntry A = E, Bq = E;
    A.e[ax] = std::min(E.e[ax], cm - 1);
    A.ep[ax] = std::min(E.ep[ax], cm);
    Bq.s[ax] = std::max(E.s[ax], cm);
    Bq.sp[ax] = std::max(E.sp[ax], cm);
    work.push_back(Bq);
    work.push_back(A);
  }
  std::stable_sort(out.begin(), out.end(),
                   [](const RfEntry& x, const RfEntry& y) { return x.blk < y.blk; });
  grp.clear();
  int maxv = 0;
  for (size_t q = 0; q < out.size(); ++q) {
    int lo[3], hi[3];
    for (int d = 0; d < 3; ++d) rf_read_range(out[q], d, lo[d], hi[d]);
    if (!grp.empty() && grp.back().blk == out[q].blk) {
      PrGroup& G = grp.back();
      int ulo[3], uhi[3];
      long long v = 1;
      for (int d = 0; d < 3; ++d) {
        ulo[d] = std::min(lo[d], G.r0[d]);
        uhi[d] = std::max(hi[d], G.r0[d] + G.rn[d] - 1);
        v *= uhi[d] - ulo[d] + 1;
      }
      if (v <= PR_LDS) {
        for (int d = 0; d < 3; ++d) {
          G.r0[d] = ulo[d];
          G.rn[d] = uhi[d] - ulo[d] + 1;
        }
        ++G.ne;
        maxv = std::max(maxv, (int)v);
        continue;
      }
    }
    PrGroup G{out[q].blk, (int)q, 1, {lo[0], lo[1], lo[2]},
              {hi[0] - lo[0] + 1, hi[1] - lo[1] + 1, hi[2] - lo[2] + 1}};
    grp.push_back(G);
    maxv = std::max(maxv, G.rn[0] * G.rn[1] * G.rn[2]);
  }
  ent.swap(out);
  return maxv;
}

// One prolongation box checked against the block's fine and coarse extents:
// every coarse vertex the 6-point stencils read and every fine vertex the
// box writes must lie in the buffers.
int make_entry(const z4c_ctx* c, const z4c_prolong_box& in, int q, RfEntry& E) {
  const std::string who = "set_prolongation: box " + std::to_string(q);
  if (in.block < 0 || in.block >= c->nblocks) return fail(Z4C_EINVAL, who + ": bad block index");
  const z4c_block& B = c->hblocks[in.block];
  const RfBlock& R = c->hrf[in.block];
  const int s[3] = {in.si, in.sj, in.sk}, e[3] = {in.ei, in.ej, in.ek};
  const int cn[3] = {R.cn1, R.cn2, R.cn3}, nn[3] = {B.nn1, B.nn2, B.nn3};
  const int cni[3] = {R.cni, R.cnj, R.cnk};
  E.blk = in.block;
  for (int a = 0; a < 3; ++a) {
    const int cmp = RF_NCG + (cni[a] - 1) / 2;  // coarse midpoint cimp
    if (s[a] > e[a]) return fail(Z4C_EINVAL, who + ": empty range");
    const int sp = s[a] > cmp ? s[a] - 1 : s[a], ep = e[a] < cmp ? e[a] + 1 : e[a];
    int rlo = s[a], rhi = e[a];            // coarse vertices read
    int flo = 2 * (s[a] - RF_H), fhi = 2 * (e[a] - RF_H);  // fine vertices written
    if (sp < ep) {
      rlo = std::min(rlo, sp - RF_H);
      rhi = std::max(rhi, ep - 1 + RF_HSZ);
      flo = std::min(flo, 2 * (sp - RF_H) + 1);
      fhi = std::max(fhi, 2 * (ep - 1 - RF_H) + 1);
    }
    if (rlo < 0 || rhi >= cn[a] || flo < 0 || fhi >= nn[a])
      return fail(Z4C_EINVAL, who + ": range leaves the coarse or fine buffer");
    E.s[a] = s[a];
    E.e[a] = e[a];
    E.sp[a] = sp;
    E.ep[a] = ep;
  }
  return Z4C_OK;
}

// The ghost update across refinement levels (z4c_mesh.hpp): block tree,
// neighbour lists, gather lists and prolongation boxes, uploaded with the
// context's coarse buffers and gather scratch (so that an exchange
// allocates nothing and can be captured).
int build_ml_exchange(z4c_ctx* c, const double* lo, const double* hi, const int* periodic) {
  c->drop_ml();
  std::vector<z4c_mesh::Geo> geo(c->nblocks);
  for (int b = 0; b < c->nblocks; ++b) {
    const z4c_block& B = c->hblocks[b];
    const int il[3] = {B.il, B.jl, B.kl}, iu[3] = {B.iu, B.ju, B.ku};
    for (int d = 0; d < 3; ++d) {
      geo[b].nx[d] = iu[d] - il[d];
      geo[b].dx[d] = B.dx[d];
      geo[b].xmin[d] = B.x0[d] + il[d] * B.dx[d];
    }
    if (B.il != z4c_mesh::MNG || B.jl != z4c_mesh::MNG || B.kl != z4c_mesh::MNG)
      return fail(Z4C_EINVAL, "set_exchange: blocks need 4 ghost layers");
  }
  z4c_mesh::Tree t;
  std::string e = t.build(geo, lo, hi, periodic);
  if (!e.empty()) return fail(Z4C_EINVAL, "set_exchange: " + e);
  z4c_mesh::Plan P;
  e = z4c_mesh::build_plan(t, P);
  if (!e.empty()) return fail(Z4C_EINVAL, "set_exchange: " + e);
  // a block that prolongates next to an open face fills its coarse ghosts
  // there with the physical fill first (ApplyPhysicalBCsOnCoarseLevel): the
  // face must carry one (z4c_block.sommerfeld_faces | outflow_faces)
  for (int b = 0; b < t.n; ++b) {
    if (!P.prolongates[b]) continue;
    const int pf = c->hblocks[b].sommerfeld_faces | c->hblocks[b].outflow_faces;
    for (int d = 0; d < 3; ++d) {
      if (t.periodic[d]) continue;
      const long long m = t.nrb0[d] << t.level[b];
      if ((t.loc[b][d] == 0 && !(pf & (1 << (2 * d)))) ||
          (t.loc[b][d] == m - 1 && !(pf & (2 << (2 * d)))))
        return fail(Z4C_EINVAL, "set_exchange: block " + std::to_string(b) +
                                    " has a coarser neighbour and an open face without a "
                                    "physical boundary condition");
    }
  }
  int rc = ensure_coarse(c);
  if (rc) return rc;
  std::vector<RfEntry> ent(P.boxes.size());
  for (size_t q = 0; q < P.boxes.size(); ++q) {
    const auto& bx = P.boxes[q];
    z4c_prolong_box box{bx[0], bx[1], bx[2], bx[3], bx[4], bx[5], bx[6]};
    rc = make_entry(c, box, (int)q, ent[q]);
    if (rc) return rc;
  }
  std::vector<PrGroup> grp;
  const int prlds = prolong_groups(ent, grp);
  if (prlds < 0) return fail(Z4C_EINVAL, "set_exchange: prolongation box too large");
  const size_t nd = P.dst.size(), ns = P.src.size();
  if (nd > (size_t)std::numeric_limits<int>::max() / NVAR)
    return fail(Z4C_EINVAL, "set_exchange: plan too large");
  auto up = [&](auto*& d, const auto* h, size_t n) {
    using T = std::remove_pointer_t<std::remove_reference_t<decltype(d)>>;
    if (n == 0) return true;
    if (hipMalloc(&d, sizeof(T) * n) != hipSuccess) return false;
    return hipMemcpy(d, h, sizeof(T) * n, hipMemcpyHostToDevice) == hipSuccess;
  };
  static_assert(sizeof(z4c_mesh::Ref) == 2 * sizeof(int), "Ref is two ints");
  bool ok = up(c->ml_dst, reinterpret_cast<const int*>(P.dst.data()), 2 * nd) &&
            up(c->ml_off, P.off.data(), P.off.size()) &&
            up(c->ml_src, reinterpret_cast<const int*>(P.src.data()), 2 * ns) &&
            up(c->ml_inv, P.inv.data(), nd) && up(c->ml_pent, ent.data(), ent.size()) &&
            up(c->ml_pgroups, grp.data(), grp.size());
  ok = ok && hipMalloc(&c->ml_coarse, sizeof(double) * NVAR * (size_t)c->rf_total) == hipSuccess;
  ok = ok && (P.n_interior == 0 ||
               hipMalloc(&c->ml_tmp, sizeof(double) * NVAR * (size_t)P.n_interior) == hipSuccess);
  if (!ok) {
    c->drop_ml();
    return fail(Z4C_ENOMEM, "set_exchange: allocation failed");
  }
  // line tables of the coarse level's physical fill (blocks that prolongate)
  for (int ax = 0; ax < 3; ++ax) {
    std::vector<PhysLine> lt;
    long long start = 0;
    for (int b = 0; b < t.n; ++b) {
      const int pf = c->hblocks[b].sommerfeld_faces | c->hblocks[b].outflow_faces;
      if (!P.prolongates[b] || !(pf & (3 << (2 * ax)))) continue;
      const RfBlock& R = c->hrf[b];
      const int is = RF_NCG, ie = RF_NCG + R.cni - 1, js = RF_NCG, je = RF_NCG + R.cnj - 1,
                ks = RF_NCG, ke = RF_NCG + R.cnk - 1;
      const int bis = is - RF_NCG, bie = ie + RF_NCG;
      const int bjs = (pf & 4) ? js : js - RF_NCG, bje = (pf & 8) ? je : je + RF_NCG;
      const int bks = (pf & 16) ? ks : ks - RF_NCG, bke = (pf & 32) ? ke : ke + RF_NCG;
      PhysLine e{};
      e.block = b;
      if (ax == 0) { e.lo0 = bjs; e.n0 = bje - bjs + 1; e.lo1 = bks; e.n1 = bke - bks + 1; }
      else if (ax == 1) { e.lo0 = bis; e.n0 = bie - bis + 1; e.lo1 = bks; e.n1 = bke - bks + 1; }
      else { e.lo0 = bis; e.n0 = bie - bis + 1; e.lo1 = js - RF_NCG; e.n1 = je - js + 1 + 2 * RF_NCG; }
      e.start = start;
      start += (long long)e.n0 * e.n1;
      lt.push_back(e);
    }
    c->mlp_nent[ax] = (int)lt.size();
    c->mlp_nlines1[ax] = start;
    if (!lt.empty() && !up(c->mlp_lines[ax], lt.data(), lt.size())) {
      c->drop_ml();
      return fail(Z4C_ENOMEM, "set_exchange: allocation failed");
    }
  }
  c->ml_ndst = (int)nd;
  c->ml_nint = (int)P.n_interior;
  c->ml_npgroups = (int)grp.size();
  c->ml_prlds = prlds;
  c->ml_nent = (int)ent.size();
  c->ml_nbrs = t.nbrs;
  c->ml_level = t.level;
  c->ml = true;
  return Z4C_OK;
}

}  // namespace

int z4c_coarse_layout(z4c_ctx* c, long long* offsets, long long* elems_per_var) {
  int rc = check_ctx(c);
  if (rc) return rc;
  rc = ensure_coarse(c);
  if (rc) return rc;
  if (offsets)
    for (int b = 0; b < c->nblocks; ++b) offsets[b] = c->hrf[b].coff;
  if (elems_per_var) *elems_per_var = c->rf_total;
  return Z4C_OK;
}

int z4c_restrict(z4c_ctx* c, int nvar, const double* u, double* coarse, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!u || !coarse || nvar <= 0) return fail(Z4C_EINVAL, "restrict: bad argument");
  rc = ensure_coarse(c);
  if (rc) return rc;
  RestrictArgs a{c->d_blocks, c->d_rf, c->d_rchunks, nvar, u, coarse};
  hipLaunchKernelGGL(k_restrict_vc, dim3(c->n_rchunks), dim3(256), 0, (hipStream_t)stream, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

int z4c_prolongation_range(z4c_ctx* c, int block, const int* ox, const long long* lx,
                           z4c_prolong_box* box) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!ox || !lx || !box || block < 0 || block >= c->nblocks)
    return fail(Z4C_EINVAL, "prolongation_range: bad argument");
  rc = ensure_coarse(c);
  if (rc) return rc;
  const RfBlock& R = c->hrf[block];
  const int cni[3] = {R.cni, R.cnj, R.cnk};
  const int pcng = NG / 2;
  int* se[3][2] = {{&box->si, &box->ei}, {&box->sj, &box->ej}, {&box->sk, &box->ek}};
  for (int a = 0; a < 3; ++a) {
    if (ox[a] < -1 || ox[a] > 1) return fail(Z4C_EINVAL, "prolongation_range: offset not in -1..1");
    const int cvs = RF_NCG, cve = RF_NCG + cni[a] - 1;
    int s, e;
    if (ox[a] > 0) {
      s = cve + 1;
      e = cve + pcng;
    } else if (ox[a] < 0) {
      s = cvs - pcng;
      e = cvs - 1;
    } else {
      s = cvs;
      e = cve;
      if ((lx[a] & 1LL) == 0)
        e += pcng;
      else
        s -= pcng;
    }
    *se[a][0] = s;
    *se[a][1] = e;
  }
  box->block = block;
  return Z4C_OK;
}

int z4c_set_prolongation(z4c_ctx* c, const z4c_prolong_box* boxes, int nbox) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (nbox < 0 || (nbox > 0 && !boxes)) return fail(Z4C_EINVAL, "set_prolongation: bad argument");
  rc = ensure_coarse(c);
  if (rc) return rc;
  std::vector<RfEntry> ent(nbox);
  for (int q = 0; q < nbox; ++q) {
    rc = make_entry(c, boxes[q], q, ent[q]);
    if (rc) return rc;
  }
  std::vector<PrGroup> grp;
  const int prlds = prolong_groups(ent, grp);
  if (prlds < 0) return fail(Z4C_EINVAL, "set_prolongation: box too large");
  if (ent.size() > (size_t)std::numeric_limits<int>::max() ||
      grp.size() > (size_t)std::numeric_limits<int>::max())
    return fail(Z4C_EINVAL, "set_prolongation: too many boxes");
  c->drop_prolongation();
  if (grp.empty()) return Z4C_OK;
  if (hipMalloc(&c->d_pent, sizeof(RfEntry) * ent.size()) != hipSuccess ||
      hipMalloc(&c->d_pgroups, sizeof(PrGroup) * grp.size()) != hipSuccess) {
    c->drop_prolongation();
    return fail(Z4C_ENOMEM, "set_prolongation: allocation failed");
  }
  HIPCALL(hipMemcpy(c->d_pent, ent.data(), sizeof(RfEntry) * ent.size(), hipMemcpyHostToDevice));
  HIPCALL(hipMemcpy(c->d_pgroups, grp.data(), sizeof(PrGroup) * grp.size(), hipMemcpyHostToDevice));
  c->n_pgroups = (int)grp.size();
  c->pr_lds = prlds;
  return Z4C_OK;
}

int z4c_prolongate(z4c_ctx* c, int nvar, const double* coarse, double* u, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!u || !coarse || nvar <= 0) return fail(Z4C_EINVAL, "prolongate: bad argument");
  if (!c->n_pgroups) return Z4C_OK;
  if (nvar > 65535) return fail(Z4C_EINVAL, "prolongate: too many fields");
  ProlongArgs a{c->d_blocks, c->d_rf, c->d_pent, c->d_pgroups, coarse, u, nvar};
  hipLaunchKernelGGL(k_prolong_vc, dim3(c->n_pgroups, nvar), dim3(256), sizeof(double) * c->pr_lds,
                     (hipStream_t)stream, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

int z4c_physical_bc(z4c_ctx* c, int nvar, double* u, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!u || nvar <= 0) return fail(Z4C_EINVAL, "physical_bc: bad argument");
  return launch_physical(c, nvar, u, (hipStream_t)stream);
}

int z4c_autotune(z4c_ctx* c, const z4c_params* p, const double* u, int reps, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || reps < 1) return fail(Z4C_EINVAL, "autotune: bad argument");
  const bool had_slots = c->dv != nullptr;
  rc = ensure_slots(c);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  std::map<std::array<int, 3>, std::vector<int>> classes;
  for (int b = 0; b < c->nblocks; ++b)
    classes[{c->hdev[b].ni, c->hdev[b].nj, c->hdev[b].nk}].push_back(b);
  hipEvent_t e0, e1;
  HIPCALL(hipEventCreate(&e0));
  HIPCALL(hipEventCreate(&e1));
  PlaneTile* d = nullptr;
  rc = Z4C_OK;
  for (auto& cl : classes) {
    int best = -1;
    float best_ms = 0.f;
    for (int q = 0; q < NSTCFG && rc == Z4C_OK; ++q) {
      std::vector<PlaneTile> tl;
      bool ok = true;
      for (int b : cl.second) ok = ok && plane_tiles(q, b, c->hdev[b].ni, c->hdev[b].nj, &tl);
      if (!ok || tl.empty()) continue;
      if (hipMalloc(&d, sizeof(PlaneTile) * tl.size()) != hipSuccess) {
        rc = fail(Z4C_ENOMEM, "autotune: allocation failed");
        break;
      }
      if (hipMemcpy(d, tl.data(), sizeof(PlaneTile) * tl.size(), hipMemcpyHostToDevice) !=
          hipSuccess) {
        rc = fail(Z4C_EHIP, "autotune: copy failed");
        break;
      }
      StencilArgs sa{c->d_blocks, d, (int)tl.size(), u, c->dv, p->diss, p->lapse_advect,
                     p->shift_advect};
      launch_stencil_cfg(q, sa, s);  // warm-up
      hipEventRecord(e0, s);
      for (int r = 0; r < reps; ++r) launch_stencil_cfg(q, sa, s);
      hipEventRecord(e1, s);
      float ms = 0.f;
      if (hipGetLastError() != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
          hipEventElapsedTime(&ms, e0, e1) != hipSuccess) {
        rc = fail(Z4C_EHIP, "autotune: timing failed");
        break;
      }
      hipFree(d);
      d = nullptr;
      if (best < 0 || ms < best_ms) {
        best = q;
        best_ms = ms;
      }
    }
    if (rc) break;
    if (best >= 0)
      for (int b : cl.second) c->blk_cfg[b] = best;
  }
  hipFree(d);
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  if (!had_slots) {  // no right-hand side of the context needed them so far
    hipFree(c->dv);
    c->dv = nullptr;
  }
  if (rc) return rc;
  return build_stencil_plan(c, c->hdev);
}

int z4c_set_stencil_threads(z4c_ctx* c, int block, int threads) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (block < -1 || block >= c->nblocks) return fail(Z4C_EINVAL, "set_stencil_threads: bad block");
  int q = -1;
  for (int k = 0; k < NSTCFG; ++k)
    if (ST_THREADS_OF[k] == threads) q = k;
  if (q < 0) return fail(Z4C_EINVAL, "set_stencil_threads: threads must be 192, 256, 320, 384, 576 or 640");
  const int b0 = block < 0 ? 0 : block, b1 = block < 0 ? c->nblocks : block + 1;
  for (int b = b0; b < b1; ++b)
    if (!plane_tiles(q, b, c->hdev[b].ni, c->hdev[b].nj, nullptr))
      return fail(Z4C_EINVAL, "set_stencil_threads: no tile of that size fits block " +
                                  std::to_string(b));
  for (int b = b0; b < b1; ++b) c->blk_cfg[b] = q;
  return build_stencil_plan(c, c->hdev);
}

int z4c_set_rhs_form(z4c_ctx* c, int form) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (form < Z4C_FORM_AUTO || form > Z4C_FORM_TWO_PASSES)
    return fail(Z4C_EINVAL, "set_rhs_form: unknown form");
  if (form == Z4C_FORM_TWO_PASSES) {
    rc = ensure_slots(c);
    if (rc) return rc;
  }
  c->invalidate_graph();
  c->form = form;
  return Z4C_OK;
}

int z4c_rhs_form(z4c_ctx* c, int* rhs, int* step) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!rhs || !step) return fail(Z4C_EINVAL, "rhs_form: null argument");
  *rhs = rhs_two(c) ? Z4C_FORM_TWO_PASSES : Z4C_FORM_ONE_KERNEL;
  *step = step_two(c) ? Z4C_FORM_TWO_PASSES : Z4C_FORM_ONE_KERNEL;
  return Z4C_OK;
}

int z4c_stencil_threads(z4c_ctx* c, int block, int* threads) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!threads || block < 0 || block >= c->nblocks)
    return fail(Z4C_EINVAL, "stencil_threads: bad argument");
  *threads = ST_THREADS_OF[c->blk_cfg[block]];
  return Z4C_OK;
}

int z4c_set_timing(z4c_ctx* c, int enable) {
  if (!c) return fail(Z4C_EINVAL, "set_timing: null context");
  c->timing = enable != 0;
  return Z4C_OK;
}

int z4c_get_timing(z4c_ctx* c, double* ms_total, long long* launches, int npass) {
  if (!c || !ms_total || !launches || npass < 0) return fail(Z4C_EINVAL, "get_timing: bad argument");
  HIPCALL(hipSetDevice(c->device));
  for (int q = 0; q < npass; ++q) {
    ms_total[q] = 0.0;
    launches[q] = 0;
  }
  int rc = Z4C_OK;
  for (auto& t : c->tev) {
    float ms = 0.f;
    if (hipEventSynchronize(t.b) != hipSuccess || hipEventElapsedTime(&ms, t.a, t.b) != hipSuccess) {
      rc = fail(Z4C_EHIP, "get_timing: event query failed");
      break;
    }
    if (t.pass >= 0 && t.pass < npass) {
      ms_total[t.pass] += t.part * ms;
      launches[t.pass] += 1;
    }
  }
  c->drop_timing();
  return rc;
}

}  // extern "C"

namespace {
int ghost_update(z4c_ctx* c, double* u, int ghosts, hipStream_t s) {
  int rc = Z4C_OK;
  if (ghosts & 1)
    rc = launch_periodic(c, NVAR, u, s);
  else if (ghosts & 2)
    rc = launch_exchange(c, NVAR, u, s);
  if (!rc && (ghosts & 4)) rc = launch_physical(c, NVAR, u, s);
  return rc;
}

// Whether the ghost update writes every ghost vertex from interior ones, so
// that no ghost of the state before it is read: across levels (zero, then the
// contributions), the exchange if every ghost has an owner, the periodic fill
// of blocks that hold their images.
bool update_fills_ghosts(const z4c_ctx* c, int ghosts) {
  if (ghosts & 2) return c->ml || c->ext_nz == c->total_pts - c->total_int;
  return (ghosts & 1) && !c->per_snap;
}

// ghosts: 0 holds the ghosts at u_n (AlgConstr(u_n), formed once); else the
// ghost update of z4c_rk4_stage after every stage (1 single-block periodic
// fill or 2 the exchange, plus 4 the physical fill), on the stage state whose
// ghosts SumBT resets to u_n, then AlgConstr of the whole block.
int launch_rk4_step(z4c_ctx* c, const z4c_params* p, double dt, double* u, double* work,
                    const double* mat, int ghosts, hipStream_t s) {
  int rc = Z4C_OK;
  const long long n = c->total_pts * NVAR;
  double* W0 = work;
  double* W1 = work + n;
  double* ACC = work + 2 * n;
  // bt_rk4 (task_list_integrators_butcher.cpp:37-49): subdiagonal of A and b
  static const double Asub[4] = {0.5, 0.5, 1.0, 0.0};
  static const double Bw[4] = {1. / 6., 1. / 3., 1. / 3., 1. / 6.};
  // In one kernel every stage reads its neighbours' vertices, so no stage
  // overwrites its input.  With ghosts held at u_n the states alternate between
  // W0 and u (u_n is kept interior-indexed in W1), and both hold the ghosts
  // AlgConstr(u_n) once stage 1 has read u_n's.  With a ghost update the
  // first three states alternate between W0 and W1, and u keeps u_n and its
  // ghosts until the last stage.  In two passes without Sommerfeld faces every
  // stage state overwrites u's interior (u_n is kept in W1 as well), and a ghost
  // update finds u_n's ghosts in W0.
  const bool two = p->cowling || with_slots(c, step_two(c));
  const bool inplace = two && !c->faces;
  const bool held = !ghosts || inplace;  // u_n kept in W1, not in u
  double* const outs[4] = {inplace ? u : W0, held ? u : W1, inplace ? u : W0, u};
  const bool all_ghosts = update_fills_ghosts(c, ghosts);
  auto copy_ghosts = [&](double* from, double* to) {
    GhostArgs gc{c->d_blocks, launch_of(c, BOX_GHOST), from, to,
                 p->eps_floor, p->tf_force_regularization, p->force_regularization};
    PassTimer t(c, Z4C_PASS_GHOSTS, s);
    hipLaunchKernelGGL(k_ghost_copy, dim3(grid_for(gc.L.ntiles)), dim3(TILE), 0, s, gc);
    HIPCALL(hipGetLastError());
    return (int)Z4C_OK;
  };
  if (ghosts && inplace && !all_ghosts) {
    rc = copy_ghosts(u, W0);
    if (rc) return rc;
  }
  for (int st = 1; st <= 4; ++st) {
    FusedArgs a{};
    a.u = st == 1 ? u : outs[st - 2];
    a.mat = mat;
    a.o = rhs_params(p);
    a.sommerfeld = 1;
    a.un = (held && st > 1) ? W1 : u;
    a.un_int = held && st > 1;
    a.acc = ACC;
    a.out = outs[st - 1];
    a.keep = (held && st == 1) ? W1 : nullptr;
    a.wa = Asub[st - 1] * dt;
    a.wb = Bw[st - 1] * dt;
    a.stage = st;
    a.cowling = p->cowling;
    a.alg = !ghosts;
    a.eps_floor = p->eps_floor;
    a.tf_force = p->tf_force_regularization;
    a.force_reg = p->force_regularization;
    rc = launch_stage(c, p, two, a, s);
    if (rc) return rc;
    if (ghosts) {
      // SumBT's ghost values (u_n) into the stage state, then the ghost
      // update and AlgConstr of the whole block (z4c_rk4_stage's order)
      double* cur = a.out;
      if (!all_ghosts && (inplace ? st > 1 : cur != u)) {
        rc = copy_ghosts(inplace ? W0 : u, cur);
        if (rc) return rc;
      }
      rc = ghost_update(c, cur, ghosts, s);
      if (!rc) rc = launch_alg(c, p, cur, nullptr, 0, s);
      if (rc) return rc;
    } else if (st == 1) {
      GhostArgs ga{c->d_blocks, launch_of(c, BOX_GHOST), u, W0, p->eps_floor,
                   p->tf_force_regularization, p->force_regularization};
      PassTimer t(c, Z4C_PASS_GHOSTS, s);
      if (inplace)
        hipLaunchKernelGGL(k_rk4_ghosts_inplace, dim3(grid_for(ga.L.ntiles)), dim3(TILE), 0, s, ga);
      else
        hipLaunchKernelGGL(k_rk4_ghosts, dim3(grid_for(ga.L.ntiles)), dim3(TILE), 0, s, ga);
      HIPCALL(hipGetLastError());
    }
  }
  return Z4C_OK;
}

int launch_wave(z4c_ctx* c, double* out, const double* in1, const double* in2, double w0,
                double w1, double w2, int mode, hipStream_t s) {
  WaveArgs a{c->d_blocks, launch_of(c, BOX_INTERIOR), NVAR, out, in1, in2, {w0, w1, w2}, mode};
  hipLaunchKernelGGL(k_wave, dim3(grid_for(a.L.ntiles)), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

int check_ls(const z4c_ls_tableau* t, bool need_2s, const char* what) {
  if (!t || t->nstages < 1 || t->nstages > Z4C_LS_MAX_STAGES)
    return fail(Z4C_EINVAL, std::string(what) + ": bad tableau");
  if (need_2s)
    for (int q = 0; q < t->nstages; ++q)
      if (t->gamma_3[q] != 0.0)
        return fail(Z4C_EINVAL, std::string(what) + ": 3S* stages (gamma_3 != 0) need u2; "
                                "use z4c_ls_stage");
  return Z4C_OK;
}

// Fused low-storage step.  In one kernel a stage reads its neighbours'
// vertices, so the stage states alternate between u and the second work
// register W; an odd number of stages ends with the interior copied from W.  In
// two passes without Sommerfeld faces every stage overwrites u's interior.  u1
// lives interior-indexed in work.  A stage's output receives its input's ghosts
// where the ghost update does not write them all; with held ghosts it receives
// AlgConstr of them (the update leaves ghosts alone; AlgConstr of the whole block
// reaches them after every stage), in one pass.
int launch_ls_step(z4c_ctx* c, const z4c_params* p, const z4c_ls_tableau* T, double dt,
                   double* u, double* work, const double* mat, int ghosts, hipStream_t s) {
  double* U1 = work;
  double* W = work + c->total_pts * NVAR;
  const bool all_ghosts = update_fills_ghosts(c, ghosts);
  // In two passes without faces the interior copy (0.03 us per 256 vertices) and
  // the ghost copies (0.026 us) fall away: a stage's share of them counts against
  // the one kernel.
  const int odd = T->nstages & 1;
  double extra = 0.0;
  if (!c->faces) {
    extra = odd * 0.03 * c->ntiles[BOX_INTERIOR];
    if (ghosts && !all_ghosts) extra += (T->nstages - odd) * 0.026 * c->ntiles[BOX_GHOST];
    extra /= T->nstages;
  }
  const bool two = p->cowling || with_slots(c, step_two(c, extra));
  const bool inplace = two && !c->faces;
  double* cur = u;
  int rc = Z4C_OK;
  for (int st = 1; st <= T->nstages; ++st) {
    double* nxt = inplace || cur == W ? u : W;
    FusedArgs a{};
    a.u = cur;
    a.mat = mat;
    a.o = rhs_params(p);
    a.sommerfeld = 1;
    a.acc = U1;
    a.out = nxt;
    a.stage = st;
    a.cowling = p->cowling;
    a.alg = !ghosts;
    a.eps_floor = p->eps_floor;
    a.tf_force = p->tf_force_regularization;
    a.force_reg = p->force_regularization;
    a.ls = 1;
    a.ls_w[0] = T->delta[st - 1];
    a.ls_w[1] = T->gamma_1[st - 1];
    a.ls_w[2] = T->gamma_2[st - 1];
    a.ls_w[3] = T->beta[st - 1] * dt;  // dt_scaled (time_integrators.hpp:37-40)
    a.ls_last = st == T->nstages;
    rc = launch_stage(c, p, two, a, s);
    if (rc) return rc;
    GhostArgs ga{c->d_blocks, launch_of(c, BOX_GHOST), cur, nxt, p->eps_floor,
                 p->tf_force_regularization, p->force_regularization};
    const dim3 gg(grid_for(ga.L.ntiles));
    if (st == T->nstages && nxt == W) {
      // u's ghosts are the ones this stage read
      const CopyArgs ca{c->d_blocks, launch_of(c, BOX_INTERIOR), W, u};
      hipLaunchKernelGGL(k_copy_interior, dim3(grid_for(ca.L.ntiles)), dim3(TILE), 0, s, ca);
      HIPCALL(hipGetLastError());
      nxt = u;
    }
    if (!ghosts) {
      PassTimer t(c, Z4C_PASS_GHOSTS, s);
      if (cur == nxt)
        hipLaunchKernelGGL(k_rk4_ghosts_inplace, gg, dim3(TILE), 0, s, ga);
      else if (st == 1)
        hipLaunchKernelGGL(k_ls_ghosts<true>, gg, dim3(TILE), 0, s, ga);
      else
        hipLaunchKernelGGL(k_ls_ghosts<false>, gg, dim3(TILE), 0, s, ga);
      HIPCALL(hipGetLastError());
    } else {
      if (cur != nxt && !all_ghosts) {
        PassTimer t(c, Z4C_PASS_GHOSTS, s);
        hipLaunchKernelGGL(k_ghost_copy, gg, dim3(TILE), 0, s, ga);
        HIPCALL(hipGetLastError());
      }
      rc = ghost_update(c, nxt, ghosts, s);
      if (!rc) rc = launch_alg(c, p, nxt, nullptr, 0, s);
      if (rc) return rc;
    }
    cur = nxt;
  }
  return Z4C_OK;
}

}  // namespace

extern "C" {

int z4c_rk4_step(z4c_ctx* c, const z4c_params* p, double dt, double* u, double* work,
                 const double* mat, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !work) return fail(Z4C_EINVAL, "rk4_step: bad argument");
  return launch_rk4_step(c, p, dt, u, work, mat, 0, (hipStream_t)stream);
}

int z4c_rk4_step_ghosts(z4c_ctx* c, const z4c_params* p, double dt, double* u, double* work,
                        const double* mat, int ghosts, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !work || ghosts < 0 || ghosts > 7 || (ghosts & 3) == 3)
    return fail(Z4C_EINVAL, "rk4_step_ghosts: bad argument");
  return launch_rk4_step(c, p, dt, u, work, mat, ghosts, (hipStream_t)stream);
}

namespace {
// The fused step (ghost update `ghosts` after every stage, 0 = ghosts held
// at u_n) replayed from a HIP graph captured once per (u, work, dt,
// parameters, ghosts).  Scratch the update needs is allocated before the
// capture, so the graph holds kernel nodes only.
int step_graph(z4c_ctx* c, const z4c_params* p, double dt, double* u, double* work, int ghosts,
               hipStream_t s, const char* who) {
  if (c->timing) return fail(Z4C_ESTATE, std::string(who) + ": the kernel timer cannot be captured");
  const bool same = c->graph_exec && c->g_u == u && c->g_work == work && c->g_dt == dt &&
                    c->g_ghosts == ghosts &&
                    std::memcmp(&c->g_params, p, sizeof(z4c_params)) == 0;
  if (!same) {
    c->invalidate_graph();
    if ((ghosts & 1) && c->per_snap) {
      const int rc0 = ensure_snapshot(c, c->total_pts * NVAR);
      if (rc0) return rc0;
    }
    if (!c->cap_stream) HIPCALL(hipStreamCreateWithFlags(&c->cap_stream, hipStreamNonBlocking));
    HIPCALL(hipStreamBeginCapture(c->cap_stream, hipStreamCaptureModeThreadLocal));
    int rc = launch_rk4_step(c, p, dt, u, work, nullptr, ghosts, c->cap_stream);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(c->cap_stream, &g);
    if (rc) {
      if (g) hipGraphDestroy(g);
      return rc;
    }
    if (e != hipSuccess || !g) return fail(Z4C_EHIP, std::string(who) + ": capture failed");
    const hipError_t ei = hipGraphInstantiate(&c->graph_exec, g, nullptr, nullptr, 0);
    hipGraphDestroy(g);
    if (ei != hipSuccess) {
      c->graph_exec = nullptr;
      return fail(Z4C_EHIP, std::string(who) + ": instantiation failed");
    }
    c->g_u = u;
    c->g_work = work;
    c->g_dt = dt;
    c->g_ghosts = ghosts;
    c->g_params = *p;
  }
  HIPCALL(hipGraphLaunch(c->graph_exec, s));
  return Z4C_OK;
}
}  // namespace

int z4c_rk4_step_graph(z4c_ctx* c, const z4c_params* p, double dt, double* u, double* work,
                       void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !work) return fail(Z4C_EINVAL, "rk4_step_graph: bad argument");
  return step_graph(c, p, dt, u, work, 0, (hipStream_t)stream, "rk4_step_graph");
}

int z4c_rk4_step_ghosts_graph(z4c_ctx* c, const z4c_params* p, double dt, double* u,
                              double* work, int ghosts, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !work || ghosts < 0 || ghosts > 6 || (ghosts & 3) == 3)
    return fail(Z4C_EINVAL, "rk4_step_ghosts_graph: bad argument");
  return step_graph(c, p, dt, u, work, ghosts, (hipStream_t)stream, "rk4_step_ghosts_graph");
}

int z4c_rk4_stage(z4c_ctx* c, const z4c_params* p, int stage, double dt, double* u,
                  const double* un, double* const* k, const double* mat,
                  int periodic, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !un || !k || stage < 1 || stage > 4)
    return fail(Z4C_EINVAL, "rk4_stage: bad argument");
  for (int s = 0; s < stage; ++s)
    if (!k[s]) return fail(Z4C_EINVAL, "rk4_stage: null k register");
  hipStream_t s = (hipStream_t)stream;
  // Butcher tableau of bt_rk4 (task_list_integrators_butcher.cpp:37-49)
  static const double A[4][4] = {{0, 0, 0, 0}, {0.5, 0, 0, 0}, {0, 0.5, 0, 0}, {0, 0, 1, 0}};
  static const double Bw[4] = {1. / 6., 1. / 3., 1. / 3., 1. / 6.};
  rc = launch_rhs(c, p, u, mat, k[stage - 1], true, s);
  if (rc) return rc;
  const double* kk[4] = {k[0], k[1], k[2], k[3]};
  if (stage < 4)
    rc = launch_bt(c, NVAR, u, un, stage, kk, A[stage], dt, s);
  else
    rc = launch_bt(c, NVAR, u, un, 4, kk, Bw, dt, s);
  if (rc) return rc;
  if (periodic & 1) {
    rc = launch_periodic(c, NVAR, u, s);
    if (rc) return rc;
  } else if (periodic & 2) {
    rc = launch_exchange(c, NVAR, u, s);
    if (rc) return rc;
  }
  if (periodic & 4) {
    rc = launch_physical(c, NVAR, u, s);
    if (rc) return rc;
  }
  rc = launch_alg(c, p, u, nullptr, 0, s);
  if (rc) return rc;
  return launch_prep(c, p, u, nullptr, s);
}

int z4c_ls_tableau_get(const char* name, z4c_ls_tableau* out) {
  if (!name || !out) return fail(Z4C_EINVAL, "ls_tableau_get: null argument");
  // (delta, gamma_1, gamma_2, gamma_3, beta) per stage,
  // task_list_integrators_low_storage.cpp:41-195 (ONE_3RD / TWO_3RD of
  // defs.hpp.in:257-258 round to 1/3 and 2/3)
  struct W { double d, g1, g2, g3, b; };
  static const std::map<std::string, std::vector<W>> tab = {
      {"vl2", {{1.0, 0.0, 1.0, 0.0, 0.5}, {0.0, 0.0, 1.0, 0.0, 1.0}}},
      {"rk1", {{1.0, 0.0, 1.0, 0.0, 1.0}}},
      {"rk2", {{1.0, 0.0, 1.0, 0.0, 1.0}, {0.0, 0.5, 0.5, 0.0, 0.5}}},
      {"rk3", {{1.0, 0.0, 1.0, 0.0, 1.0}, {0.0, 0.25, 0.75, 0.0, 0.25},
               {0.0, 2.0 / 3.0, 1.0 / 3.0, 0.0, 2.0 / 3.0}}},
      {"rk4", {{1.0, 0.0, 1.0, 0.0, 1.193743905974738},
               {0.217683334308543, 0.121098479554482, 0.721781678111411, 0.0, 0.099279895495783},
               {1.065841341361089, -3.843833699660025, 2.121209265338722, 0.0, 1.131678018054042},
               {0.0, 0.546370891121863, 0.198653035682705, 0.0, 0.310665766509336}}},
  };
  const std::string nm(name);
  if (nm == "ssprk5_4")
    return fail(Z4C_EINVAL, "ls_tableau_get: ssprk5_4 is not available with GR (the GR_Z4c "
                            "task list rejects it)");
  auto it = tab.find(nm);
  if (it == tab.end()) return fail(Z4C_EINVAL, "ls_tableau_get: unknown integrator " + nm);
  std::memset(out, 0, sizeof(*out));
  out->nstages = (int)it->second.size();
  for (int q = 0; q < out->nstages; ++q) {
    const W& w = it->second[q];
    out->delta[q] = w.d;
    out->gamma_1[q] = w.g1;
    out->gamma_2[q] = w.g2;
    out->gamma_3[q] = w.g3;
    out->beta[q] = w.b;
  }
  return Z4C_OK;
}

int z4c_ls_stage(z4c_ctx* c, const z4c_params* p, const z4c_ls_tableau* t, int stage, double dt,
                 double* u, double* u1, const double* u2, double* rhs, const double* mat,
                 int ghosts, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  rc = check_ls(t, false, "ls_stage");
  if (rc) return rc;
  if (!p || !u || !u1 || !rhs || stage < 1 || stage > t->nstages || ghosts < 0 || ghosts > 7 ||
      (ghosts & 3) == 3)
    return fail(Z4C_EINVAL, "ls_stage: bad argument");
  const int q = stage - 1;
  if (t->gamma_3[q] != 0.0 && !u2) return fail(Z4C_EINVAL, "ls_stage: gamma_3 != 0 needs u2");
  hipStream_t s = (hipStream_t)stream;
  // StartupTaskList: u1 = 0 at the beginning of each cycle
  if (stage == 1) {
    rc = fill(c, u1, 0.0, c->total_pts * NVAR, s);
    if (rc) return rc;
  }
  rc = launch_rhs(c, p, u, mat, rhs, true, s);
  if (!rc) rc = launch_wave(c, u1, u, u2, 1.0, t->delta[q], 0.0, 0, s);
  if (!rc) rc = launch_wave(c, u, u1, u2, t->gamma_1[q], t->gamma_2[q], t->gamma_3[q], 0, s);
  if (!rc) rc = launch_wave(c, u, rhs, nullptr, t->beta[q] * dt, 0.0, 0.0, 1, s);
  if (!rc) rc = ghost_update(c, u, ghosts, s);
  if (!rc) rc = launch_alg(c, p, u, nullptr, 0, s);
  if (rc) return rc;
  return launch_prep(c, p, u, nullptr, s);
}

int z4c_ls_step(z4c_ctx* c, const z4c_params* p, const z4c_ls_tableau* t, double dt, double* u,
                double* work, const double* mat, int ghosts, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  rc = check_ls(t, true, "ls_step");
  if (rc) return rc;
  if (!p || !u || !work || ghosts < 0 || ghosts > 7 || (ghosts & 3) == 3)
    return fail(Z4C_EINVAL, "ls_step: bad argument");
  return launch_ls_step(c, p, t, dt, u, work, mat, ghosts, (hipStream_t)stream);
}

int z4c_rhs_vjp(z4c_ctx* c, const z4c_params* p, const double* u, int nw, const double* w,
                double* ubar, double* pbar, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !w || !ubar || !pbar) return fail(Z4C_EINVAL, "rhs_vjp: null argument");
  rc = check_vjp_args(c, p, nw, "rhs_vjp");
  if (rc) return rc;
  return launch_rhs_vjp(c, p, u, nw, w, ubar, pbar, 0, (hipStream_t)stream);
}

int z4c_weyl(z4c_ctx* c, const z4c_params* p, const double* u, const double* adm, double* weyl,
             void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !adm || !weyl) return fail(Z4C_EINVAL, "weyl: null argument");
  hipStream_t s = (hipStream_t)stream;
  rc = launch_prep(c, p, u, nullptr, s);
  if (rc) return rc;
  rc = fill(c, weyl, std::numeric_limits<double>::quiet_NaN(), 2 * c->total_pts, s);
  if (rc) return rc;
  WeylArgs a{c->d_blocks, launch_of(c, BOX_INTERIOR), u, adm, c->d1, weyl, p->chi_psi_power,
             p->chi_div_floor};
  hipLaunchKernelGGL(k_weyl, dim3(grid_for(a.L.ntiles)), dim3(TILE), 0, s, a);
  HIPCALL(hipGetLastError());
  return Z4C_OK;
}

int z4c_hamiltonian_norm(z4c_ctx* c, const z4c_params* p, const double* u, double* J,
                         void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !J) return fail(Z4C_EINVAL, "hamiltonian_norm: null argument");
  rc = check_vjp_args(c, p, 1, "hamiltonian_norm");
  if (rc) return rc;
  return launch_hnorm(c, p, u, J, (hipStream_t)stream);
}

int z4c_hamiltonian_norm_vjp(z4c_ctx* c, const z4c_params* p, const double* u, double* ubar,
                             void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !ubar) return fail(Z4C_EINVAL, "hamiltonian_norm_vjp: null argument");
  rc = check_vjp_args(c, p, 1, "hamiltonian_norm_vjp");
  if (rc) return rc;
  double* pbar = nullptr;
  rc = ensure_buf(c->adj_stage, c->adj_stage_n, c->total_pts * NVAR, "hamiltonian_norm_vjp");
  if (rc) return rc;
  pbar = c->adj_stage;  // parameter partials are zero here; scratch target
  return launch_rhs_vjp(c, p, u, 1, nullptr, ubar, pbar, 0, (hipStream_t)stream);
}

int z4c_rk4_step_vjp(z4c_ctx* c, const z4c_params* p, double dt, const double* u, int nw,
                     const double* ubar_out, double* ubar_in, double* pbar, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !ubar_out || !ubar_in || !pbar)
    return fail(Z4C_EINVAL, "rk4_step_vjp: null argument");
  rc = check_vjp_args(c, p, nw, "rk4_step_vjp");
  if (rc) return rc;
  for (const z4c_block& b : c->hblocks)
    if (b.sommerfeld_faces & 63)
      return fail(Z4C_EINVAL, "rk4_step_vjp: Sommerfeld faces have no adjoint here");
  return launch_rk4_step_vjp(c, p, dt, u, nw, ubar_out, ubar_in, pbar, (hipStream_t)stream);
}

int z4c_rk4_step_ghosts_vjp(z4c_ctx* c, const z4c_params* p, double dt, const double* u, int nw,
                            const double* ubar_out, double* ubar_in, double* pbar, int ghosts,
                            void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!p || !u || !ubar_out || !ubar_in || !pbar)
    return fail(Z4C_EINVAL, "rk4_step_ghosts_vjp: null argument");
  rc = check_vjp_args(c, p, nw, "rk4_step_ghosts_vjp");
  if (rc) return rc;
  if (ghosts != 2 && ghosts != 6)
    return fail(Z4C_EINVAL, "rk4_step_ghosts_vjp: ghosts must be 2 (the exchange set by "
                            "z4c_set_exchange) or 6 (and the physical fill)");
  for (const z4c_block& b : c->hblocks) {
    if (b.sommerfeld_faces & 63)
      return fail(Z4C_EINVAL, "rk4_step_ghosts_vjp: Sommerfeld faces have no adjoint here");
    if ((b.outflow_faces & 63) && !(ghosts & 4))
      return fail(Z4C_EINVAL, "rk4_step_ghosts_vjp: outflow faces need ghosts = 6");
  }
  return launch_rk4_step_ghosts_vjp(c, p, dt, u, nw, ubar_out, ubar_in, pbar, ghosts,
                                    (hipStream_t)stream);
}

int z4c_exchange_vjp(z4c_ctx* c, int nvar, double* ubar, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!ubar || nvar <= 0) return fail(Z4C_EINVAL, "exchange_vjp: bad argument");
  return launch_exchange_vjp(c, nvar, ubar, (hipStream_t)stream);
}

int z4c_physical_bc_vjp(z4c_ctx* c, int nvar, double* ubar, void* stream) {
  int rc = check_ctx(c);
  if (rc) return rc;
  if (!ubar || nvar <= 0) return fail(Z4C_EINVAL, "physical_bc_vjp: bad argument");
  return launch_physical_vjp(c, nvar, ubar, (hipStream_t)stream);
}

}  // extern "C"
