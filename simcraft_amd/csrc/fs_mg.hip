// fs_mg.hip - multigrid-preconditioned CG for the pressure system.
//
// PreconditionerMethod::Multigrid is declared in the reference without an implementation
// (FluidSim/include/FluidSim/cpu/project-solver.h:117-118; setCompressedSolver reaches ERROR).
// This is the library's own multigrid; the CG loop around it is CgSolver3D::solve
// (FluidSim/src/cpu/project-solver.cc:308-346) with the same stopping rules and status codes.
//
// Hierarchy, rebuilt for every solve (the system changes every substep):
//   level 0  the assembled system on the grid: D = Adiag on active cells, Cx/Cy/Cz = the coupling
//            to the -x/-y/-z neighbour (An[Left], An[Down], An[Back]) where both cells are active,
//            else 0; a cell's +x coupling is Cx of its +x neighbour (the assembly is symmetric,
//            An[Right](i) == An[Left](i+1) bit for bit). W = omega / D where D > 0, else 0.
//   level l+1  2x2x2 aggregates of level l: the Galerkin product P^T A P of piecewise-constant
//            prolongation. D sums the children's D and twice their couplings inside the
//            aggregate; Cx sums the -x couplings of the children on the aggregate's -x face.
//            Coarsening stops at one cell.
// V-cycle on b (symmetric, so CG keeps its guarantees): two weighted-Jacobi sweeps from zero,
// the residual restricted by summation over the aggregate, the coarse cycle, the coarse solution
// added with weight alpha (over-correction, for the piecewise-constant prolongation), two
// sweeps; the coarsest level runs four sweeps.
//
// Layout: every level is a dense grid, k fastest, in the context's storage type S (FP32 in mixed
// precision); the CG vectors x, r, s, t are FP64 in both modes, so the stopping test is always
// made on an FP64 recurrence of the FP64 system. Kernels that reduce (dot products, norms) give a
// block of 256 threads one chunk of 4096 consecutive cells (thread t: cells t + 256 m, m = 0..15),
// the fixed tree; the others take one cell per thread. A cell with W = 0 (inactive) reads no
// neighbour. Sweeps that need the previous iterate of a neighbour recompute it from what is
// stored (W b for the first sweep, x + alpha x_coarse after the coarse correction), so each
// level costs four passes: two sweeps, restriction, correction with a sweep, a sweep. Dot
// products use the fixed tree of fs_reduce.h over the chunks, and the level-0 sweep that ends
// the cycle also forms z.r.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "fs_ctx.h"
#include "fs_reduce.h"

namespace {

constexpr double MG_OMEGA = 0.9;  // Jacobi weight
constexpr double MG_ALPHA = 1.8;  // coarse-correction weight
constexpr int MCH = 4096;         // cells per block of the kernels that reduce
// Up to this many blocks of them take 1024 threads instead of 256 (chunk_sum): with few blocks a
// thread's sixteen cells in turn are the kernel's time, with many the other blocks hide them. Mixed,
// us, 256 / 1024 threads, SpMV, last sweep, update: 64^3 12.5 / 8.9, 9.3 / 5.6, 8.5 / 7.5; 128^3 (512
// blocks) 15.0 / 9.8, 10.5 / 6.9, 10.9 / 8.0; 192^3 (1728) 23.6 / 25.1, 14.7 / 16.8, 17.9 / 19.2.
constexpr unsigned MG_WIDE = 1024;
// Cells in flight per thread of the 1024-thread forms: with four, FP64 operands spill (SpMV 19.2 us at
// 128^3, 13.3 with a branch per term).
template <typename S>
constexpr int MG_FLIGHT = sizeof(S) == 4 ? 4 : 2;

template <typename S>
struct Lv {
  int nx, ny, nz;
  const S *D, *Cx, *Cy, *Cz, *W;
};

__device__ __forceinline__ void decode3(int64_t c, int ny, int nz, int& i, int& j, int& k) {
  const unsigned uc = (unsigned)c;  // levels hold fewer than 2^31 cells (checked at create)
  const unsigned q = uc / (unsigned)nz;
  k = (int)(uc - q * (unsigned)nz);
  i = (int)(q / (unsigned)ny);
  j = (int)(q - (unsigned)i * (unsigned)ny);
}

// Row c of the level's operator applied to xo: diagonal, -x, -y, -z, +x, +y, +z (the order of
// applyCompressedMatrix, project-solver.cc:23-35); terms outside the grid are dropped. xo(q, i, j, k)
// gives the operand at cell q = (i, j, k). A term outside the grid reads the cell itself and is dropped
// by a select, so that a thread's reads are in flight together: a branch per term made each wait for
// the one before it (mixed, us, branches / selects: SpMV 15.6 / 8.9 at 64^3, 73 / 50 at 256^3; last sweep
// 9.6 / 5.6, 35.6 / 26.0; first sweep 43.5 / 38.2 at 256^3).
template <typename R, typename S, typename XO>
__device__ __forceinline__ R row(const Lv<S>& L, int64_t c, int i, int j, int k, XO xo) {
  const int64_t sx = (int64_t)L.ny * L.nz, sy = L.nz;
  const bool l = i > 0, d = j > 0, b = k > 0, r = i < L.nx - 1, u = j < L.ny - 1, f = k < L.nz - 1;
  const int64_t cr = r ? c + sx : c, cu = u ? c + sy : c, cf = f ? c + 1 : c;
  const R kl = (R)L.Cx[c], kd = (R)L.Cy[c], kb = (R)L.Cz[c], kr = (R)L.Cx[cr], ku = (R)L.Cy[cu], kf = (R)L.Cz[cf];
  const R x0 = xo(c, i, j, k), xl = xo(l ? c - sx : c, i - l, j, k), xd = xo(d ? c - sy : c, i, j - d, k),
          xb = xo(b ? c - 1 : c, i, j, k - b), xr = xo(cr, i + r, j, k), xu = xo(cu, i, j + u, k),
          xf = xo(cf, i, j, k + f);
  R t = (R)L.D[c] * x0;
  t = l ? t + kl * xl : t;
  t = d ? t + kd * xd : t;
  t = b ? t + kb * xb : t;
  t = r ? t + kr * xr : t;
  t = u ? t + ku * xu : t;
  t = f ? t + kf * xf : t;
  return t;
}

// ---- hierarchy ----------------------------------------------------------------------------------
template <typename S>
__global__ __launch_bounds__(256) void k_mg_level0(int nx, int ny, int nz, const S* __restrict__ adiag,
                                                   const S* __restrict__ aL, const S* __restrict__ aD,
                                                   const S* __restrict__ aB, const uint8_t* __restrict__ act,
                                                   S* __restrict__ D, S* __restrict__ Cx, S* __restrict__ Cy,
                                                   S* __restrict__ Cz, S* __restrict__ W, S* __restrict__ x,
                                                   S* __restrict__ xs) {
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (c >= (int64_t)nx * ny * nz) return;
  x[c] = S(0);  // the cycle never writes a cell with W = 0: its iterates stay 0 for the solve
  xs[c] = S(0);
  int i, j, k;
  decode3(c, ny, nz, i, j, k);
  const int64_t sx = (int64_t)ny * nz;
  S d = S(0), cx = S(0), cy = S(0), cz = S(0), w = S(0);
  if (act[c]) {
    d = adiag[c];
    if (i > 0 && act[c - sx]) cx = aL[c];
    if (j > 0 && act[c - nz]) cy = aD[c];
    if (k > 0 && act[c - 1]) cz = aB[c];
    w = d > S(0) ? (S)(MG_OMEGA / (double)d) : S(0);
  }
  D[c] = d;
  Cx[c] = cx;
  Cy[c] = cy;
  Cz[c] = cz;
  W[c] = w;
}

template <typename S>
__global__ __launch_bounds__(256) void k_mg_coarsen(Lv<S> F, int cx_, int cy_, int cz_, S* __restrict__ D,
                                                    S* __restrict__ Cx, S* __restrict__ Cy, S* __restrict__ Cz,
                                                    S* __restrict__ W, S* __restrict__ x, S* __restrict__ xs) {
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (c >= (int64_t)cx_ * cy_ * cz_) return;
  x[c] = S(0);
  xs[c] = S(0);
  int I, J, K;
  decode3(c, cy_, cz_, I, J, K);
  S d = S(0), sx = S(0), sy = S(0), sz = S(0);
  for (int di = 0; di < 2; di++)
    for (int dj = 0; dj < 2; dj++)
      for (int dk = 0; dk < 2; dk++) {
        const int i = 2 * I + di, j = 2 * J + dj, k = 2 * K + dk;
        if (i >= F.nx || j >= F.ny || k >= F.nz) continue;
        const int64_t f = ((int64_t)i * F.ny + j) * F.nz + k;
        d = d + F.D[f];
        if (di) d = d + S(2) * F.Cx[f];
        if (dj) d = d + S(2) * F.Cy[f];
        if (dk) d = d + S(2) * F.Cz[f];
        if (!di) sx = sx + F.Cx[f];
        if (!dj) sy = sy + F.Cy[f];
        if (!dk) sz = sz + F.Cz[f];
      }
  D[c] = d;
  Cx[c] = sx;
  Cy[c] = sy;
  Cz[c] = sz;
  W[c] = d > S(0) ? (S)(MG_OMEGA / (double)d) : S(0);
}

// ---- V-cycle ------------------------------------------------------------------------------------
// B is the type of the level's right-hand side: FP64 on level 0 (the CG residual), S below.
// sc (may be null): the kernels of a CG iteration return at once after the solve has stopped.
// A cell with W = 0 is never written: the level's x and xs are zeroed when the hierarchy is
// built, and stay 0 there for the whole solve.

// x = two Jacobi sweeps from zero at a live cell: x1 = W b, x = x1 + W (b - A x1).
template <typename S, typename B>
__device__ __forceinline__ S pre_cell(const Lv<S>& L, const B* __restrict__ b, int64_t c, int i, int j, int k) {
  auto xo = [&](int64_t q, int, int, int) { return L.W[q] * (S)b[q]; };
  return xo(c, i, j, k) + L.W[c] * ((S)b[c] - row<S>(L, c, i, j, k, xo));
}
// b(f) - (A x)(f) of child (bits di dj dk of q) of aggregate (I, J, K), 0 when it is off the grid or
// not live (adding it then changes no bit of the aggregate's sum, which starts at +0).
template <typename S, typename B>
__device__ __forceinline__ S restrict_child(const Lv<S>& L, const B* __restrict__ b, const S* __restrict__ x, int I,
                                            int J, int K, int q) {
  auto xo = [&](int64_t c, int, int, int) { return x[c]; };
  const int i = 2 * I + (q >> 2), j = 2 * J + ((q >> 1) & 1), k = 2 * K + (q & 1);
  if (i >= L.nx || j >= L.ny || k >= L.nz) return S(0);
  const int64_t f = ((int64_t)i * L.ny + j) * L.nz + k;
  return L.W[f] > S(0) ? (S)b[f] - row<S>(L, f, i, j, k, xo) : S(0);
}
// Sum over the children of an aggregate, which are eight consecutive lanes, in lexicographic order.
template <typename S>
__device__ __forceinline__ S restrict_sum(S r) {
  const int l0 = threadIdx.x & 56;
  S acc = S(0);
#pragma unroll
  for (int q = 0; q < 8; q++) acc = acc + __shfl(r, l0 + q, 64);
  return acc;
}
// The coarse correction x' = x + alpha xc(parent) on live cells, then one sweep at a live cell.
template <typename S, typename B>
__device__ __forceinline__ S post1_cell(const Lv<S>& L, const B* __restrict__ b, const S* __restrict__ x,
                                        const S* __restrict__ xc, int cny, int cnz, S alpha, int64_t c, int i, int j,
                                        int k) {
  auto xo = [&](int64_t q, int qi, int qj, int qk) {
    const S w = L.W[q], v = x[q], p = xc[((int64_t)(qi >> 1) * cny + (qj >> 1)) * cnz + (qk >> 1)];
    return w > S(0) ? v + alpha * p : v;
  };
  return xo(c, i, j, k) + L.W[c] * ((S)b[c] - row<S>(L, c, i, j, k, xo));
}
// One sweep x = xs + W (b - A xs) at a live cell.
template <typename S, typename B>
__device__ __forceinline__ S sweep_cell(const Lv<S>& L, const B* __restrict__ b, const S* __restrict__ xs, int64_t c,
                                        int i, int j, int k) {
  auto xo = [&](int64_t q, int, int, int) { return xs[q]; };
  return xs[c] + L.W[c] * ((S)b[c] - row<S>(L, c, i, j, k, xo));
}

// The sweeps without a dot product take one cell per thread: the coarse levels are small, and
// sixteen cells per thread would leave most of the chip idle while each thread waits on its
// loads in turn.
template <typename S, typename B>
__global__ __launch_bounds__(256) void k_mg_pre(Lv<S> L, const B* __restrict__ b, S* __restrict__ x,
                                                const PcgScalars* sc) {
  if (sc && sc->converged != STOP_RUN) return;
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (c >= (int64_t)L.nx * L.ny * L.nz || !(L.W[c] > S(0))) return;
  int i, j, k;
  decode3(c, L.ny, L.nz, i, j, k);
  x[c] = pre_cell<S, B>(L, b, c, i, j, k);
}

// CHILD: one thread per child, the aggregate's sum over eight lanes; else one thread per aggregate.
// Eight residuals of seven operands each, one after another in a thread, are the slowest sweep of a
// small level (mixed, us, an aggregate / a child per thread, with a branch per term of a row: 7.2 / 3.3
// for 64^3 -> 32^3, 11.0 / 10.0 for 128^3); above, other waves hide them and the eightfold threads and
// their shuffles cost more than they save (14.8 / 17.0 for 160^3, 39.8 / 54.5 for 256^3). The chosen
// forms take 3.7, 9.9, 11.7 and 38.1 with selects.
constexpr int64_t MG_RESTRICT_CHILD = (int64_t)1 << 18;  // aggregates up to which CHILD is taken
template <typename S, typename B, bool CHILD>
__global__ __launch_bounds__(256) void k_mg_restrict(Lv<S> L, const B* __restrict__ b, const S* __restrict__ x,
                                                     int cnx, int cny, int cnz, S* __restrict__ bc,
                                                     const PcgScalars* sc) {
  if (sc && sc->converged != STOP_RUN) return;
  const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, c = CHILD ? e >> 3 : e;
  if (c >= (int64_t)cnx * cny * cnz) return;  // uniform over the eight lanes of an aggregate
  int I, J, K;
  decode3(c, cny, cnz, I, J, K);
  if constexpr (CHILD) {
    const int q = threadIdx.x & 7;
    const S acc = restrict_sum<S>(restrict_child<S, B>(L, b, x, I, J, K, q));
    if (q == 0) bc[c] = acc;
  } else {
    S acc = S(0);
    for (int q = 0; q < 8; q++) acc = acc + restrict_child<S, B>(L, b, x, I, J, K, q);
    bc[c] = acc;
  }
}

template <typename S, typename B>
__global__ __launch_bounds__(256) void k_mg_post1(Lv<S> L, const B* __restrict__ b, const S* __restrict__ x,
                                                  const S* __restrict__ xc, int cny, int cnz, S alpha,
                                                  S* __restrict__ xs, const PcgScalars* sc) {
  if (sc && sc->converged != STOP_RUN) return;
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (c >= (int64_t)L.nx * L.ny * L.nz || !(L.W[c] > S(0))) return;
  int i, j, k;
  decode3(c, L.ny, L.nz, i, j, k);
  xs[c] = post1_cell<S, B>(L, b, x, xc, cny, cnz, alpha, c, i, j, k);
}

// One sweep from xs into x.
template <typename S, typename B>
__global__ __launch_bounds__(256) void k_mg_sweep(Lv<S> L, const B* __restrict__ b, const S* __restrict__ xs,
                                                  S* __restrict__ x, const PcgScalars* sc) {
  if (sc && sc->converged != STOP_RUN) return;
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (c >= (int64_t)L.nx * L.ny * L.nz || !(L.W[c] > S(0))) return;
  int i, j, k;
  decode3(c, L.ny, L.nz, i, j, k);
  x[c] = sweep_cell<S, B>(L, b, xs, c, i, j, k);
}

// The sweep that ends a CG cycle on level 0, from xs into x = z, with z.r over the chunk, reduced by
// the last block into sigma (FIRST: the initial sigma; else beta = sigma_new / sigma,
// sigma = sigma_new). Chunks of 4096 cells per block: the fixed reduction tree.
template <typename S, typename B, bool FIRST, int TH>
__global__ __launch_bounds__(TH) void k_mg_post2(Lv<S> L, const B* __restrict__ b, const S* __restrict__ xs,
                                                  S* __restrict__ x, double* __restrict__ part, int nchunks,
                                                  PcgScalars* sc) {
  __shared__ double sm[4];
  if (sc && sc->converged != STOP_RUN) return;
  __shared__ double terms[CHUNK_TERMS<TH>];
  const int64_t n = (int64_t)L.nx * L.ny * L.nz;
  struct V {
    S out;
    double b;
  };
  const int64_t c0 = (int64_t)blockIdx.x * MCH;
  auto at = [&](int e) { return c0 + e < n ? c0 + e : n - 1; };
  const double acc = chunk_sum<TH, V, MG_FLIGHT<S>>(
      terms,
      [&](int e) __attribute__((always_inline)) {
        const S w = L.W[at(e)];  // where it is 0, so are z and its product with r
        return c0 + e < n && w > S(0);
      },
      [&](int e) __attribute__((always_inline)) {
        const int64_t c = at(e);
        int i, j, k;
        decode3(c, L.ny, L.nz, i, j, k);
        return V{sweep_cell<S, B>(L, b, xs, c, i, j, k), (double)b[c]};
      },
      [&](int e, const V& v) __attribute__((always_inline)) {
        x[c0 + e] = v.out;
        return (double)v.out * v.b;
      });
  const double bs = block_sum256(acc, sm);
  if (threadIdx.x == 0) xstore(part + blockIdx.x, bs);
  if (blockIdx.x == gridDim.x - 1) {
    const double sig = gather256(part, nullptr, nchunks, sm, sc).sum;
    if (threadIdx.x == 0) {
      if (!FIRST) sc->beta = sig / sc->sigma;
      sc->sigma = sig;
    }
  }
}

// The levels from l0 down to the single cell and back up, in one workgroup (the small levels,
// where separate launches would cost more than the work): the same cell functions, the passes
// separated by workgroup barriers. The iterates and right-hand sides of all its levels live in
// LDS, as do the operators in FP32 (in FP64 the first level's operator, 160 KB, stays in memory):
// a pass is then a few LDS reads instead of dependent reads of the L2 (19 passes at 64^3:
// 29.5 -> 15.1 us in FP32).
constexpr int MG_TAIL_CELLS = 4096;  // levels at or below this size run in the tail kernel
constexpr int MG_TAIL_SUM = 4800;    // ... if all its levels together have no more cells than this
constexpr int MG_MAX_LEVELS = 16;
template <typename S>
struct TailLevels {
  Lv<S> L[MG_MAX_LEVELS];
  int off[MG_MAX_LEVELS + 1];  // of a level's cells in the tail's LDS arrays
  const S* b;                  // right-hand side of level l0
  S* x;                        // its solution
};
template <typename S>
__global__ __launch_bounds__(1024) void k_mg_tail(TailLevels<S> T, int l0, int nl, S alpha, const PcgScalars* sc) {
  constexpr bool ALL = sizeof(S) == 4;                    // level l0's operator in LDS as well
  constexpr int CSUM = ALL ? MG_TAIL_SUM : MG_TAIL_SUM - MG_TAIL_CELLS;
  __shared__ S cD[CSUM], cX[CSUM], cY[CSUM], cZ[CSUM], cW[CSUM], vb[MG_TAIL_SUM], vx[MG_TAIL_SUM], vs[MG_TAIL_SUM];
  if (sc && sc->converged != STOP_RUN) return;
  const int tid = threadIdx.x;
  const int n0 = T.off[l0 + 1];  // cells of level l0
  const int c0 = ALL ? 0 : n0;   // the first cell whose operator is in LDS
  for (int c = tid; c < T.off[nl]; c += 1024) {
    vx[c] = S(0);  // cells with W = 0 are never written
    vs[c] = S(0);
    vb[c] = c < n0 ? T.b[c] : S(0);
  }
  for (int l = ALL ? l0 : l0 + 1; l < nl; l++) {
    const int n = T.off[l + 1] - T.off[l], o = T.off[l] - c0;
    for (int c = tid; c < n; c += 1024) {
      cD[o + c] = T.L[l].D[c];
      cX[o + c] = T.L[l].Cx[c];
      cY[o + c] = T.L[l].Cy[c];
      cZ[o + c] = T.L[l].Cz[c];
      cW[o + c] = T.L[l].W[c];
    }
  }
  __syncthreads();
  auto in_lds = [&](int l) {
    const int o = T.off[l] - c0;
    return Lv<S>{T.L[l].nx, T.L[l].ny, T.L[l].nz, cD + o, cX + o, cY + o, cZ + o, cW + o};
  };
  auto down = [&](int l, const Lv<S>& L) __attribute__((always_inline)) {
    const int n = L.nx * L.ny * L.nz, o = T.off[l];
    for (int c = tid; c < n; c += 1024) {
      if (!(L.W[c] > S(0))) continue;
      int i, j, k;
      decode3(c, L.ny, L.nz, i, j, k);
      vx[o + c] = pre_cell<S, S>(L, vb + o, c, i, j, k);
    }
    __syncthreads();
    if (l + 1 < nl) {
      const int cny = T.L[l + 1].ny, cnz = T.L[l + 1].nz, on = T.off[l + 1], nc = T.off[l + 2] - on;
      for (int e = tid; e < 8 * nc; e += 1024) {
        int I, J, K;
        decode3(e >> 3, cny, cnz, I, J, K);
        const S acc = restrict_sum<S>(restrict_child<S, S>(L, vb + o, vx + o, I, J, K, e & 7));
        if ((e & 7) == 0) vb[on + (e >> 3)] = acc;
      }
      __syncthreads();
    }
  };
  auto sweep = [&](int l, const Lv<S>& L, const S* from, S* to) __attribute__((always_inline)) {
    const int n = L.nx * L.ny * L.nz, o = T.off[l];
    for (int c = tid; c < n; c += 1024) {
      if (!(L.W[c] > S(0))) continue;
      int i, j, k;
      decode3(c, L.ny, L.nz, i, j, k);
      to[o + c] = sweep_cell<S, S>(L, vb + o, from + o, c, i, j, k);
    }
    __syncthreads();
  };
  auto up = [&](int l, const Lv<S>& L) __attribute__((always_inline)) {
    const int cny = T.L[l + 1].ny, cnz = T.L[l + 1].nz, on = T.off[l + 1];
    const int n = L.nx * L.ny * L.nz, o = T.off[l];
    for (int c = tid; c < n; c += 1024) {
      if (!(L.W[c] > S(0))) continue;
      int i, j, k;
      decode3(c, L.ny, L.nz, i, j, k);
      vs[o + c] = post1_cell<S, S>(L, vb + o, vx + o, vx + on, cny, cnz, alpha, c, i, j, k);
    }
    __syncthreads();
    sweep(l, L, vs, vx);
  };
  if (ALL) down(l0, in_lds(l0));
  else down(l0, T.L[l0]);
  for (int l = l0 + 1; l < nl; l++) down(l, in_lds(l));
  if (ALL || nl - 1 > l0) {
    sweep(nl - 1, in_lds(nl - 1), vx, vs);
    sweep(nl - 1, in_lds(nl - 1), vs, vx);
  } else {
    sweep(l0, T.L[l0], vx, vs);
    sweep(l0, T.L[l0], vs, vx);
  }
  for (int l = nl - 2; l > l0; l--) up(l, in_lds(l));
  if (nl - 1 > l0) {
    if (ALL) up(l0, in_lds(l0));
    else up(l0, T.L[l0]);
  }
  for (int c = tid; c < n0; c += 1024) T.x[c] = vx[c];
}

// Iteration iter of a solve is finished (the thread that has written its scalars).
constexpr int MG_STOPPED = 1 << 30;
__device__ inline void report(int* prog, int iter, const PcgScalars* sc) {
  __hip_atomic_store(prog, iter | (sc->converged != STOP_RUN ? MG_STOPPED : 0), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---- CG kernels ---------------------------------------------------------------------------------
// r = rhs on active cells (0 elsewhere), x = 0; ||r||_inf, ||r||_2^2 and the stopping test at
// iteration 0.
template <typename T>
__global__ __launch_bounds__(256) void k_mg_init(int64_t n, const uint8_t* __restrict__ act,
                                                 const T* __restrict__ rhs, double* __restrict__ x,
                                                 double* __restrict__ r, double* __restrict__ s0,
                                                 double* __restrict__ s1, double* __restrict__ t,
                                                 double* __restrict__ part,
                                                 double* __restrict__ part2, int nchunks, PcgScalars* sc,
                                                 int tol_mode, double tol) {
  __shared__ double sm[4];
  double mx = 0.0, ss = 0.0;
  int na = 0;
  for (int m = 0; m < 16; m++) {
    const int64_t c = (int64_t)blockIdx.x * MCH + m * 256 + threadIdx.x;
    if (c >= n) break;
    const double v = act[c] ? (double)rhs[c] : 0.0;
    r[c] = v;
    x[c] = 0.0;
    s0[c] = 0.0;  // s and t are written on active cells only
    s1[c] = 0.0;
    t[c] = 0.0;
    ss += v * v;
    const double av = act[c] ? fabs(v) : 0.0;
    mx = (mx < av) ? av : mx;
    na += act[c] ? 1 : 0;
  }
  const double bm = block_max256(mx, sm);
  const double bs = block_sum256(ss, sm);
  const double bn = block_sum256((double)na, sm);
  if (threadIdx.x == 0) {
    xstore(part + blockIdx.x, bs);
    xstore(part2 + blockIdx.x, bm);
    atomicAdd(&sc->n_active, (unsigned long long)bn);
  }
  if (blockIdx.x == gridDim.x - 1) {
    const GatherSumMax red = gather256(part, part2, nchunks, sm, sc);
    const double tot = red.sum, mxx = red.max;
    if (threadIdx.x == 0) {
      sc->bnorm2sq = tot;
      sc->rnorm2sq = tot;
      sc->residual = mxx;
      sc->status = FS_OK;
      sc->conv_iter = 0;
      sc->sigma = sc->alpha = sc->beta = sc->sdotz = 0.0;
      const bool conv = tol_mode == FS_TOL_REL_L2 ? (sqrt(tot) <= tol * sqrt(tot)) : (mxx < tol);
      sc->converged = conv ? STOP_CONVERGED : STOP_RUN;
    }
  }
}

// s = z (iteration 1) or z + beta s_old, recomputed for the six neighbours; t = A s (the assembled
// system in FP64 on active cells); s.t reduced by the last block into alpha. Inactive cells are not
// written: s and t are zeroed when the solve starts and stay 0 there.
template <typename S, int TH>
__global__ __launch_bounds__(TH) void k_mg_spmv(Lv<S> L, const uint8_t* __restrict__ act, const S* __restrict__ z,
                                                 const double* __restrict__ s_old, double* __restrict__ s_new,
                                                 double* __restrict__ t, double* __restrict__ part, int nchunks,
                                                 PcgScalars* sc, int iter, int* prog) {
  __shared__ double sm[4];
  if (sc->converged != STOP_RUN) return;
  const int64_t n = (int64_t)L.nx * L.ny * L.nz;
  const bool first = iter == 1;
  const double beta = sc->beta;
  auto so = [&](int64_t q, int, int, int) {
    const double zq = (double)z[q], v = zq + beta * s_old[q];
    return first ? zq : v;
  };
  __shared__ double terms[CHUNK_TERMS<TH>];
  struct V {
    double s, t;
  };
  const int64_t c0 = (int64_t)blockIdx.x * MCH;
  auto at = [&](int e) { return c0 + e < n ? c0 + e : n - 1; };
  const double acc = chunk_sum<TH, V, MG_FLIGHT<S>>(
      terms,
      [&](int e) __attribute__((always_inline)) {
        const uint8_t on = act[at(e)];
        return c0 + e < n && on != 0;
      },
      [&](int e) __attribute__((always_inline)) {
        const int64_t c = at(e);
        int i, j, k;
        decode3(c, L.ny, L.nz, i, j, k);
        return V{so(c, i, j, k), row<double>(L, c, i, j, k, so)};
      },
      [&](int e, const V& v) __attribute__((always_inline)) {
        s_new[c0 + e] = v.s;
        t[c0 + e] = v.t;
        return v.s * v.t;
      });
  const double bs = block_sum256(acc, sm);
  if (threadIdx.x == 0) xstore(part + blockIdx.x, bs);
  if (blockIdx.x == gridDim.x - 1) {
    const double sdott = gather256(part, nullptr, nchunks, sm, sc).sum;
    if (threadIdx.x == 0) {
      sc->sdotz = sdott;
      if (sdott == 0.0) {
        sc->converged = STOP_ABORT;
        sc->status = FS_BREAKDOWN;
        sc->conv_iter = iter;
        report(prog, iter, sc);
      } else {
        sc->alpha = sc->sigma / sdott;
      }
    }
  }
}

// x += alpha s, r += -alpha t on active cells (saxpy, util.cc:394-402); ||r||_inf, ||r||_2^2 and the
// stopping test of iteration iter.
template <int TH>
__global__ __launch_bounds__(TH) void k_mg_update(int64_t n, const uint8_t* __restrict__ act,
                                                   double* __restrict__ x, const double* __restrict__ s,
                                                   double* __restrict__ r, const double* __restrict__ t,
                                                   double* __restrict__ part, double* __restrict__ part2,
                                                   int nchunks, PcgScalars* sc, int iter, int tol_mode, double tol,
                                                   int* prog) {
  __shared__ double sm[4];
  if (sc->converged != STOP_RUN) return;
  const double alpha = sc->alpha;
  __shared__ double terms[CHUNK_TERMS<TH>];
  double mx = 0.0;
  struct V {
    double x, r;
  };
  const int64_t c0 = (int64_t)blockIdx.x * MCH;
  auto at = [&](int e) { return c0 + e < n ? c0 + e : n - 1; };
  const double ss = chunk_sum<TH, V, 4>(
      terms,
      [&](int e) __attribute__((always_inline)) {
        const uint8_t on = act[at(e)];  // r = 0 on the others
        return c0 + e < n && on != 0;
      },
      [&](int e) __attribute__((always_inline)) {
        const int64_t c = at(e);
        return V{x[c] + alpha * s[c], r[c] + (-alpha) * t[c]};
      },
      [&](int e, const V& v) __attribute__((always_inline)) {
        x[c0 + e] = v.x;
        r[c0 + e] = v.r;
        const double av = fabs(v.r);
        mx = (mx < av) ? av : mx;
        return v.r * v.r;
      });
  mx = chunk_max<TH>(mx, terms);
  const double bm = block_max256(mx, sm);
  const double bs = block_sum256(ss, sm);
  if (threadIdx.x == 0) {
    xstore(part + blockIdx.x, bs);
    xstore(part2 + blockIdx.x, bm);
  }
  if (blockIdx.x == gridDim.x - 1) {
    const GatherSumMax red = gather256(part, part2, nchunks, sm, sc);
    const double tot = red.sum, mxx = red.max;
    if (threadIdx.x == 0) {
      sc->residual = mxx;
      sc->rnorm2sq = tot;
      const bool conv = tol_mode == FS_TOL_REL_L2 ? (sqrt(tot) <= tol * sqrt(sc->bnorm2sq)) : (mxx < tol);
      if (!(mxx <= 1.7976931348623157e308)) {
        sc->converged = STOP_ABORT;
        sc->status = FS_NONFINITE;
        sc->conv_iter = iter;
      } else if (conv) {
        sc->converged = STOP_CONVERGED;
        sc->conv_iter = iter;
      }
      report(prog, iter, sc);
    }
  }
}

template <typename T>
__global__ void k_mg_store(int64_t n, const double* __restrict__ x, T* __restrict__ out) {
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (c < n) out[c] = (T)x[c];
}

// ---- host ---------------------------------------------------------------------------------------
int ensure(fs_ctx* c, DBuf& b, size_t bytes) {
  if (b.p && b.bytes >= bytes) return FS_OK;
  fs_free(b);
  return fs_alloc(c, b, bytes);
}

template <typename S>
Lv<S> lv_of(const MgLevelBuf& B) {
  return {B.nx, B.ny, B.nz, B.D.as<S>(), B.Cx.as<S>(), B.Cy.as<S>(), B.Cz.as<S>(), B.W.as<S>()};
}

unsigned chunks_of(int64_t n) { return (unsigned)((n + MCH - 1) / MCH); }

// Levels and the hierarchy of the current assembled system.
template <typename S>
int mg_build(fs_ctx* c) {
  MgState& M = c->mg;
  std::vector<int3> dims{make_int3(c->nx, c->ny, c->nz)};
  while (dims.back().x > 1 || dims.back().y > 1 || dims.back().z > 1) {
    const int3 d = dims.back();
    dims.push_back(make_int3((d.x + 1) / 2, (d.y + 1) / 2, (d.z + 1) / 2));
  }
  M.lv.resize(dims.size());
  for (size_t l = 0; l < dims.size(); l++) {
    MgLevelBuf& B = M.lv[l];
    B.nx = dims[l].x;
    B.ny = dims[l].y;
    B.nz = dims[l].z;
    B.n = (int64_t)B.nx * B.ny * B.nz;
    const size_t bytes = (size_t)B.n * sizeof(S);
    for (DBuf* d : {&B.D, &B.Cx, &B.Cy, &B.Cz, &B.W, &B.x, &B.xs}) FS_TRY(ensure(c, *d, bytes));
    if (l > 0) FS_TRY(ensure(c, B.b, bytes));
  }
  if ((int)M.lv.size() > MG_MAX_LEVELS) {
    c->set_error("multigrid: too many levels");
    return FS_BAD_ARG;
  }
  MgLevelBuf& L0 = M.lv[0];
  k_mg_level0<S><<<fs_blocks(L0.n, 256), 256, 0, c->stream>>>(
      c->nx, c->ny, c->nz, c->adiag.as<S>(), c->an[0].as<S>(), c->an[3].as<S>(), c->an[5].as<S>(),
      c->active.as<uint8_t>(), L0.D.as<S>(), L0.Cx.as<S>(), L0.Cy.as<S>(), L0.Cz.as<S>(), L0.W.as<S>(),
      L0.x.as<S>(), L0.xs.as<S>());
  for (size_t l = 1; l < M.lv.size(); l++) {
    MgLevelBuf& B = M.lv[l];
    k_mg_coarsen<S><<<fs_blocks(B.n, 256), 256, 0, c->stream>>>(lv_of<S>(M.lv[l - 1]), B.nx, B.ny, B.nz,
                                                                  B.D.as<S>(), B.Cx.as<S>(), B.Cy.as<S>(),
                                                                  B.Cz.as<S>(), B.W.as<S>(), B.x.as<S>(),
                                                                  B.xs.as<S>());
  }
  FS_HIP(c, hipGetLastError());
  return FS_OK;
}

// One V-cycle on level 0 with right-hand side r0 (FP64). In a CG solve, sc is the solve's scalars
// and the final sweep forms sigma = z.r (FIRST: the initial sigma); z is level 0's x.
template <typename S>
int mg_cycle(fs_ctx* c, const double* r0, PcgScalars* sc, bool first) {
  MgState& M = c->mg;
  const int nl = (int)M.lv.size();
  const double na = (double)c->n_active_last;
  auto pre = [&](int l) {
    MgLevelBuf& B = M.lv[l];
    if (l == 0) k_mg_pre<S, double><<<fs_blocks(B.n, 256), 256, 0, c->stream>>>(lv_of<S>(B), r0, B.x.as<S>(), sc);
    else k_mg_pre<S, S><<<fs_blocks(B.n, 256), 256, 0, c->stream>>>(lv_of<S>(B), B.b.as<S>(), B.x.as<S>(), sc);
  };
  auto restrict_ = [&](int l) {
    MgLevelBuf &B = M.lv[l], &C = M.lv[l + 1];
    auto go = [&](auto kern, const auto* b, int64_t threads) {
      kern<<<fs_blocks(threads, 256), 256, 0, c->stream>>>(lv_of<S>(B), b, B.x.as<S>(), C.nx, C.ny, C.nz, C.b.as<S>(),
                                                           sc);
    };
    const bool child = C.n <= MG_RESTRICT_CHILD;
    if (l == 0 && child) go(k_mg_restrict<S, double, true>, r0, 8 * C.n);
    else if (l == 0) go(k_mg_restrict<S, double, false>, r0, C.n);
    else if (child) go(k_mg_restrict<S, S, true>, (const S*)B.b.as<S>(), 8 * C.n);
    else go(k_mg_restrict<S, S, false>, (const S*)B.b.as<S>(), C.n);
  };
  auto post1 = [&](int l) {
    MgLevelBuf &B = M.lv[l], &C = M.lv[l + 1];
    if (l == 0)
      k_mg_post1<S, double><<<fs_blocks(B.n, 256), 256, 0, c->stream>>>(lv_of<S>(B), r0, B.x.as<S>(), C.x.as<S>(),
                                                                         C.ny, C.nz, (S)MG_ALPHA, B.xs.as<S>(), sc);
    else
      k_mg_post1<S, S><<<fs_blocks(B.n, 256), 256, 0, c->stream>>>(lv_of<S>(B), B.b.as<S>(), B.x.as<S>(),
                                                                    C.x.as<S>(), C.ny, C.nz, (S)MG_ALPHA, B.xs.as<S>(),
                                                                    sc);
  };
  // one sweep from `from` into `to`; on level 0 of a CG cycle the sweep that ends the cycle
  // (into x) also forms sigma
  auto sweep = [&](int l, DBuf& from, DBuf& to, bool last) {
    MgLevelBuf& B = M.lv[l];
    const unsigned nb = chunks_of(B.n);
    const Lv<S> L = lv_of<S>(B);
    const unsigned nc1 = fs_blocks(B.n, 256);
    if (l > 0) {
      k_mg_sweep<S, S><<<nc1, 256, 0, c->stream>>>(L, B.b.as<S>(), from.as<S>(), to.as<S>(), sc);
    } else if (!last || !sc) {
      k_mg_sweep<S, double><<<nc1, 256, 0, c->stream>>>(L, r0, from.as<S>(), to.as<S>(), sc);
    } else {
      auto go = [&](auto kern, int th) {
        kern<<<nb, th, 0, c->stream>>>(L, r0, from.as<S>(), to.as<S>(), M.partials.as<double>(), (int)nb, sc);
      };
      const bool wide = nb <= MG_WIDE;
      if (first && wide) go(k_mg_post2<S, double, true, 1024>, 1024);
      else if (first) go(k_mg_post2<S, double, true, 256>, 256);
      else if (wide) go(k_mg_post2<S, double, false, 1024>, 1024);
      else go(k_mg_post2<S, double, false, 256>, 256);
    }
  };
  // the levels from lt on run in one workgroup (the first level small enough, with the levels
  // below it, for the tail; never level 0, whose right-hand side is the FP64 residual)
  int lt = nl;
  for (int l = 1; l < nl && lt == nl; l++) {
    int64_t sum = 0;
    for (int m = l; m < nl; m++) sum += M.lv[m].n;
    if (M.lv[l].n <= MG_TAIL_CELLS && sum <= MG_TAIL_SUM && sum - M.lv[l].n <= MG_TAIL_SUM - MG_TAIL_CELLS) lt = l;
  }
  // down
  int pf = fs_prof_begin(c, FS_KERNEL_MG_LEVEL0, (16.0 + 12.0 * sizeof(S)) * na);
  pre(0);
  if (nl > 1) restrict_(0);
  fs_prof_end(c, pf);
  // coarse levels hold about 1/7 of the active cells; 31 values per cell over the four passes
  pf = fs_prof_begin(c, FS_KERNEL_MG_COARSE, 31.0 * sizeof(S) * na / 7.0);
  for (int l = 1; l < lt; l++) {
    pre(l);
    restrict_(l);
  }
  if (lt < nl) {
    TailLevels<S> T{};
    for (int l = lt; l < nl; l++) {
      T.L[l] = lv_of<S>(M.lv[l]);
      T.off[l + 1] = T.off[l] + (int)M.lv[l].n;
    }
    T.b = M.lv[lt].b.as<S>();
    T.x = M.lv[lt].x.as<S>();
    k_mg_tail<S><<<1, 1024, 0, c->stream>>>(T, lt, nl, (S)MG_ALPHA, sc);
  }
  // up: correction and post-smoothing
  for (int l = lt - 1; l >= 1; l--) {
    post1(l);
    sweep(l, M.lv[l].xs, M.lv[l].x, false);
  }
  fs_prof_end(c, pf);
  pf = fs_prof_begin(c, FS_KERNEL_MG_LEVEL0, (16.0 + 14.0 * sizeof(S)) * na);
  if (nl > 1) {
    post1(0);
  } else {  // a single-cell grid is its own coarsest level
    sweep(0, M.lv[0].x, M.lv[0].xs, false);
  }
  sweep(0, M.lv[0].xs, M.lv[0].x, true);
  fs_prof_end(c, pf);
  FS_HIP(c, hipGetLastError());
  return FS_OK;
}

int mg_vectors(fs_ctx* c) {
  MgState& M = c->mg;
  const int64_t n = c->n_cell;
  for (DBuf* d : {&M.x, &M.r, &M.s0, &M.s1, &M.t}) FS_TRY(ensure(c, *d, (size_t)n * sizeof(double)));
  const int nc = (int)chunks_of(n);
  if (!M.scal.p) {
    FS_TRY(fs_alloc(c, M.scal, sizeof(PcgScalars)));
    FS_HIP(c, hipMemsetAsync(M.scal.p, 0, sizeof(PcgScalars), c->stream));
  }
  if (!M.host_scal) FS_HIP(c, hipHostMalloc((void**)&M.host_scal, sizeof(PcgScalars), hipHostMallocDefault));
  if (!M.prog) FS_HIP(c, hipHostMalloc((void**)&M.prog, sizeof(int), hipHostMallocMapped));
  if (!M.prog_dev) FS_HIP(c, hipHostGetDevicePointer((void**)&M.prog_dev, M.prog, 0));
  if (M.nchunks < nc || !M.partials.p) {
    FS_TRY(ensure(c, M.partials, (size_t)nc * sizeof(double)));
    FS_TRY(ensure(c, M.partials2, (size_t)nc * sizeof(double)));
    // reduction entries start unset; every reduction returns the entries it used to the sentinel
    k_fill_sentinel<<<fs_blocks(nc, 256), 256, 0, c->stream>>>(nc, M.partials.as<double>());
    k_fill_sentinel<<<fs_blocks(nc, 256), 256, 0, c->stream>>>(nc, M.partials2.as<double>());
    FS_HIP(c, hipGetLastError());
    M.nchunks = nc;
  }
  return FS_OK;
}

int mg_read_scalars(fs_ctx* c) {
  MgState& M = c->mg;
  FS_HIP(c, hipMemcpyAsync(M.host_scal, M.scal.p, sizeof(PcgScalars), hipMemcpyDeviceToHost, c->stream));
  FS_HIP(c, hipStreamSynchronize(c->stream));
  return FS_OK;
}

// Waits until iteration iter is finished or the solve has stopped.
int mg_wait(fs_ctx* c, int iter, bool* stopped) {
  for (unsigned n = 1;; n++) {
    bool idle = false;
    if (n % 1024 == 0) {  // a failed device never reports
      const hipError_t e = hipStreamQuery(c->stream);
      (void)hipGetLastError();  // "not ready" is not an error
      if (e != hipErrorNotReady) FS_HIP(c, e);
      idle = e == hipSuccess;
    }
    const int v = __atomic_load_n(c->mg.prog, __ATOMIC_RELAXED);
    *stopped = (v & MG_STOPPED) != 0;
    if (*stopped || v >= iter) return FS_OK;
    if (idle) {
      c->set_error("multigrid CG: an iteration ended without reporting");
      return FS_DEVICE_ERROR;
    }
    __builtin_ia32_pause();
  }
}

// Iterations queued beyond the last one reported. An iteration takes 60 us or more and queueing its 8 to
// 20 launches about half of that, so the device stays busy, and a solve that has stopped leaves two
// iterations of launches behind that return at once. Reading the scalars after every eighth iteration
// left up to seven, half of a solve of ten, and the device idle meanwhile (mixed, ms per pass: 64^3
// frames 14.6 / 12.9, 48^3 rollout 92 / 81, 256^3 frames alike).
constexpr int MG_AHEAD = 2;

template <typename S>
int mg_solve_t(fs_ctx* c, fs_stats* st) {
  MgState& M = c->mg;
  const int64_t n = c->n_cell;
  FS_TRY(mg_vectors(c));
  FS_TRY(mg_build<S>(c));
  const unsigned nb = chunks_of(n);
  const int nc = (int)nb;
  PcgScalars* sc = M.scal.as<PcgScalars>();
  PcgScalars* hs = M.host_scal;
  const int tmode = c->cfg.tol_mode;
  const double tol = c->cfg.cg_tolerance;
  const uint8_t* act = c->active.as<uint8_t>();
  FS_HIP(c, hipMemsetAsync(M.scal.p, 0, sizeof(PcgScalars), c->stream));
  k_mg_init<S><<<nb, 256, 0, c->stream>>>(n, act, c->rhs.as<S>(), M.x.as<double>(), M.r.as<double>(),
                                           M.s0.as<double>(), M.s1.as<double>(), M.t.as<double>(),
                                           M.partials.as<double>(), M.partials2.as<double>(), nc, sc, tmode, tol);
  FS_HIP(c, hipGetLastError());
  FS_TRY(mg_read_scalars(c));
  c->n_active_last = (int64_t)hs->n_active;
  int iters = 0, status = FS_OK;
  if (hs->converged == STOP_RUN) {
    MgLevelBuf& L0 = M.lv[0];
    const Lv<S> L = lv_of<S>(L0);
    FS_TRY(mg_cycle<S>(c, M.r.as<double>(), sc, true));
    const int maxit = c->cfg.cg_max_iterations;
    const int chk = std::max(1, c->cfg.check_interval), ahead = std::min(chk, MG_AHEAD);
    const bool timed = c->cfg.profile_stages >= 2 && c->ktime_on;  // kernels are timed one by one
    __atomic_store_n(M.prog, 0, __ATOMIC_RELAXED);  // nothing that writes it is queued
    int* prog = M.prog_dev;
    DBuf* sb[2] = {&M.s0, &M.s1};
    bool stopped = false;
    for (int it = 1; it < maxit && !stopped; it++) {
      if (!timed) {
        if (it > ahead) FS_TRY(mg_wait(c, it - ahead, &stopped));
        if (stopped) break;
      }
      const double* s_old = sb[(it + 1) & 1]->as<double>();
      double* s_new = sb[it & 1]->as<double>();
      int pf = fs_prof_begin(c, FS_KERNEL_SPMV, (24.0 + 5.0 * sizeof(S)) * c->n_active_last);
      auto spmv = [&](auto kern, int th) {
        kern<<<nb, th, 0, c->stream>>>(L, act, L0.x.as<S>(), s_old, s_new, M.t.as<double>(), M.partials.as<double>(),
                                       nc, sc, it, prog);
      };
      if (nb <= MG_WIDE) spmv(k_mg_spmv<S, 1024>, 1024);
      else spmv(k_mg_spmv<S, 256>, 256);
      fs_prof_end(c, pf);
      pf = fs_prof_begin(c, FS_KERNEL_PCG_UPDATE, 48.0 * c->n_active_last);
      auto update = [&](auto kern, int th) {
        kern<<<nb, th, 0, c->stream>>>(n, act, M.x.as<double>(), s_new, M.r.as<double>(), M.t.as<double>(),
                                       M.partials.as<double>(), M.partials2.as<double>(), nc, sc, it, tmode, tol,
                                       prog);
      };
      if (nb <= MG_WIDE) update(k_mg_update<1024>, 1024);
      else update(k_mg_update<256>, 256);
      fs_prof_end(c, pf);
      FS_TRY(mg_cycle<S>(c, M.r.as<double>(), sc, false));
      FS_HIP(c, hipGetLastError());
      if (timed && (it % chk == 0 || it + 1 == maxit)) {
        FS_TRY(mg_read_scalars(c));
        fs_prof_flush(c);
        stopped = hs->wait_timeouts != 0 || hs->converged != STOP_RUN;
      }
    }
    FS_TRY(mg_read_scalars(c));
    if (hs->wait_timeouts != 0) {
      c->set_error("multigrid CG: a reduction wait exceeded its bound");
      return FS_DEVICE_ERROR;
    }
    if (hs->converged == STOP_CONVERGED || hs->converged == STOP_ABORT) iters = hs->conv_iter;
    else iters = maxit;
    if (hs->converged == STOP_ABORT) status = hs->status;
    else if (hs->converged == STOP_RUN) status = FS_NOT_CONVERGED;
  }
  if (c->mixed)
    k_mg_store<float><<<fs_blocks(n, 256), 256, 0, c->stream>>>(n, M.x.as<double>(), c->pg.as<float>());
  else
    k_mg_store<double><<<fs_blocks(n, 256), 256, 0, c->stream>>>(n, M.x.as<double>(), c->pg.as<double>());
  FS_HIP(c, hipGetLastError());
  FS_HIP(c, hipStreamSynchronize(c->stream));
  if (st) {
    st->cg_iterations = iters;
    st->residual_inf = hs->residual;
    st->rhs_norm2 = std::sqrt(hs->bnorm2sq);
    st->residual_rel = hs->bnorm2sq > 0 ? std::sqrt(hs->rnorm2sq / hs->bnorm2sq) : 0.0;
    st->n_active = (int32_t)c->n_active_last;
    st->refinements = 0;
  }
  return status;
}

template <typename S>
int mg_apply_t(fs_ctx* c, const double* r, double* z) {
  MgState& M = c->mg;
  const int64_t n = c->n_cell;
  FS_TRY(mg_vectors(c));
  FS_TRY(mg_build<S>(c));
  // the cycle's right-hand side: r on active cells, 0 elsewhere
  std::vector<uint8_t> act(n);
  FS_HIP(c, hipMemcpyAsync(act.data(), c->active.p, n, hipMemcpyDeviceToHost, c->stream));
  FS_HIP(c, hipStreamSynchronize(c->stream));
  std::vector<double> host(n);
  for (int64_t q = 0; q < n; q++) host[q] = act[q] ? r[q] : 0.0;
  FS_HIP(c, hipMemcpyAsync(M.r.p, host.data(), n * sizeof(double), hipMemcpyHostToDevice, c->stream));
  FS_TRY(mg_cycle<S>(c, M.r.as<double>(), nullptr, false));
  return fs_download_real(c, M.lv[0].x, z, (size_t)n);
}

}  // namespace

int fs_mg_solve(fs_ctx* c, fs_stats* st) { return c->mixed ? mg_solve_t<float>(c, st) : mg_solve_t<double>(c, st); }

int fs_mg_apply_dense(fs_ctx* c, const double* r, double* z) {
  return c->mixed ? mg_apply_t<float>(c, r, z) : mg_apply_t<double>(c, r, z);
}

void fs_mg_release(fs_ctx* c) {
  MgState& M = c->mg;
  for (MgLevelBuf& B : M.lv)
    for (DBuf* d : {&B.D, &B.Cx, &B.Cy, &B.Cz, &B.W, &B.b, &B.x, &B.xs}) fs_free(*d);
  M.lv.clear();
  for (DBuf* d : {&M.x, &M.r, &M.s0, &M.s1, &M.t, &M.partials, &M.partials2, &M.scal}) fs_free(*d);
  if (M.host_scal) (void)hipHostFree(M.host_scal);
  M.host_scal = nullptr;
  if (M.prog) (void)hipHostFree(M.prog);
  M.prog = M.prog_dev = nullptr;
  M.nchunks = 0;
}
