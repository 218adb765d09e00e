// chy_mg.hip -- x-y semicoarsening multigrid preconditioner with a z-line
// smoother (-pc_type mg; PETSc's -pc_type gamg / hypre / ml map here).
//
// The electron operator couples z about 7.7e3 times more strongly than x and
// y (B along z, kappa_e = 88).  The smoother solves every z-line block of
// A(n) exactly (the cyclic tridiagonal systems of the fft2z correction,
// factored once per solve) and, damped by 0.8, removes the high x-y
// frequencies of the error; the coarse grids halve x and y only and keep every
// z plane, so the error the smoother leaves (smooth in x and y) is what they
// represent.  Level l has (N_x / 2^l, N_y / 2^l, N_z) nodes and spacings
// (2^l dx, 2^l dy, dz); its operator is the 19-point operator rediscretised
// from the density restricted to it (x-y full weighting), so every level
// runs the same stencil and z-line kernels as the fine grid.  One V(2,2)
// cycle from a zero guess per application, 8 sweeps on the coarsest level.
// Unlike the FFT preconditioners it needs no power-of-two axes, and with B along z
// its iteration counts do not grow with the grid or with the density contrast
// (a run's noise, to 1e-11: 15 on 48 x 40 x 26 and 64 x 48 x 40, 13 on 96 x 80 x
// 100).  With B oblique they do (50, 63, 93): the modes that oscillate in x and y
// and are constant along B are weak in A(n), stiff in a z-line block, and not
// represented on the coarse grids.
#include <utility>

#include "chy_internal.h"

namespace chy {

namespace {

constexpr int kMgMax = 8;
constexpr int kMgSweeps = 2;
constexpr int kMgCoarseSweeps = 8;
constexpr double kMgOmega = 0.8;

struct MgLevel {
  Grid g;
  double d[3];
  void *n = nullptr, *x = nullptr, *b = nullptr, *r = nullptr, *zf = nullptr;  // T arrays
  void *nz = nullptr, *x2 = nullptr;  // the density with z fastest, the sweeps' other x
  double *zcol = nullptr;  // per-column z-line scalars (2 per column)
};

struct Mg {
  int nlev = 0;
  MgLevel lv[kMgMax];
  bool zfast = false;   // level fields as [y][x][z] (at most kMgMaxPlanes planes)
};

// c = x-y full weighting of f (weights 1/4, 1/2, 1/4 along x and y, periodic).
// ZF: fields as [y][x][z].
template <bool ZF>
__device__ __forceinline__ int64_t mg_at(const Grid &g, int i, int j, int k)
{
  return ZF ? (int64_t)k + (int64_t)g.nz * ((int64_t)i + (int64_t)g.nx * j)
            : (int64_t)i + (int64_t)g.nx * ((int64_t)j + (int64_t)g.ny * k);
}

template <bool ZF>
__device__ __forceinline__ void mg_split(const Grid &g, int64_t q, int &i, int &j, int &k)
{
  if (ZF) {
    const uint32_t col = (uint32_t)q / (uint32_t)g.nz;  // nc < 2^31
    k = (int)((uint32_t)q - col * (uint32_t)g.nz);
    int z;
    split_cell(g, (int)col, i, j, z);
  } else {
    split_cell(g, (int)q, i, j, k);
  }
}

template <typename T, bool ZF>
__global__ __launch_bounds__(256) void k_mg_restrict(Grid gf, Grid gc, const T *__restrict__ f, T *__restrict__ c)
{
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= gc.nc) return;
  int I, J, k;
  mg_split<ZF>(gc, q, I, J, k);
  const double w[3] = {0.25, 0.5, 0.25};
  double s = 0.0;
#pragma unroll
  for (int bq = 0; bq < 3; bq++) {
    const int j = wrapi(2 * J + bq - 1, gf.ny);
#pragma unroll
    for (int a = 0; a < 3; a++) {
      const int i = wrapi(2 * I + a - 1, gf.nx);
      s += (w[bq] * w[a]) * (double)f[mg_at<ZF>(gf, i, j, k)];
    }
  }
  c[q] = (T)s;
}

// f += bilinear x-y interpolation of c.
template <typename T, bool ZF>
__global__ __launch_bounds__(256) void k_mg_prolong(Grid gf, Grid gc, const T *__restrict__ c, T *__restrict__ f)
{
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= gf.nc) return;
  int i, j, k;
  mg_split<ZF>(gf, q, i, j, k);
  const int I0 = i >> 1, J0 = j >> 1;
  const int I1 = (i & 1) ? (I0 + 1 == gc.nx ? 0 : I0 + 1) : I0, J1 = (j & 1) ? (J0 + 1 == gc.ny ? 0 : J0 + 1) : J0;
  const double v =
      0.25 * (((double)c[mg_at<ZF>(gc, I0, J0, k)] + (double)c[mg_at<ZF>(gc, I1, J0, k)]) +
              ((double)c[mg_at<ZF>(gc, I0, J1, k)] + (double)c[mg_at<ZF>(gc, I1, J1, k)]));
  f[q] = (T)((double)f[q] + v);
}

inline unsigned nb_of(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

// Level sizes: halve x and y while both stay even and at least 3 nodes.
int level_sizes(int64_t nx, int64_t ny, int64_t out[kMgMax][2])
{
  int L = 1;
  out[0][0] = nx; out[0][1] = ny;
  while (L < kMgMax && nx % 2 == 0 && ny % 2 == 0 && nx / 2 >= 3 && ny / 2 >= 3) {
    nx /= 2; ny /= 2;
    out[L][0] = nx; out[L][1] = ny;
    L++;
  }
  return L;
}

// The V-cycle on levels with z fastest: A x = b from zero; the result is in
// the returned buffer, L.x or L.x2.
template <typename T>
T *vcycle_z(chy_ctx *ctx, Mg &M, int l)
{
  MgLevel &L = M.lv[l];
  const Grid &g = L.g;
  const T *n = (const T *)L.nz, *zf = (const T *)L.zf, *b = (const T *)L.b;
  T *x = (T *)L.x, *y = (T *)L.x2;
  const bool coarsest = l == M.nlev - 1;
  launch_mg_sweep<T>(ctx, g, L.d, n, zf, L.zcol, b, (const T *)nullptr, x, kMgOmega);
  auto sweep = [&]() {
    launch_mg_sweep<T>(ctx, g, L.d, n, zf, L.zcol, b, (const T *)x, y, kMgOmega);
    std::swap(x, y);
  };
  for (int s = 1; s < (coarsest ? kMgCoarseSweeps : kMgSweeps); s++) sweep();
  if (coarsest) return x;
  MgLevel &C = M.lv[l + 1];
  launch_mg_residual<T>(ctx, g, L.d, n, b, (const T *)x, (T *)L.r);
  hipLaunchKernelGGL((k_mg_restrict<T, true>), nb_of(C.g.nc), kBlock, 0, ctx->stream, g, C.g, (const T *)L.r, (T *)C.b);
  const T *xc = vcycle_z<T>(ctx, M, l + 1);
  hipLaunchKernelGGL((k_mg_prolong<T, true>), nb_of(g.nc), kBlock, 0, ctx->stream, g, C.g, xc, x);
  for (int s = 0; s < kMgSweeps; s++) sweep();
  return x;
}

// The same with x fastest, for columns longer than kMgMaxPlanes.
template <typename T>
void vcycle(chy_ctx *ctx, Mg &M, int l, const T *b, T *x)
{
  MgLevel &L = M.lv[l];
  const Grid &g = L.g;
  const int lt = ctx->prm.lhs_type;
  const T *n = (const T *)L.n;
  T *r = (T *)L.r, *zf = (T *)L.zf;
  // first sweep from x = 0: x = omega zline^-1 b (the thread-per-column solve
  // overwrites its input, so it gets a copy)
  launch_fill<T>(ctx, g.nc, x, (T)0);
  (void)hipMemcpyAsync(r, b, sizeof(T) * g.nc, hipMemcpyDeviceToDevice, ctx->stream);
  launch_zline_apply_g<T>(ctx, g, zf, L.zcol, r, x, kMgOmega);
  auto sweep = [&]() {
    launch_residual_g<T>(ctx, g, L.d, lt, n, b, x, r);
    launch_zline_apply_g<T>(ctx, g, zf, L.zcol, r, x, kMgOmega);
  };
  const bool coarsest = l == M.nlev - 1;
  for (int s = 1; s < (coarsest ? kMgCoarseSweeps : kMgSweeps); s++) sweep();
  if (coarsest) return;
  MgLevel &C = M.lv[l + 1];
  launch_residual_g<T>(ctx, g, L.d, lt, n, b, x, r);
  hipLaunchKernelGGL((k_mg_restrict<T, false>), nb_of(C.g.nc), kBlock, 0, ctx->stream, g, C.g, (const T *)r, (T *)C.b);
  vcycle<T>(ctx, M, l + 1, (const T *)C.b, (T *)C.x);
  hipLaunchKernelGGL((k_mg_prolong<T, false>), nb_of(g.nc), kBlock, 0, ctx->stream, g, C.g, (const T *)C.x, x);
  for (int s = 0; s < kMgSweeps; s++) sweep();
}

}  // namespace

int mg_setup(chy_ctx *ctx)
{
  const chy_params &p = ctx->prm;
  Mg *M = new Mg();
  ctx->mg = M;
  int64_t sz[kMgMax][2];
  M->nlev = level_sizes(p.N[0], p.N[1], sz);
  M->zfast = p.N[2] <= kMgMaxPlanes;
  const size_t ts = ctx->mixed ? 4 : 8;
  // The finest level's fields but its factors lie in work arrays that the
  // other preconditioners use: its density in the FFT's second half (a transposed
  // solve's FFT overwrites it, and the next solve makes it anew).
  unsigned char *pcb = (unsigned char *)ctx->pc_buf, *ffb = (unsigned char *)ctx->fft_buf;
  for (int l = 0; l < M->nlev; l++) {
    MgLevel &L = M->lv[l];
    Grid &g = L.g;
    g = ctx->g;
    g.nx = (int)sz[l][0];
    g.ny = (int)sz[l][1];
    g.mx = fastdiv_magic((uint32_t)g.nx);
    g.my = fastdiv_magic((uint32_t)g.ny);
    g.nc = (int64_t)g.nx * g.ny * g.nz;
    L.d[0] = p.d[0] * (double)(p.N[0] / g.nx);
    L.d[1] = p.d[1] * (double)(p.N[1] / g.ny);
    L.d[2] = p.d[2];
    for (int a = 0; a < 3; a++) { g.d[a] = L.d[a]; g.rd[a] = 1.0 / L.d[a]; }
    const int64_t nc = g.nc, plane = (int64_t)g.nx * g.ny;
    unsigned char *q = nullptr;
    TRY(dalloc(ctx, &q, (int64_t)ts * 4 * nc)); L.zf = q;
    TRY(dalloc(ctx, &L.zcol, 2 * plane));
    if (l == 0) {
      L.x = pcb; L.x2 = pcb + ts * nc; L.b = pcb + 2 * ts * nc;
      L.r = ffb; L.nz = ffb + ts * nc;
      continue;
    }
    TRY(dalloc(ctx, &q, (int64_t)ts * nc)); L.r = q;
    TRY(dalloc(ctx, &q, (int64_t)ts * nc)); L.n = q;
    TRY(dalloc(ctx, &q, (int64_t)ts * nc)); L.x = q;
    TRY(dalloc(ctx, &q, (int64_t)ts * nc)); L.b = q;
    if (M->zfast) {
      TRY(dalloc(ctx, &q, (int64_t)ts * nc)); L.nz = q;
      TRY(dalloc(ctx, &q, (int64_t)ts * nc)); L.x2 = q;
    }
  }
  return CHY_OK;
}

void mg_release(chy_ctx *ctx)
{
  Mg *M = (Mg *)ctx->mg;
  if (!M) return;
  for (int l = 0; l < M->nlev; l++) {
    MgLevel &L = M->lv[l];
    void *own[] = {L.zf, L.zcol}, *coarse[] = {L.r, L.n, L.x, L.b, L.nz, L.x2};
    for (void *p : own) if (p) (void)hipFree(p);
    if (l == 0) continue;
    for (void *p : coarse) if (p) (void)hipFree(p);
  }
  delete M;
  ctx->mg = nullptr;
}

int mg_levels(const chy_ctx *ctx) { return ctx->mg ? ((const Mg *)ctx->mg)->nlev : 0; }

// Once per solve, before the Krylov basis holds anything: the density of every
// level and the z-line factors of every level's operator (made with x fastest in
// the basis' first four vectors).
template <typename T>
int mg_prepare(chy_ctx *ctx, const T *n)
{
  Mg *M = (Mg *)ctx->mg;
  if (!M) return set_err(ctx, CHY_ERR_LIB, "multigrid levels were not set up");
  M->lv[0].n = (void *)n;
  for (int l = 0; l < M->nlev; l++) {
    MgLevel &L = M->lv[l];
    if (l > 0)
      hipLaunchKernelGGL((k_mg_restrict<T, false>), nb_of(L.g.nc), kBlock, 0, ctx->stream, M->lv[l - 1].g, L.g,
                         (const T *)M->lv[l - 1].n, (T *)L.n);
    T *zf = M->zfast ? (T *)ctx->V : (T *)L.zf;
    launch_zline_factor_g<T>(ctx, L.g, L.d, ctx->prm.lhs_type, (const T *)L.n, zf, L.zcol);
    if (M->zfast) {
      const int64_t nc = L.g.nc;
      const T *src[5] = {(const T *)L.n, zf, zf + nc, zf + 2 * nc, zf + 3 * nc};
      T *lz = (T *)L.zf, *dst[5] = {(T *)L.nz, lz, lz + nc, lz + 2 * nc, lz + 3 * nc};
      launch_mg_transpose<T>(ctx, L.g, true, 5, src, dst);
    }
  }
  CHY_HIP(hipGetLastError());
  return CHY_OK;
}

// z = one V-cycle applied to r (level 0: the context's grid and density).
template <typename T>
int mg_apply(chy_ctx *ctx, const T *r, T *z)
{
  Mg *M = (Mg *)ctx->mg;
  if (!M || !M->lv[0].n) return set_err(ctx, CHY_ERR_LIB, "multigrid used before its set-up");
  if (M->zfast) {
    const Grid &g = M->lv[0].g;
    T *b = (T *)M->lv[0].b;
    launch_mg_transpose<T>(ctx, g, true, 1, &r, &b);
    const T *x = vcycle_z<T>(ctx, *M, 0);
    launch_mg_transpose<T>(ctx, g, false, 1, &x, &z);
  } else {
    vcycle<T>(ctx, *M, 0, r, z);
  }
  CHY_HIP(hipGetLastError());
  return CHY_OK;
}

template int mg_prepare<double>(chy_ctx *, const double *);
template int mg_prepare<float>(chy_ctx *, const float *);
template int mg_apply<double>(chy_ctx *, const double *, double *);
template int mg_apply<float>(chy_ctx *, const float *, float *);

}  // namespace chy
