// chy_grid.hip -- grid kernels for gfx950: the matrix-free 19-point electron
// operator (reference lhs.c:350-543), its residual and transpose, the node
// electric field, the forcing (rhs.c:8-303 with calculus.c stencils), and
// deterministic FP64 reductions for the Krylov solver.
//
// Every kernel is HBM-bound (no dense contraction), so the launches are
// shaped for coalesced x-fastest access; FP64 kernels use the oracle's
// operation order (the library is built with -ffp-contract=off).
#include <cmath>
#include <utility>

#include "chy_internal.h"

namespace chy {

SCoef full_scoef(const double d[3], const double K[3])
{
  const double Kx = K[0], Ky = K[1], Kz = K[2];
  const double detA = 1 + Kx * Kx + Ky * Ky + Kz * Kz;
  const double rxx = 1 + Kx * Kx, rxy = Ky * Kx - Kz, rxz = Kz * Kx + Ky;
  const double ryx = Kx * Ky + Kz, ryy = 1 + Ky * Ky, ryz = Kz * Ky - Kx;
  const double rzx = Kx * Kz - Ky, rzy = Ky * Kz + Kx, rzz = 1 + Kz * Kz;
  const double dx = d[0], dy = d[1], dz = d[2];
  const double hxx = 1.0 / (2.0 * dx * dx), hyy = 1.0 / (2.0 * dy * dy), hzz = 1.0 / (2.0 * dz * dz);
  const double hxy = 1.0 / (8.0 * dy * dx), hxz = 1.0 / (8.0 * dz * dx), hyz = 1.0 / (8.0 * dy * dz);
  const double scale = 1.0 / detA;
  SCoef s;
  s.sxx = scale * rxx * hxx; s.syy = scale * ryy * hyy; s.szz = scale * rzz * hzz;
  s.sxy = scale * rxy * hxy; s.sxz = scale * rxz * hxz; s.syz = scale * ryz * hyz;
  s.syx = scale * ryx * hxy; s.szx = scale * rzx * hxz; s.szy = scale * rzy * hyz;
  return s;
}

// Column offsets of one row, reference lhs.c:11-104.
__constant__ int kOff[19][3] = {
  {+1, 0, 0}, {-1, 0, 0}, {0, +1, 0}, {0, -1, 0}, {0, 0, +1}, {0, 0, -1},
  {+1, +1, 0}, {+1, -1, 0}, {-1, +1, 0}, {-1, -1, 0},
  {+1, 0, +1}, {+1, 0, -1}, {-1, 0, +1}, {-1, 0, -1},
  {0, +1, +1}, {0, +1, -1}, {0, -1, +1}, {0, -1, -1},
  {0, 0, 0}};
static const int hOff[19][3] = {
  {+1, 0, 0}, {-1, 0, 0}, {0, +1, 0}, {0, -1, 0}, {0, 0, +1}, {0, 0, -1},
  {+1, +1, 0}, {+1, -1, 0}, {-1, +1, 0}, {-1, -1, 0},
  {+1, 0, +1}, {+1, 0, -1}, {-1, 0, +1}, {-1, 0, -1},
  {0, +1, +1}, {0, +1, -1}, {0, -1, +1}, {0, -1, -1},
  {0, 0, 0}};

// Row coefficients from the 7-point density star (lhs.c:479-511).
template <typename C>
__host__ __device__ __forceinline__ void row_from_star(const SCoef &s, C nc, C nxp, C nxm, C nyp, C nym,
                                                       C nzp, C nzm, C v[19])
{
  const C sxx = (C)s.sxx, syy = (C)s.syy, szz = (C)s.szz, sxy = (C)s.sxy, sxz = (C)s.sxz;
  const C syz = (C)s.syz, syx = (C)s.syx, szx = (C)s.szx, szy = (C)s.szy;
  v[6] = sxy * (nxp + nc) + syx * (nyp + nc);
  v[7] = -sxy * (nxp + nc) - syx * (nc + nym);
  v[8] = -sxy * (nc + nxm) - syx * (nyp + nc);
  v[9] = sxy * (nc + nxm) + syx * (nc + nym);
  v[10] = sxz * (nxp + nc) + szx * (nzp + nc);
  v[11] = -sxz * (nxp + nc) - szx * (nc + nzm);
  v[12] = -sxz * (nc + nxm) - szx * (nzp + nc);
  v[13] = sxz * (nc + nxm) + szx * (nc + nzm);
  v[14] = syz * (nyp + nc) + szy * (nzp + nc);
  v[15] = -syz * (nyp + nc) - szy * (nc + nzm);
  v[16] = -syz * (nc + nym) - szy * (nzp + nc);
  v[17] = syz * (nc + nym) + szy * (nc + nzm);
  v[0] = sxx * (nxp + nc) + syx * (nyp - nym) + szx * (nzp - nzm);
  v[1] = sxx * (nc + nxm) - syx * (nyp - nym) - szx * (nzp - nzm);
  v[2] = syy * (nyp + nc) + sxy * (nxp - nxm) + szy * (nzp - nzm);
  v[3] = syy * (nc + nym) - sxy * (nxp - nxm) - szy * (nzp - nzm);
  v[4] = szz * (nzp + nc) + sxz * (nxp - nxm) + syz * (nyp - nym);
  v[5] = szz * (nc + nzm) - sxz * (nxp - nxm) - syz * (nyp - nym);
  v[18] = -(sxx * (nxp + 2 * nc + nxm) + syy * (nyp + 2 * nc + nym) + szz * (nzp + 2 * nc + nzm));
}

void uniform_row(int lhs_type, const double d[3], const double K[3], double nbar, double v[19])
{
  for (int q = 0; q < 19; q++) v[q] = 0.0;
  if (lhs_type == CHY_LHS_FULL) {
    const SCoef s = full_scoef(d, K);
    row_from_star<double>(s, nbar, nbar, nbar, nbar, nbar, nbar, nbar, v);
  } else if (lhs_type == CHY_LHS_LAPLACIAN) {
    const double sxx = d[1] * d[2] / d[0], syy = d[0] * d[2] / d[1], szz = d[0] * d[1] / d[2];
    v[0] = sxx; v[1] = sxx; v[2] = syy; v[3] = syy; v[4] = szz; v[5] = szz;
    v[18] = -(v[0] + v[2] + v[4] + v[1] + v[3] + v[5]);
  } else {
    v[18] = 1.0;
  }
}

// Coefficients of row c for any operator type (laplacian / identity rows are
// passed in lapv).
template <typename C, typename TN>
__device__ __forceinline__ void row_coeffs(const Grid &g, int lhs_type, const SCoef &s, const double *lapv,
                                           const TN *n, int i, int j, int k, C v[19])
{
  if (lhs_type == CHY_LHS_FULL) {
    const C nc = (C)n[lin(g, i, j, k)];
    row_from_star<C>(s, nc, (C)n[lin(g, i + 1, j, k)], (C)n[lin(g, i - 1, j, k)], (C)n[lin(g, i, j + 1, k)],
                     (C)n[lin(g, i, j - 1, k)], (C)n[lin(g, i, j, k + 1)], (C)n[lin(g, i, j, k - 1)], v);
  } else {
#pragma unroll
    for (int q = 0; q < 19; q++) v[q] = (C)lapv[q];
  }
}

struct LapRow { double v[19]; };

// kOff for compile-time indices, and f(q) for q = 0 .. 18 in order
static constexpr int cOff[19][3] = {
  {+1, 0, 0}, {-1, 0, 0}, {0, +1, 0}, {0, -1, 0}, {0, 0, +1}, {0, 0, -1},
  {+1, +1, 0}, {+1, -1, 0}, {-1, +1, 0}, {-1, -1, 0},
  {+1, 0, +1}, {+1, 0, -1}, {-1, 0, +1}, {-1, 0, -1},
  {0, +1, +1}, {0, +1, -1}, {0, -1, +1}, {0, -1, -1},
  {0, 0, 0}};
template <typename F, int... Q>
__device__ __forceinline__ void each_q(F &&f, std::integer_sequence<int, Q...>)
{
  (f(std::integral_constant<int, Q>()), ...);
}
// periodic index for i in [-2, n + 1], n >= 3
__device__ __forceinline__ int wrap2(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// y = A x (FP64: oracle order sum_q v_q x_q; FP32: difference form
// sum_q v_q (x_q - x_c), exact in exact arithmetic because rows sum to zero).
template <typename TN, typename TX, typename TY, typename C, bool DIFF>
__global__ __launch_bounds__(256) void k_lhs_apply(Grid g, int lhs_type, SCoef s, LapRow lap, const TN *__restrict__ n,
                                                   const TX *__restrict__ x, TY *__restrict__ y)
{
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.nc) return;
  const int i = (int)(c % g.nx), j = (int)((c / g.nx) % g.ny), k = (int)(c / ((int64_t)g.nx * g.ny));
  C v[19];
  row_coeffs<C, TN>(g, lhs_type, s, lap.v, n, i, j, k, v);
  C acc = (C)0;
  if (DIFF) {
    const C xc = (C)x[c];
#pragma unroll
    for (int q = 0; q < 18; q++) acc += v[q] * ((C)x[lin(g, i + kOff[q][0], j + kOff[q][1], k + kOff[q][2])] - xc);
  } else {
#pragma unroll
    for (int q = 0; q < 19; q++) acc += v[q] * (C)x[lin(g, i + kOff[q][0], j + kOff[q][1], k + kOff[q][2])];
  }
  y[c] = (TY)acc;
}

// Entry Q of row r from the densities around it, nat(dx, dy, dz) relative to
// r: row_from_star's entry alone.
template <typename C, int Q, typename F>
__device__ __forceinline__ C row_entry(const SCoef &s, F nat)
{
  C v[19];
  const C n0 = nat(0, 0, 0);
  const C xp = nat(1, 0, 0), xm = nat(-1, 0, 0), yp = nat(0, 1, 0), ym = nat(0, -1, 0), zp = nat(0, 0, 1),
          zm = nat(0, 0, -1);
  row_from_star<C>(s, n0, xp, xm, yp, ym, zp, zm, v);  // (the other entries are dead code)
  return v[Q];
}

// y = A^T x: (A^T x)_c = sum_q A[c - o_q, c] x[c - o_q]; the coefficient of
// column c in row r = c - o_q is that row's entry q.
template <typename TN, typename TX, typename TY, typename C, bool FULL>
__global__ __launch_bounds__(256) void k_lhs_apply_t(Grid g, SCoef s, LapRow lap, const TN *__restrict__ n,
                                                     const TX *__restrict__ x, TY *__restrict__ y)
{
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.nc) return;
  int i, j, k;
  split_cell(g, (int)c, i, j, k);
  // indices of the two nodes on each side (a row's star reaches one past its node)
  int64_t ox[5], oy[5], oz[5];
#pragma unroll
  for (int d = -2; d <= 2; d++) {
    ox[d + 2] = wrap2(i + d, g.nx);
    oy[d + 2] = (int64_t)g.nx * wrap2(j + d, g.ny);
    oz[d + 2] = (int64_t)g.nx * g.ny * wrap2(k + d, g.nz);
  }
  C acc = (C)0;
  auto term = [&](auto q_) {
    constexpr int q = decltype(q_)::value;
    constexpr int rx = -cOff[q][0], ry = -cOff[q][1], rz = -cOff[q][2];  // row r = c + (rx, ry, rz)
    C v;
    if constexpr (FULL)
      v = row_entry<C, q>(s, [&](int a, int b, int d) { return (C)n[ox[rx + a + 2] + oy[ry + b + 2] + oz[rz + d + 2]]; });
    else
      v = (C)lap.v[q];
    acc += v * (C)x[ox[rx + 2] + oy[ry + 2] + oz[rz + 2]];
  };
  each_q(term, std::make_integer_sequence<int, 19>());
  y[c] = (TY)acc;
}

// r = b - A x (FP64 outer residual).
template <typename TN, typename TX>
__global__ __launch_bounds__(256) void k_residual(Grid g, int lhs_type, SCoef s, LapRow lap, const TN *__restrict__ n,
                                                  const double *__restrict__ b, const TX *__restrict__ x,
                                                  double *__restrict__ r)
{
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.nc) return;
  const int i = (int)(c % g.nx), j = (int)((c / g.nx) % g.ny), k = (int)(c / ((int64_t)g.nx * g.ny));
  double v[19];
  row_coeffs<double, TN>(g, lhs_type, s, lap.v, n, i, j, k, v);
  double acc = 0.0;
#pragma unroll
  for (int q = 0; q < 19; q++) acc += v[q] * (double)x[lin(g, i + kOff[q][0], j + kOff[q][1], k + kOff[q][2])];
  r[c] = b[c] - acc;
}

// ---- LDS-tiled (2.5-D) operator apply ------------------------------------------
// A 64 x 4 thread block owns a (64 x 16) column of nodes (4 rows per thread)
// over kZChunk planes (TW = 256: a 256 x 1 block owns 256 x 8, 8 rows each).
// It keeps three z-planes of x and n, each with a one-node halo in x and y
// ((64+2) x (4+2) values), in LDS and marches up in z, loading one plane per
// step with coalesced x-fastest reads.  Output (OUT): 0 y = A x, 1 r = b - A x,
// 2 the column sums over the block's planes of b - A x, y[zc * nx * ny + col]
// for z chunk zc, plus the block's total in pl[block] (both in double),
// 3 r = b - A x and the block's sum of r^2 (in double) in pl[block], 4 as 2
// and also r = b - A x in d3.
constexpr int kTX = 64, kTY = 16, kRows = kTY / 4, kZChunk = 16;  // 64 x 4 threads, 4 rows each
constexpr int kHX = kTX + 2, kHY = kTY + 2;

// Each thread owns up to kPer elements of the (kHY x kHX) halo plane; their
// in-plane offsets are computed once (with the periodic wrap), and the next
// plane but one is prefetched into registers while the current one is
// computed from LDS, so global latency overlaps the arithmetic.
constexpr int kPer = (kHX * kHY + 255) / 256;

// Waves per SIMD asked of the compiler: the FP64 passes over an FP32 density
// fit three 64-wide tiles per CU in LDS, so their registers are held to three
// waves; the others keep the compiler's choice.
template <typename TN, typename C, int TW>
constexpr int tiled_waves() { return (sizeof(C) == 8 && sizeof(TN) == 4 && TW == 64) ? 3 : 1; }

// a * b + c: one fused multiply-add in FP32 (the mixed path's stencil); in
// FP64 the oracle's separate multiply and add (-ffp-contract=off)
template <typename C>
__device__ __forceinline__ C mad(C a, C b, C c)
{
  if constexpr (sizeof(C) == 4) return __builtin_fmaf(a, b, c);
  else return a * b + c;
}

// KZ: the full operator with B along z (K_x = K_y = 0, every workload of the
// benchmark definition): r_xz = r_zx = r_yz = r_zy = 0 (lhs.c:410-421), so
// the 8 x-z and y-z edge columns of each row (entries 10-17) and the
// cross-derivative terms of the face entries vanish, and the z +- 1 planes
// enter only through the row's own column.  A thread then takes RW
// consecutive rows and reads the x and n columns it shares between them from
// LDS once (12 LDS reads per node against 26).  The FP64 sum skips only
// exact zeros (v_q x_q = +-0 added to a non-zero sum), so it stays the
// oracle's bit for bit.
template <typename TN, typename TX, typename TY, typename C, bool DIFF, int OUT, typename TB = double, int TW = kTX,
          bool KZ = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(tiled_waves<TN, C, TW>())))
void k_lhs_tiled(Grid g, int lhs_type, SCoef s, LapRow lap,
                                                   const TN *__restrict__ n, const TX *__restrict__ x,
                                                   const TB *__restrict__ b, TY *__restrict__ y,
                                                   double *__restrict__ pl, TX *__restrict__ d3)
{
  constexpr bool ZS = OUT == 2 || OUT == 4;  // per-chunk column sums
  // tile TW x TY_ (TW = 64: 64 x 16; TW = 256, a whole x row of a 256-wide
  // grid: 256 x 8 with no x halo beyond the row's own periodic wrap), GW row
  // groups of TW threads, RW rows per thread
  constexpr int TY_ = TW == 256 ? 8 : kTY, GW = 256 / TW, RW = TY_ / GW;
  constexpr int HX = TW + 2, HY = TY_ + 2, PER = (HX * HY + 255) / 256;
  __shared__ C xs[3][HY][HX];
  // the density stays in its stored precision in LDS (FP32 density of an FP64
  // pass: half the bytes, exact on conversion at use)
  using NS = typename std::conditional<(sizeof(TN) < sizeof(C)), TN, C>::type;
  __shared__ NS ns[3][HY][HX];
  const bool full = KZ || lhs_type == CHY_LHS_FULL;
  const int tx = threadIdx.x % TW, ty0 = threadIdx.x / TW;
  // tile row of the thread's rr-th row: consecutive rows (KZ) or every GW-th
  auto row_of = [&](int rr) { return KZ ? ty0 * RW + rr : ty0 + GW * rr; };
  uint32_t bx, by, bz;
  const uint32_t tile = xcd_tile(bx, by, bz);
  const int x0 = bx * TW, y0 = by * TY_, z0 = bz * kZChunk;
  const int z1 = z0 + kZChunk < g.nz ? z0 + kZChunk : g.nz;
  const int i = x0 + tx;
  const int64_t pstride = (int64_t)g.nx * g.ny;
  // in-plane offsets and LDS slots of this thread's halo elements
  int64_t off[PER];
  int slot[PER];
#pragma unroll
  for (int q = 0; q < PER; q++) {
    const int e = threadIdx.x + 256 * q;
    slot[q] = e < HX * HY ? e : -1;
    const int hy = e / HX, hx = e - hy * HX;
    // tiles may overhang small grids by more than one period: full modulo
    int ii = x0 + hx - 1, jj = y0 + hy - 1;
    ii = ((ii % g.nx) + g.nx) % g.nx;
    jj = ((jj % g.ny) + g.ny) % g.ny;
    off[q] = (int64_t)ii + (int64_t)g.nx * jj;
  }
  C rx[PER];
  NS rn[PER];
  auto fetch = [&](int k) {
    const int64_t base = pstride * wrapi(k, g.nz);  // k in [-1, nz]
#pragma unroll
    for (int q = 0; q < PER; q++) {
      if (slot[q] >= 0) {
        rx[q] = (C)x[base + off[q]];
        if (full) rn[q] = (NS)n[base + off[q]];
      }
    }
  };
  auto store = [&](int buf) {
    C *xb = &xs[buf][0][0];
    NS *nb = &ns[buf][0][0];
#pragma unroll
    for (int q = 0; q < PER; q++) {
      if (slot[q] >= 0) {
        xb[slot[q]] = rx[q];
        if (full) nb[slot[q]] = rn[q];
      }
    }
  };
  double zs[RW];
#pragma unroll
  for (int rr = 0; rr < RW; rr++) zs[rr] = 0.0;
  // b at this thread's nodes of the current plane, and of the next one in flight
  TB rb[RW], rbn[RW];
  auto fetch_b = [&](int k, TB(&dst)[RW]) {
#pragma unroll
    for (int rr = 0; rr < RW; rr++) {
      const int j = y0 + row_of(rr);
      if (i < g.nx && j < g.ny) dst[rr] = b[(int64_t)i + (int64_t)g.nx * ((int64_t)j + (int64_t)g.ny * k)];
    }
  };
  if (OUT != 0) fetch_b(z0, rb);
  fetch(z0 - 1);
  store((z0 + 2) % 3);
  fetch(z0);
  store(z0 % 3);
  fetch(z0 + 1);
  for (int k = z0; k < z1; k++) {
    store((k + 1) % 3);
    __syncthreads();
    if (k + 1 < z1) {  // in flight while plane k is computed
      fetch(k + 2);
      if (OUT != 0) fetch_b(k + 1, rbn);
    }
    const int pm = (k + 2) % 3, pc = k % 3, pp = (k + 1) % 3;
    // the result at row rr of this plane
    auto emit = [&](int rr, int j, C acc) {
      const int64_t c = (int64_t)i + (int64_t)g.nx * ((int64_t)j + (int64_t)g.ny * k);
      if (OUT == 1) y[c] = (TY)((double)rb[rr] - (double)acc);
      else if (OUT == 2) zs[rr] += (double)rb[rr] - (double)acc;
      else if (OUT == 4) {
        const double rv = (double)rb[rr] - (double)acc;
        d3[c] = (TX)rv;
        zs[rr] += rv;
      }
      else if (OUT == 3) {
        const double rv = (double)rb[rr] - (double)acc;
        y[c] = (TY)rv;
        zs[rr] += rv * rv;
      } else y[c] = (TY)acc;
    };
    if constexpr (KZ) {
      const int hx = tx + 1, hyb = ty0 * RW + 1;
      // x at columns i-1, i, i+1 and n at column i, rows hyb-1 .. hyb+RW
      C xw[RW + 2], xo[RW + 2], xe[RW + 2], nm_[RW + 2];
#pragma unroll
      for (int r = 0; r < RW + 2; r++) {
        xw[r] = xs[pc][hyb - 1 + r][hx - 1];
        xo[r] = xs[pc][hyb - 1 + r][hx];
        xe[r] = xs[pc][hyb - 1 + r][hx + 1];
        nm_[r] = (C)ns[pc][hyb - 1 + r][hx];
      }
      const C sxx = (C)s.sxx, syy = (C)s.syy, szz = (C)s.szz, sxy = (C)s.sxy, syx = (C)s.syx;
#pragma unroll
      for (int rr = 0; rr < RW; rr++) {
        const int j = y0 + row_of(rr), hy = hyb + rr;
        if (i < g.nx && j < g.ny) {
          const C nc = nm_[rr + 1], nyp = nm_[rr + 2], nym = nm_[rr];
          const C nxp = (C)ns[pc][hy][hx + 1], nxm = (C)ns[pc][hy][hx - 1];
          const C nzp = (C)ns[pp][hy][hx], nzm = (C)ns[pm][hy][hx];
          // entries 0-9 and 18 of row_from_star with s_xz = s_yz = s_zx = s_zy = 0
          const C a = nxp + nc, bq = nc + nxm, cq = nyp + nc, dq = nc + nym;
          const C dy = nyp - nym, dx = nxp - nxm;
          C v[10];
          v[0] = mad(sxx, a, syx * dy);
          v[1] = mad(sxx, bq, -(syx * dy));
          v[2] = mad(syy, cq, sxy * dx);
          v[3] = mad(syy, dq, -(sxy * dx));
          v[4] = szz * (nzp + nc);
          v[5] = szz * (nc + nzm);
          v[6] = mad(sxy, a, syx * cq);
          v[7] = mad(-sxy, a, -(syx * dq));
          v[8] = mad(-sxy, bq, -(syx * cq));
          v[9] = mad(sxy, bq, syx * dq);
          // -((sxx X + syy Y) + szz Z), the oracle's association
          const C v18 = -(mad(szz, nzp + 2 * nc + nzm, mad(sxx, nxp + 2 * nc + nxm, syy * (nyp + 2 * nc + nym))));
          const C xv[10] = {xe[rr + 1], xw[rr + 1], xo[rr + 2], xo[rr], xs[pp][hy][hx], xs[pm][hy][hx],
                            xe[rr + 2], xe[rr], xw[rr + 2], xw[rr]};
          const C xc = xo[rr + 1];
          C acc = (C)0;
          if (DIFF) {
#pragma unroll
            for (int q = 0; q < 10; q++) acc = mad(v[q], xv[q] - xc, acc);
          } else {
#pragma unroll
            for (int q = 0; q < 10; q++) acc += v[q] * xv[q];
            acc += v18 * xc;
          }
          emit(rr, j, acc);
        }
      }
    } else {
#pragma unroll
    for (int rr = 0; rr < RW; rr++) {
      const int ty = row_of(rr), j = y0 + ty;
      if (i < g.nx && j < g.ny) {
        const int hx = tx + 1, hy = ty + 1;
        C v[19];
        if (full) {
          row_from_star<C>(s, ns[pc][hy][hx], ns[pc][hy][hx + 1], ns[pc][hy][hx - 1], ns[pc][hy + 1][hx],
                           ns[pc][hy - 1][hx], ns[pp][hy][hx], ns[pm][hy][hx], v);
        } else {
#pragma unroll
          for (int q = 0; q < 19; q++) v[q] = (C)lap.v[q];
        }
        // x at the 19 columns, in the column order of the row
        const C xv[19] = {
          xs[pc][hy][hx + 1], xs[pc][hy][hx - 1], xs[pc][hy + 1][hx], xs[pc][hy - 1][hx], xs[pp][hy][hx],
          xs[pm][hy][hx], xs[pc][hy + 1][hx + 1], xs[pc][hy - 1][hx + 1], xs[pc][hy + 1][hx - 1],
          xs[pc][hy - 1][hx - 1], xs[pp][hy][hx + 1], xs[pm][hy][hx + 1], xs[pp][hy][hx - 1], xs[pm][hy][hx - 1],
          xs[pp][hy + 1][hx], xs[pm][hy + 1][hx], xs[pp][hy - 1][hx], xs[pm][hy - 1][hx], xs[pc][hy][hx]};
        C acc = (C)0;
        if (DIFF) {
#pragma unroll
          for (int q = 0; q < 18; q++) acc = mad(v[q], xv[q] - xv[18], acc);
        } else {
#pragma unroll
          for (int q = 0; q < 19; q++) acc += v[q] * xv[q];
        }
        emit(rr, j, acc);
      }
    }
    }
    if (OUT != 0) {
#pragma unroll
      for (int rr = 0; rr < RW; rr++) rb[rr] = rbn[rr];
    }
    __syncthreads();
  }
  if (ZS || OUT == 3) {
    __shared__ double wsum[4];
    double t = 0.0;
#pragma unroll
    for (int rr = 0; rr < RW; rr++) {
      const int j = y0 + row_of(rr);
      if (i < g.nx && j < g.ny) {
        if (ZS) y[(int64_t)bz * pstride + i + (int64_t)g.nx * j] = (TY)zs[rr];
        t += zs[rr];
      }
    }
    t = wave_total(t);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0) pl[tile] = ((wsum[0] + wsum[1]) + wsum[2]) + wsum[3];
  }
}

// ---- column stencil --------------------------------------------------------------
// One thread per (i, j) column of a chunk of planes, no LDS and no barriers:
// each group of kColZ planes loads its stencil straight from the caches (the
// x-y neighbours are other lanes' centres, so L1 and L2 serve them) with every
// load of the group in flight at once, and the z neighbours are shared between
// the group's planes in registers.
//
// On grids that fit the caches the tiled kernel below is bound by its serial
// march through 16 planes (two barriers a plane) on few tiles: 8 blocks at
// 32^3, 128 at 128^3.  Here a launch has 1024 blocks where the grid gives them
// (chunks of 4 to 16 planes).  Measured, tiled -> column, us per pass of A x:
// 32^3 FP64 25.7 -> 5.3, 64^3 FP32 20.5 -> 4.6, 128^3 FP32 21.6 -> 9.4, 128^3
// FP64 28.4 -> 20.0, 256x256x64 FP32 22.9 -> 14.9; with B oblique 128^3 FP32
// 35.0 -> 10.6.  Larger grids: 15 loads a node (FP64 twice the bytes) reach
// the L1's rate before the tiles' LDS does: 256x256x64 FP64 30.3 -> 39.3,
// 256x256x128 FP32 27.9 -> 28.6 (column sums 44.7 -> 30.0), 256^3 FP32 53 ->
// 72 and FP64 99 -> 199.  col_stencil draws the line between them.  Four planes
// a group measured best or level for both types (1, 2, 4 and 8 tried).
constexpr int kColZ = 4;
constexpr int kColDots = 8;  // most dot products taken with A x
static inline bool col_stencil(const Grid &g, bool fp32) { return g.nc <= (fp32 ? (int64_t)1 << 23 : (int64_t)1 << 21); }

// Planes per chunk: 1024 blocks of columns, in whole groups, at most kZChunk
static inline int col_chunk(const Grid &g)
{
  const int64_t nb = ((int64_t)g.nx * g.ny + 255) / 256;
  const int64_t zc = (g.nz * nb + 1023) / 1024;
  return (int)std::min<int64_t>(kZChunk, (zc + kColZ - 1) / kColZ * kColZ);
}

static inline dim3 col_grid(const Grid &g)
{
  const int zc = col_chunk(g);
  return dim3((unsigned)(((int64_t)g.nx * g.ny + 255) / 256), (unsigned)((g.nz + zc - 1) / zc));
}

enum { kOpKz, kOpFull, kOpConst };  // the full operator with B along z, any B, a constant row

// Row c of A times x from the values around it.  Densities: the centre n0, the
// faces nf = x+, x-, y+, y- and z+, z- (unused with kOpConst); x: the centre
// x0, the faces xf, the x-y edges xe = ++, +-, -+, --, the z neighbours, and
// their faces xfp, xfm (the x-z and y-z edges; unused with kOpKz).  The
// oracle's order of operations in FP64; FP32 sums v_q (x_q - x_c) (DIFF).
template <typename C, bool DIFF, int OP>
__device__ __forceinline__ C row_apply(const SCoef &s, const LapRow &lap, C n0, const C (&nf)[4], C nzp, C nzm, C x0,
                                       const C (&xf)[4], const C (&xe)[4], C xzp, C xzm, const C (&xfp)[4],
                                       const C (&xfm)[4])
{
  C acc = (C)0;
  if constexpr (OP == kOpKz) {
    const C sxx = (C)s.sxx, syy = (C)s.syy, szz = (C)s.szz, sxy = (C)s.sxy, syx = (C)s.syx;
    const C nxp = nf[0], nxm = nf[1], nyp = nf[2], nym = nf[3];
    // entries 0-9 and 18 of row_from_star with s_xz = s_yz = s_zx = s_zy = 0
    const C a = nxp + n0, bq = n0 + nxm, cq = nyp + n0, dq = n0 + nym;
    const C dy = nyp - nym, dx = nxp - nxm;
    C w[10];
    w[0] = mad(sxx, a, syx * dy);
    w[1] = mad(sxx, bq, -(syx * dy));
    w[2] = mad(syy, cq, sxy * dx);
    w[3] = mad(syy, dq, -(sxy * dx));
    w[4] = szz * (nzp + n0);
    w[5] = szz * (n0 + nzm);
    w[6] = mad(sxy, a, syx * cq);
    w[7] = mad(-sxy, a, -(syx * dq));
    w[8] = mad(-sxy, bq, -(syx * cq));
    w[9] = mad(sxy, bq, syx * dq);
    // -((sxx X + syy Y) + szz Z), the oracle's association
    const C w18 = -(mad(szz, nzp + 2 * n0 + nzm, mad(sxx, nxp + 2 * n0 + nxm, syy * (nyp + 2 * n0 + nym))));
    const C xv[10] = {xf[0], xf[1], xf[2], xf[3], xzp, xzm, xe[0], xe[1], xe[2], xe[3]};
    if (DIFF) {
#pragma unroll
      for (int q = 0; q < 10; q++) acc = mad(w[q], xv[q] - x0, acc);
    } else {
#pragma unroll
      for (int q = 0; q < 10; q++) acc += w[q] * xv[q];
      acc += w18 * x0;
    }
  } else {
    C w[19];
    if constexpr (OP == kOpFull) {
      row_from_star<C>(s, n0, nf[0], nf[1], nf[2], nf[3], nzp, nzm, w);
    } else {
#pragma unroll
      for (int q = 0; q < 19; q++) w[q] = (C)lap.v[q];
    }
    const C xv[19] = {xf[0],  xf[1],  xf[2],  xf[3],  xzp,    xzm,    xe[0],  xe[1],  xe[2], xe[3],
                      xfp[0], xfm[0], xfp[1], xfm[1], xfp[2], xfm[2], xfp[3], xfm[3], x0};
    if (DIFF) {
#pragma unroll
      for (int q = 0; q < 18; q++) acc = mad(w[q], xv[q] - xv[18], acc);
    } else {
#pragma unroll
      for (int q = 0; q < 19; q++) acc += w[q] * xv[q];
    }
  }
  return acc;
}
// base + a 32-bit byte offset within a plane (a plane of 4 GB does not fit
// beside the solver's vectors), so that the plane's address stays scalar
template <typename T>
__device__ __forceinline__ T ld_off(const T *__restrict__ base, uint32_t byte_off)
{
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + byte_off);
}

template <typename TN, typename TX, typename TY, typename C, bool DIFF, int OUT, typename TB, int OP>
__global__ __launch_bounds__(256) void k_lhs_col(Grid g, int zc, SCoef s, LapRow lap, const TN *__restrict__ n,
                                                 const TX *__restrict__ x, const TB *__restrict__ b,
                                                 TY *__restrict__ y, double *__restrict__ pl, TX *__restrict__ d3,
                                                 int nv, int64_t vs)
{
  constexpr bool ZS = OUT == 2 || OUT == 4, KZ = OP == kOpKz;
  constexpr int ZR = kColZ;
  double dots[OUT == 5 ? kColDots : 1] = {};
  uint32_t bx, by, bz;
  const uint32_t tile = xcd_tile(bx, by, bz);
  const int64_t pstride = (int64_t)g.nx * g.ny;
  const int col = (int)(bx * 256 + threadIdx.x);
  const bool live = col < (int)pstride;
  int i, j, k_;
  split_cell(g, live ? col : 0, i, j, k_);
  const int ip = i + 1 == g.nx ? 0 : i + 1, im = i == 0 ? g.nx - 1 : i - 1;
  const int jp = j + 1 == g.ny ? 0 : j + 1, jm = j == 0 ? g.ny - 1 : j - 1;
  const uint32_t c0 = (uint32_t)(i + g.nx * j), cxp = (uint32_t)(ip + g.nx * j), cxm = (uint32_t)(im + g.nx * j),
                 cyp = (uint32_t)(i + g.nx * jp), cym = (uint32_t)(i + g.nx * jm),
                 cpp = (uint32_t)(ip + g.nx * jp), cpm = (uint32_t)(ip + g.nx * jm),
                 cmp = (uint32_t)(im + g.nx * jp), cmm = (uint32_t)(im + g.nx * jm);
  const int z0 = (int)by * zc, z1 = z0 + zc < g.nz ? z0 + zc : g.nz;
  double zs = 0.0;
  if (live) {
    for (int k0 = z0; k0 < z1; k0 += ZR) {
      // planes k0 - 1 .. k0 + ZR: the centre, and (unless KZ) the four face neighbours
      C xc[ZR + 2], nc[ZR + 2], xf[ZR + 2][4], xe[ZR][4], nf[ZR][4];
      TB rb[ZR];
#pragma unroll
      for (int u = 0; u < ZR + 2; u++) {
        int k = k0 - 1 + u;
        if (k > z1) k = z1;  // past the chunk: any plane in range
        const int64_t pb = pstride * wrapi(k, g.nz);
        const TX *xp = x + pb;
        const TN *np = n + pb;
        xc[u] = (C)ld_off(xp, c0 * (uint32_t)sizeof(TX));
        if (OP != kOpConst) nc[u] = (C)ld_off(np, c0 * (uint32_t)sizeof(TN));
        const bool inner = u >= 1 && u <= ZR;
        if (inner || !KZ) {
          xf[u][0] = (C)ld_off(xp, cxp * (uint32_t)sizeof(TX));
          xf[u][1] = (C)ld_off(xp, cxm * (uint32_t)sizeof(TX));
          xf[u][2] = (C)ld_off(xp, cyp * (uint32_t)sizeof(TX));
          xf[u][3] = (C)ld_off(xp, cym * (uint32_t)sizeof(TX));
        }
        if (inner) {
          const int v = u - 1;
          xe[v][0] = (C)ld_off(xp, cpp * (uint32_t)sizeof(TX));
          xe[v][1] = (C)ld_off(xp, cpm * (uint32_t)sizeof(TX));
          xe[v][2] = (C)ld_off(xp, cmp * (uint32_t)sizeof(TX));
          xe[v][3] = (C)ld_off(xp, cmm * (uint32_t)sizeof(TX));
          if (OP != kOpConst) {
            nf[v][0] = (C)ld_off(np, cxp * (uint32_t)sizeof(TN));
            nf[v][1] = (C)ld_off(np, cxm * (uint32_t)sizeof(TN));
            nf[v][2] = (C)ld_off(np, cyp * (uint32_t)sizeof(TN));
            nf[v][3] = (C)ld_off(np, cym * (uint32_t)sizeof(TN));
          }
          if (OUT != 0 && OUT != 5) rb[v] = ld_off(b + pb, c0 * (uint32_t)sizeof(TB));
        }
      }
      TY yv[ZR];
#pragma unroll
      for (int v = 0; v < ZR; v++) {
        const int u = v + 1, k = k0 + v;
        if (OUT == 5) yv[v] = (TY)0;
        if (k >= z1) break;
        const C acc = row_apply<C, DIFF, OP>(s, lap, nc[u], nf[v], nc[u + 1], nc[u - 1], xc[u], xf[u], xe[v], xc[u + 1],
                                             xc[u - 1], xf[u + 1], xf[u - 1]);
        const int64_t c = (int64_t)c0 + pstride * k;
        if (OUT == 0 || OUT == 5) {
          y[c] = (TY)acc;
          yv[v] = (TY)acc;
        } else {
          const double rv = (double)rb[v] - (double)acc;
          if (OUT == 1 || OUT == 3) y[c] = (TY)rv;
          if (OUT == 4) d3[c] = (TX)rv;
          if (ZS) zs += rv;
          if (OUT == 3) zs += rv * rv;
        }
      }
      if (OUT == 5) {
#pragma unroll
        for (int q = 0; q < kColDots; q++) {
          if (q < nv) {
            TB bv[ZR];
#pragma unroll
            for (int v = 0; v < ZR; v++) {
              const int k = k0 + v < z1 ? k0 + v : z1 - 1;  // (past the chunk: yv is 0)
              bv[v] = ld_off(b + q * vs + pstride * k, c0 * (uint32_t)sizeof(TB));
            }
#pragma unroll
            for (int v = 0; v < ZR; v++)
              if (k0 + v < z1) dots[q] += (double)bv[v] * (double)yv[v];
          }
        }
      }
    }
    if (ZS) y[(int64_t)by * pstride + c0] = (TY)zs;
  }
  if (ZS || OUT == 3) {
    __shared__ double wsum[4];
    double t = zs;
    t = wave_total(t);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0) pl[tile] = ((wsum[0] + wsum[1]) + wsum[2]) + wsum[3];
  }
  if (OUT == 5) {
    __shared__ double dsum[4][kColDots];
#pragma unroll
    for (int q = 0; q < kColDots; q++) {
      if (q < nv) {
        double t = dots[q];
        t = wave_total(t);
        if ((threadIdx.x & 63) == 0) dsum[threadIdx.x >> 6][q] = t;
      }
    }
    __syncthreads();
    if (threadIdx.x < nv)
      pl[(int64_t)tile * nv + threadIdx.x] = ((dsum[0][threadIdx.x] + dsum[1][threadIdx.x]) + dsum[2][threadIdx.x]) +
                                             dsum[3][threadIdx.x];
  }
}

static inline dim3 tiled_grid(const Grid &g, int tw = kTX)
{
  const int ty = tw == 256 ? 8 : kTY;
  return dim3((unsigned)((g.nx + tw - 1) / tw), (unsigned)((g.ny + ty - 1) / ty),
              (unsigned)((g.nz + kZChunk - 1) / kZChunk));
}

// The FP32 residual passes of the preconditioner (b - A x, and its z-chunk
// column sums) on a 256-wide grid take whole rows as tiles: the one-node x
// halo of a 64-wide tile costs two extra cache lines per row (twice the x
// traffic), a whole row's halo is its own wrap.  (A x alone, with a third
// less traffic, ran faster at the 64-wide tiles' higher occupancy.)
static inline bool wide_rows(const Grid &g, bool fp32) { return fp32 && g.nx == 256; }

static LapRow lap_row(chy_ctx *ctx, int lhs_type)
{
  LapRow L;
  uniform_row(lhs_type == CHY_LHS_FULL ? CHY_LHS_IDENTITY : lhs_type, ctx->prm.d, ctx->prm.kappa_e, 0.0, L.v);
  return L;
}

static inline unsigned nblocks(int64_t n, int b = kBlock) { return (unsigned)((n + b - 1) / b); }

// The full operator with B along z (see k_lhs_tiled's KZ).
static inline bool kz_operator(int lhs_type, const SCoef &s)
{
  return lhs_type == CHY_LHS_FULL && s.sxz == 0.0 && s.syz == 0.0 && s.szx == 0.0 && s.szy == 0.0;
}

// One stencil pass on grid g: the column kernel on grids it suits, else the tiled
// one; the B-along-z instantiation when it applies.
template <typename TN, typename TX, typename TY, typename C, bool DIFF, int OUT, typename TB = double, int TW = kTX>
static void launch_tiled_on(chy_ctx *ctx, const Grid &g, const SCoef &s, const LapRow &L, int lhs_type, const TN *n,
                            const TX *x, const TB *b, TY *y, double *pl, TX *d3 = nullptr, int nv = 0, int64_t vs = 0)
{
  if (OUT == 5 || col_stencil(g, sizeof(C) == 4)) {
#define COLK(OP)                                                                                                  \
  hipLaunchKernelGGL((k_lhs_col<TN, TX, TY, C, DIFF, OUT, TB, OP>), col_grid(g), 256, 0, ctx->stream, g, col_chunk(g), \
                     s, L, n, x, b, y, pl, d3, nv, vs)
    if (kz_operator(lhs_type, s)) COLK(kOpKz);
    else if (lhs_type == CHY_LHS_FULL) COLK(kOpFull);
    else COLK(kOpConst);
#undef COLK
    return;
  }
  if constexpr (OUT == 5) return;
  else if (kz_operator(lhs_type, s))
    hipLaunchKernelGGL((k_lhs_tiled<TN, TX, TY, C, DIFF, OUT, TB, TW, true>), tiled_grid(g, TW), kBlock, 0,
                       ctx->stream, g, lhs_type, s, L, n, x, b, y, pl, d3);
  else
    hipLaunchKernelGGL((k_lhs_tiled<TN, TX, TY, C, DIFF, OUT, TB, TW, false>), tiled_grid(g, TW), kBlock, 0,
                       ctx->stream, g, lhs_type, s, L, n, x, b, y, pl, d3);
}

// The same on the context's grid.
template <typename TN, typename TX, typename TY, typename C, bool DIFF, int OUT, typename TB = double, int TW = kTX>
static void launch_tiled(chy_ctx *ctx, int lhs_type, const TN *n, const TX *x, const TB *b, TY *y, double *pl,
                         TX *d3 = nullptr)
{
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  const LapRow L = lap_row(ctx, lhs_type);
  launch_tiled_on<TN, TX, TY, C, DIFF, OUT, TB, TW>(ctx, ctx->g, s, L, lhs_type, n, x, b, y, pl, d3);
}

template <typename TN, typename TX, typename TY>
void launch_lhs_apply(chy_ctx *ctx, int lhs_type, bool transpose, const TN *n, const TX *x, TY *y)
{
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  const LapRow L = lap_row(ctx, lhs_type);
  constexpr bool fp32 = sizeof(TX) == 4 && sizeof(TY) == 4;
  using C = typename std::conditional<fp32, float, double>::type;
  if (transpose)
  {
    if (lhs_type == CHY_LHS_FULL)
      hipLaunchKernelGGL((k_lhs_apply_t<TN, TX, TY, C, true>), nblocks(ctx->g.nc), kBlock, 0, ctx->stream, ctx->g, s,
                         L, n, x, y);
    else
      hipLaunchKernelGGL((k_lhs_apply_t<TN, TX, TY, C, false>), nblocks(ctx->g.nc), kBlock, 0, ctx->stream, ctx->g, s,
                         L, n, x, y);
  }
  else
    launch_tiled<TN, TX, TY, C, fp32, 0>(ctx, lhs_type, n, x, (const double *)nullptr, y, (double *)nullptr);
}

// y = A x with one partial of V_q . y, q < nv, per block in ctx->red; returns
// the number of partials, or 0 with nothing launched where the column kernel
// does not run or would leave more of them than the reduction buffer takes.
template <typename T>
int launch_lhs_dots(chy_ctx *ctx, int lhs_type, const T *n, const T *x, T *y, int nv, const T *V, int64_t stride)
{
  constexpr bool fp32 = sizeof(T) == 4;
  using C = typename std::conditional<fp32, float, double>::type;
  const Grid &g = ctx->g;
  const dim3 d = col_grid(g);
  if (nv > kColDots || !col_stencil(g, fp32) || (int64_t)d.x * d.y > kRedBlocks) return 0;
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  const LapRow L = lap_row(ctx, lhs_type);
  launch_tiled_on<T, T, T, C, fp32, 5, T>(ctx, g, s, L, lhs_type, n, x, V, y, ctx->red, nullptr, nv, stride);
  return (int)(d.x * d.y);
}
template int launch_lhs_dots<double>(chy_ctx *, int, const double *, const double *, double *, int, const double *, int64_t);
template int launch_lhs_dots<float>(chy_ctx *, int, const float *, const float *, float *, int, const float *, int64_t);

int lhs_zchunks(const Grid &g, bool fp32)
{
  return col_stencil(g, fp32) ? (int)col_grid(g).y : (g.nz + kZChunk - 1) / kZChunk;
}
int64_t lhs_zsum_blocks(const Grid &g, bool fp32)
{
  const dim3 d = col_stencil(g, fp32) ? col_grid(g) : tiled_grid(g, wide_rows(g, fp32) ? 256 : kTX);
  return (int64_t)d.x * d.y * d.z;
}

template <typename T>
void launch_lhs_zsum(chy_ctx *ctx, int lhs_type, const T *n, const T *x, const T *b, double *part, double *pl, T *r)
{
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  const LapRow L = lap_row(ctx, lhs_type);
  constexpr bool fp32 = sizeof(T) == 4;
  using C = typename std::conditional<fp32, float, double>::type;
  if constexpr (fp32) {
    if (wide_rows(ctx->g, fp32)) {
      if (r) launch_tiled<T, T, double, C, fp32, 4, T, 256>(ctx, lhs_type, n, x, b, part, pl, r);
      else launch_tiled<T, T, double, C, fp32, 2, T, 256>(ctx, lhs_type, n, x, b, part, pl);
      return;
    }
  }
  if (r) launch_tiled<T, T, double, C, fp32, 4, T>(ctx, lhs_type, n, x, b, part, pl, r);
  else launch_tiled<T, T, double, C, fp32, 2, T>(ctx, lhs_type, n, x, b, part, pl);
}

// r = b - A x in FP64 arithmetic, stored as TY, and one partial of |r|^2 per
// stencil block in pl (lhs_zsum_blocks(g, false) of them).
template <typename TN, typename TY>
void launch_residual_norm(chy_ctx *ctx, int lhs_type, const TN *n, const double *b, const double *x, TY *r,
                          double *pl)
{
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  const LapRow L = lap_row(ctx, lhs_type);
  launch_tiled<TN, double, TY, double, false, 3>(ctx, lhs_type, n, x, b, r, pl);
}

// r = b - A x in the inner precision (a GMRES restart's residual; the same
// arithmetic as A x followed by b - y), with one FP64 partial of |r|^2 per
// stencil block in pl; returns the number of partials
template <typename T>
int64_t launch_residual_sq(chy_ctx *ctx, int lhs_type, const T *n, const T *b, const T *x, T *r, double *pl)
{
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  const LapRow L = lap_row(ctx, lhs_type);
  constexpr bool fp32 = sizeof(T) == 4;
  using C = typename std::conditional<fp32, float, double>::type;
  if constexpr (fp32) {
    if (wide_rows(ctx->g, fp32)) {
      launch_tiled<T, T, T, C, fp32, 3, T, 256>(ctx, lhs_type, n, x, b, r, pl);
      return lhs_zsum_blocks(ctx->g, fp32);
    }
  }
  launch_tiled<T, T, T, C, fp32, 3, T>(ctx, lhs_type, n, x, b, r, pl);
  return lhs_zsum_blocks(ctx->g, fp32);
}

// y += a x, x of any precision, y FP64
template <typename TS>
__global__ __launch_bounds__(256) void k_add_scaled(int64_t n, const TS *__restrict__ x, double a, double *__restrict__ y)
{
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    y[i] = (double)x[i] * a + y[i];
}

template <typename TS>
void launch_add_scaled(chy_ctx *ctx, int64_t n, const TS *x, double a, double *y)
{
  const unsigned nb = (unsigned)std::min<int64_t>(8192, (n + kBlock - 1) / kBlock);
  hipLaunchKernelGGL((k_add_scaled<TS>), nb, kBlock, 0, ctx->stream, n, x, a, y);
}

template <typename TN, typename TX>
void launch_residual(chy_ctx *ctx, int lhs_type, const TN *n, const double *b, const TX *x, double *r)
{
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  const LapRow L = lap_row(ctx, lhs_type);
  launch_tiled<TN, TX, double, double, false, 1>(ctx, lhs_type, n, x, b, r, (double *)nullptr);
}

template <typename T>
__global__ __launch_bounds__(256) void k_jacobi(Grid g, int lhs_type, SCoef s, LapRow lap, const T *__restrict__ n,
                                                const T *__restrict__ r, T *__restrict__ z)
{
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.nc) return;
  const int i = (int)(c % g.nx), j = (int)((c / g.nx) % g.ny), k = (int)(c / ((int64_t)g.nx * g.ny));
  double v[19];
  row_coeffs<double, T>(g, lhs_type, s, lap.v, n, i, j, k, v);
  z[c] = (T)((double)r[c] / v[18]);
}

template <typename T>
void launch_jacobi(chy_ctx *ctx, int lhs_type, const T *n, const T *r, T *z)
{
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  const LapRow L = lap_row(ctx, lhs_type);
  hipLaunchKernelGGL((k_jacobi<T>), nblocks(ctx->g.nc), kBlock, 0, ctx->stream, ctx->g, lhs_type, s, L, n, r, z);
}

// Node field E = E0 - grad(phi), central differences (periodic), written
// interleaved {Ex, Ey, Ez, 0} so the gather reads one vector per node.
template <typename T>
__global__ __launch_bounds__(256) void k_efield(Grid g, double e0x, double e0y, double e0z, double hx, double hy,
                                                double hz, const double *__restrict__ phi, T *__restrict__ E4)
{
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.nc) return;
  const int i = (int)(c % g.nx), j = (int)((c / g.nx) % g.ny), k = (int)(c / ((int64_t)g.nx * g.ny));
  E4[4 * c + 0] = (T)(e0x - (phi[lin(g, i + 1, j, k)] - phi[lin(g, i - 1, j, k)]) * hx);
  E4[4 * c + 1] = (T)(e0y - (phi[lin(g, i, j + 1, k)] - phi[lin(g, i, j - 1, k)]) * hy);
  E4[4 * c + 2] = (T)(e0z - (phi[lin(g, i, j, k + 1)] - phi[lin(g, i, j, k - 1)]) * hz);
  E4[4 * c + 3] = (T)0;
}

template <typename T>
void launch_efield(chy_ctx *ctx, const double *phi, T *E4)
{
  const double *E0 = ctx->prm.E0, *d = ctx->prm.d;
  hipLaunchKernelGGL((k_efield<T>), nblocks(ctx->g.nc), kBlock, 0, ctx->stream, ctx->g, E0[0], E0[1], E0[2],
                     0.5 / d[0], 0.5 / d[1], 0.5 / d[2], phi, E4);
}

// Full forcing (rhs.c:244-285) with the intended y-z cross derivative.
template <typename T>
__global__ __launch_bounds__(256) void k_rhs_full(Grid g, RhsCoef rc, const T *__restrict__ n,
                                                  const T *__restrict__ gx, const T *__restrict__ gy,
                                                  const T *__restrict__ gz, double *__restrict__ b)
{
  // one block per 256-node segment of an x row; the (segments x ny x nz)
  // launch is relabelled XCD-contiguously, so the y and z neighbour rows come
  // from the L2 that the neighbouring rows' blocks filled
  uint32_t seg, j_, k_;
  xcd_tile(seg, j_, k_);
  const int i = (int)seg * 256 + threadIdx.x, j = (int)j_, k = (int)k_;
  if (i >= g.nx) return;
  const int ip = i + 1 == g.nx ? 0 : i + 1, im = i == 0 ? g.nx - 1 : i - 1;
  const int jp = j + 1 == g.ny ? 0 : j + 1, jm = j == 0 ? g.ny - 1 : j - 1;
  const int kp = k + 1 == g.nz ? 0 : k + 1, km = k == 0 ? g.nz - 1 : k - 1;
  auto row = [&](int jj, int kk) { return (int64_t)g.nx * ((int64_t)jj + (int64_t)g.ny * kk); };
  const int64_t r0 = row(j, k), ryp = row(jp, k), rym = row(jm, k), rzp = row(j, kp), rzm = row(j, km);
  const double n0 = (double)n[r0 + i];
  const double nxp = (double)n[r0 + ip], nxm = (double)n[r0 + im];
  const double nyp = (double)n[ryp + i], nym = (double)n[rym + i];
  const double nzp = (double)n[rzp + i], nzm = (double)n[rzm + i];
  const double dndx = (nxp - nxm) * rc.h1[0];
  const double dndy = (nyp - nym) * rc.h1[1];
  const double dndz = (nzp - nzm) * rc.h1[2];
  const double dGxdx = ((double)gx[r0 + ip] - (double)gx[r0 + im]) * rc.h1[0];
  const double dGydy = ((double)gy[ryp + i] - (double)gy[rym + i]) * rc.h1[1];
  const double dGzdz = ((double)gz[rzp + i] - (double)gz[rzm + i]) * rc.h1[2];
  double Pterm = 0.0;
  if (rc.cth != 0.0) {
    const int64_t rpp = row(jp, kp), rmp = row(jm, kp), rpm = row(jp, km), rmm = row(jm, km);
    const double d2xx = (nxp - 2.0 * n0 + nxm) * rc.h2[0];
    const double d2yy = (nyp - 2.0 * n0 + nym) * rc.h2[1];
    const double d2zz = (nzp - 2.0 * n0 + nzm) * rc.h2[2];
    const double d2xy =
        ((double)n[ryp + ip] - (double)n[ryp + im] - (double)n[rym + ip] + (double)n[rym + im]) * rc.hm[0];
    const double d2xz =
        ((double)n[rzp + ip] - (double)n[rzp + im] - (double)n[rzm + ip] + (double)n[rzm + im]) * rc.hm[1];
    const double d2yz = ((double)n[rpp + i] - (double)n[rmp + i] - (double)n[rpm + i] + (double)n[rmm + i]) * rc.hm[2];
    Pterm = rc.cth * (rc.r[0][0] * d2xx + rc.r[0][1] * d2xy + rc.r[0][2] * d2xz +
                      rc.r[1][0] * d2xy + rc.r[1][1] * d2yy + rc.r[1][2] * d2yz +
                      rc.r[2][0] * d2xz + rc.r[2][1] * d2yz + rc.r[2][2] * d2zz);
  }
  const double Eterm = rc.re[0] * dndx + rc.re[1] * dndy + rc.re[2] * dndz;
  const double Gterm = rc.detA * rc.cG * (dGxdx + dGydy + dGzdz);
  b[r0 + i] = rc.scale * (Eterm + Pterm + Gterm);
}

// Sinusoidal forcing (rhs.c:98-112); n0 is a device scalar (sum of n).
__global__ __launch_bounds__(256) void k_rhs_sin(Grid g, double dx, double dy, double dz, double fac, double inv_nc,
                                                 const double *__restrict__ nsum, double *__restrict__ b)
{
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.nc) return;
  const int i = (int)(c % g.nx), j = (int)((c / g.nx) % g.ny), k = (int)(c / ((int64_t)g.nx * g.ny));
  const double n0 = nsum[0] * inv_nc;
  const double x = ((double)i + 0.5) * dx, y = ((double)j + 0.5) * dy, z = ((double)k + 0.5) * dz;
  const double val = cos(2 * M_PI * x) * cos(2 * M_PI * y) * cos(2 * M_PI * z);
  b[c] = n0 * val * fac;
}

__global__ __launch_bounds__(256) void k_rhs_const(int64_t nc, double fac, double inv_nc, const double *__restrict__ nsum,
                                                   double *__restrict__ b)
{
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  b[c] = (nsum[0] * inv_nc) * fac;
}

// Forcing constants: magnetisation tensor R (rhs.c:205-216), cth, cG.
RhsCoef rhs_coef(const chy_ctx *ctx)
{
  const chy_params &p = ctx->prm;
  const double Kx = p.kappa_e[0], Ky = p.kappa_e[1], Kz = p.kappa_e[2];
  const double detA = 1 + Kx * Kx + Ky * Ky + Kz * Kz;
  RhsCoef rc;
  rc.r[0][0] = 1 + Kx * Kx; rc.r[0][1] = Ky * Kx - Kz; rc.r[0][2] = Kz * Kx + Ky;
  rc.r[1][0] = Kx * Ky + Kz; rc.r[1][1] = 1 + Ky * Ky; rc.r[1][2] = Kz * Ky - Kx;
  rc.r[2][0] = Kx * Kz - Ky; rc.r[2][1] = Ky * Kz + Kx; rc.r[2][2] = 1 + Kz * Kz;
  rc.detA = detA;
  rc.scale = 1.0 / detA;
  rc.cth = p.gamma_e * 1.3807e-23 * p.Te / 1.6022e-19;
  rc.cG = p.me * p.nue / 1.6022e-19;
  for (int a = 0; a < 3; a++) rc.E0[a] = p.E0[a];
  rc.dx = p.d[0]; rc.dy = p.d[1]; rc.dz = p.d[2];
  for (int a = 0; a < 3; a++) {
    rc.h1[a] = 1.0 / (2.0 * p.d[a]);
    rc.h2[a] = 1.0 / (p.d[a] * p.d[a]);
    rc.re[a] = rc.r[a][0] * p.E0[0] + rc.r[a][1] * p.E0[1] + rc.r[a][2] * p.E0[2];
  }
  rc.hm[0] = 1.0 / (4.0 * p.d[0] * p.d[1]);
  rc.hm[1] = 1.0 / (4.0 * p.d[0] * p.d[2]);
  rc.hm[2] = 1.0 / (4.0 * p.d[1] * p.d[2]);
  return rc;
}

template <typename T>
void launch_rhs(chy_ctx *ctx, int rhs_type, const T *n, const T *gx, const T *gy, const T *gz, double *b)
{
  const chy_params &p = ctx->prm;
  const double Kx = p.kappa_e[0], Ky = p.kappa_e[1], Kz = p.kappa_e[2];
  const double detA = 1 + Kx * Kx + Ky * Ky + Kz * Kz;
  const int64_t nc = ctx->g.nc;
  if (rhs_type == CHY_RHS_FULL) {
    const RhsCoef rc = rhs_coef(ctx);
    const dim3 grid((unsigned)((ctx->g.nx + 255) / 256), (unsigned)ctx->g.ny, (unsigned)ctx->g.nz);
    hipLaunchKernelGGL((k_rhs_full<T>), grid, kBlock, 0, ctx->stream, ctx->g, rc, n, gx, gy, gz, b);
  } else {
    launch_sum<T>(ctx, n, nc, ctx->red_out);
    const double fac = 2.0 * p.d[0] * p.d[1] * p.d[2] / detA;
    if (rhs_type == CHY_RHS_SINUSOIDAL)
      hipLaunchKernelGGL(k_rhs_sin, nblocks(nc), kBlock, 0, ctx->stream, ctx->g, p.d[0], p.d[1], p.d[2], fac,
                         1.0 / (double)nc, ctx->red_out, b);
    else
      hipLaunchKernelGGL(k_rhs_const, nblocks(nc), kBlock, 0, ctx->stream, nc, fac, 1.0 / (double)nc,
                         ctx->red_out, b);
  }
  if (rhs_type != CHY_RHS_CONSTANT) {
    // null-space removal (rhs.c:294-296): b -= mean(b)
    launch_sum<double>(ctx, b, nc, ctx->red_out);
    launch_shift<double>(ctx, nc, b, ctx->red_out, -1.0 / (double)nc);
  }
}

// ---- deterministic reductions ---------------------------------------------------
constexpr int kMaxDots = 32;

// partial[blk*nv + k] = sum over this block's grid-stride range of A_k . b
template <typename T, int NV>
__global__ __launch_bounds__(256) void k_mdot(int nv, const T *__restrict__ A, int64_t stride, const T *__restrict__ b,
                                              int64_t n, double *__restrict__ partial)
{
  __shared__ double sh[4][NV];
  double acc[NV];
#pragma unroll
  for (int k = 0; k < NV; k++) acc[k] = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const double bi = (double)b[i];
#pragma unroll
    for (int k = 0; k < NV; k++)
      if (k < nv) acc[k] += (double)A[k * stride + i] * bi;
  }
  const int wid = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < NV; k++) {
    if (k < nv) {
      const double s = wave_total(acc[k]);
      if ((threadIdx.x & 63) == 0) sh[wid][k] = s;
    }
  }
  __syncthreads();
  if (threadIdx.x < nv) {
    const int k = threadIdx.x;
    partial[(int64_t)blockIdx.x * nv + k] = (sh[0][k] + sh[1][k]) + (sh[2][k] + sh[3][k]);
  }
}

// Scales of a combine's outputs, passed by value with the launch.
struct DotScale {
  int on;
  double s[kMaxDots];
};

// out[k] = sum_blk partial[blk*nv + k], fixed tree order, times sc.s[k] when
// sc.on; each value also goes to mirror[k] when a mirror is given (host
// memory: the read-back of a reduced value needs no copy), and then the
// launch's number s to the host's sequence word.  A single value takes four
// waves, several take a wave each: one after another through the whole block
// they took 6.8 us where an iteration has 1 to 30 of them (multigrid on 96 x 80 x
// 50), now 3.9.
__global__ __launch_bounds__(1024) void k_combine(const double *__restrict__ partial, int nblk, int nv,
                                                  double *__restrict__ out, DotScale sc, double *__restrict__ mirror,
                                                  unsigned long long *__restrict__ seq, unsigned long long s_no)
{
  __shared__ double sh[kMaxDots];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if (nv == 1) {
    double acc = 0.0;
    for (int b = threadIdx.x; b < nblk; b += blockDim.x) acc += partial[b];
    const double s = wave_total(acc);
    if (lane == 0) sh[wid] = s;
  } else {
    for (int k = wid; k < nv; k += nw) {
      double acc = 0.0;
#pragma unroll 4
      for (int b = lane; b < nblk; b += 64) acc += partial[(int64_t)b * nv + k];
      const double s = wave_total(acc);
      if (lane == 0) sh[k] = s;
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < nv) {
    const int k = threadIdx.x;
    double t = sh[k];
    if (nv == 1)
      for (int q = 1; q < nw; q++) t += sh[q];
    const double v = sc.on ? t * sc.s[k] : t;
    out[k] = v;
    if (mirror) mirror[k] = v;
  }
  // (one wave wrote every mirror value: the fence orders them before the number)
  if (seq && threadIdx.x < 64) {
    __threadfence_system();
    if (threadIdx.x == 0) *(volatile unsigned long long *)seq = s_no;
  }
}

// The host mirror of out when out lies in the reduction output buffer.
static double *mirror_of(chy_ctx *ctx, const double *out, int nv)
{
  if (!ctx->red_mirror || out < ctx->red_out || out + nv > ctx->red_out + ctx->red_out_n) return nullptr;
  return ctx->red_mirror + (out - ctx->red_out);
}

// One combine launch: nv outputs, scaled by scale_host[k] when given (at most
// kMaxDots of them).
static void combine(chy_ctx *ctx, const double *partial, int nblk, int nv, double *out,
                    const double *scale_host = nullptr)
{
  DotScale sc;
  sc.on = scale_host != nullptr;
  for (int k = 0; k < kMaxDots; k++) sc.s[k] = (sc.on && k < nv) ? scale_host[k] : 1.0;
  double *mirror = mirror_of(ctx, out, nv);
  const int waves = nv == 1 ? 4 : std::min(nv, 16);
  hipLaunchKernelGGL(k_combine, 1, 64 * waves, 0, ctx->stream, partial, nblk, nv, out, sc, mirror,
                     mirror ? seq_word(ctx) : nullptr, mirror ? next_seq(ctx) : 0ull);
}

// Block b of 256 sums partials [b * chunk, (b + 1) * chunk) in a fixed order.
__global__ __launch_bounds__(256) void k_chunk_sum(const double *__restrict__ partial, int64_t n, int64_t chunk,
                                                   double *__restrict__ out)
{
  __shared__ double sh[4];
  const int64_t lo = (int64_t)blockIdx.x * chunk, hi = lo + chunk < n ? lo + chunk : n;
  double acc = 0.0;
#pragma unroll 8
  for (int64_t b = lo + threadIdx.x; b < hi; b += blockDim.x) acc += partial[b];
  const double t = wave_total(acc);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

void launch_combine_sum(chy_ctx *ctx, const double *partials, int nblk, int nv, double *out)
{
  if (nv == 1 && nblk > 4 * kRedBlocks) {
    // one partial per deposit block (nc / 32 of them): two levels
    constexpr int kChunks = 256;
    const int64_t chunk = ((int64_t)nblk + kChunks - 1) / kChunks;
    hipLaunchKernelGGL(k_chunk_sum, kChunks, kBlock, 0, ctx->stream, partials, (int64_t)nblk, chunk, ctx->red);
    combine(ctx, ctx->red, kChunks, 1, out);
    return;
  }
  combine(ctx, partials, nblk, nv, out);
}

template <typename T>
void launch_mdot(chy_ctx *ctx, int nv, const T *A, int64_t stride, const T *b, int64_t n, double *out_dev,
                 const double *scale)
{
  for (int k0 = 0; k0 < nv; k0 += kMaxDots) {
    const int m = (nv - k0 < kMaxDots) ? nv - k0 : kMaxDots;
    const unsigned nb = (unsigned)std::min<int64_t>(kRedBlocks, (n + kBlock - 1) / kBlock);
    if (m <= 1)
      hipLaunchKernelGGL((k_mdot<T, 1>), nb, kBlock, 0, ctx->stream, m, A + k0 * stride, stride, b, n, ctx->red);
    else if (m <= 8)
      hipLaunchKernelGGL((k_mdot<T, 8>), nb, kBlock, 0, ctx->stream, m, A + k0 * stride, stride, b, n, ctx->red);
    else
      hipLaunchKernelGGL((k_mdot<T, kMaxDots>), nb, kBlock, 0, ctx->stream, m, A + k0 * stride, stride, b, n,
                         ctx->red);
    combine(ctx, ctx->red, (int)nb, m, out_dev + k0, scale ? scale + k0 : nullptr);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_sum(const T *__restrict__ a, int64_t n, double *__restrict__ partial)
{
  __shared__ double sh[4];
  double acc = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    acc += (double)a[i];
  const double s = wave_total(acc);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

template <typename T>
void launch_sum(chy_ctx *ctx, const T *a, int64_t n, double *out_dev)
{
  const unsigned nb = (unsigned)std::min<int64_t>(kRedBlocks, (n + kBlock - 1) / kBlock);
  hipLaunchKernelGGL((k_sum<T>), nb, kBlock, 0, ctx->stream, a, n, ctx->red);
  combine(ctx, ctx->red, (int)nb, 1, out_dev);
}

// w -= sum_k h_k V_k  (h on the device, or by value in hv.s when h is null;
// accumulation in FP64)
template <typename T, int NV>
__global__ __launch_bounds__(256) void k_mgs(int nv, const T *__restrict__ V, int64_t stride,
                                             const double *__restrict__ h, DotScale hv, T *__restrict__ w, int64_t n)
{
  __shared__ double hs[NV];
  if (threadIdx.x < nv) hs[threadIdx.x] = h ? h[threadIdx.x] : hv.s[threadIdx.x];
  __syncthreads();
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    double acc = (double)w[i];
#pragma unroll
    for (int k = 0; k < NV; k++)
      if (k < nv) acc -= hs[k] * (double)V[k * stride + i];
    w[i] = (T)acc;
  }
}

// w -= sum_k h_k V_k with h on the device, or, when h_host is given, with the
// coefficients from host memory passed by value (no copy to wait for)
template <typename T>
static void mgs_update(chy_ctx *ctx, int nv, const T *V, int64_t stride, const double *h, const double *h_host, T *w,
                       int64_t n)
{
  for (int k0 = 0; k0 < nv; k0 += kMaxDots) {
    const int m = (nv - k0 < kMaxDots) ? nv - k0 : kMaxDots;
    const unsigned nb = (unsigned)std::min<int64_t>(4096, (n + kBlock - 1) / kBlock);
    DotScale hv;
    hv.on = h_host != nullptr;
    for (int k = 0; k < kMaxDots; k++) hv.s[k] = (h_host && k < m) ? h_host[k0 + k] : 0.0;
    const double *hd = h_host ? nullptr : h + k0;
    if (m <= 8)
      hipLaunchKernelGGL((k_mgs<T, 8>), nb, kBlock, 0, ctx->stream, m, V + k0 * stride, stride, hd, hv, w, n);
    else
      hipLaunchKernelGGL((k_mgs<T, kMaxDots>), nb, kBlock, 0, ctx->stream, m, V + k0 * stride, stride, hd, hv, w, n);
  }
}

template <typename T>
void launch_mgs_update(chy_ctx *ctx, int nv, const T *V, int64_t stride, const double *h, T *w, int64_t n)
{
  mgs_update<T>(ctx, nv, V, stride, h, nullptr, w, n);
}

template <typename T>
void launch_mgs_update_host(chy_ctx *ctx, int nv, const T *V, int64_t stride, const double *h_host, T *w, int64_t n)
{
  mgs_update<T>(ctx, nv, V, stride, nullptr, h_host, w, n);
}

// w -= sum_k h_k V_k as k_mgs, also accumulating ||w||^2 of the result in
// FP64 block partials (fixed grid: deterministic).
template <typename T, int NV>
__global__ __launch_bounds__(256) void k_mgs_norm(int nv, const T *__restrict__ V, int64_t stride,
                                                  const double *__restrict__ h, T *__restrict__ w, int64_t n,
                                                  double *__restrict__ partial)
{
  __shared__ double hs[NV];
  __shared__ double sh[4];
  if (threadIdx.x < nv) hs[threadIdx.x] = h[threadIdx.x];
  __syncthreads();
  double nn = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    double acc = (double)w[i];
#pragma unroll
    for (int k = 0; k < NV; k++)
      if (k < nv) acc -= hs[k] * (double)V[k * stride + i];
    const T r = (T)acc;
    w[i] = r;
    nn += (double)r * (double)r;
  }
  const double s = wave_total(nn);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

template <typename T>
void launch_mgs_norm(chy_ctx *ctx, int nv, const T *V, int64_t stride, const double *h, T *w, int64_t n,
                     double *norm2_dev)
{
  if (nv > kMaxDots) {  // rare: split, norm from the last chunk
    launch_mgs_update<T>(ctx, nv - kMaxDots, V, stride, h, w, n);
    V += (int64_t)(nv - kMaxDots) * stride;
    h += nv - kMaxDots;
    nv = kMaxDots;
  }
  const unsigned nb = (unsigned)std::min<int64_t>(kRedBlocks, (n + kBlock - 1) / kBlock);
  if (nv <= 8)
    hipLaunchKernelGGL((k_mgs_norm<T, 8>), nb, kBlock, 0, ctx->stream, nv, V, stride, h, w, n, ctx->red);
  else
    hipLaunchKernelGGL((k_mgs_norm<T, kMaxDots>), nb, kBlock, 0, ctx->stream, nv, V, stride, h, w, n, ctx->red);
  combine(ctx, ctx->red, (int)nb, 1, norm2_dev);
}

// ---- Gram-Schmidt passes with 16-byte vector loads (n % 4 == 0) -------------------
// Four consecutive elements per lane and grid-stride step; every block covers
// a fixed set of quads, so the FP64 partial sums (and the results) do not
// depend on timing.
template <typename T> struct alignas(4 * sizeof(T)) Q4 { T v[4]; };

template <typename T, int NV>
__device__ __forceinline__ void block_partials(const double (&acc)[NV], int nv, double (*sh)[NV], double *partial)
{
  const int wid = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < NV; k++) {
    if (k < nv) {
      const double s = wave_total(acc[k]);
      if ((threadIdx.x & 63) == 0) sh[wid][k] = s;
    }
  }
  __syncthreads();
  if (threadIdx.x < nv) {
    const int k = threadIdx.x;
    partial[(int64_t)blockIdx.x * nv + k] = (sh[0][k] + sh[1][k]) + (sh[2][k] + sh[3][k]);
  }
}

// partial[blk*nv + k] = A_k . b over the block's quads
template <typename T, int NV>
__global__ __launch_bounds__(256) void k_mdot4(int nv, const T *__restrict__ A, int64_t stride, const T *__restrict__ b,
                                               int64_t n4, double *__restrict__ partial)
{
  __shared__ double sh[4][NV];
  double acc[NV];
#pragma unroll
  for (int k = 0; k < NV; k++) acc[k] = 0.0;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n4; q += (int64_t)gridDim.x * blockDim.x) {
    const Q4<T> bq = reinterpret_cast<const Q4<T> *>(b)[q];
#pragma unroll
    for (int k = 0; k < NV; k++) {
      if (k < nv) {
        const Q4<T> a = reinterpret_cast<const Q4<T> *>(A + k * stride)[q];
        acc[k] += ((double)a.v[0] * (double)bq.v[0] + (double)a.v[1] * (double)bq.v[1]) +
                  ((double)a.v[2] * (double)bq.v[2] + (double)a.v[3] * (double)bq.v[3]);
      }
    }
  }
  block_partials<T, NV>(acc, nv, sh, partial);
}

// w -= sum_k h_k V_k, then partial[blk*nv + k] = V_k . w (of the new w), or
// with NORM the partial of ||w||^2 instead.  SUM: h_k is the sum of the nblk
// partials h[b*nv + k] times sc.s[k], made by every block in the same order;
// block 0 leaves them in out and its mirror, as k_combine does.
template <typename T, int NV, bool NORM, bool SUM = false>
__global__ __launch_bounds__(256) void k_gs4(int nv, const T *__restrict__ V, int64_t stride,
                                             const double *__restrict__ h, T *__restrict__ w, int64_t n4,
                                             double *__restrict__ partial, int nblk, DotScale sc,
                                             double *__restrict__ out, double *__restrict__ mirror)
{
  __shared__ double hs[NV];
  __shared__ double sh[4][NORM ? 1 : NV];
  if (SUM) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int k0 = 0; k0 < NV; k0 += 4) {
      const int k = k0 + (threadIdx.x >> 6);
      if (k < nv) {
        double t = 0.0;
#pragma unroll 4
        for (int b = lane; b < nblk; b += 64) t += h[(int64_t)b * nv + k];
        t = wave_total(t);
        if (lane == 0) {
          const double v = t * sc.s[k];
          hs[k] = v;
          if (blockIdx.x == 0) {
            out[k] = v;
            if (mirror) {
              mirror[k] = v;
              __threadfence_system();
            }
          }
        }
      }
    }
  } else if (threadIdx.x < nv) {
    hs[threadIdx.x] = h[threadIdx.x];
  }
  __syncthreads();
  double acc[NORM ? 1 : NV];
#pragma unroll
  for (int k = 0; k < (NORM ? 1 : NV); k++) acc[k] = 0.0;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n4; q += (int64_t)gridDim.x * blockDim.x) {
    Q4<T> wq = reinterpret_cast<const Q4<T> *>(w)[q];
    Q4<T> vq[NV];
    double r[4] = {(double)wq.v[0], (double)wq.v[1], (double)wq.v[2], (double)wq.v[3]};
#pragma unroll
    for (int k = 0; k < NV; k++) {
      if (k < nv) {
        vq[k] = reinterpret_cast<const Q4<T> *>(V + k * stride)[q];
#pragma unroll
        for (int e = 0; e < 4; e++) r[e] -= hs[k] * (double)vq[k].v[e];
      }
    }
#pragma unroll
    for (int e = 0; e < 4; e++) wq.v[e] = (T)r[e];
    reinterpret_cast<Q4<T> *>(w)[q] = wq;
    if (NORM) {
      acc[0] += ((double)wq.v[0] * (double)wq.v[0] + (double)wq.v[1] * (double)wq.v[1]) +
                ((double)wq.v[2] * (double)wq.v[2] + (double)wq.v[3] * (double)wq.v[3]);
    } else {
#pragma unroll
      for (int k = 0; k < (NORM ? 1 : NV); k++)
        if (k < nv)
          acc[k] += ((double)vq[k].v[0] * (double)wq.v[0] + (double)vq[k].v[1] * (double)wq.v[1]) +
                    ((double)vq[k].v[2] * (double)wq.v[2] + (double)vq[k].v[3] * (double)wq.v[3]);
    }
  }
  block_partials<T, NORM ? 1 : NV>(acc, NORM ? 1 : nv, sh, partial);
}

static inline bool quad_ok(int64_t n, int64_t stride, const void *a, const void *b)
{
  return n % 4 == 0 && stride % 4 == 0 && ((uintptr_t)a % 16) == 0 && ((uintptr_t)b % 16) == 0;
}

// The pass compiled for the next larger number of vectors (the scalar kernels,
// which took over beyond 8, need 21 us for the dots and 12.7 for the update at
// 96 x 80 x 50, these 18 and 11 with up to 32 vectors and 11 and 6 with 16)
#define GS_NV(nv, call)                                       \
  do {                                                        \
    if (nv <= 8) { constexpr int NV = 8; call; }              \
    else if (nv <= 16) { constexpr int NV = 16; call; }       \
    else { constexpr int NV = kMaxDots; call; }               \
  } while (0)

template <typename T>
void launch_gs_dots(chy_ctx *ctx, int nv, const T *V, int64_t stride, const T *w, int64_t n, double *out_dev,
                    const double *scale)
{
  if (nv > kMaxDots || !quad_ok(n, stride, V, w)) { launch_mdot<T>(ctx, nv, V, stride, w, n, out_dev, scale); return; }
  const int64_t n4 = n / 4;
  const unsigned nb = (unsigned)std::min<int64_t>(kRedBlocks, (n4 + kBlock - 1) / kBlock);
  GS_NV(nv, hipLaunchKernelGGL((k_mdot4<T, NV>), nb, kBlock, 0, ctx->stream, nv, V, stride, w, n4, ctx->red));
  combine(ctx, ctx->red, (int)nb, nv, out_dev, scale);
}

template <typename T>
void launch_gs_update_dots(chy_ctx *ctx, int nv, const T *V, int64_t stride, const double *h, T *w, int64_t n,
                           double *out_dev, const double *scale)
{
  if (nv > 8 || !quad_ok(n, stride, V, w)) {
    launch_mgs_update<T>(ctx, nv, V, stride, h, w, n);
    launch_mdot<T>(ctx, nv, V, stride, w, n, out_dev, scale);
    return;
  }
  const int64_t n4 = n / 4;
  const unsigned nb = (unsigned)std::min<int64_t>(kRedBlocks, (n4 + kBlock - 1) / kBlock);
  hipLaunchKernelGGL((k_gs4<T, 8, false>), nb, kBlock, 0, ctx->stream, nv, V, stride, h, w, n4, ctx->red, 0, DotScale(),
                     (double *)nullptr, (double *)nullptr);
  combine(ctx, ctx->red, (int)nb, nv, out_dev, scale);
}

template <typename T>
void launch_gs_update_norm(chy_ctx *ctx, int nv, const T *V, int64_t stride, const double *h, T *w, int64_t n,
                           double *norm2_dev)
{
  if (nv > kMaxDots || !quad_ok(n, stride, V, w)) { launch_mgs_norm<T>(ctx, nv, V, stride, h, w, n, norm2_dev); return; }
  const int64_t n4 = n / 4;
  const unsigned nb = (unsigned)std::min<int64_t>(kRedBlocks, (n4 + kBlock - 1) / kBlock);
  GS_NV(nv, hipLaunchKernelGGL((k_gs4<T, NV, true>), nb, kBlock, 0, ctx->stream, nv, V, stride, h, w, n4, ctx->red, 0,
                               DotScale(), (double *)nullptr, (double *)nullptr));
  combine(ctx, ctx->red, (int)nb, 1, norm2_dev);
}

// The dots of launch_lhs_dots' nblk partials, scaled, to out_dev
void launch_dots_sum(chy_ctx *ctx, int nv, int nblk, double *out_dev, const double *scale)
{
  combine(ctx, ctx->red, nblk, nv, out_dev, scale);
}

// The same, w -= V out and ||w||^2: the update adds the partials itself, in
// every block.  With the dots taken where w is made, that is two launches of
// 4.5 us an iteration fewer, for 1 to 3 us more in each of the two kernels.  us
// of a solve, dots and their sum as launches of their own -> here: 32^3 FP64 926
// -> 896, 64^3 mixed 1030 -> 994 and FP64 1030 -> 996, 64 x 128 x 64 mixed 1062
// -> 1025, 128^3 FP64 2075 -> 1985 (2020 with the sum as a launch), mixed 1580
// -> 1535.
template <typename T>
void launch_gs_sum_update_norm(chy_ctx *ctx, int nv, const T *V, int64_t stride, int nblk, double *out_dev,
                               const double *scale, T *w, int64_t n, double *norm2_dev)
{
  if (!quad_ok(n, stride, V, w)) {
    launch_dots_sum(ctx, nv, nblk, out_dev, scale);
    launch_gs_update_norm<T>(ctx, nv, V, stride, out_dev, w, n, norm2_dev);
    return;
  }
  const int64_t n4 = n / 4;
  const unsigned nb = (unsigned)std::min<int64_t>(kRedBlocks, (n4 + kBlock - 1) / kBlock);
  DotScale sc;
  sc.on = 1;
  for (int k = 0; k < kMaxDots; k++) sc.s[k] = k < nv ? scale[k] : 1.0;
  double *norms = ctx->red + (int64_t)kColDots * kRedBlocks;  // (the dots' partials are read meanwhile)
  hipLaunchKernelGGL((k_gs4<T, 8, true, true>), nb, kBlock, 0, ctx->stream, nv, V, stride, (const double *)ctx->red, w,
                     n4, norms, nblk, sc, out_dev, mirror_of(ctx, out_dev, nv));
  combine(ctx, norms, (int)nb, 1, norm2_dev);
}
template void launch_gs_sum_update_norm<double>(chy_ctx *, int, const double *, int64_t, int, double *, const double *,
                                                double *, int64_t, double *);
template void launch_gs_sum_update_norm<float>(chy_ctx *, int, const float *, int64_t, int, double *, const double *,
                                               float *, int64_t, double *);

template <typename T>
__global__ __launch_bounds__(256) void k_axpby(int64_t n, double a, const T *__restrict__ x, double b, T *__restrict__ y)
{
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    y[i] = (T)(a * (double)x[i] + (b == 0.0 ? 0.0 : b * (double)y[i]));
}

template <typename T>
void launch_axpby(chy_ctx *ctx, int64_t n, double a, const T *x, double b, T *y)
{
  const unsigned nb = (unsigned)std::min<int64_t>(8192, (n + kBlock - 1) / kBlock);
  hipLaunchKernelGGL((k_axpby<T>), nb, kBlock, 0, ctx->stream, n, a, x, b, y);
}

template <typename TS, typename TD>
__global__ __launch_bounds__(256) void k_convert(int64_t n, const TS *__restrict__ s, double scale, TD *__restrict__ d)
{
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    d[i] = (TD)((double)s[i] * scale);
}

template <typename TS, typename TD>
void launch_convert(chy_ctx *ctx, int64_t n, const TS *src, double scale, TD *dst)
{
  const unsigned nb = (unsigned)std::min<int64_t>(8192, (n + kBlock - 1) / kBlock);
  hipLaunchKernelGGL((k_convert<TS, TD>), nb, kBlock, 0, ctx->stream, n, src, scale, dst);
}

// v += scale * shift[0]
template <typename T>
__global__ __launch_bounds__(256) void k_shift(int64_t n, T *__restrict__ v, const double *__restrict__ shift, double scale)
{
  const double s = shift[0] * scale;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    v[i] = (T)((double)v[i] + s);
}

template <typename T>
void launch_shift(chy_ctx *ctx, int64_t n, T *v, const double *shift_dev, double scale)
{
  const unsigned nb = (unsigned)std::min<int64_t>(8192, (n + kBlock - 1) / kBlock);
  hipLaunchKernelGGL((k_shift<T>), nb, kBlock, 0, ctx->stream, n, v, shift_dev, scale);
}

template <typename T>
__global__ __launch_bounds__(256) void k_fill(int64_t n, T *__restrict__ v, T val)
{
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    v[i] = val;
}

template <typename T>
void launch_fill(chy_ctx *ctx, int64_t n, T *v, T val)
{
  const unsigned nb = (unsigned)std::min<int64_t>(8192, (n + kBlock - 1) / kBlock);
  if (nb) hipLaunchKernelGGL((k_fill<T>), nb, kBlock, 0, ctx->stream, n, v, val);
}

// Plain copy (counter calibration): 16-byte vector loads and stores.
__global__ __launch_bounds__(256) void k_copy(int64_t n16, const uint4 *__restrict__ a, uint4 *__restrict__ b)
{
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (int64_t)gridDim.x * blockDim.x)
    b[i] = a[i];
}

// One 16-byte element per thread, no loop: the device's streaming ceiling
// (every wave retires after one load and one store).
__global__ __launch_bounds__(256) void k_copy1(int64_t n16, const uint4 *__restrict__ a, uint4 *__restrict__ b)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n16) b[i] = a[i];
}

void launch_copy(chy_ctx *ctx, int64_t n16, const void *a, void *b)
{
  const unsigned nb = (unsigned)std::min<int64_t>(16384, (n16 + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(k_copy, nb, kBlock, 0, ctx->stream, n16, (const uint4 *)a, (uint4 *)b);
}

void launch_copy1(chy_ctx *ctx, int64_t n16, const void *a, void *b)
{
  const unsigned nb = (unsigned)((n16 + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(k_copy1, nb, kBlock, 0, ctx->stream, n16, (const uint4 *)a, (uint4 *)b);
}

// ---- adjoint pieces of the grid operators (FP64) ------------------------------------
// d/dn of mu^T A(n) phi.  Row r of A(n) is linear in the 7-point density star
// of r, so its coefficients for unit density at star slot o are constants
// (R.v[o]); node m appears at slot o of row r = m - star(o):
//   out[m] += alpha * sum_o mu[r] * sum_q R.v[o][q] phi[r + off(q)].
struct StarRows { double v[7][19]; };
__constant__ int kStar[7][3] = {{0, 0, 0}, {+1, 0, 0}, {-1, 0, 0}, {0, +1, 0}, {0, -1, 0}, {0, 0, +1}, {0, 0, -1}};

__global__ __launch_bounds__(256) void k_lhs_dn(Grid g, StarRows R, const double *__restrict__ mu,
                                                const double *__restrict__ phi, double alpha, double *__restrict__ out)
{
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= g.nc) return;
  const int i = (int)(m % g.nx), j = (int)((m / g.nx) % g.ny), k = (int)(m / ((int64_t)g.nx * g.ny));
  double acc = 0.0;
  for (int o = 0; o < 7; o++) {
    const int ri = i - kStar[o][0], rj = j - kStar[o][1], rk = k - kStar[o][2];
    const double mr = mu[lin(g, ri, rj, rk)];
    double row = 0.0;
#pragma unroll
    for (int q = 0; q < 19; q++) row += R.v[o][q] * phi[lin(g, ri + kOff[q][0], rj + kOff[q][1], rk + kOff[q][2])];
    acc += mr * row;
  }
  out[m] += alpha * acc;
}

void launch_lhs_dn(chy_ctx *ctx, const double *mu, const double *phi, double alpha, double *out)
{
  if (ctx->prm.lhs_type != CHY_LHS_FULL) return;  // laplacian and identity rows do not depend on n
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  StarRows R;
  for (int o = 0; o < 7; o++) {
    double e[7] = {0, 0, 0, 0, 0, 0, 0};
    e[o] = 1.0;
    row_from_star<double>(s, e[0], e[1], e[2], e[3], e[4], e[5], e[6], R.v[o]);
  }
  hipLaunchKernelGGL(k_lhs_dn, nblocks(ctx->g.nc), kBlock, 0, ctx->stream, ctx->g, R, mu, phi, alpha, out);
}

// Transpose of the full forcing (without its mean removal, which the caller
// applies to mu): ln += dB/dn^T mu, lG_a += dB/dG_a^T mu.  Central first
// differences are antisymmetric (D^T = -D), second differences symmetric.
__global__ __launch_bounds__(256) void k_rhs_full_adj(Grid g, RhsCoef rc, const double *__restrict__ mu,
                                                      double *__restrict__ ln, double *__restrict__ lgx,
                                                      double *__restrict__ lgy, double *__restrict__ lgz)
{
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.nc) return;
  const int i = (int)(c % g.nx), j = (int)((c / g.nx) % g.ny), k = (int)(c / ((int64_t)g.nx * g.ny));
  const double dx = rc.dx, dy = rc.dy, dz = rc.dz;
#define F(di, dj, dk) (mu[lin(g, i + (di), j + (dj), k + (dk))])
  const double Dx = (F(1, 0, 0) - F(-1, 0, 0)) / (2.0 * dx);
  const double Dy = (F(0, 1, 0) - F(0, -1, 0)) / (2.0 * dy);
  const double Dz = (F(0, 0, 1) - F(0, 0, -1)) / (2.0 * dz);
  double P = 0.0;
  if (rc.cth != 0.0) {
    const double d2xx = (F(1, 0, 0) - 2.0 * F(0, 0, 0) + F(-1, 0, 0)) / (dx * dx);
    const double d2yy = (F(0, 1, 0) - 2.0 * F(0, 0, 0) + F(0, -1, 0)) / (dy * dy);
    const double d2zz = (F(0, 0, 1) - 2.0 * F(0, 0, 0) + F(0, 0, -1)) / (dz * dz);
    const double d2xy = (F(1, 1, 0) - F(-1, 1, 0) - F(1, -1, 0) + F(-1, -1, 0)) / (4.0 * dx * dy);
    const double d2xz = (F(1, 0, 1) - F(-1, 0, 1) - F(1, 0, -1) + F(-1, 0, -1)) / (4.0 * dx * dz);
    const double d2yz = (F(0, 1, 1) - F(0, -1, 1) - F(0, 1, -1) + F(0, -1, -1)) / (4.0 * dy * dz);
    P = rc.cth * (rc.r[0][0] * d2xx + (rc.r[0][1] + rc.r[1][0]) * d2xy + (rc.r[0][2] + rc.r[2][0]) * d2xz +
                  rc.r[1][1] * d2yy + (rc.r[1][2] + rc.r[2][1]) * d2yz + rc.r[2][2] * d2zz);
  }
#undef F
  const double cx = rc.r[0][0] * rc.E0[0] + rc.r[0][1] * rc.E0[1] + rc.r[0][2] * rc.E0[2];
  const double cy = rc.r[1][0] * rc.E0[0] + rc.r[1][1] * rc.E0[1] + rc.r[1][2] * rc.E0[2];
  const double cz = rc.r[2][0] * rc.E0[0] + rc.r[2][1] * rc.E0[1] + rc.r[2][2] * rc.E0[2];
  ln[c] += rc.scale * (P - (cx * Dx + cy * Dy + cz * Dz));
  const double gG = -rc.scale * rc.detA * rc.cG;
  lgx[c] += gG * Dx;
  lgy[c] += gG * Dy;
  lgz[c] += gG * Dz;
}

void launch_rhs_full_adj(chy_ctx *ctx, const double *mu, double *ln, double *lgx, double *lgy, double *lgz)
{
  hipLaunchKernelGGL(k_rhs_full_adj, nblocks(ctx->g.nc), kBlock, 0, ctx->stream, ctx->g, rhs_coef(ctx), mu, ln, lgx,
                     lgy, lgz);
}

// Central first differences of n along x, y, z (periodic) into three arrays.
__global__ __launch_bounds__(256) void k_grad3(Grid g, const double *__restrict__ n, double *__restrict__ gx,
                                               double *__restrict__ gy, double *__restrict__ gz)
{
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.nc) return;
  const int i = (int)(c % g.nx), j = (int)((c / g.nx) % g.ny), k = (int)(c / ((int64_t)g.nx * g.ny));
  gx[c] = (n[lin(g, i + 1, j, k)] - n[lin(g, i - 1, j, k)]) / (2.0 * g.d[0]);
  gy[c] = (n[lin(g, i, j + 1, k)] - n[lin(g, i, j - 1, k)]) / (2.0 * g.d[1]);
  gz[c] = (n[lin(g, i, j, k + 1)] - n[lin(g, i, j, k - 1)]) / (2.0 * g.d[2]);
}

void launch_grad3(chy_ctx *ctx, const double *n, double *g3)
{
  const int64_t nc = ctx->g.nc;
  hipLaunchKernelGGL(k_grad3, nblocks(nc), kBlock, 0, ctx->stream, ctx->g, n, g3, g3 + nc, g3 + 2 * nc);
}

// Transpose of E = E0 - grad(phi) (central differences) for phi:
//   lphi[c] = sum_a (lE_a[c + e_a] - lE_a[c - e_a]) / (2 d_a).
__global__ __launch_bounds__(256) void k_efield_adj(Grid g, const double *__restrict__ lex,
                                                    const double *__restrict__ ley, const double *__restrict__ lez,
                                                    double *__restrict__ lphi)
{
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.nc) return;
  const int i = (int)(c % g.nx), j = (int)((c / g.nx) % g.ny), k = (int)(c / ((int64_t)g.nx * g.ny));
  const double ax = (lex[lin(g, i + 1, j, k)] - lex[lin(g, i - 1, j, k)]) * (0.5 / g.d[0]);
  const double ay = (ley[lin(g, i, j + 1, k)] - ley[lin(g, i, j - 1, k)]) * (0.5 / g.d[1]);
  const double az = (lez[lin(g, i, j, k + 1)] - lez[lin(g, i, j, k - 1)]) * (0.5 / g.d[2]);
  lphi[c] = ax + ay + az;
}

void launch_efield_adj(chy_ctx *ctx, const double *lex, const double *ley, const double *lez, double *lphi)
{
  hipLaunchKernelGGL(k_efield_adj, nblocks(ctx->g.nc), kBlock, 0, ctx->stream, ctx->g, lex, ley, lez, lphi);
}

// ---- z-averaged operator (two-level FFT preconditioner) -------------------------------
// C[o * nxy + col] = mean over k of the entries of row (col, k) whose column
// lies at x-y offset o = (dx + 1) + 3 (dy + 1); summed over k, then entries in
// row order, as the oracle.
__constant__ int kGroup19[19] = {5, 3, 7, 1, 4, 4, 8, 2, 6, 0, 5, 5, 3, 3, 7, 7, 1, 1, 4};

template <typename T>
__global__ __launch_bounds__(256) void k_zcoef(Grid g, int lhs_type, SCoef s, LapRow lap, const T *__restrict__ n,
                                               T *__restrict__ C)
{
  const int64_t nxy = (int64_t)g.nx * g.ny;
  const int64_t col = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= nxy) return;
  const int i = (int)(col % g.nx), j = (int)(col / g.nx);
  double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int k = 0; k < g.nz; k++) {
    double v[19];
    row_coeffs<double, T>(g, lhs_type, s, lap.v, n, i, j, k, v);
#pragma unroll
    for (int q = 0; q < 19; q++) acc[kGroup19[q]] += v[q];
  }
#pragma unroll
  for (int o = 0; o < 9; o++) C[o * nxy + col] = (T)(acc[o] / (double)g.nz);
}

template <typename T>
void launch_zcoef(chy_ctx *ctx, int lhs_type, const T *n, T *C)
{
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  const LapRow L = lap_row(ctx, lhs_type);
  const int64_t nxy = (int64_t)ctx->g.nx * ctx->g.ny;
  hipLaunchKernelGGL((k_zcoef<T>), nblocks(nxy), kBlock, 0, ctx->stream, ctx->g, lhs_type, s, L, n, C);
}

// ---- z-line block Jacobi and Chebyshev-Jacobi preconditioners --------------------
// z-line: one thread per (i, j) column solves the column's z-line block of
// A(n) -- diagonal v18, -z entry v5, +z entry v4, periodic -- by the
// Sherman-Morrison formula around two Thomas sweeps:
//   A = T + u w^T, u = (g, 0.., 0, c_{m-1}), w = (1, 0.., 0, a_0 / g), g = -b_0,
// T = A without the wrap entries and with b_0 - g, b_{m-1} - c_{m-1} a_0 / g.
// y = T^-1 r and q = T^-1 u share the forward sweep; z = y - q (w.y)/(1 + w.q).
// Scratch: cp and q (nc each); consecutive threads own consecutive x, so every
// sweep step is a coalesced row of the plane.
template <typename T>
__global__ __launch_bounds__(256) void k_zline(Grid g, int lhs_type, SCoef s, LapRow lap, const T *__restrict__ n,
                                               const T *__restrict__ r, T *__restrict__ z, T *__restrict__ cp,
                                               T *__restrict__ q)
{
  using C = double;
  const int64_t plane = (int64_t)g.nx * g.ny;
  const int64_t col = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= plane) return;
  const int i = (int)(col % g.nx), j = (int)(col / g.nx), m = g.nz;
  C v[19];
  row_coeffs<C, T>(g, lhs_type, s, lap.v, n, i, j, 0, v);
  const C a0 = v[5], b0 = v[18], c0 = v[4];
  if (m == 1) { z[col] = (T)((C)r[col] / b0); return; }
  row_coeffs<C, T>(g, lhs_type, s, lap.v, n, i, j, m - 1, v);
  const C al = v[5], bl = v[18], cl = v[4];
  if (m == 2) {  // both neighbours are the other node
    const C a01 = a0 + c0, a10 = al + cl, det = b0 * bl - a01 * a10;
    const C r0 = (C)r[col], r1 = (C)r[col + plane];
    z[col] = (T)((r0 * bl - a01 * r1) / det);
    z[col + plane] = (T)((b0 * r1 - a10 * r0) / det);
    return;
  }
  const C gm = -b0, ag = a0 / gm;
  C cpp = 0, yp = 0, qp = 0;
  for (int k = 0; k < m; k++) {
    C a, b, c;
    if (k == 0) { a = a0; b = b0 - gm; c = c0; }
    else if (k == m - 1) { a = al; b = bl - cl * a0 / gm; c = cl; }
    else {
      row_coeffs<C, T>(g, lhs_type, s, lap.v, n, i, j, k, v);
      a = v[5]; b = v[18]; c = v[4];
    }
    const int64_t e = col + plane * k;
    const C uk = k == 0 ? gm : (k == m - 1 ? cl : (C)0);
    const C den = k == 0 ? b : b - a * cpp;
    const C cpk = c / den;
    const C yk = k == 0 ? (C)r[e] / den : ((C)r[e] - a * yp) / den;
    const C qk = k == 0 ? uk / den : (uk - a * qp) / den;
    cp[e] = (T)cpk; z[e] = (T)yk; q[e] = (T)qk;
    cpp = cpk; yp = yk; qp = qk;
  }
  const C ylast = yp, qlast = qp;
  C yn = yp, qn = qp;
  for (int k = m - 2; k >= 0; k--) {
    const int64_t e = col + plane * k;
    const C ck = (C)cp[e];
    yn = (C)z[e] - ck * yn;
    qn = (C)q[e] - ck * qn;
    z[e] = (T)yn; q[e] = (T)qn;
  }
  const C f = (yn + ag * ylast) / ((C)1 + qn + ag * qlast);
  for (int k = 0; k < m; k++) {
    const int64_t e = col + plane * k;
    z[e] = (T)((C)z[e] - f * (C)q[e]);
  }
}

template <typename T>
void launch_zline(chy_ctx *ctx, int lhs_type, const T *n, const T *r, T *z, T *cp, T *q)
{
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  const LapRow L = lap_row(ctx, lhs_type);
  const int64_t plane = (int64_t)ctx->g.nx * ctx->g.ny;
  hipLaunchKernelGGL((k_zline<T>), nblocks(plane), kBlock, 0, ctx->stream, ctx->g, lhs_type, s, L, n, r, z, cp, q);
}

// ---- z-line correction of the two-level preconditioner (fft2z) ----------------------
// The cyclic tridiagonal system of every z-column (the diagonal and +-z entries
// of A(n), as k_zline), factored once per solve: za = the -z entry, zi = 1 /
// pivot, zc = the eliminated +z entry, zq = the Sherman-Morrison vector of the
// periodic corner; per column cag = a0 / gamma and cden = 1 + q0 + cag q_(m-1).
// An application is then forward and back substitution and the rank-one
// correction, three passes up a column with the loads of KC planes in flight.
template <typename T>
__global__ __launch_bounds__(256) void k_zline_factor(Grid g, int lhs_type, SCoef s, LapRow lap,
                                                      const T *__restrict__ n, T *__restrict__ za,
                                                      T *__restrict__ zi, T *__restrict__ zc, T *__restrict__ zq,
                                                      double *__restrict__ cag, double *__restrict__ cden)
{
  using C = double;
  const int64_t plane = (int64_t)g.nx * g.ny;
  const int64_t col = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= plane) return;
  const int i = (int)(col % g.nx), j = (int)(col / g.nx), m = g.nz;  // m >= 3
  C v[19];
  row_coeffs<C, T>(g, lhs_type, s, lap.v, n, i, j, 0, v);
  const C a0 = v[5], b0 = v[18], c0 = v[4];
  row_coeffs<C, T>(g, lhs_type, s, lap.v, n, i, j, m - 1, v);
  const C al = v[5], bl = v[18], cl = v[4];
  const C gm = -b0, ag = a0 / gm;
  C cpp = 0, qp = 0;
  for (int k = 0; k < m; k++) {
    C a, b, c;
    if (k == 0) { a = a0; b = b0 - gm; c = c0; }
    else if (k == m - 1) { a = al; b = bl - cl * a0 / gm; c = cl; }
    else {
      row_coeffs<C, T>(g, lhs_type, s, lap.v, n, i, j, k, v);
      a = v[5]; b = v[18]; c = v[4];
    }
    const int64_t e = col + plane * k;
    const C uk = k == 0 ? gm : (k == m - 1 ? cl : (C)0);
    const C den = k == 0 ? b : b - a * cpp;
    const C cpk = c / den;
    const C qk = k == 0 ? uk / den : (uk - a * qp) / den;
    za[e] = (T)a; zi[e] = (T)((C)1 / den); zc[e] = (T)cpk; zq[e] = (T)qk;
    cpp = cpk; qp = qk;
  }
  const C qlast = qp;
  C qn = qp;
  for (int k = m - 2; k >= 0; k--) {
    const int64_t e = col + plane * k;
    qn = (C)zq[e] - (C)zc[e] * qn;
    zq[e] = (T)qn;
  }
  cag[col] = ag;
  cden[col] = (C)1 + qn + ag * qlast;
}

// z += scale times the z-line solve of res (res is overwritten by the
// intermediate y)
template <typename T>
__global__ __launch_bounds__(256) void k_zline_apply(Grid g, const T *__restrict__ za, const T *__restrict__ zi,
                                                     const T *__restrict__ zc, const T *__restrict__ zq,
                                                     const double *__restrict__ cag, const double *__restrict__ cden,
                                                     T *__restrict__ res, T *__restrict__ z, double scale)
{
  constexpr int KC = 16;
  const int64_t plane = (int64_t)g.nx * g.ny;
  const int64_t col = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= plane) return;
  const int m = g.nz;
  double y = 0.0;
  for (int k0 = 0; k0 < m; k0 += KC) {  // forward substitution
    T rr[KC], aa[KC], ii[KC];
#pragma unroll
    for (int u = 0; u < KC; u++) {
      const int64_t e = col + plane * (k0 + u);
      if (k0 + u < m) { rr[u] = res[e]; aa[u] = za[e]; ii[u] = zi[e]; }
    }
#pragma unroll
    for (int u = 0; u < KC; u++) {
      if (k0 + u < m) {
        y = ((double)rr[u] - (double)aa[u] * y) * (double)ii[u];
        res[col + plane * (k0 + u)] = (T)y;
      }
    }
  }
  const double ylast = y;
  double yn = y;
  for (int k0 = m - 2; k0 >= 0; k0 -= KC) {  // back substitution, planes k0, k0 - 1, ...
    T rr[KC], cc[KC];
#pragma unroll
    for (int u = 0; u < KC; u++) {
      const int k = k0 - u;
      if (k >= 0) { rr[u] = res[col + plane * k]; cc[u] = zc[col + plane * k]; }
    }
#pragma unroll
    for (int u = 0; u < KC; u++) {
      const int k = k0 - u;
      if (k >= 0) {
        yn = (double)rr[u] - (double)cc[u] * yn;
        res[col + plane * k] = (T)yn;
      }
    }
  }
  const double f = (yn + cag[col] * ylast) / cden[col];
  for (int k0 = 0; k0 < m; k0 += KC) {  // periodic correction, added to z
    T rr[KC], qq[KC], zz[KC];
#pragma unroll
    for (int u = 0; u < KC; u++) {
      const int64_t e = col + plane * (k0 + u);
      if (k0 + u < m) { rr[u] = res[e]; qq[u] = zq[e]; zz[u] = z[e]; }
    }
#pragma unroll
    for (int u = 0; u < KC; u++) {
      if (k0 + u < m) z[col + plane * (k0 + u)] = (T)((double)zz[u] + scale * ((double)rr[u] - f * (double)qq[u]));
    }
  }
}

// The fft2z preconditioner's z-line stage with B along z (K_x = K_y = 0):
// z += e2 + zline(d0 - A(n) e2), where d0 = r - A(n) z_fft was stored by the
// column-sum pass and e2 = sum_q y2[q] Z2[q] is the 2-D correction, constant
// along z.  A(n) applied to a field constant along z keeps only the in-plane
// entries of each row (0-3 and 6-9; the z entries multiply e2_c - e2_c), and
// those are linear in the five in-plane densities, so per column
//     (A e2)(k) = Kc n_c + Kxp n_(x+1) + Kxm n_(x-1) + Kyp n_(y+1) + Kym n_(y-1)
// with the K formed once from the e2 differences de_q = e2_q - e2_c (the row
// of lhs.c:480-511 with s_xz = s_yz = s_zx = s_zy = 0, regrouped by density).
// This replaces a residual pass over r, z and n and the pass adding e2 to z.
template <typename T, int NQ>
__global__ __launch_bounds__(256) void k_zline_apply_e2(Grid g, const T *__restrict__ za, const T *__restrict__ zi,
                                                        const T *__restrict__ zc, const T *__restrict__ zq,
                                                        const double *__restrict__ cag,
                                                        const double *__restrict__ cden, T *__restrict__ res,
                                                        T *__restrict__ z, const T *__restrict__ n, SCoef s,
                                                        const T *__restrict__ Z2, const double *__restrict__ y2)
{
  constexpr int KC = 16;
  const int64_t plane = (int64_t)g.nx * g.ny;
  const int64_t col = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= plane) return;
  const int m = g.nz;
  const int i = (int)(col % g.nx), j = (int)(col / g.nx);
  const int ip = i + 1 == g.nx ? 0 : i + 1, im = i == 0 ? g.nx - 1 : i - 1;
  const int jp = j + 1 == g.ny ? 0 : j + 1, jm = j == 0 ? g.ny - 1 : j - 1;
  double yq[NQ];
#pragma unroll
  for (int q = 0; q < NQ; q++) yq[q] = y2[q];
  auto e2 = [&](int ii, int jj) {
    const int64_t c = (int64_t)ii + (int64_t)g.nx * jj;
    double e = 0.0;
#pragma unroll
    for (int q = 0; q < NQ; q++) e += yq[q] * (double)Z2[(int64_t)q * plane + c];
    return e;
  };
  const double ec = e2(i, j);
  const double de0 = e2(ip, j) - ec, de1 = e2(im, j) - ec, de2 = e2(i, jp) - ec, de3 = e2(i, jm) - ec;
  const double de6 = e2(ip, jp) - ec, de7 = e2(ip, jm) - ec, de8 = e2(im, jp) - ec, de9 = e2(im, jm) - ec;
  const double kc = s.sxx * (de0 + de1) + s.syy * (de2 + de3) + (s.sxy + s.syx) * ((de6 - de7) + (de9 - de8));
  const double kxp = s.sxx * de0 + s.sxy * (de2 - de3) + s.sxy * (de6 - de7);
  const double kxm = s.sxx * de1 - s.sxy * (de2 - de3) + s.sxy * (de9 - de8);
  const double kyp = s.syx * (de0 - de1) + s.syy * de2 + s.syx * (de6 - de8);
  const double kym = -s.syx * (de0 - de1) + s.syy * de3 + s.syx * (de9 - de7);
  const int64_t oxp = ip - i, oxm = im - i, oyp = (int64_t)g.nx * (jp - j), oym = (int64_t)g.nx * (jm - j);
  double y = 0.0;
  // (eight values per plane: half the batch of the other passes keeps the
  // loads in flight within the register file)
  constexpr int KF = KC / 2;
  for (int k0 = 0; k0 < m; k0 += KF) {  // forward substitution on d0 - A e2
    T rr[KF], aa[KF], ii[KF], nc[KF], nxp[KF], nxm[KF], nyp[KF], nym[KF];
#pragma unroll
    for (int u = 0; u < KF; u++) {
      const int64_t e = col + plane * (k0 + u);
      if (k0 + u < m) {
        rr[u] = res[e]; aa[u] = za[e]; ii[u] = zi[e];
        nc[u] = n[e]; nxp[u] = n[e + oxp]; nxm[u] = n[e + oxm]; nyp[u] = n[e + oyp]; nym[u] = n[e + oym];
      }
    }
#pragma unroll
    for (int u = 0; u < KF; u++) {
      if (k0 + u < m) {
        const double ae = kc * (double)nc[u] + kxp * (double)nxp[u] + kxm * (double)nxm[u] + kyp * (double)nyp[u] +
                          kym * (double)nym[u];
        y = (((double)rr[u] - ae) - (double)aa[u] * y) * (double)ii[u];
        res[col + plane * (k0 + u)] = (T)y;
      }
    }
  }
  const double ylast = y;
  double yn = y;
  for (int k0 = m - 2; k0 >= 0; k0 -= KC) {  // back substitution, planes k0, k0 - 1, ...
    T rr[KC], cc[KC];
#pragma unroll
    for (int u = 0; u < KC; u++) {
      const int k = k0 - u;
      if (k >= 0) { rr[u] = res[col + plane * k]; cc[u] = zc[col + plane * k]; }
    }
#pragma unroll
    for (int u = 0; u < KC; u++) {
      const int k = k0 - u;
      if (k >= 0) {
        yn = (double)rr[u] - (double)cc[u] * yn;
        res[col + plane * k] = (T)yn;
      }
    }
  }
  const double f = (yn + cag[col] * ylast) / cden[col];
  for (int k0 = 0; k0 < m; k0 += KC) {  // periodic correction; z += e2 + the solve
    T rr[KC], qq[KC], zz[KC];
#pragma unroll
    for (int u = 0; u < KC; u++) {
      const int64_t e = col + plane * (k0 + u);
      if (k0 + u < m) { rr[u] = res[e]; qq[u] = zq[e]; zz[u] = z[e]; }
    }
#pragma unroll
    for (int u = 0; u < KC; u++) {
      if (k0 + u < m) z[col + plane * (k0 + u)] = (T)(((double)zz[u] + ec) + ((double)rr[u] - f * (double)qq[u]));
    }
  }
}

// ---- z-line stage with the columns cut into segments -------------------------------
// k_zline_apply and k_zline_apply_e2 in one pass over memory: NC consecutive
// columns a block, each cut into SG segments of P planes, a thread a segment,
// whose values stay in registers from the load to the store.  The forward and
// back substitutions are first-order linear recurrences: every thread composes
// the affine map of its planes, runs through the maps before (after) it for the
// value that enters them, and then its planes with the sequential formulas.
//
// One thread a column leaves most of the chip idle (4 blocks at 32^2, 64 at
// 128^2) and reads the intermediate values back twice.  Measured with the 2-D
// correction folded in, column walk -> segments: 32^3 FP64 19.3 -> 4.7 us, 64^3
// FP32 23.1 -> 5.8, 128^3 FP32 45.6 -> 16.2 and FP64 72.7 -> 28.0, 128x128x256
// FP64 172 -> 66, 256^3 FP32 145 -> 137.  On the largest FP64 grids the walk's
// block reads longer runs of each plane: 256x256x128 137 -> 129, but 256^3 271
// -> 297, so those keep the walk, as columns beyond 256 planes do, whose values
// do not fit the registers.  Blocks of 16 columns were the faster ones but for
// FP32 columns of more than 64 planes (64-byte runs of a plane against 128);
// 8 to 64 segments were tried with 1 to 16 planes each.
template <typename T, int NC, int SG, int P, bool E2>
__global__ __launch_bounds__(NC * SG) void k_zline_seg(Grid g, const T *__restrict__ za, const T *__restrict__ zi,
                                                       const T *__restrict__ zc, const T *__restrict__ zq,
                                                       const double *__restrict__ cag,
                                                       const double *__restrict__ cden, const T *__restrict__ res,
                                                       T *__restrict__ z, const T *__restrict__ n, SCoef s,
                                                       const T *__restrict__ Z2, const double *__restrict__ y2,
                                                       double scale)
{
  __shared__ double mA[SG][NC], mB[SG][NC], ends[2][NC];
  uint32_t bx, by, bz;
  (void)xcd_tile(bx, by, bz);
  const int plane = g.nx * g.ny, m = g.nz, cx = threadIdx.x % NC, sg = threadIdx.x / NC;
  const int col = (int)bx * NC + cx;
  const bool live = col < plane;
  // (loads past the last plane or column read a valid value that is not used)
  int64_t e[P];
#pragma unroll
  for (int u = 0; u < P; u++) {
    const int k = sg * P + u;
    e[u] = (live ? col : 0) + (int64_t)plane * (k < m ? k : m - 1);
  }
  double r[P];
  T cc[P];
  double ec = 0.0;
  {
    T rr[P], aa[P], ii[P];
#pragma unroll
    for (int u = 0; u < P; u++) {
      rr[u] = res[e[u]];
      aa[u] = za[e[u]];
      ii[u] = zi[e[u]];
      cc[u] = zc[e[u]];
    }
    if constexpr (E2) {
      // (A e2)(k) from the column's five constants, as k_zline_apply_e2
      int i, j, k_;
      split_cell(g, live ? col : 0, i, j, k_);
      const int ip = i + 1 == g.nx ? 0 : i + 1, im = i == 0 ? g.nx - 1 : i - 1;
      const int jp = j + 1 == g.ny ? 0 : j + 1, jm = j == 0 ? g.ny - 1 : j - 1;
      const int64_t oxp = ip - i, oxm = im - i, oyp = (int64_t)g.nx * (jp - j), oym = (int64_t)g.nx * (jm - j);
      T nc[P], nxp[P], nxm[P], nyp[P], nym[P];
#pragma unroll
      for (int u = 0; u < P; u++) {
        nc[u] = n[e[u]];
        nxp[u] = n[e[u] + oxp]; nxm[u] = n[e[u] + oxm];
        nyp[u] = n[e[u] + oyp]; nym[u] = n[e[u] + oym];
      }
      const double y0 = y2[0], y1 = y2[1];
      auto e2 = [&](int ii, int jj) {
        const int q = ii + g.nx * jj;
        return y0 * (double)Z2[q] + y1 * (double)Z2[(int64_t)plane + q];
      };
      ec = e2(i, j);
      const double de0 = e2(ip, j) - ec, de1 = e2(im, j) - ec, de2 = e2(i, jp) - ec, de3 = e2(i, jm) - ec;
      const double de6 = e2(ip, jp) - ec, de7 = e2(ip, jm) - ec, de8 = e2(im, jp) - ec, de9 = e2(im, jm) - ec;
      const double kc = s.sxx * (de0 + de1) + s.syy * (de2 + de3) + (s.sxy + s.syx) * ((de6 - de7) + (de9 - de8));
      const double kxp = s.sxx * de0 + s.sxy * (de2 - de3) + s.sxy * (de6 - de7);
      const double kxm = s.sxx * de1 - s.sxy * (de2 - de3) + s.sxy * (de9 - de8);
      const double kyp = s.syx * (de0 - de1) + s.syy * de2 + s.syx * (de6 - de8);
      const double kym = -s.syx * (de0 - de1) + s.syy * de3 + s.syx * (de9 - de7);
#pragma unroll
      for (int u = 0; u < P; u++)
        r[u] = (double)rr[u] - (kc * (double)nc[u] + kxp * (double)nxp[u] + kxm * (double)nxm[u] + kyp * (double)nyp[u] +
                                kym * (double)nym[u]);
    } else {
#pragma unroll
      for (int u = 0; u < P; u++) r[u] = (double)rr[u];
    }
    double A = 1.0, B = 0.0;
#pragma unroll
    for (int u = 0; u < P; u++) {
      if (sg * P + u < m) {
        const double iv = (double)ii[u], al = -(double)aa[u] * iv;
        A = al * A;
        B = al * B + r[u] * iv;
      }
    }
    mA[sg][cx] = A;
    mB[sg][cx] = B;
    __syncthreads();
    double y = 0.0;
    for (int t = 0; t < sg; t++) y = mA[t][cx] * y + mB[t][cx];
#pragma unroll
    for (int u = 0; u < P; u++) {
      if (sg * P + u < m) {
        y = (r[u] - (double)aa[u] * y) * (double)ii[u];
        r[u] = y;
      }
    }
    if (sg == (m - 1) / P) ends[0][cx] = y;
  }
  __syncthreads();  // (the maps are read; the last y is known)
  const double ylast = ends[0][cx];
  double A = 1.0, B = 0.0;
#pragma unroll
  for (int u = P - 1; u >= 0; u--) {
    const int k = sg * P + u;
    if (k == m - 1) { A = 0.0; B = ylast; }
    else if (k < m - 1) { B = r[u] - (double)cc[u] * B; A = -(double)cc[u] * A; }
  }
  mA[sg][cx] = A;
  mB[sg][cx] = B;
  // the final operands are in flight while the maps are run through
  T qq[P], zz[P];
#pragma unroll
  for (int u = 0; u < P; u++) {
    qq[u] = zq[e[u]];
    zz[u] = z[e[u]];
  }
  const double ag = live ? cag[col] : 0.0, dn = live ? cden[col] : 1.0;
  __syncthreads();
  double x = 0.0;
  for (int t = SG - 1; t > sg; t--) x = mA[t][cx] * x + mB[t][cx];
#pragma unroll
  for (int u = P - 1; u >= 0; u--) {
    const int k = sg * P + u;
    if (k == m - 1) x = ylast;
    else if (k < m - 1) { x = r[u] - (double)cc[u] * x; r[u] = x; }
  }
  if (sg == 0) ends[1][cx] = x;
  __syncthreads();
  const double f = (ends[1][cx] + ag * ylast) / dn;
#pragma unroll
  for (int u = 0; u < P; u++) {
    if (live && sg * P + u < m)
      z[e[u]] = (T)(((double)zz[u] + ec) + scale * (r[u] - f * (double)qq[u]));
  }
}

// ---- multigrid levels with z fastest ----------------------------------------------
// The multigrid keeps its level fields as [y][x][z]: a group of W lanes owns a
// column, P consecutive planes a lane (W P >= nz), so that the stencil around a
// column, the column's z-line system and its solve are contiguous loads and
// register moves.  A smoothing sweep is then one launch, x' = x + omega zline^-1 (b
// - A x), the residual never stored: 4 to 6 us on 96 x 80 x 50 and its coarse
// levels (FP32), where with x fastest it took a residual pass (4 to 6 us) and a
// solve (16.6 us walking 96 x 80 columns, 4.6 us on fewer).  A preconditioner
// application there went from 65 launches to 38, 339 -> 149 us.  Whole solves
// with a run's noise, to 1e-10 (mixed) and 1e-11, B oblique: 96 x 80 x 50 mixed
// 29.3 -> 12.4 ms, 64 x 48 x 40 FP64 23.9 -> 10.4, 160 x 144 x 100 mixed 89.7 ->
// 38.8; B along z: 160 x 144 x 100 mixed 10.3 -> 4.8, 256^3 mixed 26.0 -> 16.1
// (all of the solver's changes in them).  What is left is latency: one launch
// after another on grids that a chip of 256 CUs does in a microsecond or two.
// (All sweeps of the coarsest level in one workgroup, in LDS and registers,
// took 27 to 52 us against 8 launches of 4 to 5: the scans' instructions
// bound a single CU.)

// Bases of a column and of its neighbours along x, y and diagonally
struct ColNb { int64_t c, xp, xm, yp, ym, pp, pm, mp, mm; };

__device__ __forceinline__ ColNb col_nb(const Grid &g, int col)
{
  int i, j, k_;
  split_cell(g, col, i, j, k_);
  const int ip = i + 1 == g.nx ? 0 : i + 1, im = i == 0 ? g.nx - 1 : i - 1;
  const int jp = j + 1 == g.ny ? 0 : j + 1, jm = j == 0 ? g.ny - 1 : j - 1;
  auto at = [&](int a, int b) { return ((int64_t)a + (int64_t)g.nx * b) * g.nz; };
  return {at(i, j), at(ip, j), at(im, j), at(i, jp), at(i, jm), at(ip, jp), at(ip, jm), at(im, jp), at(im, jm)};
}

// Row of A x at plane k of column q
template <typename T, typename C, bool DIFF, int OP>
__device__ __forceinline__ C zf_row(const Grid &g, const SCoef &s, const LapRow &lap, const T *__restrict__ n,
                                    const T *__restrict__ x, const ColNb &q, int k)
{
  const int kp = k + 1 == g.nz ? 0 : k + 1, km = k == 0 ? g.nz - 1 : k - 1;
  C nf[4] = {(C)0, (C)0, (C)0, (C)0}, n0 = (C)0, nzp = (C)0, nzm = (C)0;
  if (OP != kOpConst) {
    n0 = (C)n[q.c + k]; nzp = (C)n[q.c + kp]; nzm = (C)n[q.c + km];
    nf[0] = (C)n[q.xp + k]; nf[1] = (C)n[q.xm + k]; nf[2] = (C)n[q.yp + k]; nf[3] = (C)n[q.ym + k];
  }
  const C xf[4] = {(C)x[q.xp + k], (C)x[q.xm + k], (C)x[q.yp + k], (C)x[q.ym + k]};
  const C xe[4] = {(C)x[q.pp + k], (C)x[q.pm + k], (C)x[q.mp + k], (C)x[q.mm + k]};
  C xfp[4], xfm[4];
  if (OP != kOpKz) {
    xfp[0] = (C)x[q.xp + kp]; xfp[1] = (C)x[q.xm + kp]; xfp[2] = (C)x[q.yp + kp]; xfp[3] = (C)x[q.ym + kp];
    xfm[0] = (C)x[q.xp + km]; xfm[1] = (C)x[q.xm + km]; xfm[2] = (C)x[q.yp + km]; xfm[3] = (C)x[q.ym + km];
  } else {
#pragma unroll
    for (int e = 0; e < 4; e++) xfp[e] = xfm[e] = (C)0;
  }
  return row_apply<C, DIFF, OP>(s, lap, n0, nf, nzp, nzm, (C)x[q.c + k], xf, xe, (C)x[q.c + kp], (C)x[q.c + km], xfp, xfm);
}

// Inclusive scan of the affine maps y -> A y + B over groups of W lanes, lower
// lanes' maps first (UP) or higher lanes' first: four register moves within the
// rows of 16 lanes, then the row totals of the rows before it.  (Six shuffles
// of each value through LDS made a sweep take 5.3 us on 64 x 48 x 40 FP64 and 5.6
// on 96 x 80 x 50 FP32, which now takes 4.5 and 4.9; a solve there 13.2 -> 12.4
// and 14.9 -> 14.2 ms.)
template <bool UP, int W>
__device__ __forceinline__ void affine_scan(double &A, double &B)
{
  auto step = [&](auto n) {
    constexpr int ctrl = (UP ? 0x110 : 0x100) + decltype(n)::value;  // row_shr:n, row_shl:n
    const double A2 = dpp_move<ctrl>(A, 1.0), B2 = dpp_move<ctrl>(B, 0.0);
    B = A * B2 + B;
    A = A * A2;
  };
  step(std::integral_constant<int, 1>());
  step(std::integral_constant<int, 2>());
  step(std::integral_constant<int, 4>());
  step(std::integral_constant<int, 8>());
  if constexpr (W > 16) {
    const int row = (int)(threadIdx.x & 63) >> 4;
    // the maps of whole rows, in the order in which they apply: rows 0, 1, 2 (UP) or 3, 2, 1
    const double a0 = lane_value(A, UP ? 15 : 48), b0 = lane_value(B, UP ? 15 : 48);
    const double a2 = lane_value(A, UP ? 47 : 16), b2 = lane_value(B, UP ? 47 : 16);
    double a = 1.0, b = 0.0;
    if constexpr (W == 32) {
      if (UP) { if (row & 1) { a = row == 1 ? a0 : a2; b = row == 1 ? b0 : b2; } }
      else if (!(row & 1)) { a = row == 2 ? a0 : a2; b = row == 2 ? b0 : b2; }
    } else {
      const double a1 = lane_value(A, UP ? 31 : 32), b1 = lane_value(B, UP ? 31 : 32);
      const double a10 = a1 * a0, b10 = a1 * b0 + b1, a210 = a2 * a10, b210 = a2 * b10 + b2;
      const int after = UP ? row : 3 - row;  // rows whose maps come first
      a = after == 0 ? 1.0 : after == 1 ? a0 : after == 2 ? a10 : a210;
      b = after == 0 ? 0.0 : after == 1 ? b0 : after == 2 ? b10 : b210;
    }
    B = A * b + B;
    A = A * a;
  }
}

// The cyclic z-line solve of the column held by W lanes (lane L: planes L P ..
// L P + P - 1), r in and the solution in r.  The forward and back
// substitutions are first-order linear recurrences, y_k = alpha_k y_(k-1) +
// beta_k: each lane composes the affine maps of its planes, a scan over the W
// lanes gives the value entering them, and the lane then runs its planes with
// the sequential formulas.
template <typename T, int W, int P>
__device__ __forceinline__ void zline_lanes(int L, int m, double (&r)[P], const double (&a)[P], const double (&iv)[P],
                                            const double (&c)[P], const double (&q)[P], double cag, double cden)
{
  double A = 1.0, B = 0.0;
#pragma unroll
  for (int u = 0; u < P; u++) {
    if (L * P + u < m) {
      const double al = -a[u] * iv[u], be = r[u] * iv[u];
      A = al * A;
      B = al * B + be;
    }
  }
  affine_scan<true, W>(A, B);
  double yv = dpp_move<0x138>(B, 0.0);  // (wave_shr:1) the exclusive prefix applied to y_(-1) = 0
  if (L == 0) yv = 0.0;
#pragma unroll
  for (int u = 0; u < P; u++) {
    if (L * P + u < m) {
      yv = (r[u] - a[u] * yv) * iv[u];
      r[u] = yv;
    }
  }
  const double ylast = W == 64 ? lane_value(yv, (m - 1) / P) : __shfl(yv, (m - 1) / P, W);
  // backward: x_(m-1) = y_(m-1), x_k = y_k - c_k x_(k+1); higher planes first
  A = 1.0; B = 0.0;
#pragma unroll
  for (int u = P - 1; u >= 0; u--) {
    const int k = L * P + u;
    if (k == m - 1) { A = 0.0; B = ylast; }
    else if (k < m - 1) { B = -c[u] * B + r[u]; A = -c[u] * A; }
  }
  affine_scan<false, W>(A, B);
  double xv = dpp_move<0x130>(B, 0.0);  // (wave_shl:1)
  if (L == W - 1) xv = 0.0;
#pragma unroll
  for (int u = P - 1; u >= 0; u--) {
    const int k = L * P + u;
    if (k == m - 1) xv = ylast;
    else if (k < m - 1) { xv = r[u] - c[u] * xv; r[u] = xv; }
  }
  const double f = ((W == 64 ? lane_value(xv, 0) : __shfl(xv, 0, W)) + cag * ylast) / cden;
#pragma unroll
  for (int u = 0; u < P; u++) r[u] -= f * q[u];
}

// r changes from consecutive lanes on consecutive planes to the lanes' own P
// planes (to_lanes), or back, through the LDS row t of W P values.
template <int W, int P>
__device__ __forceinline__ void turn_planes(bool to_lanes, int L, double (&r)[P], double *t)
{
  if (P == 1) return;
  wave_sync();  // (earlier reads of the row)
#pragma unroll
  for (int u = 0; u < P; u++) t[to_lanes ? u * W + L : L * P + u] = r[u];
  wave_sync();
#pragma unroll
  for (int u = 0; u < P; u++) r[u] = t[to_lanes ? L * P + u : u * W + L];
}

// One column's sweep: xo = x + omega zline^-1 (b - A x), or with FIRST (x = 0)
// xo = omega zline^-1 b.  zf: the factors za, zi, zc, zq (nc each).  With
// several planes a lane, the fields are read and written with consecutive
// lanes on consecutive planes, and the residual and the solution change to and
// from the lanes' own planes through the wave's LDS row t (W P values); the
// factors of a lane's planes are consecutive in memory.
template <typename T, int W, int P, int OP, bool FIRST>
__device__ __forceinline__ void mg_sweep_col(const Grid &g, const SCoef &s, const LapRow &lap, int col, int L,
                                             const T *__restrict__ n, const T *__restrict__ zf,
                                             const double *__restrict__ zcol, const T *__restrict__ b, const T *x,
                                             T *xo, double omega, double *t)
{
  using C = typename std::conditional<sizeof(T) == 4, float, double>::type;
  const int m = g.nz;
  const ColNb nb = col_nb(g, col);
  double r[P], a[P], iv[P], c[P], q[P], xk[P];
#pragma unroll
  for (int u = 0; u < P; u++) {
    const int k = L * P + u;
    a[u] = iv[u] = c[u] = q[u] = 0.0;
    if (k < m) {
      const int64_t e = nb.c + k;
      a[u] = (double)zf[e]; iv[u] = (double)zf[g.nc + e]; c[u] = (double)zf[2 * g.nc + e]; q[u] = (double)zf[3 * g.nc + e];
    }
  }
#pragma unroll
  for (int u = 0; u < P; u++) {
    const int k = u * W + L;
    r[u] = xk[u] = 0.0;
    if (k < m) {
      const int64_t e = nb.c + k;
      r[u] = (double)b[e];
      if (!FIRST) {
        xk[u] = (double)x[e];
        r[u] -= (double)zf_row<T, C, sizeof(T) == 4, OP>(g, s, lap, n, x, nb, k);
      }
    }
  }
  const int64_t plane = (int64_t)g.nx * g.ny;
  turn_planes<W, P>(true, L, r, t);
  zline_lanes<T, W, P>(L, m, r, a, iv, c, q, zcol[col], zcol[plane + col]);
  turn_planes<W, P>(false, L, r, t);
#pragma unroll
  for (int u = 0; u < P; u++) {
    const int k = u * W + L;
    if (k < m) xo[nb.c + k] = (T)(xk[u] + omega * r[u]);
  }
}

template <typename T, int W, int P, int OP, bool FIRST>
__global__ __launch_bounds__(256) void k_mg_sweep(Grid g, SCoef s, LapRow lap, const T *__restrict__ n,
                                                  const T *__restrict__ zf, const double *__restrict__ zcol,
                                                  const T *__restrict__ b, const T *__restrict__ x, T *__restrict__ xo,
                                                  double omega)
{
  __shared__ double t[P == 1 ? 1 : 4][W * P];
  const int col = (int)(blockIdx.x * (256 / W) + threadIdx.x / W);
  if (col >= g.nx * g.ny) return;  // the column's W lanes leave together
  mg_sweep_col<T, W, P, OP, FIRST>(g, s, lap, col, (int)(threadIdx.x % W), n, zf, zcol, b, x, xo, omega,
                                   t[P == 1 ? 0 : threadIdx.x / W]);
}

// r = b - A x, one thread per node
template <typename T, int OP>
__global__ __launch_bounds__(256) void k_mg_residual(Grid g, SCoef s, LapRow lap, const T *__restrict__ n,
                                                     const T *__restrict__ b, const T *__restrict__ x,
                                                     T *__restrict__ r)
{
  using C = typename std::conditional<sizeof(T) == 4, float, double>::type;
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= g.nc) return;
  const int col = (int)((uint32_t)e / (uint32_t)g.nz), k = (int)((uint32_t)e - (uint32_t)col * (uint32_t)g.nz);
  const ColNb nb = col_nb(g, col);
  r[e] = (T)((double)b[e] - (double)zf_row<T, C, sizeof(T) == 4, OP>(g, s, lap, n, x, nb, k));
}

// dst[c][k] = src[k][c] of up to five fields (TO_Z), or the reverse
template <typename T>
struct Fields5 { const T *src[5]; T *dst[5]; };
template <typename T, bool TO_Z>
__global__ __launch_bounds__(256) void k_mg_transpose(int cols, int nz, Fields5<T> f)
{
  __shared__ T t[32][33];
  const T *__restrict__ src = f.src[blockIdx.z];
  T *__restrict__ dst = f.dst[blockIdx.z];
  const int c0 = (int)blockIdx.x * 32, k0 = (int)blockIdx.y * 32, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
#pragma unroll
  for (int u = 0; u < 32; u += 8) {
    const int c = TO_Z ? c0 + tx : c0 + ty + u, k = TO_Z ? k0 + ty + u : k0 + tx;
    if (c < cols && k < nz) t[ty + u][tx] = TO_Z ? src[(int64_t)k * cols + c] : src[(int64_t)c * nz + k];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 32; u += 8) {
    const int c = TO_Z ? c0 + ty + u : c0 + tx, k = TO_Z ? k0 + tx : k0 + ty + u;
    if (c < cols && k < nz) {
      if (TO_Z) dst[(int64_t)c * nz + k] = t[tx][ty + u];
      else dst[(int64_t)k * cols + c] = t[tx][ty + u];
    }
  }
}

template <typename T>
void launch_mg_transpose(chy_ctx *ctx, const Grid &g, bool to_z, int nf, const T *const *src, T *const *dst)
{
  Fields5<T> f = {};
  for (int q = 0; q < nf; q++) { f.src[q] = src[q]; f.dst[q] = dst[q]; }
  const int cols = g.nx * g.ny;
  const dim3 grid((unsigned)((cols + 31) / 32), (unsigned)((g.nz + 31) / 32), (unsigned)nf);
  if (to_z) hipLaunchKernelGGL((k_mg_transpose<T, true>), grid, 256, 0, ctx->stream, cols, g.nz, f);
  else hipLaunchKernelGGL((k_mg_transpose<T, false>), grid, 256, 0, ctx->stream, cols, g.nz, f);
}

// The operator kind and row constants of a level
static int mg_op(chy_ctx *ctx, const double d[3], SCoef &s, LapRow &L)
{
  const int lt = ctx->prm.lhs_type;
  s = full_scoef(d, ctx->prm.kappa_e);
  uniform_row(lt == CHY_LHS_FULL ? CHY_LHS_IDENTITY : lt, d, ctx->prm.kappa_e, 0.0, L.v);
  return kz_operator(lt, s) ? kOpKz : lt == CHY_LHS_FULL ? kOpFull : kOpConst;
}

// Lanes per column and planes per lane for nz planes (at most kMgMaxPlanes)
#define MG_WP(nz, call)                                                    \
  do {                                                                     \
    if (nz <= 16) { constexpr int W = 16, P = 1; call; }                   \
    else if (nz <= 32) { constexpr int W = 32, P = 1; call; }              \
    else if (nz <= 64) { constexpr int W = 64, P = 1; call; }              \
    else if (nz <= 128) { constexpr int W = 64, P = 2; call; }             \
    else if (nz <= 256) { constexpr int W = 64, P = 4; call; }             \
    else { constexpr int W = 64, P = 8; call; }                            \
  } while (0)
#define MG_OP(op, call)                                                    \
  do {                                                                     \
    if (op == kOpKz) { constexpr int OP = kOpKz; call; }                   \
    else if (op == kOpFull) { constexpr int OP = kOpFull; call; }          \
    else { constexpr int OP = kOpConst; call; }                            \
  } while (0)

template <typename T>
void launch_mg_sweep(chy_ctx *ctx, const Grid &g, const double d[3], const T *n, const T *zf, const double *zcol,
                     const T *b, const T *x, T *xo, double omega)
{
  SCoef s;
  LapRow L;
  const int op = mg_op(ctx, d, s, L), cols = g.nx * g.ny;
  MG_WP(g.nz, MG_OP(op, {
    const unsigned nb = (unsigned)((cols + 256 / W - 1) / (256 / W));
    if (x)
      hipLaunchKernelGGL((k_mg_sweep<T, W, P, OP, false>), nb, 256, 0, ctx->stream, g, s, L, n, zf, zcol, b, x, xo, omega);
    else
      hipLaunchKernelGGL((k_mg_sweep<T, W, P, OP, true>), nb, 256, 0, ctx->stream, g, s, L, n, zf, zcol, b, x, xo, omega);
  }));
}

template <typename T>
void launch_mg_residual(chy_ctx *ctx, const Grid &g, const double d[3], const T *n, const T *b, const T *x, T *r)
{
  SCoef s;
  LapRow L;
  const int op = mg_op(ctx, d, s, L);
  MG_OP(op, hipLaunchKernelGGL((k_mg_residual<T, OP>), nblocks(g.nc), 256, 0, ctx->stream, g, s, L, n, b, x, r));
}

#define MG_INST(T)                                                                                                  \
  template void launch_mg_transpose<T>(chy_ctx *, const Grid &, bool, int, const T *const *, T *const *);           \
  template void launch_mg_sweep<T>(chy_ctx *, const Grid &, const double[3], const T *, const T *, const double *,  \
                                   const T *, const T *, T *, double);                                              \
  template void launch_mg_residual<T>(chy_ctx *, const Grid &, const double[3], const T *, const T *, const T *, T *);
MG_INST(double)
MG_INST(float)
#undef MG_INST

// Both once-per-solve column walks of the two-level preconditioners for the
// full operator on columns beyond 256 planes (COEF: k_zcoef's z-means, FACT:
// k_zline_factor's factors, the same arithmetic in the same order), in one walk up each column with the
// density star of KC planes loaded before any is used; the back sweep of the
// Sherman-Morrison vector reads KC planes at a time too.
template <typename T, bool COEF, bool FACT>
__global__ __launch_bounds__(256) void k_zcolumn(Grid g, SCoef s, const T *__restrict__ n, T *__restrict__ Cz,
                                                 T *__restrict__ za, T *__restrict__ zi, T *__restrict__ zc,
                                                 T *__restrict__ zq, double *__restrict__ cag,
                                                 double *__restrict__ cden)
{
  using C = double;
  constexpr int KC = 8;
  const int64_t plane = (int64_t)g.nx * g.ny;
  const int64_t col = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= plane) return;
  const int i = (int)(col % g.nx), j = (int)(col / g.nx), m = g.nz;  // m >= 3
  const int64_t oxp = lin(g, i + 1, j, 0), oxm = lin(g, i - 1, j, 0), oyp = lin(g, i, j + 1, 0),
                oym = lin(g, i, j - 1, 0);
  auto nat = [&](int64_t o, int k) { return (C)n[o + plane * (int64_t)wrapi(k, m)]; };
  // rows at k = 0 and k = m - 1 (the periodic corner)
  C v[19];
  row_from_star<C>(s, nat(col, 0), nat(oxp, 0), nat(oxm, 0), nat(oyp, 0), nat(oym, 0), nat(col, 1), nat(col, -1), v);
  const C a0 = v[5], b0 = v[18], c0 = v[4];
  row_from_star<C>(s, nat(col, m - 1), nat(oxp, m - 1), nat(oxm, m - 1), nat(oyp, m - 1), nat(oym, m - 1),
                   nat(col, m), nat(col, m - 2), v);
  const C al = v[5], bl = v[18], cl = v[4];
  const C gm = -b0, ag = a0 / gm;
  C acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  C cpp = 0, qp = 0;
  for (int k0 = 0; k0 < m; k0 += KC) {
    // planes k0 - 1 .. k0 + KC of the column, and the x-y neighbours of k0 .. k0 + KC - 1
    T nc_[KC + 2], xp[KC], xm[KC], yp[KC], ym[KC];
#pragma unroll
    for (int u = 0; u < KC + 2; u++) nc_[u] = n[col + plane * (int64_t)wrapi(k0 - 1 + u < m + 1 ? k0 - 1 + u : m, m)];
#pragma unroll
    for (int u = 0; u < KC; u++) {
      const int64_t pk = plane * (int64_t)(k0 + u < m ? k0 + u : m - 1);
      xp[u] = n[oxp + pk]; xm[u] = n[oxm + pk]; yp[u] = n[oyp + pk]; ym[u] = n[oym + pk];
    }
#pragma unroll
    for (int u = 0; u < KC; u++) {
      const int k = k0 + u;
      if (k >= m) break;
      row_from_star<C>(s, (C)nc_[u + 1], (C)xp[u], (C)xm[u], (C)yp[u], (C)ym[u], (C)nc_[u + 2], (C)nc_[u], v);
      if (COEF) {
#pragma unroll
        for (int q = 0; q < 19; q++) acc[kGroup19[q]] += v[q];
      }
      if (FACT) {
        C a, b, c;
        if (k == 0) { a = a0; b = b0 - gm; c = c0; }
        else if (k == m - 1) { a = al; b = bl - cl * a0 / gm; c = cl; }
        else { a = v[5]; b = v[18]; c = v[4]; }
        const int64_t e = col + plane * k;
        const C uk = k == 0 ? gm : (k == m - 1 ? cl : (C)0);
        const C den = k == 0 ? b : b - a * cpp;
        const C cpk = c / den;
        const C qk = k == 0 ? uk / den : (uk - a * qp) / den;
        za[e] = (T)a; zi[e] = (T)((C)1 / den); zc[e] = (T)cpk; zq[e] = (T)qk;
        cpp = cpk; qp = qk;
      }
    }
  }
  if (COEF) {
#pragma unroll
    for (int o = 0; o < 9; o++) Cz[o * plane + col] = (T)(acc[o] / (double)m);
  }
  if (FACT) {
    const C qlast = qp;
    C qn = qp;
    for (int k0 = m - 2; k0 >= 0; k0 -= KC) {  // planes k0, k0 - 1, ...
      T qq[KC], cc[KC];
#pragma unroll
      for (int u = 0; u < KC; u++) {
        const int k = k0 - u >= 0 ? k0 - u : 0;
        qq[u] = zq[col + plane * k]; cc[u] = zc[col + plane * k];
      }
#pragma unroll
      for (int u = 0; u < KC; u++) {
        const int k = k0 - u;
        if (k < 0) break;
        qn = (C)qq[u] - (C)cc[u] * qn;
        zq[col + plane * k] = (T)qn;
      }
    }
    cag[col] = ag;
    cden[col] = (C)1 + qn + ag * qlast;
  }
}

// a + c + b rounded once, for a + c and -b of like size
__device__ __forceinline__ double sum3(double a, double c, double b)
{
  const double t = a + c, tz = t - a, tl = (a - (t - tz)) + (c - tz);  // (two-sums)
  const double r = b + t, rz = r - b, rl = (b - (r - rz)) + (t - rz);
  return r + (rl + tl);
}

// The same with the columns cut into segments, as k_zline_seg: NC consecutive
// columns a block, SG segments of P planes each, a thread a segment, whose rows
// stay in registers.  The pivots d_k = b_k - a_k c_(k-1) / d_(k-1) are formed
// without subtractions (Grassmann, Taksar and Heyman, "Regenerative analysis
// and steady state distributions for Markov chains", 1985), from the rows'
// excess e_k = -(a_k + b_k + c_k): -d_k = c_k + E_k, E_k = e_k + a_k E_(k-1) /
// -d_(k-1).  That is a fractional linear recurrence of E_k / -d_k: a thread
// composes the 2x2 maps of its planes (rows scaled by 1/b, so that the products
// stay between 0 and 1 in size; no entry negative where a, c and e are not), runs
// through the maps before it as a vector (num, den), and takes its planes one
// after another.  The relative error of a pivot is 1.6e-16 (geometric mean of
// the largest of a column) whatever the length and the contrast; the column
// walk's is 3e-16 (50 planes, 6 % noise) to 2e-15 (200, contrasts of 200), and
// maps of b_k - a_k cp_(k-1) itself, whose products cancel, would have 2e-15 to
// 3e-14.  The Sherman-Morrison vector and its back sweep are
// first-order linear recurrences treated alike.  us, one thread a column (bound by
// the serial chain of divisions and the few blocks) -> segments: 32^3 FP64 31 ->
// 6.5, 64^3 FP64 61 -> 11.4 and FP32 58 -> 10.8, 128^3 FP64 122 -> 29 and FP32
// 112 -> 27, 128 x 128 x 256 FP64 241 -> 71, 256^3 FP64 317 -> 296 and FP32 260 ->
// 187 (the stores of the four factors); factors alone, 64 x 48 x 40 FP64 34 -> 7.8,
// 96 x 80 x 50 FP32 41 -> 8.3.  More than 8 planes a thread spill; beyond 128
// planes 32 columns a block (239 us with 16 at 256^3 FP32), below 16 (29 and 34
// us at 128^3 FP64).  Columns beyond 256 planes keep the walk.
template <typename T, int NC, int SG, int P, bool COEF, bool FACT>
__global__ __launch_bounds__(NC * SG) void k_zcolumn_seg(Grid g, SCoef s, const T *__restrict__ n, T *__restrict__ Cz,
                                                         T *__restrict__ za, T *__restrict__ zi, T *__restrict__ zc,
                                                         T *__restrict__ zq, double *__restrict__ cag,
                                                         double *__restrict__ cden)
{
  constexpr int kMaps = FACT ? 4 : 0, kSums = COEF ? 9 : 0;
  __shared__ double sh[kMaps > kSums ? kMaps : kSums][SG][NC], ends[4][NC];
  uint32_t bx, by, bz;
  (void)xcd_tile(bx, by, bz);
  const int plane = g.nx * g.ny, m = g.nz, cx = threadIdx.x % NC, sg = threadIdx.x / NC, k0 = sg * P;
  const int col = (int)bx * NC + cx;
  const bool live = col < plane;
  int i, j, k_;
  split_cell(g, live ? col : 0, i, j, k_);
  const int c0 = i + g.nx * j;
  const int oxp = (i + 1 == g.nx ? 0 : i + 1) + g.nx * j, oxm = (i == 0 ? g.nx - 1 : i - 1) + g.nx * j;
  const int oyp = i + g.nx * (j + 1 == g.ny ? 0 : j + 1), oym = i + g.nx * (j == 0 ? g.ny - 1 : j - 1);
  // rows of the thread's planes (loads past the last plane read a valid value that is not used)
  double a[P], b[P], c[P];
  double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  {
    T nz_[P + 2], xp[P], xm[P], yp[P], ym[P];
#pragma unroll
    for (int u = 0; u < P + 2; u++) nz_[u] = n[c0 + (int64_t)plane * wrapi(k0 - 1 + u < m + 1 ? k0 - 1 + u : m, m)];
#pragma unroll
    for (int u = 0; u < P; u++) {
      const int64_t pk = (int64_t)plane * (k0 + u < m ? k0 + u : m - 1);
      xp[u] = n[oxp + pk]; xm[u] = n[oxm + pk]; yp[u] = n[oyp + pk]; ym[u] = n[oym + pk];
    }
#pragma unroll
    for (int u = 0; u < P; u++) {
      double v[19];
      row_from_star<double>(s, (double)nz_[u + 1], (double)xp[u], (double)xm[u], (double)yp[u], (double)ym[u],
                            (double)nz_[u + 2], (double)nz_[u], v);
      a[u] = v[5]; b[u] = v[18]; c[u] = v[4];
      if (COEF && k0 + u < m) {
        constexpr int grp[19] = {5, 3, 7, 1, 4, 4, 8, 2, 6, 0, 5, 5, 3, 3, 7, 7, 1, 1, 4};  // kGroup19
#pragma unroll
        for (int q = 0; q < 19; q++) acc[grp[q]] += v[q];
      }
    }
  }
  if (COEF) {
#pragma unroll
    for (int q = 0; q < 9; q++) sh[q][sg][cx] = acc[q];
    __syncthreads();
    for (int e = threadIdx.x; e < 9 * NC; e += NC * SG) {
      const int q = e / NC, cc = e % NC, cq = (int)bx * NC + cc;
      double t = 0.0;
#pragma unroll
      for (int r = 0; r < SG; r++) t += sh[q][r][cc];
      if (cq < plane) Cz[(int64_t)q * plane + cq] = (T)(t / (double)m);
    }
    __syncthreads();
  }
  if constexpr (FACT) {
    // the periodic corner: gamma = -b_0, b_0 -= gamma, b_(m-1) -= c_(m-1) a_0 / gamma
    if (sg == 0) { ends[0][cx] = a[0]; ends[1][cx] = b[0]; }
    __syncthreads();
    const double a0 = ends[0][cx], gm = -ends[1][cx];
    if (sg == 0) b[0] = b[0] - gm;
#pragma unroll
    for (int u = 0; u < P; u++)
      if (k0 + u == m - 1) b[u] = b[u] - c[u] * a0 / gm;
    // excess over the off-diagonals (in b's place from here), as the exact sum rounded
    double m00 = 1.0, m01 = 0.0, m10 = 0.0, m11 = 1.0;
#pragma unroll
    for (int u = 0; u < P; u++) {
      const double ib = -1.0 / b[u], ah = a[u] * ib, ch = c[u] * ib;
      b[u] = -sum3(a[u], c[u], b[u]);
      if (k0 + u < m) {
        const double eh = b[u] * ib;
        m00 = ah * m00 + eh * m10; m01 = ah * m01 + eh * m11;
        m10 = m00 + ch * m10; m11 = m01 + ch * m11;
      }
    }
    sh[0][sg][cx] = m00; sh[1][sg][cx] = m01; sh[2][sg][cx] = m10; sh[3][sg][cx] = m11;
    __syncthreads();
    double num = 1.0, den = 1.0;
    for (int t = 0; t < sg; t++) {
      const double x = sh[0][t][cx] * num + sh[1][t][cx] * den;
      den = sh[2][t][cx] * num + sh[3][t][cx] * den;
      num = x;
    }
    __syncthreads();  // (the maps are read)
    double ep = num / den, A = 1.0, B = 0.0, iv[P], q[P];
#pragma unroll
    for (int u = 0; u < P; u++) {
      iv[u] = 0.0;
      q[u] = 0.0;
      if (k0 + u < m) {
        const double ex = b[u] + a[u] * ep;
        iv[u] = -1.0 / (c[u] + ex);
        const double uk = k0 + u == 0 ? gm : (k0 + u == m - 1 ? c[u] : 0.0);
        ep = -ex * iv[u];
        c[u] = c[u] * iv[u];
        q[u] = uk * iv[u];
        const double al = -a[u] * iv[u];
        A = al * A;
        B = al * B + q[u];
      }
    }
    sh[0][sg][cx] = A;
    sh[1][sg][cx] = B;
    __syncthreads();
    double y = 0.0;
    for (int t = 0; t < sg; t++) y = sh[0][t][cx] * y + sh[1][t][cx];
#pragma unroll
    for (int u = 0; u < P; u++) {
      if (k0 + u < m) {
        y = q[u] - a[u] * iv[u] * y;
        q[u] = y;
      }
    }
    if (sg == (m - 1) / P) ends[2][cx] = y;
    // the back sweep x_(m-1) = q_(m-1), x_k = q_k - cp_k x_(k+1)
    A = 1.0; B = 0.0;
#pragma unroll
    for (int u = P - 1; u >= 0; u--) {
      if (k0 + u == m - 1) { A = 0.0; B = q[u]; }
      else if (k0 + u < m - 1) { B = q[u] - c[u] * B; A = -c[u] * A; }
    }
    sh[2][sg][cx] = A;
    sh[3][sg][cx] = B;
    __syncthreads();
    double x = 0.0;
    for (int t = SG - 1; t > sg; t--) x = sh[2][t][cx] * x + sh[3][t][cx];
#pragma unroll
    for (int u = P - 1; u >= 0; u--) {
      if (k0 + u < m) {
        x = k0 + u == m - 1 ? q[u] : q[u] - c[u] * x;
        q[u] = x;
      }
    }
    if (live) {
#pragma unroll
      for (int u = 0; u < P; u++) {
        if (k0 + u < m) {
          const int64_t e = col + (int64_t)plane * (k0 + u);
          za[e] = (T)a[u]; zi[e] = (T)iv[u]; zc[e] = (T)c[u]; zq[e] = (T)q[u];
        }
      }
      if (sg == 0) {
        const double ag = a0 / gm;
        cag[col] = ag;
        cden[col] = 1.0 + x + ag * ends[2][cx];
      }
    }
  }
}

// The segmented factors of the full operator on grid g where a block holds its
// columns; false: it does not.
template <typename T, bool COEF, bool FACT>
static bool launch_zcolumn_seg(chy_ctx *ctx, const Grid &g, const SCoef &s, const T *n, T *Cz, T *zbuf, double *colbuf)
{
  const int64_t nc = g.nc, plane = (int64_t)g.nx * g.ny;
  if (g.nz > 256) return false;
#define ZFAC(NC, SG, P)                                                                                                \
  hipLaunchKernelGGL((k_zcolumn_seg<T, NC, SG, P, COEF, FACT>), (unsigned)((plane + NC - 1) / NC), NC * SG, 0,         \
                     ctx->stream, g, s, n, Cz, zbuf, FACT ? zbuf + nc : zbuf, FACT ? zbuf + 2 * nc : zbuf,             \
                     FACT ? zbuf + 3 * nc : zbuf, colbuf, FACT ? colbuf + plane : colbuf)
  if (g.nz <= 32) ZFAC(16, 8, 4);
  else if (g.nz <= 64) ZFAC(16, 8, 8);
  else if (g.nz <= 128) ZFAC(16, 16, 8);
  else ZFAC(32, 32, 8);
#undef ZFAC
  return true;
}

template <typename T>
void launch_zcolumn(chy_ctx *ctx, const T *n, T *Cz, T *zbuf, double *colbuf)
{
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  const int64_t nc = ctx->g.nc, plane = (int64_t)ctx->g.nx * ctx->g.ny;
  const bool seg = Cz && zbuf ? launch_zcolumn_seg<T, true, true>(ctx, ctx->g, s, n, Cz, zbuf, colbuf)
                   : Cz       ? launch_zcolumn_seg<T, true, false>(ctx, ctx->g, s, n, Cz, zbuf, colbuf)
                   : zbuf     ? launch_zcolumn_seg<T, false, true>(ctx, ctx->g, s, n, Cz, zbuf, colbuf)
                              : true;
  if (seg) return;
  T *z4[4] = {zbuf, zbuf ? zbuf + nc : nullptr, zbuf ? zbuf + 2 * nc : nullptr, zbuf ? zbuf + 3 * nc : nullptr};
  double *c2[2] = {colbuf, colbuf ? colbuf + plane : nullptr};
#define ZCOL(A, B)                                                                                              \
  hipLaunchKernelGGL((k_zcolumn<T, A, B>), nblocks(plane), kBlock, 0, ctx->stream, ctx->g, s, n, Cz, z4[0], z4[1], \
                     z4[2], z4[3], c2[0], c2[1])
  if (Cz && zbuf) ZCOL(true, true);
  else if (Cz) ZCOL(true, false);
  else if (zbuf) ZCOL(false, true);
#undef ZCOL
}

template <typename T>
void launch_zline_factor(chy_ctx *ctx, int lhs_type, const T *n, T *zbuf, double *colbuf)
{
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  const LapRow L = lap_row(ctx, lhs_type);
  const int64_t nc = ctx->g.nc, plane = (int64_t)ctx->g.nx * ctx->g.ny;
  hipLaunchKernelGGL((k_zline_factor<T>), nblocks(plane), kBlock, 0, ctx->stream, ctx->g, lhs_type, s, L, n, zbuf,
                     zbuf + nc, zbuf + 2 * nc, zbuf + 3 * nc, colbuf, colbuf + plane);
}

template <typename T>
void launch_zline_apply(chy_ctx *ctx, const T *zbuf, const double *colbuf, T *res, T *z)
{
  launch_zline_apply_g<T>(ctx, ctx->g, zbuf, colbuf, res, z, 1.0);
}

// The segmented z-line stage where it is the faster one; false: it is not.
template <typename T, bool E2>
static bool launch_zline_seg(chy_ctx *ctx, const Grid &g, const T *zbuf, const double *colbuf, const T *res, T *z,
                             const T *n, const SCoef &s, const T *Z2, const double *y2, double scale)
{
  const int64_t nc = g.nc, plane = (int64_t)g.nx * g.ny;
  constexpr bool fp32 = sizeof(T) == 4;
  if (g.nz > 256 || (!fp32 && g.nz > 128 && nc > (int64_t)1 << 23)) return false;
#define ZSEG(NC, SG, P)                                                                                             \
  hipLaunchKernelGGL((k_zline_seg<T, NC, SG, P, E2>), (unsigned)((plane + NC - 1) / NC), NC * SG, 0, ctx->stream, g, \
                     zbuf, zbuf + nc, zbuf + 2 * nc, zbuf + 3 * nc, colbuf, colbuf + plane, res, z, n, s, Z2, y2, scale)
  if (g.nz <= 32) ZSEG(16, 8, 4);
  else if (g.nz <= 64) ZSEG(16, 8, 8);
  else if constexpr (fp32) {
    if (g.nz <= 128) ZSEG(32, 16, 8);
    else ZSEG(32, 16, 16);
  } else {
    if (g.nz <= 128) ZSEG(16, 16, 8);
    else ZSEG(16, 32, 8);
  }
#undef ZSEG
  return true;
}

template <typename T>
void launch_zline_apply_g(chy_ctx *ctx, const Grid &g, const T *zbuf, const double *colbuf, T *res, T *z,
                          double scale)
{
  const int64_t nc = g.nc, plane = (int64_t)g.nx * g.ny;
  if (launch_zline_seg<T, false>(ctx, g, zbuf, colbuf, res, z, nullptr, SCoef(), nullptr, nullptr, scale)) return;
  hipLaunchKernelGGL((k_zline_apply<T>), nblocks(plane), kBlock, 0, ctx->stream, g, zbuf, zbuf + nc,
                     zbuf + 2 * nc, zbuf + 3 * nc, colbuf, colbuf + plane, res, z, scale);
}

// fft2z's z-line stage with the 2-D correction folded in (k_zline_apply_e2):
// res holds d0 = r - A(n) z_fft on entry, Z2 the 2-D directions, y2 their
// coefficients.  Only for the full operator with B along z.
template <typename T>
void launch_zline_apply_e2(chy_ctx *ctx, const T *zbuf, const double *colbuf, T *res, T *z, const T *n, const T *Z2,
                           const double *y2)
{
  const Grid &g = ctx->g;
  const int64_t nc = g.nc, plane = (int64_t)g.nx * g.ny;
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  if (launch_zline_seg<T, true>(ctx, g, zbuf, colbuf, res, z, n, s, Z2, y2, 1.0)) return;
  hipLaunchKernelGGL((k_zline_apply_e2<T, kFft2Its>), nblocks(plane), kBlock, 0, ctx->stream, g, zbuf, zbuf + nc,
                     zbuf + 2 * nc, zbuf + 3 * nc, colbuf, colbuf + plane, res, z, n, s, Z2, y2);
}

bool zline_e2_applies(chy_ctx *ctx)
{
  return kz_operator(ctx->prm.lhs_type, full_scoef(ctx->prm.d, ctx->prm.kappa_e));
}

template <typename T>
void launch_zline_factor_g(chy_ctx *ctx, const Grid &g, const double d[3], int lhs_type, const T *n, T *zbuf,
                           double *colbuf)
{
  const SCoef s = full_scoef(d, ctx->prm.kappa_e);
  LapRow L;
  uniform_row(lhs_type == CHY_LHS_FULL ? CHY_LHS_IDENTITY : lhs_type, d, ctx->prm.kappa_e, 0.0, L.v);
  const int64_t nc = g.nc, plane = (int64_t)g.nx * g.ny;
  if (lhs_type == CHY_LHS_FULL && launch_zcolumn_seg<T, false, true>(ctx, g, s, n, nullptr, zbuf, colbuf)) return;
  hipLaunchKernelGGL((k_zline_factor<T>), nblocks(plane), kBlock, 0, ctx->stream, g, lhs_type, s, L, n, zbuf,
                     zbuf + nc, zbuf + 2 * nc, zbuf + 3 * nc, colbuf, colbuf + plane);
}

// res = b - A(n) x on grid g with spacings d, precision T (multigrid levels of
// columns beyond kMgMaxPlanes).  Where the column stencil does not take a grid, the
// tiles do also on small planes: a thread a node is level with them on thin ones
// and slower on others (twelve iterations, ms, tiles / nodes: FP64 36 x 4 x 20000
// 513 / 514, 16 x 16 x 36000 1936 / 1933, 64 x 64 x 600 55.2 / 57.0, 128 x 128 x
// 1000 129 / 149; mixed 461 / 461, 1786 / 1783, 41.5 / 41.7, 91.5 / 103)
template <typename T>
void launch_residual_g(chy_ctx *ctx, const Grid &g, const double d[3], int lhs_type, const T *n, const T *b,
                       const T *x, T *res)
{
  const SCoef s = full_scoef(d, ctx->prm.kappa_e);
  LapRow L;
  uniform_row(lhs_type == CHY_LHS_FULL ? CHY_LHS_IDENTITY : lhs_type, d, ctx->prm.kappa_e, 0.0, L.v);
  constexpr bool fp32 = sizeof(T) == 4;
  using C = typename std::conditional<fp32, float, double>::type;
  launch_tiled_on<T, T, T, C, fp32, 1, T>(ctx, g, s, L, lhs_type, n, x, b, res, (double *)nullptr);
}

// res = b - A(n) x in precision T
template <typename T>
void launch_residual_t(chy_ctx *ctx, int lhs_type, const T *n, const T *b, const T *x, T *res)
{
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  const LapRow L = lap_row(ctx, lhs_type);
  constexpr bool fp32 = sizeof(T) == 4;
  using C = typename std::conditional<fp32, float, double>::type;
  if constexpr (fp32) {
    if (wide_rows(ctx->g, fp32)) {
      launch_tiled<T, T, T, C, fp32, 1, T, 256>(ctx, lhs_type, n, x, b, res, (double *)nullptr);
      return;
    }
  }
  launch_tiled<T, T, T, C, fp32, 1, T>(ctx, lhs_type, n, x, b, res, (double *)nullptr);
}

template void launch_zcolumn<double>(chy_ctx *, const double *, double *, double *, double *);
template void launch_zcolumn<float>(chy_ctx *, const float *, float *, float *, double *);
template void launch_zline_factor<double>(chy_ctx *, int, const double *, double *, double *);
template void launch_zline_factor<float>(chy_ctx *, int, const float *, float *, double *);
template void launch_zline_apply_g<double>(chy_ctx *, const Grid &, const double *, const double *, double *,
                                           double *, double);
template void launch_zline_apply_g<float>(chy_ctx *, const Grid &, const float *, const double *, float *, float *,
                                          double);
template void launch_zline_factor_g<double>(chy_ctx *, const Grid &, const double *, int, const double *, double *,
                                            double *);
template void launch_zline_factor_g<float>(chy_ctx *, const Grid &, const double *, int, const float *, float *,
                                           double *);
template void launch_residual_g<double>(chy_ctx *, const Grid &, const double *, int, const double *, const double *,
                                        const double *, double *);
template void launch_residual_g<float>(chy_ctx *, const Grid &, const double *, int, const float *, const float *,
                                       const float *, float *);
template void launch_zline_apply<double>(chy_ctx *, const double *, const double *, double *, double *);
template void launch_zline_apply_e2<double>(chy_ctx *, const double *, const double *, double *, double *,
                                            const double *, const double *, const double *);
template void launch_zline_apply_e2<float>(chy_ctx *, const float *, const double *, float *, float *, const float *,
                                           const float *, const double *);
template void launch_zline_apply<float>(chy_ctx *, const float *, const double *, float *, float *);
template void launch_residual_t<double>(chy_ctx *, int, const double *, const double *, const double *, double *);
template void launch_residual_t<float>(chy_ctx *, int, const float *, const float *, const float *, float *);

// Chebyshev iteration on D^-1 A z = D^-1 r from z = 0 (three-term recurrence);
// the diagonal is rebuilt from n in each pass.
template <typename T>
__global__ __launch_bounds__(256) void k_cheby_init(Grid g, int lhs_type, SCoef s, LapRow lap, const T *__restrict__ n,
                                                    const T *__restrict__ r, T *__restrict__ res, T *__restrict__ dv,
                                                    T *__restrict__ z, double inv_theta)
{
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.nc) return;
  const int i = (int)(c % g.nx), j = (int)((c / g.nx) % g.ny), k = (int)(c / ((int64_t)g.nx * g.ny));
  double v[19];
  row_coeffs<double, T>(g, lhs_type, s, lap.v, n, i, j, k, v);
  const double rr = (double)r[c] / v[18];
  const double d = rr * inv_theta;
  res[c] = (T)rr; dv[c] = (T)d; z[c] = (T)d;
}

template <typename T>
__global__ __launch_bounds__(256) void k_cheby_step(Grid g, int lhs_type, SCoef s, LapRow lap, const T *__restrict__ n,
                                                    const T *__restrict__ Ad, T *__restrict__ res, T *__restrict__ dv,
                                                    T *__restrict__ z, double c1, double c2)
{
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.nc) return;
  const int i = (int)(c % g.nx), j = (int)((c / g.nx) % g.ny), k = (int)(c / ((int64_t)g.nx * g.ny));
  double v[19];
  row_coeffs<double, T>(g, lhs_type, s, lap.v, n, i, j, k, v);
  const double rr = (double)res[c] - (double)Ad[c] / v[18];
  const double d = c1 * (double)dv[c] + c2 * rr;
  res[c] = (T)rr; dv[c] = (T)d; z[c] = (T)((double)z[c] + d);
}

template <typename T>
void launch_cheby(chy_ctx *ctx, int lhs_type, bool transpose, int degree, const T *n, const T *r, T *z, T *res,
                  T *dv, T *Ad)
{
  const SCoef s = full_scoef(ctx->prm.d, ctx->prm.kappa_e);
  const LapRow L = lap_row(ctx, lhs_type);
  const double lo = 0.2, hi = 2.2, theta = 0.5 * (hi + lo), delta = 0.5 * (hi - lo), sigma = theta / delta;
  const unsigned nb = nblocks(ctx->g.nc);
  hipLaunchKernelGGL((k_cheby_init<T>), nb, kBlock, 0, ctx->stream, ctx->g, lhs_type, s, L, n, r, res, dv, z,
                     1.0 / theta);
  double rho = 1.0 / sigma;
  for (int k = 1; k < degree; k++) {
    launch_lhs_apply<T, T, T>(ctx, lhs_type, transpose, n, dv, Ad);
    const double rho1 = 1.0 / (2.0 * sigma - rho);
    hipLaunchKernelGGL((k_cheby_step<T>), nb, kBlock, 0, ctx->stream, ctx->g, lhs_type, s, L, n, Ad, res, dv, z,
                       rho1 * rho, 2.0 * rho1 / delta);
    rho = rho1;
  }
}

// explicit instantiations
template void launch_lhs_apply<double, double, double>(chy_ctx *, int, bool, const double *, const double *, double *);
template void launch_lhs_apply<float, float, float>(chy_ctx *, int, bool, const float *, const float *, float *);
template void launch_lhs_apply<float, double, double>(chy_ctx *, int, bool, const float *, const double *, double *);
template void launch_lhs_zsum<double>(chy_ctx *, int, const double *, const double *, const double *, double *,
                                      double *, double *);
template void launch_lhs_zsum<float>(chy_ctx *, int, const float *, const float *, const float *, double *, double *,
                                     float *);
template void launch_residual<double, double>(chy_ctx *, int, const double *, const double *, const double *, double *);
template void launch_residual<float, double>(chy_ctx *, int, const float *, const double *, const double *, double *);
template void launch_residual_norm<double, double>(chy_ctx *, int, const double *, const double *, const double *,
                                                   double *, double *);
template void launch_residual_norm<float, float>(chy_ctx *, int, const float *, const double *, const double *, float *,
                                                 double *);
template int64_t launch_residual_sq<double>(chy_ctx *, int, const double *, const double *, const double *, double *,
                                            double *);
template int64_t launch_residual_sq<float>(chy_ctx *, int, const float *, const float *, const float *, float *,
                                           double *);
template void launch_add_scaled<double>(chy_ctx *, int64_t, const double *, double, double *);
template void launch_add_scaled<float>(chy_ctx *, int64_t, const float *, double, double *);
template void launch_zcoef<double>(chy_ctx *, int, const double *, double *);
template void launch_zcoef<float>(chy_ctx *, int, const float *, float *);
template void launch_zline<double>(chy_ctx *, int, const double *, const double *, double *, double *, double *);
template void launch_zline<float>(chy_ctx *, int, const float *, const float *, float *, float *, float *);
template void launch_cheby<double>(chy_ctx *, int, bool, int, const double *, const double *, double *, double *,
                                   double *, double *);
template void launch_cheby<float>(chy_ctx *, int, bool, int, const float *, const float *, float *, float *, float *,
                                  float *);
template void launch_efield<double>(chy_ctx *, const double *, double *);
template void launch_efield<float>(chy_ctx *, const double *, float *);
template void launch_rhs<double>(chy_ctx *, int, const double *, const double *, const double *, const double *, double *);
template void launch_rhs<float>(chy_ctx *, int, const float *, const float *, const float *, const float *, double *);
template void launch_mdot<double>(chy_ctx *, int, const double *, int64_t, const double *, int64_t, double *,
                                  const double *);
template void launch_mdot<float>(chy_ctx *, int, const float *, int64_t, const float *, int64_t, double *,
                                 const double *);
template void launch_sum<double>(chy_ctx *, const double *, int64_t, double *);
template void launch_sum<float>(chy_ctx *, const float *, int64_t, double *);
template void launch_mgs_update<double>(chy_ctx *, int, const double *, int64_t, const double *, double *, int64_t);
template void launch_mgs_update<float>(chy_ctx *, int, const float *, int64_t, const double *, float *, int64_t);
template void launch_mgs_update_host<double>(chy_ctx *, int, const double *, int64_t, const double *, double *,
                                             int64_t);
template void launch_mgs_update_host<float>(chy_ctx *, int, const float *, int64_t, const double *, float *, int64_t);
template void launch_mgs_norm<double>(chy_ctx *, int, const double *, int64_t, const double *, double *, int64_t, double *);
template void launch_mgs_norm<float>(chy_ctx *, int, const float *, int64_t, const double *, float *, int64_t, double *);
template void launch_gs_dots<double>(chy_ctx *, int, const double *, int64_t, const double *, int64_t, double *,
                                     const double *);
template void launch_gs_dots<float>(chy_ctx *, int, const float *, int64_t, const float *, int64_t, double *,
                                    const double *);
template void launch_gs_update_dots<double>(chy_ctx *, int, const double *, int64_t, const double *, double *, int64_t,
                                            double *, const double *);
template void launch_gs_update_dots<float>(chy_ctx *, int, const float *, int64_t, const double *, float *, int64_t,
                                           double *, const double *);
template void launch_gs_update_norm<double>(chy_ctx *, int, const double *, int64_t, const double *, double *, int64_t,
                                            double *);
template void launch_gs_update_norm<float>(chy_ctx *, int, const float *, int64_t, const double *, float *, int64_t,
                                           double *);
template void launch_axpby<double>(chy_ctx *, int64_t, double, const double *, double, double *);
template void launch_axpby<float>(chy_ctx *, int64_t, double, const float *, double, float *);
template void launch_convert<double, float>(chy_ctx *, int64_t, const double *, double, float *);
template void launch_convert<float, double>(chy_ctx *, int64_t, const float *, double, double *);
template void launch_convert<double, double>(chy_ctx *, int64_t, const double *, double, double *);
template void launch_convert<float, float>(chy_ctx *, int64_t, const float *, double, float *);
template void launch_shift<double>(chy_ctx *, int64_t, double *, const double *, double);
template void launch_shift<float>(chy_ctx *, int64_t, float *, const double *, double);
template void launch_fill<double>(chy_ctx *, int64_t, double *, double);
template void launch_fill<float>(chy_ctx *, int64_t, float *, float);
template void launch_fill<uint32_t>(chy_ctx *, int64_t, uint32_t *, uint32_t);
template void launch_fill<unsigned long long>(chy_ctx *, int64_t, unsigned long long *, unsigned long long);
template void launch_jacobi<double>(chy_ctx *, int, const double *, const double *, double *);
template void launch_jacobi<float>(chy_ctx *, int, const float *, const float *, float *);

}  // namespace chy
