// chy_device.h -- device-side helpers shared by the gfx950 kernels:
// counter-based RNG, periodic cell arithmetic, CIC corner weights and the
// closed-form mean relative speed used to normalise collision probabilities.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace chy {

// Grid descriptor passed by value to kernels.  Nodes are periodic and
// node-centred: node (i,j,k) at p0 + (i,j,k)*d, linear c = i + nx*(j + ny*k).
struct Grid {
  int nx, ny, nz;
  int64_t nc;
  double p0[3], p1[3], d[3], L[3];
  double rd[3];  // 1 / d, rounded to nearest (div_rn)
  // ceil(2^64 / nx) and ceil(2^64 / ny): q = mulhi64(m, c) is c / n exactly for
  // every 32-bit c and n >= 2 (Lemire, Kaser and Kurz, "Faster remainder by
  // direct computation", 2019)
  uint64_t mx, my;
};

inline uint64_t fastdiv_magic(uint32_t n) { return ~0ull / n + 1; }

// cell -> (i, j, k) without runtime integer division
__device__ __forceinline__ void split_cell(const Grid &g, int c, int &i, int &j, int &k)
{
  const uint32_t q = (uint32_t)__umul64hi(g.mx, (uint64_t)(uint32_t)c);
  i = c - (int)q * g.nx;
  const uint32_t r = (uint32_t)__umul64hi(g.my, (uint64_t)q);
  j = (int)q - (int)r * g.ny;
  k = (int)r;
}

__device__ __forceinline__ int wrapi(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// Logical tile of this workgroup in a 3-D launch.  Workgroups are dealt to the
// 8 XCDs round-robin in linear order (x fastest); relabelling them so that XCD
// q takes the q-th contiguous eighth of the tiles keeps a tile's y and z
// neighbours, whose halo rows it reads, in the same L2.  Returns the logical
// linear index; (tx, ty, tz) are its coordinates.
__device__ __forceinline__ uint32_t xcd_tile(uint32_t &tx, uint32_t &ty, uint32_t &tz)
{
  const uint32_t gx = gridDim.x, gy = gridDim.y, nb = gx * gy * gridDim.z;
  uint32_t b = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
  if ((nb & 7u) == 0) b = (b & 7u) * (nb >> 3) + (b >> 3);
  const uint32_t p = b / gx;
  tx = b - p * gx;
  ty = p % gy;
  tz = p / gy;
  return b;
}

__device__ __forceinline__ int64_t lin(const Grid &g, int i, int j, int k)
{
  return (int64_t)wrapi(i, g.nx) + (int64_t)g.nx * ((int64_t)wrapi(j, g.ny) + (int64_t)g.ny * wrapi(k, g.nz));
}

// ---- Philox4x32-10 (Salmon et al., SC'11) ------------------------------------
struct U4 { uint32_t x, y, z, w; };

__device__ __forceinline__ U4 philox4x32_10(U4 c, uint32_t k0, uint32_t k1)
{
#pragma unroll
  for (int r = 0; r < 10; r++) {
    if (r > 0) { k0 += 0x9E3779B9u; k1 += 0xBB67AE85u; }
    const uint64_t p0 = (uint64_t)0xD2511F53u * c.x;
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c.z;
    U4 n;
    n.x = (uint32_t)(p1 >> 32) ^ c.y ^ k0;
    n.y = (uint32_t)p1;
    n.z = (uint32_t)(p0 >> 32) ^ c.w ^ k1;
    n.w = (uint32_t)p0;
    c = n;
  }
  return c;
}

// 24-bit uniform in (0,1), exactly representable in FP32 and FP64.
template <typename T>
__device__ __forceinline__ T u24(uint32_t w) { return ((T)(w >> 8) + (T)0.5) * (T)(1.0 / 16777216.0); }

// RNG streams: counter = {id, step, stream, block}, key = seed.
enum : uint32_t { STREAM_INIT = 0, STREAM_COLLIDE_A = 1, STREAM_COLLIDE_B = 2, STREAM_WEIGHT = 3 };

// ---- FP64 arithmetic of the ions ------------------------------------------------
// The FP64 ion kernels are bound by instruction issue: the push of an ion
// issued 2154 vector instructions, most of them in the library's division,
// square root, logarithm, sine and cosine, which take any argument.  These take
// the arguments that occur.

// a / d rounded to nearest, rd = 1 / d rounded to nearest: a quotient within an
// ulp corrected by its exact remainder (Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", 1990); 5 instructions
// against 12.  Finite operands, no over- or underflow.
__host__ __device__ __forceinline__ double div_rn(double a, double d, double rd)
{
  double q = a * rd;
  q = __builtin_fma(__builtin_fma(-q, d, a), rd, q);
  return __builtin_fma(__builtin_fma(-q, d, a), rd, q);
}

// The hardware's approximations of 1 / x and 1 / sqrt(x); on the host, where the
// functions below are tested, the values moved by 2^-24 of themselves
__host__ __device__ __forceinline__ double rcp_approx(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rcp(x);
#else
  return (1.0 + 0x1p-24) / x;
#endif
}

__host__ __device__ __forceinline__ double rsq_approx(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rsq(x);
#else
  return (1.0 + 0x1p-24) / __builtin_sqrt(x);
#endif
}

// a / b for normal b (not 0) whose quotient neither over- nor underflows: two
// Newton-Raphson steps y += y (1 - b y) on the hardware's reciprocal, and the
// quotient a y corrected by its exact remainder, as in div_rn (the last bit may
// differ from a / b's where that is a near tie)
__host__ __device__ __forceinline__ double div_normal(double a, double b)
{
  double y = rcp_approx(b);
  y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
  y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
  const double q = a * y;
  return __builtin_fma(__builtin_fma(-q, b, a), y, q);
}

// sin and cos of fl(2 pi u) for 0 <= u <= 1 (the rounded product, as cos(2.0 * M_PI
// * u) takes it): 4 u = k + f, |f| <= 1/2, exactly, the Taylor series of sin and
// cos(pi f / 2) with their leading terms in two parts, and the derivative times
// what the rounding of the angle left, dl.  Rounded to nearest but for 1.2 % of
// the arguments (off by an ulp); one call of about 50 instructions for both,
// against 80 for each of the library's.  A scattering whose relative velocity is
// nearly axial amplifies an ulp of its neutral's velocity by up to 1e6, so two
// implementations agree there only as far as their roundings coincide.
__host__ __device__ __forceinline__ void sincos2pi(double u, double &s, double &c)
{
  const double t = 4.0 * u, k = __builtin_rint(t), f = t - k, z = f * f, zl = __builtin_fma(f, f, -z);
  const double angle = 6.283185307179586 * u;
  const double dl = -__builtin_fma(6.283185307179586, u, -angle) - 2.4492935982947064e-16 * u;
  const double p = 1.5707963267948966 * f;
  const double pl = __builtin_fma(6.123233995736766e-17, f, __builtin_fma(1.5707963267948966, f, -p));
  double a = __builtin_fma(6.0669357311061955e-12, z, -6.688035109811468e-10);
  a = __builtin_fma(a, z, 5.692172921967927e-08);
  a = __builtin_fma(a, z, -3.598843235212085e-06);
  a = __builtin_fma(a, z, 0.00016044118478735983);
  a = __builtin_fma(a, z, -0.004681754135318688);
  a = __builtin_fma(a, z, 0.07969262624616705);
  a = __builtin_fma(a, z, -0.6459640975062463);
  double b = __builtin_fma(-5.294400200734623e-13, z, 6.565963114979473e-11);
  b = __builtin_fma(b, z, -6.386603083791852e-09);
  b = __builtin_fma(b, z, 4.710874778818172e-07);
  b = __builtin_fma(b, z, -2.5202042373060607e-05);
  b = __builtin_fma(b, z, 0.0009192602748394266);
  b = __builtin_fma(b, z, -0.02086348076335296);
  b = __builtin_fma(b, z, 0.25366950790104803);
  const double g = a * z, sf = __builtin_fma(g, f, p);
  // cos: 1 - (pi^2/8) z in two parts, the rest of the series, and -dl sin
  const double hz = 1.2337005501361697 * z, w = 1.0 - hz;
  const double wl = ((1.0 - w) - hz) - __builtin_fma(1.2337005501361697, z, -hz);
  b = w + (wl + __builtin_fma(b * z, z, -__builtin_fma(1.2337005501361697, zl,
                                                        __builtin_fma(7.831619385924639e-17, z, dl * sf))));
  a = p + __builtin_fma(g, f, __builtin_fma(dl, b, pl));
  const int q = (int)k;
  const double sn = (q & 1) ? b : a, cn = (q & 1) ? a : b;
  s = (q & 2) ? -sn : sn;
  c = ((q + 1) & 2) ? -cn : cn;
}

// log(u) for normal u in (0, 1): u = 2^e m, m in [1/sqrt 2, sqrt 2), and with f =
// m - 1, s = f / (2 + f) = (m - 1) / (m + 1) the series log m = 2 atanh s = 2 s + s
// R, R = 2/3 s^2 + 2/5 s^4 + ... (Abramowitz and Stegun, 4.1.27; to s^18: below
// 3e-17 of the logarithm).  Its leading term is not exact: since s (2 + f) = f,
// with h = f^2 / 2, 2 s = f - s f = f - h + s h, whose large terms are.  log 2 is
// in two parts of which the first has few enough bits for e, and e log 2 + f - h
// in two parts: rounded to nearest but for 0.7 % of the arguments.
__host__ __device__ __forceinline__ double log_unit(double u)
{
  int e;
#if defined(__HIP_DEVICE_COMPILE__)
  double m = __builtin_amdgcn_frexp_mant(u);
  e = __builtin_amdgcn_frexp_exp(u);
#else
  double m = __builtin_frexp(u, &e);
#endif
  if (m < 0.70710678118654752440) { m *= 2.0; e -= 1; }
  const double f = m - 1.0, d = 2.0 + f;
  double y = rcp_approx(d);
  y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
  y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
  double s = f * y;
  s = __builtin_fma(__builtin_fma(-d, s, f), y, s);
  const double z = s * s;
  double R = 2.0 / 19.0;
  R = __builtin_fma(R, z, 2.0 / 17.0);
  R = __builtin_fma(R, z, 2.0 / 15.0);
  R = __builtin_fma(R, z, 2.0 / 13.0);
  R = __builtin_fma(R, z, 2.0 / 11.0);
  R = __builtin_fma(R, z, 2.0 / 9.0);
  R = __builtin_fma(R, z, 2.0 / 7.0);
  R = __builtin_fma(R, z, 2.0 / 5.0);
  R = __builtin_fma(R, z, 2.0 / 3.0);
  R = R * z;
  const double h = 0.5 * f * f, hl = __builtin_fma(0.5 * f, f, -h), ed = (double)e;
  const double l2 = ed * 0.6931467056274414;
  const double t1 = l2 + f, t1l = f - (t1 - l2), t2 = t1 - h, t2l = (t1 - t2) - h;
  return t2 + (t2l + (t1l + __builtin_fma(s, h + R, __builtin_fma(ed, 4.7493250390316726e-07, -hl))));
}

// sqrt(x) for normal positive x, 0 for all others, NaN among them (under the
// kinematics' roots rounding may leave a little less than 0; an ion's NaN is
// seen where its state is stored): Goldschmidt's coupled iteration for g = sqrt x
// and h = 1 / (2 sqrt x) from the hardware's reciprocal root, one step (Goldschmidt,
// "Applications of division by convergence", 1964), then g twice corrected by
// its exact remainder, g += h (x - g^2) (Markstein).
__host__ __device__ __forceinline__ double sqrt_normal(double x)
{
  const double y = rsq_approx(x);
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return x > 0.0 ? g : 0.0;
}

// ---- periodic cells ----------------------------------------------------------
// Cell of an absolute coordinate, clamped to [0, n-1]; f = fraction in cell.
__device__ __forceinline__ void cell_split(double xi, int n, int &i, double &f)
{
  int ii = (int)xi;
  if (ii > n - 1) ii = n - 1;
  if (ii < 0) ii = 0;
  i = ii;
  f = xi - (double)ii;
}

__device__ __forceinline__ void cell_coord(double x, double p0, double d, double rd, int n, int &i, double &f)
{
  cell_split(div_rn(x - p0, d, rd), n, i, f);
}

// Periodic wrap into [p0, p1); a coordinate more than one period away is
// first reduced with floor, non-finite values are returned unchanged.
__device__ __forceinline__ double wrap_pos(double x, double p0, double p1, double L)
{
  if (!(x >= p0 - L && x < p1 + L)) {
    if (!isfinite(x)) return x;
    x = x - floor((x - p0) / L) * L;
  }
  if (x < p0) {
    x += L;
    if (x >= p1) x = p0;
  } else if (x >= p1) {
    x -= L;
    if (x < p0) x = p0;
  }
  return x;
}

// a*b + c: one fused multiply-add in FP32 (the mixed path, compared with the
// oracle to a tolerance); in FP64 a separate multiply and add, rounded as the
// oracle rounds them (the build turns off FMA contraction).
__device__ __forceinline__ float fmad(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fmad(double a, double b, double c) { return a * b + c; }

// Corner weights W_q = (wz*wy)*wx for q = dx + 2 dy + 4 dz.
template <typename T>
__device__ __forceinline__ void corner_weights(T fx, T fy, T fz, T W[8])
{
  const T wx[2] = {(T)1 - fx, fx}, wy[2] = {(T)1 - fy, fy}, wz[2] = {(T)1 - fz, fz};
#pragma unroll
  for (int q = 0; q < 8; q++) W[q] = (wz[q >> 2] * wy[(q >> 1) & 1]) * wx[q & 1];
}

// E|v - v_n| for v_n ~ N(vn0, vnT^2 I): mean of a non-central chi-3 variable,
// sigma [sqrt(2/pi) e^{-l^2/2} + (l + 1/l) erf(l/sqrt 2)], l = |v - vn0|/sigma.
__device__ __forceinline__ double mean_rel_speed(double vx, double vy, double vz,
                                                 double n0x, double n0y, double n0z, double vnT)
{
  const double ux = vx - n0x, uy = vy - n0y, uz = vz - n0z;
  const double mu = sqrt(ux * ux + uy * uy + uz * uz);
  if (!(vnT > 0.0)) return mu;
  const double lam = mu / vnT;
  const double c = 0.79788456080286535588;
  if (lam < 1e-3) return vnT * c * (2.0 + lam * lam / 3.0);
  return vnT * (c * exp(-0.5 * lam * lam) + (lam + 1.0 / lam) * erf(lam * 0.70710678118654752440));
}

__device__ __forceinline__ float mean_rel_speed_f(float vx, float vy, float vz, float n0x, float n0y, float n0z,
                                                  float vnT)
{
  const float ux = vx - n0x, uy = vy - n0y, uz = vz - n0z;
  const float mu = sqrtf(ux * ux + uy * uy + uz * uz);
  if (!(vnT > 0.f)) return mu;
  const float lam = mu / vnT;
  const float c = 0.79788456080286535588f;
  if (lam < 1e-2f) return vnT * c * (2.0f + lam * lam / 3.0f);
  return vnT * (c * expf(-0.5f * lam * lam) + (lam + 1.0f / lam) * erff(lam * 0.70710678118654752440f));
}

// ---- wave-level helpers (64-wide wavefronts) -----------------------------------
__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & 63); }

// Orders a wave's own LDS accesses (which the hardware keeps in order)
__device__ __forceinline__ void wave_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// x of the lane that CTRL (a DPP control) names, other where there is none in
// the row of 16 lanes (or, for a shift of the whole wave, in the wave)
template <int CTRL>
__device__ __forceinline__ double dpp_move(double x, double other)
{
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(other), __double2loint(x), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(other), __double2hiint(x), CTRL, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double lane_value(double x, int l)  // l: the same in every lane
{
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), l),
                          __builtin_amdgcn_readlane(__double2loint(x), l));
}

// Sum over the wave's 64 lanes (all active), the same in every lane
__device__ __forceinline__ double wave_total(double x)
{
  x += dpp_move<0x111>(x, 0.0);  // row_shr:1, 2, 4, 8: lane 15 of a row has its sum
  x += dpp_move<0x112>(x, 0.0);
  x += dpp_move<0x114>(x, 0.0);
  x += dpp_move<0x118>(x, 0.0);
  return (lane_value(x, 15) + lane_value(x, 31)) + (lane_value(x, 47) + lane_value(x, 63));
}

// Run-length aggregation of integer atomics over lanes holding equal keys in
// consecutive lanes: returns, for each active lane, (head lane, run length).
// Inactive lanes must pass key = -1.
__device__ __forceinline__ void key_runs(int key, int &head, int &len)
{
  const int l = lane_id();
  const int prev = __shfl_up(key, 1, 64);
  const bool is_head = (l == 0) || (prev != key);
  const uint64_t heads = __ballot(is_head);
  // head of my run: highest set bit at or below l
  const uint64_t below = heads & ((l == 63) ? ~0ull : ((2ull << l) - 1));
  head = 63 - __clzll(below);
  const uint64_t above = heads & ~((l == 63) ? ~0ull : ((2ull << l) - 1));
  const int next = above ? __ffsll((unsigned long long)above) - 1 : 64;
  len = next - head;
}

}  // namespace chy
