// chy_fft.hip -- FFT preconditioner for the periodic 19-point operator.
//
// P = A(nbar), the operator of the mean density, is a constant-coefficient
// periodic stencil with a_o = a_{-o}, hence diagonalised by the 3-D DFT with
// real symbol lam(k) = sum_o a_o cos(k.o).  z = P^+ r is computed as
// IFFT(FFT(r) / lam) with the k = 0 mode removed (the operator's constant
// null space).  All passes are LDS-resident batched radix-4 transforms:
// forward passes use decimation in frequency (natural in, bit-reversed out)
// and inverse passes decimation in time (bit-reversed in, natural out), so
// no permutation pass is needed; the z pass fuses forward FFT, the symbol
// division and the inverse FFT.  The x pass is real-to-complex (half
// spectrum, nx/2 complex values per line), so every pass moves as many bytes
// as the real field: x-fwd, y-fwd, z-fwd/scale/z-inv, y-inv, x-inv.  Grid
// sizes: powers of two.  Axes of 16 to 512 points (256 in FP64) take
// register-resident four-step transforms instead.
#include <algorithm>
#include <cmath>

#include "chy_internal.h"

namespace chy {

template <typename T> struct cpx { T x, y; };

template <typename T>
__device__ __forceinline__ cpx<T> cmul(cpx<T> a, cpx<T> b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }

__device__ __forceinline__ int bitrev(int v, int logn) { return (int)(__brev((unsigned)v) >> (32 - logn)); }

constexpr int kFftMaxN = 2048;  // longest axis handled by one LDS-resident line
constexpr int kU = 8;           // global loads batched per thread before their LDS stores

// Lines per block: the largest power of two whose padded LDS footprint
// B*(n+1) complex values stays within 64 KB, and at most `avail`.
template <typename T>
static int fft_batch(int n, int64_t avail)
{
  const int64_t E = 65536 / (int64_t)(2 * sizeof(T)) - n / 2;  // twiddles share the LDS
  int B = 1;
  while ((int64_t)(2 * B) * (n + 1) <= E && 2 * B <= avail) B *= 2;
  return B;
}

template <typename T>
static size_t fft_lds(int n, int B) { return ((size_t)B * (n + 1) + (size_t)n / 2) * 2 * sizeof(T); }

// The z pass also stages 3 doubles per line and the z table (2n doubles).
template <typename T>
static size_t fft_lds_z(int n, int B) { return fft_lds<T>(n, B) + (3 * (size_t)B + 2 * (size_t)n) * sizeof(double); }

template <typename T>
static int fft_batch_z(int n, int64_t avail)
{
  int B = fft_batch<T>(n, avail);
  while (B > 1 && fft_lds_z<T>(n, B) > 65536) B >>= 1;
  return B;
}

// One batch of B lines in LDS: s[b*(n+1) + t] (padded rows).  Twiddles
// w[j] = exp(-2 pi i j / n), j < n/2, are staged in LDS (tw).  Butterfly
// indices use shifts and masks (n is a power of two).

// Forward, decimation in frequency (natural order in, bit-reversed out):
// radix-4 stages (two radix-2 stages fused), then a final radix-2 stage when
// log2 n is odd.
template <typename T>
__device__ __forceinline__ void dif_fwd(cpx<T> *s, int B, int logn, const cpx<T> *tw, int tsh = 0)
{
  const int n = 1 << logn;
  int lg = logn;
  for (; lg >= 2; lg -= 2) {
    const int len = 1 << lg, lq = lg - 2, q = 1 << lq, step = n >> lg;
    const int nb4 = B << (logn - 2);
    for (int m = threadIdx.x; m < nb4; m += blockDim.x) {
      const int b = m >> (logn - 2), r = m & ((n >> 2) - 1);
      const int grp = r >> lq, k = r & (q - 1);
      const int i0 = b * (n + 1) + grp * len + k;
      const cpx<T> x0 = s[i0], x1 = s[i0 + q], x2 = s[i0 + 2 * q], x3 = s[i0 + 3 * q];
      const cpx<T> w1 = tw[(k * step) << tsh], w2 = tw[(2 * k * step) << tsh];
      const cpx<T> a0 = {x0.x + x2.x, x0.y + x2.y};
      const cpx<T> a1 = {x1.x + x3.x, x1.y + x3.y};
      const cpx<T> d02 = {x0.x - x2.x, x0.y - x2.y};
      const cpx<T> d13 = {x1.x - x3.x, x1.y - x3.y};
      const cpx<T> a2 = cmul<T>(d02, w1);
      const cpx<T> a3 = cmul<T>({d13.y, -d13.x}, w1);  // (x1 - x3) W^k (-i)
      s[i0] = {a0.x + a1.x, a0.y + a1.y};
      s[i0 + q] = cmul<T>({a0.x - a1.x, a0.y - a1.y}, w2);
      s[i0 + 2 * q] = {a2.x + a3.x, a2.y + a3.y};
      s[i0 + 3 * q] = cmul<T>({a2.x - a3.x, a2.y - a3.y}, w2);
    }
    __syncthreads();
  }
  if (lg == 1) {
    const int nb2 = B << (logn - 1);
    for (int m = threadIdx.x; m < nb2; m += blockDim.x) {
      const int b = m >> (logn - 1), r = m & ((n >> 1) - 1);
      const int i0 = b * (n + 1) + 2 * r;
      const cpx<T> u = s[i0], v = s[i0 + 1];
      s[i0] = {u.x + v.x, u.y + v.y};
      s[i0 + 1] = {u.x - v.x, u.y - v.y};
    }
    __syncthreads();
  }
}

// Inverse, decimation in time (bit-reversed in, natural order out, unscaled):
// a radix-2 first stage when log2 n is odd, then radix-4 stages.
template <typename T>
__device__ __forceinline__ void dit_inv(cpx<T> *s, int B, int logn, const cpx<T> *tw, int tsh = 0)
{
  const int n = 1 << logn;
  int lg = 0;
  if (logn & 1) {
    const int nb2 = B << (logn - 1);
    for (int m = threadIdx.x; m < nb2; m += blockDim.x) {
      const int b = m >> (logn - 1), r = m & ((n >> 1) - 1);
      const int i0 = b * (n + 1) + 2 * r;
      const cpx<T> u = s[i0], v = s[i0 + 1];
      s[i0] = {u.x + v.x, u.y + v.y};
      s[i0 + 1] = {u.x - v.x, u.y - v.y};
    }
    __syncthreads();
    lg = 1;
  }
  for (; lg + 2 <= logn; lg += 2) {
    const int len = 1 << (lg + 2), lq = lg, q = 1 << lq, step = n >> (lg + 2);
    const int nb4 = B << (logn - 2);
    for (int m = threadIdx.x; m < nb4; m += blockDim.x) {
      const int b = m >> (logn - 2), r = m & ((n >> 2) - 1);
      const int grp = r >> lq, k = r & (q - 1);
      const int i0 = b * (n + 1) + grp * len + k;
      const cpx<T> x0 = s[i0], x1 = s[i0 + q], x2 = s[i0 + 2 * q], x3 = s[i0 + 3 * q];
      const cpx<T> t1 = tw[(k * step) << tsh], t2 = tw[(2 * k * step) << tsh];
      const cpx<T> W = {t1.x, -t1.y}, V = {t2.x, -t2.y};  // conjugates: +2 pi i
      const cpx<T> v1 = cmul<T>(x1, V), v3 = cmul<T>(x3, V);
      const cpx<T> a0 = {x0.x + v1.x, x0.y + v1.y}, a1 = {x0.x - v1.x, x0.y - v1.y};
      const cpx<T> a2 = {x2.x + v3.x, x2.y + v3.y}, a3 = {x2.x - v3.x, x2.y - v3.y};
      const cpx<T> b2 = cmul<T>(a2, W);
      const cpx<T> wa3 = cmul<T>(a3, W);
      const cpx<T> b3 = {-wa3.y, wa3.x};  // a3 W^k (+i)
      s[i0] = {a0.x + b2.x, a0.y + b2.y};
      s[i0 + 2 * q] = {a0.x - b2.x, a0.y - b2.y};
      s[i0 + q] = {a1.x + b3.x, a1.y + b3.y};
      s[i0 + 3 * q] = {a1.x - b3.x, a1.y - b3.y};
    }
    __syncthreads();
  }
}

template <typename T>
__device__ __forceinline__ void load_twiddles(cpx<T> *tws, const double *tw, int n)
{
  for (int j = threadIdx.x; j < (n >> 1); j += blockDim.x) tws[j] = {(T)tw[2 * j], (T)tw[2 * j + 1]};
}

// Pass along x (contiguous real lines of length n = 2h) as half-length
// complex transforms.  MODE 0 (forward): z_t = r_2t + i r_2t+1, Z = FFT_h(z),
// then X_k = E_k + W_n^k O_k with E_k = (Z_k + conj Z_h-k)/2,
// O_k = (Z_k - conj Z_h-k)/(2i), written for k < h in natural order; X_0 and
// X_h are real and share slot 0 as X_0 + i X_h.  MODE 1 (inverse): the exact
// reverse (E_k = X_k + conj X_h-k, O_k = (X_k - conj X_h-k) W_n^-k,
// Z = E + i O, z = IFFT_h(Z), r_2t + i r_2t+1 = z_t), which returns n times the
// input like an unscaled length-n inverse; the real result is multiplied by
// `scale`.  LDS: twiddles W_n^j (j < h; the half-length FFT uses every other
// one) and B padded lines of h + 1 complex values.
template <typename T>
static int rfft_batch(int h, int64_t avail)
{
  const int64_t E = 65536 / (int64_t)(2 * sizeof(T)) - h;
  int B = 1;
  while ((int64_t)(2 * B) * (h + 1) <= E && 2 * B <= avail) B *= 2;
  return B;
}

template <typename T>
static size_t rfft_lds(int h, int B) { return ((size_t)B * (h + 1) + (size_t)h) * 2 * sizeof(T); }

template <typename T, int MODE>
__global__ __launch_bounds__(256) void k_rfft_x(int logn, int nlines, int B, const T *__restrict__ rin,
                                                cpx<T> *__restrict__ buf, T *__restrict__ rout,
                                                const double *__restrict__ tw, double scale, int ly, int64_t plane)
{
  // half spectrum of line l = iy + ny*iz at iy*h + iz*plane
  auto at = [&](int64_t l) { return (l & ((1 << ly) - 1)) * (int64_t)(1 << (logn - 1)) + (l >> ly) * plane; };
  extern __shared__ unsigned char smem_raw[];
  const int n = 1 << logn, lh = logn - 1, h = n >> 1;
  cpx<T> *tws = reinterpret_cast<cpx<T> *>(smem_raw);
  cpx<T> *s = tws + h;
  load_twiddles<T>(tws, tw, n);
  const int64_t l0 = (int64_t)blockIdx.x * B;
  const int nb = (int)((nlines - l0) < B ? (nlines - l0) : B);
  const cpx<T> *rin2 = reinterpret_cast<const cpx<T> *>(rin);
  if (MODE == 0) {
    // kU independent loads in flight per thread before the LDS stores
    for (int e0 = threadIdx.x; e0 < (nb << lh); e0 += kU * 256) {
      cpx<T> v[kU];
#pragma unroll
      for (int u = 0; u < kU; u++) {
        const int e = e0 + 256 * u;
        if (e < (nb << lh)) v[u] = rin2[(l0 + (e >> lh)) * h + (e & (h - 1))];
      }
#pragma unroll
      for (int u = 0; u < kU; u++) {
        const int e = e0 + 256 * u;
        if (e < (nb << lh)) s[(e >> lh) * (h + 1) + (e & (h - 1))] = v[u];
      }
    }
    __syncthreads();
    dif_fwd<T>(s, nb, lh, tws, 1);
    for (int e = threadIdx.x; e < (nb << lh); e += blockDim.x) {
      const int b = e >> lh, k = e & (h - 1);
      const cpx<T> Z = s[b * (h + 1) + (lh ? bitrev(k, lh) : 0)];
      cpx<T> X;
      if (k == 0) {
        X = {Z.x + Z.y, Z.x - Z.y};
      } else {
        const cpx<T> M = s[b * (h + 1) + bitrev(h - k, lh)];
        const cpx<T> E = {(T)0.5 * (Z.x + M.x), (T)0.5 * (Z.y - M.y)};
        const cpx<T> O = {(T)0.5 * (Z.y + M.y), (T)0.5 * (M.x - Z.x)};
        const cpx<T> WO = cmul<T>(O, tws[k]);
        X = {E.x + WO.x, E.y + WO.y};
      }
      buf[at(l0 + b) + k] = X;
    }
  } else {
    __syncthreads();  // the unpacking below reads twiddles loaded by other threads
    for (int e0 = threadIdx.x; e0 < (nb << lh); e0 += kU * 256) {
      cpx<T> X[kU], M[kU];
#pragma unroll
      for (int u = 0; u < kU; u++) {
        const int e = e0 + 256 * u;
        if (e < (nb << lh)) {
          const int b = e >> lh, k = e & (h - 1);
          const int64_t o = at(l0 + b);
          X[u] = buf[o + k];
          M[u] = buf[o + ((h - k) & (h - 1))];
        }
      }
#pragma unroll
      for (int u = 0; u < kU; u++) {
        const int e = e0 + 256 * u;
        if (e < (nb << lh)) {
          const int b = e >> lh, k = e & (h - 1);
          cpx<T> Z;
          if (k == 0) {
            Z = {X[u].x + X[u].y, X[u].x - X[u].y};
          } else {
            const cpx<T> E = {X[u].x + M[u].x, X[u].y - M[u].y};
            const cpx<T> D = {X[u].x - M[u].x, X[u].y + M[u].y};
            const cpx<T> w = tws[k];
            const cpx<T> O = cmul<T>(D, {w.x, -w.y});
            Z = {E.x - O.y, E.y + O.x};  // E + i O
          }
          s[b * (h + 1) + (lh ? bitrev(k, lh) : 0)] = Z;
        }
      }
    }
    __syncthreads();
    dit_inv<T>(s, nb, lh, tws, 1);
    cpx<T> *rout2 = reinterpret_cast<cpx<T> *>(rout);
    for (int e = threadIdx.x; e < (nb << lh); e += blockDim.x) {
      const int b = e >> lh, t = e & (h - 1);
      const cpx<T> z = s[b * (h + 1) + t];
      rout2[(l0 + b) * h + t] = {(T)((double)z.x * scale), (T)((double)z.y * scale)};
    }
  }
}

// Symbol of the constant-coefficient operator in closed form:
// lam = A0 + sum_a F_a c_a + sum_{a<b} (P_ab c_a c_b - M_ab s_a s_b),
// c_a = cos(theta_a), s_a = sin(theta_a) (faces and edges paired by a_o = a_-o).
struct Symbol {
  double A0, F[3], P[3], M[3];  // pairs ordered xy, xz, yz
  int nx, lx, ly, lz;
  int ynat;                     // y frequencies of the spectrum in natural (1) or bit-reversed (0) order
  double inv_scale;             // 1 / (nx ny nz)
};

__device__ __forceinline__ double symbol_at(const Symbol &sym, int kx, int ky, int kz, const double *__restrict__ trx,
                                            const double *__restrict__ try_, const double *__restrict__ trz)
{
  const double cx = trx[2 * kx], sx = trx[2 * kx + 1];
  const double cy = try_[2 * ky], sy = try_[2 * ky + 1];
  const double cz = trz[2 * kz], sz = trz[2 * kz + 1];
  return sym.A0 + sym.F[0] * cx + sym.F[1] * cy + sym.F[2] * cz + (sym.P[0] * cx * cy - sym.M[0] * sx * sy) +
         (sym.P[1] * cx * cz - sym.M[1] * sx * sz) + (sym.P[2] * cy * cz - sym.M[2] * sy * sz);
}

// inv_scale / lam, 0 for the null mode
__device__ __forceinline__ double symbol_factor(const Symbol &sym, int kx, int ky, int kz, const double *trx,
                                                const double *try_, const double *trz)
{
  if (kx == 0 && ky == 0 && kz == 0) return 0.0;
  const double lam = symbol_at(sym, kx, ky, kz, trx, try_, trz);
  return lam == 0.0 ? 0.0 : sym.inv_scale / lam;
}

// Pass along a strided axis: line (a, c) at base a + c*cstride, element t at
// + t*estride; a block holds B consecutive a.  MODE 0 forward, 1 inverse,
// 2 forward + symbol division + inverse (z axis) for the half-spectrum lines
// a = kx + (nx/2) * py with kx >= 1 in natural order (slot 0, which packs
// kx = 0 and nx/2, is left to k_fft_col0) and py the bit-reversed y
// frequency.
template <typename T, int MODE>
__global__ __launch_bounds__(256) void k_fft_s(int logn, int64_t A, int64_t estride, int64_t cstride, int B,
                                               cpx<T> *__restrict__ buf, const double *__restrict__ tw, Symbol sym,
                                               const double *__restrict__ trx, const double *__restrict__ try_,
                                               const double *__restrict__ trz)
{
  extern __shared__ unsigned char smem_raw[];
  const int n = 1 << logn;
  cpx<T> *tws = reinterpret_cast<cpx<T> *>(smem_raw);
  cpx<T> *s = tws + (n >> 1);
  load_twiddles<T>(tws, tw, n);
  const int64_t blocks_per_c = A / B;
  const int64_t c = blockIdx.x / blocks_per_c;
  const int64_t a0 = (blockIdx.x % blocks_per_c) * B;
  const int64_t base = a0 + c * cstride;
  const int hx = sym.nx >> 1;
  const int lb = __ffs(B) - 1;  // B is a power of two
  // in MODE 2 the lines of the packed slot (kx = 0) are not touched
  auto live = [&](int b) { return MODE != 2 || ((a0 + b) & (hx - 1)) != 0; };
  for (int e0 = threadIdx.x; e0 < B * n; e0 += kU * 256) {
    cpx<T> v[kU];
#pragma unroll
    for (int u = 0; u < kU; u++) {
      const int e = e0 + 256 * u;
      const int t = e >> lb, b = e & (B - 1);
      if (e < B * n && live(b)) v[u] = buf[base + b + (int64_t)t * estride];
    }
#pragma unroll
    for (int u = 0; u < kU; u++) {
      const int e = e0 + 256 * u;
      const int t = e >> lb, b = e & (B - 1);
      if (e < B * n && live(b)) s[b * (n + 1) + t] = v[u];
    }
  }
  __syncthreads();
  if (MODE == 1) {
    dit_inv<T>(s, B, logn, tws);
  } else {
    dif_fwd<T>(s, B, logn, tws);
    if (MODE == 3) {
      // 2-D solve: line a is the bit-reversed x frequency, element t the
      // bit-reversed y frequency, kz = 0
      for (int e = threadIdx.x; e < B * n; e += blockDim.x) {
        const int t = e >> lb, b = e & (B - 1);
        const int kx = bitrev((int)(a0 + b), sym.lx), ky = bitrev(t, sym.ly);
        const double f = symbol_factor(sym, kx, ky, 0, trx, try_, trz);
        cpx<T> &z = s[b * (n + 1) + t];
        z = {(T)((double)z.x * f), (T)((double)z.y * f)};
      }
      __syncthreads();
      dit_inv<T>(s, B, logn, tws);
    }
    if (MODE == 2) {
      // line a = kx + (nx/2)*py holds the natural x and bit-reversed y
      // frequencies, element t the bit-reversed z frequency.  Along a line the
      // symbol is la + lb cos(kz) - lc sin(kz) (the z terms of symbol_at
      // grouped): the three line constants and the z table are staged in LDS
      // after the lines (kx >= 1 here, so the null mode does not occur).
      double *lcn = reinterpret_cast<double *>(s + B * (n + 1));
      double *tz = lcn + 3 * B;
      for (int b = threadIdx.x; b < B; b += blockDim.x) {
        const int64_t a = a0 + b;
        const int kx = (int)(a & (hx - 1));
        const int py = (int)(a >> (sym.lx - 1));
        const int ky = sym.ynat ? py : bitrev(py, sym.ly);
        const double cx = trx[2 * kx], sx = trx[2 * kx + 1], cy = try_[2 * ky], sy = try_[2 * ky + 1];
        lcn[3 * b] = sym.A0 + sym.F[0] * cx + sym.F[1] * cy + (sym.P[0] * cx * cy - sym.M[0] * sx * sy);
        lcn[3 * b + 1] = sym.F[2] + sym.P[1] * cx + sym.P[2] * cy;
        lcn[3 * b + 2] = sym.M[1] * sx + sym.M[2] * sy;
      }
      for (int t = threadIdx.x; t < 2 * n; t += blockDim.x) tz[t] = trz[t];
      __syncthreads();
      for (int e = threadIdx.x; e < B * n; e += blockDim.x) {
        const int t = e >> lb, b = e & (B - 1);
        const int kz = bitrev(t, sym.lz);
        const double lam = lcn[3 * b] + lcn[3 * b + 1] * tz[2 * kz] - lcn[3 * b + 2] * tz[2 * kz + 1];
        const double f = lam == 0.0 ? 0.0 : sym.inv_scale / lam;
        cpx<T> &z = s[b * (n + 1) + t];
        z = {(T)((double)z.x * f), (T)((double)z.y * f)};
      }
      __syncthreads();
      dit_inv<T>(s, B, logn, tws);
    }
  }
  for (int e = threadIdx.x; e < B * n; e += blockDim.x) {
    const int t = e >> lb, b = e & (B - 1);
    if (live(b)) buf[base + b + (int64_t)t * estride] = s[b * (n + 1) + t];
  }
}

// The packed slot kx = 0 of the half spectrum holds X_0 + i X_h, both real in
// x, so after the y and z transforms Z = P + i Q with P = F(X_0), Q = F(X_h)
// Hermitian: P(k) = (Z(k) + conj Z(-k))/2, Q(k) = (Z(k) - conj Z(-k))/(2i).
// Block p takes the z-lines of bit-reversed y positions p and p' (ky' = -ky;
// p' == p for ky = 0, ny/2), transforms both, scales P by the symbol at
// kx = 0 and Q by the symbol at kx = nx/2, recombines and transforms back.
// Block p's share (all threads of the block): tws holds the n-point
// twiddles, s has room for 2 (n + 1) values.
template <typename T>
__device__ __forceinline__ void fft_col0_body(int p, int logn, int64_t estride, int hx, cpx<T> *__restrict__ buf,
                                              const cpx<T> *tws, cpx<T> *s, const Symbol &sym,
                                              const double *__restrict__ trx, const double *__restrict__ try_,
                                              const double *__restrict__ trz)
{
  const int n = 1 << logn;
  const int ny = 1 << sym.ly;
  const int ky = sym.ynat ? p : bitrev(p, sym.ly);
  const int pp = sym.ynat ? (ny - ky) & (ny - 1) : bitrev((ny - ky) & (ny - 1), sym.ly);
  if (pp < p) return;             // the pair is done by block pp
  const int nl = pp == p ? 1 : 2;
  const int64_t base[2] = {(int64_t)hx * p, (int64_t)hx * pp};
  for (int e = threadIdx.x; e < nl * n; e += blockDim.x) {
    const int b = e >> logn, t = e & (n - 1);
    s[b * (n + 1) + t] = buf[base[b] + (int64_t)t * estride];
  }
  __syncthreads();
  dif_fwd<T>(s, nl, logn, tws);
  // every new value needs its partner's old one: compute into registers, then write
  constexpr int kPerThread = 2 * kFftMaxN / 256;  // (shorter lines in blocks of 128 threads too)
  cpx<T> nv[kPerThread];
#pragma unroll
  for (int q = 0; q < kPerThread; q++) {
    const int e = threadIdx.x + blockDim.x * q;
    if (e >= nl * n) break;
    const int b = e >> logn, t = e & (n - 1);
    const int kyb = b == 0 ? ky : (ny - ky) & (ny - 1);
    const int kz = bitrev(t, sym.lz);
    const int tm = bitrev((n - kz) & (n - 1), sym.lz);
    const int bm = nl == 1 ? 0 : 1 - b;
    const cpx<T> Z = s[b * (n + 1) + t], M = s[bm * (n + 1) + tm];
    const double Px = 0.5 * ((double)Z.x + (double)M.x), Py = 0.5 * ((double)Z.y - (double)M.y);
    const double Qx = 0.5 * ((double)Z.y + (double)M.y), Qy = 0.5 * ((double)M.x - (double)Z.x);
    const double f0 = symbol_factor(sym, 0, kyb, kz, trx, try_, trz);
    const double fh = symbol_factor(sym, hx, kyb, kz, trx, try_, trz);
    // P f0 + i Q fh
    nv[q] = {(T)(Px * f0 - Qy * fh), (T)(Py * f0 + Qx * fh)};
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kPerThread; q++) {
    const int e = threadIdx.x + blockDim.x * q;
    if (e >= nl * n) break;
    s[(e >> logn) * (n + 1) + (e & (n - 1))] = nv[q];
  }
  __syncthreads();
  dit_inv<T>(s, nl, logn, tws);
  for (int e = threadIdx.x; e < nl * n; e += blockDim.x) {
    const int b = e >> logn, t = e & (n - 1);
    buf[base[b] + (int64_t)t * estride] = s[b * (n + 1) + t];
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_fft_col0(int logn, int64_t estride, int hx, cpx<T> *__restrict__ buf,
                                                  const double *__restrict__ tw, Symbol sym,
                                                  const double *__restrict__ trx, const double *__restrict__ try_,
                                                  const double *__restrict__ trz)
{
  extern __shared__ unsigned char smem_raw[];
  const int n = 1 << logn;
  cpx<T> *tws = reinterpret_cast<cpx<T> *>(smem_raw);
  cpx<T> *s = tws + (n >> 1);     // 2 lines, padded
  load_twiddles<T>(tws, tw, n);
  fft_col0_body<T>((int)blockIdx.x, logn, estride, hx, buf, tws, s, sym, trx, try_, trz);
}

// ---- lines of 16 to 512 points: register-resident four-step transforms --------------
// A line of N = TH R points (TH <= R: 4x4, 4x8, 8x8, 8x16, 16x16 and 16x32) is
// held by TH threads, thread j owning the elements j + TH m (m < R) in
// registers.  Each thread transforms its R values (a length-R DFT in registers
// over m), multiplies by the twiddles W_N^(j k1), and one transpose through LDS
// hands thread j the TH values of rows k1 = j + TH c (c < R/TH), whose TH-point
// DFTs over j give X[k1 + R k2].  That is element j + TH (c + (R/TH) k2): input
// and output use the same register pattern in natural order, so forward and
// inverse compose without permutations, and LDS carries each value twice per
// transform, where the radix-4 passes carry it once a stage with a barrier
// each.  Short lines are bound by that chain of LDS round trips, long ones by
// the bytes.  Measured against the radix-4 passes, us for x + y + z + y + x of
// one application with the packed column: FP64 32^3 44.2 -> 20.9, 64^3 71.5 ->
// 23.6, 128^3 122.6 -> 55.8; FP32 32^3 40.8 -> 19.4, 64^3 60.4 -> 19.8, 128^3
// 84.8 -> 39.9.
//
// LDS strides between the rows of a line (TH + 1) and between the lines of a
// block, for values split into real and imaginary arrays: with 16 threads a
// line the 64 lanes of a wave touch 64 distinct banks in both layouts (strided
// passes: lanes are 16 lines x 4 threads, x pass: 16 threads x 4 line pairs);
// shorter lines take an odd stride (strided) or an odd multiple of TH (x pass).
template <int TH, int R> constexpr int q_sbs() { return TH == 16 ? (R == 16 ? 324 : 580) : (R * (TH + 1)) | 1; }
template <int TH, int R> constexpr int q_sbx()
{
  return TH * ((R * (TH + 1) + TH - 1) / TH | 1);
}
// threads of a block: 128 where 256 threads' lines would fill half of a CU's LDS
template <typename T, int TH, int R> constexpr int q_block() { return sizeof(T) == 8 && TH * R == 128 ? 128 : 256; }

template <typename T, bool INV>
__device__ __forceinline__ void dft4(cpx<T> &a0, cpx<T> &a1, cpx<T> &a2, cpx<T> &a3)
{
  const cpx<T> t0 = {a0.x + a2.x, a0.y + a2.y}, t1 = {a0.x - a2.x, a0.y - a2.y};
  const cpx<T> t2 = {a1.x + a3.x, a1.y + a3.y}, t3 = {a1.x - a3.x, a1.y - a3.y};
  a0 = {t0.x + t2.x, t0.y + t2.y};
  a2 = {t0.x - t2.x, t0.y - t2.y};
  if (!INV) {  // X1 = t1 - i t3, X3 = t1 + i t3
    a1 = {t1.x + t3.y, t1.y - t3.x};
    a3 = {t1.x - t3.y, t1.y + t3.x};
  } else {
    a1 = {t1.x - t3.y, t1.y + t3.x};
    a3 = {t1.x + t3.y, t1.y - t3.x};
  }
}

// In-place 16-point DFT, natural order in and out: n = 4a + b, k = c + 4d.
template <typename T, bool INV>
__device__ __forceinline__ void dft16(cpx<T> (&v)[16])
{
  constexpr double c1 = 0.92387953251128674, s1 = 0.38268343236508978, h = 0.70710678118654752;  // cos, sin pi/8; sqrt 1/2
  // W_16^m = cos(2 pi m / 16) - i sin(2 pi m / 16) for the products m = b c
  constexpr double wr[10] = {1.0, c1, h, s1, 0.0, 0.0, -h, 0.0, 0.0, -c1};
  constexpr double wi[10] = {0.0, -s1, -h, -c1, -1.0, 0.0, -h, 0.0, 0.0, s1};
#pragma unroll
  for (int b = 0; b < 4; b++) dft4<T, INV>(v[b], v[4 + b], v[8 + b], v[12 + b]);
#pragma unroll
  for (int b = 1; b < 4; b++) {
#pragma unroll
    for (int c = 1; c < 4; c++) {
      const int m = b * c;
      const T x = (T)wr[m], y = INV ? (T)(-wi[m]) : (T)wi[m];
      v[4 * c + b] = cmul<T>(v[4 * c + b], {x, y});
    }
  }
#pragma unroll
  for (int c = 0; c < 4; c++) dft4<T, INV>(v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]);
  // position 4c + d holds X[c + 4d]
  cpx<T> o[16];
#pragma unroll
  for (int c = 0; c < 4; c++)
#pragma unroll
    for (int d = 0; d < 4; d++) o[c + 4 * d] = v[4 * c + d];
#pragma unroll
  for (int q = 0; q < 16; q++) v[q] = o[q];
}

// In-place 8-point DFT, natural order in and out: the 4-point DFTs of the even
// and odd elements and one radix-2 stage.
template <typename T, bool INV>
__device__ __forceinline__ void dft8(cpx<T> (&v)[8])
{
  constexpr T h = (T)0.70710678118654752;
  cpx<T> e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6], o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
  dft4<T, INV>(e0, e1, e2, e3);
  dft4<T, INV>(o0, o1, o2, o3);
  const T sg = INV ? (T)1 : (T)-1;  // W_8^k = cos(2 pi k / 8) -+ i sin(2 pi k / 8)
  o1 = cmul<T>(o1, {h, sg * h});
  o2 = {-sg * o2.y, sg * o2.x};
  o3 = cmul<T>(o3, {-h, sg * h});
  v[0] = {e0.x + o0.x, e0.y + o0.y}; v[4] = {e0.x - o0.x, e0.y - o0.y};
  v[1] = {e1.x + o1.x, e1.y + o1.y}; v[5] = {e1.x - o1.x, e1.y - o1.y};
  v[2] = {e2.x + o2.x, e2.y + o2.y}; v[6] = {e2.x - o2.x, e2.y - o2.y};
  v[3] = {e3.x + o3.x, e3.y + o3.y}; v[7] = {e3.x - o3.x, e3.y - o3.y};
}

// In-place R-point DFT (R = 4, 8, 16 or 32), natural order in and out; 32
// points as two 16-point DFTs of the even and odd elements and one radix-2
// stage.
template <typename T, bool INV, int R>
__device__ __forceinline__ void dftR(cpx<T> (&v)[R])
{
  if constexpr (R == 4) {
    dft4<T, INV>(v[0], v[1], v[2], v[3]);
  } else if constexpr (R == 8) {
    dft8<T, INV>(v);
  } else if constexpr (R == 16) {
    dft16<T, INV>(v);
  } else {
    static_assert(R == 32, "4- to 32-point register DFTs");
    cpx<T> e[16], o[16];
#pragma unroll
    for (int q = 0; q < 16; q++) { e[q] = v[2 * q]; o[q] = v[2 * q + 1]; }
    dft16<T, INV>(e);
    dft16<T, INV>(o);
    // W_32^k = cos(2 pi k / 32) -+ i sin(2 pi k / 32)
    constexpr double wc[16] = {1.0, 0.9807852804032304, 0.9238795325112867, 0.8314696123025452, 0.7071067811865476, 0.5555702330196023, 0.38268343236508984, 0.19509032201612833, 0.0, -0.1950903220161282, -0.3826834323650897, -0.555570233019602, -0.7071067811865475, -0.8314696123025453, -0.9238795325112867, -0.9807852804032304};
    constexpr double ws[16] = {0.0, 0.19509032201612825, 0.3826834323650898, 0.5555702330196022, 0.7071067811865475, 0.8314696123025452, 0.9238795325112867, 0.9807852804032304, 1.0, 0.9807852804032304, 0.9238795325112867, 0.8314696123025455, 0.7071067811865476, 0.5555702330196022, 0.3826834323650899, 0.1950903220161286};
#pragma unroll
    for (int k = 0; k < 16; k++) {
      const T wr = (T)wc[k], wi = INV ? (T)ws[k] : (T)(-ws[k]);
      const cpx<T> t = cmul<T>(o[k], {wr, wi});
      v[k] = {e[k].x + t.x, e[k].y + t.y};
      v[k + 16] = {e[k].x - t.x, e[k].y - t.y};
    }
  }
}

// The four-step transform of the line held by this thread's group (thread j
// of TH; its LDS rows start at gbase).  tws: W_N^m, m < N/2 (forward).  Every
// thread of the block calls it (two barriers); with WAVE, whole waves that hold
// their lines' threads, each ordering its own LDS accesses.
template <typename T, bool INV, int TH, int R, bool WAVE = false>
__device__ __forceinline__ void fft_line(cpx<T> (&v)[R], int j, T *lre, T *lim, int gbase, const cpx<T> *tws)
{
  constexpr int N = TH * R, H = N / 2, SK = TH + 1;
  dftR<T, INV, R>(v);
#pragma unroll
  for (int k1 = 1; k1 < R; k1++) {
    const int m = j * k1;  // < N: W^m = -W^(m-N/2) past N/2
    cpx<T> w = tws[m & (H - 1)];
    if (m & H) w = {-w.x, -w.y};
    if (INV) w.y = -w.y;
    v[k1] = cmul<T>(v[k1], w);
  }
#pragma unroll
  for (int k1 = 0; k1 < R; k1++) {
    lre[gbase + k1 * SK + j] = v[k1].x;
    lim[gbase + k1 * SK + j] = v[k1].y;
  }
  if (WAVE) wave_sync(); else __syncthreads();
#pragma unroll
  for (int c = 0; c < R / TH; c++) {
    cpx<T> u[TH];
    const int row = gbase + (j + TH * c) * SK;
#pragma unroll
    for (int n2 = 0; n2 < TH; n2++) u[n2] = {lre[row + n2], lim[row + n2]};
    dftR<T, INV, TH>(u);
#pragma unroll
    for (int k2 = 0; k2 < TH; k2++) v[c + (R / TH) * k2] = u[k2];
  }
  if (WAVE) wave_sync(); else __syncthreads();
}

// Strided N-point pass over `lines` lines: line l = a + A c (A = 2^lA) at a + c
// cstride, element t at + t estride; a block takes NL consecutive lines, thread
// (b, j) = (threadIdx % NL, threadIdx / NL).  MODE 0 forward, 1 inverse, 2
// forward + symbol division + inverse (z axis, lines a = kx + (nx/2)*py; the
// packed kx = 0 slot is left to fft_col0_body).
template <typename T, int MODE, int TH, int R>
__global__ __launch_bounds__((q_block<T, TH, R>())) void k_fftq_s(int64_t lines, int lA, int64_t estride, int64_t cstride,
                                                cpx<T> *__restrict__ buf, const double *__restrict__ tw, Symbol sym,
                                                const double *__restrict__ trx, const double *__restrict__ try_,
                                                const double *__restrict__ trz)
{
  constexpr int N = TH * R, SB = q_sbs<TH, R>(), NL = q_block<T, TH, R>() / TH;
  // (the packed column's scratch: 2 (N + 1) complex values)
  constexpr int kLds = 2 * NL * SB > 4 * (N + 1) ? 2 * NL * SB : 4 * (N + 1);
  __shared__ T lds[kLds];
  T *lre = lds, *lim = lds + NL * SB;
  __shared__ cpx<T> tws[N / 2];
  load_twiddles<T>(tws, tw, N);
  __syncthreads();
  if constexpr (MODE == 2) {
    // blocks past the lines take the packed kx = 0 column (the z lines the
    // others leave), so it needs no launch of its own
    const int64_t nmain = (lines + NL - 1) / NL;
    if ((int64_t)blockIdx.x >= nmain) {
      constexpr int kLog = N == 512 ? 9 : N == 256 ? 8 : N == 128 ? 7 : N == 64 ? 6 : N == 32 ? 5 : 4;
      fft_col0_body<T>((int)(blockIdx.x - nmain), kLog, estride, sym.nx >> 1, buf, tws, reinterpret_cast<cpx<T> *>(lds),
                       sym, trx, try_, trz);
      return;
    }
  }
  const int b = threadIdx.x % NL, j = threadIdx.x / NL;
  const int64_t l = (int64_t)blockIdx.x * NL + b, a = l & (((int64_t)1 << lA) - 1);
  const int64_t base = a + (l >> lA) * cstride;
  const int hx = sym.nx >> 1;
  const bool live = l < lines && (MODE != 2 || (a & (hx - 1)) != 0);
  cpx<T> v[R];
#pragma unroll
  for (int m = 0; m < R; m++) v[m] = live ? buf[base + (int64_t)(j + TH * m) * estride] : cpx<T>{(T)0, (T)0};
  fft_line<T, MODE == 1, TH, R>(v, j, lre, lim, b * SB, tws);
  if (MODE == 2) {
    // symbol along the line: la + lb cos(kz) - lc sin(kz), kz = j + TH m
    const int kx = (int)(a & (hx - 1));
    const int py = live ? (int)(a >> (sym.lx - 1)) : 0;
    const int ky = sym.ynat ? py : bitrev(py, sym.ly);
    const double cx = trx[2 * kx], sx = trx[2 * kx + 1], cy = try_[2 * ky], sy = try_[2 * ky + 1];
    const double la = sym.A0 + sym.F[0] * cx + sym.F[1] * cy + (sym.P[0] * cx * cy - sym.M[0] * sx * sy);
    const double lb = sym.F[2] + sym.P[1] * cx + sym.P[2] * cy;
    const double lc = sym.M[1] * sx + sym.M[2] * sy;
#pragma unroll
    for (int m = 0; m < R; m++) {
      const int kz = j + TH * m;
      // lambda in FP64 (it cancels near k = 0); the FP32 passes of 256 and 512
      // points then take its reciprocal in FP32, the shorter ones, which the
      // bytes do not bound, refine it to FP64 (one Newton step: 1e-14; the
      // FP32 quotient moves a mode by 4.8e-8 in the mean square, for at most 1 % of
      // a solve), and the FP64 pass divides exactly
      const double lam = la + lb * trz[2 * kz] - lc * trz[2 * kz + 1];
      if constexpr (sizeof(T) == 4 && N < 256) {
        const double y = (double)__builtin_amdgcn_rcpf((float)lam);
        const double f = lam == 0.0 ? 0.0 : sym.inv_scale * __builtin_fma(y, __builtin_fma(-lam, y, 1.0), y);
        v[m] = {(T)((double)v[m].x * f), (T)((double)v[m].y * f)};
      } else if constexpr (sizeof(T) == 4) {
        const float f = lam == 0.0 ? 0.0f : __builtin_amdgcn_rcpf((float)lam) * (float)sym.inv_scale;
        v[m] = {v[m].x * f, v[m].y * f};
      } else {
        const double f = lam == 0.0 ? 0.0 : sym.inv_scale / lam;
        v[m] = {(T)((double)v[m].x * f), (T)((double)v[m].y * f)};
      }
    }
    fft_line<T, true, TH, R>(v, j, lre, lim, b * SB, tws);
  }
  if (live) {
#pragma unroll
    for (int m = 0; m < R; m++) buf[base + (int64_t)(j + TH * m) * estride] = v[m];
  }
}

// x pass for nx = N, two real lines per group of TH threads (2 NL lines per
// block): z = x_a + i x_b is transformed once, and X_a = (Z_k + conj Z_-k)/2,
// X_b = (Z_k - conj Z_-k)/(2i) are written for k < N/2 (slot 0 packs X_0 and
// X_(N/2) as X_0 + i X_(N/2)), to the same layout as k_rfft_x.  MODE 1 is the
// exact reverse: Z_k = X_a + i X_b over the Hermitian extension, inverse
// transform, x_a = Re, x_b = Im (N times the input), times scale.  nlines is
// even (axes have a power of two of nodes, at least 4).
template <typename T, int MODE, int TH, int R>
__global__ __launch_bounds__((q_block<T, TH, R>())) void k_rfftq_x(int64_t nlines, const T *__restrict__ rin,
                                                 cpx<T> *__restrict__ buf, T *__restrict__ rout,
                                                 const double *__restrict__ tw, double scale, int ly, int64_t plane)
{
  constexpr int N = TH * R, H = N / 2, SB = q_sbx<TH, R>(), NL = q_block<T, TH, R>() / TH;
  static_assert(SB >= R * (TH + 1) && SB >= N, "a line's rows, and its N values in natural order");
  __shared__ T lre[NL * SB], lim[NL * SB];
  __shared__ cpx<T> tws[H];
  load_twiddles<T>(tws, tw, N);
  __syncthreads();
  const int j = threadIdx.x % TH, g = threadIdx.x / TH;
  const int64_t la = (int64_t)blockIdx.x * (2 * NL) + 2 * g, lb = la + 1;
  const bool ok = lb < nlines;
  auto at = [&](int64_t l) { return (l & ((1 << ly) - 1)) * (int64_t)H + (l >> ly) * plane; };
  const int gb = g * SB;
  cpx<T> v[R];
  if (MODE == 0) {
#pragma unroll
    for (int m = 0; m < R; m++)
      v[m] = ok ? cpx<T>{rin[la * N + j + TH * m], rin[lb * N + j + TH * m]} : cpx<T>{(T)0, (T)0};
    fft_line<T, false, TH, R>(v, j, lre, lim, gb, tws);
    // Z in natural order in LDS, for the partner values Z_-k
#pragma unroll
    for (int m = 0; m < R; m++) {
      lre[gb + j + TH * m] = v[m].x;
      lim[gb + j + TH * m] = v[m].y;
    }
    __syncthreads();
    if (ok) {
      const int64_t oa = at(la), ob = at(lb);
#pragma unroll
      for (int m = 0; m < R / 2; m++) {
        const int k = j + TH * m;
        const T zx = lre[gb + k], zy = lim[gb + k];
        cpx<T> xa, xb;
        if (k == 0) {
          xa = {zx, lre[gb + H]};
          xb = {zy, lim[gb + H]};
        } else {
          const T mx = lre[gb + N - k], my = lim[gb + N - k];
          xa = {(T)0.5 * (zx + mx), (T)0.5 * (zy - my)};
          xb = {(T)0.5 * (zy + my), (T)0.5 * (mx - zx)};
        }
        buf[oa + k] = xa;
        buf[ob + k] = xb;
      }
    }
  } else {
    const int64_t oa = ok ? at(la) : 0, ob = ok ? at(lb) : 0;
    // each half-spectrum value is read once: A_t and B_t (t < N/2) staged in
    // LDS, then Z_t = A_t + i B_t and its Hermitian partner Z_(N-t) built from
    // there (Z_0 and Z_(N/2) from the packed slot 0)
    T *are = lre + gb, *aim = lim + gb, *bre = are + H, *bim = aim + H;
#pragma unroll
    for (int m = 0; m < R / 2; m++) {
      const int t = j + TH * m;
      const cpx<T> A = ok ? buf[oa + t] : cpx<T>{(T)0, (T)0}, B = ok ? buf[ob + t] : cpx<T>{(T)0, (T)0};
      are[t] = A.x; aim[t] = A.y; bre[t] = B.x; bim[t] = B.y;
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < R; m++) {
      const int t = j + TH * m;
      cpx<T> z;
      if (t == 0) z = {are[0], bre[0]};
      else if (t == H) z = {aim[0], bim[0]};
      else if (t < H) z = {are[t] - bim[t], aim[t] + bre[t]};
      else z = {are[N - t] + bim[N - t], bre[N - t] - aim[N - t]};
      v[m] = z;
    }
    __syncthreads();
    fft_line<T, true, TH, R>(v, j, lre, lim, gb, tws);
    if (ok) {
#pragma unroll
      for (int m = 0; m < R; m++) {
        rout[la * N + j + TH * m] = (T)((double)v[m].x * scale);
        rout[lb * N + j + TH * m] = (T)((double)v[m].y * scale);
      }
    }
  }
}

// The x and y passes of one plane in one launch: a block holds the plane's row
// pairs, then its columns of the half spectrum, in LDS (a line's exchange takes
// place in its own row, SX or SY apart; its threads are lanes of one wave).
// MODE 0: real rows -> half spectrum, natural order along x and y, as k_rfftq_x<0>
// and k_fftq_s<0> leave it; MODE 1 the reverse.  On small grids a pass is one
// launch's latency, so two in one are the faster: us forward and back, four
// launches -> two: 16^3 FP64 11.2 -> 6.7, 32^3 FP64 15.9 -> 8.3 and FP32 14.3 ->
// 7.8, 64^3 FP64 18.1 -> 12.9 and FP32 15.1 -> 11.4; a solve on 16^3 FP64 843 -> 772,
// 32^3 FP64 815 -> 755, 64^3 FP64 953 -> 919, 64 x 64 x 256 mixed 1067 -> 1012.  (A
// plane of 64 x 128 fills a block for as long as the launches take: 21.0 and
// 21.1 us.)
template <typename T, int MODE, int THX, int RX, int THY, int RY>
__global__ __launch_bounds__((std::max(64, std::max(RY * THY / 2 * THX, THX * RX / 2 * THY))))
void k_fft_xy(const T *__restrict__ rin, cpx<T> *__restrict__ buf, T *__restrict__ rout,
              const double *__restrict__ twx, const double *__restrict__ twy, int64_t pstride)
{
  constexpr int NX = THX * RX, NY = THY * RY, H = NX / 2;
  constexpr int SX = (RX * (THX + 1) > NX ? RX * (THX + 1) : NX) | 1;
  constexpr int SY = (RY * (THY + 1) > NY ? RY * (THY + 1) : NY) | 1;
  constexpr int L = NY / 2 * SX > H * SY ? NY / 2 * SX : H * SY;
  __shared__ T pre[L], pim[L];
  __shared__ cpx<T> tx[NX / 2], ty[NY / 2];
  const int t = (int)threadIdx.x, g = t / THX, jx = t % THX, kx = t / THY, jy = t % THY;
  const bool xl = t < NY / 2 * THX, yl = t < H * THY;
  cpx<T> *pb = buf + (int64_t)blockIdx.x * pstride;
  const int64_t r0 = (int64_t)blockIdx.x * NX * NY + (int64_t)2 * g * NX;
  cpx<T> ax[RX], ay[RY];
  if (MODE == 0) {
    if (xl) {
#pragma unroll
      for (int m = 0; m < RX; m++) ax[m] = {rin[r0 + jx + THX * m], rin[r0 + NX + jx + THX * m]};
    }
  } else if (yl) {
#pragma unroll
    for (int m = 0; m < RY; m++) ay[m] = pb[kx + H * (jy + THY * m)];
  }
  load_twiddles<T>(tx, twx, NX);
  load_twiddles<T>(ty, twy, NY);
  __syncthreads();
  T *re = pre + g * SX, *im = pim + g * SX;
  if (MODE == 0) {
    cpx<T> xa[RX / 2], xb[RX / 2];
    if (xl) {
      fft_line<T, false, THX, RX, true>(ax, jx, pre, pim, g * SX, tx);
#pragma unroll
      for (int m = 0; m < RX; m++) { re[jx + THX * m] = ax[m].x; im[jx + THX * m] = ax[m].y; }
      wave_sync();
#pragma unroll
      for (int m = 0; m < RX / 2; m++) {
        const int k = jx + THX * m;
        const T zx = re[k], zy = im[k];
        if (k == 0) {
          xa[m] = {zx, re[H]};
          xb[m] = {zy, im[H]};
        } else {
          const T mx = re[NX - k], my = im[NX - k];
          xa[m] = {(T)0.5 * (zx + mx), (T)0.5 * (zy - my)};
          xb[m] = {(T)0.5 * (zy + my), (T)0.5 * (mx - zx)};
        }
      }
    }
    __syncthreads();
    if (xl) {
#pragma unroll
      for (int m = 0; m < RX / 2; m++) {
        const int c = (jx + THX * m) * SY + 2 * g;
        pre[c] = xa[m].x; pim[c] = xa[m].y;
        pre[c + 1] = xb[m].x; pim[c + 1] = xb[m].y;
      }
    }
    __syncthreads();
    if (yl) {
#pragma unroll
      for (int m = 0; m < RY; m++) ay[m] = {pre[kx * SY + jy + THY * m], pim[kx * SY + jy + THY * m]};
      wave_sync();
      fft_line<T, false, THY, RY, true>(ay, jy, pre, pim, kx * SY, ty);
#pragma unroll
      for (int m = 0; m < RY; m++) pb[kx + H * (jy + THY * m)] = ay[m];
    }
  } else {
    if (yl) fft_line<T, true, THY, RY, true>(ay, jy, pre, pim, kx * SY, ty);
    __syncthreads();
    if (yl) {  // row 2 g at the front of pair g's place, row 2 g + 1 H further
#pragma unroll
      for (int m = 0; m < RY; m++) {
        const int row = jy + THY * m, c = (row >> 1) * SX + (row & 1) * H + kx;
        pre[c] = ay[m].x; pim[c] = ay[m].y;
      }
    }
    __syncthreads();
    if (xl) {
#pragma unroll
      for (int m = 0; m < RX; m++) {
        const int k = jx + THX * m;
        if (k == 0) ax[m] = {re[0], re[H]};
        else if (k == H) ax[m] = {im[0], im[H]};
        else if (k < H) ax[m] = {re[k] - im[H + k], im[k] + re[H + k]};
        else ax[m] = {re[NX - k] + im[H + NX - k], re[H + NX - k] - im[NX - k]};
      }
      wave_sync();
      fft_line<T, true, THX, RX, true>(ax, jx, pre, pim, g * SX, tx);
#pragma unroll
      for (int m = 0; m < RX; m++) {
        rout[r0 + jx + THX * m] = ax[m].x;
        rout[r0 + NX + jx + THX * m] = ax[m].y;
      }
    }
  }
}

// Planes that k_fft_xy takes
static bool fft_xy_plane(int nx, int ny)
{
  auto axis = [](int n) { return n == 16 || n == 32 || n == 64; };
  return axis(nx) && axis(ny);
}

template <typename T, int MODE>
static void launch_fft_xy(chy_ctx *ctx, const T *rin, cpx<T> *buf, T *rout, int64_t pstride)
{
  const int nx = ctx->g.nx, ny = ctx->g.ny;
#define XY(THX, RX, THY, RY)                                                                                   \
  hipLaunchKernelGGL((k_fft_xy<T, MODE, THX, RX, THY, RY>), (unsigned)ctx->g.nz,                               \
                     std::max(64, std::max(RY * THY / 2 * THX, THX * RX / 2 * THY)), 0, ctx->stream, rin, buf, \
                     rout, ctx->tw[0], ctx->tw[1], pstride)
#define XY_X(THY, RY)                     \
  do {                                    \
    if (nx == 16) XY(4, 4, THY, RY);      \
    else if (nx == 32) XY(4, 8, THY, RY); \
    else XY(8, 8, THY, RY);               \
  } while (0)
  if (ny == 16) XY_X(4, 4);
  else if (ny == 32) XY_X(4, 8);
  else XY_X(8, 8);
#undef XY_X
#undef XY
}

static bool pow2(int64_t n) { return n > 0 && (n & (n - 1)) == 0; }

// Axis lengths of the four-step kernels: 16 to 512 points (512 in FP32 only:
// the FP64 tiles would not fit LDS twice per CU); the others take the radix-4
// LDS passes.
template <typename T> static bool q_axis(int n) { return pow2(n) && n >= 16 && n <= (sizeof(T) == 4 ? 512 : 256); }

// call with the axis' TH and R, and NL = the lines (x pass: line pairs) of a block
#define Q_AXIS(T, n, call)                                                                              \
  do {                                                                                                  \
    if (n == 16) { constexpr int TH = 4, R = 4, NL = q_block<T, TH, R>() / TH; call; }                  \
    else if (n == 32) { constexpr int TH = 4, R = 8, NL = q_block<T, TH, R>() / TH; call; }             \
    else if (n == 64) { constexpr int TH = 8, R = 8, NL = q_block<T, TH, R>() / TH; call; }             \
    else if (n == 128) { constexpr int TH = 8, R = 16, NL = q_block<T, TH, R>() / TH; call; }           \
    else if (n == 256) { constexpr int TH = 16, R = 16, NL = q_block<T, TH, R>() / TH; call; }          \
    else if constexpr (sizeof(T) == 4) { constexpr int TH = 16, R = 32, NL = q_block<T, TH, R>() / TH; call; } \
  } while (0)

// Complex elements between z planes of the half spectrum: (nx/2) ny plus
// 256 bytes
template <typename T>
static int64_t spec_plane(int nx, int ny) { return (int64_t)(nx / 2) * ny + 256 / (int64_t)sizeof(cpx<T>); }
static int ilog2(int64_t n) { int l = 0; while ((1ll << l) < n) l++; return l; }

int fft_setup(chy_ctx *ctx)
{
  const int64_t N[3] = {ctx->g.nx, ctx->g.ny, ctx->g.nz};
  ctx->fft_ok = pow2(N[0]) && pow2(N[1]) && pow2(N[2]) && N[0] <= kFftMaxN && N[1] <= kFftMaxN && N[2] <= kFftMaxN;
  if (!ctx->fft_ok) return CHY_OK;
  for (int a = 0; a < 3; a++) {
    std::vector<double> tw(N[a]), tr(2 * N[a]);
    for (int64_t j = 0; j < N[a] / 2; j++) {
      tw[2 * j] = cos(-2.0 * M_PI * (double)j / (double)N[a]);
      tw[2 * j + 1] = sin(-2.0 * M_PI * (double)j / (double)N[a]);
    }
    for (int64_t k = 0; k < N[a]; k++) {
      tr[2 * k] = cos(2.0 * M_PI * (double)k / (double)N[a]);
      tr[2 * k + 1] = sin(2.0 * M_PI * (double)k / (double)N[a]);
    }
    CHY_HIP(hipMalloc(&ctx->tw[a], sizeof(double) * std::max<int64_t>(2, N[a])));
    CHY_HIP(hipMalloc(&ctx->trig[a], sizeof(double) * 2 * N[a]));
    CHY_HIP(hipMemcpy(ctx->tw[a], tw.data(), sizeof(double) * N[a], hipMemcpyHostToDevice));
    CHY_HIP(hipMemcpy(ctx->trig[a], tr.data(), sizeof(double) * 2 * N[a], hipMemcpyHostToDevice));
  }
  return CHY_OK;
}

static Symbol make_symbol(const chy_ctx *ctx, const double v19[19])
{
  const int nx = ctx->g.nx, ny = ctx->g.ny, nz = ctx->g.nz;
  Symbol sym;
  sym.A0 = v19[18];
  sym.F[0] = 2.0 * v19[0]; sym.F[1] = 2.0 * v19[2]; sym.F[2] = 2.0 * v19[4];
  sym.P[0] = 2.0 * (v19[6] + v19[7]);   sym.M[0] = 2.0 * (v19[6] - v19[7]);
  sym.P[1] = 2.0 * (v19[10] + v19[11]); sym.M[1] = 2.0 * (v19[10] - v19[11]);
  sym.P[2] = 2.0 * (v19[14] + v19[15]); sym.M[2] = 2.0 * (v19[14] - v19[15]);
  sym.nx = nx;
  sym.lx = ilog2(nx); sym.ly = ilog2(ny); sym.lz = ilog2(nz);
  sym.inv_scale = 1.0 / ((double)nx * ny * nz);
  sym.ynat = 0;
  return sym;
}

template <typename T>
int fft_pc_apply(chy_ctx *ctx, const double v19[19], const T *r, T *z)
{
  const int nx = ctx->g.nx, ny = ctx->g.ny, nz = ctx->g.nz;
  cpx<T> *buf = (cpx<T> *)ctx->fft_buf;
  // symbol coefficients from the uniform-density row (column order of
  // lhs.c:11-104: faces 0..5, xy edges 6..9, xz 10..13, yz 14..17, centre 18)
  Symbol sym = make_symbol(ctx, v19);
  const int hx = nx / 2;
  // z planes of the half spectrum are spaced P = (nx/2) ny + padding apart, so
  // that the rows of a z line do not all fall at one power-of-two stride
  const int64_t P = spec_plane<T>(nx, ny);
  // the four-step kernels' y pass leaves the y frequencies in natural order
  const bool xq = q_axis<T>(nx), yq = q_axis<T>(ny), zq = q_axis<T>(nz);
  sym.ynat = yq ? 1 : 0;
  const int nlines = ny * nz;
  const int lhx = ilog2(hx);
  auto blocks = [](int64_t n, int per) { return (unsigned)((n + per - 1) / per); };
#define RFFTQ(MODE, RIN, ROUT)                                                                                        \
  Q_AXIS(T, nx, hipLaunchKernelGGL((k_rfftq_x<T, MODE, TH, R>), blocks(nlines, 2 * NL), NL * TH, 0, ctx->stream,       \
                                   (int64_t)nlines, RIN, buf, ROUT, ctx->tw[0], 1.0, ilog2(ny), P))
#define FFTQ(MODE, n, LINES, LA, EXTRA, ES, CS, TW)                                                                    \
  Q_AXIS(T, n, hipLaunchKernelGGL((k_fftq_s<T, MODE, TH, R>), blocks(LINES, NL) + EXTRA, NL * TH, 0, ctx->stream,      \
                                  (int64_t)(LINES), LA, ES, CS, buf, TW, sym, ctx->trig[0], ctx->trig[1], ctx->trig[2]))
  const bool xy = fft_xy_plane(nx, ny);
  if (xy) {
    launch_fft_xy<T, 0>(ctx, r, buf, (T *)nullptr, P);
  } else if (xq) {  // x forward: real lines -> half spectra (kx < nx/2, slot 0 packs kx = 0, nx/2)
    RFFTQ(0, r, (T *)nullptr);
  } else {
    const int B = rfft_batch<T>(hx, nlines);
    hipLaunchKernelGGL((k_rfft_x<T, 0>), (unsigned)((nlines + B - 1) / B), kBlock, rfft_lds<T>(hx, B), ctx->stream,
                       ilog2(nx), nlines, B, r, buf, (T *)nullptr, ctx->tw[0], 1.0, ilog2(ny), P);
  }
  // y forward: lines (kx, iz); A = nx/2 contiguous, c = iz with stride P
  if (xy) {
  } else if (yq) {
    FFTQ(0, ny, (int64_t)hx * nz, lhx, 0u, (int64_t)hx, P, ctx->tw[1]);
  } else {
    const int n = ny, B = fft_batch<T>(n, hx);
    hipLaunchKernelGGL((k_fft_s<T, 0>), (unsigned)((hx / B) * nz), kBlock, fft_lds<T>(n, B), ctx->stream, ilog2(n),
                       (int64_t)hx, (int64_t)hx, P, B, buf, ctx->tw[1], sym, ctx->trig[0], ctx->trig[1],
                       ctx->trig[2]);
  }
  {  // z forward + symbol + inverse: lines a = kx + (nx/2)*py, estride P
    const int n = nz;
    const int64_t A = (int64_t)hx * ny;
    if (zq) {  // (ny more blocks take the kx = 0 column)
      FFTQ(2, nz, A, ilog2(A), (unsigned)ny, P, (int64_t)0, ctx->tw[2]);
    } else {
      const int B = fft_batch_z<T>(n, A);
      hipLaunchKernelGGL((k_fft_s<T, 2>), (unsigned)(A / B), kBlock, fft_lds_z<T>(n, B), ctx->stream, ilog2(n), A, P,
                         (int64_t)0, B, buf, ctx->tw[2], sym, ctx->trig[0], ctx->trig[1], ctx->trig[2]);
      const size_t lds = ((size_t)(n >> 1) + 2 * (size_t)(n + 1)) * 2 * sizeof(T);
      hipLaunchKernelGGL((k_fft_col0<T>), (unsigned)ny, kBlock, lds, ctx->stream, ilog2(n), P, hx, buf, ctx->tw[2],
                         sym, ctx->trig[0], ctx->trig[1], ctx->trig[2]);
    }
  }
  if (xy) {
    launch_fft_xy<T, 1>(ctx, (const T *)nullptr, buf, z, P);
  } else if (yq) {  // y inverse
    FFTQ(1, ny, (int64_t)hx * nz, lhx, 0u, (int64_t)hx, P, ctx->tw[1]);
  } else {
    const int n = ny, B = fft_batch<T>(n, hx);
    hipLaunchKernelGGL((k_fft_s<T, 1>), (unsigned)((hx / B) * nz), kBlock, fft_lds<T>(n, B), ctx->stream, ilog2(n),
                       (int64_t)hx, (int64_t)hx, P, B, buf, ctx->tw[1], sym, ctx->trig[0], ctx->trig[1],
                       ctx->trig[2]);
  }
  if (xy) {
  } else if (xq) {  // x inverse: half spectra -> real lines
    RFFTQ(1, (const T *)nullptr, z);
  } else {
    const int B = rfft_batch<T>(hx, nlines);
    hipLaunchKernelGGL((k_rfft_x<T, 1>), (unsigned)((nlines + B - 1) / B), kBlock, rfft_lds<T>(hx, B), ctx->stream,
                       ilog2(nx), nlines, B, (const T *)nullptr, buf, z, ctx->tw[0], 1.0, ilog2(ny), P);
  }
#undef RFFTQ
#undef FFTQ
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_err(ctx, CHY_ERR_LIB, std::string("fft: ") + hipGetErrorString(e));
  return CHY_OK;
}

// ---- two-level preconditioner: kz = 0 correction -------------------------------------
// The 2-D inner GMRES keeps its basis unnormalised (U_q), so that no pass
// waits for a norm: a step is three launches, each leaving one partial per
// block of the sums that the next one needs (every block adds them in the same
// fixed order, so all blocks agree bit for bit).  The launches are 4 to 6 us
// each, bound by latency: seven with the final solve, where a launch per pass
// and a second Gram-Schmidt pass made fourteen.  us of a solve of 8
// iterations, fourteen -> seven launches: 64 x 128 x 64 mixed 1270 -> 1060,
// 128^3 FP64 2290 -> 2090, 128^3 mixed 1770 -> 1575, 256^3 FP64 11300 -> 11180.
constexpr int kHm = kFft2Its;
constexpr int kExtZ = 16;  // planes per block when the correction is added

// Rows of a block of the x passes: 64 blocks or more where there are rows
// enough, and with the two rows around them within 64 KB of LDS.
template <typename T>
static int rows2_of(int nx, int ny)
{
  int R = std::max(1, ny / 64);
  while (R > 1 && fft_lds<T>(nx, R + 2) > 65536) R >>= 1;
  return R;
}

static int nb2_of(const chy_ctx *ctx, bool fp32)
{
  const int nx = ctx->g.nx, ny = ctx->g.ny;
  return ny / (fp32 ? rows2_of<float>(nx, ny) : rows2_of<double>(nx, ny));
}

// x-y fields in pc2_buf (T): C (9), U (kFft2Its), Z (kFft2Its), w, and a
// complex work plane (2).
int64_t fft2_buf_elems(const chy_ctx *ctx)
{
  return (int64_t)(9 + kFft2Its + kFft2Its + 1 + 2) * ctx->g.nx * ctx->g.ny;
}

// Double workspace in pc2_h: the z-chunk column sums part[zc][nxy], the
// stencil-block sums pl[nlb], then per-block partials of the inner GMRES:
// pn[j][nb] (|U_j|^2), pd[j][q][nb] (U_q . w in step j, q <= j, and |w|^2 of
// the last step at q = m), and the coefficients y[m] of the Z_q.
struct H2 {
  double *part, *pl, *pn, *pd, *y;
  int64_t nlb;
  int nb;
};

static H2 h2_layout(const chy_ctx *ctx, bool fp32)
{
  const int64_t nxy = (int64_t)ctx->g.nx * ctx->g.ny;
  H2 h;
  h.nb = nb2_of(ctx, fp32);
  h.nlb = lhs_zsum_blocks(ctx->g, fp32);
  h.part = ctx->pc2_h;
  h.pl = h.part + (int64_t)lhs_zchunks(ctx->g, fp32) * nxy;
  h.pn = h.pl + h.nlb;
  h.pd = h.pn + (int64_t)kHm * h.nb;
  h.y = h.pd + (int64_t)kHm * (kHm + 1) * h.nb;
  return h;
}

int64_t fft2_h_elems(const chy_ctx *ctx)
{
  const int64_t nxy = (int64_t)ctx->g.nx * ctx->g.ny;
  const bool fp32 = ctx->mixed;
  const int nb = nb2_of(ctx, fp32);
  return (int64_t)lhs_zchunks(ctx->g, fp32) * nxy + lhs_zsum_blocks(ctx->g, fp32) +
         (int64_t)kHm * (kHm + 2) * nb + kHm;
}

// Block-wide sums of nv values per thread: out[q] (LDS) for q < nv.
template <int NV>
__device__ __forceinline__ void block_sums(double (&v)[NV], int nv, double *out)
{
  __shared__ double sh[16][NV];
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int q = 0; q < NV; q++) {
    if (q < nv) {
      const double t = wave_total(v[q]);
      if ((threadIdx.x & 63) == 0) sh[w][q] = t;
    }
  }
  __syncthreads();
  if (threadIdx.x < nv) {
    double t = 0.0;
    for (int k = 0; k < nw; k++) t += sh[k][threadIdx.x];
    out[threadIdx.x] = t;
  }
  __syncthreads();
}

// Direction j, forward along x.  j = 0: U_0 = r2 - mean(r2), with r2[col] =
// (1/nz) sum_k (r - A z) from the z-chunk column sums; else U_j = w less its
// parts along U_0 .. U_(j-1) (one classical Gram-Schmidt pass: what a second
// would take out, the rounding of w over |U_1|, enters z with the second
// coefficient, of the size of |U_1|.  Against the oracle's two passes, on six planes
// of 16 x 16 to 64 x 128 nodes with densities flat to 95 % contrast, an application
// is as far off as with two: mixed 2e-7 to 2e-6, FP64 the rounding of the
// symbol).  Stores U_j, |U_j|^2
// in the partials, and the rows' transforms (bit-reversed along x) in cb.
template <typename T, bool FIRST>
__global__ __launch_bounds__(256) void k2_dir(int lx, int R, int64_t nxy, int j, int nz, int nzc,
                                              const double *__restrict__ part, const double *__restrict__ pl,
                                              int64_t nlb, T *__restrict__ U, const T *__restrict__ w,
                                              cpx<T> *__restrict__ cb, const double *__restrict__ tw,
                                              double *__restrict__ pn, const double *__restrict__ pd)
{
  extern __shared__ unsigned char smem_raw[];
  const int nx = 1 << lx, nb = (int)gridDim.x;
  cpx<T> *tws = reinterpret_cast<cpx<T> *>(smem_raw);
  cpx<T> *s = tws + (nx >> 1);
  __shared__ double h[2 * kHm];
  load_twiddles<T>(tws, tw, nx);
  const int64_t c0 = (int64_t)blockIdx.x * R << lx;
  double mean = 0.0, a[1] = {0.0};
  if (FIRST) {
    for (int64_t b = threadIdx.x; b < nlb; b += blockDim.x) a[0] += pl[b];
    block_sums<1>(a, 1, h);
    mean = h[0] / ((double)nz * (double)nxy);
  } else {
    // the coefficients of the U_q: (U_q . w) / |U_q|^2
    double t[2 * kHm];
#pragma unroll
    for (int q = 0; q < 2 * kHm; q++) t[q] = 0.0;
    for (int b = threadIdx.x; b < nb; b += blockDim.x) {
#pragma unroll
      for (int q = 0; q < kHm; q++)
        if (q < j) {
          t[q] += pd[(int64_t)((j - 1) * (kHm + 1) + q) * nb + b];
          t[kHm + q] += pn[(int64_t)q * nb + b];
        }
    }
    block_sums<2 * kHm>(t, 2 * kHm, h);
  }
  a[0] = 0.0;
  for (int e = threadIdx.x; e < R << lx; e += blockDim.x) {
    const int64_t col = c0 + e;
    double x;
    if (FIRST) {
      double t = 0.0;
#pragma unroll 8
      for (int zc = 0; zc < nzc; zc++) t += part[(int64_t)zc * nxy + col];
      x = t / (double)nz - mean;
    } else {
      x = (double)w[col];
#pragma unroll
      for (int q = 0; q < kHm; q++)
        if (q < j && h[kHm + q] > 0.0) x -= h[q] / h[kHm + q] * (double)U[(int64_t)q * nxy + col];
    }
    const T xt = (T)x;
    U[(int64_t)j * nxy + col] = xt;
    s[(e >> lx) * (nx + 1) + (e & (nx - 1))] = {xt, (T)0};
    a[0] += (double)xt * (double)xt;
  }
  __syncthreads();
  dif_fwd<T>(s, R, lx, tws);
  for (int e = threadIdx.x; e < R << lx; e += blockDim.x) cb[c0 + e] = s[(e >> lx) * (nx + 1) + (e & (nx - 1))];
  block_sums<1>(a, 1, h);
  if (threadIdx.x == 0) pn[(int64_t)j * nb + blockIdx.x] = h[0];
}

// Z_j back along x and w = A2 Z_j with the z-averaged 9-point coefficients:
// a block transforms its R rows and the two around them (INV; else Z_j is
// there already), stores its rows of Z_j and of w, and leaves its parts of
// U_q . w (q <= j), in the last step of |w|^2 too.
template <typename T, bool INV>
__global__ __launch_bounds__(256) void k2_apply(int lx, int R, int ny, int j, const T *__restrict__ C,
                                                const cpx<T> *__restrict__ cb, const double *__restrict__ tw,
                                                T *__restrict__ Zj, const T *__restrict__ U, T *__restrict__ w,
                                                double *__restrict__ pd)
{
  extern __shared__ unsigned char smem_raw[];
  __shared__ double h[kHm + 1];
  const int nx = 1 << lx, nb = (int)gridDim.x;
  const int64_t nxy = (int64_t)ny << lx;
  cpx<T> *tws = reinterpret_cast<cpx<T> *>(smem_raw);
  cpx<T> *s = tws + (nx >> 1);  // line l: row r0 - 1 + l
  const int r0 = (int)blockIdx.x * R;
  if (INV) {
    load_twiddles<T>(tws, tw, nx);
    for (int e = threadIdx.x; e < (R + 2) << lx; e += blockDim.x) {
      const int l = e >> lx, t = e & (nx - 1);
      s[l * (nx + 1) + t] = cb[((int64_t)((r0 - 1 + l) & (ny - 1)) << lx) + t];
    }
    __syncthreads();
    dit_inv<T>(s, R + 2, lx, tws);
  }
  double a[kHm + 1];
#pragma unroll
  for (int q = 0; q <= kHm; q++) a[q] = 0.0;
  for (int e = threadIdx.x; e < R << lx; e += blockDim.x) {
    const int l = (e >> lx) + 1, i = e & (nx - 1);
    const int64_t col = ((int64_t)r0 << lx) + e;
    const int xs[3] = {(i - 1) & (nx - 1), i, (i + 1) & (nx - 1)};
    double acc = 0.0;
#pragma unroll
    for (int o = 0; o < 9; o++) {
      const int lo = l + o / 3 - 1;
      const T zv = INV ? s[lo * (nx + 1) + xs[o % 3]].x
                       : Zj[((int64_t)((r0 - 1 + lo) & (ny - 1)) << lx) + xs[o % 3]];
      acc += (double)C[o * nxy + col] * (double)zv;
    }
    const T wt = (T)acc;
    if (INV) Zj[col] = s[l * (nx + 1) + i].x;
    if (j + 1 < kHm) w[col] = wt;
#pragma unroll
    for (int q = 0; q < kHm; q++)
      if (q <= j) a[q] += (double)U[(int64_t)q * nxy + col] * (double)wt;
    a[kHm] += (double)wt * (double)wt;
  }
  block_sums<kHm + 1>(a, kHm + 1, h);
  if (threadIdx.x <= kHm) pd[(int64_t)(j * (kHm + 1) + (int)threadIdx.x) * nb + blockIdx.x] = h[threadIdx.x];
}

// Inverse transform along x, real part to io (lines too long for k2_apply's
// rows in LDS)
template <typename T>
__global__ __launch_bounds__(256) void k2_inv_x(int lx, int nlines, int B, T *__restrict__ io,
                                                const cpx<T> *__restrict__ cb, const double *__restrict__ tw)
{
  extern __shared__ unsigned char smem_raw[];
  const int n = 1 << lx;
  cpx<T> *tws = reinterpret_cast<cpx<T> *>(smem_raw);
  cpx<T> *s = tws + (n >> 1);
  load_twiddles<T>(tws, tw, n);
  const int64_t l0 = (int64_t)blockIdx.x * B;
  const int nbl = (int)((nlines - l0) < B ? (nlines - l0) : B);
  for (int e = threadIdx.x; e < (nbl << lx); e += blockDim.x)
    s[(e >> lx) * (n + 1) + (e & (n - 1))] = cb[(l0 << lx) + e];
  __syncthreads();
  dit_inv<T>(s, nbl, lx, tws);
  for (int e = threadIdx.x; e < (nbl << lx); e += blockDim.x)
    io[(l0 << lx) + e] = s[(e >> lx) * (n + 1) + (e & (n - 1))].x;
}

// Givens QR of the Hessenberg columns h[q][j] (q <= j) with subdiagonals
// sub[j + 1] = |V_{j+1}|, sub[0] = beta, and back substitution: y[q], q < kHm
// (zero past a breakdown).
__device__ __forceinline__ void h2_lstsq(const double (&sub)[kHm + 1], const double (&hc)[kHm][kHm], double *y)
{
  double H[kHm][kHm], g[kHm + 1], cs[kHm], sn[kHm], yy[kHm];
  for (int q = 0; q <= kHm; q++) g[q] = 0.0;
  for (int q = 0; q < kHm; q++) yy[q] = 0.0;
  int jm = 0;
  if (sub[0] > 0.0) {
    g[0] = sub[0];
    for (int j = 0; j < kHm; j++) {
      double h[kHm + 1];
      for (int q = 0; q <= j; q++) h[q] = hc[q][j];
      h[j + 1] = sub[j + 1];
      const bool more = h[j + 1] > 0.0;
      for (int q = 0; q < j; q++) {
        const double t = cs[q] * h[q] + sn[q] * h[q + 1];
        h[q + 1] = -sn[q] * h[q] + cs[q] * h[q + 1];
        h[q] = t;
      }
      const double rr = sqrt(h[j] * h[j] + h[j + 1] * h[j + 1]);
      cs[j] = rr > 0.0 ? h[j] / rr : 1.0;
      sn[j] = rr > 0.0 ? h[j + 1] / rr : 0.0;
      h[j] = rr;
      g[j + 1] = -sn[j] * g[j];
      g[j] = cs[j] * g[j];
      for (int q = 0; q <= j; q++) H[q][j] = h[q];
      jm = j + 1;
      if (!more) break;
    }
    for (int q = jm - 1; q >= 0; q--) {
      double s = g[q];
      for (int r = q + 1; r < jm; r++) s -= H[q][r] * yy[r];
      yy[q] = H[q][q] != 0.0 ? s / H[q][q] : 0.0;
    }
  }
  for (int q = 0; q < kHm; q++) y[q] = yy[q];
}

// The coefficients y[q] of the Z_q from red: |U_j|^2, j < kHm, then rows j of
// U_q . w (q <= j) and |w|^2 (see h2_layout).  The last subdiagonal entry is a
// difference: it cancels where the entry is small, and enters the least
// squares by its square.
__device__ __forceinline__ void h2_coeffs(const double *red, double *y)
{
  double sub[kHm + 1], hc[kHm][kHm], in[kHm];
  for (int j = 0; j < kHm; j++) {
    const double n2 = red[j];
    in[j] = n2 > 0.0 ? 1.0 / sqrt(n2) : 0.0;
    sub[j] = sqrt(n2) * (j > 0 ? in[j - 1] : 1.0);
  }
  const double *d = red + kHm;  // d[j (kHm + 1) + q]
  for (int j = 0; j < kHm; j++)
    for (int q = 0; q <= j; q++) hc[q][j] = d[j * (kHm + 1) + q] * in[q] * in[j];
  const int m = kHm - 1;
  double left = d[m * (kHm + 1) + kHm] * in[m] * in[m];
  for (int q = 0; q <= m; q++) left -= hc[q][m] * hc[q][m];
  sub[kHm] = left > 0.0 ? sqrt(left) : 0.0;
  h2_lstsq(sub, hc, y);
  for (int q = 0; q < kHm; q++) y[q] *= in[q];
}

// Hessenberg columns from the partials, Givens QR and back substitution
// (one block): the coefficients y[q] of the Z_q, q < kHm (zero past a
// breakdown).  The normalised basis is U_q / n_q, n_q = |U_q|; the last
// subdiagonal entry, the norm of what is left of w, comes from |w|^2 less the
// parts taken out.
constexpr int kNSums = kHm * (kHm + 2);
__global__ __launch_bounds__(64 * kNSums) void k2_solve(const double *__restrict__ p, int nb, double *__restrict__ y)
{
  // p: pn[j], then pd[j][q]; a wave a sum
  __shared__ double red[kNSums];
  const int w = threadIdx.x >> 6;
  double a = 0.0;
  for (int b = threadIdx.x & 63; b < nb; b += 64) a += p[(int64_t)w * nb + b];
  a = wave_total(a);
  if ((threadIdx.x & 63) == 0) red[w] = a;
  __syncthreads();
  if (threadIdx.x == 0) h2_coeffs(red, y);
}

// ---- the whole 2-D correction in one workgroup ------------------------------------
// On a plane of at most kPlaneMax nodes each of the correction's seven launches
// is 4 to 5 us of latency.  One workgroup does all of them: the columns it owns (P
// per thread) stay in registers, the plane being transformed sits in LDS, and
// the global sums are block sums.  k2_plane_q below takes the planes whose axes
// have 16 to 64 points, this kernel those with shorter or longer ones.  What
// bounds it is the latency of some 60 barriers and the LDS round trips of the
// transforms between them: 20 us at 32^2, but 38 (FP32) and 49 us (FP64) at 64^2,
// one CU doing the work.  512 threads (1024 make the barriers dearer: 3 to 6 % of
// a solve at 16^3).  us of a solve with one workgroup and with the launches:
// 16^3 FP64 970 and 1133, 32^3 FP64 941 and 1062, 64 x 32 x 64 mixed 900 and 955;
// 64^3 mixed 1060 and 1010, 64^3 FP64 1145 and 1023.
constexpr int kPlaneMax = 2048, kPlaneT = 512, kPlaneP = kPlaneMax / kPlaneT;
constexpr int kPlanePad = kPlaneMax / 4;  // most lines of a plane (axes of 4 nodes and more): one pad value each

// Radix-4 butterflies on x[0..3] (span 4 q; w1, w2 the forward twiddles), as
// dif_fwd and dit_inv form them.
template <typename T>
__device__ __forceinline__ void bf4_fwd(cpx<T> (&x)[4], cpx<T> w1, cpx<T> w2)
{
  const cpx<T> a0 = {x[0].x + x[2].x, x[0].y + x[2].y}, a1 = {x[1].x + x[3].x, x[1].y + x[3].y};
  const cpx<T> d02 = {x[0].x - x[2].x, x[0].y - x[2].y}, d13 = {x[1].x - x[3].x, x[1].y - x[3].y};
  const cpx<T> a2 = cmul<T>(d02, w1), a3 = cmul<T>({d13.y, -d13.x}, w1);
  x[0] = {a0.x + a1.x, a0.y + a1.y};
  x[1] = cmul<T>({a0.x - a1.x, a0.y - a1.y}, w2);
  x[2] = {a2.x + a3.x, a2.y + a3.y};
  x[3] = cmul<T>({a2.x - a3.x, a2.y - a3.y}, w2);
}

template <typename T>
__device__ __forceinline__ void bf4_inv(cpx<T> (&x)[4], cpx<T> w1, cpx<T> w2)
{
  const cpx<T> W = {w1.x, -w1.y}, V = {w2.x, -w2.y};
  const cpx<T> v1 = cmul<T>(x[1], V), v3 = cmul<T>(x[3], V);
  const cpx<T> a0 = {x[0].x + v1.x, x[0].y + v1.y}, a1 = {x[0].x - v1.x, x[0].y - v1.y};
  const cpx<T> a2 = {x[2].x + v3.x, x[2].y + v3.y}, a3 = {x[2].x - v3.x, x[2].y - v3.y};
  const cpx<T> b2 = cmul<T>(a2, W), wa3 = cmul<T>(a3, W);
  const cpx<T> b3 = {-wa3.y, wa3.x};
  x[0] = {a0.x + b2.x, a0.y + b2.y};
  x[2] = {a0.x - b2.x, a0.y - b2.y};
  x[1] = {a1.x + b3.x, a1.y + b3.y};
  x[3] = {a1.x - b3.x, a1.y - b3.y};
}

// dif_fwd (INV false) or dit_inv over the 2^lB lines at b * ls, elements es
// apart.  ROWS: a wave's threads take consecutive butterflies of a line, else
// the same butterfly of consecutive lines.  The innermost stage (spans of 4,
// or 2 when log2 n is odd) is left to the caller when SKIP is set.
template <typename T, bool ROWS, bool INV, bool SKIP>
__device__ __forceinline__ void plane_fft(cpx<T> *s, int lB, int logn, int ls, int es, const cpx<T> *tw)
{
  const int n = 1 << logn;
  auto radix2 = [&]() {
    const int nb2 = 1 << (lB + logn - 1);
    for (int m = threadIdx.x; m < nb2; m += kPlaneT) {
      const int b = ROWS ? m >> (logn - 1) : m & ((1 << lB) - 1);
      const int r = ROWS ? m & ((n >> 1) - 1) : m >> lB;
      const int i0 = b * ls + 2 * r * es;
      const cpx<T> u = s[i0], v = s[i0 + es];
      s[i0] = {u.x + v.x, u.y + v.y};
      s[i0 + es] = {u.x - v.x, u.y - v.y};
    }
    __syncthreads();
  };
  if (INV && !SKIP && (logn & 1)) radix2();
  // forward stages shrink the span from n, inverse ones grow it back
  for (int lq = INV ? (logn & 1) + (SKIP && !(logn & 1) ? 2 : 0) : logn - 2;
       INV ? lq + 2 <= logn : lq >= (SKIP && !(logn & 1) ? 2 : 0); lq += INV ? 2 : -2) {
    const int q = 1 << lq, step = n >> (lq + 2);
    const int nb4 = 1 << (lB + logn - 2);
    for (int m = threadIdx.x; m < nb4; m += kPlaneT) {
      const int b = ROWS ? m >> (logn - 2) : m & ((1 << lB) - 1);
      const int r = ROWS ? m & ((n >> 2) - 1) : m >> lB;
      const int k = r & (q - 1);
      const int i0 = b * ls + (((r >> lq) << (lq + 2)) + k) * es, dq = q * es;
      cpx<T> x[4] = {s[i0], s[i0 + dq], s[i0 + 2 * dq], s[i0 + 3 * dq]};
      if (INV) bf4_inv<T>(x, tw[k * step], tw[2 * k * step]);
      else bf4_fwd<T>(x, tw[k * step], tw[2 * k * step]);
#pragma unroll
      for (int u = 0; u < 4; u++) s[i0 + u * dq] = x[u];
    }
    __syncthreads();
  }
  if (!INV && !SKIP && (logn & 1)) radix2();
}

template <typename T>
__global__ __launch_bounds__(kPlaneT) void k2_plane(int lx, int ly, int nz, int nzc, const double *__restrict__ part,
                                                    const T *__restrict__ C, T *__restrict__ Z,
                                                    const double *__restrict__ twx, const double *__restrict__ twy,
                                                    Symbol sym, const double *__restrict__ trx,
                                                    const double *__restrict__ try_, const double *__restrict__ trz,
                                                    double *__restrict__ y)
{
  __shared__ cpx<T> s[kPlaneMax + kPlanePad];
  __shared__ cpx<T> tx[kPlanePad / 2], ty[kPlanePad / 2];
  __shared__ double cs[2 * (kPlanePad + 4)];  // cos, sin of the x and y modes
  __shared__ double red[kHm];
  const int nx = 1 << lx, ny = 1 << ly, nxy = 1 << (lx + ly), ls = nx + 1;
  load_twiddles<T>(tx, twx, nx);
  load_twiddles<T>(ty, twy, ny);
  double *csy = cs + 2 * nx;
  for (int t = threadIdx.x; t < 2 * nx; t += kPlaneT) cs[t] = trx[t];
  for (int t = threadIdx.x; t < 2 * ny; t += kPlaneT) csy[t] = try_[t];
  // the kz = 0 symbol's factor at the slot of bit-reversed frequencies (px, py)
  auto factor = [&](int px, int py) { return symbol_factor(sym, bitrev(px, lx), bitrev(py, ly), 0, cs, csy, trz); };
  auto slot = [&](int col) { return (col >> lx) * ls + (col & (nx - 1)); };
  T V[kHm + 1][kPlaneP], w[kPlaneP];
  // r2 = the z-mean of the residual, its own mean removed
  double r2[kPlaneP], a[kHm];
  a[0] = 0.0;
#pragma unroll
  for (int p = 0; p < kPlaneP; p++) {
    const int col = (int)threadIdx.x + kPlaneT * p;
    r2[p] = 0.0;
    if (col < nxy) {
      double t = 0.0;
#pragma unroll 8
      for (int zc = 0; zc < nzc; zc++) t += part[(int64_t)zc * nxy + col];
      r2[p] = t;
    }
    a[0] += r2[p];
  }
  block_sums<kHm>(a, 1, red);
  const double inz = 1.0 / (double)nz, mean = red[0] * inz / (double)nxy;
  a[0] = 0.0;
#pragma unroll
  for (int p = 0; p < kPlaneP; p++) {
    const int col = (int)threadIdx.x + kPlaneT * p;
    V[0][p] = col < nxy ? (T)(r2[p] * inz - mean) : (T)0;
    a[0] += (double)V[0][p] * (double)V[0][p];
  }
  double sub[kHm + 1], hc[kHm][kHm];
#pragma unroll
  for (int j = 0; j < kHm; j++) {
    block_sums<kHm>(a, 1, red);
    sub[j] = sqrt(red[0]);
    const double inv = sub[j] > 0.0 ? 1.0 / sub[j] : 0.0;
#pragma unroll
    for (int p = 0; p < kPlaneP; p++) {
      const int col = (int)threadIdx.x + kPlaneT * p;
      V[j][p] = (T)((double)V[j][p] * inv);
      if (col < nxy) s[slot(col)] = {V[j][p], (T)0};
    }
    __syncthreads();
    // Z_j = F2 V_j
    plane_fft<T, true, false, false>(s, ly, lx, ls, 1, tx);
    plane_fft<T, false, false, true>(s, lx, ly, 1, ls, ty);
    // the innermost stages of both y transforms touch the same values: the last
    // forward one, the symbol and the first inverse one in registers
    if (ly & 1) {
      for (int m = threadIdx.x; m < nxy / 2; m += kPlaneT) {
        const int px = m & (nx - 1), r = m >> lx, i0 = px + 2 * r * ls;
        const cpx<T> u = s[i0], v = s[i0 + ls];
        const double f0 = factor(px, 2 * r), f1 = factor(px, 2 * r + 1);
        const cpx<T> a0 = {(T)((double)(u.x + v.x) * f0), (T)((double)(u.y + v.y) * f0)};
        const cpx<T> a1 = {(T)((double)(u.x - v.x) * f1), (T)((double)(u.y - v.y) * f1)};
        s[i0] = {a0.x + a1.x, a0.y + a1.y};
        s[i0 + ls] = {a0.x - a1.x, a0.y - a1.y};
      }
    } else {
      const cpx<T> one = ty[0];
      for (int m = threadIdx.x; m < nxy / 4; m += kPlaneT) {
        const int px = m & (nx - 1), r = m >> lx, i0 = px + 4 * r * ls;
        cpx<T> x[4];
#pragma unroll
        for (int u = 0; u < 4; u++) x[u] = s[i0 + u * ls];
        bf4_fwd<T>(x, one, one);
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const double f = factor(px, 4 * r + u);
          x[u] = {(T)((double)x[u].x * f), (T)((double)x[u].y * f)};
        }
        bf4_inv<T>(x, one, one);
#pragma unroll
        for (int u = 0; u < 4; u++) s[i0 + u * ls] = x[u];
      }
    }
    __syncthreads();
    plane_fft<T, false, true, true>(s, lx, ly, 1, ls, ty);
    plane_fft<T, true, true, false>(s, ly, lx, ls, 1, tx);
    // w = A2 Z_j less its parts along V_0 .. V_j (one classical Gram-Schmidt
    // pass, as in k2_dir)
#pragma unroll
    for (int p = 0; p < kPlaneP; p++) {
      const int col = (int)threadIdx.x + kPlaneT * p;
      w[p] = (T)0;
      if (col < nxy) {
        const int i = col & (nx - 1), jy = col >> lx;
        const int xs[3] = {(i - 1) & (nx - 1), i, (i + 1) & (nx - 1)};
        const int ys[3] = {(jy - 1) & (ny - 1), jy, (jy + 1) & (ny - 1)};
        double acc = 0.0;
#pragma unroll
        for (int o = 0; o < 9; o++) acc += (double)C[o * nxy + col] * (double)s[ys[o / 3] * ls + xs[o % 3]].x;
        w[p] = (T)acc;
        Z[j * nxy + col] = s[slot(col)].x;
      }
    }
#pragma unroll
    for (int q = 0; q <= j; q++) {
      a[q] = 0.0;
#pragma unroll
      for (int p = 0; p < kPlaneP; p++) a[q] += (double)V[q][p] * (double)w[p];
    }
    block_sums<kHm>(a, j + 1, red);
#pragma unroll
    for (int q = 0; q <= j; q++) hc[q][j] = red[q];
#pragma unroll
    for (int p = 0; p < kPlaneP; p++) {
      double x = (double)w[p];
#pragma unroll
      for (int q = 0; q <= j; q++) x -= hc[q][j] * (double)V[q][p];
      w[p] = (T)x;
    }
    a[0] = 0.0;
#pragma unroll
    for (int p = 0; p < kPlaneP; p++) {
      V[j + 1][p] = w[p];
      a[0] += (double)w[p] * (double)w[p];
    }
  }
  block_sums<kHm>(a, 1, red);
  sub[kHm] = sqrt(red[0]);
  if (threadIdx.x == 0) h2_lstsq(sub, hc, y);
}

// The same on planes whose axes have 16, 32 or 64 points (NX = THX RX, NY = THY
// RY), with the four-step transforms in registers: a line's threads are lanes of
// one wave, so the transforms themselves need no barrier, only the turn from
// rows to columns does; the basis is unnormalised, as in the launches below, so
// that three block sums do; the 2-D coefficients and the symbol are loaded and
// made once.  LDS: the plane as rows (SX apart) or as columns (SY apart), with
// room for a line's exchange in its own place.  us, k2_plane -> here: 16^2 FP64
// 14.9 -> 9.7, 32^2 FP64 20.4 -> 15.7 and FP32 18.4 -> 14.2, 64 x 32 FP64 27.9 ->
// 21.4; a solve on 32^3 FP64 885 -> 820, on 16^3 FP64 908 -> 845.  (64^2 took 59
// and 42 us, more than the launches' 31: it spills.)
template <typename T, int THX, int RX, int THY, int RY>
__global__ __launch_bounds__((std::min(512, std::max(64, THX * RX * THY * RY / 4))))
void k2_plane_q(int nz, int nzc, const double *__restrict__ part, const T *__restrict__ C, T *__restrict__ Z,
                const double *__restrict__ twx, const double *__restrict__ twy, Symbol sym,
                const double *__restrict__ trx, const double *__restrict__ try_, const double *__restrict__ trz,
                double *__restrict__ y)
{
  constexpr int NX = THX * RX, NY = THY * RY, NXY = NX * NY;
  constexpr int NT = NXY / 4 < 64 ? 64 : NXY / 4 > 512 ? 512 : NXY / 4, P = NXY / NT, NW = NT / 64;
  constexpr int SX = (RX * (THX + 1) > NX ? RX * (THX + 1) : NX) | 1;
  constexpr int SY = (RY * (THY + 1) > NY ? RY * (THY + 1) : NY) | 1;
  constexpr int L = NY * SX > NX * SY ? NY * SX : NX * SY, kN = kHm + 2;
  static_assert(NY * THX <= NT && NX * THY <= NT, "a thread's share of a line fits");
  constexpr bool kKeepC = P * 9 * (int)sizeof(T) <= 320;  // the coefficients in registers (at most 80)
  __shared__ T pre[L], pim[L];
  __shared__ cpx<T> tx[NX / 2], ty[NY / 2];
  __shared__ double sums[2][NW][kN];
  const int t = (int)threadIdx.x, lane = t & 63, wid = t >> 6;
  // block-wide sums of v[0 .. n): every thread adds the waves' sums in the same order
  int flip = 0;
  auto block_sum = [&](double *v, int n) {
#pragma unroll
    for (int q = 0; q < kN; q++) {
      if (q < n) {
        const double w = wave_total(v[q]);
        if (lane == 0) sums[flip][wid][q] = w;
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kN; q++) {
      if (q < n) {
        double x = 0.0;
#pragma unroll
        for (int w = 0; w < NW; w++) x += sums[flip][w][q];
        v[q] = x;
      }
    }
    flip ^= 1;
  };
  T U[kHm][P], Ck[kKeepC ? P : 1][9], w[P];
  double r2[P], v[kN];
  v[0] = 0.0;
#pragma unroll
  for (int p = 0; p < P; p++) r2[p] = 0.0;
#pragma unroll 4
  for (int zc = 0; zc < nzc; zc++) {
#pragma unroll
    for (int p = 0; p < P; p++) r2[p] += part[(int64_t)zc * NXY + t + NT * p];
  }
  if constexpr (kKeepC) {
#pragma unroll
    for (int p = 0; p < P; p++)
#pragma unroll
      for (int o = 0; o < 9; o++) Ck[p][o] = C[o * NXY + t + NT * p];
  }
  load_twiddles<T>(tx, twx, NX);
  load_twiddles<T>(ty, twy, NY);
  // the thread's lines: row t / THX, its elements j + THX m; column kx = t / THY
  const int row = t / THX, jx = t % THX, kx = t / THY, jy = t % THY;
  const bool xl = t < NY * THX, yl = t < NX * THY;
  double f[RY];  // the kz = 0 symbol's factors at the thread's (kx, ky)
#pragma unroll
  for (int m = 0; m < RY; m++) f[m] = yl ? symbol_factor(sym, kx, jy + THY * m, 0, trx, try_, trz) : 0.0;
#pragma unroll
  for (int p = 0; p < P; p++) v[0] += r2[p];
  block_sum(v, 1);
  const double inz = 1.0 / (double)nz, mean = v[0] * inz / (double)NXY;
#pragma unroll
  for (int p = 0; p < P; p++) U[0][p] = (T)(r2[p] * inz - mean);
  double red[kNSums];
#pragma unroll
  for (int j = 0; j < kHm; j++) {
    // Z_j = F2 U_j
#pragma unroll
    for (int p = 0; p < P; p++) pre[(t + NT * p) / NX * SX + (t + NT * p) % NX] = U[j][p];
    __syncthreads();
    {
      cpx<T> a[RX];
      if (xl) {
#pragma unroll
        for (int m = 0; m < RX; m++) a[m] = {pre[row * SX + jx + THX * m], (T)0};
        wave_sync();
        fft_line<T, false, THX, RX, true>(a, jx, pre, pim, row * SX, tx);
      }
      __syncthreads();
      if (xl) {
#pragma unroll
        for (int m = 0; m < RX; m++) {
          pre[(jx + THX * m) * SY + row] = a[m].x;
          pim[(jx + THX * m) * SY + row] = a[m].y;
        }
      }
      __syncthreads();
    }
    {
      cpx<T> a[RY];
      if (yl) {
#pragma unroll
        for (int m = 0; m < RY; m++) a[m] = {pre[kx * SY + jy + THY * m], pim[kx * SY + jy + THY * m]};
        wave_sync();
        fft_line<T, false, THY, RY, true>(a, jy, pre, pim, kx * SY, ty);
#pragma unroll
        for (int m = 0; m < RY; m++) a[m] = {(T)((double)a[m].x * f[m]), (T)((double)a[m].y * f[m])};
        fft_line<T, true, THY, RY, true>(a, jy, pre, pim, kx * SY, ty);
      }
      __syncthreads();
      if (yl) {
#pragma unroll
        for (int m = 0; m < RY; m++) {
          pre[(jy + THY * m) * SX + kx] = a[m].x;
          pim[(jy + THY * m) * SX + kx] = a[m].y;
        }
      }
      __syncthreads();
    }
    if (xl) {
      cpx<T> a[RX];
#pragma unroll
      for (int m = 0; m < RX; m++) a[m] = {pre[row * SX + jx + THX * m], pim[row * SX + jx + THX * m]};
      wave_sync();
      fft_line<T, true, THX, RX, true>(a, jx, pre, pim, row * SX, tx);
#pragma unroll
      for (int m = 0; m < RX; m++) pre[row * SX + jx + THX * m] = a[m].x;
    }
    __syncthreads();
    // w = A2 Z_j and its products with U_0 .. U_j
#pragma unroll
    for (int q = 0; q < kN; q++) v[q] = 0.0;
#pragma unroll
    for (int p = 0; p < P; p++) {
      const int col = t + NT * p, i = col % NX, r = col / NX;
      const int xs[3] = {(i - 1) & (NX - 1), i, (i + 1) & (NX - 1)};
      const int ys[3] = {((r - 1) & (NY - 1)) * SX, r * SX, ((r + 1) & (NY - 1)) * SX};
      double acc = 0.0;
#pragma unroll
      for (int o = 0; o < 9; o++)
        acc += (double)(kKeepC ? Ck[kKeepC ? p : 0][o] : C[o * NXY + col]) * (double)pre[ys[o / 3] + xs[o % 3]];
      w[p] = (T)acc;
      Z[j * NXY + col] = pre[r * SX + i];
#pragma unroll
      for (int q = 0; q <= j; q++) v[q] += (double)U[q][p] * (double)w[p];
      v[kHm] += (double)w[p] * (double)w[p];
      v[kHm + 1] += (double)U[j][p] * (double)U[j][p];
    }
    block_sum(v, kN);  // (its barrier also ends the reads of the plane)
    red[j] = v[kHm + 1];
#pragma unroll
    for (int q = 0; q <= kHm; q++) red[kHm + j * (kHm + 1) + q] = v[q];
    if (j + 1 < kHm) {
#pragma unroll
      for (int p = 0; p < P; p++) {
        double x = (double)w[p];
#pragma unroll
        for (int q = 0; q <= j; q++)
          if (red[q] > 0.0) x -= v[q] / red[q] * (double)U[q][p];
        U[j + 1 < kHm ? j + 1 : 0][p] = (T)x;
      }
    }
  }
  if (t == 0) h2_coeffs(red, y);
}

// Planes that k2_plane_q takes
static bool plane_q(int nx, int ny)
{
  auto axis = [](int n) { return n == 16 || n == 32 || n == 64; };
  return axis(nx) && axis(ny) && nx * ny <= kPlaneMax;
}

// z[k * nxy + col] += sum_q y_q Z_q[col] over kExtZ planes per block
template <typename T>
__global__ __launch_bounds__(256) void k2_ext(int64_t nxy, int nz, const T *__restrict__ Z, const double *__restrict__ y,
                                              T *__restrict__ z)
{
  const int64_t col = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= nxy) return;
  double e = 0.0;
#pragma unroll
  for (int q = 0; q < kHm; q++) e += y[q] * (double)Z[(int64_t)q * nxy + col];
  const int k0 = blockIdx.y * kExtZ;
  T v[kExtZ];
#pragma unroll
  for (int u = 0; u < kExtZ; u++)
    if (k0 + u < nz) v[u] = z[(int64_t)(k0 + u) * nxy + col];
#pragma unroll
  for (int u = 0; u < kExtZ; u++)
    if (k0 + u < nz) z[(int64_t)(k0 + u) * nxy + col] = (T)((double)v[u] + e);
}

// Lines per block of a 2-D pass: at least 64 blocks when there are lines enough
template <typename T>
static int fft2_batch(int n, int64_t lines)
{
  return fft_batch<T>(n, std::max<int64_t>(1, lines / 64));
}

template <typename T>
int fft2_pc_apply(chy_ctx *ctx, const double v19[19], const T *r, T *z, T *w3, bool zline, bool *zline_done)
{
  if (zline_done) *zline_done = false;
  TRY(fft_pc_apply<T>(ctx, v19, r, z));
  if (ctx->solve_transpose) return CHY_OK;  // the correction is built for A(n), not its transpose
  // the z-line stage fused with the correction: the column-sum pass also keeps
  // r - A(n) z in w3 for it, and e2 is added by the stage itself
  const bool fused = zline && w3 && ctx->zl_buf && zline_e2_applies(ctx);
  const int nx = ctx->g.nx, ny = ctx->g.ny, nz = ctx->g.nz;
  const int64_t nxy = (int64_t)nx * ny;
  T *C = (T *)ctx->pc2_buf, *U = C + 9 * nxy, *Z = U + kFft2Its * nxy, *w = Z + kFft2Its * nxy;
  cpx<T> *cb = (cpx<T> *)(w + nxy);
  const H2 h = h2_layout(ctx, sizeof(T) == 4);
  const int nb = h.nb, nzc = lhs_zchunks(ctx->g, sizeof(T) == 4);
  // z-averaged residual of the first level
  launch_lhs_zsum<T>(ctx, ctx->prm.lhs_type, (const T *)ctx->mom[0], z, r, h.part, h.pl, fused ? w3 : nullptr);
  Symbol sym = make_symbol(ctx, v19);
  sym.inv_scale = 1.0 / (double)nxy;
  if (plane_q(nx, ny)) {
#define PLANE(THX, RX, THY, RY)                                                                                       \
  hipLaunchKernelGGL((k2_plane_q<T, THX, RX, THY, RY>), 1, std::min(512, std::max(64, nx * ny / 4)), 0, ctx->stream, nz, \
                     nzc, (const double *)h.part, (const T *)C, Z, ctx->tw[0], ctx->tw[1], sym, ctx->trig[0],          \
                     ctx->trig[1], ctx->trig[2], h.y)
#define PLANE_X(THY, RY)                          \
  do {                                            \
    if (nx == 16) PLANE(4, 4, THY, RY);           \
    else if (nx == 32) PLANE(4, 8, THY, RY);      \
    else if constexpr (THY * RY < 64) PLANE(8, 8, THY, RY); \
  } while (0)
    if (ny == 16) PLANE_X(4, 4);
    else if (ny == 32) PLANE_X(4, 8);
    else PLANE_X(8, 8);
#undef PLANE_X
#undef PLANE
  } else if (nxy <= kPlaneMax) {
    hipLaunchKernelGGL((k2_plane<T>), 1, kPlaneT, 0, ctx->stream, ilog2(nx), ilog2(ny), nz,
                       nzc, (const double *)h.part, (const T *)C, Z, ctx->tw[0],
                       ctx->tw[1], sym, ctx->trig[0], ctx->trig[1], ctx->trig[2], h.y);
  } else {
    const int R = ny / nb, lx = ilog2(nx);
    const size_t lds = fft_lds<T>(nx, R + 2);
    const int By = fft2_batch<T>(ny, nx);
    for (int j = 0; j < kFft2Its; j++) {
      T *Zj = Z + (int64_t)j * nxy;
#define DIR(FIRST)                                                                                                  \
  hipLaunchKernelGGL((k2_dir<T, FIRST>), nb, 256, fft_lds<T>(nx, R), ctx->stream, lx, R, nxy, j, nz, nzc,           \
                     (const double *)h.part, (const double *)h.pl, h.nlb, U, (const T *)w, cb, ctx->tw[0], h.pn,    \
                     (const double *)h.pd)
      if (j == 0) DIR(true);
      else DIR(false);
#undef DIR
      // 2-D FFT solve with the kz = 0 symbol: along y
      hipLaunchKernelGGL((k_fft_s<T, 3>), (unsigned)(nx / By), kBlock, fft_lds<T>(ny, By), ctx->stream, ilog2(ny),
                         (int64_t)nx, (int64_t)nx, (int64_t)0, By, cb, ctx->tw[1], sym, ctx->trig[0], ctx->trig[1],
                         ctx->trig[2]);
      if (lds <= 65536) {
        hipLaunchKernelGGL((k2_apply<T, true>), nb, 256, lds, ctx->stream, lx, R, ny, j, (const T *)C,
                           (const cpx<T> *)cb, ctx->tw[0], Zj, (const T *)U, w, h.pd);
      } else {
        const int Bx = fft2_batch<T>(nx, ny);
        hipLaunchKernelGGL((k2_inv_x<T>), (unsigned)((ny + Bx - 1) / Bx), 256, fft_lds<T>(nx, Bx), ctx->stream, lx, ny,
                           Bx, Zj, (const cpx<T> *)cb, ctx->tw[0]);
        hipLaunchKernelGGL((k2_apply<T, false>), nb, 256, 0, ctx->stream, lx, R, ny, j, (const T *)C,
                           (const cpx<T> *)cb, ctx->tw[0], Zj, (const T *)U, w, h.pd);
      }
    }
    hipLaunchKernelGGL(k2_solve, 1, 64 * kNSums, 0, ctx->stream, (const double *)h.pn, nb, h.y);
  }
  if (fused) {
    launch_zline_apply_e2<T>(ctx, (const T *)ctx->zl_buf, ctx->zl_col, w3, z, (const T *)ctx->mom[0], (const T *)Z,
                             (const double *)h.y);
    if (zline_done) *zline_done = true;
  } else {
    hipLaunchKernelGGL((k2_ext<T>), dim3((unsigned)((nxy + 255) / 256), (unsigned)((nz + kExtZ - 1) / kExtZ)), 256,
                       0, ctx->stream, nxy, nz, (const T *)Z, (const double *)h.y, z);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_err(ctx, CHY_ERR_LIB, std::string("fft2: ") + hipGetErrorString(e));
  return CHY_OK;
}

template int fft2_pc_apply<double>(chy_ctx *, const double *, const double *, double *, double *, bool, bool *);
template int fft2_pc_apply<float>(chy_ctx *, const double *, const float *, float *, float *, bool, bool *);

template int fft_pc_apply<double>(chy_ctx *, const double *, const double *, double *);
template int fft_pc_apply<float>(chy_ctx *, const double *, const float *, float *);

}  // namespace chy
