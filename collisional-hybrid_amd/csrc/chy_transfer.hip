// chy_transfer.hip -- host arrays in and out of the device.
//
// The ABI's arrays are interleaved f64 (moments {n, Gx, Gy, Gz} per node,
// positions and velocities {x, y, z, r} per ion); the device keeps one array
// per field, FP32 in mixed mode.  The layouts change on the device, in scratch
// memory: a call moves the caller's bytes once across the bus and touches them
// nowhere else.  On the host the strided loops and large copies took, in ms
// (then -> now): set_moments 7.8 -> 2.3 and get_moments 13.3 -> 2.3 at 128^3 FP64,
// 110 -> 18 and 255 -> 17 at 256^3 mixed, get_potential there 13.3 -> 4.6; setting
// 700,001 ions 10.8 -> 5.8, getting them 17.4 -> 10.1.
#include <algorithm>
#include <cstring>
#include <memory>
#include <new>
#include <system_error>
#include <thread>

#include "chy_internal.h"

namespace chy {

// Device scratch for `bytes` of a layout change, less when the caller's loop
// has to take several pieces: the Krylov basis, which holds nothing between
// solves, or for many ions on a small grid a buffer of at most kStageBytes that
// the context then keeps (the basis again, in small pieces, where the device
// has no memory left for one).
static int stage_get(chy_ctx *ctx, size_t bytes, void **p, size_t *got)
{
  constexpr size_t kEnough = (size_t)16 << 20;
  if (ctx->V_bytes >= std::min(bytes, kEnough)) {
    *p = ctx->V;
    *got = ctx->V_bytes;
    return CHY_OK;
  }
  const size_t want = std::min(bytes, kStageBytes);
  if (ctx->stage_bytes < want) {
    if (ctx->stage) (void)hipFree(ctx->stage);
    ctx->stage = nullptr;
    ctx->stage_bytes = 0;
    if (hipMalloc(&ctx->stage, want) == hipSuccess) {
      ctx->stage_bytes = want;
    } else {
      ctx->stage = nullptr;
      (void)hipGetLastError();
      *p = ctx->V;
      *got = ctx->V_bytes;
      return CHY_OK;
    }
  }
  *p = ctx->stage;
  *got = ctx->stage_bytes;
  return CHY_OK;
}

void transfer_release(chy_ctx *ctx)
{
  if (ctx->stage) (void)hipFree(ctx->stage);
  if (ctx->pin) (void)hipHostFree(ctx->pin);
  for (hipEvent_t &e : ctx->pin_ev)
    if (e) { (void)hipEventDestroy(e); e = nullptr; }
  ctx->stage = nullptr;
  ctx->pin = nullptr;
}

// Large copies to the host: a pageable destination whose pages are mostly new
// to the process takes 10 GB/s from hipMemcpy, bound by one thread's page
// faults and copies.  kPinThreads threads take alternate chunks: each enqueues
// its chunk on the context's stream into its own pinned buffer, waits for it
// and copies it on while the others' chunks cross the bus.  From 16 MB on: the
// pinned buffers cost a context 1.2 ms once and the threads 0.1 ms a copy, which
// 8 MB (0.50 ms plain, 0.38 pinned) earn back after ten copies, 128 MB (13.3 and
// 4.6 ms) at once.
int copy_to_host(chy_ctx *ctx, void *dst, const void *src, size_t bytes)
{
  constexpr size_t kMin = (size_t)16 << 20;
  bool pinned = bytes >= kMin;
  if (pinned && !ctx->pin) {
    bool ok = hipHostMalloc(&ctx->pin, kPinThreads * kPinChunk) == hipSuccess;
    for (hipEvent_t &e : ctx->pin_ev) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (!ok) {  // no pinned memory to be had: the plain copy
      if (ctx->pin) (void)hipHostFree(ctx->pin);
      ctx->pin = nullptr;
      for (hipEvent_t &e : ctx->pin_ev)
        if (e) { (void)hipEventDestroy(e); e = nullptr; }
      (void)hipGetLastError();
      pinned = false;
    }
  }
  if (!pinned) {
    // the blocking copy: an asynchronous one and a wait for the stream take 21 us
    // for 4 KB, this 13; they are level from 32 KB on
    CHY_HIP(hipMemcpyWithStream(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    return CHY_OK;
  }
  hipError_t err[kPinThreads];
  auto work = [&](int t) {
    unsigned char *buf = (unsigned char *)ctx->pin + t * kPinChunk;
    hipError_t e = hipSetDevice(ctx->device);
    for (size_t o = t * kPinChunk; e == hipSuccess && o < bytes; o += kPinThreads * kPinChunk) {
      const size_t n = std::min(kPinChunk, bytes - o);
      e = hipMemcpyAsync(buf, (const unsigned char *)src + o, n, hipMemcpyDeviceToHost, ctx->stream);
      if (e == hipSuccess) e = hipEventRecord(ctx->pin_ev[t], ctx->stream);
      if (e == hipSuccess) e = hipEventSynchronize(ctx->pin_ev[t]);
      if (e == hipSuccess) memcpy((unsigned char *)dst + o, buf, n);
    }
    err[t] = e;
  };
  std::thread th[kPinThreads];
  for (int t = 1; t < kPinThreads; t++) {
    try {
      th[t] = std::thread(work, t);
    } catch (const std::system_error &) {  // no thread to be had: this one's chunks are done below
    }
  }
  work(0);
  for (int t = 1; t < kPinThreads; t++) {
    if (th[t].joinable()) th[t].join();
    else work(t);
  }
  for (hipError_t e : err) CHY_HIP(e);
  return CHY_OK;
}

// {n, Gx, Gy, Gz} of nodes [c0, c0 + n) from or to the four moment arrays
template <typename T>
__global__ __launch_bounds__(256) void k_moments_in(int64_t n, const Vec4<double> *__restrict__ s, T *__restrict__ a,
                                                    T *__restrict__ b, T *__restrict__ c, T *__restrict__ d)
{
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const Vec4<double> v = s[i];
  a[i] = (T)v.x; b[i] = (T)v.y; c[i] = (T)v.z; d[i] = (T)v.w;
}

template <typename T>
__global__ __launch_bounds__(256) void k_moments_out(int64_t n, const T *__restrict__ a, const T *__restrict__ b,
                                                     const T *__restrict__ c, const T *__restrict__ d,
                                                     Vec4<double> *__restrict__ s)
{
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  s[i] = Vec4<double>{(double)a[i], (double)b[i], (double)c[i], (double)d[i]};
}

template <typename T>
static int moments_copy(chy_ctx *ctx, double *v, bool in)
{
  const int64_t nc = ctx->g.nc;
  void *st;
  size_t got;
  TRY(stage_get(ctx, sizeof(double) * 4 * (size_t)nc, &st, &got));
  const int64_t per = (int64_t)(got / (4 * sizeof(double)));
  T *m[4];
  for (int64_t c0 = 0; c0 < nc; c0 += per) {
    const int64_t n = std::min(per, nc - c0);
    for (int a = 0; a < 4; a++) m[a] = (T *)ctx->mom[a] + c0;
    const unsigned nb = (unsigned)((n + 255) / 256);
    const size_t bytes = sizeof(double) * 4 * (size_t)n;
    if (in) {
      CHY_HIP(hipMemcpyAsync(st, v + 4 * c0, bytes, hipMemcpyHostToDevice, ctx->stream));
      hipLaunchKernelGGL((k_moments_in<T>), nb, 256, 0, ctx->stream, n, (const Vec4<double> *)st, m[0], m[1], m[2], m[3]);
    } else {
      hipLaunchKernelGGL((k_moments_out<T>), nb, 256, 0, ctx->stream, n, (const T *)m[0], (const T *)m[1],
                         (const T *)m[2], (const T *)m[3], (Vec4<double> *)st);
      TRY(copy_to_host(ctx, v + 4 * c0, st, bytes));
    }
  }
  CHY_HIP(hipGetLastError());
  if (in) CHY_HIP(hipStreamSynchronize(ctx->stream));  // (copies to the host are complete)
  return CHY_OK;
}

int moments_upload(chy_ctx *ctx, const double *v)
{
  return ctx->mixed ? moments_copy<float>(ctx, const_cast<double *>(v), true)
                    : moments_copy<double>(ctx, const_cast<double *>(v), true);
}

int moments_download(chy_ctx *ctx, double *v)
{
  return ctx->mixed ? moments_copy<float>(ctx, v, false) : moments_copy<double>(ctx, v, false);
}

// ---- ions ------------------------------------------------------------------
// Ion base + i of the caller's arrays (positions wrapped into [p0, p1) as the
// move does); pid null: the caller's index.
__global__ __launch_bounds__(256) void k_ions_in_fp64(Grid g, int64_t n, int64_t base, const Vec4<double> *__restrict__ pos,
                                                      const Vec4<double> *__restrict__ vel,
                                                      const uint32_t *__restrict__ pid, PState<double> st)
{
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const Vec4<double> p = pos[i], v = vel[i];
  const int64_t q = base + i;
  st.x[q] = wrap_pos(p.x, g.p0[0], g.p1[0], g.L[0]);
  st.y[q] = wrap_pos(p.y, g.p0[1], g.p1[1], g.L[1]);
  st.z[q] = wrap_pos(p.z, g.p0[2], g.p1[2], g.L[2]);
  st.vx[q] = v.x; st.vy[q] = v.y; st.vz[q] = v.z;
  st.pid[q] = pid ? pid[i] : (uint32_t)q;
}

__global__ __launch_bounds__(256) void k_ions_in_mixed(Grid g, int64_t n, int64_t base, const Vec4<double> *__restrict__ pos,
                                                       const Vec4<double> *__restrict__ vel,
                                                       const double *__restrict__ w, const uint32_t *__restrict__ pid,
                                                       PState<float> st)
{
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const Vec4<double> p = pos[i], v = vel[i];
  const double x[3] = {p.x, p.y, p.z};
  const int nn[3] = {g.nx, g.ny, g.nz};
  int ci[3];
  float o[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    double f;
    cell_coord(wrap_pos(x[a], g.p0[a], g.p1[a], g.L[a]), g.p0[a], g.d[a], g.rd[a], nn[a], ci[a], f);
    o[a] = (float)f;
    if (o[a] >= 1.0f) { o[a] = 0.0f; ci[a] = ci[a] + 1 == nn[a] ? 0 : ci[a] + 1; }
  }
  const int64_t q = base + i;
  st.pos[q] = Vec4<float>{o[0], o[1], o[2], w ? (float)w[i] : 1.0f};
  st.vel[q] = Vec4<float>{(float)v.x, (float)v.y, (float)v.z, __uint_as_float(pid ? pid[i] : (uint32_t)q)};
  st.cell[q] = ci[0] + g.nx * (ci[1] + g.ny * ci[2]);
}

// Ions base .. base + n - 1 as {x, y, z, |x|} and {vx, vy, vz, |v|}
__global__ __launch_bounds__(256) void k_ions_out_fp64(int64_t n, int64_t base, PState<double> st,
                                                       Vec4<double> *__restrict__ pos, Vec4<double> *__restrict__ vel)
{
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int64_t q = base + i;
  const double x = st.x[q], y = st.y[q], z = st.z[q], a = st.vx[q], b = st.vy[q], c = st.vz[q];
  pos[i] = Vec4<double>{x, y, z, sqrt(x * x + y * y + z * z)};
  vel[i] = Vec4<double>{a, b, c, sqrt(a * a + b * b + c * c)};
}

__global__ __launch_bounds__(256) void k_ions_out_mixed(Grid g, int64_t n, int64_t base, PState<float> st,
                                                        Vec4<double> *__restrict__ pos, Vec4<double> *__restrict__ vel,
                                                        double *__restrict__ w, uint32_t *__restrict__ pid)
{
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int64_t q = base + i;
  int ci, cj, ck;
  split_cell(g, st.cell[q], ci, cj, ck);
  const Vec4<float> p = st.pos[q], v = st.vel[q];
  const double x = g.p0[0] + ((double)ci + (double)p.x) * g.d[0], y = g.p0[1] + ((double)cj + (double)p.y) * g.d[1],
               z = g.p0[2] + ((double)ck + (double)p.z) * g.d[2];
  const double a = (double)v.x, b = (double)v.y, c = (double)v.z;
  pos[i] = Vec4<double>{x, y, z, sqrt(x * x + y * y + z * z)};
  vel[i] = Vec4<double>{a, b, c, sqrt(a * a + b * b + c * c)};
  w[i] = (double)p.w;
  pid[i] = __float_as_uint(v.w);
}

// A chunk of the staging buffer: n ions' positions, velocities, weights, ids
struct IonStage {
  int64_t per;
  Vec4<double> *pos, *vel;
  double *w;
  uint32_t *pid;
};

constexpr size_t kIon = 2 * sizeof(Vec4<double>) + sizeof(double) + sizeof(uint32_t);

static int ion_stage(chy_ctx *ctx, int64_t np, IonStage &s)
{
  void *st;
  size_t got;
  TRY(stage_get(ctx, kIon * (size_t)np, &st, &got));
  s.per = std::max<int64_t>(1, std::min<int64_t>(np, (int64_t)(got / kIon)));
  s.pos = (Vec4<double> *)st;
  s.vel = s.pos + s.per;
  s.w = (double *)(s.vel + s.per);
  s.pid = (uint32_t *)(s.w + s.per);
  return CHY_OK;
}

int ions_upload(chy_ctx *ctx, int64_t np, const double *pos, const double *vel, const double *w, const uint32_t *pid)
{
  IonStage s;
  TRY(ion_stage(ctx, np, s));
  for (int64_t i0 = 0; i0 < np; i0 += s.per) {
    const int64_t n = std::min(s.per, np - i0);
    const unsigned nb = (unsigned)((n + 255) / 256);
    CHY_HIP(hipMemcpyAsync(s.pos, pos + 4 * i0, sizeof(Vec4<double>) * n, hipMemcpyHostToDevice, ctx->stream));
    CHY_HIP(hipMemcpyAsync(s.vel, vel + 4 * i0, sizeof(Vec4<double>) * n, hipMemcpyHostToDevice, ctx->stream));
    if (pid) CHY_HIP(hipMemcpyAsync(s.pid, pid + i0, sizeof(uint32_t) * n, hipMemcpyHostToDevice, ctx->stream));
    const uint32_t *dpid = pid ? s.pid : nullptr;
    if (ctx->mixed) {
      if (w) CHY_HIP(hipMemcpyAsync(s.w, w + i0, sizeof(double) * n, hipMemcpyHostToDevice, ctx->stream));
      hipLaunchKernelGGL(k_ions_in_mixed, nb, 256, 0, ctx->stream, ctx->g, n, i0, (const Vec4<double> *)s.pos,
                         (const Vec4<double> *)s.vel, w ? (const double *)s.w : nullptr, dpid, ctx->pf[ctx->cur]);
    } else {
      hipLaunchKernelGGL(k_ions_in_fp64, nb, 256, 0, ctx->stream, ctx->g, n, i0, (const Vec4<double> *)s.pos,
                         (const Vec4<double> *)s.vel, dpid, ctx->pd[ctx->cur]);
    }
  }
  if (!ctx->mixed && w)
    CHY_HIP(hipMemcpyAsync(ctx->pd[ctx->cur].w, w, sizeof(double) * np, hipMemcpyHostToDevice, ctx->stream));
  CHY_HIP(hipGetLastError());
  CHY_HIP(hipStreamSynchronize(ctx->stream));  // the caller's arrays are his again
  return CHY_OK;
}

// The staged arrays (all ions in one piece) that are wanted in one copy, where
// there are several and all of them together take at most kMost: a copy and its
// wait are some 20 us whatever they move.  us for all four weighted mixed arrays,
// a copy each -> one: 300 ions 82 -> 24, 3000 65 -> 33, 6800 66 -> 49; at 7000
// they would be level soon.  (FP64 weights and ids are not staged.)
static int ions_small(chy_ctx *ctx, const IonStage &s, double *pos, double *vel, double *w, uint32_t *pid, bool &done)
{
  constexpr size_t kMost = (size_t)512 << 10;
  const size_t n = (size_t)s.per;
  done = false;
  if (kIon * n > kMost || (pos != nullptr) + (vel != nullptr) + (w != nullptr) + (pid != nullptr) < 2) return CHY_OK;
  std::unique_ptr<unsigned char[]> h(new (std::nothrow) unsigned char[kIon * n]);
  if (!h) return CHY_OK;
  TRY(copy_to_host(ctx, h.get(), s.pos, kIon * n));
  auto part = [&](void *dst, const void *dev, size_t bytes) {
    if (dst) memcpy(dst, h.get() + ((const unsigned char *)dev - (const unsigned char *)s.pos), bytes);
  };
  part(pos, s.pos, sizeof(Vec4<double>) * n);
  part(vel, s.vel, sizeof(Vec4<double>) * n);
  part(w, s.w, sizeof(double) * n);
  part(pid, s.pid, sizeof(uint32_t) * n);
  done = true;
  return CHY_OK;
}

int ions_download(chy_ctx *ctx, int64_t np, double *pos, double *vel, double *w, uint32_t *pid)
{
  const bool own_w = ctx->weighted;  // unit weights are filled in below
  if (ctx->mixed || pos || vel) {
    IonStage s;
    TRY(ion_stage(ctx, np, s));
    for (int64_t i0 = 0; i0 < np; i0 += s.per) {
      const int64_t n = std::min(s.per, np - i0);
      const unsigned nb = (unsigned)((n + 255) / 256);
      if (ctx->mixed)
        hipLaunchKernelGGL(k_ions_out_mixed, nb, 256, 0, ctx->stream, ctx->g, n, i0, ctx->pf[ctx->cur], s.pos, s.vel,
                           s.w, s.pid);
      else
        hipLaunchKernelGGL(k_ions_out_fp64, nb, 256, 0, ctx->stream, n, i0, ctx->pd[ctx->cur], s.pos, s.vel);
      bool done = false;
      if (ctx->mixed && n == np) TRY(ions_small(ctx, s, pos, vel, own_w ? w : nullptr, pid, done));
      if (done) break;
      if (pos) TRY(copy_to_host(ctx, pos + 4 * i0, s.pos, sizeof(Vec4<double>) * n));
      if (vel) TRY(copy_to_host(ctx, vel + 4 * i0, s.vel, sizeof(Vec4<double>) * n));
      if (ctx->mixed) {
        if (w && own_w) TRY(copy_to_host(ctx, w + i0, s.w, sizeof(double) * n));
        if (pid) TRY(copy_to_host(ctx, pid + i0, s.pid, sizeof(uint32_t) * n));
      }
    }
  }
  if (!ctx->mixed) {
    if (w && own_w) TRY(copy_to_host(ctx, w, ctx->pd[ctx->cur].w, sizeof(double) * np));
    if (pid) TRY(copy_to_host(ctx, pid, ctx->pd[ctx->cur].pid, sizeof(uint32_t) * np));
  }
  if (w && !own_w) for (int64_t i = 0; i < np; i++) w[i] = 1.0;
  CHY_HIP(hipGetLastError());
  return CHY_OK;
}

}  // namespace chy
