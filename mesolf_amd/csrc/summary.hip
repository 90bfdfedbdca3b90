// Summary image of a sensor movie, 'pixelwise' detrend mode
// (summary_image_generation_module.m:62-96, :130), with the rank-1 background
// of rank_1_factorization.m:31-41 and compute_std_image.m.
//
// The movie is MATLAB column-major [npix, T] single (pixel fastest), so a
// thread per pixel walking the frames reads 64 consecutive pixels per wave
// per frame.  Arithmetic is FP64 on the FP32 samples.
//   mx = max(movie);  x = movie / mx
//   d  = x - movmean(x, window_1)            (pass 1, stored FP32)
//   y  = movmean(d, window_2) .^ poly_index  (pass 2, fused with the sums)
//   img = sqrt(sum(y.^2) / T - mean(y).^2);  summary = img / max(img)
// movmean over the window [j - a, j + b] clipped to [0, T) ('shrink'),
// a = b = (k-1)/2 for odd k, a = k/2, b = k/2 - 1 for even k, kept as a
// running FP64 sum (one sample enters and one leaves per frame; the leaving
// sample is read again, from cache).
#include <algorithm>

#include "internal.h"

namespace mlf {

namespace {

__device__ __forceinline__ double nmax(double a, double b) {
  if (a != a) return b;
  if (b != b) return a;
  return a > b ? a : b;
}

template <typename F>
__device__ double block_reduce(double v, double* sh, F op) {
  for (int off = 32; off > 0; off >>= 1) v = op(v, __shfl_down(v, off, 64));
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  __syncthreads();  // sh may still be read by a previous reduction
  if (lane == 0) sh[wid] = v;
  __syncthreads();
  double r = sh[0];
  for (int k = 1; k < (int)(blockDim.x >> 6); ++k) r = op(r, sh[k]);
  return r;  // every thread
}

constexpr int kThreads = 256;

// per-block maxima of a float array (NaN ignored)
__global__ __launch_bounds__(kThreads) void k_max_f32(const float* __restrict__ a, size_t n,
                                                      double* __restrict__ parts) {
  __shared__ double sh[kThreads / 64];
  double m = __builtin_nan("");
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    m = nmax(m, (double)a[i]);
  m = block_reduce(m, sh, nmax);
  if (threadIdx.x == 0) parts[blockIdx.x] = m;
}

// same over a 16-byte aligned array: n4 float4 and a tail of ntail floats
__global__ __launch_bounds__(kThreads) void k_max_f32x4(const float4* __restrict__ a4, size_t n4,
                                                        const float* __restrict__ tail, int ntail,
                                                        double* __restrict__ parts) {
  __shared__ double sh[kThreads / 64];
  double m = __builtin_nan("");
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n4; i += (size_t)gridDim.x * blockDim.x) {
    const float4 v = a4[i];
    m = nmax(nmax(m, (double)v.x), nmax(nmax((double)v.y, (double)v.z), (double)v.w));
  }
  if (blockIdx.x == 0 && (int)threadIdx.x < ntail) m = nmax(m, (double)tail[threadIdx.x]);
  m = block_reduce(m, sh, nmax);
  if (threadIdx.x == 0) parts[blockIdx.x] = m;
}

// scalar[0] = max of parts (one workgroup)
__global__ __launch_bounds__(kThreads) void k_fold_max(const double* __restrict__ parts, int n,
                                                       double* __restrict__ out) {
  __shared__ double sh[kThreads / 64];
  double m = __builtin_nan("");
  for (int k = threadIdx.x; k < n; k += blockDim.x) m = nmax(m, parts[k]);
  m = block_reduce(m, sh, nmax);
  if (threadIdx.x == 0) *out = m;
}

// rank-1 step 1, t~ = s' * Y: parts[j * nchunk + c] = sum over chunk c of s_i Y_ij.
// A thread keeps the s of its kChunk / kThreads pixels in registers for the
// kTdotFrames frames of its workgroup.
constexpr int kChunk = kThreads * 16;  // pixels per chunk
constexpr int kTdotFrames = 16;
__global__ __launch_bounds__(kThreads) void k_r1_tdot(const float* __restrict__ Y, size_t npix, int T,
                                                      const double* __restrict__ s,
                                                      double* __restrict__ parts) {
  constexpr int kPer = kChunk / kThreads;
  const size_t i0 = (size_t)blockIdx.x * kChunk + threadIdx.x;
  const int nchunk = gridDim.x;
  double sv[kPer];
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const size_t i = i0 + (size_t)q * kThreads;
    sv[q] = i < npix ? s[i] : 0.0;
  }
  // frames in groups of kG: the group's loads are in flight together, one
  // pair of barriers per group
  constexpr int kG = 4;
  __shared__ double shf[kG][kThreads / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  for (int j0 = blockIdx.y * kTdotFrames; j0 < T; j0 += gridDim.y * kTdotFrames) {
    for (int jg = j0; jg < j0 + kTdotFrames && jg < T; jg += kG) {
      const int nf = min(kG, T - jg);
      double acc[kG];
#pragma unroll
      for (int f = 0; f < kG; ++f) acc[f] = 0.0;
#pragma unroll
      for (int q = 0; q < kPer; ++q) {
        const size_t i = i0 + (size_t)q * kThreads;
        if (i >= npix) continue;
#pragma unroll
        for (int f = 0; f < kG; ++f)
          if (f < nf) acc[f] = fma((double)Y[i + (size_t)(jg + f) * npix], sv[q], acc[f]);
      }
#pragma unroll
      for (int f = 0; f < kG; ++f) {
        double v = acc[f];
        for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
        if (lane == 0) shf[f][wid] = v;
      }
      __syncthreads();
      if ((int)threadIdx.x < nf) {
        double r = shf[threadIdx.x][0];
        for (int k = 1; k < kThreads / 64; ++k) r += shf[threadIdx.x][k];
        parts[(size_t)(jg + threadIdx.x) * nchunk + blockIdx.x] = r;
      }
      __syncthreads();  // shf is rewritten by the next group
    }
  }
}

// rank-1 step 2a, one workgroup per frame j: t_j = (sum_c parts) / div
__global__ __launch_bounds__(kThreads) void k_r1_tsum(const double* __restrict__ parts, int nchunk, int T,
                                                      const double* __restrict__ mx,
                                                      double* __restrict__ t) {
  __shared__ double sh[kThreads / 64];
  for (int j = blockIdx.x; j < T; j += gridDim.x) {
    double v = 0.0;
    for (int c = threadIdx.x; c < nchunk; c += blockDim.x) v += parts[(size_t)j * nchunk + c];
    v = block_reduce(v, sh, [](double a, double b) { return a + b; });
    if (threadIdx.x == 0) t[j] = v / *mx;
  }
}

// rank-1 step 2b (one workgroup): t /= ||t||
__global__ __launch_bounds__(kThreads) void k_r1_tnorm(int T, double* __restrict__ t) {
  __shared__ double sh[kThreads / 64];
  double ss = 0.0;
  for (int j = threadIdx.x; j < T; j += blockDim.x) ss = fma(t[j], t[j], ss);
  const double nrm = sqrt(block_reduce(ss, sh, [](double a, double b) { return a + b; }));
  for (int j = threadIdx.x; j < T; j += blockDim.x) t[j] /= nrm;
}

// rank-1 step 3: s_i = (Y t)_i / div; per-block partial sums of s_i^2
__global__ __launch_bounds__(kThreads) void k_r1_sdot(const float* __restrict__ Y, size_t npix, int T,
                                                      const double* __restrict__ t,
                                                      const double* __restrict__ mx,
                                                      double* __restrict__ s, double* __restrict__ parts) {
  __shared__ double sh[kThreads / 64];
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  double v = 0.0;
  if (i < npix) {
#pragma unroll 8
    for (int j = 0; j < T; ++j) v = fma((double)Y[i + (size_t)j * npix], t[j], v);
    v /= *mx;
    s[i] = v;
  }
  const double ss = block_reduce(v * v, sh, [](double a, double b) { return a + b; });
  if (threadIdx.x == 0) parts[blockIdx.x] = ss;
}

// scalar[0] = sqrt(sum of parts) (one workgroup, fixed order per thread)
__global__ __launch_bounds__(kThreads) void k_fold_norm(const double* __restrict__ parts, int n,
                                                        double* __restrict__ out) {
  __shared__ double sh[kThreads / 64];
  double v = 0.0;
  for (int k = threadIdx.x; k < n; k += blockDim.x) v += parts[k];
  v = block_reduce(v, sh, [](double a, double b) { return a + b; });
  if (threadIdx.x == 0) *out = sqrt(v);
}

__global__ void k_fill_f64(double* __restrict__ v, size_t n, double value) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    v[i] = value;
}

__global__ void k_scale_div(double* __restrict__ v, size_t n, const double* __restrict__ d) {
  const double dv = *d;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    v[i] /= dv;
}

__device__ __forceinline__ void window_of(int k, int* a, int* b) {
  if (k & 1) {
    *a = *b = (k - 1) / 2;
  } else {
    *a = k / 2;
    *b = k / 2 - 1;
  }
}

// Frames j of a window walk: [0, j1) and [j2, T) take the clipped window
// (cnt varies, the updates are guarded); [j1, j2) is the steady part, where
// the window has all k samples and one enters and one leaves every frame.
// The steady loop is unrolled so that its loads (independent of the running
// sum) are issued ahead; the order of the additions is the same everywhere.
__device__ __forceinline__ void walk_bounds(int a, int b, int T, int* j1, int* j2) {
  *j1 = min(a, T);
  *j2 = max(*j1, T - b - 1);
}

// pass 1: d = x - movmean(x, w1), x = Y / mx
__global__ __launch_bounds__(kThreads) void k_detrend(const float* __restrict__ Y, size_t npix, int T,
                                                      int w1, const double* __restrict__ mx,
                                                      float* __restrict__ d) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i >= npix) return;
  // x = Y / max as a product with the reciprocal, and the steady mean as a
  // product with 1/k: within 1 ulp of the quotients, without the FP64
  // divide sequence per sample
  const double minv = 1.0 / *mx;
  int a, b;
  window_of(w1, &a, &b);
  auto x = [&](int j) { return (double)Y[i + (size_t)j * npix] * minv; };
  double S = 0.0;
  const int h0 = min(b, T - 1);
  for (int k = 0; k <= h0; ++k) S += x(k);
  auto step = [&](int j) {
    const int lo = max(j - a, 0), hi = min(j + b, T - 1);
    d[i + (size_t)j * npix] = (float)(x(j) - S / (double)(hi - lo + 1));
    if (j + b + 1 <= T - 1) S += x(j + b + 1);
    if (j - a >= 0) S -= x(j - a);
  };
  int j1, j2;
  walk_bounds(a, b, T, &j1, &j2);
  for (int j = 0; j < j1; ++j) step(j);
  const double kinv = 1.0 / (double)(a + b + 1);
#pragma unroll 8
  for (int j = j1; j < j2; ++j) {
    const double xc = x(j), xn = x(j + b + 1), xo = x(j - a);
    d[i + (size_t)j * npix] = (float)(xc - S * kinv);
    S += xn;
    S -= xo;
  }
  for (int j = j2; j < T; ++j) step(j);
}

// pass 2: y = movmean(d, w2) .^ p; img = sqrt(sum(y^2)/T - mean(y)^2)
__global__ __launch_bounds__(kThreads) void k_smooth_std(const float* __restrict__ d, size_t npix, int T,
                                                         int w2, int p, double* __restrict__ img,
                                                         double* __restrict__ parts) {
  __shared__ double sh[kThreads / 64];
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  double v = __builtin_nan("");
  if (i < npix) {
    int a, b;
    window_of(w2, &a, &b);
    auto dv = [&](int j) { return (double)d[i + (size_t)j * npix]; };
    double S = 0.0, A = 0.0, B = 0.0;
    const int h0 = min(b, T - 1);
    for (int k = 0; k <= h0; ++k) S += dv(k);
    auto acc = [&](double sm) {
      double y = 1.0;
      for (int q = 0; q < p; ++q) y *= sm;
      A = fma(y, y, A);
      B += y;
    };
    auto step = [&](int j) {
      const int lo = max(j - a, 0), hi = min(j + b, T - 1);
      acc(S / (double)(hi - lo + 1));
      if (j + b + 1 <= T - 1) S += dv(j + b + 1);
      if (j - a >= 0) S -= dv(j - a);
    };
    int j1, j2;
    walk_bounds(a, b, T, &j1, &j2);
    for (int j = 0; j < j1; ++j) step(j);
    const double kinv = 1.0 / (double)(a + b + 1);
#pragma unroll 8
    for (int j = j1; j < j2; ++j) {
      const double dn = dv(j + b + 1), dol = dv(j - a);
      acc(S * kinv);
      S += dn;
      S -= dol;
    }
    for (int j = j2; j < T; ++j) step(j);
    const double mean = B / (double)T;
    v = sqrt(A / (double)T - mean * mean);
    img[i] = v;
  }
  v = block_reduce(v, sh, nmax);
  if (threadIdx.x == 0) parts[blockIdx.x] = v;
}

// Patch movie from a sensor movie [H, W, T] (column-major): out[r + h*c + h*w*t]
// = in[(top + r) + H*(left + c) + H*W*t], one patch column per workgroup row.
__global__ __launch_bounds__(kThreads) void k_crop_movie(const float* __restrict__ in, int64_t H,
                                                         int64_t W, int64_t top, int64_t left, int h,
                                                         int w, int T, float* __restrict__ out) {
  const int c = blockIdx.y;
  for (int t = blockIdx.z; t < T; t += gridDim.z) {
    const float* src = in + (size_t)t * H * W + (size_t)(left + c) * H + top;
    float* dst = out + (size_t)t * h * w + (size_t)c * h;
    for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < h; r += gridDim.x * blockDim.x) dst[r] = src[r];
  }
}

// 'global' detrend: compute_std_image.m as written with the rank-1
// background (y_1 = s, y_2 = t) of the movie divided by its max:
// sqrt((A - s_i^2)/T - B^2 + 2 B s_i C - s_i^2 C^2), A = sum(x^2), B = mean(x),
// C = mean(t), x = Y / mx.  A negative argument gives NaN.
__global__ __launch_bounds__(kThreads) void k_std_bg(const float* __restrict__ Y, size_t npix, int T,
                                                     const double* __restrict__ mx,
                                                     const double* __restrict__ s,
                                                     const double* __restrict__ t, double* __restrict__ img,
                                                     double* __restrict__ parts) {
  __shared__ double sh[kThreads / 64];
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  double v = __builtin_nan("");
  if (i < npix) {
    const double m = *mx;
    double A = 0.0, Bs = 0.0, Cs = 0.0;
#pragma unroll 8
    for (int j = 0; j < T; ++j) {
      const double x = (double)Y[i + (size_t)j * npix] / m;
      A = fma(x, x, A);
      Bs += x;
      Cs += t[j];
    }
    const double B = Bs / (double)T, C = Cs / (double)T, y1 = s[i];
    v = sqrt((A - y1 * y1) / (double)T - B * B + 2.0 * B * y1 * C - y1 * y1 * (C * C));
    img[i] = v;
  }
  v = block_reduce(v, sh, nmax);
  if (threadIdx.x == 0) parts[blockIdx.x] = v;
}

// Rectification resample of frames [H, W] (column-major single) at the query
// coordinates yq x xq (1-based pixels): griddedInterpolant's
// 'linear' interpolation and extrapolation, i.e. the bilinear form of the
// grid cell k = clamp(floor(q), 1, size-1), which extends the boundary
// cells linearly past the image.  FP64 arithmetic.
//
// A thread makes one output row of kRectCols neighbouring columns, frames
// strided over the grid's z, with the cells and weights computed once and the
// next frame's pixels requested before this one's are stored.  Neighbouring
// output columns read the same input columns: with one column per workgroup
// they went to different XCDs, each of which fetched the input again, so an
// XCD's workgroups take one run of columns.  1515 x 1515 x 64 at step 14.8 / 15:
// 310 us (3.8 TB/s; one column per workgroup 377; 8 columns 325, 16 357, one
// frame per thread 356).  The coordinates are computed here: a table of them,
// filled, copied and freed in each call, added 12 us (a call now 314 us, was 394).
__device__ __forceinline__ double rect_coord(const RectAxis& q, int i) {
#pragma clang fp contract(off)  // the host's values: product and sum rounded apart
  const int64_t m = q.q0 + i, up = m - q.first;
  const double below = q.center + -q.step * (double)(q.first - 1 - m);
  const double above = (q.center + q.step) + q.step * (double)up;
  return up < 0 ? below : above;
}

constexpr int kRectCols = 4;
__global__ __launch_bounds__(kThreads) void k_rectify(const float* __restrict__ in, int H, int W, int n,
                                                      RectAxis yq, RectAxis xq, float* __restrict__ out) {
  const int Hq = (int)yq.size, Wq = (int)xq.size;
  const unsigned nb = gridDim.x * gridDim.y, id = blockIdx.y * gridDim.x + blockIdx.x;
  const unsigned q8 = nb / 8, rem = nb % 8, xcd = id % 8;
  const unsigned w = xcd * q8 + min(xcd, rem) + id / 8;
  const int j0 = (w / gridDim.x) * kRectCols;
  const int i = (w % gridDim.x) * blockDim.x + threadIdx.x;
  if (i >= Hq) return;
  const double y = rect_coord(yq, i);
  const int ky = min(max((int)floor(y), 1), H - 1);
  const double ty = y - ky;
  double tx[kRectCols];
  size_t o0[kRectCols];  // (row ky, column kx), 1-based
#pragma unroll
  for (int c = 0; c < kRectCols; ++c) {
    const double x = rect_coord(xq, min(j0 + c, Wq - 1));
    const int kx = __builtin_amdgcn_readfirstlane(min(max((int)floor(x), 1), W - 1));
    tx[c] = x - kx;
    o0[c] = (size_t)(kx - 1) * H;
  }
  float p[kRectCols][4];
  auto load = [&](int f) {
    const float* img = in + (size_t)f * H * W;
#pragma unroll
    for (int c = 0; c < kRectCols; ++c) {
      const float* q0 = img + o0[c];
      const float* q1 = q0 + H;
      p[c][0] = q0[ky - 1];
      p[c][1] = q0[ky];
      p[c][2] = q1[ky - 1];
      p[c][3] = q1[ky];
    }
  };
  load(min((int)blockIdx.z, n - 1));
  for (int f = blockIdx.z; f < n; f += gridDim.z) {
    float* o = out + (size_t)f * Hq * Wq + (size_t)j0 * Hq;
    float v[kRectCols];
#pragma unroll
    for (int c = 0; c < kRectCols; ++c) {
      const double v0 = (1.0 - ty) * (double)p[c][0] + ty * (double)p[c][1];
      const double v1 = (1.0 - ty) * (double)p[c][2] + ty * (double)p[c][3];
      v[c] = (float)((1.0 - tx[c]) * v0 + tx[c] * v1);
    }
    if (f + (int)gridDim.z < n) load(f + gridDim.z);
#pragma unroll
    for (int c = 0; c < kRectCols; ++c)
      if (j0 + c < Wq) o[(size_t)c * Hq + i] = v[c];
  }
}

// ---------------------------------------------------------------- tile passes
// Movies whose tiles fit LDS (up to 836 frames, which the last pass takes in tiles of 16
// pixels, from 460 on; 32 below; the rounds 32 from 549 on, 64 below): every pass over
// the movie holds one tile of P pixels x T frames in LDS, so a rank-1 round (Y t, then s'Y) reads the
// movie once instead of twice, the first pass takes the maximum along, and the
// last round's Y t, the detrend, the smoothing and the std image share one
// read with no detrended movie in memory: 6 reads of the movie for 5 rounds
// instead of 13 and a write.  765 x 750 x 400: 2.11 ms a call (the passes above:
// 4.15), 0.24 ms per round (3.8 TB/s; k_r1_tdot + k_r1_sdot 0.48).  A workgroup
// requests its next tile into registers before it computes on the one in LDS
// (tiles of 64 pixels x 400 frames leave room for one workgroup per CU; 1024
// threads rather than 512: 0.28 ms per round).  Tile passes go to
// consecutive workgroups of one XCD, so that the cache lines that two tiles
// share are read once.
//
// The rounds keep s unscaled: t is divided by its norm anyway, and a positive
// factor of s changes nothing before that.
struct TileArgs {
  const float* Y;
  size_t npix;
  int T;
  const double* mx;     // movie maximum
  const double* tt;     // unscaled temporal component [T]
  double* tparts;       // [T][workgroups]: partial s'Y
  double* parts;        // [workgroups]: partial maxima (movie, or image)
  // last pass
  double* s;            // spatial component
  double* img;
  double* t_out;        // tt / |tt|
  int w1, w2, p;
};

constexpr size_t kTileLds = 160 * 1024;
constexpr int kTileThreads = 1024;
constexpr int kRun = 8;  // frames per run of the last pass
enum TileMode { kTileFirst, kTileRound, kTileLast, kTileLastGlobal };
inline __host__ __device__ size_t tile_rows_bytes(int P, int T) { return ((size_t)T * (P + 1) * 4 + 15) / 16 * 16; }
size_t tile_lds(int P, int T, int mode) {
  const size_t common = tile_rows_bytes(P, T) + 8 * ((size_t)T + 2 * kTileThreads + P);
  return mode <= kTileRound
             ? common
             : common + tile_rows_bytes(P, T) + 8 * ((size_t)((T + kRun - 1) / kRun) * P + 2 * (size_t)T);
}

__device__ __forceinline__ double tile_reduce(double v, double* sh, bool max) {
  for (int off = 32; off > 0; off >>= 1) {
    const double o = __shfl_down(v, off, 64);
    v = max ? nmax(v, o) : v + o;
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) sh[wid] = v;
  __syncthreads();
  double r = sh[0];
  for (int k = 1; k < kTileThreads / 64; ++k) r = max ? nmax(r, sh[k]) : r + sh[k];
  return r;
}

// Registers of one tile's samples: thread (i, q) holds pixel i of frames q,
// q + G, ...  A wave's rows are uniform neighbours, so a load takes a scalar row
// address and a 32-bit lane offset.  Past the last frame or pixel a load
// repeats a valid one (its value is not used).
template <int P, int R>
struct TileRegs {
  static constexpr int G = kTileThreads / P;
  float v[R];
  __device__ __forceinline__ void load(const float* __restrict__ Y, size_t npix, int T, size_t tile) {
    const int tid = threadIdx.x;
    const size_t px = tile * P + tid % P;
    const unsigned vo = 4u * (unsigned)(px < npix ? px : npix - 1);
    const int sub = (tid & 63) / P;
    const unsigned vs = vo + 4u * (unsigned)npix * sub;
    int row = __builtin_amdgcn_readfirstlane(tid >> 6) * (64 / P);
    asm volatile("" : "+s"(row));  // else every row address is kept over the tile loop, in spilled registers
    const char* base = reinterpret_cast<const char*>(Y) + 4 * npix * (size_t)row;
#pragma unroll
    for (int k = 0; k < R; k += 8) {
      if (k * G < T) {
#pragma unroll
        for (int h = 0; h < 8; ++h) {
          const char* b = row < T ? base : reinterpret_cast<const char*>(Y);
          v[k + h] = *reinterpret_cast<const float*>(b + (P == 64 || row + sub < T ? vs : vo));
          row += G;
          base += 4 * npix * G;
        }
      }
    }
  }
};

// first tile of a workgroup: 32 consecutive tiles per XCD (blockIdx % 8) and round
__device__ __forceinline__ size_t first_tile() {
  const unsigned n = gridDim.x;
  return n % 8 == 0 ? (blockIdx.x & 7) * (n / 8) + (blockIdx.x >> 3) : blockIdx.x;
}

// tile -> LDS; each(j, x): this thread's samples x of frame j
template <int P, int R, typename F>
__device__ __forceinline__ void tile_store(const TileRegs<P, R>& regs, float* Yt, int T, bool in, F&& each) {
  constexpr int G = kTileThreads / P, LD = P + 1;
  const int i = threadIdx.x % P, q = threadIdx.x / P;
#pragma unroll
  for (int k = 0; k < R; k += 8) {
    if (k * G < T) {
#pragma unroll
      for (int h = 0; h < 8; ++h) {
        const int j = q + (k + h) * G;
        const float x = in ? regs.v[k + h] : 0.f;
        if (j < T) {
          Yt[j * LD + i] = x;
          each(j, x);
        }
      }
    }
  }
}

// t = tt / |tt| in LDS
__device__ __forceinline__ void tile_temporal(const TileArgs& g, double* td, double* red, bool write) {
  double ss = 0.0;
  for (int j = threadIdx.x; j < g.T; j += kTileThreads) ss = fma(g.tt[j], g.tt[j], ss);
  const double nrm = sqrt(tile_reduce(ss, red, false));
  for (int j = threadIdx.x; j < g.T; j += kTileThreads) {
    const double t = g.tt[j] / nrm;
    td[j] = t;
    if (write) g.t_out[j] = t;
  }
  __syncthreads();
}

// kTileFirst: partial maxima and s'Y of the constant s; kTileRound: s = Y t, then s'Y
template <int P, int R, int MODE>
__global__ __launch_bounds__(kTileThreads) void k_summary_round(TileArgs g) {
  constexpr int NT = kTileThreads, G = NT / P;
  constexpr int LD = P + 1;                      // odd: lanes along the frames fall on different banks
  constexpr int kFrames = (1200 + NT - 1) / NT;  // frames per thread of s'Y
  extern __shared__ __align__(16) char lds[];
  const int T = g.T, tid = threadIdx.x;
  float* Yt = reinterpret_cast<float*>(lds);  // [T][LD]
  double* td = reinterpret_cast<double*>(lds + tile_rows_bytes(P, T));
  double* red = td + T;        // [2 NT]
  double* vs = red + 2 * NT;   // [P]
  const size_t npix = g.npix, ntile = (npix + P - 1) / P, nwg = gridDim.x;
  TileRegs<P, R> regs;
  size_t tile = first_tile();
  if (tile < ntile) regs.load(g.Y, npix, T, tile);
  const double mx = MODE == kTileFirst ? 1.0 : *g.mx;
  if constexpr (MODE == kTileFirst) {
    if (tid < P) vs[tid] = 1.0 / sqrt((double)npix);
  } else {
    tile_temporal(g, td, red, false);
  }
  double acc[kFrames];
#pragma unroll
  for (int k = 0; k < kFrames; ++k) acc[k] = 0.0;
  float mf = __builtin_nanf("");
  for (; tile < ntile; tile += nwg) {
    const bool in = tile * P + tid % P < npix;
    double a = 0.0;
    tile_store(regs, Yt, T, in, [&](int j, float x) {
      if constexpr (MODE == kTileFirst) mf = in ? fmaxf(mf, x) : mf;  // NaN ignored
      else a = fma((double)x, td[j], a);
    });
    if constexpr (MODE == kTileRound) red[tid] = a;
    __syncthreads();
    if (tile + nwg < ntile) regs.load(g.Y, npix, T, tile + nwg);  // in flight while this tile is worked on
    if constexpr (MODE == kTileRound) {
      if (tid < P) {
        double r = red[tid];
#pragma unroll
        for (int k = 1; k < G; ++k) r += red[tid + k * P];
        vs[tid] = r / mx;
      }
      __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < kFrames; ++k) {
      const int j = tid + k * NT;
      if (j < T) {
        double r0 = 0.0, r1 = 0.0;
#pragma unroll 8
        for (int c = 0; c < P; c += 2) {
          r0 = fma((double)Yt[j * LD + c], vs[c], r0);
          r1 = fma((double)Yt[j * LD + c + 1], vs[c + 1], r1);
        }
        acc[k] += r0 + r1;
      }
    }
    __syncthreads();  // the tile, red and vs are rewritten
  }
#pragma unroll
  for (int k = 0; k < kFrames; ++k) {
    const int j = tid + k * NT;
    if (j < T) g.tparts[(size_t)j * nwg + blockIdx.x] = acc[k];
  }
  if constexpr (MODE == kTileFirst) {
    const double m = tile_reduce((double)mf, red, true);
    if (tid == 0) g.parts[blockIdx.x] = m;
  }
}

// sums of whole runs of kRun rows of pixel i, by threads (i, q)
template <int P>
__device__ __forceinline__ void run_sums(const float* rows, double* runs, int T) {
  for (int c = threadIdx.x / P; c < T / kRun; c += kTileThreads / P) {
    const float* y = rows + c * kRun * (P + 1) + threadIdx.x % P;
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < kRun; ++k) s += (double)y[k * (P + 1)];
    runs[c * P + threadIdx.x % P] = s;
  }
}
// sum of rows lo .. hi of this thread's pixel, whole runs from their sums
template <int P>
__device__ __forceinline__ double window_sum(const float* y, const double* runs, int lo, int hi) {
  double s = 0.0;
  const int c0 = (lo + kRun - 1) / kRun, c1 = (hi + 1) / kRun;
  if (c0 >= c1) {
    for (int k = lo; k <= hi; ++k) s += (double)y[k * (P + 1)];
    return s;
  }
  for (int k = lo; k < c0 * kRun; ++k) s += (double)y[k * (P + 1)];
  for (int c = c0; c < c1; ++c) s += runs[c * P];
  for (int k = c1 * kRun; k <= hi; ++k) s += (double)y[k * (P + 1)];
  return s;
}

// The last round's s = Y t and the image.  'pixelwise': the detrended tile
// (FP32, as k_detrend stores it) in LDS beside the samples; a thread walks runs
// of 8 frames, each window sum started from the sums of whole runs.  0.90 ms at
// 765 x 750 x 400 (k_r1_sdot + k_detrend + k_smooth_std: 1.23 ms), bound by the
// LDS reads and FP64 chains of the windows; one running sum over a quarter of
// the frames per thread took 2.4 ms, 512 threads instead of 1024 1.15 ms.
template <int P, int R, int MODE>
__global__ __launch_bounds__(kTileThreads) void k_summary_last(TileArgs g) {
  constexpr int NT = kTileThreads, G = NT / P, LD = P + 1;
  extern __shared__ __align__(16) char lds[];
  const int T = g.T, tid = threadIdx.x, i = tid % P, q = tid / P;
  float* Yt = reinterpret_cast<float*>(lds);                            // [T][LD]
  float* Dt = reinterpret_cast<float*>(lds + tile_rows_bytes(P, T));    // [T][LD]
  double* td = reinterpret_cast<double*>(lds + 2 * tile_rows_bytes(P, T));
  double* red = td + T;        // [2 NT]
  double* vs = red + 2 * NT;   // [P]
  double* rk1 = vs + P;        // [T] 1 / (samples in the window of frame j), window_1
  double* rk2 = rk1 + T;       // [T] window_2
  double* runs = rk2 + T;      // [T / kRun][P]
  const size_t npix = g.npix, ntile = (npix + P - 1) / P, nwg = gridDim.x;
  TileRegs<P, R> regs;
  size_t tile = first_tile();
  if (tile < ntile) regs.load(g.Y, npix, T, tile);
  const double mx = *g.mx, minv = 1.0 / mx;
  tile_temporal(g, td, red, blockIdx.x == 0);
  double tc = 0.0;  // 'global': mean of t
  if constexpr (MODE == kTileLastGlobal) {
    for (int j = 0; j < T; ++j) tc += td[j];
    tc /= (double)T;
  }
  int a1, b1, a2, b2;
  window_of(g.w1, &a1, &b1);
  window_of(g.w2, &a2, &b2);
  for (int j = tid; j < T; j += NT) {
    rk1[j] = 1.0 / (double)(min(j + b1, T - 1) - max(j - a1, 0) + 1);
    rk2[j] = 1.0 / (double)(min(j + b2, T - 1) - max(j - a2, 0) + 1);
  }
  double m = __builtin_nan("");
  for (; tile < ntile; tile += nwg) {
    const size_t px = tile * P + i;
    const bool in = px < npix;
    double a = 0.0;
    tile_store(regs, Yt, T, in, [&](int j, float x) { a = fma((double)x, td[j], a); });
    red[tid] = a;
    __syncthreads();
    if (tile + nwg < ntile) regs.load(g.Y, npix, T, tile + nwg);
    if (tid < P) {
      double r = red[tid];
#pragma unroll
      for (int k = 1; k < G; ++k) r += red[tid + k * P];
      r /= mx;
      vs[tid] = r;
      if (in) g.s[px] = r;
    }
    double A = 0.0, B = 0.0;
    if constexpr (MODE == kTileLast) {
      run_sums<P>(Yt, runs, T);
      __syncthreads();
      const float* y = Yt + i;
      float* d = Dt + i;
      for (int j0 = q * kRun; j0 < T; j0 += G * kRun) {
        double S = window_sum<P>(y, runs + i, max(j0 - a1, 0), min(j0 + b1, T - 1));
        const float* yc = y + j0 * LD;
        if (j0 >= a1 && j0 + kRun + b1 < T) {  // every window of the run is whole
          float c[kRun], n[kRun], o[kRun];
#pragma unroll
          for (int k = 0; k < kRun; ++k) {
            c[k] = yc[k * LD];
            n[k] = yc[(k + b1 + 1) * LD];
            o[k] = yc[(k - a1) * LD];
          }
#pragma unroll
          for (int k = 0; k < kRun; ++k) {
            d[(j0 + k) * LD] = (float)(((double)c[k] - S * rk1[j0 + k]) * minv);
            S += (double)n[k];
            S -= (double)o[k];
          }
        } else {
          for (int j = j0; j < min(j0 + kRun, T); ++j) {
            d[j * LD] = (float)(((double)y[j * LD] - S * rk1[j]) * minv);
            if (j + b1 + 1 <= T - 1) S += (double)y[(j + b1 + 1) * LD];
            if (j - a1 >= 0) S -= (double)y[(j - a1) * LD];
          }
        }
      }
      __syncthreads();
      run_sums<P>(Dt, runs, T);
      __syncthreads();
      for (int j0 = q * kRun; j0 < T; j0 += G * kRun) {
        double S = window_sum<P>(d, runs + i, max(j0 - a2, 0), min(j0 + b2, T - 1));
        auto add = [&](double sm) {
          double v = 1.0;
          for (int n = 0; n < g.p; ++n) v *= sm;
          A = fma(v, v, A);
          B += v;
        };
        const float* dc = d + j0 * LD;
        if (j0 >= a2 && j0 + kRun + b2 < T) {
          float n[kRun], o[kRun];
#pragma unroll
          for (int k = 0; k < kRun; ++k) {
            n[k] = dc[(k + b2 + 1) * LD];
            o[k] = dc[(k - a2) * LD];
          }
#pragma unroll
          for (int k = 0; k < kRun; ++k) {
            add(S * rk2[j0 + k]);
            S += (double)n[k];
            S -= (double)o[k];
          }
        } else {
          for (int j = j0; j < min(j0 + kRun, T); ++j) {
            add(S * rk2[j]);
            if (j + b2 + 1 <= T - 1) S += (double)d[(j + b2 + 1) * LD];
            if (j - a2 >= 0) S -= (double)d[(j - a2) * LD];
          }
        }
      }
    } else {
      __syncthreads();
      for (int j = q; j < T; j += G) {
        const double x = (double)Yt[j * LD + i] / mx;
        A = fma(x, x, A);
        B += x;
      }
    }
    red[tid] = A;
    red[NT + tid] = B;
    __syncthreads();
    if (tid < P && in) {
      for (int k = 1; k < G; ++k) {
        A += red[tid + k * P];
        B += red[NT + tid + k * P];
      }
      const double mean = B / (double)T;
      double r;
      if constexpr (MODE == kTileLast) {
        r = sqrt(A / (double)T - mean * mean);
      } else {
        const double y1 = vs[tid];
        r = sqrt((A - y1 * y1) / (double)T - mean * mean + 2.0 * mean * y1 * tc - y1 * y1 * (tc * tc));
      }
      g.img[px] = r;
      m = nmax(m, r);
    }
    __syncthreads();  // the tiles, red and vs are rewritten
  }
  m = tile_reduce(m, red, true);
  if (tid == 0) g.parts[blockIdx.x] = m;
}

typedef void (*TileKernel)(TileArgs);

// Pixels per tile of a movie of T frames: the widest rows that fit LDS (0: no
// tile does, the movie goes through the passes above).
int tile_pixels(size_t npix, int T, int mode) {
  if (npix >= (size_t)1 << 28) return 0;  // 32-bit byte offsets within four rows
  for (int P : {64, 32, 16})
    if (!(P == 64 && mode >= kTileLast) && !(P == 16 && mode <= kTileRound) && tile_lds(P, T, mode) <= kTileLds)
      return P;
  return 0;
}
// A tile of few frames is little work between its barriers, and a large frame has many
// tiles: below min(60, npix / 20000 - 2) frames the passes above are the faster ones.  Time of
// the tile passes over theirs ('pixelwise'): 400 x 400 1.07 at 4 frames, 0.67 at 16; 600 x 600 1.47 at 8,
// 0.91 at 16; 800 x 800 1.43 at 24, 0.92 at 32; 1000 x 1000 3.0 at 4, 1.25 at 32, 1.09 at 48, 0.89 at 64;
// 1515 x 1515 1.39 at 48, 0.94 at 64 (global: 1.12, 0.77).
bool tiled(size_t npix, int T) {
  return (T >= 60 || ((size_t)T + 2) * 20000 >= npix) && tile_pixels(npix, T, kTileRound) && tile_pixels(npix, T, kTileLast);
}

// 64 pixels take 16 registers for up to 256 frames, 40 up to 548; 32 pixels come
// from 549 on and take 40
template <int P, int R>
TileKernel pick_round(int mode) {
  return mode == kTileFirst ? &k_summary_round<P, R, kTileFirst> : &k_summary_round<P, R, kTileRound>;
}
template <int P>
TileKernel pick_last(int mode) {
  return mode == kTileLast ? &k_summary_last<P, 16, kTileLast> : &k_summary_last<P, 16, kTileLastGlobal>;
}

constexpr int kTileWgs = 1024;  // most workgroups of a pass

hipError_t launch_tile(const TileArgs& g, int mode, int cus, int* nwg, hipStream_t st) {
  const int P = tile_pixels(g.npix, g.T, mode);
  const size_t lds = tile_lds(P, g.T, mode);
  const TileKernel fn = mode <= kTileRound
                            ? (P == 32 ? pick_round<32, 40>(mode) : g.T <= 256 ? pick_round<64, 16>(mode) : pick_round<64, 40>(mode))
                            : (P == 32 ? pick_last<32>(mode) : pick_last<16>(mode));
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTileLds);
  if (e != hipSuccess) return e;
  const size_t ntile = (g.npix + P - 1) / P;
  const size_t per_cu = std::min<size_t>(kTileLds / lds, 2);
  *nwg = (int)std::min<size_t>(ntile, std::min<size_t>(kTileWgs, per_cu * cus));
  if (*nwg > 8) *nwg = *nwg / 8 * 8;
  hipLaunchKernelGGL(fn, dim3(*nwg), dim3(kTileThreads), lds, st, g);
  return hipGetLastError();
}

inline unsigned blocks_for(size_t n) { return (unsigned)((n + kThreads - 1) / kThreads); }

}  // namespace

size_t summary_scratch_doubles(size_t npix, int T) {
  const size_t nchunk = (npix + kChunk - 1) / kChunk;
  const size_t nblk = (npix + kThreads - 1) / kThreads;
  if (tiled(npix, T)) return 2 + 2 * (size_t)T + (size_t)T * kTileWgs + kTileWgs;
  // mx, norm, t[T], tdot parts[T * nchunk], per-block parts[max(nblk, 1024)]
  return 2 + (size_t)T + (size_t)T * nchunk + (nblk > 1024 ? nblk : 1024);
}

bool summary_needs_movie(size_t npix, int T) { return !tiled(npix, T); }

static hipError_t launch_summary_tiled(const float* Y, size_t npix, int T, int w1, int w2, int p, int bg_iter,
                                       int global, double* scratch, double* img, double* s, int cus,
                                       hipStream_t st) {
  double* mx = scratch;
  double* nrm = scratch + 1;
  double* t = scratch + 2;   // the result (summary_temporal)
  double* tt = t + T;        // unscaled
  TileArgs g{Y, npix, T, mx, tt, tt + T, tt + T + (size_t)T * kTileWgs, s, img, t, w1, w2, p};
  int nwg = 0;
  for (int it = 0; it < bg_iter; ++it) {
    const hipError_t e = launch_tile(g, it == 0 ? kTileFirst : kTileRound, cus, &nwg, st);
    if (e != hipSuccess) return e;
    if (it == 0) hipLaunchKernelGGL(k_fold_max, dim3(1), dim3(kThreads), 0, st, g.parts, nwg, mx);
    hipLaunchKernelGGL(k_r1_tsum, dim3(T), dim3(kThreads), 0, st, g.tparts, nwg, T, mx, tt);
  }
  const hipError_t e = launch_tile(g, global ? kTileLastGlobal : kTileLast, cus, &nwg, st);
  if (e != hipSuccess) return e;
  const unsigned nblk = blocks_for(npix);
  hipLaunchKernelGGL(k_fold_max, dim3(1), dim3(kThreads), 0, st, g.parts, nwg, nrm);
  hipLaunchKernelGGL(k_scale_div, dim3(nblk < 65535 ? nblk : 65535), dim3(kThreads), 0, st, img, npix, nrm);
  return hipGetLastError();
}

hipError_t launch_summary(const float* Y, size_t npix, int T, int w1, int w2, int p, int bg_iter,
                          int global, double* scratch, float* dbuf, double* img, double* s, int cus,
                          hipStream_t st) {
  if (tiled(npix, T)) return launch_summary_tiled(Y, npix, T, w1, w2, p, bg_iter, global, scratch, img, s, cus, st);
  const size_t nchunk = (npix + kChunk - 1) / kChunk;
  const unsigned nblk = blocks_for(npix);
  double* mx = scratch;
  double* nrm = scratch + 1;
  double* t = scratch + 2;
  double* tparts = t + T;
  double* parts = tparts + (size_t)T * nchunk;
  // movie max (the divisor of the background and the scale of x)
  const size_t n = npix * (size_t)T;
  const unsigned gmax = 1024;
  if (((uintptr_t)Y & 15) == 0)
    hipLaunchKernelGGL(k_max_f32x4, dim3(gmax), dim3(kThreads), 0, st, reinterpret_cast<const float4*>(Y),
                       n / 4, Y + (n & ~(size_t)3), (int)(n & 3), parts);
  else
    hipLaunchKernelGGL(k_max_f32, dim3(gmax), dim3(kThreads), 0, st, Y, n, parts);
  hipLaunchKernelGGL(k_fold_max, dim3(1), dim3(kThreads), 0, st, parts, (int)gmax, mx);
  // rank-1 background: s = ones / sqrt(npix), bg_iter rounds
  hipLaunchKernelGGL(k_fill_f64, dim3(nblk < 65535 ? nblk : 65535), dim3(kThreads), 0, st, s, npix,
                     1.0 / sqrt((double)npix));
  for (int it = 1; it <= bg_iter; ++it) {
    const int fy = (T + kTdotFrames - 1) / kTdotFrames;
    hipLaunchKernelGGL(k_r1_tdot, dim3((unsigned)nchunk, fy < 65535 ? fy : 65535), dim3(kThreads), 0, st,
                       Y, npix, T, s, tparts);
    hipLaunchKernelGGL(k_r1_tsum, dim3(T < 65535 ? T : 65535), dim3(kThreads), 0, st, tparts, (int)nchunk,
                       T, mx, t);
    hipLaunchKernelGGL(k_r1_tnorm, dim3(1), dim3(kThreads), 0, st, T, t);
    hipLaunchKernelGGL(k_r1_sdot, dim3(nblk), dim3(kThreads), 0, st, Y, npix, T, t, mx, s, parts);
    if (it < bg_iter) {
      hipLaunchKernelGGL(k_fold_norm, dim3(1), dim3(kThreads), 0, st, parts, (int)nblk, nrm);
      hipLaunchKernelGGL(k_scale_div, dim3(nblk < 65535 ? nblk : 65535), dim3(kThreads), 0, st, s, npix, nrm);
    }
  }
  // summary image
  if (global) {
    hipLaunchKernelGGL(k_std_bg, dim3(nblk), dim3(kThreads), 0, st, Y, npix, T, mx, s, t, img, parts);
  } else {
    hipLaunchKernelGGL(k_detrend, dim3(nblk), dim3(kThreads), 0, st, Y, npix, T, w1, mx, dbuf);
    hipLaunchKernelGGL(k_smooth_std, dim3(nblk), dim3(kThreads), 0, st, dbuf, npix, T, w2, p, img, parts);
  }
  hipLaunchKernelGGL(k_fold_max, dim3(1), dim3(kThreads), 0, st, parts, (int)nblk, nrm);
  hipLaunchKernelGGL(k_scale_div, dim3(nblk < 65535 ? nblk : 65535), dim3(kThreads), 0, st, img, npix, nrm);
  return hipGetLastError();
}

const double* summary_temporal(const double* scratch) { return scratch + 2; }

hipError_t launch_rectify(const float* in, int H, int W, int n, RectAxis yq, RectAxis xq, float* out,
                          hipStream_t st) {
  const unsigned gx = (unsigned)((yq.size + kThreads - 1) / kThreads);
  const unsigned gy = (unsigned)((xq.size + kRectCols - 1) / kRectCols);
  hipLaunchKernelGGL(k_rectify, dim3(gx, gy, (unsigned)(n < 16 ? n : 16)), dim3(kThreads), 0, st, in, H, W, n, yq,
                     xq, out);
  return hipGetLastError();
}

hipError_t launch_crop_movie(const float* in, int64_t H, int64_t W, int64_t top, int64_t left, int h,
                             int w, int T, float* out, hipStream_t st) {
  const unsigned gx = (unsigned)((h + kThreads - 1) / kThreads);
  hipLaunchKernelGGL(k_crop_movie, dim3(gx, (unsigned)w, (unsigned)(T < 16 ? T : 16)), dim3(kThreads), 0,
                     st, in, H, W, top, left, h, w, T, out);
  return hipGetLastError();
}

}  // namespace mlf
