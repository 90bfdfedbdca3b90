// MEX operator for odd kernel widths on the BF16 matrix pipe at FP32 precision.
//
// As in k_mex_mfma (mex_kernels.hip), outputs grouped by phase make the operator a
// GEMM: for output row y (q = y % 15), image n and x = 15 i + p
//   out = sum_{ky, t} in[15 i + t - h, y - h + ky, n] * K[t - p, ky, p, q].
// Every FP32 operand is split into three BF16 parts (8 + 8 + 8 significand bits, each
// part rounded to nearest), x = x0 + x1 + x2 exactly for |x| from 2^-110 (8e-34): below,
// x2 ends at BF16's last bit, 2^-133, and leaves up to 2^-134 out.  A product
// takes the six MFMAs x0 k0, x0 k1, x1 k0, x1 k1, x0 k2, x2 k0, all into one
// FP32 accumulator; the three left out are below 2^-24 of the product.  Six
// 16x16x32 BF16 MFMAs take 96 cycles where the FP32 pipe takes 256, and the
// accumulator is rounded 6 times per 32 taps instead of 8 or more times.
// Bound by the matrix pipe.  396 x 396 x 96, kw = 241: 8.44 ms, 1.25e15 BF16
// flop/s issued for the products alone (FP32 MFMA, k_mex_mfma: 26.8 ms); 24
// segments over 5 planes of that size: 6.3 to 8.5 ms by their slices (24.5 for the
// former); one 150 x 137 bitmap, kw = 61: 34 us (229: one wave in eight had work).
// Relative L2 error against FP64 there: 9.5e-8 / 8.7e-8 / 6.5e-8 (FP32 MFMA 8.2e-7 / 7.9e-7
// / 6.1e-7; in one chain over all rows, whose low bits the pipe cuts, 5.6e-7 / 1.8e-7 / 6.6e-8).
//
// Operand layout.  A lenslet's 15 pixels take 16 slots (slot 15 zero), so tap
// t = 15 L + s - b sits at slot s of lenslet i - a + L (h = 15 a - b) and the
// A fragment of a lane -- 8 consecutive slots of one lenslet -- is one aligned
// 16-byte LDS read, for any alignment of h.  M rows are the cells (image, i)
// counted through all images, so ragged widths waste no rows; the cells that a
// workgroup's rows read are consecutive too and are staged once per input row
// (split on the way).  N = 15 phases (16) of G output rows that share the
// input row, each with its own kernel row: G rows reuse one A fragment.
// The kernel side is a table of ready fragments built once per call
// (k_mex_split_prep) and copied to LDS by buffer loads.
//
// A value that BF16 cannot round without overflow (infinities, NaN, the last
// 2^-9 below FLT_MAX) would turn the products of its parts into NaN: the prep
// kernel marks the bitmap or the kernel set that holds one (mex_marks.h), and this
// kernel leaves a marked bitmap, or every bitmap of a marked set, to k_mex_mfma,
// launched behind it.  The other bitmaps of the call stay here.
#include <algorithm>

#include "internal.h"

namespace mlf {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

constexpr int kMaxL = 40;  // lenslets (16 slots) per kernel row, even: kw <= kMexMfmaMaxKw
constexpr int kDword3 = 0x00020000;  // raw buffer resource, 32-bit data format

__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ unsigned pk(float lo, float hi) {
  const unsigned short a = __builtin_bit_cast(unsigned short, (__bf16)lo);
  const unsigned short b = __builtin_bit_cast(unsigned short, (__bf16)hi);
  return (unsigned)a | ((unsigned)b << 16);
}
// two values -> their three parts, packed in pairs
__device__ __forceinline__ void split2(float x, float y, unsigned* w) {
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    w[k] = pk(x, y);
    x -= __builtin_bit_cast(float, w[k] << 16);
    y -= __builtin_bit_cast(float, w[k] & 0xFFFF0000u);
  }
}
// |x| rounds to infinity in BF16 (or is not finite)
__device__ __forceinline__ bool too_large(float x) {
  return (__builtin_bit_cast(unsigned, x) & 0x7FFFFFFFu) >= 0x7F7F8000u;
}

struct SplitGeo {
  int W, H, n;   // bitmap columns, rows, images of the launch
  int kw, h;     // kernel width and half width
  int nL;        // lenslets per bitmap row
  int a;         // lenslets left of an output's own that its kernel reaches
  int nks;       // K-steps (lenslet pairs) per kernel row
  int nyg, nmb;  // output row groups, M blocks
};

// Fragment table Bt[q][ky][ks][part][lane][8]: lane (p = lane % 16, lg = lane / 16)
// holds slots 8 (lg % 2) .. + 7 of lenslet L = 2 ks + lg / 2.  Past the nbt blocks that
// make it, nbi blocks look through each bitmap of `image` values.
__global__ __launch_bounds__(256) void k_mex_split_prep(const float* __restrict__ K, int kw, int b, int nks,
                                                        uintx4* __restrict__ Bt, int nbt,
                                                        const float* __restrict__ scan, size_t image, int nbi,
                                                        MexMarks marks, int set) {
  const uint32_t call = *marks.finished() + 1;
  bool bad = false;
  int img = -1;  // bitmap of this block, or the kernel set
  if ((int)blockIdx.x < nbt) {
    const size_t total = (size_t)kN * kw * nks * 64;
    for (size_t o = blockIdx.x * (size_t)256 + threadIdx.x; o < total; o += (size_t)nbt * 256) {
      const int lane = (int)(o & 63), p = lane & 15, lg = lane >> 4;
      const size_t blk = o >> 6;  // (q kw + ky) nks + ks
      const int ks = (int)(blk % nks);
      const int ky = (int)((blk / nks) % kw);
      const int q = (int)(blk / ((size_t)nks * kw));
      const int kx0 = kN * (2 * ks + (lg >> 1)) + 8 * (lg & 1) - p - b;
      const float* row = K + (size_t)kw * ky + (size_t)kw * kw * (min(p, kN - 1) + kN * q);
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int kx = kx0 + e;
        const float t = row[min(max(kx, 0), kw - 1)];
        bad = bad || too_large(t);
        v[e] = (p < kN && kx >= 0 && kx < kw && 8 * (lg & 1) + e < kN) ? t : 0.f;
      }
      unsigned w[4][3];
#pragma unroll
      for (int e = 0; e < 4; ++e) split2(v[2 * e], v[2 * e + 1], w[e]);
#pragma unroll
      for (int k = 0; k < 3; ++k) Bt[(blk * 3 + k) * 64 + lane] = uintx4{w[0][k], w[1][k], w[2][k], w[3][k]};
    }
  } else {
    img = (int)(blockIdx.x - nbt) / nbi;
    const float* s = scan + img * image;
    const size_t step = (size_t)nbi * 256;
    size_t o = ((blockIdx.x - nbt) % nbi) * (size_t)256 + threadIdx.x;
    for (; o + 3 * step < image; o += 4 * step) {
      const float v0 = s[o], v1 = s[o + step], v2 = s[o + 2 * step], v3 = s[o + 3 * step];
      bad = bad || too_large(v0) || too_large(v1) || too_large(v2) || too_large(v3);
    }
    for (; o < image; o += step) bad = bad || too_large(s[o]);
  }
  if (!bad) return;
  *marks.any() = call;
  if (img < 0) *marks.set() = MexMarks::set_mark(call, set);
  else *marks.image(img) = call;
}

// Input row r is of class r % kClasses.  Each class is summed from zero, row by
// row, and the sums of the classes are added in class order, whatever the shape
// of the workgroups: an output's bits do not depend on the shape, and so not on
// how many bitmaps share the call (a call may take any of the shapes below).
constexpr int kClasses = 8;

// WM waves along M times WK groups that share the input rows (class c goes to
// group c % WK in lap c / WK; every group keeps the sums of its laps to the end, or
// adds them up as it goes if it is the only one), MT M-tiles per wave, G output rows,
// SPB K-steps per barrier.
template <int WM, int WK, int MT, int G, int SPB>
struct SplitShape {
  static constexpr int kThreads = 64 * WM * WK;
  static constexpr int kRows = 16 * MT * WM;       // M rows (cells) per workgroup
  static constexpr int kSlots = kRows + kMaxL + 1;  // staged cells, the last always zero
  static constexpr int kHalf = kSlots * 16;         // bytes of one 8-slot half of all cells
  static constexpr int kPart = 2 * kHalf;
  static constexpr int kA = 3 * kPart;              // one input row, three parts
  static constexpr int kB = SPB * G * 3 * 1024;     // one stage of kernel fragments
  static constexpr int kGroup = 2 * kA + 2 * kB;
  static constexpr int kLaps = kClasses / WK;
  static constexpr int kSums = WK == 1 ? 1 : kLaps;  // sums kept
  static constexpr int kRed = (WK - 1) * kSums * WM * MT * G * 1024;  // the other groups' sums, at the end
  static constexpr int kLds = WK * kGroup > kRed ? WK * kGroup : kRed;
  static_assert(kClasses % WK == 0 && kLds <= 160 * 1024, "LDS");
  static constexpr int kPerCu = 160 * 1024 / kLds;  // workgroups that share a CU
};

template <int WM, int WK, int MT, int G, int SPB>
__global__ __launch_bounds__(64 * WM * WK)
__attribute__((amdgpu_waves_per_eu(SplitShape<WM, WK, MT, G, SPB>::kPerCu * WM * WK / 4)))
void k_mex_split(const float* __restrict__ in, SplitGeo g, const uintx4* __restrict__ Bt, float* __restrict__ out,
                 const int32_t* __restrict__ src, const int32_t* __restrict__ dst, MexMarks marks, int set) {
  using S = SplitShape<WM, WK, MT, G, SPB>;
  constexpr int NTH = 64 * WM;  // threads of a group
  constexpr int NU = (S::kSlots * 8 + NTH - 1) / NTH;  // pixel pairs staged per thread and row
  extern __shared__ __align__(16) char sm[];
  const uint32_t call = uni(*marks.finished()) + 1;
  if (blockIdx.x == 0 && threadIdx.x == 0) *marks.current() = call;
  const bool any = (uint32_t)uni(*marks.any()) == call;
  if (any && marks.set_marked(call, set)) return;
  const int W = g.W, H = g.H, nL = g.nL;
  const int tid = threadIdx.x, lane = tid & 63, w = uni(tid >> 6), lr = lane & 15, lg = lane >> 4;
  const int wk = w / WM, wm = w % WM, gt = tid - wk * NTH;
  char* const Ab = sm + wk * S::kGroup;
  char* const Bb = Ab + 2 * S::kA;
  // Workgroups of one row group share its kernel fragments: blockIdx % 8 is
  // the XCD, so they take consecutive turns on one XCD.  Groups in the middle
  // of the bitmap, whose kernels are cut by no border, start first.
  const int bx = blockIdx.x, turn = bx >> 3;
  const int rank = (turn / g.nmb) * 8 + (bx & 7), mb = turn % g.nmb;
  if (rank >= g.nyg) return;
  const int yg = (rank & 1) ? g.nyg / 2 - (rank + 1) / 2 : g.nyg / 2 + rank / 2;
  const int y0 = G * yg;
  const int M0 = mb * S::kRows, NC = g.n * nL;
  if (any) {  // nothing to do if every bitmap of the block is marked
    bool live = false;
    for (int i = M0 / nL; i <= (min(M0 + S::kRows, NC) - 1) / nL; ++i)
      live = live || !marks.image_marked(call, src ? src[i] : i);
    if (!live) return;
  }

  // staged pairs: pixels 15 lens + 2 k, + 1 (k = 7: pixel 14 and the zero slot)
  const int pk8 = gt & 7;
  const int ncell = S::kRows + 2 * g.nks - 1;
  int off[NU];
  unsigned ok = 0;
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int c = M0 - g.a + (gt >> 3) + u * (NTH / 8);
    const bool in0 = (gt >> 3) + u * (NTH / 8) < ncell && c >= 0 && c < NC;
    const int img = in0 ? c / nL : 0, x = kN * (in0 ? c - img * nL : 0) + 2 * pk8;
    const bool ok0 = in0 && x < W, ok1 = ok0 && pk8 < 7 && x + 1 < W;
    off[u] = ok0 ? (src ? src[img] : img) * W * H + x : 0;
    ok |= (unsigned)ok0 << u | (unsigned)ok1 << (u + 16);
  }
  static_assert(NU <= 16, "mask bits");
  float v0[NU], v1[NU];
  auto load_row = [&](int r) {
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const float* s = in + (size_t)(off[u] + r * W);
      v0[u] = s[0];
      v1[u] = s[(ok >> (u + 16)) & 1];
    }
  };
  auto store_row = [&](char* A) {
    char* d = A + (pk8 >> 2) * S::kHalf + (gt >> 3) * 16 + (pk8 & 3) * 4;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      if ((gt >> 3) + u * (NTH / 8) >= ncell) continue;
      unsigned p[3];
      split2((ok >> u) & 1 ? v0[u] : 0.f, (ok >> (u + 16)) & 1 ? v1[u] : 0.f, p);
#pragma unroll
      for (int k = 0; k < 3; ++k) *reinterpret_cast<unsigned*>(d + u * (NTH / 8) * 16 + k * S::kPart) = p[k];
    }
  };
  if (gt < 12)  // the zero slot of each buffer, part and half
    *reinterpret_cast<uintx4*>(Ab + (gt / 6) * S::kA + (gt % 6) * S::kHalf + (S::kSlots - 1) * 16) = uintx4{0, 0, 0, 0};

  // this lane's A rows
  int lens[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) lens[m] = (M0 + 16 * (wm * MT + m) + lr) % nL - g.a + (lg >> 1);
  const int slot0 = 16 * wm * MT + lr + (lg >> 1);

  floatx4 acc[MT][G], sum[S::kSums][MT][G];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int i = 0; i < G; ++i) acc[m][i] = sum[0][m][i] = floatx4{0.f, 0.f, 0.f, 0.f};

  const int rlo = max(0, y0 - g.h), rhi = min(H - 1, y0 + G - 1 + g.h);
  const int nj = (rhi - rlo) / kClasses + 1;  // rows of a class, at most
  const int ns = (g.nks + SPB - 1) / SPB;     // stages per row
  const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uintx4*>(Bt), 0, kN * g.kw * g.nks * 3 * 1024, kDword3);
  int q15[G];
#pragma unroll
  for (int i = 0; i < G; ++i) q15[i] = (y0 + i) % kN;
  auto issue_b = [&](int r, int s, char* buf) {
#pragma unroll
    for (int c0 = 0; c0 < SPB * G * 3; c0 += WM) {
      const int c = c0 + wm;
      if (c >= SPB * G * 3) break;  // wave-uniform
      const int part = c % 3, i = (c / 3) % G, kk = c / (3 * G);
      const int ky = min(max(r - y0 - i + g.h, 0), g.kw - 1);  // rows outside the kernel are copied, not used
      const int ks = min(s * SPB + kk, g.nks - 1);
      const int o = (((q15[i] * g.kw + ky) * g.nks + ks) * 3 + part) * 1024;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(br, (__attribute__((address_space(3))) void*)(buf + c * 1024), 16,
                                               lane * 16, uni(o), 0, 0);
    }
  };

  // The rows of this group, class by class.  Several groups walk nj rows of
  // each class together (past the last one a row is not used); a group alone takes
  // the rows there are.
  auto first = [&](int lap) { return rlo + ((lap * WK + wk - rlo) & (kClasses - 1)); };
  int lap = 0, j = 0, r = first(0);
  if (WK == 1)
    while (r > rhi) r = first(++lap);
  issue_b(r, 0, Bb);
  load_row(min(r, H - 1));
  store_row(Ab);
  int t = 0;
  for (int n = 0;; ++n) {
    int lap2 = lap, r2 = r + kClasses;  // the row after this one
    if (WK == 1) {
      while (r2 > rhi && ++lap2 < S::kLaps) r2 = first(lap2);
    } else if (++j == nj) {
      j = 0;
      r2 = first(++lap2);
    }
    const bool lastrow = lap2 == S::kLaps;
    const char* A = Ab + (n & 1) * S::kA;
    unsigned use = 0;  // output rows whose kernel holds this input row
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int ky = r - y0 - i + g.h;
      use |= (unsigned)(r <= rhi && y0 + i < H && ky >= 0 && ky < g.kw) << i;
    }
    use = uni(use);
    for (int s = 0; s < ns; ++s, ++t) {
      // this stage's copies and the row's staged cells are in LDS, and every
      // wave is done with the buffers that are written next
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      if (!(lastrow && s + 1 >= ns)) issue_b(s + 1 < ns ? r : r2, s + 1 < ns ? s + 1 : 0, Bb + ((t + 1) & 1) * S::kB);
      if (s == 0 && !lastrow) load_row(min(r2, H - 1));
      if (s == 1 && !lastrow) store_row(Ab + ((n + 1) & 1) * S::kA);
      const char* B = Bb + (t & 1) * S::kB + lane * 16;
#pragma unroll
      for (int kk = 0; kk < SPB; ++kk) {
        const int ks = s * SPB + kk;
        if (ks >= g.nks || !use) continue;
        bf16x8 a[MT][3];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const bool v = (unsigned)(lens[m] + 2 * ks) < (unsigned)nL;
          const char* p = A + (lg & 1) * S::kHalf + (v ? slot0 + 16 * m + 2 * ks : S::kSlots - 1) * 16;
#pragma unroll
          for (int k = 0; k < 3; ++k) a[m][k] = *reinterpret_cast<const bf16x8*>(p + k * S::kPart);
        }
#pragma unroll
        for (int i = 0; i < G; ++i) {
          if (!((use >> i) & 1)) continue;
          bf16x8 b[3];
#pragma unroll
          for (int k = 0; k < 3; ++k) b[k] = *reinterpret_cast<const bf16x8*>(B + ((kk * G + i) * 3 + k) * 1024);
          constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
          for (int q = 0; q < 6; ++q)
#pragma unroll
            for (int m = 0; m < MT; ++m)
              acc[m][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m][pa[q]], b[pb[q]], acc[m][i], 0, 0, 0);
        }
      }
      if (ns == 1 && !lastrow) store_row(Ab + ((n + 1) & 1) * S::kA);
    }
    if (lap2 != lap && (WK == 1 || !lastrow)) {  // the class is complete
#pragma unroll
      for (int p = 0; p < (WK == 1 ? 1 : S::kSums - 1); ++p)
        if (WK == 1 || p == lap)
#pragma unroll
          for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < G; ++i) sum[p][m][i] = WK == 1 ? sum[p][m][i] + acc[m][i] : acc[m][i];
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < G; ++i) acc[m][i] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    if (lastrow) break;
    lap = lap2;
    r = r2;
  }

  if constexpr (WK > 1) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int i = 0; i < G; ++i) sum[S::kSums - 1][m][i] = acc[m][i];  // the last lap's
    __syncthreads();
    // [group - 1][lap][wave][MT][G][lane]
    floatx4* red = reinterpret_cast<floatx4*>(sm) + wm * MT * G * 64 + lane;
    constexpr int kOne = WM * MT * G * 64;
    if (wk > 0) {
#pragma unroll
      for (int p = 0; p < S::kSums; ++p)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int i = 0; i < G; ++i) red[((wk - 1) * S::kSums + p) * kOne + (m * G + i) * 64] = sum[p][m][i];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int c = 1; c < kClasses; ++c)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < G; ++i)
          sum[0][m][i] += c % WK == 0 ? sum[c / WK % S::kSums][m][i]
                                      : red[((c % WK - 1) * S::kSums + c / WK) * kOne + (m * G + i) * 64];
  }
  if (lr >= kN) return;
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = M0 + 16 * (wm * MT + m) + 4 * lg + j;
      if (c >= NC) continue;
      const int img = c / nL, x = kN * (c - img * nL) + lr;
      if (x >= W || (any && marks.image_marked(call, src ? src[img] : img))) continue;
      float* o = out + (size_t)(dst ? dst[img] : img) * W * H + x;
#pragma unroll
      for (int i = 0; i < G; ++i) {
        if (y0 + i >= H) continue;
        float* d = o + (size_t)(y0 + i) * W;
        *d = dst ? *d + sum[0][m][i][j] : sum[0][m][i][j];
      }
    }
}

typedef void (*SplitKernel)(const float*, SplitGeo, const uintx4*, float*, const int32_t*, const int32_t*, MexMarks,
                            int);
struct SplitVariant {
  SplitKernel fn;
  int wm, wk, mt, g, spb, lds, per_cu;
  double step;  // matrix and LDS cycles of a K-step
};
template <int WM, int WK, int MT, int G, int SPB>
SplitVariant variant(double step) {
  using S = SplitShape<WM, WK, MT, G, SPB>;
  return {&k_mex_split<WM, WK, MT, G, SPB>, WM, WK, MT, G, SPB, S::kLds, S::kPerCu, step};
}

}  // namespace

static int split_lenslets(int kw, int* a, int* b) {
  const int h = kw / 2;
  *a = (h + kN - 1) / kN;
  *b = kN * *a - h;
  return (kw + 13 + *b) / kN + 1;
}

static int split_nks(int kw) {
  int a, b;
  return (split_lenslets(kw, &a, &b) + 1) / 2;
}

bool mex_split_takes(int64_t W, int64_t H, int64_t images, int kw) {
  // Kernels 1 and 3 pixels wide have too few products to pay for the operand table,
  // the look through the bitmaps and the two launches: the FP32 form alone takes 17
  // and 22 us for 150 x 137 (split form 23 and 28), 126 us for 396 x 396 x 96 at 3 (142);
  // at 5 it takes 26 and 192 us (25 and 126).  32-bit element offsets into the
  // bitmaps and the M row count.
  return kw % 2 == 1 && kw > 3 && kw <= kMexMfmaMaxKw && (double)W * H * images < 2147483648.0 && split_nks(kw) * 2 <= kMaxL;
}

size_t mex_split_bytes(int kw) { return (size_t)kN * kw * split_nks(kw) * 3 * 1024; }

hipError_t launch_mex_split_prep(const MexCall& c, const float* K, size_t image, hipStream_t st) {
  int a, b;
  split_lenslets(c.kw, &a, &b);
  const int nks = split_nks(c.kw);
  const size_t total = (size_t)kN * c.kw * nks * 64;
  const int nbt = (int)std::min<size_t>((total + 255) / 256, 4096);
  const int nbi = (int)std::max<size_t>(1, std::min<size_t>((image + 1023) / 1024, 2048 / c.images));
  const int64_t grid = nbt + (c.scan ? nbi * c.images : 0);
  if (grid > 0x7fffffff) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL(k_mex_split_prep, dim3((unsigned)grid), dim3(256), 0, st, K, c.kw, b, nks, (uintx4*)c.table, nbt,
                     c.scan, image, nbi, c.marks, c.sets);
  return hipGetLastError();
}

// Estimated cycles of a shape: the rounds that the XCD with the most row groups
// takes on its 32 CUs, the groups with the most input rows first.  A CU
// that holds e workgroups takes for a row the longer of all their K-steps and of
// one workgroup's chain, its own K-steps with a latency of 630 cycles each and
// 500 per barrier; a round 20000 more.  The cycles of each shape's K-step and these
// constants are fitted to 110 sizes (90 to 500 pixels, 1 to 128 bitmaps, kw 31 to 251): the
// estimates are 6 % off in the mean, and the shape chosen by them is 1.4 % slower than the
// best of 19.  396 x 396, kw = 241: 96 bitmaps take <8, 1, 2, 2, 2>, two workgroups per
// CU (8.4 ms; <8, 1, 3, 4, 2>, one per CU, 9.0), 10 bitmaps <2, 4, 2, 3, 1> (1.49; 1.95 to 2.1 with one
// group of waves), one small bitmap <1, 8, 1, 1, 1> (eight waves share the kernel's rows).
static double split_cycles(const SplitVariant& v, const SplitGeo& g, int64_t cells) {
  const int64_t nyg = (g.H + v.g - 1) / v.g, nmb = (cells + 16 * v.mt * v.wm - 1) / (16 * v.mt * v.wm);
  const int64_t wgs = (nyg + 7) / 8 * nmb, slots = 32 * v.per_cu, rounds = (wgs + slots - 1) / slots;
  const double own = g.nks * v.step, chain = own + 630.0 * g.nks + 500.0 * ((g.nks + v.spb - 1) / v.spb);
  const int64_t skip = (rounds + 63) / 64;  // of many rounds, 64 are looked at
  double t = 0.0;
  for (int64_t k = 0; k < rounds; k += skip) {
    const int64_t rank = std::min(nyg - 1, k * slots / nmb * 8);
    const int64_t y0 = v.g * ((rank & 1) ? nyg / 2 - (rank + 1) / 2 : nyg / 2 + rank / 2);
    const int64_t most = std::min<int64_t>(g.H - 1, y0 + v.g - 1 + g.h) - std::max<int64_t>(0, y0 - g.h) + 1;
    const double rows = v.wk == 1 ? (double)most : (double)(kClasses / v.wk) * ((most - 1) / kClasses + 1);
    const int64_t share = std::min<int64_t>(v.per_cu, (wgs - k * slots + 31) / 32);
    t += std::min(skip, rounds - k) * (rows * std::max(share * own, chain) + 20000.0);
  }
  return t;
}

hipError_t launch_mex_split(const MexCall& c, const float* in, int64_t W, int64_t H, int64_t n,
                            const int32_t* src, const int32_t* dst, float* out, hipStream_t st) {
  const int kw = c.kw;
  static const SplitVariant variants[] = {
      variant<8, 1, 2, 2, 2>(1190), variant<8, 1, 1, 2, 2>(600),  variant<4, 1, 3, 3, 2>(1500),
      variant<4, 1, 2, 4, 2>(1245), variant<4, 2, 2, 2, 1>(840),  variant<2, 4, 2, 3, 1>(1460),
      variant<2, 4, 3, 2, 1>(1715), variant<2, 4, 2, 2, 1>(890),  variant<1, 8, 2, 1, 1>(505),
      variant<1, 8, 1, 1, 1>(75),
  };
  static const hipError_t attr = [] {
    for (const SplitVariant& v : variants) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(v.fn),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }();
  if (attr != hipSuccess) return attr;
  SplitGeo g;
  int b;
  g.W = (int)W;
  g.H = (int)H;
  g.n = (int)n;
  g.kw = kw;
  g.h = kw / 2;
  g.nL = (int)((W + kN - 1) / kN);
  (void)split_lenslets(kw, &g.a, &b);
  g.nks = split_nks(kw);
  const int64_t cells = n * g.nL;
  const SplitVariant* best = nullptr;
  double best_t = 0.0;
  for (const SplitVariant& v : variants) {
    const double t = split_cycles(v, g, cells);
    if (!best || t < best_t) {
      best = &v;
      best_t = t;
    }
  }
  g.nyg = (int)((H + best->g - 1) / best->g);
  g.nmb = (int)((cells + 16 * best->mt * best->wm - 1) / (16 * best->mt * best->wm));
  const int64_t grid = (int64_t)((g.nyg + 7) / 8) * 8 * g.nmb;
  if (grid > 0x7fffffff) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL(best->fn, dim3((unsigned)grid), dim3(64 * best->wm * best->wk), best->lds, st, in, g,
                     (const uintx4*)c.table, out, src, dst, c.marks, c.sets);
  return hipGetLastError();
}

}  // namespace mlf
