// wgrad.hip -- the projections' weight gradients on the bf16 matrix cores, at fp32
// accuracy.
//
// P (m x k) = A (m x n) . B (k x n)^T over all n = batch * time columns, where each
// operand is a real (rows, n) array or a complex one, whose row r counts as the two
// real rows 2r (real part) and 2r + 1 (imaginary part).  The closing pass turns P
// into what the callers want:
//   complex . complex: G X^H  (rqf_models/ops/selective_scan.py:145, the autograd
//     of W @ h), from the four real products of each pair of rows;
//   real . real:       G X^T  (rqf_models/backbones/rqf/selective.py:78-97);
//   real . complex:    G [Re X; Im X]^T  (train.py:130), without the [Re; Im] copy;
//   complex . real:    [Re G; Im G] X^T  (rqf_models/ops/fbt_scan_kernel.py:993-996).
//
// The result is small and the sum is long, so the columns are cut into splits, one
// block per (tile of P, split); the partial tiles are added in order, in fp64.  Where all
// of them would take much memory, the columns go through in passes of as many splits as
// fit, each pass adding its tiles to fp64 sums.
#include "rqf_device.h"
#include "rqf_scan.h"
#include "rqf_split.h"

#include <algorithm>

using namespace rqf;

namespace {

// Both operands go through LDS: a stage is 32 columns, and a thread splits 8
// consecutive columns of one complex row (or of two real ones) into the parts of
// two 16-byte units, the operand layout of v_mfma_f32_16x16x32_bf16.  The 32-column
// instruction halves the roundings of the sum against the 16-column one, and draws
// less power (2006 against 1781 TFLOP/s on random bits, where the clock drops).
//
// T: 16-row blocks per wavefront and operand; a block is 2 x 2 wavefronts, so
// 32 T x 32 T of P.  LDS is 48 KB at T = 4 (three blocks per CU), single buffered:
// one block's splitting runs beside another's MFMAs.
constexpr int kThreadsW = 256;
constexpr int kStage = 32;
// Most columns per split: bounds the roundings one partial sum collects.
constexpr int64_t kSplitCols = 2048;

struct WgradArgs {
  const float* a;
  const float* b;
  int64_t ar, br;  // source rows
  int64_t n;
  int64_t n0, n1;  // columns of this pass
  int64_t cols;    // columns per split, a multiple of kStage
  int64_t mt, kt;  // tiles of P
  int64_t tiles;   // mt * kt * splits of the pass
  float* partial;  // (splits of the pass, mt * 32 T, kt * 32 T)
};

// Real row `row` of an operand at column n (fallback and tail).
template <bool CPLX>
__device__ __forceinline__ float one(const float* p, int64_t rows, int64_t row, int64_t n,
                                     int64_t ld, int64_t end) {
  if (n >= end) return 0.0f;
  if (CPLX) {
    const int64_t r = row >> 1 < rows ? row >> 1 : rows - 1;
    return p[2 * (r * ld + n) + (row & 1)];
  }
  return p[(row < rows ? row : rows - 1) * ld + n];
}

template <int T, bool AC, bool BC>
__global__ __launch_bounds__(kThreadsW, 2) void wgrad_kernel(const WgradArgs g) {
  constexpr int kRows = 32 * T;               // real rows of an operand tile
  constexpr int kGroup = 3 * kRows + 4;       // units of a group of 8 columns; the 4 keeps
                                              // eight lanes' stores on distinct banks
  constexpr int kUnits = 4 * kGroup;
  constexpr int kPairs = 2 * kRows;           // unit pairs of an operand's stage
  constexpr int kPer = 2 * kPairs / kThreadsW;  // pairs a thread loads and splits
  __shared__ u32x4 s_op[2][kUnits];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), w = wave_id();
  // The tiles of one split share its columns: one XCD runs them.
  const int64_t id = xcd_contiguous(blockIdx.x, g.tiles);
  const int64_t per = g.mt * g.kt, split = id / per;
  const int64_t m0 = (id % per) / g.kt * kRows, k0 = (id % per) % g.kt * kRows;
  const int64_t c0 = g.n0 + split * g.cols, c1 = std::min(c0 + g.cols, g.n1);

  // Thread t's pair u: group u % 4 of complex row u / 4, or of real rows u / 4 and
  // u / 4 + kRows / 2.  Rows past the end repeat the last one; they only reach
  // entries of P that are never read.
  const float* src[kPer][2];
  bool cx[kPer];
  int op[kPer], unit[kPer][2];
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const int v = tid + r * kThreadsW;
    op[r] = kPairs == kThreadsW ? r : __builtin_amdgcn_readfirstlane(v / kPairs);
    const int u = v % kPairs, row = u >> 2, grp = u & 3;
    cx[r] = op[r] ? BC : AC;
    const float* p = op[r] ? g.b : g.a;
    const int64_t rows = op[r] ? g.br : g.ar, t0 = op[r] ? k0 : m0;
    if (cx[r]) {
      const int64_t q = std::min(t0 / 2 + row, rows - 1);
      src[r][0] = p + 2 * (q * g.n + 8 * grp);
      src[r][1] = src[r][0] + 8;
      unit[r][0] = grp * kGroup + 2 * row;
      unit[r][1] = unit[r][0] + 1;
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int64_t q = std::min(t0 + row + h * (kRows / 2), rows - 1);
        src[r][h] = p + q * g.n + 8 * grp;
        unit[r][h] = grp * kGroup + row + h * (kRows / 2);
      }
    }
  }
  float ld[kPer][16];
  auto fetch = [&](int64_t c) {
    if (c + kStage <= c1) {
#pragma unroll
      for (int r = 0; r < kPer; ++r) {
        const int64_t o = cx[r] ? 2 * c : c;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const f4u v = *reinterpret_cast<const f4u*>(src[r][h] + o + 4 * q);
#pragma unroll
            for (int e = 0; e < 4; ++e) ld[r][8 * h + 4 * q + e] = v[e];
          }
      }
    } else {
#pragma unroll
      for (int r = 0; r < kPer; ++r) {
        const int grp = (tid + r * kThreadsW) & 3;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            // floats h * 8 + e of the pair: two per column of a complex row
            const int64_t col = c + 8 * grp + (cx[r] ? 4 * h + e / 2 : e);
            ld[r][8 * h + e] = col < c1 ? src[r][h][(cx[r] ? 2 * c : c) + e] : 0.0f;
          }
      }
    }
  };
  // The sum of the leading products and that of the five small ones: added to one
  // sum, each small product would round it once more.
  v4f acc[T][T], low[T][T];
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[i][j][v] = low[i][j][v] = 0.0f;
  const int wm = (w & 1) * 16 * T, wk = (w >> 1) * 16 * T;
  const int frag = (lane >> 4) * kGroup + (lane & 15);

  fetch(c0);
#pragma clang loop unroll(disable)
  for (int64_t c = c0; c < c1; c += kStage) {
#pragma unroll
    for (int r = 0; r < kPer; ++r)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = cx[r] ? ld[r][2 * e + h] : ld[r][8 * h + e];
        Split8 s;
        split8_scaled(x, s);
        u32x4* d = &s_op[op[r]][unit[r][h]];
        d[0] = s.h;
        d[kRows] = s.m;
        d[2 * kRows] = s.l;
      }
    __syncthreads();
    if (c + kStage < c1) fetch(c + kStage);
    Split8 b[T];
#pragma unroll
    for (int j = 0; j < T; ++j) {
      const u32x4* p = &s_op[1][frag + wk + 16 * j];
      b[j].h = p[0];
      b[j].m = p[kRows];
      b[j].l = p[2 * kRows];
    }
#pragma unroll
    for (int i = 0; i < T; ++i) {
      Split8 a;
      const u32x4* p = &s_op[0][frag + wm + 16 * i];
      a.h = p[0];
      a.m = p[kRows];
      a.l = p[2 * kRows];
#pragma unroll
      for (int t = 0; t < 5; ++t)
#pragma unroll
        for (int j = 0; j < T; ++j) low[i][j] = mfma_part(t, a, b[j], low[i][j]);
#pragma unroll
      for (int j = 0; j < T; ++j) acc[i][j] = mfma_part(5, a, b[j], acc[i][j]);
    }
    __syncthreads();
  }

  // As in the projection GEMM: a wavefront with a value that is not the sum of three
  // bf16 values computes its tile on the fp32 matrix cores.  Rows past the end repeat
  // the last row, so they decide nothing of their own.
  bool finite = true;
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        acc[i][j][v] = (acc[i][j][v] + low[i][j][v]) * kSplitUnscale;
        finite = finite && fabsf(acc[i][j][v]) <= kFltMax;
      }
  const bool redo = __ballot(!finite) != 0;
  // Lane l holds P[4*(l/16) + v][l%16] of each 16 x 16 block.
  const int64_t ldp = g.kt * kRows;
  float* out = g.partial + (split * g.mt * kRows + m0 + wm + 4 * (lane >> 4)) * ldp + k0 + wk +
               (lane & 15);
  auto store = [&](int i, int j, const v4f& c) {
#pragma unroll
    for (int v = 0; v < 4; ++v) out[(16 * i + v) * ldp + 16 * j] = c[v];
  };
  if (redo) {
#pragma clang loop unroll(disable)
    for (int ij = 0; ij < T * T; ++ij) {
      const int i = ij / T, j = ij % T;
      v4f c;
#pragma unroll
      for (int v = 0; v < 4; ++v) c[v] = 0.0f;
#pragma clang loop unroll(disable)
      for (int64_t n = c0; n < c1; n += 4) {  // lane l: row l % 16, column n + l / 16
        const int64_t q = n + (lane >> 4);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(
            one<AC>(g.a, g.ar, m0 + wm + 16 * i + (lane & 15), q, g.n, c1),
            one<BC>(g.b, g.br, k0 + wk + 16 * j + (lane & 15), q, g.n, c1), c, 0, 0, 0);
      }
      store(i, j, c);
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j) store(i, j, acc[i][j]);
}

// Sum of the splits' partials in fp64, in a fixed order, and the callers' layouts.
// A block takes 16 elements of the output (a complex value counts as one); 16
// threads share an element's splits, thread q adding q, q + 16, ... in order, so
// that hundreds of splits of a small matrix do not make one long chain of loads.
// sums: of several passes, the elements' sums of the passes before (after the first).
template <bool AC, bool BC>
__global__ __launch_bounds__(256) void wgrad_close_kernel(const float* __restrict__ partial,
                                                          int64_t splits, int64_t mp, int64_t ldp,
                                                          int64_t ar, int64_t br, bool first,
                                                          bool last, double2* __restrict__ sums,
                                                          float* __restrict__ out) {
  __shared__ double s_sum[16][16][2];
  const int64_t rows = AC && !BC ? 2 * ar : ar, cols = BC && !AC ? 2 * br : br;
  const int64_t total = rows * cols, step = mp * ldp;
  const int e = threadIdx.x & 15, q = threadIdx.x >> 4;
  for (int64_t base = (int64_t)blockIdx.x * 16; base < total; base += (int64_t)gridDim.x * 16) {
    const int64_t id = base + e;
    double re = 0.0, im = 0.0;
    if (id < total) {
      const int64_t m = id / cols, k = id % cols;
      if (AC && BC) {
        const float* p = partial + 2 * m * ldp + 2 * k;
#pragma unroll 4
        for (int64_t s = q; s < splits; s += 16) {
          const float* v = p + s * step;
          re += (double)v[0] + (double)v[ldp + 1];
          im += (double)v[ldp] - (double)v[1];
        }
      } else {
        // [Re; Im] rows (AC) or columns (BC) of the output against interleaved ones
        const int64_t pm = AC ? 2 * (m % ar) + m / ar : m, pk = BC ? 2 * (k % br) + k / br : k;
        const float* p = partial + pm * ldp + pk;
#pragma unroll 4
        for (int64_t s = q; s < splits; s += 16) re += (double)p[s * step];
      }
    }
    s_sum[q][e][0] = re;
    s_sum[q][e][1] = im;
    __syncthreads();
    if (q == 0 && id < total) {
      re = first ? 0.0 : sums[id].x;
      im = first ? 0.0 : sums[id].y;
      for (int v = 0; v < 16; ++v) {
        re += s_sum[v][e][0];
        im += s_sum[v][e][1];
      }
      if (!last) {
        sums[id] = make_double2(re, im);
      } else if (AC && BC) {
        out[2 * id] = (float)re;
        out[2 * id + 1] = (float)im;
      } else {
        out[id] = (float)re;
      }
    }
    __syncthreads();
  }
}

struct Plan {
  int t;
  int64_t mt, kt, splits, cols;
  int64_t per;   // splits per pass
  size_t sums;   // bytes of the fp64 sums, before the partials; none for a single pass
  size_t bytes;
};
// The partial tiles of one pass, unless a split's alone are more: 4096 tiles of 128 x 128.
// Complex 256 x 256 with n = 1024000 would take 512 MB at once, 4096 x 4096 134 GB.
constexpr size_t kPassBytes = (size_t)256 << 20;

// Tiles of 128 x 128, or of 64 x 64 where those would be mostly padding (192 x 128 real
// rows) or, at the 128 columns a split of small tiles may have, too few blocks for the CUs:
// real 264 x 256, n = 2048 23 us in 48 blocks of 128 x 128, 14 in 320 of 64 x 64; 520 x 512,
// n = 2048 35 / 31; complex 48 x 48, n = 4000 22 / 10.
Plan plan_of(int64_t ar, bool ac, int64_t br, bool bc, int64_t n) {
  Plan p;
  const int64_t mr = ac ? 2 * ar : ar, kr = bc ? 2 * br : br;
  const int64_t outputs = ac && bc ? ar * br : mr * kr;
  const auto area = [&](int64_t r) { return (mr + r - 1) / r * ((kr + r - 1) / r) * r * r; };
  const bool few = area(128) / (128 * 128) * (n / 128) < 512;
  p.t = few || 4 * area(64) <= 3 * area(128) ? 2 : 4;
  const int64_t r = 32 * p.t;
  p.mt = (mr + r - 1) / r;
  p.kt = (kr + r - 1) / r;
  // Three blocks for each of the 256 CUs, at most kSplitCols columns each and at least 256,
  // or 128 where that makes too few (real 16 x 16, n = 2048: 10.9 us with 256, 7.8 with 128).
  const int64_t tiles = p.mt * p.kt, fill = (768 + tiles - 1) / tiles;
  const int64_t least = p.t == 2 && tiles * (n / 128) < 512 ? 128 : 256;
  int64_t s = std::max(fill, (n + kSplitCols - 1) / kSplitCols);
  s = std::max<int64_t>(1, std::min(s, n / least));
  p.cols = ((n + s - 1) / s + kStage - 1) / kStage * kStage;
  p.splits = p.cols ? (n + p.cols - 1) / p.cols : 0;
  const size_t split = sizeof(float) * (size_t)(p.mt * r) * (size_t)(p.kt * r);
  const int64_t most = std::max<int64_t>(1, (int64_t)(kPassBytes / split));
  const int64_t passes = std::max<int64_t>(1, (p.splits + most - 1) / most);
  p.per = (p.splits + passes - 1) / passes;
  p.sums = passes > 1 ? sizeof(double2) * (size_t)outputs : 0;
  p.bytes = p.sums + split * (size_t)p.per;
  return p;
}

template <int T, bool AC, bool BC>
int launch(WgradArgs g, const Plan& p, double2* sums, float* out, hipStream_t s) {
  const int64_t total = (AC && !BC ? 2 : 1) * (BC && !AC ? 2 : 1) * g.ar * g.br;
  for (int64_t first = 0; first < p.splits; first += p.per) {
    const int64_t splits = std::min(p.per, p.splits - first);
    g.n0 = first * p.cols;
    g.n1 = std::min(g.n0 + splits * p.cols, g.n);
    g.tiles = p.mt * p.kt * splits;
    hipLaunchKernelGGL((wgrad_kernel<T, AC, BC>), dim3((unsigned)g.tiles), dim3(kThreadsW), 0, s, g);
    hipLaunchKernelGGL((wgrad_close_kernel<AC, BC>), dim3(stride_blocks((total + 15) / 16)),
                       dim3(256), 0, s, g.partial, splits, p.mt * 32 * T, p.kt * 32 * T, g.ar, g.br,
                       first == 0, first + p.per >= p.splits, sums, out);
  }
  const hipError_t err = hipGetLastError();
  return err == hipSuccess ? RQF_OK : (int)err;
}

template <bool AC, bool BC>
int launch(const WgradArgs& g, const Plan& p, double2* sums, float* out, hipStream_t s) {
  return p.t == 4 ? launch<4, AC, BC>(g, p, sums, out, s) : launch<2, AC, BC>(g, p, sums, out, s);
}

}  // namespace

extern "C" size_t rqf_weight_grad_workspace(int64_t a_rows, int32_t a_cplx, int64_t b_rows,
                                            int32_t b_cplx, int64_t n) {
  if (a_rows < 1 || b_rows < 1 || n < 1) return 0;
  return plan_of(a_rows, a_cplx != 0, b_rows, b_cplx != 0, n).bytes;
}

extern "C" int rqf_weight_grad(const float* a, int64_t a_rows, int32_t a_cplx, const float* b,
                               int64_t b_rows, int32_t b_cplx, int64_t n, float* out,
                               void* workspace, size_t workspace_bytes, rqf_stream_t stream) {
  if (a_rows < 1 || b_rows < 1 || n < 1) return RQF_ERR_ARG;
  if (!a || !b || !out) return RQF_ERR_ARG;
  if (((uintptr_t)a | (uintptr_t)b | (uintptr_t)out) & 3) return RQF_ERR_ALIGN;
  const Plan p = plan_of(a_rows, a_cplx != 0, b_rows, b_cplx != 0, n);
  if (!grid_fits(p.mt * p.kt * p.per, kThreadsW)) return RQF_ERR_ARG;
  if (!workspace || workspace_bytes < p.bytes) return RQF_ERR_WORKSPACE;
  if (p.sums && ((uintptr_t)workspace & 15)) return RQF_ERR_ALIGN;
  WgradArgs g;
  g.a = a;
  g.b = b;
  g.ar = a_rows;
  g.br = b_rows;
  g.n = n;
  g.cols = p.cols;
  g.mt = p.mt;
  g.kt = p.kt;
  double2* sums = (double2*)workspace;
  g.partial = (float*)((char*)workspace + p.sums);
  hipStream_t s = (hipStream_t)stream;
  if (a_cplx)
    return b_cplx ? launch<true, true>(g, p, sums, out, s) : launch<true, false>(g, p, sums, out, s);
  return b_cplx ? launch<false, true>(g, p, sums, out, s) : launch<false, false>(g, p, sums, out, s);
}
