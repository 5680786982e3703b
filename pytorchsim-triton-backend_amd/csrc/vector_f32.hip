// fp32 forms of the vector family for gfx950: RMSNorm over rows (and the column arm of the same
// reference case), row softmax, the SiLU gate, and the two-matmul SwiGLU block.  These serve the
// reference's own fp32 workload cases (tests/cases/workloads/{rmsnorm,softmax,swiglu}.py), which
// hold inputs and outputs in fp32 with tolerances down to rtol 1e-5: nothing is rounded below fp32.
// Rows move as 128-bit chunks of 4 floats with coalesced loads and stores; reductions are wave DPP /
// permlane steps plus one LDS pass across waves.
#include <algorithm>
#include <type_traits>

#include "ptb_common.h"

using namespace ptb;

namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ float exp_e(float x) { return __builtin_amdgcn_exp2f(x * 1.4426950408889634f); }

template <int TPR>
__device__ __forceinline__ float team_sum(float v, float* red) {
  if constexpr (TPR == kWave) return wave_sum(v);
  else return block_sum<TPR / kWave>(v, red);
}
template <int TPR>
__device__ __forceinline__ float team_max(float v, float* red) {
  if constexpr (TPR == kWave) return wave_max_nan(v);
  else return block_max_nan<TPR / kWave>(v, red);
}

// ---------------------------------------------------------------- RMSNorm over rows
// A team of TPR threads per row, VPT chunks of 4 per thread held in registers (one read, one write).
template <int TPR, int VPT>
__global__ __launch_bounds__(kBlock) void rmsnorm_rows_f32(const float* __restrict__ x, const float* __restrict__ w,
                                                           float* __restrict__ y, int64_t rows, int cols, float eps) {
  __shared__ float red[kBlock / kWave];
  constexpr int kTeams = kBlock / TPR;
  const int team = threadIdx.x / TPR, lt = threadIdx.x % TPR;
  const int64_t row = int64_t(blockIdx.x) * kTeams + team;
  const bool live = row < rows;
  const int chunks = cols >> 2;
  const f32x4v* xr = reinterpret_cast<const f32x4v*>(x + (live ? row : 0) * int64_t(cols));
  f32x4v v[VPT];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int c = lt + i * TPR;
    v[i] = (live && c < chunks) ? xr[c] : f32x4v{0.f, 0.f, 0.f, 0.f};
    ss += v[i].x * v[i].x + v[i].y * v[i].y + v[i].z * v[i].z + v[i].w * v[i].w;
  }
  ss = team_sum<TPR>(ss, red);
  const float r = 1.0f / sqrtf(ss / float(cols) + eps);
  if (!live) return;
  f32x4v* yr = reinterpret_cast<f32x4v*>(y + row * int64_t(cols));
  const f32x4v* wr = reinterpret_cast<const f32x4v*>(w);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int c = lt + i * TPR;
    if (c >= chunks) continue;
    const f32x4v wv = wr[c];
    yr[c] = f32x4v{(v[i].x * r) * wv.x, (v[i].y * r) * wv.y, (v[i].z * r) * wv.z, (v[i].w * r) * wv.w};
  }
}

// Rows too long for registers: one block per row, two passes over the row.
__global__ __launch_bounds__(kBlock) void rmsnorm_rows_f32_long(const float* __restrict__ x, const float* __restrict__ w,
                                                                float* __restrict__ y, int cols, float eps) {
  __shared__ float red[kBlock / kWave];
  const int64_t row = blockIdx.x;
  const int chunks = cols >> 2;
  const f32x4v* xr = reinterpret_cast<const f32x4v*>(x + row * int64_t(cols));
  float ss = 0.f;
  for (int c = threadIdx.x; c < chunks; c += kBlock) {
    const f32x4v a = xr[c];
    ss += a.x * a.x + a.y * a.y + a.z * a.z + a.w * a.w;
  }
  ss = block_sum<kBlock / kWave>(ss, red);
  const float r = 1.0f / sqrtf(ss / float(cols) + eps);
  f32x4v* yr = reinterpret_cast<f32x4v*>(y + row * int64_t(cols));
  const f32x4v* wr = reinterpret_cast<const f32x4v*>(w);
  for (int c = threadIdx.x; c < chunks; c += kBlock) {
    const f32x4v a = xr[c], wv = wr[c];
    yr[c] = f32x4v{(a.x * r) * wv.x, (a.y * r) * wv.y, (a.z * r) * wv.z, (a.w * r) * wv.w};
  }
}

// ---------------------------------------------------------------- column arm: rsqrt(mean_i x[i,j]^2 + eps)
// 64 columns per workgroup, its 4 waves splitting the rows; each lane walks its column.
__global__ __launch_bounds__(kBlock) void col_rms_f32(const float* __restrict__ x, float* __restrict__ c,
                                                      int64_t rows, int64_t cols, float eps) {
  __shared__ float part[4][64];
  const int64_t j = int64_t(blockIdx.x) * 64 + (threadIdx.x & 63);
  const int slice = threadIdx.x >> 6;
  float ss = 0.f;
  if (j < cols)
    for (int64_t i = slice; i < rows; i += 4) {
      const float v = x[i * cols + j];
      ss += v * v;
    }
  part[slice][threadIdx.x & 63] = ss;
  __syncthreads();
  if (slice == 0 && j < cols) {
    const float s = (part[0][threadIdx.x] + part[1][threadIdx.x]) + (part[2][threadIdx.x] + part[3][threadIdx.x]);
    c[j] = 1.0f / sqrtf(s / float(rows) + eps);
  }
}

// ---------------------------------------------------------------- row softmax
template <int TPR, int VPT>
__global__ __launch_bounds__(kBlock) void softmax_rows_f32(const float* __restrict__ x, float* __restrict__ y,
                                                           int64_t rows, int cols) {
  __shared__ float red[kBlock / kWave];
  constexpr int kTeams = kBlock / TPR;
  const int team = threadIdx.x / TPR, lt = threadIdx.x % TPR;
  const int64_t row = int64_t(blockIdx.x) * kTeams + team;
  const bool live = row < rows;
  const int chunks = cols >> 2;
  const f32x4v* xr = reinterpret_cast<const f32x4v*>(x + (live ? row : 0) * int64_t(cols));
  f32x4v v[VPT];
  float m = -__builtin_inff();
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int c = lt + i * TPR;
    const bool in = live && c < chunks;
    v[i] = in ? xr[c] : f32x4v{0.f, 0.f, 0.f, 0.f};
    if (in) m = max_nan(m, max_nan(max_nan(v[i].x, v[i].y), max_nan(v[i].z, v[i].w)));
  }
  m = team_max<TPR>(m, red);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int c = lt + i * TPR;
    if (!(live && c < chunks)) continue;
    v[i] = f32x4v{exp_e(v[i].x - m), exp_e(v[i].y - m), exp_e(v[i].z - m), exp_e(v[i].w - m)};
    s += (v[i].x + v[i].y) + (v[i].z + v[i].w);
  }
  s = team_sum<TPR>(s, red);
  if (!live) return;
  f32x4v* yr = reinterpret_cast<f32x4v*>(y + row * int64_t(cols));
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int c = lt + i * TPR;
    if (c >= chunks) continue;
    yr[c] = f32x4v{v[i].x / s, v[i].y / s, v[i].z / s, v[i].w / s};
  }
}

// Long rows: one block per row, three passes over the row.
__global__ __launch_bounds__(kBlock) void softmax_rows_f32_long(const float* __restrict__ x, float* __restrict__ y,
                                                                int cols) {
  __shared__ float red[kBlock / kWave];
  const int64_t row = blockIdx.x;
  const int chunks = cols >> 2;
  const f32x4v* xr = reinterpret_cast<const f32x4v*>(x + row * int64_t(cols));
  float m = -__builtin_inff();
  for (int c = threadIdx.x; c < chunks; c += kBlock) {
    const f32x4v a = xr[c];
    m = max_nan(m, max_nan(max_nan(a.x, a.y), max_nan(a.z, a.w)));
  }
  m = block_max_nan<kBlock / kWave>(m, red);
  float s = 0.f;
  for (int c = threadIdx.x; c < chunks; c += kBlock) {
    const f32x4v a = xr[c];
    s += (exp_e(a.x - m) + exp_e(a.y - m)) + (exp_e(a.z - m) + exp_e(a.w - m));
  }
  s = block_sum<kBlock / kWave>(s, red);
  f32x4v* yr = reinterpret_cast<f32x4v*>(y + row * int64_t(cols));
  for (int c = threadIdx.x; c < chunks; c += kBlock) {
    const f32x4v a = xr[c];
    yr[c] = f32x4v{exp_e(a.x - m) / s, exp_e(a.y - m) / s, exp_e(a.z - m) / s, exp_e(a.w - m) / s};
  }
}

// ---------------------------------------------------------------- SiLU gate
// out[r, j] = (g / (1 + exp(-g))) * u, g = gu[r, j], u = gu[r, inter + j]; 4 outputs per thread.
__global__ __launch_bounds__(kBlock) void silu_mul_f32(const float* __restrict__ gu, float* __restrict__ out,
                                                       int64_t rows, int64_t inter) {
  const int64_t q = inter >> 2;   // chunks per row
  const int64_t total = rows * q;
  for (int64_t t = int64_t(blockIdx.x) * kBlock + threadIdx.x; t < total; t += int64_t(gridDim.x) * kBlock) {
    const int64_t r = t / q, c = t - r * q;
    const f32x4v g = reinterpret_cast<const f32x4v*>(gu + r * 2 * inter)[c];
    const f32x4v u = reinterpret_cast<const f32x4v*>(gu + r * 2 * inter + inter)[c];
    reinterpret_cast<f32x4v*>(out + r * inter)[c] =
        f32x4v{(g.x / (1.0f + exp_e(-g.x))) * u.x, (g.y / (1.0f + exp_e(-g.y))) * u.y,
               (g.z / (1.0f + exp_e(-g.z))) * u.z, (g.w / (1.0f + exp_e(-g.w))) * u.w};
  }
}

// ---------------------------------------------------------------- SwiGLU block
// o = silu(x @ wg) * (x @ wu) for fp32 x [M, K], wg / wu [K, N] on v_mfma_f32_32x32x2_f32 (fp32 operands
// and accumulation): a wave owns a 32x32 block of both products, WR waves tile a workgroup's 32 WR
// rows x 32 columns and WK waves split each K slab of WK * KW columns.  Slabs pass through registers
// into two LDS buffers, the next slab's loads in flight under the current one's MFMAs; loads are dwords,
// so any size and 4-byte alignment takes this path.  Within a slab a lane's half (lane / 32) takes KW / 2
// consecutive k of its wave's KW: the order is the same for both operands, and x rows are then read
// four k at a time.  The K-split waves' sums meet in LDS, in wave order (splitting K also keeps the
// error against 64 bits below the plain fp32 sum's, 4e-7 .. 7e-7 relative against 9e-7 at K = 1024).
// Bound by the fp32 matrix rate (64 cycles an MFMA) and, per slab, by the barrier and the staging around
// its 256 .. 1024 cycles of MFMAs; measured beside its predecessor, one FMA per lane, product and k over
// 4x4 outputs a thread: 777x1024x2816 (m, k, n) 245 -> 102 us, 2048x2048x4096 1000 -> 594 (116 TFLOP/s of
// the 141 that a large fp32 library product reaches here), 1x2048x4096 395 -> 30.  Four waves of 64x64
// outputs, without the K split, were no faster and lost accuracy.
template <int WR, int WK, int KW>
struct SwShape {
  static constexpr int kThreads = 64 * WR * WK;
  static constexpr int BM = 32 * WR, BN = 32, KS = WK * KW;
  static constexpr int kPitchA = KS + 4;                      // floats: rows start 4 banks apart
  static constexpr int kA = BM * kPitchA, kB = KS * 2 * BN;   // floats; a B row is 32 gate | 32 up
  static constexpr int kSlab = kA + kB, kRed = WK * WR * 2048;
  static constexpr int kSmem = 2 * kSlab > kRed ? 2 * kSlab : kRed;
  static constexpr int kLoadA = BM * KS / kThreads, kLoadB = KS * BN / kThreads;   // kLoadB of each product
  static_assert(KW % 8 == 0 && kThreads % KS == 0 && kThreads % BN == 0, "a thread keeps its k of A and column of B");
  static_assert(BM * KS % kThreads == 0 && KS * BN % kThreads == 0, "whole loads per thread");
};
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_range(const float* p, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, uint32_t(bytes < 0xfffffffcll ? bytes : 0xfffffffcll),
                                           0x00020000);
}
__device__ __forceinline__ float buffer_f32(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
// WIDE: byte offsets within a workgroup's rows of x or a slab of the weights may pass 2^32.  Its column blocks
// run over the grid's x and z: a launch takes fewer than 2^32 threads along x.
template <int WR, int WK, int KW, bool WIDE>
__global__ __launch_bounds__(64 * WR * WK) void swiglu_f32(
    const float* __restrict__ x, const float* __restrict__ wg, const float* __restrict__ wu, float* __restrict__ o,
    int M, int N, int K) {
  using Sh = SwShape<WR, WK, KW>;
  using Off = std::conditional_t<WIDE, int64_t, uint32_t>;
  __shared__ __attribute__((aligned(16))) float smem[Sh::kSmem];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wk = wave % WK, wr = wave / WK;
  const int m0 = int(blockIdx.y) * Sh::BM;
  const int64_t nblock = WIDE ? int64_t(blockIdx.z) * gridDim.x + blockIdx.x : blockIdx.x;
  if (WIDE && nblock * Sh::BN >= N) return;   // uniform over the workgroup
  const int n0 = int(nblock * Sh::BN);
  const int col = lane & 31, h = lane >> 5;

  // Loads: thread -> k ka of rows ra0, ra0 + kThreads / KS, ... of x; column cb of rows kb0, kb0 +
  // kThreads / BN, ... of each weight.  Rows past M and columns past N repeat the last one (their
  // outputs are not stored); k past K reads as zero, which only the last slab has to test.
  constexpr int kStepA = Sh::kThreads / Sh::KS, kStepB = Sh::kThreads / Sh::BN;
  const int ka = tid % Sh::KS, ra0 = tid / Sh::KS, cb = tid % Sh::BN, kb0 = tid / Sh::BN;
  Off aoff[Sh::kLoadA], boff[Sh::kLoadB];
#pragma unroll
  for (int i = 0; i < Sh::kLoadA; ++i) aoff[i] = (Off(min(m0 + ra0 + i * kStepA, M - 1) - m0) * Off(K) + Off(ka)) * 4;
#pragma unroll
  for (int i = 0; i < Sh::kLoadB; ++i) boff[i] = (Off(kb0 + i * kStepB) * Off(N) + Off(min(n0 + cb, N - 1))) * 4;
  float ra[Sh::kLoadA], rg[Sh::kLoadB], ru[Sh::kLoadB];
  auto load = [&](int64_t k0) __attribute__((always_inline)) {
    const float* const px = x + int64_t(m0) * K + k0;
    const float* const pg = wg + k0 * N;
    const float* const pu = wu + k0 * N;
    if constexpr (WIDE) {
#pragma unroll
      for (int i = 0; i < Sh::kLoadA; ++i) ra[i] = k0 + ka < K ? px[aoff[i] / 4] : 0.f;
#pragma unroll
      for (int i = 0; i < Sh::kLoadB; ++i) {
        const bool in = k0 + kb0 + i * kStepB < K;
        rg[i] = in ? pg[boff[i] / 4] : 0.f;
        ru[i] = in ? pu[boff[i] / 4] : 0.f;
      }
    } else {
      // the ranges end at the last element: rows of the weights past K read as zero; x past K within a
      // row reads the next row and is zeroed below (an infinity there must not meet a zero weight)
      const auto rx = make_range(px, (int64_t(M - m0) * K - k0) * 4);
      const auto rwg = make_range(pg, (K - k0) * N * 4), rwu = make_range(pu, (K - k0) * N * 4);
#pragma unroll
      for (int i = 0; i < Sh::kLoadA; ++i) ra[i] = buffer_f32(rx, aoff[i]);
#pragma unroll
      for (int i = 0; i < Sh::kLoadB; ++i) rg[i] = buffer_f32(rwg, boff[i]);
#pragma unroll
      for (int i = 0; i < Sh::kLoadB; ++i) ru[i] = buffer_f32(rwu, boff[i]);
    }
  };
  // x past K, zeroed once its loads are waited for
  auto zero_tail = [&](int64_t k0) __attribute__((always_inline)) {
    if (!WIDE && k0 + Sh::KS > K) {
#pragma unroll
      for (int i = 0; i < Sh::kLoadA; ++i) ra[i] = k0 + ka < K ? ra[i] : 0.f;
    }
  };
  auto store = [&](float* slab) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < Sh::kLoadA; ++i) slab[(ra0 + i * kStepA) * Sh::kPitchA + ka] = ra[i];
    float* const b = slab + Sh::kA + kb0 * (2 * Sh::BN) + cb;
#pragma unroll
    for (int i = 0; i < Sh::kLoadB; ++i) {
      b[i * kStepB * 2 * Sh::BN] = rg[i];
      b[i * kStepB * 2 * Sh::BN + 32] = ru[i];
    }
  };
  f32x16 ag, au;
#pragma unroll
  for (int e = 0; e < 16; ++e) ag[e] = au[e] = 0.f;
  auto compute = [&](const float* slab) __attribute__((always_inline)) {
    const float* pa = slab + (32 * wr + col) * Sh::kPitchA + wk * KW + h * (KW / 2);
    const float* pb = slab + Sh::kA + (wk * KW + h * (KW / 2)) * (2 * Sh::BN) + col;
    // every fragment of the slab requested before the first MFMA, which waits for its own only
    f32x4v a[KW / 8];
    float bg[KW / 2], bu[KW / 2];
#pragma unroll
    for (int s = 0; s < KW / 2; ++s) {
      if (s % 4 == 0) a[s / 4] = *reinterpret_cast<const f32x4v*>(pa + s);
      bg[s] = pb[s * 2 * Sh::BN];
      bu[s] = pb[s * 2 * Sh::BN + 32];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < KW / 2; ++s) {
      ag = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s / 4][s % 4], bg[s], ag, 0, 0, 0);
      au = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s / 4][s % 4], bu[s], au, 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // slab s in buffer s % 2: the next slab's loads run under this one's MFMAs and go into the other
  // buffer, which every wave left before the barrier that ended the previous slab
  load(0);
  zero_tail(0);
  store(smem);
  __syncthreads();
  int buf = 0;
  for (int64_t k0 = 0; k0 < K; k0 += Sh::KS) {
    const bool more = k0 + Sh::KS < K;
    if (more) load(k0 + Sh::KS);
    compute(smem + buf * Sh::kSlab);
    buf ^= 1;
    if (more) {
      zero_tail(k0 + Sh::KS);
      store(smem + buf * Sh::kSlab);
    }
    __syncthreads();
  }
  // accumulator e of lane: row 8 (e / 4) + 4 h + e % 4 of the wave's block, column lane % 32;
  // the slabs are done with: the waves' sums take their place
  float* const red = smem + wave * 2048;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const int r = 8 * (e >> 2) + 4 * h + (e & 3);
    red[r * 32 + col] = ag[e];
    red[1024 + r * 32 + col] = au[e];
  }
  __syncthreads();
  for (int t = tid; t < Sh::BM * Sh::BN; t += Sh::kThreads) {
    const int r = t >> 5, c = t & 31;
    const float* p = smem + (r >> 5) * WK * 2048 + (r & 31) * 32 + c;
    float g = p[0], u = p[1024];
#pragma unroll
    for (int w = 1; w < WK; ++w) {
      g += p[w * 2048];
      u += p[w * 2048 + 1024];
    }
    if (m0 + r < M && n0 + c < N) o[int64_t(m0 + r) * N + n0 + c] = (g / (1.0f + exp_e(-g))) * u;
  }
}

template <int WR, int WK, int KW, bool WIDE>
int launch_swiglu_f32(const float* x, const float* wg, const float* wu, float* o, int64_t m, int64_t n, int64_t k,
                      hipStream_t s) {
  using Sh = SwShape<WR, WK, KW>;
  const int64_t gx = (n + Sh::BN - 1) / Sh::BN, gy = (m + Sh::BM - 1) / Sh::BM;
  if (gy > 65535) return PTB_ERR_GRID;
  const int64_t bx = WIDE ? std::min<int64_t>(gx, 1 << 22) : gx;
  swiglu_f32<WR, WK, KW, WIDE><<<dim3(unsigned(bx), unsigned(gy), unsigned((gx + bx - 1) / bx)), dim3(Sh::kThreads), 0,
                                 s>>>(x, wg, wu, o, int(m), int(n), int(k));
  return launch_status();
}

bool aligned_rows(const void* p, int64_t cols) { return aligned16(p) && cols % 4 == 0; }

}  // namespace

PTB_EXPORT int ptb_rmsnorm_f32(const float* x, const float* w, float* y, int64_t rows, int64_t cols, float eps,
                               void* stream) {
  if (rows < 0 || cols <= 0 || cols > (int64_t(1) << 30)) return PTB_ERR_SHAPE;
  if (rows == 0) return PTB_OK;
  if (!x || !w || !y) return PTB_ERR_NULL;
  if (!aligned_rows(x, cols) || !aligned16(w) || !aligned16(y)) return PTB_ERR_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int chunks = int(cols / 4);
  const int c = int(cols);
  if (chunks <= 64 * 8) {                      // one wave per row, 4 rows a block
    const int64_t blocks = (rows + 3) / 4;
    if (blocks > 0x7fffffff) return PTB_ERR_GRID;
    const dim3 g = dim3(unsigned(blocks)), b = dim3(kBlock);
    if (chunks <= 64 * 2) rmsnorm_rows_f32<64, 2><<<g, b, 0, s>>>(x, w, y, rows, c, eps);
    else if (chunks <= 64 * 4) rmsnorm_rows_f32<64, 4><<<g, b, 0, s>>>(x, w, y, rows, c, eps);
    else rmsnorm_rows_f32<64, 8><<<g, b, 0, s>>>(x, w, y, rows, c, eps);
  } else {
    if (rows > 0x7fffffff) return PTB_ERR_GRID;
    const dim3 g = dim3(unsigned(rows)), b = dim3(kBlock);
    if (chunks <= kBlock * 8) rmsnorm_rows_f32<kBlock, 8><<<g, b, 0, s>>>(x, w, y, rows, c, eps);
    else rmsnorm_rows_f32_long<<<g, b, 0, s>>>(x, w, y, c, eps);
  }
  return launch_status();
}

PTB_EXPORT int ptb_col_rms_f32(const float* x, float* c, int64_t rows, int64_t cols, float eps, void* stream) {
  if (rows <= 0 || cols < 0) return PTB_ERR_SHAPE;
  if (cols == 0) return PTB_OK;
  if (!x || !c) return PTB_ERR_NULL;
  const int64_t blocks = (cols + 63) / 64;
  if (blocks > 0x7fffffff) return PTB_ERR_GRID;
  col_rms_f32<<<dim3(unsigned(blocks)), dim3(kBlock), 0, static_cast<hipStream_t>(stream)>>>(x, c, rows, cols, eps);
  return launch_status();
}

PTB_EXPORT int ptb_softmax_rows_f32(const float* x, float* y, int64_t rows, int64_t cols, void* stream) {
  if (rows < 0 || cols <= 0 || cols > (int64_t(1) << 30)) return PTB_ERR_SHAPE;
  if (rows == 0) return PTB_OK;
  if (!x || !y) return PTB_ERR_NULL;
  if (!aligned_rows(x, cols) || !aligned16(y)) return PTB_ERR_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int chunks = int(cols / 4);
  const int c = int(cols);
  if (chunks <= 64 * 8) {
    const int64_t blocks = (rows + 3) / 4;
    if (blocks > 0x7fffffff) return PTB_ERR_GRID;
    const dim3 g = dim3(unsigned(blocks)), b = dim3(kBlock);
    if (chunks <= 64 * 2) softmax_rows_f32<64, 2><<<g, b, 0, s>>>(x, y, rows, c);
    else if (chunks <= 64 * 4) softmax_rows_f32<64, 4><<<g, b, 0, s>>>(x, y, rows, c);
    else softmax_rows_f32<64, 8><<<g, b, 0, s>>>(x, y, rows, c);
  } else {
    if (rows > 0x7fffffff) return PTB_ERR_GRID;
    const dim3 g = dim3(unsigned(rows)), b = dim3(kBlock);
    if (chunks <= kBlock * 8) softmax_rows_f32<kBlock, 8><<<g, b, 0, s>>>(x, y, rows, c);
    else softmax_rows_f32_long<<<g, b, 0, s>>>(x, y, c);
  }
  return launch_status();
}

PTB_EXPORT int ptb_silu_mul_f32(const float* gate_up, float* out, int64_t rows, int64_t inter, void* stream) {
  if (rows < 0 || inter <= 0) return PTB_ERR_SHAPE;
  if (rows == 0) return PTB_OK;
  if (!gate_up || !out) return PTB_ERR_NULL;
  if (inter % 4 || !aligned16(gate_up) || !aligned16(out)) return PTB_ERR_ALIGN;
  const int64_t total = rows * (inter / 4);
  const int64_t blocks = std::min<int64_t>((total + kBlock - 1) / kBlock, 65536);
  silu_mul_f32<<<dim3(unsigned(blocks)), dim3(kBlock), 0, static_cast<hipStream_t>(stream)>>>(gate_up, out, rows,
                                                                                              inter);
  return launch_status();
}

PTB_EXPORT int ptb_swiglu_f32(const float* x, const float* wg, const float* wu, float* o, int64_t m, int64_t n,
                              int64_t k, void* stream) {
  if (m < 0 || n < 0 || k < 0) return PTB_ERR_SHAPE;
  if (m == 0 || n == 0) return PTB_OK;
  if (!x || !wg || !wu || !o) return PTB_ERR_NULL;
  if (m > 0x7fffffff || n > 0x7fffffff || k > 0x7fffffff) return PTB_ERR_SHAPE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // By the number of 32x32 output blocks: up to two a CU, one block a workgroup of eight waves (few
  // rows are bound by the latency of the weights: 1x2048x4096 30 us against 38 with four waves); to nine
  // a CU, one block to four waves (200x1024x2816 38 us against 41 with eight); past it 64x32 outputs to
  // four waves, which read less per product (2048x2048x4096 594 us against 668 with 32x32).  64-bit
  // offsets only where a workgroup's rows of x or a slab of the weights may pass 4 GB.
  const int64_t blocks = ((m + 31) / 32) * ((n + 31) / 32);
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (k >= (int64_t(1) << 24) || n >= (int64_t(1) << 24))
    return launch_swiglu_f32<2, 2, 16, true>(x, wg, wu, o, m, n, k, s);
  if (blocks <= 2 * int64_t(cus)) return launch_swiglu_f32<1, 8, 8, false>(x, wg, wu, o, m, n, k, s);
  // Where K is short enough for the first of the waves that split it, the others only add the sum through the LDS:
  // 128x32 outputs to four waves, each with all of K (no larger error).  4096x4096 outputs: K = 8 32.7 us before the
  // matrix instruction, 43.9 split, 24.3 so, K = 16 33.0, 44.5, 29.6; 363x4230 outputs: K = 8 7.6, 8.3, 6.2.
  if (k <= (blocks > 9 * int64_t(cus) ? 16 : 8)) return launch_swiglu_f32<4, 1, 8, false>(x, wg, wu, o, m, n, k, s);
  if (blocks <= 9 * int64_t(cus)) return launch_swiglu_f32<1, 4, 8, false>(x, wg, wu, o, m, n, k, s);
  return launch_swiglu_f32<2, 2, 16, false>(x, wg, wu, o, m, n, k, s);
}
