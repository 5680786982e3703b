// bf16 GEMM on gfx950 matrix cores: C[M,N] = A[M,K] * B[K,N] (+ R[M,N]), all row-major, fp32
// accumulation, one bf16 rounding at the store.
//
// Workgroup tiles of 256x256, 256x192, 256x128, 128x256, 128x128 or 64x128 (Shape below), 4 waves in
// a 2x2 arrangement, each wave owning WM x WN v_mfma_f32_32x32x16_bf16 accumulators (256 fp32 per
// lane for 256x256 tiles, held in AGPRs).
//
// Operands move HBM -> LDS with buffer_load_dwordx4 ... lds (no VGPR staging), 64 K columns at a time
// (a whole 128-byte line of every A row): 256x128 and 128x256 tiles in a ring of three slots, 256x256
// and 256x192 tiles in rings of three A slots and two B slots (160 / 144 KB), 128x128 and 64x128 tiles
// in rings of four.  Each stage's DMAs run two (or three)
// stages ahead and spread over a whole K step's MFMAs, into the slots the previous step's barrier
// freed.  A and B keep their global layouts in LDS with 16-byte chunks XOR-swizzled per row, so
// every fragment read is bank-conflict free:
//   A fragments (8 consecutive k of one row per lane) are plain 128-bit LDS reads; row m keeps
//   chunk c in slot c ^ ((m >> 1) & 7);
//   B fragments (8 consecutive k of one column per lane, while B is N-contiguous) come from two
//   ds_read_b64_tr_b16 transposing reads; row k keeps chunk c in slot c ^ (4 * (k & 3)) (rows of
//   384 bytes: c ^ (4 * ((k >> 1) & 1))).
// The fragments of the next 16-wide K slice are read while the MFMAs of the current one run, and
// the main loop runs a whole number of ring turns a trip, so every slot address is a constant.
// The MFMA is issued with B as its first operand, so each accumulator holds a 32x32 block of C^T.
// The epilogue stages each wave's 32-row blocks of fp32 results through a private, padded LDS
// region (the rings are free by then) so that stores, and residual loads, cover whole rows; buffer
// resources drop rows and columns outside C.
//
// Modes: plain (+ residual), split-K into fp32 partials (splitk_finish sums them) and SwiGLU (the gate
// and up columns of the same outputs meet in one wave; the epilogue stores silu(gate) * up).  The MoE
// grouped GEMM (a program table maps row tiles to weights) is a kernel of its own on the same stages.
//
// Tile order is XCD-aware: hardware hands workgroup i to XCD i % 8, so ids are remapped to give
// each XCD a contiguous range of tiles, walked in groups of 8 tile-rows for L2 reuse; split-K walks
// one K slice's tiles after the other, so that an XCD's workgroups share their slice's panels.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "ptb_common.h"

using namespace ptb;



namespace {

constexpr int kThreads = 256;
constexpr int kGroupM = 8;
// K past the end the DMA stream may address: two 64-deep stages, or three in the four-slot rings
constexpr int kRunAhead = 128, kRunAheadDeep = 192;
// Widest C (columns) the epilogue addresses: a 256-row tile of it stays within 2^31 bytes, so its
// 32-bit store offsets, and the 0x80000000 that marks a column outside C, stay in range.
constexpr int64_t kMaxOutCols = int64_t(1) << 22;

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

// Tile shape: the 4 waves sit 2x2, each owning WM x WN blocks of 32x32, so the workgroup tile is
// BM = 64*WM rows by BN = 64*WN columns (256x256, 256x192, 256x128, 128x256, 128x128 or 64x128).  A
// stage holds BK of K: 64 (a whole 128-byte line of every A row: the L2 serves a request per line,
// and a half-line request costs a whole one) in rings of 3 slots (256x128, 128x256), of 3 A slots and
// 2 B slots (256x256, 256x192) or of 4 slots (128x128, 64x128: a workgroup of these is alone on its
// CU and its step's MFMAs are short, so a third stage in flight pays: 4.5% over 3 slots).  Against
// 32-deep stages these took one-round shapes of 128x128 tiles from 53 to 42 us (640x4096x6144) and 48
// to 39 us (1024x4096x4096).  Stage kt + DIST, DIST = NSA - 1 = 2 or 3, refills the slots of stage kt-1, which the barrier of step
// kt-1 freed, so the stage's DMAs spread over all of step kt's MFMAs; with two B slots, its B part
// waits for the barrier of step kt and spreads over the slice after it.
// RING: NSA; 64x128 and 128x128 tiles also come in rings of 3 for short K ranges (see make_plan).
template <int WM, int WN, int RING = (WM * WN >= 8 ? 3 : 4)>
struct Shape {
  static constexpr int BK = 64;
  // A and B live in rings of their own: NSA and NSB slots.  256x256 and 256x192 tiles with 64-deep
  // stages have room for three A slots and two B slots only (160 / 144 KB), so their B ring
  // refills a slot only after the barrier that frees it (the "hybrid" schedule below); every other
  // ring is one slot deeper than its DMA distance.
  static constexpr bool kHybrid = WM * WN >= 12;
  static constexpr int NSA = RING;
  static constexpr int NSB = kHybrid ? 2 : NSA;
  static constexpr int NS = NSA;
  static constexpr int DIST = NSA - 1;
  static constexpr int SPS = BK / 16;                    // 16-wide K slices per stage
  static constexpr int BM = 64 * WM, BN = 64 * WN;
  static constexpr int kRowBytes = BK * 2;               // bytes of an A row in a stage
  static constexpr int kChunks = BK / 8;                 // 16-byte chunks of an A row in a stage
  static constexpr int kABytes = BM * BK * 2;
  static constexpr int kBBytes = BK * BN * 2;
  static constexpr int kDmaA = kABytes / 4096;           // buffer_load ... lds per wave per stage
  static constexpr int kDmaB = kBBytes / 4096;
  static constexpr int kDma = kDmaA + kDmaB;
  static constexpr int kARowsPerKB = 1024 / kRowBytes;   // A rows per DMA instruction
  static constexpr int kMfma = WM * WN;                  // MFMAs per wave per 16-wide K slice
  static constexpr int kPieces = WM + 2 * WN;            // LDS reads per wave per K slice
  static constexpr int kBSlots = BN / 8;                 // 16-byte chunks per B row
  static constexpr int kSmemBytes = NSA * kABytes + NSB * kBBytes;
  static_assert(kSmemBytes <= 160 * 1024, "the rings fit the LDS");
  static_assert(kABytes % 4096 == 0 && kBBytes % 4096 == 0, "whole 1 KB DMA instructions per wave");
  static_assert(DIST == NS - 1 && DIST >= 2, "the DMA refills the slot freed a step earlier");
};
// A row m keeps chunk c in slot c ^ a_swz(m): the 16 rows a 16-lane phase reads land in 16 distinct
// bank groups.
__device__ __forceinline__ int a_swz(int m) { return (m >> 1) & 7; }
// B row k keeps chunk c in slot c ^ b_swz(k).  A transposing read takes 64 bytes of each of 4
// consecutive rows k0..k0+3 (k0 % 4 == 0) per 32 lanes.  Rows of 512 or 256 bytes all start at
// bank 0, so the rows shift by 64 bytes each: 4 * (k & 3).  Rows of 384 bytes (BN 192) start 32
// banks apart in turn, so only k0+2 and k0+3 shift, by 64 bytes: 4 * ((k >> 1) & 1).  Either way
// the 4 rows' 64 bytes take 64 distinct banks, and the XOR stays inside the row's chunks.
template <int BN>
__device__ __forceinline__ int b_swz(int k) { return BN == 192 ? 4 * ((k >> 1) & 1) : 4 * (k & 3); }

// The column of B (from the tile's first gate column; up columns I further) that a SwiGLU tile of BN
// columns stages as its 16-byte chunk c: BN / 2 gate columns, then their up columns, so that the DMAs
// take whole 128-byte lines of both one after the other (32-column blocks of gate and up in turn, in
// 64-byte pieces, were 0.7% slower on an MLP of 200 tokens and 0.5% on the 640-token layer).
template <int BN>
__device__ __forceinline__ int swiglu_col(int c, int inter) {
  return c < BN / 16 ? 8 * c : inter + 8 * (c - BN / 16);
}
// The staged column of column n (0 .. 31) of block j of wave column wn.  Even WN: a wave's blocks 2jp and
// 2jp + 1 are the gate and up of the same 32 outputs.  WN = 3 (48 outputs a wave): block 0 its first 32
// gate columns, block 2 their up columns, block 1 the last 16 gate columns, then their up columns, which
// a lane holds 8 accumulator registers apart.
template <int WN>
__device__ __forceinline__ int swiglu_staged(int wn, int j, int n) {
  constexpr int kUp = 32 * WN;   // BN / 2
  if constexpr (WN == 3) return 48 * wn + (j == 0 ? n : j == 2 ? kUp + n : n < 16 ? 32 + n : kUp + 16 + n);
  else return (j & 1) * kUp + 32 * (wn * (WN / 2) + (j >> 1)) + n;
}

// Split-K mode: workgroup (tile, slice s) multiplies K columns [s*kchunk, s*kchunk + kchunk) and
// stores its fp32 partial tile at part + s*M*N; splitk_finish sums the partials.
// SwiGLU mode (the gate_up GEMM with silu(gate) * up fused into its epilogue): B is [K, 2*I] with
// gate columns [0, I) and up columns [I, 2I); a workgroup tile's BN columns of B are the gate and up
// columns of the same BN / 2 output columns, laid out so that a lane holds both of every output (see
// swiglu_staged), and the epilogue stores bf16(silu(bf16(gate)) * bf16(up)), as a separate silu_mul
// would compute it from the bf16 GEMM.
enum { kPlain = 0, kSplit = 1, kSwiGLU = 2 };
// Up to this many outputs the partials of 64x128 tiles in rings of 3 leave straight from the accumulators, without the barrier
// and the LDS pass: 348x2048x40 5.69 -> 5.42 us, 3x2816x8 5.54 -> 5.23, 544x1600x48 6.02 -> 5.78.  Past it whole
// rows a store instruction are worth them: 1024x2048x128 7.74 us staged, 8.09 direct; 193x3008x576 7.51 / 7.84.
constexpr int64_t kDirectPartials = 32768;


// PERSIST (plain 256x256 tiles, no residual): one workgroup per CU walks the tiles
// blockIdx.x, blockIdx.x + gridDim.x, ...; the next tile's first stage goes out halfway through the
// current tile's epilogue, so its latency hides behind the stores (see the epilogue).
template <int WM, int WN, bool RESID, int MODE, bool PERSIST = false, int RING = Shape<WM, WN>::NSA>
__global__ __launch_bounds__(kThreads, (WM * WN >= 12 ? 1 : 2)) void gemm_bf16_kernel(
    const uint16_t* __restrict__ A_in, const uint16_t* __restrict__ B_in, const uint16_t* __restrict__ R,
    uint16_t* __restrict__ C, int M, int N, int K, int tiles_m, int tiles_n, int xcd_grid, float* __restrict__ part,
    int kchunk) {
  using Sh = Shape<WM, WN, RING>;
  constexpr int BM = Sh::BM, BN = Sh::BN, kABytes = Sh::kABytes;
  constexpr int BK = Sh::BK, NS = Sh::NS, DIST = Sh::DIST, NSA = Sh::NSA, NSB = Sh::NSB;
  constexpr bool kHybrid = Sh::kHybrid;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[Sh::kSmemBytes];

  // ---- tile selection: tile id -> (first row, first column); ids are spread so that each XCD
  //      takes a contiguous range of tiles, walked in groups of kGroupM tile-rows
  const int ntiles = tiles_m * tiles_n;
  // XCD x takes ids x, x + 8, ...: the n / 8 (one more for the first n % 8) consecutive positions
  // from x * (n / 8) + min(x, n % 8)
  auto xcd_position = [](int id, int n) __attribute__((always_inline)) {
    const int x = id & 7;
    return x * (n >> 3) + min(x, n & 7) + (id >> 3);
  };
  auto tile_origin = [&](int pid, int& tm0, int& tn0) __attribute__((always_inline)) {
    const int width = kGroupM * tiles_n;
    const int first_m = (pid / width) * kGroupM;
    const int gsize = min(tiles_m - first_m, kGroupM);
    const int tm = first_m + (pid % width) % gsize;
    const int tn = (pid % width) / gsize;
    tm0 = tm * BM;
    tn0 = MODE == kSwiGLU ? tn * (BN / 2) : tn * BN;   // SwiGLU: the output (and gate) column base
  };
  const uint16_t* A = A_in;
  const uint16_t* B = B_in;
  int m0, n0;
  int Kl = K;    // the K columns this workgroup multiplies
  int slice = 0; // split-K: this workgroup's K slice
  // xcd_grid: the workgroups of the launch (the tiles of a persistent walk), 0: positions by workgroup id
  int pid = blockIdx.x;
  if (MODE != kPlain || xcd_grid > 0) pid = xcd_position(pid, xcd_grid);
  if constexpr (MODE == kSplit) {
    slice = pid / ntiles;
    pid -= slice * ntiles;
    const int k0 = slice * kchunk;
    Kl = min(kchunk, K - k0);
    A = A_in + k0;
    B = B_in + int64_t(k0) * N;
  }
  tile_origin(pid, m0, n0);

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  // ---- loaders: A tile rows past M read as zero (num_records); B columns past N are read from
  //      the next row or as zero, and only feed columns of C that are never stored
  const int koff = MODE == kSplit ? slice * kchunk : 0;   // this slice's first K column
  auto make_rsrc_a = [&](int tm0) __attribute__((always_inline)) {
    return make_rsrc(A + int64_t(tm0) * K, uint32_t(int64_t(min(BM, M - tm0)) * K - koff) * 2u);
  };
  auto make_rsrc_b = [&](int tn0) __attribute__((always_inline)) {
    return make_rsrc(B + tn0, uint32_t((int64_t(K - koff) * N - tn0) * 2));
  };
  i32x4 rsrc_a = make_rsrc_a(m0);
  i32x4 rsrc_b = make_rsrc_b(n0);
  // A: instruction t of this wave covers rows kARowsPerKB*(kDmaA*wave + t) + lane/kChunks; lane ->
  //    slot lane%kChunks, holding chunk slot ^ a_swz(row)
  // B: instruction t covers the stage's 16-byte pieces 64*(kDmaB*wave + t) + lane in row-major order,
  //    piece i -> row i/kBSlots, slot i%kBSlots holding chunk slot ^ b_swz(row)
  uint32_t a_voff[Sh::kDmaA], b_voff[Sh::kDmaB];
#pragma unroll
  for (int t = 0; t < Sh::kDmaA; ++t) {
    const int row = (wave * Sh::kDmaA + t) * Sh::kARowsPerKB + lane / Sh::kChunks;
    const int chunk = (lane % Sh::kChunks) ^ a_swz(row);
    a_voff[t] = uint32_t(row * K + chunk * 8) * 2u;
  }
#pragma unroll
  for (int t = 0; t < Sh::kDmaB; ++t) {
    const int piece = 64 * (wave * Sh::kDmaB + t) + lane;
    const int k = piece / Sh::kBSlots;
    const int bchunk = (piece % Sh::kBSlots) ^ b_swz<BN>(k);
    const int bcol = MODE == kSwiGLU ? swiglu_col<BN>(bchunk, N / 2) : bchunk * 8;
    b_voff[t] = uint32_t(k * N + bcol) * 2u;
  }
  const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(smem));
  const uint32_t wave_a = __builtin_amdgcn_readfirstlane(uint32_t(wave * Sh::kDmaA * 1024));
  const uint32_t wave_b = __builtin_amdgcn_readfirstlane(uint32_t(wave * Sh::kDmaB * 1024));
  // t-th of this wave's A (or B) DMA instructions of stage kt into A slot sa (B slot sb); the slots
  // are compile-time constants at every call (the main loop runs a whole number of ring turns a
  // trip), so the LDS addresses are constants plus scalar offsets and the fragment reads take them
  // as immediate offsets
  const uint32_t lds_b0 = lds0 + uint32_t(NSA * kABytes);
  auto dma_a = [&](int kt, int t, auto sa) __attribute__((always_inline)) {
    dma16(rsrc_a, lds0 + uint32_t(decltype(sa)::value) * kABytes + wave_a + t * 1024, a_voff[t],
          uint32_t(kt * BK) * 2u);
  };
  auto dma_b = [&](int kt, int t, auto sb) __attribute__((always_inline)) {
    dma16(rsrc_b, lds_b0 + uint32_t(decltype(sb)::value) * Sh::kBBytes + wave_b + t * 1024, b_voff[t],
          uint32_t(kt * BK) * uint32_t(N) * 2u);
  };
  // the t-th DMA of a stage, A first, then B
  auto dma_one = [&](int kt, int t, auto sa, auto sb) __attribute__((always_inline)) {
    if (t < Sh::kDmaA) dma_a(kt, t, sa);
    else dma_b(kt, t - Sh::kDmaA, sb);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  using I4 = std::integral_constant<int, 4>;
  using I5 = std::integral_constant<int, 5>;

  f32x16 acc[WM][WN];

  // ---- fragment addressing
  const int fr = lane & 31, h = lane >> 5;
  // A: row m (this lane's), chunk 2*ks + h, swizzled by a_swz(m)
  int a_row_off[WM], a_sw[WM];
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int m = wm * (BM / 2) + i * 32 + fr;
    a_row_off[i] = m * Sh::kRowBytes;
    a_sw[i] = a_swz(m);
  }
  // B (transposing reads): group g = lane/16 -> k half g/2, column half 16*(g%2); in-group lane
  // 4*jj + q supplies row 8h + 4r + jj (+16 ks), columns +4q..+4q+3
  const int g16 = (lane >> 4) & 1, l16 = lane & 15, jj = l16 >> 2, q = l16 & 3;
  int b_off[WN][2];
#pragma unroll
  for (int j = 0; j < WN; ++j) {
    const int nb = 16 * g16 + 4 * q;
    const int n = MODE == kSwiGLU ? swiglu_staged<WN>(wn, j, nb) : wn * (BN / 2) + j * 32 + nb;
    const int chunk = n >> 3;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int k = 8 * h + 4 * r + jj;  // + 16*ks, which keeps k & 3
      b_off[j][r] = k * (2 * BN) + ((chunk ^ b_swz<BN>(k)) << 4) + (q & 1) * 8;
    }
  }

  // One K slice's fragments, read in kPieces pieces (WM A reads, 2*WN B half-reads) so that the
  // reads can be spread between MFMAs.
  struct Slice {
    bf16x8 a[WM];
    bf16x8 b[WN];
    i16x4 blo[WN];
  };
  auto read_piece = [&](const uint8_t* sta, const uint8_t* stb, int ks, int p, Slice& f) __attribute__((always_inline)) {
    if (p < WM) {
      f.a[p] = *reinterpret_cast<const bf16x8*>(sta + a_row_off[p] + (((2 * ks + h) ^ a_sw[p]) << 4));
    } else {
      const int j = (p - WM) >> 1, r = (p - WM) & 1;
      const i16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(stb + b_off[j][r] + ks * 16 * 2 * BN));
      if (r == 0) f.blo[j] = v;
      else f.b[j] = __builtin_bit_cast(bf16x8, i16x8{f.blo[j][0], f.blo[j][1], f.blo[j][2], f.blo[j][3], v[0], v[1], v[2], v[3]});
    }
  };
  auto mfma_one = [&](const Slice& f, int u) __attribute__((always_inline)) {
    const int i = u / WN, j = u % WN;
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.b[j], f.a[i], acc[i][j], 0, 0, 0);
  };

  // The DMA stream runs DIST stages ahead of the MFMAs and does not stop at the last K step:
  // stages past the end read zeros (num_records) into slots nobody reads any more, which keeps the
  // loop free of branches; everything is drained before the epilogue.
  constexpr int U = Sh::kMfma, P = Sh::kPieces, D = Sh::kDma, SPS = Sh::SPS;
  constexpr bool kOneReadPerMfma = P <= U;
  // stage kt+DIST's DMAs go out one every SLOTS/D MFMAs of step kt (bunched after the barrier they
  // would queue behind each other in the address unit and stall the MFMAs)
  constexpr int SLOTS = SPS * U;
  // Hybrid schedule (two B slots): stage kt+2's A DMAs spread over step kt before its barrier, into
  // the A slot step kt-1 freed; its B DMAs go into the B slot step kt's barrier frees, spread over
  // step kt's last slice (one per two MFMAs, against the A DMAs' one per six).  Splitting the B
  // DMAs between that slice and the next step's first MFMAs measured no faster.
  constexpr int NPRE = [] {   // DMAs of stage kt+DIST issued before step kt's barrier
    int n = 0;
    if (kHybrid) return Sh::kDmaA;
    for (int o = 0; o < D; ++o)
      if (o * SLOTS / D < (SPS - 1) * U) ++n;
    return n;
  }();
  const int nk = Kl / BK;
  const uint8_t* const smem_b = smem + NSA * kABytes;
  static_assert(!PERSIST || (WM == 4 && WN == 4 && !RESID && MODE == kPlain),
                "the persistent walk is for plain 256x256 tiles (the SwiGLU form has no registers to spare)");
  // stores of the epilogue's second half, issued after the next tile's stage-0 DMAs
  constexpr int kStoresAfter = (WM / 2) * 4 * WN;
  int tile_id = blockIdx.x;
  bool pre0 = false;   // this tile's stage 0 went out during the previous tile's epilogue
  for (;;) {
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  if (!pre0) {
#pragma unroll
    for (int t = 0; t < D; ++t) dma_one(0, t, I0{}, I0{});
  }
#pragma unroll
  for (int t = 0; t < D; ++t) dma_one(1, t, I1{}, std::integral_constant<int, 1 % NSB>{});
  if constexpr (DIST > 2) {
#pragma unroll
    for (int t = 0; t < D; ++t) dma_one(2, t, I2{}, std::integral_constant<int, 2 % NSB>{});
  }
  // stage 0 landed (this wave's part): after it went out, the stages above and, when it was
  // prefetched, the epilogue's last kStoresAfter stores (memory operations count down in order)
  if (pre0) wait_vmcnt<(DIST - 1) * D + (PERSIST ? kStoresAfter : 0)>();
  else wait_vmcnt<(DIST - 1) * D>();
  __syncthreads();                  // ... and everyone's
  Slice sl[2];
#pragma unroll
  for (int p = 0; p < P; ++p) read_piece(smem, smem_b, 0, p, sl[0]);

  // Each K step: slices 0 .. SPS-2, each with the next slice's reads and a share of the DMAs folded
  // in; the barrier that publishes stage kt+1 (and frees stage kt's slots); the last slice with the
  // rest of the DMAs and the reads of stage kt+1's slice 0 folded in.  sched_barrier(0) pins that
  // interleave, so the matrix core is fed between memory instructions.
  auto step = [&](int kt, auto sa, auto sb) __attribute__((always_inline)) {
    constexpr int SA = decltype(sa)::value, SB = decltype(sb)::value;   // kt % NSA, kt % NSB
    using FarA = std::integral_constant<int, (SA + DIST) % NSA>;
    using FarB = std::integral_constant<int, (SB + DIST) % NSB>;
    const uint8_t* sta = smem + SA * kABytes;
    const uint8_t* stb = smem_b + SB * Sh::kBBytes;
#pragma unroll
    for (int q = 0; q + 1 < SPS; ++q) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        mfma_one(sl[q & 1], u);
#pragma unroll
        for (int p = 0; p < P; ++p)
          if (kOneReadPerMfma ? p == u : (p >= u * P / U && p < (u + 1) * P / U)) read_piece(sta, stb, q + 1, p, sl[(q + 1) & 1]);
        if constexpr (kHybrid) {
#pragma unroll
          for (int o = 0; o < Sh::kDmaA; ++o)
            if (o * (SPS - 1) * U / Sh::kDmaA == q * U + u) dma_a(kt + DIST, o, FarA{});
        } else {
#pragma unroll
          for (int o = 0; o < D; ++o)
            if (o * SLOTS / D == q * U + u) dma_one(kt + DIST, o, FarA{}, FarB{});
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // stage kt+1 landed (later stages' DMAs may still be in flight); past this barrier no wave
    // reads stage kt
    wait_vmcnt<(DIST - 2) * D + NPRE>();
    __syncthreads();
    const uint8_t* nsta = smem + ((SA + 1) % NSA) * kABytes;
    const uint8_t* nstb = smem_b + ((SB + 1) % NSB) * Sh::kBBytes;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      mfma_one(sl[(SPS - 1) & 1], u);
      // the stage's remaining DMAs, and the next stage's first reads spread evenly
      if constexpr (kHybrid) {
#pragma unroll
        for (int o = 0; o < Sh::kDmaB; ++o)
          if (o * U / Sh::kDmaB == u) dma_b(kt + DIST, o, FarB{});   // into the B slot this barrier freed
      } else {
#pragma unroll
        for (int o = 0; o < D; ++o)
          if (o * SLOTS / D == (SPS - 1) * U + u) dma_one(kt + DIST, o, FarA{}, FarB{});
      }
#pragma unroll
      for (int p = 0; p < P; ++p)
        if (p >= u * P / U && p < (u + 1) * P / U) read_piece(nsta, nstb, 0, p, sl[0]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // L steps a trip: a whole number of turns of both rings, so every slot is a constant
  constexpr int L = kHybrid ? 6 : NSA;
  auto stepc = [&](int k, auto i) __attribute__((always_inline)) {
    constexpr int I = decltype(i)::value;
    step(k, std::integral_constant<int, I % NSA>{}, std::integral_constant<int, I % NSB>{});
  };
  int kt = 0;
  for (; kt + L <= nk; kt += L) {
    stepc(kt, I0{});
    stepc(kt + 1, I1{});
    stepc(kt + 2, I2{});
    if constexpr (L > 3) stepc(kt + 3, I3{});
    if constexpr (L > 4) stepc(kt + 4, I4{});
    if constexpr (L > 5) stepc(kt + 5, I5{});
  }
  if (kt < nk) stepc(kt, I0{});
  if (kt + 1 < nk) stepc(kt + 1, I1{});
  if constexpr (L > 3) {
    if (kt + 2 < nk) stepc(kt + 2, I2{});
  }
  if constexpr (L > 4) {
    if (kt + 3 < nk) stepc(kt + 3, I3{});
  }
  if constexpr (L > 5) {
    if (kt + 4 < nk) stepc(kt + 4, I4{});
  }
  wait_vmcnt<0>();

  // the next tile of a persistent walk, and its stage-0 DMAs into A slot 0 and B slot 0 (free:
  // every DMA has landed and, past the epilogue's barrier, no wave reads a stage)
  const int next_id = tile_id + int(gridDim.x);
  const bool has_next = PERSIST && next_id < ntiles;
  int nm0 = 0, nn0 = 0;
  if (has_next) tile_origin(xcd_position(next_id, ntiles), nm0, nn0);
  auto prefetch_next = [&]() __attribute__((always_inline)) {
    if (has_next) {
      rsrc_a = make_rsrc_a(nm0);
      rsrc_b = make_rsrc_b(nn0);
#pragma unroll
      for (int t = 0; t < D; ++t) dma_one(0, t, I0{}, I0{});
    }
  };

  // ---- epilogue: accumulator (i, j, r) of lane holds C row m0 + wm*BM/2 + i*32 + lane%32,
  //      column n0 + wn*BN/2 + j*32 + 8*(r/4) + 4*(lane/32) + r%4: 4 consecutive columns per r/4
  // Tiles leave through the LDS, which is free now (every DMA has landed
  // and, past the barrier, no wave reads a stage): a wave writes one 32-row block of its results
  // (bf16; fp32 where a residual is still to be added, and in the persistent walk) (NG groups of
  // 8 columns; value(i, gg) gives the 4 fp32 columns 8gg + 4*(lane/32) .. +3 for row lane%32) into a private, padded region and reads it back 4 columns a lane, so
  // each store writes whole rows of its block (in the accumulator layout one store instruction
  // writes 16 bytes into each of 32 rows, which took 12% of a 256x256 tile's time) and the
  // residual is read the same way.  The region is the wave's own and LDS operations of a wave
  // complete in order, so no barrier separates its writes from its reads.  Rows past M and columns
  // past `cols` fall outside the buffer resources (stores dropped, loads 0): no branches.
  const bool direct = MODE == kSplit && WM == 1 && RING == 3 && int64_t(M) * N <= kDirectPartials;
  if (!direct) __syncthreads();
  auto store_staged = [&](auto ng, auto value, uint16_t* out, int ldc, int cols, int col0) __attribute__((always_inline)) {
    constexpr int NG = decltype(ng)::value;
    constexpr int WC = NG * 8;            // columns of a wave's block
    // without a residual to add, each value is rounded to bf16 before it is staged (the rounding
    // the store would make anyway), halving the staged bytes; with one, the fp32 sum needs fp32.
    // The persistent walk keeps fp32 staging: its bf16 form needs registers it does not have
    // (632 bytes of spills)
    constexpr bool kF32Stage = RESID || PERSIST;
    constexpr int kEl = kF32Stage ? 4 : 2;   // bytes per staged value
    constexpr int kPitch = WC * kEl + 16; // bytes per staged row: rows start 4 banks apart
    constexpr int LPR = WC / 4;           // lanes per row, 4 columns each
    // rows per instruction (96 columns: 2 rows on 48 lanes; 48 columns: 4 rows on 48 lanes)
    constexpr int RPI = LPR == 12 ? 4 : 64 / LPR;
    static_assert(32 % RPI == 0, "whole instructions per 32-row block");
    static_assert(4 * 32 * kPitch <= Sh::kSmemBytes, "the staging regions fit in the ring's LDS");
    // a persistent walk keeps A slot 0 and B slot 0 free for the next tile's first stage: waves 0-2
    // stage in A slots 1-2, wave 3 in B slot 1
    static_assert(!PERSIST || (3 * 32 * kPitch <= 2 * kABytes && 32 * kPitch <= Sh::kBBytes),
                  "the persistent staging regions fit beside the next tile's first stage");
    uint8_t* const stage = !PERSIST ? smem + wave * (32 * kPitch)
                           : wave < 3 ? smem + kABytes + wave * (32 * kPitch)
                                      : smem + NSA * kABytes + Sh::kBBytes;
    const bool lane_on = lane < RPI * LPR;     // lanes past the last whole row store nothing
    const int rl = lane_on ? lane / LPR : 0, c4 = lane % LPR;
    const int gcol = col0 + 4 * c4;
    const uint32_t tile_bytes = uint32_t(min(BM, M - m0)) * uint32_t(ldc) * 2u;
    const __amdgpu_buffer_rsrc_t rsrc_c =
        __builtin_amdgcn_make_buffer_rsrc(out + int64_t(m0) * ldc, 0, tile_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_r =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(RESID ? R + int64_t(m0) * ldc : out), 0, tile_bytes,
                                          0x00020000);
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      const int r0 = wm * (BM / 2) + i * 32 + rl;   // tile row of this lane's first row
      uint32_t voff[32 / RPI];
#pragma unroll
      for (int t = 0; t < 32 / RPI; ++t)
        voff[t] = lane_on && gcol < cols ? (uint32_t(r0 + t * RPI) * uint32_t(ldc) + uint32_t(gcol)) * 2u
                                         : 0x80000000u;
      u32x2 rr[32 / RPI];
      if constexpr (RESID) {   // issued before the staging writes so their latency overlaps them
#pragma unroll
        for (int t = 0; t < 32 / RPI; ++t) rr[t] = __builtin_amdgcn_raw_buffer_load_b64(rsrc_r, voff[t], 0, 0);
      }
#pragma unroll
      for (int gg = 0; gg < NG; ++gg) {
        const f32x4v v = value(i, gg);
        if constexpr (kF32Stage)
          *reinterpret_cast<f32x4v*>(stage + fr * kPitch + (8 * gg + 4 * h) * 4) = v;
        else
          *reinterpret_cast<u32x2*>(stage + fr * kPitch + (8 * gg + 4 * h) * 2) =
              u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      }
      // every staged row of the block read back before the first conversion: the reads' latencies
      // overlap instead of adding up pair by pair
      using Staged = std::conditional_t<kF32Stage, f32x4v, u32x2>;
      Staged sv[32 / RPI];
#pragma unroll
      for (int t = 0; t < 32 / RPI; ++t)
        sv[t] = *reinterpret_cast<const Staged*>(stage + (t * RPI + rl) * kPitch + c4 * 4 * kEl);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < 32 / RPI; ++t) {
        u32x2 packed;
        if constexpr (kF32Stage) {
          f32x4v v = sv[t];
          if constexpr (RESID) {
            v[0] += bf16_lo(rr[t][0]);
            v[1] += bf16_hi(rr[t][0]);
            v[2] += bf16_lo(rr[t][1]);
            v[3] += bf16_hi(rr[t][1]);
          }
          packed = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        } else {
          packed = sv[t];
        }
        __builtin_amdgcn_raw_buffer_store_b64(packed, rsrc_c, voff[t], 0, 0);
      }
      if constexpr (PERSIST) {
        static_assert(32 / RPI * (WM - WM / 2) == kStoresAfter, "the prologue's wait counts these stores");
        if (i == WM / 2 - 1) prefetch_next();   // half the stores out: the next tile's stage 0
      }
    }
  };
  if (direct) {
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      const int row = m0 + wm * (BM / 2) + i * 32 + fr;
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int col = n0 + wn * (BN / 2) + j * 32 + 8 * g + 4 * h;
          if (row < M && col < N)   // N % 8 == 0: a 4-column group is all in or all out
            *reinterpret_cast<f32x4v*>(part + int64_t(slice) * M * N + int64_t(row) * N + col) =
                f32x4v{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
        }
    }
  } else if constexpr (MODE == kSplit) {
    // the slice's fp32 partial sums, staged the same way: whole rows of WN * 128 bytes a store
    // instruction (16 bytes into each of 32 rows straight from the accumulators)
    constexpr int WC = WN * 32, kPitch = WC * 4 + 16, LPR = WC / 4, RPI = 64 / LPR;
    static_assert(64 % LPR == 0, "whole rows per instruction (no split-K form of 96-column waves)");
    static_assert(4 * 32 * kPitch <= Sh::kSmemBytes, "the staging regions fit in the ring's LDS");
    uint8_t* const stage = smem + wave * (32 * kPitch);
    const int rl = lane / LPR, c4 = lane % LPR;
    const int gcol = n0 + wn * (BN / 2) + 4 * c4;
    const __amdgpu_buffer_rsrc_t rsrc_p =
        __builtin_amdgcn_make_buffer_rsrc(part + int64_t(slice) * M * N + int64_t(m0) * N, 0,
                                          uint32_t(min(BM, M - m0)) * uint32_t(N) * 4u, 0x00020000);
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      const int r0 = wm * (BM / 2) + i * 32 + rl;
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<f32x4v*>(stage + fr * kPitch + (j * 32 + 8 * g + 4 * h) * 4) =
              f32x4v{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
      u32x4 sv[32 / RPI];
#pragma unroll
      for (int t = 0; t < 32 / RPI; ++t)
        sv[t] = *reinterpret_cast<const u32x4*>(stage + (t * RPI + rl) * kPitch + c4 * 16);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < 32 / RPI; ++t) {
        const uint32_t off = gcol < N ? (uint32_t(r0 + t * RPI) * uint32_t(N) + uint32_t(gcol)) * 4u : 0x80000000u;
        __builtin_amdgcn_raw_buffer_store_b128(sv[t], rsrc_p, off, 0, 0);
      }
    }
  } else if constexpr (MODE == kSwiGLU) {
    // output columns n0 + wn*BN/4 + 8*gg + 4*(lane/32) + e of C [M, N/2]: gate and up where swiglu_staged
    // put them
    store_staged(std::integral_constant<int, 2 * WN>{}, [&](int i, int gg) __attribute__((always_inline)) {
      const int gj = WN == 3 ? gg >> 2 : 2 * (gg >> 2), uj = WN == 3 ? (gg < 4 ? 2 : 1) : gj + 1;
      const int gr = 4 * (gg & 3), ur = WN == 3 && gg >= 4 ? gr + 8 : gr;
      float gv[4], uv[4], bv[4], q[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        gv[e] = bf16_to_f32(f32_to_bf16(acc[i][gj][gr + e]));
        uv[e] = bf16_to_f32(f32_to_bf16(acc[i][uj][ur + e]));
        bv[e] = __builtin_amdgcn_exp2f(-gv[e] * 1.4426950408889634f) + 1.0f;
        q[e] = silu_quotient(gv[e], bv[e]);
      }
      // one test per four outputs for the rare denominators past 2^126 (fmaxf skips a NaN b, whose
      // quotient the fixup already made NaN)
      if (__builtin_expect(fmaxf(fmaxf(bv[0], bv[1]), fmaxf(bv[2], bv[3])) >= 0x1p126f, 0)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) q[e] = gv[e] / bv[e];
      }
      f32x4v o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = q[e] * uv[e];
      return o;
    }, C, N / 2, N / 2, n0 + wn * (BN / 4));
  } else {
    store_staged(std::integral_constant<int, 4 * WN>{}, [&](int i, int gg) __attribute__((always_inline)) {
      const int j = gg >> 2, g = gg & 3;
      return f32x4v{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
    }, C, N, N, n0 + wn * (BN / 2));
  }
  if (!has_next) break;
  __syncthreads();   // every wave has read its staged rows back: the next stages may land there
  tile_id = next_id;
  m0 = nm0;
  n0 = nn0;
  pre0 = true;
  }   // tile walk
}

// ---------------------------------------------------------------- grouped GEMM
// Program p of the launch multiplies group g = grp[p]'s rows [gstart[g], gstart[g] + grows[g]) of A by
// weight g of B (row-major K x N at B + g*sbg) into the same rows of C.  Table entries that do not
// describe rows inside A (or a weight inside B) count as empty.
struct Groups {
  const int32_t* grp;
  const int32_t* gstart;
  const int32_t* grows;
  int nprog, ntab, nweights, a_rows;
  int64_t sbg;
};
constexpr int kMaxPrograms = 256;
constexpr int kMaxDedupGroups = 1024;   // group tables up to this size have repeated programs skipped

// The read of the weights bounds it while groups are small, so its DMA stream does not stop between
// tiles: WGS workgroups a CU walk the tiles of all programs, and a cursor of its own (tile, K step) runs
// DIST stages ahead of the MFMAs, over tile borders, so the next tile's first stages land during this
// tile's last steps and epilogue.  (One workgroup a 128x128 tile, two a CU, paid a table scan, the first
// stage's latency and a drained epilogue in each.)  Ring slots are runtime values here, as a tile's K
// steps are no whole number of ring turns; that costs 16 address adds a stage.  Tiles are numbered
// program by program, column by column, rows fastest, and XCD x takes a contiguous range, so row tiles
// that share a weight panel run side by side on one L2.  128 experts, gate_up (2048 -> 1536) and down
// (768 -> 2048) together: 64 routed rows 91 -> 81 us, 512 203 -> 190, 2048 243 -> 226, 4096 273 -> 268,
// 8192 315 -> 274, 16384 406 -> 320, 32768 617 -> 441.
// STREAM (see grouped_plan): the weights of a group with one row tile go by the streaming policy.  On
// another box, with skewed groups, both GEMMs without and with it: 128 routed rows 132 -> 118 us, 256 183 ->
// 165, 1024 214 -> 188, 4096 239 -> 219, 8192 279 -> 256.
template <int WM, int WN, int NS, int WGS, bool STREAM>
__global__ __launch_bounds__(kThreads, WGS) void grouped_gemm_kernel(const uint16_t* __restrict__ A,
                                                                   const uint16_t* __restrict__ B,
                                                                   uint16_t* __restrict__ C, int N, int K, int tiles_n,
                                                                   Groups gp) {
  using Sh = Shape<WM, WN>;
  constexpr int BM = Sh::BM, BN = Sh::BN, BK = Sh::BK, kABytes = Sh::kABytes, kBBytes = Sh::kBBytes;
  constexpr int DIST = NS - 1, SPS = Sh::SPS, D = Sh::kDma, U = Sh::kMfma, P = Sh::kPieces;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[NS * (kABytes + kBBytes)];
  __shared__ __attribute__((aligned(16))) int pref[kMaxPrograms + 1];   // tiles of the programs before
  __shared__ int pstart[kMaxPrograms], prows[kMaxPrograms], pgroup[kMaxPrograms];
  __shared__ int wsum[kThreads / 64];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  // the first program listing each group (the ring is still free)
  int* const first_prog = reinterpret_cast<int*>(smem);
  static_assert(kMaxDedupGroups * 4 <= NS * (kABytes + kBBytes), "the group table fits the ring");
  const bool dedup = gp.ntab <= kMaxDedupGroups;
  if (dedup)
    for (int i = tid; i < gp.ntab; i += kThreads) first_prog[i] = kMaxPrograms;
  __syncthreads();
  const int gt = tid < gp.nprog ? gp.grp[tid] : -1;
  const bool in_table = gt >= 0 && gt < gp.ntab;
  if (dedup && in_table) atomicMin(&first_prog[gt], tid);
  const int gs = in_table ? gp.gstart[gt] : 0, gr = in_table ? gp.grows[gt] : 0;
  __syncthreads();
  // a program repeating an earlier program's group would write the same rows with the same values: it
  // takes no tiles
  unsigned cnt = 0;
  if (in_table && (!dedup || first_prog[gt] == tid) && gr > 0 && gs >= 0 && int64_t(gs) + gr <= gp.a_rows &&
      gt < gp.nweights)
    cnt = unsigned(min(uint64_t((unsigned(gr) + BM - 1) / BM) * unsigned(tiles_n), uint64_t(0x7fffffff)));
  // inclusive scan over the 256 programs, within waves, then across them (sums stop at 2^31 - 1 tiles)
  auto sat = [](unsigned a, unsigned b) __attribute__((always_inline)) { return min(a + b, 0x7fffffffu); };
  unsigned v = cnt;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const unsigned u = unsigned(__shfl_up(int(v), off, 64));
    if (lane >= off) v = sat(v, u);
  }
  if (lane == 63) wsum[wave] = int(v);
  __syncthreads();
  for (int i = 0; i < wave; ++i) v = sat(v, unsigned(wsum[i]));
  unsigned total = 0;
  for (int i = 0; i < kThreads / 64; ++i) total = sat(total, unsigned(wsum[i]));
  total = unsigned(__builtin_amdgcn_readfirstlane(int(total)));
  pref[tid + 1] = int(v);
  if (tid == 0) pref[0] = 0;
  pstart[tid] = gs;
  prows[tid] = gr;
  pgroup[tid] = gt;
  __syncthreads();
  unsigned tile = blockIdx.x;
  if (tile >= total) return;   // uniform over the workgroup, before the stream starts

  // tile id -> its group's weight, first row of A, rows and first column.  The last program with
  // pref[p] <= id: each lane looks at four
  struct Tile {
    int first, rows, n0, g;
    bool once;   // the group's only row tile: no other tile reads its weight columns
  };
  auto locate = [&](unsigned id) __attribute__((always_inline)) {
    const unsigned x = id & 7, n8 = total >> 3;
    const int pos = int(x * n8 + min(x, total & 7) + (id >> 3));
    typedef int i32x4v __attribute__((ext_vector_type(4)));
    const i32x4v pr = *reinterpret_cast<const i32x4v*>(&pref[4 * lane]);
    int p = -1;
#pragma unroll
    for (int e = 0; e < 4; ++e) p += __builtin_popcountll(__ballot(pr[e] <= pos));
    const int rows = __builtin_amdgcn_readfirstlane(prows[p]);
    const int rt = int((unsigned(rows) + BM - 1) / BM);
    const int qn = pos - __builtin_amdgcn_readfirstlane(pref[p]);
    const int tn = qn / rt, mt = qn - tn * rt;
    Tile t;
    t.first = __builtin_amdgcn_readfirstlane(pstart[p]) + mt * BM;
    t.rows = min(BM, rows - mt * BM);
    t.n0 = tn * BN;
    t.once = rt == 1;
    t.g = __builtin_amdgcn_readfirstlane(pgroup[p]);
    return t;
  };

  // ---- loaders: as the plain kernel's; A rows past the tile's read as zero, B columns past N read the
  //      next row or zero and only feed columns of C that are never stored
  uint32_t a_voff[Sh::kDmaA], b_voff[Sh::kDmaB];
#pragma unroll
  for (int t = 0; t < Sh::kDmaA; ++t) {
    const int row = (wave * Sh::kDmaA + t) * Sh::kARowsPerKB + lane / Sh::kChunks;
    a_voff[t] = uint32_t(row * K + ((lane % Sh::kChunks) ^ a_swz(row)) * 8) * 2u;
  }
#pragma unroll
  for (int t = 0; t < Sh::kDmaB; ++t) {
    const int piece = 64 * (wave * Sh::kDmaB + t) + lane, k = piece / Sh::kBSlots;
    b_voff[t] = uint32_t(k * N + ((piece % Sh::kBSlots) ^ b_swz<BN>(k)) * 8) * 2u;
  }
  const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(smem));
  const uint32_t wave_a = __builtin_amdgcn_readfirstlane(lds0 + uint32_t(wave * Sh::kDmaA * 1024));
  const uint32_t wave_b = __builtin_amdgcn_readfirstlane(lds0 + uint32_t(NS * kABytes + wave * Sh::kDmaB * 1024));
  const int nk = K / BK;

  // the stream's cursor: the tile and K step of the next stage to go out, and the slot it goes to.
  // Past the last tile its resources are empty: such stages write zeros nobody reads
  unsigned next_load = tile;
  int lkt = nk, lslot = 0;
  bool lonce = false;
  i32x4 rsrc_a = make_rsrc(A, 0), rsrc_b = make_rsrc(B, 0);
  auto advance = [&]() __attribute__((always_inline)) {   // before a stage's DMAs
    if (lkt == nk) {
      lkt = 0;
      if (next_load < total) {
        const Tile t = locate(next_load);
        lonce = STREAM && t.once;
        rsrc_a = make_rsrc(A + int64_t(t.first) * K, uint32_t(int64_t(t.rows) * K) * 2u);
        rsrc_b = make_rsrc(B + int64_t(t.g) * gp.sbg + t.n0, uint32_t((int64_t(K) * N - t.n0) * 2));
        next_load += gridDim.x;
      } else {
        rsrc_a = make_rsrc(A, 0);
        rsrc_b = make_rsrc(B, 0);
        lkt = nk + 1;   // no further tile: never nk again
      }
    }
  };
  auto dma_one = [&](int t) __attribute__((always_inline)) {
    const uint32_t kt = lkt > nk ? 0u : uint32_t(lkt);
    if (t < Sh::kDmaA) {
      dma16(rsrc_a, wave_a + uint32_t(lslot * kABytes + t * 1024), a_voff[t], kt * (BK * 2u));
    } else {
      const int b = t - Sh::kDmaA;
      const uint32_t at = wave_b + uint32_t(lslot * kBBytes + b * 1024), soff = kt * (BK * 2u) * uint32_t(N);
      if (STREAM && lonce) dma16_once(rsrc_b, at, b_voff[b], soff);
      else dma16(rsrc_b, at, b_voff[b], soff);
    }
  };
  auto stage_out = [&]() __attribute__((always_inline)) {   // after a stage's DMAs
    lkt += lkt < nk ? 1 : 0;
    lslot = lslot + 1 == NS ? 0 : lslot + 1;
  };

  // ---- fragment addressing: as the plain kernel's
  const int fr = lane & 31, h = lane >> 5;
  int a_off[WM][SPS], b_off[WN][2];
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int m = wm * (BM / 2) + i * 32 + fr;
#pragma unroll
    for (int ks = 0; ks < SPS; ++ks) a_off[i][ks] = m * Sh::kRowBytes + (((2 * ks + h) ^ a_swz(m)) << 4);
  }
  const int g16 = (lane >> 4) & 1, l16 = lane & 15, jj = l16 >> 2, q = l16 & 3;
#pragma unroll
  for (int j = 0; j < WN; ++j)
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int n = wn * (BN / 2) + j * 32 + 16 * g16 + 4 * q, k = 8 * h + 4 * r + jj;
      b_off[j][r] = k * (2 * BN) + (((n >> 3) ^ b_swz<BN>(k)) << 4) + (q & 1) * 8;
    }
  struct Slice {
    bf16x8 a[WM];
    bf16x8 b[WN];
    i16x4 blo[WN];
  };
  const uint8_t* const smem_b = smem + NS * kABytes;
  auto read_piece = [&](int slot, int ks, int p, Slice& f) __attribute__((always_inline)) {
    if (p < WM) {
      f.a[p] = *reinterpret_cast<const bf16x8*>(smem + slot * kABytes + a_off[p][ks]);
    } else {
      const int j = (p - WM) >> 1, r = (p - WM) & 1;
      const i16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_i16x4*)(smem_b + slot * kBBytes + b_off[j][r] + ks * 16 * 2 * BN));
      if (r == 0) f.blo[j] = x;
      else f.b[j] = __builtin_bit_cast(bf16x8, i16x8{f.blo[j][0], f.blo[j][1], f.blo[j][2], f.blo[j][3], x[0], x[1], x[2], x[3]});
    }
  };
  f32x16 acc[WM][WN];
  auto mfma_one = [&](const Slice& f, int u) __attribute__((always_inline)) {
    const int i = u / WN, j = u % WN;
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.b[j], f.a[i], acc[i][j], 0, 0, 0);
  };
  constexpr int SLOTS = SPS * U;
  constexpr int NPRE = [] {   // DMAs of a step's stage issued before its barrier
    int n = 0;
    for (int o = 0; o < D; ++o)
      if (o * SLOTS / D < (SPS - 1) * U) ++n;
    return n;
  }();

  // ---- epilogue geometry: each wave stages a 32-row block in bf16 in the slot of the tile's last stage
  // (past that step's barrier no wave reads it, and the next step's DMAs are the first into it): waves
  // 0-2 in its B part, wave 3 in its A part
  constexpr int WC = WN * 32, kPitch = WC * 2 + 16, LPR = WC / 4, RPI = 64 / LPR;
  static_assert(3 * 32 * kPitch <= kBBytes && 32 * kPitch <= kABytes, "the staging regions fit one slot");
  constexpr int kStores = WM * (32 / RPI);
  static_assert((DIST - 2) * D + NPRE + kStores < 64, "the wait counts in six bits");
  const int rl = lane / LPR, c4 = lane % LPR;

#pragma unroll
  for (int i = 0; i < DIST; ++i) {
    advance();
#pragma unroll
    for (int t = 0; t < D; ++t) dma_one(t);
    stage_out();
  }
  wait_vmcnt<(DIST - 1) * D>();
  __syncthreads();
  Slice sl[2];
#pragma unroll
  for (int p = 0; p < P; ++p) read_piece(0, 0, p, sl[0]);
  int slot = 0;            // of the stage the MFMAs work on
  bool first_tile = true;
  for (; tile < total; tile += gridDim.x) {
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    for (int kt = 0; kt < nk; ++kt) {
      const int nslot = slot + 1 == NS ? 0 : slot + 1;
      advance();
#pragma unroll
      for (int s = 0; s + 1 < SPS; ++s) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          mfma_one(sl[s & 1], u);
#pragma unroll
          for (int p = 0; p < P; ++p)
            if (p >= u * P / U && p < (u + 1) * P / U) read_piece(slot, s + 1, p, sl[(s + 1) & 1]);
#pragma unroll
          for (int o = 0; o < D; ++o)
            if (o * SLOTS / D == s * U + u) dma_one(o);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      // the next stage landed.  The stages waited for in a tile's first DIST - 1 steps went out before
      // the previous tile's stores, which may still be on their way
      if (first_tile || kt >= DIST - 1) wait_vmcnt<(DIST - 2) * D + NPRE>();
      else wait_vmcnt<(DIST - 2) * D + NPRE + kStores>();
      __syncthreads();
#pragma unroll
      for (int u = 0; u < U; ++u) {
        mfma_one(sl[(SPS - 1) & 1], u);
#pragma unroll
        for (int o = 0; o < D; ++o)
          if (o * SLOTS / D == (SPS - 1) * U + u) dma_one(o);
#pragma unroll
        for (int p = 0; p < P; ++p)
          if (p >= u * P / U && p < (u + 1) * P / U) read_piece(nslot, 0, p, sl[0]);
        __builtin_amdgcn_sched_barrier(0);
      }
      stage_out();
      slot = nslot;
    }
    first_tile = false;

    // ---- epilogue: accumulator (i, j, r) of lane holds tile row wm*BM/2 + i*32 + lane%32, column
    //      wn*BN/2 + j*32 + 8*(r/4) + 4*(lane/32) + r%4; whole rows of a wave's block a store
    const Tile t = locate(tile);
    const int fslot = slot == 0 ? NS - 1 : slot - 1;
    uint8_t* const stage = wave < 3 ? smem + NS * kABytes + fslot * kBBytes + wave * (32 * kPitch) : smem + fslot * kABytes;
    const int gcol = t.n0 + wn * (BN / 2) + 4 * c4;
    const __amdgpu_buffer_rsrc_t rsrc_c = __builtin_amdgcn_make_buffer_rsrc(
        C + int64_t(t.first) * N, 0, uint32_t(t.rows) * uint32_t(N) * 2u, 0x00020000);
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      const int r0 = wm * (BM / 2) + i * 32 + rl;
#pragma unroll
      for (int gg = 0; gg < 4 * WN; ++gg) {
        const int j = gg >> 2, e = 4 * (gg & 3);
        *reinterpret_cast<u32x2*>(stage + fr * kPitch + (8 * gg + 4 * h) * 2) =
            u32x2{pack_bf16x2(acc[i][j][e], acc[i][j][e + 1]), pack_bf16x2(acc[i][j][e + 2], acc[i][j][e + 3])};
      }
      u32x2 sv[32 / RPI];
#pragma unroll
      for (int x = 0; x < 32 / RPI; ++x)
        sv[x] = *reinterpret_cast<const u32x2*>(stage + (x * RPI + rl) * kPitch + c4 * 8);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < 32 / RPI; ++x)
        __builtin_amdgcn_raw_buffer_store_b64(
            sv[x], rsrc_c,
            gcol < N ? (uint32_t(r0 + x * RPI) * uint32_t(N) + uint32_t(gcol)) * 2u : 0x80000000u, 0, 0);
    }
    __syncthreads();   // every wave has read its staged rows back: the next step's DMAs may land there
  }
  wait_vmcnt<0>();     // no stage of the stream lands in LDS that is no longer this workgroup's
}

int cu_count();

template <int WM, int WN, int RING = Shape<WM, WN>::NSA>
int launch_gemm(const void* a, const void* b, const void* residual, void* c, int64_t m, int64_t n, int64_t k,
                bool by_xcd, hipStream_t s) {
  using Sh = Shape<WM, WN, RING>;
  const int64_t tm = (m + Sh::BM - 1) / Sh::BM, tn = (n + Sh::BN - 1) / Sh::BN;
  if (tm * tn > 0x7fffffff) return PTB_ERR_GRID;
  const dim3 grid(unsigned(tm * tn)), block(kThreads);
  if constexpr (WM == 4 && WN == 4) {
    // two or more rounds of 256x256 tiles: one workgroup per CU walks its tiles
    const int64_t cus = cu_count();
    if (!residual && tm * tn >= 2 * cus) {
      gemm_bf16_kernel<4, 4, false, kPlain, true><<<dim3(unsigned(cus)), block, 0, s>>>(
          static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(b), nullptr, static_cast<uint16_t*>(c),
          int(m), int(n), int(k), int(tm), int(tn), int(tm * tn), nullptr, 0);
      return launch_status();
    }
  }
  if (residual)
    gemm_bf16_kernel<WM, WN, true, kPlain, false, RING><<<grid, block, 0, s>>>(
        static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(b), static_cast<const uint16_t*>(residual),
        static_cast<uint16_t*>(c), int(m), int(n), int(k), int(tm), int(tn), by_xcd ? int(tm * tn) : 0, nullptr, 0);
  else
    gemm_bf16_kernel<WM, WN, false, kPlain, false, RING><<<grid, block, 0, s>>>(
        static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(b), nullptr, static_cast<uint16_t*>(c), int(m),
        int(n), int(k), int(tm), int(tn), by_xcd ? int(tm * tn) : 0, nullptr, 0);
  return launch_status();
}

int cu_count() {
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess) hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  return cus;
}

// Tile shape (BM = 64 wm rows by BN = 64 wn columns) and K split of a GEMM.
struct GemmPlan {
  int wm, wn, splits;
  int64_t kchunk;   // K columns per split
  int ring;         // slots of the ring (chosen for 64x128 and 128x128 tiles, given by the others' shape)
  bool by_xcd;      // consecutive tiles to one XCD (one pass; see xcd_order)
};

// Whether the tiles of one pass that fits one round go to the XCDs by consecutive runs.  A run is compact where
// the tiles are many columns wide: an XCD then fetches few columns of B (178x704x10360 11.7 us in the order of the
// workgroup ids, 6.4 by runs).  Over few columns a run reaches into two groups of kGroupM tile-rows, and the
// ids' order, which gives an XCD the same row of every group, fetches less: 3146x2176x296 13.7 us by runs, 10.4 by
// ids, 1067x5760x160 27.3 / 20.1, 2105x1088x1120 10.2 / 8.8.  By ids where the most rows and columns that one XCD
// fetches are over 10% more by runs: of 26 such sizes 24 were faster by ids or within 0.5%, and nearly all others by
// runs.  Tile counts that divide by 8 keep to runs.
bool xcd_order(int bm, int bn, int tiles_m, int tiles_n, int64_t cus) {
  const int n = tiles_m * tiles_n;
  if (n % 8 == 0 || n > cus || tiles_m < 12 || tiles_m <= tiles_n || tiles_m > 256) return true;
  int most[2] = {0, 0};   // by ids, by runs
  for (int runs = 0; runs < 2; ++runs) {
    for (int x = 0; x < 8; ++x) {
      const int count = n / 8 + (x < n % 8 ? 1 : 0), first = x * (n / 8) + std::min(x, n % 8);
      bool row[256] = {}, col[256] = {};
      int fetched = 0;
      for (int i = 0; i < count; ++i) {
        const int pid = runs ? first + i : x + 8 * i, group = pid / (kGroupM * tiles_n), in = pid % (kGroupM * tiles_n);
        const int rows = std::min(tiles_m - group * kGroupM, kGroupM), r = group * kGroupM + in % rows, c = in / rows;
        fetched += (row[r] ? 0 : bm) + (col[c] ? 0 : bn);
        row[r] = col[c] = true;
      }
      most[runs] = std::max(most[runs], fetched);
    }
  }
  return 10 * most[1] <= 11 * most[0];
}

// Cost model of a plan, in us.  A round of workgroups (one a CU) costs `step` per 64-deep K step
// plus `load` x (share of the CUs busy: they share the chip's power and L2 bandwidth) and `fixed` for
// its prologue and epilogue.  Reading the operands and writing C takes kMemUs plus kMemUsPerMB; the
// two overlap partly, which their root sum of squares follows.  A split adds the finish launch,
// kFinishUs, and writing and reading 4 bytes per output and slice at kPartialUsPerMB.  Fitted by
// least squares to 3969 (shape, tile, split) times on MI355X over 239 shapes with M 1 .. 4096, K
// 64 .. 12288 and N 128 .. 24576: 4.7% rms error, and the plans picked by the fit as it came out (before 256x256's
// constants were raised, below, and splits had to beat one pass by kSplitMargin) ran within 0.9% (geometric
// mean) of the best measured plan of each shape, 1.23x faster than the previous rule's plans (one
// pass of 128x128 tiles where those covered 3/4 of the CUs, splits of 64x128 tiles only; both with
// 32-deep stages): 640x12288x4096 147 -> 71 us, 1280x12288x4096 237 -> 114, 384x12288x4096 105 -> 50,
// 640x4096x6144 53 -> 42, 2048x4096x12288 173 -> 150, 32x4096x6144 16 -> 14.5, 3000x8192x512 65 -> 36.
struct TileCost {
  int wm, wn;
  double step, load, fixed;
};
constexpr TileCost kTiles[] = {{4, 4, 0.830, 0.500, 6.29}, {4, 3, 0.620, 0.511, 5.89}, {4, 2, 0.555, 0.203, 3.72},
                               {2, 4, 0.592, 0.250, 3.92}, {2, 2, 0.358, 0.196, 2.42}, {1, 2, 0.296, 0.141, 1.68}};
// (256x256's step and load a little above the fit's 0.816 and 0.464: at 1664x12288x4096 the fit took two
// slices of 256x256 tiles, 1.4% of the layer slower than one pass of 256x128 ones)
constexpr double kMemUs = 3.3, kMemUsPerMB = 0.106, kFinishUs = 1.9, kPartialUsPerMB = 0.148;
// A split that nobody has to bring a workspace for (required_slices) has to beat one pass by these factors, taller
// outputs than wide by the larger one: the fit took their one pass in an order over the XCDs that they no longer
// run in.  Of 128 sizes at which the model saw a split ahead by less than 1.3, the 37 that it put less than this
// ahead ran 7% slower split (geometric mean; 3954x2368x160 11.7 us in one pass, 14.6 split, 492x2496x2304 13.0 /
// 16.7), the others 10% faster (270x7488x7720 52.6 / 48.0, 293x3520x2728 20.5 / 16.5).
constexpr double kSplitMarginTall = 1.12, kSplitMargin = 1.07;
constexpr int kMaxSplits = 8;
constexpr int64_t kFitK = 16384;   // past it (the fit ends at 12288) splits keep to the narrow rule below

// The K slices that ptb_gemm_bf16_ws asks a caller's workspace for: those of 64x128 tiles on at most half
// of the CUs where a workgroup's operand stream (90 GB/s; 2.5 us to launch) gets shorter by more than the
// finish launch (1.5 us) and the partials' traffic (2.5 TB/s) take.  Part of the call's contract, not of the plan: such a call is refused without
// the room for them, and every other one runs with the room it has.
int required_slices(int64_t m, int64_t n, int64_t k, int64_t cus) {
  const int64_t t64 = ((m + 63) / 64) * ((n + 127) / 128);
  auto stream = [&](int sp) { return 2.5 + double(k) / sp * (64 + 128) * 2 / 90e3; };
  int best = 1;
  double best_us = stream(1);
  for (int sp = 2; sp <= 8 && k >= 1024 && k / sp >= 256 && t64 * sp <= cus; sp *= 2) {
    const double us = stream(sp) + (1.5 + sp * double(m) * double(n) * 8 / 2.5e6);
    if (us < best_us) {
      best_us = us;
      best = sp;
    }
  }
  const int64_t kc = ((k + best - 1) / best + 63) / 64 * 64;
  return int((k + kc - 1) / kc);
}

// The cheapest plan by the model.  Splits: K at least 1024 and slices at least 128 deep (below, the
// finish launch costs more than the shorter slices save), all in one round of workgroups; a K past
// the fitted range is split only when 128x128 tiles would leave a quarter of the CUs idle.  256-row
// and 128-row tiles need 256 rows of A within the 32-bit buffer offsets, and the four-slot rings
// their deeper run past the end of a slice of B.  The partials take at most `room` bytes (kAnyRoom: what
// they need; 0: one pass).
constexpr size_t kAnyRoom = ~size_t(0);
GemmPlan make_plan(int64_t m, int64_t n, int64_t k, size_t room, int64_t cus) {
  auto tiles = [&](int64_t bm, int64_t bn) { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn); };
  const bool may_split = room > 0 && k >= 1024 && (k <= kFitK || 4 * tiles(128, 128) < 3 * cus);
  const double mem = kMemUs + kMemUsPerMB * 2e-6 * (double(k) * double(n) + double(m) * (double(k) + double(n)));
  const double partial = kPartialUsPerMB * 8e-6 * double(m) * double(n);
  const bool tall = int64_t(256) * k * 2 < (int64_t(1) << 32);
  const double margin = !may_split || required_slices(m, n, k, cus) > 1 ? 1.0 : m > n ? kSplitMarginTall : kSplitMargin;
  GemmPlan best{1, 2, 1, k, 4, true};
  double best_t = -1.0;
  for (const TileCost& c : kTiles) {
    if (c.wm > 1 && !tall) continue;
    const int64_t t = tiles(64 * c.wm, 64 * c.wn);
    const int run_ahead = c.wm * c.wn >= 8 ? kRunAhead : kRunAheadDeep;
    for (int sp = 1; sp <= (may_split && c.wn != 3 ? kMaxSplits : 1); ++sp) {
      if (sp > 1 && (t * sp > cus || k / sp < 128)) break;
      const int64_t kc = sp == 1 ? k : ((k + sp - 1) / sp + 63) / 64 * 64;
      const int64_t splits = (k + kc - 1) / kc;
      if (splits > 1 && size_t(splits) * size_t(m) * size_t(n) * sizeof(float) > room) break;
      if ((kc + run_ahead) * n * 2 >= (int64_t(1) << 32)) continue;
      const int64_t w = t * splits, full = (w - 1) / cus;
      const double steps = double((kc + 63) / 64), last = double(w - full * cus) / double(cus);
      const double body = double(full) * (steps * (c.step + c.load) + c.fixed) + steps * (c.step + c.load * last) + c.fixed;
      double us = std::sqrt(body * body + mem * mem);
      if (splits > 1) us += kFinishUs + partial * double(splits);
      if (splits > 1) us *= margin;
      if (best_t < 0.0 || us < best_t) {
        best_t = us;
        best = GemmPlan{c.wm, c.wn, int(splits), kc, 4, true};
      }
    }
  }
  // 64x128 tiles of few K steps, or of a moderate number on few CUs, take rings of 3 slots: the fourth one's 24 KB
  // cost 0.3 us of a launch, which only longer ranges, with more of the chip asking for operands, make up for.
  // 3 against 4 slots: 3x128x272 2.94 us / 3.26, 302x704x8 4.67 / 4.94, 2048x768x768 5.52 / 5.79, 330x832x1056 5.20
  // / 5.48, 9x1600x120 6.99 / 7.22; but 2x896x7856 (62 workgroups of 14 steps) 6.35 / 5.65, 97x1728x8896 11.7 / 9.3.
  const int64_t steps = (best.kchunk + 63) / 64, wgs = tiles(64, 128) * best.splits;
  if (best.wm == 1 && (steps <= 12 || (steps <= 32 && wgs <= 48))) best.ring = 3;
  // 128x128 tiles in one pass likewise (128 KB of LDS against 96): 727x64x2880 4.19 us / 4.40, 469x320x7120 5.74 /
  // 6.07, 935x768x3072 7.25 / 7.46, 3301x1088x728 8.36 / 8.74; 137x2560x11712 (40 steps) 19.3 / 18.3.
  if (best.wm == 2 && best.wn == 2 && best.splits == 1 && steps <= 16) best.ring = 3;
  if (best.splits == 1 && tiles(64 * best.wm, 64 * best.wn) <= cus)
    best.by_xcd = xcd_order(64 * best.wm, 64 * best.wn, int((m + 64 * best.wm - 1) / (64 * best.wm)),
                            int((n + 64 * best.wn - 1) / (64 * best.wn)), cus);
  return best;
}

// The plan of a size is asked for twice a call, by the workspace query and by the launch (with other room where no
// split is wanted), and a model comes back to a few sizes: a thread keeps the last plan of each of 64 places that
// sizes are spread over.
GemmPlan gemm_plan(int64_t m, int64_t n, int64_t k, size_t room) {
  struct Last {
    int64_t m = -1, n = 0, k = 0, cus = 0;
    size_t room = 0;
    GemmPlan plan{};
  };
  static thread_local Last kept[64];
  const int64_t cus = cu_count();
  const uint64_t h = (uint64_t(m) * 0x9e3779b97f4a7c15u + uint64_t(n)) * 0xc2b2ae3d27d4eb4fu + uint64_t(k) + room;
  Last& last = kept[(h * 0x9e3779b97f4a7c15u) >> 58];
  if (last.m != m || last.n != n || last.k != k || last.room != room || last.cus != cus)
    last = Last{m, n, k, cus, room, make_plan(m, n, k, room, cus)};
  return last.plan;
}

int launch_planned(const GemmPlan& p, const void* a, const void* b, const void* residual, void* c, int64_t m,
                   int64_t n, int64_t k, hipStream_t s) {
  if (p.wm == 4 && p.wn == 3) return launch_gemm<4, 3>(a, b, residual, c, m, n, k, p.by_xcd, s);
  if (p.wm == 4 && p.wn == 4) return launch_gemm<4, 4>(a, b, residual, c, m, n, k, p.by_xcd, s);
  if (p.wm == 4 && p.wn == 2) return launch_gemm<4, 2>(a, b, residual, c, m, n, k, p.by_xcd, s);
  if (p.wm == 2 && p.wn == 4) return launch_gemm<2, 4>(a, b, residual, c, m, n, k, p.by_xcd, s);
  if (p.wm == 2 && p.wn == 2 && p.ring == 3) return launch_gemm<2, 2, 3>(a, b, residual, c, m, n, k, p.by_xcd, s);
  if (p.wm == 2 && p.wn == 2) return launch_gemm<2, 2>(a, b, residual, c, m, n, k, p.by_xcd, s);
  if (p.ring == 3) return launch_gemm<1, 2, 3>(a, b, residual, c, m, n, k, p.by_xcd, s);
  return launch_gemm<1, 2>(a, b, residual, c, m, n, k, p.by_xcd, s);
}

}  // namespace

PTB_EXPORT int ptb_gemm_bf16(const void* a, const void* b, const void* residual, void* c, int64_t m,
                             int64_t n, int64_t k, void* stream) {
  if (m < 0 || n < 0 || k < 0) return PTB_ERR_SHAPE;
  if (m == 0 || n == 0) return PTB_OK;
  if (!a || !b || !c) return PTB_ERR_NULL;
  if (k == 0) return PTB_ERR_UNSUPPORTED;
  if (m > 0x7fffffff || n > 0x7fffffff || k > 0x7fffffff) return PTB_ERR_SHAPE;
  if (k % 64 || n % 8) return PTB_ERR_UNSUPPORTED;
  // buffer offsets are 32-bit: B and one 256-row panel of A must each stay under 4 GB
  if ((k + kRunAhead) * n * 2 >= (int64_t(1) << 32) || int64_t(256) * k * 2 >= (int64_t(1) << 32) ||
      n > kMaxOutCols)
    return PTB_ERR_UNSUPPORTED;
  if (!aligned16(a) || !aligned16(b) || !aligned16(c) || (residual && !aligned16(residual)))
    return PTB_ERR_ALIGN;
  return launch_planned(gemm_plan(m, n, k, 0), a, b, residual, c, m, n, k, static_cast<hipStream_t>(stream));
}

namespace {

// C = bf16(sum_s P[s] (+ R)), 4 consecutive elements per thread, the slices in order, P_0 + P_1 + ...;
// all S loads go out before the first add.
template <int S>
__global__ __launch_bounds__(256) void splitk_finish(const float* __restrict__ P, int64_t mn,
                                                     const uint16_t* __restrict__ R, uint16_t* __restrict__ C) {
  const int64_t q = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (q >= mn) return;
  f32x4v v[S];
#pragma unroll
  for (int u = 0; u < S; ++u) v[u] = *reinterpret_cast<const f32x4v*>(P + int64_t(u) * mn + q);
  f32x4v acc = v[0];
#pragma unroll
  for (int u = 1; u < S; ++u) acc = acc + v[u];
  if (R) {
    const u32x2 rr = *reinterpret_cast<const u32x2*>(R + q);
    acc.x += bf16_lo(rr[0]);
    acc.y += bf16_hi(rr[0]);
    acc.z += bf16_lo(rr[1]);
    acc.w += bf16_hi(rr[1]);
  }
  *reinterpret_cast<u32x2*>(C + q) = u32x2{pack_bf16x2(acc.x, acc.y), pack_bf16x2(acc.z, acc.w)};
}

template <int WM, int WN, int RING = Shape<WM, WN>::NSA>
int launch_split(const GemmPlan& p, const uint16_t* a, const uint16_t* b, const uint16_t* residual, uint16_t* c,
                 float* part, int64_t m, int64_t n, int64_t k, hipStream_t s) {
  using Sh = Shape<WM, WN, RING>;
  const int64_t tm = (m + Sh::BM - 1) / Sh::BM, tn = (n + Sh::BN - 1) / Sh::BN;   // at most a tile a CU
  gemm_bf16_kernel<WM, WN, false, kSplit, false, RING><<<dim3(unsigned(tm * tn * p.splits)), dim3(kThreads), 0, s>>>(
      a, b, nullptr, nullptr, int(m), int(n), int(k), int(tm), int(tn), int(tm * tn * p.splits), part,
      int(p.kchunk));
  const int64_t mn = m * n;
  const dim3 grid(unsigned((mn / 4 + 255) / 256)), block(256);
  static_assert(kMaxSplits == 8, "a finish kernel for every split count");
  switch (p.splits) {
    case 2: splitk_finish<2><<<grid, block, 0, s>>>(part, mn, residual, c); break;
    case 3: splitk_finish<3><<<grid, block, 0, s>>>(part, mn, residual, c); break;
    case 4: splitk_finish<4><<<grid, block, 0, s>>>(part, mn, residual, c); break;
    case 5: splitk_finish<5><<<grid, block, 0, s>>>(part, mn, residual, c); break;
    case 6: splitk_finish<6><<<grid, block, 0, s>>>(part, mn, residual, c); break;
    case 7: splitk_finish<7><<<grid, block, 0, s>>>(part, mn, residual, c); break;
    default: splitk_finish<8><<<grid, block, 0, s>>>(part, mn, residual, c); break;
  }
  return launch_status();
}

size_t plan_workspace(const GemmPlan& p, int64_t m, int64_t n) {
  return p.splits < 2 ? 0 : size_t(p.splits) * size_t(m) * size_t(n) * sizeof(float);
}

}  // namespace

PTB_EXPORT int ptb_gemm_bf16_plan(int64_t m, int64_t n, int64_t k, int split, int32_t* plan) {
  if (!plan) return PTB_ERR_NULL;
  if (m <= 0 || n <= 0 || k <= 0 || m > 0x7fffffff || n > 0x7fffffff || k > 0x7fffffff) return PTB_ERR_SHAPE;
  const GemmPlan p = gemm_plan(m, n, k, split ? kAnyRoom : 0);
  plan[0] = 64 * p.wm;
  plan[1] = 64 * p.wn;
  plan[2] = p.splits;
  return PTB_OK;
}

PTB_EXPORT size_t ptb_gemm_bf16_workspace_bytes(int64_t m, int64_t n, int64_t k) {
  if (m <= 0 || n <= 0 || k <= 0 || m > 0x7fffffff || n > 0x7fffffff || k > 0x7fffffff) return 0;
  return plan_workspace(gemm_plan(m, n, k, kAnyRoom), m, n);
}

PTB_EXPORT int ptb_gemm_bf16_ws(const void* a, const void* b, const void* residual, void* c, int64_t m, int64_t n,
                                int64_t k, void* workspace, size_t workspace_bytes, void* stream) {
  if (m <= 0 || n <= 0 || k <= 0 || k % 64 || n % 8 || m > 0x7fffffff || n > 0x7fffffff || k > 0x7fffffff)
    return ptb_gemm_bf16(a, b, residual, c, m, n, k, stream);   // refused or trivial there
  GemmPlan p = gemm_plan(m, n, k, kAnyRoom);
  if (p.splits > 1) {
    const size_t need = plan_workspace(p, m, n);
    const size_t room = workspace && aligned16(workspace) ? workspace_bytes : 0;
    const int required = required_slices(m, n, k, cu_count());
    if (required > 1) {
      if (!a || !b || !c || !workspace) return PTB_ERR_NULL;
      if (workspace_bytes < std::min(need, size_t(required) * size_t(m) * size_t(n) * sizeof(float)))
        return PTB_ERR_WORKSPACE;
      if (!aligned16(workspace)) return PTB_ERR_ALIGN;
    }
    if (room < need) p = make_plan(m, n, k, room, cu_count());
  }
  if (p.splits < 2) return ptb_gemm_bf16(a, b, residual, c, m, n, k, stream);   // one pass
  if (!a || !b || !c) return PTB_ERR_NULL;
  // B and a tile's rows of A within 32-bit buffer offsets (the plan takes 64-row tiles past K = 2^23)
  if ((k + kRunAhead) * n * 2 >= (int64_t(1) << 32) || int64_t(64) * k * 2 >= (int64_t(1) << 32))
    return PTB_ERR_UNSUPPORTED;
  if (!aligned16(a) || !aligned16(b) || !aligned16(c) || (residual && !aligned16(residual))) return PTB_ERR_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto ap = static_cast<const uint16_t*>(a), bp = static_cast<const uint16_t*>(b);
  auto rp = static_cast<const uint16_t*>(residual);
  auto cp = static_cast<uint16_t*>(c);
  float* part = static_cast<float*>(workspace);
  if (p.wm == 4 && p.wn == 4) return launch_split<4, 4>(p, ap, bp, rp, cp, part, m, n, k, s);
  if (p.wm == 4) return launch_split<4, 2>(p, ap, bp, rp, cp, part, m, n, k, s);
  if (p.wm == 2 && p.wn == 4) return launch_split<2, 4>(p, ap, bp, rp, cp, part, m, n, k, s);
  if (p.wm == 2) return launch_split<2, 2>(p, ap, bp, rp, cp, part, m, n, k, s);
  if (p.ring == 3) return launch_split<1, 2, 3>(p, ap, bp, rp, cp, part, m, n, k, s);
  return launch_split<1, 2>(p, ap, bp, rp, cp, part, m, n, k, s);
}

namespace {

template <int WM, int WN>
int launch_swiglu(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k, hipStream_t s) {
  using Sh = Shape<WM, WN>;
  const int64_t tm = (m + Sh::BM - 1) / Sh::BM, tn = (n + Sh::BN - 1) / Sh::BN;
  if (tm * tn > 0x7fffffff) return PTB_ERR_GRID;
  gemm_bf16_kernel<WM, WN, false, kSwiGLU><<<dim3(unsigned(tm * tn)), dim3(kThreads), 0, s>>>(
      static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(b), nullptr, static_cast<uint16_t*>(c), int(m),
      int(n), int(k), int(tm), int(tn), int(tm * tn), nullptr, 0);
  return launch_status();
}

// The groups that `rows` rows hit, spread over them at random with popularities of log-normal deviation `skew`
// (0: all alike): the mean over eight equal shares of the groups.
double groups_hit(double groups, double rows, double skew) {
  static const double share[] = {-1.534, -0.887, -0.489, -0.157, 0.157, 0.489, 0.887, 1.534};   // normal quantiles
  double sum = 0.0;
  for (const double z : share) sum += 1.0 - std::exp(-rows / groups * std::exp(skew * z - 0.5 * skew * skew));
  return groups * sum / 8.0;
}

// The tile of a grouped GEMM: 0 128x256, 1 128x128 (one workgroup a CU), 2 64x128 (two).  The host does
// not see the row counts: a hit group of m rows takes m / BM + 1/2 row tiles, or one up to m = BM / 2, and the
// cost of those rounds is the plain GEMM's (its step, load and fixed per tile; 128x128 steps 0.34 here).  Nor does
// it see how evenly the rows are routed: the tile that is cheapest for evenly popular groups gives way to the one
// with the least product of costs for even and strongly skewed popularities where that product is less than
// 1 / 1.3 of its own.  (By even popularities alone the wide tile ran where skewed rows hit too few groups to fill the
// CUs with it: 32 rows of 16 groups, 4096 -> 2816, 6 of them hit, 56.8 us, now 42.0; 57 rows of 32, 2048 -> 1536,
// 25.1, now 18.2.)  Over 1040 points (2 to 128 groups, 17 to 8192 rows, four weights, deviations of 0 to 1.5) the
// pick runs within 1.6% (geometric mean) of the best tile and 12% faster than a workgroup a 128x128 tile.
struct GroupedPlan {
  int tile;
  bool stream;
};
// The weights go by the streaming policy, tile by tile where a group has one row tile, if
// - a group's mean rows fit one (128 experts, gate_up / down: 4 rows each 137.0 -> 119.9 / 75.0 -> 65.4 us, 60
//   156.4 -> 145.0 / 87.9 -> 80.6; at 200 rows 255 -> 262 / 145 -> 146);
// - the table's weights pass kStreamBytes, so that the groups of the next call are not all in the cache; and
// - a fifth of the groups are expected to be hit.  Fewer stay in the cache up to the next call, through an expert
//   block's two GEMMs in turn: with the same rows in each call 17 rows over 128 experts' gate_up and down (146 MB of
//   1.2 GB) 28.3 -> 35.8 us, with other rows routed to the same weights 36.9 either way; past the line 32 rows (283
//   MB) 53.1 -> 53.8 and 54.6 -> 53.2, 48 rows with other rows 73.0 -> 67.2, 96 rows 125.1 -> 114.0 and 117.5 ->
//   107.3.  (A GEMM by itself on the same 100 to 250 MB in each call loses up to 9% of what the block gains.)
GroupedPlan grouped_plan(int64_t groups, int64_t a_rows, int64_t n, int64_t k, int64_t cus) {
  struct {
    int bm, bn;
    double step, load, fixed;
  } const tiles[] = {{128, 256, 0.592, 0.250, 3.92}, {128, 128, 0.340, 0.196, 2.42}, {64, 128, 0.296, 0.141, 1.68}};
  if (groups <= 0) return {2, false};
  const double hit = double(groups) * (1.0 - std::exp(-double(a_rows) / double(groups)));
  const double hits[] = {hit, groups_hit(double(groups), double(a_rows), 2.0)};
  const double mean = double(a_rows) / hit, steps = double(k / 64);
  double t[3][2];
  int even = 0, both = 0;   // the cheapest for even popularities, and by the product
  for (int i = 0; i < 3; ++i) {
    const auto& c = tiles[i];
    for (int j = 0; j < 2; ++j) {
      const double m = double(a_rows) / hits[j];
      const double w = hits[j] * (m > c.bm / 2 ? m / c.bm + 0.5 : 1.0) * double((n + c.bn - 1) / c.bn);
      const double full = std::ceil(w / double(cus)) - 1.0, last = w / double(cus) - full;
      t[i][j] = full * (steps * (c.step + c.load) + c.fixed) + steps * (c.step + c.load * last) + c.fixed;
    }
    if (t[i][0] < t[even][0]) even = i;
    if (t[i][0] * t[i][1] < t[both][0] * t[both][1]) both = i;
  }
  const int best = t[even][0] * t[even][1] > 1.3 * t[both][0] * t[both][1] ? both : even;
  const double table = double(groups) * double(n) * double(k) * 2.0;
  return {best, mean <= tiles[best].bm && table > double(kStreamBytes) && 5.0 * hit > double(groups)};
}

// A workgroup for each of the tiles there can be, up to the CUs' WGS each.
template <int WM, int WN, int NS, int WGS>
int launch_grouped(bool stream, const void* a, const void* b, void* c, int64_t n, int64_t k, const Groups& gp,
                   hipStream_t s) {
  using Sh = Shape<WM, WN>;
  const int64_t tn = (n + Sh::BN - 1) / Sh::BN, tm = (int64_t(gp.a_rows) + Sh::BM - 1) / Sh::BM + gp.nprog;
  const int64_t grid = std::min<int64_t>(tm * tn, WGS * cu_count());
  const auto kernel = stream ? grouped_gemm_kernel<WM, WN, NS, WGS, true> : grouped_gemm_kernel<WM, WN, NS, WGS, false>;
  kernel<<<dim3(unsigned(grid)), dim3(kThreads), 0, s>>>(
      static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(b), static_cast<uint16_t*>(c), int(n), int(k),
      int(tn), gp);
  return launch_status();
}

}  // namespace

PTB_EXPORT int ptb_gemm_swiglu_bf16(const void* a, const void* b, void* c, int64_t m, int64_t inter, int64_t k,
                                    void* stream) {
  if (m < 0 || inter < 0 || k < 0) return PTB_ERR_SHAPE;
  if (m == 0 || inter == 0) return PTB_OK;
  if (!a || !b || !c) return PTB_ERR_NULL;
  if (k == 0 || k % 64 || inter % 128) return PTB_ERR_UNSUPPORTED;
  const int64_t n = 2 * inter;
  if (m > 0x7fffffff || n > 0x7fffffff || k > 0x7fffffff) return PTB_ERR_SHAPE;
  if ((k + kRunAhead) * n * 2 >= (int64_t(1) << 32) || int64_t(256) * k * 2 >= (int64_t(1) << 32) ||
      n > kMaxOutCols)
    return PTB_ERR_UNSUPPORTED;
  if (!aligned16(a) || !aligned16(b) || !aligned16(c)) return PTB_ERR_ALIGN;
  // The tiles of the [m, 2*inter] product by the plain GEMM's model, whose pick was within 0.2%
  // (geometric mean) of the best tile over 100 (tokens, hidden, inter) points and 1.7x faster than
  // 256x256 tiles throughout: 1 token of 4096 -> 12288 84 -> 46 us (96 workgroups of which one row is
  // wanted -> 192 of 64x128), 200 tokens 84.5 -> 65 (192 of 256x128), 640 167 -> 130 (128x256), 1024
  // 184 -> 171 (two even rounds of 256x192), 2048 unchanged.
  const GemmPlan p = gemm_plan(m, n, k, 0);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (p.wm == 4 && p.wn == 4) return launch_swiglu<4, 4>(a, b, c, m, n, k, s);
  if (p.wm == 4 && p.wn == 3) return launch_swiglu<4, 3>(a, b, c, m, n, k, s);
  if (p.wm == 4) return launch_swiglu<4, 2>(a, b, c, m, n, k, s);
  if (p.wm == 2 && p.wn == 4) return launch_swiglu<2, 4>(a, b, c, m, n, k, s);
  if (p.wm == 2) return launch_swiglu<2, 2>(a, b, c, m, n, k, s);
  return launch_swiglu<1, 2>(a, b, c, m, n, k, s);
}

PTB_EXPORT int ptb_grouped_gemm_plan(int64_t groups, int64_t a_rows, int64_t k, int64_t n, int32_t* plan) {
  if (!plan) return PTB_ERR_NULL;
  if (groups <= 0 || a_rows <= 0 || k <= 0 || n <= 0 || a_rows > 0x7fffffff || k > 0x7fffffff || n > 0x7fffffff)
    return PTB_ERR_SHAPE;
  const GroupedPlan p = grouped_plan(groups, a_rows, n, k, cu_count());
  plan[0] = p.tile == 2 ? 64 : 128;
  plan[1] = p.tile == 0 ? 256 : 128;
  plan[2] = p.stream;
  return PTB_OK;
}

PTB_EXPORT int ptb_grouped_gemm_bf16(const void* a, const void* b, const int32_t* group, const int32_t* start,
                                     const int32_t* rows, void* c, int64_t nprog, int64_t ntab, int64_t a_rows,
                                     int64_t nweights, int64_t k, int64_t n, int64_t weight_stride, void* stream) {
  if (nprog < 0 || ntab < 0 || a_rows < 0 || nweights < 0 || k < 0 || n < 0) return PTB_ERR_SHAPE;
  if (nprog == 0 || a_rows == 0 || n == 0) return PTB_OK;
  if (!a || !b || !group || !start || !rows || !c) return PTB_ERR_NULL;
  if (k == 0 || k % 64 || n % 8 || nprog > kMaxPrograms) return PTB_ERR_UNSUPPORTED;
  if (weight_stride < k * n || a_rows > 0x7fffffff || ntab > 0x7fffffff || nweights > 0x7fffffff) return PTB_ERR_SHAPE;
  if ((k + kRunAhead) * n * 2 >= (int64_t(1) << 32) || int64_t(128) * k * 2 >= (int64_t(1) << 32) ||
      n > kMaxOutCols)
    return PTB_ERR_UNSUPPORTED;
  if (!aligned16(a) || !aligned16(b) || !aligned16(c) || (weight_stride % 8)) return PTB_ERR_ALIGN;
  // a bound on the 128x128 tiles of every program together: each program's rows lie inside A
  if (((a_rows + 127) / 128 + nprog) * ((n + 127) / 128) > 0x7fffffff) return PTB_ERR_GRID;
  const Groups gp{group, start, rows, int(nprog), int(ntab), int(nweights), int(a_rows), weight_stride};
  hipStream_t s = static_cast<hipStream_t>(stream);
  const GroupedPlan p = grouped_plan(std::min(nprog, std::min(ntab, nweights)), a_rows, n, k, cu_count());
  switch (p.tile) {
    case 0: return launch_grouped<2, 4, 3, 1>(p.stream, a, b, c, n, k, gp, s);
    case 1: return launch_grouped<2, 2, 4, 1>(p.stream, a, b, c, n, k, gp, s);
    default: return launch_grouped<1, 2, 3, 2>(p.stream, a, b, c, n, k, gp, s);
  }
}
