// Projections of many rows at once (a prompt's prefill, a server's batch):
// y = x W^T over M rows as a tiled GEMM on the matrix cores, for bf16 weights
// and for 8-bit ones (int8 or fp8-e4m3fn codes with an fp32 scale per row).
//
//  * block = four waves on an output tile of TM rows x 128 weight rows, or
//    eight on TM rows x 256. The waves stand 2 x 2 or 2 x 4 (TM = 32 NT: each
//    wave 16 NT rows x 64 weight rows) or, for tiles of at most 48 rows, 1 x 4
//    (TM = 16 NT: all rows x 32 weight rows);
//  * each 64-deep k step stages the x tile (TM rows x 128 bytes) and the
//    weight tile (128 or 256 rows of 128 bytes, or 64 for 8-bit codes) into LDS
//    with LDS-direct loads, a ring of kStages steps deep: as many as leave room
//    for two four-wave blocks per CU or one of eight waves, because what bounds
//    a few hundred rows is the weight stream, i.e. the bytes in flight, and what
//    bounds more is the matrix cores, which need other waves while some wait at
//    a barrier. A wave waits only for the step it is about to multiply (vmcnt
//    counts the later steps' loads, the same number in every step: steps past
//    the end are loaded through an empty descriptor, as zeros);
//  * x chunk c (16 bytes) of row r sits at column c ^ (r & 7), weight chunk c
//    of an 8-bit row at c ^ ((r >> 2) & 3), so the fragment reads of eight
//    consecutive lanes hit eight different column groups;
//  * D^T = W X^T on v_mfma_f32_16x16x32_bf16 (weight rows as M, x rows as N):
//    a lane ends with four consecutive output columns of one row (8-byte
//    stores). 8-bit codes become bf16 in registers (exact for both formats)
//    after one 16-byte read per lane and step: lane quad q holds k
//    16 q .. 16 q + 15 and x is read in the same permuted order, which leaves
//    each dot product unchanged. The row scale multiplies the fp32 sum, as in
//    the batch-one GEMVs;
//  * SwiGLU tiles interleave gate and up rows in groups of 16 (32 with two
//    waves along the rows), so a lane holds the gate and up dot products of the
//    same outputs;
//  * when the tiles leave block slots empty, each tile's k range splits over
//    up to 12 blocks; they store fp32 partial sums and a second launch adds
//    them in split order and applies the epilogue (with the next RMSNorm, when
//    the caller wants it);
//  * blocks are laid out XCD-major: the blocks of one weight tile share an
//    XCD (block L runs on XCD L % 8), so its L2 serves the tile to all of them.
//
// Epilogues keep the batch-one GEMV's bf16 boundaries (store, + residual,
// SwiGLU, argmax keys); fp32 accumulation over k in 64-wide steps.
//
// Measured per 8B layer at 201 rows, bf16, against two 128-row launches of the
// strips (gemm_rows.hip): QKV 99 -> 28 us, O 72 -> 24 (with the next norm),
// gate/up 190 -> 67 (605 TFLOP/s, 3.0 TB/s), down 170 -> 51; 0.6B at 100 rows
// 10 / 13 / 12 / 14 -> 8 / 10 / 8 / 11. 4B at 300 rows, fp8, against the GEMV
// row by row: 8.4 ms -> 23 + 25 + 42 + 39 us (gate/up 712 TFLOP/s). What bounds
// them: a CU stages some 50 bytes per ns, x and weights together, whatever the
// ring's depth (a step of 18 KB for 16 rows takes 0.36 us, of 36 KB for 160
// rows 0.9). All 256 CUs at that rate would take 12.8 TB/s, twice what the
// weights come from HBM at: a launch of few rows on every CU is bound by that
// stream, one that leaves CUs without a block, or whose rows make the x tile
// most of what is staged, by its CUs. Hence narrow tiles on every CU for few
// rows and wide ones for many.
#include "common.h"

namespace htn {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_ptr_t;

constexpr int kTk = 64;                   // k per staged step
constexpr int kMaxTm = 256;               // x rows per block, at most
constexpr int kCuLds = 160 * 1024;        // a CU's LDS
constexpr int kFinishThreads = 1024;      // of the finish with the norm
constexpr int kMaxNormCols = 8192;        // a row the finish with the norm holds in LDS

struct TileArgs {
  const bf16_t* x; long x_rs;
  const unsigned char* w;
  const float* scale;  // 8-bit weights: one per weight row
  const bf16_t* res; long res_rs;
  bf16_t* y; long y_rs;
  int M, N, K;        // N: output columns (gate columns for SwiGLU)
  int mtiles, ntiles; // output tiles along M and N
  int ksplit, steps;  // k splits per tile, 64-wide k steps per split
  int wide;           // y rows take 8-byte stores
  float* part;        // K-split partial sums [ksplit][M][part_rs]
  long part_rs;       // round4(N), twice that for SwiGLU (gate, then up sums)
  uint64_t* keys;     // argmax: [ntiles][M]
  // Residual epilogue fused with the next RMSNorm (K-split finish only).
  const bf16_t* ngain; float neps;
  bf16_t* normed;
};

// k steps between the starts of neighbouring weight tiles' ranges: weight rows
// a power of two apart (8 KB at K = 4096) put one k step's rows of every tile
// on a few memory channels while all blocks walk k together. A copy of this
// staging alone, 268 MB in 256 tiles: all from k = 0 4.4 TB/s, rotated 6.05,
// rotated and past the caches (one row tile) 6.7.
constexpr int kRotate = 37;
// Weights of this size or more are streamed past the caches by the tiles of at
// most 48 rows, bf16 ones of any size from kStreamRows rows on.
// From HBM streaming is faster: 4B int8, one tile, QKV of 15.7 MB 10.1 -> 9.3
// us, O of 10.5 MB 11.4 -> 10.6; 8B at 32 rows in two tiles, O 15.0 -> 14.5,
// down 35.7 -> 34.5. Smaller weights belong to small models, where the last-level
// cache still holds a part from the pass before: the more, the less the larger
// ones put there. Three 0.6B models' 125 MB in turn, rows: all cached / from
// 10 MB on (gate/up) / all streamed: 40 rows 152 / 146 / 153 us, 64 157 / 152 /
// 159, 128 170 / 161 / 174, 200 187 / 178 / 189; one model alone 140 / 147 / 155
// and 171 / 177 / 189. From 256 rows on gate/up goes through the library, whose
// loads fill the cache, and the rest is streamed: 256 rows 218 / 214 / 208, 300
// 240 / 239 / 231, 400 255 / 255 / 252 (alone 193 / 192 / 207 and 234 for each).
// 8-bit gate/up stays here: 256 rows 206 / 205 / 211, 300 229 / 228 / 233.
constexpr long kStreamBytes = 10L << 20, kStreamRows = 256;
constexpr int kMinSplitSteps = 8;     // k steps each split keeps at least
constexpr int kMaxSplit = 12;

// A tile's shape: waves along the rows (WM) and the weight rows (WN), 16-row x
// tiles per wave (NT), weight format.
template <int WM, int WN, int NT, int WF>
struct Shape {
  static constexpr int kTm = 16 * NT * WM;
  static constexpr int kWaves = WM * WN;
  static constexpr int kWt = 2 * WM;                       // 16-row weight tiles per wave
  static constexpr int kTn = 16 * kWt * WN;                // weight rows per block
  static constexpr int kXl = (kTm / 8 + kWaves - 1) / kWaves;  // staging loads per wave: x
  static constexpr int kWl = WF == WF_BF16 ? 4 : 2;        // and weights
  static constexpr int kWRow = WF == WF_BF16 ? 128 : 64;   // bytes of a staged weight row
  static constexpr int kXBytes = kTm * kTk * 2;
  static constexpr int kStage = kXBytes + kTn * kWRow;
  static constexpr int kBlocks = kWaves == 8 ? 1 : 2;      // resident per CU
  static constexpr int kFit = kCuLds / kBlocks / kStage;
  static constexpr int kStages = kFit < 2 ? 2 : (kFit > 8 ? 8 : kFit);
};

// Operand fragments are read by inline asm: the compiler would wait for every
// LDS-direct load in flight before an ordinary LDS read of such a buffer.
// Reads are issued without their wait; wait_frags waits and names every
// fragment as an operand, so no use of one moves above it.
template <int OFF>
__device__ __forceinline__ void issue_frag(uint32_t addr, u32x4& f) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(f) : "v"(addr), "n"(OFF) : "memory");
}

template <int N, int STRIDE, int I = 0>
__device__ __forceinline__ void issue_frags(uint32_t addr, u32x4* f) {
  if constexpr (I < N) {
    issue_frag<I * STRIDE>(addr, f[I]);
    issue_frags<N, STRIDE, I + 1>(addr, f);
  }
}

template <int N>
__device__ __forceinline__ void wait_frags(u32x4 (&f)[N]) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f[0]) : : "memory");
#pragma unroll
  for (int i = 1; i < N; ++i) asm volatile("" : "+v"(f[i]) : : "memory");
}

// Eight 8-bit codes (k ascending) as eight bf16 values, exactly.
template <int WF>
__device__ __forceinline__ u32x4 codes_to_bf16(uint32_t lo, uint32_t hi) {
  u32x4 o;
  const uint32_t d[2] = {lo, hi};
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if constexpr (WF == WF_INT8) {
      const int v = static_cast<int>(d[j]);
      o[2 * j] = pack_exact_bf2(static_cast<float>(static_cast<signed char>(v)),
                                static_cast<float>(static_cast<signed char>(v >> 8)));
      o[2 * j + 1] = pack_exact_bf2(static_cast<float>(static_cast<signed char>(v >> 16)),
                                    static_cast<float>(v >> 24));
    } else {
      o[2 * j] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(
                                                  static_cast<int>(d[j]), 1.0f, false));
      o[2 * j + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(
                                                      static_cast<int>(d[j]), 1.0f, true));
    }
  }
  return o;
}

__device__ __forceinline__ f32x4_t mfma(u32x4 w, u32x4 x, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w),
                                                 __builtin_bit_cast(bf16x8_t, x), c, 0, 0, 0);
}

// The fp32 dot products of output columns n .. n + 3 (weight rows row0 + n ..):
// 8-bit weights' row scales applied.
template <int WF>
__device__ __forceinline__ f32x4_t scaled(const TileArgs& a, f32x4_t v, int row0, int n) {
  if constexpr (WF != WF_BF16) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] *= n + e < a.N ? a.scale[row0 + n + e] : 0.f;
  }
  return v;
}

// Four output columns n .. n + 3 of row m (fewer at the right edge).
__device__ __forceinline__ void store4(const TileArgs& a, int m, int n, const float (&o)[4]) {
  bf16_t* dst = a.y + static_cast<long>(m) * a.y_rs + n;
  if (a.wide && n + 4 <= a.N) {
    *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf2(o[0], o[1]), pack_bf2(o[2], o[3]));
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < a.N) dst[e] = static_cast<bf16_t>(f2bf(o[e]));
  }
}

// The epilogue of four outputs: g holds the (gate) dot products, u the up ones.
template <int EPI, int WF>
__device__ __forceinline__ void finish4(const TileArgs& a, int m, int n, f32x4_t g, f32x4_t u) {
  g = scaled<WF>(a, g, 0, n);
  float o[4];
  if constexpr (EPI == HTN_EPI_SWIGLU) {
    u = scaled<WF>(a, u, a.N, n);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = silu_bf(round_bf(g[e])) * round_bf(u[e]);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] = g[e];
      if (EPI == HTN_EPI_RESIDUAL)
        o[e] = round_bf(o[e]) +
               (n + e < a.N ? bf2f(a.res[static_cast<long>(m) * a.res_rs + n + e]) : 0.f);
    }
  }
  store4(a, m, n, o);
}

// A uniform pointer kept in scalar registers: a descriptor in vector registers
// makes every load through it a per-lane descriptor loop.
__device__ __forceinline__ const unsigned char* uniform_ptr(const unsigned char* ptr) {
  const uint64_t p = reinterpret_cast<uint64_t>(ptr);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(p));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(p >> 32));
  return reinterpret_cast<const unsigned char*>((static_cast<uint64_t>(hi) << 32) | lo);
}

// One k step into ring slot `slot` (empty past the split's last step): eight x
// rows (1 KB) per load, weight rows eight (bf16) or sixteen (8-bit) per load.
template <int WM, int WN, int NT, int WF, int AUX>
__device__ __forceinline__ void stage_tiles(unsigned char* st, int ks, bool live, int wave,
                                            const bf16_t* xb, uint32_t xrange,
                                            const unsigned char* const (&wb)[2],
                                            const uint32_t (&wrange)[2],
                                            const uint32_t* xoff,
                                            const uint32_t (&woff)[2]) {
  using S = Shape<WM, WN, NT, WF>;
  const uint32_t kx = live ? static_cast<uint32_t>(ks) * kTk * 2u : 0u;
  const uint32_t kw = live ? static_cast<uint32_t>(ks) * S::kWRow : 0u;
  const __amdgpu_buffer_rsrc_t xrs = buffer_rsrc(xb, live ? xrange : 0u);
#pragma unroll
  for (int u = 0; u < S::kXl; ++u) {
    int li = wave + S::kWaves * u;  // where loads and waves do not divide, some repeat
    if ((S::kTm / 8) % S::kWaves != 0) li %= S::kTm / 8;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, (lds_ptr_t*)(st + li * 1024), 16, xoff[u], kx, 0, 0);
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {  // the wave's two 16-row groups of the weight tile
    const __amdgpu_buffer_rsrc_t wrs = buffer_rsrc(wb[h], live ? wrange[h] : 0u);
    unsigned char* dst = st + S::kXBytes + (2 * wave + h) * 16 * S::kWRow;
#pragma unroll
    for (int u = 0; u < S::kWl / 2; ++u)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (lds_ptr_t*)(dst + u * 1024), 16, woff[u], kw, 0, AUX);
  }
}

// AUX: the weight loads' cache policy (kStreamBytes).
template <int EPI, int WM, int WN, int NT, int WF, int AUX>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_tiles_kernel(TileArgs a) {
  using S = Shape<WM, WN, NT, WF>;
  constexpr bool SW = EPI == HTN_EPI_SWIGLU;
  constexpr int WT = S::kWt, TM = S::kTm;
  // Arguments in scalar registers at entry: one round of scalar loads.
  asm volatile("" ::"s"(a.x), "s"(a.x_rs), "s"(a.w), "s"(a.scale), "s"(a.res), "s"(a.res_rs),
               "s"(a.y), "s"(a.y_rs), "s"(a.M), "s"(a.N), "s"(a.K), "s"(a.mtiles), "s"(a.ntiles),
               "s"(a.ksplit), "s"(a.steps), "s"(a.part), "s"(a.part_rs));
  extern __shared__ __align__(16) unsigned char lds[];  // kStages x and weight tiles
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = WM == 2 ? wave & 1 : 0, wn = WM == 2 ? wave >> 1 : wave;
  const int col = lane & 15, quad = lane >> 4;
  // XCD-major layout: block L on XCD L % 8 takes weight tile
  // nt = (L / 8 / (mtiles ksplit)) * 8 + L % 8, row tile (L / 8) % mtiles and
  // k split (L / 8 / mtiles) % ksplit.
  const int L = blockIdx.x, j = L >> 3, per = a.mtiles * a.ksplit;
  const int g = j / per, q = j - g * per, s = q / a.mtiles;
  const int nt = g * 8 + (L & 7), mt = q - s * a.mtiles;
  if (nt >= a.ntiles) return;
  const int m0 = mt * TM;
  // Weight rows of the tile: kTn rows from n0, or for SwiGLU kTn / 2 output
  // columns from n0 as 16-row groups: gate, gate, up, up, ... with two waves
  // along the rows, else gate, up, ....
  const int n0 = nt * (SW ? S::kTn / 2 : S::kTn);

  // Staging: a lane of load li takes x row 8 li + lane / 8 and writes position
  // lane % 8 of it, loading source chunk (lane % 8) ^ (row & 7); weights the
  // same, or for 8-bit rows 16 rows per load, row lane / 4, chunk
  // (lane % 4) ^ ((row >> 2) & 3). Operands go through descriptors whose range
  // ends at the last real row, so rows past M or the weight's end read zeros.
  const long mrows = a.M - m0 < TM ? a.M - m0 : TM;
  const bf16_t* xb = a.x + static_cast<long>(m0) * a.x_rs;
  const uint32_t xrange = static_cast<uint32_t>(((mrows - 1) * a.x_rs + a.K) * 2);
  const long wrow_bytes = static_cast<long>(a.K) * (WF == WF_BF16 ? 2 : 1);
  const unsigned char* wb[2];
  uint32_t wrange[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int gi = 2 * wave + h;
    int first = n0 + 16 * gi, base = first;  // output column, weight row
    if (SW) {
      first = WM == 2 ? n0 + 32 * (gi >> 2) + 16 * (gi & 1) : n0 + 16 * (gi >> 1);
      base = first + ((WM == 2 ? (gi & 2) : (gi & 1)) ? a.N : 0);
    }
    const int rows = a.N - first < 16 ? (a.N - first > 0 ? a.N - first : 0) : 16;
    wb[h] = uniform_ptr(a.w + (rows > 0 ? base : 0) * wrow_bytes);
    wrange[h] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(rows * wrow_bytes));
  }
  uint32_t xoff[S::kXl], woff[2];
#pragma unroll
  for (int u = 0; u < S::kXl; ++u) {
    int li = wave + S::kWaves * u;
    if ((TM / 8) % S::kWaves != 0) li %= TM / 8;
    const int r = 8 * li + (lane >> 3);
    xoff[u] = static_cast<uint32_t>(r) * static_cast<uint32_t>(a.x_rs) * 2u +
              (((lane & 7) ^ (r & 7)) * 16);
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int r = WF == WF_BF16 ? 8 * u + (lane >> 3) : (lane >> 2);
    woff[u] = static_cast<uint32_t>(r) * static_cast<uint32_t>(wrow_bytes) +
              (WF == WF_BF16 ? ((lane & 7) ^ (r & 7)) * 16 : ((lane & 3) ^ ((r >> 2) & 3)) * 16);
  }

  // Fragment addresses in ring slot 0, per k half: x and bf16 weights, chunk
  // 4 h + quad (8-bit: 2 quad + h) of row 16 t + col; 8-bit weights, chunk
  // quad, both halves in one read. Row tiles are 2048 (1024) bytes apart.
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr_t*)lds));
  uint32_t xa[2], wa[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int c = WF == WF_BF16 ? 4 * h + quad : 2 * quad + h;
    xa[h] = lds0 + static_cast<uint32_t>((16 * NT * wm + col) * 128 + ((c ^ (col & 7)) * 16));
    wa[h] = lds0 + S::kXBytes +
            static_cast<uint32_t>(WF == WF_BF16
                                      ? (16 * WT * wn + col) * 128 + ((c ^ (col & 7)) * 16)
                                      : (16 * WT * wn + col) * 64 + ((quad ^ ((col >> 2) & 3)) * 16));
  }

  f32x4_t acc[WT][NT];  // [weight tile][x tile]: D^T rows = weight rows, columns = x rows
#pragma unroll
  for (int i = 0; i < WT; ++i)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int nk = a.K / kTk;
  const int k0 = s * a.steps, k1 = nk < k0 + a.steps ? nk : k0 + a.steps;
  int left = k1 - k0;                  // steps still to stage
  int kn = k0 + (nt * kRotate) % left;  // the next one
  auto stage_next = [&](int slot) {
    stage_tiles<WM, WN, NT, WF, AUX>(lds + slot * S::kStage, kn, left > 0, wave, xb, xrange, wb,
                                       wrange, xoff, woff);
    kn = kn + 1 == k1 ? k0 : kn + 1;
    --left;
  };
#pragma unroll
  for (int u = 0; u < S::kStages - 1; ++u) stage_next(u);
  int rd = 0, wr = S::kStages - 1;
  for (int ks = k0; ks < k1; ++ks) {
    // This wave's part of step ks has landed (the later steps' loads may still
    // be in flight); after the barrier everyone's has, and every wave has
    // finished step ks - 1, whose slot the next load takes.
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S::kStages - 2) * (S::kXl + S::kWl)) : "memory");
    asm volatile("s_barrier" ::: "memory");
    stage_next(wr);
    const uint32_t so = static_cast<uint32_t>(rd * S::kStage);
    rd = rd + 1 == S::kStages ? 0 : rd + 1;
    wr = wr + 1 == S::kStages ? 0 : wr + 1;
    if constexpr (WF == WF_BF16) {
      u32x4 f0[WT + NT], f1[WT + NT];
      issue_frags<WT, 2048>(wa[0] + so, f0);
      issue_frags<NT, 2048>(xa[0] + so, f0 + WT);
      wait_frags(f0);
      issue_frags<WT, 2048>(wa[1] + so, f1);
      issue_frags<NT, 2048>(xa[1] + so, f1 + WT);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = mfma(f0[i], f0[WT + t], acc[i][t]);
      __builtin_amdgcn_sched_barrier(0);
      wait_frags(f1);
#pragma unroll
      for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = mfma(f1[i], f1[WT + t], acc[i][t]);
    } else {
      u32x4 f0[WT + NT], f1[NT];  // codes of both halves and x of the first; x of the second
      issue_frags<WT, 1024>(wa[0] + so, f0);
      issue_frags<NT, 2048>(xa[0] + so, f0 + WT);
      wait_frags(f0);
      issue_frags<NT, 2048>(xa[1] + so, f1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < WT; ++i) {
        const u32x4 w = codes_to_bf16<WF>(f0[i][0], f0[i][1]);
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = mfma(w, f0[WT + t], acc[i][t]);
      }
      __builtin_amdgcn_sched_barrier(0);
      wait_frags(f1);
#pragma unroll
      for (int i = 0; i < WT; ++i) {
        const u32x4 w = codes_to_bf16<WF>(f0[i][2], f0[i][3]);
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = mfma(w, f1[t], acc[i][t]);
      }
    }
  }
  // Every staging load has landed before the block's LDS is reused or released.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // Lane (col, quad) holds, per weight tile i and x tile t, row mb + 16 t + col
  // and weight rows 16 (WT wn + i) + 4 quad + (0..3) of the tile; for SwiGLU
  // the first half of a wave's weight tiles are gate, the second up rows.
  const int mb = m0 + 16 * NT * wm;
  constexpr int OT = SW ? WT / 2 : WT;  // 16-column output tiles per wave
  const int nb = n0 + 16 * OT * wn + 4 * quad;
  if constexpr (EPI == HTN_EPI_ARGMAX) {
    // The best (bf16 logit, lowest id) key of the tile's columns per row: over
    // the lane's columns, the four quads, then the waves.
    uint64_t* best = reinterpret_cast<uint64_t*>(lds);  // [4 waves][NT * 16]
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      uint64_t key = 0;
#pragma unroll
      for (int i = 0; i < WT; ++i) {
        const f32x4_t v = scaled<WF>(a, acc[i][t], 0, nb + 16 * i);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int n = nb + 16 * i + e;
          const uint64_t k = n < a.N ? argmax_key(f2bf(v[e]), static_cast<uint32_t>(n)) : 0ull;
          key = k > key ? k : key;
        }
      }
#pragma unroll
      for (int d = 16; d <= 32; d += d) {
        const uint64_t o = __shfl_xor(key, d, kWave);
        key = o > key ? o : key;
      }
      if (quad == 0) best[wave * (NT * 16) + 16 * t + col] = key;
    }
    __syncthreads();
    for (int r = tid; r < TM; r += 64 * S::kWaves) {
      const int w0 = WM == 2 ? r / (16 * NT) : 0, rr = r - w0 * 16 * NT;
      uint64_t key = 0;
      for (int w = w0; w < 4; w += WM) {
        const uint64_t k = best[w * (NT * 16) + rr];
        key = k > key ? k : key;
      }
      if (m0 + r < a.M) a.keys[static_cast<long>(nt) * a.M + m0 + r] = key;
    }
    return;
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int m = mb + 16 * t + col;
    if (m >= a.M) continue;
    // K-split partials, unrounded and unscaled, at part[(s M + m) part_rs + c],
    // c = the output column, or for SwiGLU c = n for the gate sums and
    // part_rs / 2 + n for the up sums. The four columns of a lane end before
    // round4(N), so every store is whole.
    float* row = a.part + (static_cast<long>(s) * a.M + m) * a.part_rs;
#pragma unroll
    for (int i = 0; i < OT; ++i) {
      const int n = nb + 16 * i;
      if (n >= a.N) continue;
      const f32x4_t u = SW ? acc[SW ? i + OT : i][t] : f32x4_t{};
      if (a.ksplit > 1) {
        *reinterpret_cast<f32x4_t*>(row + n) = acc[i][t];
        if (SW) *reinterpret_cast<f32x4_t*>(row + a.part_rs / 2 + n) = u;
      } else {
        finish4<EPI, WF>(a, m, n, acc[i][t], u);
      }
    }
  }
}

// The k splits' partial sums of columns n .. n + 3 of row m, in split order.
__device__ __forceinline__ f32x4_t sum_parts(const TileArgs& a, long m, long n) {
  const long stride = static_cast<long>(a.M) * a.part_rs;
  const float* p = a.part + m * a.part_rs + n;
  f32x4_t v = *reinterpret_cast<const f32x4_t*>(p);
#pragma unroll 4
  for (int s = 1; s < a.ksplit; ++s) v += *reinterpret_cast<const f32x4_t*>(p + s * stride);
  return v;
}

// K-split sum + epilogue: thread i takes output columns 4 (i % n4) .. + 3 of
// row i / n4, n4 = round4(N) / 4.
template <int EPI, int WF>
__global__ __launch_bounds__(256) void gemm_tiles_finish(TileArgs a) {
  asm volatile("" ::"s"(a.res), "s"(a.res_rs), "s"(a.y), "s"(a.y_rs), "s"(a.M), "s"(a.N),
               "s"(a.ksplit), "s"(a.part), "s"(a.part_rs));
  constexpr bool SW = EPI == HTN_EPI_SWIGLU;
  const long n4 = (SW ? a.part_rs / 2 : a.part_rs) / 4;
  const long i = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
  const long m = i / n4;
  if (m >= a.M) return;
  const int n = static_cast<int>(i - m * n4) * 4;
  const f32x4_t g = sum_parts(a, m, n);
  const f32x4_t u = SW ? sum_parts(a, m, a.part_rs / 2 + n) : f32x4_t{};
  finish4<EPI, WF>(a, static_cast<int>(m), n, g, u);
}

// K-split finish of the residual epilogue with the next RMSNorm, one block of
// sixteen waves per row: y = bf16(bf16(sum) + residual) to memory and LDS, then
// wave 0 forms the sum of squares in the row-wise RMSNorm's order (lane l over
// vectors l, l + 64, ..., element by element, one wave reduction), so `normed`
// is bit-identical to running that norm on y. A thread takes four columns and
// has all its splits' loads in flight: few rows are few blocks, and the chain
// of loads, not the bytes, is their time (8B at 16 rows, against 256 threads of eight columns that
// load split by split: O 15.1 -> 13.2 us with its finish, down 29.9 -> 25.8).
template <int WF>
__global__ __launch_bounds__(kFinishThreads) void gemm_tiles_finish_norm(TileArgs a) {
  asm volatile("" ::"s"(a.res), "s"(a.res_rs), "s"(a.y), "s"(a.y_rs), "s"(a.M), "s"(a.N),
               "s"(a.ksplit), "s"(a.part), "s"(a.part_rs), "s"(a.ngain), "s"(a.neps),
               "s"(a.normed));
  __shared__ uint2 ys[kMaxNormCols / 4];
  __shared__ float inv_s;
  const int tid = threadIdx.x, m = blockIdx.x, nv = a.N >> 2;
  const long stride = static_cast<long>(a.M) * a.part_rs;
  for (int v = tid; v < nv; v += kFinishThreads) {
    const float* p = a.part + m * a.part_rs + 4 * v;
    f32x4_t part[kMaxSplit];
#pragma unroll
    for (int s = 0; s < kMaxSplit; ++s)
      if (s < a.ksplit) part[s] = *reinterpret_cast<const f32x4_t*>(p + s * stride);
    const uint2 r = *reinterpret_cast<const uint2*>(a.res + m * a.res_rs + v * 4);
    f32x4_t t = part[0];
#pragma unroll
    for (int s = 1; s < kMaxSplit; ++s)
      if (s < a.ksplit) t += part[s];
    t = scaled<WF>(a, t, 0, 4 * v);
    const uint2 yv = make_uint2(pack_bf2(round_bf(t[0]) + bf_lo(r.x), round_bf(t[1]) + bf_hi(r.x)),
                                pack_bf2(round_bf(t[2]) + bf_lo(r.y), round_bf(t[3]) + bf_hi(r.y)));
    *reinterpret_cast<uint2*>(a.y + m * a.y_rs + v * 4) = yv;
    ys[v] = yv;
  }
  __syncthreads();
  if (tid < kWave) {
    float ss = 0.f;
    for (int v = tid; v < a.N >> 3; v += kWave) {
      float f[8];
      const uint2 lo = ys[2 * v], hi = ys[2 * v + 1];
      unpack8(make_uint4(lo.x, lo.y, hi.x, hi.y), f);
#pragma unroll
      for (int i = 0; i < 8; ++i) ss = fmaf(f[i], f[i], ss);
    }
    const float inv = 1.0f / sqrtf(wave_sum(ss) / static_cast<float>(a.N) + a.neps);
    if (tid == 0) inv_s = inv;
  }
  __syncthreads();
  const float inv = inv_s;
  for (int v = tid; v < nv; v += kFinishThreads) {
    const uint2 x = ys[v], g = *reinterpret_cast<const uint2*>(a.ngain + v * 4);
    *reinterpret_cast<uint2*>(a.normed + static_cast<long>(m) * a.N + v * 4) =
        make_uint2(pack_bf2(bf_lo(g.x) * round_bf(bf_lo(x.x) * inv), bf_hi(g.x) * round_bf(bf_hi(x.x) * inv)),
                   pack_bf2(bf_lo(g.y) * round_bf(bf_lo(x.y) * inv), bf_hi(g.y) * round_bf(bf_hi(x.y) * inv)));
  }
}

// Per-row argmax over the weight tiles' keys.
__global__ __launch_bounds__(256) void gemm_tiles_argmax(const uint64_t* __restrict__ keys,
                                                         int tiles, int M, int64_t* tokens) {
  __shared__ uint64_t wbest[4];
  const int m = blockIdx.x;
  uint64_t b = 0;
  for (int i = threadIdx.x; i < tiles; i += 256) {
    const uint64_t k = keys[static_cast<long>(i) * M + m];
    b = k > b ? k : b;
  }
  b = wave_max_u64(b);
  if ((threadIdx.x & 63) == 0) wbest[threadIdx.x >> 6] = b;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t r = wbest[0];
    for (int i = 1; i < 4; ++i) r = wbest[i] > r ? wbest[i] : r;
    tokens[m] = static_cast<int64_t>(argmax_key_index(r));
  }
}

// Launch shape: the row tile, and the k split.
struct TilePlan {
  int wm, wn, nt;     // waves along the rows and the weight rows, 16-row tiles per wave
  int ksplit, steps;
  long blocks, ntiles, part_rs, keys_bytes;
};

// The tiles and what one k step of a block on them takes, in us, alone on its
// CU (step[0]) and beside a second block (step[1]; eight waves stand alone):
// bf16, then 8-bit weights. Measured over the QKV, O, gate/up and down
// projections of the 0.6B, 4B and 8B shapes at 5 to 1000 rows, every tile with
// 1 to 12 k splits (1200 launches, weights from HBM), as the coefficients that
// fit those times best; the plan below then picks launches 1% slower than the
// fastest of each sweep on average, 16% at most.
struct TileShape { int wm, wn, nt; float step[2][2]; };
constexpr TileShape kShapes[] = {
    {1, 4, 1, {{.36f, .72f}, {.32f, .68f}}}, {1, 4, 2, {{.38f, .84f}, {.35f, .78f}}},
    {1, 4, 3, {{.45f, .94f}, {.41f, .89f}}}, {2, 2, 2, {{.47f, .81f}, {.47f, .73f}}},
    {2, 2, 3, {{.80f, .93f}, {.59f, .83f}}}, {2, 2, 4, {{.85f, 1.08f}, {.69f, .97f}}},
    {2, 2, 5, {{.89f, 1.16f}, {.84f, 1.08f}}}, {2, 4, 4, {{.96f, .96f}, {1.06f, 1.06f}}},
    {2, 4, 5, {{1.11f, 1.11f}, {1.20f, 1.20f}}}, {2, 4, 7, {{1.50f, 1.50f}, {1.52f, 1.52f}}},
    {2, 4, 8, {{1.54f, 1.54f}, {1.68f, 1.68f}}}};

// 8-bit weights are never best on the eight-wave tiles of 128 and 160 rows: two
// four-wave blocks on a CU do the same rows by 256 weight rows in less (0.97
// and 1.08 us a step against 1.06 and 1.20).
constexpr bool built_w8(int wm, int wn, int nt) { return wm * wn < 8 || nt > 5; }

// A launch's time by those coefficients: per XCD, `blocks` blocks of `steps`
// k steps in rounds of two per CU (one, for eight waves), no less than the
// weights take from HBM, the launch itself, and for a k split its finish: a
// launch, the partial sums' bytes, and for the finish with a norm (a block per
// row) its chain over the splits.
float tile_cost(const TileShape& sh, long blocks, long steps, long ks, double part_mb,
                double weight_mb, bool residual, int format) {
  const long cus = device_cus() / 8 > 0 ? device_cus() / 8 : 1;
  const long per = cus * (sh.wm * sh.wn == 8 ? 1 : 2);
  const float* step = sh.step[format != 0];
  const long rest = blocks % per;
  float t = blocks / per * step[1];
  if (rest > 0) t += rest <= cus ? step[0] : step[1];
  t *= steps;
  const float stream = static_cast<float>(weight_mb) / 6.f;  // the weights at 6 TB/s
  t = (t > stream ? t : stream) + 3.3f;
  if (ks > 1) t += 2.6f + .43f * static_cast<float>(part_mb) + (residual ? .3f * ks : 0.f);
  else if (residual) t += 6.4f;  // the norm's own launch
  return t;
}

TilePlan plan_tiles(long rows, long n, long k, int epilogue, int format) {
  const bool sw = epilogue == HTN_EPI_SWIGLU, argmax = epilogue == HTN_EPI_ARGMAX;
  const long nk = k / kTk;
  // bf16 prompts whose 128 x 128 tiles alone give every CU its two blocks keep
  // whole k ranges: their callers need no scratch.
  const bool full = format == 0 && ((rows + 127) / 128) * ((n * (sw ? 2 : 1) + 127) / 128) >=
                                       2L * device_cus();
  TilePlan p{};
  p.part_rs = (sw ? 2 : 1) * ((n + 3) / 4 * 4);
  float best = 0.f;
  for (const TileShape& sh : kShapes) {
    if (argmax && (sh.wm != 1 || sh.nt > 2)) continue;
    if (format != 0 && !built_w8(sh.wm, sh.wn, sh.nt)) continue;
    const long tm = 16L * sh.nt * sh.wm, tn = 32L * sh.wm * sh.wn / (sw ? 2 : 1);
    const long ntiles = (n + tn - 1) / tn;
    const long per_xcd = (ntiles + 7) / 8 * ((rows + tm - 1) / tm);
    for (long ks = 1; ks <= kMaxSplit; ++ks) {
      if (ks > 1 && (argmax || full || nk / ks < kMinSplitSteps)) break;
      const long steps = (nk + ks - 1) / ks;
      if ((nk + steps - 1) / steps != ks) continue;  // a split would be empty
      const float cost = tile_cost(sh, per_xcd * ks, steps, ks, ks * rows * p.part_rs * 4e-6,
                                   p.part_rs * k * (format ? 1e-6 : 2e-6),
                                   epilogue == HTN_EPI_RESIDUAL, format);
      if (p.ksplit == 0 || cost < best) {
        best = cost;
        p.wm = sh.wm; p.wn = sh.wn; p.nt = sh.nt;
        p.ntiles = ntiles;
        p.ksplit = static_cast<int>(ks);
        p.steps = static_cast<int>(steps);
        p.blocks = 8 * per_xcd * ks;
      }
    }
  }
  p.keys_bytes = argmax ? p.ntiles * rows * 8 : 0;
  return p;
}

long tiles_scratch_bytes(const TilePlan& p, long rows) {
  return p.ksplit > 1 ? static_cast<long>(p.ksplit) * rows * p.part_rs * 4 : p.keys_bytes;
}

// Whether tiles of one wave along the rows load a [n, k] weight (twice n rows
// for SwiGLU) past the caches.
bool streamed(long rows, long n, long k, int epilogue, int format) {
  const long bytes = (epilogue == HTN_EPI_SWIGLU ? 2 : 1) * n * k * (format == 0 ? 2 : 1);
  return bytes >= kStreamBytes || (format == 0 && rows >= kStreamRows);
}

template <int EPI, int WM, int WN, int NT, int WF, int AUX>
int launch_policy(const TileArgs& a, long blocks, hipStream_t st) {
  using S = Shape<WM, WN, NT, WF>;
  constexpr int bytes = S::kStages * S::kStage;
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&gemm_tiles_kernel<EPI, WM, WN, NT, WF, AUX>),
      hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  (void)attr;  // a refused size surfaces as a launch error
  hipLaunchKernelGGL((gemm_tiles_kernel<EPI, WM, WN, NT, WF, AUX>),
                     dim3(static_cast<unsigned>(blocks)), dim3(64 * S::kWaves), bytes, st, a);
  return launch_status();
}

template <int EPI, int WM, int WN, int NT, int WF>
int launch_shape(TileArgs& a, long blocks, hipStream_t st) {
  constexpr int TM = Shape<WM, WN, NT, WF>::kTm;
  a.mtiles = (a.M + TM - 1) / TM;
  if constexpr (WM == 1) {
    if (streamed(a.M, a.N, a.K, EPI, WF))
      return launch_policy<EPI, WM, WN, NT, WF, 2>(a, blocks, st);
  }
  return launch_policy<EPI, WM, WN, NT, WF, 0>(a, blocks, st);
}

template <int EPI, int WF>
int launch_tiles(TileArgs& a, const TilePlan& p, hipStream_t st) {
  if constexpr (EPI == HTN_EPI_ARGMAX) {
    return p.nt == 1 ? launch_shape<EPI, 1, 4, 1, WF>(a, p.blocks, st)
                     : launch_shape<EPI, 1, 4, 2, WF>(a, p.blocks, st);
  } else {
    switch (100 * p.wm + 10 * p.wn + p.nt) {
      case 141: return launch_shape<EPI, 1, 4, 1, WF>(a, p.blocks, st);
      case 142: return launch_shape<EPI, 1, 4, 2, WF>(a, p.blocks, st);
      case 143: return launch_shape<EPI, 1, 4, 3, WF>(a, p.blocks, st);
      case 222: return launch_shape<EPI, 2, 2, 2, WF>(a, p.blocks, st);
      case 223: return launch_shape<EPI, 2, 2, 3, WF>(a, p.blocks, st);
      case 224: return launch_shape<EPI, 2, 2, 4, WF>(a, p.blocks, st);
      case 225: return launch_shape<EPI, 2, 2, 5, WF>(a, p.blocks, st);
      case 247: return launch_shape<EPI, 2, 4, 7, WF>(a, p.blocks, st);
      case 248: return launch_shape<EPI, 2, 4, 8, WF>(a, p.blocks, st);
      default: break;
    }
    if constexpr (WF == WF_BF16)
      return p.nt == 4 ? launch_shape<EPI, 2, 4, 4, WF>(a, p.blocks, st)
                       : launch_shape<EPI, 2, 4, 5, WF>(a, p.blocks, st);
    return HTN_EUNSUPPORTED;  // the plan picks no other shape
  }
}

template <int EPI, int WF>
int finish_tiles(TileArgs& a, hipStream_t st) {
  const long groups = static_cast<long>(a.M) * ((a.N + 3) / 4);
  hipLaunchKernelGGL((gemm_tiles_finish<EPI, WF>), dim3(static_cast<unsigned>((groups + 255) / 256)),
                     dim3(256), 0, st, a);
  return launch_status();
}

template <int WF>
int run_tiles(TileArgs& a, const TilePlan& p, int epilogue, int64_t* tokens, hipStream_t st) {
  int rc;
  switch (epilogue) {
    case HTN_EPI_STORE: rc = launch_tiles<HTN_EPI_STORE, WF>(a, p, st); break;
    case HTN_EPI_RESIDUAL: rc = launch_tiles<HTN_EPI_RESIDUAL, WF>(a, p, st); break;
    case HTN_EPI_SWIGLU: rc = launch_tiles<HTN_EPI_SWIGLU, WF>(a, p, st); break;
    default: rc = launch_tiles<HTN_EPI_ARGMAX, WF>(a, p, st); break;
  }
  if (rc != HTN_OK) return rc;
  if (epilogue == HTN_EPI_ARGMAX) {
    hipLaunchKernelGGL(gemm_tiles_argmax, dim3(a.M), dim3(256), 0, st, a.keys, a.ntiles, a.M, tokens);
    return launch_status();
  }
  if (a.ksplit == 1) return HTN_OK;
  if (a.normed) {
    hipLaunchKernelGGL((gemm_tiles_finish_norm<WF>), dim3(a.M), dim3(kFinishThreads), 0, st, a);
    return launch_status();
  }
  switch (epilogue) {
    case HTN_EPI_STORE: return finish_tiles<HTN_EPI_STORE, WF>(a, st);
    case HTN_EPI_RESIDUAL: return finish_tiles<HTN_EPI_RESIDUAL, WF>(a, st);
    default: return finish_tiles<HTN_EPI_SWIGLU, WF>(a, st);
  }
}

bool known_epilogue(int e, int format) {
  return e == HTN_EPI_STORE || e == HTN_EPI_RESIDUAL || e == HTN_EPI_SWIGLU ||
         (e == HTN_EPI_ARGMAX && format != 0);
}

int tiles(const void* x, int64_t x_stride, const void* w, const float* scale, int format, int64_t n,
          int64_t k, int64_t rows, int epilogue, const void* residual, int64_t res_stride, void* y,
          int64_t y_stride, const void* gain, float eps, void* normed, int64_t* tokens,
          void* scratch, hipStream_t st) {
  if (!x || !w || rows <= 0 || n <= 0 || k <= 0) return HTN_EINVAL;
  if (format < 0 || format > HTN_WEIGHT_FP8_E4M3 || (format != 0 && !scale)) return HTN_EINVAL;
  if (!known_epilogue(epilogue, format)) return HTN_EINVAL;
  const bool argmax = epilogue == HTN_EPI_ARGMAX;
  if (argmax ? !tokens : !y) return HTN_EINVAL;
  if (epilogue == HTN_EPI_RESIDUAL && (!residual || res_stride < n)) return HTN_EINVAL;
  if ((!argmax && y_stride < n) || x_stride < k) return HTN_EINVAL;  // rows must not overlap
  // 64-wide k steps of 16-byte chunks; 32-bit offsets.
  if (k % kTk || k > (1L << 20) || x_stride % 8 || !aligned16(x) || !aligned16(w))
    return HTN_EUNSUPPORTED;
  const long wrows = epilogue == HTN_EPI_SWIGLU ? 2 * n : n;
  if (static_cast<long>(kMaxTm) * x_stride * 2 >= (1L << 32) || wrows >= (1L << 31) ||
      rows >= (1L << 31) || (argmax && rows > HTN_GEMM_TILES_ARGMAX_ROWS))
    return HTN_EUNSUPPORTED;
  if (!aligned16(scratch)) return HTN_EUNSUPPORTED;
  TilePlan p = plan_tiles(rows, n, k, epilogue, format);
  if (!scratch) {  // no scratch: every tile sums its whole k range
    if (argmax) return HTN_EINVAL;
    p.blocks /= p.ksplit;
    p.ksplit = 1;
    p.steps = static_cast<int>(k / kTk);
  }
  TileArgs a{};
  a.x = static_cast<const bf16_t*>(x); a.x_rs = x_stride;
  a.w = static_cast<const unsigned char*>(w);
  a.scale = scale;
  a.res = static_cast<const bf16_t*>(residual); a.res_rs = res_stride;
  a.y = static_cast<bf16_t*>(y); a.y_rs = y_stride;
  a.M = static_cast<int>(rows); a.N = static_cast<int>(n); a.K = static_cast<int>(k);
  a.ntiles = static_cast<int>(p.ntiles);
  a.ksplit = p.ksplit;
  a.steps = p.steps;
  a.wide = y_stride % 4 == 0 && aligned8(y);
  a.part = static_cast<float*>(scratch);
  a.part_rs = p.part_rs;
  a.keys = static_cast<uint64_t*>(scratch);
  // The finish with the norm holds a row of y in LDS as 8-element vectors.
  const bool fused = gain && p.ksplit > 1 && n % 8 == 0 && n <= kMaxNormCols &&
                     res_stride % 8 == 0 && y_stride % 8 == 0 && aligned16(residual) &&
                     aligned16(y) && aligned16(gain) && aligned16(normed);
  if (fused) {
    a.ngain = static_cast<const bf16_t*>(gain);
    a.neps = eps;
    a.normed = static_cast<bf16_t*>(normed);
  }
  const int rc = format == 0              ? run_tiles<WF_BF16>(a, p, epilogue, tokens, st)
                 : format == HTN_WEIGHT_INT8 ? run_tiles<WF_INT8>(a, p, epilogue, tokens, st)
                                             : run_tiles<WF_FP8>(a, p, epilogue, tokens, st);
  if (rc != HTN_OK || !gain || fused) return rc;
  return htn_rms_norm(y, y_stride, gain, normed, rows, n, eps, st);
}

}  // namespace
}  // namespace htn

using namespace htn;

extern "C" int64_t htn_gemm_tiles_scratch_bytes(int64_t rows, int64_t n, int64_t k,
                                                int epilogue) {
  return htn_gemm_tiles_w8_scratch_bytes(rows, n, k, epilogue, 0);
}

extern "C" int64_t htn_gemm_tiles_w8_scratch_bytes(int64_t rows, int64_t n, int64_t k, int epilogue,
                                                   int format) {
  if (rows <= 0 || n <= 0 || k <= 0 || k % kTk || format < 0 || format > HTN_WEIGHT_FP8_E4M3 ||
      !known_epilogue(epilogue, format))
    return 0;
  return tiles_scratch_bytes(plan_tiles(rows, n, k, epilogue, format), rows);
}

extern "C" int htn_gemm_tiles_plan(int64_t rows, int64_t n, int64_t k, int epilogue,
                                   int weight_format, int32_t* plan) {
  if (!plan || rows <= 0 || n <= 0 || k <= 0 || k % kTk || weight_format < 0 ||
      weight_format > HTN_WEIGHT_FP8_E4M3 || !known_epilogue(epilogue, weight_format))
    return HTN_EINVAL;
  const TilePlan p = plan_tiles(rows, n, k, epilogue, weight_format);
  const long tm = 16L * p.nt * p.wm;
  plan[0] = static_cast<int32_t>(tm);
  plan[1] = 32 * p.wm * p.wn;
  plan[2] = p.ksplit;
  plan[3] = p.wm == 1 && streamed(rows, n, k, epilogue, weight_format);
  return HTN_OK;
}

extern "C" int htn_gemm_tiles(const void* x, int64_t x_stride, const void* w, int64_t n,
                              int64_t k, int64_t rows, int epilogue, const void* residual,
                              int64_t res_stride, void* y, int64_t y_stride, void* scratch,
                              htn_stream_t stream) {
  if (epilogue == HTN_EPI_ARGMAX) return HTN_EINVAL;
  if (y_stride % 4 || !aligned8(y)) return y && y_stride >= n ? HTN_EUNSUPPORTED : HTN_EINVAL;
  return tiles(x, x_stride, w, nullptr, 0, n, k, rows, epilogue, residual, res_stride, y, y_stride,
               nullptr, 0.f, nullptr, nullptr, scratch, static_cast<hipStream_t>(stream));
}

extern "C" int htn_gemm_tiles_w8(const void* x, int64_t x_stride, const void* w,
                                 const float* w_scale, int weight_format, int64_t n, int64_t k,
                                 int64_t rows, int epilogue, const void* residual,
                                 int64_t res_stride, void* y, int64_t y_stride, int64_t* tokens,
                                 void* scratch, htn_stream_t stream) {
  if (weight_format != HTN_WEIGHT_INT8 && weight_format != HTN_WEIGHT_FP8_E4M3) return HTN_EINVAL;
  return tiles(x, x_stride, w, w_scale, weight_format, n, k, rows, epilogue, residual, res_stride,
               y, y_stride, nullptr, 0.f, nullptr, tokens, scratch,
               static_cast<hipStream_t>(stream));
}

extern "C" int htn_gemm_tiles_residual_norm(const void* x, int64_t x_stride, const void* w,
                                            const float* w_scale, int weight_format, int64_t n,
                                            int64_t k, int64_t rows, const void* residual,
                                            int64_t res_stride, void* y, int64_t y_stride,
                                            const void* gain, float eps, void* normed,
                                            void* scratch, htn_stream_t stream) {
  if (!gain || !normed) return HTN_EINVAL;
  return tiles(x, x_stride, w, w_scale, weight_format, n, k, rows, HTN_EPI_RESIDUAL, residual,
               res_stride, y, y_stride, gain, eps, normed, nullptr, scratch,
               static_cast<hipStream_t>(stream));
}
