// Prefill attention for gfx950 (head_dim 128): causal attention over many
// queries per sequence, on the matrix cores.
//
// These kernels are a code object of their own. The decode kernels of
// attention.hip run between streams of weights and cache that leave little
// else in the caches, and where their code lies costs time: with the
// long-prompt kernels in their object (the same instructions elsewhere) a
// 4B fp8 decode slice at 30 K slots took 268.2 us in place of 265.9.
#include "attention.h"

#include <type_traits>

namespace htn {

// The kernel arguments read before the first vector load, named as scalar
// operands at entry: one round of scalar loads.
__device__ __forceinline__ void preload_prefill(const PrefillArgs& a) {
  asm volatile("" ::"s"(a.Hkv), "s"(a.B), "s"(a.G), "s"(a.cap), "s"(a.keys), "s"(a.values),
               "s"(a.pos), "s"(a.q), "s"(a.q_sb), "s"(a.q_sh), "s"(a.q_st), "s"(a.Q));
}

// Operand reads of the prefill kernel's staged tiles (LDS-direct data, read
// by inline asm: the compiler would wait for every load in flight before an
// ordinary LDS read of such a buffer), issued without their waits: issue, run
// other work, then a wait that names the registers as operands so no use of
// them moves above it. K: one 32-dim step for the four 16-slot M-tiles of a
// 64-slot tile; V^T: transpose reads as attention.hip's read_vt_tr.
template <int OFF>
__device__ __forceinline__ void issue_k_pf(uint32_t addr, u32x4 (&k)[4]) {
  asm volatile(
      "ds_read_b128 %0, %4 offset:%5\n\t"
      "ds_read_b128 %1, %4 offset:%6\n\t"
      "ds_read_b128 %2, %4 offset:%7\n\t"
      "ds_read_b128 %3, %4 offset:%8"
      : "=&v"(k[0]), "=&v"(k[1]), "=&v"(k[2]), "=&v"(k[3])
      : "v"(addr), "n"(OFF), "n"(OFF + 4096), "n"(OFF + 8192), "n"(OFF + 12288)
      : "memory");
}

typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));

template <int OFF>
__device__ __forceinline__ void issue_vt_tr(const uint32_t (&va)[8], u32x2_t (&w)[8]) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8 offset:%16\n\t"
      "ds_read_b64_tr_b16 %1, %9 offset:%16\n\t"
      "ds_read_b64_tr_b16 %2, %10 offset:%16\n\t"
      "ds_read_b64_tr_b16 %3, %11 offset:%16\n\t"
      "ds_read_b64_tr_b16 %4, %12 offset:%16\n\t"
      "ds_read_b64_tr_b16 %5, %13 offset:%16\n\t"
      "ds_read_b64_tr_b16 %6, %14 offset:%16\n\t"
      "ds_read_b64_tr_b16 %7, %15 offset:%16"
      : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]), "=&v"(w[4]), "=&v"(w[5]),
        "=&v"(w[6]), "=&v"(w[7])
      : "v"(va[0]), "v"(va[1]), "v"(va[2]), "v"(va[3]), "v"(va[4]), "v"(va[5]), "v"(va[6]),
        "v"(va[7]), "n"(OFF)
      : "memory");
}

__device__ __forceinline__ void wait_k16(u32x4 (&k)[4][4]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(k[0][0]), "+v"(k[0][1]), "+v"(k[0][2]), "+v"(k[0][3]), "+v"(k[1][0]),
                 "+v"(k[1][1]), "+v"(k[1][2]), "+v"(k[1][3]), "+v"(k[2][0]), "+v"(k[2][1]),
                 "+v"(k[2][2]), "+v"(k[2][3]), "+v"(k[3][0]), "+v"(k[3][1]), "+v"(k[3][2]),
                 "+v"(k[3][3])
               :
               : "memory");
}

__device__ __forceinline__ void wait_v32(u32x2_t (&w)[4][8]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(w[0][0]), "+v"(w[0][1]), "+v"(w[0][2]), "+v"(w[0][3]), "+v"(w[0][4]),
                 "+v"(w[0][5]), "+v"(w[0][6]), "+v"(w[0][7]), "+v"(w[1][0]), "+v"(w[1][1]),
                 "+v"(w[1][2]), "+v"(w[1][3]), "+v"(w[1][4]), "+v"(w[1][5]), "+v"(w[1][6]),
                 "+v"(w[1][7]), "+v"(w[2][0]), "+v"(w[2][1]), "+v"(w[2][2]), "+v"(w[2][3]),
                 "+v"(w[2][4]), "+v"(w[2][5]), "+v"(w[2][6]), "+v"(w[2][7]), "+v"(w[3][0]),
                 "+v"(w[3][1]), "+v"(w[3][2]), "+v"(w[3][3]), "+v"(w[3][4]), "+v"(w[3][5]),
                 "+v"(w[3][6]), "+v"(w[3][7])
               :
               : "memory");
}

__device__ __forceinline__ void wait_v16(u32x2_t (&w)[2][8]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(w[0][0]), "+v"(w[0][1]), "+v"(w[0][2]), "+v"(w[0][3]), "+v"(w[0][4]),
                 "+v"(w[0][5]), "+v"(w[0][6]), "+v"(w[0][7]), "+v"(w[1][0]), "+v"(w[1][1]),
                 "+v"(w[1][2]), "+v"(w[1][3]), "+v"(w[1][4]), "+v"(w[1][5]), "+v"(w[1][6]),
                 "+v"(w[1][7])
               :
               : "memory");
}

constexpr int kPfQ = 64;                          // queries per prefill block
constexpr int kPfTileBytes = 2 * kSplit * D * 2;  // K then V of one staged 64-slot tile

// Causal attention over many queries per sequence (a prompt's prefill): one
// launch per layer, no split, no merge. Block = (64-query tile, query head h,
// batch b), four waves of 16 queries. The block stages each 64-slot K/V tile
// of kv head h / G once for its waves (a quarter each, LDS-direct, K and V; the
// next tile in flight), then every wave multiplies all 64 slots against its
// queries on the matrix cores as the decode kernel does per 16-slot
// group: S^T = K Q^T (slots as M, queries as N: four 16-slot M-tiles x four
// 32-dim steps), an online softmax per query in base 2, O^T += V^T P^T with P
// as hi/lo bf16 halves (weights keep ~16 bits; the denominator sums the fp32
// weights). A query sees slots <= its own position (masked per lane); the
// block reads tiles up to its largest position, the latest query tiles
// first. K rows are staged rotated (chunk c of slot s at column (c + s) % 16)
// and V rows by two chunks per slot (c + 2 (s % 8)); V^T operands come from
// transpose reads, one per 16 dims and 16 slots.
__global__ __launch_bounds__(kBlock) void attention_prefill(PrefillArgs a) {
  preload_prefill(a);
  constexpr int NW = kBlock / kWave;
  extern __shared__ __align__(16) unsigned char ring[];  // two staged tiles
  __shared__ int wave_pos[NW];
  const int tid = threadIdx.x, lane = tid & 63;
  // The bound on the wave, which a block of four waves does not tell the
  // compiler, is worth 2% (64 queries over 1064 slots: 29.3 -> 28.5 us).
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & (NW - 1);
  const int col = lane & 15, quad = lane >> 4;
  const int ntq = (a.Q + kPfQ - 1) / kPfQ;
  const int qt = ntq - 1 - static_cast<int>(blockIdx.x);  // latest queries first
  const int h = blockIdx.y, b = blockIdx.z, kvh = h / a.G;
  const int t = qt * kPfQ + wave * 16 + col;  // this lane's query
  const int tq = t < a.Q ? t : a.Q - 1;
  // Visible slots [0, pos]; a position past the cache sees every slot, a
  // negative one (and a padding query) none.
  const int64_t pv = a.pos[tq];
  const int pos = t >= a.Q || pv < 0 ? -1 : (pv >= a.cap ? static_cast<int>(a.cap) - 1 : static_cast<int>(pv));
  // B operand of S^T = K Q^T: dims 32 ks + 8 quad .. + 7 of this lane's query.
  const bf16_t* qrow = a.q + b * a.q_sb + h * a.q_sh + tq * a.q_st + 8 * quad;
  u32x4 qf[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) qf[ks] = *reinterpret_cast<const u32x4*>(qrow + 32 * ks);
  const float wmax = wave_max(static_cast<float>(pos));     // exact: |pos| < 2^24
  const float wmin = -wave_max(-static_cast<float>(pos));
  if (lane == 0) wave_pos[wave] = static_cast<int>(wmax);
  lds_barrier();
  int bmax = wave_pos[0];
#pragma unroll
  for (int w = 1; w < NW; ++w) bmax = wave_pos[w] > bmax ? wave_pos[w] : bmax;
  const int nkt = bmax < 0 ? 0 : bmax / kSplit + 1;  // tiles [0, nkt) hold every visible slot
  const int wave_last = static_cast<int>(wmax), wave_first = static_cast<int>(wmin);

  // Staging: wave w loads slots 16 w .. 16 w + 15 of each tile (K, then V),
  // through descriptors over the slots up to the block's largest position:
  // later slots (the cache may hold anything there, NaN included) read as
  // zeros, so masked weights never multiply NaN.
  const long kv_base = (static_cast<long>(b) * a.Hkv + kvh) * a.cap * D;
  const uint32_t range = static_cast<uint32_t>(bmax + 1) * D * 2;  // block-uniform (from LDS)
  const __amdgpu_buffer_rsrc_t krs = uniform_rsrc(a.keys + kv_base, range);
  const __amdgpu_buffer_rsrc_t vrs = uniform_rsrc(a.values + kv_base, range);
  uint32_t kvoff[4], vvoff[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int sl = 4 * u + (lane >> 4);
    kvoff[u] = static_cast<uint32_t>(sl * 256 + (((lane & 15) - sl) & 15) * 16);
    vvoff[u] = static_cast<uint32_t>(sl * 256 + (((lane & 15) - 2 * (sl & 7)) & 15) * 16);
  }
  auto stage = [&](int kt) {
    unsigned char* tb = ring + (kt & 1) * kPfTileBytes + wave * 4096;
    const uint32_t off = static_cast<uint32_t>(kt * kSplit + wave * 16) * D * 2;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(krs, (lds_void_t*)(tb + u * 1024), 16, kvoff[u], off, 0, 0);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(vrs, (lds_void_t*)(tb + kSplit * D * 2 + u * 1024), 16,
                                               vvoff[u], off, 0, 0);
  };
  if (nkt > 0) stage(0);

  // Operand addresses in tile buffer 0 (buffer 1 is kPfTileBytes further):
  // K slot 16 mt + col, chunk 4 ks + quad, rotated by the slot; for the V^T
  // transpose reads, slot 16 mt + r (r = 4 quad + col / 4), dims
  // 16 j + 4 (col % 4) .. + 3: 8 bytes of chunk 2 j + (col % 4) / 2, whose
  // position the slot rotates by 2 (r % 8).
  const uint32_t ring_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_t*)ring));
  uint32_t kaddr[4], vaddr[8];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    kaddr[ks] = ring_base + static_cast<uint32_t>(col * 256 + (((4 * ks + quad + col) & 15) * 16));
  const int vr = 4 * quad + (col >> 2);
#pragma unroll
  for (int j = 0; j < 8; ++j)
    vaddr[j] = ring_base + kSplit * D * 2 +
               static_cast<uint32_t>(vr * 256 + (((2 * j + ((col & 3) >> 1) + 2 * (vr & 7)) & 15) * 16) +
                                     (col & 1) * 8);

  const float scale2 = a.scale * 1.4426950408889634f;  // log2(e) / sqrt(D)
  f32x4_t acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  for (int kt = 0; kt < nkt; ++kt) {
    // This wave's part of tile kt has landed; after the barrier everyone's
    // has, and every wave has finished tile kt - 1, whose buffer tile kt + 1
    // now takes (in flight during this tile's work).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    if (kt + 1 < nkt) stage(kt + 1);
    const int s0 = kt * kSplit;
    if (s0 <= wave_last) {  // wave-uniform: some slot of the tile is visible to the wave
      const uint32_t tb = static_cast<uint32_t>((kt & 1) * kPfTileBytes);
      // All sixteen K fragments at once, then the scores.
      u32x4 kf[4][4];
      issue_k_pf<0>(kaddr[0] + tb, kf[0]);
      issue_k_pf<0>(kaddr[1] + tb, kf[1]);
      issue_k_pf<0>(kaddr[2] + tb, kf[2]);
      issue_k_pf<0>(kaddr[3] + tb, kf[3]);
      wait_k16(kf);
      f32x4_t st[4];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) st[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
          st[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kf[ks][mt]),
                                                           __builtin_bit_cast(bf16x8_t, qf[ks]),
                                                           st[mt], 0, 0, 0);
      // The V^T operands of the whole tile in flight during the softmax.
      uint32_t va[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) va[j] = vaddr[j] + tb;
      u32x2_t vw[4][8];
      issue_vt_tr<0>(va, vw[0]);
      issue_vt_tr<4096>(va, vw[1]);
      issue_vt_tr<8192>(va, vw[2]);
      issue_vt_tr<12288>(va, vw[3]);
      // Scores in base 2; slots past the query's position masked unless the
      // whole tile is visible to every query of the wave (a wave-uniform
      // branch: the mask is computed only on the tiles that need it).
      float sc[4][4];
      float tmax = -INFINITY;
      if (__builtin_expect(s0 + kSplit - 1 <= wave_first, 1)) {
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            sc[mt][i] = st[mt][i] * scale2;
            tmax = fmaxf(tmax, sc[mt][i]);
          }
      } else {
        // Slot s0 + 16 mt + 4 quad + i is visible iff 16 mt + i <= lim.
        const int lim = pos - s0 - 4 * quad;
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float v = st[mt][i] * scale2;
            sc[mt][i] = 16 * mt + i <= lim ? v : -INFINITY;
            tmax = fmaxf(tmax, sc[mt][i]);
          }
      }
      tmax = quad_max(tmax);
      const float m_new = fmaxf(m, tmax);
      // A query with nothing visible yet keeps weight 0 (no inf - inf).
      const float ms = m_new == -INFINITY ? 0.f : m_new;
      // Where no lane's max moved, alpha is exactly 1 (or 0 on an all-zero
      // state) and the products are identities: the wave skips them.
      if (!__all(m_new == m)) {
        const float alpha = __builtin_amdgcn_exp2f(m - ms);  // 0 while m is -inf
        l *= alpha;
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] *= alpha;
      }
      m = m_new;
      uint4 phl[4];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = __builtin_amdgcn_exp2f(sc[mt][i] - ms);
        l += (p[0] + p[1]) + (p[2] + p[3]);
        const uint2 pb = make_uint2(pack_bf2(p[0], p[1]), pack_bf2(p[2], p[3]));
        const uint2 pl = make_uint2(pack_bf2(p[0] - bf_lo(pb.x), p[1] - bf_hi(pb.x)),
                                    pack_bf2(p[2] - bf_lo(pb.y), p[3] - bf_hi(pb.y)));
        phl[mt] = make_uint4(pb.x, pb.y, pl.x, pl.y);
      }
      wait_v32(vw);
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8_t, make_uint4(vw[mt][j].x, vw[mt][j].y, vw[mt][j].x, vw[mt][j].y)),
              __builtin_bit_cast(bf16x8_t, phl[mt]), acc[j], 0, 0, 0);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // O[query][dim 16 j + 4 quad + i] = acc[j][i] / (the four quads' sums).
  const float ln = quad_sum(l);
  if (t < a.Q) {
    bf16_t* dst = a.out + b * a.o_sb + h * a.o_sh + static_cast<long>(t) * a.o_st + 4 * quad;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      *reinterpret_cast<uint2*>(dst + 16 * j) =
          make_uint2(pack_bf2(acc[j][0] / ln, acc[j][1] / ln), pack_bf2(acc[j][2] / ln, acc[j][3] / ln));
  }
}

template <typename T>
__device__ __forceinline__ void swap(T& a, T& b) {
  const T t = a;
  a = b;
  b = t;
}

// Causal attention over long prompts: as attention_prefill, but every wave
// takes 32 queries (two 16-query N tiles), so each K and V^T operand read from
// LDS feeds two products. Block = four waves: HPB query heads of one kv head
// (2, or 1 for an odd group) x 64 / 128 queries sharing each staged tile; two
// blocks per CU, whose waves overlap one's softmax with the other's products.
//
// Bit-identical to attention_prefill (the same tiles, products and sums per
// query), also where V holds infinities or NaN: of a tile, a query weighs the
// slots that its 16-query group and its 64-query tile reach there. Per layer,
// 32 query heads on 8 kv heads: 1500 queries 72 -> 56 us, 2048 126 -> 72, 5000
// 497 -> 305 (672 TFLOP/s counted once, 1.5 times that on the matrix cores,
// since the weights multiply as two halves); 4 sequences of 512 39 -> 25. What
// bounds it: per wave and tile 96 products (1536 cycles) and some 370 vector
// instructions with 32 exponentials (1900 cycles), which two waves per SIMD
// (244 registers) hardly overlap: raising the priority of either phase, or
// interleaving one group's products with the next one's weights, measured the
// same or slower (5000 queries: 302, 330 us).
template <int HPB>
__global__ __launch_bounds__(kBlock, 2) void attention_prefill_long(PrefillArgs a) {
  preload_prefill(a);
  constexpr int QW = 4 / HPB;       // 32-query groups per head
  constexpr int BQ = 32 * QW;       // queries per block
  extern __shared__ __align__(16) unsigned char ring[];  // two staged tiles
  __shared__ int wave_pos[4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, quad = lane >> 4;
  // Block L takes head unit L % units (units of one kv head a multiple of Hkv
  // apart: on one XCD where Hkv is a multiple of 8) and query rank L / units.
  // Ranks run from the latest queries, the longest, to the first; where every
  // block is resident at once (two per CU), the second half runs the other
  // way, so that a CU's two blocks sum to the same work.
  const int units = a.B * a.Hq / HPB, ntq = (a.Q + BQ - 1) / BQ;
  const int u = static_cast<int>(blockIdx.x) % units;
  int rank = static_cast<int>(blockIdx.x) / units;
  if (rank >= a.turn) rank = ntq - 1 - (rank - a.turn);
  const int qt = ntq - 1 - rank;
  const int b = u / (a.Hq / HPB), hu = u % (a.Hq / HPB);
  const int kvh = hu % a.Hkv;
  const int h = kvh * a.G + (hu / a.Hkv) * HPB + wave / QW;
  const int t0 = qt * BQ + (wave % QW) * 32 + col;  // this lane's queries: t0, t0 + 16
  // Visible slots [0, pos]; a position past the cache sees every slot, a
  // negative one (and a padding query) none.
  int pos[2];
  u32x4 qf[2][4];
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const int t = t0 + 16 * n, tq = t < a.Q ? t : a.Q - 1;
    const int64_t pv = a.pos[tq];
    pos[n] = t >= a.Q || pv < 0 ? -1 : (pv >= a.cap ? static_cast<int>(a.cap) - 1 : static_cast<int>(pv));
    // B operand of S^T = K Q^T: dims 32 ks + 8 quad .. + 7 of the query.
    const bf16_t* qrow = a.q + b * a.q_sb + h * a.q_sh + tq * a.q_st + 8 * quad;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) qf[n][ks] = *reinterpret_cast<const u32x4*>(qrow + 32 * ks);
  }
  // The last slot each 16-query group of the wave sees (exact: |pos| < 2^24).
  auto wave_top = [](int v) {
    return __builtin_amdgcn_readfirstlane(static_cast<int>(wave_max(static_cast<float>(v))));
  };
  const int last0 = wave_top(pos[0]), last1 = wave_top(pos[1]);
  const int wave_first = -wave_top(pos[0] < pos[1] ? -pos[0] : -pos[1]);
  if (lane == 0) wave_pos[wave] = last0 > last1 ? last0 : last1;
  lds_barrier();
  int bmax = wave_pos[0];
#pragma unroll
  for (int w = 1; w < 4; ++w) bmax = wave_pos[w] > bmax ? wave_pos[w] : bmax;
  const int nkt = bmax < 0 ? 0 : bmax / kSplit + 1;  // tiles [0, nkt) hold every visible slot
  // The last slot that the 64 queries around the wave's see: with one head per
  // block, the other 64 may see more of a tile.
  const int near = __builtin_amdgcn_readfirstlane(
      wave_pos[wave & 2] > wave_pos[wave | 1] ? wave_pos[wave & 2] : wave_pos[wave | 1]);

  // Staging and operand addresses as attention_prefill's four-wave block.
  const long kv_base = (static_cast<long>(b) * a.Hkv + kvh) * a.cap * D;
  const uint32_t range = static_cast<uint32_t>(bmax + 1) * D * 2;  // block-uniform (from LDS)
  const __amdgpu_buffer_rsrc_t krs = uniform_rsrc(a.keys + kv_base, range);
  const __amdgpu_buffer_rsrc_t vrs = uniform_rsrc(a.values + kv_base, range);
  uint32_t kvoff[4], vvoff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int sl = 4 * i + (lane >> 4);
    kvoff[i] = static_cast<uint32_t>(sl * 256 + (((lane & 15) - sl) & 15) * 16);
    vvoff[i] = static_cast<uint32_t>(sl * 256 + (((lane & 15) - 2 * (sl & 7)) & 15) * 16);
  }
  auto stage = [&](int kt) {
    unsigned char* tb = ring + (kt & 1) * kPfTileBytes + wave * 4096;
    const uint32_t off = static_cast<uint32_t>(kt * kSplit + wave * 16) * D * 2;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(krs, (lds_void_t*)(tb + i * 1024), 16, kvoff[i], off, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(vrs, (lds_void_t*)(tb + kSplit * D * 2 + i * 1024), 16,
                                               vvoff[i], off, 0, 0);
  };
  if (nkt > 0) stage(0);

  const uint32_t ring_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_t*)ring));
  uint32_t kaddr[4], vaddr[8];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    kaddr[ks] = ring_base + static_cast<uint32_t>(col * 256 + (((4 * ks + quad + col) & 15) * 16));
  const int vr = 4 * quad + (col >> 2);
#pragma unroll
  for (int j = 0; j < 8; ++j)
    vaddr[j] = ring_base + kSplit * D * 2 +
               static_cast<uint32_t>(vr * 256 + (((2 * j + ((col & 3) >> 1) + 2 * (vr & 7)) & 15) * 16) +
                                     (col & 1) * 8);

  const float scale2 = a.scale * 1.4426950408889634f;  // log2(e) / sqrt(D)
  f32x4_t acc[2][8];
  float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};
#pragma unroll
  for (int n = 0; n < 2; ++n)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[n][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // The work of one tile for the wave's groups N0 and 1.
  auto tile = [&](int kt, auto n0) {
    constexpr int N0 = decltype(n0)::value;
    const int s0 = kt * kSplit;
    const uint32_t tb = static_cast<uint32_t>((kt & 1) * kPfTileBytes);
    u32x4 kf[4][4];
    issue_k_pf<0>(kaddr[0] + tb, kf[0]);
    issue_k_pf<0>(kaddr[1] + tb, kf[1]);
    issue_k_pf<0>(kaddr[2] + tb, kf[2]);
    issue_k_pf<0>(kaddr[3] + tb, kf[3]);
    wait_k16(kf);
    f32x4_t st[2][4];
#pragma unroll
    for (int n = N0; n < 2; ++n)
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) st[n][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int n = N0; n < 2; ++n)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
          st[n][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8_t, kf[ks][mt]), __builtin_bit_cast(bf16x8_t, qf[n][ks]),
              st[n][mt], 0, 0, 0);
    // The V^T operands of half the tile in flight during the softmax.
    uint32_t va[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) va[j] = vaddr[j] + tb;
    u32x2_t vw[2][8];
    issue_vt_tr<0>(va, vw[0]);
    issue_vt_tr<4096>(va, vw[1]);
    uint4 phl[2][4];
#pragma unroll
    for (int n = N0; n < 2; ++n) {
      float sc[4][4];
      float tmax = -INFINITY;
      if (__builtin_expect(s0 + kSplit - 1 <= wave_first, 1)) {
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            sc[mt][i] = st[n][mt][i] * scale2;
            tmax = fmaxf(tmax, sc[mt][i]);
          }
      } else {
        const int lim = pos[n] - s0 - 4 * quad;  // slot s0 + 16 mt + 4 quad + i visible iff 16 mt + i <= lim
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float v = st[n][mt][i] * scale2;
            sc[mt][i] = 16 * mt + i <= lim ? v : -INFINITY;
            tmax = fmaxf(tmax, sc[mt][i]);
          }
      }
      tmax = quad_max(tmax);
      const float m_new = fmaxf(m[n], tmax);
      // A query with nothing visible yet keeps weight 0 (no inf - inf).
      const float ms = m_new == -INFINITY ? 0.f : m_new;
      if (!__all(m_new == m[n])) {
        const float alpha = __builtin_amdgcn_exp2f(m[n] - ms);  // 0 while m is -inf
        l[n] *= alpha;
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[n][j] *= alpha;
      }
      m[n] = m_new;
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = __builtin_amdgcn_exp2f(sc[mt][i] - ms);
        l[n] += (p[0] + p[1]) + (p[2] + p[3]);
        const uint2 pb = make_uint2(pack_bf2(p[0], p[1]), pack_bf2(p[2], p[3]));
        const uint2 pl = make_uint2(pack_bf2(p[0] - bf_lo(pb.x), p[1] - bf_hi(pb.x)),
                                    pack_bf2(p[2] - bf_lo(pb.y), p[3] - bf_hi(pb.y)));
        phl[n][mt] = make_uint4(pb.x, pb.y, pl.x, pl.y);
      }
    }
    auto weigh = [&](const u32x2_t (&v2)[2][8], int mt0) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        // With one head per block, slots past `near` as zeros: the lane's
        // slots are 0 .. e of the four from s0 + 16 (mt0 + mt) + 4 quad.
        uint32_t lo = ~0u, hi = ~0u;
        if constexpr (HPB == 1 && N0 == 1) {
          const int e = near - s0 - 16 * (mt0 + mt) - 4 * quad;
          lo = e < 0 ? 0u : (e == 0 ? 0xffffu : ~0u);
          hi = e < 2 ? 0u : (e == 2 ? 0xffffu : ~0u);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint32_t x = v2[mt][j].x & lo, y = v2[mt][j].y & hi;
          const u32x4 v = {x, y, x, y};
#pragma unroll
          for (int n = N0; n < 2; ++n)
            acc[n][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8_t, v), __builtin_bit_cast(bf16x8_t, phl[n][mt0 + mt]),
                acc[n][j], 0, 0, 0);
        }
      }
    };
    wait_v16(vw);
    u32x2_t vx[2][8];
    issue_vt_tr<8192>(va, vx[0]);
    issue_vt_tr<12288>(va, vx[1]);
    __builtin_amdgcn_sched_barrier(0);
    weigh(vw, 0);
    __builtin_amdgcn_sched_barrier(0);
    wait_v16(vx);
    weigh(vx, 2);
  };
  auto next_tile = [&](int kt) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    if (kt + 1 < nkt) stage(kt + 1);
  };
  // A weight of zero times an infinite or NaN V is NaN, so a group takes part
  // in the tiles it sees a slot of and no others, and weighs no slot past
  // `near`: first the tiles that both groups see and that end by `near`, both
  // groups at once, then the few others one group at a time, as group 1. Every
  // wave passes nkt barriers, wherever its two loops part.
  const int first_last = last0 < last1 ? last0 : last1;
  int whole = first_last < 0 ? 0 : first_last / kSplit + 1;
  if (HPB == 1 && whole > (near + 1) / kSplit) whole = (near + 1) / kSplit;
  for (int kt = 0; kt < whole; ++kt) {
    next_tile(kt);
    tile(kt, std::integral_constant<int, 0>{});
  }
  for (int kt = whole; kt < nkt; ++kt) {
    next_tile(kt);
#pragma unroll 1
    for (int g = 1; g >= 0; --g) {
      if (kt * kSplit <= (g == 1 ? last1 : last0)) tile(kt, std::integral_constant<int, 1>{});
#pragma unroll
      for (int j = 0; j < 8; ++j) swap(acc[0][j], acc[1][j]);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) swap(qf[0][ks], qf[1][ks]);
      swap(pos[0], pos[1]);
      swap(m[0], m[1]);
      swap(l[0], l[1]);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // O[query][dim 16 j + 4 quad + i] = acc[j][i] / (the four quads' sums).
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const float ln = quad_sum(l[n]);
    const int t = t0 + 16 * n;
    if (t >= a.Q) continue;
    bf16_t* dst = a.out + b * a.o_sb + h * a.o_sh + static_cast<long>(t) * a.o_st + 4 * quad;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      *reinterpret_cast<uint2*>(dst + 16 * j) =
          make_uint2(pack_bf2(acc[n][j][0] / ln, acc[n][j][1] / ln), pack_bf2(acc[n][j][2] / ln, acc[n][j][3] / ln));
  }
}

namespace {

template <int HPB>
int launch_prefill_long(const PrefillArgs& a, long blocks, size_t lds, hipStream_t st) {
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&attention_prefill_long<HPB>),
      hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
  (void)attr;  // a refused size surfaces as a launch error
  hipLaunchKernelGGL(attention_prefill_long<HPB>, dim3(static_cast<unsigned>(blocks)), dim3(kBlock),
                     lds, st, a);
  return launch_status();
}

}  // namespace

int prefill_attention(PrefillArgs& a, hipStream_t st) {
  if (a.B <= 0 || a.cap <= 0 || a.Q > (1 << 30) || a.Hq > 65535 || a.B > 65535)
    return HTN_EUNSUPPORTED;
  if (a.cap > (1L << 31) / (D * 2) - 2 * kSplit) return HTN_EUNSUPPORTED;  // 32-bit byte offsets
  if ((reinterpret_cast<uintptr_t>(a.q) & 15u) || ((a.q_sb | a.q_sh | a.q_st) & 7) ||
      (reinterpret_cast<uintptr_t>(a.out) & 7u) || ((a.o_sb | a.o_sh | a.o_st) & 3))
    return HTN_EUNSUPPORTED;
  a.scale = 1.0f / sqrtf(static_cast<float>(D));
  const size_t lds = 2 * static_cast<size_t>(kPfTileBytes);
  // Long prompts: two heads of a kv head (one, for an odd group) per block
  // with 32 queries per wave, as soon as its blocks outnumber the CUs (8B,
  // 1024 queries, 256 blocks: 38 us either way; 1500 72 -> 56; 512 16.5 -> 21).
  // One head's blocks hold 128 queries, twice the short kernel's: they take
  // grids that they pad by at most a tenth more (24 heads on 8 kv heads, 16
  // sequences of 64 queries 8.2 us short, 10.7 long; 4 of 300 15.5 / 17.6; 4 of
  // 512 33 / 25; 2 of 700 31 / 29).
  const int hpb = a.G % 2 == 0 ? 2 : 1;
  const long units = static_cast<long>(a.B) * a.Hq / hpb;
  const long bq = 128 / hpb, nq = (a.Q + bq - 1) / bq, cus = device_cus();
  const long padded = bq * nq, padded_short = (a.Q + kPfQ - 1) / kPfQ * kPfQ;
  if (units * nq > cus && units * nq * hpb < (1L << 31) && 10 * padded <= 11 * padded_short) {
    a.turn = static_cast<int>(units * nq <= 2 * cus ? (cus + units - 1) / units : nq);
    return hpb == 2 ? launch_prefill_long<2>(a, units * nq, lds, st)
                    : launch_prefill_long<1>(a, units * nq, lds, st);
  }
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&attention_prefill), hipFuncAttributeMaxDynamicSharedMemorySize,
      static_cast<int>(lds));
  (void)attr;  // a refused size surfaces as a launch error
  const dim3 grid(static_cast<unsigned>((a.Q + kPfQ - 1) / kPfQ), static_cast<unsigned>(a.Hq),
                  static_cast<unsigned>(a.B));
  hipLaunchKernelGGL(attention_prefill, grid, dim3(kBlock), lds, st, a);
  return launch_status();
}

}  // namespace htn
