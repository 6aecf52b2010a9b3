// Y[M,N] = X[M,K] . dequant(W[N,K])^T on tiles.
//
// W never passes through LDS: a 32-k chunk of a column is what one lane of an
// MFMA operand needs over a 64-deep stage once the k order is permuted (lane
// half h takes the stage's chunk h; k step t multiplies elements 8t .. 8t + 7
// of both chunks), so each lane loads its column's chunk and dequantizes it
// into operands.  Only X goes through LDS (a ring of 3 stages).  The first
// form of this kernel dequantized into LDS for all waves to read; its LDS
// traffic (2304 cycles per stage of a 256 x 256 tile against 2048 of MFMA)
// bounded it.  Here a 256 x 256 tile moves 1280 cycles' worth, and the WM waves
// of a column block repeat its dequantization.  Counted: 5.9 VALU per MFMA on
// 128 x 256 tiles at 4 bits (2048 x 12288 x 4096, MFMA busy 51 %), 5.0 on 256 x
// 256 at 8 bits (777 x 12288 x 4096, 38 %); no LDS bank conflicts.
#include <algorithm>

#include "qmm_tile.hpp"

namespace cpq {
namespace tile {
namespace {

template <typename TT_, int BITS_, int BM_, int BN_, int WM_, int WN_>
struct TCfg {
  using TT = TT_;
  static constexpr int BITS = BITS_, BM = BM_, BN = BN_, WM = WM_, WN = WN_;
  static constexpr int THREADS = 64 * WM * WN;
  static constexpr int MB = BM / WM / 32, NB = BN / WN / 32;  // 32 x 32 blocks of a wave
  static constexpr int SLOT = BM * BK * 2, SLOTS = 3;
  static constexpr int COPIES = SLOT / 1024 / (THREADS / 64);  // 1-KiB copies per wave and stage
  static constexpr int LOADS = kWordLoads<BITS> * NB;          // loads of a stage's chunks
  // Constants: a ring of 16 groups (slot = group % 16) of (scale | bias << 16)
  // words, one per column.
  static constexpr int CBASE = SLOTS * SLOT;
  static constexpr int LDS = CBASE + 16 * BN * 4;
  static_assert(THREADS == 2 * BN, "one block of scales or biases per thread");
  static_assert(COPIES * 1024 * (THREADS / 64) == SLOT, "whole copies");
};

// A lane's chunks of one stage, one per column block.
template <typename C>
struct TChunks {
  uint32_t w[C::NB][C::BITS];
};

template <typename C>
__device__ __forceinline__ void keep(const TChunks<C>& c) {
#pragma unroll
  for (int j = 0; j < C::NB; ++j)
#pragma unroll
    for (int i = 0; i < C::BITS; ++i) asm volatile("" ::"v"(c.w[j][i]));
}

// 8 groups of one column's scales or biases, read as the 5 aligned words
// around them (a row of G values starts on any 2 bytes) and shifted.  Read one
// group at a time they would fetch their cache line once per stage.
struct CstBlock {
  u32x4 v;
  uint32_t e;
};

template <typename C>
struct TGeom {
  unsigned char* smem;
  Rsrc xr, wr, cr;
  uint32_t xoff[C::COPIES];
  uint32_t woff[C::NB];        // this lane's chunks of stage 0
  uint32_t coff, cput, cget;   // constants: element it loads, where they go, its own columns'
  uint32_t aget;               // X operand of row block 0 at k step 0, within a slot
  int wave, half, gs_shift, groups;
};

template <typename C>
__device__ __forceinline__ void load_chunks(const TGeom<C>& g, int st, TChunks<C>& c) {
#pragma unroll
  for (int j = 0; j < C::NB; ++j) load_words<C::BITS>(g.wr, g.woff[j] + (uint32_t)st * (2 * 4 * C::BITS), c.w[j]);
}

template <typename C>
__device__ __forceinline__ void load_cst(const TGeom<C>& g, int block, CstBlock& c) {
  const uint32_t at = (g.coff + (uint32_t)block * 8u) * 2u & ~3u;
  c.v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(g.cr, at, 0, 0));
  c.e = __builtin_amdgcn_raw_buffer_load_b32(g.cr, at + 16u, 0, 0);
}

// Groups past the row's end (the second chunk of a last stage of 32 k) are
// stored as zeros: their weights are then zero.
template <typename C>
__device__ __forceinline__ void put_cst(const TGeom<C>& g, int block, const CstBlock& c) {
  const uint32_t sh = (g.coff & 1u) << 4;
  uint16_t* at = reinterpret_cast<uint16_t*>(g.smem + C::CBASE + (block & 1) * (8 * C::BN * 4) + g.cput);
  const uint32_t w[5] = {c.v.x, c.v.y, c.v.z, c.v.w, c.e};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t p = __builtin_amdgcn_alignbit(w[i + 1], w[i], sh);
    at[(2 * i) * (C::BN * 2)] = (uint16_t)(8 * block + 2 * i < g.groups ? p : 0u);
    at[(2 * i + 1) * (C::BN * 2)] = (uint16_t)(8 * block + 2 * i + 1 < g.groups ? p >> 16 : 0u);
  }
}

// Raw (scale | bias << 16) of this lane's chunks of stage st.
template <typename C>
__device__ __forceinline__ void raw_cst(const TGeom<C>& g, int st, uint32_t (&sb)[C::NB]) {
  const uint32_t gi = (uint32_t)((st * BK + 32 * g.half) >> g.gs_shift);
  const unsigned char* p = g.smem + C::CBASE + g.cget + (gi & 15u) * (uint32_t)(C::BN * 4);
#pragma unroll
  for (int j = 0; j < C::NB; ++j) sb[j] = *reinterpret_cast<const uint32_t*>(p + j * 128);
}

template <typename C>
__device__ __forceinline__ void make_cst(const uint32_t (&sb)[C::NB], SubCst (&cst)[C::NB], uint32_t& top) {
#pragma unroll
  for (int j = 0; j < C::NB; ++j) cst[j] = cst_of<typename C::TT>(sb[j] & 0xffffu, sb[j] >> 16, top);
}

template <typename C, int G, typename K>
__device__ __forceinline__ void dequant(const TChunks<C>& c, const K (&cst)[C::NB], u32x4 (&w)[C::NB]) {
#pragma unroll
  for (int j = 0; j < C::NB; ++j) {
    w[j] = sub_group<typename C::TT, C::BITS, G>(c.w[j], cst[j]);
    asm volatile("" : "+v"(w[j]));  // here, not where it is used (behind the next barrier)
  }
}

// X operands of k step t from the slot at `slot` (bytes): piece 4 half + t.
template <typename C>
__device__ __forceinline__ void get(const TGeom<C>& g, uint32_t slot, int t, u32x4 (&x)[C::MB]) {
  const unsigned char* p = g.smem + ((g.aget + slot) ^ (uint32_t)(t << 4));
#pragma unroll
  for (int i = 0; i < C::MB; ++i) x[i] = *reinterpret_cast<const u32x4*>(p + i * 4096);
}

template <typename C>
__device__ __forceinline__ uint32_t next_slot(uint32_t slot) {
  return slot == 2 * C::SLOT ? 0u : slot + C::SLOT;
}

// Stage s, its X in `slot`: `cur` holds W(s), whose first 8 k per lane are
// already operands (w0, constants cst); `nxt` holds W(s + 1).  X(s + 2) is
// copied into the slot of stage s - 1, W(s + 2) is loaded into `cur` once that
// is used up (both clamped to the last stage, so that every stage issues the
// same).  Behind the copies of X(s) come W(s - 0) .. : a stage issues COPIES
// copies, then LOADS loads, so at its start all but the last COPIES + 2 LOADS
// operations done means X(s) landed.  The previous stage's last k step (x1, w1)
// is multiplied behind the barrier, while this stage's operands are on their
// way.
template <typename C>
__device__ __forceinline__ void stage(const TGeom<C>& g, int s, int last, uint32_t slot, TChunks<C>& cur,
                                      const TChunks<C>& nxt, CstBlock& cb, SubCst (&cst)[C::NB], u32x4 (&x0)[C::MB],
                                      u32x4 (&x1)[C::MB], u32x4 (&w0)[C::NB], u32x4 (&w1)[C::NB],
                                      Acc<C::MB, C::NB>& acc, uint32_t& top) {
  using TT = typename C::TT;
  fence();
  stage_barrier<C::COPIES + 2 * C::LOADS>();
  get<C>(g, slot, 0, x0);
  fence();
  // Constants: 2^spb stages use a block of 8 groups.  Once stage s + 1 starts
  // one, the block before it is done with, and the block after it is loaded;
  // the next stage stores it.
  {
    const int spb = g.gs_shift - 3, in = s & ((1 << spb) - 1), block = s >> spb;
    if (in == 0)
      put_cst<C>(g, block + 1, cb);
    else if (in == (1 << spb) - 1)
      load_cst<C>(g, block + 2, cb);
  }
  order();
  fence();
  const uint32_t ahead = slot == 0 ? 2 * C::SLOT : slot - C::SLOT;
  copy_x(g.xr, g.smem + ahead, g.wave, g.xoff, min(s + 2, last));
  order();
  fence();
  multiply<TT>(x1, w1, acc);
  dequant<C, 1>(cur, cst, w1);
  fence();
  get<C>(g, slot, 1, x1);
  fence();
  multiply<TT>(x0, w0, acc);
  dequant<C, 2>(cur, cst, w0);
  fence();
  get<C>(g, slot, 2, x0);
  fence();
  multiply<TT>(x1, w1, acc);
  dequant<C, 3>(cur, cst, w1);
  fence();
  uint32_t sb[C::NB];
  raw_cst<C>(g, s + 1, sb);
  get<C>(g, slot, 3, x1);
  order();
  fence();
  load_chunks<C>(g, min(s + 2, last), cur);
  order();
  fence();
  multiply<TT>(x0, w0, acc);
  make_cst<C>(sb, cst, top);
  dequant<C, 0>(nxt, cst, w0);
}

template <typename C>
__global__ __launch_bounds__(C::THREADS) __attribute__((amdgpu_waves_per_eu(2))) void qmm_tile_t_kernel(const Args a) {
  using TT = typename C::TT;
  constexpr int BITS = C::BITS, MB = C::MB, NB = C::NB;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ unsigned int flag;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / C::WN, wn = wave % C::WN, l32 = lane & 31;
  const int v = xcd_order(blockIdx.x, a.tiles_m * a.tiles_n * a.split);
  const int kh = v % a.split, t = v / a.split;
  const int row0 = (t % a.tiles_m) * C::BM, col0 = (t / a.tiles_m) * C::BN;
  const int S = (a.k + BK - 1) / BK, per = (S + a.split - 1) / a.split;
  const int s0 = kh * per, s1 = min(S, s0 + per), last = s1 - 1;
  const int G = a.k >> a.gs_shift;

  TGeom<C> g;
  g.smem = smem;
  g.wave = wave;
  g.half = lane >> 5;
  g.gs_shift = a.gs_shift;
  g.groups = G;
  g.xr = rsrc(a.x + (size_t)row0 * a.k, (uint64_t)(a.m - row0) * a.k * 2);
  copy_sources(a, row0, wave, lane, g.xoff);
  const uint64_t rowbytes = (uint64_t)a.k * BITS / 8;
  // Columns past N read zeros (never stored).
  g.wr = rsrc(reinterpret_cast<const unsigned char*>(a.w) + (uint64_t)col0 * rowbytes, (uint64_t)(a.n - col0) * rowbytes);
#pragma unroll
  for (int j = 0; j < NB; ++j)
    g.woff[j] = (uint32_t)((uint64_t)(32 * (wn * NB + j) + l32) * rowbytes) + (uint32_t)(g.half * 4 * BITS);
  {
    // The table this wave loads constants from, from the aligned word holding
    // the tile's first group (the last word may reach 2 bytes past the table).
    const bool is_b = wave >= C::BN / 64;
    const int col = tid & (C::BN - 1);
    const uintptr_t tab = reinterpret_cast<uintptr_t>(is_b ? a.biases : a.scales) + (uint64_t)col0 * G * 2;
    const uint32_t skew = (uint32_t)(tab >> 1) & 1u;
    g.cr = rsrc(reinterpret_cast<const void*>(tab & ~(uintptr_t)3), ((uint64_t)(a.n - col0) * G + skew + 1) / 2 * 4);
    g.coff = (uint32_t)col * (uint32_t)G + skew;
    g.cput = (uint32_t)col * 4u + (is_b ? 2u : 0u);
    g.cget = (uint32_t)(32 * wn * NB + l32) * 4u;
  }
  g.aget = (uint32_t)(32 * wm * MB + l32) * 128u + (((uint32_t)(4 * g.half) ^ (uint32_t)row_key(l32)) << 4);

  TChunks<C> ca, cb;
  CstBlock blk;
  SubCst cst[NB];
  u32x4 x0[MB], x1[MB], w0[NB], w1[NB];
  Acc<MB, NB> acc;
  uint32_t top = 0;
  const int spb = a.gs_shift - 3;
  clear<MB, NB>(acc);
  // Constants and chunks of the first stages, then (in the stage's own order)
  // X(s0), W(s0), X(s0 + 1), W(s0 + 1).
  {
    CstBlock c;
    load_cst<C>(g, s0 >> spb, c);
    load_cst<C>(g, (s0 >> spb) + 1, blk);
    order();
    fence();
    copy_x(g.xr, smem, wave, g.xoff, s0);
    order();
    fence();
    load_chunks<C>(g, s0, ca);
    order();
    fence();
    copy_x(g.xr, smem + C::SLOT, wave, g.xoff, min(s0 + 1, last));
    order();
    fence();
    load_chunks<C>(g, min(s0 + 1, last), cb);
    order();
    fence();
    put_cst<C>(g, s0 >> spb, c);
    put_cst<C>(g, (s0 >> spb) + 1, blk);
    lds_barrier();
    uint32_t sb[NB];
    raw_cst<C>(g, s0, sb);
    make_cst<C>(sb, cst, top);
    dequant<C, 0>(ca, cst, w0);
  }
#pragma unroll
  for (int i = 0; i < MB; ++i) x1[i] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
  for (int j = 0; j < NB; ++j) w1[j] = u32x4{0u, 0u, 0u, 0u};
  // Stages s0 .. last - 1 in pairs (the chunk sets change roles).
  uint32_t slot = 0;
  int s = s0;
#pragma clang loop unroll(disable)
  for (; s + 1 < last; s += 2) {
    stage<C>(g, s, last, slot, ca, cb, blk, cst, x0, x1, w0, w1, acc, top);
    slot = next_slot<C>(slot);
    stage<C>(g, s + 1, last, slot, cb, ca, blk, cst, x0, x1, w0, w1, acc, top);
    slot = next_slot<C>(slot);
  }
  if (s < last) {
    stage<C>(g, s, last, slot, ca, cb, blk, cst, x0, x1, w0, w1, acc, top);
    slot = next_slot<C>(slot);
    ca = cb;
  }
  keep<C>(ca);
  keep<C>(cb);
  // The last stage: every copy landed, nothing left to prepare.
  fence();
  stage_barrier<0>();
  if (a.k - last * BK < BK) {
    clear_pieces<C::BM, C::THREADS>(smem + slot, 4);
    __syncthreads();
  }
  get<C>(g, slot, 0, x0);
  multiply<TT>(x1, w1, acc);
  multiply<TT>(x0, w0, acc);
  get<C>(g, slot, 1, x1);
  dequant<C, 1>(ca, cst, w1);
  multiply<TT>(x1, w1, acc);
  get<C>(g, slot, 2, x0);
  dequant<C, 2>(ca, cst, w0);
  multiply<TT>(x0, w0, acc);
  get<C>(g, slot, 3, x1);
  dequant<C, 3>(ca, cst, w1);
  multiply<TT>(x1, w1, acc);

  // A scale too large for the subnormal form (bf16 only): once more from the
  // start, one stage at a time.
  if constexpr (Sig16<TT>::bf16) {
    if (__syncthreads_or(top >= kSubScaleLimit<TT> ? 1 : 0)) {
      clear<MB, NB>(acc);
      for (s = s0; s < s1; ++s) {
        __syncthreads();
        copy_x(g.xr, smem, wave, g.xoff, s);
        CstBlock c;
        load_cst<C>(g, s >> spb, c);
        load_chunks<C>(g, s, ca);
        put_cst<C>(g, s >> spb, c);
        stage_barrier<0>();
        if (a.k - s * BK < BK) {
          clear_pieces<C::BM, C::THREADS>(smem, 4);
          __syncthreads();
        }
        uint32_t sb[NB];
        raw_cst<C>(g, s, sb);
        BigCst big[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j)
          big[j] = BigCst{TT::to_f32((uint16_t)(sb[j] & 0xffffu)), TT::to_f32((uint16_t)(sb[j] >> 16))};
        get<C>(g, 0, 0, x0);
        dequant<C, 0>(ca, big, w0);
        multiply<TT>(x0, w0, acc);
        get<C>(g, 0, 1, x0);
        dequant<C, 1>(ca, big, w0);
        multiply<TT>(x0, w0, acc);
        get<C>(g, 0, 2, x0);
        dequant<C, 2>(ca, big, w0);
        multiply<TT>(x0, w0, acc);
        get<C>(g, 0, 3, x0);
        dequant<C, 3>(ca, big, w0);
        multiply<TT>(x0, w0, acc);
      }
    }
  }
  if (a.split > 1 && !exchange<MB, NB, C::THREADS>(a, t, kh, acc, &flag)) return;
  store_tile<TT>(a, row0 + 32 * wm * MB, col0 + 32 * wn * NB, lane, acc);
}

template <typename C>
hipError_t launch_t(hipStream_t st, const Args& a) {
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&qmm_tile_t_kernel<C>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
  if (attr != hipSuccess) return attr;
  return launch_kernel(qmm_tile_t_kernel<C>, C::LDS, C::THREADS, st, a);
}


// Stage times at 4-bit, group size 64 (N = 4096 / 12288, M = 32 .. 2048).
const Shape kShapes[] = {
    {256, 256, 1, 1.38f, 1.67f}, {128, 256, 1, 0.80f, 1.10f}, {128, 128, 2, 0.56f, 0.58f},
    {64, 128, 4, 0.50f, 0.38f},  {32, 128, 4, 0.44f, 0.35f},
};

template <typename TT, int BITS>
hipError_t launch_shape(int cfg, hipStream_t s, const Args& a) {
  switch (cfg) {
    case 0: return launch_t<TCfg<TT, BITS, 256, 256, 2, 4>>(s, a);
    case 1: return launch_t<TCfg<TT, BITS, 128, 256, 1, 8>>(s, a);
    case 2: return launch_t<TCfg<TT, BITS, 128, 128, 1, 4>>(s, a);
    case 3: return launch_t<TCfg<TT, BITS, 64, 128, 1, 4>>(s, a);
    case 4: return launch_t<TCfg<TT, BITS, 32, 128, 1, 4>>(s, a);
    default: return hipErrorInvalidValue;
  }
}

template <typename TT>
hipError_t launch_bits(int bits, int cfg, hipStream_t s, const Args& a) {
  switch (bits) {
    case 2: return launch_shape<TT, 2>(cfg, s, a);
    case 3: return launch_shape<TT, 3>(cfg, s, a);
    case 4: return launch_shape<TT, 4>(cfg, s, a);
    case 5: return launch_shape<TT, 5>(cfg, s, a);
    case 6: return launch_shape<TT, 6>(cfg, s, a);
    case 8: return launch_shape<TT, 8>(cfg, s, a);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace
}  // namespace tile

TilePlan qmm_tile_t_plan(const QuantArgs& q, int m, int n, int k, int cu_count, size_t scratch_cap) {
  // 32 columns are stored together.  K past 2^21 leaves the smaller tiles, past
  // about 2^24 none (4-bit 8 x 256, K = 2^21 + 1024: general kernel 58 ms, tiles 1.0).
  if (m < 1 || n < 32 || n % 32 != 0 || k < 32) return TilePlan{-1, 1, 0, 0.f};
  return tile::plan_tiles(tile::kShapes, (int)(sizeof(tile::kShapes) / sizeof(tile::kShapes[0])), m, n, k, q.bits,
                          cu_count, scratch_cap);
}

// The plan's time as measured, to compare with other kernels' (the plan itself
// only ranks tiles): a tile's calls take this share of their estimate, unsplit
// and split (4-bit, 639 shapes: 5th to 95th percentile within 0.91 .. 1.14
// after it), and where several workgroups share a CU the wider words cost more
// per stage (5, 6 bits 1.5, 8 bits 1.45 times; 8-bit 3 x 20544 x 10336 79.8 us,
// plan 47.8).
float qmm_tile_t_us(const QuantArgs& q, const TilePlan& p, int m, int n, int k, int cu_count) {
  static const float kMeasured[][2] = {{1.04f, 0.90f}, {0.90f, 0.83f}, {1.06f, 0.95f}, {0.97f, 0.87f}, {0.85f, 0.84f}};
  const tile::Shape& sh = tile::kShapes[p.cfg];
  const long cus = cu_count > 0 ? cu_count : 256;
  const long tiles = (long)((m + sh.bm - 1) / sh.bm) * ((n + sh.bn - 1) / sh.bn);
  const long load = (tiles * p.split + cus - 1) / cus, rounds = (load + sh.resident - 1) / sh.resident;
  const int S = (k + tile::BK - 1) / tile::BK, per = (S + p.split - 1) / p.split;
  const float wide = q.bits == 8 ? 1.45f : q.bits >= 5 ? 1.5f : 1.f;
  const float alone = sh.alone * (float)rounds, each = sh.each * (float)load;
  const float us = p.us + (float)per * (std::max(alone, each * wide) - std::max(alone, each));
  return us * kMeasured[p.cfg][p.split > 1];
}

hipError_t launch_qmm_tile_t(hipStream_t s, const TilePlan& p, void* scratch, const QuantArgs& q, const void* x,
                             void* y, int m, int n, int k) {
  if (p.cfg < 0 || (p.split > 1 && !scratch)) return hipErrorInvalidValue;
  const tile::Args a = tile::make_args(tile::kShapes[p.cfg], p, scratch, q, x, y, m, n, k);
  if (q.dtype == CPQ_DTYPE_BF16) return tile::launch_bits<dev::BF16>(q.bits, p.cfg, s, a);
  if (q.dtype == CPQ_DTYPE_F16) return tile::launch_bits<dev::F16>(q.bits, p.cfg, s, a);
  return hipErrorInvalidValue;
}

}  // namespace cpq
