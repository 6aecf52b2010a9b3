// Tiled quantized GEMM for gfx950, every width and both weight directions.
//
//   qmm_tile_t.hip:  Y[M,N] = X[M,K] . dequant(W[N,K])^T   (affine_qmm_t)
//   qmm_tile_n.hip:  Y[M,N] = X[M,K] . dequant(W[K,N])     (affine_qmm_n)
//
// This file: what both share, and the choice of tile and K split.
//
// Reference ops: qmm_t_impl / qmm_n_impl (kernels-mlx/mlx/backend/metal/
// kernels/quantized.h:1087-1213, 1215-1349).  Numerics as every path here:
// each weight dequantized to T (RNE of fmaf(s, q, b)), fp32 accumulation on
// the matrix cores, one rounding to T.
//
// A workgroup owns a BM x BN tile over a range of 64-deep K stages; X is copied
// into LDS by buffer_load ... lds as rows of 64 k (128 bytes), the 16-byte piece
// c of row r at c ^ ((r >> 1) & 7).  One ds_read_b128 serves lanes {0-3, 12-15,
// 20-27}, {4-11, 16-19, 28-31} and the same of the upper half together, one
// ds_read_b64_tr_b16 lanes 0-31 and 32-63 (measured lane by lane): operand reads
// of 32 rows at one piece are conflict-free.
//
// MFMA 32x32x16 with W as the A operand: D[n][m] in lane m + 32 ((n/4) % 2),
// register 4 (n/8) + n % 4, so a lane's registers are 4 consecutive columns of
// one output row: 8-byte stores.
#pragma once

#include <algorithm>

#include "../cpq_internal.hpp"
#include "subnormal.hpp"

namespace cpq {
namespace tile {

using namespace dev;

constexpr int BK = 64;
constexpr int SC1 = 16;  // cache policy: through to the memory side

// Split-K words at the head of the scratch: arrivals of tile t at [t].  Zero
// between launches.
constexpr int kMaxTiles = (int)(kWideCounterBytes / 4);

struct Args {
  const uint32_t* w;
  const uint16_t* scales;
  const uint16_t* biases;
  const uint16_t* x;
  uint16_t* y;
  int m, n, k, gs_shift, tiles_m, tiles_n, split;
  float* part;
  unsigned int* counters;
};

constexpr uint64_t kRange = 0x7ffffff0ull;  // bytes addressed through one buffer at most

__device__ __forceinline__ Rsrc rsrc(const void* p, uint64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0,
                                           (int)(bytes > kRange ? (uint32_t)kRange : (uint32_t)bytes), 0x00020000);
}

template <typename TT>
__device__ __forceinline__ f32x16 mma(const u32x4& a, const u32x4& b, const f32x16& c) {
  if constexpr (Sig16<TT>::bf16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
}

// Wait for all but N vector-memory operations of this wave and for its LDS
// operations, then the workgroup barrier.
template <int N>
__device__ __forceinline__ void stage_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (0 << 8) | ((N >> 4) << 14));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// One 1-KiB copy of a wave into LDS (16 bytes a lane).
__device__ __forceinline__ void copy_1k(Rsrc r, unsigned char* lds, uint32_t off, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, off, soff, 0, 0);
}

typedef short s16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ u32x2 read_tr(const unsigned char* lds) {
  return __builtin_bit_cast(u32x2,
                            __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)lds));
}

__device__ __forceinline__ int row_key(int r) { return (r >> 1) & 7; }

// Vector-memory instructions that load a chunk's words.
template <int BITS>
constexpr int kWordLoads = BITS >= 5 ? 2 : 1;

// Keeps the operand reads ahead of the MFMAs they are to hide behind (left
// alone, the compiler sinks them next to their uses).
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }

__device__ __forceinline__ void order() { asm volatile("" ::: "memory"); }

// Workgroup -> (tile, k part): each XCD (linear ids congruent mod 8) takes a
// contiguous run of (tile, part) pairs, part fastest, then M tiles, so a run
// shares panels of W.
__device__ __forceinline__ int xcd_order(int id, int count) {
  const int q = count >> 3, r = count & 7, x = id & 7;
  return x * q + min(x, r) + (id >> 3);
}

template <int MB, int NB>
using Acc = f32x16[MB][NB];

template <int MB, int NB>
__device__ __forceinline__ void clear(Acc<MB, NB>& acc) {
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
}

// One k step of a wave's tile: W is the MFMA's A operand.
template <typename TT, int MB, int NB>
__device__ __forceinline__ void multiply(const u32x4 (&x)[MB], const u32x4 (&w)[NB], Acc<MB, NB>& acc) {
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int i = 0; i < MB; ++i) acc[i][j] = mma<TT>(w[j], x[i], acc[i][j]);
}

// Split K: every part parks its fp32 tile through to the memory side, waits
// until its stores are complete and only then counts its arrival; the last to
// arrive adds the parts in k order (the result does not depend on who that
// is), clears the counter for the next launch and returns true.  It reads 16
// vectors a thread at once, of several parts where a tile has fewer: a part
// at a time cost a memory round trip each.
template <int MB, int NB, int THREADS>
__device__ __forceinline__ bool exchange(const Args& a, int t, int kh, Acc<MB, NB>& acc, unsigned int* flag) {
  constexpr int NV = MB * NB * 4, U = NV >= 16 ? 1 : 16 / NV;
  const int tid = threadIdx.x;
  const uint64_t bytes = (uint64_t)a.split * NV * THREADS * 16;
  const Rsrc pr = rsrc(reinterpret_cast<const char*>(a.part) + t * bytes, bytes);
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const f32x16& b = acc[v / 4 / NB][v / 4 % NB];
    const int q = v & 3;
    const f32x4 p{b[4 * q], b[4 * q + 1], b[4 * q + 2], b[4 * q + 3]};
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, p), pr, tid * 16u, (kh * NV + v) * (THREADS * 16),
                                           SC1);
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (tid == 0) *flag = __hip_atomic_fetch_add(&a.counters[t], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (*flag != (unsigned int)(a.split - 1)) return false;
  clear<MB, NB>(acc);
#pragma clang loop unroll(disable)
  for (int kk = 0; kk < a.split; kk += U) {
    f32x4 p[U][NV];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int v = 0; v < NV; ++v)
        p[u][v] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(pr, tid * 16u,
                                                         (min(kk + u, a.split - 1) * NV + v) * (THREADS * 16), SC1));
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (kk + u >= a.split) break;
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[v / 4 / NB][v / 4 % NB][4 * (v & 3) + e] += p[u][v][e];
    }
  }
  if (tid == 0) __hip_atomic_store(&a.counters[t], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// Registers 4q .. 4q + 3 of a block are columns 8q + 4 (lane / 32) .. + 3 of
// output row lane % 32 (N is a multiple of 32, so they exist together).
template <typename TT, int MB, int NB>
__device__ __forceinline__ void store_tile(const Args& a, int row0, int col0, int lane, const Acc<MB, NB>& acc) {
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int row = row0 + 32 * i + (lane & 31);
    if (row >= a.m) continue;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int cb = col0 + 32 * j;
      if (cb >= a.n) continue;
      uint16_t* out = a.y + (size_t)row * a.n + cb + 4 * (lane >> 5);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<u32x2*>(out + 8 * q) = u32x2{TT::pack2(acc[i][j][4 * q], acc[i][j][4 * q + 1]),
                                                       TT::pack2(acc[i][j][4 * q + 2], acc[i][j][4 * q + 3])};
    }
  }
}

// Clears the pieces [from, 8) of every row of an X stage (K ends inside it).
template <int BM, int THREADS>
__device__ __forceinline__ void clear_pieces(unsigned char* stage, int from) {
  for (int i = threadIdx.x; i < BM * 8; i += THREADS) {
    const int r = i >> 3, c = i & 7;
    if (c >= from) *reinterpret_cast<u32x4*>(stage + r * 128 + ((c ^ row_key(r)) << 4)) = u32x4{0u, 0u, 0u, 0u};
  }
}

// Sources of a wave's activation copies (1 KiB each: 8 rows), at stage 0.
// Rows past M re-read row M - 1 (never stored).
template <int COPIES>
__device__ __forceinline__ void copy_sources(const Args& a, int row0, int wave, int lane, uint32_t (&xoff)[COPIES]) {
#pragma unroll
  for (int j = 0; j < COPIES; ++j) {
    const int r = (wave * COPIES + j) * 8 + (lane >> 3);
    const int c = (lane & 7) ^ row_key(r);
    xoff[j] = ((uint32_t)min(r, a.m - 1 - row0) * (uint32_t)a.k + (uint32_t)(c * 8)) * 2u;
  }
}

template <int COPIES>
__device__ __forceinline__ void copy_x(Rsrc xr, unsigned char* slot, int wave, const uint32_t (&xoff)[COPIES], int st) {
#pragma unroll
  for (int j = 0; j < COPIES; ++j)
    copy_1k(xr, slot + (wave * COPIES + j) * 1024, xoff[j], (uint32_t)st * (BK * 2));
}

// A chunk's constants; `top` keeps the largest scale magnitude seen.
template <typename TT>
__device__ __forceinline__ SubCst cst_of(uint32_t sv, uint32_t bv, uint32_t& top) {
  top = max(top, sv & 0x7fffu);
  return SubCst{TT::to_f32((uint16_t)sv) * 16777216.0f, TT::to_f32((uint16_t)bv)};
}

// ---------------------------------------------------------------------------
// Host side: tile and split by estimated time
// ---------------------------------------------------------------------------

// One tile size: resident workgroups per CU, and the time of a 64-deep stage
// (us) of a workgroup by itself (alone: latency) and of each of several on one
// CU (each: throughput), from measured calls that differ in their tile count.
struct Shape {
  int bm, bn, resident;
  float alone, each;
};

// The cheapest (tile, split) for m x n x k: rounds of workgroups, each its
// stages plus about 4 us of launch, prologue and store; a split adds an
// exchange of 1 us + 0.35 us per part + its parked bytes, written and read, at
// about 4 TB/s.  A tile's rows of X, and of W at w_bits per weight (0: addressed
// some other way), lie within a buffer's 31-bit range.  cfg < 0 where nothing
// fits.  CPQ_TILE_CFG and CPQ_QMM_SPLIT
// force the tile and the split (test hooks, read per call).
inline TilePlan plan_tiles(const Shape* shapes, int count, int m, int n, int k, int w_bits, int cu_count,
                           size_t scratch_cap) {
  const int cus = cu_count > 0 ? cu_count : 256, S = (int)(((unsigned)k + BK - 1) / BK);
  const int only = env_int("CPQ_TILE_CFG", -1), forced = env_int("CPQ_QMM_SPLIT", 0);
  // The splits worth a look (no empty part, two stages at least) and their stages.
  // Every op that may take a tile comes here: 32-bit divisions, and few.
  int splits[16], pers[16], ways = 0;
  for (int want = 1; want <= 16; ++want) {
    if (forced > 0 && want != std::min(forced, 16)) continue;
    const int per = (S + want - 1) / want, split = (S + per - 1) / per;
    if (split > 1 && per < 2 && forced <= 0) break;
    if (ways && split == splits[ways - 1]) continue;
    splits[ways] = split;
    pers[ways++] = per;
  }
  TilePlan best{-1, 1, 0, 0.f};
  for (int c = 0; c < count; ++c) {
    if (only >= 0 && only < count && c != only) continue;
    const Shape& sh = shapes[c];
    if ((uint64_t)std::max(16 * sh.bm, w_bits * sh.bn) * (uint64_t)k / 8 > kRange) continue;
    const long all = (long)(((unsigned)m + sh.bm - 1) / (unsigned)sh.bm) * (long)(((unsigned)n + sh.bn - 1) / (unsigned)sh.bn);
    if (all > (1L << 30)) continue;
    const unsigned tiles = (unsigned)all;
    for (int i = 0; i < ways; ++i) {
      const int split = splits[i], per = pers[i];
      size_t bytes = 0;
      float us = 0.f;
      if (split > 1) {
        if (tiles > (unsigned)kMaxTiles) break;
        const size_t parts = (size_t)tiles * split * sh.bm * sh.bn * sizeof(float);
        bytes = kWideCounterBytes + parts;
        if (bytes > scratch_cap) break;
        us = 1.f + 0.35f * (float)split + 2.f * (float)parts / 4e6f;
      }
      const unsigned load = (tiles * (unsigned)split + (unsigned)cus - 1) / (unsigned)cus;
      const unsigned rounds = (load + (unsigned)sh.resident - 1) / (unsigned)sh.resident;
      us += (float)per * std::max(sh.alone * (float)rounds, sh.each * (float)load) + 3.f + (float)rounds;
      if (best.cfg < 0 || us < best.us) best = TilePlan{c, split, bytes, us};
    }
  }
  return best;
}

inline Args make_args(const Shape& sh, const TilePlan& p, void* scratch, const QuantArgs& q, const void* x, void* y,
                      int m, int n, int k) {
  Args a;
  a.w = q.w;
  a.scales = static_cast<const uint16_t*>(q.scales);
  a.biases = static_cast<const uint16_t*>(q.biases);
  a.x = static_cast<const uint16_t*>(x);
  a.y = static_cast<uint16_t*>(y);
  a.m = m;
  a.n = n;
  a.k = k;
  a.gs_shift = q.gs == 32 ? 5 : q.gs == 64 ? 6 : 7;
  a.tiles_m = (m + sh.bm - 1) / sh.bm;
  a.tiles_n = (n + sh.bn - 1) / sh.bn;
  a.split = p.split;
  a.counters = static_cast<unsigned int*>(scratch);
  a.part = scratch ? reinterpret_cast<float*>(static_cast<char*>(scratch) + kWideCounterBytes) : nullptr;
  return a;
}

template <typename K>
hipError_t launch_kernel(K kernel, int lds, int threads, hipStream_t st, const Args& a) {
  hipLaunchKernelGGL(kernel, dim3((unsigned)(a.tiles_m * a.tiles_n * a.split)), dim3((unsigned)threads), (size_t)lds,
                     st, a);
  return hipGetLastError();
}

}  // namespace tile
}  // namespace cpq
