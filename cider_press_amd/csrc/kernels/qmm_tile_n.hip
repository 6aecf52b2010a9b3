// Y[M,N] = X[M,K] . dequant(W[K,N]) on tiles (transpose=false).
//
// A row of W is contiguous along n while the matrix cores want 8 consecutive
// k of a column, so W goes through LDS: per 64-deep stage each thread
// dequantizes one 32-column chunk of one k row into the stage's [k][n] image,
// and the operands are read back transposed (ds_read_b64_tr_b16: 16 lanes' 4 k
// x 16 columns come back as one column of 4 k per lane).  A weight is thus
// dequantized once per BM rows.  X and W are double buffered, one barrier per
// stage: while stage s is multiplied, X(s + 1) is copied, W(s + 1) goes from
// registers through the dequantizer to LDS and W(s + 2) is loaded.
//
// W image: row k holds its 32-column chunk c at c ^ (k & 3), that chunk's
// 16-byte piece i at i ^ piece_key, which spreads both the transposed reads
// (4 rows x 32 columns at a time) and the writes (8 chunks of a row, one piece
// each) over the banks.  Counted at 512 x 4096, K = 12288: MFMA busy 37 %, 15 % of
// a wave's life waiting for LDS, bank conflicts 1.3 %.
#include "qmm_tile.hpp"

namespace cpq {
namespace tile {
namespace {

template <typename TT_, int BITS_, int BM_, int BN_, int WM_, int WN_>
struct NCfg {
  using TT = TT_;
  static constexpr int BITS = BITS_, BM = BM_, BN = BN_, WM = WM_, WN = WN_;
  static constexpr int THREADS = 64 * WM * WN;
  static constexpr int MB = BM / WM / 32, NB = BN / WN / 32;  // 32 x 32 blocks of a wave
  static constexpr int ABYTES = BM * BK * 2, BBYTES = BN * BK * 2;
  static constexpr int LDS = 2 * (ABYTES + BBYTES);
  static constexpr int COPIES = ABYTES / 1024 / (THREADS / 64);  // 1-KiB copies per wave and stage
  static constexpr int LOADS = kWordLoads<BITS> + 2;             // loads of a chunk
  static_assert(THREADS == 2 * BN, "one 32-element chunk per thread and stage");
  static_assert(COPIES * 1024 * (THREADS / 64) == ABYTES, "whole copies");
};

// One thread's raw chunk with its (scale, bias).
template <int BITS>
struct NChunk {
  uint32_t w[BITS];
  uint32_t s, b;
};

// Keeps the loads of a chunk that nothing uses any more: the stage barriers
// count on them.
template <int BITS>
__device__ __forceinline__ void keep(const NChunk<BITS>& c) {
#pragma unroll
  for (int i = 0; i < BITS; ++i) asm volatile("" ::"v"(c.w[i]));
  asm volatile("" ::"v"(c.s), "v"(c.b));
}

template <int BN>
__device__ __forceinline__ int piece_key(int k, int c) {
  return BN == 128 ? (k & 3) : ((c >> 2) ^ ((k & 1) << 1));
}

template <typename C>
struct NGeom {
  unsigned char* smem;
  Rsrc xr, sr, br;
  const unsigned char* wbase;  // row 0 of W at the tile's first column
  uint64_t wbytes;             // bytes from wbase to the end of W
  uint32_t xoff[C::COPIES];
  uint32_t woff, soff;   // this thread's chunk: bytes into W, (scale, bias) element, stage 0
  uint32_t wstep, srow;  // bytes per 64 rows of W; groups per row
  uint32_t bput, wkey;   // place and key of the chunk's row
  uint32_t aget, akey, bget[C::NB];
  int wave, lane;
};

template <typename C>
__device__ __forceinline__ void load_chunk(const NGeom<C>& g, int st, NChunk<C::BITS>& c) {
  const uint64_t at = (uint64_t)st * g.wstep;
  load_words<C::BITS>(rsrc(g.wbase + at, g.wbytes - at), g.woff, c.w);
  const uint32_t so = (g.soff + (uint32_t)st * BK * g.srow) * 2u;
  c.s = __builtin_amdgcn_raw_buffer_load_b16(g.sr, so, 0, 0);
  c.b = __builtin_amdgcn_raw_buffer_load_b16(g.br, so, 0, 0);
}

template <typename C>
__device__ __forceinline__ void put_piece(const NGeom<C>& g, int buf, int i, const u32x4& v) {
  *reinterpret_cast<u32x4*>(g.smem + 2 * C::ABYTES + buf * C::BBYTES + g.bput + (((uint32_t)i ^ g.wkey) << 4)) = v;
}

template <typename C, int G>
__device__ __forceinline__ void put_group(const NGeom<C>& g, int buf, const NChunk<C::BITS>& c, const SubCst& cst) {
  put_piece<C>(g, buf, G, sub_group<typename C::TT, C::BITS, G>(c.w, cst));
}

template <typename C>
struct NOps {
  u32x4 x[C::MB], w[C::NB];
};

// Operands of k step t (16 k).
template <typename C>
__device__ __forceinline__ void get(const NGeom<C>& g, int buf, int t, NOps<C>& o) {
  const unsigned char* pa = g.smem + buf * C::ABYTES + g.aget + (((uint32_t)(2 * t + (g.lane >> 5)) ^ g.akey) << 4);
  const unsigned char* pb = g.smem + 2 * C::ABYTES + buf * C::BBYTES + t * (16 * C::BN * 2);
#pragma unroll
  for (int j = 0; j < C::NB; ++j) {
    const u32x2 h0 = read_tr(pb + g.bget[j]), h1 = read_tr(pb + g.bget[j] + 4 * (C::BN * 2));
    o.w[j] = u32x4{h0.x, h0.y, h1.x, h1.y};
  }
#pragma unroll
  for (int i = 0; i < C::MB; ++i) o.x[i] = *reinterpret_cast<const u32x4*>(pa + i * 4096);
}

// Stage s (buffers P) while stage s + 1 is prepared in the other buffers:
// `cur` holds W(s + 1), `nxt` receives W(s + 2) (clamped to the last stage, so
// that every stage issues the same loads).  The copies are issued before W's
// loads, so all but those loads done means X(s + 1) landed.  The previous
// stage's last k step (in f1) is multiplied behind the barrier, while this
// stage's first operands are on their way.
template <typename C, int P>
__device__ __forceinline__ void stage(const NGeom<C>& g, int s, int last, const NChunk<C::BITS>& cur,
                                      NChunk<C::BITS>& nxt, NOps<C>& f0, NOps<C>& f1, Acc<C::MB, C::NB>& acc,
                                      uint32_t& top) {
  using TT = typename C::TT;
  get<C>(g, P, 0, f0);
  fence();
  copy_x(g.xr, g.smem + (P ^ 1) * C::ABYTES, g.wave, g.xoff, s + 1);
  order();
  fence();
  load_chunk<C>(g, min(s + 2, last), nxt);
  order();
  fence();
  const SubCst cst = cst_of<TT>(cur.s, cur.b, top);
  multiply<TT>(f1.x, f1.w, acc);
  put_group<C, 0>(g, P ^ 1, cur, cst);
  fence();
  get<C>(g, P, 1, f1);
  fence();
  multiply<TT>(f0.x, f0.w, acc);
  put_group<C, 1>(g, P ^ 1, cur, cst);
  fence();
  get<C>(g, P, 2, f0);
  fence();
  multiply<TT>(f1.x, f1.w, acc);
  put_group<C, 2>(g, P ^ 1, cur, cst);
  fence();
  get<C>(g, P, 3, f1);
  fence();
  multiply<TT>(f0.x, f0.w, acc);
  put_group<C, 3>(g, P ^ 1, cur, cst);
  stage_barrier<C::LOADS>();
  fence();
}

// The range's last stage (kv of its 64 k exist; K is a multiple of 8, rows of
// W past K read zeros).
template <typename C>
__device__ __forceinline__ void last_stage(const NGeom<C>& g, int kv, NOps<C>& f, Acc<C::MB, C::NB>& acc) {
  if (kv & 8) {
    clear_pieces<C::BM, C::THREADS>(g.smem, kv >> 3);
    __syncthreads();
  }
  for (int t = 0; t < (kv + 15) >> 4; ++t) {
    get<C>(g, 0, t, f);
    multiply<typename C::TT>(f.x, f.w, acc);
  }
}

template <typename C>
__global__ __launch_bounds__(C::THREADS) __attribute__((amdgpu_waves_per_eu(2))) void qmm_tile_n_kernel(const Args a) {
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
  const int s0 = kh * per, s1 = min(S, s0 + per);
  const int G = a.n >> a.gs_shift;

  NGeom<C> g;
  g.smem = smem;
  g.wave = wave;
  g.lane = lane;
  g.xr = rsrc(a.x + (size_t)row0 * a.k, (uint64_t)(a.m - row0) * a.k * 2);
  copy_sources(a, row0, wave, lane, g.xoff);
  {
    constexpr int PER = C::BN / 32;
    const int kr = tid / PER, sub = tid % PER;
    const uint64_t rowbytes = (uint64_t)a.n * BITS / 8, skip = (uint64_t)col0 * BITS / 8;
    g.wbase = reinterpret_cast<const unsigned char*>(a.w) + skip;
    g.wbytes = (uint64_t)a.k * rowbytes - skip;
    g.wstep = (uint32_t)(BK * rowbytes);
    g.woff = (uint32_t)(kr * rowbytes) + (uint32_t)(sub * 4 * BITS);
    g.srow = (uint32_t)G;
    g.soff = (uint32_t)kr * (uint32_t)G + (uint32_t)((col0 + 32 * sub) >> a.gs_shift);
    g.sr = rsrc(a.scales, (uint64_t)a.k * G * 2);
    g.br = rsrc(a.biases, (uint64_t)a.k * G * 2);
    g.bput = (uint32_t)(kr * C::BN * 2 + ((sub ^ (kr & 3)) << 6));
    g.wkey = (uint32_t)piece_key<C::BN>(kr, sub);
  }
  g.aget = (uint32_t)(32 * wm * MB + l32) * 128u;
  g.akey = (uint32_t)row_key(l32);
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int cb = wn * NB + j;
    const int kr = 8 * (lane >> 5) + ((lane & 15) >> 2), i = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
    g.bget[j] = (uint32_t)(kr * C::BN * 2 + ((cb ^ (kr & 3)) << 6) + ((i ^ piece_key<C::BN>(kr, cb)) << 4) +
                           (lane & 1) * 8);
  }

  // Stages s0 .. last - 1 in pairs of buffers (0, 1), the last one in buffers
  // 0; an odd number of them starts with one in buffers 1.
  NChunk<BITS> c0, c1;  // W for the stage in buffers 0, 1
  NOps<C> f0, f1;
  Acc<MB, NB> acc;
  uint32_t top = 0;
  const int last = s1 - 1, odd = (last - s0) & 1;
  const int kv = min(BK, a.k - last * BK);
  clear<MB, NB>(acc);
  {
    NChunk<BITS> first;
    load_chunk<C>(g, s0, first);
    order();
    fence();
    copy_x(g.xr, smem + odd * C::ABYTES, wave, g.xoff, s0);
    order();
    fence();
    if (odd)
      load_chunk<C>(g, min(s0 + 1, last), c0);
    else
      load_chunk<C>(g, min(s0 + 1, last), c1);
    order();
    const SubCst cst = cst_of<TT>(first.s, first.b, top);
    put_group<C, 0>(g, odd, first, cst);
    put_group<C, 1>(g, odd, first, cst);
    put_group<C, 2>(g, odd, first, cst);
    put_group<C, 3>(g, odd, first, cst);
  }
  stage_barrier<C::LOADS>();
  fence();
#pragma unroll
  for (int i = 0; i < MB; ++i) f1.x[i] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
  for (int j = 0; j < NB; ++j) f1.w[j] = u32x4{0u, 0u, 0u, 0u};
  int s = s0;
  if (odd) {
    stage<C, 1>(g, s, last, c0, c1, f0, f1, acc, top);
    ++s;
  }
#pragma clang loop unroll(disable)
  for (; s < last; s += 2) {
    stage<C, 0>(g, s, last, c1, c0, f0, f1, acc, top);
    stage<C, 1>(g, s + 1, last, c0, c1, f0, f1, acc, top);
  }
  multiply<TT>(f1.x, f1.w, acc);
  last_stage<C>(g, kv, f0, acc);
  keep(c0);
  keep(c1);

  // A scale too large for the subnormal form (bf16 only): once more from the
  // start, one stage at a time.
  if constexpr (Sig16<TT>::bf16) {
    if (__syncthreads_or(top >= kSubScaleLimit<TT> ? 1 : 0)) {
      clear<MB, NB>(acc);
      for (s = s0; s < s1; ++s) {
        __syncthreads();
        copy_x(g.xr, smem, wave, g.xoff, s);
        load_chunk<C>(g, s, c0);
        const BigCst big{TT::to_f32((uint16_t)c0.s), TT::to_f32((uint16_t)c0.b)};
        put_piece<C>(g, 0, 0, sub_group<TT, BITS, 0>(c0.w, big));
        put_piece<C>(g, 0, 1, sub_group<TT, BITS, 1>(c0.w, big));
        put_piece<C>(g, 0, 2, sub_group<TT, BITS, 2>(c0.w, big));
        put_piece<C>(g, 0, 3, sub_group<TT, BITS, 3>(c0.w, big));
        stage_barrier<0>();
        last_stage<C>(g, s == last ? kv : BK, f0, acc);
      }
    }
  }
  if (a.split > 1 && !exchange<MB, NB, C::THREADS>(a, t, kh, acc, &flag)) return;
  store_tile<TT>(a, row0 + 32 * wm * MB, col0 + 32 * wn * NB, lane, acc);
}

template <typename C>
hipError_t launch_n(hipStream_t st, const Args& a) {
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&qmm_tile_n_kernel<C>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
  if (attr != hipSuccess) return attr;
  return launch_kernel(qmm_tile_n_kernel<C>, C::LDS, C::THREADS, st, a);
}


// Stage times at 4-bit, group size 64.  A workgroup dequantizes each weight once
// and stages both operands: the widest tile costs least per multiply, the
// narrowest starts most workgroups.
const Shape kShapes[] = {
    {256, 256, 1, 1.48f, 1.75f}, {128, 256, 1, 0.98f, 1.20f}, {128, 128, 2, 0.78f, 0.58f},
    {64, 128, 3, 0.68f, 0.42f},  {32, 128, 4, 0.55f, 0.38f},
};

template <typename TT, int BITS>
hipError_t launch_shape(int cfg, hipStream_t s, const Args& a) {
  switch (cfg) {
    case 0: return launch_n<NCfg<TT, BITS, 256, 256, 2, 4>>(s, a);
    case 1: return launch_n<NCfg<TT, BITS, 128, 256, 2, 4>>(s, a);
    case 2: return launch_n<NCfg<TT, BITS, 128, 128, 2, 2>>(s, a);
    case 3: return launch_n<NCfg<TT, BITS, 64, 128, 2, 2>>(s, a);
    case 4: return launch_n<NCfg<TT, BITS, 32, 128, 1, 4>>(s, a);
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

TilePlan qmm_tile_n_plan(const QuantArgs& q, int m, int n, int k, int cu_count, size_t scratch_cap) {
  // 256 rows of X, 64 rows of W and the whole scale table within the 31-bit
  // ranges of their buffers.
  if (m < 1 || k < 1 || k % 8 != 0 || n % 32 != 0 || k > (1 << 21) || n > (1 << 24) ||
      (uint64_t)k * (n / q.gs) * 2 >= 0x7ffffff0ull)
    return TilePlan{-1, 1, 0, 0.f};
  return tile::plan_tiles(tile::kShapes, (int)(sizeof(tile::kShapes) / sizeof(tile::kShapes[0])), m, n, k, 0, cu_count,
                          scratch_cap);
}

hipError_t launch_qmm_tile_n(hipStream_t s, const TilePlan& p, void* scratch, const QuantArgs& q, const void* x,
                             void* y, int m, int n, int k) {
  if (p.cfg < 0 || (p.split > 1 && !scratch)) return hipErrorInvalidValue;
  const tile::Args a = tile::make_args(tile::kShapes[p.cfg], p, scratch, q, x, y, m, n, k);
  if (q.dtype == CPQ_DTYPE_BF16) return tile::launch_bits<dev::BF16>(q.bits, p.cfg, s, a);
  if (q.dtype == CPQ_DTYPE_F16) return tile::launch_bits<dev::F16>(q.bits, p.cfg, s, a);
  return hipErrorInvalidValue;
}

}  // namespace cpq
