// Decode matmul for gfx950, up to 16 rows, every width and group count:
//   Y[M,N] = X[M,K] . dequant(W[N,K])^T,  K a multiple of 32.
//
// Reference ops: affine_qmv / affine_qmv_fast (kernels-mlx/mlx/backend/metal/
// kernels/quantized.h:749-975).  Each weight is dequantized to T (RNE of
// fmaf(s, q, b)), products accumulate in fp32, one rounding to T.
//
// One row at 4/8 bits shares this with qmv.hip (its lean layout, K in whole
// 512s, and its shared staging, some K in whole 256s); every other width is its
// own.  What it avoids is a chain of dependent waits: the
// dequantization through f16 subnormals needs no look at the constants before
// the stream starts, so a wave issues its activations, constants and first
// weights together, and waits for the rest of the workgroup only to add the
// K parts.
//
// A workgroup owns 16 columns; its waves split K into ranges of whole 128-k
// steps.  Lane (column c = lane % 16, g = lane / 16) streams the 32-k chunk
// 4 step + g of its column (BITS words) and feeds it as four MFMA 16x16x32
// operands (W's k order is permuted inside the step; the activations follow):
//   x: the wave's range of each row in LDS (in phases where the workgroup's
//      rows exceed it: a wave refills its own part, no barrier), a step's
//      16-byte pieces of row r at p ^ swz_key(r) (conflict-free for
//      ds_read_b128's lane groups);
//   scales, biases: the 4 steps' groups of a column read as aligned words
//      around them and shifted (rows of group counts start on any 2 bytes);
//   4 steps in flight, the next 4 requested before they are used.
#include <algorithm>
#include <type_traits>

#include "../cpq_internal.hpp"
#include "subnormal.hpp"

namespace cpq {
namespace {

using namespace dev;

constexpr int STEP = 128, BATCH = 4, MAXW = 12;

__device__ __forceinline__ Rsrc range(const void* p, uint64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)(uint32_t)bytes, 0x00020000);
}

// The words holding a table's groups of BATCH steps, one more for the skew.
template <int GS_SHIFT>
constexpr int kCstWords = BATCH * STEP / (1 << GS_SHIFT) / 2;

template <int GS_SHIFT>
struct Cst {
  uint32_t w[kCstWords<GS_SHIFT> + 1];
};

template <int GS_SHIFT>
__device__ __forceinline__ void load_cst(Rsrc r, uint32_t off, Cst<GS_SHIFT>& c) {
  constexpr int W = kCstWords<GS_SHIFT>;
  if constexpr (W == 2) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b96(r, off, 0, 0);
    c.w[0] = v[0]; c.w[1] = v[1]; c.w[2] = v[2];
  } else {
#pragma unroll
    for (int i = 0; i < W; i += 4) {
      const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off + 4 * i, 0, 0));
      c.w[i] = v.x; c.w[i + 1] = v.y; c.w[i + 2] = v.z; c.w[i + 3] = v.w;
    }
    c.w[W] = __builtin_amdgcn_raw_buffer_load_b32(r, off + 4 * W, 0, 0);
  }
}

// The 16-bit constant of step j's chunk g; `sh` = 16 where the table row
// starts in the upper half of a word.
template <int GS_SHIFT, int J>
__device__ __forceinline__ uint32_t cst_at(const Cst<GS_SHIFT>& c, uint32_t sh, int g) {
  auto word = [&](int i) { return __builtin_amdgcn_alignbit(c.w[i + 1], c.w[i], sh); };
  if constexpr (GS_SHIFT == 5) {  // 4 groups a step
    const uint32_t v = g >= 2 ? word(2 * J + 1) : word(2 * J);
    return (v >> ((g & 1) * 16)) & 0xffffu;
  } else if constexpr (GS_SHIFT == 6) {  // 2 groups a step
    return (word(J) >> ((g >> 1) * 16)) & 0xffffu;
  } else {  // 1 group a step
    return (word(J >> 1) >> ((J & 1) * 16)) & 0xffffu;
  }
}

template <int BITS, int GS_SHIFT>
struct Batch {
  uint32_t w[BATCH][BITS];
  Cst<GS_SHIFT> s, b;
};

struct Geom {
  Rsrc wr, sr, br;
  uint32_t woff;        // this lane's chunk at step 0 of the wave
  uint32_t soff, boff;  // aligned byte offsets of its groups there
  uint32_t ssh, bsh;    // 16 where they start in a word's upper half
  const unsigned char* xrow;  // its row of x in LDS
  int key, g, chunks, chunk0;  // chunks past `chunks` do not exist
};

template <int BITS, int GS_SHIFT>
__device__ __forceinline__ void load_batch(const Geom& q, int t0, Batch<BITS, GS_SHIFT>& p) {
  constexpr uint32_t GB = STEP / (1 << GS_SHIFT) * 2;  // table bytes per step
  load_cst<GS_SHIFT>(q.sr, q.soff + t0 * GB, p.s);
  load_cst<GS_SHIFT>(q.br, q.boff + t0 * GB, p.b);
#pragma unroll
  for (int j = 0; j < BATCH; ++j)
    load_words<BITS>(q.wr, q.woff + (uint32_t)(t0 + j) * (4 * 4 * BITS), p.w[j]);
}

// One step.  A chunk past the row's end gets zero constants: zero weights (its
// activations are zeros too).
template <typename TT, int BITS, int GS_SHIFT, int J, bool BIG>
__device__ __forceinline__ void step(const Geom& q, int t, const Batch<BITS, GS_SHIFT>& p, f32x4& acc, uint32_t& top) {
  const bool live = q.chunk0 + 4 * t < q.chunks;
  const uint32_t sv = live ? cst_at<GS_SHIFT, J>(p.s, q.ssh, q.g) : 0u;
  const uint32_t bv = live ? cst_at<GS_SHIFT, J>(p.b, q.bsh, q.g) : 0u;
  const float s = TT::to_f32((uint16_t)sv), b = TT::to_f32((uint16_t)bv);
  top = max(top, sv & 0x7fffu);
  const unsigned char* xs = q.xrow + t * (STEP * 2);
  using C = std::conditional_t<BIG, BigCst, SubCst>;
  const C c{BIG ? s : s * 16777216.0f, b};
  const u32x4 w[4] = {sub_group<TT, BITS, 0>(p.w[J], c), sub_group<TT, BITS, 1>(p.w[J], c),
                      sub_group<TT, BITS, 2>(p.w[J], c), sub_group<TT, BITS, 3>(p.w[J], c)};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const u32x4 xa = *reinterpret_cast<const u32x4*>(xs + (((4 * q.g + i) ^ q.key) << 4));
    acc = Mfma16<TT>::run(xa, w[i], acc);
  }
}

template <typename TT, int BITS, int GS_SHIFT, bool BIG>
__device__ __forceinline__ void use_batch(const Geom& q, int t0, int nt, const Batch<BITS, GS_SHIFT>& p, f32x4& acc,
                                          uint32_t& top) {
  step<TT, BITS, GS_SHIFT, 0, BIG>(q, t0, p, acc, top);
  if (t0 + 1 < nt) step<TT, BITS, GS_SHIFT, 1, BIG>(q, t0 + 1, p, acc, top);
  if (t0 + 2 < nt) step<TT, BITS, GS_SHIFT, 2, BIG>(q, t0 + 2, p, acc, top);
  if (t0 + 3 < nt) step<TT, BITS, GS_SHIFT, 3, BIG>(q, t0 + 3, p, acc, top);
}

template <typename TT, int BITS, int GS_SHIFT, bool PHASED>
__global__ __launch_bounds__(64 * MAXW) void decode_kernel(const uint32_t* __restrict__ w,
                                                           const uint16_t* __restrict__ scales,
                                                           const uint16_t* __restrict__ biases,
                                                           const uint16_t* __restrict__ x, uint16_t* __restrict__ y,
                                                           int m, int n, int k, int steps, int hold) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.x * 16, c = lane & 15, g = lane >> 4;
  const int S = (k + STEP - 1) / STEP;
  const int u0 = wave * steps, nt = min(steps, S - u0);  // this wave's steps (none where nt <= 0)
  const int G = k >> GS_SHIFT;
  const uint64_t rowbytes = (uint64_t)k * BITS / 8;

  f32x4 acc{0.f, 0.f, 0.f, 0.f};
  uint32_t top = 0;
  Geom q;
  if (nt > 0) {
    // Columns past N read zeros (never stored).
    q.wr = range(reinterpret_cast<const unsigned char*>(w) + n0 * rowbytes, (uint64_t)min(16, n - n0) * rowbytes);
    q.woff = (uint32_t)(c * rowbytes) + (uint32_t)(4 * u0 + g) * (4 * BITS);
    const uintptr_t st = reinterpret_cast<uintptr_t>(scales) + (uint64_t)n0 * G * 2;
    const uintptr_t bt = reinterpret_cast<uintptr_t>(biases) + (uint64_t)n0 * G * 2;
    const uint32_t tab = (uint32_t)min(16, n - n0) * (uint32_t)G * 2u;
    // From the aligned word holding the first group; the last word may reach
    // 2 bytes past the table.
    q.sr = range(reinterpret_cast<const void*>(st & ~(uintptr_t)3), (tab + (uint32_t)(st & 2) + 3u) & ~3u);
    q.br = range(reinterpret_cast<const void*>(bt & ~(uintptr_t)3), (tab + (uint32_t)(bt & 2) + 3u) & ~3u);
    const uint32_t at = ((uint32_t)c * (uint32_t)G + (uint32_t)((u0 * STEP) >> GS_SHIFT)) * 2u;
    q.soff = (at + (uint32_t)(st & 2)) & ~3u;
    q.boff = (at + (uint32_t)(bt & 2)) & ~3u;
    q.ssh = ((at + (uint32_t)(st & 2)) & 2u) << 3;
    q.bsh = ((at + (uint32_t)(bt & 2)) & 2u) << 3;
    q.g = g;
    q.chunks = k / 32;
    q.chunk0 = 4 * u0 + g;
    const int row = min(c, m - 1);
    if constexpr (!PHASED) hold = steps;
    unsigned char* xw = smem + (size_t)wave * m * hold * (STEP * 2);
    q.xrow = xw + (size_t)row * hold * (STEP * 2);
    q.key = swz_key(row);

    // Activations of up to 4 rows first, then the first batch, then the other
    // rows: what is waited for first was asked for first.
    const Rsrc xr = range(x, (uint64_t)m * k * 2);
    const int pieces = min(nt, hold) * 16;
    auto xoff = [&](int r, int p) {
      const int kk = u0 * STEP + p * 8;
      return p < pieces && kk < k ? ((uint32_t)r * (uint32_t)k + (uint32_t)kk) * 2u : 0xfffffff0u;
    };
    auto xput = [&](int r, int p, const u32x4& v) {
      if (p < pieces)
        *reinterpret_cast<u32x4*>(xw + ((size_t)r * hold + (p >> 4)) * (STEP * 2) + (((p & 15) ^ swz_key(r)) << 4)) = v;
    };
    // The phase of steps t0 .. t0 + hold - 1 takes the place of the one before
    // (the wave's own LDS, no barrier: other lanes read what this one writes, so
    // the phases' reads and writes are kept in order within the wave).
    auto next_phase = [&](int t0) {
      const int held = min(hold, nt - t0) * 16;
      wave_lds_order();
      for (int r0 = 0; r0 < m; r0 += 4)
        for (int p = lane; p < held; p += 64) {
          const int kk = (u0 + t0) * STEP + p * 8;
          u32x4 v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (r0 + r < m)
              v[r] = __builtin_bit_cast(
                  u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                             xr, kk < k ? ((uint32_t)(r0 + r) * (uint32_t)k + (uint32_t)kk) * 2u : 0xfffffff0u, 0, 0));
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (r0 + r < m)
              *reinterpret_cast<u32x4*>(xw + ((size_t)(r0 + r) * hold + (p >> 4)) * (STEP * 2) +
                                        (((p & 15) ^ swz_key(r0 + r)) << 4)) = v[r];
        }
      wave_lds_order();
      q.xrow -= hold * (STEP * 2);
    };
    Batch<BITS, GS_SHIFT> b0, b1;
    {
      u32x4 v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (r < m) v[r] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, xoff(r, lane), 0, 0));
      asm volatile("" ::: "memory");
      load_batch<BITS, GS_SHIFT>(q, 0, b0);
      asm volatile("" ::: "memory");
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (r < m) xput(r, lane, v[r]);
    }
    for (int r0 = 0; r0 < m; r0 += 4)
      for (int p0 = r0 == 0 ? 64 : 0; p0 < pieces; p0 += 64) {
        u32x4 v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (r0 + r < m)
            v[r] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, xoff(r0 + r, p0 + lane), 0, 0));
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (r0 + r < m) xput(r0 + r, p0 + lane, v[r]);
      }
    wave_lds_order();  // lanes read what other lanes staged
    for (int t0 = 0; t0 < nt; t0 += 2 * BATCH) {
      if (PHASED && t0 && t0 % hold == 0) next_phase(t0);
      if (t0 + BATCH < nt) load_batch<BITS, GS_SHIFT>(q, t0 + BATCH, b1);
      use_batch<TT, BITS, GS_SHIFT, false>(q, t0, nt, b0, acc, top);
      if (t0 + BATCH >= nt) break;
      if (PHASED && (t0 + BATCH) % hold == 0) next_phase(t0 + BATCH);
      if (t0 + 2 * BATCH < nt) load_batch<BITS, GS_SHIFT>(q, t0 + 2 * BATCH, b0);
      use_batch<TT, BITS, GS_SHIFT, false>(q, t0 + BATCH, nt, b1, acc, top);
    }
    // A scale too large for the subnormal form (bf16 only): this wave's range
    // once more.
    if constexpr (Sig16<TT>::bf16) {
      if (__builtin_amdgcn_ballot_w64(top >= kSubScaleLimit<TT>) != 0) {
        acc = f32x4{0.f, 0.f, 0.f, 0.f};
        q.xrow = xw + (size_t)row * hold * (STEP * 2) + (PHASED ? hold * (STEP * 2) : 0);
        for (int t0 = 0; t0 < nt; t0 += BATCH) {
          if (PHASED && t0 % hold == 0) next_phase(t0);
          load_batch<BITS, GS_SHIFT>(q, t0, b0);
          use_batch<TT, BITS, GS_SHIFT, true>(q, t0, nt, b0, acc, top);
        }
      }
    }
  }

  // K parts in wave order: lane (column c, rows 4g .. 4g + 3) of every wave.
  f32x4* parts = reinterpret_cast<f32x4*>(smem + (size_t)waves * m * (PHASED ? hold : steps) * (STEP * 2));
  parts[tid] = acc;
  __syncthreads();
  if (tid < 64 && 4 * g < m && n0 + c < n) {
    f32x4 sum = parts[lane];
    for (int i = 1; i < waves; ++i) sum += parts[i * 64 + lane];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (4 * g + e < m) y[(size_t)(4 * g + e) * n + n0 + c] = TT::from_f32(sum[e]);
  }
}

// Waves per workgroup and 128-k steps per wave: a batch of 4 steps each (all of
// a wave's loads in flight at once), up to 12 waves, up to 8 where the grid
// fills the chip twice (6-bit, us at 4 / 8 / 12 waves: 2048 x 2048 4.8 / 5.6 /
// 5.6, 2048 x 6144 9.8 / 9.9 / 7.5, 9984 x 3520 4-bit 9.5 / 8.7 / 11.2).
// CPQ_DECODE_WAVES sets their limit, 1 .. 12 (test hook).
void decode_split(int n, int k, int* waves, int* steps) {
  const int S = (k + STEP - 1) / STEP;
  const int most = (n + 15) / 16 >= 512 ? 8 : MAXW;
  const int limit = std::max(1, std::min(MAXW, env_int("CPQ_DECODE_WAVES", most)));
  const int w = std::min(limit, (S + BATCH - 1) / BATCH);
  *steps = (S + w - 1) / w;
  *waves = (S + *steps - 1) / *steps;
}

size_t decode_lds(int m, int waves, int steps) {
  return (size_t)waves * m * steps * (STEP * 2) + (size_t)waves * 64 * 16;
}

// The same with activations staged in phases: as many waves as hold a batch of
// steps each, and the steps a wave holds at once (whole batches, phases of
// about one length).  A refill costs a wave one round trip with nothing else
// of its own in flight: 8 rows of 12288 in two phases 20.0 us at 8 bits, against
// 16.8 for 4 rows in one.  Activations in registers instead (each lane its own
// row's pieces, no LDS) 21.5, and 25.7 against 19.4 at 12288 x 4096.
void decode_phases(int m, int k, int* waves, int* steps, int* hold) {
  const int S = (k + STEP - 1) / STEP, batch = m * BATCH * STEP * 2;
  const int w = std::min({MAXW, (160 * 1024 - MAXW * 64 * 16) / batch, (S + BATCH - 1) / BATCH});
  *steps = (S + w - 1) / w;
  *waves = (S + *steps - 1) / *steps;
  const int fit = (160 * 1024 - *waves * 64 * 16) / (*waves * batch), all = (*steps + BATCH - 1) / BATCH;
  const int phases = (all + fit - 1) / fit;
  *hold = (all + phases - 1) / phases * BATCH;
}

template <typename TT, int BITS, int GS_SHIFT, bool PHASED>
hipError_t launch_gs(hipStream_t s, const QuantArgs& q, const void* x, void* y, int m, int n, int k) {
  static const hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void*>(&decode_kernel<TT, BITS, GS_SHIFT, PHASED>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  if (attr != hipSuccess) return attr;
  int waves, steps;
  decode_split(n, k, &waves, &steps);
  int hold = steps;
  if constexpr (PHASED) decode_phases(m, k, &waves, &steps, &hold);
  hipLaunchKernelGGL((decode_kernel<TT, BITS, GS_SHIFT, PHASED>), dim3((unsigned)((n + 15) / 16)), dim3((unsigned)(64 * waves)),
                     decode_lds(m, waves, hold), s, q.w, static_cast<const uint16_t*>(q.scales),
                     static_cast<const uint16_t*>(q.biases), static_cast<const uint16_t*>(x),
                     static_cast<uint16_t*>(y), m, n, k, steps, hold);
  return hipGetLastError();
}

template <typename TT, int BITS, bool PHASED>
hipError_t launch_bits(hipStream_t s, const QuantArgs& q, const void* x, void* y, int m, int n, int k) {
  if (q.gs == 32) return launch_gs<TT, BITS, 5, PHASED>(s, q, x, y, m, n, k);
  if (q.gs == 64) return launch_gs<TT, BITS, 6, PHASED>(s, q, x, y, m, n, k);
  return launch_gs<TT, BITS, 7, PHASED>(s, q, x, y, m, n, k);
}

template <typename TT, bool PHASED>
hipError_t launch_t(hipStream_t s, const QuantArgs& q, const void* x, void* y, int m, int n, int k) {
  switch (q.bits) {
    case 2: return launch_bits<TT, 2, PHASED>(s, q, x, y, m, n, k);
    case 3: return launch_bits<TT, 3, PHASED>(s, q, x, y, m, n, k);
    case 4: return launch_bits<TT, 4, PHASED>(s, q, x, y, m, n, k);
    case 5: return launch_bits<TT, 5, PHASED>(s, q, x, y, m, n, k);
    case 6: return launch_bits<TT, 6, PHASED>(s, q, x, y, m, n, k);
    case 8: return launch_bits<TT, 8, PHASED>(s, q, x, y, m, n, k);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

namespace {

bool decode_takes(const QuantArgs& q, int m, int n, int k, const void* x) {
  // 16 rows of X and of W within the 32-bit ranges of their buffers.
  if (m < 1 || m > 16 || n < 1 || k < 32 || k % 32 != 0 || k > (1 << 25)) return false;
  if (q.gs != 32 && q.gs != 64 && q.gs != 128) return false;
  return ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(q.w)) & 15u) == 0;
}

}  // namespace

bool decode_fits(const QuantArgs& q, int m, int n, int k, const void* x) {
  if (!decode_takes(q, m, n, k, x)) return false;
  int waves, steps;
  decode_split(n, k, &waves, &steps);
  return decode_lds(m, waves, steps) <= 160 * 1024;
}

hipError_t launch_decode(hipStream_t s, const QuantArgs& q, const void* x, void* y, int m, int n, int k) {
  if (!decode_fits(q, m, n, k, x)) return hipErrorInvalidValue;
  if (q.dtype == CPQ_DTYPE_BF16) return launch_t<BF16, false>(s, q, x, y, m, n, k);
  if (q.dtype == CPQ_DTYPE_F16) return launch_t<F16, false>(s, q, x, y, m, n, k);
  return hipErrorInvalidValue;
}

bool decode_phased_fits(const QuantArgs& q, int m, int n, int k, const void* x) {
  return decode_takes(q, m, n, k, x);
}

hipError_t launch_decode_phased(hipStream_t s, const QuantArgs& q, const void* x, void* y, int m, int n, int k) {
  if (!decode_phased_fits(q, m, n, k, x)) return hipErrorInvalidValue;
  if (q.dtype == CPQ_DTYPE_BF16) return launch_t<BF16, true>(s, q, x, y, m, n, k);
  if (q.dtype == CPQ_DTYPE_F16) return launch_t<F16, true>(s, q, x, y, m, n, k);
  return hipErrorInvalidValue;
}

}  // namespace cpq
