// torque_hip.hip -- MI355X (gfx950) kernels and C ABI for the packed rotated
// KV-cache decode path.  Declarations and the reference interfaces each entry
// point replaces are in include/torque_hip.h.
//
// Kernels
//   fwht_kernel          structured Hadamard rotation, one wavefront per row
//   append_kernel        rotate -> quantize -> bit-pack (or dequantize), 16
//                        elements of a row to a lane, packed words written in
//                        place into the [L, Hkv, capacity, W] slab
//   unpack_kernel        packed slab -> dense float32 centroid values
//   decode_kernel<Fmt>   split-K decode attention: each workgroup owns one
//                        (layer, KV head, query-head group) and one split of
//                        the sequence (row blocks dealt out cyclically) and
//                        writes its partial (max, sum, accumulator); with a
//                        single split it finishes the rows itself.  Fmt
//                        selects packed 2/3/4-bit or dense fp16/fp32 rows;
//                        packed rows with groups of 4 query heads run their
//                        products on the matrix cores.
//   merge_kernel         log-sum-exp merge of the splits of one query head
//                        (partials arrive rotated back), current token,
//                        normalisation.
//   score / softmax / accumulate kernels   the three stages of the
//                        reference's split path, for profiling and the op API.

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdio>
#include <mutex>
#include <string>
#include <type_traits>

#include "torque_hip.h"
#include "tq_device.hpp"

using namespace tq;

namespace {

thread_local std::string g_last_error;

int fail(int code, const std::string& msg) {
  g_last_error = msg;
  return code;
}

int launch_status(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TQ_ERR_LAUNCH, std::string(what) + ": " + hipGetErrorString(e));
  g_last_error.clear();
  return TQ_OK;
}

bool valid_bits(int b) { return b == 2 || b == 3 || b == 4; }
bool valid_head_dim(int d) { return d == 64 || d == 128 || d == 256; }

int check_geometry(int head_dim, int bits) {
  if (!valid_head_dim(head_dim))
    return fail(TQ_ERR_UNSUPPORTED, "Unsupported head dimension: " + std::to_string(head_dim));
  if (bits != 0 && !valid_bits(bits)) return fail(TQ_ERR_UNSUPPORTED, "Unsupported bit width: " + std::to_string(bits));
  return TQ_OK;
}

int packed_words(int head_dim, int bits) { return (head_dim * bits + 31) / 32; }

float sqrt_f32(int head_dim) { return static_cast<float>(std::sqrt(static_cast<double>(head_dim))); }

constexpr float kLog2e = 1.4426950408889634f;
// Lazy rescale threshold for the online softmax, in log2 units: the running
// reference maximum is only raised when a score exceeds it by more than this,
// so partial weights stay below 2^8.
constexpr float kRescaleThreshold = 8.0f;
constexpr int kMaxSplits = 256;
constexpr int kTokensPerIter = 2;  // tokens per lane group per loop iteration
constexpr int kWideTokensPerIter = 3;  // the same, in the instances of wide_iter_shape
constexpr int kPrefetchIters = 1;  // loop iterations whose loads are in flight ahead
constexpr int kScoreChains = 2;    // independent score product chains per token (matrix-core mode)
constexpr bool kPhaseFences = true;  // matrix-core mode: no interleaving of products with VALU work

// ============================================================== rotation


template <int D, typename T>
__global__ __launch_bounds__(kBlock) void fwht_kernel(const T* __restrict__ x, float* __restrict__ y, int64_t rows,
                                                      const float* __restrict__ s_first,
                                                      const float* __restrict__ s_second, float sqrt_d) {
  constexpr int E = D / kWave;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;  // whole wavefront exits together
  const int lane = lane_id();
  float v[E];
  const T* src = x + row * D + lane * E;
#pragma unroll
  for (int i = 0; i < E; ++i) v[i] = to_f32(src[i]);
  wave_rotate<D>(v, s_first, s_second, sqrt_d);
  float* dst = y + row * D + lane * E;
#pragma unroll
  for (int i = 0; i < E; ++i) dst[i] = v[i];
}

// ============================================================== append


// Division of a 32-bit row number by the tokens per group, as a multiply-high
// and a shift with constants from the host (d >= 1, n < 2^31): Granlund and
// Montgomery's division by invariant integers.
struct FastDiv {
  uint32_t mul, shift, d;
  __device__ uint32_t quot(uint32_t n) const { return (__umulhi(n, mul) + n) >> shift; }
};
FastDiv make_fast_div(uint32_t d) {
  uint32_t s = 0;
  while ((uint64_t(1) << s) < d) ++s;
  return {static_cast<uint32_t>(((uint64_t(1) << 32) * ((uint64_t(1) << s) - d)) / d + 1), s, d};
}

struct AppendArgs {
  const void* keys;  // [rows, D] per stream, rows (l, h, t) in [L, Hkv, seq_new] order
  const void* values;
  uint32_t rows;
  FastDiv seq_new;
  int rotate_keys, rotate_values;
  int wide;  // sources and outputs 16-byte aligned: vector loads and stores
  const float* signs_left;
  const float* signs_right;
  float sqrt_d;
  const float* key_bnd;
  const float* value_bnd;
  const float* key_cent;
  const float* value_cent;
  uint32_t* key_codes;
  uint32_t* value_codes;
  int64_t capacity, offset;
  float* key_out;
  float* value_out;
  float* key_scales;
  float* value_scales;
};

// Neighbouring floats by their order: key(x) counts the floats below x, with
// both zeros at 0.
__device__ __forceinline__ int float_key(float x) {
  const int i = __float_as_int(x);
  return i >= 0 ? i : INT_MIN - i;
}
__device__ __forceinline__ float key_float(int k) { return __int_as_float(k >= 0 ? k : INT_MIN - k); }

// x / sqrt(D) as wave_rotate_signs rounds it.
template <int D>
__device__ __forceinline__ float div_sqrt_d(float x, float sqrt_d) {
  if constexpr (D == 64) return __fmul_rn(x, 0.125f);
  if constexpr (D == 256) return __fmul_rn(x, 0.0625f);
  return __fdiv_rn(x, sqrt_d);
}

// v[i] += pair * (the partner lane's v[i]) for 16 elements, one operation
// each: the compiler leaves the DPP move and the fma apart.  The two wait
// states in front are what a DPP read needs after a VALU write.
template <int CTRL>
__device__ __forceinline__ void pair_step(float (&v)[16], float pair) {
#define TQ_PAIR(i, mode) "v_fmac_f32_dpp %" #i ", %" #i ", %16 " mode " row_mask:0xf bank_mask:0xf\n\t"
#define TQ_PAIRS(mode)                                                                                             \
  asm("s_nop 1\n\t" TQ_PAIR(0, mode) TQ_PAIR(1, mode) TQ_PAIR(2, mode) TQ_PAIR(3, mode) TQ_PAIR(4, mode)           \
          TQ_PAIR(5, mode) TQ_PAIR(6, mode) TQ_PAIR(7, mode) TQ_PAIR(8, mode) TQ_PAIR(9, mode) TQ_PAIR(10, mode)   \
              TQ_PAIR(11, mode) TQ_PAIR(12, mode) TQ_PAIR(13, mode) TQ_PAIR(14, mode) TQ_PAIR(15, mode)            \
      : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]),            \
        "+v"(v[8]), "+v"(v[9]), "+v"(v[10]), "+v"(v[11]), "+v"(v[12]), "+v"(v[13]), "+v"(v[14]), "+v"(v[15])       \
      : "v"(pair))
  if constexpr (CTRL == kDppXor1) TQ_PAIRS("quad_perm:[1,0,3,2]");
  if constexpr (CTRL == kDppXor2) TQ_PAIRS("quad_perm:[2,3,0,1]");
  if constexpr (CTRL == kDppHalfMirror) TQ_PAIRS("row_half_mirror");
  if constexpr (CTRL == kDppRor8) TQ_PAIRS("row_ror:8");
#undef TQ_PAIRS
#undef TQ_PAIR
}

constexpr int kAppendBuckets = 64;
// Rows (of all streams) up to which append_few_kernel runs: append_kernel's
// tables cost 1.5 to 3 us, its rows less than half.  The lines lie where the
// two cross on MI355X (us, append_few_kernel / append_kernel, rows of two
// streams each).  Packing: head_dim 64, 4-bit 3000 rows 4.3 / 4.4, 4096 4.6 /
// 4.5, 2-bit 3500 4.6 / 4.8, 4096 5.0 / 4.6; 128, 4-bit 2049 4.1 / 4.7, 3000 4.7 /
// 4.8, scaled 2049 4.7 / 4.9; 256, 4-bit 2049 4.8 / 4.8, 2-bit 3000 4.9 / 5.4, 4096
// 5.7 / 5.5.  Writing centroid values: 64, 4-bit 6000 5.0 / 5.5, 8000 5.9 / 5.8,
// 2-bit 34000 12.3 / 13.4; 128, 4-bit 4000 5.7 / 6.3, 3-bit 18000 12.2 / 13.4, 2-bit
// 34000 18.2 / 21.6; 256, 4-bit 2049 5.5 / 6.0, 3-bit 24000 21.3 / 24.8, 2-bit 70000
// 61.2 / 63.7, scaled 24000 21.7 / 24.3.
template <int D, int BITS, bool DEQUANT, bool SCALED>
constexpr int64_t append_few_rows() {
  if (!DEQUANT) {
    if (SCALED || BITS == 3) return (SCALED ? BITS == 4 && D < 256 : D == 64) ? 4608 : 4096;
    return D == 64 ? 7168 : D == 128 ? 6144 : BITS == 2 ? 8192 : 4096;
  }
  if (BITS == 4) return D == 256 ? 5120 : SCALED ? 8192 : 12288;
  if (BITS == 3) return SCALED ? (D == 256 ? 8192 : 12288) : D == 64 ? 20480 : D == 128 ? 40960 : 57344;
  if (SCALED) return D == 256 ? 57344 : 20480;
  return D == 64 ? 81920 : D == 128 ? 98304 : 163840;
}
constexpr int kAppendMaxBlocks = 2048;  // 8 wavefronts per SIMD on 256 CUs: one resident wave of workgroups

// Rotate -> quantize -> pack (or dequantize) rows of one stream (grid y: keys,
// values), D / 16 lanes to a row and 16 elements to a lane.
// SCALED (per-vector scales): the rotated row x is quantized as x / s with
// s = sqrt(mean(x^2)) (1 for a zero row); s is stored at the token's slot of
// the [L, Hkv, capacity] scale slab, or multiplied into the dequantized
// values.
//
// A prompt's append moves 2 D bytes in and D b / 8 out per fp16 row, so the
// work per element has to stay near 20 VALU operations to keep up with HBM.
// Layout: a lane holds the elements 8 l .. 8 l + 7 and D / 2 + 8 l .. of its
// row, l its place among the row's lanes, so a load is 16 contiguous bytes a
// lane, a chunk's 8 codes are one word at 4 bits, and of the transform's
// log2(D) steps the first three and the last stay in registers.  The steps in
// between are one DPP fma each, own + (+-1) other: l = 4..7 sit mirrored (lane
// 7 - l + 4), which makes the step 4 apart a row_half_mirror, and the upper
// lane of a pair keeps the negated difference, right - left.  Its sign is the
// same on both lanes of every later pair and is undone by the second sign
// multiply, so every value is wave_fwht's up to the sign of a zero, which no
// code, mean square or centroid depends on.
// Quantizer: code(x) = #{k : x > b_k}.  The division by sqrt(D) is monotone,
// so x / sqrt(D) > b is x > T with T the largest float whose quotient does
// not exceed b: found once per workgroup, it takes the division (11
// operations at head_dim 128) out of the loop.  Signs other than +-1 take the
// division per element instead.  The thresholds are looked up through
// kAppendBuckets affine buckets of x: with at most one threshold to a bucket,
// code = (thresholds in lower buckets) + (x > the bucket's own), one 8-byte
// LDS read and 5 operations against 30 for 15 comparisons; a rounded affine
// map is monotone, so the count is exact for every x.  Codebooks that put two
// thresholds into one bucket are counted one threshold at a time.
// Measured: 24 x 8 x 8192 fp16 tokens at head_dim 128, 4-bit (1.0 GB read and
// written): 230 us, 4.3 TB/s, against 1160 us for a wavefront per row
// (append_few_kernel); 4 x 8 x 4096 float32 tokens 27 us, 5.5 TB/s (a large
// device copy reaches 5.1).  fp16 rows are bound by the 15 operations an
// element, float32 rows by memory.  With per-vector scales the two divisions
// an element remain (2.1 to 2.8 TB/s for fp16).
template <int D, int BITS, typename T, bool DEQUANT, bool SCALED>
__global__ __launch_bounds__(kBlock) void append_kernel(const AppendArgs a) {
  constexpr int LPR = D / 16;           // lanes per row: 4, 8, 16
  constexpr int RPW = kWave / LPR;      // rows per wavefront
  constexpr int RPB = RPW * kWavesPerBlock;
  constexpr int W = D * BITS / 32;
  constexpr int NL = (1 << BITS) - 1;   // thresholds
  constexpr int NB = kAppendBuckets;
  __shared__ float s_thr[NL];
  __shared__ int s_at[NL];              // bucket of each threshold
  __shared__ float2 s_bucket[NB];       // (threshold or +inf, code below it)
  __shared__ float s_cent[NL + 1];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
  const bool is_v = blockIdx.y != 0;
  const bool rotate = (is_v ? a.rotate_values : a.rotate_keys) != 0;
  const float* bnd = is_v ? a.value_bnd : a.key_bnd;

  // this lane's place among its row's lanes
  const int pl = lane & (LPR - 1);
  const int l = LPR >= 8 && (pl & 4) ? (pl & 8) + 11 - (pl & 7) : pl;
  auto dim = [&](int i) { return (i >> 3) * (D / 2) + 8 * l + (i & 7); };  // element i of 16
  float sg_first[16], sg_second[16];
  bool unit = true;  // signs are +-1
  if (rotate) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      sg_first[i] = a.signs_right[dim(i)];
      sg_second[i] = a.signs_left[dim(i)];
      unit = unit && fabsf(sg_second[i]) == 1.f;
      if (__builtin_popcount(l) & 1) sg_second[i] = -sg_second[i];  // an odd number of negated differences
    }
  }
  // Thresholds apply to the undivided transform (`folded`) or to the rotated
  // value itself.
  const bool folded = !SCALED && rotate && __syncthreads_and(unit) != 0;
  if (tid < NL) {
    const float b = bnd[tid];
    float t = b == b ? b : INFINITY;  // nothing exceeds a NaN boundary
    if (folded && fabsf(t) < INFINITY) {
      int k = float_key(t * a.sqrt_d);
      while (k < float_key(INFINITY) && div_sqrt_d<D>(key_float(k + 1), a.sqrt_d) <= t) ++k;
      while (div_sqrt_d<D>(key_float(k), a.sqrt_d) > t) --k;
      t = key_float(k);
    }
    s_thr[tid] = t;
  }
  if (DEQUANT && tid <= NL) s_cent[tid] = (is_v ? a.value_cent : a.key_cent)[tid];
  __syncthreads();
  float lo = s_thr[0], hi = s_thr[0];
#pragma unroll
  for (int k = 1; k < NL; ++k) {
    lo = fminf(lo, s_thr[k]);
    hi = fmaxf(hi, s_thr[k]);
  }
  // bucket(x): an affine map rounded to an integer by adding 2^23, whose
  // mantissa then holds it
  constexpr float kInt = 8388608.f;
  const float slope = (NB - 2) / (hi - lo), shift = fmaf(-lo, slope, kInt + 1.f);
  auto bucket = [&](float x) {
    return __float_as_uint(fminf(fmaxf(fmaf(x, slope, shift), kInt), kInt + (NB - 1))) - 0x4B000000u;
  };
  const bool affine = fabsf(slope) < INFINITY && fabsf(shift) < INFINITY;  // uniform
  if (affine && tid < NL) s_at[tid] = static_cast<int>(bucket(s_thr[tid]));
  __syncthreads();
  bool single = affine;  // at most one threshold to a bucket
  if (affine && tid < NB) {
    int below = 0, own = 0;
    float t = INFINITY;
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      below += s_at[k] < tid;
      own += s_at[k] == tid;
      if (s_at[k] == tid) t = s_thr[k];
    }
    s_bucket[tid] = make_float2(t, __int_as_float(below));
    single = own <= 1;
  }
  const bool lookup = __syncthreads_and(single) != 0;

  const T* src = static_cast<const T*>(is_v ? a.values : a.keys);
  uint32_t* codes = is_v ? a.value_codes : a.key_codes;
  float* scales = is_v ? a.value_scales : a.key_scales;
  float* out = is_v ? a.value_out : a.key_out;
  // the partner's sign in each step between lanes
  const float pair1 = (l & 1) ? -1.f : 1.f, pair2 = (l & 2) ? -1.f : 1.f;
  const float pair4 = (l & 4) ? -1.f : 1.f, pair8 = (l & 8) ? -1.f : 1.f;

  for (uint32_t r0 = blockIdx.x * RPB; r0 < a.rows; r0 += gridDim.x * RPB) {
    const uint32_t mine = r0 + wave * RPW + lane / LPR;
    const uint32_t r = min(mine, a.rows - 1);  // lanes past the end repeat the last row and store nothing
    alignas(16) T e[16];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const T* p = src + static_cast<int64_t>(r) * D + c * (D / 2) + 8 * l;
      if (a.wide) {
#pragma unroll
        for (int q = 0; q < static_cast<int>(sizeof(T) / 2); ++q)
          reinterpret_cast<uint4*>(e + 8 * c)[q] = reinterpret_cast<const uint4*>(p)[q];
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) e[8 * c + i] = p[i];
      }
    }
    float v[16];
    if (!rotate) {
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = to_f32(e[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = fmaf(to_f32(e[i]), sg_first[i], -0.f);  // the product, in one operation from fp16
#pragma unroll
      for (int st = 1; st < 8; st <<= 1)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if ((i & st) == 0) {
            const float x = v[i], y = v[i + st];
            v[i] = __fadd_rn(x, y);
            v[i + st] = __fsub_rn(x, y);
          }
      pair_step<kDppXor1>(v, pair1);
      pair_step<kDppXor2>(v, pair2);
      if constexpr (LPR >= 8) pair_step<kDppHalfMirror>(v, pair4);
      if constexpr (LPR >= 16) pair_step<kDppRor8>(v, pair8);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float x = v[i], y = v[i + 8];
        v[i] = __fadd_rn(x, y);
        v[i + 8] = __fsub_rn(x, y);
      }
      if (!folded) {
        asm volatile("");  // keeps this a branch: the compiler would divide always and select
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = div_sqrt_d<D>(v[i], a.sqrt_d);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = __fmul_rn(v[i], sg_second[i]);
    }
    float scale = 1.f;
    if constexpr (SCALED) {
      // mean square in the order of a wavefront's lanes holding D / 64
      // consecutive elements each: a chain over those, then pairs
      constexpr int E = D / kWave;
      float ss[16 / E];
#pragma unroll
      for (int j = 0; j < 16 / E; ++j) {
        ss[j] = 0.f;
#pragma unroll
        for (int i = 0; i < E; ++i) ss[j] = fmaf(v[j * E + i], v[j * E + i], ss[j]);
      }
      constexpr int H = 8 / E;  // partial sums per chunk
#pragma unroll
      for (int st = 1; st < H; st <<= 1)
#pragma unroll
        for (int j = 0; j < 2 * H; j += 2 * st) ss[j] += ss[j + st];
      float s0 = ss[0], s1 = ss[H];
      s0 = group_sum<LPR>(s0);  // pairs, quads, 8 and 16 lanes: l's bits in order
      s1 = group_sum<LPR>(s1);
      const float rms = sqrtf((s0 + s1) / static_cast<float>(D));
      scale = rms > 0.f ? rms : 1.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = v[i] / scale;
    }
    uint32_t code[16];
    if (lookup) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float2 e = s_bucket[bucket(v[i])];
        code[i] = __float_as_uint(e.y) + (v[i] > e.x ? 1u : 0u);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) code[i] = 0;
      for (int k = 0; k < NL; ++k) {
        const float t = s_thr[k];
#pragma unroll
        for (int i = 0; i < 16; ++i) code[i] += v[i] > t ? 1u : 0u;
      }
    }
    const bool active = mine < a.rows;
    if constexpr (DEQUANT) {
      if (active) {
        float* row = out + static_cast<int64_t>(r) * D;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          float* p = row + c * (D / 2) + 8 * l;
          float e[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) e[i] = SCALED ? s_cent[code[8 * c + i]] * scale : s_cent[code[8 * c + i]];
          if (a.wide) {
            reinterpret_cast<float4*>(p)[0] = make_float4(e[0], e[1], e[2], e[3]);
            reinterpret_cast<float4*>(p)[1] = make_float4(e[4], e[5], e[6], e[7]);
          } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) p[i] = e[i];
          }
        }
      }
    } else {
      uint32_t chunk[2];  // 8 codes: 8 * BITS bits
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        uint32_t w = code[8 * c];
#pragma unroll
        for (int i = 1; i < 8; ++i) w |= code[8 * c + i] << (BITS * i);
        chunk[c] = w;
      }
      const uint32_t lh = a.seq_new.quot(r), t = r - lh * a.seq_new.d;
      const int64_t slot = static_cast<int64_t>(lh) * a.capacity + a.offset + t;
      uint32_t* dst = codes + slot * W;
      if constexpr (BITS == 4) {
        if (active) {
          dst[l] = chunk[0];
          dst[W / 2 + l] = chunk[1];
        }
      } else {
        // the chunk of the next place, l + 1: lane + 1, or lane - 1 in the mirrored half
        auto next = [&](uint32_t x) {
          const int y = static_cast<int>(x);
          const int above = __builtin_amdgcn_mov_dpp(y, 0xF9, 0xF, 0xF, true);   // quad_perm [1,2,3,3]
          if constexpr (LPR < 8) return static_cast<uint32_t>(above);
          const int below = __builtin_amdgcn_mov_dpp(y, 0x90, 0xF, 0xF, true);   // quad_perm [0,0,1,2]
          return static_cast<uint32_t>((l & 4) ? below : above);
        };
        const uint32_t n0 = next(chunk[0]), n1 = next(chunk[1]);
        if constexpr (BITS == 3) {
          // four chunks of 24 bits are three words
          const int j = l & 3, w = 3 * (l >> 2) + j;
          if (active && j < 3) {
            dst[w] = (chunk[0] >> (8 * j)) | (n0 << (24 - 8 * j));
            dst[W / 2 + w] = (chunk[1] >> (8 * j)) | (n1 << (24 - 8 * j));
          }
        } else {
          if (active && (l & 1) == 0) {
            dst[l >> 1] = chunk[0] | (n0 << 16);
            dst[W / 2 + (l >> 1)] = chunk[1] | (n1 << 16);
          }
        }
      }
      if (SCALED && active && l == 0) scales[slot] = scale;
    }
  }
}

// The same for a few rows (append_few_rows): one wavefront per row, D / 64
// elements to a lane, codes counted one boundary at a time and packed through
// LDS.  It has no tables to set up: one token x 4 heads at head_dim 256 takes
// 2.9 us against append_kernel's 4.3, 64 tokens x 8 heads at 64 3.4 against
// 5.0, but 512 x 8 at 128 5.8 against 5.6 and 1999 x 4 at 64 8.1 against 5.0.
template <int D, int BITS, typename T, bool DEQUANT, bool SCALED>
__global__ __launch_bounds__(kBlock) void append_few_kernel(const AppendArgs a) {
  constexpr int E = D / kWave;
  constexpr int W = D * BITS / 32;
  __shared__ uint8_t s_codes[kWavesPerBlock][D];
  const int wave = threadIdx.x >> 6, lane = lane_id();
  const uint32_t r = blockIdx.x * kWavesPerBlock + wave;
  const bool active = r < a.rows;
  const bool is_v = blockIdx.y != 0;
  float scale = 1.f;  // per-vector scale (SCALED)
  if (active) {
    const T* src = static_cast<const T*>(is_v ? a.values : a.keys) + static_cast<int64_t>(r) * D + lane * E;
    float v[E];
#pragma unroll
    for (int i = 0; i < E; ++i) v[i] = to_f32(src[i]);
    if (is_v ? a.rotate_values : a.rotate_keys) wave_rotate<D>(v, a.signs_right, a.signs_left, a.sqrt_d);
    const float* bnd = is_v ? a.value_bnd : a.key_bnd;
    if constexpr (SCALED) {
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < E; ++i) ss = fmaf(v[i], v[i], ss);
      ss = group_sum<kWave>(ss);
      const float rms = sqrtf(ss / static_cast<float>(D));
      scale = rms > 0.f ? rms : 1.f;
#pragma unroll
      for (int i = 0; i < E; ++i) v[i] = v[i] / scale;
    }
    if constexpr (DEQUANT) {
      const float* cent = is_v ? a.value_cent : a.key_cent;
      float* dst = (is_v ? a.value_out : a.key_out) + static_cast<int64_t>(r) * D + lane * E;
      // every load before the first store, which might alias the tables
#pragma unroll
      for (int i = 0; i < E; ++i) {
        v[i] = cent[quantize_count<BITS>(v[i], bnd)];
        if (SCALED) v[i] = v[i] * scale;
      }
#pragma unroll
      for (int i = 0; i < E; ++i) dst[i] = v[i];
    } else {
#pragma unroll
      for (int i = 0; i < E; ++i) s_codes[wave][lane * E + i] = static_cast<uint8_t>(quantize_count<BITS>(v[i], bnd));
    }
  }
  if constexpr (!DEQUANT) {
    __syncthreads();
    if (active && lane < W) {
      const uint32_t word = pack_word<BITS, D>(s_codes[wave], lane);
      const uint32_t lh = a.seq_new.quot(r), t = r - lh * a.seq_new.d;
      const int64_t slot = static_cast<int64_t>(lh) * a.capacity + a.offset + t;
      (is_v ? a.value_codes : a.key_codes)[slot * W + lane] = word;
      if (SCALED && lane == 0) (is_v ? a.value_scales : a.key_scales)[slot] = scale;
    }
  }
}

// ============================================================== unpack


// scales (or null): per-token scale slab [groups, capacity] multiplied in.
template <int BITS>
__global__ __launch_bounds__(kBlock) void unpack_kernel(const uint32_t* __restrict__ codes, int64_t groups,
                                                        int64_t capacity, int64_t seq_len, int head_dim,
                                                        const float* __restrict__ cent,
                                                        const float* __restrict__ scales, float* __restrict__ out) {
  const int W = head_dim * BITS / 32;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  const int64_t total = groups * seq_len * head_dim;
  if (idx >= total) return;
  const int d = static_cast<int>(idx % head_dim);
  const int64_t tok = idx / head_dim;
  const int64_t g = tok / seq_len, t = tok - g * seq_len;
  const uint32_t* row = codes + (g * capacity + t) * W;
  const float c = cent[unpack_code<BITS>(row, d)];
  out[idx] = scales != nullptr ? c * scales[g * capacity + t] : c;
}

// ============================================================== decode


struct DecodeArgs {
  const void* q;
  int q_f16;
  const uint8_t* k;  // slab [L, Hkv, cap, row_bytes]
  const uint8_t* v;
  int64_t cap;
  int64_t seq_len;
  int num_layers, query_heads, kv_heads, group, n_hgroups;
  const float* cent_k;
  const float* cent_v;
  const float* signs_left;
  const float* signs_right;
  float sqrt_d;
  float q_scale;  // log2(e) / sqrt(D): scores come out in log2 units
  int rotate_query, inverse_output;
  // Append mode (new_k != null): the token new_k/new_v [L, Hkv, D] (float16
  // when new_f16, else float32) is rotated, quantized and packed into the
  // slabs at row seq_len by the split-0 workgroups, and joins the softmax as
  // the current token.
  const void* new_k;
  const void* new_v;
  int new_f16;
  const float* bnd_k;
  const float* bnd_v;
  uint32_t* k_slab;
  uint32_t* v_slab;
  int rotate_new_k, rotate_new_v;
  const float* cur_k;  // [L, Hkv, D] or null
  const float* cur_v;
  int n_splits;
  // Splits that read rows: n_splits, or in append mode n_splits - 1 when
  // split 0 (which also packs the new token) takes no rows and the others
  // cover every block with no more blocks each than a deal over all splits.
  int row_splits;
  float* ws_ml;   // [L * Hq, n_splits, 2]  (max, sum) of each split, log2 units
  float* ws_acc;  // [L * Hq, n_splits, D]  value accumulator of each split
  float* ws_cur_s; // [L * Hq]              score of the current token (log2 units)
  float* ws_cur_v; // [L * Hkv, D]          current token's value, rotated back when requested
  float* out;     // [L, Hq, D]
  // Per-vector scales (SCALED kernels): [L, Hkv, cap] float32 per stream; a
  // token's score is multiplied by its key scale, its value by its value
  // scale.
  const float* k_scales;
  const float* v_scales;
  int wide_iter;  // host side only: launch the kWideTokensPerIter instance
};

// Finish one output row held by a wavefront: optional extra dense token
// (decode-with-current), normalisation, optional inverse rotation, store.
// A[D]: accumulator relative to max M (log2 units), L: softmax sum.
template <int D>
__device__ __forceinline__ void finish_row(const float* A, float M, float L, const float* qs, const float* ck,
                                           const float* cv, int inverse, const float (&sg_left)[D / kWave],
                                           const float (&sg_right)[D / kWave], float sqrt_d, float* dst) {
  constexpr int E = D / kWave;
  const int lane = lane_id();
  float e[E];
#pragma unroll
  for (int i = 0; i < E; ++i) e[i] = A[lane * E + i];
  if (ck != nullptr) {
    float dot = 0.f;
#pragma unroll
    for (int i = 0; i < E; ++i) dot = fmaf(qs[lane * E + i], ck[lane * E + i], dot);
    dot = group_sum<kWave>(dot);
    const float mn = fmaxf(M, dot);
    const float f_old = L > 0.f ? fast_exp2(M - mn) : 0.f;
    const float f_cur = fast_exp2(dot - mn);
#pragma unroll
    for (int i = 0; i < E; ++i) e[i] = e[i] * f_old + cv[lane * E + i] * f_cur;
    L = L * f_old + f_cur;
  }
#pragma unroll
  for (int i = 0; i < E; ++i) e[i] = L > 0.f ? e[i] / L : 0.f;
  if (inverse) wave_rotate_signs<D>(e, sg_left, sg_right, sqrt_d);
#pragma unroll
  for (int i = 0; i < E; ++i) dst[lane * E + i] = e[i];
}

// One reduce-scatter step over lane pairs (i, i xor LM): the lower lane of a
// pair gets x_i + x_partner, the upper lane y_i + y_partner.
template <int LM>
__device__ __forceinline__ float scatter_pair(float x, float y, int lane) {
  if constexpr (LM == 16 || LM == 32) {
    const LanePair r = permlane_swap<LM>(x, y);
    return r.first + r.second;
  } else if constexpr (LM == 8) {
    const float sx = x + dpp_move<kDppRor8>(x);
    const float sy = y + dpp_move<kDppRor8>(y);
    return (lane & 8) ? sy : sx;
  } else {
    const bool upper = (lane & LM) != 0;
    const float send = upper ? x : y;
    const float keep = upper ? y : x;
    return keep + xor_partner<LM>(send, lane);
  }
}

// Reduce-scatter of buf[0, 2*LEN) over the lanes that differ in lane bits
// LM, LM/2, ..., LO (one step per bit, highest first): each step halves the
// live length, the upper lane of a pair keeping the upper half.  Afterwards a
// lane holds, summed over its partners, the chunk of the original buffer that
// its lane bits LO..LM select (bit LM weighs half the buffer).
template <int LO, int LM, int LEN, int NV>
__device__ __forceinline__ void reduce_scatter(float (&buf)[NV], int lane) {
#pragma unroll
  for (int k = 0; k < LEN; ++k) buf[k] = scatter_pair<LM>(buf[k], buf[k + LEN], lane);
  if constexpr (LM > LO) reduce_scatter<LO, LM / 2, LEN / 2, NV>(buf, lane);
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Matrix-core score products leave on lane l, register i, the partial score
// of token 4 * ((l / 4) / LPT) + i over slice (l / 4) % LPT.  Sum over the
// LPT slices (lane bits 2 .. 2 + log2(LPT) - 1) and keep on lane l the token
// of its value layout, l / LPT, i.e. register (l / LPT) % 4: a reduce-scatter
// over lane bits log2(LPT) + 1 and log2(LPT) (which select that register)
// and an all-reduce over the slice bits below them.
template <int LPT>
__device__ __forceinline__ float slice_sum_select(f32x4 c, int lane) {
  static_assert(LPT == 4 || LPT == 8 || LPT == 16, "4, 8 or 16 slices per token");
  float buf[4] = {c[0], c[1], c[2], c[3]};
  reduce_scatter<LPT, 2 * LPT, 2, 4>(buf, lane);
  float v = buf[0];
  if constexpr (LPT >= 8) v += xor_partner<4>(v, lane);
  if constexpr (LPT >= 16) v += xor_partner<8>(v, lane);
  return v;
}

// U: tokens per lane group per loop iteration -- kTokensPerIter, or
// kWideTokensPerIter in the instances wide_iter_instance() names.
template <class Fmt, int D, int HG, bool QF16, bool SCALED, int U = kTokensPerIter>
__global__ __launch_bounds__(kBlock, 2) void decode_kernel(const DecodeArgs a) {
  constexpr int SD = Fmt::kSliceDims;
  constexpr int LPT = D / SD;        // lanes per token
  constexpr int TPW = kWave / LPT;   // tokens (lane groups) per wavefront
  constexpr int TPB = kWavesPerBlock * TPW;
  constexpr int PF = kPrefetchIters;
  constexpr int NB = PF + 1;         // ring of iteration slots
  constexpr int STRIDE = U * TPB;    // tokens per workgroup iteration
  constexpr int E = D / kWave;
  constexpr int ROW = Fmt::template row_bytes<D>();
  constexpr int NV = HG * SD;        // accumulator values per lane
  using Raw = typename Fmt::Raw;

  __shared__ typename Fmt::LutT s_lut[2][Fmt::kLutEntries];
  __shared__ float s_q[HG][D];
  __shared__ float s_red[kWavesPerBlock][HG * D];
  __shared__ float s_mw[kWavesPerBlock][HG];
  __shared__ float s_lw[kWavesPerBlock][HG];
  // append mode: the new token's dequantized rotated key / value, and its codes
  __shared__ float s_cur[2][Fmt::kHasLut ? D : 1];
  __shared__ uint8_t s_codes[2][Fmt::kHasLut ? D : 1];

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & (kWave - 1);
  const int gi = lane / LPT, slice = lane % LPT;

  // ---- work item.  Consecutive workgroup ids land on different XCDs
  // (round robin over 8); remap so the splits of one head group are
  // dispatched to the same XCD and share its L2.  XCD x receives the ids
  // x, x + 8, ...: nblk / 8 of them, one more for x < nblk % 8, and takes
  // that many consecutive work items starting at x (nblk / 8) + min(x,
  // nblk % 8), so every work item is taken exactly once for any nblk
  // (3 head groups x 170 splits: float32-kernel median 12.4-12.6 ->
  // 12.0-12.1 us against the remap only for multiples of 8).
  const int units = a.num_layers * a.kv_heads * a.n_hgroups;
  const int64_t nblk = static_cast<int64_t>(units) * a.n_splits;
  int64_t g = blockIdx.x;
  g = (g & 7) * (nblk >> 3) + min(g & 7, nblk & 7) + (g >> 3);
  const int unit = static_cast<int>(g / a.n_splits);
  const int split = static_cast<int>(g - static_cast<int64_t>(unit) * a.n_splits);
  const int lkv = unit / a.n_hgroups;
  const int hg = unit - lkv * a.n_hgroups;
  const int layer = lkv / a.kv_heads, kvh = lkv - layer * a.kv_heads;
  const int qh0 = kvh * a.group + hg * HG;
  // Query heads of this head group: fewer than HG in the last one of a group
  // that is no multiple of 4.  The missing heads' slots repeat the last head
  // and are not stored.
  const int heads = min(HG, a.group - hg * HG);

  // ---- tokens of this wavefront.  The sequence is cut into blocks of
  // STRIDE rows (one workgroup iteration) dealt out cyclically: split s takes
  // blocks s, s + n_splits, s + 2 n_splits, ..., so at any moment the splits
  // of a head group read neighbouring blocks (one contiguous window of
  // n_splits blocks per stream) rather than n_splits separate streams, which
  // keeps HBM rows open (measured: main loop 10.0 -> 9.0 us at M).  In
  // iteration i, lane group gi takes tokens first + gi + u * TPB + i * BSTRIDE
  // (u < U): one wavefront load covers TPW consecutive rows.  Token offsets
  // are 32-bit (the host keeps capacity * ROW below 2^31).  Every block but
  // the sequence's last is full.
  //
  // In append mode split 0 also quantizes the new token and finishes its
  // score and value, which sets the kernel's end when it reads rows too.  So
  // the rows go to splits 1.. only (deal index split - 1 over row_splits =
  // n_splits - 1) where that gives no split more blocks than a deal over
  // all of them, and split 0 deals past the last block; otherwise split 0
  // takes the lightest share (the one split n_splits - 1 would take) and
  // splits 1.. the shares of splits 0.. (24-layer 8K decode loop at 64
  // splits: 320 -> 289 us per step for the lightest share, 274 -> 249 for
  // none).
  const int t1 = static_cast<int>(a.seq_len);
  const int n_blocks = (t1 + STRIDE - 1) / STRIDE;
  const bool app_deal = Fmt::kHasLut && a.new_k != nullptr;
  const int row_splits = app_deal ? a.row_splits : a.n_splits;  // splits that read rows
  const int deal = !app_deal ? split : split > 0 ? split - 1 : row_splits < a.n_splits ? n_blocks : a.n_splits - 1;
  const int64_t t0 = static_cast<int64_t>(deal) * STRIDE;
  const int BSTRIDE = row_splits * STRIDE;
  const int first = static_cast<int>(t0) + wave * TPW;
  const int n_iter = deal < n_blocks ? (n_blocks - deal + row_splits - 1) / row_splits : 0;  // uniform per workgroup
  const uint8_t* kbase = a.k + static_cast<int64_t>(lkv) * a.cap * ROW;
  const uint8_t* vbase = a.v + static_cast<int64_t>(lkv) * a.cap * ROW;

  // Iteration i reads through buffer resources over rows
  // [t0 + i * STRIDE, t1): the workgroup-uniform part of a row's offset sits
  // in the resource base (scalar arithmetic), the lane's part in a fixed
  // per-token offset, and rows past the end of the split read as zeros and
  // are masked out when processed, so loads need no clamp and no branch.
  //
  // Matrix-core mode (packed rows, groups of 4 query heads): scores and value
  // updates run as 4x4x1 fp32 outer products (v_mfma_f32_4x4x1_16b_f32, 16
  // blocks of 4 lanes; block b = lanes 4b..4b+3, output element (i, j) of a
  // block in register i of lane 4b + j, A operand of row i from lane 4b + i,
  // B operand of column j from lane 4b + j).  Key rows are then read in a
  // second lane layout: a lane quad holds 4 consecutive tokens of one slice
  // (lane l: token 4 * ((l / 4) / LPT) + l % 4, slice (l / 4) % LPT), so one
  // product per slice dimension gives 4 tokens x 4 heads of partial scores.
  // Value rows keep the token-major layout (lane l: token l / LPT, slice
  // l % LPT), where a quad holds 4 slices of one token and one product per
  // slice dimension adds weight(head i) x value(dim of lane j).
  constexpr bool kMfma = Fmt::kHasLut && HG == 4;
  const int tk = kMfma ? 4 * ((lane >> 2) / LPT) + (lane & 3) : gi;
  const int sk = kMfma ? (lane >> 2) % LPT : slice;
  int lane_off_k[U], lane_off_v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    lane_off_k[u] = (wave * TPW + u * TPB + tk) * ROW + Fmt::slice_offset(sk);
    lane_off_v[u] = (wave * TPW + u * TPB + gi) * ROW + Fmt::slice_offset(slice);
  }
  // Every iteration's loads are issued unconditionally -- an iteration past
  // the end of the split gets an empty range and reads zeros without touching
  // memory -- so the compiler can count the loads in flight and wait only for
  // the iteration being processed, not for the prefetched ones.
  auto iter_rsrc = [&](const uint8_t* base, int i) {
    const int64_t row0 = min(t0 + static_cast<int64_t>(i) * BSTRIDE, static_cast<int64_t>(t1));
    return make_rsrc(base + row0 * ROW, static_cast<uint32_t>(t1 - row0) * ROW);
  };
  auto load_k = [&](int i, Raw (&kr)[U]) {
    const BufferRsrc rk = iter_rsrc(kbase, i);
#pragma unroll
    for (int u = 0; u < U; ++u) kr[u] = Fmt::load(rk, lane_off_k[u]);
  };
  auto load_v = [&](int i, Raw (&vr)[U]) {
    const BufferRsrc rv = iter_rsrc(vbase, i);
#pragma unroll
    for (int u = 0; u < U; ++u) vr[u] = Fmt::load(rv, lane_off_v[u]);
  };
  // Scaled mode: the key and value scales of the lane's value tokens
  // (lane group gi), loaded with the rows they belong to.
  const float* ksbase = SCALED ? a.k_scales + static_cast<int64_t>(lkv) * a.cap : nullptr;
  const float* vsbase = SCALED ? a.v_scales + static_cast<int64_t>(lkv) * a.cap : nullptr;
  auto load_scales = [&](int i, float (&ks)[U], float (&vs)[U]) {
    const int64_t row0 = min(t0 + static_cast<int64_t>(i) * BSTRIDE, static_cast<int64_t>(t1));
    const uint32_t bytes = static_cast<uint32_t>(t1 - row0) * 4u;
    const BufferRsrc rk = make_rsrc(ksbase + row0, bytes), rv = make_rsrc(vsbase + row0, bytes);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int off = (wave * TPW + u * TPB + gi) * 4;
      ks[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rk, off, 0, kRowLoadPolicy));
      vs[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rv, off, 0, kRowLoadPolicy));
    }
  };
  auto load_iter = [&](int i, Raw (&kr)[U], Raw (&vr)[U], float (&ks)[U], float (&vs)[U]) {
    load_k(i, kr);
    load_v(i, vr);
    if constexpr (SCALED) load_scales(i, ks, vs);
  };

  // ---- set-up loads first: this thread's centroid-table entry, the query
  // row and its rotation signs.  Loads complete in order, so waiting for
  // these below does not wait for the K/V rows requested after them.
  typename Fmt::LutT lut_kv[2];
  if constexpr (Fmt::kHasLut) {
    static_assert(Fmt::kLutEntries <= kBlock, "one table entry per thread");
    if (tid < Fmt::kLutEntries) {
      lut_kv[0] = Fmt::lut_entry(tid, a.cent_k);
      lut_kv[1] = Fmt::lut_entry(tid, a.cent_v);
    }
  }
  // Append mode: the split-0 workgroups quantize the new token (wavefront 0
  // the key, 1 the value) while their first K/V rows are in flight.
  const bool appending = Fmt::kHasLut && a.new_k != nullptr;
  const bool appender = appending && split == 0 && wave < 2;
  constexpr int kLevels = Fmt::kHasLut ? (1 << Fmt::kBits) - 1 : 1;
  float tok[E], bnd[kLevels];
  if (appender) {
    const int64_t toff = static_cast<int64_t>(lkv) * D + lane * E;
    const void* src = wave == 0 ? a.new_k : a.new_v;
#pragma unroll
    for (int i = 0; i < E; ++i)
      tok[i] = a.new_f16 ? __half2float(static_cast<const __half*>(src)[toff + i]) : static_cast<const float*>(src)[toff + i];
    const float* b = wave == 0 ? a.bnd_k : a.bnd_v;
#pragma unroll
    for (int k = 0; k < kLevels; ++k) bnd[k] = b[k];
  }

  // Query bits are loaded raw and converted after the K/V requests below, so
  // the conversion does not hold those requests back.
  // A lane's query values as raw 32-bit words: E floats, or (E + 1) / 2 words
  // of fp16 pairs.
  float qe[E], sg_first[E], sg_second[E];
  uint32_t qw[E];
  if (wave < HG) {
    const int64_t qoff = (static_cast<int64_t>(layer) * a.query_heads + qh0 + min(wave, heads - 1)) * D + lane * E;
    if constexpr (!QF16) {
      const uint32_t* q = static_cast<const uint32_t*>(a.q) + qoff;
#pragma unroll
      for (int i = 0; i < E; ++i) qw[i] = q[i];
    } else if constexpr (E == 1) {
      qw[0] = static_cast<const unsigned short*>(a.q)[qoff];
    } else {
      const uint32_t* q = reinterpret_cast<const uint32_t*>(static_cast<const unsigned short*>(a.q) + qoff);
#pragma unroll
      for (int i = 0; i < E / 2; ++i) qw[i] = q[i];
    }
  }
  // Signs are kept in registers: the query rotation uses (right, left), the
  // inverse rotation of the result (left, right).
  if ((wave < HG && (a.rotate_query || a.inverse_output)) || appender) {
#pragma unroll
    for (int i = 0; i < E; ++i) {
      sg_first[i] = a.signs_right[lane * E + i];
      sg_second[i] = a.signs_left[lane * E + i];
    }
  }

  // Software pipeline over a ring of NB = PF + 1 iteration slots: the loads of
  // iteration i + PF are in flight while iteration i is processed.  The first
  // PF iterations are requested here, so their latency overlaps the set-up.
  Raw kr[NB][U], vr[NB][U];
  float ksr[NB][U], vsr[NB][U];  // scaled mode only
#pragma unroll
  for (int j = 0; j < PF; ++j) load_iter(j, kr[j], vr[j], ksr[j], vsr[j]);

  // ---- centroid tables
  if constexpr (Fmt::kHasLut) {
    if (tid < Fmt::kLutEntries) {
      s_lut[0][tid] = lut_kv[0];
      s_lut[1][tid] = lut_kv[1];
    }
  }

  // ---- append mode: rotate (as on append) and quantize the new token.
  if constexpr (Fmt::kHasLut) {
    if (appender) {
      if (wave == 1 ? a.rotate_new_v : a.rotate_new_k) wave_rotate_signs<D>(tok, sg_first, sg_second, a.sqrt_d);
#pragma unroll
      for (int i = 0; i < E; ++i) s_codes[wave][lane * E + i] = static_cast<uint8_t>(quantize_count<Fmt::kBits>(tok[i], bnd));
    }
  }

  // ---- queries: optional rotation (bit-identical to the reference), then
  // the softmax scale and log2(e) folded in, so scores are in log2 units.
  if (wave < HG) {
#pragma unroll
    for (int i = 0; i < E; ++i)
      qe[i] = QF16 ? __half2float(__ushort_as_half(static_cast<unsigned short>(qw[i / 2] >> (16 * (i % 2)))))
                   : __builtin_bit_cast(float, qw[i]);
    if (a.rotate_query) wave_rotate_signs<D>(qe, sg_first, sg_second, a.sqrt_d);
#pragma unroll
    for (int i = 0; i < E; ++i) s_q[wave][lane * E + i] = qe[i] * a.q_scale;
  }
  lds_barrier();  // LDS-only exchange: the prefetched rows stay in flight
  if constexpr (Fmt::kHasLut) {
    if (appender) {
      // Dequantized values through the centroid table (entry c holds centroid
      // c first); one head group writes the packed words (all compute them).
#pragma unroll
      for (int i = 0; i < E; ++i) s_cur[wave][lane * E + i] = Fmt::first_centroid(s_lut[wave][s_codes[wave][lane * E + i]]);
      constexpr int W = D * Fmt::kBits / 32;
      if (hg == 0 && lane < W) {
        uint32_t* dst = (wave == 0 ? a.k_slab : a.v_slab) + (static_cast<int64_t>(lkv) * a.cap + a.seq_len) * W + lane;
        *dst = pack_word<Fmt::kBits, D>(s_codes[wave], lane);
      }
    }
  }

  // ---- head slots.  With HG == 4 the softmax runs in quad mode
  // (see process): the lane at quad position q4 owns head q4 ^ slot_x -- it
  // sums that head's score, exponentiates it and keeps its softmax sum -- and
  // its per-head registers (query slice, accumulators, running maxima) hold,
  // in slot r, head ((q4 + r) & 3) ^ slot_x.  With that rotation the lane
  // that owns a head is reached by one fixed quad_perm rotation per slot, so
  // the quad reduction and the weight broadcast need no selects; slot_x = 3
  // in the odd quads of a token's lanes makes the row_half_mirror / row_mirror
  // partners (quad position p <-> 3 - p) own the same head.  Other modes use
  // slot r = head r.
  constexpr bool kQuad = HG == 4 && !kMfma;
  const int q4 = lane & 3;
  const int slot_x = (kQuad && LPT >= 8 && ((lane >> 2) & 1)) ? 3 : 0;
  auto head_of = [&](int r) { return kQuad ? (((q4 + r) & 3) ^ slot_x) : r; };

  float qv[HG][SD];
  if constexpr (!kMfma) {
#pragma unroll
    for (int r = 0; r < HG; ++r)
#pragma unroll
      for (int i = 0; i < SD; ++i) qv[r][i] = s_q[head_of(r)][slice * SD + i];
  }

  float m[HG], lsum[HG], acc[HG][SD];
#pragma unroll
  for (int r = 0; r < HG; ++r) {
    m[r] = -INFINITY;
    lsum[r] = 0.f;  // quad and matrix-core modes use lsum[0] for the lane's own head
#pragma unroll
    for (int i = 0; i < SD; ++i) acc[r][i] = 0.f;
  }

  // Matrix-core mode: the lane's query slice of head lane % 4 (the B operand
  // of the score products), and the value accumulators cv[k] = (head 0..3) at
  // dimension slice * SD + k.  m[0] and lsum[0] belong to head lane % 4 and
  // the lane's value token; m[0] is wavefront-wide per head.
  float qk[SD];
  f32x4 cv[SD];
  if constexpr (kMfma) {
#pragma unroll
    for (int k = 0; k < SD; ++k) {
      qk[k] = s_q[lane & 3][sk * SD + k];
      cv[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }

  const typename Fmt::LutT* lut_k = s_lut[0];
  const typename Fmt::LutT* lut_v = s_lut[1];

  // Matrix-core mode, three parts of an iteration.  score_products: the
  // 4 x 4 x 1 products of one iteration's key rows, kScoreChains independent
  // chains per token (dimension k goes to chain k % kScoreChains).
  // score_reduce: the chains and then the slices are summed and each lane
  // keeps the score of its own (head, value token).  softmax_values: online
  // softmax update and value products of one iteration.
  constexpr int SC = kScoreChains;
  // Matrix ops and VALU ops issued interleaved in one wavefront cost more on
  // this part than the two issued in separate runs (measured: 634 against
  // 453 cycles for 16 products and 32 FMAs at two wavefronts per SIMD), so
  // each phase is fenced off from the compiler's scheduler: table decode,
  // then the products, then the reductions.
  auto score_products = [&](const Raw (&kr)[U], f32x4 (&c)[U][SC]) {
    float x[U][SD];
#pragma unroll
    for (int u = 0; u < U; ++u) Fmt::decode(kr[u], sk, lut_k, x[u]);
    if constexpr (kPhaseFences) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int k = 0; k < SD; ++k)
        c[u][k % SC] = __builtin_amdgcn_mfma_f32_4x4x1f32(x[u][k], qk[k],
                                                          k < SC ? f32x4{0.f, 0.f, 0.f, 0.f} : c[u][k % SC], 0, 0, 0);
    if constexpr (kPhaseFences) __builtin_amdgcn_sched_barrier(0);
  };
  auto score_reduce = [&](f32x4 (&c)[U][SC], float (&s_own)[U]) {
    if constexpr (kMfma) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int w = SC / 2; w >= 1; w /= 2)
#pragma unroll
          for (int j = 0; j < w; ++j) c[u][j] += c[u][j + w];
        s_own[u] = slice_sum_select<LPT>(c[u][0], lane);
      }
    }
  };
  auto softmax_values = [&](const Raw (&vr)[U], const float (&s_own)[U], const float (&vs)[U], int i, auto full) {
    constexpr bool FULL = decltype(full)::value;
    bool valid[U];
#pragma unroll
    for (int u = 0; u < U; ++u) valid[u] = FULL || first + i * BSTRIDE + u * TPB + gi < t1;
    float xv[U][SD];
#pragma unroll
    for (int u = 0; u < U; ++u) Fmt::decode(vr[u], slice, lut_v, xv[u]);
    bool need = false;
#pragma unroll
    for (int u = 0; u < U; ++u) need = need || (valid[u] && s_own[u] > m[0] + kRescaleThreshold);
    if (__builtin_amdgcn_ballot_w64(need) != 0) {
      // A running maximum moves: one maximum per head over the wavefront
      // (lanes sharing lane % 4), accumulators of head r rescaled by the
      // factor of the lanes that hold head r.
      float mx = -INFINITY;
#pragma unroll
      for (int u = 0; u < U; ++u) mx = valid[u] ? fmaxf(mx, s_own[u]) : mx;
      mx = strided_reduce<4, OpMax>(mx);
      float alpha = 1.f;
      if (mx > m[0] + kRescaleThreshold) {
        alpha = fast_exp2(m[0] - mx);  // 0 before the first maximum: nothing accumulated yet
        m[0] = mx;
      }
      lsum[0] *= alpha;
      const float a0 = quad_broadcast_t<0>(alpha), a1 = quad_broadcast_t<1>(alpha);
      const float a2 = quad_broadcast_t<2>(alpha), a3 = quad_broadcast_t<3>(alpha);
#pragma unroll
      for (int k = 0; k < SD; ++k) cv[k] *= f32x4{a0, a1, a2, a3};
    }
    float p[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      p[u] = valid[u] ? fast_exp2(s_own[u] - m[0]) : 0.f;
      lsum[0] += p[u];
      if constexpr (SCALED) p[u] *= vs[u];  // the value products take weight x value scale
    }
    if constexpr (kPhaseFences) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int k = 0; k < SD; ++k) cv[k] = __builtin_amdgcn_mfma_f32_4x4x1f32(p[u], xv[u][k], cv[k], 0, 0, 0);
    if constexpr (kPhaseFences) __builtin_amdgcn_sched_barrier(0);
  };

  // Partial dot products of this lane's slice: part[u][s] for token u, slot s.
  auto partial_scores = [&](const Raw (&kr)[U], float (&part)[U][HG]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float x[SD];
      Fmt::decode(kr[u], slice, lut_k, x);
#pragma unroll
      for (int s = 0; s < HG; ++s) {
        float d = 0.f;
#pragma unroll
        for (int k = 0; k < SD; ++k) d = fmaf(qv[s][k], x[k], d);
        part[u][s] = d;
      }
    }
  };

  // One iteration: U tokens per lane group -- U x HG partial scores, their
  // reduction over the group's lanes, one online-softmax update per head and
  // U value updates.  FULL iterations skip the validity masks.
  auto process = [&](const Raw (&kr)[U], const Raw (&vr)[U], const float (&ks)[U], const float (&vs)[U], int i,
                     auto full) {
    constexpr bool FULL = decltype(full)::value;
    bool valid[U];
#pragma unroll
    for (int u = 0; u < U; ++u) valid[u] = FULL || first + i * BSTRIDE + u * TPB + gi < t1;
    float part[U][HG];
    partial_scores(kr, part);
    // Value rows are decoded (LDS table reads issued) before the softmax so
    // the table latency overlaps it.
    float xv[U][SD];
#pragma unroll
    for (int u = 0; u < U; ++u) Fmt::decode(vr[u], slice, lut_v, xv[u]);
    if constexpr (kQuad) {
      // Quad reduction: slot r of the lane r positions back holds this
      // lane's own head, so three rotations add the quad's partials; the
      // other quads of the group are added after.  Each lane then
      // exponentiates its head for both tokens, and the value update takes
      // the weight of slot r from the lane r positions ahead.
      float own[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        own[u] = cross_quad_sum<LPT>(part[u][0] + quad_rotate_from<1>(part[u][1]) + quad_rotate_from<2>(part[u][2]) +
                                     quad_rotate_from<3>(part[u][3]));
      if constexpr (SCALED) {
#pragma unroll
        for (int u = 0; u < U; ++u) own[u] *= ks[u];
      }
      bool need = false;
#pragma unroll
      for (int u = 0; u < U; ++u) need = need || (valid[u] && own[u] > m[0] + kRescaleThreshold);
      if (__builtin_amdgcn_ballot_w64(need) != 0) {
        // Some running maximum moves (first iteration, rare afterwards).
        // The maxima are kept wavefront-wide: slot r holds the same head on
        // every lane group, and one maximum per head over all the groups'
        // tokens moves far less often than one per group would.
#pragma unroll
        for (int r = 0; r < HG; ++r) {
          float mx = -INFINITY;
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const float v = quad_rotate_to(own[u], r);
            mx = valid[u] ? fmaxf(mx, v) : mx;
          }
          mx = strided_reduce<LPT, OpMax>(mx);
          if (mx > m[r] + kRescaleThreshold) {
            if (m[r] != -INFINITY) {  // nothing accumulated before the first maximum
              const float alpha = fast_exp2(m[r] - mx);
#pragma unroll
              for (int k = 0; k < SD; ++k) acc[r][k] *= alpha;
              if (r == 0) lsum[0] *= alpha;
            }
            m[r] = mx;
          }
        }
      }
      float p_own[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        p_own[u] = valid[u] ? fast_exp2(own[u] - m[0]) : 0.f;
        lsum[0] += p_own[u];
        if constexpr (SCALED) p_own[u] *= vs[u];
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int r = 0; r < HG; ++r) {
          const float p = quad_rotate_to(p_own[u], r);
#pragma unroll
          for (int k = 0; k < SD; ++k) acc[r][k] = fmaf(p, xv[u][k], acc[r][k]);
        }
    } else {
      // Every lane of the group reduces and exponentiates every pair.
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int s = 0; s < HG; ++s) part[u][s] = SCALED ? group_sum<LPT>(part[u][s]) * ks[u] : group_sum<LPT>(part[u][s]);
      // Wavefront-wide running maxima, moved only when some score passes
      // one by more than the threshold (as in quad mode).
      bool need = false;
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int s = 0; s < HG; ++s) need = need || (valid[u] && part[u][s] > m[s] + kRescaleThreshold);
      if (__builtin_amdgcn_ballot_w64(need) != 0) {
#pragma unroll
        for (int s = 0; s < HG; ++s) {
          float mx = -INFINITY;
#pragma unroll
          for (int u = 0; u < U; ++u) mx = valid[u] ? fmaxf(mx, part[u][s]) : mx;
          mx = strided_reduce<LPT, OpMax>(mx);
          if (mx > m[s] + kRescaleThreshold) {
            if (m[s] != -INFINITY) {  // nothing accumulated before the first maximum
              const float alpha = fast_exp2(m[s] - mx);
              lsum[s] *= alpha;
#pragma unroll
              for (int k = 0; k < SD; ++k) acc[s][k] *= alpha;
            }
            m[s] = mx;
          }
        }
      }
      float p[U][HG];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int s = 0; s < HG; ++s) {
          p[u][s] = valid[u] ? fast_exp2(part[u][s] - m[s]) : 0.f;
          lsum[s] += p[u][s];
          if constexpr (SCALED) p[u][s] *= vs[u];
        }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int s = 0; s < HG; ++s)
#pragma unroll
          for (int k = 0; k < SD; ++k) acc[s][k] = fmaf(p[u][s], xv[u][k], acc[s][k]);
    }
  };

  // The ring is unrolled NB times with no exit inside it, so the waits for
  // each slot are the same on every trip and leave the PF prefetched slots in
  // flight; loads for iterations past n_iter get an empty range and read
  // nothing, and their compute is skipped (a wavefront-uniform branch: the
  // longest splits of the 24-layer 8K decode loop run 3 iterations, not 4).
  for (int it = 0; it < n_iter; it += NB) {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int i = it + j;
      load_iter(i + PF, kr[(j + PF) % NB], vr[(j + PF) % NB], ksr[(j + PF) % NB], vsr[(j + PF) % NB]);
      if (j > 0 && i >= n_iter) continue;
      const bool full = first + i * BSTRIDE + (U - 1) * TPB + TPW <= t1;
      if constexpr (kMfma) {
        f32x4 c[U][SC];
        float s_own[U];
        score_products(kr[j], c);
        score_reduce(c, s_own);
        if constexpr (SCALED) {
#pragma unroll
          for (int u = 0; u < U; ++u) s_own[u] *= ksr[j][u];
        }
        if (full)
          softmax_values(vr[j], s_own, vsr[j], i, std::true_type{});
        else
          softmax_values(vr[j], s_own, vsr[j], i, std::false_type{});
      } else {
        if (full)
          process(kr[j], vr[j], ksr[j], vsr[j], i, std::true_type{});
        else
          process(kr[j], vr[j], ksr[j], vsr[j], i, std::false_type{});
      }
    }
  }

  // ---- combine the lane groups of this workgroup (log-sum-exp).
  // The running maxima are wavefront-wide: m[r] is the same on every lane
  // that holds the same head in slot r, and lane 0 holds head r in slot r.
  // So the lane groups' sums share one reference per head and add without
  // rescaling: the softmax sums over the lanes of one slice (in quad mode a
  // lane holds only its own head's sum and takes slot r's from the lane r
  // positions ahead; the sums are equal on the lanes of a group that hold the
  // same head in the same slot), the accumulators by a reduce-scatter.  The
  // wavefronts' partials are weighted against the workgroup maximum when
  // they are added after the barrier.
  if constexpr (kMfma) {
    // Matrix-core mode: lane l holds head l % 4 and value token l / LPT; the
    // LPT / 4 lanes of a token that hold the same head add each weight once.
    const float ls = (lane % LPT) < 4 ? lsum[0] : 0.f;
    const float lw = strided_reduce<4, OpSum>(ls);
    if (lane < 4) {
      s_mw[wave][lane] = m[0];
      s_lw[wave][lane] = lw;
    }
  } else {
#pragma unroll
    for (int r = 0; r < HG; ++r) {
      const float ls = !kQuad || r == 0 ? lsum[kQuad ? 0 : r] : quad_rotate_to(lsum[0], r);
      const float lw = strided_reduce<LPT, OpSum>(ls);
      if (lane == 0) {
        s_mw[wave][r] = m[r];
        s_lw[wave][r] = lw;
      }
    }
  }
  // Reduce-scatter the accumulators over the TPW lane groups of the
  // wavefront: afterwards lane (gi, slice) holds values
  // [gi * NV / TPW, (gi + 1) * NV / TPW) of its slice, summed over groups.
  {
    float buf[NV];
#pragma unroll
    for (int r = 0; r < HG; ++r)
#pragma unroll
      for (int k = 0; k < SD; ++k) buf[r * SD + k] = kMfma ? cv[k][r] : acc[r][k];
    if constexpr (TPW > 1) reduce_scatter<LPT, kWave / 2, NV / 2, NV>(buf, lane);
    constexpr int W = NV / TPW;
#pragma unroll
    for (int k = 0; k < W; ++k) {
      const int v = gi * W + k;
      const int r = v / SD, d = v - r * SD;
      s_red[wave][head_of(r) * D + slice * SD + d] = buf[k];
    }
  }
  __syncthreads();
  // Weight of each wavefront's partial for head h against the workgroup
  // maximum (zero for a wavefront that saw no token); returns that maximum.
  auto wave_weights = [&](int h, float (&f)[kWavesPerBlock]) {
    float M = s_mw[0][h];
#pragma unroll
    for (int w = 1; w < kWavesPerBlock; ++w) M = fmaxf(M, s_mw[w][h]);
#pragma unroll
    for (int w = 0; w < kWavesPerBlock; ++w) f[w] = s_mw[w][h] == -INFINITY ? 0.f : fast_exp2(s_mw[w][h] - M);
    return M;
  };
  // Sum of the wavefronts' accumulators into s_red[0], weighted.
  auto combine_waves = [&]() {
    for (int o = tid; o < HG * D; o += kBlock) {
      float f[kWavesPerBlock];
      wave_weights(o / D, f);
      float v = s_red[0][o] * f[0];
#pragma unroll
      for (int w = 1; w < kWavesPerBlock; ++w) v = fmaf(s_red[w][o], f[w], v);
      s_red[0][o] = v;
    }
    __syncthreads();
  };

  // ---- one split: this workgroup holds the whole result and finishes it.
  const int64_t qhg0 = static_cast<int64_t>(layer) * a.query_heads + qh0;
  if (a.n_splits == 1) {
    combine_waves();
    if (wave < heads) {
      float f[kWavesPerBlock];
      const float M = wave_weights(wave, f);
      float l = 0.f;
#pragma unroll
      for (int w = 0; w < kWavesPerBlock; ++w) l = fmaf(s_lw[w][wave], f[w], l);
      const float* ck = appending ? s_cur[0] : a.cur_k ? a.cur_k + static_cast<int64_t>(lkv) * D : nullptr;
      const float* cv = appending ? s_cur[1] : a.cur_v ? a.cur_v + static_cast<int64_t>(lkv) * D : nullptr;
      finish_row<D>(&s_red[0][wave * D], M, l, s_q[wave], ck, cv, a.inverse_output, sg_second, sg_first, a.sqrt_d,
                    a.out + (qhg0 + wave) * D);
    }
    return;
  }

  // ---- several splits: publish this split's partial for merge_kernel.  The
  // accumulator is stored inverse-rotated already: the rotation is linear, so
  // the merge is a plain weighted sum per dimension.  Split 0 also publishes
  // the current token's score per query head and its value per KV head.
  // Wavefront h < HG sums head h's row over the 4 wavefronts' partials
  // straight from LDS (no combining pass, no second barrier).
  if (wave < heads) {
    float f[kWavesPerBlock];
    const float M = wave_weights(wave, f);
    float e[E];
#pragma unroll
    for (int i = 0; i < E; ++i) {
      float v = s_red[0][wave * D + lane * E + i] * f[0];
#pragma unroll
      for (int w = 1; w < kWavesPerBlock; ++w) v = fmaf(s_red[w][wave * D + lane * E + i], f[w], v);
      e[i] = v;
    }
    if (a.inverse_output) wave_rotate_signs<D>(e, sg_second, sg_first, a.sqrt_d);
    float* dst = a.ws_acc + ((qhg0 + wave) * a.n_splits + split) * D + lane * E;
#pragma unroll
    for (int i = 0; i < E; ++i) dst[i] = e[i];
    if (lane == 0) {
      float l = 0.f;
#pragma unroll
      for (int w = 0; w < kWavesPerBlock; ++w) l = fmaf(s_lw[w][wave], f[w], l);
      a.ws_ml[((qhg0 + wave) * a.n_splits + split) * 2] = M;
      a.ws_ml[((qhg0 + wave) * a.n_splits + split) * 2 + 1] = l;
    }
    if (split == 0 && (appending || a.cur_k != nullptr)) {
      const float* ck = (appending ? s_cur[0] : a.cur_k + static_cast<int64_t>(lkv) * D) + lane * E;
      float dot = 0.f;
#pragma unroll
      for (int i = 0; i < E; ++i) dot = fmaf(s_q[wave][lane * E + i], ck[i], dot);
      dot = group_sum<kWave>(dot);
      if (lane == 0) a.ws_cur_s[qhg0 + wave] = dot;
      if (wave == 0 && hg == 0) {
        float v[E];
        const float* cv = (appending ? s_cur[1] : a.cur_v + static_cast<int64_t>(lkv) * D) + lane * E;
#pragma unroll
        for (int i = 0; i < E; ++i) v[i] = cv[i];
        if (a.inverse_output) wave_rotate_signs<D>(v, sg_second, sg_first, a.sqrt_d);
#pragma unroll
        for (int i = 0; i < E; ++i) a.ws_cur_v[static_cast<int64_t>(lkv) * D + lane * E + i] = v[i];
      }
    }
  }
}

#include "decode_mx.hpp"

// Log-sum-exp merge of the splits: M = max(max_s M_s, current score),
// L = sum_s L_s 2^(M_s - M) (+ 2^(score - M)), out = (sum_s A_s 2^(M_s - M)
// (+ 2^(score - M) value)) / L.  The split accumulators A_s are already
// rotated back, so every dimension is independent: one workgroup per (query
// head, kMergeDims dimensions), its threads split the splits into kMergeGroups
// strided groups and issue all their loads before the (max, sum) reduction.
constexpr int kMergeDims = 16;  // 16: M -0.6 us per step against 32 (8 equal, 64 +2 us)
constexpr int kMergeGroups = kBlock / kMergeDims;
constexpr int kMergePerThread = kMaxSplits / kMergeGroups;

struct MergeArgs {
  int query_heads, kv_heads, group, n_splits;
  const float* ws_ml;   // [L * Hq, n_splits, 2]
  const float* ws_acc;  // [L * Hq, n_splits, D]
  const float* cur_s;   // [L * Hq] or null
  const float* cur_v;   // [L * Hkv, D]
  float* out;           // [L, Hq, D]
};

template <int D>
__global__ __launch_bounds__(kBlock) void merge_kernel(const MergeArgs a) {
  constexpr int CH = D / kMergeDims;
  __shared__ float s_f[kMaxSplits];
  __shared__ float s_red[kWavesPerBlock];
  __shared__ float s_part[kMergeGroups][kMergeDims];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & (kWave - 1);
  // Same XCD remap as the split kernel: XCD x takes the x-th eighth of the
  // query heads, whose partials that kernel wrote through the same XCD's L2
  // (measured: C5 loop 336 -> 332 us per step, M unchanged).
  int64_t mb = blockIdx.x;
  const int64_t nmb = gridDim.x;
  mb = (mb & 7) * (nmb >> 3) + min(mb & 7, nmb & 7) + (mb >> 3);
  const int64_t qhg = mb / CH;
  const int c = static_cast<int>(mb - qhg * CH);
  const int ns = a.n_splits;
  const int d = tid % kMergeDims, grp = tid / kMergeDims;
  const float* ml = a.ws_ml + qhg * ns * 2;
  const float* acc = a.ws_acc + qhg * ns * D + c * kMergeDims + d;

  float vals[kMergePerThread];
#pragma unroll
  for (int k = 0; k < kMergePerThread; ++k) {
    const int sp = grp + k * kMergeGroups;
    vals[k] = sp < ns ? acc[static_cast<int64_t>(sp) * D] : 0.f;
  }
  const float ms = tid < ns ? ml[tid * 2] : -INFINITY;
  const float ls = tid < ns ? ml[tid * 2 + 1] : 0.f;
  float cs = -INFINITY;
  if (a.cur_s != nullptr) cs = a.cur_s[qhg];

  const float mx = group_reduce<kWave, OpMax>(ms);
  if (lane == 0) s_red[wave] = mx;
  __syncthreads();
  const float M = fmaxf(fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3])), cs);
  const float f = ls > 0.f ? fast_exp2(ms - M) : 0.f;
  if (tid < ns) s_f[tid] = f;
  const float lw = group_sum<kWave>(ls * f);
  __syncthreads();
  if (lane == 0) s_red[wave] = lw;
  float part = 0.f;
#pragma unroll
  for (int k = 0; k < kMergePerThread; ++k) {
    const int sp = grp + k * kMergeGroups;
    if (sp < ns) part = fmaf(vals[k], s_f[sp], part);
  }
  s_part[grp][d] = part;
  __syncthreads();
  if (tid < kMergeDims) {
    float L = s_red[0] + s_red[1] + s_red[2] + s_red[3];
    float v = s_part[0][d];
#pragma unroll
    for (int g = 1; g < kMergeGroups; ++g) v += s_part[g][d];
    if (a.cur_s != nullptr) {
      const int layer = static_cast<int>(qhg / a.query_heads);
      const int qh = static_cast<int>(qhg - static_cast<int64_t>(layer) * a.query_heads);
      const int64_t lkv = static_cast<int64_t>(layer) * a.kv_heads + qh / a.group;
      const float fc = fast_exp2(cs - M);
      v = fmaf(fc, a.cur_v[lkv * D + c * kMergeDims + d], v);
      L += fc;
    }
    a.out[qhg * D + c * kMergeDims + d] = L > 0.f ? v / L : 0.f;
  }
}

// ============================================================== split path stages


template <class Fmt, int D>
__global__ __launch_bounds__(kBlock) void score_kernel(const float* __restrict__ q, const uint8_t* __restrict__ codes,
                                                       int64_t seq_len, const float* __restrict__ cent,
                                                       float* __restrict__ scores) {
  constexpr int SD = Fmt::kSliceDims;
  constexpr int LPT = D / SD;
  constexpr int TPW = kWave / LPT;
  constexpr int ROW = Fmt::template row_bytes<D>();
  __shared__ typename Fmt::LutT s_lut[Fmt::kLutEntries];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & (kWave - 1);
  const int gi = lane / LPT, slice = lane % LPT;
  const int b = blockIdx.y;
  for (int e = tid; e < Fmt::kLutEntries; e += kBlock) s_lut[e] = Fmt::lut_entry(e, cent);
  __syncthreads();
  float qv[SD];
#pragma unroll
  for (int i = 0; i < SD; ++i) qv[i] = q[static_cast<int64_t>(b) * D + slice * SD + i];
  const int64_t t = (static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + wave) * TPW + gi;
  float x[SD];
  float s = 0.f;
  if (t < seq_len) {
    const auto r = Fmt::load(codes + (static_cast<int64_t>(b) * seq_len + t) * ROW, slice);
    Fmt::decode(r, slice, s_lut, x);
#pragma unroll
    for (int i = 0; i < SD; ++i) s = fmaf(qv[i], x[i], s);
  }
  s = group_sum<LPT>(s);
  if (t < seq_len && slice == 0) scores[static_cast<int64_t>(b) * seq_len + t] = s;
}

__global__ __launch_bounds__(kBlock) void softmax_kernel(const float* __restrict__ scores, int64_t seq_len,
                                                         float scale, float* __restrict__ w) {
  __shared__ float s_red[kWavesPerBlock];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & (kWave - 1);
  const float* row = scores + static_cast<int64_t>(blockIdx.x) * seq_len;
  float* orow = w + static_cast<int64_t>(blockIdx.x) * seq_len;
  float mx = -INFINITY;
  for (int64_t t = tid; t < seq_len; t += kBlock) mx = fmaxf(mx, row[t] * scale);
  mx = group_reduce<kWave, OpMax>(mx);
  if (lane == 0) s_red[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
  __syncthreads();
  float sum = 0.f;
  for (int64_t t = tid; t < seq_len; t += kBlock) sum += expf(row[t] * scale - mx);
  sum = group_sum<kWave>(sum);
  if (lane == 0) s_red[wave] = sum;
  __syncthreads();
  sum = s_red[0] + s_red[1] + s_red[2] + s_red[3];
  for (int64_t t = tid; t < seq_len; t += kBlock) orow[t] = expf(row[t] * scale - mx) / sum;
}

template <class Fmt, int D>
__global__ __launch_bounds__(kBlock) void accumulate_kernel(const float* __restrict__ w,
                                                            const uint8_t* __restrict__ codes, int64_t seq_len,
                                                            const float* __restrict__ cent, float* __restrict__ out) {
  constexpr int SD = Fmt::kSliceDims;
  constexpr int LPT = D / SD;
  constexpr int TPW = kWave / LPT;
  constexpr int TPB = kWavesPerBlock * TPW;
  constexpr int ROW = Fmt::template row_bytes<D>();
  __shared__ typename Fmt::LutT s_lut[Fmt::kLutEntries];
  __shared__ float s_part[TPB][D];  // one row per lane group: summed in a fixed order
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & (kWave - 1);
  const int gi = lane / LPT, slice = lane % LPT;
  const int b = blockIdx.x;
  for (int e = tid; e < Fmt::kLutEntries; e += kBlock) s_lut[e] = Fmt::lut_entry(e, cent);
  __syncthreads();
  float acc[SD];
#pragma unroll
  for (int i = 0; i < SD; ++i) acc[i] = 0.f;
  float x[SD];
  for (int64_t t = wave * TPW + gi; t < seq_len; t += TPB) {
    const float wt = w[static_cast<int64_t>(b) * seq_len + t];
    const auto r = Fmt::load(codes + (static_cast<int64_t>(b) * seq_len + t) * ROW, slice);
    Fmt::decode(r, slice, s_lut, x);
#pragma unroll
    for (int i = 0; i < SD; ++i) acc[i] = fmaf(wt, x[i], acc[i]);
  }
#pragma unroll
  for (int i = 0; i < SD; ++i) s_part[wave * TPW + gi][slice * SD + i] = acc[i];
  __syncthreads();
  for (int d = tid; d < D; d += kBlock) {
    float v = 0.f;
    for (int r = 0; r < TPB; ++r) v += s_part[r][d];
    out[static_cast<int64_t>(b) * D + d] = v;
  }
}

// ============================================================== attention layer


#include "attention_layer.hpp"

// ============================================================== measurement


constexpr int kStreamThreads = 512;  // streaming-read probe: 512 threads, one workgroup per CU

// Streaming-read probe (the bench's HBM ceiling): every thread keeps four
// nontemporal 16-byte loads in flight over a grid-stride pass.  The shape is
// the best of a sweep on MI355X (grid-stride and per-workgroup chunks; 1, 2,
// 4, 8, 16 loads in flight; 256 / 512 / 1024 threads; 1-16 workgroups per
// CU; with and without the nontemporal bit): 6.9-7.0 TB/s over a 768 MiB
// pass, against 6.3-6.5 for the best cached-load shapes.  The store happens
// only if the xor of everything read equals a fixed pattern, which keeps the
// loads live without writing in practice.
__global__ __launch_bounds__(kStreamThreads) void stream_read_kernel(const uint4* __restrict__ p, int64_t n16,
                                                                     float* __restrict__ sink) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const u32x4* q = reinterpret_cast<const u32x4*>(p);
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kStreamThreads;
  int64_t i = static_cast<int64_t>(blockIdx.x) * kStreamThreads + threadIdx.x;
  uint32_t acc = 0;
  for (; i + 3 * stride < n16; i += 4 * stride) {
    const u32x4 a = __builtin_nontemporal_load(q + i), b = __builtin_nontemporal_load(q + i + stride);
    const u32x4 c = __builtin_nontemporal_load(q + i + 2 * stride), d = __builtin_nontemporal_load(q + i + 3 * stride);
    const u32x4 x = a ^ b ^ c ^ d;
    acc ^= x.x ^ x.y ^ x.z ^ x.w;
  }
  for (; i < n16; i += stride) {
    const u32x4 a = __builtin_nontemporal_load(q + i);
    acc ^= a.x ^ a.y ^ a.z ^ a.w;
  }
  if (acc == 0x9E3779B9u) sink[blockIdx.x] = 1.f;
}

// ============================================================== host helpers


// Query heads per work unit.  A unit reads its KV head's rows once, so groups
// of 3 and more that are no multiple of 4 are cut into units of 4, the last
// one with slots to spare (the matrix-core products cost the same whatever
// the heads in them), where that saves enough rows (elements) to pay for the
// longer set-up and combine of a 4-head unit.  Measured on MI355X against
// units that divide the group: 8 KV heads, 3-bit rows at head_dim 128, 32768
// tokens: groups of 3 25.2 -> 17.0 us, 5 38.6 -> 26.2, 6 32.7 -> 26.3, 7 48.3
// -> 26.0; 16 x 8 heads at 64, 23236 tokens, groups of 3 124 -> 57; 10 M
// elements saved 18.6 -> 16.1, but 4.2 M 9.3 -> 10.1 and 5.1 M (dense rows)
// 7.5 -> 8.4.
// Dense rows, which units of 1 and 2 read without table lookups, are cut from
// 768 tokens on: 64 units x 7 heads x 520 tokens at 128 11.2 -> 13.5, 5 heads
// 11.5 -> 12.9, but at 768 14.4 -> 14.1 and 14.8 -> 13.5.
constexpr int64_t kMinSavedElements = int64_t(1) << 23;
constexpr int64_t kMinCutDenseTokens = 768;

int head_groups(int group, int hg) { return (group + hg - 1) / hg; }
int even_hg(int group) { return group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1; }
bool packed_rows(int fmt) { return fmt == 2 || fmt == 3 || fmt == 4; }
int pick_hg(int group, int64_t kv_units, int64_t seq_len, int fmt, int head_dim) {
  const int hg = even_hg(group);
  if (hg == 4 || group < 3 || (!packed_rows(fmt) && seq_len < kMinCutDenseTokens)) return hg;
  const int64_t saved = kv_units * (head_groups(group, hg) - head_groups(group, 4)) * seq_len * head_dim;
  return saved >= kMinSavedElements ? 4 : hg;
}

// The split kernel a decode call runs: the float32 kernel (decode_kernel,
// 4x4x1 fp32 matrix products or VALU FMAs, 256 threads, two workgroups per
// CU) or, for 4-bit packed rows in groups of 4 query heads at head_dim 64 or
// 128, decode_mx_kernel (16x16x32 products of exact f16 splits, 768 threads,
// one workgroup per CU) unless TQ_F32_PRODUCTS asks for the former.
enum class SplitKernel { Fp32, Mx };

struct Plan {
  int hg, n_hgroups, units, n_splits;
  SplitKernel kernel;
  int block_rows;  // rows per workgroup iteration (the unit the sequence is dealt out in)
  int tokens_per_iter;  // decode_kernel: tokens per lane group per iteration
};

constexpr int kMinTokensPerSplit = 128;

// Most workgroups per CU of a plan whose workgroups do not all run at once
// (see balanced_splits), and the work of a workgroup besides its blocks, in
// blocks: 4 heads at head_dim 256 take twice the set-up and combine for half
// the rows of a block.
constexpr int kMaxLoad = 6;
int load_overhead(int head_dim, int hg) { return head_dim == 256 && hg == 4 ? 12 : 5; }
constexpr int kMergeWork = 12;  // the merge launch that more than one split adds

// Splits of a call with many units.  One resident round of workgroups leaves
// CUs with one workgroup less than others when units does not divide it (192
// units: 384 workgroups, 2 on half of the CUs and 1 on the rest); a CU works
// through its workgroups at the same rate whether one or two are resident, so
// what counts is the work of the CU with the most.  Starting from the
// one-round count ns0, take the count that makes it smallest, if that is at
// least 1/16 less (1/4 for dense rows, whose one-round plans read memory at
// 5.5 to 6.3 TB/s already).  Measured on MI355X, 24 layers x 8 KV heads: 3-bit rows at
// head_dim 128 x 8192 tokens, groups of 4, 74 us at 2 splits, 60 at 4 (768
// workgroups, 3 to a CU), 64 at 5, 63 at 8; 4-bit rows, groups of 1, 57, 45,
// 47, 44; at head_dim 64, groups of 2, 36, 30, 31, 31.  Over 24 random shapes
// whose count it changes: 1.03 to 1.41 times as fast.  The overheads keep it
// from short sequences, where more splits lose (3-bit rows at head_dim 256,
// groups of 4: 384 units x 1536 tokens 53 us at 1 split, 62 at 2, 640 x 3072
// 143 and 161).  Dense rows at 256, groups of 4: 384 units x 768 tokens 51 and
// 69, x 2048 129 and 148; 300 x 3072 172 at 1, 167 at 3, groups of 1 172 and 145 at 5.
struct Work {
  int units;
  int64_t blocks;  // of one sequence
  int overhead, num_cus;
  int64_t of(int64_t ns) const {
    return ((units * ns + num_cus - 1) / num_cus) * (overhead + (blocks + ns - 1) / ns) + (ns > 1 ? kMergeWork : 0);
  }
};
int balanced_splits(const Work& work, int ns0, bool packed) {
  const int64_t limit = (packed ? 15 : 12) * work.of(ns0);
  int best = ns0;
  const int64_t most = std::min<int64_t>({static_cast<int64_t>(kMaxLoad) * work.num_cus / work.units, work.blocks, kMaxSplits});
  for (int64_t ns = ns0 + 1; ns <= most; ++ns)
    if (16 * work.of(ns) <= limit && work.of(ns) < work.of(best)) best = static_cast<int>(ns);
  return best;
}

int default_splits(int units, int64_t seq_len, int num_cus, int wgs_per_cu) {
  if (num_cus <= 0) num_cus = 256;
  const int64_t target = static_cast<int64_t>(wgs_per_cu) * num_cus;
  // Whole waves only: rounding target / units up would overshoot the target
  // when units does not divide it, and the few workgroups past it run as a
  // second wave.  Measured on MI355X, 3 head groups x 64K tokens: matrix
  // kernel 86 splits 16.6-17.1 us against 11.3-11.9 at 85, float32 kernel
  // 171 splits 15.3-16.0 us against 12.8-13.5 at 170.
  int64_t ns = std::max<int64_t>(1, target / units);
  const int64_t by_len = std::max<int64_t>(1, (seq_len + kMinTokensPerSplit - 1) / kMinTokensPerSplit);
  ns = std::min(ns, by_len);
  // A length cap just above one workgroup per CU (8192 + t tokens over 4 KV
  // heads: 65 splits, 260 workgroups) leaves a few CUs running two, and
  // those end the kernel late; one workgroup per CU with an extra block on
  // a few splits ends sooner.  Measured on MI355X, a 4 x 8192-token layer:
  // 10.0 us per decode at 64 splits, 11.2 at 63 (four splits with an extra
  // block), 12.6 at 65 (260 workgroups); a 24-layer 8K decode loop 375 ->
  // 340 us per step.
  if (units * ns > num_cus && units * ns <= num_cus + num_cus / 8)
    ns = std::max<int64_t>(1, num_cus / units);
  ns = std::max<int64_t>(1, std::min<int64_t>(ns, kMaxSplits));
  return static_cast<int>(ns);
}

int device_cu_count() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 256;
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) return 256;
  return cus;
}

// Workspace layout: [ml: Lq * ns * 2][acc: Lq * ns * D][cur_s: Lq][cur_v: Lkv * D]
// floats, Lq = layers * query heads, Lkv = layers * KV heads, each section
// 256-byte aligned.
struct WsLayout {
  size_t ml, acc, cur_s, cur_v, total;
};

size_t align256(size_t v) { return (v + 255) / 256 * 256; }

WsLayout workspace_layout(int64_t lq, int64_t lkv, int head_dim, int n_splits) {
  WsLayout w;
  w.ml = 0;
  w.acc = align256(static_cast<size_t>(lq) * n_splits * 2 * sizeof(float));
  w.cur_s = w.acc + align256(static_cast<size_t>(lq) * n_splits * head_dim * sizeof(float));
  w.cur_v = w.cur_s + align256(static_cast<size_t>(lq) * sizeof(float));
  w.total = w.cur_v + align256(static_cast<size_t>(lkv) * head_dim * sizeof(float));
  return w;
}

// ---- static scratch of the no-allocation decode entry point.
// One array per GPU in device memory, held until the process ends; every
// tq_decode_noalloc call on a GPU uses that GPU's copy as its split-K
// workspace (which needs no initialisation: each call writes every partial it
// later reads), so calls that overlap on one GPU race.  In host code
// `scratch` only names the symbol: its device address comes from
// hipGetSymbolAddress, looked up once per device with that device current.
constexpr size_t kScratchBytes = size_t(8) << 20;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// The current device's scratch address in *out (looked up on the first call
// on that device), or an error code with the message set.  The lookup is not a stream
// operation, but it may load the code object, which a stream capture does not
// allow: a first call on a device made inside a capture is refused with a
// message, before anything is enqueued.
int device_scratch(hipStream_t stream, void** out) {
  int dev = -1;
  const hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    return fail(TQ_ERR_LAUNCH, std::string("tq_decode_noalloc: no current HIP device: ") + hipGetErrorString(e));
  }
  if (dev < 0 || dev >= kMaxDevices) {
    return fail(TQ_ERR_UNSUPPORTED, "tq_decode_noalloc: device index " + std::to_string(dev) + " out of range");
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cap) == hipSuccess && cap != hipStreamCaptureStatusNone) {
      return fail(TQ_ERR_BAD_ARG, "tq_decode_noalloc: the first call on device " + std::to_string(dev) +
                                      " is inside a stream capture; make one call on that device outside capture first");
    }
    void* ptr = nullptr;
    const hipError_t r = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (r != hipSuccess || ptr == nullptr) {
      return fail(TQ_ERR_LAUNCH, std::string("tq_decode_noalloc: hipGetSymbolAddress(scratch) failed: ") +
                                     hipGetErrorString(r));
    }
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return TQ_OK;
}

// Rows per workgroup iteration of decode_kernel for `fmt` (2/3/4 packed
// bits, 16 dense fp16, 32 dense fp32): tokens per lane group x lane groups
// per wavefront (64 / (D / slice dims)) x wavefronts; packed slices hold 16
// dimensions, fp16 rows 8, fp32 rows 4.
int decode_block_rows(int fmt, int head_dim, int tokens_per_iter = kTokensPerIter) {
  const bool packed = packed_rows(fmt);
  const int slice_dims = packed ? 16 : (fmt == 16 ? 8 : 4);
  return tokens_per_iter * kWavesPerBlock * kWave * slice_dims / head_dim;
}

// decode_kernel also has instances with kWideTokensPerIter tokens per lane
// group for 4-bit rows at head_dim 256 in groups of 4 query heads (48 rows
// per workgroup iteration against 32; 211 VGPRs, no spills).
template <class Fmt, int D, int HG>
constexpr bool wide_iter_instance() {
  return std::is_same_v<Fmt, PackedB4> && D == 256 && HG == 4;
}
bool wide_iter_shape(int fmt, int head_dim, int hg) { return fmt == 4 && head_dim == 256 && hg == 4; }

// Tokens per lane group per iteration of a decode_kernel call over seq_len
// rows and at most `ns_cap` splits.  Two measurements on MI355X (4 KV heads,
// 64 splits) put a wide iteration at about 1.6 narrow ones: at 8193-8320
// rows (5 iterations of 32 rows on the longest split against 3 of 48) a
// 24-layer decode loop takes 275 against 289 us per step, at 8192 rows (4
// against 3) one layer 11.2 against 10.0 us.  So the wide instance runs
// where 1.6 x its iterations stay below the narrow count: where the last
// narrow iteration is a nearly empty one, not on long sequences.
int fp32_tokens_per_iter(int fmt, int head_dim, int hg, int64_t seq_len, int64_t ns_cap) {
  if (!wide_iter_shape(fmt, head_dim, hg)) return kTokensPerIter;
  auto iters = [&](int u) {
    const int64_t rows = decode_block_rows(fmt, head_dim, u);
    const int64_t blocks = std::max<int64_t>(1, (seq_len + rows - 1) / rows);
    const int64_t ns = std::max<int64_t>(1, std::min(blocks, ns_cap));
    return (blocks + ns - 1) / ns;
  };
  return 8 * iters(kWideTokensPerIter) < 5 * iters(kTokensPerIter) ? kWideTokensPerIter : kTokensPerIter;
}

// Shapes the matrix-core split kernel takes: groups of a multiple of 4 query
// heads with 4-bit rows at head_dim 64 / 128 / 256 or 2-bit rows at head_dim 128.
bool mx_shape(int fmt, int head_dim, int group) {
  return group % 4 == 0 && ((fmt == 4 && (head_dim == 64 || head_dim == 128 || head_dim == 256)) ||
                            (fmt == 2 && head_dim == 128));
}

// Fewest 128-row blocks per split, in units of 4 heads, at which the
// matrix-core kernel runs by default.  Measured on MI355X (wall time per decode, each kernel on its own
// default split plan): at head_dim 128 it is level with the float32 kernel at
// 2 blocks per split and ahead from 4 (0.6 us at 16K tokens x 8 KV heads,
// 1.6 us at 32K); at head_dim 256 it trails at 1-4 blocks (0.2-1.6 us) and
// leads at 8 (2.5 us at 64K x 4 and 128K x 2).  With less work per
// workgroup, writing its 128 KB of tables costs more than its loop saves.
int mx_min_blocks_per_split(int head_dim) { return head_dim == 256 ? 8 : 4; }

// Short packed sequences take one split: the workgroup of a head group reads
// them in few iterations and finishes its rows itself, so the call is one
// launch.  The line is where that is as fast on the GPU.  Measured on MI355X
// (graphs of decodes), one split against the splits of 128 tokens: at head_dim
// 64 every case up to 512 tokens (4 iterations; 8 heads 5.3 us against 6.4);
// at 128, groups of 1, 384 tokens (6) 6.6 against 7.1 but 448 7.2 against 7.1,
// larger units 320 tokens (5) 7.5 against 7.7 but 384 3-bit tokens 8.1 against
// 7.75; at 256, groups of 1, 256 tokens (8) 7.9 against 8.3, larger units 192
// tokens (6) 8.0 against 8.5 but 256 9.2 against 9.0.  With more units than
// half of the CUs the splits do not run side by side and one is faster up to
// 512 tokens (24 layers x 8 heads, 512 3-bit tokens at 128 9.6 against 15.5);
// so it is for a group cut into units of 4 whose own units are more than the
// CUs (40 x 7 heads, 341 4-bit tokens at 128 8.4 in units of 1, 9.3 in 3 splits).
// A caller whose host pays for the second launch asks for TQ_ONE_LAUNCH: 512
// tokens x 8 heads at head_dim 128 take 7.6 us on the GPU in one split and 7.1
// in 4, and 8.6 against 11.6 with the Python call around them.
constexpr int kShortTokens = 512;
constexpr int kShortIterations = 8;

bool one_split(int64_t seq_len, int fmt, int head_dim, int hg, bool many_units, bool one_launch) {
  if (!packed_rows(fmt)) return false;
  int iterations = kShortIterations;
  if (!one_launch && !many_units) iterations = (head_dim == 256 ? 8 : 6) - (hg > 1);
  return seq_len <= std::min(kShortTokens, iterations * decode_block_rows(fmt, head_dim));
}

// Whether ns splits of units of 8 heads pay for the merge that they need where
// units of 4 fill the CUs with one split each: the blocks they take off a
// workgroup against partial results in proportion to the units.  Measured on
// MI355X, units of 8 in one split / in ns (units of 4): 128 units, 4-bit rows
// at head_dim 128, 1024 tokens 10.4 / 17.8 us (10.7), 4096 24.5 / 27.4 (29.7),
// 6144 35.1 / 33.7 (41.2); 96 units 3072 18.4 / 20.4 (19.4), 4096 22.7 / 22.7
// (24.1); 72 units, 3 splits 2048 13.8 / 15.6 (13.9), 3072 18.2 / 17.1 (18.8);
// the same lines at head_dim 64 and for 2-bit rows; at 256, 128 units, 3072
// tokens 39.0 / 42.0 (43.6), 4096 49.7 / 48.6 (54.1).
bool splits_pay_units_of_8(int units, int ns, int64_t blocks, int head_dim) {
  return blocks * (ns - 1) * (head_dim == 256 ? 8 : 6) >= static_cast<int64_t>(units) * ns;
}

// Split kernel, split count and heads per unit of a decode over kv_units
// (layers x KV heads) with decode `flags` (n_splits <= 0: the default count
// for the chosen kernel).
struct KernelChoice {
  SplitKernel kernel;
  int n_splits;
  int hg;  // query heads per unit
};
KernelChoice choose_kernel(int64_t kv_units, int64_t seq_len, int n_splits, int fmt, int head_dim, int group, int flags,
                           int num_cus) {
  if (num_cus <= 0) num_cus = 256;
  int hg = pick_hg(group, kv_units, seq_len, fmt, head_dim);
  // An explicit count with which units of 4 save no round of workgroups over
  // the CUs only makes each workgroup longer.  Of an odd group: 4 KV heads x
  // 30000 3-bit tokens at head_dim 64, groups of 7, 8 splits (224 workgroups)
  // 22.9 us in units of 1, 26.4 in units of 4, 11 splits (308) 20.7 and 21.2,
  // 23 (644) 15.9 and 13.7; 8 x 32768 at 128, groups of 3, 9 splits (216) 34.7
  // and 39.1, 11 (264) 40.3 and 33.5.  Of dense rows: 8 x 52384 at 128, groups
  // of 6, 1 split (24) 647 in units of 2 and 710, 10 x 13139, 3 splits (240)
  // 62.5 and 67.5.  Packed rows in units of 2 lose to units of 4 within one
  // round (24 workgroups 120.7 and 111.0, 240 41.6 and 38.5), but not within
  // two (480, 8197 rows at 64: 27.5 and 29.3).  Dense splits shorter than the
  // default's shortest are set-up for the most part: 64 x 1558 at 128, groups
  // of 6, 48 splits 38.3 in units of 2 and 42.0.
  if (n_splits > 0 && hg > even_hg(group)) {
    const int own = even_hg(group);
    auto rounds = [&](int h) { return (kv_units * head_groups(group, h) * n_splits + num_cus - 1) / num_cus; };
    const bool dense = !packed_rows(fmt);
    if (rounds(own) == rounds(hg) && (own == 1 || dense || rounds(own) > 1)) hg = own;
    if (dense && own > 1 && seq_len < static_cast<int64_t>(n_splits) * kMinTokensPerSplit) hg = own;
  }
  const int units = static_cast<int>(kv_units * head_groups(group, hg));
  const bool forced = (flags & TQ_MATRIX_PRODUCTS) != 0;
  const bool takes_mx = mx_shape(fmt, head_dim, group) && (flags & TQ_F32_PRODUCTS) == 0;
  const int64_t blocks = std::max<int64_t>(1, (seq_len + mx::kStride - 1) / mx::kStride);
  const int min_blocks = mx_min_blocks_per_split(head_dim);
  const int ns4 = default_splits(units, seq_len, num_cus, 1);
  const bool one_launch = forced || (flags & TQ_ONE_LAUNCH) != 0;
  const bool many_units = 2 * units > num_cus || kv_units * head_groups(group, even_hg(group)) > num_cus;
  if (n_splits <= 0 && one_split(seq_len, fmt, head_dim, hg, many_units, one_launch)) {
    // the matrix kernel where its own plan is one split of enough blocks: 24
    // layers x 8 KV heads x 512 4-bit tokens in groups of 4 at head_dim 128
    // 7.3 us against 9.0, at 64 6.2 against 6.3, 2-bit rows 7.2 against 8.2
    if (!forced && !(takes_mx && blocks / std::min<int64_t>(blocks, ns4) >= min_blocks)) return {SplitKernel::Fp32, 1, hg};
    n_splits = 1;
  }
  if (takes_mx) {
    const int ns = n_splits > 0 ? n_splits : ns4;
    const bool runs = forced || blocks / std::min<int64_t>(blocks, ns) >= min_blocks;
    // Units of 8 heads where units of 4 would run: one read of the rows and
    // one lookup of every code for 8 heads, in products whose columns 4 heads
    // fill by half.  Measured on MI355X, units of 4 -> 8: 4 KV heads x 30001
    // 4-bit tokens at head_dim 128 13.6 -> 11.6 us, 8 x 32768 in groups of 16
    // 28.8 -> 19.6, 12 layers x 8 x 8192 45.5 -> 34.2, 2 x 131072 at 256 31.5
    // -> 23.8, 24 layers x 2 x 8192 at 256 59.7 -> 33.4.  An explicit count
    // has to give more than half of the CUs a workgroup.
    if (group % 8 == 0) {
      int ns8 = default_splits(units / 2, seq_len, num_cus, 1);
      if (ns4 == 1 && !splits_pay_units_of_8(units / 2, ns8, blocks, head_dim)) ns8 = 1;
      if (n_splits <= 0 || n_splits == ns8) {
        if (forced || blocks / std::min<int64_t>(blocks, ns4) >= min_blocks) return {SplitKernel::Mx, ns8, 8};
      } else if (forced || (runs && static_cast<int64_t>(units / 2) * n_splits > num_cus / 2)) {
        return {SplitKernel::Mx, n_splits, 8};
      }
    }
    if (runs) return {SplitKernel::Mx, ns, hg};
  }
  if (n_splits > 0) return {SplitKernel::Fp32, n_splits, hg};
  // one split per kMinTokensPerSplit tokens at most, as in default_splits
  const int64_t by_len = (seq_len + kMinTokensPerSplit - 1) / kMinTokensPerSplit;
  const bool packed = packed_rows(fmt);
  const int64_t rows = decode_block_rows(packed ? fmt : 16, head_dim);  // dense rows: one plan for both types
  const Work work{units, (seq_len + rows - 1) / rows, load_overhead(head_dim, hg), num_cus};
  int ns0 = default_splits(units, seq_len, num_cus, 2);
  if (ns0 < by_len) ns0 = static_cast<int>(std::min<int64_t>(balanced_splits(work, ns0, packed), by_len));
  // Groups cut into units of 4: where the units that divide the group fill the
  // CUs with one split each, the splits that fewer units take have to pay for
  // a merge of their own.  Below 2/3 of the work one split is the faster one:
  // 96 units x 5 heads, 3-bit rows at head_dim 128, 768 tokens 12.6 us in units
  // of 1, 16.3 cut with 2 splits, 12.6 cut with one, 1536 tokens 20.2, 22.2 and
  // 20.5; 128 x 3 heads 768 tokens 12.4, 13.2, 12.5, 1024 15.1, 14.0, 15.2; 64 x 7
  // heads 4-bit at 64, 768 tokens 9.0, 10.6, 7.9.  Fewer units than a third of
  // the CUs leave too many of them idle: 64 x 3 heads 768 tokens 11.7, 10.7, 12.6.
  const int own = even_hg(group);
  if (hg > own && 3 * units >= num_cus && 3 * work.of(1) <= 2 * work.of(ns0)) ns0 = 1;
  // As with explicit counts: 160 x 6 heads, 1311 4-bit scaled tokens at 128 24.8
  // us in one split of 480 units of 2, 25.9 in one of 320 units of 4.
  if (hg > own && ns0 == 1 && units > num_cus && kv_units * head_groups(group, own) <= 2 * num_cus) hg = own;
  return {SplitKernel::Fp32, ns0, hg};
}

// Fills the split plan of a decode call over `fmt` rows (see
// decode_block_rows) with decode `flags`; every split gets at least one block.
int make_plan(int num_layers, int kv_heads, int query_heads, int64_t seq_len, int n_splits, int fmt, int head_dim,
              int flags, Plan* p) {
  if (num_layers <= 0 || kv_heads <= 0 || query_heads <= 0)
    return fail(TQ_ERR_BAD_ARG, "num_layers, kv_heads and query_heads must be positive");
  if (query_heads % kv_heads != 0)
    return fail(TQ_ERR_BAD_ARG, "query head count " + std::to_string(query_heads) + " must be divisible by kv_heads " +
                                    std::to_string(kv_heads));
  if (seq_len < 0) return fail(TQ_ERR_BAD_ARG, "seq_len must be non-negative");
  const int group = query_heads / kv_heads;
  const int64_t kv_units = static_cast<int64_t>(num_layers) * kv_heads;
  p->hg = pick_hg(group, kv_units, seq_len, fmt, head_dim);
  p->n_hgroups = head_groups(group, p->hg);
  // One launch holds at most 2^32 - 1 work-items: units x splits workgroups.
  const int64_t max_wg = ((int64_t(1) << 32) - 1) / kBlock;
  int64_t units = kv_units * p->n_hgroups;
  if (units > max_wg)
    return fail(TQ_ERR_BAD_ARG, "num_layers x kv_heads x head groups exceeds one launch; decode fewer layers per call");
  if ((flags & TQ_F32_PRODUCTS) != 0 && (flags & TQ_MATRIX_PRODUCTS) != 0)
    return fail(TQ_ERR_BAD_ARG, "TQ_F32_PRODUCTS and TQ_MATRIX_PRODUCTS exclude each other");
  const KernelChoice kc = choose_kernel(kv_units, seq_len, n_splits, fmt, head_dim, group, flags, device_cu_count());
  p->kernel = kc.kernel;
  p->hg = kc.hg;
  p->n_hgroups = head_groups(group, p->hg);
  units = kv_units * p->n_hgroups;
  p->units = static_cast<int>(units);
  const int ns = kc.n_splits;
  if (ns > kMaxSplits) return fail(TQ_ERR_BAD_ARG, "n_splits must be at most " + std::to_string(kMaxSplits));
  p->tokens_per_iter = p->kernel == SplitKernel::Mx
                           ? 0
                           : fp32_tokens_per_iter(fmt, head_dim, p->hg, seq_len, std::min<int64_t>(ns, max_wg / units));
  p->block_rows = p->kernel == SplitKernel::Mx ? mx::kStride : decode_block_rows(fmt, head_dim, p->tokens_per_iter);
  const int64_t blocks = std::max<int64_t>(1, (seq_len + p->block_rows - 1) / p->block_rows);
  p->n_splits = static_cast<int>(std::min<int64_t>({blocks, static_cast<int64_t>(ns), max_wg / units}));
  return TQ_OK;
}

template <class Fmt, int D, int HG, bool QF16, bool SC, int U>
void launch_decode_u(const DecodeArgs& a, int nblk, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  if (start != nullptr || stop != nullptr)
    hipExtLaunchKernelGGL((decode_kernel<Fmt, D, HG, QF16, SC, U>), dim3(nblk), dim3(kBlock), 0, stream, start, stop,
                          0, a);
  else
    hipLaunchKernelGGL((decode_kernel<Fmt, D, HG, QF16, SC, U>), dim3(nblk), dim3(kBlock), 0, stream, a);
}

template <class Fmt, int D, int HG, bool QF16, bool SC>
void launch_decode_q(const DecodeArgs& a, int nblk, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  if constexpr (wide_iter_instance<Fmt, D, HG>()) {
    if (a.wide_iter) return launch_decode_u<Fmt, D, HG, QF16, SC, kWideTokensPerIter>(a, nblk, stream, start, stop);
  }
  launch_decode_u<Fmt, D, HG, QF16, SC, kTokensPerIter>(a, nblk, stream, start, stop);
}

// Scaled kernels exist for packed rows only (the host never passes scales
// with dense rows).
template <class Fmt, int D, int HG, bool QF16>
void launch_decode_s(const DecodeArgs& a, int nblk, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  if constexpr (Fmt::kHasLut) {
    if (a.k_scales != nullptr) return launch_decode_q<Fmt, D, HG, QF16, true>(a, nblk, stream, start, stop);
  }
  launch_decode_q<Fmt, D, HG, QF16, false>(a, nblk, stream, start, stop);
}

template <class Fmt, int D, int HG>
void launch_decode(const DecodeArgs& a, int nblk, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  if (a.q_f16)
    launch_decode_s<Fmt, D, HG, true>(a, nblk, stream, start, stop);
  else
    launch_decode_s<Fmt, D, HG, false>(a, nblk, stream, start, stop);
}

template <class Fmt, int D>
int dispatch_hg(const DecodeArgs& a, int hg, int nblk, hipStream_t s, hipEvent_t e0, hipEvent_t e1) {
  switch (hg) {
    case 1:
      launch_decode<Fmt, D, 1>(a, nblk, s, e0, e1);
      break;
    case 2:
      launch_decode<Fmt, D, 2>(a, nblk, s, e0, e1);
      break;
    case 4:
      launch_decode<Fmt, D, 4>(a, nblk, s, e0, e1);
      break;
    default:
      return fail(TQ_ERR_UNSUPPORTED, "unsupported query-head group");
  }
  return TQ_OK;
}

template <class Fmt>
int dispatch_d(const DecodeArgs& a, int head_dim, int hg, int nblk, hipStream_t s, hipEvent_t e0, hipEvent_t e1) {
  switch (head_dim) {
    case 64:
      return dispatch_hg<Fmt, 64>(a, hg, nblk, s, e0, e1);
    case 128:
      return dispatch_hg<Fmt, 128>(a, hg, nblk, s, e0, e1);
    case 256:
      return dispatch_hg<Fmt, 256>(a, hg, nblk, s, e0, e1);
    default:
      return fail(TQ_ERR_UNSUPPORTED, "Unsupported head dimension: " + std::to_string(head_dim));
  }
}

// Common front end of tq_decode / tq_decode_dense.  fmt: 2/3/4 packed bits,
// 16 dense fp16, 32 dense fp32.
// The new token of tq_decode_append.
struct AppendSpec {
  const void* keys;
  const void* values;
  int dtype;  // TQ_F32 or TQ_F16
  const float* key_boundaries;
  const float* value_boundaries;
  int flags;  // TQ_ROTATE_KEYS | TQ_ROTATE_VALUES
};

int launch_fp32(const DecodeArgs& a, int fmt, int head_dim, int hg, int nblk, hipStream_t stream, hipEvent_t start,
                hipEvent_t stop);
struct ProfileEvents {
  hipEvent_t start = nullptr, stop = nullptr;
};
int launch_merge(const MergeArgs& m, int num_layers, int query_heads, int head_dim, hipStream_t stream,
                 bool profiled, const ProfileEvents* caller_events);

template <int D, bool QF16, int BITS, int HG>
void launch_mx_t(const DecodeArgs& a, dim3 grid, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  if (start != nullptr || stop != nullptr)
    hipExtLaunchKernelGGL((decode_mx_kernel<D, QF16, BITS, HG>), grid, dim3(mx::threads_of<D>()), 0, stream, start,
                          stop, 0, a);
  else
    hipLaunchKernelGGL((decode_mx_kernel<D, QF16, BITS, HG>), grid, dim3(mx::threads_of<D>()), 0, stream, a);
}

template <int D, int BITS>
void launch_mx_d(const DecodeArgs& a, dim3 grid, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  const bool eight = a.n_hgroups * 8 == a.group;
  if (a.q_f16)
    eight ? launch_mx_t<D, true, BITS, 8>(a, grid, stream, start, stop)
          : launch_mx_t<D, true, BITS, 4>(a, grid, stream, start, stop);
  else
    eight ? launch_mx_t<D, false, BITS, 8>(a, grid, stream, start, stop)
          : launch_mx_t<D, false, BITS, 4>(a, grid, stream, start, stop);
}

// Grid (split, head group, layer x KV head) of decode_mx_kernel.
int launch_mx(const DecodeArgs& a, int fmt, int head_dim, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  constexpr int kMaxGridYZ = 65535;
  const int lkv = a.num_layers * a.kv_heads;
  if (lkv > kMaxGridYZ || a.n_hgroups > kMaxGridYZ)
    return fail(TQ_ERR_BAD_ARG, "num_layers x kv_heads must be at most 65535 per call; decode fewer layers per call");
  const dim3 grid(a.n_splits, a.n_hgroups, lkv);
  if (fmt == 2 && head_dim == 128) {
    launch_mx_d<128, 2>(a, grid, stream, start, stop);
    return TQ_OK;
  }
  if (fmt != 4) return fail(TQ_ERR_UNSUPPORTED, "decode_mx_kernel: unsupported bit width " + std::to_string(fmt));
  switch (head_dim) {
    case 64:
      launch_mx_d<64, 4>(a, grid, stream, start, stop);
      return TQ_OK;
    case 128:
      launch_mx_d<128, 4>(a, grid, stream, start, stop);
      return TQ_OK;
    case 256:
      launch_mx_d<256, 4>(a, grid, stream, start, stop);
      return TQ_OK;
    default:
      return fail(TQ_ERR_UNSUPPORTED, "decode_mx_kernel: unsupported head dimension " + std::to_string(head_dim));
  }
}

int decode_common(int fmt, const void* query, int query_dtype, int num_layers, int query_heads, int kv_heads,
                  int head_dim, const void* keys, const void* values, int64_t capacity, int64_t seq_len,
                  const float* cent_k, const float* cent_v, const float* signs_left, const float* signs_right,
                  int flags, const float* cur_k, const float* cur_v, int n_splits, void* workspace,
                  size_t workspace_bytes, float* out, hipStream_t stream, hipEvent_t start, hipEvent_t stop,
                  const AppendSpec* app = nullptr,
                  const float* k_scales = nullptr, const float* v_scales = nullptr,
                  const ProfileEvents* merge_events = nullptr) {
  int rc = check_geometry(head_dim, 0);
  if (rc) return rc;
  if ((k_scales == nullptr) != (v_scales == nullptr))
    return fail(TQ_ERR_BAD_ARG, "key_scales and value_scales must both be given or both be null");
  if (k_scales != nullptr && app != nullptr)
    return fail(TQ_ERR_BAD_ARG, "per-vector scales are not supported by the fused append + decode");
  if (query == nullptr || out == nullptr || workspace == nullptr)
    return fail(TQ_ERR_BAD_ARG, "query, out and workspace must be non-null");
  if (query_dtype != TQ_F32 && query_dtype != TQ_F16) return fail(TQ_ERR_BAD_ARG, "query dtype must be F32 or F16");
  if (seq_len > 0 && (keys == nullptr || values == nullptr))
    return fail(TQ_ERR_BAD_ARG, "key and value slabs must be non-null");
  if (capacity < seq_len) return fail(TQ_ERR_BAD_ARG, "capacity must be >= seq_len");
  if ((cur_k == nullptr) != (cur_v == nullptr))
    return fail(TQ_ERR_BAD_ARG, "current_keys and current_values must both be given or both be null");
  if (app != nullptr) {
    if (app->keys == nullptr || app->values == nullptr || app->key_boundaries == nullptr ||
        app->value_boundaries == nullptr || keys == nullptr || values == nullptr)
      return fail(TQ_ERR_BAD_ARG, "new keys/values, boundaries and both slabs must be non-null");
    if (seq_len >= capacity) return fail(TQ_ERR_BAD_ARG, "slab is full: seq_len must be below capacity");
    if (app->dtype != TQ_F32 && app->dtype != TQ_F16) return fail(TQ_ERR_BAD_ARG, "new key/value dtype must be F32 or F16");
    if ((app->flags & (TQ_ROTATE_KEYS | TQ_ROTATE_VALUES)) && (signs_left == nullptr || signs_right == nullptr))
      return fail(TQ_ERR_BAD_ARG, "rotation flags need signs_left and signs_right");
  }
  if ((flags & (TQ_ROTATE_QUERY | TQ_INVERSE_OUTPUT)) && (signs_left == nullptr || signs_right == nullptr))
    return fail(TQ_ERR_BAD_ARG, "rotation flags need signs_left and signs_right");
  const bool packed = fmt == 2 || fmt == 3 || fmt == 4;
  if (packed && (cent_k == nullptr || cent_v == nullptr))
    return fail(TQ_ERR_BAD_ARG, "key and value centroids must be non-null");
  const int64_t row_bytes = packed ? static_cast<int64_t>(packed_words(head_dim, fmt)) * 4
                                   : static_cast<int64_t>(head_dim) * (fmt == 16 ? 2 : 4);
  if (capacity * row_bytes >= (1LL << 31))
    return fail(TQ_ERR_BAD_ARG, "capacity * row bytes must stay below 2 GiB per (layer, KV head)");
  Plan p;
  rc = make_plan(num_layers, kv_heads, query_heads, seq_len, n_splits, fmt, head_dim, flags, &p);
  if (rc) return rc;
  if (p.n_splits > 1 &&
      static_cast<int64_t>(num_layers) * query_heads * (head_dim / kMergeDims) > ((int64_t(1) << 32) - 1) / kBlock)
    return fail(TQ_ERR_BAD_ARG, "num_layers x query_heads exceeds one merge launch; decode fewer layers per call");

  uint8_t* ws = static_cast<uint8_t*>(workspace);
  const WsLayout wl = workspace_layout(static_cast<int64_t>(num_layers) * query_heads,
                                      static_cast<int64_t>(num_layers) * kv_heads, head_dim, p.n_splits);
  if (workspace_bytes < wl.total)
    return fail(TQ_ERR_BAD_ARG, "workspace of " + std::to_string(workspace_bytes) + " bytes is smaller than the " +
                                    std::to_string(wl.total) + " bytes this call needs (" +
                                    std::to_string(p.n_splits) + " splits)");

  DecodeArgs a{};
  a.q = query;
  a.q_f16 = query_dtype == TQ_F16;
  a.k = static_cast<const uint8_t*>(keys);
  a.v = static_cast<const uint8_t*>(values);
  a.cap = capacity;
  a.seq_len = seq_len;
  a.num_layers = num_layers;
  a.query_heads = query_heads;
  a.kv_heads = kv_heads;
  a.group = query_heads / kv_heads;
  a.n_hgroups = p.n_hgroups;
  a.cent_k = cent_k;
  a.cent_v = cent_v;
  a.signs_left = signs_left;
  a.signs_right = signs_right;
  a.sqrt_d = sqrt_f32(head_dim);
  a.q_scale = static_cast<float>(1.4426950408889634 / std::sqrt(static_cast<double>(head_dim)));
  a.rotate_query = (flags & TQ_ROTATE_QUERY) != 0;
  a.inverse_output = (flags & TQ_INVERSE_OUTPUT) != 0;
  a.cur_k = cur_k;
  a.cur_v = cur_v;
  a.k_scales = k_scales;
  a.v_scales = v_scales;
  if (app != nullptr) {
    a.new_k = app->keys;
    a.new_v = app->values;
    a.new_f16 = app->dtype == TQ_F16;
    a.bnd_k = app->key_boundaries;
    a.bnd_v = app->value_boundaries;
    a.k_slab = const_cast<uint32_t*>(static_cast<const uint32_t*>(keys));
    a.v_slab = const_cast<uint32_t*>(static_cast<const uint32_t*>(values));
    a.rotate_new_k = (app->flags & TQ_ROTATE_KEYS) != 0;
    a.rotate_new_v = (app->flags & TQ_ROTATE_VALUES) != 0;
  }
  a.n_splits = p.n_splits;
  a.row_splits = p.n_splits;
  if (app != nullptr && p.n_splits > 1) {
    // split 0 packs the new token; it reads no rows when the other splits
    // can take them all without a longer share
    const int64_t blocks = (seq_len + p.block_rows - 1) / p.block_rows;
    const int64_t n = p.n_splits;
    if ((blocks + n - 2) / (n - 1) <= (blocks + n - 1) / n) a.row_splits = p.n_splits - 1;
  }
  a.wide_iter = p.tokens_per_iter == kWideTokensPerIter;
  a.ws_ml = reinterpret_cast<float*>(ws + wl.ml);
  a.ws_acc = reinterpret_cast<float*>(ws + wl.acc);
  a.ws_cur_s = reinterpret_cast<float*>(ws + wl.cur_s);
  a.ws_cur_v = reinterpret_cast<float*>(ws + wl.cur_v);
  a.out = out;
  const int nblk = p.units * p.n_splits;
  MergeArgs m{};
  m.query_heads = query_heads;
  m.kv_heads = kv_heads;
  m.group = a.group;
  m.n_splits = p.n_splits;
  m.ws_ml = a.ws_ml;
  m.ws_acc = a.ws_acc;
  m.cur_s = (cur_k != nullptr || app != nullptr) ? a.ws_cur_s : nullptr;
  m.cur_v = a.ws_cur_v;
  m.out = out;

  if (p.kernel == SplitKernel::Mx) {
    rc = launch_mx(a, fmt, head_dim, stream, start, stop);
  } else {
    rc = launch_fp32(a, fmt, head_dim, p.hg, nblk, stream, start, stop);
  }
  if (rc) return rc;
  rc = launch_status("decode_kernel");
  if (rc || p.n_splits == 1) return rc;
  return launch_merge(m, num_layers, query_heads, head_dim, stream, start != nullptr || stop != nullptr, merge_events);
}

int launch_fp32(const DecodeArgs& a, int fmt, int head_dim, int hg, int nblk, hipStream_t stream, hipEvent_t start,
                hipEvent_t stop) {
  int rc;
  switch (fmt) {
    case 2:
      rc = dispatch_d<PackedB2>(a, head_dim, hg, nblk, stream, start, stop);
      break;
    case 3:
      rc = dispatch_d<PackedB3>(a, head_dim, hg, nblk, stream, start, stop);
      break;
    case 4:
      rc = dispatch_d<PackedB4>(a, head_dim, hg, nblk, stream, start, stop);
      break;
    case 16:
      rc = dispatch_d<DenseF16>(a, head_dim, hg, nblk, stream, start, stop);
      break;
    case 32:
      rc = dispatch_d<DenseF32>(a, head_dim, hg, nblk, stream, start, stop);
      break;
    default:
      return fail(TQ_ERR_UNSUPPORTED, "Unsupported bit width: " + std::to_string(fmt));
  }
  return rc;
}

// Events of the merge launch of a timed call whose caller passes none, one
// pair per device (created on first use with that device current; never
// read, and shared by every stream of the device).  A timed call launches
// the merge kernel with profiling too: a dispatch launched with profiling
// events right after one launched without starts on six of the eight XCDs
// about 1.2 us after the other two (measured on MI355X for the split kernel
// after an unprofiled merge: median workgroup start skew 1.25 us, against
// 0.13 us with no events and 0.15 us with every dispatch profiled), and the
// split kernel's events would count that delay as its own time.
std::mutex g_profile_mutex;
ProfileEvents g_merge_events[kMaxDevices];

int merge_profile_events(ProfileEvents* ev) {
  int dev = -1;
  const hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(TQ_ERR_LAUNCH, std::string("no current HIP device: ") + hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices)
    return fail(TQ_ERR_UNSUPPORTED, "device index " + std::to_string(dev) + " out of range");
  std::lock_guard<std::mutex> lock(g_profile_mutex);
  ProfileEvents& p = g_merge_events[dev];
  if (p.start == nullptr) {
    hipEvent_t a = nullptr, b = nullptr;
    hipError_t r = hipEventCreate(&a);
    if (r == hipSuccess) r = hipEventCreate(&b);
    if (r != hipSuccess) {
      if (a != nullptr) (void)hipEventDestroy(a);
      return fail(TQ_ERR_LAUNCH, std::string("hipEventCreate failed: ") + hipGetErrorString(r));
    }
    p.start = a;
    p.stop = b;
  }
  *ev = p;
  return TQ_OK;
}

template <int D>
void launch_merge_d(const MergeArgs& m, unsigned mblk, hipStream_t stream, const ProfileEvents* ev) {
  if (ev != nullptr)
    hipExtLaunchKernelGGL(merge_kernel<D>, dim3(mblk), dim3(kBlock), 0, stream, ev->start, ev->stop, 0, m);
  else
    hipLaunchKernelGGL(merge_kernel<D>, dim3(mblk), dim3(kBlock), 0, stream, m);
}

int launch_merge(const MergeArgs& m, int num_layers, int query_heads, int head_dim, hipStream_t stream,
                 bool profiled, const ProfileEvents* caller_events) {
  const unsigned mblk =
      static_cast<unsigned>(static_cast<int64_t>(num_layers) * query_heads * (head_dim / kMergeDims));
  ProfileEvents ev;
  if (caller_events != nullptr) {
    ev = *caller_events;
  } else if (profiled) {
    const int rc = merge_profile_events(&ev);
    if (rc) return rc;
  }
  const ProfileEvents* evp = (profiled || caller_events != nullptr) ? &ev : nullptr;
  switch (head_dim) {
    case 64:
      launch_merge_d<64>(m, mblk, stream, evp);
      break;
    case 128:
      launch_merge_d<128>(m, mblk, stream, evp);
      break;
    default:
      launch_merge_d<256>(m, mblk, stream, evp);
      break;
  }
  return launch_status("merge_kernel");
}

template <template <int> class Body, typename... Args>
int with_d(int head_dim, Args&&... args) {
  switch (head_dim) {
    case 64:
      return Body<64>::run(args...);
    case 128:
      return Body<128>::run(args...);
    case 256:
      return Body<256>::run(args...);
  }
  return fail(TQ_ERR_UNSUPPORTED, "Unsupported head dimension: " + std::to_string(head_dim));
}

// Workgroups per launch of the row kernels (fwht, append, unpack, rotary,
// gate).  A HIP launch holds at most 2^32 - 1 work-items; larger calls are cut
// into launches of at most this many workgroups, in stream order.
constexpr int64_t kMaxLaunchBlocks = int64_t(1) << 20;

// Grid of one launch of a kernel with a wavefront per row, `rows` left to do.
dim3 row_grid(int64_t rows) {
  return dim3(static_cast<unsigned>(std::min((rows + kWavesPerBlock - 1) / kWavesPerBlock, kMaxLaunchBlocks)));
}

template <int D>
struct FwhtBody {
  static int run(const void* x, int x_dtype, float* y, int64_t rows, const float* s_first, const float* s_second,
                 hipStream_t stream) {
    const float sd = sqrt_f32(D);
    const int64_t chunk = kMaxLaunchBlocks * kWavesPerBlock;  // one wavefront per row
    for (int64_t r0 = 0; r0 < rows; r0 += chunk) {
      const int64_t n = std::min(chunk, rows - r0);
      const unsigned nblk = static_cast<unsigned>((n + kWavesPerBlock - 1) / kWavesPerBlock);
      if (x_dtype == TQ_F16)
        hipLaunchKernelGGL((fwht_kernel<D, __half>), dim3(nblk), dim3(kBlock), 0, stream,
                           static_cast<const __half*>(x) + r0 * D, y + r0 * D, n, s_first, s_second, sd);
      else
        hipLaunchKernelGGL((fwht_kernel<D, float>), dim3(nblk), dim3(kBlock), 0, stream,
                           static_cast<const float*>(x) + r0 * D, y + r0 * D, n, s_first, s_second, sd);
      const int rc = launch_status("fwht_kernel");
      if (rc) return rc;
    }
    return TQ_OK;
  }
};

struct AppendParams {
  const void* keys;
  const void* values;
  int dtype;
  int64_t rows;
  int streams;
  int64_t seq_new;
  int rotate_keys, rotate_values;
  const float* signs_left;
  const float* signs_right;
  const float* key_bnd;
  const float* value_bnd;
  const float* key_cent;
  const float* value_cent;
  uint32_t* key_codes;
  uint32_t* value_codes;
  int64_t capacity, offset;
  float* key_out;
  float* value_out;
  bool dequant;
  // per-vector scales (scaled mode): scale slabs [L, Hkv, capacity] written
  // by the packing path; the dequantizing path multiplies them in.
  bool scaled;
  float* key_scales;
  float* value_scales;
};

// One launch over rows [g0 * seq_new + t0, + rows) of p: `groups` whole
// (layer, head) groups from group g0 (t0 = 0), or `rows` tokens of group g0
// from token t0.
template <int D, int BITS, typename T, bool DQ, bool SC>
int launch_append_part(const AppendParams& p, int64_t g0, int64_t t0, int64_t seq_part, int64_t rows,
                       hipStream_t stream) {
  constexpr int W = D * BITS / 32;
  constexpr int RPB = kBlock / (D / 16);
  const int64_t row0 = g0 * p.seq_new + t0;
  AppendArgs a{};
  a.keys = static_cast<const T*>(p.keys) + row0 * D;
  a.values = static_cast<const T*>(p.values) + row0 * D;
  a.rows = static_cast<uint32_t>(rows);
  a.seq_new = make_fast_div(static_cast<uint32_t>(seq_part));
  a.rotate_keys = p.rotate_keys;
  a.rotate_values = p.rotate_values;
  a.signs_left = p.signs_left;
  a.signs_right = p.signs_right;
  a.sqrt_d = sqrt_f32(D);
  a.key_bnd = p.key_bnd;
  a.value_bnd = p.value_bnd;
  a.key_cent = p.key_cent;
  a.value_cent = p.value_cent;
  a.key_codes = p.key_codes ? p.key_codes + g0 * p.capacity * W : nullptr;
  a.value_codes = p.value_codes ? p.value_codes + g0 * p.capacity * W : nullptr;
  a.capacity = p.capacity;
  a.offset = p.offset + t0;
  a.key_out = p.key_out ? p.key_out + row0 * D : nullptr;
  a.value_out = p.value_out ? p.value_out + row0 * D : nullptr;
  a.key_scales = p.key_scales ? p.key_scales + g0 * p.capacity : nullptr;
  a.value_scales = p.value_scales ? p.value_scales + g0 * p.capacity : nullptr;
  const uintptr_t bits = reinterpret_cast<uintptr_t>(a.keys) | reinterpret_cast<uintptr_t>(a.values) |
                         reinterpret_cast<uintptr_t>(a.key_out) | reinterpret_cast<uintptr_t>(a.value_out);
  a.wide = bits % 16 == 0;
  if (rows * p.streams <= append_few_rows<D, BITS, DQ, SC>()) {
    const unsigned few = static_cast<unsigned>((rows + kWavesPerBlock - 1) / kWavesPerBlock);
    hipLaunchKernelGGL((append_few_kernel<D, BITS, T, DQ, SC>), dim3(few, p.streams), dim3(kBlock), 0, stream, a);
    return launch_status("append_few_kernel");
  }
  const int64_t nblk = std::min<int64_t>((rows + RPB - 1) / RPB, kAppendMaxBlocks / p.streams);
  hipLaunchKernelGGL((append_kernel<D, BITS, T, DQ, SC>), dim3(static_cast<unsigned>(nblk), p.streams), dim3(kBlock),
                     0, stream, a);
  return launch_status("append_kernel");
}

// rows = groups * seq_new items per stream; at most kMaxAppendRows rows of a
// stream per launch, cut at whole groups, or at tokens when one group alone is
// larger: row numbers are 32-bit, and a wavefront per row of both streams has to
// stay within one launch's work-items.  Cut at 2^21 rows, a call of 2.3 M took
// 312 us against 302.
constexpr int64_t kMaxAppendRows = int64_t(1) << 23;

template <int D, int BITS, typename T, bool DQ, bool SC>
int launch_append(const AppendParams& p, hipStream_t stream) {
  const int64_t max_rows = kMaxAppendRows;
  const int64_t groups = p.rows / p.seq_new;
  if (p.seq_new <= max_rows) {
    const int64_t per = max_rows / p.seq_new;
    for (int64_t g0 = 0; g0 < groups; g0 += per) {
      const int64_t ng = std::min(per, groups - g0);
      const int rc = launch_append_part<D, BITS, T, DQ, SC>(p, g0, 0, p.seq_new, ng * p.seq_new, stream);
      if (rc) return rc;
    }
    return TQ_OK;
  }
  for (int64_t g = 0; g < groups; ++g)
    for (int64_t t0 = 0; t0 < p.seq_new; t0 += max_rows) {
      const int64_t nt = std::min(max_rows, p.seq_new - t0);
      const int rc = launch_append_part<D, BITS, T, DQ, SC>(p, g, t0, nt, nt, stream);
      if (rc) return rc;
    }
  return TQ_OK;
}

template <int D, int BITS, typename T>
int append_mode(const AppendParams& p, hipStream_t stream) {
  if (p.scaled)
    return p.dequant ? launch_append<D, BITS, T, true, true>(p, stream) : launch_append<D, BITS, T, false, true>(p, stream);
  return p.dequant ? launch_append<D, BITS, T, true, false>(p, stream) : launch_append<D, BITS, T, false, false>(p, stream);
}

template <int D, int BITS>
int append_dtype(const AppendParams& p, hipStream_t stream) {
  return p.dtype == TQ_F16 ? append_mode<D, BITS, __half>(p, stream) : append_mode<D, BITS, float>(p, stream);
}

template <int D>
struct AppendBody {
  static int run(const AppendParams& p, int bits, hipStream_t stream) {
    switch (bits) {
      case 2:
        return append_dtype<D, 2>(p, stream);
      case 3:
        return append_dtype<D, 3>(p, stream);
      case 4:
        return append_dtype<D, 4>(p, stream);
      default:
        return fail(TQ_ERR_UNSUPPORTED, "Unsupported bit width: " + std::to_string(bits));
    }
  }
};

template <int D>
struct StageBody {
  // op 0: score, op 2: accumulate
  template <class Fmt>
  static void go(int op, const float* a, const uint8_t* codes, int batch, int64_t seq_len, const float* cent,
                 float* out, hipStream_t stream) {
    constexpr int LPT = D / Fmt::kSliceDims;
    constexpr int TPB = kWavesPerBlock * (kWave / LPT);
    if (op == 0) {
      const int64_t nx = (seq_len + TPB - 1) / TPB;
      hipLaunchKernelGGL((score_kernel<Fmt, D>), dim3(static_cast<unsigned>(nx), batch), dim3(kBlock), 0, stream, a,
                         codes, seq_len, cent, out);
    } else {
      hipLaunchKernelGGL((accumulate_kernel<Fmt, D>), dim3(batch), dim3(kBlock), 0, stream, a, codes, seq_len, cent,
                         out);
    }
  }
  static int run(int op, int bits, const float* a, const uint8_t* codes, int batch, int64_t seq_len,
                 const float* cent, float* out, hipStream_t stream) {
    switch (bits) {
      case 2:
        go<PackedB2>(op, a, codes, batch, seq_len, cent, out, stream);
        break;
      case 3:
        go<PackedB3>(op, a, codes, batch, seq_len, cent, out, stream);
        break;
      case 4:
        go<PackedB4>(op, a, codes, batch, seq_len, cent, out, stream);
        break;
      default:
        return fail(TQ_ERR_UNSUPPORTED, "Unsupported bit width: " + std::to_string(bits));
    }
    return launch_status(op == 0 ? "score_kernel" : "accumulate_kernel");
  }
};

template <int D>
struct UnpackBody {
  // One launch: `groups` groups of seq_len tokens (group stride `capacity`
  // rows) into out [groups, seq_len, D].
  template <int BITS>
  static int part(const uint32_t* codes, int64_t groups, int64_t capacity, int64_t seq_len, const float* cent,
                  const float* scales, float* out, hipStream_t stream) {
    const unsigned nblk = static_cast<unsigned>((groups * seq_len * D + kBlock - 1) / kBlock);
    hipLaunchKernelGGL(unpack_kernel<BITS>, dim3(nblk), dim3(kBlock), 0, stream, codes, groups, capacity, seq_len, D,
                       cent, scales, out);
    return launch_status("unpack_kernel");
  }
  // At most kMaxLaunchBlocks workgroups (one thread per output value) per
  // launch: cut at whole groups, or at tokens when one group alone is larger.
  template <int BITS>
  static int chunks(const uint32_t* codes, int64_t groups, int64_t capacity, int64_t seq_len, const float* cent,
                    const float* scales, float* out, hipStream_t stream) {
    constexpr int W = D * BITS / 32;
    const int64_t max_tokens = kMaxLaunchBlocks * kBlock / D;
    if (seq_len <= max_tokens) {
      const int64_t per = max_tokens / seq_len;
      for (int64_t g0 = 0; g0 < groups; g0 += per) {
        const int64_t ng = std::min(per, groups - g0);
        const int rc = part<BITS>(codes + g0 * capacity * W, ng, capacity, seq_len, cent,
                                  scales ? scales + g0 * capacity : nullptr, out + g0 * seq_len * D, stream);
        if (rc) return rc;
      }
      return TQ_OK;
    }
    for (int64_t g = 0; g < groups; ++g)
      for (int64_t t0 = 0; t0 < seq_len; t0 += max_tokens) {
        const int64_t nt = std::min(max_tokens, seq_len - t0);
        const int rc = part<BITS>(codes + (g * capacity + t0) * W, 1, capacity, nt, cent,
                                  scales ? scales + g * capacity + t0 : nullptr, out + (g * seq_len + t0) * D, stream);
        if (rc) return rc;
      }
    return TQ_OK;
  }
  static int run(const uint32_t* codes, int64_t groups, int64_t capacity, int64_t seq_len, int bits,
                 const float* cent, const float* scales, float* out, hipStream_t stream) {
    switch (bits) {
      case 2:
        return chunks<2>(codes, groups, capacity, seq_len, cent, scales, out, stream);
      case 3:
        return chunks<3>(codes, groups, capacity, seq_len, cent, scales, out, stream);
      case 4:
        return chunks<4>(codes, groups, capacity, seq_len, cent, scales, out, stream);
      default:
        return fail(TQ_ERR_UNSUPPORTED, "Unsupported bit width: " + std::to_string(bits));
    }
  }
};

int append_impl(const void* keys, const void* values, int dtype, int num_layers, int kv_heads, int64_t seq_new,
                int head_dim, int bits, const float* signs_left, const float* signs_right, int flags,
                const float* key_boundaries, const float* value_boundaries, uint32_t* key_codes,
                uint32_t* value_codes, int64_t capacity, int64_t offset, float* key_scales, float* value_scales,
                hipStream_t stream) {
  int rc = check_geometry(head_dim, bits);
  if (rc) return rc;
  if (num_layers <= 0 || kv_heads <= 0) return fail(TQ_ERR_BAD_ARG, "num_layers and kv_heads must be positive");
  if (seq_new < 0 || offset < 0) return fail(TQ_ERR_BAD_ARG, "seq_new and offset must be non-negative");
  if (offset + seq_new > capacity) return fail(TQ_ERR_BAD_ARG, "append past slab capacity");
  if (seq_new == 0) return TQ_OK;
  if (!keys || !values || !key_boundaries || !value_boundaries || !key_codes || !value_codes)
    return fail(TQ_ERR_BAD_ARG, "null pointer argument");
  if ((flags & (TQ_ROTATE_KEYS | TQ_ROTATE_VALUES)) && (!signs_left || !signs_right))
    return fail(TQ_ERR_BAD_ARG, "rotation flags need signs_left and signs_right");
  if (dtype != TQ_F32 && dtype != TQ_F16) return fail(TQ_ERR_BAD_ARG, "dtype must be F32 or F16");
  AppendParams p{};
  p.keys = keys;
  p.values = values;
  p.dtype = dtype;
  p.rows = static_cast<int64_t>(num_layers) * kv_heads * seq_new;
  p.streams = 2;
  p.seq_new = seq_new;
  p.rotate_keys = (flags & TQ_ROTATE_KEYS) != 0;
  p.rotate_values = (flags & TQ_ROTATE_VALUES) != 0;
  p.signs_left = signs_left;
  p.signs_right = signs_right;
  p.key_bnd = key_boundaries;
  p.value_bnd = value_boundaries;
  p.key_codes = key_codes;
  p.value_codes = value_codes;
  p.capacity = capacity;
  p.offset = offset;
  p.scaled = key_scales != nullptr;
  p.key_scales = key_scales;
  p.value_scales = value_scales;
  return with_d<AppendBody>(head_dim, p, bits, stream);
}

int qdq_impl(const void* keys, const void* values, int dtype, int64_t rows, int head_dim, int bits,
             const float* signs_left, const float* signs_right, int flags, const float* key_boundaries,
             const float* value_boundaries, const float* key_centroids, const float* value_centroids,
             float* key_out, float* value_out, bool scaled, hipStream_t stream) {
  int rc = check_geometry(head_dim, bits);
  if (rc) return rc;
  if (rows < 0) return fail(TQ_ERR_BAD_ARG, "rows must be non-negative");
  if (rows == 0) return TQ_OK;
  if (!keys || !key_boundaries || !key_centroids || !key_out) return fail(TQ_ERR_BAD_ARG, "null key argument");
  const bool two = values != nullptr;
  if (two && (!value_boundaries || !value_centroids || !value_out))
    return fail(TQ_ERR_BAD_ARG, "null value argument");
  if ((flags & (TQ_ROTATE_KEYS | TQ_ROTATE_VALUES)) && (!signs_left || !signs_right))
    return fail(TQ_ERR_BAD_ARG, "rotation flags need signs_left and signs_right");
  if (dtype != TQ_F32 && dtype != TQ_F16) return fail(TQ_ERR_BAD_ARG, "dtype must be F32 or F16");
  AppendParams p{};
  p.keys = keys;
  p.values = two ? values : keys;
  p.dtype = dtype;
  p.rows = rows;
  p.streams = two ? 2 : 1;
  p.seq_new = rows;
  p.rotate_keys = (flags & TQ_ROTATE_KEYS) != 0;
  p.rotate_values = (flags & TQ_ROTATE_VALUES) != 0;
  p.signs_left = signs_left;
  p.signs_right = signs_right;
  p.key_bnd = key_boundaries;
  p.value_bnd = two ? value_boundaries : key_boundaries;
  p.key_cent = key_centroids;
  p.value_cent = two ? value_centroids : key_centroids;
  p.key_out = key_out;
  p.value_out = two ? value_out : key_out;
  p.dequant = true;
  p.scaled = scaled;
  return with_d<AppendBody>(head_dim, p, bits, stream);
}

int unpack_impl(const uint32_t* codes, int64_t groups, int64_t capacity, int64_t seq_len, int head_dim, int bits,
                const float* centroids, const float* scales, float* out, hipStream_t stream) {
  int rc = check_geometry(head_dim, bits);
  if (rc) return rc;
  if (groups < 0 || seq_len < 0 || capacity < seq_len) return fail(TQ_ERR_BAD_ARG, "bad unpack extents");
  if (groups == 0 || seq_len == 0) return TQ_OK;
  if (!codes || !centroids || !out) return fail(TQ_ERR_BAD_ARG, "null pointer argument");
  return with_d<UnpackBody>(head_dim, codes, groups, capacity, seq_len, bits, centroids, scales, out, stream);
}

}  // namespace

// ============================================================== C ABI

extern "C" {

int tq_abi_version(void) { return TQ_ABI_VERSION; }

const char* tq_last_error(void) { return g_last_error.c_str(); }

int tq_fwht(const void* x, int x_dtype, float* y, int64_t rows, int head_dim, const float* signs_left,
            const float* signs_right, int inverse, hipStream_t stream) {
  int rc = check_geometry(head_dim, 0);
  if (rc) return rc;
  if (rows < 0) return fail(TQ_ERR_BAD_ARG, "rows must be non-negative");
  if (rows == 0) return TQ_OK;
  if (!x || !y || !signs_left || !signs_right) return fail(TQ_ERR_BAD_ARG, "null pointer argument");
  if (x_dtype != TQ_F32 && x_dtype != TQ_F16) return fail(TQ_ERR_BAD_ARG, "x dtype must be F32 or F16");
  const float* first = inverse ? signs_left : signs_right;
  const float* second = inverse ? signs_right : signs_left;
  return with_d<FwhtBody>(head_dim, x, x_dtype, y, rows, first, second, stream);
}

int tq_quantize_pack(const float* values, int64_t rows, int head_dim, int bits, const float* boundaries,
                     uint32_t* packed, hipStream_t stream) {
  int rc = check_geometry(head_dim, bits);
  if (rc) return rc;
  if (rows < 0) return fail(TQ_ERR_BAD_ARG, "rows must be non-negative");
  if (rows == 0) return TQ_OK;
  if (!values || !boundaries || !packed) return fail(TQ_ERR_BAD_ARG, "null pointer argument");
  AppendParams p{};
  p.keys = values;
  p.values = values;
  p.dtype = TQ_F32;
  p.rows = rows;
  p.streams = 1;
  p.seq_new = rows;
  p.key_bnd = boundaries;
  p.value_bnd = boundaries;
  p.key_codes = packed;
  p.value_codes = packed;
  p.capacity = rows;
  p.offset = 0;
  return with_d<AppendBody>(head_dim, p, bits, stream);
}

int tq_append(const void* keys, const void* values, int dtype, int num_layers, int kv_heads, int64_t seq_new,
              int head_dim, int bits, const float* signs_left, const float* signs_right, int flags,
              const float* key_boundaries, const float* value_boundaries, uint32_t* key_codes,
              uint32_t* value_codes, int64_t capacity, int64_t offset, hipStream_t stream) {
  return append_impl(keys, values, dtype, num_layers, kv_heads, seq_new, head_dim, bits, signs_left, signs_right, flags,
                     key_boundaries, value_boundaries, key_codes, value_codes, capacity, offset, nullptr, nullptr,
                     stream);
}

int tq_append_scaled(const void* keys, const void* values, int dtype, int num_layers, int kv_heads, int64_t seq_new,
                     int head_dim, int bits, const float* signs_left, const float* signs_right, int flags,
                     const float* key_boundaries, const float* value_boundaries, uint32_t* key_codes,
                     uint32_t* value_codes, float* key_scales, float* value_scales, int64_t capacity,
                     int64_t offset, hipStream_t stream) {
  if (key_scales == nullptr || value_scales == nullptr)
    return fail(TQ_ERR_BAD_ARG, "key_scales and value_scales must be non-null");
  return append_impl(keys, values, dtype, num_layers, kv_heads, seq_new, head_dim, bits, signs_left, signs_right, flags,
                     key_boundaries, value_boundaries, key_codes, value_codes, capacity, offset, key_scales,
                     value_scales, stream);
}

int tq_quantize_dequantize(const void* keys, const void* values, int dtype, int64_t rows, int head_dim, int bits,
                           const float* signs_left, const float* signs_right, int flags,
                           const float* key_boundaries, const float* value_boundaries,
                           const float* key_centroids, const float* value_centroids, float* key_out,
                           float* value_out, hipStream_t stream) {
  return qdq_impl(keys, values, dtype, rows, head_dim, bits, signs_left, signs_right, flags, key_boundaries,
                  value_boundaries, key_centroids, value_centroids, key_out, value_out, false, stream);
}

int tq_quantize_dequantize_scaled(const void* keys, const void* values, int dtype, int64_t rows, int head_dim,
                                  int bits, const float* signs_left, const float* signs_right, int flags,
                                  const float* key_boundaries, const float* value_boundaries,
                                  const float* key_centroids, const float* value_centroids, float* key_out,
                                  float* value_out, hipStream_t stream) {
  return qdq_impl(keys, values, dtype, rows, head_dim, bits, signs_left, signs_right, flags, key_boundaries,
                  value_boundaries, key_centroids, value_centroids, key_out, value_out, true, stream);
}

int tq_unpack_dequantize(const uint32_t* codes, int64_t groups, int64_t capacity, int64_t seq_len, int head_dim,
                         int bits, const float* centroids, float* out, hipStream_t stream) {
  return unpack_impl(codes, groups, capacity, seq_len, head_dim, bits, centroids, nullptr, out, stream);
}

int tq_unpack_dequantize_scaled(const uint32_t* codes, const float* scales, int64_t groups, int64_t capacity,
                                int64_t seq_len, int head_dim, int bits, const float* centroids, float* out,
                                hipStream_t stream) {
  if (scales == nullptr) return fail(TQ_ERR_BAD_ARG, "scales must be non-null");
  return unpack_impl(codes, groups, capacity, seq_len, head_dim, bits, centroids, scales, out, stream);
}

int tq_decode_default_splits(int num_layers, int kv_heads, int query_heads, int head_dim, int bits, int flags,
                             int64_t seq_len, int num_cus) {
  if (num_layers <= 0 || kv_heads <= 0 || query_heads <= 0 || query_heads % kv_heads != 0)
    return fail(TQ_ERR_BAD_ARG, "bad head configuration");
  if ((flags & TQ_F32_PRODUCTS) != 0 && (flags & TQ_MATRIX_PRODUCTS) != 0)
    return fail(TQ_ERR_BAD_ARG, "TQ_F32_PRODUCTS and TQ_MATRIX_PRODUCTS exclude each other");
  const int group = query_heads / kv_heads;
  if (num_cus <= 0) num_cus = device_cu_count();
  const int64_t kv_units = static_cast<int64_t>(num_layers) * kv_heads;
  return choose_kernel(kv_units, seq_len, 0, bits, head_dim, group, flags, num_cus).n_splits;
}

const char* tq_decode_split_kernel(int num_layers, int kv_heads, int query_heads, int head_dim, int bits, int flags,
                                   int query_dtype, int64_t seq_len, int n_splits, int num_cus) {
  if (num_layers <= 0 || kv_heads <= 0 || query_heads <= 0 || query_heads % kv_heads != 0 ||
      !valid_head_dim(head_dim) || seq_len < 0) {
    fail(TQ_ERR_BAD_ARG, "bad head configuration");
    return nullptr;
  }
  const bool packed = bits == 2 || bits == 3 || bits == 4;
  if (!packed) {
    fail(TQ_ERR_UNSUPPORTED, "split kernel names cover packed rows (bits 2, 3, 4)");
    return nullptr;
  }
  if ((flags & TQ_F32_PRODUCTS) != 0 && (flags & TQ_MATRIX_PRODUCTS) != 0) {
    fail(TQ_ERR_BAD_ARG, "TQ_F32_PRODUCTS and TQ_MATRIX_PRODUCTS exclude each other");
    return nullptr;
  }
  const int group = query_heads / kv_heads;
  if (num_cus <= 0) num_cus = device_cu_count();
  const int64_t kv_units = static_cast<int64_t>(num_layers) * kv_heads;
  static thread_local std::string name;
  const KernelChoice kc = choose_kernel(kv_units, seq_len, n_splits, bits, head_dim, group, flags, num_cus);
  if (kc.kernel == SplitKernel::Mx)
    name = "decode_mx_kernel<" + std::to_string(head_dim) + "," + (query_dtype == TQ_F16 ? "true" : "false") +
           (kc.hg == 8 ? "," + std::to_string(bits) + ",8>" : bits == 4 ? ">" : "," + std::to_string(bits) + ">");
  else if (fp32_tokens_per_iter(bits, head_dim, kc.hg, seq_len, kc.n_splits) == kWideTokensPerIter)
    name = "decode_kernel<PackedB4,256,4," + std::to_string(kWideTokensPerIter) + ">";
  else
    name = "decode_kernel<PackedB" + std::to_string(bits) + "," + std::to_string(head_dim) + "," +
           std::to_string(kc.hg) + ">";
  return name.c_str();
}

size_t tq_decode_workspace_bytes(int num_layers, int kv_heads, int query_heads, int head_dim, int n_splits,
                                 int num_cus) {
  if (num_layers <= 0 || kv_heads <= 0 || query_heads <= 0 || query_heads % kv_heads != 0) return 0;
  if (!valid_head_dim(head_dim)) return 0;
  const int group = query_heads / kv_heads;
  // the fewest units a group is cut into, so the most splits
  const int units = num_layers * kv_heads * head_groups(group, group >= 3 ? 4 : group);
  int ns = n_splits;
  // the larger of the two split kernels' defaults (two workgroups per CU, or
  // kMaxLoad where they are not all resident at once)
  if (ns <= 0) {
    ns = default_splits(units, static_cast<int64_t>(kMaxSplits) * kMinTokensPerSplit, num_cus, 2);
    ns = std::max(ns, kMaxLoad * (num_cus > 0 ? num_cus : 256) / units);
  }
  ns = std::min(ns, kMaxSplits);
  return workspace_layout(static_cast<int64_t>(num_layers) * query_heads, static_cast<int64_t>(num_layers) * kv_heads,
                          head_dim, ns)
      .total;
}

int tq_decode(const void* query, int query_dtype, int num_layers, int query_heads, int kv_heads, int head_dim,
              int bits, const uint32_t* key_codes, const uint32_t* value_codes, int64_t capacity, int64_t seq_len,
              const float* key_centroids, const float* value_centroids, const float* signs_left,
              const float* signs_right, int flags, const float* current_keys, const float* current_values,
              int n_splits, void* workspace, size_t workspace_bytes, float* out, hipStream_t stream) {
  return tq_decode_timed(query, query_dtype, num_layers, query_heads, kv_heads, head_dim, bits, key_codes,
                         value_codes, capacity, seq_len, key_centroids, value_centroids, signs_left, signs_right,
                         flags, current_keys, current_values, n_splits, workspace, workspace_bytes, out, stream,
                         nullptr, nullptr);
}

int tq_decode_noalloc(const void* query, int query_dtype, int num_layers, int query_heads, int kv_heads,
                      int head_dim, int bits, const uint32_t* key_codes, const uint32_t* value_codes,
                      int64_t capacity, int64_t seq_len, const float* key_centroids, const float* value_centroids,
                      const float* signs_left, const float* signs_right, int flags, const float* current_keys,
                      const float* current_values, int n_splits, float* out, hipStream_t stream) {
  if (!valid_bits(bits)) return fail(TQ_ERR_UNSUPPORTED, "Unsupported bit width: " + std::to_string(bits));
  int rc = check_geometry(head_dim, bits);
  if (rc) return rc;
  // The split plan this call resolves to, and the scratch it needs, before
  // anything touches the device.
  Plan p;
  rc = make_plan(num_layers, kv_heads, query_heads, seq_len, n_splits, bits, head_dim, flags, &p);
  if (rc) return rc;
  const size_t need = workspace_layout(static_cast<int64_t>(num_layers) * query_heads,
                                       static_cast<int64_t>(num_layers) * kv_heads, head_dim, p.n_splits)
                          .total;
  if (need > kScratchBytes)
    return fail(TQ_ERR_BAD_ARG, "tq_decode_noalloc: this call needs " + std::to_string(need) +
                                    " bytes of scratch (" + std::to_string(p.n_splits) +
                                    " splits) but the static scratch holds " + std::to_string(kScratchBytes) +
                                    "; pass fewer splits or decode fewer layers per call");
  void* ws = nullptr;
  rc = device_scratch(stream, &ws);
  if (rc) return rc;
  return decode_common(bits, query, query_dtype, num_layers, query_heads, kv_heads, head_dim, key_codes,
                       value_codes, capacity, seq_len, key_centroids, value_centroids, signs_left, signs_right, flags,
                       current_keys, current_values, n_splits, ws, kScratchBytes, out, stream, nullptr, nullptr);
}

int tq_decode_scaled(const void* query, int query_dtype, int num_layers, int query_heads, int kv_heads, int head_dim,
                     int bits, const uint32_t* key_codes, const uint32_t* value_codes, const float* key_scales,
                     const float* value_scales, int64_t capacity, int64_t seq_len, const float* key_centroids,
                     const float* value_centroids, const float* signs_left, const float* signs_right, int flags,
                     const float* current_keys, const float* current_values, int n_splits, void* workspace,
                     size_t workspace_bytes, float* out, hipStream_t stream) {
  return tq_decode_scaled_timed(query, query_dtype, num_layers, query_heads, kv_heads, head_dim, bits, key_codes,
                                value_codes, key_scales, value_scales, capacity, seq_len, key_centroids,
                                value_centroids, signs_left, signs_right, flags, current_keys, current_values,
                                n_splits, workspace, workspace_bytes, out, stream, nullptr, nullptr);
}

int tq_decode_scaled_timed(const void* query, int query_dtype, int num_layers, int query_heads, int kv_heads,
                           int head_dim, int bits, const uint32_t* key_codes, const uint32_t* value_codes,
                           const float* key_scales, const float* value_scales, int64_t capacity, int64_t seq_len,
                           const float* key_centroids, const float* value_centroids, const float* signs_left,
                           const float* signs_right, int flags, const float* current_keys,
                           const float* current_values, int n_splits, void* workspace, size_t workspace_bytes,
                           float* out, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  if (!valid_bits(bits)) return fail(TQ_ERR_UNSUPPORTED, "Unsupported bit width: " + std::to_string(bits));
  if (seq_len > 0 && (key_scales == nullptr || value_scales == nullptr))
    return fail(TQ_ERR_BAD_ARG, "key_scales and value_scales must be non-null");
  // Per-vector scales multiply the softmax weights, which the f16-split
  // kernel cannot hold for a factor of unknown size: always float32 products.
  return decode_common(bits, query, query_dtype, num_layers, query_heads, kv_heads, head_dim, key_codes, value_codes,
                       capacity, seq_len, key_centroids, value_centroids, signs_left, signs_right,
                       flags | TQ_F32_PRODUCTS, current_keys, current_values, n_splits, workspace, workspace_bytes,
                       out, stream, start, stop, nullptr,
                       seq_len > 0 ? key_scales : nullptr, seq_len > 0 ? value_scales : nullptr);
}

int tq_decode_append(const void* query, int query_dtype, const void* new_keys, const void* new_values, int kv_dtype,
                     int num_layers, int query_heads, int kv_heads, int head_dim, int bits, uint32_t* key_codes,
                     uint32_t* value_codes, int64_t capacity, int64_t seq_len, const float* key_centroids,
                     const float* value_centroids, const float* key_boundaries, const float* value_boundaries,
                     const float* signs_left, const float* signs_right, int append_flags, int decode_flags,
                     int n_splits, void* workspace, size_t workspace_bytes, float* out, hipStream_t stream) {
  int rc = check_geometry(head_dim, bits);
  if (rc) return rc;
  const AppendSpec app{new_keys, new_values, kv_dtype, key_boundaries, value_boundaries, append_flags};
  return decode_common(bits, query, query_dtype, num_layers, query_heads, kv_heads, head_dim, key_codes, value_codes,
                       capacity, seq_len, key_centroids, value_centroids, signs_left, signs_right, decode_flags,
                       nullptr, nullptr, n_splits, workspace, workspace_bytes, out, stream, nullptr, nullptr, &app);
}

int tq_decode_timed(const void* query, int query_dtype, int num_layers, int query_heads, int kv_heads,
                    int head_dim, int bits, const uint32_t* key_codes, const uint32_t* value_codes,
                    int64_t capacity, int64_t seq_len, const float* key_centroids, const float* value_centroids,
                    const float* signs_left, const float* signs_right, int flags, const float* current_keys,
                    const float* current_values, int n_splits, void* workspace, size_t workspace_bytes, float* out,
                    hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  if (!valid_bits(bits)) return fail(TQ_ERR_UNSUPPORTED, "Unsupported bit width: " + std::to_string(bits));
  return decode_common(bits, query, query_dtype, num_layers, query_heads, kv_heads, head_dim, key_codes,
                       value_codes, capacity, seq_len, key_centroids, value_centroids, signs_left, signs_right, flags,
                       current_keys, current_values, n_splits, workspace, workspace_bytes, out, stream, start, stop);
}

int tq_decode_step_timed(const void* query, int query_dtype, int num_layers, int query_heads, int kv_heads,
                         int head_dim, int bits, const uint32_t* key_codes, const uint32_t* value_codes,
                         int64_t capacity, int64_t seq_len, const float* key_centroids, const float* value_centroids,
                         const float* signs_left, const float* signs_right, int flags, const float* current_keys,
                         const float* current_values, int n_splits, void* workspace, size_t workspace_bytes,
                         float* out, hipStream_t stream, hipEvent_t split_start, hipEvent_t split_stop,
                         hipEvent_t merge_start, hipEvent_t merge_stop) {
  if (!valid_bits(bits)) return fail(TQ_ERR_UNSUPPORTED, "Unsupported bit width: " + std::to_string(bits));
  if ((merge_start == nullptr) != (merge_stop == nullptr))
    return fail(TQ_ERR_BAD_ARG, "merge_start and merge_stop must both be given or both be null");
  ProfileEvents mev;
  mev.start = merge_start;
  mev.stop = merge_stop;
  return decode_common(bits, query, query_dtype, num_layers, query_heads, kv_heads, head_dim, key_codes,
                       value_codes, capacity, seq_len, key_centroids, value_centroids, signs_left, signs_right, flags,
                       current_keys, current_values, n_splits, workspace, workspace_bytes, out, stream, split_start,
                       split_stop, nullptr, nullptr, nullptr, merge_start != nullptr ? &mev : nullptr);
}

int tq_decode_dense(const void* query, int query_dtype, const void* keys, const void* values, int kv_dtype,
                    int num_layers, int query_heads, int kv_heads, int head_dim, int64_t capacity, int64_t seq_len,
                    const float* signs_left, const float* signs_right, int flags, int n_splits, void* workspace,
                    size_t workspace_bytes, float* out, hipStream_t stream) {
  return tq_decode_dense_timed(query, query_dtype, keys, values, kv_dtype, num_layers, query_heads, kv_heads,
                               head_dim, capacity, seq_len, signs_left, signs_right, flags, n_splits, workspace,
                               workspace_bytes, out, stream, nullptr, nullptr);
}

int tq_decode_dense_timed(const void* query, int query_dtype, const void* keys, const void* values, int kv_dtype,
                          int num_layers, int query_heads, int kv_heads, int head_dim, int64_t capacity,
                          int64_t seq_len, const float* signs_left, const float* signs_right, int flags,
                          int n_splits, void* workspace, size_t workspace_bytes, float* out, hipStream_t stream,
                          hipEvent_t start, hipEvent_t stop) {
  if (kv_dtype != TQ_F16 && kv_dtype != TQ_F32) return fail(TQ_ERR_BAD_ARG, "kv dtype must be F32 or F16");
  return decode_common(kv_dtype == TQ_F16 ? 16 : 32, query, query_dtype, num_layers, query_heads, kv_heads, head_dim,
                       keys, values, capacity, seq_len, nullptr, nullptr, signs_left, signs_right, flags, nullptr,
                       nullptr, n_splits, workspace, workspace_bytes, out, stream, start, stop);
}

int tq_score_packed(const float* query, const uint32_t* codes, int batch, int64_t seq_len, int head_dim, int bits,
                    const float* centroids, float* scores, hipStream_t stream) {
  int rc = check_geometry(head_dim, bits);
  if (rc) return rc;
  if (batch < 0 || seq_len < 0) return fail(TQ_ERR_BAD_ARG, "batch and seq_len must be non-negative");
  if (batch == 0 || seq_len == 0) return TQ_OK;
  if (!query || !codes || !centroids || !scores) return fail(TQ_ERR_BAD_ARG, "null pointer argument");
  return with_d<StageBody>(head_dim, 0, bits, query, reinterpret_cast<const uint8_t*>(codes), batch, seq_len,
                           centroids, scores, stream);
}

int tq_softmax_rows(const float* scores, int batch, int64_t seq_len, float scale, float* weights,
                    hipStream_t stream) {
  if (batch < 0 || seq_len < 0) return fail(TQ_ERR_BAD_ARG, "batch and seq_len must be non-negative");
  if (batch == 0 || seq_len == 0) return TQ_OK;
  if (!scores || !weights) return fail(TQ_ERR_BAD_ARG, "null pointer argument");
  hipLaunchKernelGGL(softmax_kernel, dim3(batch), dim3(kBlock), 0, stream, scores, seq_len, scale, weights);
  return launch_status("softmax_kernel");
}

int tq_accumulate_packed(const float* weights, const uint32_t* codes, int batch, int64_t seq_len, int head_dim,
                         int bits, const float* centroids, float* out, hipStream_t stream) {
  int rc = check_geometry(head_dim, bits);
  if (rc) return rc;
  if (batch < 0 || seq_len < 0) return fail(TQ_ERR_BAD_ARG, "batch and seq_len must be non-negative");
  if (batch == 0) return TQ_OK;
  if (!weights || !codes || !centroids || !out) return fail(TQ_ERR_BAD_ARG, "null pointer argument");
  return with_d<StageBody>(head_dim, 2, bits, weights, reinterpret_cast<const uint8_t*>(codes), batch, seq_len,
                           centroids, out, stream);
}

int tq_rotary(const void* query, const void* key, int x_dtype, int query_heads, int key_heads, int64_t tokens,
              int head_dim, int64_t q_head_stride, int64_t q_token_stride, int64_t k_head_stride,
              int64_t k_token_stride, const void* cos, const void* sin, int table_dtype, int64_t cos_stride,
              int64_t sin_stride, int rotary_dim, void* query_out, void* key_out, int out_dtype, hipStream_t stream) {
  if (query_heads < 0 || key_heads < 0 || tokens < 0 || head_dim <= 0)
    return fail(TQ_ERR_BAD_ARG, "heads and tokens must be non-negative, head_dim positive");
  if (rotary_dim < 0 || rotary_dim % 2 != 0 || rotary_dim > head_dim)
    return fail(TQ_ERR_BAD_ARG, "rotary_dim must be even and at most head_dim");
  for (int type : {x_dtype, table_dtype, out_dtype})
    if (type < TQ_F32 || type > TQ_BF16) return fail(TQ_ERR_BAD_ARG, "dtypes must be F32, F16 or BF16");
  const int64_t rows = (static_cast<int64_t>(query_heads) + key_heads) * tokens;
  if (rows == 0) return TQ_OK;
  if (!query || !key || !cos || !sin || !query_out || !key_out) return fail(TQ_ERR_BAD_ARG, "null pointer argument");
  RotaryArgs a{};
  a.x[0] = {query, x_dtype, query_heads, q_head_stride, q_token_stride};
  a.x[1] = {key, x_dtype, key_heads, k_head_stride, k_token_stride};
  a.out[0] = query_out;
  a.out[1] = key_out;
  a.out_type = out_dtype;
  a.cos = cos;
  a.sin = sin;
  a.table_type = table_dtype;
  a.cos_stride = cos_stride;
  a.sin_stride = sin_stride;
  a.tokens = tokens;
  a.head_dim = head_dim;
  a.rotary_dim = rotary_dim;
  for (a.row0 = 0; a.row0 < rows; a.row0 += kMaxLaunchBlocks * kWavesPerBlock) {
    hipLaunchKernelGGL(rotary_kernel, row_grid(rows - a.row0), dim3(kBlock), 0, stream, a);
    const int rc = launch_status("rotary_kernel");
    if (rc) return rc;
  }
  return TQ_OK;
}

int tq_unrotate_gate(const float* attn, int heads, int64_t tokens, int head_dim, int64_t head_stride,
                     int64_t token_stride, const void* gate, int gate_dtype, int64_t gate_head_stride,
                     int64_t gate_token_stride, const float* signs_left, const float* signs_right, void* out,
                     int out_dtype, hipStream_t stream) {
  const int rc = check_geometry(head_dim, 0);
  if (rc) return rc;
  if (heads < 0 || tokens < 0) return fail(TQ_ERR_BAD_ARG, "heads and tokens must be non-negative");
  for (int type : {gate_dtype, out_dtype})
    if (type < TQ_F32 || type > TQ_BF16) return fail(TQ_ERR_BAD_ARG, "dtypes must be F32, F16 or BF16");
  const int64_t rows = heads * tokens;
  if (rows == 0) return TQ_OK;
  if (!attn || !gate || !signs_left || !signs_right || !out) return fail(TQ_ERR_BAD_ARG, "null pointer argument");
  GateArgs a{};
  a.attn = {attn, kTypeF32, heads, head_stride, token_stride};
  a.gate = {gate, gate_dtype, heads, gate_head_stride, gate_token_stride};
  a.out = out;
  a.out_type = out_dtype;
  a.tokens = tokens;
  a.signs_left = signs_left;
  a.signs_right = signs_right;
  a.sqrt_d = sqrt_f32(head_dim);
  for (a.row0 = 0; a.row0 < rows; a.row0 += kMaxLaunchBlocks * kWavesPerBlock) {
    const dim3 grid = row_grid(rows - a.row0);
    if (head_dim == 64)
      hipLaunchKernelGGL(unrotate_gate_kernel<64>, grid, dim3(kBlock), 0, stream, a);
    else if (head_dim == 128)
      hipLaunchKernelGGL(unrotate_gate_kernel<128>, grid, dim3(kBlock), 0, stream, a);
    else
      hipLaunchKernelGGL(unrotate_gate_kernel<256>, grid, dim3(kBlock), 0, stream, a);
    const int rc_launch = launch_status("unrotate_gate_kernel");
    if (rc_launch) return rc_launch;
  }
  return TQ_OK;
}

int tq_stream_read(const void* data, size_t bytes, float* sink, int n_blocks, hipStream_t stream, hipEvent_t start,
                   hipEvent_t stop) {
  if (data == nullptr || sink == nullptr) return fail(TQ_ERR_BAD_ARG, "data and sink must be non-null");
  if (bytes % 16 != 0 || reinterpret_cast<uintptr_t>(data) % 16 != 0)
    return fail(TQ_ERR_BAD_ARG, "bytes and the data address must be multiples of 16");
  if (n_blocks <= 0) n_blocks = device_cu_count();
  const int64_t n16 = static_cast<int64_t>(bytes / 16);
  if (start != nullptr || stop != nullptr)
    hipExtLaunchKernelGGL(stream_read_kernel, dim3(n_blocks), dim3(kStreamThreads), 0, stream, start, stop, 0,
                          static_cast<const uint4*>(data), n16, sink);
  else
    hipLaunchKernelGGL(stream_read_kernel, dim3(n_blocks), dim3(kStreamThreads), 0, stream,
                       static_cast<const uint4*>(data), n16, sink);
  return launch_status("stream_read_kernel");
}

}  // extern "C"
