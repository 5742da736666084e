// Causal attention of a prompt chunk over the dense keys and values, float32
// accuracy on the float16 matrix cores.
//
// Included by torque_hip.hip (after attention_layer.hpp).
//
// Arithmetic.  Operands are split into float16 pairs, x = hi + lo with hi =
// f16(x) and lo = f16(x - hi) (|x - hi - lo| <= 2^-23 |x|), after exact
// power-of-two scales that put the largest magnitude of a query row, a 32-key
// tile of keys or of values, and the weights at 2^14: no overflow, and lo
// stays clear of subnormals down to 2^-28 of that magnitude.  A product is
// hi hi + hi lo + lo hi in float32 sums; the lo lo left out is below 2^-22 of
// a term, as is a float32 product's own rounding over the chain of sums.
// 16x16x32 float16 products run at 16 times the rate of float32 ones, so three
// of them still do 5 times the work.
//
// Layout.  A wavefront takes 16 rows of one query head and computes S^T = K
// Q^T and O^T = V^T P^T, so that a query is one column, lane mod 16, in every
// result: its maximum and sum need two lane swaps, its rescaling none.  The
// 16x16 scores leave keys 4g .. 4g + 3 of two 16-key halves on lane group g =
// lane / 16, which is an operand's 8 k-slots in another key order, and V is
// packed in that order: weights go from one product to the next without
// moving.  pack_kv_kernel writes the splits in operand order, 1 KB to a
// wavefront read, so a tile moves to LDS by direct loads while the one before
// it is used, and is shared by the 4 wavefronts of a workgroup (rows of the
// query heads of one KV head).
// Measured, both kernels and their launches, against torch's attention with a
// mask (float32): 1024 tokens, 16 / 4 heads of 256, 113 us against 567; 1500,
// 8 / 8 heads of 128, 85 against 500; 4096, 32 / 8 heads of 128, 541 against
// 4799 (its error against float64 2e-7 to 8e-7 where torch's is 2e-7 to
// 1.4e-6).  At head_dim 256 a tile takes ~2.9 us of a workgroup against 0.75
// of products: one wavefront per SIMD waits for its LDS reads.
#pragma once

namespace prompt {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTileKeys = 32;
constexpr int kRows = 16;  // query rows of a wavefront
// 16-byte operands of one tile, per lane: keys [half][D / 32][hi, lo], then
// values [D / 16][hi, lo].
template <int D>
constexpr int tile_frags() {
  return 2 * (D / 32) * 2 + (D / 16) * 2;
}
constexpr size_t tile_bytes(int head_dim) { return static_cast<size_t>(kTileKeys) * head_dim * 2 * 2 * 2; }

struct Split {
  _Float16 hi, lo;
};
__device__ __forceinline__ Split split_f16(float x) {
  const _Float16 hi = static_cast<_Float16>(x);
  return {hi, static_cast<_Float16>(x - static_cast<float>(hi))};
}
// Power of two that puts a magnitude into [2^14, 2^15), at most 2^100, which
// is what all-zero operands take (a tile of them then sets no other's scale).
__device__ __forceinline__ int shift_of(float maxabs) { return maxabs == 0.f ? 100 : min(100, mx::scale_shift(maxabs)); }

}  // namespace prompt

struct PromptArgs {
  RowView q, k, v;
  int64_t tokens, keys;  // query rows, keys
  int64_t offset;        // row i attends keys 0 .. offset + i
  float scale;
  int group;             // query heads per KV head
  int tiles;             // key tiles
  uint4* packed;         // [KV heads, tiles, tile_frags * 64]
  int2* shifts;          // [KV heads, tiles] (key, value) scale exponents
  float* out;            // contiguous [query heads, tokens, D]
};

// One workgroup per (tile, KV head).  Keys past the end are zeros.
template <int D>
__global__ __launch_bounds__(kBlock) void pack_kv_kernel(const PromptArgs a) {
  using namespace prompt;
  __shared__ float s_k[kTileKeys][D + 4], s_v[kTileKeys][D + 4];
  __shared__ float s_max[2][kWavesPerBlock];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & (kWave - 1);
  const int64_t tile = blockIdx.x, h = blockIdx.y;
  float mk = 0.f, mv = 0.f;
  for (int i = tid; i < kTileKeys * D; i += kBlock) {
    const int r = i / D, d = i % D;
    const int64_t key = tile * kTileKeys + r;
    float x = 0.f, y = 0.f;
    if (key < a.keys) {
      x = load_as_f32(a.k.data, h * a.k.head_stride + key * a.k.token_stride + d, a.k.type);
      y = load_as_f32(a.v.data, h * a.v.head_stride + key * a.v.token_stride + d, a.v.type);
    }
    s_k[r][d] = x;
    s_v[r][d] = y;
    mk = fmaxf(mk, fabsf(x));
    mv = fmaxf(mv, fabsf(y));
  }
  mk = group_reduce<kWave, OpMax>(mk);
  mv = group_reduce<kWave, OpMax>(mv);
  if (lane == 0) {
    s_max[0][wave] = mk;
    s_max[1][wave] = mv;
  }
  __syncthreads();
  auto over = [&](int s) { return fmaxf(fmaxf(s_max[s][0], s_max[s][1]), fmaxf(s_max[s][2], s_max[s][3])); };
  const int sk = shift_of(over(0)), sv = shift_of(over(1));
  const int64_t at = h * a.tiles + tile;
  if (tid == 0) a.shifts[at] = make_int2(sk, sv);
  uint4* dst = a.packed + at * (tile_frags<D>() * kWave);
  const int n = lane & 15, g = lane >> 4;
  constexpr int kKey = 2 * (D / 32);  // key operand pairs, then value operand pairs
  for (int f = wave; f < kKey + D / 16; f += kWavesPerBlock) {
    f16x8 hi, lo;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float x;
      if (f < kKey)
        x = ldexpf(s_k[16 * (f / (D / 32)) + n][32 * (f % (D / 32)) + 8 * g + j], sk);
      else
        x = ldexpf(s_v[(j < 4 ? 0 : 12) + 4 * g + j][16 * (f - kKey) + n], sv);
      const Split s = split_f16(x);
      hi[j] = s.hi;
      lo[j] = s.lo;
    }
    dst[(2 * f) * kWave + lane] = __builtin_bit_cast(uint4, hi);
    dst[(2 * f + 1) * kWave + lane] = __builtin_bit_cast(uint4, lo);
  }
}

// Grid (row groups, KV heads), the longest rows first.  Wavefront w of row
// group b takes item 4 b' + w of the KV head's (row tile, query head) pairs,
// query head fastest, b' counted from the end.
template <int D>
__global__ __launch_bounds__(kBlock, D == 256 ? 1 : 2) void prompt_attention_kernel(const PromptArgs a) {
  using namespace prompt;
  constexpr int KS = D / 32, NV = D / 16;
  constexpr int FR = tile_frags<D>();
  constexpr float kWeightScale = 16384.f;  // 2^14
  __shared__ uint4 s_tile[2 * FR * kWave];  // two tiles: one in use, one on its way
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int64_t h = blockIdx.y;
  const int64_t row_tiles = (a.tokens + kRows - 1) / kRows;
  const int64_t items = row_tiles * a.group;
  const int64_t base = (static_cast<int64_t>(gridDim.x) - 1 - blockIdx.x) * kWavesPerBlock;
  const int64_t item = base + wave;
  const bool active = item < items;  // whole wavefront
  const int64_t rt = min(item, items - 1) / a.group;
  const int64_t qh = h * a.group + (min(item, items - 1) - rt * a.group);
  const int64_t row = min(rt * kRows + n, a.tokens - 1);  // rows past the end repeat the last and are not stored
  const int64_t limit = min(a.offset + row, a.keys - 1);  // last key of this lane's row
  auto last_tile = [&](int64_t r) {
    return static_cast<int>(min(a.offset + min(r * kRows + kRows - 1, a.tokens - 1), a.keys - 1) / kTileKeys);
  };
  const int my_last = last_tile(rt);
  const int last = last_tile(min(base + kWavesPerBlock - 1, items - 1) / a.group);  // of the workgroup: its last item's

  // ---- queries: log2(e) * scale folded in, then the split, column n, dims 32 ks + 8 g ..
  f16x8 qh8[KS], ql8[KS];
  float score_scale;  // raw score -> log2 units, without the keys' exponent
  {
    float x[KS][8];
    float mx = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        x[ks][j] = load_as_f32(a.q.data, qh * a.q.head_stride + row * a.q.token_stride + 32 * ks + 8 * g + j, a.q.type) *
                   (a.scale * kLog2e);
        mx = fmaxf(mx, fabsf(x[ks][j]));
      }
    mx = xor_reduce<16, OpMax>(mx);
    mx = xor_reduce<32, OpMax>(mx);
    const int sq = shift_of(mx);
    score_scale = ldexpf(1.f, -sq);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const Split s = split_f16(ldexpf(x[ks][j], sq));
        qh8[ks][j] = s.hi;
        ql8[ks][j] = s.lo;
      }
  }

  const uint4* packed = a.packed + h * a.tiles * static_cast<int64_t>(FR * kWave);
  auto load_tile = [&](int t, int buf) {
    const uint4* src = packed + static_cast<int64_t>(t) * (FR * kWave);
    for (int f = wave; f < FR; f += kWavesPerBlock)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(src + f * kWave + lane),
          (__attribute__((address_space(3))) void*)(s_tile + (buf * FR + f) * kWave), 16, 0, 0);
  };

  f32x4 acc[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  int ref = 127;  // value exponent of the accumulators

  load_tile(0, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (int t = 0; t <= last; ++t) {
    const int buf = t & 1;
    if (t < last) load_tile(t + 1, buf ^ 1);
    if (active && t <= my_last) {
      const f16x8* frag = reinterpret_cast<const f16x8*>(s_tile + buf * FR * kWave) + lane;
      const int2 shift = a.shifts[h * a.tiles + t];
      f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const f16x8 k0h = frag[(2 * ks) * kWave], k0l = frag[(2 * ks + 1) * kWave];
        const f16x8 k1h = frag[(2 * (KS + ks)) * kWave], k1l = frag[(2 * (KS + ks) + 1) * kWave];
        s0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(k0h, qh8[ks], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(k1h, qh8[ks], s1, 0, 0, 0);
        s0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(k0l, qh8[ks], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(k1l, qh8[ks], s1, 0, 0, 0);
        s0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(k0h, ql8[ks], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(k1h, ql8[ks], s1, 0, 0, 0);
      }
      // ---- softmax, log2 units; keys past a row's limit get weight zero
      const float f = score_scale * ldexpf(1.f, -shift.x);
      const int64_t key0 = static_cast<int64_t>(t) * kTileKeys + 4 * g;
      float s[8];
      float mx = -INFINITY;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float raw = j < 4 ? s0[j] : s1[j - 4];
        s[j] = key0 + (j < 4 ? j : 12 + j) <= limit ? raw * f : -INFINITY;
        mx = fmaxf(mx, s[j]);
      }
      mx = xor_reduce<16, OpMax>(mx);
      mx = xor_reduce<32, OpMax>(mx);
      const float mn = fmaxf(m, mx);
      const int new_ref = min(ref, shift.y);
      const float alpha = fast_exp2(m - mn);  // 0 at the first tile: nothing accumulated
      const float rescale = ref == new_ref ? alpha : alpha * ldexpf(1.f, new_ref - ref);
      l *= alpha;
      m = mn;
      ref = new_ref;
      if (__builtin_amdgcn_ballot_w64(rescale != 1.f) != 0) {
#pragma unroll
        for (int j = 0; j < NV; ++j) acc[j] *= rescale;
      }
      const float weight = kWeightScale * ldexpf(1.f, ref - shift.y);
      f16x8 ph, pl;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float p = fast_exp2(s[j] - m);
        l += p;
        const Split w = split_f16(p * weight);
        ph[j] = w.hi;
        pl[j] = w.lo;
      }
      const f16x8* vfrag = frag + 4 * KS * kWave;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const f16x8 vh = vfrag[(2 * j) * kWave], vl = vfrag[(2 * j + 1) * kWave];
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, ph, acc[j], 0, 0, 0);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vl, ph, acc[j], 0, 0, 0);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, pl, acc[j], 0, 0, 0);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the next tile is in LDS
    __syncthreads();
  }

  l = xor_reduce<16, OpSum>(l);
  l = xor_reduce<32, OpSum>(l);
  if (active && rt * kRows + n < a.tokens) {
    const float inv = ldexpf(1.f / l, -14);
    float* dst = a.out + (qh * a.tokens + row) * D + 4 * g;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      float4 o;
      o.x = ldexpf(acc[j][0] * inv, -ref);
      o.y = ldexpf(acc[j][1] * inv, -ref);
      o.z = ldexpf(acc[j][2] * inv, -ref);
      o.w = ldexpf(acc[j][3] * inv, -ref);
      *reinterpret_cast<float4*>(dst + 16 * j) = o;
    }
  }
}
