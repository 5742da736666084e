// The elementwise stages of a gated attention layer around the packed cache:
// rotary embedding of queries and keys, and the way from the attention output
// to the output projection's input (inverse rotation, gate, cast).
//
// Included by torque_hip.hip.  As torch operations they are 14 and 6 launches
// a layer and step, each of which costs a decode step more than its own work
// (one token x 20 heads is 10 KB): they take 95 us of host time where the two
// launches here take 12.  Every operation is rounded as the torch operation it
// stands for, in the same order, so the rotary output is bit-identical.
#pragma once

// Element types of the layer's tensors.
enum { kTypeF32 = 0, kTypeF16 = 1, kTypeBF16 = 2 };

__device__ __forceinline__ float load_as_f32(const void* p, int64_t i, int type) {
  if (type == kTypeF32) return static_cast<const float*>(p)[i];
  const uint16_t h = static_cast<const uint16_t*>(p)[i];
  return type == kTypeF16 ? __half2float(__ushort_as_half(h)) : __uint_as_float(static_cast<uint32_t>(h) << 16);
}
// Bits of x rounded to nearest even in bfloat16 (a NaN stays one).
__device__ __forceinline__ uint16_t bf16_bits(float x) {
  const uint32_t u = __float_as_uint(x);
  if (x != x) return static_cast<uint16_t>((u >> 16) | 0x40u);
  return static_cast<uint16_t>((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}
__device__ __forceinline__ float round_as(float x, int type) {
  if (type == kTypeF32) return x;
  if (type == kTypeF16) return __half2float(__float2half(x));
  return __uint_as_float(static_cast<uint32_t>(bf16_bits(x)) << 16);
}
__device__ __forceinline__ void store_as(void* p, int64_t i, float x, int type) {
  if (type == kTypeF32)
    static_cast<float*>(p)[i] = x;
  else if (type == kTypeF16)
    static_cast<__half*>(p)[i] = __float2half(x);
  else
    static_cast<uint16_t*>(p)[i] = bf16_bits(x);
}

// [heads, tokens, D] rows with unit stride along D.
struct RowView {
  const void* data;
  int type, heads;
  int64_t head_stride, token_stride;
};

struct RotaryArgs {
  RowView x[2];       // queries, keys
  void* out[2];       // contiguous [heads, tokens, D] of out_type
  int out_type;
  const void* cos;    // [tokens, rotary_dim], rows token_stride apart
  const void* sin;
  int table_type;
  int64_t cos_stride, sin_stride;
  int64_t tokens, row0;  // row0: first row of this launch
  int head_dim, rotary_dim;
};

// One wavefront per row of queries (then keys): x cos + rotate_half(x) sin on
// the first rotary_dim dimensions, the rest copied.  At prompt sizes it reads
// and writes each row once and is bound by memory.
__global__ __launch_bounds__(kBlock) void rotary_kernel(const RotaryArgs a) {
  int64_t row = a.row0 + static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + (threadIdx.x >> 6);
  const int64_t q_rows = static_cast<int64_t>(a.x[0].heads) * a.tokens;
  const int s = row >= q_rows;
  if (s) row -= q_rows;
  const RowView x = s ? a.x[1] : a.x[0];
  if (row >= static_cast<int64_t>(x.heads) * a.tokens) return;
  const int64_t h = row / a.tokens, t = row - h * a.tokens;
  const int64_t base = h * x.head_stride + t * x.token_stride;
  void* out = s ? a.out[1] : a.out[0];
  const int half = a.rotary_dim / 2;
  for (int d = lane_id(); d < a.head_dim; d += kWave) {
    const float v = load_as_f32(x.data, base + d, x.type);
    float y = v;
    if (d < a.rotary_dim) {
      const float w = d < half ? -load_as_f32(x.data, base + d + half, x.type) : load_as_f32(x.data, base + d - half, x.type);
      const float c = load_as_f32(a.cos, t * a.cos_stride + d, a.table_type);
      const float sn = load_as_f32(a.sin, t * a.sin_stride + d, a.table_type);
      y = round_as(__fadd_rn(round_as(__fmul_rn(v, c), a.out_type), round_as(__fmul_rn(w, sn), a.out_type)), a.out_type);
    }
    store_as(out, row * a.head_dim + d, y, a.out_type);
  }
}

struct GateArgs {
  RowView attn;       // float32 attention output, in the rotated basis
  RowView gate;
  void* out;          // contiguous [tokens, heads * D] of out_type
  int out_type;
  int64_t tokens, row0;  // row0: first row of this launch
  const float* signs_left;
  const float* signs_right;
  float sqrt_d;
};

// One wavefront per (head, token): inverse rotation, times sigmoid(gate),
// stored at the token's row of the projection's input.
template <int D>
__global__ __launch_bounds__(kBlock) void unrotate_gate_kernel(const GateArgs a) {
  constexpr int E = D / kWave;
  const int64_t row = a.row0 + static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + (threadIdx.x >> 6);
  if (row >= static_cast<int64_t>(a.attn.heads) * a.tokens) return;  // whole wavefront exits together
  const int64_t t = row / a.attn.heads, h = row - t * a.attn.heads;
  const int d0 = lane_id() * E;
  const int64_t src = h * a.attn.head_stride + t * a.attn.token_stride + d0;
  const int64_t g = h * a.gate.head_stride + t * a.gate.token_stride + d0;
  float v[E];
#pragma unroll
  for (int i = 0; i < E; ++i) v[i] = static_cast<const float*>(a.attn.data)[src + i];
  wave_rotate<D>(v, a.signs_left, a.signs_right, a.sqrt_d);
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const float s = __fdiv_rn(1.f, 1.f + expf(-load_as_f32(a.gate.data, g + i, a.gate.type)));
    store_as(a.out, row * D + d0 + i, __fmul_rn(v[i], s), a.out_type);
  }
}
