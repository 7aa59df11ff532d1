// Decode attention of the decoder and its SiLU gate, each as one launch
// (gfx950, 16-bit data).
//
// Attention of one new token per sequence over a static KV cache: rotary on q
// and k, the new key and value into the cache, scores, masked softmax and the
// weighted sum of the values.  As torch operations these were eleven launches
// a layer of 3 to 10 us each, most of them launch latency at decode sizes;
// the arithmetic here is fp32 throughout, rounded where the cache or the
// output stores it (the separate launches also rounded q, the scores and the
// probabilities to 16 bits).
//
// Workgroup = (sequence, key head) with its REP query heads, eight waves.
// The cache holds keys transposed, [kv_heads, D, L]: a lane takes four
// neighbouring positions and a wave an eighth of D, so every load is
// contiguous over the wave, and the waves' sums meet in LDS.  Values are
// [kv_heads, L, D]: D / 8 lanes take a row, the workgroup's groups of lanes
// the positions in turn.  Bound by the dependent round trips of these phases
// (launch, rows, keys and values, scores, softmax, sums) and, for long caches,
// by the cache's bytes.  32 sequences, 16 heads of 4 key heads, 208 positions:
// 13.2 us for one launch against 44.8 us for torch's eleven (34 us with four
// waves a workgroup and the keys and values requested phase by phase); 64
// sequences, 32 heads of 8 key heads: 57 against 96 us at 520 positions, 166
// against 204 at 2048 (3.2 TB/s of cache).  A decoder's step of four layers
// (hidden 2048, 32 sequences): 684 -> 499 us with the SiLU gate below (1088 x
// 14336: 17.7 against 38.9 us).
#include "kernels.h"
#include "loads.h"

namespace mlora {

namespace {

constexpr int kAttnWaves = kAttnThreads / kWave;
constexpr int kAttnChunk = 256;  // positions a pass

template <int D, int REP>
struct AttnLds {
  float q[REP][D];
  float k[D];
  float v[D];
  float new_score[REP];
  float score[REP][kAttnMaxLen];
  // A pass's scores by wave (a part of D each), then the output by wave (a
  // part of the positions each).
  union {
    float part[kAttnWaves][REP][kAttnChunk];
    float out[kAttnWaves][REP][D];
  };
};

template <class T, int D, int REP>
__global__ __launch_bounds__(kAttnThreads) void decode_attn_kernel(AttnArgs a) {
  using raw = typename T::raw_t;
  constexpr int DW = D / kAttnWaves;           // key rows a wave
  constexpr int LPR = D / 8;                   // lanes a value row
  constexpr int G = kAttnThreads / LPR;        // value rows read at once
  constexpr int VR = (kAttnChunk + G - 1) / G; // value rows a thread and pass
  constexpr int ROT = ((REP + 2) * D + kAttnThreads - 1) / kAttnThreads;
  __shared__ AttnLds<D, REP> s;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int b = blockIdx.x / a.kv_heads;
  const int kh = blockIdx.x - b * a.kv_heads;
  const raw* q = static_cast<const raw*>(a.q) + b * a.q_stride + kh * REP * D;
  const raw* k = static_cast<const raw*>(a.k) + b * a.k_stride + kh * D;
  const raw* v = static_cast<const raw*>(a.v) + b * a.v_stride + kh * D;
  const raw* cs = static_cast<const raw*>(a.cos) + b * a.rot_stride;
  const raw* sn = static_cast<const raw*>(a.sin) + b * a.rot_stride;
  const int64_t head = static_cast<int64_t>(b) * a.kv_heads + kh;
  raw* keys = static_cast<raw*>(a.keys) + head * D * a.len;
  raw* values = static_cast<raw*>(a.values) + head * D * a.len;
  const bool vec4 = (a.len & 3) == 0 && (reinterpret_cast<uintptr_t>(a.keys) & 7) == 0;

  // Everything the first pass needs is requested at once: the rows to
  // rotate, then the keys and values of positions [0, kAttnChunk).
  const int64_t p64 = *a.pos;
  raw xe[ROT], xo[ROT], ce[ROT], se[ROT];
#pragma unroll
  for (int z = 0; z < ROT; ++z) {
    const int i = min(tid + z * kAttnThreads, (REP + 2) * D - 1);
    const int r = i / D;
    const int e = i - r * D;
    const raw* x = r < REP ? q + r * D : r == REP ? k : v;
    xe[z] = x[e];
    xo[z] = x[e ^ (D / 2)];
    ce[z] = cs[e];
    se[z] = sn[e];
  }
  uint2 kreg[DW];
  u32x4 vreg[VR];
  auto load_keys = [&](int l0) {
    const int l = l0 + lane * 4;
#pragma unroll
    for (int e = 0; e < DW; ++e) {
      const raw* row = keys + static_cast<int64_t>(wave * DW + e) * a.len;
      if (vec4) {
        kreg[e] = *reinterpret_cast<const uint2*>(row + min(l, a.len - 4));
      } else {
        uint32_t h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = row[min(l + i, a.len - 1)];
        kreg[e].x = h[0] | (h[1] << 16);
        kreg[e].y = h[2] | (h[3] << 16);
      }
    }
  };
  const int grp = tid / LPR;
  const int c = tid - grp * LPR;
  auto load_values = [&](int l0) {
#pragma unroll
    for (int i = 0; i < VR; ++i)
      vreg[i] = ld_chunk(values + static_cast<int64_t>(min(l0 + grp + G * i, a.len - 1)) * D + c * 8);
  };
  load_keys(0);
  load_values(0);

  // rotate(x) = x * cos + (x rolled by D / 2) * sin (sin signed).
  const int pos = p64 >= 0 && p64 < a.len ? static_cast<int>(p64) : -1;
#pragma unroll
  for (int z = 0; z < ROT; ++z) {
    const int i = tid + z * kAttnThreads;
    if (i >= (REP + 2) * D) break;
    const int r = i / D;
    const int e = i - r * D;
    if (r == REP + 1) {
      s.v[e] = T::to_f32(xe[z]);
      if (pos >= 0) values[static_cast<int64_t>(pos) * D + e] = xe[z];
      continue;
    }
    const float f = T::to_f32(xe[z]) * T::to_f32(ce[z]) + T::to_f32(xo[z]) * T::to_f32(se[z]);
    if (r < REP) {
      s.q[r][e] = f;
    } else {
      const raw w = T::from_f32(f);
      s.k[e] = T::to_f32(w);
      if (pos >= 0) keys[static_cast<int64_t>(e) * a.len + pos] = w;
    }
  }
  lds_barrier();
  // The new token's own scores (and below its value) come from here, not from
  // the cache lines being written.
  for (int r = wave; r < REP; r += kAttnWaves) {
    float f = 0.f;
#pragma unroll
    for (int e = 0; e < D; e += kWave) f += s.q[r][e + lane] * s.k[e + lane];
    for (int off = 1; off < kWave; off <<= 1) f += __shfl_xor(f, off, kWave);
    if (lane == 0) s.new_score[r] = f;
  }

  for (int l0 = 0; l0 < a.len; l0 += kAttnChunk) {
    if (l0 > 0) load_keys(l0);
    float acc[REP][4];
#pragma unroll
    for (int r = 0; r < REP; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[r][i] = 0.f;
#pragma unroll
    for (int e = 0; e < DW; ++e) {
      const float kv[4] = {T::to_f32(static_cast<raw>(kreg[e].x & 0xffffu)), T::to_f32(static_cast<raw>(kreg[e].x >> 16)),
                           T::to_f32(static_cast<raw>(kreg[e].y & 0xffffu)), T::to_f32(static_cast<raw>(kreg[e].y >> 16))};
#pragma unroll
      for (int r = 0; r < REP; ++r) {
        const float qv = s.q[r][wave * DW + e];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[r][i] += qv * kv[i];
      }
    }
#pragma unroll
    for (int r = 0; r < REP; ++r)
      *reinterpret_cast<f32x4*>(&s.part[wave][r][lane * 4]) = f32x4{acc[r][0], acc[r][1], acc[r][2], acc[r][3]};
    lds_barrier();
    for (int i = tid; i < REP * kAttnChunk; i += kAttnThreads) {
      const int r = i / kAttnChunk;
      const int lc = i - r * kAttnChunk;
      const int l = l0 + lc;
      if (l >= a.len) continue;
      float f = 0.f;
#pragma unroll
      for (int w = 0; w < kAttnWaves; ++w) f += s.part[w][r][lc];
      if (l == pos) f = s.new_score[r];
      s.score[r][l] = a.hide[b * a.hide_stride + l] != 0 ? -INFINITY : f * a.scale;
    }
    lds_barrier();
  }

  for (int r = wave; r < REP; r += kAttnWaves) {
    float m = -INFINITY;
    for (int l = lane; l < a.len; l += kWave) m = fmaxf(m, s.score[r][l]);
    for (int off = 1; off < kWave; off <<= 1) m = fmaxf(m, __shfl_xor(m, off, kWave));
    float sum = 0.f;
    for (int l = lane; l < a.len; l += kWave) {
      const float e = expf(s.score[r][l] - m);
      s.score[r][l] = e;
      sum += e;
    }
    for (int off = 1; off < kWave; off <<= 1) sum += __shfl_xor(sum, off, kWave);
    const float inv = 1.f / sum;
    for (int l = lane; l < a.len; l += kWave) s.score[r][l] *= inv;
  }
  lds_barrier();

  float acc[REP][8];
#pragma unroll
  for (int r = 0; r < REP; ++r)
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[r][i] = 0.f;
  for (int l0 = 0; l0 < a.len; l0 += kAttnChunk) {
    if (l0 > 0) load_values(l0);
#pragma unroll
    for (int z = 0; z < VR; ++z) {
      const int l = l0 + grp + G * z;
      if (grp + G * z >= kAttnChunk || l >= a.len) continue;
      float f[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] = l == pos ? s.v[c * 8 + i] : chunk_elem<T>(vreg[z], i);
#pragma unroll
      for (int r = 0; r < REP; ++r) {
        const float p = s.score[r][l];
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[r][i] += p * f[i];
      }
    }
  }
  // The lane groups of a wave, then the waves.
#pragma unroll
  for (int r = 0; r < REP; ++r)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      for (int off = LPR; off < kWave; off <<= 1) acc[r][i] += __shfl_xor(acc[r][i], off, kWave);
      if (lane < LPR) s.out[wave][r][c * 8 + i] = acc[r][i];
    }
  lds_barrier();
  raw* out = static_cast<raw*>(a.out) + b * a.out_stride + kh * REP * D;
  for (int i = tid; i < REP * D; i += kAttnThreads) {
    const int r = i / D;
    const int e = i - r * D;
    float f = 0.f;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) f += s.out[w][r][e];
    // A position outside the cache: the token's key and value have no place,
    // and attention without them is no answer.
    out[i] = T::from_f32(pos >= 0 ? f : NAN);
  }
}

template <class T, int D>
hipError_t launch_rep(const AttnArgs& a, int rep, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(a.batch * a.kv_heads));
  switch (rep) {
    case 1: hipLaunchKernelGGL((decode_attn_kernel<T, D, 1>), grid, dim3(kAttnThreads), 0, stream, a); break;
    case 2: hipLaunchKernelGGL((decode_attn_kernel<T, D, 2>), grid, dim3(kAttnThreads), 0, stream, a); break;
    case 4: hipLaunchKernelGGL((decode_attn_kernel<T, D, 4>), grid, dim3(kAttnThreads), 0, stream, a); break;
    default: hipLaunchKernelGGL((decode_attn_kernel<T, D, 8>), grid, dim3(kAttnThreads), 0, stream, a); break;
  }
  return hipGetLastError();
}

// out = silu(gate) * up, fp32 math, one rounding.  Thread = 8 columns of a row.
template <class T>
__global__ __launch_bounds__(256) void silu_mul_kernel(const void* gate, const void* up, int64_t in_stride, void* out,
                                                       int rows, int chunks) {
  using raw = typename T::raw_t;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= static_cast<int64_t>(rows) * chunks) return;
  const int64_t r = i / chunks;
  const int64_t c = (i - r * chunks) * 8;
  const u32x4 g = ld_chunk(static_cast<const raw*>(gate) + r * in_stride + c);
  const u32x4 u = ld_chunk(static_cast<const raw*>(up) + r * in_stride + c);
  float f[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float x = chunk_elem<T>(g, e);
    f[e] = x / (1.f + expf(-x)) * chunk_elem<T>(u, e);
  }
  st_chunk(static_cast<raw*>(out) + r * chunks * 8 + c, pack_chunk<T>(f));
}

}  // namespace

hipError_t launch_decode_attn(const AttnArgs& a, int dtype, int head_dim, int rep, hipStream_t stream) {
  if (dtype == MLORA_BF16) return head_dim == 64 ? launch_rep<BF16, 64>(a, rep, stream) : launch_rep<BF16, 128>(a, rep, stream);
  return head_dim == 64 ? launch_rep<F16, 64>(a, rep, stream) : launch_rep<F16, 128>(a, rep, stream);
}

hipError_t launch_silu_mul(const void* gate, const void* up, int64_t in_stride, void* out, int rows, int width, int dtype,
                           hipStream_t stream) {
  const int64_t blocks = (static_cast<int64_t>(rows) * (width / 8) + 255) / 256;
  if (blocks <= 0) return hipSuccess;
  if (!grid_fits(blocks)) return hipErrorInvalidConfiguration;
  const dim3 grid(static_cast<unsigned>(blocks));
  if (dtype == MLORA_BF16)
    hipLaunchKernelGGL((silu_mul_kernel<BF16>), grid, dim3(256), 0, stream, gate, up, in_stride, out, rows, width / 8);
  else
    hipLaunchKernelGGL((silu_mul_kernel<F16>), grid, dim3(256), 0, stream, gate, up, in_stride, out, rows, width / 8);
  return hipGetLastError();
}

}  // namespace mlora
