// The parts of a decoder layer's decode step around its quantized linears
// (DecodeRunner.step): residual add + RMSNorm, one-token attention over a
// static bf16 K/V cache with the rotary embedding and the cache write in the
// same launch, and SiLU(gate) * up.
//
// What bounds them: at decode batches each moves a few KB to a few MB, so
// launches and dependent round trips are the cost, not bytes. As separate
// library launches (casts, products, concatenations, copies, softmax: about 22
// a layer, 4-5 us each in a graph) they took 100 us of a 133 us layer at
// batch 1; here four launches a layer.

#include "pe_internal.h"

namespace pe {

constexpr int kNormMaxThreads = 1024;
constexpr int kNormMaxIter = 4;

__device__ __forceinline__ void unpack_bf8(const uint4 u, float v[8]) {
  const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = __builtin_bit_cast(float, w[i] << 16);
    v[2 * i + 1] = __builtin_bit_cast(float, w[i] & 0xffff0000u);
  }
}
__device__ __forceinline__ uint4 pack_bf8(const float v[8]) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = pack16x2(v[2 * i], v[2 * i + 1], true);
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// ---------------------------------------------------------------------------
// x_out = bf16(x + r) (when r is given), h = bf16(x_out / rms(x_out) * w): one
// workgroup per row, the row in registers (8 columns a thread and pass, one
// 16-byte load), so each value is read once. IT: passes over the row.
// ---------------------------------------------------------------------------
template <int IT>
__global__ __launch_bounds__(kNormMaxThreads) void add_rms_norm_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ r, const uint16_t* __restrict__ w,
    int cols, float eps, uint16_t* __restrict__ x_out, uint16_t* __restrict__ h) {
  __shared__ float sums[kNormMaxThreads / 64];
  const int64_t row = (int64_t)blockIdx.x * cols;
  float v[IT][8];
  float ss = 0.f;
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int c = (it * (int)blockDim.x + (int)threadIdx.x) * 8;
    if (c >= cols) {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[it][i] = 0.f;
      continue;
    }
    unpack_bf8(*reinterpret_cast<const uint4*>(x + row + c), v[it]);
    if (r) {
      float a[8];
      unpack_bf8(*reinterpret_cast<const uint4*>(r + row + c), a);
#pragma unroll
      for (int i = 0; i < 8; ++i) v[it][i] = bf2f(f2bf_rne(v[it][i] + a[i]));
      *reinterpret_cast<uint4*>(x_out + row + c) = pack_bf8(v[it]);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) ss = __builtin_fmaf(v[it][i], v[it][i], ss);
  }
  ss = wave_sum_dpp(ss);
  if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6] = ss;
  __syncthreads();
  float total = 0.f;
  for (int i = 0; i < (int)blockDim.x / 64; ++i) total += sums[i];
  const float scale = 1.f / __builtin_sqrtf(total / (float)cols + eps);
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int c = (it * (int)blockDim.x + (int)threadIdx.x) * 8;
    if (c >= cols) continue;
    float g[8];
    unpack_bf8(*reinterpret_cast<const uint4*>(w + c), g);
#pragma unroll
    for (int i = 0; i < 8; ++i) g[i] *= v[it][i] * scale;
    *reinterpret_cast<uint4*>(h + row + c) = pack_bf8(g);
  }
}

// out[row, c] = bf16(silu(gu[row, c]) * gu[row, cols + c]), 8 columns a thread
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ gu,
                                                       int64_t groups, int cols8,
                                                       uint16_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= groups) return;
  const int64_t row = i / cols8;
  const int c = (int)(i - row * cols8);
  const uint4* src = reinterpret_cast<const uint4*>(gu) + row * 2 * cols8 + c;
  float g[8], u[8];
  unpack_bf8(src[0], g);
  unpack_bf8(src[cols8], u);
#pragma unroll
  for (int k = 0; k < 8; ++k) g[k] = g[k] / (1.f + expf(-g[k])) * u[k];
  reinterpret_cast<uint4*>(out)[i] = pack_bf8(g);
}

// ---------------------------------------------------------------------------
// One-token attention. Workgroup (split, b * KVH + kvh) of four waves takes the
// positions of one split, 64 a step, for the GRP query heads of its KV head:
//  * scores: lane = position, the waves share the D dimensions (K is stored
//    [D][L], so a wave's load of one dimension is one run of 64 positions and
//    no score needs a cross-lane sum); the rotated query is broadcast from LDS;
//  * softmax of the step: one wave per query head, running maximum and sum;
//  * values: a wave takes 16 positions, 16 bytes of a row per lane, GRP x 8
//    fp32 sums per lane, added across lanes and waves once at the end.
// The loads of the next step's K go out as soon as this step's scores are done
// with theirs, those of V after the values: each is in flight over the rest.
// The query, the new key and the new value of the position come from the qkv
// row; every workgroup rotates its own query (D x GRP values), and the
// workgroup that owns the position stores key and value into the cache and
// uses them from LDS. Scores, probabilities and sums are fp32.
//
// Splits: as many as give about kAttnTargetWgs workgroups, at least one step
// each, divided by the position (read on the device, so a captured launch
// serves every position); with more than one, each writes its unnormalised sums
// with coherent stores and the last one of a (sequence, KV head) to finish adds
// them in split order.
// ---------------------------------------------------------------------------
constexpr int kAttnStep = 64;
constexpr int kAttnMaxSplits = 64;
constexpr int kAttnTargetWgs = 512;
constexpr float kLog2e = 1.4426950408889634f;

// maximum over the 64 lanes, in every lane (DPP inside 16-lane rows, readlane across)
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, lane_xor<1>(v));
  v = fmaxf(v, lane_xor<2>(v));
  v = fmaxf(v, lane_xor<4>(v));
  v = fmaxf(v, lane_xor<8>(v));
  const int b = __builtin_bit_cast(int, v);
  return fmaxf(fmaxf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 0)),
                     __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 16))),
               fmaxf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 32)),
                     __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 48))));
}

// raw buffer over `bytes` bytes at p (bounds-checked by the hardware); the
// coherent form (sc1) reads and writes what every XCD sees alike
constexpr int kAttnSC1 = 16;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t attn_buf(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}

// fp32 words of one split's sums: GRP x D values, then GRP maxima and GRP sums
template <int D, int GRP>
constexpr int attn_part_words() { return GRP * D + (2 * GRP + 3) / 4 * 4; }

template <int D, int GRP>
__global__ __launch_bounds__(256) void decode_attn_kernel(
    const uint16_t* __restrict__ qkv, const float* __restrict__ rope,
    const int64_t* __restrict__ pos_p, uint16_t* __restrict__ kc, uint16_t* __restrict__ vc,
    uint16_t* __restrict__ out, int KVH, int L, int NS, float scale, float* __restrict__ part,
    uint32_t* __restrict__ cnt) {
  constexpr int LPR = D / 8;       // lanes per value row
  constexpr int RPI = 64 / LPR;    // value rows per load
  constexpr int NV = 16 / RPI;     // value loads per step and wave
  constexpr int KD = D / 4;        // dimensions per wave
  constexpr int GW = (GRP + 3) / 4;  // query heads per wave in the softmax
  constexpr int PW = attn_part_words<D, GRP>();
  constexpr int Q = GRP * D / 4;   // 16-byte quads of the output
  constexpr int SL = Q < 256 ? 256 / Q : 1;  // slices of the splits in the last sum
  constexpr int QI = Q > 256 ? Q / 256 : 1;
  __shared__ __align__(16) float qs[GRP][D];
  __shared__ float kn[D], vn[D];
  __shared__ float sc[4][GRP][kAttnStep];
  __shared__ float pr[GRP][kAttnStep];
  __shared__ float alpha[GRP], mfin[GRP], lfin[GRP];
  __shared__ __align__(16) float ob[4][GRP * D < 256 ? 256 : GRP * D];
  __shared__ float wt[GRP][kAttnMaxSplits];
  __shared__ uint32_t last;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int y = blockIdx.y;
  const int b = y / KVH, kvh = y - b * KVH;
  const int64_t pos64 = *pos_p;
  if (pos64 < 0 || pos64 >= L) return;
  const int pos = (int)pos64;
  const int steps = pos / kAttnStep + 1;
  const int per = (steps + NS - 1) / NS;
  const int s0 = blockIdx.x * per, s1 = min(steps, s0 + per);
  if (s0 >= s1) return;
  const int active = (steps + per - 1) / per;

  const int H = KVH * GRP;
  const uint16_t* qrow = qkv + (int64_t)b * (H + 2 * KVH) * D;
  uint16_t* kb = kc + (int64_t)y * D * L;
  uint16_t* vb = vc + (int64_t)y * L * D;
  const __amdgpu_buffer_rsrc_t kbuf = attn_buf(kb, (uint32_t)D * L * 2);
  const __amdgpu_buffer_rsrc_t vbuf = attn_buf(vb, (uint32_t)D * L * 2);
  const int r0 = lane / LPR, dc = (lane - r0 * LPR) * 8;

  // positions past pos read the row of pos (their scores are masked below)
  uint16_t kr[KD];
  u32x4v vr[NV];
  auto load_k = [&](int st) {
    const int off = min(st * kAttnStep + lane, pos) * 2;
#pragma unroll
    for (int d = 0; d < KD; ++d)
      kr[d] = __builtin_amdgcn_raw_buffer_load_b16(kbuf, off, (wave * KD + d) * L * 2, 0);
  };
  auto load_v = [&](int st) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int row = min(st * kAttnStep + 16 * wave + i * RPI + r0, pos);
      vr[i] = __builtin_bit_cast(
          u32x4v, __builtin_amdgcn_raw_buffer_load_b128(vbuf, (row * D + dc) * 2, 0, 0));
    }
  };
  load_k(s0);
  load_v(s0);

  // rotate the query heads (scaled, in log2 units) and the new key
  const bool owner = s1 == steps;
  for (int i = tid; i < (GRP + 1) * (D / 2); i += 256) {
    const int hd = i / (D / 2), j = i - hd * (D / 2);
    const uint16_t* src = qrow + (int64_t)(hd < GRP ? kvh * GRP + hd : H + kvh) * D;
    const float a = bf2f(src[j]), c = bf2f(src[j + D / 2]);
    const float cs = rope[j], sn = rope[D / 2 + j];
    const float o1 = a * cs - c * sn, o2 = c * cs + a * sn;
    if (hd < GRP) {
      qs[hd][j] = o1 * (scale * kLog2e);
      qs[hd][j + D / 2] = o2 * (scale * kLog2e);
    } else {
      const uint16_t k1 = f2bf_rne(o1), k2 = f2bf_rne(o2);
      kn[j] = bf2f(k1);
      kn[j + D / 2] = bf2f(k2);
      if (owner) {
        kb[(int64_t)j * L + pos] = k1;
        kb[(int64_t)(j + D / 2) * L + pos] = k2;
      }
    }
  }
  if (owner && tid < D) {
    const uint16_t v = qrow[(int64_t)(H + KVH + kvh) * D + tid];
    vn[tid] = bf2f(v);
    vb[(int64_t)pos * D + tid] = v;
  }
  __syncthreads();

  float m_run[GW], l_run[GW], s_new[GW];  // s_new: the new position's score
#pragma unroll
  for (int k = 0; k < GW; ++k) {
    m_run[k] = -__builtin_inff();
    l_run[k] = s_new[k] = 0.f;
    const int g = wave + 4 * k;
    if (owner && g < GRP) {
      float t = 0.f;
#pragma unroll
      for (int d = 0; d < D; d += 64) t = __builtin_fmaf(qs[g][d + lane], kn[d + lane], t);
      s_new[k] = wave_sum_dpp(t);
    }
  }
  float acc[GRP][8];
#pragma unroll
  for (int g = 0; g < GRP; ++g)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[g][j] = 0.f;

  for (int st = s0; st < s1; ++st) {
    const int p = st * kAttnStep + lane;
    float s[GRP];
#pragma unroll
    for (int g = 0; g < GRP; ++g) s[g] = 0.f;
#pragma unroll
    for (int d = 0; d < KD; d += 4) {
      float kf[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) kf[u] = bf2f(kr[d + u]);
#pragma unroll
      for (int g = 0; g < GRP; ++g) {
        const float4 q = *reinterpret_cast<const float4*>(&qs[g][wave * KD + d]);
        s[g] = __builtin_fmaf(q.x, kf[0], s[g]);
        s[g] = __builtin_fmaf(q.y, kf[1], s[g]);
        s[g] = __builtin_fmaf(q.z, kf[2], s[g]);
        s[g] = __builtin_fmaf(q.w, kf[3], s[g]);
      }
    }
#pragma unroll
    for (int g = 0; g < GRP; ++g) sc[wave][g][lane] = s[g];
    if (st + 1 < s1) load_k(st + 1);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < GW; ++k) {
      const int g = wave + 4 * k;
      if (g < GRP) {
        float t = (sc[0][g][lane] + sc[1][g][lane]) + (sc[2][g][lane] + sc[3][g][lane]);
        if (p == pos) t = s_new[k];
        if (p > pos) t = -__builtin_inff();
        const float mn = fmaxf(m_run[k], wave_max(t));
        const float ms = mn == -__builtin_inff() ? 0.f : mn;  // no score above -inf so far
        const float e = __builtin_amdgcn_exp2f(t - ms);
        const float al = __builtin_amdgcn_exp2f(m_run[k] - ms);
        l_run[k] = l_run[k] * al + wave_sum_dpp(e);
        m_run[k] = mn;
        pr[g][lane] = e;
        if (lane == 0) alpha[g] = al;
      }
    }
    __syncthreads();
    if (st != s0) {
#pragma unroll
      for (int g = 0; g < GRP; ++g) {
        const float al = alpha[g];
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[g][j] *= al;
      }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int rl = 16 * wave + i * RPI + r0;
      float v[8];
      unpack_bf8(make_uint4(vr[i][0], vr[i][1], vr[i][2], vr[i][3]), v);
      bool live = true;
      if (st == steps - 1) {  // the step that holds pos
        const int row = st * kAttnStep + rl;
        live = row <= pos;
        if (row == pos) {
#pragma unroll
          for (int j = 0; j < 8; ++j) v[j] = vn[dc + j];
        }
      }
      if (live) {
#pragma unroll
        for (int g = 0; g < GRP; ++g) {
          const float w = pr[g][rl];
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[g][j] = __builtin_fmaf(w, v[j], acc[g][j]);
        }
      }
    }
    if (st + 1 < s1) load_v(st + 1);
  }

  // sums of the workgroup
#pragma unroll
  for (int g = 0; g < GRP; ++g)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
#pragma unroll
      for (int off = LPR; off < 64; off <<= 1) acc[g][j] += __shfl_xor(acc[g][j], off, 64);
      if (r0 == 0) ob[wave][g * D + dc + j] = acc[g][j];
    }
#pragma unroll
  for (int k = 0; k < GW; ++k)
    if (wave + 4 * k < GRP && lane == 0) {
      mfin[wave + 4 * k] = m_run[k];
      lfin[wave + 4 * k] = l_run[k];
    }
  __syncthreads();
  uint16_t* orow = out + ((int64_t)b * H + (int64_t)kvh * GRP) * D;
  auto ob_quad = [&](int q) {
    float4v t;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      t[u] = (ob[0][4 * q + u] + ob[1][4 * q + u]) + (ob[2][4 * q + u] + ob[3][4 * q + u]);
    return t;
  };
  auto store_quad = [&](int q, float4v t) {
    *reinterpret_cast<uint2*>(orow + 4 * q) =
        make_uint2(pack16x2(t[0], t[1], true), pack16x2(t[2], t[3], true));
  };
  if (active == 1) {
    for (int q = tid; q < Q; q += 256) {
      const float l = lfin[4 * q / D];
      float4v t = ob_quad(q);
#pragma unroll
      for (int u = 0; u < 4; ++u) t[u] /= l;
      store_quad(q, t);
    }
    return;
  }
  const __amdgpu_buffer_rsrc_t pbuf = attn_buf(part + (int64_t)y * NS * PW, (uint32_t)NS * PW * 4);
  const int mine = (int)blockIdx.x * PW * 4;
  for (int q = tid; q < Q; q += 256)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4v, ob_quad(q)), pbuf, q * 16,
                                           mine, kAttnSC1);
  if (tid < GRP) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, mfin[tid]), pbuf,
                                          (GRP * D + tid) * 4, mine, kAttnSC1);
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, lfin[tid]), pbuf,
                                          (GRP * D + GRP + tid) * 4, mine, kAttnSC1);
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (tid == 0) last = atomicAdd(&cnt[y], 1u) + 1 == (uint32_t)active ? 1u : 0u;
  __syncthreads();
  if (!last) return;
  // weight of each split, exp2(m_s - max m) / total; the first sums' loads are
  // already on their way
  const int slice = SL > 1 ? tid / Q : 0;
  constexpr int kBatch = 8;
  u32x4v t[kBatch];
  auto load_parts = [&](int q, int first) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
      t[u] = __builtin_bit_cast(
          u32x4v, __builtin_amdgcn_raw_buffer_load_b128(
                      pbuf, min(first + u * SL, active - 1) * (PW * 4) + q * 16, 0, kAttnSC1));
  };
  load_parts(tid & (Q - 1), slice);
  for (int g = wave; g < GRP; g += 4) {
    float m = -__builtin_inff(), l = 0.f;
    if (lane < active) {
      m = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                        pbuf, (lane * PW + GRP * D + g) * 4, 0, kAttnSC1));
      l = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                        pbuf, (lane * PW + GRP * D + GRP + g) * 4, 0, kAttnSC1));
    }
    const float mm = wave_max(m);
    const float e = __builtin_amdgcn_exp2f(m - (mm == -__builtin_inff() ? 0.f : mm));
    const float total = wave_sum_dpp(e * l);
    wt[g][lane] = e / total;
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < QI; ++it) {
    const int q = (tid & (Q < 256 ? Q - 1 : 255)) + 256 * it;
    const int g = 4 * q / D;
    if (it > 0) load_parts(q, slice);
    float4v o = {0.f, 0.f, 0.f, 0.f};
    for (int s = slice; s < active; s += kBatch * SL) {
      if (s != slice) load_parts(q, s);
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
        if (s + u * SL < active) {
          const float w = wt[g][s + u * SL];
          const float4v tf = __builtin_bit_cast(float4v, t[u]);
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = __builtin_fmaf(w, tf[i], o[i]);
        }
    }
    if constexpr (SL == 1) {
      store_quad(q, o);
    } else {
      float* red = &ob[0][0];  // SL x Q quads: 4 KB, within ob
      *reinterpret_cast<float4v*>(red + tid * 4) = o;
      __syncthreads();
      if (tid < Q) {
#pragma unroll
        for (int k = 1; k < SL; ++k) {
          const float4v z = *reinterpret_cast<const float4v*>(red + (k * Q + tid) * 4);
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] += z[i];
        }
        store_quad(tid, o);
      }
    }
  }
  if (tid == 0) __hip_atomic_store(&cnt[y], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------------
// lm_head: logits[m, n] = x[m] . w[n] for a few rows, bf16 in, fp32 out. Bound
// by reading w once. A persistent workgroup of eight waves takes tiles of 16
// rows of w; the waves split K, so a wave reads K / 4 consecutive bytes of each
// row, R 16-byte loads a lane in flight, the next tile's behind this one's
// across the barrier that ends a tile. v_mfma_f32_16x16x32_bf16 with w as A, x
// (in LDS, rows padded by 16 bytes) as B; the eight partial tiles meet in LDS
// and leave as fp32 (no rounding to bf16 on the way). K: a multiple of 256 R.
//
// Measured, 151936 x 4096 bf16 (library product and conversion to fp32 -> this):
// 1 row 246 -> 196 us (6.3 TB/s), 4 rows 248 -> 205, 16 rows 258 -> 229; x 2048:
// 203 -> 103 and 207 -> 124 us; 2000 x 1024 24 -> 9 us. Non-temporal loads 212 us
// at 1 row, 8 or 16 loads in flight level at 4096 and 5% slower at 2048 columns,
// tiles of 32 rows 242-257, a run of neighbouring tiles per workgroup 202.
// ---------------------------------------------------------------------------
constexpr int kHeadWaves = 8;
constexpr int kHeadTile = 16;
constexpr int kHeadMaxRows = 16;
constexpr int kHeadLoads = 4;
static size_t head_lds(int64_t M, int K) {
  return (size_t)M * (K * 2 + 16) + 2 * kHeadWaves * kHeadTile * 16 * 4;
}

__global__ __launch_bounds__(kHeadWaves * 64) void head_kernel(const uint16_t* __restrict__ x,
                                                               const uint16_t* __restrict__ w,
                                                               int M, int N, int K,
                                                               float* __restrict__ y) {
  extern __shared__ __align__(16) unsigned char head_smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int R = kHeadLoads;
  const int xrow = K * 2 + 16;
  float* red = reinterpret_cast<float*>(head_smem + M * xrow);
  const int tiles = (N + kHeadTile - 1) / kHeadTile;
  const int blocks = K / (kHeadWaves * 32 * R);  // groups of R k-steps per tile and wave
  const int voff = (lane & 15) * K * 2 + wave * (K / kHeadWaves * 2) + (lane >> 4) * 16;
  auto tile_buf = [&](int t) {
    // rows past N read as zeros; past the last tile nothing is read
    const int rows = t < tiles ? min(kHeadTile, N - t * kHeadTile) : 0;
    return attn_buf(w + (int64_t)(t < tiles ? t : 0) * kHeadTile * K, (uint32_t)rows * K * 2);
  };
  auto load = [&](__amdgpu_buffer_rsrc_t buf, int off) {
    return __builtin_bit_cast(u32x4v, __builtin_amdgcn_raw_buffer_load_b128(buf, voff, off, 0));
  };
  u32x4v a[R];
  int t = blockIdx.x;
  __amdgpu_buffer_rsrc_t buf = tile_buf(t);
#pragma unroll
  for (int i = 0; i < R; ++i) a[i] = load(buf, i * 64);
  for (int i = tid; i < M * (K / 8); i += kHeadWaves * 64) {
    const int m = i / (K / 8), c = i - m * (K / 8);
    *reinterpret_cast<uint4*>(head_smem + m * xrow + c * 16) =
        reinterpret_cast<const uint4*>(x)[i];
  }
  __syncthreads();
  const unsigned char* xl = head_smem + min(lane & 15, M - 1) * xrow + wave * (K / kHeadWaves * 2) +
                            (lane >> 4) * 16;
  for (int par = 0; t < tiles; t += gridDim.x, par ^= 1) {
    const __amdgpu_buffer_rsrc_t next = tile_buf(t + (int)gridDim.x);
    float4v acc = {0.f, 0.f, 0.f, 0.f};
    for (int b = 0; b < blocks; ++b) {
      const bool here = b + 1 < blocks;  // uniform: the loads behind these
      const __amdgpu_buffer_rsrc_t src = here ? buf : next;
      const int s0 = here ? (b + 1) * R * 64 : 0;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const bf16x8v xb = *reinterpret_cast<const bf16x8v*>(xl + (b * R + i) * 64);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8v, a[i]), xb, acc, 0, 0, 0);
        a[i] = load(src, s0 + i * 64);
      }
    }
    buf = next;
    // lane: batch row lane % 16, w rows 4 (lane / 16) .. + 3 of the tile
    float* part = red + par * (kHeadWaves * 16 * kHeadTile);
    *reinterpret_cast<float4v*>(part + wave * (16 * kHeadTile) + (lane & 15) * kHeadTile +
                                (lane >> 4) * 4) = acc;
    __syncthreads();
    if (tid < kHeadTile * M) {
      float s = 0.f;
#pragma unroll
      for (int k = 0; k < kHeadWaves; ++k) s += part[k * (16 * kHeadTile) + tid];
      const int n = t * kHeadTile + (tid & (kHeadTile - 1));
      if (n < N) y[(int64_t)(tid / kHeadTile) * N + n] = s;
    }
  }
}

static bool attn_shape_ok(int64_t batch, int kv_heads, int group, int head_dim, int64_t max_len) {
  if (batch < 1 || kv_heads < 1 || max_len < 1 || batch * kv_heads > 65535) return false;
  if (group != 1 && group != 2 && group != 4 && group != 8) return false;
  if (head_dim != 64 && head_dim != 128 && head_dim != 256) return false;
  return max_len <= INT32_MAX / (2 * head_dim);  // one head's cache is one 32-bit buffer
}

// splits of one (sequence, KV head); one where the counters do not reach
static int attn_splits(int64_t batch, int kv_heads, int64_t max_len) {
  const int64_t rows = batch * kv_heads;
  if (rows > kWsCounters) return 1;
  int64_t ns = (kAttnTargetWgs + rows - 1) / rows;
  ns = ns < kAttnMaxSplits ? ns : kAttnMaxSplits;
  const int64_t steps = (max_len + kAttnStep - 1) / kAttnStep;
  return (int)(ns < steps ? ns : steps);
}

template <int D>
static int launch_attn(int grp, dim3 grid, hipStream_t st, const uint16_t* qkv, const float* rope,
                       const int64_t* pos, uint16_t* kc, uint16_t* vc, uint16_t* out, int kvh,
                       int L, int ns, float scale, float* part, uint32_t* cnt) {
  switch (grp) {
    case 1: decode_attn_kernel<D, 1><<<grid, 256, 0, st>>>(qkv, rope, pos, kc, vc, out, kvh, L, ns, scale, part, cnt); break;
    case 2: decode_attn_kernel<D, 2><<<grid, 256, 0, st>>>(qkv, rope, pos, kc, vc, out, kvh, L, ns, scale, part, cnt); break;
    case 4: decode_attn_kernel<D, 4><<<grid, 256, 0, st>>>(qkv, rope, pos, kc, vc, out, kvh, L, ns, scale, part, cnt); break;
    default: decode_attn_kernel<D, 8><<<grid, 256, 0, st>>>(qkv, rope, pos, kc, vc, out, kvh, L, ns, scale, part, cnt); break;
  }
  return launch_status();
}

}  // namespace pe

using namespace pe;

extern "C" int pe_add_rms_norm(const void* x, const void* r, const void* w, int64_t rows, int cols,
                               float eps, void* x_out, void* h, void* stream) {
  if (!x || !w || !h || (r && !x_out)) return PE_ERR_NULL;
  if (rows < 0 || rows > INT32_MAX || cols <= 0 || cols % 8 ||
      cols > 8 * kNormMaxThreads * kNormMaxIter)
    return PE_ERR_DIMS;
  if (!aligned16(x) || !aligned16(w) || !aligned16(h) || (r && (!aligned16(r) || !aligned16(x_out))))
    return PE_ERR_ALIGN;
  if (rows == 0) return PE_OK;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const uint16_t *xp = reinterpret_cast<const uint16_t*>(x), *rp = reinterpret_cast<const uint16_t*>(r),
                 *wp = reinterpret_cast<const uint16_t*>(w);
  uint16_t *xo = reinterpret_cast<uint16_t*>(x_out), *hp = reinterpret_cast<uint16_t*>(h);
  const int threads = cols / 8 < kNormMaxThreads ? (cols / 8 + 63) / 64 * 64 : kNormMaxThreads;
  if (cols <= 8 * kNormMaxThreads)
    add_rms_norm_kernel<1><<<(unsigned)rows, threads, 0, st>>>(xp, rp, wp, cols, eps, xo, hp);
  else
    add_rms_norm_kernel<kNormMaxIter><<<(unsigned)rows, threads, 0, st>>>(xp, rp, wp, cols, eps, xo, hp);
  return launch_status();
}

extern "C" int pe_silu_mul(const void* gate_up, int64_t rows, int cols, void* out, void* stream) {
  if (!gate_up || !out) return PE_ERR_NULL;
  if (rows < 0 || cols <= 0 || cols % 8 || rows > ((int64_t)INT32_MAX * 256) / (cols / 8))
    return PE_ERR_DIMS;
  if (!aligned16(gate_up) || !aligned16(out)) return PE_ERR_ALIGN;
  if (rows == 0) return PE_OK;
  const int64_t groups = rows * (cols / 8);
  silu_mul_kernel<<<(unsigned)((groups + 255) / 256), 256, 0, reinterpret_cast<hipStream_t>(stream)>>>(
      reinterpret_cast<const uint16_t*>(gate_up), groups, cols / 8, reinterpret_cast<uint16_t*>(out));
  return launch_status();
}

extern "C" size_t pe_decode_attention_workspace_size(int64_t batch, int kv_heads, int group,
                                                     int head_dim, int64_t max_len) {
  if (!attn_shape_ok(batch, kv_heads, group, head_dim, max_len)) return 0;
  const int ns = attn_splits(batch, kv_heads, max_len);
  return kWsCounterBytes + (size_t)batch * kv_heads * ns * (group * head_dim + (2 * group + 3) / 4 * 4) * 4;
}

extern "C" int pe_decode_attention(const void* qkv, const float* rope, const int64_t* pos,
                                   void* k_cache, void* v_cache, void* out, int64_t batch,
                                   int kv_heads, int group, int head_dim, int64_t max_len,
                                   float scale, void* workspace, size_t workspace_bytes,
                                   void* stream) {
  if (!qkv || !rope || !pos || !k_cache || !v_cache || !out) return PE_ERR_NULL;
  if (!attn_shape_ok(batch, kv_heads, group, head_dim, max_len)) return PE_ERR_DIMS;
  if (!aligned16(v_cache)) return PE_ERR_ALIGN;
  const size_t need = pe_decode_attention_workspace_size(batch, kv_heads, group, head_dim, max_len);
  if (!workspace || workspace_bytes < need) return PE_ERR_WORKSPACE;
  if (!aligned16(workspace)) return PE_ERR_ALIGN;
  const int ns = attn_splits(batch, kv_heads, max_len);
  const dim3 grid((unsigned)ns, (unsigned)(batch * kv_heads));
  uint32_t* cnt = reinterpret_cast<uint32_t*>(workspace);
  float* part = reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + kWsCounterBytes);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  auto q = reinterpret_cast<const uint16_t*>(qkv);
  auto kc = reinterpret_cast<uint16_t*>(k_cache), vc = reinterpret_cast<uint16_t*>(v_cache);
  auto o = reinterpret_cast<uint16_t*>(out);
  const int L = (int)max_len;
  if (head_dim == 64) return launch_attn<64>(group, grid, st, q, rope, pos, kc, vc, o, kv_heads, L, ns, scale, part, cnt);
  if (head_dim == 128) return launch_attn<128>(group, grid, st, q, rope, pos, kc, vc, o, kv_heads, L, ns, scale, part, cnt);
  return launch_attn<256>(group, grid, st, q, rope, pos, kc, vc, o, kv_heads, L, ns, scale, part, cnt);
}

extern "C" int pe_lm_head_fits(int64_t M, int64_t N, int K) {
  return M >= 1 && M <= kHeadMaxRows && N >= 1 && N <= INT32_MAX - kHeadTile && K >= 1024 &&
         K % 1024 == 0 && K <= 16384 && head_lds(M, K) <= (size_t)160 * 1024;
}

extern "C" int pe_lm_head(const void* x, const void* w, int64_t M, int64_t N, int K, float* y,
                          void* stream) {
  if (!x || !w || !y) return PE_ERR_NULL;
  if (!pe_lm_head_fits(M, N, K)) return PE_ERR_DIMS;
  if (!aligned16(x) || !aligned16(w)) return PE_ERR_ALIGN;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const size_t lds = head_lds(M, K);
  const int64_t tiles = (N + kHeadTile - 1) / kHeadTile;
  const int64_t wgs = (int64_t)num_cus() * (lds <= (size_t)80 * 1024 ? 2 : 1);
  const unsigned grid = (unsigned)(tiles < wgs ? tiles : wgs);
  auto xp = reinterpret_cast<const uint16_t*>(x), wp = reinterpret_cast<const uint16_t*>(w);
  if (lds > (size_t)64 * 1024 &&
      hipFuncSetAttribute(reinterpret_cast<const void*>(head_kernel),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return PE_ERR_LAUNCH;
  head_kernel<<<grid, kHeadWaves * 64, lds, st>>>(xp, wp, (int)M, (int)N, K, y);
  return launch_status();
}
