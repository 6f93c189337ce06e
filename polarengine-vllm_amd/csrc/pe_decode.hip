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
// K and V loads of a step are issued together, before the scores.
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

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

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
  constexpr int PS = GRP * (D + 2);  // fp32 words of one split's sums
  __shared__ __align__(16) float qs[GRP][D];
  __shared__ float kn[D], vn[D];
  __shared__ float sc[4][GRP][kAttnStep];
  __shared__ float pr[GRP][kAttnStep];
  __shared__ float alpha[GRP], mfin[GRP], lfin[GRP];
  __shared__ float ob[4][GRP][D];
  __shared__ float wt[GRP][kAttnMaxSplits];
  __shared__ uint32_t last;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int y = blockIdx.y;
  const int b = y / KVH, kvh = y - b * KVH;
  const int64_t pos64 = *pos_p;
  if (pos64 < 0 || pos64 >= L) return;  // refused by the caller's table lookup; never out of range here
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
  const bool owner = s1 == steps;

  // rotate the query heads (scaled, in log2 units) and the new key
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
  if (tid < D) {
    const uint16_t v = qrow[(int64_t)(H + KVH + kvh) * D + tid];
    vn[tid] = bf2f(v);
    if (owner) vb[(int64_t)pos * D + tid] = v;
  }

  const int r0 = lane / LPR, dc = (lane - r0 * LPR) * 8;
  float m_run[(GRP + 3) / 4], l_run[(GRP + 3) / 4];
#pragma unroll
  for (int k = 0; k < (GRP + 3) / 4; ++k) {
    m_run[k] = -__builtin_inff();
    l_run[k] = 0.f;
  }
  float acc[GRP][8];
#pragma unroll
  for (int g = 0; g < GRP; ++g)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[g][j] = 0.f;

  for (int st = s0; st < s1; ++st) {
    const int p = st * kAttnStep + lane;
    const uint16_t* kp = kb + (int64_t)(wave * KD) * L + min(p, pos);
    uint16_t kr[KD];
#pragma unroll
    for (int d = 0; d < KD; ++d) kr[d] = kp[(int64_t)d * L];
    uint4 vr[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int row = st * kAttnStep + 16 * wave + i * RPI + r0;
      vr[i] = *reinterpret_cast<const uint4*>(vb + (int64_t)min(row, pos) * D + dc);
    }
    if (st == s0) __syncthreads();  // qs, kn, vn
    float s[GRP];
#pragma unroll
    for (int g = 0; g < GRP; ++g) s[g] = 0.f;
#pragma unroll
    for (int d = 0; d < KD; d += 4) {
      float kf[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) kf[u] = p == pos ? kn[wave * KD + d + u] : bf2f(kr[d + u]);
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
    __syncthreads();
#pragma unroll
    for (int k = 0; k < (GRP + 3) / 4; ++k) {
      const int g = wave + 4 * k;
      if (g < GRP) {
        float t = (sc[0][g][lane] + sc[1][g][lane]) + (sc[2][g][lane] + sc[3][g][lane]);
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
#pragma unroll
    for (int g = 0; g < GRP; ++g) {
      const float al = alpha[g];
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[g][j] *= al;
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int rl = 16 * wave + i * RPI + r0;
      float v[8];
      unpack_bf8(vr[i], v);
      if (st * kAttnStep + rl == pos) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = vn[dc + j];
      }
      if (st * kAttnStep + rl <= pos) {
#pragma unroll
        for (int g = 0; g < GRP; ++g) {
          const float w = pr[g][rl];
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[g][j] = __builtin_fmaf(w, v[j], acc[g][j]);
        }
      }
    }
  }

  // sums of the workgroup
#pragma unroll
  for (int g = 0; g < GRP; ++g)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
#pragma unroll
      for (int off = LPR; off < 64; off <<= 1) acc[g][j] += __shfl_xor(acc[g][j], off, 64);
      if (r0 == 0) ob[wave][g][dc + j] = acc[g][j];
    }
#pragma unroll
  for (int k = 0; k < (GRP + 3) / 4; ++k)
    if (wave + 4 * k < GRP && lane == 0) {
      mfin[wave + 4 * k] = m_run[k];
      lfin[wave + 4 * k] = l_run[k];
    }
  __syncthreads();
  uint16_t* orow = out + ((int64_t)b * H + (int64_t)kvh * GRP) * D;
  if (active == 1) {
    for (int i = tid; i < GRP * D; i += 256) {
      const int g = i / D, d = i - g * D;
      orow[i] = f2bf_rne(((ob[0][g][d] + ob[1][g][d]) + (ob[2][g][d] + ob[3][g][d])) / lfin[g]);
    }
    return;
  }
  uint32_t* mine = reinterpret_cast<uint32_t*>(part) + ((int64_t)y * NS + blockIdx.x) * PS;
  for (int i = tid; i < GRP * D; i += 256) {
    const int g = i / D, d = i - g * D;
    st_dev32(mine + i, __builtin_bit_cast(uint32_t, (ob[0][g][d] + ob[1][g][d]) +
                                                        (ob[2][g][d] + ob[3][g][d])));
  }
  if (tid < GRP) {
    st_dev32(mine + GRP * D + tid, __builtin_bit_cast(uint32_t, mfin[tid]));
    st_dev32(mine + GRP * D + GRP + tid, __builtin_bit_cast(uint32_t, lfin[tid]));
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (tid == 0) last = atomicAdd(&cnt[y], 1u) + 1 == (uint32_t)active ? 1u : 0u;
  __syncthreads();
  if (!last) return;
  const uint32_t* all = reinterpret_cast<const uint32_t*>(part) + (int64_t)y * NS * PS;
  // weight of each split: exp2(m_s - max m) / total
  for (int g = wave; g < GRP; g += 4) {
    float m = -__builtin_inff(), l = 0.f;
    if (lane < active) {
      m = __builtin_bit_cast(float, ld_dev32(all + lane * PS + GRP * D + g));
      l = __builtin_bit_cast(float, ld_dev32(all + lane * PS + GRP * D + GRP + g));
    }
    const float mm = wave_max(m);
    const float e = __builtin_amdgcn_exp2f(m - (mm == -__builtin_inff() ? 0.f : mm));
    const float total = wave_sum_dpp(e * l);
    wt[g][lane] = e / total;
  }
  __syncthreads();
  for (int i = tid; i < GRP * D; i += 256) {
    const int g = i / D;
    float o = 0.f;
    for (int s = 0; s < active; s += 8) {
      float t[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        t[u] = __builtin_bit_cast(float, ld_dev32(all + (int64_t)min(s + u, active - 1) * PS + i));
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (s + u < active) o = __builtin_fmaf(wt[g][s + u], t[u], o);
    }
    orow[i] = f2bf_rne(o);
  }
  if (tid == 0) __hip_atomic_store(&cnt[y], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

static bool attn_shape_ok(int64_t batch, int kv_heads, int group, int head_dim, int64_t max_len) {
  if (batch < 1 || kv_heads < 1 || max_len < 1 || batch * kv_heads > 65535) return false;
  if (group != 1 && group != 2 && group != 4 && group != 8) return false;
  if (head_dim != 64 && head_dim != 128 && head_dim != 256) return false;
  return max_len <= INT32_MAX / 2;
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
  return kWsCounterBytes + (size_t)batch * kv_heads * ns * group * (head_dim + 2) * 4;
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
