// PolarQuant quantizer on gfx950: weight [N, K] -> codes + fp16 block norms,
// one 16-lane group per (row, 128-block).
//
// Replaces PolarQuantizer.quantize_tensor (polarengine_vllm/quantizer.py:
// 206-257): pad K to the block with zeros, per-block L2 norm clamped at
// 1e-10, unit block rotated by the Hadamard transform and scaled by
// sqrt(128) -- i.e. the unnormalised transform H v with entries +-1 -- and
// code = the first index of the smallest |r - ct[l]| over the raw Lloyd-Max
// centroids; norms are stored as fp16 (round to nearest even).
//
// The transform is the butterfly (DPP across the 16 lanes, each lane holding 8
// consecutive positions) in fp32; the reference's fp32 matmul
// rounds differently, so a code can differ where r sits within a few ulps of
// the midpoint between two centroids. pack = 1 writes the half-block nibble
// layout directly (bits <= 4).

#include "pe_internal.h"

namespace pe {

template <int DT>
__device__ __forceinline__ float load_w(const void* w, int64_t i) {
  if constexpr (DT == PE_DTYPE_F16) return h2f(reinterpret_cast<const uint16_t*>(w)[i]);
  else if constexpr (DT == PE_DTYPE_BF16) return bf2f(reinterpret_cast<const uint16_t*>(w)[i]);
  else return reinterpret_cast<const float*>(w)[i];
}

// ---------------------------------------------------------------------------
// Codes by cell. The scan's answer is a step function of r: for ascending
// centroids the fp32 comparison |r - ct[l+1]| < |r - ct[l]| turns true once and
// stays true as r grows, so T[l], the largest float for which it is false, is
// an exact threshold (found by bisection over the floats between the two) and
// the code is the number of thresholds below r. The range is cut into kCells
// cells by a monotone map (scale by a power of two, clamp, round to integer);
// entry c holds the thresholds in lower cells and the one in c (+inf if none),
// so a code is one LDS read and one comparison whatever the number of levels.
// Centroids that do not ascend, or that put two thresholds in a cell, take the
// scan itself.
// ---------------------------------------------------------------------------
constexpr int kCells = 1024;
constexpr float kCellHi = kCells / 2 - 1, kCellLo = -kCellHi;
constexpr float kRoundMagic = 12582912.f;  // 1.5 * 2^23: the sum's low bits are the rounded integer

struct QuantCells {
  uint2 cell[kCells];  // {thresholds below, the cell's threshold / w as bits}
  float thr[256];
  int at[256];
  float ct[256];
};

// cell of a value given in cells (already divided by w)
__device__ __forceinline__ int cell_of(float t) {
  const float c = __builtin_amdgcn_fmed3f(t, kCellLo, kCellHi);  // a NaN goes to the lowest cell
  return (int)(__builtin_bit_cast(uint32_t, c + kRoundMagic) - 0x4B400000u) + kCells / 2;
}

// floats in ascending order <-> integers in ascending order
__device__ __forceinline__ int ordered(float f) {
  const int i = __builtin_bit_cast(int, f);
  return i >= 0 ? i : (int)(0x80000000u - (uint32_t)i);
}
__device__ __forceinline__ float from_ordered(int i) {
  return __builtin_bit_cast(float, i >= 0 ? i : (int)(0x80000000u - (uint32_t)i));
}

// The whole workgroup (it ends in a barrier). Returns 1 / w, 0 where the scan
// has to be used. A chain of dependent steps that every workgroup waits for: the
// bisection in 32 bits and the ranks by ballots, against 64 bits and a binary
// search in LDS for each cell, take 1.0-1.3 us off every call (1500 x 4000 fp16
// at 32 levels 12.4 -> 11.3 us, 4096 x 4096 20.6 -> 19.3).
__device__ float quant_cells_setup(QuantCells& q, const float* __restrict__ ct, int n_levels) {
  __shared__ int bad;
  const int tid = threadIdx.x;
  if (tid == 0) bad = 0;
  if (tid < n_levels) q.ct[tid] = ct[tid];
  __syncthreads();
  const int n = n_levels - 1;  // thresholds
  if (tid < n) {
    const float a = q.ct[tid], b = q.ct[tid + 1];
    if (!(a < b) || !(__builtin_fabsf(a) < 1e30f) || !(__builtin_fabsf(b) < 1e30f)) {
      bad = 1;
    } else {
      // false at a, true at b
      uint32_t lo = (uint32_t)ordered(a), hi = (uint32_t)ordered(b);  // hi - lo fits 32 bits
      while (hi - lo > 1) {
        const uint32_t mid = lo + ((hi - lo) >> 1);
        const float r = from_ordered((int)mid);
        if (__builtin_fabsf(r - b) < __builtin_fabsf(r - a)) hi = mid;
        else lo = mid;
      }
      q.thr[tid] = from_ordered((int)lo);
    }
  }
  __syncthreads();
  if (bad) return 0.f;  // uniform
  // smallest power of two w with every threshold inside the clamp
  const float amax = fmaxf(__builtin_fabsf(q.thr[0]), __builtin_fabsf(q.thr[n - 1]));
  int e = 0;
  (void)frexpf(amax / (kCellHi - 1.f), &e);
  if (e < -100) e = -100;
  const float inv_w = ldexpf(1.f, -e);
  for (int c = tid; c < kCells; c += 256) q.cell[c].x = 0;
  if (tid < n) q.at[tid] = cell_of(q.thr[tid] * inv_w);
  __syncthreads();
  if (tid + 1 < n && q.at[tid] >= q.at[tid + 1]) bad = 1;
  __syncthreads();
  if (bad) return 0.f;
  if (tid < n) q.cell[q.at[tid]].x = 1;  // the cells that hold a threshold
  __syncthreads();
  // a wave fills 64 consecutive cells at a time: thresholds below them, then
  // their own marks, counted by ballots
  const int lane = tid & 63;
  for (int c0 = tid - lane; c0 < kCells; c0 += 256) {
    int lo = 0;
    for (int l = lane; l - lane < n; l += 64)
      lo += __popcll(__ballot(l < n && q.at[l] < c0));
    const bool here = q.cell[c0 + lane].x != 0;
    const uint64_t marks = __ballot(here);
    lo += __popcll(marks & ((1ull << lane) - 1));
    const float t = here ? q.thr[lo] * inv_w : __builtin_inff();
    q.cell[c0 + lane] = make_uint2((uint32_t)lo, __builtin_bit_cast(uint32_t, t));
  }
  __syncthreads();
  return inv_w;
}

// One butterfly stage over the lane pairing XOR, as one multiply-add per value:
// each lane keeps its value up to a sign that it carries along (`sg`, exact),
// chosen so that its own value enters with +1. Lower lane of a pair: a + b;
// upper: a - b.
template <int XOR>
__device__ __forceinline__ float pair_get(float v) {
  const int i = __builtin_bit_cast(int, v);
  constexpr int ctrl = XOR == 1 ? 0xB1 : XOR == 2 ? 0x4E : XOR == 7 ? 0x141 : 0x128;  // quad_perm, quad_perm, row_half_mirror, row_ror:8
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, i, ctrl, 0xF, 0xF, true));
}
template <int XOR>
__device__ __forceinline__ void signed_stage(float (&v)[8], float& sg, bool upper) {
  const float so = pair_get<XOR>(sg);
  const float f = upper ? -(sg * so) : sg * so;
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = __builtin_fmaf(pair_get<XOR>(v[i]), f, v[i]);
  if (upper) sg = -sg;
}

// VEC: rows of 16-byte aligned 8-value groups with K a multiple of 8 (one or
// two 16-byte loads a lane); otherwise value by value with the edge checked.
// The 16 lanes of a group hold the block's positions 8 p .. 8 p + 7 with
// p = lane bits (b0 ^ b2, b1 ^ b2, b2, b3): the pairings that flip one bit of p
// are then lane xor 1, 2, 7 and 8, all DPP moves.
//
// Bound by VALU: about 25 vector operations a value against 3 bytes of
// traffic. Weight 12288 x 4096, fp16, 32 levels: 50 us (3.0 TB/s, traced)
// against 265 us with the scan over the levels, 2-byte loads and one block per
// lane group and workgroup; the call 48.9 against 278 us, bit-identical.
template <int DT, bool PACK, bool VEC>
__global__ __launch_bounds__(256) void quantize_kernel(const void* __restrict__ w, int64_t ldw,
                                                       int N, int K, int nb,
                                                       const float* __restrict__ ct, int n_levels,
                                                       uint8_t* __restrict__ codes,
                                                       uint16_t* __restrict__ norms) {
  __shared__ QuantCells cells;
  const float inv_w = quant_cells_setup(cells, ct, n_levels);
  const int l16 = threadIdx.x & 15;
  const int p = l16 ^ ((l16 & 4) ? 3 : 0);
  const int64_t items = (int64_t)N * nb;
  const int64_t step = (int64_t)gridDim.x * 16;
  for (int64_t item = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
       item - (threadIdx.x >> 4) < items; item += step) {
    const bool live = item < items;
    const int64_t it = live ? item : items - 1;  // dead groups repeat the last block, store nothing
    const int n = (int)(it / nb), b = (int)(it - (int64_t)n * nb);
    const int k0 = b * kBlock + 8 * p;
    float v[8];
    if constexpr (VEC) {
      constexpr int ES = DT == PE_DTYPE_F32 ? 4 : 2;
      if (k0 < K) {
        load8<DT>(reinterpret_cast<const char*>(w) + ((int64_t)n * ldw + k0) * ES, v);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = 0.f;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        v[i] = (k0 + i < K) ? load_w<DT>(w, (int64_t)n * ldw + k0 + i) : 0.f;
    }

    // L2 norm of the block: lane partial, then across the 16 lanes
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) ss = __builtin_fmaf(v[i], v[i], ss);
    ss += pair_get<1>(ss);
    ss += pair_get<2>(ss);
    ss += pair_get<7>(ss);
    ss += pair_get<8>(ss);
    float nrm = __builtin_sqrtf(ss);
    nrm = nrm > 1e-10f ? nrm : 1e-10f;

    // v / nrm, correctly rounded. From the correctly rounded reciprocal one
    // residual correction gives the rounded quotient (Markstein) as long as no
    // step leaves the normal range: nrm below 2^20 and every value zero or at
    // least 2^-100.
    bool plain = nrm < 0x1p20f;
    if constexpr (DT != PE_DTYPE_F16) {
      uint32_t least = 0xffffffffu;  // of the magnitudes, zero as the largest
#pragma unroll
      for (int i = 0; i < 8; ++i)
        least = min(least, (__builtin_bit_cast(uint32_t, v[i]) << 1) - 1u);
      plain = plain && least >= (27u << 24) - 1u;  // 2^-100: biased exponent 27
    }
    if (__all(plain)) {
      const float y = 1.f / nrm;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float q = v[i] * y;
        v[i] = __builtin_fmaf(__builtin_fmaf(-nrm, q, v[i]), y, q);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = v[i] / nrm;
    }

#pragma unroll
    for (int h = 1; h < 8; h <<= 1) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if ((i & h) == 0) {
          const float c = v[i], d = v[i + h];
          v[i] = c + d;
          v[i + h] = c - d;
        }
      }
    }
    float sg = 1.f;
    signed_stage<1>(v, sg, p & 1);
    signed_stage<2>(v, sg, p & 2);
    signed_stage<7>(v, sg, p & 4);
    signed_stage<8>(v, sg, p & 8);

    uint32_t c[8];
    if (inv_w != 0.f) {  // uniform
      const float scale = sg * inv_w;
      float t[8];
      uint2 e[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        t[i] = v[i] * scale;
        e[i] = cells.cell[cell_of(t[i])];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) c[i] = e[i].x + (t[i] > __builtin_bit_cast(float, e[i].y) ? 1u : 0u);
    } else {
      // first index of the nearest centroid, whatever their order
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float r = v[i] * sg;
        float best = __builtin_fabsf(r - cells.ct[0]);
        uint32_t bi = 0;
        for (int l = 1; l < n_levels; ++l) {
          const float d = __builtin_fabsf(r - cells.ct[l]);
          if (d < best) {
            best = d;
            bi = (uint32_t)l;
          }
        }
        c[i] = bi;
      }
    }
    const uint32_t lo = c[0] | (c[1] << 8) | (c[2] << 16) | (c[3] << 24);
    const uint32_t hi = c[4] | (c[5] << 8) | (c[6] << 16) | (c[7] << 24);
    if (live && l16 == 0) norms[it] = f2h_bits(nrm);
    if constexpr (!PACK) {
      if (live) *reinterpret_cast<uint2*>(codes + (int64_t)n * nb * kBlock + k0) = make_uint2(lo, hi);
    } else {
      // byte 64 b + i = code[128 b + 64 + i] << 4 | code[128 b + i]: lanes p < 8
      // hold positions 8p..8p+7 of the low half, lane xor 8 the same of the high
      const uint32_t olo = __builtin_bit_cast(uint32_t, pair_get<8>(__builtin_bit_cast(float, lo)));
      const uint32_t ohi = __builtin_bit_cast(uint32_t, pair_get<8>(__builtin_bit_cast(float, hi)));
      if (live && p < 8)
        *reinterpret_cast<uint2*>(codes + (int64_t)n * nb * 64 + b * 64 + 8 * p) =
            make_uint2(lo | (olo << 4), hi | (ohi << 4));
    }
  }
}

constexpr int kQuantWgsPerCu = 8;  // grid-stride beyond that: the cell table is built once a workgroup

template <int DT, bool PACK>
static int launch_quant(const void* w, int64_t ldw, int N, int K, int nb, const float* ct,
                        int n_levels, void* codes, uint16_t* norms, hipStream_t st) {
  const int64_t wgs = ((int64_t)N * nb + 15) / 16, cap = (int64_t)num_cus() * kQuantWgsPerCu;
  const unsigned grid = (unsigned)(wgs < cap ? wgs : cap);
  uint8_t* c = reinterpret_cast<uint8_t*>(codes);
  const int es = DT == PE_DTYPE_F32 ? 4 : 2;
  if (aligned16(w) && (ldw * es) % 16 == 0 && K % 8 == 0)
    quantize_kernel<DT, PACK, true><<<grid, 256, 0, st>>>(w, ldw, N, K, nb, ct, n_levels, c, norms);
  else
    quantize_kernel<DT, PACK, false><<<grid, 256, 0, st>>>(w, ldw, N, K, nb, ct, n_levels, c, norms);
  return launch_status();
}

template <int DT>
static int launch_quant(const void* w, int64_t ldw, int N, int K, int nb, const float* ct,
                        int n_levels, int pack, void* codes, uint16_t* norms, hipStream_t st) {
  return pack ? launch_quant<DT, true>(w, ldw, N, K, nb, ct, n_levels, codes, norms, st)
              : launch_quant<DT, false>(w, ldw, N, K, nb, ct, n_levels, codes, norms, st);
}

}  // namespace pe

extern "C" int pe_quantize(const void* w, int w_dtype, int64_t N, int K, int64_t ldw,
                           const float* ct, int n_levels, int pack, void* codes,
                           uint16_t* norms_f16, void* stream) {
  if (!w || !ct || !codes || !norms_f16) return PE_ERR_NULL;
  if (N < 0 || K <= 0 || ldw < K || N > INT32_MAX) return PE_ERR_DIMS;
  if (n_levels < 2 || n_levels > 256 || (pack && n_levels > 16) || (pack & ~1)) return PE_ERR_BITS;
  if (reinterpret_cast<uintptr_t>(codes) & 7) return PE_ERR_ALIGN;
  if (N == 0) return PE_OK;
  const int nb = (K + pe::kBlock - 1) / pe::kBlock;
  if ((int64_t)N * nb > ((int64_t)1 << 35)) return PE_ERR_DIMS;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  switch (w_dtype) {
    case PE_DTYPE_F16: return pe::launch_quant<PE_DTYPE_F16>(w, ldw, (int)N, K, nb, ct, n_levels, pack, codes, norms_f16, st);
    case PE_DTYPE_BF16: return pe::launch_quant<PE_DTYPE_BF16>(w, ldw, (int)N, K, nb, ct, n_levels, pack, codes, norms_f16, st);
    case PE_DTYPE_F32: return pe::launch_quant<PE_DTYPE_F32>(w, ldw, (int)N, K, nb, ct, n_levels, pack, codes, norms_f16, st);
    default: return PE_ERR_DTYPE;
  }
}
