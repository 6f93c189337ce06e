// Prefill GEMM for gfx950: Y[M, N] = X_tf[M, K] . W~[N, K]^T with
// W~[n, k] = ct[code[n, k]] * norm[n, k / 128], fp16 operands on MFMA
// (v_mfma_f32_32x32x16_f16), fp32 accumulate.
//
// Replaces polar_gemm / polar_gemm_packed (kernels/polar_gemm.py:81-171,
// 211-418), which gather ct per tile and run tl.dot on fp32 tiles.
//
// Structure (a workgroup of WM x WN waves, wave tile 32*TMW x 32*TNW; the
// dispatcher uses 1 x WN rows of waves, see pick_gemm_tile):
//  * K advances in half-blocks of 64 activations = 32 pairs; pair p of a
//    128-block is (x[p], x[p + 64]), the two positions one nibble byte codes;
//  * the activation tile (BM rows x 32 pairs, pair-f16) is staged global ->
//    registers -> LDS, double-buffered, rows padded to 144 B so the
//    ds_read_b128 of 8 consecutive rows hit distinct banks;
//  * the weight operand never touches LDS as data: every wave loads its own
//    codes (one dwordx4 per row per half-block for nibbles) one half-block
//    ahead, and dequantizes in registers through the per-lane LDS codebook
//    table (one v_perm + one ds_read_b32 per code byte) and a v_pk_mul_f16 by
//    the block norm;
//  * k-order inside an MFMA is the pair order: lane half h of slab t carries
//    pairs 16h + 4t + j, j = 0..3, as (lo, hi) halves, identically for A and B.
//  * workgroup ids are remapped so that each XCD (ids round-robin over 8)
//    walks a contiguous range of tiles (M-tile fastest) and shares A/B in its
//    own L2.

#include <type_traits>

#include "pe_internal.h"

namespace pe {

constexpr int kAStride = 144;  // bytes per A-tile row in LDS (128 + 16 pad)

// OM_F16: 16-bit output, bfloat16 when ybf (bias of the same type)
template <int OM>
__device__ __forceinline__ void store_out(void* y, int64_t ldy, int m, int n, float v,
                                          const uint16_t* bias, bool ybf) {
  if constexpr (OM == 0) {
    reinterpret_cast<float*>(y)[(int64_t)m * ldy + n] = v;
  } else {
    reinterpret_cast<uint16_t*>(y)[(int64_t)m * ldy + n] = out16(v, bias, n, ybf);
  }
}

// Dequantize one slab worth of B for one MFMA n-tile: 4 pair dwords.
template <bool NIB>
__device__ __forceinline__ half8v dequant_slab(const char* tbl, uint32_t wlo, uint32_t whi,
                                               uint32_t lane4, half2v nrm2) {
  uint32_t p[4];
  if constexpr (NIB) {
    p[0] = lds_ld32(tbl_addr<0>(wlo, lane4));
    p[1] = lds_ld32(tbl_addr<1>(wlo, lane4));
    p[2] = lds_ld32(tbl_addr<2>(wlo, lane4));
    p[3] = lds_ld32(tbl_addr<3>(wlo, lane4));
  } else {
    const uint32_t a0 = lds_ld32(tbl_addr<0>(wlo, lane4));
    const uint32_t a1 = lds_ld32(tbl_addr<1>(wlo, lane4));
    const uint32_t a2 = lds_ld32(tbl_addr<2>(wlo, lane4));
    const uint32_t a3 = lds_ld32(tbl_addr<3>(wlo, lane4));
    const uint32_t b0 = lds_ld32(tbl_addr<0>(whi, lane4));
    const uint32_t b1 = lds_ld32(tbl_addr<1>(whi, lane4));
    const uint32_t b2 = lds_ld32(tbl_addr<2>(whi, lane4));
    const uint32_t b3 = lds_ld32(tbl_addr<3>(whi, lane4));
    // (lo16 of a, lo16 of b): bytes a0,a1,b0,b1 -> selector 0x05040100 over {b, a}
    p[0] = __builtin_amdgcn_perm(b0, a0, 0x05040100u);
    p[1] = __builtin_amdgcn_perm(b1, a1, 0x05040100u);
    p[2] = __builtin_amdgcn_perm(b2, a2, 0x05040100u);
    p[3] = __builtin_amdgcn_perm(b3, a3, 0x05040100u);
  }
  half8v r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const half2v v = as_h2(p[j]) * nrm2;
    r[2 * j] = v[0];
    r[2 * j + 1] = v[1];
  }
  return r;
}

// B operand registers of one half-block K-tile for the wave's TNW n-tiles
template <bool NIB, int TNW>
struct BTile {
  u32x4v lo[TNW];
  u32x4v hi[TNW];  // int8 codes only: bytes at +64 (the pair's second position)
  uint16_t nrm[TNW];
};

template <bool NIB, int TNW>
__device__ __forceinline__ void load_btile(BTile<NIB, TNW>& t, const uint8_t* const (&b_row)[TNW],
                                           const uint16_t* const (&n_row)[TNW], int kt,
                                           int64_t c_blk, int64_t n_blk) {
  const int b = kt >> 1, half = kt & 1;
#pragma unroll
  for (int j = 0; j < TNW; ++j) {
    const uint8_t* pc = b_row[j] + b * c_blk + half * 32;
    t.lo[j] = ld_nt16v(pc);
    if constexpr (!NIB) t.hi[j] = ld_nt16v(pc + 64);
    t.nrm[j] = n_row[j][b * n_blk];
  }
}

template <int KA>
__device__ __forceinline__ void load_atile(u32x4v (&r)[KA], const uint32_t* const (&a_src)[KA],
                                           int kt) {
  const int off = (kt >> 1) * 64 + (kt & 1) * 32;
#pragma unroll
  for (int i = 0; i < KA; ++i) r[i] = *reinterpret_cast<const u32x4v*>(a_src[i] + off);
}

template <int KA>
__device__ __forceinline__ void store_atile(char* dst, const u32x4v (&r)[KA],
                                            const int (&a_dst)[KA]) {
#pragma unroll
  for (int i = 0; i < KA; ++i) *reinterpret_cast<u32x4v*>(dst + a_dst[i]) = r[i];
}

// One half-block K-tile of MFMA work on LDS A buffer `abase`.
template <bool NIB, int TMW, int TNW>
__device__ __forceinline__ void mma_ktile(float16v (&acc)[TMW][TNW], const BTile<NIB, TNW>& bt,
                                          const char* abase, const char* tbl, uint32_t lane4,
                                          uint32_t code_mask) {
  half2v nrm2[TNW];
#pragma unroll
  for (int j = 0; j < TNW; ++j) {
    const _Float16 nh = __builtin_bit_cast(_Float16, bt.nrm[j]);
    nrm2[j] = half2v{nh, nh};
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    half8v af[TMW];
#pragma unroll
    for (int i = 0; i < TMW; ++i)
      af[i] = __builtin_bit_cast(half8v, *reinterpret_cast<const u32x4v*>(abase + i * 32 * kAStride + 16 * t));
#pragma unroll
    for (int j = 0; j < TNW; ++j) {
      const uint32_t wl = bt.lo[j][t] & code_mask;
      uint32_t wh = 0;
      if constexpr (!NIB) wh = bt.hi[j][t] & code_mask;
      const half8v bf = dequant_slab<NIB>(tbl, wl, wh, lane4, nrm2[j]);
#pragma unroll
      for (int i = 0; i < TMW; ++i)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], bf, acc[i][j], 0, 0, 0);
    }
  }
}

// WM x WN waves, wave tile 32 TMW x 32 TNW.
template <bool NIB, int TMW, int TNW, int WM, int WN, int OM>
__global__ __launch_bounds__(WM * WN * 64) void gemm_kernel(
    const uint8_t* __restrict__ codes, const uint16_t* __restrict__ norms,
    const float* __restrict__ ct, int n_levels, uint32_t code_mask, int tbl_entries,
    const uint32_t* __restrict__ xp, void* __restrict__ y, const uint16_t* __restrict__ bias,
    int M, int N, int nb, int64_t ldy, int tiles_m, int tiles_total, WLayout lay, int ybf) {
  constexpr int NT = WM * WN * 64;
  constexpr int BM = WM * TMW * 32;
  constexpr int BN = WN * TNW * 32;
  constexpr int KA = BM * 8 / NT;  // uint4 of A per thread per half-block
  static_assert(KA * NT == BM * 8, "A tile must split evenly over the threads");
  extern __shared__ uint4 smem4[];
  char* smem = reinterpret_cast<char*>(smem4);
  char* tbl = smem;
  char* abuf = smem + tbl_entries * 256;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int h = lane >> 5, l32 = lane & 31;
  const uint32_t lane4 = (uint32_t)lane << 2;

  // XCD-aware tile order: ids are dealt round-robin to 8 XCDs; give each XCD a
  // contiguous range of logical tiles.
  int wid = blockIdx.x;
  if ((tiles_total & 7) == 0) wid = (wid & 7) * (tiles_total >> 3) + (wid >> 3);
  const int tm = wid % tiles_m, tn = wid / tiles_m;
  const int m0 = tm * BM, n0 = tn * BN;

  // codebook values now, the table once the first A and B loads are issued
  float cbr[4];
  codebook_regs(cbr, ct, n_levels);

  // K range of this workgroup: gridDim.z groups split the 128-blocks; with
  // more than one, each writes fp32 partial sums to its slab [M][ldy] of y
  // (one group: the whole K range, y itself)
  const int kb0 = (int)((int64_t)nb * blockIdx.z / gridDim.z);
  const int nbz = (int)((int64_t)nb * (blockIdx.z + 1) / gridDim.z) - kb0;
  y = reinterpret_cast<char*>(y) + (int64_t)blockIdx.z * M * ldy * (OM == 0 ? 4 : 2);

  // A loader: thread t moves uint4 q = t + NT i (row q >> 3, 16-byte col q & 7)
  const int64_t xrow_u32 = (int64_t)nb * 64;
  const uint32_t* a_src[KA];
  int a_dst[KA];
#pragma unroll
  for (int i = 0; i < KA; ++i) {
    const int q = tid + NT * i;
    const int r = q >> 3, c = q & 7;
    int m = m0 + r;
    if (m >= M) m = M - 1;  // clamped rows feed discarded outputs only
    a_src[i] = xp + (int64_t)m * xrow_u32 + (int64_t)kb0 * 64 + c * 4;
    a_dst[i] = r * kAStride + c * 16;
  }
  // B rows of this wave
  const uint8_t* b_row[TNW];
  const uint16_t* n_row[TNW];
#pragma unroll
  for (int j = 0; j < TNW; ++j) {
    int n = n0 + wn * TNW * 32 + j * 32 + l32;
    if (n >= N) n = N - 1;
    b_row[j] = codes + lay.codes_off(n) + 16 * h + (int64_t)kb0 * lay.c_blk;
    n_row[j] = norms + lay.norms_off(n) + (int64_t)kb0 * lay.n_blk;
  }

  float16v acc[TMW][TNW];
#pragma unroll
  for (int i = 0; i < TMW; ++i)
#pragma unroll
    for (int j = 0; j < TNW; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  const int nkt = 2 * nbz;  // half-block K-tiles of this K range (always even)
  const int a_off = (wm * TMW * 32 + l32) * kAStride + 64 * h;
  u32x4v ar[KA];
  BTile<NIB, TNW> b0, b1;

  // prologue: A(0) -> LDS 0, A(1) -> regs, B(0), B(1) -> regs
  load_atile<KA>(ar, a_src, 0);
  load_btile<NIB, TNW>(b0, b_row, n_row, 0, lay.c_blk, lay.n_blk);
  load_btile<NIB, TNW>(b1, b_row, n_row, 1, lay.c_blk, lay.n_blk);
  if constexpr (NIB) fill_codebook_from<TBL_NIB_H2>(0, cbr, tbl_entries, NT / 64);
  else fill_codebook_from<TBL_F16>(0, cbr, tbl_entries, NT / 64);
  store_atile<KA>(abuf, ar, a_dst);
  load_atile<KA>(ar, a_src, 1);
  __syncthreads();

  for (int kt = 0; kt < nkt; kt += 2) {
    // ---- even half-block: B from b0, A from LDS buffer 0
    {
      const BTile<NIB, TNW> cur = b0;
      if (kt + 2 < nkt) load_btile<NIB, TNW>(b0, b_row, n_row, kt + 2, lay.c_blk, lay.n_blk);
      mma_ktile<NIB, TMW, TNW>(acc, cur, abuf + a_off, tbl, lane4, code_mask);
      store_atile<KA>(abuf + BM * kAStride, ar, a_dst);  // A(kt+1) -> LDS 1
      if (kt + 2 < nkt) load_atile<KA>(ar, a_src, kt + 2);
      __syncthreads();
    }
    // ---- odd half-block: B from b1, A from LDS buffer 1
    {
      const BTile<NIB, TNW> cur = b1;
      if (kt + 3 < nkt) load_btile<NIB, TNW>(b1, b_row, n_row, kt + 3, lay.c_blk, lay.n_blk);
      mma_ktile<NIB, TMW, TNW>(acc, cur, abuf + BM * kAStride + a_off, tbl, lane4, code_mask);
      if (kt + 2 < nkt) {
        store_atile<KA>(abuf, ar, a_dst);  // A(kt+2) -> LDS 0
        load_atile<KA>(ar, a_src, kt + 3);
      }
      __syncthreads();
    }
  }

  // ---- epilogue: acc[i][j][e] -> row 8*(e/4) + 4*h + e%4, col l32
#pragma unroll
  for (int i = 0; i < TMW; ++i) {
#pragma unroll
    for (int j = 0; j < TNW; ++j) {
      const int n = n0 + wn * TNW * 32 + j * 32 + l32;
      if (n >= N) continue;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + wm * TMW * 32 + i * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
        if (m < M) store_out<OM>(y, ldy, m, n, acc[i][j][e], bias, ybf != 0);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Four-wave variant: one wave per SIMD, each wave owning BM = 32 TMW rows x
// 32 NTW columns (NTW 32-column n-tiles: 2 or 3), workgroup tile BM x 128 NTW.
// Per MFMA it moves (TMW + NTW) / (NTW TMW) KB of operands through LDS instead
// of (TMW + 1) / TMW, and every weight column is still dequantized by exactly
// one wave; NTW = 3 (384 columns) cuts the LDS reads, A-tile stores and
// barriers per MFMA by a further quarter to a third where its tiles fill the
// CUs in as few rounds.
//  * A half-block tiles sit in a ring of six LDS buffers (96 KB beside the
//    64 KB table), stored four half-blocks ahead, with one barrier per two
//    half-blocks: the tile of half-block kt + 1 is complete before the barrier
//    that precedes kt, so the first slab of kt + 1 is read ahead while kt
//    still computes.
//  * Within a half-block every slab's operands (A fragments and codebook
//    lookups) are issued one slab ahead of its MFMAs.
//  * Codes ride a ring of four half-block slots (issued three half-blocks
//    ahead), activations a ring of two register stages (loaded six ahead,
//    stored four ahead); the loop
//    body covers four half-blocks so every ring index is static. Loads past the
//    end are clamped to the last half-block, so each wait count is static too.
// An odd 128-block count ends in half a loop body.
// ---------------------------------------------------------------------------
// Codes of one half-block for the wave's NTW n-tiles. Norms are kept
// zero-extended to 32 bits: 16-bit members next to vectors made the compiler
// keep the slot in memory.
template <bool NIB, int NTW>
struct BSlot4 {
  u32x4v lo[NTW];
  u32x4v hi[NIB ? 1 : NTW];  // int8 codes only: bytes at +64
  uint32_t nrm[NTW];
};

template <bool NIB, int TMW, int NTW>
struct Frag4 {
  half8v a[TMW];
  uint32_t raw[NTW][NIB ? 4 : 8];
};

// A tiles of the four-wave kernel: 128-byte rows (32 pairs), 16-byte chunk c
// of row r stored at chunk c ^ ((r >> 1) & 7). A ds_read_b128 phase serves 16
// lanes (rows r0..r0+15, one chunk each) from the 64 four-byte banks: a row
// spans half the banks (even rows the low half, odd rows the high half), so
// the eight rows of each parity need eight distinct chunks. The plain
// c ^ (r & 7) repeats after eight rows and made every A read a 2-way conflict.
constexpr int kARow4 = 128;
// A half-block tiles in the four-wave kernel's LDS ring (16 KB each at 128
// rows): A(kt + 4) is stored while A(kt) is read, one barrier per two tiles
constexpr int kA4Ring = 6;
__device__ __forceinline__ uint32_t a4_swz(int r) { return (uint32_t)((r >> 1) & 7); }

// ACT <= TMW: the m-tiles that hold live rows (the others' A fragments are
// not read and their MFMAs not issued; their accumulators stay zero)
template <bool NIB, int TMW, int NTW, bool MASK, int ACT = TMW>
__device__ __forceinline__ void issue_frag4(Frag4<NIB, TMW, NTW>& f, uint32_t aaddr, int t,
                                            const BSlot4<NIB, NTW>& bt, uint32_t lane4,
                                            uint32_t code_mask) {
  // aaddr: this lane's row and swizzled chunk of slab t in m-tile 0
#pragma unroll
  for (int i = 0; i < ACT; ++i)
    f.a[i] = __builtin_bit_cast(half8v, lds_ld128(aaddr + i * 32 * kARow4));
#pragma unroll
  for (int j = 0; j < NTW; ++j) {
    uint32_t wl = bt.lo[j][t];
    if constexpr (MASK) wl &= code_mask;
    f.raw[j][0] = lds_ld32(tbl_addr<0>(wl, lane4));
    f.raw[j][1] = lds_ld32(tbl_addr<1>(wl, lane4));
    f.raw[j][2] = lds_ld32(tbl_addr<2>(wl, lane4));
    f.raw[j][3] = lds_ld32(tbl_addr<3>(wl, lane4));
    if constexpr (!NIB) {
      uint32_t wh = bt.hi[j][t];
      if constexpr (MASK) wh &= code_mask;
      f.raw[j][4] = lds_ld32(tbl_addr<0>(wh, lane4));
      f.raw[j][5] = lds_ld32(tbl_addr<1>(wh, lane4));
      f.raw[j][6] = lds_ld32(tbl_addr<2>(wh, lane4));
      f.raw[j][7] = lds_ld32(tbl_addr<3>(wh, lane4));
    }
  }
}

template <bool NIB, int TMW, int NTW, int ACT = TMW>
__device__ __forceinline__ void mma_frag4(float16v (&acc)[TMW][NTW], const Frag4<NIB, TMW, NTW>& f,
                                          const BSlot4<NIB, NTW>& bt) {
#pragma unroll
  for (int j = 0; j < NTW; ++j) {
    const _Float16 nh = __builtin_bit_cast(_Float16, (uint16_t)bt.nrm[j]);
    const half2v nrm2{nh, nh};
    half8v bf;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t p = f.raw[j][q];
      // int8: (lo16 of the first-position entry, lo16 of the second)
      if constexpr (!NIB) p = __builtin_amdgcn_perm(f.raw[j][4 + q], p, 0x05040100u);
      const half2v v = as_h2(p) * nrm2;
      bf[2 * q] = v[0];
      bf[2 * q + 1] = v[1];
    }
    // weights as the MFMA's A operand: the accumulator comes out transposed,
    // lane = output row, four consecutive output columns per register group
#pragma unroll
    for (int i = 0; i < ACT; ++i)
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bf, f.a[i], acc[i][j], 0, 0, 0);
  }
}

// Output tile through LDS: the transposed accumulators (lane = row m, groups
// of four consecutive columns) are written as 8- or 16-byte pieces into a
// row-major staging tile, then copied to y in 16-byte coalesced stores.
template <int TMW, int NTW, int OM>
__device__ __forceinline__ void store_tile4(const float16v (&acc)[TMW][NTW], void* __restrict__ y,
                                            int64_t ldy, const uint16_t* __restrict__ bias, int M,
                                            int N, int m0, int n0, int vec_ok, bool ybf) {
  constexpr int BM = TMW * 32, BN = 128 * NTW;
  constexpr int ES = OM == OM_F16 ? 2 : 4;
  constexpr uint32_t OSTR = BN * ES + 16;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int h = lane >> 5, l32 = lane & 31;
  __syncthreads();  // every wave is done with the ring and the table
#pragma unroll
  for (int i = 0; i < TMW; ++i)
#pragma unroll
    for (int j = 0; j < NTW; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const uint32_t addr = (uint32_t)(32 * i + l32) * OSTR +
                              (uint32_t)(wave * 32 * NTW + 32 * j + 8 * g + 4 * h) * ES;
        // element values first: a bit_cast applied to a vector element
        // lvalue reads element 0 of the vector with this compiler
        const float v0 = acc[i][j][4 * g], v1 = acc[i][j][4 * g + 1];
        const float v2 = acc[i][j][4 * g + 2], v3 = acc[i][j][4 * g + 3];
        if constexpr (OM == OM_F16) {
          lds_st64(addr, u32x2v{pack16x2(v0, v1, ybf), pack16x2(v2, v3, ybf)});
        } else {
          lds_st128(addr, u32x4v{__builtin_bit_cast(uint32_t, v0), __builtin_bit_cast(uint32_t, v1),
                                 __builtin_bit_cast(uint32_t, v2), __builtin_bit_cast(uint32_t, v3)});
        }
      }
  __syncthreads();
  // bias of the two columns n, n + 1 (zero past N) onto a rounded pair
  auto with_bias = [&](uint32_t w, int n) -> uint32_t {
    const float b0 = n < N ? f16or_bf(bias[n], ybf) : 0.f, b1 = n + 1 < N ? f16or_bf(bias[n + 1], ybf) : 0.f;
    return pack16x2(f16or_bf((uint16_t)(w & 0xffff), ybf) + b0, f16or_bf((uint16_t)(w >> 16), ybf) + b1, ybf);
  };
  if (!vec_ok) {
    // rows that do not start on 16 bytes (a column count that is no multiple
    // of 8): consecutive lanes store consecutive dwords, or halves of them
    // where rows start on odd halves (eight 2-byte stores of one 16-byte chunk
    // per lane touched every line eight times: 10003 columns at M = 2996, 2048
    // deep, 201 -> 181 us for the 128 x 256 tiles)
    constexpr int DPR = BN * ES / 4;  // dwords per row
    const bool dw = OM != OM_F16 || ((ldy & 1) == 0 && ((uintptr_t)y & 3) == 0);
    for (int q = tid; q < BM * DPR; q += 256) {
      const int r = q / DPR, c = q % DPR;
      const int m = m0 + r, n = n0 + c * (4 / ES);
      if (m >= M || n >= N) continue;
      uint32_t v = lds_ld32((uint32_t)r * OSTR + (uint32_t)c * 4u);
      char* dst = reinterpret_cast<char*>(y) + ((int64_t)m * ldy + n) * ES;
      if constexpr (OM == OM_F16) {
        if (bias) v = with_bias(v, n);
        if (dw && n + 1 < N) {
          *reinterpret_cast<uint32_t*>(dst) = v;
        } else {
          reinterpret_cast<uint16_t*>(dst)[0] = (uint16_t)v;
          if (n + 1 < N) reinterpret_cast<uint16_t*>(dst)[1] = (uint16_t)(v >> 16);
        }
      } else {
        *reinterpret_cast<uint32_t*>(dst) = v;
      }
    }
    return;
  }
  constexpr int CPR = BN * ES / 16;  // 16-byte chunks per row
  constexpr int EPC = 16 / ES;       // elements per chunk
  for (int q = tid; q < BM * CPR; q += 256) {
    const int r = q / CPR, c = q % CPR;
    const int m = m0 + r, n = n0 + c * EPC;
    if (m >= M || n >= N) continue;
    u32x4v v = lds_ld128((uint32_t)r * OSTR + (uint32_t)c * 16u);
    if constexpr (OM == OM_F16) {
      if (bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = with_bias(v[e], n + 2 * e);
      }
    }
    char* dst = reinterpret_cast<char*>(y) + ((int64_t)m * ldy + n) * ES;
    if (n + EPC <= N) {
      *reinterpret_cast<u32x4v*>(dst) = v;
    } else {
      const int cnt = N - n < EPC ? N - n : EPC;
      for (int e = 0; e < cnt; ++e) {
        if constexpr (OM == OM_F16)
          reinterpret_cast<uint16_t*>(dst)[e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
        else
          reinterpret_cast<uint32_t*>(dst)[e] = v[e];
      }
    }
  }
}

// Grouped form (experts): the row tiles of all groups, in group order, are
// numbered consecutively; tile t of the grid belongs to the group whose tiles
// cover t. A wave finds it from the group offsets with a prefix sum over the
// lanes (64 groups per step). False past the last tile.
template <int BM>
__device__ __forceinline__ bool group_tile(const GemmGroup& g, int t, int lane, int& e_out,
                                           int& mt_out) {
  int base = 0;
  for (int q = 0; q * 64 < g.groups; ++q) {  // uniform
    const int e = q * 64 + lane;
    const int cnt = e < g.groups ? g.offsets[e + 1] - g.offsets[e] : 0;
    const int tiles = (cnt + BM - 1) / BM;
    int incl = tiles;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(incl, d, 64);
      if (lane >= d) incl += v;
    }
    const int first = base + incl - tiles;
    const unsigned long long hit = __ballot(tiles > 0 && t >= first && t < first + tiles);
    if (hit) {
      const int l = __ffsll((long long)hit) - 1;
      e_out = __builtin_amdgcn_readfirstlane(q * 64 + l);
      mt_out = __builtin_amdgcn_readfirstlane(t - __shfl(first, l, 64));
      return true;
    }
    base += __shfl(incl, 63, 64);
  }
  return false;
}

// SwiGLU epilogue of the grouped four-wave kernel: h = silu(gate) * up for
// the tile's 128 columns (one 128-block of h) into an fp16 LDS tile [BM][128],
// then each row through the FWHT-128 (16 lanes per row) into pair-f16 x_tf
// layout at y + (row0 + m) * (ldy / 2) u32, block n0 / 128. Columns >= I are
// zero.
template <int TMW>
__device__ __forceinline__ void swiglu_xtf_tile4(const float16v (&acc)[TMW][2], uint32_t* __restrict__ y,
                                                 int64_t ldy, int M, int I, int64_t row0, int m0, int n0) {
  constexpr int BM = TMW * 32;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int h = lane >> 5, l32 = lane & 31;
  __syncthreads();  // every wave is done with the ring and the table
#pragma unroll
  for (int i = 0; i < TMW; ++i)
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
      const int col = wave * 32 + 8 * gq + 4 * h;  // four consecutive columns
      float hv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float s = acc[i][0][4 * gq + e], u = acc[i][1][4 * gq + e];
        hv[e] = n0 + col + e < I ? s / (1.f + __expf(-s)) * u : 0.f;
      }
      const uint32_t addr = (uint32_t)(32 * i + l32) * 256u + (uint32_t)col * 2u;
      lds_st64(addr, u32x2v{pack16x2(hv[0], hv[1], false), pack16x2(hv[2], hv[3], false)});
    }
  __syncthreads();
  const int q = tid & 15;  // 16 groups of 16 lanes: rows tid / 16 + 16 k
#pragma unroll
  for (int k = 0; k < BM / 16; ++k) {
    const int r = (tid >> 4) + 16 * k;
    float v[8];
    {
      const u32x4v w = lds_ld128((uint32_t)r * 256u + (uint32_t)q * 16u);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        v[2 * c] = h2f((uint16_t)(w[c] & 0xffff));
        v[2 * c + 1] = h2f((uint16_t)(w[c] >> 16));
      }
    }
    fwht128_group16(v, q);
    const int m = m0 + r;
    const bool live = m < M;
    const int64_t prow = live ? row0 + m : row0;  // no address past the expert's rows
    store_pair_block(v, q, y + prow * (ldy / 2) + (int64_t)(n0 / 128) * 64, live);
  }
}

// GRP 0: one matrix. GRP 1 / 2 (grouped experts, GemmGroup g): blockIdx.x is
// a row tile of some expert (group_tile), blockIdx.y the column tile; the
// activation rows are gathered (g.a_rows) and the expert's codes and norms
// start at codes / norms + e * stride. GRP 1 writes fp32 rows of y at the
// expert's pair rows; GRP 2 (SwiGLU, NTW = 2) takes gate rows n and up rows
// I + n for the same 128 columns n of h, and writes silu(gate) * up through
// the FWHT-128 as pair-f16 rows (the next product's activations).
template <bool NIB, int TMW, int NTW, bool MASK, int OM, int GRP>
__global__ __launch_bounds__(256) void gemm4_kernel(
    const uint8_t* __restrict__ codes, const uint16_t* __restrict__ norms,
    const float* __restrict__ ct, int n_levels, uint32_t code_mask, int tbl_entries,
    const uint32_t* __restrict__ xp, void* __restrict__ y, const uint16_t* __restrict__ bias,
    int M, int N, int nb, int64_t ldy, int tiles_m, int tiles_total, WLayout lay, int vec_ok,
    int ybf, GemmGroup g) {
  constexpr int NT = 256;
  constexpr int BM = TMW * 32;
  constexpr int BN = 128 * NTW;
  constexpr int KA = BM * 8 / NT;
  constexpr uint32_t ABUF = BM * kARow4;
  static_assert(KA * NT == BM * 8, "A tile must split evenly over the threads");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int h = lane >> 5, l32 = lane & 31;
  const uint32_t lane4 = (uint32_t)lane << 2;

  static_assert(GRP != 2 || NTW == 2, "SwiGLU tiles: one gate and one up n-tile per wave");
  static_assert(GRP == 0 || TMW > 2, "grouped tiles: 1, 2 or TMW live m-tiles");
  int m0, n0;
  int64_t row0 = 0;  // grouped: the expert's first pair row
  if constexpr (GRP == 0) {
    // XCD-aware tile order: ids are dealt round-robin to 8 XCDs; give each
    // XCD a contiguous range of logical tiles (M-tile fastest).
    int wid = blockIdx.x;
    if ((tiles_total & 7) == 0) wid = (wid & 7) * (tiles_total >> 3) + (wid >> 3);
    const int tm = wid % tiles_m, tn = wid / tiles_m;
    m0 = tm * BM;
    n0 = tn * BN;
  } else {
    int e, mt;
    if (!group_tile<BM>(g, blockIdx.x, lane, e, mt)) return;  // uniform
    row0 = g.offsets[e];
    M = g.offsets[e + 1] - (int)row0;  // this expert's rows
    m0 = mt * BM;
    n0 = blockIdx.y * (GRP == 2 ? 128 : BN);
    codes += (int64_t)e * g.codes_stride;
    norms += (int64_t)e * g.norms_stride;
  }

  // codebook values now, the table once the first A and B loads are issued
  // (the values' round trip overlaps theirs)
  float cbr[4];
  codebook_regs(cbr, ct, n_levels);
  const uint32_t abuf = (uint32_t)tbl_entries * 256u;

  // K range of this workgroup, in pairs of 128-blocks (the loop takes four
  // half-blocks per step; the last group also takes an odd last block):
  // gridDim.z groups; with more than one, fp32 partial sums go to slab
  // blockIdx.z [M][ldy] of y
  const int kb0 = GRP ? 0 : 2 * (int)((int64_t)(nb / 2) * blockIdx.z / gridDim.z);
  const int nbz = GRP || blockIdx.z + 1 == gridDim.z
                      ? nb - kb0
                      : 2 * (int)((int64_t)(nb / 2) * (blockIdx.z + 1) / gridDim.z) - kb0;
  if constexpr (GRP == 0) y = reinterpret_cast<char*>(y) + (int64_t)blockIdx.z * M * ldy * (OM == OM_F16 ? 2 : 4);

  // Loads through buffer resources based at this workgroup's first row of x
  // and first column of the weights: per-lane offsets in VGPRs, the K
  // position in the scalar offset (no 64-bit address arithmetic in the K
  // loop). Every extent is below 2 GiB (host check).
  const int64_t xrow_u32 = (int64_t)nb * 64;
  const int mlast = (m0 + BM <= M ? m0 + BM : M) - 1;
  // grouped: the whole activation matrix (rows gathered per lane)
  const __amdgpu_buffer_rsrc_t ra =
      GRP ? __builtin_amdgcn_make_buffer_rsrc((void*)xp, (short)0, (int)(g.a_total_rows * xrow_u32 * 4), 0x00020000)
          : __builtin_amdgcn_make_buffer_rsrc((void*)(xp + (int64_t)m0 * xrow_u32), (short)0,
                                              (int)((mlast - m0 + 1) * xrow_u32 * 4), 0x00020000);
  uint32_t a_voff[KA];
  uint32_t a_dst[KA];
#pragma unroll
  for (int i = 0; i < KA; ++i) {
    const int q = tid + NT * i;
    const int r = q >> 3, c = q & 7;
    int m = m0 + r;
    if (m >= M) m = M - 1;  // clamped rows feed discarded outputs only
    if constexpr (GRP) {
      const int64_t pr = row0 + m;  // pair row
      const int64_t src = g.a_rows ? (int64_t)g.a_rows[pr] : pr;
      a_voff[i] = (uint32_t)((src * xrow_u32 + c * 4) * 4);
    } else {
      a_voff[i] = (uint32_t)(((int64_t)(m - m0) * xrow_u32 + c * 4) * 4);
    }
    a_dst[i] = (uint32_t)(r * kARow4 + (((uint32_t)c ^ a4_swz(r)) << 4));
  }
  // grouped: resources over the expert's whole codes and norms
  const int nlast = (n0 + BN <= N ? n0 + BN : N) - 1;
  const int64_t cb0 = GRP ? 0 : lay.codes_off(n0), nb0 = GRP ? 0 : lay.norms_off(n0);
  const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(codes + cb0), (short)0,
      GRP ? (int)g.codes_stride
          : (int)(lay.codes_off(nlast) + (int64_t)(nb - 1) * lay.c_blk + (NIB ? 64 : 128) - cb0), 0x00020000);
  const __amdgpu_buffer_rsrc_t rn = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(norms + nb0), (short)0,
      GRP ? (int)(g.norms_stride * 2)
          : (int)((lay.norms_off(nlast) + (int64_t)(nb - 1) * lay.n_blk + 1 - nb0) * 2),
      0x00020000);
  uint32_t b_voff[NTW], n_voff[NTW];
#pragma unroll
  for (int j = 0; j < NTW; ++j) {
    int n;
    if constexpr (GRP == 2) {
      // gate row (j = 0) or up row (j = 1) of column c of h
      int c = n0 + wave * 32 + l32;
      if (c >= g.I) c = g.I - 1;
      n = j == 0 ? c : g.I + c;
    } else {
      n = n0 + wave * 32 * NTW + j * 32 + l32;
      if (n >= N) n = N - 1;
    }
    b_voff[j] = (uint32_t)(lay.codes_off(n) - cb0) + 16 * h;
    n_voff[j] = (uint32_t)((lay.norms_off(n) - nb0) * 2);
  }
  uint32_t a_off[4];  // lane's row l32, chunk 4h + t, swizzled
#pragma unroll
  for (int t = 0; t < 4; ++t) a_off[t] = (uint32_t)(l32 * kARow4 + (((uint32_t)(4 * h + t) ^ a4_swz(l32)) << 4));

  const int nkt = 2 * nbz;  // half-blocks of this K range
  // loads past the last half-block re-read it (in bounds, never used)
  auto ldb = [&](BSlot4<NIB, NTW>& sl, int kt) {
    kt = kt < nkt ? kt : nkt - 1;
    const int bk = kb0 + (kt >> 1), half = kt & 1;
    const int sc = bk * (int)lay.c_blk + half * 32, sn = bk * (int)lay.n_blk * 2;
#pragma unroll
    for (int j = 0; j < NTW; ++j) {
      sl.lo[j] = __builtin_bit_cast(u32x4v, __builtin_amdgcn_raw_buffer_load_b128(rc, b_voff[j], sc, 0));
      if constexpr (!NIB)
        sl.hi[j] = __builtin_bit_cast(u32x4v, __builtin_amdgcn_raw_buffer_load_b128(rc, b_voff[j], sc + 64, 0));
      sl.nrm[j] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(rn, n_voff[j], sn, 0);
    }
  };
  auto lda = [&](u32x4v (&rg)[KA], int kt) {
    kt = kt < nkt ? kt : nkt - 1;
    const int sa = (kb0 * 64 + (kt >> 1) * 64 + (kt & 1) * 32) * 4;
#pragma unroll
    for (int i = 0; i < KA; ++i)
      rg[i] = __builtin_bit_cast(u32x4v, __builtin_amdgcn_raw_buffer_load_b128(ra, a_voff[i], sa, 0));
  };
  auto sta = [&](uint32_t buf, const u32x4v (&rg)[KA]) {
#pragma unroll
    for (int i = 0; i < KA; ++i) lds_st128(buf + a_dst[i], rg[i]);
  };

  float16v acc[TMW][NTW];
#pragma unroll
  for (int i = 0; i < TMW; ++i)
#pragma unroll
    for (int j = 0; j < NTW; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  BSlot4<NIB, NTW> slot[4];
  u32x4v stg[2][KA], pre[2][KA];  // pre: prologue only
  lda(stg[0], 0);
  lda(stg[1], 1);
  lda(pre[0], 2);
  lda(pre[1], 3);
  ldb(slot[0], 0);
  ldb(slot[1], 1);
  ldb(slot[2], 2);
  if constexpr (NIB) fill_codebook_from<TBL_NIB_H2>(0, cbr, tbl_entries, NT / 64);
  else fill_codebook_from<TBL_F16>(0, cbr, tbl_entries, NT / 64);
  __syncthreads();  // codebook table written
  sta(abuf, stg[0]);
  sta(abuf + ABUF, stg[1]);
  sta(abuf + 2 * ABUF, pre[0]);
  sta(abuf + 3 * ABUF, pre[1]);
  lda(stg[0], 4);
  lda(stg[1], 5);
  __syncthreads();

  auto ring_next = [](uint32_t b) { return b == (kA4Ring - 1) * ABUF ? 0u : b + ABUF; };
  // the K loop, computing the first ACT m-tiles
  auto k_loop = [&](auto ACT_) {
    constexpr int ACT = decltype(ACT_)::value;
    Frag4<NIB, TMW, NTW> f;
    issue_frag4<NIB, TMW, NTW, MASK, ACT>(f, abuf + a_off[0], 0, slot[0], lane4, code_mask);
    uint32_t bcur = 0;  // ring offset (bytes) of half-block kt's A buffer

    auto half_step = [&](auto S_, int kt) {
      constexpr int S = decltype(S_)::value;
      const uint32_t bnext = ring_next(bcur);
      const uint32_t bst = ring_next(ring_next(ring_next(bnext)));  // where A(kt - 2) was
      ldb(slot[(S + 3) & 3], kt + 3);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        Frag4<NIB, TMW, NTW> fn;
        // this slab's operands (issued one slab ago) are in: wait for them
        // before the next slab's reads go out
        __builtin_amdgcn_s_waitcnt(0xc07f);
        if (t < 3)
          issue_frag4<NIB, TMW, NTW, MASK, ACT>(fn, abuf + bcur + a_off[t + 1], t + 1, slot[S], lane4, code_mask);
        else
          issue_frag4<NIB, TMW, NTW, MASK, ACT>(fn, abuf + bnext + a_off[0], 0, slot[(S + 1) & 3], lane4, code_mask);
        // keep the next slab's reads ahead of this slab's MFMAs
        __builtin_amdgcn_sched_barrier(0);
        mma_frag4<NIB, TMW, NTW, ACT>(acc, f, slot[S]);
        f = fn;
      }
      sta(abuf + bst, stg[S & 1]);  // A(kt + 4)
      lda(stg[S & 1], kt + 6);
      bcur = bnext;
      // one barrier per 128-block: between two of them the waves read A(kt),
      // A(kt + 1) and the first slab of A(kt + 2) while A(kt + 4), A(kt + 5)
      // go into the buffers of A(kt - 2), A(kt - 1), read before the last one
      if constexpr (S & 1) __syncthreads();
    };
    int kt = 0;
    for (; kt + 4 <= nkt; kt += 4) {
      half_step(std::integral_constant<int, 0>{}, kt);
      half_step(std::integral_constant<int, 1>{}, kt + 1);
      half_step(std::integral_constant<int, 2>{}, kt + 2);
      half_step(std::integral_constant<int, 3>{}, kt + 3);
    }
    if (kt < nkt) {  // an odd block count: its last block
      half_step(std::integral_constant<int, 0>{}, kt);
      half_step(std::integral_constant<int, 1>{}, kt + 1);
    }
  };
  if constexpr (GRP != 0) {
    // an expert's last row tile often holds a few rows: compute only the
    // m-tiles that hold live rows (uniform: M and m0 are per workgroup)
    const int live = M - m0;
    if (live <= 32) k_loop(std::integral_constant<int, 1>{});
    else if (live <= 64) k_loop(std::integral_constant<int, 2>{});
    else k_loop(std::integral_constant<int, TMW>{});
  } else {
    k_loop(std::integral_constant<int, TMW>{});
  }

  if constexpr (GRP == 2) {
    swiglu_xtf_tile4<TMW>(acc, reinterpret_cast<uint32_t*>(y), ldy, M, g.I, row0, m0, n0);
  } else if constexpr (GRP == 1) {
    store_tile4<TMW, NTW, OM>(acc, reinterpret_cast<char*>(y) + row0 * ldy * (OM == OM_F16 ? 2 : 4), ldy,
                              bias, M, N, m0, n0, vec_ok, ybf != 0);
  } else {
    store_tile4<TMW, NTW, OM>(acc, y, ldy, bias, M, N, m0, n0, vec_ok, ybf != 0);
  }
}

// LDS of the four-wave kernel (16-bit or fp32 rows out)
template <int ES>
static size_t gemm4_lds(int entries, int tmw, int ntw) {
  const size_t bm = 32 * (size_t)tmw, bn = 128 * (size_t)ntw;
  const size_t loop = (size_t)entries * 256 + kA4Ring * bm * kARow4, out = bm * (bn * ES + 16);
  return loop > out ? loop : out;
}

template <bool NIB, int TMW, int NTW, bool MASK, int OM>
static int launch_gemm4_t(const GemmArgs& a, hipStream_t st, int ksplit = 1) {
  constexpr int BM = TMW * 32, BN = 128 * NTW;
  auto kern = gemm4_kernel<NIB, TMW, NTW, MASK, OM, 0>;
  const int entries = table_entries(NIB, a.n_levels);
  constexpr int ES = OM == OM_F16 ? 2 : 4;
  const size_t lds = gemm4_lds<ES>(entries, TMW, NTW);
  if (lds > 160 * 1024) return PE_ERR_DIMS;
  static const bool attr_ok = [&] {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                               hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) == hipSuccess;
  }();
  (void)attr_ok;
  const int tiles_m = (a.M + BM - 1) / BM;
  const int tiles_n = (a.N + BN - 1) / BN;
  const int64_t total = (int64_t)tiles_m * tiles_n;
  if (total > INT32_MAX) return PE_ERR_DIMS;
  // one workgroup's rows of x and columns of codes and norms are addressed by
  // 32-bit buffer offsets
  const int64_t w_span = a.lay.codes_off(BN - 1) + (int64_t)a.nb * a.lay.c_blk + 128;
  if ((int64_t)BM * a.nb * 256 >= ((int64_t)1 << 31) || w_span >= ((int64_t)1 << 31)) return PE_ERR_DIMS;
  const uint8_t mb = NIB ? (uint8_t)((a.n_levels - 1) * 0x11) : (uint8_t)(a.n_levels - 1);
  // 16-byte stores need aligned rows; with a K split, aligned slab starts too
  const int vec_ok = ((uintptr_t)a.y % 16 == 0) && ((a.ldy * (int64_t)ES) % 16 == 0) &&
                     (ksplit == 1 || ((int64_t)a.M * a.ldy * (int64_t)ES) % 16 == 0);
  kern<<<dim3((unsigned)total, 1, (unsigned)ksplit), dim3(256), lds, st>>>(
      a.codes, a.norms, a.ct, a.n_levels, 0x01010101u * mb, entries,
      reinterpret_cast<const uint32_t*>(a.xp), a.y, a.bias, a.M, a.N, a.nb, a.ldy, tiles_m,
      (int)total, a.lay, vec_ok, a.ybf, GemmGroup{});
  return launch_status();
}

// Grouped expert products on the four-wave kernel, 128 x 256 tiles: GRP 1
// (SE_F32 / SE_F16) fp32 or 16-bit rows y[pair][N]; GRP 2 (SE_SWIGLU_XTF) the
// transformed silu(gate) * up as pair-f16 rows of I / 128 blocks.
template <bool NIB, bool MASK, int GRP, int OMX = OM_F32>
static int launch_moe_gemm4_t(const MoeGemmArgs& a, hipStream_t st) {
  constexpr int TMW = 4, NTW = 2, BM = TMW * 32, BN = 128 * NTW;
  constexpr int OM = GRP == 1 ? OMX : OM_F16;
  auto kern = gemm4_kernel<NIB, TMW, NTW, MASK, OM, GRP>;
  const int entries = table_entries(NIB, a.n_levels);
  const size_t lds_loop = (size_t)entries * 256 + kA4Ring * (size_t)BM * kARow4;
  const size_t lds_out = GRP == 1 ? (size_t)BM * (BN * 4 + 16) : (size_t)BM * 256;
  const size_t lds = lds_loop > lds_out ? lds_loop : lds_out;
  if (lds > 160 * 1024) return PE_ERR_DIMS;
  static const bool attr_ok = [&] {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                               hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) == hipSuccess;
  }();
  (void)attr_ok;
  // at least the sum over the groups of ceil(rows / BM); the surplus
  // workgroups find no tile and leave
  const int64_t tiles_m = a.g.groups + (a.P + BM - 1) / BM;
  const int64_t tiles_n = GRP == 2 ? a.g.I / 128 : (a.N + BN - 1) / BN;
  if (tiles_m > INT32_MAX || tiles_n > 65535 || tiles_n < 1) return PE_ERR_DIMS;
  const uint8_t mb = NIB ? (uint8_t)((a.n_levels - 1) * 0x11) : (uint8_t)(a.n_levels - 1);
  const int vec_ok = GRP == 1 && (uintptr_t)a.y % 16 == 0 && (a.ldy * (OM == OM_F16 ? 2 : 4)) % 16 == 0;
  kern<<<dim3((unsigned)tiles_m, (unsigned)tiles_n), dim3(256), lds, st>>>(
      a.codes, a.norms, a.ct, a.n_levels, 0x01010101u * mb, entries,
      reinterpret_cast<const uint32_t*>(a.xp), a.y, nullptr, 0, a.N, a.nb, a.ldy, 0, 0, a.lay, vec_ok,
      GRP == 1 && OM == OM_F16 ? a.ybf : 0, a.g);
  return launch_status();
}

bool moe_gemm4_fits(const MoeGemmArgs& a, int epilogue) {
  const int64_t lim = (int64_t)1 << 31;
  if (epilogue == SE_SWIGLU_XTF && (a.g.I <= 0 || a.g.I % 128 || a.ldy % 128)) return false;
  return a.nb >= 1 && a.g.groups >= 1 && a.g.codes_stride < lim && a.g.norms_stride * 2 < lim &&
         a.g.a_total_rows * a.nb * 256 < lim && a.P < lim;
}

int moe_gemm4(bool nibble, int epilogue, const MoeGemmArgs& a, hipStream_t st) {
  if (!a.g.offsets || !moe_gemm4_fits(a, epilogue)) return PE_ERR_DIMS;
  const bool mask = nibble ? a.n_levels != 16 : a.n_levels != 256;
  if (epilogue == SE_F32) {
    if (nibble) return mask ? launch_moe_gemm4_t<true, true, 1>(a, st) : launch_moe_gemm4_t<true, false, 1>(a, st);
    return mask ? launch_moe_gemm4_t<false, true, 1>(a, st) : launch_moe_gemm4_t<false, false, 1>(a, st);
  }
  if (epilogue == SE_F16) {
    if (nibble)
      return mask ? launch_moe_gemm4_t<true, true, 1, OM_F16>(a, st) : launch_moe_gemm4_t<true, false, 1, OM_F16>(a, st);
    return mask ? launch_moe_gemm4_t<false, true, 1, OM_F16>(a, st) : launch_moe_gemm4_t<false, false, 1, OM_F16>(a, st);
  }
  if (epilogue == SE_SWIGLU_XTF) {
    if (nibble) return mask ? launch_moe_gemm4_t<true, true, 2>(a, st) : launch_moe_gemm4_t<true, false, 2>(a, st);
    return mask ? launch_moe_gemm4_t<false, true, 2>(a, st) : launch_moe_gemm4_t<false, false, 2>(a, st);
  }
  return PE_ERR_DTYPE;
}

template <bool NIB, int TMW, int TNW, int WM, int WN, int OM>
static int launch_gemm_t(const GemmArgs& a, hipStream_t st, int ksplit = 1) {
  constexpr int BM = WM * TMW * 32, BN = WN * TNW * 32;
  auto kern = gemm_kernel<NIB, TMW, TNW, WM, WN, OM>;
  const int entries = table_entries(NIB, a.n_levels);
  const size_t lds = (size_t)entries * 256 + 2 * (size_t)BM * kAStride;
  if (lds > 160 * 1024) return PE_ERR_DIMS;
  static const bool attr_ok = [&] {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                               hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) == hipSuccess;
  }();
  (void)attr_ok;
  const int tiles_m = (a.M + BM - 1) / BM;
  const int tiles_n = (a.N + BN - 1) / BN;
  const int64_t total = (int64_t)tiles_m * tiles_n;
  if (total > INT32_MAX) return PE_ERR_DIMS;
  const uint8_t mb = NIB ? (uint8_t)((a.n_levels - 1) * 0x11) : (uint8_t)(a.n_levels - 1);
  kern<<<dim3((unsigned)total, 1, (unsigned)ksplit), dim3(WM * WN * 64), lds, st>>>(
      a.codes, a.norms, a.ct, a.n_levels, 0x01010101u * mb, entries,
      reinterpret_cast<const uint32_t*>(a.xp), a.y, a.bias, a.M, a.N, a.nb, a.ldy, tiles_m,
      (int)total, a.lay, a.ybf);
  return launch_status();
}

// Tile shape. Waves sit in one row (1 x WN), each owning 32 TMW rows x 32
// columns, so every weight column is dequantized by exactly one wave and two
// waves share a SIMD (8 waves). A workgroup's time grows with its tile area
// and tiles run in rounds of one workgroup per CU: the cost of a shape is
// rounds x area x a penalty for short tiles (the dequantization is amortised
// over BM rows; measured ~13% per halving of BM) or for 4-wave workgroups
// (one wave per SIMD hides no latency).
struct GemmShape {
  int tmw, wn;
};
static GemmShape pick_gemm_tile(int M, int N) {
  const int cus = num_cus();
  const GemmShape cand[] = {{8, 8}, {4, 8}, {2, 8}, {8, 4}, {4, 4}, {2, 4}};
  GemmShape best = cand[0];
  double best_cost = -1;
  for (const GemmShape& c : cand) {
    const int bm = 32 * c.tmw, bn = 32 * c.wn;
    if (c.tmw > 2 && M <= bm / 2) continue;  // no tile more than twice as tall as needed
    const int64_t tiles = (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
    const int64_t rounds = (tiles + cus - 1) / cus;
    const double pen = (c.tmw == 8 ? 1.0 : c.tmw == 4 ? 1.13 : 1.3) * (c.wn == 8 ? 1.0 : 1.25);
    const double cost = (double)rounds * bm * bn * pen;
    if (best_cost < 0 || cost < best_cost * 0.999) {
      best_cost = cost;
      best = c;
    }
  }
  return best;
}

// ---------------------------------------------------------------------------
// Which kernel, tile and K split one product takes: the cheapest by a cost
// model in microseconds. Its constants are fitted to 135,000 timings of every
// form on 10,677 shapes (M 33..8192, N 256..24576, 3..112 128-blocks, 2..8 bits,
// spread over their logarithms, odd sizes and layer shapes among them), each
// as the mean of a repeated call and of calls whose weights come from HBM (HIP
// graphs; 500 of the shapes: profiles/gemm_form_timings.txt). Over those
// shapes the choice is 1.1% above the fastest form on average, and 1.5% of them
// are more than 5% slower than by thresholds on tile counts tuned on layer
// shapes (which were 29% slower on average). A model fitted to repeated calls
// alone, without the terms for ragged rows, weight reads and co-resident fixed
// parts, was 2.5% above the fastest, with 4.2% of the shapes behind the
// thresholds and some by 1.4 times.
//  * tiles on the busiest CU, each a fixed part (table fill, ring fill,
//    epilogue; more where rows do not start on 16 bytes and are stored by
//    dwords) and a cost per 128-block of its form, more with every CU busy
//    (clock, memory), less where the last round is partly empty;
//  * two co-resident workgroups (64-row tiles whose LDS fits twice) overlap most
//    of their fixed parts and some of their loops;
//  * every row of tiles reads the weight once: its bytes;
//  * K split: a smaller epilogue, the partial sums' bytes and the reduction's
//    launch.
// ---------------------------------------------------------------------------
struct TileCost {
  double block, fixed;  // us per 128-block and per tile
  double pair_fixed, pair_loop;  // two tiles of a CU, in units of one
  double ragged, busy;
};

// us of one product as tiles of bm x bn in z K groups of at most nbz blocks
static double tiles_cost(const TileCost& t, int cus, int M, int N, int bm, int bn, int z, int nbz,
                         int entries, int row_bytes) {
  const double rows = (M + bm - 1) / bm, wgs = rows * ((N + bn - 1) / bn) * z;
  const int64_t per = (int64_t)((wgs + cus - 1) / cus);
  const double area = bm * bn / 32768.0, odd = (double)(per & 1);
  const double fixed = t.fixed + 0.0063 * entries + (t.ragged - (z > 1 ? 4.1 : 0.0)) * area;
  const double loop = nbz * t.block * (1.0 + t.busy * (wgs < cus ? wgs / cus : 1.0));
  const double last = per > 1 ? 0.3 * ((double)per - wgs / cus) : 0.0;
  return ((double)(per / 2) * t.pair_fixed + odd) * fixed +
         ((double)(per / 2) * t.pair_loop + odd - last) * loop + rows * N * (double)row_bytes / 56e6 +
         (z > 1 ? 3.46 + (double)z * M * N * 8 / 5.6e6 : 0.0);
}

// partial_limit: most bytes of partial sums; cost: of the choice
static MmPlan gemm_plan(bool nibble, int n_levels, int om, int M, int N, int nb,
                        size_t partial_limit, double* cost) {
  struct Form {
    int tmw, ntw;
    double block_nib, fixed_nib, block_int8, fixed_int8;
  };
  static const Form forms[] = {{4, 3, 1.91, 8.9, 0.0, 0.0},     {4, 2, 1.31, 6.55, 1.74, 7.15},
                               {4, 1, 0.782, 3.95, 0.985, 4.2}, {2, 3, 1.06, 3.25, 0.0, 0.0},
                               {2, 2, 0.769, 3.82, 1.12, 4.75}, {2, 1, 0.488, 1.68, 0.663, 2.2}};
  // the eight-wave kernel's tiles: 32 tmw rows x 32 ntw columns
  static const Form eight[] = {{8, 8, 2.58, 9.4, 3.5, 10.9},  {4, 8, 1.46, 4.85, 2.66, 4.7},
                               {2, 8, 1.01, 1.25, 2.57, -2.4}, {8, 4, 1.98, 8.3, 2.39, 10.4},
                               {4, 4, 1.155, 6.05, 1.72, 3.6}, {2, 4, 0.983, 0.05, 1.43, 2.7}};
  static const int splits[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24};
  const int cus = num_cus();
  const int64_t max_wgs = 5 * (int64_t)cus / 2;  // of a K split
  const int entries = table_entries(nibble, n_levels), row_bytes = nb * (nibble ? 64 : 128);
  auto tiles = [&](int bm, int bn) { return (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  auto split_ok = [&](int z, int64_t t) {
    return om == OM_F16 && z <= nb / 2 && t * z <= max_wgs && (size_t)z * M * N * 4 <= partial_limit;
  };
  *cost = 0;
  // the four-wave kernel addresses its rows of x by 31-bit offsets
  if (nb >= 65536) return MmPlan{0, 0, 1};
  MmPlan best{4, 2, 1};
  *cost = -1;
  auto offer = [&](const MmPlan& p, double c) {
    if (*cost < 0 || c < *cost) {
      *cost = c;
      best = p;
    }
  };
  for (const Form& f : forms) {
    // 384 columns: nibble codes with 16-bit output only (the int8 variant
    // spills, fp32 rows do not fit the output staging)
    if (f.ntw == 3 && (!nibble || om != OM_F16)) continue;
    const int bm = 32 * f.tmw, bn = 128 * f.ntw;
    const bool twice = f.tmw == 2 && f.ntw < 3 && 2 * gemm4_lds<2>(entries, f.tmw, f.ntw) <= 160 * 1024;
    TileCost t{nibble ? f.block_nib : f.block_int8, nibble ? f.fixed_nib : f.fixed_int8,
               twice ? 1.24 : 2.0, twice ? 1.74 : 2.0, 0.0, nibble ? 0.384 : 0.30};
    for (int z : splits) {
      if (z > 1 && (f.ntw == 3 || !split_ok(z, tiles(bm, bn)))) break;
      // fp32 rows (output or partial sums), 16-bit rows
      t.ragged = z > 1 || om != OM_F16 ? (N % 4 ? 7.1 : 0.0) : N % 8 ? (f.ntw == 3 ? 6.2 : 4.7) : 0.0;
      const int nbz = z > 1 ? 2 * ((nb / 2 + (nb & 1) + z - 1) / z) : nb;
      offer(MmPlan{f.tmw, f.ntw, z}, tiles_cost(t, cus, M, N, bm, bn, z, nbz, entries, row_bytes));
    }
  }
  if (nb <= 40) {  // the eight-wave kernel: a small fixed part, but slower per block
    const GemmShape g = pick_gemm_tile(M, N);
    const int bm = 32 * g.tmw, bn = 32 * g.wn;
    const bool twice = g.tmw < 8 && 2 * (entries * 256 + 2 * bm * kAStride) <= 160 * 1024;
    for (const Form& f : eight) {
      if (f.tmw != g.tmw || f.ntw != g.wn) continue;
      TileCost t{nibble ? f.block_nib : f.block_int8, nibble ? f.fixed_nib : f.fixed_int8, 2.0,
                 twice ? 1.56 : 2.0, 0.0, 0.48};
      for (int z : splits) {
        if (z > 1 && (M > 128 || !split_ok(z, tiles(bm, bn)))) break;
        t.ragged = z == 1 && N % 8 ? 0.5 : 0.0;
        offer(MmPlan{0, 0, z},
              tiles_cost(t, cus, M, N, bm, bn, z, (nb + z - 1) / z, entries, row_bytes));
      }
    }
  }
  return best;
}

template <bool NIB, int OM>
static int launch_gemm_eight(const GemmArgs& a, hipStream_t st, int ksplit) {
  const GemmShape g = pick_gemm_tile(a.M, a.N);
  switch (g.tmw * 16 + g.wn) {
    case 8 * 16 + 8: return launch_gemm_t<NIB, 8, 1, 1, 8, OM>(a, st, ksplit);
    case 4 * 16 + 8: return launch_gemm_t<NIB, 4, 1, 1, 8, OM>(a, st, ksplit);
    case 2 * 16 + 8: return launch_gemm_t<NIB, 2, 1, 1, 8, OM>(a, st, ksplit);
    case 8 * 16 + 4: return launch_gemm_t<NIB, 8, 1, 1, 4, OM>(a, st, ksplit);
    case 4 * 16 + 4: return launch_gemm_t<NIB, 4, 1, 1, 4, OM>(a, st, ksplit);
    default: return launch_gemm_t<NIB, 2, 1, 1, 4, OM>(a, st, ksplit);
  }
}

// the four-wave kernel with the code mask its codebook size needs
template <bool NIB, int TMW, int NTW, int OM>
static int launch_gemm4_m(const GemmArgs& a, hipStream_t st, int ksplit = 1) {
  const bool mask = NIB ? a.n_levels != 16 : a.n_levels != 256;
  return mask ? launch_gemm4_t<NIB, TMW, NTW, true, OM>(a, st, ksplit)
              : launch_gemm4_t<NIB, TMW, NTW, false, OM>(a, st, ksplit);
}

// OM: the product's output; a K split runs in fp32 and is reduced to 16 bits
template <bool NIB, int OM>
static int launch_gemm4_form(const GemmArgs& a, hipStream_t st, const MmPlan& p) {
  if constexpr (NIB && OM == OM_F16) {
    if (p.ntw == 3)
      return p.tmw == 4 ? launch_gemm4_m<NIB, 4, 3, OM>(a, st, p.z) : launch_gemm4_m<NIB, 2, 3, OM>(a, st, p.z);
  }
  if (p.tmw == 4)
    return p.ntw == 2 ? launch_gemm4_m<NIB, 4, 2, OM>(a, st, p.z) : launch_gemm4_m<NIB, 4, 1, OM>(a, st, p.z);
  return p.ntw == 2 ? launch_gemm4_m<NIB, 2, 2, OM>(a, st, p.z) : launch_gemm4_m<NIB, 2, 1, OM>(a, st, p.z);
}

template <bool NIB, int OM>
static int launch_gemm_shape(const MmPlan& p, const GemmArgs& a, hipStream_t st, void* ws, size_t ws_bytes) {
  if (p.z == 1)
    return p.tmw ? launch_gemm4_form<NIB, OM>(a, st, p) : launch_gemm_eight<NIB, OM>(a, st, 1);
  if (!ws || !aligned16(ws) || ws_bytes < mm_partials(p, a.M, a.N)) return PE_ERR_WORKSPACE;
  GemmArgs g = a;
  g.y = ws;
  g.ldy = a.N;
  g.bias = nullptr;
  if (int rc = p.tmw ? launch_gemm4_form<NIB, OM_F32>(g, st, p) : launch_gemm_eight<NIB, OM_F32>(g, st, p.z))
    return rc;
  return split_reduce(reinterpret_cast<const float*>(ws), p.z, a.M, a.N, a.bias, a.y, a.ldy, st,
                      a.ybf != 0);
}

// Matmul on a pair-f16 x_tf, used by the linear entry points for M > 1. The
// small-M kernel up to 32 rows, and up to 64 for fp32 output or where K and N
// are short (over 745 shapes of up to 4096 columns it takes 0.88 of the fastest
// GEMM form's time up to 7 blocks, 1.05 at 8 and 9, 1.2 at 10 to 13; past 4096
// columns the GEMM is 1.9 to 2.8 times faster).
static bool mm_small(int64_t M, int N, int nb, int out_mode) {
  if (M <= 32) return true;
  if (M > kSmallMaxRows) return false;
  return out_mode != OM_F16 || (nb <= 9 && N <= 4096);
}

MmPlan mm_plan(bool nibble, int n_levels, int64_t M, int N, int nb, int out_mode) {
  if (M > INT32_MAX || mm_small(M, N, nb, out_mode)) return MmPlan{0, 0, 0};
  double cost = 0, cost_fit = 0;
  const MmPlan best = gemm_plan(nibble, n_levels, out_mode, (int)M, N, nb, SIZE_MAX, &cost);
  // Partial sums that fit the allocation-free entry point's scratch beside x_tf,
  // where the model puts them within 5% (that call then runs in one part; over
  // 66 timed shapes the two took the same time on average, 0.89 to 1.11).
  const size_t fixed = kWsCounterBytes + (size_t)M * nb * (kBlock * 2) + 512;  // 512: rounding
  if (fixed >= kScratchBytes || fixed + mm_partials(best, M, N) <= kScratchBytes) return best;
  const MmPlan fit = gemm_plan(nibble, n_levels, out_mode, (int)M, N, nb, kScratchBytes - fixed, &cost_fit);
  return cost_fit <= 1.05 * cost ? fit : best;
}

void mm_form(const MmPlan& p, int64_t M, int N, int form[4]) {
  form[0] = form[1] = form[2] = 0;
  form[3] = 1;
  if (!p.z) return;
  const GemmShape g = pick_gemm_tile((int)M, N);
  form[0] = p.tmw ? 2 : 1;
  form[1] = 32 * (p.tmw ? p.tmw : g.tmw);
  form[2] = p.tmw ? 128 * p.ntw : 32 * g.wn;
  form[3] = p.z;
}

int mm_xtf(const MmPlan& plan, bool nibble, bool tiled, const void* codes, const uint16_t* norms,
           const float* ct, int n_levels, const void* x_pair, int64_t M, int N, int nb, void* y,
           int out_mode, int64_t ldy, const uint16_t* bias, void* ws, size_t ws_bytes,
           hipStream_t st, bool ybf) {
  if (M > INT32_MAX) return PE_ERR_DIMS;
  const WLayout lay = wlayout(nibble, tiled, nb);
  if (!plan.z) {
    SmallArgs s{reinterpret_cast<const uint8_t*>(codes), norms, ct, n_levels,
                reinterpret_cast<const uint32_t*>(x_pair), nullptr, nullptr, 0, 0, y, ldy, bias,
                (int)M, N, nb, lay, ybf ? 1 : 0};
    return gemm_small(nibble, out_mode == OM_F32 ? SE_F32 : SE_F16, s, st);
  }
  GemmArgs a{reinterpret_cast<const uint8_t*>(codes), norms, ct, n_levels, x_pair, y, bias,
             (int)M, N, nb, ldy, lay, ybf ? 1 : 0};
  if (nibble)
    return out_mode == OM_F32 ? launch_gemm_shape<true, OM_F32>(plan, a, st, ws, ws_bytes)
                              : launch_gemm_shape<true, OM_F16>(plan, a, st, ws, ws_bytes);
  return out_mode == OM_F32 ? launch_gemm_shape<false, OM_F32>(plan, a, st, ws, ws_bytes)
                            : launch_gemm_shape<false, OM_F16>(plan, a, st, ws, ws_bytes);
}

}  // namespace pe
