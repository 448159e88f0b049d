// mmq_planes.hip -- the prompt MMQ of the super-block formats from a weight's
// plane image and an activation image (int8 MFMA, exact integers); all of them
// but Q4_K, whose prompts read its fragment image.
//
// Plane image.  Every value of a super-block format enters its block integer
// as p = scale * value, an integer (Q6_K int8 scale x [-32, 31],
// kernels256.c:200-212, :720-738; Q5_K 6 bits x 5 bits, :605-629; IQ4_XS 6
// signed bits x codebook, iq_kernels.c:967-1001; IQ3_XXS / IQ3_S odd scale x
// signed grid value, :612-643, :1728-1772; Q3_K 6 signed bits x [-4, 3],
// kernels256.c:349-369; Q2_K 4 bits x 2 bits, :232-257).  The
// image holds p as one int8 plane where it fits (Q2_K at most 45; Q3_K as -p
// in [-128, 124] with -d), else split exactly as p = 64 hi + lo (lo = p & 63,
// hi = p >> 6: |p| < 2^13).  Per 32-row group and super-block: each plane's 8
// KB (the 16 values 16 v ..+15 of row i at 512 v + 16 i), the 32 rows' f32
// scales d; formats with mins add the rows' f32 dmin and the mins of the
// 16-value groups as f16 (row 16 h + i, groups 4 k ..+3 at 512 h + 8 (i + 16
// k)).
//
// Activation image (k_quantize_mmq_act): the Q8_K quantization of x, bit for
// bit, in the order this kernel copies it: per 32-token group and super-block
// the quants (8 KB, as above with tokens for rows), the 16-value sums as f16
// (exact: at most 2032; 1 KB, as the mins), the tokens' f32 scales -- 9344
// bytes, the Q8_K size.  A workgroup's copy into LDS is then whole aligned 1 KB
// pieces, and the 16-byte pieces of an MFMA fragment are runs of 256 contiguous
// bytes, in memory and in LDS (conflict free).
#include "qhip_device.hpp"
#include "qhip_internal.hpp"

#include "../../include/qwen35_hip.h"

namespace qhip {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

// planes and mins of a format; image bytes per 32-row group and super-block
constexpr int pl_planes(int tt) { return tt == TT_Q3_K || tt == TT_Q2_K ? 1 : 2; }
constexpr bool pl_mins(int tt) { return tt == TT_Q5_K || tt == TT_Q2_K; }
constexpr int pl_grp(int planes, bool mins) { return 8192 * planes + 128 + (mins ? 128 + 1024 : 0); }
constexpr int kActGrp = 9344;       // activation image bytes per 32-token group and super-block
constexpr int kActSums = 8192, kActScale = 9216;

// ---- the activation image ----------------------------------------------------------------
// One workgroup per 32-token group and super-block; wave w quantizes tokens 4
// w ..+3, one super-block per wave and step (lane l: values 4 l ..+3, as the
// Q8_K quantizer), into an LDS copy of the group, which leaves in 16-byte
// pieces.  LDS piece rows are 528 bytes apart (512 + 16), so a wave's 64 dword
// writes fall in 64 banks.  Tokens past the end are zeros.
template <bool ALIGNED>
__global__ __launch_bounds__(512) void k_quantize_mmq_act(const float* __restrict__ x, uint8_t* __restrict__ out,
                                                           int cols, int nsb, int tokens) {
  constexpr int kRow = 528, kSums = 16 * kRow;
  __shared__ __attribute__((aligned(16))) uint8_t sm[kSums + 1024 + 128];
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int sb = blockIdx.x, tg = blockIdx.y;
  float v[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = 32 * tg + 4 * wv + i;
    const float* p = x + (long)(t < tokens ? t : 0) * cols + 256 * sb + 4 * l;
    if constexpr (ALIGNED) {
      const f32x4 f = *(const f32x4*)p;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[i][j] = f[j];
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[i][j] = p[j];
    }
    if (t >= tokens)
#pragma unroll
      for (int j = 0; j < 4; ++j) v[i][j] = 0.0f;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int tl = 4 * wv + i, g = l >> 2;
    int gsum;
    float scale;
    const uint32_t packed = quant_q8_K_lane(v[i], gsum, scale);
    *(uint32_t*)(sm + kRow * g + 16 * tl + 4 * (l & 3)) = packed;
    if ((l & 3) == 0) *(_Float16*)(sm + kSums + 512 * (tl >> 4) + 8 * ((tl & 15) + 16 * (g >> 2)) + 2 * (g & 3)) = (_Float16)(float)gsum;
    if (l == 0) *(float*)(sm + kSums + 1024 + 4 * tl) = scale;
  }
  __syncthreads();
  uint8_t* o = out + ((long)tg * nsb + sb) * kActGrp;
  for (int j = threadIdx.x; j < kActGrp / 16; j += 512)
    *(uint4*)(o + 16 * j) = *(const uint4*)(sm + (j < 512 ? kRow * (j >> 5) + 16 * (j & 31) : kSums + 16 * (j - 512)));
}

long planes_act_bytes(int cols, int tokens) { return (long)((tokens + 31) / 32) * (cols / 256) * kActGrp; }

hipError_t launch_quantize_mmq_act(const float* x, void* out, int cols, int tokens, hipStream_t s) {
  if (tokens <= 0) return hipSuccess;
  const long ntg = (tokens + 31) / 32;
  if (cols <= 0 || cols % 256 || ntg > 65535 || ((uintptr_t)out & 15u)) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(cols / 256), (unsigned)ntg);
  if (((uintptr_t)x & 15u) == 0)
    hipLaunchKernelGGL(k_quantize_mmq_act<true>, grid, dim3(512), 0, s, x, (uint8_t*)out, cols, cols / 256, tokens);
  else
    hipLaunchKernelGGL(k_quantize_mmq_act<false>, grid, dim3(512), 0, s, x, (uint8_t*)out, cols, cols / 256, tokens);
  return hipGetLastError();
}

// ---- the plane image ---------------------------------------------------------------------
bool planes_format(int ttype) {
  switch (ttype) {
    case TT_Q6_K: case TT_Q5_K: case TT_Q3_K: case TT_Q2_K: case TT_IQ4_XS: case TT_IQ3_XXS: case TT_IQ3_S:
      return true;
    default: return false;
  }
}

long planes_image_bytes(int ttype, int rows, int cols) {
  if (!planes_format(ttype) || rows < 0 || cols <= 0 || cols % 256) return -1;
  return (long)((rows + 31) / 32) * (cols / 256) * pl_grp(pl_planes(ttype), pl_mins(ttype));
}

__device__ __forceinline__ uint32_t pl_ld16(const uint8_t* p) { return (uint32_t)p[0] | ((uint32_t)p[1] << 8); }

// 6-bit scale and min j of the 12 packed bytes (kernels256.c:105-125)
__device__ __forceinline__ void pl_k_scale(const uint8_t* s12, int j, int& sc, int& mn) {
  if (j < 4) {
    sc = s12[j] & 63;
    mn = s12[j + 4] & 63;
  } else {
    sc = (s12[j + 4] & 15) | ((s12[j - 4] >> 6) << 4);
    mn = (s12[j + 4] >> 4) | ((s12[j] >> 6) << 4);
  }
}

// The integer scale of values 16 g ..+15 (g = e0 / 16) of a super-block, its
// f32 d, and value e of it.
template <int TT>
__device__ __forceinline__ int pl_scale(const uint8_t* blk, int e0) {
  const int s = e0 >> 5, g = e0 >> 4;
  int sc = 0, mn;
  if constexpr (TT == TT_Q6_K) sc = (int)(int8_t)blk[192 + g];
  else if constexpr (TT == TT_Q5_K) pl_k_scale(blk + 4, s, sc, mn);
  else if constexpr (TT == TT_IQ4_XS)
    sc = (int)(((blk[4 + s / 2] >> (4 * (s % 2))) & 15u) | (((pl_ld16(blk + 2) >> (2 * s)) & 3u) << 4)) - 32;
  else if constexpr (TT == TT_IQ3_XXS) sc = 2 * (int)(pl_ld16(blk + 68 + 4 * s) >> 12) + 1;
  else if constexpr (TT == TT_IQ3_S) sc = 2 * (int)((blk[106 + s / 2] >> (4 * (s % 2))) & 15u) + 1;
  else if constexpr (TT == TT_Q3_K)
    sc = (int)(((blk[96 + (g & 7)] >> (4 * (g >> 3))) & 15u) | (((blk[104 + (g & 3)] >> (2 * (g >> 2))) & 3u) << 4)) - 32;
  else sc = (int)(blk[g] & 15u);  // Q2_K
  return sc;
}
template <int TT>
__device__ __forceinline__ float pl_d(const uint8_t* blk) {
  if constexpr (TT == TT_Q6_K) return h2f(pl_ld16(blk + 208));
  else if constexpr (TT == TT_Q3_K) return -h2f(pl_ld16(blk + 108));  // the image holds -p
  else if constexpr (TT == TT_Q2_K) return h2f(pl_ld16(blk + 80));
  else if constexpr (TT == TT_IQ3_XXS) return h2f(pl_ld16(blk)) * 0.25f;
  else return h2f(pl_ld16(blk));
}
template <int TT>
__device__ __forceinline__ int pl_value(const uint8_t* blk, int e) {
  const int s = e >> 5, l = e & 31, h = e >> 7, q = s & 3;
  if constexpr (TT == TT_Q6_K) {
    uint32_t lq = blk[64 * h + 32 * (q & 1) + l];
    lq = q >= 2 ? (lq >> 4) : (lq & 15u);
    return (int)(lq | (((blk[128 + 32 * h + l] >> (2 * q)) & 3u) << 4)) - 32;
  } else if constexpr (TT == TT_Q5_K) {
    const uint32_t b = blk[48 + 32 * (s >> 1) + l];
    return (int)((s & 1) ? (b >> 4) : (b & 15u)) | ((int)((blk[16 + l] >> s) & 1u) << 4);
  } else if constexpr (TT == TT_IQ4_XS) {
    const uint32_t b = blk[8 + 16 * s + (l & 15)];
    const uint32_t nib = l < 16 ? (b & 15u) : (b >> 4);
    const uint32_t tab = nib < 4 ? IQ4_T0 : nib < 8 ? IQ4_T1 : nib < 12 ? IQ4_T2 : IQ4_T3;
    return sext8(tab >> (8 * (nib & 3)));
  } else if constexpr (iq3(TT)) {
    const int k = l >> 2;  // grid entry k of the sub-block, its signs' half
    uint32_t ent, s8;
    if constexpr (TT == TT_IQ3_XXS) {
      const uint32_t aux = pl_ld16(blk + 66 + 4 * s) | (pl_ld16(blk + 68 + 4 * s) << 16);
      ent = kIq3xxsGrid[blk[2 + 8 * s + k]];
      s8 = iq_sign8((aux >> (7 * (k >> 1))) & 127u);
    } else {
      ent = kIq3sGrid[blk[2 + 8 * s + k] | (((blk[66 + s] >> k) & 1u) << 8)];
      s8 = blk[74 + 4 * s + (k >> 1)];
    }
    const int v = (int)((ent >> (8 * (l & 3))) & 255u);
    return (s8 >> (4 * (k & 1) + (l & 3))) & 1u ? -v : v;
  } else if constexpr (TT == TT_Q3_K) {
    // minus the value: q2 - 4 unless its hmask bit is set
    return (((blk[l] >> s) & 1u) ? 0 : 4) - (int)((blk[32 + 32 * h + l] >> (2 * q)) & 3u);
  } else {
    return (int)((blk[16 + 32 * h + l] >> (2 * q)) & 3u);
  }
}

// One thread per (32-row group, super-block, sub-block s, lane L): the 16
// values 32 s + 16 (L / 32) .. +15 of row 32 group + L % 32 in every plane,
// and for s = 0 the row's scales and mins.  Rows past the end: zeros.
template <int TT>
__global__ __launch_bounds__(256) void k_planes_prepare(const uint8_t* __restrict__ W, uint8_t* __restrict__ IMG,
                                                         int rows, long row_bytes, int nsb, long nthreads) {
  constexpr bool MINS = pl_mins(TT);
  constexpr int PL = pl_planes(TT);
  const long gid = (long)blockIdx.x * 256 + threadIdx.x;
  if (gid >= nthreads) return;
  const int Lq = (int)(gid & 63), s = (int)((gid >> 6) & 7);
  const long gs = gid >> 9;  // group * nsb + sb
  const long grp = gs / nsb;
  const int sb = (int)(gs - grp * nsb);
  const long row = grp * 32 + (Lq & 31);
  const int e0 = 32 * s + 16 * (Lq >> 5);
  uint32_t hi[4] = {0, 0, 0, 0}, lo[4] = {0, 0, 0, 0};
  float d = 0.0f, dmin = 0.0f;
  f16x4 mins[2] = {};
  if (row < rows) {
    const uint8_t* blk = W + row * row_bytes + (row_bytes / nsb) * sb;
    const int sc = pl_scale<TT>(blk, e0);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int pv = sc * pl_value<TT>(blk, e0 + i);
      if constexpr (PL == 1) {
        hi[i >> 2] |= ((uint32_t)pv & 255u) << (8 * (i & 3));
      } else {
        hi[i >> 2] |= ((uint32_t)(pv >> 6) & 255u) << (8 * (i & 3));  // arithmetic shift: floor
        lo[i >> 2] |= (uint32_t)(pv & 63) << (8 * (i & 3));
      }
    }
    d = pl_d<TT>(blk);
    if constexpr (MINS) {
      dmin = h2f(pl_ld16(blk + (TT == TT_Q2_K ? 82 : 2)));
      if (s == 0)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int g = 8 * (Lq >> 5) + k;  // groups 8 (L / 32) ..+7 of the row
          int c, m;
          if constexpr (TT == TT_Q2_K) m = blk[g] >> 4;
          else pl_k_scale(blk + 4, g >> 1, c, m);
          mins[k >> 2][k & 3] = (_Float16)(float)m;
        }
    }
  }
  uint8_t* b = IMG + gs * pl_grp(PL, MINS);
  *(uint4*)(b + 1024 * s + 16 * Lq) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
  if constexpr (PL == 2) *(uint4*)(b + 8192 + 1024 * s + 16 * Lq) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
  if (s == 0) {
    if (Lq < 32) *(float*)(b + 8192 * PL + 4 * Lq) = d;
    if constexpr (MINS) {
      if (Lq < 32) *(float*)(b + 8192 * PL + 128 + 4 * Lq) = dmin;
#pragma unroll
      for (int k = 0; k < 2; ++k)
        *(f16x4*)(b + 8192 * PL + 256 + 512 * ((Lq >> 4) & 1) + 8 * ((Lq & 15) + 16 * (2 * (Lq >> 5) + k))) = mins[k];
    }
  }
}

hipError_t launch_planes_prepare(int ttype, const void* w, long row_bytes, int rows, int cols, void* img,
                                 hipStream_t s) {
  if (planes_image_bytes(ttype, rows, cols) < 0) return hipErrorInvalidValue;
  const long n = (long)((rows + 31) / 32) * (cols / 256) * 512;
  if (n == 0) return hipSuccess;
  const dim3 grid((unsigned)((n + 255) / 256));
  return dispatch_type(ttype, [&](auto tt) {
    constexpr int TT = decltype(tt)::value;
    if constexpr (act32(TT) || TT == TT_Q4_K) return hipErrorInvalidValue;
    else {
      hipLaunchKernelGGL(k_planes_prepare<TT>, grid, dim3(256), 0, s, (const uint8_t*)w, (uint8_t*)img, rows, row_bytes,
                         cols / 256, n);
      return hipGetLastError();
    }
  });
}

// ---- the product -------------------------------------------------------------------------
// Tiles of 32 NW rows x TK = 32 NA tokens: 128 x 64 (four waves, two workgroups
// per CU) or 256 x 128 (eight waves, one per CU; planes_plan).  Wave w takes row
// group w and all TK tokens, 16 at a time.  A super-block's 16
// plane fragments stay in registers; each activation fragment read from LDS
// (16 tokens x 64 values) feeds four v_mfma_i32_16x16x64_i8 (two row halves,
// two planes), isum = 64 C_hi + C_lo: the reference's per-super-block integer
// exactly (|isum| < 2^27).  The 16 x 16 form draws less power than the 32 x 32
// one: register-only loops on random int8 data run at 4.06 against 3.50 POP/s
// (2.19 against 1.73 GHz, the chip being at its power limit), and its four
// accumulators hold 16 registers, so a sub-tile's float epilogue can be written
// between the next one's MFMAs (a second accumulator set) at no cost in
// registers.  On the last sub-tile each plane fragment's register is reloaded
// with the next super-block's fragment as soon as its MFMAs are issued.  The
// activations of the next super-block are copied into the other LDS stage
// meanwhile.
//
// Grid: workgroups [0, nwhole) take whole tiles, as many full rounds of
// resident workgroups as there are; the remaining tiles come last
// and are cut into P slices over K, so that they fill the final, partial round.
// P minimises the work of the busiest workgroup (at least four super-blocks a
// slice).  Within each part a block's tile is XCD-contiguous (block b is
// dispatched to XCD b % 8): the token tiles of one row tile, which share the
// weights, run side by side on one XCD; the slices are ordered (group of ntt
// tiles, slice, tile) for the same reason.  Blocks are dispatched as others
// finish: the 256 x 128 tiles of one round take 60-90 us each at [16384, 5120]
// x 2048 (contention, not work), and a persistent grid with a fixed share per
// workgroup, though it saves each tile's prologue, was no faster than one
// block per tile (387-411 against 372 us).  A sliced tile is finished
// deterministically: each slice writes its partial tile to the workspace, the
// last to arrive adds the P partials in slice order and writes the outputs.
struct PlPlan {
  int ntt, nsb;
  int nwhole;    // tiles computed whole
  int sk_tiles;  // sliced tiles
  int P;         // slices per sliced tile
  int gw;        // sliced tiles per piece group
};

// piece p of the sliced tiles -> (sliced tile u, slice)
__device__ __forceinline__ void pl_piece(const PlPlan& q, int p, int& u, int& slice) {
  const int full = q.sk_tiles / q.gw, rem = q.sk_tiles - full * q.gw;
  if (p < full * q.P * q.gw) {
    const int g = p / (q.P * q.gw), loc = p - g * q.P * q.gw;
    slice = loc / q.gw;
    u = g * q.gw + loc % q.gw;
  } else {
    const int loc = p - full * q.P * q.gw;
    slice = loc / rem;
    u = full * q.gw + loc % rem;
  }
}

// Block b of n -> its place in an order in which each XCD (block b is dispatched
// to XCD b % 8) has a contiguous run, the first n % 8 of them one longer.  In
// plain block order the token tiles of a row tile read its weights in up to
// eight L2s: with n a multiple of 8 only mapped, 5 x 20 tiles of [2560, 9728]
// x 300 in 5 slices took 63 us against 36 mapped, 258 tiles of [11008, 4096] x
// 150 58 against 44.
__device__ __forceinline__ int pl_xcd(int b, int n) {
  const int x = b & 7, r = n & 7;
  return x * (n >> 3) + (x < r ? x : r) + (b >> 3);
}

// The workgroup barrier between units: s_waitcnt vmcnt(N) lgkmcnt(0), then
// s_barrier.  Vector memory loads complete in issue order, so vmcnt(N) means
// everything but this wave's N most recent loads has landed; __syncthreads
// would wait for all of them (its release fence is vmcnt(0)).  The compiler
// barriers keep LDS accesses on their side of the s_barrier.
template <int N>
__device__ __forceinline__ void pl_sync() {
  static_assert(N >= 0 && N < 64, "vmcnt is six bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | (0x7 << 4) | ((N >> 4) << 14));
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// global_load_lds through inline assembly: lane l's 16 / 4 bytes at base +
// voff land at LDS M0 + 16 l / 4 l.  Invisible to the compiler's wait
// insertion, which otherwise makes every later LDS read of the same array
// wait for all copies in flight; pl_sync orders them.  (M0 is saved and
// restored around the copy: the compiler keeps it reserved.)
__device__ __forceinline__ uint32_t pl_lds(const void* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p);
}
__device__ __forceinline__ void pl_copy16(const void* base, uint32_t voff, const void* lds_dst) {
  uint32_t keep;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
      : "=&s"(keep)
      : "v"(voff), "s"(base), "s"(pl_lds(lds_dst))
      : "memory");
}
__device__ __forceinline__ void pl_copy4(const void* base, uint32_t voff, const void* lds_dst) {
  uint32_t keep;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2\n\ts_mov_b32 m0, %0"
      : "=&s"(keep)
      : "v"(voff), "s"(base), "s"(pl_lds(lds_dst))
      : "memory");
}

template <int NW, int NA, int PL, bool MINS>
__global__ __launch_bounds__(64 * NW, 2) void k_mmq_planes(const uint8_t* __restrict__ IMG, const uint8_t* __restrict__ XA,
                                                        float* __restrict__ Y, int rows, int tokens, PlPlan P,
                                                        float* __restrict__ part, unsigned* __restrict__ cnt) {
  constexpr int TK = 32 * NA, STAGE = kActGrp * NA, GRP = pl_grp(PL, MINS), D0 = 8192 * PL;
  static_assert(NW == 2 * NA, "a wave copies half a token group");
  constexpr int kLoads = 8 * PL + 2 + (MINS ? 4 : 0);   // loads a wave issues after a super-block's copy
  constexpr long PT = 32L * NW * TK;                // floats per partial tile
  __shared__ __attribute__((aligned(16))) uint8_t act[2][STAGE];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  const uint32_t fo = 512 * lk + 16 * lr;  // this lane's 16 bytes of a fragment
  const int nsb = P.nsb, ngrp = (rows + 31) >> 5, ntg = (tokens + 31) >> 5;
  // this workgroup's tile and super-blocks
  int tile, sb0 = 0, sb1 = nsb, u = 0, slice = 0;
  if ((int)blockIdx.x < P.nwhole) {
    tile = pl_xcd((int)blockIdx.x, P.nwhole);
  } else {
    pl_piece(P, pl_xcd((int)blockIdx.x - P.nwhole, P.sk_tiles * P.P), u, slice);
    tile = P.nwhole + u;
    sb0 = slice * nsb / P.P;
    sb1 = (slice + 1) * nsb / P.P;
  }
  const int rt = tile / P.ntt, tt = tile - rt * P.ntt;
  // The copy of a super-block's activations (a token group past the end
  // re-reads the last one): wave w half w % 2 of group w / 2's quants, and for
  // w < NA group w's sums and scales.
  auto group = [&](int a) { return XA + (long)(tt * NA + a < ntg ? tt * NA + a : ntg - 1) * nsb * kActGrp; };
  const uint8_t* const xq = group(wv >> 1) + 4096 * (wv & 1);
  const uint8_t* const xs = group(wv < NA ? wv : 0);
  auto issue_act = [&](int sb, uint8_t* st) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      pl_copy16(xq + (long)kActGrp * sb + 1024 * i, 16 * lane, st + (wv >> 1) * kActGrp + 4096 * (wv & 1) + 1024 * i);
    if (wv < NA) {
      if constexpr (MINS) pl_copy16(xs + (long)kActGrp * sb + kActSums, 16 * lane, st + wv * kActGrp + kActSums);
      if (lane < 32) pl_copy4(xs + (long)kActGrp * sb + kActScale, 4 * lane, st + wv * kActGrp + kActScale);
    }
  };
  // this wave's 32-row group in the image (a group past the end re-reads the last)
  const int grp = NW * rt + wv < ngrp ? NW * rt + wv : ngrp - 1;
  const uint8_t* const wimg = IMG + (long)grp * nsb * GRP;

  f32x4 acc[2 * NA][2];  // [16-token sub-tile][row half]
#pragma unroll
  for (int a = 0; a < 2 * NA; ++a)
#pragma unroll
    for (int r = 0; r < 2; ++r) acc[a][r] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const i32x4 zero = {};
  const f32x4 fzero = {};
  // the current super-block's plane fragments [row half][64-value step] and
  // the rows' scales and mins
  i32x4 ph[2][4], pq[2][4];
  float dw[2], dmn[2] = {0.0f, 0.0f};
  f16x4 mn[2] = {};
  auto load_scales = [&](const uint8_t* b) {
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      dw[r] = *(const float*)(b + D0 + 64 * r + 4 * lr);
      if constexpr (MINS) {
        dmn[r] = *(const float*)(b + D0 + 128 + 64 * r + 4 * lr);
        mn[r] = *(const f16x4*)(b + D0 + 256 + 512 * r + 8 * lane);
      }
    }
  };
  issue_act(sb0, &act[0][0]);
  {
    const uint8_t* b = wimg + (long)sb0 * GRP;
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        ph[r][s] = *(const i32x4*)(b + 2048 * s + 256 * r + fo);
        if constexpr (PL == 2) pq[r][s] = *(const i32x4*)(b + 8192 + 2048 * s + 256 * r + fo);
      }
    load_scales(b);
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  for (int sb = sb0; sb < sb1; ++sb) {
    const uint8_t* A = &act[(sb - sb0) & 1][0];
    uint8_t* const nxt = &act[((sb - sb0) & 1) ^ 1][0];
    const int ns = sb + 1 < sb1 ? sb + 1 : sb;  // the last super-block re-reads its own operands
    const uint8_t* nb = wimg + (long)ns * GRP;
    const float d[2] = {dw[0], dw[1]}, ndm[2] = {-dmn[0], -dmn[1]};
    // the products of this sub-tile and of the one before, whose epilogue is
    // written between this one's MFMAs
    i32x4 ch[2][2], cl[2][2];
    f32x4 dy, cm[2];
    // a sub-tile's activation fragments, read one sub-tile ahead: with the
    // reads beside their MFMAs a third of the waves' cycles were waits (512
    // tokens of [17408, 5120]: Q3_K 84 -> 80 us, Q5_K 133 -> 131)
    i32x4 af[2][4];
    auto read_act = [&](int a) {
#pragma unroll
      for (int s = 0; s < 4; ++s) af[a & 1][s] = *(const i32x4*)(A + (a >> 1) * kActGrp + 2048 * s + 256 * (a & 1) + fo);
    };
    read_act(0);
#pragma unroll
    for (int a = 0; a <= 2 * NA; ++a) {
      const int c = a & 1;
      // The copy of the next super-block's activations goes out once this
      // one's planes have landed (the first sub-tile's MFMAs wait for them):
      // the compiler's waits for the planes do not count the copy, and would
      // wait for it too if it were in flight.  No load of the next weights may
      // be issued ahead of it: pl_sync counts those as the last kLoads.
      if (a == 2) {
        // the row scales' and mins' wait comes first too
        asm volatile("" ::"v"(d[0]), "v"(d[1]));
        if constexpr (MINS) asm volatile("" ::"v"(ndm[0]), "v"(ndm[1]), "v"(mn[0]), "v"(mn[1]));
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        issue_act(ns, nxt);
        asm volatile("" ::: "memory");
      }
      if (a > 0) {
        // sub-tile a - 1: lane element e holds token 4 (lane / 16) + e.
        // summs[t][r] = sum_g bsum[t][g] * min[r][g / 2]: operands below 2048,
        // sums below 2^24, exact in the f16 MFMA
        const uint8_t* G = A + ((a - 1) >> 1) * kActGrp;
        dy = *(const f32x4*)(G + kActScale + 64 * ((a - 1) & 1) + 16 * lk);
        if constexpr (MINS) {
          const f16x4 bs = *(const f16x4*)(G + kActSums + 512 * ((a - 1) & 1) + 8 * lane);
#pragma unroll
          for (int r = 0; r < 2; ++r) cm[r] = __builtin_amdgcn_mfma_f32_16x16x16f16(bs, mn[r], fzero, 0, 0, 0);
        }
      }
      if (a + 1 < 2 * NA) {
        read_act(a + 1);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (a < 2 * NA) {
#pragma unroll
          for (int r = 0; r < 2; ++r) {
            ch[c][r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[c][s], ph[r][s], s == 0 ? zero : ch[c][r], 0, 0, 0);
            if constexpr (PL == 2)
              cl[c][r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[c][s], pq[r][s], s == 0 ? zero : cl[c][r], 0, 0, 0);
            if (a == 2 * NA - 1) {
              ph[r][s] = *(const i32x4*)(nb + 2048 * s + 256 * r + fo);
              if constexpr (PL == 2) pq[r][s] = *(const i32x4*)(nb + 8192 + 2048 * s + 256 * r + fo);
            }
          }
        }
        if (a > 0) {
          // acc += dy * (d * isum - dmin * summs) for two elements of row half s / 2
          const int r = s >> 1;
#pragma unroll
          for (int e = 2 * (s & 1); e < 2 * (s & 1) + 2; ++e) {
            int isum = ch[c ^ 1][r][e];
            if constexpr (PL == 2) {
              const int lv = cl[c ^ 1][r][e];
              isum = (isum << 6) + lv;
            }
            const float is = (float)isum;
            const float inner = MINS ? __builtin_fmaf(d[r], is, ndm[r] * cm[r][e]) : d[r] * is;
            acc[a - 1][r][e] = __builtin_fmaf(dy[e], inner, acc[a - 1][r][e]);
          }
        }
      }
    }
    load_scales(nb);
    // the next activations are in LDS once this wave's copy has landed; the
    // weight loads issued after it may stay in flight
    pl_sync<kLoads>();
  }
  if ((int)blockIdx.x >= P.nwhole && P.P > 1) {
    float* pp = part + ((long)u * P.P + slice) * PT + (long)wv * (1024 * NA) + lane;
#pragma unroll
    for (int a = 0; a < 2 * NA; ++a)
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e) sk_store(pp + ((a * 2 + r) * 4 + e) * 64, acc[a][r][e]);
    if (!sk_arrive(cnt + u, (unsigned)P.P)) return;
#pragma unroll
    for (int a = 0; a < 2 * NA; ++a)
#pragma unroll
      for (int r = 0; r < 2; ++r) acc[a][r] = fzero;
    const float* q0 = part + (long)u * P.P * PT + (long)wv * (1024 * NA) + lane;
    for (int sl = 0; sl < P.P; ++sl) {
      const float* qq = q0 + sl * PT;
      f32x4 v[2 * NA][2];
#pragma unroll
      for (int a = 0; a < 2 * NA; ++a)
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[a][r][e] = sk_load(qq + ((a * 2 + r) * 4 + e) * 64);
#pragma unroll
      for (int a = 0; a < 2 * NA; ++a)
#pragma unroll
        for (int r = 0; r < 2; ++r) acc[a][r] += v[a][r];
    }
    sk_reset(cnt + u);
  }
  const int row = 32 * (NW * rt + wv) + lr, t0 = tt * TK + 4 * lk;
#pragma unroll
  for (int a = 0; a < 2 * NA; ++a)
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int t = t0 + 16 * a + e;
        if (row + 16 * r < rows && t < tokens) Y[(long)t * rows + row + 16 * r] = acc[a][r][e];
      }
}

// A launch with tiles of 32 NA tokens (and 64 NA rows, 2 NA waves).  split =
// false: no tile is cut over K (no workspace needed).
struct PlLaunch {
  PlPlan p;
  int na;
  long steps;  // super-blocks of the busiest workgroup slot
};
static PlLaunch planes_shape(int rows, int cols, int tokens, bool split, int na) {
  PlLaunch l{};
  PlPlan& p = l.p;
  const int tk = 32 * na, nw = 2 * na;
  l.na = na;
  p.nsb = cols / 256;
  p.ntt = (tokens + tk - 1) / tk;
  const int ntiles = p.ntt * ((rows + 32 * nw - 1) / (32 * nw));
  const int cus = qhip_gpu_cu_count();
  const int slots = 8 / nw * (cus > 0 ? cus : 256);  // resident workgroups: eight waves per CU
  p.nwhole = ntiles / slots * slots;
  p.sk_tiles = ntiles - p.nwhole;
  p.P = 1;
  p.gw = 1;
  l.steps = (long)(p.nwhole / slots + (p.sk_tiles > 0)) * p.nsb;
  if (p.sk_tiles > 0 && split && p.sk_tiles <= kSkMaxTiles) {
    // the slice count with the least work on the busiest workgroup (ties:
    // fewer slices), at least four super-blocks a slice; a slice costs its
    // super-blocks plus about two for writing and adding its partial tile
    long best = -1;
    const int pmax = p.nsb / 4 > 1 ? p.nsb / 4 : 1;
    for (int q = 1; q <= pmax && q <= 64; ++q) {
      const long per = (long)p.sk_tiles * q;
      const long m = ((per + slots - 1) / slots) * ((p.nsb + q - 1) / q + (q > 1 ? 2 : 0));
      if (best < 0 || m < best) {
        best = m;
        p.P = q;
      }
    }
    l.steps = (long)(p.nwhole / slots) * p.nsb + best;
    p.gw = p.ntt < p.sk_tiles ? p.ntt : p.sk_tiles;
  }
  if (p.P == 1) {  // nothing is sliced
    p.nwhole = ntiles;
    p.sk_tiles = 0;
  }
  return l;
}

// Tiles of 128 x 64 up to 256 tokens, else of 256 x 128.  The large tile's
// workgroup has a CU to itself and does twice the work per CU of two of the
// small ones in 1.5 to 1.7 times their time, so below 2^25 weights, whose grid
// may not fill the CUs with it, it is taken where it saves a third of the
// steps.  us, small / large: Q5_K [1024, 1024] x 300 15.1 / 23.6, [2560, 2560]
// x 300 22.0 / 34.5, x 2048 50.8 / 49.8, [9728, 2560] x 300 33.7 / 38.8, x 700
// 62.9 / 52.0, x 2048 160 / 136; [14336, 4096] x 300 69.8 / 76.7, x 512 101 /
// 78, x 2048 338 / 268 (from 2^25 weights always the large one).
static PlLaunch planes_plan(int rows, int cols, int tokens, bool split) {
  if (tokens <= 256) return planes_shape(rows, cols, tokens, split, 2);
  if ((long)rows * cols < (1L << 25) &&
      3 * planes_shape(rows, cols, tokens, true, 4).steps >= 2 * planes_shape(rows, cols, tokens, true, 2).steps)
    return planes_shape(rows, cols, tokens, split, 2);
  return planes_shape(rows, cols, tokens, split, 4);
}

// Workspace of the plane-image MMQ: tile counters, then one partial tile per
// piece (none when no tile is sliced).
long planes_work_bytes(int rows, int cols, int tokens) {
  if (rows <= 0 || tokens <= 0 || cols <= 0 || cols % 256) return 0;
  const PlLaunch l = planes_plan(rows, cols, tokens, true);
  if (l.p.P <= 1) return 0;
  return kSkCountBytes + (long)l.p.sk_tiles * l.p.P * (64L * l.na) * (32 * l.na) * 4;
}

hipError_t launch_mmq_planes(int ttype, const void* img, const void* xa, float* out, int rows, int cols, int tokens,
                             void* work, long work_bytes, hipStream_t s) {
  if (rows <= 0 || tokens <= 0) return hipSuccess;
  if (!planes_format(ttype) || cols % 256 || ((uintptr_t)img & 15u) || ((uintptr_t)xa & 15u) ||
      (long)tokens * ((rows + 127) / 128) > 0x3FFFFFFFL)
    return hipErrorInvalidValue;
  const long need = planes_work_bytes(rows, cols, tokens);
  const PlLaunch l = planes_plan(rows, cols, tokens, need > 0 && work && work_bytes >= need);
  const PlPlan& p = l.p;
  unsigned* cnt = (unsigned*)work;
  float* part = work ? (float*)((uint8_t*)work + kSkCountBytes) : nullptr;
#define QHIP_PLANES(NW, NA, PL, MINS)                                                                            \
  hipLaunchKernelGGL((k_mmq_planes<NW, NA, PL, MINS>), dim3((unsigned)(p.nwhole + p.sk_tiles * p.P)),            \
                     dim3(64 * NW), 0, s, (const uint8_t*)img, (const uint8_t*)xa, out, rows, tokens, p, part, cnt)
#define QHIP_PLANES_SIZE(PL, MINS)              \
  if (l.na == 2)                                \
    QHIP_PLANES(4, 2, PL, MINS);                \
  else                                          \
    QHIP_PLANES(8, 4, PL, MINS)
  const bool mins = pl_mins(ttype);
  if (pl_planes(ttype) == 1) {
    if (mins) {
      QHIP_PLANES_SIZE(1, true);
    } else {
      QHIP_PLANES_SIZE(1, false);
    }
  } else if (mins) {
    QHIP_PLANES_SIZE(2, true);
  } else {
    QHIP_PLANES_SIZE(2, false);
  }
#undef QHIP_PLANES_SIZE
#undef QHIP_PLANES
  return hipGetLastError();
}

}  // namespace qhip
