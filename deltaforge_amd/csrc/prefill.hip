// Prompt prefill for gfx950: every token of the prompt in one pass per layer.
//
// Kernels:
// - the int4 GEMM on MFMA, with a store or a SwiGLU epilogue;
// - the 4-tap causal conv over a sequence;
// - the chunked gated delta rule;
// - GatedRMSNorm over rows;
// - q/k RMSNorm + partial RoPE over rows, which also writes the KV cache;
// - causal GQA attention in one pass over the keys.
//
// Every rounding point is the reference's forward over a sequence (reference.py:496-550,
// 610-677, 692-735), but one: from the 33rd position on, attention rounds exp(s - m) to bf16 and
// divides by the sum after the product, where the reference rounds the quotient (the same relative
// rounding). Otherwise only fp32 summation order differs.
#include <float.h>
#include <math.h>

#include <algorithm>

#include "common.h"
#include "deltaforge_hip.h"
#include "int4_block.h"

namespace df {
namespace pf {

DF_DEVICE df_f32x4 mfma(const uint4& a, const uint4& b, df_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(df_bf16x8, a), __builtin_bit_cast(df_bf16x8, b),
                                                 c, 0, 0, 0);
}

DF_DEVICE float readlane(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// ---------------------------------------------------------------------------------------
// int4 GEMM: out[m][n] = bf16( sum_k x[m][k] * bf16((nibble - 8) * scale) ), fp32 sums
// ---------------------------------------------------------------------------------------
//
// The weight is in the library's device tiling (df_int4_repack). A 1 KB block is 16 columns x
// one 128-group, and lane L of a 64-lane read owns its bytes [16 L, 16 L + 16): four words of
// column L % 16. Word i holds k = 32 (L / 16) + 8 i + e, e < 8, which is exactly the B operand
// of v_mfma_f32_16x16x32_bf16 number i, whose A operand is then x[row][32 (L / 16) + 8 i ..+8]
// (the decode GEMV's products).
//
// A workgroup computes tiles of RB row blocks of 32 x WN * CP column pairs (two 16-column tiles,
// 32 columns) on v_mfma_f32_32x32x16_bf16. Step n of a group takes word n % 4 of slots
// 2 (n / 4) and 2 (n / 4) + 1 (lanes 0..31 and 32..63): B operand as loaded, and
// x[row][128 g + 32 slot + 8 (n % 4) ..+8] as A. Its 2 WN waves are two sets: set s sums the
// groups g = s, s + 2, .. of the tile in order, and the result is set 0's sum plus set 1's, in
// every launch shape. So an output's bits do not depend on M, N or the shape chosen (a prompt
// filled in chunks equals one pass).
// - A stage is one group of each set. x rows go to LDS by global_load_lds (no registers), NBUF
//   stages in a ring, one barrier per stage; a row's 16-byte chunk c sits in slot
//   c ^ (row % 16), so the rows of an A operand read spread over the banks.
// - WREG shapes (long prompts): each wave loads its blocks and scales of the next stage into
//   registers. Otherwise blocks and scales go through the LDS ring too, NBUF - 1 stages ahead:
//   the narrow shapes' stages are shorter than a memory round trip.
// - Every wave dequantises its own blocks (17 VALU per 8 weights), the next step's during the
//   products of this one; A operands are read a step (narrow shapes: more) ahead.
// - WREG workgroups are persistent, one per CU: the next tile's first stage loads while the
//   sums of this one meet in LDS, 32 rows at a time, and leave as 16-byte stores.
// What bounds it: of a SIMD's cycles in the 4096 x 2560 x 18432 SwiGLU product (128 x 256 tiles) the matrix
// cores are busy in 51 %, other VALU (mostly the dequant) takes 42 %, 23 % run both; waves wait for their turn
// to issue 42 % of the time and for LDS, DMA and barriers 26 %. The clock averages 1.85 GHz of 2.4 there.
// LDS hands out 36 bytes a cycle and CU. Before (128 x 128 tiles, each wave all 128 rows x 32
// columns on 16 x 16 x 32 products, x through registers, one group's weights ahead) -> now, us: gate|up
// 4096 x 2560 x 18432 433 -> 373 (1038 TFLOP/s; a plain bf16 library product of that shape 368), down 4096 x
// 9216 x 2560 257 -> 201, at 100 rows 36.0 -> 23.5 and 104 -> 28.5. Tried and not kept: 16 x 16 x 32 products (same
// time, twice the operand reads), forcing products and VALU to alternate one by one (1 to 3 %
// slower), wave priorities (no change), 320-column tiles (spill).

constexpr int kGmMaxLds = 160 * 1024;
constexpr int kCUs = 256;
typedef float f32x16 __attribute__((ext_vector_type(16)));
DF_DEVICE f32x16 mfma32(const uint4& a, const uint4& b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(df_bf16x8, a), __builtin_bit_cast(df_bf16x8, b),
                                                 c, 0, 0, 0);
}

struct GemmGeom {
  int mblocks, nblocks;  // workgroups along M and N
  int flags;             // kGmVecOut, kGmScale4
};
constexpr int kGmVecOut = 1;  // out and ldo allow 16-byte stores
constexpr int kGmScale4 = 2;  // s is 4-byte aligned (the scale DMA moves dwords)

template <int RB, int CP, int WN, int NBUF, bool WREG>
struct GemmShape {
  static constexpr int BM = 32 * RB, BN = 32 * CP * WN, kThreads = 128 * WN;
  static constexpr int kTiles = 2 * CP * WN;             // 16-column tiles
  static constexpr int kRegion = BM * 256;               // one group of the x rows
  static constexpr int kXBytes = 2 * kRegion;            // both sets' groups
  static constexpr int kXOps = BM / (4 * WN);            // x DMAs per wave and stage
  static constexpr int kWBytes = WREG ? 0 : kTiles * 2048;
  static constexpr int kSOps = (kTiles + 3) / 4;        // scale DMAs (4 tiles each) per stage
  static constexpr int kSBytes = WREG ? 0 : kSOps * 256;
  static constexpr int kStage = kXBytes + kWBytes + kSBytes;
  static constexpr int kOps = kXOps + (WREG ? 0 : 2 * CP + 1);  // DMAs per wave and stage
  static constexpr int kPitch = BN + 4;                  // fp32 row pitch of the epilogue
  static constexpr int kEpi = 2 * 32 * kPitch * 4;
  // WREG: the sums meet past the first buffer, which already receives the next tile's rows
  static constexpr int kEpiOff = WREG ? kStage : 0;
  static constexpr int kLds = NBUF * kStage > kEpiOff + kEpi ? NBUF * kStage : kEpiOff + kEpi;
  static_assert(BM % (8 * WN) == 0 && kLds <= kGmMaxLds && (!WREG || NBUF == 2), "shape");
};

// 16 (4) bytes per lane from global memory to LDS at lds_base + 16 (4) * lane. Inline asm, so
// that the compiler does not wait for all of them before any LDS read; the kernel waits itself.
DF_DEVICE void dma16(const void* gaddr, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(gaddr), "s"(lds_base)
               : "memory", "m0");
}
DF_DEVICE void dma4(const void* gaddr, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(gaddr), "s"(lds_base)
               : "memory", "m0");
}
// The same with the global address as a uniform base plus the lane's offset.
DF_DEVICE void dma16s(const void* base, uint32_t offset, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(offset), "s"(base), "s"(lds_base)
               : "memory", "m0");
}
// y[i] = x / (1 + e^-x) of N values where y is rounded to bf16 at once: from the hardware's exp2 and a
// reciprocal with one Newton step instead of expf and an IEEE division, 8 VALU instead of about 40. Far
// out, where the quotient nears fp32's smallest numbers, it is silu() (one branch for the N: one for each
// took 10 us of the 717 x 2560 x 18432 SwiGLU product's 82). Of the 65536 bf16 inputs every one gives the
// same bf16 as silu(). With silu() the SwiGLU epilogue takes 6 us more of a 128 x 256 tile's 40, the conv
// 17 more of 25 (4096 tokens, 8192 channels).
template <int N>
DF_DEVICE void silu_fast(const float (&x)[N], float (&y)[N]) {
  float low = x[0];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float d = 1.0f + __builtin_amdgcn_exp2f(-1.44269504f * x[i]);
    const float r = __builtin_amdgcn_rcpf(d);
    y[i] = x[i] * fmaf(fmaf(-d, r, 1.0f), r, r);
    low = fminf(low, x[i]);
  }
  if (__builtin_expect(low < -80.0f, 0)) {
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (x[i] < -80.0f) y[i] = silu(x[i]);
  }
}
// The same where y goes on in fp32, in about 19 VALU: every finite bf16 input gives silu()'s own bits. e^-x
// is 2^n 2^f with the product -x log2 e in two parts (silu_fast rounds it: up to 3e-6 of the quotient
// at -80, 3e-7 at -4), and a residual step each corrects the reciprocal and the quotient.
template <int N>
DF_DEVICE void silu_bits(const float (&x)[N], float (&y)[N]) {
#pragma clang fp contract(off)
  float low = x[0];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float c = fminf(x[i], 104.0f);  // e^-x is nothing beside 1 long before
    const float t = -1.44269504f * c, n = rintf(t);
    const float f = (t - n) + fmaf(-1.92596299e-8f, c, fmaf(-1.44269504f, c, -t));
    const float d = 1.0f + ldexpf(__builtin_amdgcn_exp2f(f), static_cast<int>(n));
    const float r0 = __builtin_amdgcn_rcpf(d), r = fmaf(fmaf(-d, r0, 1.0f), r0, r0);
    const float q = x[i] * r;
    const float quot = copysignf(fmaf(fmaf(-d, q, x[i]), r, q), x[i]);  // (-0 stays so)
    y[i] = x[i] > 104.0f ? x[i] : quot;                                 // (and +inf)
    low = fminf(low, x[i]);
  }
  if (__builtin_expect(low < -80.0f, 0)) {
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (x[i] < -80.0f) y[i] = silu(x[i]);
  }
}
template <int N>
DF_DEVICE void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

typedef __attribute__((address_space(3))) unsigned char lds_byte;
DF_DEVICE uint32_t lds_offset(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const lds_byte*)p));
}

// A transposing LDS read: each 16 lanes give the addresses of four rows of 16 values, 4 lanes a
// row (8 bytes each), and lane i gets column i of the four.
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
DF_DEVICE s16x4 read_tr(uint32_t at) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_s16x4*>(at));
}

template <int EPI, int RB, int CP, int WN, int NBUF, bool WREG>
__global__ __launch_bounds__(128 * WN, 1) void int4_gemm_kernel(DfInt4GemmArgs p, GemmGeom geo) {
  using SH = GemmShape<RB, CP, WN, NBUF, WREG>;
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kset = wave / WN, wn = wave % WN;
  const int G = p.K / 128, ntiles = p.N / 16, stages = G / 2;

  // Workgroups go to XCDs round-robin by index. Each XCD takes a contiguous run of the tile
  // order, which walks 8 row blocks down before the next column block, so that the workgroups
  // of an XCD share x rows and weight blocks in its L2. WREG workgroups are one per CU and
  // walk their XCD's run; the others have one tile.
  const int total = geo.mblocks * geo.nblocks, xcd = blockIdx.x & 7;
  const int run = (total >> 3) * xcd + min(xcd, total & 7), run_end = run + (total >> 3) + (xcd < (total & 7) ? 1 : 0);
  const int stride = static_cast<int>(gridDim.x) < total ? static_cast<int>(gridDim.x) >> 3 : total;
  int tile = run + (blockIdx.x >> 3);
  if (tile >= run_end) return;

  // x: this thread's 16-byte chunks of a stage. Chunk i of thread tid lands at byte
  // (i * threads + tid) * 16 of the stage: row (i * 8 WN + tid / 16) % BM of a set's group,
  // slot tid % 16. Rows past M read row M - 1 (their results are not stored).
  const unsigned char* xp[SH::kXOps / 2];
  int m0, tile0, t0;
  auto start_tile = [&](int t) {
    const int per = 8 * geo.nblocks, grp = t / per, in = t - grp * per;
    const int rows = min(8, geo.mblocks - grp * 8);
    const int nb = in / rows, mb = grp * 8 + (in - nb * rows);
    m0 = mb * SH::BM;
    tile0 = nb * SH::kTiles;
    t0 = tile0 + wn * 2 * CP;
#pragma unroll
    for (int i = 0; i < SH::kXOps / 2; ++i) {
      const int r = i * 8 * WN + (tid >> 4);
      const int c = (tid & 15) ^ (r & 15);
      xp[i] = reinterpret_cast<const unsigned char*>(p.x + (size_t)min(m0 + r, p.M - 1) * p.ldx) + c * 16;
    }
  };
  start_tile(tile);
  const uint32_t lds0 = lds_offset(smem) + wave * 1024;
  auto issue_x = [&](int st, int buf) {
    const uint32_t base = lds0 + buf * SH::kStage;
#pragma unroll
    for (int i = 0; i < SH::kXOps; ++i) {
      const int set = i / (SH::kXOps / 2);
      dma16(xp[i % (SH::kXOps / 2)] + (size_t)st * 512 + set * 256, base + i * (SH::kThreads * 16));
    }
  };
  // Blocks through LDS: wave's DMA j moves block wave * 2 CP + j of [tile][group of the stage];
  // a tile's two groups are contiguous in memory. Scales: [tile][group][16], 4 tiles per DMA.
  auto issue_w = [&](int st, int buf) {
    const uint32_t base = lds_offset(smem) + buf * SH::kStage + SH::kXBytes;
#pragma unroll
    for (int j = 0; j < 2 * CP; ++j) {
      const int blk = wave * 2 * CP + j, t = min(tile0 + (blk >> 1), ntiles - 1);
      dma16(p.w + ((size_t)t * G + 2 * st + (blk & 1)) * 1024 + lane * 16, base + blk * 1024);
    }
    const int op = wave % SH::kSOps, t = min(tile0 + op * 4 + (lane >> 4), ntiles - 1);
    const uint16_t* src = p.s + ((size_t)t * G + 2 * st) * 16 + (lane & 15) * 2;
    const uint32_t dst = base + SH::kWBytes + op * 256;
    if (geo.flags & kGmScale4) {
      dma4(src, dst);
    } else {
      const uint32_t v = src[0] | (static_cast<uint32_t>(src[1]) << 16);
      *reinterpret_cast<uint32_t*>(smem + (dst - lds_offset(smem)) + lane * 4) = v;
    }
  };

  // Column lane % 32 of pair cp is column lane % 16 of tile 2 cp + (lane / 16) % 2; the lane's
  // half (lane / 32) holds slots h and 2 + h of its block, 16 bytes each.
  const int half = lane >> 5, odd = (lane >> 4) & 1, lcol = lane & 15, lrow = lane & 31;
  const uint32_t woff = half * 256 + lcol * 16;
  uint4 wq[CP][2];
  uint32_t sq[CP];
  auto load_w = [&](int st) {
    const int g = 2 * st + kset;
#pragma unroll
    for (int c = 0; c < CP; ++c) {
      const size_t blk = (size_t)min(t0 + 2 * c + odd, ntiles - 1) * G + g;
      wq[c][0] = load16(p.w + blk * 1024 + woff);
      wq[c][1] = load16(p.w + blk * 1024 + 512 + woff);
      sq[c] = p.s[blk * 16 + lcol];
    }
  };

  f32x16 acc[RB][CP];
  const DqK K = dq_consts();
  uint4 wr[CP][2];      // this set's group of the stage: the wave's blocks
  GroupScale gs[CP];
  // Operands of step n: a[n % (kAhead + 1)], read kAhead steps before, and b[n & 1].
  constexpr int kAhead = RB >= 3 ? 1 : RB == 2 ? 3 : 7;
  uint4 a[kAhead + 1][RB], b[2][CP];
  auto word = [&](int c, int n) {
    const uint4 v = wr[c][n >> 2];
    return (n & 3) == 0 ? v.x : (n & 3) == 1 ? v.y : (n & 3) == 2 ? v.z : v.w;
  };
  // takes over the blocks loaded by load_w: the compiler waits for them here and not later, when
  // its wait would include DMAs that it does not count
  auto take_w = [&](int c) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      asm volatile("" : "+v"(wq[c][h].x), "+v"(wq[c][h].y), "+v"(wq[c][h].z), "+v"(wq[c][h].w));
      wr[c][h] = wq[c][h];
    }
    asm volatile("" : "+v"(sq[c]));
    gs[c] = group_scale(static_cast<uint16_t>(sq[c]));
  };
  auto first_stages = [&]() {
    if constexpr (WREG) {
      load_w(0);
      issue_x(0, 0);
    } else {
#pragma unroll
      for (int n = 0; n < NBUF - 1; ++n)
        if (n < stages) {
          issue_x(n, n);
          issue_w(n, n);
        }
    }
  };
  first_stages();
  for (;;) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int c = 0; c < CP; ++c)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[rb][c][e] = 0.f;
    if constexpr (WREG) {
#pragma unroll
      for (int c = 0; c < CP; ++c) {
        take_w(c);
        b[0][c] = dequant8(word(c, 0), gs[c], K);
      }
    }
    int buf = 0;
    for (int st = 0; st < stages; ++st) {
      // This wave's part of stage st is in LDS: later stages' DMAs may still be in flight.
      if (st + NBUF - 2 < stages)
        wait_vm<(NBUF - 2) * SH::kOps>();
      else
        wait_vm<0>();
      // every wave's part is, and every wave is done with the buffer that is filled next
      __syncthreads();
      if (st + NBUF - 1 < stages) {
        const int next = buf == 0 ? NBUF - 1 : buf - 1;
        if constexpr (WREG) load_w(st + 1);
        issue_x(st + NBUF - 1, next);
        if constexpr (!WREG) issue_w(st + NBUF - 1, next);
      }
      const unsigned char* sb = smem + buf * SH::kStage;
      const unsigned char* xs = sb + kset * SH::kRegion + lrow * 256;
      auto read_a = [&](int n) {
        const uint32_t at = ((8 * (n >> 2) + 4 * half + (n & 3)) ^ lcol) << 4;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) a[n % (kAhead + 1)][rb] = *reinterpret_cast<const uint4*>(xs + rb * 8192 + at);
      };
#pragma unroll
      for (int n = 0; n < kAhead; ++n) read_a(n);
      if constexpr (!WREG) {
#pragma unroll
        for (int c = 0; c < CP; ++c) {
          const int blk = 2 * (wn * 2 * CP + 2 * c + odd) + kset;
          const unsigned char* w = sb + SH::kXBytes + blk * 1024 + woff;
          wr[c][0] = *reinterpret_cast<const uint4*>(w);
          wr[c][1] = *reinterpret_cast<const uint4*>(w + 512);
          gs[c] = group_scale(*reinterpret_cast<const uint16_t*>(sb + SH::kXBytes + SH::kWBytes + blk * 32 + lcol * 2));
          b[0][c] = dequant8(word(c, 0), gs[c], K);
        }
      }
      // 8 steps of 16 k: a step's A operands are read kAhead steps before and its B operands
      // dequantised between the products of the step before.
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        if (n + kAhead < 8) read_a(n + kAhead);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
          for (int c = 0; c < CP; ++c) acc[rb][c] = mfma32(a[n % (kAhead + 1)][rb], b[n & 1][c], acc[rb][c]);
#pragma unroll
        for (int c = 0; c < CP; ++c) {
          if (n < 7) {
            b[(n + 1) & 1][c] = dequant8(word(c, n + 1), gs[c], K);
          } else if (WREG) {
            take_w(c);
            b[0][c] = dequant8(word(c, 0), gs[c], K);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      buf = buf + 1 == NBUF ? 0 : buf + 1;
    }

    // The sets' sums, 32 rows at a time: lane holds D[(e % 4) + 8 (e / 4) + 4 (lane / 32)][lane % 32]
    // of each 32 x 32 product; 8 columns of a row leave together.
    const int em0 = m0, etile0 = tile0;
    __syncthreads();
    tile += stride;
    if (tile < run_end) {  // the next tile's first stage arrives during the stores
      start_tile(tile);
      first_stages();
    }
    float* ep = reinterpret_cast<float*>(smem + SH::kEpiOff);
    constexpr int kOutCols = EPI == DF_EPI_SWIGLU ? SH::BN / 2 : SH::BN;
    const int out_col0 = EPI == DF_EPI_SWIGLU ? etile0 * 8 : etile0 * 16;
    const int out_n = EPI == DF_EPI_SWIGLU ? p.N / 2 : p.N;
#pragma unroll
    for (int h = 0; h < RB; ++h) {
      if (h > 0) __syncthreads();
#pragma unroll
      for (int c = 0; c < CP; ++c)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          ep[(kset * 32 + (e & 3) + 8 * (e >> 2) + 4 * half) * SH::kPitch + (wn * CP + c) * 32 + lrow] = acc[h][c][e];
      __syncthreads();
      for (int u = tid; u < 32 * kOutCols / 8; u += SH::kThreads) {
        const int row = u / (kOutCols / 8), c = (u - row * (kOutCols / 8)) * 8;
        const int m = em0 + h * 32 + row, col = out_col0 + c;
        if (m >= p.M || col >= out_n) continue;
        float y[8];
        if constexpr (EPI == DF_EPI_SWIGLU) {
          // tiles alternate gate, up: bf16(bf16(silu(bf16(g))) * bf16(u)) (reference.py:692-693)
          const float* g = ep + row * SH::kPitch + (c / 16) * 32 + (c & 15);
          const float* g1 = g + 32 * SH::kPitch;
#pragma unroll
          for (int e = 0; e < 8; ++e) y[e] = round_bf(g[e] + g1[e]);
          float act[8];
          silu_fast(y, act);
#pragma unroll
          for (int e = 0; e < 8; ++e) y[e] = round_bf(act[e]) * round_bf(g[16 + e] + g1[16 + e]);
        } else {
          const float* g = ep + row * SH::kPitch + c;
          const float* g1 = g + 32 * SH::kPitch;
#pragma unroll
          for (int e = 0; e < 8; ++e) y[e] = g[e] + g1[e];
        }
        uint16_t* dst = p.out + (size_t)m * p.ldo + col;
        if (geo.flags & kGmVecOut) {
          *reinterpret_cast<uint4*>(dst) = make_uint4(pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3]),
                                                      pack_bf16(y[4], y[5]), pack_bf16(y[6], y[7]));
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) dst[e] = f2bf(y[e]);
        }
      }
    }
    if (tile >= run_end) break;
  }
}

// ---------------------------------------------------------------------------------------
// causal conv over the sequence (reference.py:496-510)
// ---------------------------------------------------------------------------------------

// out[t][c] = bf16(silu(bf16(sum_j w[c][j] x(p - 3 + j)))) for position p = pos0 + t, taps in
// order with fp32 sums (the decode step's arithmetic); x(q) is row q - pos0 of the input for
// q >= pos0, else the history ring (slot q mod 4, zero for positions before the first).
//
// A thread walks `per` tokens of V channels, four rows in flight and the window in registers, so a row
// is read 1 + 3 / per times; the threads of the first tokens also put the last three inputs into the
// ring, after they have read it. 8192 channels of a wider projection's rows, with the ring, us before (a
// thread to an element, four loads each, and a launch for the ring) -> now: 17 tokens 4.2 -> 2.8, 717 tokens
// 14.7 -> 7.6, 4096 tokens, 134 MB, 92 -> 32, 16384 tokens 352 -> 108.
template <int V>
__global__ __launch_bounds__(256) void conv_seq_kernel(const uint16_t* __restrict__ x, int ldx, int tokens,
                                                       int channels, const uint16_t* __restrict__ w,
                                                       uint16_t* __restrict__ ring, int pos0,
                                                       uint16_t* __restrict__ out, int ldo, int per) {
#pragma clang fp contract(off)
  struct alignas(2 * V) Row {
    uint16_t v[V];
  };
  const int c = (blockIdx.x * 256 + threadIdx.x) * V;
  if (c >= channels) return;
  const int t0 = blockIdx.y * per, t1 = min(t0 + per, tokens);
  float wk[V][4];
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const uint2 wt = *reinterpret_cast<const uint2*>(w + (size_t)(c + v) * 4);
    wk[v][0] = __uint_as_float(wt.x << 16), wk[v][1] = __uint_as_float(wt.x & 0xFFFF0000u);
    wk[v][2] = __uint_as_float(wt.y << 16), wk[v][3] = __uint_as_float(wt.y & 0xFFFF0000u);
  }
  float h[V][7];  // rows t - 3 .. t + 3
  auto load = [&](int t, int i) {
    const Row r = *reinterpret_cast<const Row*>(x + (size_t)t * ldx + c);
#pragma unroll
    for (int v = 0; v < V; ++v) h[v][i] = bf2f(r.v[v]);
  };
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int t = t0 - 3 + j;
    if (t >= 0) {
      load(t, j);
    } else {
#pragma unroll
      for (int v = 0; v < V; ++v) h[v][j] = bf2f(ring[(size_t)(c + v) * 4 + ((pos0 + t) & 3)]);
    }
  }
  for (int t = t0; t < t1; t += 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) load(min(t + i, tokens - 1), 3 + i);
    Row o[4];
#pragma unroll
    for (int v = 0; v < V; ++v) {
      float s[4], y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float acc = h[v][i] * wk[v][0];
        acc = acc + h[v][i + 1] * wk[v][1];
        acc = acc + h[v][i + 2] * wk[v][2];
        acc = acc + h[v][i + 3] * wk[v][3];
        s[i] = round_bf(acc);
      }
      silu_fast(s, y);
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i].v[v] = f2bf(y[i]);
#pragma unroll
      for (int j = 0; j < 3; ++j) h[v][j] = h[v][j + 4];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (t + i < t1) *reinterpret_cast<Row*>(out + (size_t)(t + i) * ldo + c) = o[i];
  }
  if (t0 == 0) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int t = tokens - 3 + j;
      if (t < 0) continue;
#pragma unroll
      for (int v = 0; v < V; ++v) ring[(size_t)(c + v) * 4 + ((pos0 + t) & 3)] = x[(size_t)t * ldx + c + v];
    }
  }
}

// Tokens a thread walks: long walks read fewer rows twice, short ones fill the chip.
static int conv_tokens(int tokens, int channels) { return (long)tokens * channels >= 1 << 23 ? 16 : 4; }
// Channels to a thread: two make longer runs of memory, which long prompts are bound by (8192 channels, 4096
// tokens 33.7 -> 31.7 us, 16384 118 -> 108; four are as fast), and a longer chain of ring accesses and
// SiLUs, which short ones are (1024 tokens 11.6 -> 12.7; four: 17 tokens 2.8 -> 5.6).
static bool conv_pairs(int tokens, int channels) { return (long)tokens * channels >= 1 << 24; }

// ---------------------------------------------------------------------------------------
// chunked gated delta rule (reference.py:403-461 over a sequence)
// ---------------------------------------------------------------------------------------
//
// Within a chunk of C = 64 tokens, with cumulative log-decay gamma_t = g_1 + ... + g_t and
// the chunk's initial state S0 (Dk x Dv), the token-by-token rule
//   S <- exp(g_t) S;  delta_t = beta_t (v_t - S^T k_t);  S <- S + k_t delta_t^T;  o_t = S^T q_t
// is, exactly in real arithmetic:
//   A'[t][j] = beta_t exp(gamma_t - gamma_j) (k_t . k_j), j < t      (strictly lower)
//   T        = (I + A')^-1                                            (unit lower)
//   QK[t][j] = exp(gamma_t - gamma_j) (q_t . k_j), j <= t
//   delta    = T R,  R = diag(beta) V - diag(beta e^gamma) K S0
//   O        = diag(e^gamma) Q S0 + QK delta
//   S_C      = e^gamma_C S0 + K^T diag(exp(gamma_C - gamma)) delta
// with q, k the L2-normalised rows (q also / sqrt(Dk)). T and QK do not depend on the state:
// delta_prep_kernel forms them for every (chunk, value head) at once, with the per-token
// factors. delta_scan_kernel then walks the chunks in order.
//
// The rows are kept raw, as the bf16 the conv wrote, and their norms go into the per-token
// factors. So K K^T and Q K^T are exact products of bf16 on the matrix core with fp32 sums, and
// K S0, Q S0 and K^T delta are too once the fp32 operand is written as three bf16 (8 + 8 + 8
// significant bits, every remainder exact): three products at 1 / 16 of the fp32 product's
// cost. T R and QK delta, where both sides are fp32, stay on v_mfma_f32_16x16x4_f32.
// Padding tokens past the prompt get g = beta = 0 (their rows repeat the last token's), so their
// rows of A', R and delta are zero and the state does not see them.

constexpr int kCk = 64;             // tokens per chunk
constexpr int kDk = 128;            // key (and value) head dim
constexpr int kBlk = 256;           // floats of a 16 x 16 block
constexpr int kTri = 10;            // lower block triangle of 4 x 4 blocks
// One (chunk, value head) in the scratch, in floats: T's blocks (b, c <= b) at b (b + 1) / 2 + c,
// each [j / 4][t][j % 4] (the fp32 product's A operand, lane by lane), QK's likewise, then
// per token beta e^gamma rk | beta | exp(gamma_C - gamma) rk | e^gamma rq / sqrt(Dk), then e^gamma_C.
constexpr int kPrepQk = kTri * kBlk;
constexpr int kPrepTok = 2 * kTri * kBlk;
constexpr int kPrepEc = kPrepTok + 4 * kCk;
constexpr int kPrepFloats = kPrepEc + 16;  // (16 copies: a vector load, in order with the others)

DF_DEVICE size_t prep_base(int chunk, int h, int hv) { return ((size_t)chunk * hv + h) * kPrepFloats; }
DF_DEVICE int tri(int b, int c) { return b * (b + 1) / 2 + c; }
DF_DEVICE df_f32x4 mfma4(float a, float b, df_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// acc += A B over one 16-wide block of the sum: a = A[row][4 q ..+3], b = B[4 q ..+3][col]
DF_DEVICE df_f32x4 mfma16(const float4& a, const float4& b, df_f32x4 acc) {
  acc = mfma4(a.x, b.x, acc);
  acc = mfma4(a.y, b.y, acc);
  acc = mfma4(a.z, b.z, acc);
  return mfma4(a.w, b.w, acc);
}
// 16 bytes from an address that may be only 4-byte aligned.
DF_DEVICE uint4 load16u(const uint16_t* p, bool aligned) {
  if (aligned) return *reinterpret_cast<const uint4*>(p);
  const uint32_t* w = reinterpret_cast<const uint32_t*>(p);
  return make_uint4(w[0], w[1], w[2], w[3]);
}
DF_DEVICE void store16u(uint16_t* p, const uint4& v, bool aligned) {
  if (aligned) {
    *reinterpret_cast<uint4*>(p) = v;
    return;
  }
  uint32_t* w = reinterpret_cast<uint32_t*>(p);
  w[0] = v.x, w[1] = v.y, w[2] = v.z, w[3] = v.w;
}
DF_DEVICE void unpack8(const uint4& v, float (&x)[8]) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[2 * i] = __uint_as_float(w[i] << 16);
    x[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
  }
}

// Four waves; wave w owns tokens 16 w .. + 15. K K^T and Q K^T on 16 x 16 x 32 products (their
// diagonals and Q Q^T's give the norms), A' into LDS, then T block by block: each wave inverts
// its diagonal block by forward substitution (lane = column), and the blocks below follow by
// diagonals, T_ba = -T_bb sum_{a <= c < b} A'_bc T_ca. 4096 tokens: 507 us with fp32 VALU products
// of all of R's columns and 335 MB of results -> 45 us and 44 MB.
struct PrepLds {
  uint4 k[kCk * 16], q[kCk * 16];   // raw rows, 16-byte chunk c of row t in slot c ^ (t % 16)
  float a[kTri][16][20];            // A' blocks, [t][j]
  float tt[kTri][16][20];           // T blocks transposed, [j][t]
  float td[4][16][20];              // T's diagonal blocks, [t][j]
  float pt[3][16][20];              // a product on its way from result to operand, transposed
  float gam[kCk], beta[kCk], nk[kCk], nq[kCk];
};

__global__ __launch_bounds__(256) void delta_prep_kernel(DfDeltaPrefillArgs p, float* __restrict__ scratch, int aligned) {
  __shared__ __align__(16) PrepLds L;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int chunk = blockIdx.x, h = blockIdx.y;
  const int c0 = chunk * kCk;
  const int kh = h / (p.num_v_heads / p.num_k_heads);
  const int key_dim = p.num_k_heads * kDk;
  const int n16 = lane & 15, q4 = lane >> 4;
  float* base = scratch + prep_base(chunk, h, p.num_v_heads);

  {
    uint4 kr[4], qr[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = i * 16 + (tid >> 4);
      const uint16_t* row = p.mixed + (size_t)min(c0 + t, p.tokens - 1) * p.ld_mixed + kh * kDk + (tid & 15) * 8;
      qr[i] = load16u(row, aligned);
      kr[i] = load16u(row + key_dim, aligned);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = i * 16 + (tid >> 4), at = t * 16 + ((tid & 15) ^ (t & 15));
      L.q[at] = qr[i];
      L.k[at] = kr[i];
    }
  }
  float gam = 0.0f;
  if (wave == 0) {
    const int T = c0 + lane;
    float beta = 0.0f;
    if (T < p.tokens) {
      const float av = bf2f(p.a[(size_t)T * p.ld_ab + h]), bv = bf2f(p.b[(size_t)T * p.ld_ab + h]);
      beta = round_bf(sigmoid(bv));                                         // bf16 sigmoid
      gam = -expf(bf2f(p.A_log[h])) * softplus(av + bf2f(p.dt_bias[h]));   // fp32 (reference.py:528-532)
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {  // inclusive prefix sum over the chunk
      const float o = __shfl_up(gam, off, 64);
      if (lane >= off) gam += o;
    }
    L.gam[lane] = gam;
    L.beta[lane] = beta;
  }
  __syncthreads();

  // lane: rows 16 wave + 4 q4 + r, column 16 c + n16 of block (wave, c)
  auto operand = [&](const uint4* m, int blk, int s) { return m[(blk * 16 + n16) * 16 + ((4 * s + q4) ^ n16)]; };
  df_f32x4 kk[4], qk[4], qq = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < 4; ++c) kk[c] = qk[c] = df_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const uint4 ka = operand(L.k, wave, s), qa = operand(L.q, wave, s);
    qq = mfma(qa, qa, qq);
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (c <= wave) {
        const uint4 kb = operand(L.k, c, s);
        kk[c] = mfma(ka, kb, kk[c]);
        qk[c] = mfma(qa, kb, qk[c]);
      }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (4 * q4 + r == n16) {
      float dk = 0.0f;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (c == wave) dk = kk[c][r];
      L.nk[16 * wave + n16] = 1.0f / sqrtf(dk + 1e-6f);
      L.nq[16 * wave + n16] = 1.0f / sqrtf(qq[r] + 1e-6f) / sqrtf(static_cast<float>(kDk));
    }
  __syncthreads();
  float gt[4], bt[4], nkt[4], nqt[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int t = 16 * wave + 4 * q4 + r;
    gt[r] = L.gam[t], bt[r] = L.beta[t], nkt[r] = L.nk[t], nqt[r] = L.nq[t];
  }
#pragma unroll
  for (int c = 0; c < 4; ++c)
    if (c <= wave) {
      const int j = 16 * c + n16;
      const float gj = L.gam[j], nj = L.nk[j];
      float* qout = base + kPrepQk + tri(wave, c) * kBlk + (n16 >> 2) * 64 + (n16 & 3);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * wave + 4 * q4 + r;
        const float d = j <= t ? expf(gt[r] - gj) * nj : 0.0f;
        L.a[tri(wave, c)][4 * q4 + r][n16] = j < t ? bt[r] * (kk[c][r] * nkt[r] * d) : 0.0f;
        qout[(4 * q4 + r) * 4] = qk[c][r] * nqt[r] * d;
      }
    }
  if (wave == 0) {
    const float last = readlane(gam, 63), eg = expf(gam), nk = L.nk[lane];
    base[kPrepTok + lane] = L.beta[lane] * eg * nk;
    base[kPrepTok + kCk + lane] = L.beta[lane];
    base[kPrepTok + 2 * kCk + lane] = expf(last - gam) * nk;
    base[kPrepTok + 3 * kCk + lane] = eg * L.nq[lane];
    if (lane < 16) base[kPrepEc + lane] = expf(last);
  }
  // the wave's own block of A' is complete for the wave: its inverse, column n16 in registers
  {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int d = tri(wave, wave);
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) x[t] = t == n16 ? 1.0f : 0.0f;
#pragma unroll
    for (int t = 1; t < 16; ++t) {
      float row[16];
#pragma unroll
      for (int j = 0; j < t; j += 4) {
        const float4 v = *reinterpret_cast<const float4*>(&L.a[d][t][j]);
        row[j] = v.x, row[j + 1] = v.y, row[j + 2] = v.z, row[j + 3] = v.w;
      }
#pragma unroll
      for (int j = 0; j < t; ++j) x[t] = fmaf(-row[j], x[j], x[t]);
    }
    if (q4 == 0) {
#pragma unroll
      for (int t = 0; t < 16; t += 4)
        *reinterpret_cast<float4*>(&L.tt[d][n16][t]) = make_float4(x[t], x[t + 1], x[t + 2], x[t + 3]);
    }
    if (q4 == 1) {
#pragma unroll
      for (int t = 0; t < 16; ++t) L.td[wave][t][n16] = x[t];
    }
  }
  __syncthreads();
#pragma unroll
  for (int dist = 1; dist < 4; ++dist) {
    if (wave >= dist) {
      const int b = wave, a = wave - dist;
      df_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < dist; ++i) {
        const int c = a + i;
        acc = mfma16(*reinterpret_cast<const float4*>(&L.a[tri(b, c)][n16][4 * q4]),
                     *reinterpret_cast<const float4*>(&L.tt[tri(c, a)][n16][4 * q4]), acc);
      }
      *reinterpret_cast<float4*>(&L.pt[wave - 1][n16][4 * q4]) = make_float4(acc[0], acc[1], acc[2], acc[3]);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      df_f32x4 t = {0.f, 0.f, 0.f, 0.f};
      t = mfma16(*reinterpret_cast<const float4*>(&L.td[b][n16][4 * q4]),
                 *reinterpret_cast<const float4*>(&L.pt[wave - 1][n16][4 * q4]), t);
      *reinterpret_cast<float4*>(&L.tt[tri(b, a)][n16][4 * q4]) = make_float4(-t[0], -t[1], -t[2], -t[3]);
    }
    __syncthreads();
  }
  // T out: float (j / 4, t, j % 4) of a block from its transposed [j][t]
#pragma unroll
  for (int i = 0; i < kTri; ++i)
    base[i * kBlk + tid] = L.tt[i][(tid >> 6) * 4 + (tid & 3)][(tid >> 2) & 15];
}

// Two fp32 as three bf16 each, whose sums they are: 8 significant bits apiece, every remainder
// exact. Component i holds both values' part i, packed.
DF_DEVICE void split3(float a, float b, uint32_t (&part)[3]) {
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    part[i] = pack_bf16(a, b);
    a -= __uint_as_float(part[i] << 16);
    b -= __uint_as_float(part[i] & 0xFFFF0000u);
  }
}

// The scan: one workgroup per (value head, 16 value columns), eight waves, the chunks in order.
// Wave w holds state rows 16 w .. + 15 in the product's result layout; S0 lies in LDS as
// three bf16 planes, transposed. Per chunk, a barrier after each:
//   1. waves 0..3 (16 tokens each): Y = K S0 and Z = Q S0 from one read of the planes,
//      R = beta V - (beta e^gamma rk) Y and Z into LDS;
//      waves 4..7: the next chunk's K rows by global_load_lds, this chunk's QK blocks into
//      registers, and the outputs of the chunk before, O = (e^gamma rq / sqrt(Dk)) Z + QK delta;
//   2. waves 0..3: delta = T R, into LDS in fp32 and, times exp(gamma_C - gamma) rk, in three planes;
//   3. every wave: S = e^gamma_C S + K^T delta (K read transposed by ds_read_tr16_b64), its planes.
// Every operand that is a lane's own is loaded a chunk ahead into registers.
// A serial chain of three steps a chunk, 2.5 us: 256 workgroups for 32 heads are one per CU, so
// wider column tiles would idle CUs. Waves wait 58 % of the time and the matrix cores are busy in 20 % of a
// SIMD's cycles. Without any loads the loop takes about 95 of
// the 157 us (4096 tokens, 32 heads), without T R too about 75. 319 us with the rows in fp32
// and every product on the fp32 unit. The T, Q and V loads are issued after step 2's products:
// at the start of step 1 they cost 12 us more, after its products 13.
constexpr int kScanVs = 16;
constexpr int kScanThreads = 512;

struct ScanLds {
  uint4 k[2][kCk * 16];              // raw K rows, 16-byte chunk c of row t in slot c ^ (t % 16)
  uint16_t s[3][kScanVs][kDk];       // S0's planes transposed, 16-byte chunk c of column n in slot c ^ n
  float r[kScanVs][kCk + 4];         // R transposed
  float d[2][kScanVs][kCk + 4];      // delta transposed, two chunks
  float4 z[2][4][64];                // Z as the lanes of waves 0..3 hold it, two chunks
  uint16_t dp[3][kScanVs][kCk + 8];  // the scaled delta's planes, transposed
};

__global__ __launch_bounds__(kScanThreads) void delta_scan_kernel(DfDeltaPrefillArgs p, const float* __restrict__ scratch,
                                                                  int aligned) {
  __shared__ __align__(1024) ScanLds L;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = blockIdx.x, hv = p.num_v_heads;
  const int col0 = blockIdx.y * kScanVs;
  const int nchunks = (p.tokens + kCk - 1) / kCk;
  const int n16 = lane & 15, q4 = lane >> 4;
  const bool kwave = wave < 4;
  const int w4 = wave & 3, t4 = 16 * w4 + 4 * q4;  // the wave's token block, the lane's 4 result tokens
  const int qoff = h / (hv / p.num_k_heads) * kDk, koff = qoff + p.num_k_heads * kDk;
  const int voff = 2 * p.num_k_heads * kDk + h * kDk + col0 + n16;
  float* gstate = p.state + (size_t)h * kDk * kDk;
  const uint32_t lds_k = lds_offset(&L.k[0][0]);

  df_f32x4 S;  // rows 16 wave + 4 q4 + r, column n16
#pragma unroll
  for (int r = 0; r < 4; ++r) S[r] = gstate[(size_t)(16 * wave + 4 * q4 + r) * kDk + col0 + n16];
  auto put4 = [&](uint16_t* plane, int stride, float v0, float v1, float v2, float v3) {  // into the three planes
    uint32_t a[3], b[3];
    split3(v0, v1, a);
    split3(v2, v3, b);
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<uint2*>(plane + i * stride) = make_uint2(a[i], b[i]);
  };
  auto put_state = [&]() {
    const int k = 16 * wave + 4 * q4;
    put4(&L.s[0][n16][((k >> 3) ^ n16) * 8 + (k & 7)], kScanVs * kDk, S[0], S[1], S[2], S[3]);
  };

  // K rows of a chunk, by waves 4..7: rows i * 16 + (tid - 256) / 16, slot tid % 16
  auto issue_k = [&](int chunk) {
    const int at = chunk * kCk, last = p.tokens - 1 - at;
    const uint16_t* rows = p.mixed + (size_t)at * p.ld_mixed + koff;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = i * 16 + ((tid >> 4) & 15), c = (tid & 15) ^ (row & 15);
      const uint16_t* src = rows + (size_t)min(row, last) * p.ld_mixed + c * 8;
      if (aligned)
        dma16(src, lds_k + (chunk & 1) * (kCk * 256) + w4 * 1024 + i * 4096);
      else
        L.k[chunk & 1][i * 256 + (tid & 255)] = load16u(src, false);
    }
  };
  // A lane's operands of a chunk. Waves 0..3: T blocks (w4, c <= w4), the factors beta e^gamma rk,
  // beta and exp(gamma_C - gamma) rk at tokens t4 .. + 3, V there, and Q's row 16 w4 + n16, dims
  // 32 s + 8 q4 ..+7.
  struct Ops {
    float4 t[4], f0, f1, f2;
    uint32_t v[4];
    uint4 q[4];
  };
  const size_t v_at = (size_t)t4 * p.ld_mixed + voff, q_at = (size_t)(16 * w4 + n16) * p.ld_mixed + qoff + q4 * 8;
  auto fetch = [&](int chunk) {
    Ops o;
    const float* base = scratch + prep_base(chunk, h, hv);
    const float* blk = base + tri(w4, 0) * kBlk + lane * 4;
#pragma unroll
    for (int c = 0; c < 4; ++c) o.t[c] = *reinterpret_cast<const float4*>(blk + min(c, w4) * kBlk);
    const float* tok = base + kPrepTok + t4;
    o.f0 = *reinterpret_cast<const float4*>(tok);
    o.f1 = *reinterpret_cast<const float4*>(tok + kCk);
    o.f2 = *reinterpret_cast<const float4*>(tok + 2 * kCk);
    const int at = chunk * kCk, last = p.tokens - 1 - at;
    const uint16_t* rows = p.mixed + (size_t)at * p.ld_mixed;
    if (last >= kCk - 1) {  // a full chunk: uniform bases and the lane's offsets, no address arithmetic
#pragma unroll
      for (int r = 0; r < 4; ++r) o.v[r] = rows[(size_t)r * p.ld_mixed + v_at];
#pragma unroll
      for (int s = 0; s < 4; ++s) o.q[s] = load16u(rows + s * 32 + q_at, aligned);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) o.v[r] = rows[(size_t)min(t4 + r, last) * p.ld_mixed + voff];
      const uint16_t* row = rows + (size_t)min(16 * w4 + n16, last) * p.ld_mixed + qoff + q4 * 8;
#pragma unroll
      for (int s = 0; s < 4; ++s) o.q[s] = load16u(row + s * 32, aligned);
    }
    return o;
  };
  // Waves 4..7: QK blocks (w4, c <= w4) and the factor e^gamma rq / sqrt(Dk) at tokens t4 .. + 3.
  struct Outs {
    float4 qk[4], f;
  };
  auto fetch_out = [&](int chunk) {
    Outs o;
    const float* base = scratch + prep_base(chunk, h, hv);
    const float* blk = base + kPrepQk + tri(w4, 0) * kBlk + lane * 4;
#pragma unroll
    for (int c = 0; c < 4; ++c) o.qk[c] = *reinterpret_cast<const float4*>(blk + min(c, w4) * kBlk);
    o.f = *reinterpret_cast<const float4*>(base + kPrepTok + 3 * kCk + t4);
    return o;
  };
  auto outputs = [&](const Outs& o, int chunk) {
    df_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (c <= w4)
        acc = mfma16(o.qk[c], *reinterpret_cast<const float4*>(&L.d[chunk & 1][n16][16 * c + 4 * q4]), acc);
    const float4 z = L.z[chunk & 1][w4][lane];
    const float v[4] = {fmaf(o.f.x, z.x, acc[0]), fmaf(o.f.y, z.y, acc[1]), fmaf(o.f.z, z.z, acc[2]),
                        fmaf(o.f.w, z.w, acc[3])};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int T = chunk * kCk + t4 + r;
      if (T < p.tokens) p.out[(size_t)T * p.ld_out + h * kDk + col0 + n16] = f2bf(v[r]);
    }
  };

  put_state();
  const float* ecp = scratch + kPrepEc + (lane & 15);
  float ec_next = ecp[prep_base(0, h, hv)];
  Ops next;
  Outs out;
  if (kwave)
    next = fetch(0);
  else
    issue_k(0);
  for (int chunk = 0; chunk < nchunks; ++chunk) {
    wait_vm<0>();     // this wave's operands and K rows have arrived
    __syncthreads();  // every wave's K rows and S0's planes are in LDS
    const float ec = ec_next;
    const int ahead = min(chunk + 1, nchunks - 1);
    Ops cur;
    // ---- 1: Y, Z and R; the outputs of the chunk before
    if (kwave) {
      cur = next;
      df_f32x4 y[3], z[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) y[i] = z[i] = df_f32x4{0.f, 0.f, 0.f, 0.f};
      const uint4* kt = &L.k[chunk & 1][(16 * w4 + n16) * 16];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int slot = (4 * s + q4) ^ n16;
        const uint4 ka = kt[slot];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const uint4 b = *reinterpret_cast<const uint4*>(&L.s[i][n16][slot * 8]);
          y[i] = mfma(ka, b, y[i]);
          z[i] = mfma(cur.q[s], b, z[i]);
        }
      }
      const df_f32x4 ys = y[0] + (y[1] + y[2]), zs = z[0] + (z[1] + z[2]);  // smallest first
      *reinterpret_cast<float4*>(&L.r[n16][t4]) = make_float4(fmaf(-cur.f0.x, ys[0], cur.f1.x * bf2f(cur.v[0])),
                                                              fmaf(-cur.f0.y, ys[1], cur.f1.y * bf2f(cur.v[1])),
                                                              fmaf(-cur.f0.z, ys[2], cur.f1.z * bf2f(cur.v[2])),
                                                              fmaf(-cur.f0.w, ys[3], cur.f1.w * bf2f(cur.v[3])));
      L.z[chunk & 1][w4][lane] = make_float4(zs[0], zs[1], zs[2], zs[3]);
    } else {
      if (chunk + 1 < nchunks) issue_k(chunk + 1);
      const Outs mine = out;
      out = fetch_out(chunk);
      if (chunk > 0) outputs(mine, chunk - 1);  // (the wait at the next chunk's top takes its stores in)
    }
    __syncthreads();
    // ---- 2: delta
    ec_next = ecp[prep_base(ahead, h, hv)];
    if (kwave) {
      df_f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (c <= w4) d = mfma16(cur.t[c], *reinterpret_cast<const float4*>(&L.r[n16][16 * c + 4 * q4]), d);
      next = fetch(ahead);  // issued while the products run
      *reinterpret_cast<float4*>(&L.d[chunk & 1][n16][t4]) = make_float4(d[0], d[1], d[2], d[3]);
      put4(&L.dp[0][n16][t4], kScanVs * (kCk + 8), d[0] * cur.f2.x, d[1] * cur.f2.y, d[2] * cur.f2.z, d[3] * cur.f2.w);
    }
    __syncthreads();
    // ---- 3: the state
    df_f32x4 add[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) add[i] = df_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      // K^T: dims 16 wave + n16, tokens 32 s + 8 q4 ..+7 (two transposed reads of 4 tokens x 16 dims)
      uint2 a[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int t = 32 * s + 8 * q4 + 4 * i + (n16 >> 2), c = 2 * wave + ((n16 & 3) >> 1);
        const uint32_t at = t * 256 + ((c ^ (t & 15)) << 4) + (n16 & 1) * 8;
        a[i] = __builtin_bit_cast(uint2, read_tr(lds_k + (chunk & 1) * (kCk * 256) + at));
      }
      const uint4 av = make_uint4(a[0].x, a[0].y, a[1].x, a[1].y);
#pragma unroll
      for (int i = 0; i < 3; ++i)
        add[i] = mfma(av, *reinterpret_cast<const uint4*>(&L.dp[i][n16][32 * s + 8 * q4]), add[i]);
    }
    const df_f32x4 sum = add[0] + (add[1] + add[2]);
#pragma unroll
    for (int r = 0; r < 4; ++r) S[r] = fmaf(ec, S[r], sum[r]);
    put_state();
  }
  if (!kwave) outputs(out, nchunks - 1);
#pragma unroll
  for (int r = 0; r < 4; ++r) gstate[(size_t)(16 * wave + 4 * q4 + r) * kDk + col0 + n16] = S[r];
}

// The outputs from the scratch to `out`, for an `out` over `mixed`'s memory, which every workgroup of the
// scan reads to the end: [tokens][width], 4 channels a thread.
__global__ __launch_bounds__(256) void delta_out_kernel(const uint16_t* __restrict__ from, int tokens, int width,
                                                        uint16_t* __restrict__ out, int ldo) {
  const int per = width / 4, t = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
  if (c >= per) return;
  for (int row = t; row < tokens; row += gridDim.y)
    *reinterpret_cast<uint2*>(out + (size_t)row * ldo + c * 4) =
        *reinterpret_cast<const uint2*>(from + (size_t)row * width + c * 4);
}

// ---------------------------------------------------------------------------------------
// GatedRMSNorm over rows (reference.py:115-121)
// ---------------------------------------------------------------------------------------

// Sixteen lanes to a head, 8 dims each (16-byte accesses where `aligned`, else 4-byte ones), so
// the sum is four exchanges. 4096 tokens of 32 heads, 101 MB: 38 us (a wave to a head) -> 21 (24 with silu()
// for the gate).
__global__ __launch_bounds__(256) void gated_norm_rows_kernel(const uint16_t* __restrict__ x, int ldx,
                                                              const uint16_t* __restrict__ z, int ldz,
                                                              const uint16_t* __restrict__ w, float eps, int tokens,
                                                              int heads, uint16_t* __restrict__ out, int ldo,
                                                              int aligned) {
  const long unit = (long)blockIdx.x * 16 + (threadIdx.x >> 4);
  if (unit >= (long)tokens * heads) return;
  const int t = unit / heads, hh = unit - (long)t * heads;
  const int d = (threadIdx.x & 15) * 8, at = hh * 128 + d;
  float xv[8], zv[8], wv[8];
  unpack8(load16u(x + (size_t)t * ldx + at, aligned), xv);
  unpack8(load16u(z + (size_t)t * ldz + at, aligned), zv);
  unpack8(load16u(w + d, aligned), wv);
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) ss = fmaf(xv[i], xv[i], ss);
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
  const float r = 1.0f / sqrtf(ss / 128.0f + eps);
  float gate[8];
  silu_bits(zv, gate);
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float y[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) y[e] = round_bf(wv[2 * i + e] * round_bf(xv[2 * i + e] * r)) * gate[2 * i + e];
    o[i] = pack_bf16(y[0], y[1]);
  }
  store16u(out + (size_t)t * ldo + at, make_uint4(o[0], o[1], o[2], o[3]), aligned);
}

// ---------------------------------------------------------------------------------------
// q/k RMSNorm (1 + w) + partial RoPE over rows; K/V cache rows written
// ---------------------------------------------------------------------------------------

constexpr int kHd = 256;
constexpr int kQkTokens = 4;  // the most tokens a workgroup takes

// 16 bytes where rows may be only 8-byte aligned.
DF_DEVICE uint4 load16h(const uint16_t* p, bool aligned) {
  if (aligned) return *reinterpret_cast<const uint4*>(p);
  const uint2 a = *reinterpret_cast<const uint2*>(p), b = *reinterpret_cast<const uint2*>(p + 4);
  return make_uint4(a.x, a.y, b.x, b.y);
}
DF_DEVICE void store16h(uint16_t* p, const uint4& v, bool aligned) {
  if (aligned) {
    *reinterpret_cast<uint4*>(p) = v;
    return;
  }
  *reinterpret_cast<uint2*>(p) = make_uint2(v.x, v.y);
  *reinterpret_cast<uint2*>(p + 4) = make_uint2(v.z, v.w);
}

DF_DEVICE void load4(const uint16_t* src, float x[4]) {
  const uint2 v = *reinterpret_cast<const uint2*>(src);
  x[0] = __uint_as_float(v.x << 16);
  x[1] = __uint_as_float(v.x & 0xFFFF0000u);
  x[2] = __uint_as_float(v.y << 16);
  x[3] = __uint_as_float(v.y & 0xFFFF0000u);
}
DF_DEVICE void store4(uint16_t* dst, const float x[4]) {
  *reinterpret_cast<uint2*>(dst) =
      make_uint2(static_cast<uint32_t>(f2bf(x[0])) | (static_cast<uint32_t>(f2bf(x[1])) << 16),
                 static_cast<uint32_t>(f2bf(x[2])) | (static_cast<uint32_t>(f2bf(x[3])) << 16));
}

// One thread group of 32 lanes per (token, slot), 8 dims a lane: slots < Hq are query heads
// (normed, roped -> q_out), the next Hkv are KV heads (key normed and roped, value copied, both
// into the cache at pos0 + t). The arithmetic is the decode kernel's norm_rope4 (attention.hip).
// A workgroup takes `per` tokens and `sper` of their slots, whose angles' cosines and sines, a token's in
// common, are computed once. 8192 tokens of 16 + 4 heads, 201 MB: 103 us (a wave to a slot, every
// angle in every head) -> 41; 717 tokens 13.1 -> 8.5; 17 tokens 3.9 -> 4.0 (6.9 where a workgroup goes
// through all 20 slots in three turns).
__global__ __launch_bounds__(256) void qk_rows_kernel(DfQkPrefillArgs p, int per, int sper, int aligned) {
  __shared__ float2 cs[kQkTokens * kHd / 2];
  const int l = threadIdx.x & 31, half = p.rotary_dim / 2;
  const int s0 = blockIdx.y * sper, slots = min(sper, p.num_q_heads + p.num_kv_heads - s0);
  const int t0 = blockIdx.x * per, count = min(per, p.tokens - t0);
  for (int i = threadIdx.x; i < count * half; i += 256) {
    const int t = i / half;
    const float ang = static_cast<float>(p.pos0 + t0 + t) * p.inv_freq[i - t * half];
    cs[i] = make_float2(round_bf(cosf(ang)), round_bf(sinf(ang)));
  }
  float wq[8], wkey[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    wq[i] = 1.0f + bf2f(p.q_norm[l * 8 + i]);
    wkey[i] = 1.0f + bf2f(p.k_norm[l * 8 + i]);
  }
  __syncthreads();
  for (int u = threadIdx.x >> 5; u < count * slots; u += 8) {
    const int t = u / slots, sl = s0 + u - t * slots, g = sl - p.num_q_heads;
    const bool query = g < 0;
    const uint16_t* row = p.proj + (size_t)(t0 + t) * p.ld_proj + l * 8;
    const size_t cache = ((size_t)(query ? 0 : g) * p.max_len + p.pos0 + t0 + t) * kHd + l * 8;
    float x[8];
    // head sl's [query | gate]: the query half
    unpack8(load16h(row + (query ? sl * 2 * kHd : p.k_col + g * kHd), aligned), x);
    if (!query) store16h(p.v_cache + cache, load16h(row + p.v_col + g * kHd, aligned), aligned);
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) ss = fmaf(x[i], x[i], ss);
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
    const float r = 1.0f / sqrtf(ss / static_cast<float>(kHd) + p.eps);
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = round_bf((x[i] * r) * (query ? wq[i] : wkey[i]));
    float partner[8];  // of dim d: d ^ half
#pragma unroll
    for (int i = 0; i < 8; ++i) partner[i] = half >= 8 ? __shfl_xor(x[i], half >> 3, 64) : x[i ^ 4];
    const float2* tab = cs + t * half;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int dim = l * 8 + i;
      if (dim < p.rotary_dim) {
        const float2 a = tab[dim & (half - 1)];
        const float rotated = dim < half ? -partner[i] : partner[i];
        x[i] = round_bf(x[i] * a.x) + round_bf(rotated * a.y);
      }
    }
    uint16_t* dst = query ? p.q_out + ((size_t)(t0 + t) * p.num_q_heads + sl) * kHd + l * 8 : p.k_cache + cache;
    store16h(dst, make_uint4(pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3]), pack_bf16(x[4], x[5]), pack_bf16(x[6], x[7])),
             aligned);
  }
}

// ---------------------------------------------------------------------------------------
// causal GQA attention over the prompt (reference.py:645-677)
// ---------------------------------------------------------------------------------------
//
// scores = bf16(bf16(q . k) * scale), masked above the diagonal; p = softmax over fp32; o = p V
// with p rounded to bf16 for the product; out = bf16(bf16(o) * bf16(gate_fn(gate))).
//
// A workgroup owns 32 query positions of one KV head. Wave w is query head 4 g + w % 4 and key
// set w / 4, which takes every other 32 keys; the two sets' (m, l, O) are merged at the end.
// Keys and values pass through LDS in blocks of 64 (32 for each set), two buffers, filled by
// global_load_lds a block ahead. One pass over the keys, on v_mfma_f32_32x32x16_bf16 with the
// keys as rows: S^T = K Q^T leaves a query's scores in its lane's registers (column
// lane % 32), so max and sum need one exchange with lane + 32, and exp(S^T) is at once the B
// operand of O^T = V^T P^T: lane half h holds keys 4 h + {0..3, 8..11} of 16, and V^T comes in
// that key order from ds_read_tr16_b64, which transposes 4 keys x 16 dims of the row-major
// tile. K's 16-byte chunks are XORed with key % 16 and V's with 4 (key % 8), so that both
// reads spread over the banks.
//
// p is exp(s - m) with m a running maximum that moves only when a block exceeds it by more
// than 2^8 (p and l then stay far inside fp32); bf16(p) has the relative rounding that the
// normalised bf16 probability has, and l sums the unrounded p. The first 32 positions, whose
// few weights are large, know their sum before the product and round p / l as the reference
// does. A row's result depends only on its own scores in blocks of 32 keys from key 0, so a
// prompt filled in chunks equals one pass.
//
// The next block's K products run between this block's softmax. No unit is full (8192 tokens): of a SIMD's
// cycles the matrix cores are busy in 41 %, other VALU takes 29 %, 15 % run both, LDS hands out 53 bytes a
// cycle and CU; waves wait for LDS, DMA and barriers 39 % of the time and for their turn to issue 27 %.
// Causal prompts, us before (two passes over the keys, 16 query rows to a wave) -> now: 8192
// tokens 3106 -> 573 (959 TFLOP/s), 717 tokens 114 -> 38; 2000 tokens after 20 000 keys 675 (1019 TFLOP/s).
// Measured and not kept: 64 positions to a workgroup and no key sets (8192 tokens 562, 717 tokens 55), two
// barriers with K and V two blocks ahead (595), reading an operand right before its product (597).

constexpr int kAtKeys = 64;
constexpr int kAtTile = kAtKeys * kHd * 2;  // bytes of a K or V block
constexpr int kAtThreads = 512;
constexpr int kAtMl = 4 * kAtTile;          // byte offset of the sets' (m, l) exchange
constexpr int kAtLds = kAtMl + 8 * 32 * 8;
constexpr float kLog2e = 1.44269504088896f;
constexpr int kAtPow2Scale = 1;  // scale is a positive power of two: bf16(s * scale) is exact
constexpr int kAtVecGate = 2;    // gate rows allow 8-byte loads
constexpr int kAtVecOut = 4;     // out rows allow 8-byte stores

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;

__global__ __launch_bounds__(kAtThreads, 1) void attn_prefill_kernel(DfAttnPrefillArgs p, int flags) {
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, q = lane & 31;
  // KV head fastest, so that an XCD (workgroups i mod 8) reads one head's keys; the last
  // positions, which have the most keys, first
  const int g = blockIdx.x % p.num_kv_heads;
  const int qblocks = (p.tokens + 31) / 32;
  const int h = g * 4 + (wave & 3), kset = wave >> 2, t0 = (qblocks - 1 - blockIdx.x / p.num_kv_heads) * 32;
  const uint32_t lds0 = lds_offset(smem);

  const int nkeys = p.pos0 + min(t0 + 32, p.tokens);  // keys any row of the block attends
  const int nkb = (nkeys + kAtKeys - 1) / kAtKeys;
  const unsigned char* kbase = reinterpret_cast<const unsigned char*>(p.k_cache + (size_t)g * p.max_len * kHd);
  const unsigned char* vbase = reinterpret_cast<const unsigned char*>(p.v_cache + (size_t)g * p.max_len * kHd);
  constexpr int kOps = kAtTile / (kAtThreads * 16);  // DMAs per wave and block of K or V
  constexpr int kAhead = 2;                          // LDS operands in flight
  // This thread's chunk of DMA i: key 16 i + tid / 32 of the block, slot tid % 32. Full blocks go
  // by a uniform base and a per-thread offset; in the last one keys past the end repeat the last.
  const uint32_t krow = (tid >> 5) * (kHd * 2), kchunk = ((tid & 31) ^ (tid >> 5)) << 4;
  const uint32_t vchunk = ((tid & 31) ^ (((tid >> 5) & 7) << 2)) << 4;
  auto issue = [&](const unsigned char* base, uint32_t chunk, int kb, uint32_t at) {
    const unsigned char* block = base + (size_t)kb * kAtTile;
    if (kb * kAtKeys + kAtKeys <= nkeys) {
#pragma unroll
      for (int i = 0; i < kOps; ++i)
        dma16s(block + i * (16 * kHd * 2), krow + chunk, at + i * (kAtThreads * 16));
    } else {
#pragma unroll
      for (int i = 0; i < kOps; ++i) {
        const int key = min(i * 16 + (tid >> 5), nkeys - 1 - kb * kAtKeys);
        dma16s(block, key * (kHd * 2) + chunk, at + i * (kAtThreads * 16));
      }
    }
  };
  auto issue_k = [&](int kb) { issue(kbase, kchunk, kb, lds0 + (kb & 1) * 2 * kAtTile + wave * 1024); };
  auto issue_v = [&](int kb) { issue(vbase, vchunk, kb, lds0 + (kb & 1) * 2 * kAtTile + kAtTile + wave * 1024); };
  // B operands of K Q^T: step n takes dims 16 n + 8 half ..+7. Rows past the prompt repeat its last
  // one and are not stored.
  uint4 qf[16];
  {
    const uint16_t* src = p.q + ((size_t)min(t0 + q, p.tokens - 1) * p.num_q_heads + h) * kHd + half * 8;
#pragma unroll
    for (int n = 0; n < 16; ++n) qf[n] = *reinterpret_cast<const uint4*>(src + n * 16);
#pragma unroll
    for (int n = 0; n < 16; ++n)
      asm volatile("" : "+v"(qf[n].x), "+v"(qf[n].y), "+v"(qf[n].z), "+v"(qf[n].w));  // waited for here
  }
  issue_k(0);
  issue_v(0);
  if (nkb > 1) issue_k(1);
  const int pos = p.pos0 + t0 + q;
  const int pos_lo = p.pos0 + t0, pos_hi = pos_lo + 31;  // the wave's positions
  const bool pow2 = flags & kAtPow2Scale;
  const float cexp = pow2 ? p.scale * kLog2e : kLog2e;
  const float masked = p.scale < 0.0f ? INFINITY : -INFINITY;  // a score that the scale makes -inf

  f32x16 o[8];
#pragma unroll
  for (int db = 0; db < 8; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[db][e] = 0.f;
  float m = -INFINITY, l = 0.0f;  // m: the maximum in use, in units of log2(e) (scaled)

  // LDS addresses of this lane: K row q, chunk half ^ (q % 16) (step n: ^ 32 n); V key
  // 4 half + (lane % 16) / 4, dims 16 ((lane / 16) % 2) + 4 (lane % 4) (dim block db: ^ 64 db)
  const uint32_t ka = q * (kHd * 2) + ((half ^ (q & 15)) << 4);
  const int vkey = 4 * half + ((lane & 15) >> 2);
  const uint32_t va = vkey * (kHd * 2) + (vkey << 6) + ((lane >> 4) & 1) * 32 + (lane & 3) * 8;

  // blocks in which this set has keys that some row attends
  const int live = pos_hi < kset * 32 ? 0 : min(nkb, (pos_hi - kset * 32) / kAtKeys + 1);
  auto k_at = [&](int kb) {
    uint32_t at = lds0 + (kb & 1) * 2 * kAtTile + kset * (32 * kHd * 2) + ka;
    asm volatile("" : "+v"(at));  // the 16 addresses are made from it block by block: kept, they would spill
    return at;
  };
  auto read_k = [&](uint32_t at, int n) { return *reinterpret_cast<const lds_u32x4*>(at ^ (n << 5)); };
  // lane: query q, keys key0 + (e % 4) + 8 (e / 4) + 4 half
  auto mask = [&](f32x16& s, int kb) {
    const int key0 = kb * kAtKeys + kset * 32;
    if (key0 + 31 > pos_lo) {
#pragma unroll
      for (int e = 0; e < 16; ++e)
        s[e] = key0 + (e & 3) + 8 * (e >> 2) + 4 * half <= pos ? s[e] : masked;
    }
  };
  auto prob = [&](float r, float mc) { return __builtin_amdgcn_exp2f(fmaf(r, cexp, -mc)); };
  // One block: the products of the next block's scores (sn) run between the VALU work of this
  // block's softmax (s), two scores a product; then this block's values.
  // After the last block the products read a stale buffer and their result is dropped.
  auto step = [&](f32x16& s, int kb) {
    u32x4 kf[kAhead];
    f32x16 sn;
    const uint32_t kat = k_at(kb + 1);
#pragma unroll
    for (int e = 0; e < 16; ++e) sn[e] = 0.f;
#pragma unroll
    for (int n = 0; n < kAhead; ++n) kf[n] = read_k(kat, n);
    __builtin_amdgcn_sched_barrier(0);
    auto product = [&](int n) {
      sn = mfma32(__builtin_bit_cast(uint4, kf[n % kAhead]), qf[n], sn);
      if (n + kAhead < 16) kf[n % kAhead] = read_k(kat, n + kAhead);
    };
    float mx = -INFINITY;
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      product(n);
      const uint32_t two = pack_bf16(s[2 * n], s[2 * n + 1]);
      s[2 * n] = __uint_as_float(two << 16);
      s[2 * n + 1] = __uint_as_float(two & 0xFFFF0000u);
      if (!pow2) {
        s[2 * n] = round_bf(s[2 * n] * p.scale);
        s[2 * n + 1] = round_bf(s[2 * n + 1] * p.scale);
      }
      mx = fmaxf(fmaxf(mx, s[2 * n]), s[2 * n + 1]);
      __builtin_amdgcn_sched_barrier(0);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * cexp;
    const bool move = mx > m + 8.0f;
    if (__any(move)) {
      const float mn = move ? mx : m;
      const float alpha = move ? __builtin_amdgcn_exp2f(m - mn) : 1.0f;
      m = mn;
      l *= alpha;
#pragma unroll
      for (int db = 0; db < 8; ++db)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[db][e] *= alpha;
    }
    const float mc = m == -INFINITY ? 0.0f : m;
    float sum = 0.0f;
    uint32_t pk[8];
#pragma unroll
    for (int n = 8; n < 16; ++n) {
      product(n);
      const int e = 2 * (n - 8);
      const float p0 = prob(s[e], mc), p1 = prob(s[e + 1], mc);
      sum += p0 + p1;
      pk[n - 8] = pack_bf16(p0, p1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (kb == 0 && kset == 0 && pos_lo < 32) {
      // a row whose keys all lie in the first 32 is normalised before the rounding
      const float total = sum + __shfl_xor(sum, 32, 64);
      const float norm = pos >= 32 ? 1.0f : total == 0.0f ? 0.0f : 1.0f / total;
      if (pos < 32) sum = 0.5f;
#pragma unroll
      for (int e = 0; e < 16; e += 2) pk[e / 2] = pack_bf16(prob(s[e], mc) * norm, prob(s[e + 1], mc) * norm);
    }
    l += sum;
    mask(sn, kb + 1);
    // O^T += V^T P^T: keys 16 kk + 4 half + {0..3, 8..11} are the lane's values 8 kk .. 8 kk + 7
    uint32_t vat = lds0 + (kb & 1) * 2 * kAtTile + kAtTile + kset * (32 * kHd * 2) + va;
    asm volatile("" : "+v"(vat));
    auto read_v = [&](int u) {  // unit u: dims 32 (u / 2) .. + 31, keys 16 (u % 2) .. + 15
      const uint32_t at = (vat ^ ((u >> 1) << 6)) + (u & 1) * (16 * kHd * 2);
      const uint2 a0 = __builtin_bit_cast(uint2, read_tr(at));
      const uint2 a1 = __builtin_bit_cast(uint2, read_tr(at + 8 * (kHd * 2)));
      return make_uint4(a0.x, a0.y, a1.x, a1.y);
    };
    uint4 vf[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) vf[u] = read_v(u);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int kk = u & 1;
      const uint4 pv = make_uint4(pk[4 * kk], pk[4 * kk + 1], pk[4 * kk + 2], pk[4 * kk + 3]);
      o[u >> 1] = mfma32(vf[u % kAhead], pv, o[u >> 1]);
      if (u + kAhead < 16) vf[u % kAhead] = read_v(u + kAhead);
      __builtin_amdgcn_sched_barrier(0);
    }
    s = sn;
  };
  f32x16 sa;
  wait_vm<0>();
  __syncthreads();
  if (live > 0) {
    const uint32_t kat = k_at(0);
#pragma unroll
    for (int e = 0; e < 16; ++e) sa[e] = 0.f;
#pragma unroll
    for (int n = 0; n < 16; ++n) sa = mfma32(__builtin_bit_cast(uint4, read_k(kat, n)), qf[n], sa);
    mask(sa, 0);
  }
  for (int kb = 0; kb < nkb; ++kb) {
    wait_vm<0>();     // this wave's part of K (kb + 1) and V (kb) is in LDS
    __syncthreads();  // every wave's is, and every wave is done with K (kb) and V (kb - 1)
    if (kb + 2 < nkb) issue_k(kb + 2);
    if (kb + 1 < nkb) issue_v(kb + 1);
    if (kb < live) step(sa, kb);
  }
  l += __shfl_xor(l, 32, 64);  // the two halves summed their own keys

  // ---- the sets' merge: each set finishes half of the head's dims -----------------------
  // The gates this wave will need (rows 2 i + lane / 32, 4 dims) are loaded ahead.
  const int d0 = kset * 128 + (lane & 31) * 4;
  uint2 gr[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int t = min(t0 + 2 * i + half, p.tokens - 1);
    const uint16_t* src = p.gate + (size_t)t * p.ld_gate + h * p.gate_head_stride + d0;
    if (flags & kAtVecGate) {
      gr[i] = *reinterpret_cast<const uint2*>(src);
    } else {
      gr[i].x = src[0] | (static_cast<uint32_t>(src[1]) << 16);
      gr[i].y = src[2] | (static_cast<uint32_t>(src[3]) << 16);
    }
  }
  __syncthreads();  // every wave is done with the keys and values
  float2* ml = reinterpret_cast<float2*>(smem + kAtMl);
  if (half == 0) ml[wave * 32 + q] = make_float2(m, l);
  const int partner = wave ^ 4;
  float4* give = reinterpret_cast<float4*>(smem + partner * 16384) + lane;
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const f32x16 v = kset ? o[db] : o[4 + db];
      give[(db * 4 + e) * 64] = make_float4(v[4 * e], v[4 * e + 1], v[4 * e + 2], v[4 * e + 3]);
    }
  __syncthreads();
  const float2 other = ml[partner * 32 + q];
  const float mm = fmaxf(m, other.x);
  const float a_own = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mm);
  const float a_oth = other.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(other.x - mm);
  // set 0's term first, whichever set adds them
  const float l0 = kset ? a_oth * other.y : a_own * l, l1 = kset ? a_own * l : a_oth * other.y;
  const float den = l0 + l1, inv = den == 0.0f ? 0.0f : 1.0f / den;
  const float w_own = a_own * inv, w_oth = a_oth * inv;
  const float4* take = reinterpret_cast<const float4*>(smem + wave * 16384) + lane;
  float y[4][16];
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const f32x16 v = kset ? o[4 + db] : o[db];
      const float4 u = take[(db * 4 + e) * 64];
      const float uu[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) y[db][4 * e + i] = fmaf(v[4 * e + i], w_own, uu[i] * w_oth);
    }
  // bf16(o) through this wave's part of LDS to whole rows, times bf16(gate_fn(gate))
  constexpr int kPitch = 128 * 2 + 16;
  unsigned char* ot = smem + wave * 16384;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      *reinterpret_cast<uint2*>(ot + q * kPitch + (db * 32 + e * 8 + half * 4) * 2) =
          make_uint2(pack_bf16(y[db][4 * e], y[db][4 * e + 1]), pack_bf16(y[db][4 * e + 2], y[db][4 * e + 3]));
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int t = t0 + 2 * i + half;
    if (t >= p.tokens) break;
    float v[4], gx[4];
    load4(reinterpret_cast<const uint16_t*>(ot + (2 * i + half) * kPitch) + (lane & 31) * 4, v);
    load4(reinterpret_cast<const uint16_t*>(&gr[i]), gx);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] *= round_bf(p.gate_kind == 0 ? sigmoid(gx[j]) : silu(gx[j]));
    uint16_t* orow = p.out + (size_t)t * p.ld_out + h * kHd + d0;
    if (flags & kAtVecOut) {
      store4(orow, v);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) orow[j] = f2bf(v[j]);
    }
  }
}

}  // namespace pf
}  // namespace df

using namespace df;
using namespace df::pf;

template <int EPI, int RB, int CP, int WN, int NBUF, bool WREG>
static hipError_t launch_gemm_shape(const DfInt4GemmArgs& a, hipStream_t stream) {
  using SH = GemmShape<RB, CP, WN, NBUF, WREG>;
  GemmGeom geo;
  geo.mblocks = (a.M + SH::BM - 1) / SH::BM;
  geo.nblocks = (a.N / 16 + SH::kTiles - 1) / SH::kTiles;
  geo.flags = (((reinterpret_cast<uintptr_t>(a.out) & 15) == 0 && a.ldo % 8 == 0) ? kGmVecOut : 0) |
              ((reinterpret_cast<uintptr_t>(a.s) & 3) == 0 ? kGmScale4 : 0);
  const long total = (long)geo.mblocks * geo.nblocks;
  if (total > 0x7FFFFFFF) return hipErrorInvalidValue;
  const unsigned grid = WREG && total > kCUs ? kCUs : (unsigned)total;
  hipLaunchKernelGGL((int4_gemm_kernel<EPI, RB, CP, WN, NBUF, WREG>), dim3(grid), dim3(SH::kThreads), SH::kLds, stream,
                     a, geo);
  return hipGetLastError();
}

// The shapes, and the cost of one workgroup in each: start and epilogue, and a stage (ns). A launch
// takes as many rounds of one workgroup per CU as it has tiles, so the shape taken is the one
// with the least rounds * (start + stages * stage). Of 65 products (the model's five projections at 17 ..
// 8192 rows, all seven shapes timed) it is the fastest in 64 and 0.6 % slower than that in one. As a time
// the cost is up to 15 % low where the clock falls (320 us for 376), alike for the wide shapes. Wide ones serve
// long prompts (2560 x 18432 at 4096 rows: 9 full rounds of 128 x 256, 376 us against 443 with 128 x 128), 96
// rows where they pack better (9216 x 2560 at 4096 rows: 197 us against 229), narrow ones reach more CUs
// with a short prompt (9216 x 2560 at 100 rows: 27.3 us with 32 x 64 against 97 with 128 x 256).
struct GemmCost {
  int bm, bn, start, stage;
};
constexpr GemmCost kGemmCosts[] = {{128, 256, 9000, 2650}, {128, 128, 5000, 1750}, {96, 256, 7000, 2250},
                                   {96, 128, 4000, 1350},  {64, 128, 3200, 1100},  {64, 64, 2000, 880},
                                   {32, 64, 1500, 710}};

static int gemm_plan(int M, int K, int N) {
  int best = 0;
  double best_cost = 0;
  for (int i = 0; i < static_cast<int>(sizeof(kGemmCosts) / sizeof(kGemmCosts[0])); ++i) {
    const GemmCost& c = kGemmCosts[i];
    const long tiles = (long)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn);
    const double cost = (double)((tiles + kCUs - 1) / kCUs) * (c.start + (double)c.stage * (K / 256));
    if (i == 0 || cost < best_cost) best = i, best_cost = cost;
  }
  return best;
}

template <int EPI>
static hipError_t launch_gemm(const DfInt4GemmArgs& a, int shape, hipStream_t stream) {
  switch (shape) {
    case 0: return launch_gemm_shape<EPI, 4, 2, 4, 2, true>(a, stream);
    case 1: return launch_gemm_shape<EPI, 4, 1, 4, 2, true>(a, stream);
    case 2: return launch_gemm_shape<EPI, 3, 2, 4, 2, true>(a, stream);
    case 3: return launch_gemm_shape<EPI, 3, 1, 4, 2, true>(a, stream);
    case 4: return launch_gemm_shape<EPI, 2, 1, 4, 2, true>(a, stream);
    case 5: return launch_gemm_shape<EPI, 2, 1, 2, 3, false>(a, stream);
    default: return launch_gemm_shape<EPI, 1, 1, 2, 4, false>(a, stream);
  }
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

extern "C" {

int df_int4_gemm(const DfInt4GemmArgs* a, hipStream_t stream) {
  if (!a || !a->x || !a->w || !a->s || !a->out || a->M < 1 || a->K < 256 || a->K % 256 || a->N < 16 || a->N % 16)
    return DF_BAD_ARGUMENT;
  if (a->epilogue != DF_EPI_STORE && a->epilogue != DF_EPI_SWIGLU) return DF_BAD_ARGUMENT;
  if (a->epilogue == DF_EPI_SWIGLU && a->N % 32) return DF_BAD_ARGUMENT;
  const int out_cols = a->epilogue == DF_EPI_SWIGLU ? a->N / 2 : a->N;
  if (a->ldx < a->K || a->ldx % 8 || a->ldo < out_cols || !aligned16(a->x) || !aligned16(a->w))
    return DF_BAD_ARGUMENT;
  // (8.4 M rows: tile and row counts stay far inside int)
  if ((a->M + 127) / 128 > 65535) return DF_BAD_ARGUMENT;
  const int shape = gemm_plan(a->M, a->K, a->N);
  const hipError_t e = a->epilogue == DF_EPI_SWIGLU ? launch_gemm<DF_EPI_SWIGLU>(*a, shape, stream)
                                                    : launch_gemm<DF_EPI_STORE>(*a, shape, stream);
  return e == hipSuccess ? DF_OK : DF_LAUNCH_FAILED;
}
int df_causal_conv_prefill(const uint16_t* x, int ldx, int tokens, int channels, const uint16_t* weight,
                           uint16_t* ring, int pos0, uint16_t* out, int ldo, hipStream_t stream) {
  if (!x || !weight || !ring || !out || tokens < 1 || channels < 1 || ldx < channels || ldo < channels || pos0 < 0 ||
      (reinterpret_cast<uintptr_t>(weight) & 7) || tokens > 65535)
    return DF_BAD_ARGUMENT;
  const int per = conv_tokens(tokens, channels);
  const bool pairs = conv_pairs(tokens, channels) && channels % 2 == 0 && ldx % 2 == 0 && ldo % 2 == 0 &&
                     !(reinterpret_cast<uintptr_t>(x) & 3) && !(reinterpret_cast<uintptr_t>(out) & 3);
  const int width = pairs ? 512 : 256;  // channels a workgroup
  hipLaunchKernelGGL(pairs ? conv_seq_kernel<2> : conv_seq_kernel<1>,
                     dim3((channels + width - 1) / width, (tokens + per - 1) / per), dim3(256), 0, stream, x, ldx, tokens,
                     channels, weight, ring, pos0, out, ldo, per);
  DF_RETURN_LAUNCH_STATUS();
}

size_t df_delta_rule_prefill_workspace_bytes(int tokens, int num_v_heads) {
  if (tokens < 1 || num_v_heads < 1) return 0;
  const size_t chunks = (size_t)(tokens + kCk - 1) / kCk;
  return chunks * num_v_heads * (kPrepFloats * sizeof(float) + kCk * kDk * sizeof(uint16_t));
}

// Whether two sets of `rows` rows (lda and ldb elements apart, wa and wb long) share memory. Rows of one
// stride whose columns lie beside each other do not.
static bool rows_overlap(const uint16_t* a, int lda, int wa, const uint16_t* b, int ldb, int wb, int rows) {
  const uintptr_t a0 = reinterpret_cast<uintptr_t>(a), b0 = reinterpret_cast<uintptr_t>(b);
  if (a0 + ((size_t)(rows - 1) * lda + wa) * 2 <= b0 || b0 + ((size_t)(rows - 1) * ldb + wb) * 2 <= a0) return false;
  if (lda != ldb) return true;
  const size_t ld = (size_t)lda * 2, apart = b0 >= a0 ? (b0 - a0) % ld : (ld - (a0 - b0) % ld) % ld;
  return apart < (size_t)wa * 2 || apart + (size_t)wb * 2 > ld;
}

int df_delta_rule_prefill(const DfDeltaPrefillArgs* a, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (!a || !a->mixed || !a->a || !a->b || !a->A_log || !a->dt_bias || !a->state || !a->out || a->tokens < 1)
    return DF_BAD_ARGUMENT;
  if (a->num_k_heads < 1 || a->num_v_heads < 1 || a->num_v_heads % a->num_k_heads) return DF_BAD_ARGUMENT;
  const int channels = 2 * a->num_k_heads * kDk + a->num_v_heads * kDk;
  if (a->ld_mixed < channels || a->ld_mixed % 2 || a->ld_out < a->num_v_heads * kDk || a->ld_out % 4 ||
      a->ld_ab < a->num_v_heads || (reinterpret_cast<uintptr_t>(a->mixed) & 3) ||
      (reinterpret_cast<uintptr_t>(a->out) & 7) || (reinterpret_cast<uintptr_t>(a->state) & 15))
    return DF_BAD_ARGUMENT;
  if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 15) ||
      workspace_bytes < df_delta_rule_prefill_workspace_bytes(a->tokens, a->num_v_heads))
    return DF_WORKSPACE_TOO_SMALL;
  const int chunks = (a->tokens + kCk - 1) / kCk;
  float* scratch = reinterpret_cast<float*>(workspace);
  const int aligned = aligned16(a->mixed) && a->ld_mixed % 8 == 0;  // rows allow 16-byte loads
  hipLaunchKernelGGL(delta_prep_kernel, dim3(chunks, a->num_v_heads), dim3(256), 0, stream, *a, scratch, aligned);
  const int width = a->num_v_heads * kDk;
  DfDeltaPrefillArgs scan = *a;
  const bool staged = rows_overlap(a->mixed, a->ld_mixed, channels, a->out, a->ld_out, width, a->tokens);
  if (staged) {
    scan.out = reinterpret_cast<uint16_t*>(scratch + (size_t)chunks * a->num_v_heads * kPrepFloats);
    scan.ld_out = width;
  }
  hipLaunchKernelGGL(delta_scan_kernel, dim3(a->num_v_heads, kDk / kScanVs), dim3(kScanThreads), 0, stream, scan,
                     static_cast<const float*>(scratch), aligned);
  if (staged)
    hipLaunchKernelGGL(delta_out_kernel, dim3((width / 4 + 255) / 256, std::min(a->tokens, 65535)), dim3(256), 0, stream,
                       scan.out, a->tokens, width, a->out, a->ld_out);
  DF_RETURN_LAUNCH_STATUS();
}

int df_gated_rms_norm_rows(const uint16_t* x, int ldx, const uint16_t* z, int ldz, const uint16_t* weight, float eps,
                           int tokens, int heads, uint16_t* out, int ldo, hipStream_t stream) {
  if (!x || !z || !weight || !out || tokens < 1 || heads < 1 || ldx < heads * 128 || ldz < heads * 128 ||
      ldo < heads * 128 || ldx % 2 || ldz % 2 || ldo % 2 || (reinterpret_cast<uintptr_t>(x) & 3) ||
      (reinterpret_cast<uintptr_t>(z) & 3) || (reinterpret_cast<uintptr_t>(out) & 3) ||
      (reinterpret_cast<uintptr_t>(weight) & 3))
    return DF_BAD_ARGUMENT;
  const long units = (long)tokens * heads;
  const int aligned = aligned16(x) && aligned16(z) && aligned16(weight) && aligned16(out) && ldx % 8 == 0 &&
                      ldz % 8 == 0 && ldo % 8 == 0;
  hipLaunchKernelGGL(gated_norm_rows_kernel, dim3((units + 15) / 16), dim3(256), 0, stream, x, ldx, z, ldz, weight, eps,
                     tokens, heads, out, ldo, aligned);
  DF_RETURN_LAUNCH_STATUS();
}

int df_qk_norm_rope_prefill(const DfQkPrefillArgs* a, hipStream_t stream) {
  if (!a || !a->proj || !a->q_norm || !a->k_norm || !a->inv_freq || !a->q_out || !a->k_cache || !a->v_cache ||
      a->tokens < 1 || a->num_q_heads < 1 || a->num_kv_heads < 1 || a->pos0 < 0 ||
      a->pos0 + a->tokens > a->max_len)
    return DF_BAD_ARGUMENT;
  const int half = a->rotary_dim / 2;
  if (a->rotary_dim > kHd || half < 4 || (half & (half - 1))) return DF_BAD_ARGUMENT;
  if (a->ld_proj % 4 || a->k_col % 4 || a->v_col % 4 || (reinterpret_cast<uintptr_t>(a->proj) & 7) ||
      a->ld_proj < a->num_q_heads * 2 * kHd || a->k_col + a->num_kv_heads * kHd > a->ld_proj ||
      a->v_col + a->num_kv_heads * kHd > a->ld_proj)
    return DF_BAD_ARGUMENT;
  const int aligned = aligned16(a->proj) && a->ld_proj % 8 == 0 && a->k_col % 8 == 0 && a->v_col % 8 == 0 &&
                      aligned16(a->q_out) && aligned16(a->k_cache) && aligned16(a->v_cache);
  // Long prompts: four tokens to a workgroup, all their slots. Short ones need the workgroups: one
  // token and, where they still leave the chip's latency bare, as many slots as a workgroup has thread groups
  // (20 slots: 512 tokens 7.8 -> 6.7 us, 717 as long, 1500 12.5 -> 13.8 of recomputed angles; 10 slots: 1024
  // tokens 7.0 -> 6.5).
  const int slots = a->num_q_heads + a->num_kv_heads, per = a->tokens >= 2048 ? kQkTokens : 1;
  const int sper = (long)a->tokens * slots <= 12288 ? 8 : slots;
  hipLaunchKernelGGL(qk_rows_kernel, dim3((a->tokens + per - 1) / per, (slots + sper - 1) / sper), dim3(256), 0, stream, *a,
                     per, sper, aligned);
  DF_RETURN_LAUNCH_STATUS();
}

int df_attention_prefill(const DfAttnPrefillArgs* a, hipStream_t stream) {
  if (!a || !a->q || !a->k_cache || !a->v_cache || !a->gate || !a->out || a->tokens < 1 || a->pos0 < 0 ||
      a->pos0 + a->tokens > a->max_len || a->num_kv_heads < 1 || a->num_q_heads != 4 * a->num_kv_heads)
    return DF_BAD_ARGUMENT;
  if (!aligned16(a->q) || !aligned16(a->k_cache) || !aligned16(a->v_cache) || a->ld_out < a->num_q_heads * kHd ||
      a->gate_kind < 0 || a->gate_kind > 1)
    return DF_BAD_ARGUMENT;
  DfAttnPrefillArgs args = *a;
  // A scale of zero would turn a masked score into NaN. The smallest normal number leaves every
  // exp(s - m) of scores below 1e29 at 1, as zero does.
  if (args.scale == 0.0f) args.scale = FLT_MIN;
  int e = 0;
  const bool pow2 = args.scale > 0.0f && frexpf(args.scale, &e) == 0.5f;
  auto mult = [](const void* ptr, int ld, int align) {
    return (reinterpret_cast<uintptr_t>(ptr) % align) == 0 && ld % (align / 2) == 0;
  };
  const int flags = (pow2 ? kAtPow2Scale : 0) |
                    (mult(a->gate, a->ld_gate, 8) && a->gate_head_stride % 4 == 0 ? kAtVecGate : 0) |
                    (mult(a->out, a->ld_out, 8) ? kAtVecOut : 0);
  hipLaunchKernelGGL(attn_prefill_kernel, dim3((a->tokens + 31) / 32 * a->num_kv_heads), dim3(kAtThreads), kAtLds,
                     stream, args, flags);
  DF_RETURN_LAUNCH_STATUS();
}

}  // extern "C"
