// Group-128 int4 dequantise-GEMV for gfx950, with fused norm prologues and epilogues.
//
// Interchange format (reference kernels/tiled_gemv.py:242-288): packed uint8 [K/2][N],
// byte [j][n] = nibble(k=j) | nibble(k=j+K/2) << 4, each stored +8; scales [K/128][N].
// At install time the weight is repacked once into a device tiling:
//
//   block (t, g) = 1024 bytes for output columns 16t..16t+15 and k in group g
//                = [slot s 0..3][column c 0..15][16 bytes]
//   16 bytes     = 4 dwords d; dword d holds k = 128g + 32s + 8d + e, e = 0..7, with
//                  nibble e=2j at bits 4j..4j+3 and e=2j+1 at bits 16+4j..16+4j+3.
//   blocks are ordered [t][g], so one tile's whole K range is contiguous.
//
// Work split: a workgroup of 8 waves owns NT 16-column tiles; the 8/NT waves that share a
// tile split its K range, and their fp32 partials are summed in LDS in a fixed order. Each
// wave keeps up to 10 groups in flight, 1 KB of weights each. Each group
// is one fully coalesced 1 KB load (64 lanes x 16 B).
//
// Arithmetic is the reference's (kernels/visible_int4_head.py:187-199): every weight is
// dequantised to bf16((nibble - 8) * scale) -- (nibble - 8) * scale is exact in fp32 and
// the bf16 conversion is one round-to-nearest-even (v_cvt_pk_bf16_f32) -- and multiplied by
// the bf16 activations with fp32 accumulation on MFMA (v_mfma_f32_16x16x32_bf16; up to 16
// activation rows, the dequantised weights as the B operand). Only the summation order
// differs from the reference.
//
// When even that leaves too few waves, the K range is also split across workgroups
// (blockIdx.y); those write fp32 partials and a second kernel sums them in split order and
// runs the epilogue. Nothing uses atomics, so results are bit-identical run to run.
#include "common.h"
#include "deltaforge_hip.h"
#include "int4_block.h"

namespace df {

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
constexpr int kMaxRows = 16;
// Groups in flight per wave (kLongRow: kLongDepth), or half as many where a wave has no more: the
// decode's shapes have 4 to 10 groups a wave at 1 row and 9 to 20 at 16, so a range is one or two full
// sets with few repeats. Against 12 for all but the head's 8: down 9216 x 2560 6.6 -> 6.3 us at 1 row,
// head 71.2 -> 68.6, a 4096 x 2560 product (4 groups a wave) 6.1 -> 5.6.
constexpr int kDepth = 10;
constexpr int kNormChunks = 3;  // RMSNorm prologue: K <= kNormChunks * kThreads * 8 = 12288
constexpr int kRowChunks = 5;   // ... one wave per row when K <= kRowChunks * 64 * 8 = 2560
constexpr int kFewChunks = 2;   // ... K <= 1024
// A prologue's forms: one chunk of a row to a thread, several (norms of K > 4096), a wave to a row (more
// than 4 rows), the same for norms of K <= 1024
constexpr int kShortRow = 0, kLongRow = 1, kManyRows = 2, kManyShort = 3;
// kLongRow's chunks leave registers for 8 groups at its two workgroups a CU (10 spill, and cost 4 % at
// 16 rows of 4352 and 5120).
constexpr int kLongDepth = 8;
constexpr int kGemvLds = 100 * 1024;  // LDS bytes a workgroup may take

struct GemvSmem {
  int xs_ld;  // bf16 elements per LDS row of x
  int ybuf_off, red_off, total;
};

// LDS holds the activation rows plus, when rows < 16, one zero row that the MFMA lanes of
// absent rows read (so the inner loop has no divergent branch).
__host__ __device__ inline GemvSmem gemv_smem(int rows, int kx, int nt) {
  GemvSmem s;
  s.xs_ld = kx + 8;
  const int rows_alloc = rows < kMaxRows ? rows + 1 : rows;
  const int xs_bytes = ((rows_alloc * s.xs_ld * 2) + 15) & ~15;
  s.ybuf_off = xs_bytes;
  s.red_off = s.ybuf_off + (kWaves / nt) * rows * nt * kTileCols * 4;
  s.total = s.red_off + 64;
  return s;
}

// ---------------------------------------------------------------------------------------
// Prologues: this workgroup's K range of the bf16 activation rows, into LDS.
// ---------------------------------------------------------------------------------------

// A prologue's operands go into registers before the weight loads are issued: loads return in
// order, so a norm whose row was asked for after the weights would wait for all of them, and the
// sum, its barrier and the scaling (with the norm weight's own round trip after the sum) came on top
// of the stream instead of under it. What does not fit here is loaded in pro_finish.
// 1 row, weights in cache where they fit: in_proj 2560 x 12352 8.5 -> 6.9 us, gate|up 2560 x 18432
// 11.3 -> 10.5, head 2560 x 248320 74.3 -> 68.6; 16 rows: in_proj 13.0 -> 11.2, gate|up 15.0 -> 14.0; 8 rows
// of the head 117 -> 95 (with kDepth's change). The plain copy keeps its loads behind the weights':
// before them they delay the stream and have no sum to hide (down, 4 rows, 7.6 -> 8.1 us).
template <int PRO, int EPI, int FORM>
struct Pro {
  static constexpr bool WROWS = FORM >= kManyRows;
  static constexpr bool kNorm = PRO == DF_PRO_RMSNORM || PRO == DF_PRO_ADD_RMSNORM;
  static constexpr bool kTwo = PRO == DF_PRO_ADD_RMSNORM || PRO == DF_PRO_GATED_RMSNORM;
  // 16-byte chunks of the rows a thread takes early: the gated norm's of all rows, the norms' of one
  // row (a wave's row with WROWS); the plain copy takes none
  static constexpr int kNormX[4] = {1, kNormChunks, kRowChunks, kFewChunks};
  static constexpr int kX = kNorm ? kNormX[FORM] : WROWS ? 4 : 1;
  static constexpr int kEarly = kNorm && !WROWS ? 1 : kX;  // (4096 elements; longer rows' other chunks later)
  static constexpr int kRows = kNorm && WROWS && EPI != DF_EPI_LOGITS ? 2 : 1;  // rows a wave takes early
  uint4 x[kRows][kX], r[kTwo ? kRows : 1][kTwo ? kX : 1], w[PRO == DF_PRO_NONE ? 1 : kX];
};

template <int PRO, int EPI, int FORM>
DF_DEVICE void pro_issue(const DfInt4GemvArgs& p, Pro<PRO, EPI, FORM>& o, int k0, int kc) {
  using P = Pro<PRO, EPI, FORM>;
  constexpr bool WROWS = P::WROWS;
  const int tid = threadIdx.x;
  if constexpr (PRO == DF_PRO_NONE) return;
  if constexpr (P::kNorm) {
    const int first = WROWS ? tid & 63 : tid, step = WROWS ? 64 : kThreads, nchunks = p.K / 8;
#pragma unroll
    for (int i = 0; i < P::kRows; ++i) {
      const int m = WROWS ? (tid >> 6) + i * kWaves : 0;
#pragma unroll
      for (int j = 0; j < P::kEarly; ++j) {
        const int c = first + j * step;
        o.x[i][j] = make_uint4(0u, 0u, 0u, 0u);
        if constexpr (P::kTwo) o.r[i][j] = make_uint4(0u, 0u, 0u, 0u);
        if (c < nchunks && m < p.rows) {
          o.x[i][j] = load16(p.x + (size_t)m * p.ldx + c * 8);
          if constexpr (P::kTwo) o.r[i][j] = load16(p.x2 + (size_t)m * p.ldx2 + c * 8);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < P::kEarly; ++j) {
      const int k = (first + j * step) * 8;
      o.w[j] = make_uint4(0u, 0u, 0u, 0u);
      if (k >= k0 && k < k0 + kc) o.w[j] = load16(p.norm_w + k);
    }
  } else {
    const int per = kc / 8;
#pragma unroll
    for (int j = 0; j < P::kX; ++j) {
      const int u = tid + j * kThreads;
      if (u < p.rows * per) {
        const int m = u / per, k = k0 + (u - m * per) * 8;
        o.x[0][j] = load16(p.x + (size_t)m * p.ldx + k);
        o.r[0][j] = load16(p.x2 + (size_t)m * p.ldx2 + k);
        o.w[j] = load16(p.norm_w + (k % kGroup));
      }
    }
  }
}

// bf16(x + residual) of 8 elements (reference.py:735 feeding the next norm)
DF_DEVICE uint4 add8(const uint4& x, const uint4& r) {
  const uint32_t a[4] = {x.x, x.y, x.z, x.w}, b[4] = {r.x, r.y, r.z, r.w};
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    o[i] = pack_bf16(__uint_as_float(a[i] << 16) + __uint_as_float(b[i] << 16),
                     __uint_as_float(a[i] & 0xFFFF0000u) + __uint_as_float(b[i] & 0xFFFF0000u));
  return make_uint4(o[0], o[1], o[2], o[3]);
}
DF_DEVICE float sum_squares(const uint4& x, float ss) {
  const uint32_t a[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float lo = __uint_as_float(a[i] << 16), hi = __uint_as_float(a[i] & 0xFFFF0000u);
    ss += lo * lo;
    ss += hi * hi;
  }
  return ss;
}
// bf16((x r) (1 + w)) (reference.py:92-96)
DF_DEVICE uint4 scale8(const uint4& x, const uint4& w, float r) {
  const uint32_t a[4] = {x.x, x.y, x.z, x.w}, b[4] = {w.x, w.y, w.z, w.w};
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    o[i] = pack_bf16(__uint_as_float(a[i] << 16) * r * (1.0f + __uint_as_float(b[i] << 16)),
                     __uint_as_float(a[i] & 0xFFFF0000u) * r * (1.0f + __uint_as_float(b[i] & 0xFFFF0000u)));
  return make_uint4(o[0], o[1], o[2], o[3]);
}

template <int PRO, int EPI, int FORM>
DF_DEVICE void pro_finish(const DfInt4GemvArgs& p, Pro<PRO, EPI, FORM>& o, uint16_t* xs, int xs_ld, float* red, int k0,
                          int kc) {
  using P = Pro<PRO, EPI, FORM>;
  constexpr bool WROWS = P::WROWS;
  const int tid = threadIdx.x;
  if (p.rows < kMaxRows) {
    for (int kk = tid * 8; kk < kc; kk += kThreads * 8)
      *reinterpret_cast<uint4*>(xs + p.rows * xs_ld + kk) = make_uint4(0u, 0u, 0u, 0u);
  }
  if constexpr (PRO == DF_PRO_NONE) {
    for (int m = 0; m < p.rows; ++m) {
      const uint16_t* src = p.x + (size_t)m * p.ldx + k0;
      for (int kk = tid * 8; kk < kc; kk += kThreads * 8)
        *reinterpret_cast<uint4*>(xs + m * xs_ld + kk) = load16(src + kk);
    }
  } else if constexpr (P::kNorm) {
    // RMSNorm with the (1 + w) scale over the whole row; with ADD the row is first
    // bf16(x + residual). Few rows: every thread holds chunks of the row and the sum is the
    // workgroup's. WROWS, many rows: one wave per row (rows w, w + 8, ...), its sum reduced within
    // the wave, so rows proceed in parallel with no block-wide reduction; it holds more
    // registers, which costs more than it saves for one row. The two orders of the sum
    // differ only in fp32 rounding.
    const bool write_h = (PRO == DF_PRO_ADD_RMSNORM) && p.h_out && blockIdx.x == 0 && blockIdx.y == 0;
    const int first = WROWS ? tid & 63 : tid, step = WROWS ? 64 : kThreads, nchunks = p.K / 8;
    auto row = [&](int m, uint4 (&x)[P::kX], const uint4* r) {
      float ss = 0.0f;
#pragma unroll
      for (int j = 0; j < P::kX; ++j) {
        const int c = first + j * step;
        if constexpr (P::kTwo) x[j] = add8(x[j], r[j]);
        ss = sum_squares(x[j], ss);  // absent chunks are zero
        if (write_h && c < nchunks) *reinterpret_cast<uint4*>(p.h_out + (size_t)m * p.K + c * 8) = x[j];
      }
      ss = WROWS ? wave_sum(ss) : block_sum<kWaves>(ss, red);
      const float rs = 1.0f / sqrtf(ss / static_cast<float>(p.K) + p.eps);
#pragma unroll
      for (int j = 0; j < P::kX; ++j) {
        const int k = (first + j * step) * 8;
        if (k >= k0 && k < k0 + kc) *reinterpret_cast<uint4*>(xs + m * xs_ld + (k - k0)) = scale8(x[j], o.w[j], rs);
      }
    };
    if constexpr (P::kEarly < P::kX) {
#pragma unroll
      for (int j = P::kEarly; j < P::kX; ++j) {
        const int c = first + j * step, k = c * 8;
        o.x[0][j] = o.w[j] = make_uint4(0u, 0u, 0u, 0u);
        if constexpr (P::kTwo) o.r[0][j] = o.x[0][j];
        if (c < nchunks) {
          o.x[0][j] = load16(p.x + k);
          if constexpr (P::kTwo) o.r[0][j] = load16(p.x2 + k);
        }
        if (k >= k0 && k < k0 + kc) o.w[j] = load16(p.norm_w + k);
      }
    }
    int m = WROWS ? tid >> 6 : 0;
    const int next = WROWS ? kWaves : 1;
#pragma unroll
    for (int i = 0; i < P::kRows; ++i, m += next)
      if (m < p.rows) row(m, o.x[i], P::kTwo ? o.r[i] : nullptr);
    for (; m < p.rows; m += next) {
      uint4 x[P::kX], r[P::kX];
#pragma unroll
      for (int j = 0; j < P::kX; ++j) {
        const int c = first + j * step;
        x[j] = r[j] = make_uint4(0u, 0u, 0u, 0u);
        if (c < nchunks) {
          x[j] = load16(p.x + (size_t)m * p.ldx + c * 8);
          if constexpr (P::kTwo) r[j] = load16(p.x2 + (size_t)m * p.ldx2 + c * 8);
        }
      }
      row(m, x, r);
    }
  } else {
    const int per = kc / 8, total = p.rows * per;
    auto put = [&](int u, const uint4& x, const uint4& z, const uint4& w) {
      const int m = u / per, c = u - m * per;
      // one 128-group is one value head (reference.py:115-121): 16 consecutive lanes, 8 elements each
      float ss = sum_squares(x, 0.0f);
#pragma unroll
      for (int off = 1; off < 16; off <<= 1) ss += __shfl_xor(ss, off, 64);
      const float r = 1.0f / sqrtf(ss / 128.0f + p.eps);
      const uint32_t xw[4] = {x.x, x.y, x.z, x.w}, zw[4] = {z.x, z.y, z.z, z.w}, ww[4] = {w.x, w.y, w.z, w.w};
      uint32_t out[4];
#pragma unroll
      for (int e2 = 0; e2 < 4; ++e2) {
        float g[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float xe = bf2f(static_cast<uint16_t>(xw[e2] >> (16 * h)));
          const float t = round_bf(bf2f(static_cast<uint16_t>(ww[e2] >> (16 * h))) * round_bf(xe * r));
          g[h] = t * silu(bf2f(static_cast<uint16_t>(zw[e2] >> (16 * h))));
        }
        out[e2] = pack_bf16(g[0], g[1]);
      }
      *reinterpret_cast<uint4*>(xs + m * xs_ld + c * 8) = make_uint4(out[0], out[1], out[2], out[3]);
    };
#pragma unroll
    for (int j = 0; j < P::kX; ++j) {
      const int u = tid + j * kThreads;
      if (u < total) put(u, o.x[0][j], o.r[0][j], o.w[j]);
    }
    for (int u = tid + P::kX * kThreads; u < total; u += kThreads) {
      const int m = u / per, k = k0 + (u - m * per) * 8;
      put(u, load16(p.x + (size_t)m * p.ldx + k), load16(p.x2 + (size_t)m * p.ldx2 + k),
          load16(p.norm_w + (k % kGroup)));
    }
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------------------
// Epilogues over the `cols` columns x rows results of this workgroup (fp32, in LDS).
// ---------------------------------------------------------------------------------------

template <int EPI>
DF_DEVICE void gemv_epilogue(const DfInt4GemvArgs& p, const float* y, int col0, int cols) {
  for (int e = threadIdx.x; e < p.rows * cols; e += blockDim.x) {
    const int m = e / cols, c = e % cols;
    const float v = y[m * cols + c];
    if constexpr (EPI == DF_EPI_STORE || EPI == DF_EPI_LOGITS) {
      p.out[(size_t)m * p.ldo + col0 + c] = f2bf(v);
    } else if constexpr (EPI == DF_EPI_RESIDUAL) {
      // bf16(residual + bf16(y)) (reference.py:730, 735). In place is allowed.
      const size_t at = (size_t)m * p.ldo + col0 + c;
      p.out[at] = f2bf(bf2f(p.res[at]) + round_bf(v));
    } else {  // DF_EPI_SWIGLU: 16-column gate / up tiles alternate
      if ((c & 16) == 0) {
        const float g = round_bf(v);
        const float u = round_bf(y[m * cols + c + 16]);
        const int oc = (col0 + c) / 32 * 16 + (c & 15);
        p.out[(size_t)m * p.ldo + oc] = f2bf(round_bf(silu(g)) * u);
      }
    }
  }
}

template <int PRO, int EPI, int NT, int FORM, int DEPTH>
__global__ __launch_bounds__(kThreads, FORM >= kManyRows || PRO == DF_PRO_NONE ? 2 : 4)
void w4_gemv_kernel(DfInt4GemvArgs p) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int KS = kWaves / NT;
  constexpr int COLS = NT * kTileCols;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tsub = wave % NT, kpart = wave / NT;
  const int G = p.K / kGroup;
  const int gx0 = blockIdx.y * p.groups_per_split;
  const int ngx = min(p.groups_per_split, G - gx0);
  const int per = (ngx + KS - 1) / KS;
  const int g_lo = min(kpart * per, ngx), g_hi = min(g_lo + per, ngx);
  const GemvSmem L = gemv_smem(p.rows, ngx * kGroup, NT);
  uint16_t* xs = reinterpret_cast<uint16_t*>(smem);
  float* ybuf = reinterpret_cast<float*>(smem + L.ybuf_off);
  float* red = reinterpret_cast<float*>(smem + L.red_off);

  const int tile = blockIdx.x * NT + tsub;
  const unsigned char* wp = p.w + ((size_t)tile * G + gx0) * kBlockBytes + lane * 16;
  const uint16_t* sp = p.s + ((size_t)tile * G + gx0) * kTileCols + (lane & 15);

  // The prologue's operands, then the first groups of weights, all in flight at once; the
  // prologue then waits for its own loads only (no branch around the weights', which would make
  // the wait one for everything). Refills are clamped to the last group of the range (a
  // repeat read of a cached block) so the pipeline is branch-free; a wave without groups reads one.
  Pro<PRO, EPI, FORM> pro;
  pro_issue<PRO, EPI, FORM>(p, pro, gx0 * kGroup, ngx * kGroup);
  const int g_last = max(g_hi - 1, 0);
  uint4 wb[DEPTH];
  uint16_t sb[DEPTH];
#pragma unroll
  for (int u = 0; u < DEPTH; ++u) {
    const int g = min(g_lo + u, g_last);
    wb[u] = load16(wp + (size_t)g * kBlockBytes);
    sb[u] = sp[g * kTileCols];
  }

  pro_finish<PRO, EPI, FORM>(p, pro, xs, L.xs_ld, red, gx0 * kGroup, ngx * kGroup);

  const int col = lane & 15;   // A row, B/C column, scale column
  const int slot = lane >> 4;  // K slot of A and B; C row block
  const uint16_t* xrow = xs + min(col, p.rows) * L.xs_ld + slot * 32;  // absent rows read zeros
  df_f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  const DqK K = dq_consts();

  auto group_mac = [&](const uint4 wv, const uint16_t sraw, const int g) {
    const GroupScale gs = group_scale(sraw);
    const uint32_t words[4] = {wv.x, wv.y, wv.z, wv.w};
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const uint4 bw = dequant8(words[d], gs, K);
      const uint4 aw = *reinterpret_cast<const uint4*>(xrow + g * kGroup + d * 8);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(df_bf16x8, aw),
                                                    __builtin_bit_cast(df_bf16x8, bw), acc, 0, 0, 0);
    }
  };

  int g0 = g_lo;
  for (; g0 + DEPTH < g_hi; g0 += DEPTH) {
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) {
      const uint4 wv = wb[u];
      const uint16_t sv = sb[u];
      const int gn = min(g0 + u + DEPTH, g_last);
      wb[u] = load16(wp + (size_t)gn * kBlockBytes);
      sb[u] = sp[gn * kTileCols];
      group_mac(wv, sv, g0 + u);
    }
  }
  // Tail: the remaining groups are already in wb[0 .. g_hi - g0).
#pragma unroll
  for (int u = 0; u < DEPTH; ++u) {
    if (g0 + u < g_hi) group_mac(wb[u], sb[u], g0 + u);
  }

  // K parts of a tile -> LDS, then a fixed-order sum.
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = slot * 4 + i;
    if (m < p.rows) ybuf[(kpart * p.rows + m) * COLS + tsub * kTileCols + col] = acc[i];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < p.rows * COLS; e += kThreads) {
    float v = ybuf[e];
#pragma unroll
    for (int k = 1; k < KS; ++k) v += ybuf[k * p.rows * COLS + e];
    ybuf[e] = v;
  }
  __syncthreads();
  const int col0 = blockIdx.x * COLS;
  if (gridDim.y == 1) {
    gemv_epilogue<EPI>(p, ybuf, col0, COLS);
  } else {
    for (int e = threadIdx.x; e < p.rows * COLS; e += kThreads) {
      const int m = e / COLS, c = e % COLS;
      p.part[((size_t)blockIdx.y * p.rows + m) * p.N + col0 + c] = ybuf[e];
    }
  }
}

// Sum of the cross-workgroup K splits (in split order) + the epilogue. 64 columns per block.
template <int EPI>
__global__ __launch_bounds__(256) void w4_reduce_kernel(DfInt4GemvArgs p) {
  __shared__ float y[kMaxRows * 64];
  const int col0 = blockIdx.x * 64;
  for (int e = threadIdx.x; e < p.rows * 64; e += 256) {
    const int m = e / 64, c = e % 64;
    const float* src = p.part + (size_t)m * p.N + col0 + c;
    const size_t stride = (size_t)p.rows * p.N;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    int s = 0;
    for (; s + 4 <= p.ksplit; s += 4) {
      const float a0 = src[(s + 0) * stride], a1 = src[(s + 1) * stride];
      const float a2 = src[(s + 2) * stride], a3 = src[(s + 3) * stride];
      v[0] = ((v[0] + a0) + a1) + a2;
      v[0] = v[0] + a3;
    }
    for (; s < p.ksplit; ++s) v[0] += src[s * stride];
    y[e] = v[0];
  }
  __syncthreads();
  gemv_epilogue<EPI>(p, y, col0, 64);
}

// ---------------------------------------------------------------------------------------
// Install-time repack and the bit-exact dequant (debug / parity entry point).
// ---------------------------------------------------------------------------------------

__global__ void w4_repack_kernel(const uint8_t* __restrict__ packed, const uint16_t* __restrict__ scale,
                                 int K, int N, uint32_t* __restrict__ wt, uint16_t* __restrict__ st) {
  const int G = K / kGroup;
  const size_t total = (size_t)(N / kTileCols) * G * 256;
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const int d = idx & 3, lane = (idx >> 2) & 63;
  const size_t tg = idx >> 8;
  const int g = tg % G, t = tg / G;
  const int s = lane >> 4, c = lane & 15, n = t * kTileCols + c;
  const int half = K / 2;
  uint32_t word = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int k = g * kGroup + s * 32 + d * 8 + e;
    const uint32_t byte = k < half ? packed[(size_t)k * N + n] : packed[(size_t)(k - half) * N + n];
    const uint32_t nib = k < half ? (byte & 15u) : (byte >> 4);
    const int pos = (e & 1) ? 16 + 4 * (e >> 1) : 4 * (e >> 1);
    word |= nib << pos;
  }
  wt[idx] = word;
  if (s == 0 && d == 0) st[tg * kTileCols + c] = scale[(size_t)g * N + n];
}

// W[k][n] = bf16((nibble - 8) * scale), read back from the tiled layout with the GEMV's own
// dequant routine: proves the repack and the dequant arithmetic together (reference
// tiled_gemv.py:281-288 then .to(bf16)).
__global__ void w4_dequant_kernel(const uint32_t* __restrict__ wt, const uint16_t* __restrict__ st, int K,
                                  int N, uint16_t* __restrict__ out) {
  const int G = K / kGroup;
  const size_t total = (size_t)(N / kTileCols) * G * 256;
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const int d = idx & 3, lane = (idx >> 2) & 63;
  const size_t tg = idx >> 8;
  const int g = tg % G, t = tg / G;
  const int s = lane >> 4, c = lane & 15, n = t * kTileCols + c;
  const uint4 q = dequant8(wt[idx], group_scale(st[tg * kTileCols + c]), dq_consts());
  const uint32_t pairs[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int k = g * kGroup + s * 32 + d * 8 + e;
    out[(size_t)k * N + n] = static_cast<uint16_t>(pairs[e >> 1] >> (16 * (e & 1)));
  }
}

template <int PRO, int EPI, int NT>
static hipError_t launch_gemv(const DfInt4GemvArgs& a, hipStream_t stream) {
  const int G = a.K / kGroup;
  const int gps = a.groups_per_split;
  const GemvSmem L = gemv_smem(a.rows, min(gps, G) * kGroup, NT);
  dim3 grid(a.N / (NT * kTileCols), a.ksplit);
  constexpr bool kNorm = PRO == DF_PRO_RMSNORM || PRO == DF_PRO_ADD_RMSNORM;
  const int per = (min(gps, G) + kWaves / NT - 1) / (kWaves / NT);  // groups a wave
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(kThreads), L.total, stream, a); };
  [&] {
    if constexpr (kNorm)
      if (a.rows > 4 && a.K <= kFewChunks * 64 * 8) return go(w4_gemv_kernel<PRO, EPI, NT, kManyShort, kDepth>);
    if constexpr (PRO != DF_PRO_NONE)
      if (a.rows > 4 && (!kNorm || a.K <= kRowChunks * 64 * 8)) return go(w4_gemv_kernel<PRO, EPI, NT, kManyRows, kDepth>);
    if constexpr (kNorm)
      if (a.K > kThreads * 8) return go(w4_gemv_kernel<PRO, EPI, NT, kLongRow, kLongDepth>);
    if (per <= kDepth / 2) return go(w4_gemv_kernel<PRO, EPI, NT, kShortRow, kDepth / 2>);
    go(w4_gemv_kernel<PRO, EPI, NT, kShortRow, kDepth>);
  }();
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || a.ksplit == 1) return e;
  hipLaunchKernelGGL((w4_reduce_kernel<EPI>), dim3(a.N / 64), dim3(256), 0, stream, a);
  return hipGetLastError();
}

template <int PRO, int EPI>
static hipError_t launch_nt(const DfInt4GemvArgs& a, hipStream_t stream) {
  switch (a.tiles_per_workgroup) {
    case 1: return launch_gemv<PRO, EPI, 1>(a, stream);
    case 2: return launch_gemv<PRO, EPI, 2>(a, stream);
    case 4: return launch_gemv<PRO, EPI, 4>(a, stream);
    case 8: return launch_gemv<PRO, EPI, 8>(a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace df

using namespace df;

extern "C" {

size_t df_int4_gemv_workspace_bytes(int rows, int N, int ksplit) {
  return ksplit > 1 ? (size_t)ksplit * rows * N * sizeof(float) : 0;
}

int df_int4_gemv_plan(int rows, int K, int N, int epilogue, int target_waves, int* tiles_per_workgroup,
                      int* ksplit, int* groups_per_split, size_t* workspace_bytes) {
  if (rows < 1 || rows > kMaxRows || K % 256 || N % 64 || K <= 0 || !tiles_per_workgroup || !ksplit ||
      !groups_per_split || !workspace_bytes)
    return DF_BAD_ARGUMENT;
  if (target_waves <= 0) target_waves = 2048;
  const int G = K / kGroup;
  const int tiles = N / kTileCols;
  // Widest workgroup (most tiles, least K splitting) that divides the tiles and still
  // reaches the wave target; SwiGLU pairs a gate tile with an up tile, so at least 2.
  const int min_nt = epilogue == DF_EPI_SWIGLU ? 2 : 1;
  // A workgroup's LDS (the activation rows of its K range, partial sums) must fit kGemvLds of
  // gfx950's 160 KB: 16 rows of K = 2560 fit, so that shape needs no K split, partials or
  // reduce launch.
  auto split_for = [&](int nt_, int& gps_, int& ks_) {
    gps_ = G;
    while (gps_ > 1 && gemv_smem(rows, gps_ * kGroup, nt_).total > kGemvLds) --gps_;
    ks_ = (G + gps_ - 1) / gps_;
    gps_ = (G + ks_ - 1) / ks_;
  };
  int nt = 8;
  while (nt > min_nt && (tiles % nt || (tiles / nt) * kWaves < target_waves)) nt /= 2;
  if (rows > 4) {
    // Many rows: every workgroup stages all rows of its K range, so fewer, wider workgroups
    // stage them fewer times. Take the most workgroups up to one per CU (measured best at 8
    // and 16 rows: gate|up 2560 x 18432 in 144 workgroups of 8 tiles, 17.7 against 23.9 us at
    // 16 rows and 16.2 against 20.3 us at 8 rows with 288 of 4; down 9216 x 2560 in 160
    // workgroups, 13.8 against 20.7 us at 16 rows (4 tiles x 4 K splits, not 1 tile) and 14.0
    // against 16.1 us at 8 rows (2 tiles x 2 splits)).
    int best = 0, best_wgs = 0;
    for (int c = 8; c >= min_nt; c /= 2) {
      if (tiles % c) continue;
      int gps_, ks_;
      split_for(c, gps_, ks_);
      const int wgs = (tiles / c) * ks_;
      if (wgs <= 256 && wgs > best_wgs) best = c, best_wgs = wgs;
    }
    if (best) nt = best;
  }
  int gps, ks;
  split_for(nt, gps, ks);
  *tiles_per_workgroup = nt;
  *ksplit = ks;
  *groups_per_split = gps;
  *workspace_bytes = df_int4_gemv_workspace_bytes(rows, N, ks);
  return DF_OK;
}

int df_int4_gemv(const DfInt4GemvArgs* args, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (!args) return DF_BAD_ARGUMENT;
  DfInt4GemvArgs a = *args;
  const int G = a.K / kGroup;
  if (a.rows < 1 || a.rows > kMaxRows || a.K <= 0 || a.K % 256 || a.N <= 0 || a.N % 64 || !a.w || !a.s || !a.x ||
      !a.out)
    return DF_BAD_ARGUMENT;
  const int nt = a.tiles_per_workgroup;
  if (nt != 1 && nt != 2 && nt != 4 && nt != 8) return DF_BAD_ARGUMENT;
  if ((a.N / kTileCols) % nt) return DF_BAD_ARGUMENT;
  if (a.ksplit < 1 || a.groups_per_split < 1 || (long)a.ksplit * a.groups_per_split < G ||
      (long)(a.ksplit - 1) * a.groups_per_split >= G)
    return DF_BAD_ARGUMENT;
  if (a.ldx < a.K || a.ldx % 8) return DF_BAD_ARGUMENT;
  if (a.epilogue == DF_EPI_SWIGLU && (nt < 2 || a.N % 32)) return DF_BAD_ARGUMENT;
  const int out_cols = a.epilogue == DF_EPI_SWIGLU ? a.N / 2 : a.N;
  if (a.ldo < out_cols) return DF_BAD_ARGUMENT;
  if (gemv_smem(a.rows, min(a.groups_per_split, G) * kGroup, nt).total > kGemvLds) return DF_BAD_ARGUMENT;
  if ((a.prologue == DF_PRO_ADD_RMSNORM || a.prologue == DF_PRO_GATED_RMSNORM) && !a.x2) return DF_BAD_ARGUMENT;
  if (a.prologue != DF_PRO_NONE && !a.norm_w) return DF_BAD_ARGUMENT;
  if (a.epilogue == DF_EPI_RESIDUAL && !a.res) return DF_BAD_ARGUMENT;
  if (reinterpret_cast<uintptr_t>(a.x) % 16 || reinterpret_cast<uintptr_t>(a.w) % 16) return DF_BAD_ARGUMENT;
  // The norm prologues read x2 and the norm weight with 16-byte loads.
  if (a.prologue != DF_PRO_NONE && reinterpret_cast<uintptr_t>(a.norm_w) % 16) return DF_BAD_ARGUMENT;
  if ((a.prologue == DF_PRO_ADD_RMSNORM || a.prologue == DF_PRO_GATED_RMSNORM) &&
      (reinterpret_cast<uintptr_t>(a.x2) % 16 || a.ldx2 % 8))
    return DF_BAD_ARGUMENT;
  if ((a.prologue == DF_PRO_RMSNORM || a.prologue == DF_PRO_ADD_RMSNORM) && a.K > kNormChunks * kThreads * 8)
    return DF_BAD_ARGUMENT;
  if (a.h_out && reinterpret_cast<uintptr_t>(a.h_out) % 16) return DF_BAD_ARGUMENT;
  if (a.ksplit > 1) {
    if (!workspace || workspace_bytes < df_int4_gemv_workspace_bytes(a.rows, a.N, a.ksplit))
      return DF_WORKSPACE_TOO_SMALL;
    a.part = reinterpret_cast<float*>(workspace);
  }
  hipError_t e = hipErrorInvalidValue;
#define DF_GEMV_CASE(PRO, EPI) \
  if (a.prologue == PRO && a.epilogue == EPI) e = launch_nt<PRO, EPI>(a, stream);
  DF_GEMV_CASE(DF_PRO_NONE, DF_EPI_STORE)
  DF_GEMV_CASE(DF_PRO_NONE, DF_EPI_RESIDUAL)
  DF_GEMV_CASE(DF_PRO_NONE, DF_EPI_SWIGLU)
  DF_GEMV_CASE(DF_PRO_RMSNORM, DF_EPI_STORE)
  DF_GEMV_CASE(DF_PRO_RMSNORM, DF_EPI_SWIGLU)
  DF_GEMV_CASE(DF_PRO_RMSNORM, DF_EPI_LOGITS)
  DF_GEMV_CASE(DF_PRO_ADD_RMSNORM, DF_EPI_STORE)
  DF_GEMV_CASE(DF_PRO_ADD_RMSNORM, DF_EPI_LOGITS)
  DF_GEMV_CASE(DF_PRO_GATED_RMSNORM, DF_EPI_STORE)
  DF_GEMV_CASE(DF_PRO_GATED_RMSNORM, DF_EPI_RESIDUAL)
#undef DF_GEMV_CASE
  if (e == hipErrorInvalidValue) return DF_BAD_ARGUMENT;
  return e == hipSuccess ? DF_OK : DF_LAUNCH_FAILED;
}

int df_int4_repack(const uint8_t* packed, const uint16_t* scale, int K, int N, uint8_t* w_tiled,
                   uint16_t* s_tiled, hipStream_t stream) {
  if (!packed || !scale || !w_tiled || !s_tiled || K % 256 || N % kTileCols || K <= 0 || N <= 0)
    return DF_BAD_ARGUMENT;
  const size_t total = (size_t)(N / kTileCols) * (K / kGroup) * 256;
  hipLaunchKernelGGL(w4_repack_kernel, dim3((total + 255) / 256), dim3(256), 0, stream, packed, scale, K, N,
                     reinterpret_cast<uint32_t*>(w_tiled), s_tiled);
  DF_RETURN_LAUNCH_STATUS();
}

int df_int4_dequant(const uint8_t* w_tiled, const uint16_t* s_tiled, int K, int N, uint16_t* out,
                    hipStream_t stream) {
  if (!w_tiled || !s_tiled || !out || K % 256 || N % kTileCols || K <= 0 || N <= 0) return DF_BAD_ARGUMENT;
  const size_t total = (size_t)(N / kTileCols) * (K / kGroup) * 256;
  hipLaunchKernelGGL(w4_dequant_kernel, dim3((total + 255) / 256), dim3(256), 0, stream,
                     reinterpret_cast<const uint32_t*>(w_tiled), s_tiled, K, N, out);
  DF_RETURN_LAUNCH_STATUS();
}

}  // extern "C"
