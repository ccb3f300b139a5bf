// Prompt-block contraction of q4nx tiles on the matrix cores (gfx950), weights and activations
// as fp16 operands: Y[m][n] = R[m][n] + sum_k W[n][k] X[m][k], and [gate, up, SwiGLU].
//
// Replaces, for prompt blocks, the torch fallback that reference/npu.py:118-122, 138-140 takes
// for more than one row.
//
// Arithmetic, q4. Per column n and 32-K group g, with the Q4_1 factoring of granite_gemv.h:19-29 and
// an offset o[n][g] near 7.5 d[n][g],
//   y[m][n] = sum_k (d[n][g] c[n][k] - o[n][g]) x[m][k] + sum_g u[n][g] S[m][g]
//   S[m][g] = sum_{k in g} x[m][k]     u[n][g] = m[n][g] + o[n][g]
// A code's four bits under a fixed fp16 exponent are the value B + c (B = 1024 for a low nibble,
// 64 for a high one), so d c - o is one fp16 multiply-add, d (B + c) + A with A the fp16 value
// of -(B + 7.5) d. d has 8 significant bits and A is a multiple of at most 128 of their last
// place, so the result is a multiple of that place below 2^11 of them: exact. A's own rounding
// is in o = -(B d + A), hence in u. x is an exact fp16 value under a power of two per row, d
// under one per column (what that leaves out: below, "Range"). The first sum is therefore v_mfma_f32_16x16x32_f16 alone, one per 16x16 block and
// group with exact products: no per-group scale on the VALU, and no large offset to cancel
// afterwards. The second sum is a contraction over the groups (32 per MFMA), S and u each in two
// fp16 terms (the product of the two low terms, 2^-22, is left out). A one-hot row still gives
// the float32 dequantised column bit for bit, as long as u fits its two terms: |m| down to 2^-14 of
// 8 |d|, below that it is kept to 2^-23 of 8 |d| (in fp32, m - 16 d was kept to 2^-24 of 16 |d|). The
// 128-row tile adds the two terms one after the other to the codes' sum: one more rounding, none
// where m = -8 d.
//
// Arithmetic, q8: y[m][n] = sum_g s[n][g] sum_{k in g} q[n][k] x[m][k]. s q has 15 bits, more than
// one fp16 value holds, so the operand is the code alone (q = (1152 + q) - 1152, the byte under a
// fixed exponent less a constant) and one MFMA from zero per 16x16 block and group gives the
// inner sum, which four FMAs per lane scale into the total. (Two MFMAs on s = s1 + s2, four bits
// each, and no FMA took 555 us for 512 rows of 248320 x 1024, this 406.) x and s under powers of two
// as above.
//
// Range. Under a row's power of two an entry of x is exact down to 2^-31 of the row's largest and
// is rounded at 2^-39 of it below; d is exact down to 2^-22 of what the column's largest |m| and 8
// |d| allow (d below 2^5, |m| below 2^8), S and u are kept to 2^-23 of themselves and 2^-33, 2^-39
// of the largest. All of that is below the fp32 rounding of a sum to which the large groups
// contribute: 16 d x of some group is within 2^-10 of the largest d times the largest x as soon as
// either the row's or the column's groups all lie within 2^-10 of its largest one. The pre-pass marks
// the rows and the columns of which that is not so, and a workgroup that has both adds up its tile
// on bf16 operands with one fp32 scale per group instead (exact_tile): no loss at any range. (Marking
// takes 0.3 to 0.4 us of the pre-pass, looking 0.3 to 3 us of the contraction.)
//
// What bounds it: see pq_kernel.
#include "common.h"
#include "gemm.h"
#include "gemm_fmt.h"

namespace q4nx {

namespace {

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef unsigned short us2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x4_t mfma_f16(const u32x4_t& a, const u32x4_t& b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t pk_max_u16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(us2_t, a),
                                                                __builtin_bit_cast(us2_t, b)));
}
__device__ __forceinline__ uint32_t pk_min_u16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(us2_t, a),
                                                                __builtin_bit_cast(us2_t, b)));
}
__device__ __forceinline__ uint32_t pk_add_u16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(us2_t, a) + __builtin_bit_cast(us2_t, b));
}
// two fp32 values as packed fp16, towards zero (one instruction); to nearest
__device__ __forceinline__ uint32_t pk_f16z(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(lo, hi));
}
__device__ __forceinline__ uint32_t pk_f16(float lo, float hi) {
  return h2_bits(half2_t{(_Float16)lo, (_Float16)hi});
}
// v = hi + lo to 2^-22: the two terms of a pair of values as packed fp16 words
__device__ __forceinline__ void split2(float v0, float v1, uint32_t& hi, uint32_t& lo) {
  const half2_t h = {(_Float16)v0, (_Float16)v1};
  const half2_t r = {(_Float16)(v0 - (float)h.x), (_Float16)(v1 - (float)h.y)};
  hi = h2_bits(h);
  lo = h2_bits(r);
}

constexpr int kPqChunkTiles = 4;      // K-tiles (32 groups) per minimum-term contraction
// LDS bytes of half a tile: codes of 128 K, then their scales
template <int KIND>
constexpr int kPqHalf = KIND == 4 ? 2560 : 4352;
constexpr int kPqXTop = 141;          // 141 - exponent field: the row's largest x in [2^14, 2^15)
constexpr int kPqWTop = 135;          // |u| of a column below 2^9, its 8 |d| below 2^8
constexpr int kPqSum = 6;             // S is kept 2^6 below its row's scale, u 2^6 above its column's
constexpr int kPqSTop = 131;          // a q8 column's largest scale in [2^4, 2^5)
constexpr float kPqLow = -1031.5f, kPqHigh = -71.5f;   // A / d of the low and the high nibbles
constexpr int kPqSpan = 10;           // a "wide" row or column: a group below 2^-10 of its largest
constexpr int kPqSlack = 64 << 10;    // bytes after x that steps past its end read (never used)

// The pre-pass's output (workspace), all in the order the contraction's operands take it: x as
// fp16, its group sums, every column's u, and the powers of two.
struct PqX {
  u32x4_t* xt;      // [m-tile][32-K step][row % 16][k / 8 ^ row / 2 % 4]: 8 fp16 values; after
                    // the steps, two of sums (hi, lo) per chunk of 32 groups, k the group
  u32x4_t* u;       // [tensor][tile-row][chunk][hi, lo][even, odd column][lane]
  uint2* scale;     // [tensor][tile-row][group][lane % 16]: fp16 d of the even and odd column, A
                    // (q4 only)
  int* xshift;      // [row]: the power of two of x, times two, + 1 for a wide row
  int* wshift;      // [tensor][column]: that of d, A and u (q8: of s), + 1 for a wide column
  uint16_t* xe;     // with an RMSNorm whose rows the caller does not take: [row][K], wide rows only
  const uint16_t* exact;    // bf16 rows for exact_tile, exact_stride entries apart: all of them,
  int64_t exact_stride;     // or the wide ones
  bool exact_all;
  int m_blocks, c_groups;   // the launch's row blocks, its groups of columns
  bool rows_first;  // the order of its workgroups: row blocks first, within an eighth of them
};

// The larger of each lane's value and its DPP / permlane partner's, over the whole wave
template <int CTRL>
__device__ __forceinline__ uint32_t umax_dpp(uint32_t v) {
  const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
  return pk_max_u16(v, o);
}
__device__ __forceinline__ uint32_t rows_max(uint32_t v) {    // across the four rows of 16 lanes
  const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = pk_max_u16(a[0], a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return pk_max_u16(b[0], b[1]);
}

__device__ __forceinline__ uint32_t rows_min(uint32_t v) {
  const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = pk_min_u16(a[0], a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return pk_min_u16(b[0], b[1]);
}
// the smallest over the wave of 32-bit values that the four lanes of a quad share
template <int CTRL>
__device__ __forceinline__ uint32_t umin_dpp(uint32_t v) {
  return min(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ uint32_t quads_min(uint32_t v) {
  v = umin_dpp<kDppRor8>(umin_dpp<kDppHalfMirror>(v));
  const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = min(a[0], a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return min(b[0], b[1]);
}
// whether the smallest of a row's or column's groups lies more than kPqSpan binary orders below
// its largest (bf16 exponent fields; 0 is the smallest normal numbers' binade or less, which the
// largest power of two lifts whole into range)
__device__ __forceinline__ int span_wide(int largest, int smallest) {
  return max(largest, 1) - max(smallest, 1) > kPqSpan;
}

// 2^e as a float, -126 <= e <= 127
__device__ __forceinline__ float exp2i(int e) { return __int_as_float((e + 127) << 23); }

// chunks of 32 groups of the minimum term (q8 has none)
template <int KIND>
__host__ __device__ constexpr int pq_chunks(int k_t) {
  return KIND == 4 ? (k_t + kPqChunkTiles - 1) / kPqChunkTiles : 0;
}

// One row of x per NT threads (a workgroup, or one wave of it): x (or RMSNorm of the fp32 residual,
// to bf16 first, as every consumer rounds it) to fp16 under the row's power of two, the sums per
// 32-K group, and whether the row is wide (a wide row of a norm is also kept as bf16). Each thread
// keeps C chunks of 8 entries (K <= 8 NT C; longer rows are read again for the second
// pass). Every load is unconditional, through a buffer resource over the row: entries past its
// end read zeros. Rows past m_rows stay unwritten: a row of an operand reaches its own row of
// the result only. The code is kept short: a wave runs it once, so its instruction fetches are
// not amortised (eight rows per workgroup, a wave each with up to 16 chunks, took 2.5 times as
// long).
template <int KIND, bool NORM, int C, int NT>
__device__ __forceinline__ void prep_row(const GemmArgs& a, const PqX& o, int row,
                                         float* __restrict__ sg, uint32_t* __restrict__ smx) {
  const int tid = threadIdx.x & (NT - 1), l = tid & 63, wave = tid >> 6;
  auto meet = [] {                              // of the row's threads
    if constexpr (NT > 64) __syncthreads();
    else __builtin_amdgcn_wave_barrier();
  };
  const int K = a.k_t * kTileK, n_q = K / 8;
  const int n_ch = pq_chunks<KIND>(a.k_t);
  auto ld = [](__amdgpu_buffer_rsrc_t r, uint32_t off) {
    const v4i_t t = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
    return u32x4_t{(uint32_t)t.x, (uint32_t)t.y, (uint32_t)t.z, (uint32_t)t.w};
  };
  const __amdgpu_buffer_rsrc_t xr =
      NORM ? make_rsrc(a.hres + (int64_t)row * a.x_stride, (uint32_t)K * 4u)
           : make_rsrc(a.x + (int64_t)row * a.x_stride, (uint32_t)K * 2u);
  u32x4_t v[C];
  uint32_t mx = 0, mn = ~0u;                    // the row's largest entry; the smallest group's
  auto see = [&](const u32x4_t& w) {            // largest, less 1 (a group of zeros: none)
    uint32_t g = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) g = pk_max_u16(g, w[j] & 0x7FFF7FFFu);
    mx = pk_max_u16(mx, g);
    g = umax_dpp<kDppXor2>(umax_dpp<kDppXor1>(g));
    mn = min(mn, max(g >> 16, g & 0xFFFFu) - 1u);
  };
  if constexpr (NORM) {
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(a.norm_w, (uint32_t)K * 2u);
    const int n_ss = K / kSsqRows;              // <= 512
    u32x4_t h0[C], h1[C], w[C];
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const uint32_t q = tid + NT * i;
      h0[i] = ld(xr, 32 * q);
      h1[i] = ld(xr, 32 * q + 16);
      w[i] = ld(wr, 16 * q);
    }
    float4 sq[2];
    ssq_load<2>(a.ssq_in + (int64_t)row * n_ss, l, n_ss, sq);
    const float inv = rms_inv(wave_sum(ssq_lane_sum<2>(sq, l, n_ss)), K, a.eps);
#pragma unroll
    for (int i = 0; i < C; ++i) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const u32x4_t& h = j < 2 ? h0[i] : h1[i];
        const int e = (j & 1) * 2;
        v[i][j] = pack_bf16x2((__uint_as_float(h[e]) * inv) * bf16lo(w[i][j]),
                              (__uint_as_float(h[e + 1]) * inv) * bf16hi(w[i][j]));
      }
      const int q = tid + NT * i;
      if (a.xn_out != nullptr && q < n_q)
        *(u32x4_t*)(a.xn_out + (int64_t)row * a.x_stride + 8 * q) = v[i];
    }
  } else {
#pragma unroll
    for (int i = 0; i < C; ++i) v[i] = ld(xr, 16 * (tid + NT * i));
    for (int q = tid + NT * C; q < n_q; q += NT) see(ld(xr, 16 * q));
  }
#pragma unroll
  for (int i = 0; i < C; ++i) see(v[i]);
  mx = umax_dpp<kDppXor1>(mx);
  mx = umax_dpp<kDppXor2>(mx);
  mx = umax_dpp<kDppHalfMirror>(mx);
  mx = rows_max(umax_dpp<kDppRor8>(mx));
  mn = quads_min(mn);
  if constexpr (NT > 64) {
    if (l == 0) smx[2 * wave] = mx, smx[2 * wave + 1] = mn;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) mx = pk_max_u16(mx, smx[2 * i]), mn = min(mn, smx[2 * i + 1]);
  }
  // exponent field of the row's largest entry; a row with an infinity or a NaN is left
  // unscaled (its sums carry the NaN into every output of the row)
  const int ex = (int)max(mx >> 16, mx & 0xFFFFu) >> 7;
  const int sh = ex == 255 ? 0 : min(kPqXTop - max(ex, 1), 127);
  const float sc = exp2i(sh);
  const int wide = ex < 255 && mn != ~0u && span_wide(ex, (int)(mn + 1) >> 7);
  if (tid == 0) o.xshift[row] = 2 * sh + wide;
  if constexpr (NORM) {
    if (wide && a.xn_out == nullptr) {
#pragma unroll
      for (int i = 0; i < C; ++i) {
        const int q = tid + NT * i;
        if (q < n_q) *(u32x4_t*)(o.xe + (size_t)row * K + 8 * q) = v[i];
      }
    }
  }
  const int r16 = row & 15, swz = (r16 >> 1) & 3;
  u32x4_t* xt = o.xt + (size_t)(row >> 4) * (a.k_t * 8 + n_ch * 2) * 64 + r16 * 4;
  u32x4_t* sm = xt + (size_t)a.k_t * 8 * 64;
  for (int i0 = 0; i0 * 8 * NT < K; i0 += C) {
    if (KIND == 4 && i0 > 0) meet();   // the sums of the section before are read
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const int q = tid + NT * (i0 + i);
      u32x4_t w = v[i];
      if (!NORM && i0 > 0) w = ld(xr, 16 * q);
      u32x4_t h;
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // entries k, k + 2 of a group of four share a word, as the codes do (below)
        const int e = j & 2;
        const float x0 = ((j & 1) ? bf16hi(w[e]) : bf16lo(w[e])) * sc;
        const float x1 = ((j & 1) ? bf16hi(w[e + 1]) : bf16lo(w[e + 1])) * sc;
        h[j] = pk_f16(x0, x1);
        s += x0 + x1;
      }
      if (q < n_q) xt[(size_t)(q >> 2) * 64 + ((q & 3) ^ swz)] = h;
      if constexpr (KIND == 4) {
        s += dpp<kDppXor1>(s);
        s += dpp<kDppXor2>(s);                  // the group's sum, in its four lanes
        if ((l & 3) == 0) sg[NT / 4 * i + (tid >> 2)] = s;
      }
    }
    if constexpr (KIND != 4) continue;
    meet();
    // eight groups per thread (groups past K hold zeros, which the last chunk keeps)
    const int g = NT / 4 * i0 + 8 * tid;
    if (tid < NT / 32 * C && g < 32 * n_ch) {
      u32x4_t hi, lo;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t th, tl;
        split2(sg[8 * tid + 2 * j] * exp2i(-kPqSum), sg[8 * tid + 2 * j + 1] * exp2i(-kPqSum), th, tl);
        hi[j] = th;
        lo[j] = tl;
      }
      u32x4_t* d = sm + (size_t)(g >> 5) * 2 * 64 + (((g >> 3) & 3) ^ swz);
      d[0] = hi;
      d[64] = lo;
    }
  }
}

// Weight tile-row: its columns' powers of two and u = m + 8 d in the minimum term's B operand
// order. NW waves per tile-row, a chunk of 32 groups each: lane (c, s) holds columns
// (c / 8) 16 + 2 (c % 8), + 1 at groups 8 s + j (K-tile 4 ch + s).
template <int NW>
__device__ __forceinline__ void prep_tile_row(const GemmArgs& a, const PqX& o, int tensor, int tr,
                                              uint32_t* __restrict__ sm) {
  constexpr int CACHED = 2;                     // chunks a wave keeps: K <= 2048 NW
  const int l = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = l & 15, s = l >> 4, n_tr = a.n_tr[0];
  const int n_ch = pq_chunks<4>(a.k_t);
  const uint8_t* wr = a.w[tensor] + (size_t)tr * a.k_t * kQ4TileBytes +
                      2 * ((c >> 3) * 16 + 2 * (c & 7));
  uint32_t dv[CACHED][8], mv[CACHED][8], dm = 0, mm = 0;
  uint32_t mn = ~0u;                            // the smallest group's larger of |m| and 8 |d|
  auto fetch = [&](int ch, uint32_t (&d)[8], uint32_t (&m)[8]) {
    const int kt = kPqChunkTiles * ch + s;
    const uint8_t* t = wr + (size_t)min(kt, a.k_t - 1) * kQ4TileBytes;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      d[j] = *(const uint32_t*)(t + j * 64);
      m[j] = *(const uint32_t*)(t + kMetaBytes + j * 64);
    }
  };
  auto clip = [&](int ch, uint32_t (&d)[8], uint32_t (&m)[8]) {   // groups past K: zero
    const bool in = kPqChunkTiles * ch + s < a.k_t;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      d[j] = in ? d[j] : 0u;
      m[j] = in ? m[j] : 0u;
    }
  };
  auto see = [&](int ch, const uint32_t (&d)[8], const uint32_t (&m)[8]) {
    const uint32_t past = kPqChunkTiles * ch + s < a.k_t ? 0u : ~0u;   // groups past K: none
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t da = d[j] & 0x7FFF7FFFu, ma = m[j] & 0x7FFF7FFFu;
      dm = pk_max_u16(dm, da);
      mm = pk_max_u16(mm, ma);
      mn = pk_min_u16(mn, pk_max_u16(pk_add_u16(da, 0x01800180u), ma) | past);
    }
  };
#pragma unroll
  for (int i = 0; i < CACHED; ++i)
    if (w + NW * i < n_ch) fetch(w + NW * i, dv[i], mv[i]);
#pragma unroll
  for (int i = 0; i < CACHED; ++i)
    if (w + NW * i < n_ch) {
      clip(w + NW * i, dv[i], mv[i]);
      see(w + NW * i, dv[i], mv[i]);
    }
  for (int ch = w + NW * CACHED; ch < n_ch; ch += NW) {
    uint32_t d[8], m[8];
    fetch(ch, d, m);
    clip(ch, d, m);
    see(ch, d, m);
  }
  dm = rows_max(dm);
  mm = rows_max(mm);
  mn = rows_min(mn);
  if (l < 16) {
    sm[w * 48 + l] = dm;
    sm[w * 48 + 16 + l] = mm;
    sm[w * 48 + 32 + l] = mn;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    dm = pk_max_u16(dm, sm[i * 48 + c]);
    mm = pk_max_u16(mm, sm[i * 48 + 16 + c]);
    mn = pk_min_u16(mn, sm[i * 48 + 32 + c]);
  }
  int sh[2], wide[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int ed = (int)((dm >> (16 * h + 7)) & 0xFF), em = (int)((mm >> (16 * h + 7)) & 0xFF);
    // |u| <= |m| + 8 |d| < 2^(max(em, ed + 3) + 1 - 126)
    const bool finite = ed < 255 && em < 255;
    sh[h] = finite ? min(kPqWTop - 1 - max(em, ed + 3), 127 - kPqSum) : 0;
    wide[h] = finite && span_wide(max(em, ed + 3), (int)((mn >> (16 * h + 7)) & 0x1FF));
  }
  if (w == 0 && l < 16)
    *(int2*)(o.wshift + ((size_t)tensor * n_tr + tr) * 32 + (c >> 3) * 16 + 2 * (c & 7)) =
        make_int2(2 * sh[0] + wide[0], 2 * sh[1] + wide[1]);
  const float sd[2] = {exp2i(sh[0]), exp2i(sh[1])};
  auto put = [&](int ch, const uint32_t (&d)[8], const uint32_t (&m)[8]) {
    u32x4_t* du = o.u + ((((size_t)tensor * n_tr + tr) * n_ch + ch) * 4) * 64 + l;
    uint2* ds = o.scale + (((size_t)tensor * n_tr + tr) * a.k_t + kPqChunkTiles * ch + s) * 128 + c;
    u32x4_t hi[2], lo[2];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float u[2][2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint32_t dd = d[2 * j + e], mw = m[2 * j + e];
        const float d0 = bf16lo(dd) * sd[0], d1 = bf16hi(dd) * sd[1];
        const uint32_t dp = pk_f16z(d0, d1), ap = pk_f16z(d0 * kPqLow, d1 * kPqHigh);
        const half2_t dh = as_h2(dp), ah = as_h2(ap);
        if (kPqChunkTiles * ch + s < a.k_t) ds[(2 * j + e) * 16] = make_uint2(dp, ap);
        u[0][e] = (bf16lo(mw) * sd[0] - fmaf(1024.f, (float)dh.x, (float)ah.x)) * (1 << kPqSum);
        u[1][e] = (bf16hi(mw) * sd[1] - fmaf(64.f, (float)dh.y, (float)ah.y)) * (1 << kPqSum);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint32_t th, tl;
        split2(u[h][0], u[h][1], th, tl);
        hi[h][j] = th;
        lo[h][j] = tl;
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      du[h * 64] = hi[h];
      du[(2 + h) * 64] = lo[h];
    }
  };
#pragma unroll
  for (int i = 0; i < CACHED; ++i)
    if (w + NW * i < n_ch) put(w + NW * i, dv[i], mv[i]);
  for (int ch = w + NW * CACHED; ch < n_ch; ch += NW) {
    uint32_t d[8], m[8];
    fetch(ch, d, m);
    clip(ch, d, m);
    put(ch, d, m);
  }
}

// Of a q8 tile-row: the columns' powers of two. Each wave takes K-tiles, lane (c, s) the scales of
// columns 2 c and 2 c + 1 at groups 2 s and 2 s + 1.
template <int NW>
__device__ __forceinline__ void prep_tile_row_q8(const GemmArgs& a, const PqX& o, int tr,
                                                 uint32_t* __restrict__ sm) {
  const int l = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = l & 15, s = l >> 4;
  const uint8_t* wr = a.w[0] + (size_t)tr * a.k_t * kQ8TileBytes + 128 * s + 4 * c;
  uint32_t mx = 0, mn = ~0u;
  for (int kt = w; kt < a.k_t; kt += NW)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const uint32_t v = *(const uint32_t*)(wr + (size_t)kt * kQ8TileBytes + 64 * e) & 0x7FFF7FFFu;
      mx = pk_max_u16(mx, v);
      mn = pk_min_u16(mn, v);
    }
  mx = rows_max(mx);
  mn = rows_min(mn);
  if (l < 16) {
    sm[w * 32 + l] = mx;
    sm[w * 32 + 16 + l] = mn;
  }
  __syncthreads();
  if (w > 0 || l >= 16) return;
#pragma unroll
  for (int i = 1; i < NW; ++i) {
    mx = pk_max_u16(mx, sm[32 * i + c]);
    mn = pk_min_u16(mn, sm[32 * i + 16 + c]);
  }
  int sh[2], wide[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int e = (int)((mx >> (16 * h + 7)) & 0xFF);
    sh[h] = e < 255 ? min(kPqSTop - max(e, 1), 127) : 0;
    wide[h] = e < 255 && span_wide(e, (int)((mn >> (16 * h + 7)) & 0xFF));
  }
  *(int2*)(o.wshift + (size_t)tr * 32 + 2 * c) = make_int2(2 * sh[0] + wide[0], 2 * sh[1] + wide[1]);
}

// First a weight tile-row per workgroup, over both tensors of [gate, up] -- the longer ones -- then
// ROWS rows of x each.
// What bounds it: the latency of one workgroup (3 us launched empty-handed; 80 tile-rows of K =
// 8192 took 8.9 us in four waves, 5.4 in the eight of K > 4096) and, with many rows, their bytes
// (2048 x 2560, 21 MB in and out, 8.2 us). Rows of K <= 1024 leave most of a workgroup idle and
// are a wave each, so a workgroup's 64-byte pieces of x also fill whole cache lines (3000 rows of
// K = 512 8.2 -> 6.8 us, and with 12288 columns the contraction after it 61 -> 57); two or four
// longer rows per workgroup gain nothing (2048 x 2560 9.1 -> 10.1, 9.9).
template <int KIND, bool NORM, int C, int NT, int ROWS>
__global__ __launch_bounds__(NT) void pq_prep_kernel(GemmArgs a, PqX o, int tile_rows) {
  __shared__ float sg[KIND == 4 ? NT / 4 * C : 1];
  __shared__ uint32_t sm[NT / 64 * 48];         // (a tile-row's: 48 words of a wave)
  const int t = blockIdx.x, n = a.n_tr[0];
  if (t >= tile_rows) {
    constexpr int TR = NT / ROWS;                 // threads of a row: one wave, or all
    const int sub = ROWS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / TR);
    // (past the last row: that row again, in step with the others)
    prep_row<KIND, NORM, C, TR>(a, o, min((t - tile_rows) * ROWS + sub, a.m_rows - 1),
                                sg + (KIND == 4 ? TR / 4 * C * sub : 0), sm + TR / 64 * sub);
  } else {
    if constexpr (KIND == 4) prep_tile_row<NT / 64>(a, o, t / n, t % n, sm);
    else prep_tile_row_q8<NT / 64>(a, o, t, sm);
  }
}

constexpr int vm_wait_pq(int n) {
  return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) & 3) << 14;
}

// The workgroup's waves meet; nothing is waited for (the reads of LDS in flight are of buffers
// that are written again a whole step later at the earliest, after their use)
__device__ __forceinline__ void step_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}

__device__ __forceinline__ void pin_acc(f32x4_t& v) { asm volatile("" : "+v"(v)); }

// 16 bytes (4: one dword) per lane from uniform base + offset + lane offset to LDS at lds + off
// + 16 (4) lane
template <int OFF>
__device__ __forceinline__ void ldl16(const void* base, uint32_t voff, uint32_t lds, int add) {
  asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:%4"
               :: "s"(lds), "v"(voff), "s"(base), "i"(add - OFF), "i"(OFF) : "memory", "scc");
}
__device__ __forceinline__ void ldl16d(const void* base, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :: "s"(lds), "v"(voff), "s"(base) : "memory");
}
template <int OFF>
__device__ __forceinline__ void ldl4(const void* base, uint32_t voff, uint32_t lds, int add) {
  asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2 offset:%4"
               :: "s"(lds), "v"(voff), "s"(base), "i"(add - OFF), "i"(OFF) : "memory", "scc");
}

// A wave's tile without the powers of two, for rows and columns whose groups differ too far in size
// (above, "Range"): per 32-K group the bf16 rows of x on exact bf16 codes (c - 8, or q) from zero, and
// one FMA per output with the group's fp32 scale (q4: another with m + 8 d and the group's sum of x),
// added up per K-tile. Everything comes through the caches as it is needed; the weights' tile goes
// through the wave's LDS slot for the transposing read. All of K, MC m-tiles at a time, which the
// waves of the K parts share out, each pass handed to `out`. One to two times the batched kernel's
// time where every row is wide (8192 x 2560, 2048 rows 277 / 214 us, q8 324 / 349).
template <int KIND, int MT, int RT, int WK, typename OUT>
__device__ __forceinline__ void exact_tile(const GemmArgs& a, const PqX& p, uint8_t* slot,
                                           const uint8_t* const (&wr)[RT], int m0, int wk, OUT&& out) {
  constexpr int MW = MT > WK ? MT / WK : 1, MC = MW * RT > 4 ? 4 / RT : MW;
  constexpr int TB = GemmFmt<KIND>::kTile, NLD = GemmFmt<KIND>::kLoads;
  const int l = threadIdx.x & 63, c = l & 15, s = l >> 4;
  const int tr_off = KIND == 4
      ? GemmFmt<4>::kCodes + (c & 1) * 2048 + (8 * s + (c >> 1)) * 8
      : GemmFmt<8>::kCodes + (8 * s + (c >> 1)) * 16 + (c & 1) * 8;
  const int meta_off = KIND == 4 ? 2 * ((c >> 3) * 16 + 2 * (c & 7)) : 2 * c;
  const int unit_steps = a.k_t * 8 + pq_chunks<KIND>(a.k_t) * 2;
  const u32x4_t ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int mp = wk * MC; mp < MT; mp += WK * MC) {
    f32x4_t acc[RT][MC][2];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int mt = 0; mt < MC; ++mt) acc[r][mt][0] = acc[r][mt][1] = zero;
    // the lane's row of each m-tile: its bf16 entries, or (a row of a fused norm that is not wide)
    // the pre-pass's fp16 ones under the power of two sh
    const uint8_t* xr[MC];
    int step[MC], sh[MC];
#pragma unroll
    for (int mt = 0; mt < MC; ++mt) {
      const int row = min(m0 + 16 * (mp + mt) + c, a.m_rows - 1), r16 = row & 15;
      const int x = p.exact_all ? 1 : p.xshift[row];
      sh[mt] = x & 1 ? 256 : x >> 1;             // 256: bf16
      step[mt] = x & 1 ? 64 : 1024;
      xr[mt] = x & 1 ? (const uint8_t*)(p.exact + row * p.exact_stride + 8 * s)
                     : (const uint8_t*)(p.xt + (size_t)(row >> 4) * unit_steps * 64 + r16 * 4 +
                                        (s ^ ((r16 >> 1) & 3)));
    }
#pragma unroll 1
    for (int kt = 0; kt < a.k_t; ++kt) {
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
          const int o = 16 * (64 * i + l);
          if (o < TB) *(u32x4_t*)(slot + r * TB + o) = *(const u32x4_t*)(wr[r] + (size_t)kt * TB + o);
        }
      f32x4_t prt[RT][MC][2];
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int mt = 0; mt < MC; ++mt) prt[r][mt][0] = prt[r][mt][1] = zero;
#pragma unroll 1
      for (int kb = 0; kb < 8; ++kb) {
        u32x4_t op[RT][2];
        float d[RT][2], u[RT][2];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          const uint8_t* sl = slot + r * TB;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const i32x2_t cb = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                (lds_i32x2_t*)(sl + tr_off + (KIND == 4 ? kb * 256 : h * 4096 + kb * 512)));
#pragma unroll
            for (int j = 0; j < 4; ++j) {        // entries 2 j and 2 j + 1
              const uint32_t w = ((uint32_t)(j < 2 ? cb.x : cb.y)) >> (16 * (j & 1));
              float f0, f1;
              if constexpr (KIND == 4) {
                f0 = (float)((w >> (4 * h)) & 15u) - 8.f;
                f1 = (float)((w >> (8 + 4 * h)) & 15u) - 8.f;
              } else {
                f0 = (float)(int)(int8_t)w;
                f1 = (float)(int)(int8_t)(w >> 8);
              }
              op[r][h][j] = perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
            }
            if constexpr (KIND == 4) {
              d[r][h] = bf16_to_f32(*(const uint16_t*)(sl + kb * 64 + meta_off + 2 * h));
              u[r][h] = fmaf(8.f, d[r][h], bf16_to_f32(*(const uint16_t*)(sl + kMetaBytes + kb * 64 + meta_off + 2 * h)));
            } else {
              d[r][h] = bf16_to_f32(*(const uint16_t*)(sl + kb * 64 + h * 32 + meta_off));
            }
          }
        }
#pragma unroll
        for (int mt = 0; mt < MC; ++mt) {
          u32x4_t x = *(const u32x4_t*)(xr[mt] + (size_t)(kt * 8 + kb) * step[mt]);
          if (sh[mt] < 256) {                    // entries k, k + 2 share a word there
            u32x4_t y;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const half2_t e0 = as_h2(x[j & 2]), e1 = as_h2(x[(j & 2) + 1]);
              const float f0 = ldexpf((float)(j & 1 ? e0.y : e0.x), -sh[mt]);
              const float f1 = ldexpf((float)(j & 1 ? e1.y : e1.x), -sh[mt]);
              y[j] = perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
            }
            x = y;
          }
          f32x4_t sx;
          if constexpr (KIND == 4) sx = mfma_bf16(x, ones, zero);
#pragma unroll
          for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const f32x4_t t = mfma_bf16(x, op[r][h], zero);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                prt[r][mt][h][e] = fmaf(d[r][h], t[e], prt[r][mt][h][e]);
                if constexpr (KIND == 4) prt[r][mt][h][e] = fmaf(u[r][h], sx[e], prt[r][mt][h][e]);
              }
            }
        }
      }
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int mt = 0; mt < MC; ++mt)
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[r][mt][h][e] += prt[r][mt][h][e];
    }
    out(acc, m0 + 16 * mp);
  }
}

// A workgroup of WN x WK waves takes 16 MT rows of X; wave (wn, wk) owns RT tile-rows (GATEUP:
// the same tile-row of gate and of up) over K part wk, so nothing is shared between waves but
// the staged x of their K part, and the parts are added through LDS at the end in part order.
// x (a ring of RING 32-K steps) and the codes (a K-tile in two halves) go from memory to LDS by
// direct loads, counted by hand, with no registers in between; the step's operands are built
// beside its MFMAs, in 18 VALU instructions per tile-row, so the matrix cores set the pace.
// What bounds it (2048 rows of 8192 x 2560, 83 us): more K adds at 1.23 to 1.30 PFLOP/s, with the
// clock held at 2.0 to 2.1 GHz under that load and the matrix cores busy 0.51 of the time (0.59 at K
// = 5120); 17 us of the launch -- the first loads and the outputs, all of its workgroups' at once --
// and the pre-pass's 9 are not overlapped with it. Calls, pre-pass included, before (scale after the
// MFMA, one FMA per output and group; below 512 workgroups and [gate, up] the batched kernel) and now,
// us, N x K, rows: 8192 x 2560, 2048 rows 124 -> 86; 2560 x 8192, 333 rows 57 -> 31; [gate, up] 8192 x
// 2560, 500 rows 126 -> 55, 2048 rows 477 -> 185. Error against 64 bits: 2048 rows, K = 2560 1.05e-6 ->
// 3.2e-7, 333 rows, K = 8192 3.1e-7 -> 1.2e-7, [gate, up], K = 2560 2.6e-7 -> 2.2e-7.
template <int KIND, int OP, int MT, int RT, int WN, int WK, int RING, int OCC>
__global__ __launch_bounds__(64 * WN * WK, OCC) void pq_kernel(GemmArgs a, PqX p) {
  constexpr int TB = GemmFmt<KIND>::kTile, HALF = kPqHalf<KIND>;
  constexpr int NR = KIND == 4 ? 1 : 2;        // transposing reads of a step's codes
  constexpr int NC = KIND == 4 ? 2 : 4;        // direct loads of half a tile's codes
  constexpr int U = MT / WN;                   // x units (1 KB: one m-tile, one step) per wave
  constexpr int XD = RING - 1;                 // steps of x in flight ahead of use
  constexpr bool LOOK = RING == 8;             // x read from LDS ahead across the step boundary
  constexpr int WL = (NC + (KIND == 4 ? 2 : 1)) * RT;            // direct loads of half a weight tile
  static_assert(MT % WN == 0, "every wave stages as many m-tiles");
  static_assert(8 % RING == 0, "a step's ring slot is known at compile time");
  static_assert(OP == GOP_PLAIN || (KIND == 4 && RT == 2), "gate and up");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

  const int tid = threadIdx.x, l = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, wk = wave / WN;
  const int c = l & 15, s = l >> 4;
  const int n_tr = a.n_tr[0];
  const int n_ch = pq_chunks<KIND>(a.k_t);
  const int unit_steps = a.k_t * 8 + n_ch * 2;  // per m-tile: the steps of x, then of the sums
  int cgrp, mblk;
  if (p.rows_first) {
    const int tile = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    cgrp = tile / p.m_blocks;
    mblk = tile - cgrp * p.m_blocks;
  } else {
    mblk = blockIdx.x / p.c_groups;
    cgrp = blockIdx.x - mblk * p.c_groups;
  }
  const int unit = cgrp * WN + wn;             // RT tile-rows, or one pair
  if (cgrp >= p.c_groups || mblk >= p.m_blocks) return;   // the grid is a multiple of 8
  const int m0 = mblk * 16 * MT;
  // this wave's K part (a wave whose part ends early, or is empty, keeps the others' barriers)
  const int kq = (a.k_t + WK - 1) / WK;
  const int kt0 = min(wk * kq, a.k_t - 1), kt1 = min(a.k_t, wk * kq + kq);
  const int nt = kt1 - wk * kq;                // its K-tiles (0 or less: none)
  const uint8_t* wr[RT];
  int tr[RT], col0[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int ten = OP == GOP_PLAIN ? 0 : r;
    tr[r] = OP == GOP_PLAIN ? unit * RT + r : unit;
    const int trc = min(tr[r], n_tr - 1);
    wr[r] = a.w[ten] + (size_t)trc * a.k_t * TB;
    col0[r] = ten * n_tr + trc;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  const uint32_t xring = wk * RING * MT * 1024;                       // this part's x ring
  constexpr int WBUF = RT * 2 * HALF;       // one K-tile of the wave's tile-rows
  const uint32_t wslot = WK * RING * MT * 1024 + wave * WBUF;
  const uint32_t l16 = 16 * l, l4 = 4 * l;
  const uint32_t xm0 = lds0 + xring + wn * 1024, wm0 = lds0 + wslot;
  const uint8_t* xp[U];                        // m-tile wn + WN j at a multiple of four steps
#pragma unroll
  for (int j = 0; j < U; ++j)
    xp[j] = (const uint8_t*)p.xt +
            ((size_t)(mblk * MT + wn + WN * j) * unit_steps + kt0 * 8) * 1024;
  // the part's chunks of the minimum term, and from its last x step to its sums
  const int ch0 = kt0 / kPqChunkTiles, nc = nt > 0 ? (kt1 + kPqChunkTiles - 1) / kPqChunkTiles - ch0 : 0;
  const int64_t to_sums = KIND == 4 ? (int64_t)((a.k_t - kt1) * 8 + ch0 * 2 + 4) * 1024 : 4096;
  const uint8_t *up[RT], *sp[RT];              // its u, its scales
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    up[r] = (const uint8_t*)(p.u + ((size_t)col0[r] * n_ch + ch0) * 4 * 64);
    sp[r] = (const uint8_t*)(p.scale + (size_t)col0[r] * a.k_t * 128);
  }

  // x of a step, `ks` (mod 8) its place in its K-tile; the part's sums follow its last K-tile,
  // and loads past them read the next bytes of the workspace, never used
  auto x_load = [&](auto ksc, bool last) {
    constexpr int ks = decltype(ksc)::value;
    if constexpr ((ks & 3) == 0) {
      const int64_t go = ks == 0 && last ? to_sums : 4096;
#pragma unroll
      for (int j = 0; j < U; ++j) xp[j] += go;
    }
#pragma unroll
    for (int j = 0; j < U; ++j)
      ldl16<(ks & 3) * 1024>(xp[j], l16, xm0, ((ks % RING) * MT + WN * j) * 1024);
  };
  // half of the part's K-tile t: 128 K of codes and their scales; after the last tile, in as many
  // loads, the high (low) terms of the part's first chunk of u in their place (q8: that tile
  // again, never used)
  auto w_load = [&](int t, auto halfc) {
    constexpr int half = decltype(halfc)::value;
    const bool more = t < nt;
    const int kt = KIND == 4 ? kt0 + t : kt0 + (more ? t : max(nt - 1, 0));
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const uint8_t* w = wr[r] + (size_t)kt * TB;
      const uint8_t* q = sp[r] + (size_t)kt * 1024 + half * 512;
      const int d = (r * 2 + half) * HALF;
      if constexpr (KIND == 4) {
        const uint8_t* u = up[r] + half * 2048;
        ldl16<0>(more ? w + 1024 + half * 1024 : u, l16, wm0, d);
        ldl16<0>(more ? w + 3072 + half * 1024 : u + 1024, l16, wm0, d + 1024);
        q = more ? q : u;
        ldl4<256>(q, l4, wm0, d + NC * 1024 + 256);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)            // each row block's 2 KB
          ldl16<0>(w + kMetaBytes + (i >> 1) * 4096 + half * 2048 + (i & 1) * 1024, l16, wm0,
                   d + i * 1024);
        q = w + half * 256;
      }
      ldl4<0>(q, l4, wm0, d + NC * 1024);
    }
  };
#pragma unroll
  for (int j = 0; j < U; ++j) xp[j] -= 4096;
  x_load(std::integral_constant<int, 0>{}, false);
  w_load(0, std::integral_constant<int, 0>{});
  w_load(0, std::integral_constant<int, 1>{});
  static_for<1, XD>([&](auto i) { x_load(i, false); });

  f32x4_t acc[RT][MT][2];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[r][mt][0] = acc[r][mt][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // Short accumulation chains where the registers allow: a K-tile's sum starts from zero and is
  // added to the total on the VALU. The matrix cores' own accumulation rounds more coarsely: one
  // chain over K = 1024 / 2560 / 8192 is 2.0 / 3.2 / 5.9e-7 off the 64-bit result, in K-tiles 1.0 /
  // 1.1 / 1.4e-7. The 128-row q4 tile has no registers for that; in two K parts it is 1.4 / 2.2 /
  // 4.1e-7 off, the batched kernel 1.9 / 2.6 / 4.2e-7 (which tile a launch may take: pq_plain).
  constexpr bool FLUSH = KIND == 4 && MT * RT <= 8;
  f32x4_t prt[FLUSH ? RT : 1][FLUSH ? MT : 1][2];
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  // the lane's two columns of a tile-row (its even and odd column, or column c of each row block)
  const int cols[2] = {KIND == 4 ? (c >> 3) * 16 + 2 * (c & 7) : c,
                       KIND == 4 ? (c >> 3) * 16 + 2 * (c & 7) + 1 : 16 + c};
  int shw[RT][2];                              // the columns' powers of two
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    shw[r][0] = p.wshift[(size_t)col0[r] * 32 + cols[0]] >> 1;
    shw[r][1] = p.wshift[(size_t)col0[r] * 32 + cols[1]] >> 1;
  }
  // whether a row of the block is wide: lane l looks at rows 2 l and 2 l + 1 (past X: anything)
  const int row2 = m0 + 2 * min(l, 8 * MT - 1);
  const int2 rows2 = *(const int2*)(p.xshift + row2);
  const int wide_r = (row2 < a.m_rows ? rows2.x : 0) | (row2 + 1 < a.m_rows ? rows2.y : 0);
  // q8: the inner sums on their way to the totals (each LAG MFMAs after its own), the scales of
  // the steps of either parity, the columns' powers of two
  constexpr int LAG = 3;
  f32x4_t inner[4] = {zero, zero, zero, zero};
  float scl[2][RT][2] = {}, wsc[RT][2];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int h = 0; h < 2; ++h) wsc[r][h] = exp2i(shw[r][h]);
  // ---- operands: the transposing LDS read gives lane (c, s) the 8 code bytes at k = 8 s .. of
  // row pair c % 8 of row-block c / 8, low nibbles the even row, high the odd one (q8: of row c
  // of one row block per read)
  const uint8_t* const trp = lds + wslot + (KIND == 4 ? (c & 1) * 1024 + (8 * s + (c >> 1)) * 8
                                                      : (8 * s + (c >> 1)) * 16 + (c & 1) * 8);
  const uint8_t* const scp = lds + wslot + NC * 1024 + (KIND == 4 ? 8 : 2) * c;
  struct Raw {
    i32x2_t cb[NR];
    uint2 sc;                                  // fp16 (d even, d odd), (A even, A odd); q8: bf16
  } raw[2][RT];                                // of steps of either parity
  auto read_raw = [&](int kb) {
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const int b = (r * 2 + (kb >> 2)) * HALF;
#pragma unroll
      for (int h = 0; h < NR; ++h)
        raw[kb & 1][r].cb[h] = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
            (lds_i32x2_t*)(trp + b + h * 2048 + (kb & 3) * (KIND == 4 ? 256 : 512)));
      if constexpr (KIND == 4) raw[kb & 1][r].sc = *(const uint2*)(scp + b + (kb & 3) * 128);
      else
        raw[kb & 1][r].sc = make_uint2(*(const uint16_t*)(scp + b + (kb & 3) * 64),
                                       *(const uint16_t*)(scp + b + (kb & 3) * 64 + 32));
    }
  };
  // The operands of a step, in 8 NR RT half pieces: the first half of a piece takes two code
  // bytes (0 and 2, or 1 and 3) of a word to fp16 B + c -- their low and their high nibbles (q8:
  // the bytes) -- the second multiplies and adds (q8: subtracts).
  u32x4_t ops[2][RT][2];
  uint32_t msk_l, msk_h, exp_l, exp_h, tE = 0, tO = 0;
  asm("v_mov_b32 %0, 0x000f000f" : "=v"(msk_l));
  asm("v_mov_b32 %0, 0x00f000f0" : "=v"(msk_h));
  asm("s_mov_b32 %0, 0x64006400" : "=s"(exp_l));
  asm("s_mov_b32 %0, 0x54005400" : "=s"(exp_h));
  auto half_piece = [&](int b, int i) {        // into ops[b] from raw[b]
    const int r = i / (8 * NR), col = (i >> 3) & (NR - 1), h = (i >> 2) & 1, q = (i >> 1) & 1;
    const i32x2_t cb = raw[b][r].cb[col];
    if constexpr (KIND == 4) {
      const uint32_t w = h ? (uint32_t)cb.y : (uint32_t)cb.x;
      if ((i & 1) == 0) {
        tE = ((w >> (8 * q)) & msk_l) | exp_l;
        tO = ((w >> (8 * q)) & msk_h) | exp_h;
        return;
      }
      const half2_t d = as_h2(raw[b][r].sc.x), A = as_h2(raw[b][r].sc.y);
      const half2_t dE = {d.x, d.x}, dO = {d.y, d.y}, aE = {A.x, A.x}, aO = {A.y, A.y};
      ops[b][r][0][2 * h + q] = h2_bits(__builtin_elementwise_fma(as_h2(tE), dE, aE));
      ops[b][r][1][2 * h + q] = h2_bits(__builtin_elementwise_fma(as_h2(tO), dO, aO));
    } else {
      if ((i & 3) == 0) tO = (h ? (uint32_t)cb.y : (uint32_t)cb.x) ^ 0x80808080u;
      if ((i & 1) == 0) {
        tE = __builtin_amdgcn_perm(exp_l, tO, q ? 0x07030701u : 0x07020700u);   // 0x64 code bytes
        return;
      }
      const half2_t k = {(_Float16)1152.f, (_Float16)1152.f};
      uint32_t o = h2_bits(as_h2(tE) - k);
      asm volatile("" : "+v"(o));
      ops[b][r][col][2 * h + q] = o;
    }
  };
  auto scales = [&](int b) {                   // q8: scl[b] from raw[b]
    if constexpr (KIND == 8)
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        scl[b][r][0] = __uint_as_float(raw[b][r].sc.x << 16) * wsc[r][0];
        scl[b][r][1] = __uint_as_float(raw[b][r].sc.y << 16) * wsc[r][1];
      }
  };
  // q8: MFMA f's inner sums, a step of parity b, into the totals
  auto fold = [&](int f, int b) {
    const int h = f & 1, r = (f >> 1) % RT, mt = (f >> 1) / RT;
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[r][mt][h][e] = fmaf(scl[b][r][h], inner[f & 3][e], acc[r][mt][h][e]);
    pin_acc(acc[r][mt][h]);
  };

  // ---- outputs: the lane's two columns are adjacent, so the 16 lanes of a row write 128
  // contiguous bytes (64 of bf16; q8: 64 bytes per row block)
  // (an output's address is a uniform row 16 mt + e plus the lane's 32-bit offset)
  const uint32_t ly = (uint32_t)(4 * s * (OP == GOP_PLAIN ? a.y_stride : a.h_stride) + cols[0]);
  // (v: RT x any number of m-tiles x 2, from row mb on; full: every row of them is one of X)
  auto store_rows = [&](auto& v, int mb, auto fullc) {
    constexpr bool FULL = decltype(fullc)::value;
#pragma unroll
    for (int mt = 0; mt < (int)(sizeof(v[0]) / sizeof(v[0][0])); ++mt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int mu = mb + 16 * mt + e, m = mu + 4 * s;
        const bool row_live = FULL || m < a.m_rows;
        if constexpr (OP == GOP_PLAIN) {
#pragma unroll
          for (int r = 0; r < RT; ++r) {
            if (tr[r] >= n_tr) continue;
            const int64_t o = (int64_t)mu * a.y_stride + (int64_t)tr[r] * 32;
            float2 o2 = make_float2(v[r][mt][0][e], v[r][mt][1][e]);
            if (row_live) {
              if (a.residual != nullptr) {
                const float* rr = a.residual + o;
                if constexpr (KIND == 4) {
                  const float2 t = *(const float2*)(rr + ly);
                  o2.x += t.x;
                  o2.y += t.y;
                } else {
                  o2.x += rr[ly];
                  o2.y += rr[ly + 16];
                }
              }
              if (a.y != nullptr) {
                float* yy = a.y + o;
                if constexpr (KIND == 4) *(float2*)(yy + ly) = o2;
                else {
                  yy[ly] = o2.x;
                  yy[ly + 16] = o2.y;
                }
              }
            }
            if (a.ssq_out != nullptr) {        // per 16-row block: 8 lanes (q8: 16, a column each)
              float* so = a.ssq_out + (int64_t)m * n_tr * 2 + tr[r] * 2;
              if constexpr (KIND == 4) {
                float q = fmaf(o2.x, o2.x, o2.y * o2.y);
                q += dpp<kDppXor1>(q);
                q += dpp<kDppXor2>(q);
                q += dpp<kDppHalfMirror>(q);
                if (row_live && (c & 7) == 0) so[c >> 3] = q;
              } else {
                const float q0 = group16_sum(o2.x * o2.x), q1 = group16_sum(o2.y * o2.y);
                if (row_live && c == 0) so[0] = q0, so[1] = q1;
              }
            }
          }
        } else {
          if (tr[0] >= n_tr || !row_live) continue;
          const int64_t N = (int64_t)n_tr * 32, n = (int64_t)tr[0] * 32;
          const float g0 = v[0][mt][0][e], g1 = v[0][mt][1][e];
          const float u0 = v[1][mt][0][e], u1 = v[1][mt][1][e];
          *(uint32_t*)(a.h_out + (int64_t)mu * a.h_stride + n + ly) =
              pack_bf16x2(swiglu(round_bf16_op(g0), round_bf16_op(u0)),
                          swiglu(round_bf16_op(g1), round_bf16_op(u1)));
          if (a.raw_out != nullptr) {
            float* ro = a.raw_out + (int64_t)m * 2 * N + n + cols[0];
            *(float2*)ro = make_float2(g0, g1);
            *(float2*)(ro + N) = make_float2(u0, u1);
          }
        }
      }
  };
  auto store = [&](auto& v, int mb, int rows) {
    if (mb + rows <= a.m_rows) store_rows(v, mb, std::true_type{});
    else store_rows(v, mb, std::false_type{});
  };

  __builtin_amdgcn_s_waitcnt(vm_wait_pq(0));
  __syncthreads();
  if (__builtin_expect(__any(wide_r & 1), 0)) {
    // a column of the workgroup too: the tile by other means
    int wide_c = 0;
#pragma unroll
    for (int i = 0; i < WN * RT * 32; i += 64) {
      const int t = (i + l) >> 5;                // of the group's tile-rows (gate's, then up's)
      const int ten = OP == GOP_PLAIN ? 0 : t / WN;
      const int u = OP == GOP_PLAIN ? cgrp * WN * RT + t : cgrp * WN + t % WN;
      if (i + l < WN * RT * 32 && u < n_tr) wide_c |= p.wshift[((size_t)ten * n_tr + u) * 32 + (l & 31)];
    }
    if (__any(wide_c & 1)) {
      exact_tile<KIND, MT, RT, WK>(a, p, lds + wslot, wr, m0, wk, [&](auto& v, int mb) {
        store_rows(v, mb, std::false_type{});
      });
      return;
    }
  }
  read_raw(0);
  read_raw(1);
#pragma unroll
  for (int i = 0; i < 8 * NR * RT; ++i) half_piece(0, i);
  scales(0);
  // x fragments are read from LDS D m-tiles ahead of their use (LOOK: across the step boundary
  // too) and a step's operand data two steps ahead
  constexpr int D = MT < 3 ? MT : 3;
  u32x4_t xa[4];
  const uint8_t* const xl = lds + xring + c * 64 + ((s ^ (c >> 1)) & 3) * 16;
  if constexpr (LOOK) {
#pragma unroll
    for (int f = 0; f < D; ++f) xa[f] = *(const u32x4_t*)(xl + f * 1024);
  }

  // ---- main loop over the part's K-tiles
  for (int t = 0; t < nt; ++t) {
    static_for<0, 8>([&](auto kbc) {
      constexpr int kb = decltype(kbc)::value;
      constexpr int cur = kb & 1, nxt = cur ^ 1;
      constexpr int cs = (kb % RING) * MT * 1024, ns = ((kb + 1) % RING) * MT * 1024;
      if constexpr (!LOOK) {
#pragma unroll
        for (int f = 0; f < D; ++f) xa[(kb * MT + f) & 3] = *(const u32x4_t*)(xl + cs + f * 1024);
      }
      read_raw((kb + 2) & 7);
      x_load(std::integral_constant<int, (kb + XD) & 7>{}, t == nt - 1);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        if (mt + D < MT) xa[(kb * MT + mt + D) & 3] = *(const u32x4_t*)(xl + cs + (mt + D) * 1024);
        else if (LOOK) xa[(kb * MT + mt + D) & 3] = *(const u32x4_t*)(xl + ns + (mt + D - MT) * 1024);
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            constexpr int F = MT * RT * 2;
            const int f = (mt * RT + r) * 2 + h;
            const u32x4_t& x = xa[(kb * MT + mt) & 3];
            if constexpr (KIND == 8) {
              inner[f & 3] = mfma_f16(x, ops[cur][r][h], zero);
              if (f >= LAG) fold(f - LAG, cur);
              else fold(F + f - LAG, nxt);     // the step before's (before the first: zeros)
              if (f == LAG) scales(nxt);
            } else if constexpr (!FLUSH) {
              acc[r][mt][h] = mfma_f16(x, ops[cur][r][h], acc[r][mt][h]);
            } else {
              prt[r][mt][h] = mfma_f16(x, ops[cur][r][h], kb == 0 ? zero : prt[r][mt][h]);
            }
            // one MFMA, then the part of the operand build that fits beside it: a wave issues in
            // order, so MFMAs back to back would hold the build up until the last has started
#pragma unroll
            for (int i = f * 4 * NR / MT; i < (f + 1) * 4 * NR / MT; ++i) half_piece(nxt, i);
            __builtin_amdgcn_sched_barrier(0);
          }
        // the half tile whose last operand data this step's build has used is loaded again
        if constexpr (kb == 2) {
          if (mt == 0) w_load(t + 1, std::integral_constant<int, 0>{});
        } else if constexpr (kb == 6) {
          if (mt == 0) w_load(t + 1, std::integral_constant<int, 1>{});
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (FLUSH && kb == 7) {
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[r][mt][h][e] += prt[r][mt][h][e];
      }
      // x of the steps that the next step reads (its own, and with LOOK the one after it) has
      // landed when at most the loads issued after it are in flight: x of the LATE steps last
      // issued, and the half tiles loaded since; the half tile whose operand data the next step
      // begins to read (kb 2, 6) when x of three steps is all that follows it
      constexpr int LATE = LOOK ? XD - 2 : XD - 1, AGO = (kb - 2) & 3;
      constexpr int X = LATE * U + ((AGO <= LATE) + (AGO + 4 <= LATE)) * WL;
      constexpr int N = AGO == 3 && X > 3 * U ? 3 * U : X;
      __builtin_amdgcn_s_waitcnt(vm_wait_pq(N));
      step_barrier();
    });
  }
  if constexpr (KIND == 8)
#pragma unroll
    for (int f = MT * RT * 2 - LAG; f < MT * RT * 2; ++f) fold(f, 1);
  for (int t = nt > 0 ? nt : 0; t < kq; ++t)   // a shorter part: the others' barriers
#pragma unroll
    for (int kb = 0; kb < 8; ++kb) step_barrier();

  // ---- the minimum term, in the same scale: A holds the S terms (ring steps after the last of
  // x), B u of the lane's two columns at groups 32 ch + 8 s + j (K-tile 4 ch + s; zero outside
  // the part). The next chunk's are loaded while this one's are used.
  const int nc_all = KIND != 4 ? 0 : WK == 1 ? nc : (kq + 2 * kPqChunkTiles - 2) / kPqChunkTiles;   // any part's, at most
  const uint8_t* sx[U];
#pragma unroll
  for (int j = 0; j < U; ++j)
    sx[j] = (const uint8_t*)p.xt + ((size_t)(mblk * MT + wn + WN * j) * unit_steps +
                                    a.k_t * 8 + ch0 * 2) * 1024;
  for (int i = 0; i < nc_all; ++i) {
    __builtin_amdgcn_s_waitcnt(vm_wait_pq(0));
    __syncthreads();
    if (i >= nc) continue;
    const int kt = kPqChunkTiles * (ch0 + i) + s;
    const bool in = WK == 1 || (kt >= kt0 && kt < kt1);
    u32x4_t uu[RT][2][2];                      // [hi, lo][even, odd column]
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const u32x4_t v = *(const u32x4_t*)(lds + wslot + (r * 2 + (e >> 1)) * HALF +
                                            (e & 1) * 1024 + l16);
        uu[r][e >> 1][e & 1] = in ? v : u32x4_t{0, 0, 0, 0};
      }
    if (i + 1 < nc) {
#pragma unroll
      for (int e = 2; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < U; ++j)
          ldl16d(sx[j] + (size_t)(2 * i + e) * 1024, l16,
                 xm0 + (((2 * i + e) & (RING - 1)) * MT + WN * j) * 1024);
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {              // the sums' high terms, then the low ones
      const uint8_t* xs = xl + ((2 * i + e) & (RING - 1)) * MT * 1024;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const u32x4_t x = *(const u32x4_t*)(xs + mt * 1024);
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            f32x4_t& t = FLUSH ? prt[FLUSH ? r : 0][FLUSH ? mt : 0][h] : acc[r][mt][h];
            if (e == 0) t = mfma_f16(x, uu[r][1][h], FLUSH && i == 0 ? zero : t);
            t = mfma_f16(x, uu[r][0][h], t);
          }
      }
      if (e == 0 && i + 1 < nc) {              // u is in registers: its slots are free
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int k = 0; k < 4; ++k)
            ldl16d(up[r] + (size_t)(i + 1) * 4096 + k * 1024, l16,
                   wm0 + (r * 2 + (k >> 1)) * HALF + (k & 1) * 1024);
      }
    }
  }
  if constexpr (FLUSH && KIND == 4) {
    if (nc > 0) {
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[r][mt][h][e] += prt[r][mt][h][e];
    }
  }
  __builtin_amdgcn_s_waitcnt(vm_wait_pq(0));   // the loads past the end have landed
  __syncthreads();

  // ---- to the true scale: rows 4 s + e of each m-tile
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int4 xs = *(const int4*)(p.xshift + m0 + 16 * mt + 4 * s);
    const int xsh[4] = {xs.x >> 1, xs.y >> 1, xs.z >> 1, xs.w >> 1};
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[r][mt][h][e] = ldexpf(acc[r][mt][h][e], -(shw[r][h] + xsh[e]));
  }

  // ---- the K parts, added in part order by part 0's wave
  if constexpr (WK > 1) {
    constexpr int REC = RT * MT * 2;           // f32x4 per lane
    f32x4_t* red = (f32x4_t*)lds;
    if (wk > 0) {
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            red[(((wk - 1) * WN + wn) * REC + (r * MT + mt) * 2 + h) * 64 + l] = acc[r][mt][h];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll 1
    for (int k = 1; k < WK; ++k)
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const f32x4_t v = red[(((k - 1) * WN + wn) * REC + (r * MT + mt) * 2 + h) * 64 + l];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[r][mt][h][e] += v[e];
          }
  }

  store(acc, m0, 16 * MT);
}

// ---------------------------------------------------------------- host side

size_t pq_align(size_t b) { return (b + 255) & ~(size_t)255; }
int pq_mtiles(int m_rows) { return (m_rows + 127) / 128 * 8; }   // whole 128-row blocks

// The pre-pass's buffers in a workspace (nullptr: their total size)
size_t pq_layout(void* ws, int kind, int tensors, int n_tr, int k_t, int m_rows, bool xe, PqX* x) {
  const size_t mt = pq_mtiles(m_rows), tr = (size_t)tensors * n_tr;
  const size_t ch = kind == Q4NX_KIND_Q4 ? pq_chunks<4>(k_t) : pq_chunks<8>(k_t);
  size_t off = 0;
  auto take = [&](size_t bytes) {
    uint8_t* b = (uint8_t*)ws + off;
    off += pq_align(bytes);
    return b;
  };
  x->xt = (u32x4_t*)take(mt * (k_t * 8 + ch * 2) * 1024 + kPqSlack);
  x->u = (u32x4_t*)take(tr * ch * 4 * 1024);
  x->scale = (uint2*)take(kind == Q4NX_KIND_Q4 ? tr * k_t * 1024 : 0);
  x->xshift = (int*)take(mt * 16 * 4);
  x->wshift = (int*)take(tr * 32 * 4);
  x->xe = (uint16_t*)take(xe ? (size_t)m_rows * k_t * kTileK * 2 : 0);
  return off;
}

template <int KIND, int OP, int MT, int RT, int WN, int WK, int RING, int OCC>
void pq_go(const GemmArgs& a, PqX x, hipStream_t st) {
  constexpr int ring = WK * RING * MT * 1024 + WN * WK * RT * 2 * kPqHalf<KIND>;
  constexpr int red = (WK - 1) * WN * RT * MT * 2 * 1024;
  constexpr int lds = ring > red ? ring : red;
  static_assert(lds <= 160 * 1024);
  const int units = OP == GOP_PLAIN ? (a.n_tr[0] + RT - 1) / RT : a.n_tr[0];
  x.m_blocks = (a.m_rows + 16 * MT - 1) / (16 * MT);
  x.c_groups = (units + WN - 1) / WN;
  // Weights beyond the eight L2s (4 MB each) would be read from memory again for every row block.
  // The dispatcher deals workgroups to the XCDs in turn, so each XCD then takes an eighth of the
  // tiles, all row blocks of a group of columns before the next group. Columns first / rows first,
  // us: 248320 x 1024 (q8, 258 MB), 512 rows 443..471 / 406, 200 rows 225 / 209; 163200 x 2048 (q4,
  // 199 MB), 102 rows 143 / 134; 26272 x 2304 (q4, 36 MB), 300 rows 74.5 / 72.5; smaller weights stay
  // in column order: 8192 x 4096 (q4, 20 MB), 1000 rows 75.3 / 74.8, 2560 x 8192 (12 MB) 70 / 81.
  x.rows_first = (size_t)a.n_tr[0] * (OP == GOP_PLAIN ? 1 : 2) * a.k_t * GemmFmt<KIND>::kTile > (32u << 20);
  const int tiles = x.c_groups * x.m_blocks;
  const dim3 grid((unsigned)((tiles + 7) / 8 * 8));
  hipLaunchKernelGGL((pq_kernel<KIND, OP, MT, RT, WN, WK, RING, OCC>), grid, dim3(64 * WN * WK),
                     lds, st, a, x);
}

template <int KIND, bool NORM>
void pq_prep(const GemmArgs& a, const PqX& x, int tensors, hipStream_t st) {
  const int tile_rows = a.n_tr[0] * tensors;
  const auto go = [&](auto rows, auto threads) {
    constexpr int ROWS = decltype(rows)::value, NT = decltype(threads)::value;
    hipLaunchKernelGGL((pq_prep_kernel<KIND, NORM, 2, NT, ROWS>),
                       dim3((unsigned)((a.m_rows + ROWS - 1) / ROWS + tile_rows)), dim3(NT), 0, st,
                       a, x, tile_rows);
  };
  if (a.k_t <= 4) go(std::integral_constant<int, 4>{}, std::integral_constant<int, 256>{});
  else if (a.k_t <= 16) go(std::integral_constant<int, 1>{}, std::integral_constant<int, 256>{});
  else go(std::integral_constant<int, 1>{}, std::integral_constant<int, 512>{});
}

}  // namespace

size_t pq_ws_bytes(int kind, int op, int n_tile_rows, int k_t, int m_rows, bool own_norm) {
  PqX x;
  return pq_layout(nullptr, kind, op == GOP_GATEUP ? 2 : 1, n_tile_rows, k_t, m_rows, own_norm, &x);
}

bool pq_use(int kind, int op, const GemmArgs& a) {
  if (op == GOP_QKV || a.m_rows < kPqRows || a.argmax_keys != nullptr) return false;
  // a lane's offset in its 16 rows has 32 bits
  constexpr int64_t kMaxStride = 1 << 25;
  if (op == GOP_PLAIN) {
    if (a.y_stride >= kMaxStride) return false;
    // q4: a lane's two columns are adjacent and are read and written as one 8-byte pair (q8: they
    // lie in different row blocks)
    return kind == Q4NX_KIND_Q8 ||
           (Q4NX_ALIGNED(a.y, 8) && Q4NX_ALIGNED(a.residual, 8) && a.y_stride % 2 == 0);
  }
  // pairs of bf16 as one word, pairs of fp32 as one 8-byte piece
  return a.h_stride < kMaxStride && Q4NX_ALIGNED(a.h_out, 4) && a.h_stride % 2 == 0 &&
         Q4NX_ALIGNED(a.raw_out, 8);
}

// Whether w workgroups that take a CU each leave at most an eighth of their rounds idle
static bool fills_cus(int w) { return w >= 224 && w * 8 >= (w + 255) / 256 * 256 * 7; }

// Tile by the workgroups it gives a chip of 256 CUs, two on each: the largest that fills it.
// Measured over N x K of 512 x 1024 to 12288 x 4096 (q8: to 248320 x 1024) and 65 to 3000 rows; us
// at the side of each line where the two are closest (N x K, rows):
PqTile pq_plain_tile(int kind, int n_tr, int k_t, int m_rows, bool ssq) {
  const auto wgs = [&](int rows, int trs) {
    return ((m_rows + rows - 1) / rows) * ((n_tr + trs - 1) / trs);
  };
  const int w64 = wgs(64, 4);
  if (kind == Q4NX_KIND_Q4) {
    // 128 rows x 8 tile-rows, eight waves with K in two parts, one workgroup per CU, against the
    // same in one part and 64 x 4 (workgroups): 8192 x 2560 256 55.5 / 54.9 / 58.3, 512 100 / 86 /
    // 103; 4096 x 4096 256 73.9 / 74.8 / 84.6; 2560 x 8192, 3000 rows (240) 133 / 140 / 161; one that
    // leaves CUs idle in its last round loses (10240 x 4096 320 125 / 109 / 101). Its chains over K
    // are half as long, so launches with sums of squares, formerly the batched kernel's, take it
    // or 64 x 4 (768 144 / 148) where one chain is the less exact, from K = 1024 on.
    const bool exact = ssq && k_t >= 4;
    const int w0 = m_rows < 128 ? 0 : wgs(128, 8);
    if (k_t >= 8 && fills_cus(w0) && (w0 <= 256 || exact))
      return {128, 8, 2};
    // the same in one part against 64 x 4: 640 rows (160) 53 / 47; a short K does not repay the
    // larger block's epilogue (6144 x 1024, 1500 rows (288) 44 / 38), and with fewer rows than the
    // block has the others are as fast and nearer to the 64-bit result
    if (!exact && (w0 >= 512 || (w0 >= 240 && k_t >= 8)))
      return {128, 8, 1};
    // 64 x 4 against 64 x 2 with K in two parts: 2560 x 8192, 1500 rows (480) 90 / 99, 1000 rows
    // (320) 80 / 72
    if (w64 >= 440) return {64, 4, 1};
  } else {
    // 128 rows x 4 tile-rows (eight would take the LDS of both workgroups of a CU) against the
    // next: 8192 x 2560, 1000 rows (512) 68 / 79, 768 rows (384) 65 / 65, 640 rows (320) 64 / 60
    if (wgs(128, 4) >= 384) return {128, 4, 1};
    // 64 x 4 when it fills the chip once, against 64 x 2 with K in two parts: 8192 x 2560, 400
    // rows (448) 40 / 43, 320 rows (320) 39 / 37, 640 rows (640) 62 / 60
    if (w64 >= 440 && w64 <= 512) return {64, 4, 1};
  }
  // two parts against four: 2560 x 8192, 400 rows (280) q4 50 / 56, q8 61 / 68, 256 rows (160)
  // q4 40 / 36, q8 46 / 40
  if (wgs(64, 2) > 256) return {64, 2, 2};
  // 64 x 2 in four parts against 32 x 2: 2560 x 8192, 256 rows (160) q4 36 / 48, q8 40 / 52, 192
  // rows (120) q4 35 / 31, q8 39 / 32
  if (wgs(64, 2) >= 160) return {64, 2, 4};
  // 32 x 2 in four parts against 32 x 1 in eight: 2560 x 2560, 128 rows (320) q4 16 / 22, q8 16 /
  // 21, 96 rows (240) q4 16 / 14, q8 16 / 14
  if (wgs(32, 1) > 256) return {32, 2, 4};
  return {32, 1, 8};
}

template <int KIND>
static void pq_plain(const GemmArgs& a, const PqX& x, hipStream_t st) {
  const PqTile t = pq_plain_tile(KIND, a.n_tr[0], a.k_t, a.m_rows, a.ssq_out != nullptr);
  const auto is = [&](int rows, int trs, int parts) {
    return t.rows == rows && t.tile_rows == trs && t.parts == parts;
  };
  if constexpr (KIND == 4) {
    if (is(128, 8, 2)) return pq_go<4, GOP_PLAIN, 8, 2, 4, 2, 4, 2>(a, x, st);
    if (is(128, 8, 1)) return pq_go<4, GOP_PLAIN, 8, 2, 4, 1, 4, 2>(a, x, st);
  } else {
    if (is(128, 4, 1)) return pq_go<8, GOP_PLAIN, 8, 1, 4, 1, 4, 2>(a, x, st);
  }
  if (is(64, 4, 1)) return pq_go<KIND, GOP_PLAIN, 4, 1, 4, 1, 8, 2>(a, x, st);
  if (is(64, 2, 2)) return pq_go<KIND, GOP_PLAIN, 4, 1, 2, 2, 4, 2>(a, x, st);
  if (is(64, 2, 4)) return pq_go<KIND, GOP_PLAIN, 4, 1, 2, 4, 4, 2>(a, x, st);
  if (is(32, 2, 4)) return pq_go<KIND, GOP_PLAIN, 2, 1, 2, 4, 8, 2>(a, x, st);
  pq_go<KIND, GOP_PLAIN, 2, 1, 1, 8, 4, 2>(a, x, st);
}

static void pq_gateup(const GemmArgs& a, const PqX& x, hipStream_t st) {
  const auto wgs = [&](int rows, int trs) {
    return ((a.m_rows + rows - 1) / rows) * ((a.n_tr[0] + trs - 1) / trs);
  };
  // 128 rows x 4 pairs, eight waves with K in two parts, one workgroup per CU, against 64 x 4 in one
  // part (128-row workgroups, us): 8192 x 2560 256 54.8 / 57.1, 1024 185 / 186; 4096 x 4096 224 67 /
  // 76, 512 135 / 146; 2560 x 8192 480 240 / 278; 10240 x 4096 400 121 / 111, 960 253 / 277; 6144 x 1536
  // 768 105 / 96. (In one part it takes 155 us for the 1024, but its chain over K is 3.2e-7 off at
  // K = 2560 where the batched kernel was 2.6e-7.)
  if (a.k_t >= 8 && a.m_rows >= 128 && fills_cus(wgs(128, 4)))
    return pq_go<4, GOP_GATEUP, 8, 2, 4, 2, 4, 2>(a, x, st);
  // 64 rows x 4 pairs, whole K, against 64 x 2 in two parts, which fill a last round of the 512
  // workgroups the chip holds more evenly (64 x 4 workgroups): 8192 x 2560 448 54 / 59, 576 75 / 72,
  // 640 76 / 74, 832 93 / 96; 4096 x 4096 320 72 / 66, 416 75 / 80, 608 110 / 102; 10240 x 4096 720
  // 111 / 118; a short K does not repay the parts: 2048 x 1024 144 19.6 / 19.3, 384 28.6 / 30.9, 6144
  // x 1536 144 26.2 / 26.7, 432 37 / 43
  const int w64 = wgs(64, 4);
  if (a.k_t <= 6 ? w64 >= 144 : w64 >= 400 && (w64 <= 512 || w64 >= 704))
    return pq_go<4, GOP_GATEUP, 4, 2, 4, 1, 4, 2>(a, x, st);
  // 64 x 2 against 32 x 2 in four parts: 2560 x 8192, 256 rows (160) 58 / 70, 192 rows (120)
  // 58 / 44
  if (wgs(64, 2) >= 160) return pq_go<4, GOP_GATEUP, 4, 2, 2, 2, 4, 2>(a, x, st);
  // 32 x 2 against 32 x 1 in eight parts: 2560 x 2560, 128 rows (320) 23 / 28, 96 rows (240)
  // 22 / 18
  if (wgs(32, 1) > 256) return pq_go<4, GOP_GATEUP, 2, 2, 2, 4, 4, 2>(a, x, st);
  pq_go<4, GOP_GATEUP, 2, 2, 1, 8, 4, 2>(a, x, st);
}

void pq_launch(int kind, int op, const GemmArgs& a, void* ws, hipStream_t st) {
  PqX x;
  const int tensors = op == GOP_GATEUP ? 2 : 1;
  const bool norm = a.norm_w != nullptr, own = norm && a.xn_out == nullptr;
  pq_layout(ws, kind, tensors, a.n_tr[0], a.k_t, a.m_rows, own, &x);
  x.exact = !norm ? a.x : own ? x.xe : a.xn_out;
  x.exact_stride = own ? (int64_t)a.k_t * kTileK : a.x_stride;
  x.exact_all = !own;
  if (kind == Q4NX_KIND_Q8) norm ? pq_prep<8, true>(a, x, tensors, st) : pq_prep<8, false>(a, x, tensors, st);
  else norm ? pq_prep<4, true>(a, x, tensors, st) : pq_prep<4, false>(a, x, tensors, st);
  if (op == GOP_GATEUP) pq_gateup(a, x, st);
  else if (kind == Q4NX_KIND_Q4) pq_plain<4>(a, x, st);
  else pq_plain<8>(a, x, st);
}

}  // namespace q4nx
