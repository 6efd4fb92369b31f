// Building blocks of the chunked gated delta rule, shared by the fused prefill
// kernel (gdn_prefill.hip, whose head states the algebra, the MFMA operand
// layouts and the precision) and the split one (gdn_prefill_split.hip): chunk
// tiles in LDS, their loads, the Gram products, T = (I + A)^-1 and P.
#ifndef GDN_CHUNK_H_
#define GDN_CHUNK_H_
#include "gdn_common.h"

namespace {


constexpr int C = 64;      // chunk
constexpr int KD = 128;    // key head dim
constexpr int VD = 128;    // value head dim
constexpr int LDK = 136;   // fp16 row stride of the K/Q tiles
constexpr int LDV = 144;   // bf16 row stride of the V tile (conflict-free transposed reads)
constexpr int LDH = 68;    // fp16 row stride of T_hi/T_lo/P

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct PrefillArgs {
  const bf16_t* q; const bf16_t* k; const bf16_t* v; const float* g; const void* beta;
  float* state; const void* idx; const void* cu; bf16_t* out;
  int64_t q_s0, q_s1, k_s0, k_s1, v_s0, v_s1, g_s0, g_s1, b_s0, b_s1, o_s0, o_s1;
  int64_t st_slot, st_head;
  int64_t T, nseq, num_slots;
  int32_t Hv, r;
  int32_t b_dtype;
  float scale;
  int32_t spin_limit;  // bound of a producer wait (sleep iterations)
  int32_t per_wg;      // 0: one item per workgroup, longest first; > 0: runs of work ids dealt by cost
  int32_t kd, vd;      // key and value head dims (multiples of 8 up to 128; smaller ones run zero-padded)
  int32_t flags;       // GDN_PREFILL_ZERO_INIT | GDN_PREFILL_ACCUM_STATE | GDN_PREFILL_ACCUM_OUT
  bool idx64, cu64;
};

// On-chip data.  The state waves work on chunk c while the producers stage
// chunk c + 1 and solve the diagonal blocks of T for chunk c + 2:
//  * per-chunk tiles, double-buffered by chunk parity (44,816 bytes each);
//  * T of three consecutive chunks, rotating (17,408 bytes each);
//  * one V tile: the state waves signal when they have read chunk c's
//    values, and only then is chunk c + 1's written.
struct ChunkTiles {
  f16_t k[C * LDK];
  f16_t q[C * LDK];  // chunk queries (the output is staged in the V tile)
  f16_t p[C * LDH];  // P (fp16), lower triangle
  alignas(16) float gam[C];
  alignas(16) float eg[C];    // e^gamma
  alignas(16) float ieg[C];   // e^-gamma
  alignas(16) float edec[C];  // e^(gamma_L - gamma), 0 past the chunk's last token
  alignas(16) float beta[C];
  float gam_last;
  int32_t fact;  // every |gamma| < 80: e^(gamma_i - gamma_j) = e^gamma_i e^-gamma_j (both normal)
};

// T = (I + A)^-1 as fp16 hi + lo.  Block (0,1) (rows 0..31,
// columns 32..63) is zero and never read by the state waves; the producers
// keep A_10 there, and while the diagonal blocks are being solved the two
// off-diagonal blocks hold the fp32 working copies of the diagonal blocks.
struct TBuf {
  f16_t hi[C * LDH];
  f16_t lo[C * LDH];
};

static_assert(sizeof(ChunkTiles) == 44816 && sizeof(TBuf) == 17408, "tile sizes as documented above");

GDN_DEVICE f32x16 mfma32(f16x8 a, f16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
GDN_DEVICE f32x4 mfma16(f16x4 a, f16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
}

GDN_DEVICE f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int j = 0; j < 16; ++j) z[j] = 0.f;
  return z;
}

GDN_DEVICE f16x8 cat4(f16x4 lo, f16x4 hi) {
  return (f16x8){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

// Fragment of a row-major fp16 LDS matrix M: lane holds M[r0 + n][k-step
// slots] -- an A operand (rows of M are the M dim) or a B operand of M^T.
GDN_DEVICE f16x8 frag_rows(const f16_t* M, int ld, int r0, int kbase, int lane) {
  const f16_t* p = M + (r0 + (lane & 31)) * ld + kbase + 4 * (lane >> 5);
  return cat4(*reinterpret_cast<const f16x4*>(p), *reinterpret_cast<const f16x4*>(p + 8));
}

// Transposed read of a row-major 16-bit LDS matrix (ds_read_b64_tr_b16: each
// 16-lane group reads a 4x16 block, lane i gets column i).
GDN_DEVICE s16x4 tr_read(const void* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
}
// Fragment of the transpose of a row-major fp16 LDS matrix M: lane holds
// M[k-step slots][c0 + n].
GDN_DEVICE f16x8 frag_cols(const f16_t* M, int ld, int c0, int kbase, int lane) {
  const int j = lane & 15, qd = lane >> 4;
  const f16_t* p = M + (kbase + 4 * (qd >> 1) + (j >> 2)) * ld + c0 + 16 * (qd & 1) + 4 * (j & 3);
  return cat4(__builtin_bit_cast(f16x4, tr_read(p)), __builtin_bit_cast(f16x4, tr_read(p + 8 * ld)));
}

// K and Q tiles are stored with the middle two 4-element quads of every
// 16-column group swapped (logical quad q at stored quad kq_quad(q)), so that
// the 8 k-values a lane takes for one 16-wide k-step (logical columns 4g..4g+3
// and 8+4g..8+4g+3) are 16 contiguous bytes: one ds_read_b128 per fragment
// instead of two ds_read_b64 (a wave issues one LDS read per ~35 cycles
// whatever its width, so the count of reads is what costs).  A Gram of two
// such tiles needs nothing else; the transposed reads of K (K^T as an A
// operand, whose rows are K's columns) permute their quad addresses so the
// lanes still receive logical columns in order.
GDN_DEVICE int kq_quad(int q) { return ((q & 1) << 1) | (q >> 1); }
GDN_DEVICE f16x8 frag_rows_kq(const f16_t* M, int r0, int kbase, int lane) {
  return *reinterpret_cast<const f16x8*>(M + (r0 + (lane & 31)) * LDK + kbase + 8 * (lane >> 5));
}
GDN_DEVICE f16x8 frag_cols_kq(const f16_t* M, int c0, int kbase, int lane) {
  const int j = lane & 15, qd = lane >> 4;
  const f16_t* p = M + (kbase + 4 * (qd >> 1) + (j >> 2)) * LDK + c0 + 16 * (qd & 1) + 4 * kq_quad(j & 3);
  return cat4(__builtin_bit_cast(f16x4, tr_read(p)), __builtin_bit_cast(f16x4, tr_read(p + 8 * LDK)));
}

// Per-row vector entries for C-layout rows r0 + 8i + 4g + (0..3).
GDN_DEVICE f32x4 rows4(const float* vec, int r0, int i, int lane) {
  return *reinterpret_cast<const f32x4*>(vec + r0 + 8 * i + 4 * (lane >> 5));
}

// Maximum of |x| over one value column of the wave's `nt` C tiles.  In the
// C layout lanes l and l ^ 32 hold the two row halves of column l % 32, so
// the per-lane maximum (a tree of a few dependent operations) needs one
// exchange between the wave halves; no wave-wide reduction.  Non-negative
// floats order like their bit patterns, so the exchange takes the maximum on
// integers.
GDN_DEVICE float col_max(const f32x16* t, int nt) {
  float m[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    m[j] = fabsf(t[0][j]);
    for (int i = 1; i < nt; ++i) m[j] = fmaxf(m[j], fabsf(t[i][j]));
  }
#pragma unroll
  for (int w = 8; w >= 1; w >>= 1)
#pragma unroll
    for (int j = 0; j < w; ++j) m[j] = fmaxf(m[j], m[j + w]);
  const uint32_t v = __builtin_bit_cast(uint32_t, m[0]);
  const auto sw = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return __builtin_bit_cast(float, max(sw[0], sw[1]));
}

// Exponent E with max|x| in [2^(E-1), 2^E) over one value column, kNone
// when the column is zero.
constexpr int kNone = -4096;
GDN_DEVICE int col_max_exp(const f32x16* t, int nt) {
  const float mx = col_max(t, nt);
  return mx > 0.f ? __builtin_amdgcn_frexp_expf(mx) : kNone;
}

// Power-of-two exponent e with max|x| * 2^-e in [2^9, 2^10) over one value
// column (0 when the column is zero).
GDN_DEVICE int col_scale_exp(const f32x16* t, int nt) {
  const int e = col_max_exp(t, nt);
  return e == kNone ? 0 : e - 10;
}

// Inclusive prefix sum over the 64 lanes (DPP row shifts, then the row
// broadcasts of the last lane of each row).
GDN_DEVICE float wave_inclusive_scan(float x) {
  x += __builtin_amdgcn_update_dpp(0.f, x, 0x111, 0xF, 0xF, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0.f, x, 0x112, 0xF, 0xF, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0.f, x, 0x114, 0xF, 0xF, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0.f, x, 0x118, 0xF, 0xF, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0.f, x, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1, 3
  x += __builtin_amdgcn_update_dpp(0.f, x, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2, 3
  return x;
}

// Maximum over the 64 lanes of a non-negative float (bit patterns order like the values).
GDN_DEVICE float wave_max(float x) {
  int v = __builtin_bit_cast(int, x);
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false));  // row_shr:1
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false));  // row_shr:2
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false));  // row_shr:4
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false));  // row_shr:8
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false));  // row_bcast:15
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false));  // row_bcast:31
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(v, 63));
}

// hi/lo fp16 splits: hi = fp16(x) (round to nearest even), lo = fp16(x - hi).
// hi is converted once and its bits are pinned through an empty asm, so the
// x - hi below is taken from exactly the bits that are stored as hi.  (If the
// compiler is left to convert x twice it may pick the packed and the scalar
// float->fp16 instructions for the two uses, and those can disagree on exact
// rounding ties, which leaves lo referenced to a different hi.)
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
GDN_DEVICE void split_pair(float x0, float x1, f16_t& h0, f16_t& h1, f16_t& l0, f16_t& l1) {
  const f32x2 x = {x0, x1};
  uint32_t hb = __builtin_bit_cast(uint32_t, __builtin_convertvector(x, f16x2));
  asm volatile("" : "+v"(hb));
  const f16x2 h = __builtin_bit_cast(f16x2, hb);
  const f32x2 r = {x0 - (float)h[0], x1 - (float)h[1]};
  const f16x2 l = __builtin_convertvector(r, f16x2);
  h0 = h[0];
  h1 = h[1];
  l0 = l[0];
  l1 = l[1];
}

// Scaled fp16 hi/lo pairs: hi = fp16(x s) and lo = fp16(x s - hi) (s a
// power of two times a per-element factor, so x s - hi is exact in fp32 and
// each half is rounded once).  hi's bits are pinned through an empty asm, so
// lo is referenced to exactly the stored hi bits whichever conversion
// instructions the compiler picks for the two uses.  (Plain code rather than
// hand-written v_fma_mix* instructions: the compiler pads an MFMA's operand
// reads after VALU writes only for instructions it generated itself.)  A
// scale per element lets a per-row factor ride along (C-layout neighbours
// are adjacent rows).
GDN_DEVICE uint32_t mix_hi_pair(float x0, float s0, float x1, float s1) {
  const f16x2 h = {(f16_t)(x0 * s0), (f16_t)(x1 * s1)};
  uint32_t hb = __builtin_bit_cast(uint32_t, h);
  asm volatile("" : "+v"(hb));
  return hb;
}
GDN_DEVICE uint32_t mix_lo_pair(float x0, float s0, float x1, float s1, uint32_t hb) {
  const f16x2 h = __builtin_bit_cast(f16x2, hb);
  const f16x2 l = {(f16_t)__builtin_fmaf(x0, s0, -(float)h[0]), (f16_t)__builtin_fmaf(x1, s1, -(float)h[1])};
  return __builtin_bit_cast(uint32_t, l);
}

// split of registers 8h..8h+7 of a C tile, times sc
GDN_DEVICE void split8(const f32x16& c, int h, float sc, f16x8& hi, f16x8& lo) {
  uint32_t H[4], L[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    H[m] = mix_hi_pair(c[8 * h + 2 * m], sc, c[8 * h + 2 * m + 1], sc);
    L[m] = mix_lo_pair(c[8 * h + 2 * m], sc, c[8 * h + 2 * m + 1], sc, H[m]);
  }
  hi = __builtin_bit_cast(f16x8, (u32x4){H[0], H[1], H[2], H[3]});
  lo = __builtin_bit_cast(f16x8, (u32x4){L[0], L[1], L[2], L[3]});
}
// the same unscaled: hi = fp16(x), lo = fp16(fma(x, one, -hi)) with one = 1
// held opaque by the caller (the compiler would otherwise fold the fma into a
// subtraction and convert hi back to fp32 first)
GDN_DEVICE void split8u(const f32x16& c, int h, float one, f16x8& hi, f16x8& lo) {
  uint32_t H[4], L[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const f16x2 hv = {(f16_t)c[8 * h + 2 * m], (f16_t)c[8 * h + 2 * m + 1]};
    H[m] = __builtin_bit_cast(uint32_t, hv);
    asm volatile("" : "+v"(H[m]));
    L[m] = mix_lo_pair(c[8 * h + 2 * m], one, c[8 * h + 2 * m + 1], one, H[m]);
  }
  hi = __builtin_bit_cast(f16x8, (u32x4){H[0], H[1], H[2], H[3]});
  lo = __builtin_bit_cast(f16x8, (u32x4){L[0], L[1], L[2], L[3]});
}
// the same with one factor per register (f[m] scales register 8h + m)
GDN_DEVICE void split8f(const f32x16& c, int h, const float (&f)[8], f16x8& hi, f16x8& lo) {
  uint32_t H[4], L[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    H[m] = mix_hi_pair(c[8 * h + 2 * m], f[2 * m], c[8 * h + 2 * m + 1], f[2 * m + 1]);
    L[m] = mix_lo_pair(c[8 * h + 2 * m], f[2 * m], c[8 * h + 2 * m + 1], f[2 * m + 1], H[m]);
  }
  hi = __builtin_bit_cast(f16x8, (u32x4){H[0], H[1], H[2], H[3]});
  lo = __builtin_bit_cast(f16x8, (u32x4){L[0], L[1], L[2], L[3]});
}
template <int N>
GDN_DEVICE void split_vec(const float* x, f16_t* hi, f16_t* lo) {
  static_assert(N % 2 == 0, "pairs");
#pragma unroll
  for (int m = 0; m < N; m += 2) split_pair(x[m], x[m + 1], hi[m], hi[m + 1], lo[m], lo[m + 1]);
}

// ---- T = (I + A)^-1 pieces ---------------------------------------------------------
//
// With A = strict_lower(beta_i k_i.k_j e^(gamma_i - gamma_j)), T = (I + A)^-1 is
// unit lower triangular and block lower triangular over the two 32-token
// halves, and its off-diagonal block satisfies
//   T_10 = -T_11 A_10 T_00,
// so each diagonal block is solved on its own (one wave each) and the
// off-diagonal block needs only the fp16 hi/lo of T_00, T_11 and A_10.  (beta
// scales the rows of R instead of the columns of T: with T' = T diag(beta)
// a small beta pushed T' into fp16's subnormal range, where its split lost
// precision.)

// fp32 working copy of a 32x32 diagonal block, kept in the two fp16 arrays
// of an off-diagonal block of the same T buffer: row i's columns 0..15 in
// the hi array, 16..31 in the lo array (64 bytes each, 8-byte aligned).
struct Scratch {
  // byte address of the block's row 0 in the hi array; the lo array follows
  // the hi array at a fixed distance, so a lane-dependent half is an integer
  // offset (a select between two pointers went through private memory and
  // turned the LDS accesses into flat ones)
  char* hi;
  static constexpr int kLoOff = C * LDH * (int)sizeof(f16_t);
  GDN_DEVICE float* row(int i, int half) const { return reinterpret_cast<float*>(hi + half * kLoOff + i * (2 * LDH)); }
  GDN_DEVICE float& at(int i, int j) const { return row(i, j >> 4)[j & 15]; }
};
static_assert(offsetof(TBuf, lo) == Scratch::kLoOff, "TBuf: lo follows hi");
// diagonal block blk (0 or 1) of tb is worked on in its off-diagonal block (0,1) or (1,0)
GDN_DEVICE Scratch scratch_of(TBuf& tb, int blk) {
  const int off = blk == 0 ? 32 : 32 * LDH;  // halves
  return {reinterpret_cast<char*>(tb.hi + off)};
}
GDN_DEVICE f32x4 load4(const float* p) {
  const f32x2 a = *reinterpret_cast<const f32x2*>(p), b = *reinterpret_cast<const f32x2*>(p + 2);
  return (f32x4){a[0], a[1], b[0], b[1]};
}

// 16x16 diagonal blocks of a 32x32 strictly lower block A (fp32) by
// right-looking forward substitution, in place: lane (b, c) = ((lane / 16) % 2,
// lane % 16) computes column c of block b; lanes 32..63 repeat lanes 0..31 and
// do not store.
GDN_DEVICE void invert_diag16(const Scratch& A, int lane) {
  const int b = (lane >> 4) & 1, c = lane & 15;
  float y[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) y[i] = i == c ? 1.f : 0.f;
#pragma unroll
  for (int kk = 0; kk < 16; kk += 2) {  // two columns of A per read
    f32x2 ak[16];
#pragma unroll
    for (int i = kk + 1; i < 16; ++i) ak[i] = *reinterpret_cast<const f32x2*>(A.row(16 * b + i, b) + kk);
#pragma unroll
    for (int i = kk + 1; i < 16; ++i) y[i] = fmaf(-ak[i][0], y[kk], y[i]);
#pragma unroll
    for (int i = kk + 2; i < 16; ++i) y[i] = fmaf(-ak[i][1], y[kk + 1], y[i]);
  }
  if (lane < 32) {
#pragma unroll
    for (int i = 0; i < 16; ++i) A.row(16 * b + i, b)[c] = y[i];
  }
}

GDN_DEVICE void split4(f32x4 x, f16x4& hi, f16x4& lo) {
  float xs[4] = {x[0], x[1], x[2], x[3]};
  f16_t h[4], l[4];
  split_vec<4>(xs, h, l);
  hi = (f16x4){h[0], h[1], h[2], h[3]};
  lo = (f16x4){l[0], l[1], l[2], l[3]};
}

// 16 -> 32 merge inside a 32x32 block whose diagonal 16-blocks hold their
// inverses: T_10 = -T_11 A_10 T_00, with 16x16x16 MFMAs on hi/lo splits.
GDN_DEVICE void merge16(const Scratch& A, int lane) {
  const int n = lane & 15, g4 = 4 * (lane >> 4);
  f16x4 ah, al, bh, bl;
  // M = A_10 T_00: A operand = rows of A_10, B operand = columns of T_00
  split4(load4(A.row(16 + n, 0) + g4), ah, al);
  {
    f32x4 y;
#pragma unroll
    for (int m = 0; m < 4; ++m) y[m] = A.row(g4 + m, 0)[n];
    split4(y, bh, bl);
  }
  f32x4 M = {0.f, 0.f, 0.f, 0.f};
  M = mfma16(ah, bh, M);
  M = mfma16(ah, bl, M);
  M = mfma16(al, bh, M);
  // T_10 = -T_11 M: A operand = rows of T_11, B operand = M (C layout rows == k)
  split4(load4(A.row(16 + n, 1) + g4), ah, al);
  split4(M, bh, bl);
  f32x4 R = {0.f, 0.f, 0.f, 0.f};
  R = mfma16(ah, bh, R);
  R = mfma16(ah, bl, R);
  R = mfma16(al, bh, R);
#pragma unroll
  for (int m = 0; m < 4; ++m) A.row(16 + g4 + m, 0)[n] = -R[m];
}

// Where a (sequence, v-head) reads its chunks from.
struct ChunkSource {
  const PrefillArgs* a;
  const bf16_t* kg;  // k-head base
  const bf16_t* qg;  // k-head base
  const bf16_t* vg;  // v-head base
  int h;             // v-head
  int64_t e;         // end token of the sequence
};

GDN_DEVICE int chunk_rows(const ChunkSource& src, int64_t c0) {
  const int64_t rem = src.e - c0;
  return (int)(rem < C ? rem : C);
}

// Rows past the chunk's last token are loaded from the last token instead
// (no divergent loads, so nothing waits on them early): they are inert
// because their g, beta and e^(gamma_L - gamma) are set to zero, which zeroes
// their rows of R and their rows and columns of A (T keeps a unit row and
// column for them) and their share of the state update, and their output rows
// are not stored.
//
// 16 bytes of row `row` of a chunk (uniform base pointer of the chunk's first
// token + a 32-bit lane offset; the host guarantees 64 token strides fit).
GDN_DEVICE bf16x8 load_row_piece(const bf16_t* chunk_base, uint32_t stride, int row, int col, int Lc) {
  const uint32_t rc = (uint32_t)(row < Lc ? row : Lc - 1);
  const uint32_t byte_off = (rc * stride + (uint32_t)col) * (uint32_t)sizeof(bf16_t);
  return *reinterpret_cast<const bf16x8*>(reinterpret_cast<const char*>(chunk_base) + byte_off);
}

// A whole 64 x 128 chunk tile in one wave's registers: vector u of lane l is
// row l / 16 + 4u, columns 8 (l % 16) .. +7.
struct TileLoad {
  bf16x8 r[16];
};
// With a head dim below 128 (dim), a lane whose columns lie past it reads
// column 0 instead (in bounds); staging zeroes them.
GDN_DEVICE void load_tile(TileLoad& tl, const bf16_t* head_base, int64_t stride, int64_t c0, int Lc, int lane,
                          int dim = KD) {
  const bf16_t* b = head_base + c0 * stride;
  const int col = 8 * (lane & 15) < dim ? 8 * (lane & 15) : 0;
#pragma unroll
  for (int u = 0; u < 16; ++u) tl.r[u] = load_row_piece(b, (uint32_t)stride, (lane >> 4) + 4 * u, col, Lc);
}

// g and beta (raw bits) of token `lane` of a chunk.
struct DecayLoad {
  float g;
  ScalarRaw b;
};
GDN_DEVICE void load_decay(DecayLoad& dl, const ChunkSource& src, int64_t c0, int Lc, int lane) {
  const PrefillArgs& a = *src.a;
  const int64_t t = c0 + (lane < Lc ? lane : Lc - 1);
  dl.g = a.g[t * a.g_s0 + src.h * a.g_s1];
  dl.b = load_scalar_raw(a.beta, t * a.b_s0 + src.h * a.b_s1, a.b_dtype);
}

// K fragments of a diagonal block's 32 rows (lane (n, g) holds row 32 blk + n,
// columns 16 ks + 8 g .. +7) and the chunk's decays.
struct DiagLoad {
  bf16x8 kf[8];
  DecayLoad d;
};
GDN_DEVICE void load_diag(DiagLoad& dl, const ChunkSource& src, int64_t c0, int blk, int lane, int dim = KD) {
  const PrefillArgs& a = *src.a;
  const int Lc = chunk_rows(src, c0);
  const bf16_t* kb = src.kg + c0 * a.k_s0;
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) {
    const int col = 16 * ks + 8 * (lane >> 5);
    dl.kf[ks] = load_row_piece(kb, (uint32_t)a.k_s0, 32 * blk + (lane & 31), col < dim ? col : 0, Lc);
  }
  load_decay(dl.d, src, c0, Lc, lane);
}

// bf16 -> fp16 of 8 values (exact for |x| in the fp16 normal range): the
// bf16 bits widened to fp32 by a shift or mask, then one packed conversion
// per pair.
GDN_DEVICE f16x8 bf16x8_to_f16x8(bf16x8 x) {
  const u32x4 w = __builtin_bit_cast(u32x4, x);
  u32x4 o;
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const f32x2 f = {__builtin_bit_cast(float, w[m] << 16), __builtin_bit_cast(float, w[m] & 0xffff0000u)};
    o[m] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2));
  }
  return __builtin_bit_cast(f16x8, o);
}

// The kernel reads q/k/v and writes o as 16-bit floats of one type: bf16
// (F16 = false) or fp16 (F16 = true).  Loads and the V tile move raw bits;
// these convert at the points of use.
template <bool F16>
GDN_DEVICE f16x8 to_f16x8(bf16x8 raw) {
  if constexpr (F16) return __builtin_bit_cast(f16x8, raw);
  else return bf16x8_to_f16x8(raw);
}
template <bool F16>
GDN_DEVICE f32x4 to_f32x4(s16x4 raw) {
  f32x4 r;
  if constexpr (F16) {
    const f16x4 h = __builtin_bit_cast(f16x4, raw);
#pragma unroll
    for (int m = 0; m < 4; ++m) r[m] = (float)h[m];
  } else {
    const bf16x4 h = __builtin_bit_cast(bf16x4, raw);
#pragma unroll
    for (int m = 0; m < 4; ++m) r[m] = (float)h[m];
  }
  return r;
}
template <bool F16>
GDN_DEVICE s16x4 from_f32x4(f32x4 x) {
  if constexpr (F16) {
    const f16x4 h = {(f16_t)x[0], (f16_t)x[1], (f16_t)x[2], (f16_t)x[3]};
    return __builtin_bit_cast(s16x4, h);
  } else {
    const bf16x4 h = {(bf16_t)x[0], (bf16_t)x[1], (bf16_t)x[2], (bf16_t)x[3]};
    return __builtin_bit_cast(s16x4, h);
  }
}

// gamma = in-chunk cumsum of g (one token per lane) and the per-token decay
// vectors; g and beta of tokens past the chunk end are taken as zero.
// Whether every lane's |gamma| < 80, so that e^gamma and e^-gamma are both
// normal floats and e^(gamma_i - gamma_j) = e^gamma_i e^-gamma_j loses nothing
// (one rounding per factor instead of an exponential per element).  Wave-uniform.
GDN_DEVICE bool factorable(float gm) {
  return __builtin_amdgcn_ballot_w64(!(fabsf(gm) < 80.f)) == 0;
}

GDN_DEVICE float chunk_gamma(const DecayLoad& dl, int L, int lane, float& gl) {
  const float gm = wave_inclusive_scan(lane < L ? dl.g : 0.f);
  gl = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, gm), 63));  // gamma at token L-1
  return gm;
}

// Gram tile (mt, nt) of rows of M1 against rows of M2 (K = 128): C layout,
// lane holds column 32nt + n, rows 32mt + 8i + 4g + r.
GDN_DEVICE f32x16 gram_tile(const f16_t* M1, const f16_t* M2, int mt, int nt, int lane) {
  f32x16 G = zero16();
#pragma unroll
  for (int ks = 0; ks < KD / 16; ++ks)
    G = mfma32(frag_rows_kq(M1, 32 * mt, 16 * ks, lane), frag_rows_kq(M2, 32 * nt, 16 * ks, lane), G);
  return G;
}

// kk^T of a diagonal block's rows from the register fragments, in k's own
// 16-bit type (which holds k exactly)
template <bool F16>
GDN_DEVICE f32x16 gram_regs(const bf16x8 (&kf)[8]) {
  f32x16 G = zero16();
#pragma unroll
  for (int ks = 0; ks < KD / 16; ++ks) {
    if constexpr (F16) {
      const f16x8 h = __builtin_bit_cast(f16x8, kf[ks]);
      G = mfma32(h, h, G);
    } else {
      G = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[ks], kf[ks], G, 0, 0, 0);
    }
  }
  return G;
}

// e^(gamma_i - gamma_j) for token i of the lane and the tokens j = j0 + 8 i4 + 4g + r of its registers
GDN_DEVICE void row_decays(float (&d)[16], const float* gam, const float* eg, const float* ieg, bool fact, int i, int j0,
                           int lane) {
  if (fact) {
    const float ei = eg[i];
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const f32x4 ej = rows4(ieg, j0, i4, lane);
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) d[4 * i4 + rr] = ei * ej[rr];
    }
  } else {
    const float gi = gam[i];
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const f32x4 gj = rows4(gam, j0, i4, lane);
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) d[4 * i4 + rr] = __expf(gi - gj[rr]);
    }
  }
}

// Diagonal block `blk` of T: A_bb = strict_lower(beta_i k_i.k_j e^(g_i - g_j))
// from its kk^T tile, solved in fp32 in the off-diagonal block of the same
// T buffer (16x16 substitution + one MFMA merge), then T_bb written as fp16
// hi/lo.  One wave, no workgroup synchronisation: the wave's
// LDS accesses complete in program order.  gam and beta: the chunk's vectors.
GDN_DEVICE void solve_diag_block(TBuf& tb, const float* gam, const float* beta, const float* eg, const float* ieg,
                                 bool fact, const f32x16& G, int blk, int lane) {
  const int n = lane & 31, gq = lane >> 5, o = 32 * blk;
  const Scratch A = scratch_of(tb, blk);
  // (kk^T is symmetric to the bit, so the lane's column is taken as row n and
  // its registers as four consecutive columns at a time: two 8-byte writes)
  const float bn = beta[o + n];
  float d[16];
  row_decays(d, gam, eg, ieg, fact, o + n, o, lane);
#pragma unroll
  for (int i4 = 0; i4 < 4; ++i4) {
    const int j = 8 * i4 + 4 * gq;
    float x[4];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) x[rr] = n > j + rr ? bn * G[4 * i4 + rr] * d[4 * i4 + rr] : 0.f;
    float* p = &A.at(n, j);
    *reinterpret_cast<f32x2*>(p) = (f32x2){x[0], x[1]};
    *reinterpret_cast<f32x2*>(p + 2) = (f32x2){x[2], x[3]};
  }
  invert_diag16(A, lane);
  merge16(A, lane);
  // T_bb (unit diagonal) as fp16 hi/lo: lane -> row lane / 2, 16 columns
  const int i = lane >> 1, half = lane & 1, j0 = 16 * half;
  float tv[16];
#pragma unroll
  for (int m = 0; m < 16; m += 4) {
    const f32x4 x = load4(A.row(i, half) + m);
#pragma unroll
    for (int z = 0; z < 4; ++z) tv[m + z] = x[z];
  }
  f16_t th[16], tl[16];
  split_vec<16>(tv, th, tl);
#pragma unroll
  for (int m = 0; m < 16; m += 4) {
    const int off = (o + i) * LDH + o + j0 + m;
    *reinterpret_cast<f16x4*>(tb.hi + off) = (f16x4){th[m], th[m + 1], th[m + 2], th[m + 3]};
    *reinterpret_cast<f16x4*>(tb.lo + off) = (f16x4){tl[m], tl[m + 1], tl[m + 2], tl[m + 3]};
  }
}

// A_10 = beta_i k_i.k_j e^(g_i - g_j) for tokens i in 32..63, j in 0..31
// (always i > j), as fp16 hi/lo in block (0,1) of the T arrays: A_10[i][j] at
// row i, column 32 + j.  |A_10| <= beta_i |k_i| |k_j| (<= 1 for unit keys and
// beta <= 1), split unscaled.
template <typename Tiles>
GDN_DEVICE void b10_block(const Tiles& ct, TBuf& tb, int lane) {
  const int n = lane & 31, gq = lane >> 5;
  // (the transposed tile: lane column = token 32 + n, registers = four
  // consecutive tokens j at a time)
  const f32x16 G = gram_tile(ct.k, ct.k, 0, 1, lane);
  const bool fact = __builtin_amdgcn_readfirstlane(ct.fact) != 0;
  const float bn = ct.beta[32 + n];
  float d[16];
  row_decays(d, ct.gam, ct.eg, ct.ieg, fact, 32 + n, 0, lane);
#pragma unroll
  for (int i4 = 0; i4 < 4; ++i4) {
    float x[4];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) x[rr] = G[4 * i4 + rr] * (d[4 * i4 + rr] * bn);
    f16_t hi[4], lo[4];
    split_vec<4>(x, hi, lo);
    const int off = n * LDH + 32 + 8 * i4 + 4 * gq;
    *reinterpret_cast<f16x4*>(tb.hi + off) = (f16x4){hi[0], hi[1], hi[2], hi[3]};
    *reinterpret_cast<f16x4*>(tb.lo + off) = (f16x4){lo[0], lo[1], lo[2], lo[3]};
  }
}

// T_10 = -T_11 A_10 T_00 from the fp16 hi/lo blocks (lo x lo dropped).  One wave.
GDN_DEVICE void merge_offdiag(TBuf& tb, int lane) {
  const int n = lane & 31, gq = lane >> 5;
  const f16_t* th = tb.hi;
  const f16_t* tl = tb.lo;
  // M = A_10 T_00: A operand = rows of A_10, B operand = columns of T_00
  f32x16 M = zero16();
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const f16x8 bh = frag_rows(th, LDH, 0, 32 + 16 * ks, lane), bl = frag_rows(tl, LDH, 0, 32 + 16 * ks, lane);
    const f16x8 ch = frag_cols(th, LDH, 0, 16 * ks, lane), cl = frag_cols(tl, LDH, 0, 16 * ks, lane);
    M = mfma32(bh, ch, M);
    M = mfma32(bh, cl, M);
    M = mfma32(bl, ch, M);
  }
  // (T_11 M)^T = M^T T_11^T: A operand = M^T (M's C layout as it lies), B
  // operand = rows of T_11; lane column = row of T_10, registers = four
  // consecutive columns at a time
  f32x16 R = zero16();
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const f16x8 ah = frag_rows(th, LDH, 32, 32 + 16 * ks, lane), al = frag_rows(tl, LDH, 32, 32 + 16 * ks, lane);
    f16x8 mh, ml;
    split8(M, ks, 1.f, mh, ml);
    R = mfma32(mh, ah, R);
    R = mfma32(ml, ah, R);
    R = mfma32(mh, al, R);
  }
#pragma unroll
  for (int i4 = 0; i4 < 4; ++i4) {
    float x[4];
    f16_t hi[4], lo[4];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) x[rr] = -R[4 * i4 + rr];
    split_vec<4>(x, hi, lo);
    const int off = (32 + n) * LDH + 8 * i4 + 4 * gq;
    *reinterpret_cast<f16x4*>(tb.hi + off) = (f16x4){hi[0], hi[1], hi[2], hi[3]};
    *reinterpret_cast<f16x4*>(tb.lo + off) = (f16x4){lo[0], lo[1], lo[2], lo[3]};
  }
}

// (Q K^T) tile (mt, nt) -> P = lower(q_i.k_j e^(g_i - g_j)) as fp16, C layout
// (element 4 i4 + rr of the tile at row 32mt + 8 i4 + 4g + rr).
GDN_DEVICE f16x8 qk_half(const f32x16& G, const ChunkTiles& ct, bool fact, int mt, int nt, int h, int lane) {
  const int n = lane & 31, gq = lane >> 5;
  const int j = 32 * nt + n;
  f16x8 out;
  if (fact) {
    const float ej = ct.ieg[j];
#pragma unroll
    for (int i4 = 2 * h; i4 < 2 * h + 2; ++i4) {
      const f32x4 ei = rows4(ct.eg, 32 * mt, i4, lane);
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int i = 32 * mt + 8 * i4 + 4 * gq + rr;
        out[4 * (i4 - 2 * h) + rr] = (f16_t)(i >= j ? G[4 * i4 + rr] * (ei[rr] * ej) : 0.f);
      }
    }
  } else {
    const float gj = ct.gam[j];
#pragma unroll
    for (int i4 = 2 * h; i4 < 2 * h + 2; ++i4) {
      const f32x4 gi = rows4(ct.gam, 32 * mt, i4, lane);
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int i = 32 * mt + 8 * i4 + 4 * gq + rr;
        out[4 * (i4 - 2 * h) + rr] = (f16_t)(i >= j ? G[4 * i4 + rr] * __expf(gi[rr] - gj) : 0.f);
      }
    }
  }
  return out;
}
GDN_DEVICE void p_tile(ChunkTiles& ct, int mt, int nt, int lane) {
  const f32x16 G = gram_tile(ct.q, ct.k, mt, nt, lane);
  const bool fact = __builtin_amdgcn_readfirstlane(ct.fact) != 0;
  const f16x8 h0 = qk_half(G, ct, fact, mt, nt, 0, lane), h1 = qk_half(G, ct, fact, mt, nt, 1, lane);
  const int n = lane & 31, gq = lane >> 5;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const int i = 32 * mt + 8 * (e >> 2) + 4 * gq + (e & 3);
    ct.p[i * LDH + 32 * nt + n] = e < 8 ? h0[e] : h1[e - 8];
  }
}

// Stage a tile held in registers into LDS (fp16 for K/Q, the raw 16-bit
// elements for V).
template <bool F16>
GDN_DEVICE void stage_f16(f16_t* dst, const TileLoad& tl, int lane, bool keep = true) {
  // lane's 8 logical columns 8a..8a+7 (a = lane % 16) are quads 2a', 2a'+1 of
  // 16-column group a / 2 (a' = a % 2), stored at quads kq_quad(2a'), kq_quad(2a'+1)
  const int a = lane & 15, grp = 16 * (a >> 1), q0 = 2 * (a & 1);
  const int off0 = grp + 4 * kq_quad(q0), off1 = grp + 4 * kq_quad(q0 + 1);
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const f16x8 v = keep ? to_f16x8<F16>(tl.r[u]) : f16x8{};  // (keep: the lane's columns lie inside the head dim)
    f16_t* row = dst + ((lane >> 4) + 4 * u) * LDK;
    *reinterpret_cast<f16x4*>(row + off0) = (f16x4){v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f16x4*>(row + off1) = (f16x4){v[4], v[5], v[6], v[7]};
  }
}
GDN_DEVICE void stage_v(bf16_t* dst, const TileLoad& tl, int lane, bool keep = true) {
#pragma unroll
  for (int u = 0; u < 16; ++u)
    *reinterpret_cast<bf16x8*>(dst + ((lane >> 4) + 4 * u) * LDV + 8 * (lane & 15)) = keep ? tl.r[u] : bf16x8{};
}

// Decay vectors of a chunk for the state waves and the producers' epilogues.
template <typename Tiles>
GDN_DEVICE void stage_decay(Tiles& ct, const DecayLoad& dl, int L, int b_dtype, int lane) {
  float gl;
  const float gm = chunk_gamma(dl, L, lane, gl);
  ct.gam[lane] = gm;
  ct.eg[lane] = __expf(gm);
  ct.ieg[lane] = __expf(-gm);
  const bool fact = factorable(gm);
  if (lane == 0) ct.fact = fact;
  ct.edec[lane] = lane < L ? __expf(gl - gm) : 0.f;
  ct.beta[lane] = lane < L ? scalar_raw_f32(dl.b, b_dtype) : 0.f;
  if (lane == 0) ct.gam_last = gl;
}

// Kernel arguments of a call (tensors checked by the caller).
inline PrefillArgs prefill_args(const gdn_tensor* q, const gdn_tensor* k, const gdn_tensor* v, const gdn_tensor* g,
                                const gdn_tensor* beta, gdn_tensor* state, const gdn_tensor* idx,
                                const gdn_tensor* cu, gdn_tensor* out, float scale) {
  PrefillArgs a{};
  a.q = reinterpret_cast<const bf16_t*>(q->data);
  a.k = reinterpret_cast<const bf16_t*>(k->data);
  a.v = reinterpret_cast<const bf16_t*>(v->data);
  a.g = reinterpret_cast<const float*>(g->data);
  a.beta = beta->data;
  a.state = reinterpret_cast<float*>(state->data);
  a.idx = idx->data;
  a.cu = cu->data;
  a.out = reinterpret_cast<bf16_t*>(out->data);
  a.q_s0 = q->stride[0]; a.q_s1 = q->stride[1];
  a.k_s0 = k->stride[0]; a.k_s1 = k->stride[1];
  a.v_s0 = v->stride[0]; a.v_s1 = v->stride[1];
  a.g_s0 = g->stride[0]; a.g_s1 = g->stride[1];
  a.b_s0 = beta->stride[0]; a.b_s1 = beta->stride[1];
  a.o_s0 = out->stride[0]; a.o_s1 = out->stride[1];
  a.st_slot = state->stride[0]; a.st_head = state->stride[1];
  a.T = q->shape[0];
  a.nseq = cu->shape[0] - 1;
  a.num_slots = state->shape[0];
  a.Hv = (int32_t)v->shape[1];
  a.r = (int32_t)(v->shape[1] / q->shape[1]);
  a.b_dtype = beta->dtype;
  a.scale = scale;
  a.idx64 = idx->dtype == GDN_DTYPE_I64;
  a.cu64 = cu->dtype == GDN_DTYPE_I64;
  a.kd = (int32_t)q->shape[2];
  a.vd = (int32_t)v->shape[2];
  return a;
}

}  // namespace
#endif  // GDN_CHUNK_H_
