// Chunked gated-delta-rule prefill in two launches, for batches with few
// (sequence, v-head) items.
//
// The fused kernel (gdn_prefill.hip) walks an item's chunks in one workgroup,
// about 4.8 us per chunk, whatever the chip is doing otherwise: one prompt of
// 2,943 tokens keeps 32 of 256 CUs busy for 222 us.  Here everything that does
// not depend on the state is computed by one workgroup per (chunk, v-head)
// first, into a workspace, and the walk over the chunks that is left runs one
// workgroup per (item, 16 or 32 value columns): no product mixes value columns,
// so an item's column groups are independent.  That prompt takes 95 us: 37 to
// prepare 1,472 (chunk, v-head) pairs, 56 to scan 46 chunks.
//
// gdn_prepare_kernel, per chunk (notation of gdn_prefill.hip):
//   T = (I + A)^-1,  P                     as in the fused kernel
//   W = T diag(beta e^gamma) K,  U = T diag(beta) V
// gdn_scan_kernel, per chunk:
//   V' = U - W S
//   O  = scale [diag(e^gamma) Q S + P V']
//   S  = e^gamma_L S + K^T diag(e^(gamma_L - gamma)) V'
// so the chain from one state to the next is two products deep.
//
// What bounds the scan is that chain's latency, so everything on it is short:
// the state sits in the registers of four waves (wave w: keys
// 32w..32w+31 of the columns), each wave computes 16 rows of V' and its own
// keys of the update, the operands that come from the workspace are stored as
// the MFMA fragments of the wave that reads them (16 bytes per lane,
// contiguous) and are loaded a chunk ahead, and only S and V' cross the
// workgroup, through LDS: two barriers per chunk.
//
// Precision: as in the fused kernel every fp32 operand that feeds the state is
// split into fp16 hi + lo (lo x lo dropped) after scaling by a power of two,
// and products that only feed o use the hi part.  T diag(beta) multiplies V in
// V's own type (bf16: three terms of T, 24 bits), T diag(beta e^gamma) is
// scaled per row, W per chunk, S per wave and column (each of the four
// k-steps has its own accumulator, combined in fp32), V' per column by a bound
// from max |U|, max |W| and max |S| that all waves work out alike.
//
// 16x16x32 MFMA operands: A lane holds row l % 16, B lane column l % 16, both
// the 8 contraction slots 8 (l / 16)..+7; C lane holds column l % 16, rows
// 4 (l / 16)..+3.  Slot 8q + 4a + r of a 32-wide k-step stands for index
// 16a + 4q + r, so that two C tiles of 16 rows are a B operand as they lie.
#include "gdn_chunk.h"

namespace {

constexpr int kCols = 16;                    // value columns of a column group
constexpr int kGroups = VD / kCols;          // column groups per item
constexpr int kTouch = 4;                    // chunks a record is read into L2 ahead of its use
constexpr int kOneGroupItems = 32;           // items up to which a workgroup takes one column group
constexpr int kMaxSplitSeqs = 64;            // one lane per sequence
constexpr int kPieceBytes = 64 * 16;         // one fragment of a wave

// Workspace record of a (chunk, v-head), in bytes
constexpr int64_t kRecWhi = 0;                                 // [wave][k-step][lane]
constexpr int64_t kRecWlo = kRecWhi + 16 * kPieceBytes;
constexpr int64_t kRecU = kRecWlo + 16 * kPieceBytes;          // [column group][wave][lane], fp32
constexpr int64_t kRecP = kRecU + 4 * kGroups * kPieceBytes;   // [wave][k-step][lane]
constexpr int64_t kRecVec = kRecP + 8 * kPieceBytes;           // e^gamma, e^(gamma_L - gamma), max |U| per column, misc
constexpr int64_t kRecBytes = kRecVec + 1280;
constexpr int kVecDec = C, kVecU = 2 * C, kVecMisc = 2 * C + VD;  // float offsets in the vectors
// Workspace record of a (chunk, k-head): K^T [16-key tile][k-step][lane], Q [wave][k-step][lane]
constexpr int64_t kKRecQ = 16 * kPieceBytes;
constexpr int64_t kKRecBytes = 32 * kPieceBytes;

struct SplitArgs {
  PrefillArgs p;
  char* ws;       // records of (slot, v-head), then of (slot, k-head); slot = the chunk's index in the batch
  int64_t slots;  // chunk slots of the workspace
  int32_t Hk;
};

// Chunks of the batch, one sequence per lane: start of each sequence's slots
// and its number of chunks (padding sequences have theirs too: their lengths
// alone place the others).
struct ChunkMap {
  int32_t base, nc;
};
GDN_DEVICE ChunkMap chunk_map(const PrefillArgs& a, int lane) {
  ChunkMap m;
  m.nc = 0;
  if (lane < a.nseq) {
    int64_t s, e;
    seq_range(a.cu, a.cu64, lane, a.T, s, e);
    m.nc = (int32_t)((e - s + C - 1) / C);
  }
  m.base = wave_inclusive_scan_i32(m.nc) - m.nc;
  return m;
}

// Workgroup barrier over LDS only: global loads and stores stay in flight.
GDN_DEVICE void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

constexpr int kLdt = 72;  // row stride of the terms of T diag(..)

// The tile members of ChunkTiles that the prepare kernel has (its helpers take
// K and the decay vectors only).
struct PrepSmem {
  alignas(16) f16_t k[C * LDK];  // K, later V
  union {
    TBuf tb;
    alignas(16) f16_t terms[3 * C * kLdt];  // later the terms of T diag(..), quads swapped like K's
  };
  alignas(16) float gam[C];
  alignas(16) float eg[C];
  alignas(16) float ieg[C];
  alignas(16) float edec[C];
  alignas(16) float beta[C];
  float gam_last;
  int32_t fact;
  alignas(16) float dvec[2][4][C];  // waves 0, 1: gamma, beta, e^gamma, e^-gamma
  alignas(16) float rowf[2][C];     // row scales undone on W's and U's accumulators
  float wmax[4];
};
static_assert(3 * sizeof(PrepSmem) <= 160 * 1024, "three workgroups per CU");

// 2^e for a float's exponent, within the range that keeps every factor finite
GDN_DEVICE int bound_exp(float mx) {
  const int e = __builtin_amdgcn_frexp_expf(mx);
  return e < -100 ? -100 : e;
}

// maximum of |x| over a row's four lanes
GDN_DEVICE float quad_max(float x) {
  x = fmaxf(x, dpp_f32<0xB1>(x));
  return fmaxf(x, dpp_f32<0x4E>(x));
}

// One row's 16 entries x * 2^e as fp16 hi + lo at row i, columns j0.. of two arrays
GDN_DEVICE void put_split16(f16_t* dst, int i, int j0, const float (&x)[16], float sc) {
  float y[16];
  f16_t hi[16], lo[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) y[m] = x[m] * sc;
  split_vec<16>(y, hi, lo);
#pragma unroll
  for (int m = 0; m < 2; ++m) {  // stored quads 0, 2 and 1, 3 of the 16 columns
    const int a = 4 * m, b = a + 8;
    f16_t* p = dst + i * kLdt + j0 + 8 * m;
    *reinterpret_cast<f16x8*>(p) =
        (f16x8){hi[a], hi[a + 1], hi[a + 2], hi[a + 3], hi[b], hi[b + 1], hi[b + 2], hi[b + 3]};
    *reinterpret_cast<f16x8*>(p + C * kLdt) =
        (f16x8){lo[a], lo[a + 1], lo[a + 2], lo[a + 3], lo[b], lo[b + 1], lo[b + 2], lo[b + 3]};
  }
}
GDN_DEVICE f16x8 term_rows(const f16_t* M, int r0, int kbase, int lane) {
  return *reinterpret_cast<const f16x8*>(M + (r0 + (lane & 31)) * kLdt + kbase + 8 * (lane >> 5));
}

// The same as three bf16 terms (24 bits, fp32's range) in three arrays
GDN_DEVICE void put_bf16x3(f16_t* dst, int i, int j0, const float (&x)[16]) {
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    bf16x8 t[3];
#pragma unroll
    for (int z = 0; z < 8; ++z) {
      float r = x[4 * m + (z & 3) + 8 * (z >> 2)];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        t[k][z] = (bf16_t)r;
        r -= (float)t[k][z];
      }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) *reinterpret_cast<bf16x8*>(dst + k * C * kLdt + i * kLdt + j0 + 8 * m) = t[k];
  }
}

// 32 rows of a 64 x 128 tile as eight fp16 fragments in the k order of
// frag_rows_kq: lane (n, g) loads columns 8g..8g+7 of every 16, and its halves
// trade places with lane n + 32's so that it holds 4g..4g+3 and 8+4g..8+4g+3.
template <bool F16>
GDN_DEVICE void rows_kq(const bf16x8 (&raw)[8], f16x8 (&out)[8]) {
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) {
    const u32x4 x = __builtin_bit_cast(u32x4, to_f16x8<F16>(raw[ks]));
    const auto a = __builtin_amdgcn_permlane32_swap(x[0], x[2], false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(x[1], x[3], false, false);
    out[ks] = __builtin_bit_cast(f16x8, (u32x4){a[0], b[0], a[1], b[1]});
  }
}

// One workgroup of 256 threads per (chunk slot, v-head).  Bound by the latency
// of the chain Gram -> diagonal blocks -> T -> W, U; three workgroups per CU
// (47 KB of LDS: Q stays in registers and P is formed transposed, so that its
// accumulators are the scan's fragments).
template <bool F16, bool OUT32>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void gdn_prepare_kernel(SplitArgs sa) {
  __shared__ PrepSmem sm;
  const PrefillArgs& a = sa.p;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t bid = blockIdx.x;
  if (!(a.flags & GDN_PREFILL_ACCUM_OUT))
    zero_uncovered_rows<OUT32 ? 4 : 2>(a.out, a.o_s0, a.o_s1, a.Hv, VD, a.cu, a.cu64, a.nseq, a.T, bid, gridDim.x, tid, 256);
  // the two v-heads of a k-head on one XCD, as in the fused kernel
  const int64_t work = 2 * ((bid >> 4) * 8 + (bid & 7)) + ((bid >> 3) & 1);
  const int64_t slot = work / a.Hv;
  const int h = (int)(work - slot * a.Hv);
  if (slot >= sa.slots) return;
  const ChunkMap cm = chunk_map(a, lane);
  const uint64_t own = __builtin_amdgcn_ballot_w64(slot >= cm.base && slot < (int64_t)cm.base + cm.nc);
  if (own == 0) return;
  const int seq = __builtin_ctzll(own);
  const int64_t st_slot = load_index(a.idx, seq, a.idx64);
  if (st_slot < 0 || st_slot >= a.num_slots) return;  // a padding sequence: nothing to prepare
  int64_t s0, s1;
  seq_range(a.cu, a.cu64, seq, a.T, s0, s1);
  const int64_t c0 = s0 + (int64_t)C * (slot - __builtin_amdgcn_readlane(cm.base, seq));
  const int kh = h / a.r;
  const ChunkSource src{&a, a.k + kh * a.k_s1, a.q + kh * a.q_s1, a.v + h * a.v_s1, h, s1};
  const int L = chunk_rows(src, c0);
  char* const rec = sa.ws + (slot * a.Hv + h) * kRecBytes;
  char* const krec = sa.ws + sa.slots * a.Hv * kRecBytes + (slot * sa.Hk + kh) * kKRecBytes;
  PrepSmem& ct = sm;
  const int n = lane & 31, g2 = lane >> 5, l16 = lane & 15, q4 = lane >> 4;

  f16x8 qf[2][8];  // wave 3: Q
  if (w < 2) {
    DiagLoad dl;
    load_diag(dl, src, c0, w, lane);
    float gl;
    const float gm = chunk_gamma(dl.d, L, lane, gl);
    sm.dvec[w][0][lane] = gm;
    sm.dvec[w][1][lane] = lane < L ? scalar_raw_f32(dl.d.b, a.b_dtype) : 0.f;
    sm.dvec[w][2][lane] = __expf(gm);
    sm.dvec[w][3][lane] = __expf(-gm);
    const bool fact = factorable(gm);
    const f32x16 G = gram_regs<F16>(dl.kf);
    solve_diag_block(sm.tb, sm.dvec[w][0], sm.dvec[w][1], sm.dvec[w][2], sm.dvec[w][3], fact, G, w, lane);
  } else if (w == 2) {
    TileLoad kl;
    DecayLoad dl;
    load_tile(kl, src.kg, a.k_s0, c0, L, lane);
    load_decay(dl, src, c0, L, lane);
    stage_f16<F16>(ct.k, kl, lane);
    stage_decay(ct, dl, L, a.b_dtype, lane);
  } else {
    const bf16_t* qb = src.qg + c0 * a.q_s0;
    bf16x8 raw[2][8];
#pragma unroll
    for (int it = 0; it < 2; ++it)
#pragma unroll
      for (int ks = 0; ks < 8; ++ks)
        raw[it][ks] = load_row_piece(qb, (uint32_t)a.q_s0, 32 * it + n, 16 * ks + 8 * g2, L);
#pragma unroll
    for (int it = 0; it < 2; ++it) rows_kq<F16>(raw[it], qf[it]);
  }
  __syncthreads();
  if (w == 2) {
    b10_block(ct, sm.tb, lane);
    merge_offdiag(sm.tb, lane);
  } else if (w == 3) {
    // P^T tiles (key tile jt, query tile it): lane column = query 32 it + n, so
    // four accumulators are four consecutive keys of the query's row of P
    const bool fact = __builtin_amdgcn_readfirstlane(ct.fact) != 0;
#pragma unroll
    for (int tl = 0; tl < 3; ++tl) {
      const int jt = tl == 2, it = tl >= 1;
      f32x16 G = zero16();
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) G = mfma32(frag_rows_kq(ct.k, 32 * jt, 16 * ks, lane), qf[it][ks], G);
      const int i = 32 * it + n;
      f16x4 p[4];
      if (fact) {
        const float ei = ct.eg[i];
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          const f32x4 ej = rows4(ct.ieg, 32 * jt, i4, lane);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            p[i4][r] = (f16_t)(32 * jt + 8 * i4 + 4 * g2 + r <= i ? G[4 * i4 + r] * (ei * ej[r]) : 0.f);
        }
      } else {
        const float gi = ct.gam[i];
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          const f32x4 gj = rows4(ct.gam, 32 * jt, i4, lane);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            p[i4][r] = (f16_t)(32 * jt + 8 * i4 + 4 * g2 + r <= i ? G[4 * i4 + r] * __expf(gi - gj[r]) : 0.f);
        }
      }
#pragma unroll
      for (int f = 0; f < 2; ++f)
        *reinterpret_cast<f16x8*>(rec + kRecP + (2 * (2 * it + (n >> 4)) + jt) * kPieceBytes +
                                  16 * (16 * (2 * f + g2) + (n & 15))) = cat4(p[f], p[2 + f]);
    }
    if (h - kh * a.r == 0) {  // the k-head's Q fragments
#pragma unroll
      for (int it = 0; it < 2; ++it)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          const f16x8 x = qf[it][2 * ks], y = qf[it][2 * ks + 1];
          char* p = krec + kKRecQ + ((2 * it + (n >> 4)) * 4 + ks) * kPieceBytes + 16 * (n & 15);
          *reinterpret_cast<f16x8*>(p + 256 * g2) = (f16x8){x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
          *reinterpret_cast<f16x8*>(p + 256 * (2 + g2)) = (f16x8){x[4], x[5], x[6], x[7], y[4], y[5], y[6], y[7]};
        }
    }
  } else if (h - kh * a.r == 0) {  // the k-head's K^T fragments
#pragma unroll
    for (int f = 8 * w; f < 8 * w + 8; ++f) {
      const f16_t* p = ct.k + (32 * (f & 1) + 4 * q4 + (l16 >> 2)) * LDK + 16 * (f >> 1) + 4 * kq_quad(l16 & 3);
      *reinterpret_cast<f16x8*>(krec + f * kPieceBytes + 16 * lane) =
          cat4(__builtin_bit_cast(f16x4, tr_read(p)), __builtin_bit_cast(f16x4, tr_read(p + 16 * LDK)));
    }
  }
  __syncthreads();
  // V rows 16w + lane / 16 + 4u, in flight until the K tile is done with
  bf16x8 vr[4];
  {
    const bf16_t* vb = src.vg + c0 * a.v_s0;
#pragma unroll
    for (int u = 0; u < 4; ++u) vr[u] = load_row_piece(vb, (uint32_t)a.v_s0, 16 * w + q4 + 4 * u, 8 * l16, L);
  }
  // this lane's 16 entries of T (row ti, columns tj..)
  const int ti = 16 * w + (lane >> 2), tj = 16 * (lane & 3);
  float tbeta[16], tw[16];
#pragma unroll
  for (int m = 0; m < 16; m += 4) {
    const f16x4 hv = *reinterpret_cast<const f16x4*>(sm.tb.hi + ti * LDH + tj + m);
    const f16x4 lv = *reinterpret_cast<const f16x4*>(sm.tb.lo + ti * LDH + tj + m);
    const f32x4 bv = *reinterpret_cast<const f32x4*>(ct.beta + tj + m);
    const f32x4 ev = *reinterpret_cast<const f32x4*>(ct.eg + tj + m);
#pragma unroll
    for (int z = 0; z < 4; ++z) {
      const bool in = tj + m + z <= ti;  // (block (0,1) holds A_10)
      tbeta[m + z] = in ? ((float)hv[z] + (float)lv[z]) * bv[z] : 0.f;
      tw[m + z] = tbeta[m + z] * ev[z];
    }
  }
  f16_t* const terms = sm.terms;
  auto row_exp = [&](const float (&x)[16]) __attribute__((always_inline)) {
    float m = 0.f;
#pragma unroll
    for (int j = 0; j < 16; ++j) m = fmaxf(m, fabsf(x[j]));
    return bound_exp(quad_max(m)) - 10;
  };
  const int we = row_exp(tw);
  const int ue = F16 ? row_exp(tbeta) : 0;
  if ((lane & 3) == 0) {
    sm.rowf[0][ti] = __builtin_amdgcn_ldexpf(1.f, we);
    sm.rowf[1][ti] = __builtin_amdgcn_ldexpf(1.f, ue);
  }
  __syncthreads();
  put_split16(terms, ti, tj, tw, __builtin_amdgcn_ldexpf(1.f, -we));
  __syncthreads();
  // W^T = K^T (T diag(beta e^gamma))^T on this wave's 32 keys: lane column = token 32 nt + n
  f32x16 acc[2] = {zero16(), zero16()};
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const f16x8 kf = frag_cols_kq(ct.k, 32 * w, 16 * ks, lane);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int nt = ks >> 1; nt < 2; ++nt)
        acc[nt] = mfma32(kf, term_rows(terms + t * C * kLdt, 32 * nt, 16 * ks, lane), acc[nt]);
    }
  }
  float mx = 0.f;
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const float f = sm.rowf[0][32 * nt + n];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      acc[nt][j] *= f;
      mx = fmaxf(mx, fabsf(acc[nt][j]));
    }
  }
  mx = wave_max(mx);
  if (lane == 0) sm.wmax[w] = mx;
  __syncthreads();  // (and every wave has read the K tile and the terms)
  mx = fmaxf(fmaxf(sm.wmax[0], sm.wmax[1]), fmaxf(sm.wmax[2], sm.wmax[3]));
  const int wexp = bound_exp(mx);
  {
    const float sc = __builtin_amdgcn_ldexpf(1.f, 14 - wexp);
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      f32x16 x;  // registers in fragment order: quad-rows 0, 2, 1, 3
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x[r] = acc[nt][r];
        x[4 + r] = acc[nt][8 + r];
        x[8 + r] = acc[nt][4 + r];
        x[12 + r] = acc[nt][12 + r];
      }
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        f16x8 hi, lo;
        split8(x, f, sc, hi, lo);
        char* p = rec + ((2 * nt + (n >> 4)) * 4 + w) * kPieceBytes + 16 * (16 * (2 * f + g2) + (n & 15));
        *reinterpret_cast<f16x8*>(p + kRecWhi) = hi;
        *reinterpret_cast<f16x8*>(p + kRecWlo) = lo;
      }
    }
  }
  // V into the K tile, T diag(beta) into the terms
  bf16_t* const vt = reinterpret_cast<bf16_t*>(ct.k);
#pragma unroll
  for (int u = 0; u < 4; ++u)
    *reinterpret_cast<bf16x8*>(vt + (16 * w + q4 + 4 * u) * LDK + 8 * l16) = vr[u];
  if constexpr (F16) put_split16(terms, ti, tj, tbeta, __builtin_amdgcn_ldexpf(1.f, -ue));
  else put_bf16x3(terms, ti, tj, tbeta);
  __syncthreads();
  // U on this wave's 32 value columns
  f32x16 U[2] = {zero16(), zero16()};
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const f16x8 vf = frag_cols(reinterpret_cast<const f16_t*>(vt), LDK, 32 * w, 16 * ks, lane);
#pragma unroll
    for (int t = 0; t < (F16 ? 2 : 3); ++t) {
#pragma unroll
      for (int mt = ks >> 1; mt < 2; ++mt) {
        const f16x8 tf = term_rows(terms + t * C * kLdt, 32 * mt, 16 * ks, lane);
        if constexpr (F16) U[mt] = mfma32(tf, vf, U[mt]);
        else
          U[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, tf), __builtin_bit_cast(bf16x8, vf),
                                                          U[mt], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      f32x4 x;
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = U[mt][4 * i4 + r];
      if constexpr (F16) {
        const f32x4 f = rows4(sm.rowf[1], 32 * mt, i4, lane);
#pragma unroll
        for (int r = 0; r < 4; ++r) U[mt][4 * i4 + r] = x[r] = x[r] * f[r];
      }
      const int cg = 2 * w + (n >> 4), ww = 2 * mt + (i4 >> 1), qq = 2 * (i4 & 1) + g2;
      *reinterpret_cast<f32x4*>(rec + kRecU + (cg * 4 + ww) * kPieceBytes + 16 * (16 * qq + (n & 15))) = x;
    }
  float* const vec = reinterpret_cast<float*>(rec + kRecVec);
  const float um = col_max(U, 2);
  if (lane < 32) vec[kVecU + 32 * w + n] = um;
  if (w == 0) vec[lane] = ct.eg[lane];
  if (w == 1) vec[kVecDec + lane] = ct.edec[lane];
  if (tid == 128) {
    vec[kVecMisc] = __builtin_amdgcn_ldexpf(1.f, wexp - 14);
    vec[kVecMisc + 1] = mx * (float)(KD << 13);  // 2^13 times a bound of sum_j |W_ij|
    vec[kVecMisc + 2] = __expf(ct.gam_last);
    vec[kVecMisc + 3] = 0.f;
  }
}

// What a lane of chain wave w and of output wave w read of one chunk.
template <int NT>
struct ChainLoad {
  f16x8 whi[4], wlo[4], kt[2][2];
  f32x4 u[NT], edec, misc;
  float un[NT];
};
struct OutLoad {
  f16x8 q[4], p[2];
  f32x4 eg;
};

struct ScanSmem {
  f16x8 shi[4][64], slo[4][64];  // S of wave w as B fragments, in units of sfac
  alignas(16) float sfac[kCols][4];
  float vu[kCols];               // units of V'
  f16x4 vhi[2][64][2];           // V', and e^(gamma_L - gamma) V' as hi and lo: fragments of two waves' rows
  f16x4 dhi[2][64][2], dlo[2][64][2];
};

// Biased exponent E of a non-negative float's bits, at least 2^-100's, with
// x < 2^(E - 126); and 2^k as a float from k + 127.
GDN_DEVICE int biased_exp(uint32_t bits) { return max((int)(bits >> 23), 27); }
GDN_DEVICE float pow2_biased(int k) { return __builtin_bit_cast(float, (uint32_t)k << 23); }

// One workgroup per (item, NT groups of 16 value columns); see the file's head.  Waves 0..3
// run the chain from state to state, waves 4..7 follow it a barrier behind with
// the output rows (they share the SIMDs, so the chain does not wait for their
// products, loads and stores).  One prompt of 2,943 tokens, 32 heads: 1.28 us per
// chunk against 1.67 with four waves doing both and all loads at the end.
// An item's column groups run on one XCD (workgroups are dealt
// round-robin), which reads its chunks' records from HBM once.
template <bool F16, int NT, bool OUT32>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void gdn_scan_kernel(SplitArgs sa) {
  __shared__ ScanSmem smt[NT];
  constexpr int kWgs = kGroups / NT;  // workgroups per item
  const PrefillArgs& a = sa.p;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), w = wave & 3;
  const int64_t bid = blockIdx.x >> 3;
  const int cg = NT * (int)(bid % kWgs);  // first column group
  const int64_t work = 2 * (bid / (2 * kWgs) * 8 + (blockIdx.x & 7)) + (bid / kWgs & 1);
  if (work >= a.nseq * a.Hv) return;
  const int rank = (int)(work / a.Hv), h = (int)(work - (int64_t)rank * a.Hv);
  const ChunkMap cm = chunk_map(a, lane);
  // sequences longest first
  int rk = 0;
  for (int j = 0; j < (int)a.nseq; ++j) {
    const int nj = __builtin_amdgcn_readlane(cm.nc, j);
    rk += nj > cm.nc || (nj == cm.nc && j < lane);
  }
  const uint64_t own = __builtin_amdgcn_ballot_w64(lane < a.nseq && rk == rank);
  const int seq = __builtin_ctzll(own);
  const int64_t slot0 = __builtin_amdgcn_readlane(cm.base, seq);
  int nc = __builtin_amdgcn_readlane(cm.nc, seq);
  if (slot0 + nc > sa.slots) nc = (int)(sa.slots > slot0 ? sa.slots - slot0 : 0);  // (only for offsets that decrease)
  int64_t s0, s1;
  seq_range(a.cu, a.cu64, seq, a.T, s0, s1);
  const int64_t st_slot = load_index(a.idx, seq, a.idx64);
  const int c = lane & 15, q = lane >> 4;
  // (byte addresses: the output holds 16-bit elements, or fp32 ones with OUT32)
  constexpr uint32_t kOut = OUT32 ? 4 : 2;
  char* const ob = reinterpret_cast<char*>(a.out) + (h * a.o_s1 + kCols * cg) * kOut;
  if (st_slot < 0 || st_slot >= a.num_slots) {  // a padding sequence: zero rows, no state
    if (a.flags & GDN_PREFILL_ACCUM_OUT) return;  // (nothing to add)
    for (int64_t t = s0 + (tid >> 4); t < s1; t += 32)
      for (int nt = 0; nt < NT; ++nt) {
        char* p = ob + (t * a.o_s0 + kCols * nt + c) * kOut;
        if constexpr (OUT32) *reinterpret_cast<float*>(p) = 0.f;
        else *reinterpret_cast<uint16_t*>(p) = 0;
      }
    return;
  }
  if (nc == 0) return;
  // records through one descriptor of the workspace (at most 1 GiB): uniform
  // 32-bit record offsets, 16 bytes per lane
  const int kh = h / a.r;
  const uint32_t rec_step = (uint32_t)(a.Hv * kRecBytes), krec_step = (uint32_t)(sa.Hk * kKRecBytes);
  const uint32_t krecs = (uint32_t)(sa.slots * a.Hv * kRecBytes);
  const __amdgpu_buffer_rsrc_t rws = __builtin_amdgcn_make_buffer_rsrc(
      sa.ws, 0, krecs + (uint32_t)(sa.slots * sa.Hk * kKRecBytes), 0x00020000);
  const uint32_t rec0 = (uint32_t)slot0 * rec_step + (uint32_t)(h * kRecBytes);
  const uint32_t krec0 = krecs + (uint32_t)slot0 * krec_step + (uint32_t)(kh * kKRecBytes);
  const uint32_t l16b = 16u * lane;
  auto piece = [&](uint32_t lane_off, uint32_t off) __attribute__((always_inline)) {
    return __builtin_amdgcn_raw_buffer_load_b128(rws, lane_off, off, 0);
  };
  auto frag = [&](uint32_t lane_off, uint32_t off) __attribute__((always_inline)) {
    return __builtin_bit_cast(f16x8, piece(lane_off, off));
  };
  const f32x4 z = {0.f, 0.f, 0.f, 0.f};
  // (each role keeps two chunks' operands in registers, a chunk's loaded while
  // the one before it is worked on; past the end the last is read again)
  auto next = [&](int ch) __attribute__((always_inline)) { return ch + 1 < nc ? ch + 1 : nc - 1; };

  if (wave >= 4) {
    auto load = [&](OutLoad& d, int ch) __attribute__((always_inline)) {
      const uint32_t rec = rec0 + (uint32_t)ch * rec_step;
      const uint32_t krec = krec0 + (uint32_t)ch * krec_step + (uint32_t)(kKRecQ + 4 * w * kPieceBytes);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) d.q[ks] = frag(l16b + ks * kPieceBytes, krec);
      d.eg = __builtin_bit_cast(f32x4, piece(16u * q, rec + (uint32_t)(kRecVec + 64 * w)));
      // (waves 0 and 1 have no second k-step: they read their first again)
      const uint32_t pr = rec + (uint32_t)(kRecP + 2 * w * kPieceBytes);
      d.p[0] = frag(l16b, pr);
      d.p[1] = frag(l16b, pr + (w >= 2 ? kPieceBytes : 0));
    };
    // output rows 16w + 4q + r of a chunk, through a descriptor that ends with
    // this workgroup's columns of its last row (64 whole rows of the largest
    // token stride, 2^24, are 2^32 bytes of fp32)
    const uint32_t orow = (uint32_t)a.o_s0 * kOut;
    const uint32_t ooff = (uint32_t)(16 * w + 4 * q) * orow + kOut * c;
    // A touch reads one dword of each 128-byte line of a chunk's records into
    // L2, kTouch chunks before they are loaded for use, the lines dealt over
    // the item's output waves.  Without it every one of the item's workgroups
    // waited out HBM's latency for the same lines, more of them than
    // a CU keeps in flight.  Its registers are folded into an accumulator one
    // touch later, so that no wave waits for one.
    constexpr int kRecLines = (int)(kRecBytes / 128), kLines = kRecLines + (int)(kKRecBytes / 128);
    static_assert(kRecBytes % 128 == 0 && kLines <= 4 * kWgs * 64, "a touch covers the records");
    const int line = 4 * kWgs * lane + 4 * (cg / NT) + w;
    const uint32_t toff = line < kRecLines ? 128u * line : 128u * (line - kRecLines);
    uint32_t tv = 0, tacc = 0;
    auto touch = [&](int ch) __attribute__((always_inline)) {
      if (ch >= nc) return;
      tacc |= tv;
      const uint32_t base = line < kRecLines ? rec0 + (uint32_t)ch * rec_step : krec0 + (uint32_t)ch * krec_step;
      tv = __builtin_amdgcn_raw_buffer_load_b32(rws, line < kLines ? base + toff : 0xfffffff0u, 0, 0);
    };
    OutLoad la, lb;
    load(la, 0);
    for (int ch = 1; ch < kTouch; ++ch) touch(ch);
    auto step = [&](const OutLoad& d, OutLoad& dn, int ch) __attribute__((always_inline)) {
      touch(ch + kTouch);
      lds_barrier();
      f32x4 QS[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const ScanSmem& sm = smt[nt];
        f32x4 qa[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
          qa[ks] = __builtin_amdgcn_mfma_f32_16x16x32_f16(d.q[ks], sm.shi[ks][lane], z, 0, 0, 0);
        const f32x4 sf = *reinterpret_cast<const f32x4*>(sm.sfac[c]);
        QS[nt] = z;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
          for (int r = 0; r < 4; ++r) QS[nt][r] = fmaf(qa[ks][r], sf[ks], QS[nt][r]);
      }
      lds_barrier();
      const int64_t t0 = s0 + (int64_t)C * ch;
      const uint32_t rows = (uint32_t)(s1 - t0 < C ? s1 - t0 : C);
      const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
          ob + t0 * (int64_t)orow, 0, (rows - 1) * orow + kOut * kCols * NT, 0x00020000);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const ScanSmem& sm = smt[nt];
        const float vu = sm.vu[c];
        f32x4 O = __builtin_amdgcn_mfma_f32_16x16x32_f16(d.p[0], *reinterpret_cast<const f16x8*>(sm.vhi[0][lane]), z, 0, 0, 0);
        if (w >= 2)
          O = __builtin_amdgcn_mfma_f32_16x16x32_f16(d.p[1], *reinterpret_cast<const f16x8*>(sm.vhi[1][lane]), O, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float o = a.scale * fmaf(d.eg[r], QS[nt][r], O[r] * vu);
          if constexpr (OUT32) {
            float y = o;
            if (a.flags & GDN_PREFILL_ACCUM_OUT)
              y += __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ro, ooff + r * orow, kOut * kCols * nt, 0));
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, y), ro, ooff + r * orow, kOut * kCols * nt, 0);
          } else {
            uint16_t ov;
            if constexpr (F16) ov = __builtin_bit_cast(uint16_t, (f16_t)o);
            else ov = __builtin_bit_cast(uint16_t, (bf16_t)o);
            __builtin_amdgcn_raw_buffer_store_b16(ov, ro, ooff + r * orow, kOut * kCols * nt, 0);
          }
        }
      }
      load(dn, next(ch));
    };
    int ch = 0;
    for (; ch + 1 < nc; ch += 2) {
      step(la, lb, ch);
      step(lb, la, ch + 1);
    }
    if (ch < nc) step(la, lb, ch);
    asm volatile("" ::"v"(tacc | tv));
    return;
  }

  auto load_whi = [&](ChainLoad<NT>& d, int ch) __attribute__((always_inline)) {
    const uint32_t rec = rec0 + (uint32_t)ch * rec_step + (uint32_t)(kRecWhi + 4 * w * kPieceBytes);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) d.whi[ks] = frag(l16b + ks * kPieceBytes, rec);
  };
  auto load_wlo = [&](ChainLoad<NT>& d, int ch) __attribute__((always_inline)) {
    const uint32_t rec = rec0 + (uint32_t)ch * rec_step + (uint32_t)(kRecWlo + 4 * w * kPieceBytes);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) d.wlo[ks] = frag(l16b + ks * kPieceBytes, rec);
  };
  auto load_kt = [&](ChainLoad<NT>& d, int ch) __attribute__((always_inline)) {
    const uint32_t krec = krec0 + (uint32_t)ch * krec_step + (uint32_t)(4 * w * kPieceBytes);
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int s = 0; s < 2; ++s) d.kt[mt][s] = frag(l16b + (2 * mt + s) * kPieceBytes, krec);
  };
  auto load_vec = [&](ChainLoad<NT>& d, int ch) __attribute__((always_inline)) {
    const uint32_t rec = rec0 + (uint32_t)ch * rec_step;
    const uint32_t vec = rec + kRecVec;
    d.misc = __builtin_bit_cast(f32x4, piece(0, vec + 4 * kVecMisc));
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      d.u[nt] = __builtin_bit_cast(f32x4, piece(l16b, rec + (uint32_t)(kRecU + (4 * (cg + nt) + w) * kPieceBytes)));
      d.un[nt] = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(rws, 4u * c, vec + 4 * (kVecU + kCols * (cg + nt)), 0));
    }
    d.edec = __builtin_bit_cast(f32x4, piece(16u * q, vec + 4 * kVecDec + 64 * w));
  };
  ChainLoad<NT> la, lb;
  load_whi(la, 0);
  load_wlo(la, 0);
  load_vec(la, 0);
  load_kt(la, 0);

  // state: keys 32w + 16mt + 4q + r, value column 16 (cg + nt) + c
  float* const sg = a.state + st_slot * a.st_slot + (int64_t)h * a.st_head + (32 * w + 4 * q) * VD + kCols * cg + c;
  f32x4 S[NT][2];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        S[nt][mt][r] = a.flags & GDN_PREFILL_ZERO_INIT ? 0.f : sg[(16 * mt + r) * VD + kCols * nt];
  // The next chunk's loads go out in four groups, each behind the LDS reads or
  // MFMAs that the wave is about to wait for (the scheduling barriers keep them
  // there): all at once they held up the chain for as long as they took to issue.
  auto step = [&](const ChainLoad<NT>& d, ChainLoad<NT>& dn, int ch) __attribute__((always_inline)) {
    const int cn = next(ch);
    // S of this wave: units from its column maximum over the wave's keys, hi + lo fragments
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      ScanSmem& sm = smt[nt];
      uint32_t m = 0;
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float x = S[nt][mt][r];  // (a bit cast of a vector's element would read its first)
          m = max(m, __builtin_bit_cast(uint32_t, x) & 0x7fffffffu);
        }
      const auto m1 = __builtin_amdgcn_permlane16_swap(m, m, false, false);
      m = max(m1[0], m1[1]);
      const auto m2 = __builtin_amdgcn_permlane32_swap(m, m, false, false);
      m = max(m2[0], m2[1]);
      const int e = biased_exp(m);
      const float sc = pow2_biased(266 - e);  // 2^13 / 2^(e - 126)
      uint32_t H[4], Lo[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float x0 = S[nt][k >> 1][2 * (k & 1)], x1 = S[nt][k >> 1][2 * (k & 1) + 1];
        H[k] = mix_hi_pair(x0, sc, x1, sc);
        Lo[k] = mix_lo_pair(x0, sc, x1, sc, H[k]);
      }
      sm.shi[w][lane] = __builtin_bit_cast(f16x8, (u32x4){H[0], H[1], H[2], H[3]});
      sm.slo[w][lane] = __builtin_bit_cast(f16x8, (u32x4){Lo[0], Lo[1], Lo[2], Lo[3]});
      sm.sfac[c][w] = pow2_biased(e - 12);  // 2^(e - 126 - 13)
    }
    lds_barrier();
    float vu[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      ScanSmem& sm = smt[nt];
      // W S, one accumulator per k-step (each has its own units)
      f16x8 shi[4], slo[4];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) shi[ks] = sm.shi[ks][lane];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) slo[ks] = sm.slo[ks][lane];
      const f32x4 sf = *reinterpret_cast<const f32x4*>(sm.sfac[c]);
      if (nt == 0) {
        __builtin_amdgcn_sched_barrier(0);
        load_whi(dn, cn);
        __builtin_amdgcn_sched_barrier(0);
      }
      f32x4 X = z;
      f32x4 xa[4];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) xa[ks] = __builtin_amdgcn_mfma_f32_16x16x32_f16(d.whi[ks], shi[ks], z, 0, 0, 0);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) xa[ks] = __builtin_amdgcn_mfma_f32_16x16x32_f16(d.wlo[ks], shi[ks], xa[ks], 0, 0, 0);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) xa[ks] = __builtin_amdgcn_mfma_f32_16x16x32_f16(d.whi[ks], slo[ks], xa[ks], 0, 0, 0);
      if (nt == NT - 1) {
        __builtin_amdgcn_sched_barrier(0);
        load_wlo(dn, cn);
        __builtin_amdgcn_sched_barrier(0);
      }
      // V' and its units: |V'| <= max |U| + sum_j |W_ij| max |S|, |S| < 2^13 sfac
      const float vb = fmaf(d.misc[1], fmaxf(fmaxf(sf[0], sf[1]), fmaxf(sf[2], sf[3])), d.un[nt]);
      const int ve = biased_exp(__builtin_bit_cast(uint32_t, vb));
      const float vs = pow2_biased(267 - ve);  // 2^14 / 2^(ve - 126), and its inverse:
      vu[nt] = pow2_biased(ve - 13);
      float v[4], f[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) f[r] = vs * d.edec[r];
      sm.vu[c] = vu[nt];  // (the four waves' are equal)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int r = 0; r < 4; ++r) X[r] = fmaf(xa[ks][r], sf[ks], X[r]);
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = fmaf(-d.misc[0], X[r], d.u[nt][r]);
      const uint32_t h0 = mix_hi_pair(v[0], f[0], v[1], f[1]), h1 = mix_hi_pair(v[2], f[2], v[3], f[3]);
      const uint32_t l0 = mix_lo_pair(v[0], f[0], v[1], f[1], h0), l1 = mix_lo_pair(v[2], f[2], v[3], f[3], h1);
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      sm.dhi[w >> 1][lane][w & 1] = __builtin_bit_cast(f16x4, (u32x2){h0, h1});
      sm.dlo[w >> 1][lane][w & 1] = __builtin_bit_cast(f16x4, (u32x2){l0, l1});
      sm.vhi[w >> 1][lane][w & 1] =
          (f16x4){(f16_t)(v[0] * vs), (f16_t)(v[1] * vs), (f16_t)(v[2] * vs), (f16_t)(v[3] * vs)};
    }
    lds_barrier();
    // S = e^gamma_L S + K^T (..): this wave's keys
    const float dec = d.misc[2];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const ScanSmem& sm = smt[nt];
      f32x4 up[2] = {z, z};
      f16x8 dh[2], dl[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) dh[s] = *reinterpret_cast<const f16x8*>(sm.dhi[s][lane]);
#pragma unroll
      for (int s = 0; s < 2; ++s) dl[s] = *reinterpret_cast<const f16x8*>(sm.dlo[s][lane]);
      if (nt == 0) {
        __builtin_amdgcn_sched_barrier(0);
        load_kt(dn, cn);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) up[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(d.kt[mt][s], dh[s], up[mt], 0, 0, 0);
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) up[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(d.kt[mt][s], dl[s], up[mt], 0, 0, 0);
      if (nt == NT - 1) {
        __builtin_amdgcn_sched_barrier(0);
        load_vec(dn, cn);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[nt][mt][r] = fmaf(S[nt][mt][r], dec, up[mt][r] * vu[nt]);
    }
  };
  int ch = 0;
  for (; ch + 1 < nc; ch += 2) {
    step(la, lb, ch);
    step(lb, la, ch + 1);
  }
  if (ch < nc) step(la, lb, ch);
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float* p = sg + (16 * mt + r) * VD + kCols * nt;
        *p = a.flags & GDN_PREFILL_ACCUM_STATE ? *p + S[nt][mt][r] : S[nt][mt][r];
      }
}

}  // namespace

// Floats of the workspace with which a prefill of these sizes runs split, 0
// when the fused kernel serves it.  Split wins where the fused kernel's items
// leave most CUs idle for a few chunks.  Measured, fused -> split, prompts x
// tokens at 16 / 32 heads: 1 x 128 21 -> 20 us, 1 x 192 27 -> 22, 1 x 384 40 ->
// 26, 1 x 1,024 88 -> 45, 1 x 2,943 223 -> 95, 1 x 16,384 1,186 -> 618, 2 x
// 256 32 -> 28, 2 x 512 51 -> 41, 2 x 1,500 126 -> 95, 2 x 2,943 226 -> 202,
// and past 64 items 3 x 1,000 91 -> 104, 4 x 2,048 164 -> 276: the records
// (91 KB per chunk and head, written and read once) then cost more than the
// idle CUs.  Up to 32 items a scan workgroup takes 16 columns (256 workgroups;
// 32 columns: 2,943 tokens at 16 heads 74 -> 102 us), past that 32 (each record
// is read four times instead of eight: 2 x 2,943 226 -> 202 us, where a CU's
// L2 reads, about 50 GB/s, bound the scan).
int64_t gdn_chunk_prefill_split_floats(int64_t T, int64_t nseq, int64_t Hk, int64_t Hv, int64_t kd, int64_t vd) {
  if (T <= 0 || nseq <= 0 || nseq > kMaxSplitSeqs || Hk <= 0 || Hv <= 0 || kd != KD || vd != VD) return 0;
  const int64_t items = nseq * Hv;
  if (items > 2 * kOneGroupItems || T < (items <= kOneGroupItems ? 192 : 256) * nseq) return 0;
  const int64_t bytes = (T / C + nseq) * (Hv * kRecBytes + Hk * kKRecBytes);
  return bytes <= (int64_t(1) << 30) ? bytes / 4 : 0;
}

namespace {
template <bool F16, bool OUT32>
hipError_t launch_split(const SplitArgs& sa, int nt, hipStream_t st) {
  // (the work maps cover whole groups of 16)
  const dim3 pgrid((unsigned)((sa.slots * sa.p.Hv + 15) / 16 * 16));
  const dim3 sgrid((unsigned)((sa.p.nseq * sa.p.Hv + 15) / 16 * 16 * (kGroups / nt)));
  gdn_prepare_kernel<F16, OUT32><<<pgrid, dim3(256), 0, st>>>(sa);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (nt == 1) gdn_scan_kernel<F16, 1, OUT32><<<sgrid, dim3(512), 0, st>>>(sa);
  else gdn_scan_kernel<F16, 2, OUT32><<<sgrid, dim3(512), 0, st>>>(sa);
  return hipGetLastError();
}
}  // namespace

hipError_t gdn_chunk_prefill_split_launch(const gdn_tensor* q, const gdn_tensor* k, const gdn_tensor* v,
                                          const gdn_tensor* g, const gdn_tensor* beta, gdn_tensor* state,
                                          const gdn_tensor* idx, const gdn_tensor* cu, gdn_tensor* out,
                                          float* workspace, float scale, int32_t flags, hipStream_t st) {
  SplitArgs sa;
  sa.p = prefill_args(q, k, v, g, beta, state, idx, cu, out, scale);
  sa.p.flags = flags;
  sa.ws = reinterpret_cast<char*>(workspace);
  sa.slots = sa.p.T / C + sa.p.nseq;
  sa.Hk = (int32_t)q->shape[1];
  const int nt = sa.p.nseq * sa.p.Hv <= kOneGroupItems ? 1 : 2;
  if (out->dtype == GDN_DTYPE_F32) return launch_split<true, true>(sa, nt, st);  // (q, k, v fp16: checked by the caller)
  return q->dtype == GDN_DTYPE_F16 ? launch_split<true, false>(sa, nt, st) : launch_split<false, false>(sa, nt, st);
}
