// Split-K shared-KV decode attention, device side (decode.hip's header comment has the scheme): shared by
// the decode kernels and by the mixed-step kernel that runs decode rows beside prefill tiles.
#pragma once
#include <algorithm>

#include "attn_common.h"
#include "common.h"
#include "runtime.h"

namespace lkv {

constexpr int kDecodeWaves = 4;
constexpr float kDecodeNegInf = -__builtin_inff();
constexpr int kInterleaveBlocks = 3072;  // (96K keys; see decode_split_body)
constexpr float kLazyRaise = 8.f;  // exp2 units a block maximum may exceed m before m is raised

struct DecodeParams {
  const uint16_t* q;
  int64_t q_sb, q_st;
  uint16_t* out;
  int64_t out_sb, out_st;
  float* lse;
  SegParams seg;
  const float* vscale;
  const float* out_scale;  // [Hkv] or nullptr: out = bf16(bf16(o) * out_scale[kvh])
  float* ws_o;
  float* ws_ml;
  int32_t batch, hq, group, splits;
  int32_t L, causal;  // query tokens per sequence (1 for decode calls) and bottom-right causality
  float scale_log2;
  // ragged query rows (short-prefill calls): sequence b's tokens are rows cu[b] .. cu[b + 1] - 1 of
  // q / out (nullptr: L tokens per sequence); rows = the call's total row count.  Only sequences
  // with col_lo < tokens * group <= col_hi run in this launch.  Their split count is `splits` when
  // dyn_splits is 0, else chosen per launch on the device from the number n of sequences in the
  // class, min(splits, max(1, floor(cus / (n * Hkv)))); their split states are laid out by the sequence's
  // rank in the class, lmax token rows each.
  const int32_t* cu;
  int32_t rows, col_lo, col_hi;
  int32_t dyn_splits, cus, lmax;
  int32_t interleave;  // tiled caches: sequences of more than kInterleaveBlocks key blocks interleave their splits
};

// Query tokens of sequence b (kMulti calls) and the flattened row of its token 0 (the q / out / lse
// / split-state row index is row0 + token).
struct MultiRows {
  int L;
  int64_t row0;
};

__device__ inline MultiRows multi_rows(const DecodeParams& p, int b) {
  if (p.cu == nullptr) return MultiRows{p.L, static_cast<int64_t>(b) * p.L};
  const int s0 = min(max(p.cu[b], 0), p.rows);
  return MultiRows{min(min(max(p.cu[b + 1], s0), p.rows) - s0, p.L), s0};
}

__device__ inline bool in_column_class(const DecodeParams& p, int L) {
  const int cols = L * p.group;
  return L > 0 && cols > p.col_lo && cols <= p.col_hi;
}

// Ragged calls: the number of sequences in this launch's column class and b's rank among them (every
// wave counts them itself, 64 sequences per ballot), and the class's split count.
struct ClassRank {
  int n, rank, splits;
};

__device__ inline ClassRank class_rank(const DecodeParams& p, int b, int hkv) {
  const int lane = threadIdx.x & 63;
  int n = 0, rank = 0;
  for (int i0 = 0; i0 < p.batch; i0 += 64) {
    const int i = i0 + lane;
    const bool in = i < p.batch && in_column_class(p, multi_rows(p, i).L);
    const uint64_t m = __builtin_amdgcn_ballot_w64(in);
    n += __builtin_popcountll(m);
    if (b >= i0) rank += __builtin_popcountll(b - i0 >= 64 ? m : (m & ((uint64_t{1} << (b - i0)) - 1)));
  }
  int splits = p.splits;
  if (p.dyn_splits && n > 0) splits = min(p.splits, max(1, p.cus / (n * hkv)));
  return ClassRank{n, rank, splits};
}

// Ragged calls with the split count chosen on the device run on a compact grid: workgroup
// (kv head fastest) u-th (sequence, split) pair of the class, sequences in order, each with the
// class's split count S.  Returns false past the class's n * S pairs.
struct ClassPick {
  int b, rank, split, splits;
};

__device__ inline bool class_pick(const DecodeParams& p, int u, int hkv, ClassPick& r) {
  const int lane = threadIdx.x & 63;
  int n = 0;
  for (int i0 = 0; i0 < p.batch; i0 += 64) {
    const int i = i0 + lane;
    n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(i < p.batch && in_column_class(p, multi_rows(p, i).L)));
  }
  if (n == 0) return false;
  r.splits = min(p.splits, max(1, p.cus / (n * hkv)));
  r.rank = u / r.splits;
  r.split = u - r.rank * r.splits;
  if (r.rank >= n) return false;
  int base = 0;  // class sequences before this step's 64
  for (int i0 = 0; i0 < p.batch; i0 += 64) {
    const int i = i0 + lane;
    const bool in = i < p.batch && in_column_class(p, multi_rows(p, i).L);
    const uint64_t m = __builtin_amdgcn_ballot_w64(in);
    const int c = __builtin_popcountll(m);
    if (r.rank < base + c) {  // the (rank - base)-th class sequence of these 64
      const int below = __builtin_popcountll(m & ((uint64_t{1} << lane) - 1));
      r.b = i0 + __builtin_ctzll(__builtin_amdgcn_ballot_w64(in && below == r.rank - base));
      return true;
    }
    base += c;
  }
  return false;
}

// The bf16 output of a normalised fp32 value x of kv head kvh: bf16(x), or bf16(bf16(x) * s) with
// an output scale (the reference rescales its bf16 attention output by s in fp32).
__device__ inline uint16_t out_bits(float x, const float* out_scale, int kvh) {
  if (out_scale == nullptr) return f32_to_bf16_bits(x);
  return f32_to_bf16_bits(bf16_bits_to_f32(f32_to_bf16_bits(x)) * out_scale[kvh]);
}

struct BlockFrags {
  uint4 k[2][4];
  uint4 v[8];
};

template <bool kNT>
__device__ inline uint4 load_frag(const uint16_t* p) {
  return kNT ? load_nt(p) : *reinterpret_cast<const uint4*>(p);
}

// kNT: non-temporal loads (K/V read once and not again before they would be evicted anyway).
template <bool kNT>
__device__ inline void load_block(BlockFrags& f, const BlockRef& r, int n16, int g4) {
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
      f.k[u][kb] = load_frag<kNT>(r.k + ((u * 4 + kb) * 16 + n16) * 32 + 8 * g4);
#pragma unroll
  for (int nb = 0; nb < 8; ++nb) f.v[nb] = load_frag<kNT>(r.v + (16 * nb + n16) * 32 + 8 * g4);
}

struct SoftmaxState {
  float m, l;
  f32x4 o[8];  // O rows (heads 4*g4 + i) x dims 16*nb + n16
};

// kMulti: the columns are (query token, head) pairs; lim is this lane's column's last visible local
// token and lim_min the smallest over the columns (local blocks past it need the causal mask).
template <bool kVScale, bool kMulti>
__device__ inline void compute_block(const BlockFrags& f, const BlockRef& r, const uint4 (&qf)[4], float vs,
                                     float scale_log2, int n16, int g4, int lim, int lim_min, SoftmaxState& st) {
  f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    s0 = mfma_bf16(f.k[0][kb], qf[kb], s0);
    s1 = mfma_bf16(f.k[1][kb], qf[kb], s1);
  }
  // lane (n16 = head column, g4) holds the scores of tokens 8*g4 + j, j = 0..7
  float s[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    s[i] = s0[i] * scale_log2;
    s[4 + i] = s1[i] * scale_log2;
  }
  if (r.lo > 0 || r.hi < kBlockTokens || (kMulti && !r.older && r.seg_tok + kBlockTokens - 1 > lim_min)) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (8 * g4 + j < r.lo || 8 * g4 + j >= r.hi || (kMulti && !r.older && r.seg_tok + 8 * g4 + j > lim)) s[j] = kDecodeNegInf;
  }
  float mx = s[0];
#pragma unroll
  for (int j = 1; j < 8; ++j) mx = fmaxf(mx, s[j]);
  mx = wave_max_across_rows(mx);
  // Lazy reference: a column's m moves (and O and l are rescaled) only in a wave-uniform branch
  // taken when some column's block maximum exceeds its m by more than kLazyRaise (exp2 units), the
  // first block with a visible key included (m = -inf).  Otherwise P = 2^(s - m) stays below
  // 2^kLazyRaise; its bf16 hi + lo split keeps ~16 bits at any magnitude and O, l are fp32.
  float alpha = 1.f;
  if (__builtin_amdgcn_ballot_w64(mx > st.m + kLazyRaise)) {
    const float m_new = fmaxf(st.m, mx);
    alpha = m_new == kDecodeNegInf ? 1.f : fast_exp2(st.m - m_new);
    st.m = m_new;
    // rows of this lane's O accumulators are heads 4*g4 + i; their factors live in lanes 4*g4 + i
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float a = __shfl(alpha, 4 * g4 + i);
#pragma unroll
      for (int nb = 0; nb < 8; ++nb) st.o[nb][i] *= a;
    }
  }
  float p[8];
  if (st.m == kDecodeNegInf) {
#pragma unroll
    for (int j = 0; j < 8; ++j) p[j] = 0.f;
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) p[j] = fast_exp2(s[j] - st.m);
  }
  float rs = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
  rs = wave_sum_across_rows(rs);
  st.l = st.l * alpha + rs;
  uint4 phi, plo;
  float hi[8];
  phi.x = pack_bf16x2(p[0], p[1]);
  phi.y = pack_bf16x2(p[2], p[3]);
  phi.z = pack_bf16x2(p[4], p[5]);
  phi.w = pack_bf16x2(p[6], p[7]);
  hi[0] = bf16_lo(phi.x);
  hi[1] = bf16_hi(phi.x);
  hi[2] = bf16_lo(phi.y);
  hi[3] = bf16_hi(phi.y);
  hi[4] = bf16_lo(phi.z);
  hi[5] = bf16_hi(phi.z);
  hi[6] = bf16_lo(phi.w);
  hi[7] = bf16_hi(phi.w);
  plo.x = pack_bf16x2(p[0] - hi[0], p[1] - hi[1]);
  plo.y = pack_bf16x2(p[2] - hi[2], p[3] - hi[3]);
  plo.z = pack_bf16x2(p[4] - hi[4], p[5] - hi[5]);
  plo.w = pack_bf16x2(p[6] - hi[6], p[7] - hi[7]);
  const bool scale_v = kVScale && r.older;
#pragma unroll
  for (int nb = 0; nb < 8; ++nb) {
    const uint4 v = scale_v ? scale_frag(f.v[nb], vs) : f.v[nb];
    st.o[nb] = mfma_bf16(phi, v, st.o[nb]);
    st.o[nb] = mfma_bf16(plo, v, st.o[nb]);
  }
}

// LDS of one decode workgroup: the waves' states of the columns each holds, indexed by the column inside
// the wave's own range (with kPairs each wave pair stages only its half of the columns, so the staging
// takes 64 KiB at most and two workgroups fit on a CU).
template <int CG>
struct DecodeShared {
  float m[kDecodeWaves][16 * CG];
  float l[kDecodeWaves][16 * CG];
  float o[kDecodeWaves][16 * CG][kHeadDim];
};

// One (sequence, kv head, key split): its workgroup's share of the call.
struct DecodeItem {
  int b, kvh, split, S;
  int64_t ws_row0;  // ragged calls: split-state row of the sequence's token 0 (its rank in the class)
  MultiRows mr;     // ragged calls: this sequence's query tokens
};

// The work item of this workgroup (wg: its index among the launch's decode workgroups, on the compact 1-D
// grid of a class whose split count is chosen on the device; grid z / y / x otherwise); false: none.
template <bool kMulti>
__device__ inline bool decode_item(const DecodeParams& p, int wg, DecodeItem& it) {
  const int hkv = p.hq / p.group;
  it.S = p.splits;
  it.ws_row0 = 0;
  if (kMulti && p.dyn_splits) {
    // the class's (sequence, split) pairs on a compact 1-D grid (the split count, chosen from the
    // number of sequences in the class, is not known to the host; a grid of every sequence at the
    // largest count would mostly exit, and with the split as its fastest dimension the exiting
    // workgroups were whole XCDs: 2 splits left 6 of 8 idle)
    it.kvh = wg % hkv;
    ClassPick cp;
    if (!class_pick(p, wg / hkv, hkv, cp)) return false;  // (workgroup-uniform)
    it.b = cp.b;
    it.split = cp.split;
    it.S = cp.splits;
    it.ws_row0 = static_cast<int64_t>(cp.rank) * p.lmax;
  } else {
    it.split = blockIdx.x;
    it.kvh = blockIdx.y;
    it.b = blockIdx.z;
  }
  // ragged calls: this sequence's query tokens (workgroup-uniform; sequences of another column
  // class run in another launch)
  it.mr = kMulti ? multi_rows(p, it.b) : MultiRows{1, it.b};
  if (kMulti && !in_column_class(p, it.mr.L)) return false;
  if (!(kMulti && p.cu != nullptr)) {
    it.ws_row0 = it.mr.row0;
  } else if (!p.dyn_splits) {  // a fixed split count over a (splits, Hkv, B) grid
    it.ws_row0 = static_cast<int64_t>(class_rank(p, it.b, hkv).rank) * p.lmax;
  }
  return true;
}

// kMulti: L > 1 query tokens per sequence, column c = (token c / G, head c % G) for c < G * L <=
// 16 * CG (CG <= 2 per wave: four groups spill), in CG groups of 16 columns that share each block's K/V fragments (short prefill calls);
// otherwise column c = head c (L = 1, CG = 1).
// kPairs (with kMulti): 32 * CG columns; waves 0-1 take column groups [0, CG), waves 2-3 groups
// [CG, 2 CG), and each pair walks all of the split's blocks (every block is fetched by both pairs,
// the second time normally from L2), so no wave holds more than CG groups of state.
// kFold: see the loop (64 more registers; the instance that shares its SIMDs with other waves goes without).
template <bool kVScale, bool kNT, bool kMulti, int CG, bool kPairs, bool kFold>
__device__ __attribute__((always_inline)) inline void decode_split_body(const DecodeParams& p, const DecodeItem& it,
                                                                        DecodeShared<CG>& sm) {
  constexpr int kWaveCols = 16 * CG;  // columns one wave holds (a pair's share with kPairs)
  constexpr int kStride = kPairs ? 2 : kDecodeWaves;  // block stride of one wave
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n16 = lane & 15, g4 = lane >> 4;
  const int G = p.group, kvh = it.kvh, b = it.b, split = it.split, S = it.S;
  const int64_t ws_row0 = it.ws_row0;
  const MultiRows mr = it.mr;
  const int Lq = mr.L;

  const SeqView sv = make_seq_view(p.seg, b, kvh);
  const int nbt = sv.nb0 + (sv.n1 > 0 ? (sv.lead + sv.n1 + kBlockTokens - 1) / kBlockTokens : 0);
  // Long sequences in tiled caches interleave their splits: wave w of split s takes blocks s * kStride + w, + S * kStride, ...,
  // so that the workgroups of one (sequence, kv head) walk one window of its K and V together: fewer DRAM
  // pages are open at once than with a contiguous range per split.  At 128K keys, us with ranges and
  // interleaved: 1, 2 and 4 sequences of 8 kv heads 95.2 / 84.0, 175 / 166, 345 / 325, of 4 heads 50.6 / 48.9,
  // 96.8 / 86.7, 178 / 166, of 12 heads 129 / 124, 253 / 247, 492 / 482.  At 64K the two are within 2 % (4
  // sequences of 8 heads 164 / 167.5), at 8K ranges are ahead (16 sequences 86.5 / 91.6).  The line is a
  // sequence's own key count, so that its bits do not change with the call's other sequences or the size
  // of its cache.  Paged segments keep ranges: a block's page id would come from another cache line of the table
  // than the wave's last (9 sequences at 16K: 104.6 with ranges, 107.3 interleaved).
  const int bps = (nbt + S - 1) / S;
  const bool interleave = p.interleave && nbt > kInterleaveBlocks;
  const int step = interleave ? S * kStride : kStride;
  const int blk_begin = interleave ? split * kStride : split * bps;
  const int blk_end = interleave ? nbt : min(blk_begin + bps, nbt);

  const int cols = kMulti ? G * Lq : G;
  uint4 qf[CG][4];
  int lim[CG], lim_min = 0;  // causal limits (local token index) of this lane's columns and of column 0
  if (kMulti) lim_min = p.causal ? sv.n1 - Lq : sv.n1 - 1;
  const int cg0 = kPairs ? (wave >> 1) * CG : 0;  // this wave's first column group
#pragma unroll
  for (int cg = 0; cg < CG; ++cg) {
    const int c = 16 * (cg0 + cg) + n16;
    const int t = kMulti ? c / G : 0, h = c - t * G;
    const uint16_t* qrow = p.q + (kMulti && p.cu ? mr.row0 * p.q_st : b * p.q_sb) + (kMulti ? t * p.q_st : 0) +
                           static_cast<int64_t>(kvh * G + h) * kHeadDim;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
      qf[cg][kb] = c < cols ? *reinterpret_cast<const uint4*>(qrow + 32 * kb + 8 * g4) : make_uint4(0, 0, 0, 0);
    lim[cg] = kMulti && p.causal ? lim_min + t : lim_min;
  }
  const float vs = kVScale ? p.vscale[kvh] : 1.f;

  SoftmaxState st[CG];
#pragma unroll
  for (int cg = 0; cg < CG; ++cg) {
    st[cg].m = kDecodeNegInf;
    st[cg].l = 0.f;
#pragma unroll
    for (int nb = 0; nb < 8; ++nb) st[cg].o[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  auto compute = [&](const BlockFrags& f, const BlockRef& r) __attribute__((always_inline)) {
#pragma unroll
    for (int cg = 0; cg < CG; ++cg)
      compute_block<kVScale, kMulti>(f, r, qf[cg], vs, p.scale_log2, n16, g4, lim[cg], lim_min, st[cg]);
  };

  // this wave's blocks: first + step * t, t < nw; block t + 1 is loaded while block t is computed.  The
  // loop runs while two or more blocks remain, so its loads are unconditional (the compiler then counts
  // them exactly for s_waitcnt); the last one or two blocks follow it.
  const int first = blk_begin + (kPairs ? (wave & 1) : wave);
  if (first < blk_end) {
    int nw = (blk_end - 1 - first) / step + 1;
    // A wave with one block more than the workgroup's last wave (the split's block count is not a
    // multiple of the waves) fetches that last block together with its first one and computes it
    // after the loop, so its extra block adds compute but no round trip to memory: the loop, whose
    // iterations are bound by load latency, then runs as many iterations in every wave.
    const int last_first = blk_begin + kStride - 1;
    const int nw_last = last_first < blk_end ? (blk_end - 1 - last_first) / step + 1 : 0;
    const bool fold = kFold && nw > nw_last && nw >= 2;
    BlockFrags fa, fb, fc;
    BlockRef ra = block_ref(sv, first), rc{};
    load_block<kNT>(fa, ra, n16, g4);
    if (fold) {
      rc = block_ref(sv, first + step * (nw - 1));
      load_block<kNT>(fc, rc, n16, g4);
      --nw;
    }
    int t = 0;
    // (the scheduling barriers keep the block being computed from moving above the next block's
    // loads, where reusing its registers would make the loads wait for it)
    for (; t + 2 < nw; t += 2) {
      const BlockRef rb = block_ref(sv, first + step * (t + 1));
      load_block<kNT>(fb, rb, n16, g4);
      __builtin_amdgcn_sched_barrier(0);
      compute(fa, ra);
      ra = block_ref(sv, first + step * (t + 2));
      load_block<kNT>(fa, ra, n16, g4);
      __builtin_amdgcn_sched_barrier(0);
      compute(fb, rb);
    }
    if (t + 1 < nw) {
      const BlockRef rb = block_ref(sv, first + step * (t + 1));
      load_block<kNT>(fb, rb, n16, g4);
      compute(fa, ra);
      compute(fb, rb);
    } else {
      compute(fa, ra);
    }
    if (fold) compute(fc, rc);
  }

  // merge the four waves' states
#pragma unroll
  for (int cg = 0; cg < CG; ++cg) {
    if (g4 == 0 && 16 * (cg0 + cg) + n16 < cols) {
      sm.m[wave][16 * cg + n16] = st[cg].m;
      sm.l[wave][16 * cg + n16] = st[cg].l;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int hl = 16 * cg + 4 * g4 + i;  // column 16 * cg0 + hl
      if (16 * cg0 + hl < cols) {
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) sm.o[wave][hl][16 * nb + n16] = st[cg].o[nb][i];
      }
    }
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < cols * kHeadDim; idx += 256) {
    const int h = idx >> 7, d = idx & (kHeadDim - 1);  // column h = (token tq, head hh)
    const int tq = kMulti ? h / G : 0, hh = h - tq * G;
    const int64_t row_q = (mr.row0 + tq) * p.hq + kvh * G + hh;  // [rows, Hq] row
    // the waves that hold column h: all four, or the pair of its column group
    const int pair = kPairs ? h / kWaveCols : 0;
    const int w0 = 2 * pair, hl = h - pair * kWaveCols;  // its waves and its column inside their range
    constexpr int kMergeWaves = kPairs ? 2 : kDecodeWaves;
    float M = sm.m[w0][hl];
#pragma unroll
    for (int w = w0 + 1; w < w0 + kMergeWaves; ++w) M = fmaxf(M, sm.m[w][hl]);
    float L = 0.f, O = 0.f;
#pragma unroll
    for (int w = w0; w < w0 + kMergeWaves; ++w) {
      const float f = sm.m[w][hl] == kDecodeNegInf ? 0.f : fast_exp2(sm.m[w][hl] - M);
      L += f * sm.l[w][hl];
      O += f * sm.o[w][hl][d];
    }
    if (S == 1) {
      p.out[(kMulti && p.cu ? mr.row0 * p.out_st : b * p.out_sb) + (kMulti ? tq * p.out_st : 0) +
            static_cast<int64_t>(kvh * G + hh) * kHeadDim + d] =
          out_bits(L > 0.f ? O / L : 0.f, p.out_scale, kvh);
      if (p.lse != nullptr && d == 0) p.lse[row_q] = L > 0.f ? (M + __log2f(L)) * kLn2 : kDecodeNegInf;
    } else {
      const int64_t row = ((ws_row0 + tq) * p.hq + kvh * G + hh) * S + split;
      p.ws_o[row * kHeadDim + d] = O;
      if (d == 0) {
        p.ws_ml[row * 2] = M;
        p.ws_ml[row * 2 + 1] = L;
      }
    }
  }
}

// Key tokens a call can read per sequence (lengths read from device memory bounded by the
// capacities); Args is lkv_decode_args or lkv_prefill_args (same segment fields).
template <typename Args>
inline int64_t call_key_tokens(const Args* a) {
  const int64_t ring_tokens = static_cast<int64_t>(a->local_ring_blocks) * kBlockTokens;
  const int64_t older = a->older_k == nullptr ? 0
                                              : (a->older_len != nullptr ? a->older_capacity_tokens
                                                                         : std::min(a->older_len_const, a->older_capacity_tokens));
  const int64_t local = a->local_k == nullptr
                            ? 0
                            : (a->local_len != nullptr ? ring_tokens : std::min<int64_t>(a->local_len_const, ring_tokens));
  return std::max<int64_t>(older, 0) + std::max<int64_t>(local, 0);
}

// The launch of a ragged or short prefill call's sequences of one column class (col_lo < group * tokens <=
// col_hi) on the decode kernels.
struct ShortRowsPlan {
  DecodeParams p;
  dim3 grid;
  int cg;           // 16-column groups of the instance: 1, 2 or 4 (two wave pairs)
  bool vscale, nt;
  int out_rows;     // combine grid: one block per output row (uniform calls)
  bool empty;       // no sequence can fall in the class
  int64_t items;    // (kv head, sequence, split) work items when the host knows the class's count, else 0
  int64_t state_bytes;  // of ws the split states take
};

// Fills the plan with the split states in ws (ws_bytes bytes); class_n: the number of the ragged call's
// sequences in the class when the host knows it, else -1.
int32_t plan_short_rows(const lkv_prefill_args* a, const SegParams& seg, int32_t group, int32_t col_lo, int32_t col_hi,
                        int32_t class_n, void* ws, int64_t ws_bytes, ShortRowsPlan& plan);

// Merges the key splits of a launched plan (nothing to do for one split).
int32_t combine_short_rows(const ShortRowsPlan& plan, hipStream_t s, const char* what);

}  // namespace lkv
