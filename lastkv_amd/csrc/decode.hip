// Split-K shared-KV decode attention for gfx950.
//
// One workgroup = 4 waves = one (sequence, kv head, key split).  Each wave streams 32-token
// blocks of the tiled K/V cache straight from HBM into registers with 16-byte loads (each load
// instruction of the wave covers one contiguous 1 KiB run), double-buffered so that the next
// block is in flight while the current one is computed:
//   S^T[32 tok x 16 col] = K_tile * Q^T   two 16x16x32 bf16 MFMAs per 32 dims, 8 per block;
//                                          columns are the (<=16) query heads of the GQA group
//   online softmax in the exp2 domain, row max / row sum over the four 16-lane rows (DPP)
//   O[16 x 128] += P * V                  P split into bf16 hi + lo parts, 16 MFMAs per block,
//                                          so P*V carries ~16 mantissa bits instead of 8
// The waves of a workgroup merge their (m, l, O) states through LDS.  With one split the
// workgroup writes the normalised bf16 output; otherwise it writes an unnormalised partial
// state and lkv_decode_combine merges the splits.
#include <algorithm>
#include <atomic>

#include "attn_common.h"
#include "common.h"
#include "decode_body.h"
#include "runtime.h"

namespace lkv {
namespace {

constexpr float kNegInf = kDecodeNegInf;

template <bool kVScale, bool kNT, bool kMulti, int CG = 1, bool kPairs = false>
__global__ __launch_bounds__(256) void decode_split_kernel(const DecodeParams p) {
  __shared__ DecodeShared<CG> sm;
  DecodeItem it;
  if (!decode_item<kMulti>(p, blockIdx.x, it)) return;  // (workgroup-uniform)
  decode_split_body<kVScale, kNT, kMulti, CG, kPairs, true>(p, it, sm);
}

// Merges the per-split states of one (sequence, query head); one thread per head dim.  The splits'
// (m, l) pairs are staged in LDS and reduced in parallel (maximum, then the weights 2^(m_s - M)
// and L), so the per-dim accumulation over the splits has no dependent loads and keeps several
// partial-O loads in flight.
constexpr int kCombineThreads = kHeadDim;
constexpr int kMaxSplits = 1024;

// Merges the S split states (ml: (m, l) pairs, o: partial O rows) of one (query token, head) into
// its output row and optional LSE; every thread of the block calls it (one per head dim).
__device__ inline void combine_row(const DecodeParams& p, const float* ml, const float* o, int S, uint16_t* out_row,
                                   float* lse, int kvh, float* sm_w, float* sm_red) {
  const int d = threadIdx.x;
  float mx = kNegInf;
  for (int s = d; s < S; s += kCombineThreads) {
    const float m = ml[2 * s];
    sm_w[s] = m;
    mx = fmaxf(mx, m);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
  if ((d & 63) == 0) sm_red[d >> 6] = mx;
  __syncthreads();
  const float M = fmaxf(sm_red[0], sm_red[1]);
  __syncthreads();
  float lsum = 0.f;
  for (int s = d; s < S; s += kCombineThreads) {
    const float m = sm_w[s];
    const float f = m == kNegInf ? 0.f : fast_exp2(m - M);
    sm_w[s] = f;
    lsum += f * ml[2 * s + 1];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off);
  if ((d & 63) == 0) sm_red[d >> 6] = lsum;
  __syncthreads();
  const float L = sm_red[0] + sm_red[1];
  float O[4] = {0.f, 0.f, 0.f, 0.f};
  int s = 0;
  for (; s + 4 <= S; s += 4) {
#pragma unroll
    for (int j = 0; j < 4; ++j) O[j] += sm_w[s + j] * o[(s + j) * kHeadDim + d];
  }
  for (; s < S; ++s) O[0] += sm_w[s] * o[s * kHeadDim + d];
  const float Ot = (O[0] + O[1]) + (O[2] + O[3]);
  out_row[d] = out_bits(L > 0.f ? Ot / L : 0.f, p.out_scale, kvh);
  if (lse != nullptr && d == 0) *lse = L > 0.f ? (M + __log2f(L)) * kLn2 : kNegInf;
  __syncthreads();  // (sm_w and sm_red are reused by the caller's next row)
}

// Uniform calls: one block per [B, L, Hq] row.  Ragged calls: one block per (head, sequence, query
// token) of the launch's column class (its split count and split-state rows come from the
// sequence's rank in the class, as in the split kernel; with one split that kernel wrote the output).
__global__ __launch_bounds__(kCombineThreads) void decode_combine_kernel(const DecodeParams p) {
  __shared__ float sm_w[kMaxSplits];
  __shared__ float sm_red[kCombineThreads / 64];
  if (p.cu != nullptr) {
    const int h = blockIdx.x, b = blockIdx.y, tq = blockIdx.z;
    const MultiRows mr = multi_rows(p, b);
    if (!in_column_class(p, mr.L) || tq >= mr.L) return;  // (uniform over the block)
    const ClassRank cr = class_rank(p, b, p.hq / p.group);
    const int S = cr.splits;
    if (S == 1) return;
    const int64_t ws_row = (static_cast<int64_t>(cr.rank) * p.lmax + tq) * p.hq + h;
    const int64_t out_row = mr.row0 + tq;
    combine_row(p, p.ws_ml + ws_row * S * 2, p.ws_o + ws_row * S * kHeadDim, S,
                p.out + out_row * p.out_st + static_cast<int64_t>(h) * kHeadDim,
                p.lse != nullptr ? p.lse + out_row * p.hq + h : nullptr, h / p.group, sm_w, sm_red);
    return;
  }
  const int bh = blockIdx.x;  // [B, L, Hq] row
  const int row = bh / p.hq, h = bh % p.hq;
  const int b = row / p.L, tq = row % p.L;
  const int S = p.splits;
  combine_row(p, p.ws_ml + static_cast<int64_t>(bh) * S * 2, p.ws_o + static_cast<int64_t>(bh) * S * kHeadDim, S,
              p.out + b * p.out_sb + tq * p.out_st + static_cast<int64_t>(h) * kHeadDim,
              p.lse != nullptr ? p.lse + bh : nullptr, h / p.group, sm_w, sm_red);
}

// Non-temporal K/V loads when a call's K/V exceed 384 MiB (more than the 256 MB last-level cache
// could keep for the next layer's call over the same shared cache); hint 1 / 2 force a policy.
bool use_nontemporal(int32_t hint, int64_t kv_bytes) { return hint == 2 || (hint == 0 && kv_bytes > (int64_t{384} << 20)); }

template <int CG, bool kPairs = false>
void launch_multi(const DecodeParams& p, dim3 grid, bool vscale, bool nt, hipStream_t s) {
  if (vscale && nt)
    decode_split_kernel<true, true, true, CG, kPairs><<<grid, 256, 0, s>>>(p);
  else if (vscale)
    decode_split_kernel<true, false, true, CG, kPairs><<<grid, 256, 0, s>>>(p);
  else if (nt)
    decode_split_kernel<false, true, true, CG, kPairs><<<grid, 256, 0, s>>>(p);
  else
    decode_split_kernel<false, false, true, CG, kPairs><<<grid, 256, 0, s>>>(p);
}

int32_t launch_combine(const DecodeParams& p, int rows, hipStream_t s, const char* what) {
  if (p.splits <= 1) return LKV_OK;
  const dim3 grid = p.cu != nullptr ? dim3(p.hq, p.batch, p.lmax) : dim3(rows);
  decode_combine_kernel<<<grid, kCombineThreads, 0, s>>>(p);
  return check_launch(what);
}

// cg: 0 for decode calls (one column per head), else the 16-column groups of a short prefill call
int32_t launch_decode(const DecodeParams& p, dim3 grid, bool vscale, bool nt, int cg, int rows, hipStream_t s,
                      const char* what) {
  if (cg == 1) {
    launch_multi<1>(p, grid, vscale, nt, s);
  } else if (cg == 2) {
    launch_multi<2>(p, grid, vscale, nt, s);
  } else if (cg == 4) {  // two wave pairs of two groups each
    launch_multi<2, true>(p, grid, vscale, nt, s);
  } else {
    if (vscale && nt)
      decode_split_kernel<true, true, false><<<grid, 256, 0, s>>>(p);
    else if (vscale)
      decode_split_kernel<true, false, false><<<grid, 256, 0, s>>>(p);
    else if (nt)
      decode_split_kernel<false, true, false><<<grid, 256, 0, s>>>(p);
    else
      decode_split_kernel<false, false, false><<<grid, 256, 0, s>>>(p);
  }
  if (const int32_t st = check_launch(what)) return st;
  return launch_combine(p, rows, s, what);
}

}  // namespace

int64_t ragged_split_state_rows(int32_t batch, int32_t num_q_heads, int32_t num_kv_heads, int32_t lmax, int32_t cap,
                                int32_t fixed, int32_t cus) {
  int64_t worst = 0;
  for (int64_t n = 1; n <= batch; ++n) {
    const int64_t S = fixed > 0 ? fixed : std::min<int64_t>(cap, std::max<int64_t>(1, cus / (n * num_kv_heads)));
    if (S > 1) worst = std::max(worst, n * lmax * num_q_heads * S);
  }
  return worst;
}

int32_t plan_short_rows(const lkv_prefill_args* a, const SegParams& seg, int32_t group, int32_t col_lo, int32_t col_hi,
                        int32_t class_n, void* ws, int64_t ws_bytes, ShortRowsPlan& plan) {
  DecodeParams& p = plan.p;
  p.seg = seg;
  p.q = static_cast<const uint16_t*>(a->q);
  p.q_sb = a->q_stride_b;
  p.q_st = a->q_stride_t;
  p.out = static_cast<uint16_t*>(a->out);
  p.out_sb = a->out_stride_b;
  p.out_st = a->out_stride_t;
  p.lse = a->lse;
  p.vscale = a->vscale;
  p.out_scale = a->out_scale;
  p.batch = a->batch;
  p.hq = a->num_q_heads;
  p.group = group;
  p.cu = a->cu_seqlens_q;
  p.rows = a->tokens;
  p.L = a->cu_seqlens_q ? std::min(a->max_seqlen_q, a->tokens) : a->tokens;
  p.col_lo = col_lo;
  p.col_hi = col_hi;
  p.causal = a->causal;
  p.scale_log2 = a->sm_scale * kLog2e;
  const bool ragged = p.cu != nullptr;
  // a ragged call's sequences of this class have at most lmax query tokens
  p.lmax = ragged ? std::min(col_hi / group, p.L) : p.L;
  plan.empty = p.lmax < 1;  // (no sequence fits the class)
  if (plan.empty) return LKV_OK;
  const int64_t tokens = call_key_tokens(a);
  const int64_t blocks = (tokens + 2 * kBlockTokens - 1) / kBlockTokens;  // (+1 for a ring start inside a block)
  const int64_t pairs = static_cast<int64_t>(a->batch) * a->num_kv_heads;
  const int64_t cus = device_cu_count() > 0 ? device_cu_count() : 256;
  p.cus = static_cast<int32_t>(cus);
  // as many splits as fit one round of workgroups (one per CU), at least 4 blocks per split, partial
  // states within the workspace; a ragged call's launch caps the count at what one sequence alone
  // would take (and kRaggedSplitCap) and each launch divides the CUs among the sequences it finds in
  // its class
  int64_t splits = std::min<int64_t>({ragged ? std::min<int64_t>(std::max<int64_t>(1, cus / a->num_kv_heads), kRaggedSplitCap)
                                             : std::max<int64_t>(1, cus / pairs),
                                      std::max<int64_t>(blocks / 4, 1), 1024});
  // split-state rows x splits: [B, L, Hq] rows for uniform calls, the class's sequences by rank
  // (lmax rows each) for ragged ones
  auto state = [&](int64_t cap, int32_t fixed) -> int64_t {
    if (ragged) return ragged_split_state_rows(a->batch, a->num_q_heads, a->num_kv_heads, p.lmax, cap, fixed, p.cus);
    const int64_t S = fixed > 0 ? fixed : cap;
    return S > 1 ? static_cast<int64_t>(a->batch) * a->tokens * a->num_q_heads * S : 0;
  };
  if (a->num_splits > 0) {  // fixed by the caller (lkv_prefill_workspace_bytes counted its states)
    splits = a->num_splits;
    const int64_t need = state(splits, a->num_splits) * (kHeadDim + 2) * 4;
    if (need > ws_bytes)
      return fail(LKV_ERR_WORKSPACE, "prefill with %d decode splits needs %lld bytes of workspace, got %lld", a->num_splits,
                  static_cast<long long>(need), static_cast<long long>(ws_bytes));
  }
  while (splits > 1 && state(splits, a->num_splits > 0 ? static_cast<int32_t>(splits) : 0) * (kHeadDim + 2) * 4 >
                           ws_bytes)
    splits = (splits + 1) / 2;
  p.splits = static_cast<int32_t>(splits);
  p.dyn_splits = ragged && a->num_splits == 0;
  const int64_t state_rows = state(splits, a->num_splits > 0 ? static_cast<int32_t>(splits) : 0);
  plan.state_bytes = state_rows * (kHeadDim + 2) * 4;
  p.ws_o = state_rows > 0 ? static_cast<float*>(ws) : nullptr;
  p.ws_ml = state_rows > 0 ? p.ws_o + state_rows * kHeadDim : nullptr;
  // the class's split count when the host knows how many sequences it holds: the count the split
  // kernel derives from them (so one split launches no merge); a cap the kernel cannot exceed
  if (p.dyn_splits && class_n > 0)
    p.splits = static_cast<int32_t>(std::min<int64_t>(p.splits, std::max<int64_t>(1, cus / (int64_t{class_n} * a->num_kv_heads))));
  plan.items = class_n > 0 ? int64_t{class_n} * a->num_kv_heads * p.splits : 0;
  plan.vscale = a->older_vscale_mode == 1;
  plan.nt = use_nontemporal(0, pairs * tokens * kHeadDim * 2 * 2);
  p.interleave = seg.o_tab == nullptr && seg.l_tab == nullptr;
  // the instance holds the class's widest sequence: 16, 32 or 64 columns
  const int64_t cols = std::min<int64_t>(col_hi, static_cast<int64_t>(group) * p.L);
  plan.cg = cols <= 16 ? 1 : cols <= 32 ? 2 : 4;
  plan.out_rows = static_cast<int>((ragged ? static_cast<int64_t>(a->tokens) : static_cast<int64_t>(a->batch) * a->tokens) *
                                   a->num_q_heads);  // ([rows, Hq] ragged, [B, L, Hq] uniform)
  // split counts chosen on the device: n sequences x S(n) splits <= ceil(CUs / Hkv) + B pairs per kv head
  plan.grid = p.dyn_splits
                  ? dim3(static_cast<unsigned>(a->num_kv_heads * ((cus + a->num_kv_heads - 1) / a->num_kv_heads + a->batch)))
                  : dim3(p.splits, a->num_kv_heads, a->batch);
  return LKV_OK;
}

int32_t combine_short_rows(const ShortRowsPlan& plan, hipStream_t s, const char* what) {
  return launch_combine(plan.p, plan.out_rows, s, what);
}

int32_t prefill_on_decode_kernel(const lkv_prefill_args* a, const SegParams& seg, int32_t group, int32_t col_lo,
                                 int32_t col_hi, int32_t class_n, hipStream_t s) {
  ShortRowsPlan plan;
  if (const int32_t st = plan_short_rows(a, seg, group, col_lo, col_hi, class_n, a->workspace, a->workspace_bytes, plan))
    return st;
  if (plan.empty) return LKV_OK;
  return launch_decode(plan.p, plan.grid, plan.vscale, plan.nt, plan.cg, plan.out_rows, s,
                       "lkv_prefill_attn (short call on the decode kernel)");
}

}  // namespace lkv

extern "C" int64_t lkv_decode_workspace_bytes(int32_t batch, int32_t num_q_heads, int32_t num_splits) {
  if (batch <= 0 || num_q_heads <= 0 || num_splits <= 1) return 0;
  return static_cast<int64_t>(batch) * num_q_heads * num_splits * (lkv::kHeadDim + 2) * 4;
}

namespace lkv {
namespace {

// Argument checks of lkv_decode_attn and lkv_decode_attn_noalloc (no device calls).
int32_t check_decode_args(const lkv_decode_args* a) {
  LKV_REQUIRE(a != nullptr, "null args");
  LKV_REQUIRE(a->struct_size == static_cast<int32_t>(sizeof(lkv_decode_args)),
              "lkv_decode_args size mismatch (caller %d, library %d)", a->struct_size,
              static_cast<int32_t>(sizeof(lkv_decode_args)));
  LKV_REQUIRE(a->head_dim == kHeadDim, "head_dim must be 128, got %d", a->head_dim);
  LKV_REQUIRE(a->batch >= 0 && a->num_kv_heads > 0 && a->num_q_heads > 0, "bad sizes");
  LKV_REQUIRE(a->num_q_heads % a->num_kv_heads == 0, "num_q_heads must be a multiple of num_kv_heads");
  LKV_REQUIRE(a->num_q_heads / a->num_kv_heads <= 64, "GQA group %d exceeds 64", a->num_q_heads / a->num_kv_heads);
  LKV_REQUIRE(a->num_splits >= 1 && a->num_splits <= 1024, "num_splits must be in [1, 1024]");
  LKV_REQUIRE(a->older_vscale_mode == 0 || a->older_vscale_mode == 1, "older_vscale_mode must be 0 or 1");
  LKV_REQUIRE(a->older_vscale_mode == 0 || a->vscale != nullptr, "older_vscale_mode 1 needs vscale");
  LKV_REQUIRE(a->kv_cache_hint >= 0 && a->kv_cache_hint <= 2, "kv_cache_hint must be 0, 1 or 2, got %d", a->kv_cache_hint);
  LKV_REQUIRE(a->q != nullptr && a->out != nullptr, "null q/out");
  LKV_REQUIRE((a->q_stride_b % 8) == 0 && (reinterpret_cast<uintptr_t>(a->q) & 15) == 0,
              "q rows must be 16-byte aligned");
  return LKV_OK;
}

// The decode call of checked args with the split partials in `ws` (ws_bytes bytes).
int32_t run_decode(const lkv_decode_args* a, void* ws, int64_t ws_bytes, hipStream_t stream) {
  DecodeParams p;
  if (const int32_t st = fill_segments(a, p.seg)) return st;
  if (a->batch == 0) return LKV_OK;
  const int group = a->num_q_heads / a->num_kv_heads;
  const int64_t need = lkv_decode_workspace_bytes(a->batch, a->num_q_heads, a->num_splits);
  if (need > 0) {
    if (ws == nullptr || ws_bytes < need)
      return fail(LKV_ERR_WORKSPACE, "decode workspace needs %lld bytes, got %lld", static_cast<long long>(need),
                  static_cast<long long>(ws_bytes));
    if ((reinterpret_cast<uintptr_t>(ws) & 15) != 0) return fail(LKV_ERR_INVALID_ARGUMENT, "workspace must be 16-byte aligned");
  }
  p.q = static_cast<const uint16_t*>(a->q);
  p.q_sb = a->q_stride_b;
  p.q_st = 0;
  p.out = static_cast<uint16_t*>(a->out);
  p.out_sb = a->out_stride_b;
  p.out_st = 0;
  p.L = 1;
  p.causal = 0;
  p.cu = nullptr;
  p.rows = a->batch;
  p.col_lo = 0;
  p.col_hi = 1 << 30;
  p.dyn_splits = 0;
  p.cus = 0;
  p.lmax = 1;
  p.batch = a->batch;
  p.lse = a->lse;
  p.vscale = a->vscale;
  p.out_scale = a->out_scale;
  p.ws_o = static_cast<float*>(ws);
  p.ws_ml = need > 0 ? p.ws_o + static_cast<int64_t>(a->batch) * a->num_q_heads * a->num_splits * kHeadDim : nullptr;
  p.hq = a->num_q_heads;
  p.group = group;
  p.splits = a->num_splits;
  p.scale_log2 = a->sm_scale * kLog2e;
  const int64_t kv_bytes = static_cast<int64_t>(a->batch) * a->num_kv_heads * call_key_tokens(a) * kHeadDim * 2 * 2;
  p.interleave = p.seg.o_tab == nullptr && p.seg.l_tab == nullptr;
  // groups above 16 query heads per kv head take the multi-column instances (columns = heads)
  const int cg = group <= 16 ? 0 : group <= 32 ? 2 : 4;
  return launch_decode(p, dim3(a->num_splits, a->num_kv_heads, a->batch), a->older_vscale_mode == 1,
                       use_nontemporal(a->kv_cache_hint, kv_bytes), cg, a->batch * a->num_q_heads, stream,
                       "lkv_decode_attn");
}

// Scratch of the allocation-free entry point: the split partials of one call, in a static device
// array that each GPU holds for the life of the process.  Host code must not use the array's name
// as a device address (it is a host-side stand-in): the address on a device comes from
// hipGetSymbolAddress, taken once per device with that device current and kept here.
constexpr int64_t kNoAllocScratchBytes = LKV_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];
constexpr int kMaxScratchDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxScratchDevices];

// Device address of the current device's scratch.
int32_t current_device_scratch(void** out) {
  int dev = -1;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return fail(LKV_ERR_HIP, "hipGetDevice: %s", hipGetErrorString(err));
  if (dev < 0 || dev >= kMaxScratchDevices) return fail(LKV_ERR_UNSUPPORTED, "device %d beyond the scratch table", dev);
  void* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (ptr == nullptr) {
    err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (err != hipSuccess || ptr == nullptr)
      return fail(LKV_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(err));
    g_scratch_ptr[dev].store(ptr, std::memory_order_release);
  }
  *out = ptr;
  return LKV_OK;
}

}  // namespace
}  // namespace lkv

extern "C" int32_t lkv_decode_attn(const lkv_decode_args* a, lkv_stream_t stream) {
  using namespace lkv;
  if (const int32_t st = check_decode_args(a)) return st;
  return run_decode(a, a->workspace, a->workspace_bytes, as_stream(stream));
}

extern "C" int32_t lkv_decode_attn_noalloc(const lkv_decode_args* a, lkv_stream_t stream) {
  using namespace lkv;
  if (const int32_t st = check_decode_args(a)) return st;
  LKV_REQUIRE(a->workspace == nullptr && a->workspace_bytes == 0,
              "lkv_decode_attn_noalloc uses the library's static scratch: workspace must be NULL and workspace_bytes 0");
  const int64_t need = lkv_decode_workspace_bytes(a->batch, a->num_q_heads, a->num_splits);
  LKV_REQUIRE(need <= kNoAllocScratchBytes,
              "%d splits of %d x %d query heads need %lld bytes of split state, more than the %lld bytes of static "
              "scratch: use fewer splits, or lkv_decode_attn with a workspace",
              a->num_splits, a->batch, a->num_q_heads, static_cast<long long>(need),
              static_cast<long long>(kNoAllocScratchBytes));
  void* ws = nullptr;
  if (need > 0 && a->batch > 0) {
    if (const int32_t st = current_device_scratch(&ws)) return st;
  }
  return run_decode(a, ws, kNoAllocScratchBytes, as_stream(stream));
}
