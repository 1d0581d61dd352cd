// C entry points of the prefill (kernels: prefill_kernel.h, prefill_split.hip).
#include "prefill_kernel.h"

namespace tmopt {
namespace {

template <int REP, bool REL>
void launch_src(const PrefillArgs& a, int src, dim3 grid, size_t lds,
                hipStream_t st) {
  if (src == kPacked)
    hipLaunchKernelGGL((prefill_kernel<REP, REL, kPacked>), grid, dim3(512), lds, st,
                       a);
  else if (src == kPaged)
    hipLaunchKernelGGL((prefill_kernel<REP, REL, kPaged>), grid, dim3(512), lds, st,
                       a);
  else if (src == kMixed)
    hipLaunchKernelGGL((prefill_kernel<REP, REL, kMixed>), grid, dim3(512), lds, st,
                       a);
  else
    hipLaunchKernelGGL((prefill_kernel<REP, REL, kPackedCM>), grid, dim3(512), lds, st,
                       a);
}

// Work-groups of one level of the grid: HKV * items per head, rounded up to
// whole XCD rounds.
int64_t level_wgs(int HKV, int BQ, int S, int max_seqlen) {
  const int64_t items = (int64_t)S * ((max_seqlen + BQ - 1) / BQ);
  if (HKV <= 8 && 8 % HKV == 0) return 8 * ((items + 8 / HKV - 1) / (8 / HKV));
  return HKV * items;
}

// Levels of a launch (1: keys are not split): split where the items are at
// most half the compute units and a query may see `min_tiles` tiles of keys
// (`max_keys` keys at most). Between half and all of them the pieces' start
// and merge cost more than the idle units give (one 777-token prompt, 200
// items: 49.9 us per call in one launch, 67.5 us split); a larger grid fills
// the chip by itself, its heaviest items first. Without cached context the
// longest run's length is known and its blocks see half of it on average, so
// the line lies higher (2000 tokens, 16 query heads, 32 tiles: 46.4 us in one
// launch, 51.4 us split); with one, the row width of the block table is only a
// bound, and the device decides item by item.
int split_levels(int64_t n_base, int BQ, int64_t max_keys, int window,
                 int min_tiles) {
  const int cus = device_cus();
  if (2 * n_base > cus) return 1;
  int64_t keys = max_keys;
  if (window > 0 && keys > (int64_t)window + BQ + kBN) keys = window + BQ + kBN;
  const int64_t tiles = (keys + kBN - 1) / kBN;
  if (tiles < min_tiles) return 1;
  int64_t n = 2 * cus / n_base;
  if (n > 64) n = 64;
  if (n > tiles / kMinPiece + 1) n = tiles / kMinPiece + 1;
  return (int)n;
}

// The same from the arguments of a launch: keys a query may see, by the run's
// own length or the row width of a block table (with a ring, which is read
// under a window, the window bounds them).
int split_levels(int64_t n_base, int BQ, int max_seqlen, int64_t bt_stride,
                 int table_wrap, int window) {
  if (bt_stride <= 0)
    return split_levels(n_base, BQ, max_seqlen, window, 48);
  const int64_t keys =
      table_wrap > 0 ? 0x3fffffff : bt_stride * kPage + max_seqlen;
  return split_levels(n_base, BQ, keys, window, kMinSplit);
}

constexpr int64_t kSlotBytes = (256 * kD + 256) * sizeof(float);
int64_t workspace_bytes_of(int levels, int64_t n_base) {
  return levels * n_base * kSlotBytes + ((n_base * 4 + 15) & ~(int64_t)15);
}

template <int REP>
void launch(const PrefillArgs& a, int src, size_t lds, hipStream_t st) {
  const dim3 grid((unsigned)a.n_base);
  if (a.rel)
    launch_src<REP, true>(a, src, grid, lds, st);
  else
    launch_src<REP, false>(a, src, grid, lds, st);
}

// One work-group: *reject = 1 unless q_pos[i] - q_pos[0] == i and
// kv_pos[i] - q_pos[0] == i for every i < T (always written, so the flag
// needs no clearing).
__global__ __launch_bounds__(1024) void positions_check_kernel(
    const int64_t* __restrict__ q_pos, const int64_t* __restrict__ kv_pos,
    int64_t T, int32_t* __restrict__ reject) {
  const int64_t p0 = q_pos[0];
  int bad = 0;
  for (int64_t i = threadIdx.x; i < T; i += blockDim.x)
    bad |= (q_pos[i] - p0 != i) | (kv_pos[i] - p0 != i);
  bad = __syncthreads_or(bad);
  if (threadIdx.x == 0) reject[0] = bad ? 1 : 0;
}

}  // namespace
}  // namespace tmopt

using namespace tmopt;

extern "C" int tmopt_prefill_check_positions(const int64_t* q_positions,
                                             const int64_t* kv_positions,
                                             int64_t T, int32_t* reject,
                                             tmopt_stream_t stream) {
  clear_error();
  TMOPT_REQUIRE(q_positions && kv_positions && reject, TMOPT_EINVAL,
                "prefill_check_positions: null pointer");
  TMOPT_REQUIRE(T > 0, TMOPT_EINVAL,
                "prefill_check_positions: T must be positive (got %lld)",
                (long long)T);
  hipLaunchKernelGGL(positions_check_kernel, dim3(1), dim3(1024), 0,
                     (hipStream_t)stream, q_positions, kv_positions, T,
                     reject);
  return check_launch("prefill_check_positions");
}

// Query heads per work-group: the largest of 8, 4, 2, 1 dividing HQ/HKV; a
// ratio above it runs as several scheduled heads per stored KV head (its keys
// then load once per group of that many query heads).
static int query_group(int ratio) {
  return ratio % 8 == 0 ? 8 : ratio % 4 == 0 ? 4 : ratio % 2 == 0 ? 2 : 1;
}

extern "C" size_t tmopt_attn_prefill_workspace_size(int num_seqs,
                                                    int max_seqlen_q, int HQ,
                                                    int HKV, int64_t bt_stride,
                                                    int table_wrap,
                                                    int window) {
  if (num_seqs <= 0 || max_seqlen_q <= 0 || HKV <= 0 || HQ <= 0 ||
      HQ % HKV != 0)
    return 0;
  const int rep = query_group(HQ / HKV);
  const int64_t hkv = HQ / rep;
  if (hkv > 65535) return 0;
  const int bq = 256 / rep;
  const int64_t n = level_wgs((int)hkv, bq, num_seqs, max_seqlen_q);
  const int levels =
      split_levels(n, bq, max_seqlen_q, bt_stride, table_wrap, window);
  return levels > 1 ? (size_t)workspace_bytes_of(levels, n) : 0;
}

static int prefill_impl(
    const void* q, int64_t q_stride_tok, int64_t q_stride_head, const void* k,
    int64_t k_stride_run, int64_t k_stride_tok, int64_t k_stride_head,
    int64_t k_stride_dim, const void* v, int64_t v_stride_run,
    int64_t v_stride_tok, int64_t v_stride_head, int64_t v_stride_dim,
    const int32_t* cu_seqlens_q,
    const int32_t* prior_lens, int num_seqs, int max_seqlen_q,
    const void* k_pool, const void* v_pool, const int32_t* block_table,
    int64_t bt_stride, int table_wrap, int page_size, int64_t num_pages,
    int HQ, int HKV, int D, int window, float scale, const void* rel,
    int64_t rel_stride_tok, int64_t rel_stride_head, int rel_extent,
    void* out, int64_t o_stride_tok, int64_t o_stride_head, float* lse,
    const int32_t* reject, void* workspace, size_t workspace_bytes,
    tmopt_stream_t stream) {
  clear_error();
  if (num_seqs == 0 || max_seqlen_q == 0) return TMOPT_OK;
  TMOPT_REQUIRE(num_seqs > 0 && num_seqs <= 65535 && max_seqlen_q > 0,
                TMOPT_EINVAL, "prefill: num_seqs=%d max_seqlen_q=%d", num_seqs,
                max_seqlen_q);
  TMOPT_REQUIRE(q && out && cu_seqlens_q, TMOPT_EINVAL,
                "prefill: null q/out/cu_seqlens");
  TMOPT_REQUIRE(D == kD, TMOPT_EUNSUPPORTED, "prefill: D=%d (only 128)", D);
  TMOPT_REQUIRE(HKV > 0 && HQ > 0 && HQ % HKV == 0 && HKV <= 65535,
                TMOPT_EINVAL, "prefill: HQ=%d HKV=%d", HQ, HKV);
  const int ratio = HQ / HKV;
  const int rep = query_group(ratio);
  const int kv_div = ratio / rep;
  TMOPT_REQUIRE((int64_t)HKV * kv_div <= 65535, TMOPT_EUNSUPPORTED,
                "prefill: HKV=%d x %d query-head groups exceeds 65535", HKV,
                kv_div);
  TMOPT_REQUIRE(window >= 0, TMOPT_EINVAL, "prefill: window=%d", window);
  TMOPT_REQUIRE(scale > 0.0f, TMOPT_EINVAL, "prefill: scale must be > 0");
  TMOPT_REQUIRE(rel == nullptr || rel_extent > 0, TMOPT_EINVAL,
                "prefill: rel_extent=%d", rel_extent);
  TMOPT_REQUIRE(rel == nullptr ||
                    (rel_stride_tok >= rel_extent && rel_stride_head >= 0 &&
                     (64 * rel_stride_tok + 2 * (int64_t)rel_extent) <
                         kOob),
                TMOPT_EUNSUPPORTED,
                "prefill: rel rows must not overlap, and 32 rows must span "
                "less than 2 GiB (stride_tok=%lld, extent=%d)",
                (long long)rel_stride_tok, rel_extent);
  {
    const int bq = 256 / rep;
    const int64_t blocks =
        (int64_t)HKV * kv_div * num_seqs * ((max_seqlen_q + bq - 1) / bq) +
        8 * 8;
    TMOPT_REQUIRE(blocks < 0x7fffffffll, TMOPT_EUNSUPPORTED,
                  "prefill: %lld work-groups exceed the grid limit",
                  (long long)blocks);
  }
  const bool pooled = block_table != nullptr;
  const bool own = k != nullptr || v != nullptr;
  const bool cm = own && (k_stride_dim != 1 || v_stride_dim != 1);
  const int src = !pooled ? (cm ? kPackedCM : kPacked)
                          : (own ? kMixed : kPaged);
  if (pooled) {
    TMOPT_REQUIRE(k_pool && v_pool && page_size > 0 && bt_stride > 0 &&
                      num_pages > 0 && table_wrap >= 0,
                  TMOPT_EINVAL,
                  "prefill: paged source needs pools, page_size, bt_stride");
    TMOPT_REQUIRE(page_size == kPage, TMOPT_EUNSUPPORTED,
                  "prefill: page_size=%d (only 16)", page_size);
    TMOPT_REQUIRE(((uintptr_t)k_pool | (uintptr_t)v_pool) % 16 == 0,
                  TMOPT_EINVAL, "prefill: pools must be 16-byte aligned");
    TMOPT_REQUIRE((int64_t)kPage * HKV * kD * 2 < (1ll << 31),
                  TMOPT_EUNSUPPORTED, "prefill: page too large");
    // A ring holds the last table_wrap * 16 positions: the run's own keys
    // would overwrite the prior context they must be read beside, so a
    // ring is read for the prior context only (mixed source), under a
    // window no wider than the ring.
    TMOPT_REQUIRE(table_wrap == 0 ||
                      (src == kMixed && table_wrap <= bt_stride && window > 0 &&
                       (int64_t)window <= (int64_t)table_wrap * kPage),
                  TMOPT_EINVAL,
                  "prefill: a ring table (table_wrap=%d) needs packed k/v for "
                  "the run's own keys and 0 < window <= %lld",
                  table_wrap, (long long)table_wrap * kPage);
  } else {
    TMOPT_REQUIRE(prior_lens == nullptr && table_wrap == 0, TMOPT_EINVAL,
                  "prefill: prior context needs a block table");
  }
  if (own) {
    TMOPT_REQUIRE(k && v, TMOPT_EINVAL, "prefill: k and v go together");
    TMOPT_REQUIRE(k_stride_run >= 0 && v_stride_run >= 0 &&
                      k_stride_run % 8 == 0 && v_stride_run % 8 == 0 &&
                      k_stride_head % 8 == 0 && v_stride_head % 8 == 0 &&
                      ((uintptr_t)k | (uintptr_t)v) % 16 == 0,
                  TMOPT_EINVAL,
                  "prefill: k/v runs and heads must start 16-byte aligned "
                  "(run and head strides %% 8)");
    if (cm) {
      // channel-major: tokens contiguous, dim rows 16-byte aligned and not
      // overlapping, runs placed by the run stride (a run's first token
      // must be 16-byte aligned, which cu_seqlens offsets do not promise)
      TMOPT_REQUIRE(!pooled, TMOPT_EUNSUPPORTED,
                    "prefill: channel-major k/v only as the packed source");
      TMOPT_REQUIRE(k_stride_tok == 1 && v_stride_tok == 1 &&
                        k_stride_dim != 1 && v_stride_dim != 1,
                    TMOPT_EINVAL,
                    "prefill: k and v must both be token-major (stride_dim "
                    "1) or both channel-major (stride_tok 1)");
      TMOPT_REQUIRE(k_stride_run > 0 && v_stride_run > 0, TMOPT_EINVAL,
                    "prefill: channel-major k/v need a run stride");
      TMOPT_REQUIRE(k_stride_dim % 8 == 0 && v_stride_dim % 8 == 0 &&
                        k_stride_dim >= max_seqlen_q &&
                        v_stride_dim >= max_seqlen_q,
                    TMOPT_EINVAL,
                    "prefill: channel-major dim rows must be 16-byte aligned "
                    "and hold max_seqlen_q tokens (stride_dim %% 8, >= %d)",
                    max_seqlen_q);
      const int64_t sd = k_stride_dim > v_stride_dim ? k_stride_dim
                                                     : v_stride_dim;
      TMOPT_REQUIRE(((kD - 1) * sd + max_seqlen_q) * 2 < kOob,
                    TMOPT_EUNSUPPORTED,
                    "prefill: a run's channel-major k/v span must stay below "
                    "2 GiB");
    } else {
      TMOPT_REQUIRE(((int64_t)max_seqlen_q * (k_stride_tok > v_stride_tok
                                                  ? k_stride_tok
                                                  : v_stride_tok) +
                     kD) * 2 < kOob,
                    TMOPT_EUNSUPPORTED,
                    "prefill: a run's packed k/v span must stay below 2 GiB");
      TMOPT_REQUIRE(k_stride_tok % 8 == 0 && v_stride_tok % 8 == 0,
                    TMOPT_EINVAL,
                    "prefill: k/v rows must be 16-byte aligned (strides %% 8)");
    }
  }
  TMOPT_REQUIRE(((int64_t)max_seqlen_q * q_stride_tok + kD) * 2 < kOob,
                TMOPT_EUNSUPPORTED,
                "prefill: a run's q span must stay below 2 GiB");
  TMOPT_REQUIRE(q_stride_tok % 8 == 0 && q_stride_head % 8 == 0 &&
                    o_stride_tok % 4 == 0 && o_stride_head % 4 == 0 &&
                    (uintptr_t)q % 16 == 0 && (uintptr_t)out % 8 == 0,
                TMOPT_EINVAL, "prefill: q/out rows misaligned");
  PrefillArgs a;
  a.q = (const __bf16*)q;
  a.q_st = q_stride_tok;
  a.q_sh = q_stride_head;
  a.k = (const __bf16*)k;
  a.k_st = k_stride_tok;
  a.k_sh = k_stride_head;
  a.v = (const __bf16*)v;
  a.v_st = v_stride_tok;
  a.v_sh = v_stride_head;
  a.k_sd = own ? k_stride_dim : 1;
  a.v_sd = own ? v_stride_dim : 1;
  a.k_sr = own ? k_stride_run : 0;
  a.v_sr = own ? v_stride_run : 0;
  a.cu = cu_seqlens_q;
  a.prior = prior_lens;
  a.kpool = (const __bf16*)k_pool;
  a.vpool = (const __bf16*)v_pool;
  a.bt = block_table;
  a.bt_stride = bt_stride;
  a.bt_width = bt_stride > 0x7fffffff ? 0x7fffffff : (int)bt_stride;
  a.table_wrap = table_wrap;
  a.num_pages = num_pages > 0x7fffffff ? 0x7fffffff : (int)num_pages;
  a.page_size = page_size > 0 ? page_size : 16;
  a.HQ = HQ;
  a.HKV = HKV * kv_div;
  a.kv_div = kv_div;
  a.HKV_stored = HKV;
  a.window = window;
  a.scale = scale;
  a.scale_log2 = scale * kLog2e;
  a.out = (__bf16*)out;
  a.o_st = o_stride_tok;
  a.o_sh = o_stride_head;
  a.lse = lse;
  a.S = num_seqs;
  a.rel = (const __bf16*)rel;
  a.r_st = rel_stride_tok;
  a.r_sh = rel_stride_head;
  a.rel_extent = rel ? rel_extent : 0;
  a.reject = reject;
  a.n_base = (int)level_wgs(a.HKV, 256 / rep, num_seqs, max_seqlen_q);
  a.split_wgs = device_cus();
  a.nsplit = workspace == nullptr
                 ? 1
                 : split_levels(a.n_base, 256 / rep, max_seqlen_q,
                                pooled ? bt_stride : 0, table_wrap, window);
  const int64_t slots = (int64_t)a.nsplit * a.n_base;
  const int64_t need = workspace_bytes_of(a.nsplit, a.n_base);
  TMOPT_REQUIRE(a.nsplit <= 1 || ((int64_t)workspace_bytes >= need &&
                                  (uintptr_t)workspace % 16 == 0),
                TMOPT_EWORKSPACE,
                "prefill: workspace %zu bytes < %lld needed (or unaligned)",
                workspace_bytes, (long long)need);
  a.part_o = (float*)workspace;
  a.part_lse = a.part_o + slots * 256 * kD;
  a.part_n = (int*)(a.part_lse + slots * 256);
  a.nqb_max = (max_seqlen_q + 256 / rep - 1) / (256 / rep);
  hipStream_t st = (hipStream_t)stream;
  const size_t lds = kNStage * kStage + (a.rel ? 8 * kBiasB : 0);
  if (a.nsplit > 1)
    launch_prefill_split(a, rep, src, lds, st);
  else if (rep == 8)
    launch<8>(a, src, lds, st);
  else if (rep == 4)
    launch<4>(a, src, lds, st);
  else if (rep == 2)
    launch<2>(a, src, lds, st);
  else
    launch<1>(a, src, lds, st);
  return check_launch("prefill");
}

extern "C" int tmopt_attn_prefill_varlen(
    const void* q, int64_t q_stride_tok, int64_t q_stride_head, const void* k,
    int64_t k_stride_run, int64_t k_stride_tok, int64_t k_stride_head,
    int64_t k_stride_dim, const void* v, int64_t v_stride_run,
    int64_t v_stride_tok, int64_t v_stride_head, int64_t v_stride_dim,
    const int32_t* cu_seqlens_q,
    const int32_t* prior_lens, int num_seqs, int max_seqlen_q,
    const void* k_pool, const void* v_pool, const int32_t* block_table,
    int64_t bt_stride, int table_wrap, int page_size, int64_t num_pages,
    int HQ, int HKV, int D, int window, float scale, const void* rel,
    int64_t rel_stride_tok, int64_t rel_stride_head, int rel_extent,
    void* out, int64_t o_stride_tok, int64_t o_stride_head, float* lse,
    const int32_t* reject, tmopt_stream_t stream) {
  return prefill_impl(
      q, q_stride_tok, q_stride_head, k, k_stride_run, k_stride_tok,
      k_stride_head, k_stride_dim, v, v_stride_run, v_stride_tok,
      v_stride_head, v_stride_dim, cu_seqlens_q, prior_lens, num_seqs,
      max_seqlen_q, k_pool, v_pool, block_table, bt_stride, table_wrap,
      page_size, num_pages, HQ, HKV, D, window, scale, rel, rel_stride_tok,
      rel_stride_head, rel_extent, out, o_stride_tok, o_stride_head, lse,
      reject, nullptr, 0, stream);
}

extern "C" int tmopt_attn_prefill_varlen_split(
    const void* q, int64_t q_stride_tok, int64_t q_stride_head, const void* k,
    int64_t k_stride_run, int64_t k_stride_tok, int64_t k_stride_head,
    int64_t k_stride_dim, const void* v, int64_t v_stride_run,
    int64_t v_stride_tok, int64_t v_stride_head, int64_t v_stride_dim,
    const int32_t* cu_seqlens_q,
    const int32_t* prior_lens, int num_seqs, int max_seqlen_q,
    const void* k_pool, const void* v_pool, const int32_t* block_table,
    int64_t bt_stride, int table_wrap, int page_size, int64_t num_pages,
    int HQ, int HKV, int D, int window, float scale, const void* rel,
    int64_t rel_stride_tok, int64_t rel_stride_head, int rel_extent,
    void* out, int64_t o_stride_tok, int64_t o_stride_head, float* lse,
    const int32_t* reject, void* workspace, size_t workspace_bytes,
    tmopt_stream_t stream) {
  return prefill_impl(
      q, q_stride_tok, q_stride_head, k, k_stride_run, k_stride_tok,
      k_stride_head, k_stride_dim, v, v_stride_run, v_stride_tok,
      v_stride_head, v_stride_dim, cu_seqlens_q, prior_lens, num_seqs,
      max_seqlen_q, k_pool, v_pool, block_table, bt_stride, table_wrap,
      page_size, num_pages, HQ, HKV, D, window, scale, rel, rel_stride_tok,
      rel_stride_head, rel_extent, out, o_stride_tok, o_stride_head, lse,
      reject, workspace, workspace_bytes, stream);
}
