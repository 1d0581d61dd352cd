// Persistent split-KV paged decode attention for gfx950 (CDNA4).
//
// Replaces _attn_decode_kernel (engine/pyengine/kernels/attn_swa.py:49-117):
// one query token per sequence against its paged K/V history, a GQA group
// of REP query heads per KV head, fp32 online softmax, probabilities rounded
// to bf16 for the P.V product (attn_swa.py:110-112), one bf16 rounding of
// the output. What is different, and why (MI355X):
//
//  * Balanced persistent grid. The visible pages of all sequences are laid
//    end to end (U pages in total) and work-group i of G processes the
//    contiguous range [i*C, (i+1)*C), C = max(ceil(U / G), min_pages). Every
//    work-group therefore streams the same number of bytes whatever the
//    length distribution, and the grid is fixed (G = 3/4 of the CUs by
//    default), so one launch shape serves every step of a captured
//    hipGraph.
//  * Only pages holding visible keys are touched: [lo/16, ceil(n/16)) where
//    lo = max(0, n - window) on sliding-window layers, 0 on global ones.
//  * A sequence cut by work-group boundaries leaves one normalised partial
//    (O, LSE) per piece, in slot b + i of the workspace (unique: work-groups
//    and sequences are both in order); decode_combine_kernel then merges
//    the pieces of each such sequence in work-group order. No atomics and no
//    cross-work-group fences (a device-scope release/acquire pair writes
//    back and invalidates a whole XCD L2 on MI355X), and a fixed merge
//    order, so repeated runs are bitwise identical. A sequence that one
//    work-group covers alone is written in place and skipped by the merge.
//  * One wave per KV head. The four waves of a work-group read the four
//    256-byte head slices of the same token rows, so together they stream
//    whole 16 KB pages.
//  * K and V go from global memory straight into LDS (buffer_load ... lds,
//    1 KB per instruction, no registers), per wave into two stages of one
//    step (two pages, 32 tokens) each. A step's fragments are read into
//    registers first, which frees its stage for the step after next: two
//    steps (32 KB per wave) fly while one is computed. The resource of a
//    load is the rows of one page that hold visible keys: other rows (a
//    window's first page, a sequence's last one, a missing page, steps past
//    the range) read as zeros and cost no memory traffic, so every step
//    issues the same number of loads (no branch around them) and the waits
//    count exactly.
//  * Coalesced loads: each group of 16 lanes reads one token's 256-byte
//    head slice. The tiles are XOR-swizzled (by permuting which 16 bytes a
//    lane fetches) so that the fragment reads do not conflict on 64 banks;
//    V^T fragments are transposed reads. Loading the MFMA layout directly
//    (16 tokens per instruction, lanes 1 KB apart) cost 12-15 % of the
//    bandwidth.
//  * The page ids of a work-group's range are fetched before the walk, one
//    page per thread, into LDS.
//  * Scores and P.V run on MFMA (v_mfma_f32_16x16x32_bf16). S^T = K.Q^T puts
//    16 tokens on the M axis and the REP heads (padded to 16) on N, so each
//    lane owns 8 scores of one head: the running max needs two cross-lane
//    steps (xor 16, xor 32) and the running sum stays lane-local until the
//    end of a piece. P^T is then already in the B-operand layout of
//    O^T = V^T.P^T. Any GQA ratio up to 16 fills that many columns (one
//    read of the pages); a larger one runs as groups of its largest divisor
//    up to 16, each group a scheduled KV head of its own.
//
// What bounds it: HBM on large batches (6.2-6.45 TB/s at 64-128 sequences);
// on small ones, and beside another kernel, the rate at which one compute
// unit streams. See the walk for what that rate is made of.
//
// Per step (tile t = page t):
//  S^T: lane (r, g) reads row 16t + r, dims 32kk + 8g..+7 (one 16-byte read).
//  P.V: the A operand of lane (r, g) is dim 16 blk + r of tokens 4g..4g+3
//  and 16+4g..16+4g+3 (two transposed reads), matching the P^T lane layout
//  (element 4t + i <-> token 16t + 4g + i).
#include <mutex>

#include "common.h"

namespace tmopt {
namespace {

constexpr int kD = 128;
constexpr int kPS = 16;                      // tokens per page
constexpr int kRowB = 256;                   // one token's head slice
constexpr int kTileB = 2 * kPS * kRowB;      // 32 tokens: 8 KB
constexpr int kBiasB = 5 * 256;              // bias windows of a step, per wave
// LDS of a wave: two stages of one step each (K tile, V tile, bias windows),
// then the query rows of a piece
constexpr int stage_bytes(bool rel) { return 2 * kTileB + (rel ? kBiasB : 0); }
constexpr int wave_lds(bool rel) { return 2 * stage_bytes(rel) + kPS * kRowB; }
constexpr int kMaxB = 8192;                  // prefix table lives in LDS
// page ids of a range kept in LDS, beside four waves' tiles
constexpr int ids_kept(bool rel) { return rel ? 1500 : 4000; }
struct DecodeArgs {
  const __bf16* q;
  const __bf16* kpool;
  const __bf16* vpool;
  const int32_t* bt;
  int64_t bt_stride;
  int bt_width;      // entries a row may be read at: min(bt_stride, 2^31-1)
  int table_wrap;
  const int32_t* ctx_lens;
  // the engine's own index tensors instead of a block table and lengths,
  // with pos64 [B] int64 query positions (keys = pos + 1): kind 1
  // (tmopt_attn_decode_flat) = per-token pool rows [B, bt_stride] int64 (page
  // lp = row 16 lp / 16; bt_width counts its pages), kind 2
  // (tmopt_attn_decode_ring) = ring slots [B] int64 (page slot * table_wrap +
  // lp % table_wrap)
  int bt_kind;
  const int64_t* rows64;
  const int64_t* pos64;
  int B, HQ;
  int HKV;           // KV heads as scheduled (HKV_stored * kv_div)
  int num_pages;     // clamped to INT32_MAX: page ids are int32
  int window;
  float scale_log2;  // scale * log2(e)
  const __bf16* rel;
  int rel_extent;
  int min_pages;     // lower bound of pages per work-group
  int seqs_per_wg;   // > 0: work-group i takes whole sequences
                     // [i * seqs_per_wg, (i + 1) * seqs_per_wg), no merge
  __bf16* out;
  float* lse;
  float* part_o;     // [B + G, HQ, D] fp32
  float* part_lse;   // [B + G, HQ]
  int* geo;          // [B + 2]: C, then the page-stream prefix pref[0..B]
  int ids_off;       // LDS byte offset of the range's page ids
  // read by the REP 0 kernels only (any other REP implies rep == REP,
  // kv_div == 1, HKV_stored == HKV)
  int rep;           // query heads per scheduled KV head (1..16)
  int kv_div;        // scheduled KV heads per stored one: 1 unless HQ/HKV
                     // is above 16 (then kv_div groups of `rep` query
                     // heads each read the stored head's pages)
  int HKV_stored;    // KV heads of a pool token row
};

__device__ __forceinline__ int vis_lo(int n, int window) {
  return (window > 0 && n > window) ? n - window : 0;
}

// visible pages of a sequence holding n tokens
__device__ __forceinline__ int vis_pages(int n, int window) {
  if (n <= 0) return 0;
  return (n + kPS - 1) / kPS - vis_lo(n, window) / kPS;
}

// The kernel's arguments in the argument segment. `rare`: read again there
// (the pointer is opaque to the compiler) where they are needed rarely, at a
// new sequence or a piece's end: held over the walk they cost more scalar
// registers than there are.
typedef const __attribute__((address_space(4))) DecodeArgs* ArgsPtr;
__device__ __forceinline__ ArgsPtr kernel_args(bool rare) {
  auto p = (ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
  if (rare) asm volatile("" : "+s"(p));
  return p;
}

// keys of sequence b (its query sits at position n - 1)
template <int KIND>
__device__ __forceinline__ int seq_n(ArgsPtr a, int b) {
  if constexpr (KIND != 0) return (int)(as_const(a->pos64)[b] + 1);
  return as_const(a->ctx_lens)[b];
}

template <int KIND>
__device__ __forceinline__ int page_id(ArgsPtr a, int b, int lp) {
  const int idx = a->table_wrap > 0 ? lp % a->table_wrap : lp;
  int v;
  if constexpr (KIND == 2) {
    v = (int)as_const(a->rows64)[b] * a->table_wrap + idx;
  } else {
    // a logical page past the row's width has no entry: its keys are absent
    // (reading on would return the next row's page ids)
    if ((unsigned)idx >= (unsigned)a->bt_width) return -1;
    if constexpr (KIND == 1)
      v = (int32_t)(as_const(a->rows64)[(int64_t)b * a->bt_stride +
                                        (int64_t)kPS * idx] / kPS);
    else
      v = as_const(a->bt)[(int64_t)b * a->bt_stride + idx];
  }
  return (unsigned)v < (unsigned)a->num_pages ? v : -1;
}

// One 32-token step of the flattened page stream (wave-uniform; small, since
// three of them are held in scalar registers).
struct Step {
  int b;       // sequence (-1: past the end of this work-group's range)
  int n;       // its context length
  int pg;      // first logical page
  int flags;
};
enum : int {
  kFirst = 1,   // first step of this piece: the query rows come with it
  kLast = 2,    // last step of this piece of sequence b
  kFull = 4,    // both pages present and all 32 tokens visible
  kPage0 = 8,   // the pages are there
  kPage1 = 16,
  kWhole = 32,  // the piece is the whole sequence
};

// distance of the step's first token
__device__ __forceinline__ int rel_dist(const Step& st) {
  return st.n - 1 - st.pg * kPS;
}

// The bias of tile t's four scores of a lane out of the three dwords it
// fetched: rel[d - i] for i = 0..3, zero from d - i = E on (the band's end).
__device__ __forceinline__ void bias_values(const DecodeArgs& a, const Step& st,
                                            const uint32_t (&w)[3], int t,
                                            int sh, int g, float (&v)[4]) {
  const uint32_t z0 = __builtin_amdgcn_alignbyte(w[1], w[0], sh);
  const uint32_t z1 = __builtin_amdgcn_alignbyte(w[2], w[1], sh);
  const uint32_t b[4] = {z1 & 0xffff0000u, z1 << 16, z0 & 0xffff0000u,
                         z0 << 16};
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = __builtin_bit_cast(float, b[i]);
  const int d0 = rel_dist(st) - 16 * t;   // of the tile's oldest token
  if (d0 >= a.rel_extent) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[i] = d0 - 4 * g - i < a.rel_extent ? v[i] : 0.0f;
  }
}

// One work-group per CU by its LDS, one wave per SIMD. 256 registers: O^T then
// stays in vector registers (given the whole register file the compiler kept
// it in the accumulator half and moved all 32 values back and forth each step).
template <int REP, bool REL, int KIND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void decode_kernel(DecodeArgs a) {
  extern __shared__ __align__(16) char smem[];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = blockDim.x >> 6;
  const int r = lane & 15;  // MFMA row / column index
  const int g = lane >> 4;  // MFMA k-group
  const int wg = blockIdx.x;
  const int G = gridDim.x;
  const int kvh = blockIdx.y * nw + w;
  // the tables of the batch (prefix of visible pages, lengths) are only read
  // before the walk; the per-wave K / V tiles then reuse the same LDS (a
  // barrier separates the two uses). The range's page ids follow both.
  int* pref = reinterpret_cast<int*>(smem);  // [B + 1]
  int* wsum = pref + a.B + 1;                // [4]
  int* nlen = wsum + 4;                      // [B]
  int* ids = reinterpret_cast<int*>(smem + a.ids_off);   // [ids_kept + 2]

  // ---- 1. prefix sums of visible pages: pref[b] = first unit of seq b ----
  {
    int carry = 0;
    for (int b0 = 0; b0 < a.B; b0 += blockDim.x) {
      const int b = b0 + threadIdx.x;
      const int nb = b < a.B ? seq_n<KIND>(kernel_args(false), b) : 0;
      const int v = vis_pages(nb, a.window);
      if (b < a.B) nlen[b] = nb;
      // inclusive scan over the wave by DPP (VALU, no LDS round trips):
      // within each 16-lane row by shifts of 1, 2, 4, 8, then row 0's
      // total into row 1 and row 2's into row 3, then rows 0-1's total into
      // rows 2-3
      int x = v;
      x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, true);  // shr 1
      x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, true);  // shr 2
      x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, true);  // shr 4
      x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, true);  // shr 8
      x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false); // bcast 15
      x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false); // bcast 31
      if (lane == 63) wsum[w] = x;
      __syncthreads();
      int before = carry;
      for (int j = 0; j < w; ++j) before += wsum[j];
      if (b < a.B) pref[b + 1] = before + x;
      int tot = 0;
      for (int j = 0; j < nw; ++j) tot += wsum[j];
      carry += tot;
      __syncthreads();
    }
    if (threadIdx.x == 0) pref[0] = 0;
    __syncthreads();
  }
  const int U = __builtin_amdgcn_readfirstlane(pref[a.B]);
  int C = (U + G - 1) / G;
  if (C < a.min_pages) C = a.min_pages;
  // publish the split geometry for the combine kernel
  if (wg == 0 && blockIdx.y == 0) {
    for (int i = threadIdx.x; i <= a.B; i += blockDim.x) a.geo[1 + i] = pref[i];
    if (threadIdx.x == 0) a.geo[0] = C;
  }
  // this work-group's page range: an equal share of the page stream, or
  // (seqs_per_wg > 0) the pages of whole sequences, so that no sequence is
  // split and the merge has nothing to do
  int u0, u1;
  if (a.seqs_per_wg > 0) {
    const int b0 = min(wg * a.seqs_per_wg, a.B);
    const int b1 = min(b0 + a.seqs_per_wg, a.B);
    u0 = __builtin_amdgcn_readfirstlane(pref[b0]);
    u1 = __builtin_amdgcn_readfirstlane(pref[b1]);
  } else {
    u0 = min(wg * C, U);
    u1 = min(u0 + C, U);
  }
  // REP 1, 2, 4, 8, 16: that many query heads per KV head; REP 0: a.rep
  // of them (any count up to the 16 MFMA columns) and a.kv_div scheduled
  // heads per stored one
  const int rep = REP > 0 ? REP : a.rep;
  const int hq = kvh * rep + r;  // query head owned as MFMA column r
  const bool head_ok = r < rep;

  // ---- 2. sequences with no visible key: output 0, LSE -inf -------------
  for (int b = wg; b < a.B; b += G) {
    if (pref[b + 1] != pref[b] || !head_ok) continue;
    __bf16* o = a.out + ((int64_t)b * a.HQ + hq) * kD;
#pragma unroll
    for (int blk = 0; blk < 8; ++blk)
      *reinterpret_cast<u32x2*>(o + 16 * blk + 4 * g) = u32x2{0, 0};
    if (a.lse && g == 0) a.lse[(int64_t)b * a.HQ + hq] = -INFINITY;
  }
  if (u0 >= u1) return;

  constexpr int kStageB = stage_bytes(REL);
  // ---- 3. the step stream of [u0, u1) -----------------------------------
  // Everything about the step stream is wave-uniform and lives in SGPRs. The
  // page ids of the whole range are fetched here, one page per thread, into
  // LDS: looked up step by step (a dependent scalar load or two per step,
  // each waited for before the step's loads could go out) they cost every
  // step several hundred cycles. The walk reads them one step ahead. In a
  // range of more than kIds pages (a caller's own small grid, or contexts
  // adding up to millions of tokens) the later ones are looked up step by
  // step. Lengths of later sequences come from scalar loads.
  constexpr int kIds = ids_kept(REL);
  auto seq_of = [&](int u) {   // first sequence with pref[b + 1] > u
    int lo = 0, hi = a.B - 1;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (pref[mid + 1] > u) hi = mid; else lo = mid + 1;
    }
    return lo;
  };
  const int nids = min(u1 - u0, kIds);
  for (int i = threadIdx.x; i < nids; i += blockDim.x) {
    const int b = seq_of(u0 + i);
    ids[i] = page_id<KIND>(kernel_args(false), b,
                           vis_lo(nlen[b], a.window) / kPS +
                               (u0 + i - pref[b]));
  }
  int cb = __builtin_amdgcn_readfirstlane(seq_of(u0));
  int seq_start = __builtin_amdgcn_readfirstlane(pref[cb]);
  int cur_n = __builtin_amdgcn_readfirstlane(nlen[cb]);
  int seq_end = seq_start + vis_pages(cur_n, a.window);
  int pg_of = vis_lo(cur_n, a.window) / kPS - seq_start;   // page of unit u
  int cu = u0;
  int last_b = -1;  // sequence of the previous step handed out
  __syncthreads();  // the ids are there; every wave is done with the tables
  // LDS address of the next step's ids (a range's first step is at least one
  // page; what lies past its last page is read and not used)
  uint32_t ids_at =
      (uint32_t)(uintptr_t)((__attribute__((address_space(3))) int*)ids);
  const uint32_t ids_end = ids_at + 4 * kIds;
  int id0 = (int)lds_ld32(ids_at), id1 = (int)lds_ld32(ids_at + 4);
  // The next step, and the pages it reads (-1: none).
  auto next_step = [&](Step& st, int& phys0, int& phys1)
      __attribute__((always_inline)) {
    st.b = -1;
    st.n = st.pg = st.flags = 0;
    phys0 = phys1 = -1;
    if (cu >= u1) return;
    if (seq_end <= cu) {   // the next sequence that has a page
      const ArgsPtr ra = kernel_args(true);
      do {
        ++cb;
        seq_start = seq_end;
        cur_n = seq_n<KIND>(ra, cb);
        seq_end = seq_start + vis_pages(cur_n, a.window);
      } while (seq_end <= cu);
      pg_of = vis_lo(cur_n, a.window) / kPS - seq_start;
    }
    const int cnt = min(2, min(seq_end, u1) - cu);
    st.b = cb;
    st.n = cur_n;
    st.pg = cu + pg_of;
    phys0 = __builtin_amdgcn_readfirstlane(id0);
    phys1 = __builtin_amdgcn_readfirstlane(id1);
    if (ids_at + 4 * cnt > ids_end) {
      const ArgsPtr ra = kernel_args(true);
      phys0 = page_id<KIND>(ra, cb, st.pg);
      phys1 = cnt > 1 ? page_id<KIND>(ra, cb, st.pg + 1) : -1;
    }
    if (cnt < 2) phys1 = -1;
    cu += cnt;
    ids_at = min(ids_at + 4 * cnt, ids_end);
    id0 = (int)lds_ld32(ids_at);
    id1 = (int)lds_ld32(ids_at + 4);
    // every token visible: not before the window, not past the end
    const int past = st.n - (st.pg + 2) * kPS;
    const bool full = (phys0 | phys1) >= 0 && past >= 0 &&
                      (a.window <= 0 || past + 2 * kPS <= a.window);
    st.flags = (cb != last_b ? kFirst : 0) |
               (cu == min(seq_end, u1) ? kLast : 0) | (full ? kFull : 0) |
               (phys0 >= 0 ? kPage0 : 0) | (phys1 >= 0 ? kPage1 : 0) |
               (seq_start >= u0 && seq_end <= u1 ? kWhole : 0);
    last_b = cb;
  };

  const int row_elems = (REP > 0 ? a.HKV : a.HKV_stored) * kD;
  const int kvs = REP > 0 ? kvh : kvh / a.kv_div;   // the stored KV head
  const int row_bytes = row_elems * 2;
  // Tiles in LDS: 32 token rows of 256 B each for K, then for V. K row x
  // keeps 16-byte chunk c at slot c ^ (x & 15), V row x keeps 32-byte unit u
  // at slot u ^ (x & 7): conflict-free for the K fragment reads (16 rows, one
  // chunk) and for the transposed V reads (8 rows, one unit, per 32 lanes).
  // They arrive by direct loads, 4 rows per instruction: lane l fills row
  // l >> 4, physical slot l & 15, and fetches the chunk that belongs there
  // (a group of 16 lanes reads one token's whole 256-byte head slice).
  const int wtok = lane >> 4, wslot = lane & 15;
  int koff[4], voff[4];   // byte offsets in a page of rows 4i + wtok, less
                          // the 1024 i that the instruction's own offset adds
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int x = 4 * i + wtok;
    const int base = x * row_bytes + kvs * kRowB - 1024 * i;
    koff[i] = base + 16 * (wslot ^ x);
    voff[i] = base + 32 * ((wslot >> 1) ^ (x & 7)) + 16 * (wslot & 1);
  }
  const uint32_t lds_w =
      (uint32_t)(uintptr_t)((__attribute__((address_space(3))) char*)smem) +
      w * wave_lds(REL);
  const uint32_t lds_q = lds_w + 2 * kStageB;
  // K fragment (t, kk) of lane (r, g): row 16t + r, chunk 4kk + g (queries
  // alike: row = head)
  const uint32_t kr0 = lds_w + r * kRowB + 16 * (g ^ r);
  // transposed V reads: rows 4g + (s >> 2) (+16), unit blk, dims 4 (s & 3)
  const int x0 = 4 * g + (wslot >> 2);
  const uint32_t vr0 = lds_w + kTileB + x0 * kRowB + 32 * (x0 & 7) +
                       8 * (wslot & 3);

  // ---- direct loads of one step --------------------------------------------
  // Always kNK for K and the bias, then 8 for V, whatever the step holds, so
  // that the waits below can count: rows of a page that hold no visible key
  // (and missing pages, and steps past the range) are outside the resource,
  // arrive as zeros and are not fetched, so nothing has to be zeroed before
  // P.V. (A page of the walk holds a visible key; a step's second page never
  // holds the first one.)
  constexpr int kRepMax = REP > 0 ? REP : 16;
  constexpr int kNB = (kRepMax + 3) / 4 + 1;   // bias window loads
  constexpr int kNK = REL ? 8 + kNB : 8, kNS = kNK + 8;
  auto page_dma = [&](const __bf16* pool, const Step& st, int phys0, int phys1,
                      uint32_t dst, const int (&off)[4])
      __attribute__((always_inline)) {
    const int past = st.n - st.pg * kPS;   // tokens from the step's first on
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int phys = t == 0 ? phys0 : phys1;
      const int r_lo = t == 0 && a.window > 0 ? max(0, past - a.window) : 0;
      const int r_hi = min(kPS, past - kPS * t);
      const uint64_t base = (uint64_t)(uint32_t)max(phys, 0) *
                                (uint32_t)(kPS * row_bytes) +
                            (uint32_t)(r_lo * row_bytes);
      const i32x4 rs =
          make_rsrc(reinterpret_cast<const char*>(pool) + base,
                    phys >= 0 ? (uint32_t)((r_hi - r_lo) * row_bytes) : 0u);
      if (t == 0 && r_lo > 0) {   // the window's first page
        const int d = r_lo * row_bytes;
        dma4_nt<false>(rs, dst, off[0] - d, off[1] + 1024 - d,
                       off[2] + 2048 - d, off[3] + 3072 - d);
      } else {
        dma4_nt<true>(rs, dst + t * kPS * kRowB, off[0], off[1], off[2],
                      off[3]);
      }
    }
  };
  // Bias: of each head's row, the 32 values the step's tokens take (distances
  // D - 31 .. D, D that of the first token): 17 dwords from the one that holds
  // rel[D - 31]. 16 lanes fetch a head's first 16, four heads per load, into
  // 64 bytes per head; one more load takes the 17th dwords. Dwords before the
  // sequence's rows read as zeros; what they, or another row's values, put
  // into a score past the band or masked is dropped. A step wholly past the
  // band fetches nothing.
  // byte offset of the 16-lane group's head row; padded heads: past every
  // resource, whatever the distance adds
  auto rel_row = [&](int hr) {
    return hr < rep ? (kvh * rep + hr) * a.rel_extent * 2 : 0x60000000;
  };
  // byte offset of the sequence's first bias value in its dword (0 or 2), and
  // the offset of distance D - 31 of a row, from the dword that holds it
  auto rel_mis = [&](const Step& st) {
    return (int)(((uintptr_t)a.rel +
                  (int64_t)max(st.b, 0) * a.HQ * a.rel_extent * 2) & 3);
  };
  auto issue_k = [&](const Step& st, int phys0, int phys1, int stage)
      __attribute__((always_inline)) {
    const uint32_t dst = lds_w + stage * kStageB;
    page_dma(a.kpool, st, phys0, phys1, dst, koff);
    if constexpr (REL) {
      const char* row = reinterpret_cast<const char*>(a.rel) +
                        (int64_t)max(st.b, 0) * a.HQ * a.rel_extent * 2;
      const int mis = rel_mis(st);
      const bool band = st.b >= 0 && rel_dist(st) - 31 < a.rel_extent;
      const i32x4 rs = make_rsrc(
          row - mis,
          band ? (uint32_t)((a.HQ * a.rel_extent * 2 + mis + 3) & ~3) : 0u);
      const int d = 2 * (rel_dist(st) - 31) + mis;
#pragma unroll
      for (int j = 0; j + 1 < kNB; ++j)
        dma32(rs, dst + 2 * kTileB + 256 * j,
              (uint32_t)(((rel_row(4 * j + wtok) + d) & ~3) + 4 * wslot));
      dma32(rs, dst + 2 * kTileB + 256 * (kNB - 1),
            (uint32_t)(((rel_row(lane) + d) & ~3) + 64));
    }
  };
  auto issue_v = [&](const Step& st, int phys0, int phys1, int stage)
      __attribute__((always_inline)) {
    page_dma(a.vpool, st, phys0, phys1, lds_w + stage * kStageB + kTileB, voff);
  };
  // where lane (r, g) finds the dwords of its scores of tile t (tokens
  // 16t + 4g + i, i = 0..3: values 28 - 16t - 4g .. 31 - 16t - 4g of the
  // window, from its dword 14 - 8t - 2g on): two adjacent ones and a third,
  // which for t = g = 0 is the row's 17th (padded heads read the last row)
  const int rr = min(r, rep - 1);
  const uint32_t bias0 = lds_w + 2 * kTileB + 64 * rr + 4 * (14 - 2 * g);
  const uint32_t bias2 =
      g == 0 ? lds_w + 2 * kTileB + 256 * (kNB - 1) + 4 * rr : bias0 + 8;
  // the 16 query rows of a piece (padded heads: zeros)
  auto issue_q = [&](int b) __attribute__((always_inline)) {
    const i32x4 rs = make_rsrc(
        a.q + ((int64_t)b * a.HQ + (int64_t)kvh * rep) * kD,
        (uint32_t)(rep * kRowB));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int x = 4 * i + wtok;
      dma(rs, lds_q + 1024 * i, x * kRowB + 16 * (wslot ^ x));
    }
  };
  // this wave's LDS reads are complete: what they read may be overwritten
  auto lds_done = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));   // lgkmcnt 0
    asm volatile("" ::: "memory");
  };

  // ---- per-piece state ----------------------------------------------------
  f32x4 o_acc[8];
#pragma unroll
  for (int blk = 0; blk < 8; ++blk) o_acc[blk] = f32x4{0, 0, 0, 0};
  float m_run = -INFINITY;
  float l_part = 0.0f;
  bf16x8 qf[4];   // query fragments

  // End of a piece of sequence b: write the result (whole sequence) or a
  // normalised partial that decode_combine_kernel merges.
  auto finish_piece = [&](const Step& st) {
    const int b = st.b;
    float l_tot = l_part;
    l_tot = lane_pair(lane_pair(l_tot, 16, false), 32, false);
    const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    const float lse_nat =
        l_tot > 0.0f ? (m_run + fast_log2(l_tot)) * kLn2 : -INFINITY;
    // Buffer stores with a per-row (wave-uniform) base: the lane offsets
    // stay 32-bit, and padded heads / the LSE of lanes g != 0 / a missing
    // LSE output get an out-of-range offset or an empty resource (dropped),
    // so there is no divergent branch and no 64-bit address to keep live.
    // (The lane's offset is opaque to the compiler, which would otherwise
    // keep every store's offset in a register across the walk.)
    const ArgsPtr ra = kernel_args(true);
    const int HQ = ra->HQ;
    const int bad = 0x7ffff000;
    int eo = head_ok ? hq * kD + 4 * g : bad / 4;   // element of blk 0
    int lo4 = head_ok && g == 0 ? hq * 4 : bad;
    asm volatile("" : "+v"(eo), "+v"(lo4));
    if (st.flags & kWhole) {
      const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
          reinterpret_cast<char*>(ra->out + (int64_t)b * HQ * kD), (short)0,
          HQ * kD * 2, 0x00020000);
      float* const lse = ra->lse;
      const __amdgpu_buffer_rsrc_t rl = __builtin_amdgcn_make_buffer_rsrc(
          reinterpret_cast<char*>(lse ? lse + (int64_t)b * HQ : nullptr),
          (short)0, lse ? HQ * 4 : 0, 0x00020000);
#pragma unroll
      for (int blk = 0; blk < 8; ++blk) {
        const uint32_t w0 =
            pack_bf16x2(f32_to_bf16_bits(o_acc[blk][0] * inv),
                        f32_to_bf16_bits(o_acc[blk][1] * inv));
        const uint32_t w1 =
            pack_bf16x2(f32_to_bf16_bits(o_acc[blk][2] * inv),
                        f32_to_bf16_bits(o_acc[blk][3] * inv));
        __builtin_amdgcn_raw_buffer_store_b64(
            u32x2{w0, w1}, ro, eo * 2 + 32 * blk, 0, 0);
      }
      __builtin_amdgcn_raw_buffer_store_b32(
          __builtin_bit_cast(uint32_t, lse_nat), rl,
          lo4, 0, 0);
    } else {
      // one piece of a longer sequence: slot b + wg is unique because
      // work-groups and sequences are both laid out in order
      const int64_t slot0 = (int64_t)(b + wg) * HQ;
      const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
          reinterpret_cast<char*>(ra->part_o + slot0 * kD), (short)0,
          HQ * kD * 4, 0x00020000);
      const __amdgpu_buffer_rsrc_t rl = __builtin_amdgcn_make_buffer_rsrc(
          reinterpret_cast<char*>(ra->part_lse + slot0), (short)0, HQ * 4,
          0x00020000);
#pragma unroll
      for (int blk = 0; blk < 8; ++blk)
        __builtin_amdgcn_raw_buffer_store_b128(
            __builtin_bit_cast(u32x4, o_acc[blk] * inv), ro,
            eo * 4 + 64 * blk, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b32(
          __builtin_bit_cast(uint32_t, lse_nat), rl,
          lo4, 0, 0);
    }
#pragma unroll
    for (int blk = 0; blk < 8; ++blk) o_acc[blk] = f32x4{0, 0, 0, 0};
    m_run = -INFINITY;
    l_part = 0.0f;
  };

  // ---- 4. software-pipelined walk ------------------------------------------
  // Step s sits in stage s & 1. Its fragments are read into registers first,
  // each tile then makes room for step s + 2 at once, so two steps (32 KB per
  // wave) are in flight while one is computed. With one wave per SIMD nothing
  // hides a step's chain (fragment reads, score MFMAs, softmax, P.V MFMAs), so
  // its length and its instruction count (4 cycles each) set how fast a
  // compute unit streams: page rows do not pass through registers, V^T is
  // read under the softmax, the next step's scalar work goes under the K
  // reads, and steps whose 32 tokens are all visible skip the masks. Measured
  // per step of 32 keys and 4 KV heads, one work-group: 1.60 us with its pages
  // in the L2 and from HBM alike for the form that loaded page rows into
  // registers one step ahead, looked up page ids step by step and zeroed,
  // masked and rescaled on every step (1.86 us with the bias, then 8 two-byte
  // loads per lane); here 0.65 us in the L2 (the chain; 1.12 us with the bias)
  // and 1.06 us from HBM: the loads of one compute unit, 62 GB/s (41 before),
  // now bound it. Among 128 work-groups one streams 46 GB/s (39 before), among
  // 192 the HBM's share, 36. attn_swa at B = 4, 64Q/16KV (one ring per work-group): 37.3 ->
  // 24.6 us; B = 96: 72.6 -> 65.3 us.
  // Queries: those of the next step, if it starts a piece, go out at the top
  // of this one.
  Step cur, nx, nn;
  int p0, p1;   // pages of the step whose loads go out
  next_step(cur, p0, p1);
  issue_q(cur.b);
  issue_k(cur, p0, p1, 0);
  issue_v(cur, p0, p1, 0);
  next_step(nx, p0, p1);
  issue_k(nx, p0, p1, 1);
  issue_v(nx, p0, p1, 1);
  auto read_q = [&]() __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
      qf[kk] = lds_ld128((kr0 ^ (64u * kk)) + 2 * kStageB);
    lds_done();
  };
  wait_vm<2 * kNS>();
  read_q();
  cur.flags &= ~kFirst;
  for (;;) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint32_t so = k * kStageB;
      if (cur.flags & kFirst) {
        wait_vm<kNS>();
        read_q();
      }
      if (nx.flags & kFirst) issue_q(nx.b);
      // ---- K fragments, bias dwords --------------------------------------------
      wait_vm<8 + kNS>();   // after K(s), in flight: V(s) and step s + 1
      asm volatile("" ::: "memory");
      bf16x8 kf[2][4];
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          kf[t][kk] = lds_ld128((kr0 ^ (64u * kk)) + so + 16 * t * kRowB);
      [[maybe_unused]] uint32_t bw[2][3];
      if constexpr (REL) {
        const u32x2 y0 = lds_ld64(bias0 + so), y1 = lds_ld64(bias0 + so - 32);
        bw[0][0] = y0[0];
        bw[0][1] = y0[1];
        bw[0][2] = lds_ld32(bias2 + so);
        bw[1][0] = y1[0];
        bw[1][1] = y1[1];
        bw[1][2] = lds_ld32(bias0 + so - 24);
      }
      next_step(nn, p0, p1);
      lds_done();
      // ---- S^T = K.Q^T for the two 16-token tiles -------------------------
      f32x4 sc[2] = {f32x4{0, 0, 0, 0}, f32x4{0, 0, 0, 0}};
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          sc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][kk], qf[kk],
                                                          sc[t], 0, 0, 0);
      issue_k(nn, p0, p1, k);
      // ---- V^T fragments -------------------------------------------------------
      // A operand (dims 16 blk + r, tokens 4g..4g+3 and 16+4g..16+4g+3) by two
      // transposed reads: source lane s of each 16-lane group names token
      // base + (s >> 2) and dims 16 blk + 4 (s & 3)..+3
      wait_vm<kNS + kNK>();   // after V(s): step s + 1 and K(s + 2)
      asm volatile("" ::: "memory");
      bf16x8 vf[8];
#pragma unroll
      for (int blk = 0; blk < 8; ++blk) {
        const uint32_t va = (vr0 ^ (32u * blk)) + so;
        const bf16x4 lo4 = lds_tr16(va);
        const bf16x4 hi4 = lds_tr16(va + 16 * kRowB);
        vf[blk] = __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7);
      }
      __builtin_amdgcn_sched_barrier(0);   // (or the reads sink to their uses)
      // ---- bias, mask, running max ----------------------------------------
      float x[2][4];
      float mx = -INFINITY;
      [[maybe_unused]] int sh = 0;
      if constexpr (REL)
        sh = (rel_row(rr) + 2 * (rel_dist(cur) - 31) + rel_mis(cur)) & 2;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float bias[4];
        if constexpr (REL) bias_values(a, cur, bw[t], t, sh, g, bias);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          x[t][i] = sc[t][i] * a.scale_log2;
          if constexpr (REL) x[t][i] += bias[i] * kLog2e;
        }
      }
      if (!(cur.flags & kFull)) {
        const int lo = vis_lo(cur.n, a.window);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const bool page_ok = cur.flags & (t == 0 ? kPage0 : kPage1);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int kpos = (cur.pg + t) * kPS + 4 * g + i;
            const bool ok = page_ok && kpos >= lo && kpos < cur.n;
            x[t][i] = ok ? x[t][i] : -INFINITY;
          }
        }
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, x[t][i]);
      mx = lane_pair(lane_pair(mx, 16, true), 32, true);
      // O^T and l move to a new maximum only on the steps that have one (a
      // reference that lags the maximum would skip more of them, but the
      // largest probabilities are then no longer exact in bf16: 10% more error)
      const bool move = mx > m_run;
      if (__builtin_amdgcn_ballot_w64(move)) {
        const float m_new = move ? mx : m_run;
        const float alpha = move ? fast_exp2(m_run - m_new) : 1.0f;
        m_run = m_new;
        l_part *= alpha;
#pragma unroll
        for (int blk = 0; blk < 8; ++blk) o_acc[blk] = o_acc[blk] * alpha;
      }
      const float m_use = m_run == -INFINITY ? 0.0f : m_run;
      // ---- probabilities: fp32 sum, bf16 operand --------------------------
      // B-operand element j = 4t + i  <->  token 16t + 4g + i
      float p[2][4];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) p[t][i] = fast_exp2(x[t][i] - m_use);
      l_part += ((p[0][0] + p[0][1]) + (p[0][2] + p[0][3])) +
                ((p[1][0] + p[1][1]) + (p[1][2] + p[1][3]));
      uint32_t pw[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        pw[j] = pack_bf16x2_rn(p[j >> 1][2 * (j & 1)],
                               p[j >> 1][2 * (j & 1) + 1]);
      const bf16x8 pf =
          __builtin_bit_cast(bf16x8, u32x4{pw[0], pw[1], pw[2], pw[3]});
      // ---- O^T += V^T.P^T ------------------------------------------------------
      lds_done();
#pragma unroll
      for (int blk = 0; blk < 8; ++blk)
        o_acc[blk] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            vf[blk], pf, o_acc[blk], 0, 0, 0);
      issue_v(nn, p0, p1, k);
      if (cur.flags & kLast) finish_piece(cur);
      cur = nx;
      nx = nn;
      if (cur.b < 0) {
        wait_vm<0>();   // no direct load outlives the wave
        return;
      }
    }
  }
}

// Merge the pieces of every sequence that several work-groups shared, in a
// fixed order (deterministic, no atomics): grid (B, ceil(HQ / H)), H heads per
// work-group, S groups of 32 lanes per head (4 dims per lane). Group s takes
// pieces s, s + S, ..., eight pieces' loads in flight at a time; the S results
// then merge through LDS in group order. The load latency, not the bytes, is
// what this kernel waits on: S is chosen so that the pieces of an average
// sequence take one round (one 50,001-token sequence cut into 184 pieces:
// 19.3 us with S = 1, 23 rounds in a chain, 5.8 us with S = 32). A long sequence
// among many short ones still merges in a chain, since the host knows the
// average alone (50,001 tokens beside 31 sequences of 300: 42.6 us a call,
// alone 26.0).
template <int H, int S>
__global__ __launch_bounds__(32 * H * S) void decode_combine_kernel(
    DecodeArgs a) {
  const int b = blockIdx.x;
  const int C = as_const(a.geo)[0];
  const int s0 = as_const(a.geo)[1 + b];
  const int s1 = as_const(a.geo)[2 + b];
  if (s1 <= s0) return;                  // no visible key: written already
  const int wfirst = s0 / C;
  const int np = (s1 - 1) / C - wfirst + 1;
  if (np <= 1) return;                   // one piece: written in place
  const int grp = threadIdx.x >> 5;
  const int sub = grp % S;
  const int h = blockIdx.y * H + grp / S;
  const bool hok = h < a.HQ;
  const int d0 = 4 * (threadIdx.x & 31);
  const int64_t slot0 = (int64_t)(b + wfirst) * a.HQ + (hok ? h : 0);
  float m = -INFINITY, sum = 0.0f;
  f32x4 acc = f32x4{0, 0, 0, 0};
  auto add = [&](float l, float w1, f32x4 o) {   // a piece (LSE l, weight w1)
    const float m_new = fmaxf(m, l);
    const float m_use = m_new == -INFINITY ? 0.0f : m_new;
    const float keep = fast_exp2((m - m_use) * kLog2e);
    const float w = fast_exp2((l - m_use) * kLog2e);
    sum = sum * keep + w * w1;
    acc = acc * keep + o * w;
    m = m_new;
  };
  constexpr int kBatch = 8;
  for (int k = sub; k < np; k += kBatch * S) {
    float l4[kBatch];
    f32x4 o4[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const bool in = k + j * S < np;
      const int64_t slot = slot0 + (int64_t)(in ? k + j * S : 0) * a.HQ;
      l4[j] = in ? a.part_lse[slot] : -INFINITY;
      o4[j] = *reinterpret_cast<const f32x4*>(a.part_o + slot * kD + d0);
    }
#pragma unroll
    for (int j = 0; j < kBatch; ++j)     // (0 x infinity: weight 0 won't do)
      add(l4[j], 1.0f, k + j * S < np ? o4[j] : f32x4{0, 0, 0, 0});
  }
  if constexpr (S > 1) {
    // (m, sum, acc) of every group but the head's first, then merged by it
    __shared__ float part[H * S][6][32];
    const int l = threadIdx.x & 31;
    if (sub > 0) {
      part[grp][0][l] = m;
      part[grp][1][l] = sum;
#pragma unroll
      for (int i = 0; i < 4; ++i) part[grp][2 + i][l] = acc[i];
    }
    __syncthreads();
    if (sub > 0) return;
    const int n = min(np, S);
    for (int j = 1; j < n; ++j) {
      f32x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = part[grp + j][2 + i][l];
      add(part[grp + j][0][l], part[grp + j][1][l], o);
    }
  }
  if (!hok) return;
  const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
  __bf16* o = a.out + ((int64_t)b * a.HQ + h) * kD + d0;
  *reinterpret_cast<u32x2*>(o) =
      u32x2{pack_bf16x2_rn(acc[0] * inv, acc[1] * inv),
            pack_bf16x2_rn(acc[2] * inv, acc[3] * inv)};
  if (a.lse && d0 == 0)
    a.lse[(int64_t)b * a.HQ + h] =
        sum > 0.0f ? (m == -INFINITY ? 0.0f : m) + fast_log2(sum) * kLn2
                   : -INFINITY;
}

// The merge's shape, from the number of pieces of an average sequence (at most
// one more than its share of the grid's G ranges). Heads per work-group times
// the grid's y dimension (65,536 at most) must hold every head, so more of them
// than that take the shape of eight. Groups of lanes per head cost waves, which
// a prefill beside the decode makes wait: with 1 / 4 / 8 of them, us, 32Q/4KV, 4
// sequences of 4K-8K 20.0 / 16.5 / 16.5, 9 up to 4.7K 17.9 / 16.6 / 17.2, 20 of
// 4K-8K 43.4 / 43.5 / 44.9; a mixed step (four layers, two 1285-token chunks, 9
// decode rows) 445.8 / 448.0 / 453.8, against 452.1 before the merge had groups.
void launch_combine(const DecodeArgs& a, int G, hipStream_t st) {
  const int np = a.HQ > 65535 ? 1 : 1 + G / a.B;
  if (np <= 8)
    hipLaunchKernelGGL((decode_combine_kernel<8, 1>),
                       dim3(a.B, (a.HQ + 7) / 8), dim3(256), 0, st, a);
  else if (np <= 64)
    hipLaunchKernelGGL((decode_combine_kernel<2, 4>),
                       dim3(a.B, (a.HQ + 1) / 2), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((decode_combine_kernel<1, 32>), dim3(a.B, a.HQ),
                       dim3(1024), 0, st, a);
}

int waves_per_wg(int HKV) { return HKV % 4 == 0 ? 4 : (HKV % 2 == 0 ? 2 : 1); }

// Three work-groups per four CUs (one wave per SIMD where they run). 160 / 176
// / 192 / 208 / 256 / 512 work-groups, us: 64 sequences of 1K-8K (32Q/4KV) 98.8
// / 96.7 / 96.5 / 96.7 / 99.0 / 110.5, window 4096 at 128 sequences 168.9 /
// 164.6 / 165.1 / 166.2 / 170.7 / 178.5.
int default_wgs(int HKV) {
  const int ny = HKV / waves_per_wg(HKV);
  const int g = 3 * device_cus() / (4 * ny);
  return g > 0 ? g : 1;
}

size_t ws_layout(int B, int HQ, int G, size_t* off_lse, size_t* off_geo) {
  const size_t slots = (size_t)B + G;
  const size_t o_bytes = slots * HQ * kD * sizeof(float);
  const size_t l_bytes = (slots * HQ * sizeof(float) + 255) & ~(size_t)255;
  const size_t g_bytes = (((size_t)B + 2) * sizeof(int) + 255) & ~(size_t)255;
  if (off_lse) *off_lse = o_bytes;
  if (off_geo) *off_geo = o_bytes + l_bytes;
  return o_bytes + l_bytes + g_bytes;
}

template <int REP, int KIND>
void launch_kind(const DecodeArgs& a, dim3 grid, int nw, size_t lds,
                 hipStream_t st) {
  if (a.rel)
    hipLaunchKernelGGL((decode_kernel<REP, true, KIND>), grid,
                       dim3(64 * nw), lds, st, a);
  else
    hipLaunchKernelGGL((decode_kernel<REP, false, KIND>), grid,
                       dim3(64 * nw), lds, st, a);
}

template <int REP>
void launch(const DecodeArgs& a, int G, int nw, size_t lds, hipStream_t st) {
  const dim3 grid(G, a.HKV / nw);
  if (a.bt_kind == 2) launch_kind<REP, 2>(a, grid, nw, lds, st);
  else if (a.bt_kind == 1) launch_kind<REP, 1>(a, grid, nw, lds, st);
  else launch_kind<REP, 0>(a, grid, nw, lds, st);
}

// ---- static scratch of the allocation-free entry point -------------------
// Device memory for tmopt_attn_decode_paged_noalloc's workspace: a fixed
// array in the library's code object, so the call needs no allocation.
// Every GPU the library runs on holds its own copy until the process ends.
constexpr size_t kScratchBytes = size_t(16) << 20;   // 16 MiB per GPU
static __device__ __align__(256) char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_addr[kMaxDevices] = {};

// Device address of the current device's copy of `scratch`. The array's
// name is a host-side stand-in in host code, never a device address: it is
// resolved here, once per device with that device current, and only the
// resolved address is passed to kernels.
int scratch_address(void** addr) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  TMOPT_REQUIRE(e == hipSuccess && dev >= 0 && dev < kMaxDevices,
                TMOPT_ELAUNCH, "decode_noalloc: no current device (%s)",
                hipGetErrorString(e));
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_addr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    TMOPT_REQUIRE(e == hipSuccess && p != nullptr, TMOPT_ELAUNCH,
                  "decode_noalloc: hipGetSymbolAddress failed on device %d: "
                  "%s", dev, hipGetErrorString(e));
    g_scratch_addr[dev] = p;
  }
  *addr = g_scratch_addr[dev];
  return TMOPT_OK;
}

// The block table of attn_global's per-token rows (model.py:938-945: flat
// [b, j] = table[b][j / 16] * 16 + j % 16 for live j, 0 past the length):
// table[b][i] = flat[b][16 i] / 16, and ctx_lens[b] = pos[b] + 1. One thread
// per table entry (entries of pages past a row's length are 0, never read).
__global__ __launch_bounds__(256) void table_from_flat_kernel(
    const int64_t* __restrict__ flat, int64_t Lg, const int64_t* __restrict__ pos,
    int npages, int32_t* __restrict__ table, int64_t table_stride,
    int32_t* __restrict__ ctx_lens) {
  const int b = blockIdx.y;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < npages)
    table[(int64_t)b * table_stride + i] =
        (int32_t)(flat[(int64_t)b * Lg + (int64_t)kPS * i] / kPS);
  if (i == 0) ctx_lens[b] = (int32_t)(pos[b] + 1);
}

}  // namespace
}  // namespace tmopt

using namespace tmopt;

extern "C" int tmopt_attn_decode_default_workgroups(int HKV) {
  if (HKV <= 0) return 0;
  return default_wgs(HKV);
}

extern "C" size_t tmopt_attn_decode_workspace_size(int B, int HQ, int HKV,
                                                   int D, int num_workgroups) {
  (void)D;
  if (B <= 0 || HQ <= 0 || HKV <= 0) return 0;
  const int G = num_workgroups > 0 ? num_workgroups : default_wgs(HKV);
  return ws_layout(B, HQ, G, nullptr, nullptr);
}

// The decode launch behind the entry points: `kind` 0 = int32 block table
// + int32 lengths (block_table, ctx_lens), 1 = per-token flat rows + int64
// positions (rows64, pos64), 2 = ring slots + int64 positions. (Flat rows,
// one page id per 128 bytes, cost nothing over a table since a range's ids
// are fetched at once: looked up step by step they measured 17% slower, and a
// launch that makes a table of them first takes 4.8 us: 60.1 against 58.1 us
// per call at 16 sequences of 1K-8K, 64Q/8KV.)
static int decode_impl(
    int kind, const void* q, const void* k_pool, const void* v_pool,
    const int32_t* block_table, const int64_t* rows64, int64_t bt_stride,
    int table_wrap, const int32_t* ctx_lens, const int64_t* pos64, int B,
    int HQ, int HKV, int D, int page_size, int64_t num_pages, int window,
    float scale, const void* rel, int rel_extent, int min_pages,
    int num_workgroups, int seqs_per_wg, void* out, float* lse,
    void* workspace, size_t workspace_bytes, tmopt_stream_t stream) {
  if (B == 0) return TMOPT_OK;
  TMOPT_REQUIRE(B > 0, TMOPT_EINVAL, "decode: B=%d", B);
  TMOPT_REQUIRE(B <= kMaxB, TMOPT_EUNSUPPORTED, "decode: B=%d above %d", B,
                kMaxB);
  TMOPT_REQUIRE(q && k_pool && v_pool && out &&
                    (kind == 0 ? block_table && ctx_lens : rows64 && pos64),
                TMOPT_EINVAL, "decode: null tensor pointer");
  TMOPT_REQUIRE(D == kD, TMOPT_EUNSUPPORTED, "decode: D=%d (only 128)", D);
  TMOPT_REQUIRE(page_size == kPS, TMOPT_EUNSUPPORTED,
                "decode: page_size=%d (only 16)", page_size);
  TMOPT_REQUIRE(HKV > 0 && HQ > 0 && HQ % HKV == 0, TMOPT_EINVAL,
                "decode: HQ=%d HKV=%d", HQ, HKV);
  // Query heads per scheduled KV head: the whole ratio up to 16 (the MFMA
  // columns), else its largest divisor up to 16, the stored head then
  // scheduled kv_div times (each reading its pages once per group).
  const int ratio = HQ / HKV;
  int rep = ratio;
  while (rep > 16 || ratio % rep != 0) --rep;
  const int kv_div = ratio / rep;
  TMOPT_REQUIRE((int64_t)HKV * kv_div <= 65535, TMOPT_EUNSUPPORTED,
                "decode: HKV=%d x %d query-head groups exceeds 65535", HKV,
                kv_div);
  TMOPT_REQUIRE((int64_t)kPS * HKV * kD * 2 < (1ll << 31), TMOPT_EUNSUPPORTED,
                "decode: page too large");
  TMOPT_REQUIRE(num_pages > 0 && bt_stride > 0 && table_wrap >= 0 &&
                    (table_wrap == 0 || table_wrap <= bt_stride),
                TMOPT_EINVAL,
                "decode: num_pages=%lld bt_stride=%lld table_wrap=%d",
                (long long)num_pages, (long long)bt_stride, table_wrap);
  TMOPT_REQUIRE(window >= 0, TMOPT_EINVAL, "decode: window=%d", window);
  // a ring table holds the last table_wrap * 16 positions: a wider (or no)
  // window would read rows the ring has already overwritten
  TMOPT_REQUIRE(table_wrap == 0 ||
                    (window > 0 && (int64_t)window <= (int64_t)table_wrap * kPS),
                TMOPT_EINVAL, "decode: window=%d outside a ring of %d pages",
                window, table_wrap);
  TMOPT_REQUIRE(min_pages > 0 && num_workgroups >= 0, TMOPT_EINVAL,
                "decode: min_pages=%d num_workgroups=%d", min_pages,
                num_workgroups);
  TMOPT_REQUIRE(rel == nullptr || rel_extent > 0, TMOPT_EINVAL,
                "decode: rel_extent=%d", rel_extent);
  TMOPT_REQUIRE(((uintptr_t)q | (uintptr_t)k_pool | (uintptr_t)v_pool |
                 (uintptr_t)out) % 16 == 0,
                TMOPT_EINVAL, "decode: tensors must be 16-byte aligned");
  const int G = num_workgroups > 0 ? num_workgroups : default_wgs(HKV);
  TMOPT_REQUIRE(G <= 65535, TMOPT_EINVAL, "decode: num_workgroups=%d", G);
  TMOPT_REQUIRE(seqs_per_wg >= 0 &&
                    (seqs_per_wg == 0 || (int64_t)seqs_per_wg * G >= B),
                TMOPT_EINVAL,
                "decode: %d work-groups of %d whole sequences do not cover "
                "B=%d",
                G, seqs_per_wg, B);
  size_t off_lse = 0, off_geo = 0;
  const size_t need = ws_layout(B, HQ, G, &off_lse, &off_geo);
  TMOPT_REQUIRE(workspace && workspace_bytes >= need &&
                    (uintptr_t)workspace % 16 == 0,
                TMOPT_EWORKSPACE,
                "decode: workspace %zu bytes < %zu needed (or unaligned)",
                workspace_bytes, need);

  DecodeArgs a;
  a.q = (const __bf16*)q;
  a.kpool = (const __bf16*)k_pool;
  a.vpool = (const __bf16*)v_pool;
  a.bt = block_table;
  a.bt_stride = bt_stride;
  const int64_t width = kind == 1 ? (bt_stride + kPS - 1) / kPS : bt_stride;
  a.bt_width = width > 0x7fffffff ? 0x7fffffff : (int)width;
  a.table_wrap = table_wrap;
  a.ctx_lens = ctx_lens;
  a.bt_kind = kind;
  a.rows64 = rows64;
  a.pos64 = pos64;
  a.B = B;
  a.HQ = HQ;
  a.HKV = HKV * kv_div;
  a.rep = rep;
  a.kv_div = kv_div;
  a.HKV_stored = HKV;
  a.num_pages = num_pages > 0x7fffffff ? 0x7fffffff : (int)num_pages;
  a.window = window;
  a.scale_log2 = scale * kLog2e;
  a.rel = (const __bf16*)rel;
  a.rel_extent = rel ? rel_extent : 0;
  a.min_pages = min_pages;
  a.seqs_per_wg = seqs_per_wg;
  a.out = (__bf16*)out;
  a.lse = lse;
  a.part_o = (float*)workspace;
  a.part_lse = (float*)((char*)workspace + off_lse);
  a.geo = (int*)((char*)workspace + off_geo);

  const int nw = waves_per_wg(a.HKV);
  const size_t tab = ((2 * (size_t)B + 1 + 4) * sizeof(int) + 15) & ~(size_t)15;
  const size_t tiles = (size_t)nw * wave_lds(rel != nullptr);
  a.ids_off = (int)(tab > tiles ? tab : tiles);
  const size_t lds = a.ids_off + (ids_kept(rel != nullptr) + 2) * sizeof(int);
  hipStream_t st = (hipStream_t)stream;
  switch (kv_div == 1 ? rep : 0) {
    case 1: launch<1>(a, G, nw, lds, st); break;
    case 2: launch<2>(a, G, nw, lds, st); break;
    case 4: launch<4>(a, G, nw, lds, st); break;
    case 8: launch<8>(a, G, nw, lds, st); break;
    case 16: launch<16>(a, G, nw, lds, st); break;
    default: launch<0>(a, G, nw, lds, st); break;
  }
  int rc = check_launch("decode");
  if (rc || seqs_per_wg > 0) return rc;   // whole sequences: nothing to merge
  launch_combine(a, G, st);
  return check_launch("decode_combine");
}

extern "C" int tmopt_attn_decode_paged(
    const void* q, const void* k_pool, const void* v_pool,
    const int32_t* block_table, int64_t bt_stride, int table_wrap,
    const int32_t* ctx_lens, int B, int HQ, int HKV, int D, int page_size,
    int64_t num_pages, int window, float scale, const void* rel,
    int rel_extent, int min_pages, int num_workgroups, void* out, float* lse,
    void* workspace, size_t workspace_bytes, tmopt_stream_t stream) {
  clear_error();
  return decode_impl(0, q, k_pool, v_pool, block_table, nullptr, bt_stride,
                     table_wrap, ctx_lens, nullptr, B, HQ, HKV, D, page_size,
                     num_pages, window, scale, rel, rel_extent, min_pages,
                     num_workgroups, 0, out, lse, workspace, workspace_bytes,
                     stream);
}

extern "C" int tmopt_attn_decode_ring(
    const void* q, const void* k_pool, const void* v_pool,
    const int64_t* slots, int ring_pages, const int64_t* pos, int B, int HQ,
    int HKV, int D, int64_t num_pages, int window, float scale,
    const void* rel, int rel_extent, int min_pages, int num_workgroups,
    int seqs_per_workgroup, void* out, float* lse, void* workspace,
    size_t workspace_bytes, tmopt_stream_t stream) {
  clear_error();
  TMOPT_REQUIRE(ring_pages > 0, TMOPT_EINVAL, "decode_ring: ring_pages=%d",
                ring_pages);
  return decode_impl(2, q, k_pool, v_pool, nullptr, slots, ring_pages,
                     ring_pages, nullptr, pos, B, HQ, HKV, D, kPS, num_pages,
                     window, scale, rel, rel_extent, min_pages,
                     num_workgroups, seqs_per_workgroup, out, lse, workspace,
                     workspace_bytes, stream);
}

extern "C" int tmopt_attn_decode_flat(
    const void* q, const void* k_pool, const void* v_pool,
    const int64_t* flat, int64_t Lg, const int64_t* pos, int B, int HQ,
    int HKV, int D, int page_size, int64_t num_pages, float scale,
    const void* rel, int rel_extent, int min_pages, int num_workgroups,
    void* out, float* lse, void* workspace, size_t workspace_bytes,
    tmopt_stream_t stream) {
  clear_error();
  return decode_impl(1, q, k_pool, v_pool, nullptr, flat, Lg, 0, nullptr, pos,
                     B, HQ, HKV, D, page_size, num_pages, 0, scale, rel,
                     rel_extent, min_pages, num_workgroups, 0, out, lse,
                     workspace, workspace_bytes, stream);
}

extern "C" int tmopt_attn_decode_paged_noalloc(
    const void* q, const void* k_pool, const void* v_pool,
    const int32_t* block_table, int64_t bt_stride, int table_wrap,
    const int32_t* ctx_lens, int B, int HQ, int HKV, int D, int page_size,
    int64_t num_pages, int window, float scale, const void* rel,
    int rel_extent, int min_pages, int num_workgroups, void* out, float* lse,
    tmopt_stream_t stream) {
  clear_error();
  if (B == 0) return TMOPT_OK;
  // the workspace this launch shape needs (0 for arguments the full entry
  // point rejects: it reports them)
  const size_t need =
      tmopt_attn_decode_workspace_size(B, HQ, HKV, D, num_workgroups);
  TMOPT_REQUIRE(need <= kScratchBytes, TMOPT_EWORKSPACE,
                "decode_noalloc: the launch needs %zu bytes of scratch, above "
                "the %zu-byte static buffer (use tmopt_attn_decode_paged with "
                "a workspace)",
                need, kScratchBytes);
  void* ws = nullptr;
  const int rc = scratch_address(&ws);
  if (rc != TMOPT_OK) return rc;
  return tmopt_attn_decode_paged(q, k_pool, v_pool, block_table, bt_stride,
                                 table_wrap, ctx_lens, B, HQ, HKV, D,
                                 page_size, num_pages, window, scale, rel,
                                 rel_extent, min_pages, num_workgroups, out,
                                 lse, ws, kScratchBytes, stream);
}

extern "C" int tmopt_decode_table_from_flat(const int64_t* flat, int64_t Lg,
                                            const int64_t* pos, int B,
                                            int32_t* block_table,
                                            int64_t bt_stride,
                                            int32_t* ctx_lens,
                                            tmopt_stream_t stream) {
  clear_error();
  if (B == 0) return TMOPT_OK;
  TMOPT_REQUIRE(B > 0 && B <= 65535 && Lg > 0, TMOPT_EINVAL,
                "table_from_flat: B=%d Lg=%lld", B, (long long)Lg);
  TMOPT_REQUIRE(flat && pos && block_table && ctx_lens, TMOPT_EINVAL,
                "table_from_flat: null pointer");
  const int64_t npages = (Lg + kPS - 1) / kPS;
  TMOPT_REQUIRE(npages <= 0x7fffffff && bt_stride >= npages, TMOPT_EINVAL,
                "table_from_flat: bt_stride=%lld < %lld pages",
                (long long)bt_stride, (long long)npages);
  hipLaunchKernelGGL(table_from_flat_kernel,
                     dim3((unsigned)((npages + 255) / 256), B), dim3(256), 0,
                     (hipStream_t)stream, flat, Lg, pos, (int)npages,
                     block_table, bt_stride, ctx_lens);
  return check_launch("table_from_flat");
}
