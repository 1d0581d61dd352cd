// Prefill launches whose keys are split over work-groups (see key_pieces in
// prefill_kernel.h): the split kernel and the merge of its pieces.
#define TMOPT_PREFILL_PIECES
#include "prefill_kernel.h"

namespace tmopt {
namespace {

// prefill_kernel with split keys (items that stay whole included). The number
// of pieces goes to the merge through memory: it comes of fp32 arithmetic next
// to rounding edges, which another kernel need not contract the same way (fma
// or not, 64 + 256 queries after 7,936 and 7,680 keys give 12 or 13 pieces),
// and the merge must read exactly the slots that were written. Every work-group
// of this kernel runs the same instructions on the same lengths.
template <int REP, bool REL, int SRC>
__global__ __launch_bounds__(512) void prefill_split_kernel(PrefillArgs a) {
  constexpr int BQ = 256 / REP;
  const int lane = threadIdx.x & 63;
  const int level = (int)blockIdx.x / a.n_base;
  const Work wk = schedule(a, BQ, lane, (int)blockIdx.x - level * a.n_base);
  const bool first = level == 0 && threadIdx.x == 0;
  if (wk.seq < 0) {
    if (first) a.part_n[blockIdx.x] = 0;
    return;
  }
  const Tiles tl = item_tiles(a, BQ, wk.prior, wk.len, wk.qb);
  const Pieces pc = key_pieces(a, BQ, lane, wk, tl);
  if (level >= pc.nall) return;
  if (first) a.part_n[blockIdx.x] = pc.nall;
  const int t0 = pc.begin(level, tl.n), t1 = pc.begin(level + 1, tl.n);
  const int slot = pc.nall > 1 ? (int)blockIdx.x : -1;
  if constexpr (REL) {
    if (level < pc.np && pc.nall > 1) {
      prefill_item<REP, false, SRC>(a, wk, tl.k_lo, t0, t1, slot);
      return;
    }
  }
  prefill_item<REP, REL, SRC>(a, wk, tl.k_lo, t0, t1, slot);
}

// A 32-row block of outputs on its way through LDS, query-major: 256-byte
// rows, 16-byte chunks swizzled by row & 15, so neither the 8-byte writes nor
// the 16-byte reads conflict. Chunk c (dims 8c..8c+7) of row lane & 31, half
// lane >> 5, from four fp32 values.
__device__ __forceinline__ void rows_to_lds(uint32_t ob, int lane, int c,
                                            float x0, float x1, float x2,
                                            float x3) {
  const int r = lane & 31;
  lds_st64(ob + r * kRowB + 16 * (c ^ (r & 15)) + 8 * (lane >> 5),
           u32x2{pack_bf16x2(f32_to_bf16_bits(x0), f32_to_bf16_bits(x1)),
                 pack_bf16x2(f32_to_bf16_bits(x2), f32_to_bf16_bits(x3))});
}
// Rows r0, r0 + STEP, ... (N of them) from there to the output, 16-byte chunk
// c16 of each (a store instruction covers 4 complete rows: 16 lanes x 16 bytes
// each).
template <int N, int STEP>
__device__ __forceinline__ void rows_from_lds(const PrefillArgs& a, uint32_t ob,
                                              int r0, int c16, int qrow0,
                                              int len, int t0, int head) {
  const bool al16 = ((a.o_st | a.o_sh) & 7) == 0 &&
                    ((uintptr_t)a.out & 15) == 0;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int r = STEP * i + r0;
    const u32x4 x = __builtin_bit_cast(
        u32x4, lds_ld128(ob + r * kRowB + 16 * (c16 ^ (r & 15))));
    if (qrow0 + r < len) {
      __bf16* const dst = a.out + (int64_t)(t0 + qrow0 + r) * a.o_st +
                          (int64_t)head * a.o_sh + 8 * c16;
      if (al16) {
        *reinterpret_cast<u32x4*>(dst) = x;
      } else {
        reinterpret_cast<u32x2*>(dst)[0] = u32x2{x[0], x[1]};
        reinterpret_cast<u32x2*>(dst)[1] = u32x2{x[2], x[3]};
      }
    }
  }
}

// Combine the pieces of the items that were split: grid (n_base, 8), one
// work-group per 32-row block of an item, wave db the dims 32 db .. +31; eight
// pieces' loads in flight at a time, combined in piece order.
template <int REP>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillArgs a) {
  constexpr int BQ = 256 / REP, QSUB = BQ / 32;
  __shared__ __align__(256) char rows[32 * kRowB];
  const int lane = threadIdx.x & 63;
  const int db = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31;
  const int np = min(as_const(a.part_n)[blockIdx.x], a.nsplit);
  if (np <= 1) return;                        // no item, or written in place
  const Work wk = schedule(a, BQ, lane, blockIdx.x);
  const int w = blockIdx.y;                   // row block = wave of the item
  const int qrow0 = wk.qb * BQ + 32 * (w % QSUB);
  const int head = wk.kvh * REP + w / QSUB;
  float m = -INFINITY, sum = 0.0f;
  f32x4 acc[4] = {};
  constexpr int kBatch = 8;
  for (int s0 = 0; s0 < np; s0 += kBatch) {
    float l[kBatch];
    f32x4 o[kBatch][4];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const int s = min(s0 + j, np - 1);
      const int64_t pw = ((int64_t)s * a.n_base + blockIdx.x) * 8 + w;
      l[j] = s0 + j < np ? a.part_lse[pw * 32 + l32] : -INFINITY;
      const float* po = a.part_o + ((pw * 16 + 4 * db) * 64 + lane) * 4;
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4)
        o[j][g4] = *reinterpret_cast<const f32x4*>(po + g4 * 256);
    }
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      if (s0 + j >= np) break;       // (0 x infinity: weight 0 won't do)
      const float m_new = fmaxf(m, l[j]);
      const float m_use = m_new == -INFINITY ? 0.0f : m_new;
      const float keep = fast_exp2((m - m_use) * kLog2e);
      const float wt = fast_exp2((l[j] - m_use) * kLog2e);
      sum = sum * keep + wt;
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) acc[g4] = acc[g4] * keep + o[j][g4] * wt;
      m = m_new;
    }
  }
  // (a rejected launch's pieces are NaN, and so is their sum)
  const bool rejected = a.reject != nullptr && as_const(a.reject)[0] != 0;
  const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
  const int qi = qrow0 + l32;
  if (a.lse && db == 0 && lane < 32 && qi < wk.len)
    a.lse[(int64_t)head * wk.total + wk.t0 + qi] =
        rejected ? __builtin_nanf("")
        : sum > 0.0f ? m + fast_log2(sum) * kLn2 : -INFINITY;
  const uint32_t ob =
      (uint32_t)(uintptr_t)((__attribute__((address_space(3))) char*)rows);
#pragma unroll
  for (int g4 = 0; g4 < 4; ++g4)
    rows_to_lds(ob, lane, 4 * db + g4, acc[g4][0] * inv, acc[g4][1] * inv,
                acc[g4][2] * inv, acc[g4][3] * inv);
  __syncthreads();
  rows_from_lds<2, 16>(a, ob, 4 * db + (lane >> 4), lane & 15, qrow0, wk.len,
                       wk.t0, head);
}

template <int REP, bool REL>
void launch_src(const PrefillArgs& a, int src, dim3 grid, size_t lds,
                hipStream_t st) {
  if (src == kPacked)
    hipLaunchKernelGGL((prefill_split_kernel<REP, REL, kPacked>), grid, dim3(512), lds, st,
                       a);
  else if (src == kPaged)
    hipLaunchKernelGGL((prefill_split_kernel<REP, REL, kPaged>), grid, dim3(512), lds, st,
                       a);
  else if (src == kMixed)
    hipLaunchKernelGGL((prefill_split_kernel<REP, REL, kMixed>), grid, dim3(512), lds, st,
                       a);
  else
    hipLaunchKernelGGL((prefill_split_kernel<REP, REL, kPackedCM>), grid, dim3(512), lds, st,
                       a);
}

template <int REP>
void launch(const PrefillArgs& a, int src, size_t lds, hipStream_t st) {
  const dim3 grid((unsigned)(a.n_base * a.nsplit));
  if (a.rel)
    launch_src<REP, true>(a, src, grid, lds, st);
  else
    launch_src<REP, false>(a, src, grid, lds, st);
  hipLaunchKernelGGL((prefill_merge_kernel<REP>), dim3(a.n_base, 8), dim3(256),
                     0, st, a);
}

}  // namespace

void launch_prefill_split(const PrefillArgs& a, int rep, int src, size_t lds,
                          hipStream_t st) {
  if (rep == 8)
    launch<8>(a, src, lds, st);
  else if (rep == 4)
    launch<4>(a, src, lds, st);
  else if (rep == 2)
    launch<2>(a, src, lds, st);
  else
    launch<1>(a, src, lds, st);
}

}  // namespace tmopt
