// Single-token decode attention for gfx950: paged KV pool and contiguous KV cache.
//
// Replaces axlearn/common/flash_attention/gpu_paged_attention.py:38-152 (`_paged_attention_kernel`)
// with its launcher and XLA combine (:164-296), and axlearn/common/flash_attention/
// gpu_decoding.py:71-283 (`_attn_forward_kernel`, `_decode_attn_unbatched`).
//
// The operation is bound by HBM: every K and V byte of the live context is read exactly once.
//   * split-K over the context, by one of two rules (DecArgs::even):
//     calls whose context capacity gives a workgroup at most 256 tiles of 16 tokens: the live tiles of all
//     (sequence, kv head) pairs form one list and every workgroup (two of 4 wavefronts per CU) takes an
//     equal, contiguous share of it.  Nothing is drawn, so there is no counter, no kernel that zeroes it and
//     no half-empty last round;
//     other calls: blocks of `chunk_pages` tiles of one pair.  The split kernel is persistent: every workgroup derives the list of live blocks from the lengths and
//     draws runs of consecutive blocks from a global counter, long runs first and single blocks at the
//     end, so that blocks past a sequence's length cost nothing and CUs that are served faster by the
//     memory system take more of the work (over the milliseconds of such a call that is worth 4 %);
//   * K and V pages stream from HBM straight into a private LDS ring per wavefront
//     (global_load_lds), so the bytes in flight cost no registers; a stage is refilled as soon as
//     its fragments sit in registers.  The pages of a run are handed to the 4 wavefronts through a
//     counter in LDS, so they finish together;
//   * per page a wavefront computes S^T = K Q^T (v_mfma_f32_16x16x32_bf16) for all query heads of
//     the kv head (padded to 16 columns) and O^T += V^T P^T (v_mfma_f32_16x16x16_bf16, V^T through
//     transposing LDS reads); the accumulator layout of the first product is the operand layout
//     of the second, so probabilities never leave registers;
//   * each run inside one (sequence, kv head) yields one partial record (o, m, l) in an fp32
//     workspace (the reference stores partial o in the query dtype, gpu_paged_attention.py:272)
//     and a second small kernel merges the records of a (sequence, kv head) in context order; short
//     calls do without it, the last workgroup of a pair merges them (finish_pairs).
// Work is handed out by timing, so the grouping of the fp32 partial sums - not the set of keys -
// can differ between two calls; the AXL_DECODE_DETERMINISTIC flag of the call (or
// AXL_DECODE_DETERMINISTIC=1 in the environment, read once, as the default for every call) selects
// a fixed decomposition (equal shares, or one block per record; pages dealt round-robin) whose result is
// reproducible bit for bit.
// Keys at index >= length are masked (gpu_paged_attention.py:100, gpu_decoding.py:109); the query
// position is length-1, so a sliding window w also masks keys with (length-1) - j > w.  A page
// index outside the pool reads as zeros and a negative one counts from the end of the pool, as the
// reference's gather does (kv_cache/paged_kv_cache.py:32).
#include <algorithm>
#include <atomic>
#include <mutex>
#include <random>

#include "common.h"

namespace axl {

struct DecArgs {
  const __bf16* q;        // [B, Hq, D]
  const __bf16* k;        // paged: [Hkv, P, page_size, D]; contiguous: [B, S, Hkv, D] (strided)
  const __bf16* v;
  const int32_t* page_tables;  // [B, pt_stride] (paged only)
  const char* lengths;         // [B] at `len_stride` bytes: lengths, or positions of the query (len_add = 1)
  int64_t len_stride;
  int len_i64, len_add;        // int64 instead of int32; what to add to get the length
  __bf16* out;                 // [B, Hq, D]
  float* ws_o;                 // [records, GP, D]; at most B * Hkv * NCH records
  float* ws_m;                 // [records, GP]
  float* ws_l;                 // [records, GP]
  int32_t* ws_tab;             // [B, Hkv, NCH]: record that starts at this live chunk, or -1; every live
                               // chunk's entry is written by the workgroup that streams the chunk
  Strides3 ks, vs;             // contiguous only
  int B, Hq, Hkv, G;
  int ngrp, Hv;                // groups of 16 query heads per kv head; Hv = Hkv * ngrp "virtual" kv heads:
                               // a kv head with more than 16 query heads is streamed once per group
  int num_pages, pps;          // pool pages; 16-token tiles per sequence (ceil(S/16) if contiguous)
  int page_shift, pt_stride;   // a pool page holds 16 << page_shift tokens; entries per page-table row
  int d_real;                  // head_dim of the tensors (a multiple of 8, <= the compiled width D)
  int kv_len;                  // key positions a sequence can address (cache rows / table capacity)
  const char* bias;            // [B|1, Hq|1, kv_len] additive logit bias, bf16 or fp32, or nullptr
  int64_t bias_sb, bias_sh;    // BYTES per batch / query head (0 broadcasts)
  int bias_f32;
  float inv_scale;             // 1 / scale: the bias joins the raw (unscaled) logits
  int chunk_pages, nch;
  int window;
  float scale;
  int* ticket;                 // [0] blocks handed out: zero when the split kernel starts (zeroed by
                               // decode_plan_kernel, or left at zero by the previous call's combine kernel)
  int deterministic;           // fixed work decomposition: results reproducible bit for bit
  int even;                    // equal shares of the live tiles instead of blocks (see the head of this file)
  int n_wg;                    // ... over this many workgroups
  int min_share;               // ... of at least this many tiles
  uint64_t call_id;            // ... of the split kernel that merges its records itself (finish_pairs; else 0)
  uint64_t* ws_flag;           // ... [records]: call_id once the record is complete
};

// Tokens per tile: the unit the kernels stream and compute on.  A pool page of 16 << page_shift
// tokens is that many consecutive tiles (the reference gathers gpu_block_size / page_size pages per
// compute block, gpu_paged_attention.py:91-94; here the compute block is a tile and a page spans
// several).
constexpr int kPage = 16;

// One element of the bias row of (sequence b, query head h) at key position t, in raw-logit units.
__device__ __forceinline__ float decode_bias_at(const DecArgs& a, int b, int h, int t) {
  const char* row = a.bias + b * a.bias_sb + h * a.bias_sh;
  const float x = a.bias_f32 ? ((const float*)row)[t] : (float)((const __bf16*)row)[t];
  return x * a.inv_scale;
}

// XOR swizzle of the 16-byte chunks of a K row inside an LDS tile, so that 16 lanes reading the
// same logical chunk of 16 different rows hit 16 different bank groups.
template <int D>
__device__ __forceinline__ int k_swizzle(int row) {
  if (D == 128) return ((row & 3) << 2) | ((row >> 2) & 3);
  return (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
}

// The same for V rows: the transposing read of a 16-column block touches 32 bytes of 16 rows;
// rows 0..7 (and 8..15) are spread over all banks.
template <int D>
__device__ __forceinline__ int v_swizzle(int row) {
  if (D == 128) return 2 * (row & 7);
  return 2 * ((row >> 1) & 3);
}

// Records per (sequence, kv head) pair: bounds the combine kernel's LDS tables.
constexpr int kMaxChunks = 256;

// Sequences per launch: bounds the work-item tables each workgroup keeps in LDS.
constexpr int kMaxBatch = 512;

// Length of sequence b.  Lengths outside [0, capacity] are clamped: a sequence cannot hold more keys than
// its page table (or its cache rows) can address, and a non-positive length is an empty context.
__device__ __forceinline__ int length_of(const DecArgs& a, int b) {
  const char* p = a.lengths + b * a.len_stride;
  const int64_t len = (a.len_i64 ? *(const int64_t*)p : (int64_t)*(const int32_t*)p) + a.len_add;
  return (int)max((int64_t)0, min(len, (int64_t)a.kv_len));
}

// Live tiles [t0, t1) of a sequence of length `len`.
__device__ __forceinline__ void live_tiles(const DecArgs& a, int len, int& t0, int& t1) {
  t0 = a.window >= 0 ? max(0, len - 1 - a.window) / kPage : 0;
  t1 = max(t0, min((len + kPage - 1) / kPage, a.pps));
}
// Live units of work [u0, u1) of a sequence, a unit being `unit` tiles (numbered from the first of the cache).
__device__ __forceinline__ void live_units(const DecArgs& a, int len, int unit, int& u0, int& u1) {
  int t0, t1;
  live_tiles(a, len, t0, t1);
  u0 = t0 / unit;
  u1 = max(u0, (t1 + unit - 1) / unit);
}
// Equal shares (DecArgs::even): the unit and the units per workgroup, from the call's live blocks and tiles.
// No more blocks than workgroups: a block each, the decomposition of AXL_DECODE_DETERMINISTIC.  Otherwise
// tiles, in whole rounds of the 4 wavefronts.
struct EvenPlan {
  int unit, share;
};
__device__ __forceinline__ EvenPlan even_plan(const DecArgs& a, int blocks, int tiles) {
  if (blocks <= a.n_wg) return EvenPlan{a.chunk_pages, 1};
  return EvenPlan{1, max(a.min_share, ((tiles + a.n_wg - 1) / a.n_wg + 3) & ~3)};
}

template <int D, int GP, int NST>
struct DecTile {
  static constexpr int ROW_BYTES = D * 2;
  static constexpr int TILE_BYTES = kPage * ROW_BYTES;   // K (or V) of one page
  static constexpr int STAGE_BYTES = 2 * TILE_BYTES;     // K then V
  static constexpr int RING_BYTES = 4 * NST * STAGE_BYTES;
  static constexpr int RED_BYTES = 2 * 4 * 16 * 4;
  static constexpr int RED_BASE = RING_BYTES;
  static constexpr int PFX_BASE = RED_BASE + RED_BYTES;   // int[kMaxBatch + 4]: work-item prefix
  static constexpr int LEN_BASE = PFX_BASE + (kMaxBatch + 4) * 4;  // int[kMaxBatch]: sequence lengths
  static constexpr int NEXT_BASE = LEN_BASE + kMaxBatch * 4;       // int[4]: next run, record index
  static constexpr int LDS_BYTES = NEXT_BASE + 16;
  static constexpr int RED_O_PITCH = D + 4;              // floats per (wave, head) row of the epilogue
  static_assert(4 * GP * RED_O_PITCH * 4 <= RING_BYTES, "epilogue staging must fit in the ring");
  static_assert(256 * 24 <= RING_BYTES, "a merge's exchange must fit in the ring");
};

// Partial results between workgroups: written and read past the XCD's own L2 where another workgroup of the same
// launch reads them (DEVICE; the L2s are not coherent inside a launch), else as everything is.
template <bool DEVICE>
__device__ __forceinline__ float read_record(const float* p) {
  if constexpr (DEVICE) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else return *p;
}
template <bool DEVICE>
__device__ __forceinline__ float4 read_record4(const float* p) {
  if constexpr (DEVICE) {
    union { unsigned long long u[2]; float4 f; } x;
    x.u[0] = __hip_atomic_load((const unsigned long long*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    x.u[1] = __hip_atomic_load((const unsigned long long*)p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return x.f;
  } else {
    return *(const float4*)p;
  }
}
__device__ __forceinline__ void write_record(float* p, float x, bool device) {
  if (device) __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = x;
}

// The threads' partial sums in a merge, with their maxima and row sums.
template <int NT>
struct MergeLds {
  float4 part[NT];
  float m[NT], l[NT];
};

constexpr int kMergeBatch = 8;   // records in flight per thread

// Merges `nl` records of pair (b, hv), the i-th of them record_of(i), in that order, by NT threads: the result.
template <typename E, int D, int GP, int NT, bool DEVICE, typename F>
__device__ __forceinline__ void merge_records(const DecArgs& a, int b, int hv, int nl, F record_of, MergeLds<NT>& lds, int tid) {
  // Output: G*D floats = n4 groups of four.  With fewer groups than threads the records are dealt
  // to `ways` slices of threads (record ci to slice ci % ways), kBatch of them in flight per thread,
  // and the slices' partial results are merged in slice order.
  constexpr int kBatch = kMergeBatch;
  const float c = a.scale * kLog2e;
  const int hk = hv / a.ngrp, grp = hv - hk * a.ngrp;
  const int gcount = min(16, a.G - 16 * grp);   // query heads of this group
  const int hbase = hk * a.G + 16 * grp;
  const int n4 = gcount * D / 4;
  const int per = min(n4, NT);
  const int ways = NT / per;
  for (int base = 0; base < n4; base += per) {
    const int way = tid / per, col = base + tid % per;
    const bool live = way < ways && col < n4;
    const int gq = live ? (4 * col) / D : 0;
    float4 acc = {0.f, 0.f, 0.f, 0.f};
    float m = kNegInf, l = 0.f;
    if (live) {
      for (int c0 = way; c0 < nl; c0 += kBatch * ways) {
        float4 o[kBatch];
        float mb[kBatch], lb[kBatch];
#pragma unroll
        for (int i = 0; i < kBatch; i++) {
          // past the end: the batch's first record again, with a weight of zero
          const int ci = c0 + i * ways;
          const int64_t r = record_of(ci < nl ? ci : c0);
          o[i] = read_record4<DEVICE>(a.ws_o + r * (GP * D) + 4 * col);
          mb[i] = read_record<DEVICE>(a.ws_m + r * GP + gq);
          lb[i] = read_record<DEVICE>(a.ws_l + r * GP + gq);
        }
        float mn = m;
#pragma unroll
        for (int i = 0; i < kBatch; i++) mn = fmaxf(mn, mb[i]);
        const float f0 = fast_exp2((m - mn) * c);
        acc.x *= f0; acc.y *= f0; acc.z *= f0; acc.w *= f0;
        l *= f0;
        m = mn;
#pragma unroll
        for (int i = 0; i < kBatch; i++) {
          if (c0 + i * ways < nl) {
            const float f = fast_exp2((mb[i] - mn) * c);
            acc.x += o[i].x * f; acc.y += o[i].y * f; acc.z += o[i].z * f; acc.w += o[i].w * f;
            l += lb[i] * f;
          }
        }
      }
    }
    if (base > 0) __syncthreads();  // the exchange of the previous pass has been read
    lds.part[tid] = acc;
    lds.m[tid] = m;
    lds.l[tid] = l;
    __syncthreads();
    if (live && way == 0) {
      float mw = m;
      for (int w = 1; w < ways; w++) mw = fmaxf(mw, lds.m[w * per + tid]);
      const float f0 = fast_exp2((m - mw) * c);
      acc.x *= f0; acc.y *= f0; acc.z *= f0; acc.w *= f0;
      l *= f0;
      for (int w = 1; w < ways; w++) {
        const float4 p = lds.part[w * per + tid];
        const float f = fast_exp2((lds.m[w * per + tid] - mw) * c);
        acc.x += p.x * f; acc.y += p.y * f; acc.z += p.z * f; acc.w += p.w * f;
        l += lds.l[w * per + tid] * f;
      }
      // An empty context (length 0, or no key inside the window) has no record: the output is zeros,
      // as with the reference's o / (l + eps) (gpu_decoding.py:282, gpu_paged_attention.py:291-293).
      const float inv = l > 0.f ? 1.f / l : 0.f;
      const int dcol = 4 * col - gq * D;   // column inside the head: the ones past head_dim are padding
      const int64_t at = ((int64_t)b * a.Hq + hbase + gq) * a.d_real + dcol;
      if (dcol < a.d_real) {
        if constexpr (std::is_same_v<E, ElemF32>) {
          *(float4*)((float*)a.out + at) = float4{acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv};
        } else {
          union { bf16x2 p[2]; uint2 u; } pk;
          pk.p[0] = E::pack(acc.x * inv, acc.y * inv);
          pk.p[1] = E::pack(acc.z * inv, acc.w * inv);
          *(uint2*)(a.out + at) = pk.u;
        }
      }
    }
  }
}

// Equal shares, merged by the split kernel itself (MERGE): the workgroup calls this with the (at most two) pairs of which
// it left a record, after its threads' record stores.  It marks its records as complete and merges a pair whose records all
// are: of the workgroups of a pair the last one to mark finds all the others' marks, for a mark is at the memory that
// all XCDs share before the marks are read.  (Two that mark at the same time may both find all: they store the same bits.)
// A mark is the number of the call, which no workspace can hold from before, so nothing has to be zeroed; a captured launch, which
// is replayed with its number, takes the merge kernel (launch_common).  Saves that kernel and its launch: decode of one sequence of 1024
// tokens, 8 heads, 12.6 -> 11.0 us, 4 sequences in 128-token pages under a window of 1024, 8 heads of 64, with their page insert
// 19.6 -> 18.0.
template <typename E, int D, int GP>
__device__ __forceinline__ void finish_pairs(const DecArgs& a, const int* pfx, const int* lens, int unit, int share,
                                             const int (&pairs)[2], int n_pairs, MergeLds<256>& lds, int tid) {
  wait_vmem_le<0>();   // this thread's records are complete
  __syncthreads();
  if (tid < n_pairs)
    __hip_atomic_store(&a.ws_flag[blockIdx.x + pairs[tid]], a.call_id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  wait_vmem_le<0>();
  __syncthreads();
  for (int i = 0; i < n_pairs; i++) {
    const int pair = i == 0 ? pairs[0] : pairs[1], b = pair / a.Hv, hv = pair - b * a.Hv;
    int u0, u1;
    live_units(a, lens[b], unit, u0, u1);
    const int first = pfx[b] * a.Hv + hv * (u1 - u0);
    const int w0 = first / share, n = (first + u1 - u0 - 1) / share - w0 + 1;   // its workgroups, at most kMaxChunks
    bool done = true;
    if (tid < n) done = __hip_atomic_load(&a.ws_flag[w0 + tid + pair], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.call_id;
    if (!__syncthreads_and(done)) continue;
    merge_records<E, D, GP, 256, true>(a, b, hv, n, [&](int j) { return w0 + j + pair; }, lds, tid);
    __syncthreads();
  }
}

// Split-K kernel.  Per page a wavefront computes
//   S^T = K Q^T     (v_mfma_f32_16x16x32_bf16, A = K rows from LDS, B = Q^T held in registers),
//   O^T += V^T P^T  (v_mfma_f32_16x16x16_bf16, A = V^T through transposing LDS reads, B = P^T),
// in the "transposed" form where lane l owns query head l%16 and the tokens 4*(l/16)..+3 of the
// page: the accumulator layout of S^T is exactly the B-operand layout of the second product, so
// probabilities never leave registers, and every softmax statistic is per lane.
//
// MERGE: equal shares, whose records the kernel merges itself.  A form of its own: as a run-time branch it cost the long calls, which
// draw their blocks, 1.3 us (5 sequences of up to 13568 tokens, 32 heads, 128.9 -> 130.5 us).
template <typename E, int D, int GP, bool PAGED, int NST, bool BIAS, bool MERGE>
__global__ __launch_bounds__(256) void decode_split_kernel(const DecArgs a) {
  using Tile = DecTile<D, GP, NST>;
  constexpr int KSTEPS = D / 32;        // MFMA k-steps over head_dim for S^T
  constexpr int NB = D / 16;            // 16-row blocks of O^T
  constexpr int SL = D / 8;             // 16-byte slices per token row
  constexpr int TPL = 64 / SL;          // token rows covered by one wave-wide load
  constexpr int NLOAD = kPage / TPL;    // wave-wide loads per K (or V) page
  constexpr int LPP = 2 * NLOAD;        // loads in flight per page
  static_assert(LPP * (NST - 1) <= 63, "vmcnt is 6 bits");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float(*red_o)[Tile::RED_O_PITCH] = (float(*)[Tile::RED_O_PITCH])smem;  // [wave*GP + head][d], aliases the ring
  float(*red_m)[16] = (float(*)[16])(smem + Tile::RED_BASE);
  float(*red_l)[16] = red_m + 4;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  // ---- every workgroup builds the same exclusive prefix of live-block counts over the batch.
  int* pfx = (int*)(smem + Tile::PFX_BASE);
  int* lens = (int*)(smem + Tile::LEN_BASE);
  int unit = a.chunk_pages, share = 0;
  {
    constexpr int PER = kMaxBatch / 256;  // consecutive sequences per thread
    int cnt[PER], cnt_t[PER], tsum = 0, tsum_t = 0;   // live blocks, live tiles
#pragma unroll
    for (int i = 0; i < PER; i++) {
      const int bi = tid * PER + i;
      int n = 0, nt = 0;
      if (bi < a.B) {
        const int l = length_of(a, bi);
        lens[bi] = l;
        int u0, u1;
        live_units(a, l, a.chunk_pages, u0, u1);
        n = u1 - u0;
        live_tiles(a, l, u0, u1);
        nt = u1 - u0;
      }
      cnt[i] = n;
      cnt_t[i] = nt;
      tsum += n;
      tsum_t += nt;
    }
    int incl = tsum, incl_t = tsum_t;  // inclusive scans over the wavefront
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(incl, d, 64), up_t = __shfl_up(incl_t, d, 64);
      if (lane >= d) {
        incl += up;
        incl_t += up_t;
      }
    }
    int* wsum = (int*)(smem + Tile::RED_BASE);
    if (lane == 63) {
      wsum[wave] = incl;
      wsum[4 + wave] = incl_t;
    }
    __syncthreads();
    int run = incl - tsum;
    if (a.even) {
      const EvenPlan p = even_plan(a, (wsum[0] + wsum[1] + wsum[2] + wsum[3]) * a.Hv,
                                   (wsum[4] + wsum[5] + wsum[6] + wsum[7]) * a.Hv);
      unit = p.unit;
      share = p.share;
      if (unit == 1) {
        run = incl_t - tsum_t;
        wsum += 4;
#pragma unroll
        for (int i = 0; i < PER; i++) cnt[i] = cnt_t[i];
      }
    }
    for (int w = 0; w < wave; w++) run += wsum[w];
#pragma unroll
    for (int i = 0; i < PER; i++) {
      const int bi = tid * PER + i;
      if (bi <= a.B) pfx[bi] = run;
      run += cnt[i];
    }
    if (tid == 255) pfx[kMaxBatch] = run;
    __syncthreads();
  }
  // ---- work distribution.  The unit of work is a block of `chunk_pages` pages of one (sequence,
  // kv head); blocks are numbered sequence-major, then kv head, then position.  A workgroup draws
  // runs of consecutive blocks from a global counter - long runs while plenty of work is left,
  // single blocks at the end (guided self-scheduling) - so that workgroups on CUs that get more
  // of the memory system take more of the work.  The part of a run inside one (sequence, kv head)
  // is a segment: one contiguous page range, streamed without a break, one partial record.
  const int n_blocks = pfx[a.B] * a.Hv;
  const int n_wg = gridDim.x;
  // The ids of at most 256 pages are kept in registers.  A fixed decomposition (one block per
  // record, pages dealt round-robin) makes the result independent of timing.
  const int max_run = a.deterministic ? 1 : max(1, 256 / a.chunk_pages);
  const int run0 = a.even ? share : min(max_run, max(1, n_blocks / (2 * n_wg)));
  int* s_next = (int*)(smem + Tile::NEXT_BASE);
  int* s_page = s_next + 3;  // next page of the segment to hand to a wavefront
  if (tid == 0) *s_page = 4 * NST;
  __syncthreads();
  int merge_pairs[2] = {0, 0}, n_merge = 0;   // pairs of which this workgroup leaves a record
  int run_e = blockIdx.x * run0;
  int run_end = min(run_e + run0, n_blocks);
  int handed = n_wg * run0;  // estimate of how many blocks have been handed out
  while (run_e < n_blocks) {
  bool first_segment = true;
  int next_e = 0, next_n = 0;
  while (run_e < run_end) {
  int b = 0;
  for (int hi = a.B; hi - b > 1;) {  // last b with Hv * pfx[b] <= run_e
    const int mid = (b + hi) >> 1;
    if (pfx[mid] * a.Hv <= run_e) b = mid; else hi = mid;
  }
  const int len = lens[b];
  int ch0, ch1;
  live_units(a, len, unit, ch0, ch1);
  const int rem = run_e - pfx[b] * a.Hv;
  const int hv = rem / (ch1 - ch0), cl = rem % (ch1 - ch0);
  // Virtual head -> kv head and group of (at most) 16 of its query heads.
  const int hk = a.ngrp == 1 ? hv : hv / a.ngrp;
  const int grp = hv - hk * a.ngrp;
  const int gcount = min(16, a.G - 16 * grp);
  const int hbase = hk * a.G + 16 * grp;
  const int seg = min(run_end - run_e, ch1 - ch0 - cl);
  int t0, t1;
  live_tiles(a, len, t0, t1);
  const int c_begin = max((ch0 + cl) * unit, t0), c_end = min((ch0 + cl + seg) * unit, t1);
  // Pages of the segment are numbered 0 .. n_pg-1.  A wavefront starts with pages wave + 4*i,
  // i < NST, and draws further ones from a counter in LDS whenever a ring stage frees up, so that
  // the 4 wavefronts finish together however unevenly the memory system serves them.
  const int n_pg = c_end - c_begin;

  // Draw the next run; the round trip overlaps the loads of Q and of the page ids below.  The
  // segment's record slot is the number of its first block: unique, and below the B * Hkv * NCH
  // records the workspace holds.  With equal shares it is workgroup + pair: from one segment of the list
  // to the next one of the two or both go up, so it is unique too, and the records of a pair lie side
  // by side in context order.
  const int rec = a.even ? (int)blockIdx.x + b * a.Hv + hv : run_e;
  const bool whole = a.even && seg == ch1 - ch0;   // all of the pair's keys: the result, not a record
  if (tid == 0 && first_segment) {
    next_n = min(max_run, max(1, (n_blocks - handed) / (4 * n_wg)));
    next_e = a.even ? n_blocks : atomicAdd(&a.ticket[0], next_n);
  }
  first_segment = false;

  // Q^T as MFMA B operand: lane (head column = lane%16, k-group = lane/16) holds d = 32s + 8kg .. +7.
  const int head = lane & 15, kg = lane >> 4;
  bf16x8 qf[KSTEPS];
#pragma unroll
  for (int s = 0; s < KSTEPS; s++) {
    if (head < gcount && 32 * s + 8 * kg < a.d_real) {
      qf[s] = *(const bf16x8*)(a.q + ((int64_t)b * a.Hq + hbase + head) * a.d_real + 32 * s + 8 * kg);
    } else {
#pragma unroll
      for (int e = 0; e < 8; e++) qf[s][e] = (__bf16)0.f;
    }
  }
  // Pool page of each tile of the segment (at most 256 tiles): register r, lane l holds tile 64r + l.
  int seg_pages[4] = {0, 0, 0, 0};
  if (PAGED) {
#pragma unroll
    for (int r = 0; r < 4; r++)
      if (64 * r + lane < n_pg)
        seg_pages[r] = a.page_tables[(int64_t)b * a.pt_stride + ((c_begin + 64 * r + lane) >> a.page_shift)];
  }
  auto page_id = [&](int idx) -> int {
    int pg = __builtin_amdgcn_readlane(seg_pages[0], idx & 63);
#pragma unroll
    for (int r = 1; r < 4; r++)
      if ((idx >> 6) == r) pg = __builtin_amdgcn_readlane(seg_pages[r], idx & 63);
    if (pg < 0) pg += a.num_pages;  // negative indices count from the end, as in the reference's gather
    return pg;
  };

  const int vslice = lane % SL;       // load layout: 16-byte slice of the row
  const int vtok = lane / SL;         // load layout: token row within a load
  const float c = a.scale * kLog2e;

  float m_run = kNegInf, l_run = 0.f;
  floatx4 o[NB];                      // O^T rows d = 16nb + 4kg + r, column = head
#pragma unroll
  for (int nb = 0; nb < NB; nb++) o[nb] = floatx4{0.f, 0.f, 0.f, 0.f};

  // Per-lane source offsets (elements) of the wave-wide loads of a page, and LDS read offsets.
  // Both tiles are stored with their 16-byte chunks XOR-swizzled by a function of the row, which
  // makes the K reads (16 lanes = 16 rows, same chunk) and the transposing V reads (rows 0..7 of
  // the same 32-byte column window) hit distinct banks.
  const int64_t k_row_stride = PAGED ? a.d_real : a.ks.s;
  const int64_t v_row_stride = PAGED ? a.d_real : a.vs.s;
  // A head_dim below the compiled width: the slices past it are fetched from slice 0 of the same row
  // instead.  Those LDS columns then hold finite copies of real data; the Q columns they meet are
  // zero, and the output rows they produce are never written.
  const int real_slices = a.d_real >> 3;
  int k_src[NLOAD], v_src[NLOAD];
#pragma unroll
  for (int i = 0; i < NLOAD; i++) {
    const int row = TPL * i + vtok;
    const int ksl = vslice ^ k_swizzle<D>(row), vsl = vslice ^ v_swizzle<D>(row);
    k_src[i] = (ksl < real_slices ? ksl : 0) * 8;     // + row * stride, added per page
    v_src[i] = (vsl < real_slices ? vsl : 0) * 8;
  }
  int k_rd[KSTEPS];
#pragma unroll
  for (int s = 0; s < KSTEPS; s++) k_rd[s] = (lane & 15) * Tile::ROW_BYTES + (((4 * s + kg) ^ k_swizzle<D>(lane & 15)) << 4);
  // Transposing V read for block nb: this lane points at row 4kg + (lane%16)/4, columns
  // 16nb + 4*(lane%4) .. +3, i.e. chunk 2nb + (lane%4)/2, half (lane%4)%2.
  const int vrow = 4 * kg + ((lane & 15) >> 2);
  const int v_rd0 = vrow * Tile::ROW_BYTES + ((lane & 2) << 3) + ((lane & 1) << 3);
  const int v_xor = v_swizzle<D>(vrow) << 4;
  const unsigned ring_lds = lds_address(smem) +
                            wave * (NST * Tile::STAGE_BYTES);
  char* ring = smem + wave * (NST * Tile::STAGE_BYTES);

  // Everything the compiler tracks has landed before the first untracked load is issued.
  wait_all_vmem();

  // Issues the 2*NLOAD loads of page `idx` of the segment into ring stage `st`.
  auto issue = [&](int idx, int st) {
    const int j = c_begin + idx;
    const __bf16 *kb, *vb;
    if (PAGED) {
      int pg = page_id(idx);
      if ((unsigned)pg >= (unsigned)a.num_pages) pg = 0;  // reads as zeros: see `valid` below
      // tile (j mod tiles-per-page) of pool page pg of kv head hk
      const int64_t tile = ((((int64_t)hk * a.num_pages + pg) << a.page_shift) + (j & ((1 << a.page_shift) - 1)));
      const int64_t off = tile * (kPage * a.d_real);
      kb = a.k + off;
      vb = a.v + off;
    } else {
      kb = a.k + b * a.ks.b + hk * a.ks.h;
      vb = a.v + b * a.vs.b + hk * a.vs.h;
    }
    const unsigned dst = __builtin_amdgcn_readfirstlane(ring_lds + st * Tile::STAGE_BYTES);
#pragma unroll
    for (int i = 0; i < NLOAD; i++) {
      // Rows past the end of a contiguous cache are clamped to its last row; they are masked.
      const int row = PAGED ? TPL * i + vtok : min(j * kPage + TPL * i + vtok, a.kv_len - 1);
      dma16(kb + row * k_row_stride + k_src[i], dst + i * 1024);
    }
#pragma unroll
    for (int i = 0; i < NLOAD; i++) {
      const int row = PAGED ? TPL * i + vtok : min(j * kPage + TPL * i + vtok, a.kv_len - 1);
      dma16(vb + row * v_row_stride + v_src[i], dst + Tile::TILE_BYTES + i * 1024);
    }
  };

  int ring_idx[NST];     // page held (or awaited) by each ring stage
  int issued = 0;
#pragma unroll
  for (int i = 0; i < NST; i++) {
    ring_idx[i] = wave + 4 * i;
    if (ring_idx[i] < n_pg) {
      issue(ring_idx[i], i);
      issued++;
    }
  }
  bool exhausted = issued < NST;
  int st = 0;
  for (int consumed = 0; consumed < issued; consumed++) {
    int idx = ring_idx[0];
#pragma unroll
    for (int i = 1; i < NST; i++)
      if (st == i) idx = ring_idx[i];
    const int j = c_begin + idx;
    // Wait for this page; the younger pages stay in flight.
    const int younger = issued - consumed - 1;
    if (NST > 3 && younger == 3) wait_vmem_le<(NST > 3 ? 3 : 0) * LPP>();
    else if (NST > 2 && younger == 2) wait_vmem_le<(NST > 2 ? 2 : 0) * LPP>();
    else if (NST > 1 && younger == 1) wait_vmem_le<(NST > 1 ? 1 : 0) * LPP>();
    else wait_vmem_le<0>();
    bool valid = true;
    if (PAGED) valid = (unsigned)page_id(idx) < (unsigned)a.num_pages;
    const char* kt = ring + st * Tile::STAGE_BYTES;
    const char* vt = kt + Tile::TILE_BYTES;
    bf16x8 kf[KSTEPS];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) kf[ks] = *(const bf16x8*)(kt + k_rd[ks]);
    shortx4 vf[NB];
#pragma unroll
    for (int nb = 0; nb < NB; nb++) vf[nb] = lds_read_tr16(vt + v_rd0 + ((nb * 32) ^ v_xor));
    // The stage is free as soon as its fragments sit in registers: refill it right away so that
    // the loads of page it+NST overlap the arithmetic of this one.
    wait_lds_reads();
    if (!exhausted) {
      int nxt = idx + 4 * NST;
      if (!a.deterministic) {
        if (lane == 0) nxt = atomicAdd(s_page, 1);
        nxt = __builtin_amdgcn_readfirstlane(nxt);
      }
      if (nxt < n_pg) {
        issue(nxt, st);
#pragma unroll
        for (int i = 0; i < NST; i++)
          if (st == i) ring_idx[i] = nxt;
        issued++;
      } else {
        exhausted = true;
      }
    }
    // ---- scores: S^T[token][head]; this lane: head = lane%16, tokens 4kg + r
    floatx4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) s = E::mfma_16x16x32(kf[ks], qf[ks], s);
    if constexpr (BIAS) {
      // logits = scale * q.k + bias (gpu_decoding.py:117-121, gpu_paged_attention.py:103-106): in raw
      // units, bias / scale.  Positions past the row's end are masked below; their reads are clamped.
      if (head < gcount) {
#pragma unroll
        for (int r = 0; r < 4; r++)
          s[r] += decode_bias_at(a, b, hbase + head, min(j * kPage + 4 * kg + r, a.kv_len - 1));
      }
    }
    // A page that straddles the length (or the window start) holds tokens whose probability is
    // exactly 0; their V rows may be uninitialised pool memory, and 0 * NaN would poison the sum,
    // so those rows are replaced by zeros, as are all rows of a page outside the pool.
    const bool boundary = (j * kPage + kPage > len) || (a.window >= 0 && len - 1 - j * kPage > a.window);
    if (boundary || !valid) {
      if (!valid) s = floatx4{0.f, 0.f, 0.f, 0.f};  // a page outside the pool reads as zeros
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int tpos = j * kPage + 4 * kg + r;
        bool keep = tpos < len;
        if (a.window >= 0) keep = keep && (len - 1 - tpos <= a.window);
        s[r] = keep ? s[r] : kMasked;
        if (!keep || !valid) {
#pragma unroll
          for (int nb = 0; nb < NB; nb++) vf[nb][r] = 0;
        }
      }
    }
    float mx = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m_run, mx);
    const bool changed = mn != m_run;
    const float corr = fast_exp2((m_run - mn) * c);
    m_run = mn;
    float psum = 0.f;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      s[r] = fast_exp2((s[r] - mn) * c);
      psum += s[r];
    }
    l_run = l_run * corr + psum;
    union { shortx4 v; bf16x2 p[2]; } pf;
    pf.p[0] = E::pack(s[0], s[1]);
    pf.p[1] = E::pack(s[2], s[3]);
    if (__builtin_amdgcn_ballot_w64(changed) != 0) {
#pragma unroll
      for (int nb = 0; nb < NB; nb++) o[nb] *= corr;
    }
    // ---- O^T += V^T P^T
#pragma unroll
    for (int nb = 0; nb < NB; nb++)
      o[nb] = E::mfma_16x16x16(vf[nb], pf.v, o[nb]);
    st = (st + 1 == NST) ? 0 : st + 1;
  }

  // ---- merge the 4 wavefronts of this workgroup.
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);
  if (kg == 0) {
    red_m[wave][head] = m_run;
    red_l[wave][head] = l_run;
  }
  __syncthreads();  // also: every wavefront is done with its ring, which red_o aliases
  {
    const float mw = fmaxf(fmaxf(red_m[0][head], red_m[1][head]), fmaxf(red_m[2][head], red_m[3][head]));
    const float f_wave = fast_exp2((m_run - mw) * c);
    if (head < GP) {
#pragma unroll
      for (int nb = 0; nb < NB; nb++)
        *(float4*)&red_o[wave * GP + head][16 * nb + 4 * kg] =
            float4{o[nb][0] * f_wave, o[nb][1] * f_wave, o[nb][2] * f_wave, o[nb][3] * f_wave};
    }
  }
  __syncthreads();
  const int64_t slot = rec;
  float* out_ws = a.ws_o + slot * (GP * D);
  if (whole) {
    for (int idx = tid; idx < GP * D / 2; idx += 256) {
      const int gq = 2 * idx / D, d = 2 * idx % D;
      if (gq >= gcount || d >= a.d_real) continue;
      const float mw = fmaxf(fmaxf(red_m[0][gq], red_m[1][gq]), fmaxf(red_m[2][gq], red_m[3][gq]));
      float lw = 0.f;
#pragma unroll
      for (int w = 0; w < 4; w++) lw += red_l[w][gq] * fast_exp2((red_m[w][gq] - mw) * c);
      const float inv = lw > 0.f ? 1.f / lw : 0.f;
      float x[2];
#pragma unroll
      for (int j = 0; j < 2; j++)
        x[j] = (red_o[gq][d + j] + red_o[GP + gq][d + j] + red_o[2 * GP + gq][d + j] + red_o[3 * GP + gq][d + j]) * inv;
      *(bf16x2*)(a.out + ((int64_t)b * a.Hq + hbase + gq) * a.d_real + d) = E::pack(x[0], x[1]);
    }
  } else {
    for (int idx = tid; idx < GP * D; idx += 256) {
      const int gq = idx / D, d = idx % D;
      write_record(out_ws + idx, red_o[gq][d] + red_o[GP + gq][d] + red_o[2 * GP + gq][d] + red_o[3 * GP + gq][d], MERGE);
    }
  }
  if (!whole && tid < GP) {
    const float mw = fmaxf(fmaxf(red_m[0][tid], red_m[1][tid]), fmaxf(red_m[2][tid], red_m[3][tid]));
    float lw = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) lw += red_l[w][tid] * fast_exp2((red_m[w][tid] - mw) * c);
    write_record(a.ws_m + slot * GP + tid, mw, MERGE);
    write_record(a.ws_l + slot * GP + tid, lw, MERGE);
  }
  if (MERGE && !whole) {
    merge_pairs[n_merge > 0] = b * a.Hv + hv;
    n_merge++;
  }
  // Table entries of the segment's chunks: the record at its first chunk, "none" at the others.
  for (int i = tid; i < seg && !a.even; i += 256) a.ws_tab[((int64_t)b * a.Hv + hv) * a.nch + cl + i] = i == 0 ? (int)slot : -1;
  if (tid == 0) *s_page = 4 * NST;
  __syncthreads();  // the ring (and red_m/red_l) are reused by the next segment
  run_e += seg;
  }  // segments of the run
  if (tid == 0) { s_next[0] = n_wg * run0 + next_e; s_next[1] = next_n; }
  __syncthreads();
  run_e = s_next[0];
  run_end = min(run_e + s_next[1], n_blocks);
  handed = run_e + s_next[1];
  __syncthreads();  // s_next is rewritten at the end of the next run
  }  // runs
  if constexpr (MERGE) {
    if (blockIdx.x == 0 && tid == 0) a.ticket[0] = 0;   // as the merge kernel leaves it
    // Pairs without a live key belong to no workgroup.
    for (int pair = blockIdx.x; pair < a.B * a.Hv; pair += n_wg) {
      const int b = pair / a.Hv;
      int t0, t1;
      live_tiles(a, lens[b], t0, t1);
      if (t0 == t1) merge_records<E, D, GP, 256, true>(a, b, pair - b * a.Hv, 0, [](int) { return 0; }, *(MergeLds<256>*)smem, tid);
    }
    if (n_merge > 0) finish_pairs<E, D, GP>(a, pfx, lens, unit, share, merge_pairs, n_merge, *(MergeLds<256>*)smem, tid);
  }
}

// Zeroes the work counter ahead of the split kernel when the workspace comes with unknown contents
// (a kernel rather than a memset so that the sequence can be captured into a graph).  A workspace
// that the caller declares reused skips it: the combine kernel leaves the counter at zero.
__global__ __launch_bounds__(64) void decode_plan_kernel(int* ticket) {
  if (threadIdx.x == 0) ticket[0] = 0;
}

// Merges the per-chunk partials of one (sequence, kv head): the "final round of flash"
// (gpu_paged_attention.py:287-296, gpu_decoding.py:277-283).
//
// A few tens of KB per workgroup: bound by the chain of dependent round trips to memory.  Every thread fetches
// its slice of a record together with the record's statistics and keeps a running (m, l, o) of its own, so
// that after the list of records there is one round trip and one exchange through LDS (statistics first, then
// weights, then slices: three round trips and eight barriers).  8 x 8 pairs of 8 records 7.4 -> 5.3 us, 64 x 8 pairs of
// up to 64 records 17.2 -> 12.0 us.
template <typename E, int D, int GP, int NT>
__global__ __launch_bounds__(NT) void decode_combine_kernel(const DecArgs a) {
  __shared__ int s_raw[kMaxChunks];       // the record table row
  __shared__ int s_list[kMaxChunks];      // records of this (sequence, kv head), in chunk order
  __shared__ int s_count;
  __shared__ MergeLds<NT> lds;
  const int hv = blockIdx.x, b = blockIdx.y;
  const int tid = threadIdx.x;
  const int len = length_of(a, b);
  int ch0, ch1;
  live_units(a, len, a.chunk_pages, ch0, ch1);
  int nc = ch1 - ch0;                     // live chunks = upper bound on records of this (b, hk)
  // The split kernel has finished: leave the work counter at zero for the next call on this workspace.
  if (hv == 0 && b == 0 && tid == 0) a.ticket[0] = 0;
  if (a.even) {
    // Where the pair's units lie in the list says which workgroups took them.
    int before[2] = {0, 0}, all[2] = {0, 0};   // of blocks, of tiles
    for (int i = tid; i < a.B; i += NT) {
      const int l = length_of(a, i);
#pragma unroll
      for (int k = 0; k < 2; k++) {
        int u0, u1;
        live_units(a, l, k == 0 ? a.chunk_pages : 1, u0, u1);
        all[k] += u1 - u0;
        before[k] += i < b ? u1 - u0 : 0;
      }
    }
    constexpr int W = NT / 64;
    __shared__ int s_sum[4][W];
#pragma unroll
    for (int k = 0; k < 2; k++) {
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        before[k] += __shfl_xor(before[k], o);
        all[k] += __shfl_xor(all[k], o);
      }
      if ((tid & 63) == 0) {
        s_sum[k][tid >> 6] = before[k];
        s_sum[2 + k][tid >> 6] = all[k];
      }
    }
    __syncthreads();
    auto sum = [&](int k) {
      int x = 0;
#pragma unroll
      for (int w = 0; w < W; w++) x += s_sum[k][w];
      return x;
    };
    const EvenPlan p = even_plan(a, sum(2) * a.Hv, sum(3) * a.Hv);
    live_units(a, len, p.unit, ch0, ch1);
    nc = ch1 - ch0;
    const int first = sum(p.unit == 1 ? 1 : 0) * a.Hv + hv * nc;
    const int w0 = first / p.share, w1 = nc > 0 ? (first + nc - 1) / p.share : w0 - 1;
    if (w0 == w1) return;                 // one workgroup had all of it and stored the result
    const int n = min(w1 - w0 + 1, kMaxChunks);
    if (tid < n) s_list[tid] = w0 + tid + b * a.Hv + hv;
    if (tid == 0) s_count = n;
  } else {
  // The whole table row in one round trip, then compacted in chunk order by one wavefront.
  if (tid < kMaxChunks) s_raw[tid] = tid < nc ? a.ws_tab[((int64_t)b * a.Hv + hv) * a.nch + tid] : -1;
  __syncthreads();
  if (tid < 64) {
    int count = 0;
    for (int base = 0; base < nc; base += 64) {
      const int r = s_raw[base + tid];
      const unsigned long long mask = __builtin_amdgcn_ballot_w64(r >= 0);
      if (r >= 0) s_list[count + __builtin_popcountll(mask & ((1ull << tid) - 1))] = r;
      count += __builtin_popcountll(mask);
    }
    if (tid == 0) s_count = count;
  }
  }
  __syncthreads();
  merge_records<E, D, GP, NT, false>(a, b, hv, s_count, [&](int i) { return s_list[i]; }, lds, tid);
}

// ---------------------------------------------------------------------------------------------
// fp32 decode (the reference's decode tests run float32, decoding_test.py:33): plain fp32
// multiply-adds and the accurate exponential, one workgroup per live block of `chunk_pages` pages of
// a (sequence, kv head), a fixed decomposition.  A token row is spread over 16 lanes; each 16-lane
// group keeps a running (m, l, o) per query head over the tokens it visits, the groups are merged at
// the end and leave one record in the same format as the 16-bit kernel's, for the same merge kernel.
// For parity with float32 callers, not for speed.
// ---------------------------------------------------------------------------------------------
template <int D, int GP, bool PAGED>
__global__ __launch_bounds__(256) void decode_split_f32_kernel(const DecArgs a) {
  constexpr int SL = D / 16;  // floats of a row per lane
  __shared__ float q_lds[GP * D];
  __shared__ float red_o[4][GP][D];
  __shared__ float red_m[4][GP], red_l[4][GP];
  const int c = blockIdx.x, hv = blockIdx.y, b = blockIdx.z;
  const int hk = hv / a.ngrp, grp = hv - hk * a.ngrp;
  const int gcount = min(16, a.G - 16 * grp);   // query heads of this group
  const int hbase = hk * a.G + 16 * grp;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, sub = lane >> 4, l16 = lane & 15;
  const int len = length_of(a, b);
  int ch0, ch1;
  live_units(a, len, a.chunk_pages, ch0, ch1);
  if (ch0 + c >= ch1) return;
  const int npages = min((len + kPage - 1) / kPage, a.pps);
  const int first_page = a.window >= 0 ? max(0, len - 1 - a.window) / kPage : 0;
  const int p_begin = max((ch0 + c) * a.chunk_pages, first_page);
  const int p_end = min((ch0 + c + 1) * a.chunk_pages, npages);
  const float* qg = (const float*)a.q + ((int64_t)b * a.Hq + hbase) * a.d_real;
  for (int i = tid; i < GP * D; i += 256) {
    const int h = i / D, d = i % D;   // columns past head_dim and heads past the group are zero
    q_lds[i] = (h < gcount && d < a.d_real) ? qg[h * a.d_real + d] : 0.f;
  }
  __syncthreads();

  float m[GP], l[GP], o[GP][SL];
#pragma unroll
  for (int h = 0; h < GP; h++) {
    m[h] = kNegInf;
    l[h] = 0.f;
#pragma unroll
    for (int i = 0; i < SL; i++) o[h][i] = 0.f;
  }
  for (int tok = p_begin * kPage + wave * 4 + sub; tok < p_end * kPage; tok += 16) {
    const float *kr, *vr;
    bool valid = true;
    if (PAGED) {
      const int page_tokens = kPage << a.page_shift;
      int pg = a.page_tables[(int64_t)b * a.pt_stride + tok / page_tokens];
      if (pg < 0) pg += a.num_pages;  // negative indices count from the end, as in the reference's gather
      valid = (unsigned)pg < (unsigned)a.num_pages;  // a page outside the pool reads as zeros
      const int64_t off = (((int64_t)hk * a.num_pages + (valid ? pg : 0)) * page_tokens + tok % page_tokens) * a.d_real;
      kr = (const float*)a.k + off;
      vr = (const float*)a.v + off;
    } else {
      const int row = min(tok, a.kv_len - 1);  // rows past the cache are masked below
      kr = (const float*)a.k + b * a.ks.b + (int64_t)row * a.ks.s + hk * a.ks.h;
      vr = (const float*)a.v + b * a.vs.b + (int64_t)row * a.vs.s + hk * a.vs.h;
    }
    bool keep = tok < len;
    if (a.window >= 0) keep = keep && (len - 1 - tok <= a.window);
    if (!keep) continue;  // uniform over the 16 lanes of the token
    float kx[SL], vx[SL];
#pragma unroll
    for (int i = 0; i < SL; i += 4) {
      const bool in = valid && SL * l16 + i < a.d_real;   // head_dim is a multiple of 8: whole groups of 4
      const float4 x = in ? *(const float4*)(kr + SL * l16 + i) : float4{0.f, 0.f, 0.f, 0.f};
      const float4 y = in ? *(const float4*)(vr + SL * l16 + i) : float4{0.f, 0.f, 0.f, 0.f};
      kx[i] = x.x; kx[i + 1] = x.y; kx[i + 2] = x.z; kx[i + 3] = x.w;
      vx[i] = y.x; vx[i + 1] = y.y; vx[i + 2] = y.z; vx[i + 3] = y.w;
    }
#pragma unroll
    for (int h = 0; h < GP; h++) {
      float dot = 0.f;
#pragma unroll
      for (int i = 0; i < SL; i++) dot = __builtin_fmaf(q_lds[h * D + SL * l16 + i], kx[i], dot);
      dot += __shfl_xor(dot, 1, 64);
      dot += __shfl_xor(dot, 2, 64);
      dot += __shfl_xor(dot, 4, 64);
      dot += __shfl_xor(dot, 8, 64);
      if (a.bias && h < gcount) dot += decode_bias_at(a, b, hbase + h, tok);
      const float mn = fmaxf(m[h], dot);
      const float corr = expf((m[h] - mn) * a.scale);
      const float pr = expf((dot - mn) * a.scale);
      m[h] = mn;
      l[h] = l[h] * corr + pr;
#pragma unroll
      for (int i = 0; i < SL; i++) o[h][i] = __builtin_fmaf(pr, vx[i], o[h][i] * corr);
    }
  }
  // ---- merge the four 16-lane groups of the wavefront, then the four wavefronts.
#pragma unroll
  for (int h = 0; h < GP; h++) {
    float mw = fmaxf(m[h], __shfl_xor(m[h], 16, 64));
    mw = fmaxf(mw, __shfl_xor(mw, 32, 64));
    const float f = expf((m[h] - mw) * a.scale);
    float lw = l[h] * f;
    lw += __shfl_xor(lw, 16, 64);
    lw += __shfl_xor(lw, 32, 64);
#pragma unroll
    for (int i = 0; i < SL; i++) {
      float x = o[h][i] * f;
      x += __shfl_xor(x, 16, 64);
      x += __shfl_xor(x, 32, 64);
      if (sub == 0) red_o[wave][h][SL * l16 + i] = x;
    }
    if (lane == 0) {
      red_m[wave][h] = mw;
      red_l[wave][h] = lw;
    }
  }
  __syncthreads();
  const int64_t rec = ((int64_t)b * a.Hv + hv) * a.nch + c;
  for (int idx = tid; idx < GP * D; idx += 256) {
    const int h = idx / D, d = idx % D;
    const float mw = fmaxf(fmaxf(red_m[0][h], red_m[1][h]), fmaxf(red_m[2][h], red_m[3][h]));
    float acc = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) acc += red_o[w][h][d] * expf((red_m[w][h] - mw) * a.scale);
    a.ws_o[rec * (GP * D) + idx] = acc;
  }
  if (tid < GP) {
    const float mw = fmaxf(fmaxf(red_m[0][tid], red_m[1][tid]), fmaxf(red_m[2][tid], red_m[3][tid]));
    float lw = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) lw += red_l[w][tid] * expf((red_m[w][tid] - mw) * a.scale);
    a.ws_m[rec * GP + tid] = mw;
    a.ws_l[rec * GP + tid] = lw;
    if (tid == 0) a.ws_tab[rec] = (int)rec;
  }
}

// Ring depth (pages in flight per wavefront).  head_dim 128: 2 x 8 KB per wavefront, 69 KB per
// workgroup, two workgroups per CU.
constexpr int kStages128 = 2;
constexpr int kStages64 = 4;

// Workgroups the split kernel keeps resident on the GPU it is tuned for (two on each of 256 CUs).
constexpr int kSplitSlots = 512;

// Pages per block of work.  `rows` = (sequence, kv head group) pairs of the call.
static int pick_chunk_pages(int pps, int64_t rows) {
  // 32 pages = 512 tokens = 256 KB of K+V per workgroup at head_dim 128.
  int cp = 32;
  // A small call (one sequence, a short context) has fewer such blocks than the GPU has workgroup slots
  // and is bound by the latency of a block's few rounds of loads: shorter blocks, about one per slot,
  // down to 8 pages (one round of the four wavefronts' rings).
  if (rows > 0 && rows * ((pps + cp - 1) / cp) < kSplitSlots) {
    const int64_t per_row = kSplitSlots / rows;
    cp = (int)(((pps + per_row - 1) / per_row + 3) / 4 * 4);
    cp = cp < 8 ? 8 : (cp > 32 ? 32 : cp);
  }
  if (pps < cp) cp = ((pps + 3) / 4) * 4;
  if (pps > cp * kMaxChunks) cp = ((pps + kMaxChunks - 1) / kMaxChunks + 3) / 4 * 4;
  return cp < 4 ? 4 : cp;
}

constexpr int kWsHeaderFloats = 64;  // 256 bytes ahead of the records: the work counter

static size_t ws_bytes(int B, int Hkv, int nch, int gp, int D) {
  return (size_t)B * Hkv * nch * ((size_t)gp * D + 2 * gp + 1) * sizeof(float) + kWsHeaderFloats * sizeof(float);
}

// Query-head columns a record holds: the heads of a group padded to 4 / 8 / 16.  The kernels that add
// a bias are compiled for 16 only.
static int gp_of(int G, bool bias) { return bias || G > 8 ? 16 : (G <= 4 ? 4 : 8); }
// Groups of at most 16 query heads per kv head ("virtual" kv heads per kv head).
static int groups_of(int G) { return (G + 15) / 16; }
// Compiled head_dim width that serves a head_dim (a multiple of 8, at most 128).
static int width_of(int d) { return d <= 64 ? 64 : 128; }
// log2(page_size / 16), or -1 if the page size is not 16 times a power of two.
static int page_shift_of(int page_size) {
  for (int sh = 0; sh < 16; sh++)
    if (page_size == (kPage << sh)) return sh;
  return -1;
}

// Tiles of a (sequence, kv head) pair that a call can have to read, from its shapes.
static int64_t capacity_tiles(int tiles, int window) {
  const int64_t w = window >= 0 ? (int64_t)window / kPage + 2 : tiles;
  return w < tiles ? w : tiles;
}

// Workspace of equal shares: one record per workgroup and pair at most.  The size does not depend on the window
// (a query may leave it out): with one there are no more tiles, in shares of 8 or more.
static size_t even_ws_bytes(int64_t pairs, int tiles, int gp, int width) {
  const int64_t wgs = (pairs * tiles + 7) / 8, slots = 2 * (int64_t)cu_count();
  const int records = (int)((wgs < slots ? wgs : slots) + pairs);
  return ws_bytes(1, 1, records, gp, width) + (size_t)records * sizeof(uint64_t);   // behind the table, which is not used: flags
}
// The workgroups' records must not push a call whose blocks fit it past the buffer of axl_paged_decode_static
// (thousands of pairs of a block each; blocks are drawn there).
static bool even_fits(size_t even, size_t drawn) { return even <= drawn || even <= AXL_PAGED_DECODE_STATIC_MAX_BYTES; }

// The split kernel merges the records itself (finish_pairs) where its workgroups are short and a pair's records are a
// round or two of loads: the marks and the records' way past the L2 take 1.5 us more there than in a kernel of its own, which costs 3 us
// and its launch; 4 us and more where the memory system is loaded, and one workgroup of 256 threads is slow with many
// records.  (Call, own kernel / by the split kernel: 420 tiles in shares of 8, 9 records 12.9 / 11.0 us; 10 280 tiles in shares of 20
// 25.1 / 24.1; 9552 in 20, 31 records 21.9 / 21.1; 16 384 in 36 30.4 / 32.5; 8 sequences of 2000 to 8190 tokens, shares of 64,
// 40.6 / 42.1; shares of 8, 39 records of 8 heads 25.1 / 29.8.)  A workgroup whose share ends inside a pair is the last one of
// two pairs as often as not and merges one after the other.  In shares of 8 that takes longer than the kernel (16 heads, one
// sequence of 1000 tokens in a cache of 1006, 126 shares for 128 blocks, 14.7 / 16.6 us; window 1024 of 6000, 8 heads 14.7 / 16.4; 4
// sequences of 991, 16 heads 17.8 / 20.8), so there every block the call can have must find a workgroup, and not all that the
// GPU holds at once (512 blocks of 32 heads 14.1 / 14.9).  In shares of 12 to 20 the two are even, and the call gains where it
// turns out to have fewer blocks than workgroups (4224 to 8448 tiles: 0.92 to 1.03; in 24 up to 1.08).  The kernel of its own
// takes 1024 threads from four rounds on
// (108 records of 8 heads 24.0 -> 18.8 us, 240 40.2 -> 26.6, 8 pairs of 65 65.8 -> 60.5; with few records, or hundreds of
// pairs of them, it would lose 1 to 3 us).
constexpr int kMergeShare = 20, kMergeRounds = 2, kManyRounds = 4, kManyThreads = 1024;

// Equal shares (see the head of this file) where the capacity makes them at most 256 tiles, the page ids a
// segment keeps in registers.  Measured at 8 sequences of 2000 to 8190 tokens, 8 kv heads (40 tiles a
// workgroup): split kernel 42.8 us drawing blocks of 32 tiles (640 blocks for 512 workgroups), 39.6 us in
// equal shares, and the call is two launches instead of three; at 64 sequences of up to 32768 tokens (1024
// tiles a workgroup) drawing is 4 % faster.  Fills in the launch's part of `a`; a.B, a.Hv, a.pps, a.window
// and a.nch are set.
static void plan_even(DecArgs& a, bool deterministic, int& merge_rounds, bool& merge_here) {
  const int64_t pair = capacity_tiles(a.pps, a.window), total = pair * a.B * a.Hv;
  const int slots = 2 * cu_count();
  // at least 8 tiles (one round of the wavefronts' rings: a shorter share ends no sooner), and few enough
  // records per pair for the tables of the combine kernel
  const int64_t by_table = (pair + kMaxChunks - 2) / (kMaxChunks - 1);
  a.min_share = (int)((by_table > 8 ? by_table : 8) + 3) & ~3;
  a.n_wg = (int)(total < (int64_t)slots * a.min_share ? (total + a.min_share - 1) / a.min_share : slots);
  const int64_t share = ((total + a.n_wg - 1) / a.n_wg + 3) & ~(int64_t)3;
  a.even = a.B <= kMaxBatch && share <= 256 && a.min_share <= 256;
  // records a pair can have, by equal shares or a block each, and the rounds of loads in which 256 threads merge them
  const int64_t records = std::max((pair + share - 1) / share + 1, std::min<int64_t>(pair / a.chunk_pages + 2, a.n_wg));
  merge_rounds = (int)((records * std::min(a.G, 16) * width_of(a.d_real) / 4 + kMergeBatch * 256 - 1) / (kMergeBatch * 256));
  // blocks a pair can have: under a window they may begin and end inside one
  const int64_t blocks = a.window >= 0 ? std::min<int64_t>(a.nch, (pair + a.chunk_pages - 2) / a.chunk_pages + 1) : a.nch;
  const bool block_each = blocks * a.B * a.Hv <= a.n_wg && a.n_wg < slots;
  merge_here = !a.bias && merge_rounds <= kMergeRounds && share <= kMergeShare && (block_each || share > a.min_share);
  // A deterministic call keeps to the blocks, whose bits depend on a pair's own keys alone: equal shares only
  // where the shapes leave no more blocks than workgroups.
  if (deterministic && (int64_t)a.B * a.Hv * a.nch > a.n_wg) a.even = 0;
  const int gp = gp_of(a.G, a.bias != nullptr), width = width_of(a.d_real);
  if (!even_fits(even_ws_bytes((int64_t)a.B * a.Hv, a.pps, gp, width), ws_bytes(a.B, a.Hv, a.nch, gp, width))) a.even = 0;
  if (!a.even) {
    merge_rounds = 1;   // runs, mostly of several blocks: few records
    merge_here = false;
  }
}

static size_t ws_bytes_for(int batch, int hq, int hkv, int d, int tiles, bool bias, int dtype) {
  const int G = hq / hkv;
  const int cp = pick_chunk_pages(tiles, (int64_t)batch * hkv * groups_of(G));
  const int nch = (tiles + cp - 1) / cp;
  const size_t drawn = ws_bytes(batch, hkv * groups_of(G), nch, gp_of(G, bias), width_of(d));
  if (dtype == AXL_F32 || batch > kMaxBatch) return drawn;
  const size_t even = even_ws_bytes((int64_t)batch * hkv * groups_of(G), tiles, gp_of(G, bias), width_of(d));
  return even > drawn && even_fits(even, drawn) ? even : drawn;
}

size_t paged_decode_workspace_bytes(const AxlPagedDecodeParams& p) {
  const int sh = page_shift_of(p.page_size);
  if (p.pages_per_seq <= 0 || p.num_kv_heads <= 0 || p.num_q_heads < p.num_kv_heads || sh < 0) return 0;
  return ws_bytes_for(p.batch, p.num_q_heads, p.num_kv_heads, p.head_dim, p.pages_per_seq << sh, p.bias.bias != nullptr,
                      p.dtype);
}

size_t decode_workspace_bytes(const AxlDecodeParams& p) {
  if (p.kv_len <= 0 || p.num_kv_heads <= 0 || p.num_q_heads < p.num_kv_heads) return 0;
  return ws_bytes_for(p.batch, p.num_q_heads, p.num_kv_heads, p.head_dim, (p.kv_len + kPage - 1) / kPage,
                      p.bias.bias != nullptr, p.dtype);
}

static void set_lengths(DecArgs& a, const int32_t* lengths, int64_t stride, int flags) {
  a.lengths = (const char*)lengths;
  a.len_i64 = (flags & AXL_DECODE_LENGTHS_I64) != 0;
  a.len_add = (flags & AXL_DECODE_LENGTHS_ARE_POSITIONS) != 0;
  const bool strided = a.len_i64 || a.len_add;
  a.len_stride = (strided ? stride : 1) * (a.len_i64 ? 8 : 4);
}

static void set_bias(DecArgs& a, const AxlDecodeBias& x, float scale) {
  const int es = x.dtype == AXL_F32 ? 4 : 2;
  a.bias = (const char*)x.bias;
  a.bias_sb = x.batch_stride * es;
  a.bias_sh = x.head_stride * es;
  a.bias_f32 = x.dtype == AXL_F32;
  a.inv_scale = 1.0f / scale;
}

// AXL_DECODE_DETERMINISTIC in the environment, read once: the default for calls that do not set the flag.
static bool deterministic_by_default() {
  static const bool v = [] {
    const char* det = getenv("AXL_DECODE_DETERMINISTIC");
    return det && det[0] != '\0' && det[0] != '0';
  }();
  return v;
}

// A number of its own for every call of every process: marks of an earlier call, or whatever else a workspace holds, are
// not taken for this call's.
static uint64_t next_call_id() {
  static std::atomic<uint64_t> next{[] {
    std::random_device r;
    return ((uint64_t)r() << 32) ^ r();
  }()};
  const uint64_t id = next.fetch_add(1, std::memory_order_relaxed);
  return id ? id : next.fetch_add(1, std::memory_order_relaxed);
}

// Whether what is enqueued becomes part of a graph (also where that cannot be asked).
static bool is_captured(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &status) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return status != hipStreamCaptureStatusNone;
}

template <typename E, bool PAGED>
static int launch_common(DecArgs a, int flags, hipStream_t stream, const char* who) {
  const int D = width_of(a.d_real);
  const bool bias = a.bias != nullptr;
  const int gp = gp_of(a.G, bias);
  a.ngrp = groups_of(a.G);
  a.Hv = a.Hkv * a.ngrp;
  a.chunk_pages = pick_chunk_pages(a.pps, (int64_t)a.B * a.Hv);
  if (a.chunk_pages > 256)
    return set_error(AXL_ERR_UNSUPPORTED, "%s: context longer than %d tokens", who, 256 * kMaxChunks * kPage);
  a.nch = (a.pps + a.chunk_pages - 1) / a.chunk_pages;
  // Workspace: a 256-byte header (the work counter, at the same place whatever the shapes), then the
  // records, their statistics and the record table.
  a.ticket = (int*)a.ws_o;
  a.ws_o += kWsHeaderFloats;
  float* ws = a.ws_o;
  a.deterministic = (flags & AXL_DECODE_DETERMINISTIC) != 0 || deterministic_by_default();
  int merge_rounds;
  bool merge_here;
  plan_even(a, a.deterministic, merge_rounds, merge_here);
  const size_t records = a.even ? (size_t)a.n_wg + (size_t)a.B * a.Hv : (size_t)a.B * a.Hv * a.nch;
  const size_t n_o = records * gp * D, n_s = records * gp;
  a.ws_m = ws + n_o;
  a.ws_l = ws + n_o + n_s;
  a.ws_tab = (int32_t*)(ws + n_o + 2 * n_s);
  a.ws_flag = (uint64_t*)(ws + n_o + 2 * n_s);
  a.call_id = merge_here && !is_captured(stream) ? next_call_id() : 0;
  // Two workgroups fit a CU (LDS); the split kernel is persistent and strides over its work items.
  const dim3 grid(a.even ? a.n_wg : 2 * cu_count());
  hipError_t err = hipSuccess;
  if (!(flags & AXL_DECODE_WORKSPACE_REUSED) && !a.even)
    hipLaunchKernelGGL(decode_plan_kernel, dim3(1), dim3(64), 0, stream, a.ticket);
#define AXL_DEC(E, DD, GG, NS, BB)                                                              \
  do {                                                                                          \
    using Tile = DecTile<DD, GG, NS>;                                                           \
    auto kern = BB || !s.call_id ? decode_split_kernel<E, DD, GG, PAGED, NS, BB, false>         \
                                 : decode_split_kernel<E, DD, GG, PAGED, NS, BB, !BB>;          \
    err = allow_dynamic_lds((const void*)kern, Tile::LDS_BYTES);                                \
    if (err == hipSuccess) {                                                                    \
      hipLaunchKernelGGL(kern, grid, dim3(256), Tile::LDS_BYTES, stream, s);                    \
      if (s.call_id) break;                                                                     \
      if (merge_rounds >= kManyRounds)                                                          \
        hipLaunchKernelGGL((decode_combine_kernel<E, DD, GG, kManyThreads>), cgrid, dim3(kManyThreads), 0, stream, s); \
      else                                                                                      \
        hipLaunchKernelGGL((decode_combine_kernel<E, DD, GG, 256>), cgrid, dim3(256), 0, stream, s); \
    }                                                                                           \
  } while (0)
  // The kernels keep per-sequence tables in LDS: larger batches go in slices of kMaxBatch (each
  // slice's combine kernel leaves the shared work counter at zero for the next slice).
  for (int b0 = 0; b0 < a.B && err == hipSuccess; b0 += kMaxBatch) {
    DecArgs s = a;
    s.B = a.B - b0 < kMaxBatch ? a.B - b0 : kMaxBatch;
    s.q = a.q + (size_t)b0 * a.Hq * a.d_real;
    s.out = a.out + (size_t)b0 * a.Hq * a.d_real;
    s.lengths = a.lengths + b0 * a.len_stride;
    if (PAGED) s.page_tables = a.page_tables + (size_t)b0 * a.pt_stride;
    else { s.k = a.k + b0 * a.ks.b; s.v = a.v + b0 * a.vs.b; }
    if (bias) s.bias = a.bias + b0 * a.bias_sb;
    s.ws_o = a.ws_o + (size_t)b0 * a.Hv * a.nch * gp * D;
    s.ws_m = a.ws_m + (size_t)b0 * a.Hv * a.nch * gp;
    s.ws_l = a.ws_l + (size_t)b0 * a.Hv * a.nch * gp;
    s.ws_tab = a.ws_tab + (size_t)b0 * a.Hv * a.nch;
    const dim3 cgrid(a.Hv, s.B);
    if (bias && D == 128) AXL_DEC(E, 128, 16, kStages128, true);
    else if (bias) AXL_DEC(E, 64, 16, kStages64, true);
    else if (D == 128 && gp == 4) AXL_DEC(E, 128, 4, kStages128, false);
    else if (D == 128 && gp == 8) AXL_DEC(E, 128, 8, kStages128, false);
    else if (D == 128) AXL_DEC(E, 128, 16, kStages128, false);
    else if (gp == 4) AXL_DEC(E, 64, 4, kStages64, false);
    else if (gp == 8) AXL_DEC(E, 64, 8, kStages64, false);
    else AXL_DEC(E, 64, 16, kStages64, false);
  }
#undef AXL_DEC
  if (err == hipSuccess) err = hipGetLastError();
  if (err != hipSuccess)
    return set_error(AXL_ERR_LAUNCH, "%s: launch failed: %s", who, hipGetErrorString(err));
  return AXL_OK;
}

template <bool PAGED>
static int launch_f32(DecArgs a, hipStream_t stream, const char* who) {
  const int D = width_of(a.d_real);
  const int gp = gp_of(a.G, a.bias != nullptr);
  a.ngrp = groups_of(a.G);
  a.Hv = a.Hkv * a.ngrp;
  a.chunk_pages = pick_chunk_pages(a.pps, (int64_t)a.B * a.Hv);
  if (a.chunk_pages > 256)
    return set_error(AXL_ERR_UNSUPPORTED, "%s: context longer than %d tokens", who, 256 * kMaxChunks * kPage);
  if (a.B > 65535) return set_error(AXL_ERR_UNSUPPORTED, "%s: more than 65535 sequences in fp32", who);
  a.nch = (a.pps + a.chunk_pages - 1) / a.chunk_pages;
  a.ticket = (int*)a.ws_o;
  a.ws_o += kWsHeaderFloats;
  float* ws = a.ws_o;
  const size_t n_o = (size_t)a.B * a.Hv * a.nch * gp * D;
  const size_t n_s = (size_t)a.B * a.Hv * a.nch * gp;
  a.ws_m = ws + n_o;
  a.ws_l = ws + n_o + n_s;
  a.ws_tab = (int32_t*)(ws + n_o + 2 * n_s);
  a.deterministic = 1;
  // One workgroup per live chunk writes that chunk's table entry; the work counter is not used (the
  // combine kernel still leaves it at zero).
  const dim3 grid(a.nch, a.Hv, a.B), cgrid(a.Hv, a.B);
#define AXL_DEC32(DD, GG)                                                                          \
  do {                                                                                              \
    hipLaunchKernelGGL((decode_split_f32_kernel<DD, GG, PAGED>), grid, dim3(256), 0, stream, a);    \
    hipLaunchKernelGGL((decode_combine_kernel<ElemF32, DD, GG, 256>), cgrid, dim3(256), 0, stream, a); \
  } while (0)
  if (D == 128 && gp == 4) AXL_DEC32(128, 4);
  else if (D == 128 && gp == 8) AXL_DEC32(128, 8);
  else if (D == 128) AXL_DEC32(128, 16);
  else if (gp == 4) AXL_DEC32(64, 4);
  else if (gp == 8) AXL_DEC32(64, 8);
  else AXL_DEC32(64, 16);
#undef AXL_DEC32
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return set_error(AXL_ERR_LAUNCH, "%s: launch failed: %s", who, hipGetErrorString(err));
  return AXL_OK;
}

int launch_paged_decode(const AxlPagedDecodeParams& p, hipStream_t stream) {
  DecArgs a{};
  a.q = (const __bf16*)p.q; a.k = (const __bf16*)p.k_pages; a.v = (const __bf16*)p.v_pages;
  a.page_tables = p.page_tables; a.out = (__bf16*)p.out;
  set_lengths(a, p.lengths, p.lengths_stride, p.flags);
  a.ws_o = (float*)p.workspace;
  a.B = p.batch; a.Hq = p.num_q_heads; a.Hkv = p.num_kv_heads; a.G = p.num_q_heads / p.num_kv_heads;
  a.page_shift = page_shift_of(p.page_size);   // the entry point has checked the page size
  a.pt_stride = p.pages_per_seq;
  a.num_pages = p.num_pages; a.pps = p.pages_per_seq << a.page_shift; a.kv_len = p.pages_per_seq * p.page_size;
  a.d_real = p.head_dim;
  a.window = p.sliding_window < 0 ? -1 : p.sliding_window;
  a.scale = p.softmax_scale;
  set_bias(a, p.bias, p.softmax_scale);
  if (p.dtype == AXL_F32) return launch_f32<true>(a, stream, "axl_paged_decode");
  return p.dtype == AXL_F16 ? launch_common<ElemF16, true>(a, p.flags, stream, "axl_paged_decode")
                            : launch_common<ElemBf16, true>(a, p.flags, stream, "axl_paged_decode");
}

// ---------------------------------------------------------------------------------------------
// Allocation-free variant of the paged decode: the split-K workspace (partial records, record table,
// work counter) is this file-scope device array instead of caller memory.  Every GPU the library runs
// on holds its own copy until the process ends; `scratch` itself is a host-side stand-in, the device
// address comes from hipGetSymbolAddress, once per device.
// ---------------------------------------------------------------------------------------------
constexpr size_t kStaticScratchBytes = AXL_PAGED_DECODE_STATIC_MAX_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxDevices];  // device address of `scratch` on each device, once resolved

// Device address of this device's copy of `scratch` (the current device is the one the call runs on).
static int static_scratch(void** ptr, const char* who) {
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return set_error(AXL_ERR_LAUNCH, "%s: hipGetDevice: %s", who, hipGetErrorString(err));
  if (dev < 0 || dev >= kMaxDevices) return set_error(AXL_ERR_UNSUPPORTED, "%s: device index %d", who, dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (err != hipSuccess || !p)
      return set_error(AXL_ERR_LAUNCH, "%s: hipGetSymbolAddress(scratch): %s", who, hipGetErrorString(err));
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return AXL_OK;
}

int launch_paged_decode_static(const AxlPagedDecodeParams& p, hipStream_t stream) {
  const char* who = "axl_paged_decode_static";
  const size_t need = paged_decode_workspace_bytes(p);
  if (need > kStaticScratchBytes)
    return set_error(AXL_ERR_WORKSPACE,
                     "%s: these shapes need %zu bytes of split-K scratch, the built-in buffer holds %zu "
                     "(use axl_paged_decode with a caller workspace)", who, need, kStaticScratchBytes);
  void* ws = nullptr;
  const int rc = static_scratch(&ws, who);
  if (rc != AXL_OK) return rc;
  AxlPagedDecodeParams q = p;
  q.workspace = ws;  // the resolved device address, never the array's name
  q.workspace_bytes = kStaticScratchBytes;
  // The buffer keeps the previous call's contents (possibly of other shapes, possibly of a call that
  // was captured and never replayed): the work counter is zeroed by a kernel on every call.
  q.flags &= ~AXL_DECODE_WORKSPACE_REUSED;
  return launch_paged_decode(q, stream);
}

int launch_decode(const AxlDecodeParams& p, hipStream_t stream) {
  DecArgs a{};
  a.q = (const __bf16*)p.q; a.k = (const __bf16*)p.k; a.v = (const __bf16*)p.v;
  a.page_tables = nullptr; a.out = (__bf16*)p.out;
  set_lengths(a, p.lengths, p.lengths_stride, p.flags);
  a.ws_o = (float*)p.workspace;
  a.ks = Strides3{p.k_strides.batch, p.k_strides.seq, p.k_strides.head};
  a.vs = Strides3{p.v_strides.batch, p.v_strides.seq, p.v_strides.head};
  a.B = p.batch; a.Hq = p.num_q_heads; a.Hkv = p.num_kv_heads; a.G = p.num_q_heads / p.num_kv_heads;
  a.num_pages = 0; a.pps = (p.kv_len + kPage - 1) / kPage; a.kv_len = p.kv_len;
  a.page_shift = 0; a.pt_stride = 0;
  a.d_real = p.head_dim;
  a.window = p.sliding_window < 0 ? -1 : p.sliding_window;
  a.scale = p.softmax_scale;
  set_bias(a, p.bias, p.softmax_scale);
  if (p.dtype == AXL_F32) return launch_f32<false>(a, stream, "axl_decode");
  return p.dtype == AXL_F16 ? launch_common<ElemF16, false>(a, p.flags, stream, "axl_decode")
                            : launch_common<ElemBf16, false>(a, p.flags, stream, "axl_decode");
}

}  // namespace axl
