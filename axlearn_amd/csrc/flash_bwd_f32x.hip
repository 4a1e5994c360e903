// fp32 flash-attention backward for gfx950 with every fp32 product formed from bf16 parts
// (flash_bwd_f32x.h): dK/dV, and dQ from the dS that the dK/dV kernel leaves in the workspace.
// (dQ without a dS workspace, and the kernels on the fp32 matrix instruction: flash_bwd_f32.hip.)
//
// Replaces the float32 case of axlearn/common/flash_attention/gpu_attention.py:621-786
// (`_mha_backward`) with
//   p  = exp(scale * q k^T + bias - lse)                    (:507, :599)
//   dp = dO v^T, zeroed where dropped and scaled by 1/(1-rate)   (:508-512, :600-603)
//   ds = p * (dp - delta)                                   (:514, :604)
//   dv += (p after dropout)^T dO,  dk += scale * ds^T q,  dq += scale * ds k   (:513, :518, :608)
#include "flash_bwd_f32x.h"

namespace axl {

// ---------------------------------------------------------------------------------------------
// dK/dV.  A workgroup owns 128 keys of one kv head and loops over 32-query tiles of the heads of its group.
//   S[q][key] = Q K^T and dP[q][key] = dO V^T (A = Q / dO row of the tile, B = K / V row l32), so
//   lane (l32, g) holds key l32 and, in register r, query 16 (r/8) + 8g + r%8;
//   dV^T[d][key] += dO^T[d][q] P[q][key],  dK^T[d][key] += Q^T[d][q] dS[q][key].
//
// Bound by the matrix cores (24 bf16 products per pair and element of d), as long as the rest hides behind
// them: per tile and key a lane forms 32 exponent / dS values, splits them, and splits its share of the
// next tile.  One wavefront per SIMD doing all of it in turn kept the matrix cores busy a fifth of the time.
// So 32 keys belong to TWO wavefronts of the same SIMD, each with half of the products and all of its
// stationary operand in registers:
//   wavefronts 0..3 ("P")   S(e) from their K rows, P(e), dV += P(e)^T dO(e)
//   wavefronts 4..7 ("dS")  dP(e) from their V rows, dS(e) = P(e) (dP(e) - delta), dK += dS(e)^T Q(e)
// P(e) goes from one to the other through LDS in fp32.  The dS wavefront is one tile behind with its second
// half: in iteration e it forms dS(e-1), multiplies it, then starts dP(e); one barrier per tile, and
// one wavefront's vector arithmetic falls on the other's matrix instructions.  Neither keeps more
// than one accumulator set (64 registers), so both operands fit 256 registers and two wavefronts a SIMD.
// Rings: Q planes of three tiles (e-1, e, e+1), dO planes of two, P of two, statistics of three.
//
// B2 H32 T4096 D128 causal: 2.55 ms, matrix cores 73 % busy (at the 1.7 GHz that the power limit leaves; one wavefront
// per SIMD: 6.4 ms, 20 %).
// ---------------------------------------------------------------------------------------------
template <int D>
struct DkdvF32x : TileF32x<D> {
  using Base = TileF32x<D>;
  static constexpr int NT = 512;
  static constexpr int ROWS = 128;
  static constexpr int P_GROUP = 32 * 32 * 4;                 // P of one tile and 32 keys
  static constexpr int DO_BASE = 3 * Base::TENSOR;
  static constexpr int P_BASE = DO_BASE + 2 * Base::TENSOR;
  static constexpr int STAT_BASE = P_BASE + 2 * 4 * P_GROUP;
  static constexpr int STAT_BYTES = 2 * Base::TILE * 4;       // lse and delta of a tile's queries
  static constexpr int LDS_BYTES = STAT_BASE + 3 * STAT_BYTES;
  static constexpr int FETCH = Base::TENSOR / 4;              // bytes of a tile that a wavefront fetches
  static_assert(FETCH % 1024 == 0, "whole direct-to-LDS instructions");
  static_assert(LDS_BYTES <= 160 * 1024, "the rings fit the LDS");
};

// c += A B over the head dim: A = rows of the tile's planes, B = the lane's stationary row.  The fragments
// of the next step are read ahead of the current step's MFMAs.
template <int D>
__device__ __forceinline__ floatx16 multiply_rows(const char* planes, const TileReadOffsets<D>& off,
                                                  const bf16x8 (&mine)[D / 16][3]) {
  constexpr int KSTEPS = D / 16;
  floatx16 c;
#pragma unroll
  for (int r = 0; r < 16; r++) c[r] = 0.f;
  bf16x8 f[2][3];
  read_rows<D>(f[0], planes, off, 0);
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ks++) {
    if (ks + 1 < KSTEPS) read_rows<D>(f[(ks + 1) & 1], planes, off, ks + 1);
    __builtin_amdgcn_sched_barrier(0);
    c = mfma_split(f[ks & 1], mine[ks], c);
    __builtin_amdgcn_sched_barrier(0);
  }
  return c;
}

// acc[dt] += A B over the tile's 32 rows: A = columns 32 dt .. of the tile's planes (transposing reads),
// B = the accumulator column x, split.
template <int D>
__device__ __forceinline__ void multiply_columns(floatx16 (&acc)[D / 32], const char* planes,
                                                 const TileReadOffsets<D>& off, const floatx16& x) {
  constexpr int DT = D / 32;
  bf16x8 f[2][3], b[3];
  read_transposed<D>(f[0], planes, off, 0, 0);
#pragma unroll
  for (int n = 0; n < 2 * DT; n++) {
    if (n % DT == 0) split_column(b, x, n / DT);
    if (n + 1 < 2 * DT) read_transposed<D>(f[(n + 1) & 1], planes, off, (n + 1) / DT, (n + 1) % DT);
    __builtin_amdgcn_sched_barrier(0);
    acc[n % DT] = mfma_split(f[n & 1], b, acc[n % DT]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// SPILL (causal or sliding-window mask, q_off 0, T == S): dS is also stored, for flash_bwd_dq_ds_f32_kernel.
// AUX: with a dense bias and / or a dropout mask (the plain form has no registers to spare for their addresses).
template <int D, bool SPILL, bool AUX>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void flash_bwd_dkdv_f32x_kernel(const BwdArgs a) {
  using Tile = DkdvF32x<D>;
  constexpr int DT = D / 32, KSTEPS = D / 16;
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
  const bool p_wave = wave < 4;
  const int kg = wave & 3;                           // the wavefront's 32 keys of the workgroup's 128
  const int G = a.Hq / a.Hkv;
  const int nkb = a.S / Tile::ROWS, nkb_wg = nkb / a.kb_per_wg, npairs = a.B * a.Hkv;
  // Workgroup i runs on XCD i % 8; an XCD takes one (batch, kv head) pair after the other, so the workgroups
  // that run together read the same Q and dO rows through its L2.
  int kb0, pair;
  if (npairs % 8 == 0) {
    const int slot = blockIdx.x >> 3;
    pair = (blockIdx.x & 7) + 8 * (slot / nkb_wg);
    kb0 = slot % nkb_wg;
  } else {
    kb0 = blockIdx.x / npairs;
    pair = blockIdx.x % npairs;
  }
  const int b = pair / a.Hkv, hk = pair % a.Hkv;

  const int32_t* seg_q = a.seg ? a.seg + (int64_t)b * a.T : nullptr;
  // The P wavefronts fetch the Q planes, the dS wavefronts the dO planes, a quarter each; wavefronts 0 and 4 also
  // the tile's lse (negated, log2 units) and -delta.
  const int nqt = a.T / Tile::TILE;
  const int64_t head0 = (int64_t)b * a.stat_hq + hk * G;
  const char* const planes = (p_wave ? a.q_planes : a.do_planes) + head0 * nqt * Tile::TENSOR + kg * Tile::FETCH;
  const char* const stats = (const char*)((p_wave ? a.lse2 : a.ndelta) + head0 * a.T);
  const unsigned lds0 = lds_address(smem);

  for (int pass = 0; pass < a.kb_per_wg; pass++) {
    // With two key blocks per workgroup the second is the first one's mirror image (complementary shares of
    // the queries under a causal mask), walked the other way: see the 16-bit kernel.
    const int kb = pass == 0 ? kb0 : nkb - 1 - kb0;
    const int k0_wg = kb * Tile::ROWS, k0 = k0_wg + kg * 32;
    const int kpos = k0 + l32;

    bf16x8 mine[KSTEPS][3];   // P: the lane's K row; dS: its V row
    {
      const float* row = p_wave ? (const float*)a.k + b * a.ks.b + hk * a.ks.h + (int64_t)kpos * a.ks.s
                                : (const float*)a.v + b * a.vs.b + hk * a.vs.h + (int64_t)kpos * a.vs.s;
#pragma unroll
      for (int s = 0; s < KSTEPS; s++) {
        const float4 lo = *(const float4*)(row + 16 * s + 8 * g), hi = *(const float4*)(row + 16 * s + 8 * g + 4);
        const float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        Split3x8 sp;
        split3x8(x, sp);
#pragma unroll
        for (int p = 0; p < 3; p++) mine[s][p] = sp.part[p].v;
      }
    }

    // Query rows that can see a key of this block: qpos >= first key, qpos <= last key + window.
    int q_begin = 0, q_end = a.T;
    if (a.mask_kind != AXL_MASK_NONE) {
      q_begin = min(a.T, max(0, k0_wg - a.q_off));
      if (a.mask_kind == AXL_MASK_SLIDING_WINDOW)
        q_end = max(q_begin, (int)min((int64_t)a.T, (int64_t)k0_wg + Tile::ROWS + a.window - a.q_off));
    }
    const int t_begin = q_begin / Tile::TILE;
    const int nt = max((q_end + Tile::TILE - 1) / Tile::TILE - t_begin, 0);
    const int seg_k = a.seg ? a.seg[(int64_t)b * a.T + kpos] : 0;
    const int steps = nt * G;
    // Steps: query tile (outer; the first pass from the last one down to the diagonal, the second pass up) x
    // query head (inner), so that the workgroups of a pair walk the tiles together.
    const int dir = pass == 0 ? -1 : 1;
    const int t_first = t_begin + (dir < 0 ? max(nt - 1, 0) : 0);

    floatx16 acc[DT];         // P: dV^T, dS: dK^T
#pragma unroll
    for (int i = 0; i < DT; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][r] = 0.f;

    // Tile t of head h into ring slots i3 (Q, statistics) and i2 (dO): direct global->LDS loads.
    auto fetch = [&](int t, int h, int i3, int i2, unsigned lane16) __attribute__((always_inline)) {
      const char* src = planes + ((int64_t)h * nqt + t) * Tile::TENSOR;
      const unsigned dst = lds0 + (p_wave ? i3 * Tile::TENSOR : Tile::DO_BASE + i2 * Tile::TENSOR) + kg * Tile::FETCH;
      constexpr int N = Tile::FETCH / 1024;
#pragma unroll
      for (int i = 0; i + 1 < N; i += 2) dma16x2(lane16, lane16, src + 1024 * i, dst + 1024 * i);
      if (N % 2) dma16s(lane16, src + 1024 * (N - 1), dst + 1024 * (N - 1));
      if (kg == 0)
        dma16s_first8(lane16, stats + ((int64_t)h * a.T + t * Tile::TILE) * 4,
                      lds0 + Tile::STAT_BASE + i3 * Tile::STAT_BYTES + (p_wave ? 0 : Tile::TILE * 4));
    };
    // Does the mask leave no query of tile t any of the wavefront's keys?  Does it leave every query all of them?
    auto skipped = [&](int t) __attribute__((always_inline)) {
      const int qt0 = t * Tile::TILE + a.q_off;
      if (a.mask_kind == AXL_MASK_NONE) return false;
      return qt0 + 31 < k0 || (a.mask_kind == AXL_MASK_SLIDING_WINDOW && qt0 - (k0 + 31) > a.window);
    };
    auto is_interior = [&](int t) __attribute__((always_inline)) {
      const int qt0 = t * Tile::TILE + a.q_off;
      return a.mask_kind == AXL_MASK_NONE ||
             (qt0 >= k0 + 31 && (a.mask_kind != AXL_MASK_SLIDING_WINDOW || qt0 + 31 - k0 <= a.window));
    };
    // Slots of the rings in iteration e: Q and statistics e % 3, dO and P e % 2.
    auto q_slot = [&](int i) __attribute__((always_inline)) { return smem + i * Tile::TENSOR; };
    auto do_slot = [&](int i) __attribute__((always_inline)) { return smem + Tile::DO_BASE + i * Tile::TENSOR; };
    auto p_slot = [&](int i) __attribute__((always_inline)) { return smem + Tile::P_BASE + (4 * i + kg) * Tile::P_GROUP; };
    auto stat_slot = [&](int i) __attribute__((always_inline)) { return (float*)(smem + Tile::STAT_BASE + i * Tile::STAT_BYTES); };

    int t = t_first, h = 0;              // tile and head (of the group) of step e
    int t_prev = t_first, h_prev = 0;    // ... of step e - 1
    int s3 = 0, s3_prev = 2;             // e % 3, (e - 1) % 3
    wait_all_vmem();                     // what the compiler tracks has landed before the untracked loads
    if (steps > 0) fetch(t, h, 0, 0, 16 * lane);
    wait_all_vmem();
    __syncthreads();
    auto walk = [&](auto p_role) __attribute__((always_inline)) {
    constexpr bool P_ROLE = decltype(p_role)::value;
    floatx16 x;   // dS wavefronts: dP of step e - 1
    for (int e = 0; e <= steps && steps > 0; e++) {
      int t_nx = t, h_nx = h + 1;
      if (h_nx == G) {
        h_nx = 0;
        t_nx += dir;
      }
      const int s3_nx = s3 == 2 ? 0 : s3 + 1, s2 = e & 1;
      const bool more = e + 1 < steps;
      bool stored = false;
      // Whatever depends on the lane alone is formed anew in every step: kept, it would not fit the registers, and a
      // reload from scratch memory waits for the tile loads that were issued before it.
      int ln = lane;
      asm volatile("" : "+v"(ln));
      const int l32 = ln & 31, g = ln >> 5, kpos = k0 + l32;
      TileReadOffsets<D> off;
      off.init(ln);
      if (more) fetch(t_nx, h_nx, s3_nx, s2 ^ 1, 16 * ln);  // the round trip runs under this step's MFMAs
      if constexpr (P_ROLE) {
        if (e < steps && !skipped(t)) {
          x = multiply_rows<D>(q_slot(s3), off, mine);
          const float* lse = stat_slot(s3);                 // -lse
          const int qt0 = t * Tile::TILE;
          float4* const p_out = (float4*)p_slot(s2) + ln;
          if constexpr (AUX) {
            if (a.aux.bias) {
              const char* col = a.aux.bias + b * a.aux.bias_sb + (hk * G + h) * a.aux.bias_sh + (int64_t)(qt0 + 8 * g) * a.aux.bias_sr;
#pragma unroll
              for (int r = 0; r < 16; r++) x[r] += bias_at(a.aux, col + (16 * (r / 8) + r % 8) * a.aux.bias_sr, kpos) * kLog2e;
            }
          }
#pragma unroll
          for (int r = 0; r < 16; r++) x[r] = fast_exp2(x[r] + lse[16 * (r / 8) + 8 * g + (r % 8)]);
          if (!is_interior(t)) {
            const int diff0 = qt0 + 8 * g + a.q_off - kpos;
            const unsigned limit = a.mask_kind == AXL_MASK_SLIDING_WINDOW ? (unsigned)a.window : 0x7fffffffu;
#pragma unroll
            for (int r = 0; r < 16; r++) x[r] = (unsigned)(diff0 + 16 * (r / 8) + (r % 8)) <= limit ? x[r] : 0.f;
          }
          if (seg_q) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
              const intx4 id = *(const intx4*)(seg_q + qt0 + 16 * (i / 2) + 8 * g + 4 * (i % 2));
#pragma unroll
              for (int j = 0; j < 4; j++) x[4 * i + j] = id[j] == seg_k ? x[4 * i + j] : 0.f;
            }
          }
#pragma unroll
          for (int i = 0; i < 4; i++) {
            float4 w = {x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]};
            p_out[64 * i] = w;
          }
          if constexpr (AUX) {       // dV takes P after dropout
            if (a.aux.drop) {
              const uint8_t* col = a.aux.drop + b * a.aux.drop_sb + (hk * G + h) * a.aux.drop_sh + (int64_t)(qt0 + 8 * g) * a.aux.drop_sr + kpos;
#pragma unroll
              for (int r = 0; r < 16; r++) x[r] = col[(16 * (r / 8) + r % 8) * a.aux.drop_sr] ? 0.f : x[r] * a.aux.keep_scale;
            }
          }
          multiply_columns<D>(acc, do_slot(s2), off, x);
        }
      } else {
        if (e > 0 && !skipped(t_prev)) {
          const float* delta = stat_slot(s3_prev) + Tile::TILE;   // -delta
          const float4* const p_in = (const float4*)p_slot(s2 ^ 1) + ln;
          if constexpr (AUX) {
            if (a.aux.drop) {
              const uint8_t* col = a.aux.drop + b * a.aux.drop_sb + (hk * G + h_prev) * a.aux.drop_sh + (int64_t)(t_prev * Tile::TILE + 8 * g) * a.aux.drop_sr + kpos;
#pragma unroll
              for (int r = 0; r < 16; r++) x[r] = col[(16 * (r / 8) + r % 8) * a.aux.drop_sr] ? 0.f : x[r] * a.aux.keep_scale;
            }
          }
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const float4 p = p_in[64 * i];
            const float* dl = delta + 16 * (i / 2) + 8 * g + 4 * (i % 2);
            x[4 * i + 0] = p.x * (x[4 * i + 0] + dl[0]);  // dS
            x[4 * i + 1] = p.y * (x[4 * i + 1] + dl[1]);
            x[4 * i + 2] = p.z * (x[4 * i + 2] + dl[2]);
            x[4 * i + 3] = p.w * (x[4 * i + 3] + dl[3]);
          }
          if constexpr (SPILL) {
            // the block of (query tile, 32 keys): quad i of lane (key, g) at 16-byte slot 64 i + 32 g + (key ^ (2 i + g))
            const char* const blk = (const char*)a.ds +
                (ds32_run_start(pair, a.T, G, t_prev, h_prev) + 4 * kb + kg) * (kDs32BlockElems * 4);
#pragma unroll
            for (int i = 0; i < 4; i++) {
              const floatx4 w = {x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]};
              store16_stream(16u * (32 * g + (l32 ^ (2 * i + g))), blk + 1024 * i, w);
            }
            stored = true;
          }
          multiply_columns<D>(acc, q_slot(s3_prev), off, x);
        }
        if (e < steps && !skipped(t)) x = multiply_rows<D>(do_slot(s2), off, mine);
      }
      // The next tile has landed; the four dS stores went out after its loads.
      if (SPILL && stored) wait_vmem_le<4>();
      else wait_all_vmem();
      __syncthreads();
      t_prev = t; h_prev = h; s3_prev = s3;
      t = t_nx; h = h_nx; s3 = s3_nx;
    }
    };
    // Two copies of the loop, one per kind of wavefront; both meet at every barrier.
    if (p_wave) walk(std::true_type{});
    else walk(std::false_type{});

    float* out = p_wave ? (float*)a.dv + b * a.dvs.b + (int64_t)kpos * a.dvs.s + hk * a.dvs.h
                        : (float*)a.dk + b * a.dks.b + (int64_t)kpos * a.dks.s + hk * a.dks.h;
    const float mult = p_wave ? 1.f : 1.f / kLog2e;   // the Q planes carry scale * log2(e)
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int rq = 0; rq < 4; rq++) {
        float4 w = {acc[dt][4 * rq + 0] * mult, acc[dt][4 * rq + 1] * mult, acc[dt][4 * rq + 2] * mult,
                    acc[dt][4 * rq + 3] * mult};
        *(float4*)(out + 32 * dt + 8 * rq + 4 * g) = w;
      }
  }
}

// ---------------------------------------------------------------------------------------------
// dQ from stored dS: dQ^T[d][q] += K^T[d][key] dS^T[key][q], one product instead of the three of the
// recomputing kernel (axlearn/common/flash_attention/gpu_attention.py:533-616).  A workgroup of 8 wavefronts
// owns 256 queries of one head, 32 per wavefront (one query tile), and walks 32-key tiles: the K tile, split
// by all threads, in two LDS buffers; every wavefront's own 4 KB block of dS through 4 KB of LDS of its own,
// which turns it around (stored with a lane per key, needed with a lane per query; the slot exchange of the
// store keeps the reads free of bank conflicts).  K rows and dS blocks travel through registers, requested
// two tiles ahead.  Bound by the matrix cores (six bf16 products per pair and
// element of d) with dS read from HBM once, 4 bytes per visible pair.
//
// B2 H32 T4096 D128 causal: 0.94 ms, matrix cores 53 % busy (recomputing S and dP: 4.3 ms).
// ---------------------------------------------------------------------------------------------
template <int D>
struct DqDsF32 : TileF32x<D> {
  using Base = TileF32x<D>;
  static constexpr int NT = 512;
  static constexpr int TILES = 8;                      // query tiles of a workgroup
  static constexpr int DS_BASE = 2 * Base::TENSOR;
  static constexpr int LDS_BYTES = DS_BASE + TILES * kDs32BlockElems * 4;
  static constexpr int LD4 = Base::LD4(NT);
};

template <int D>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void flash_bwd_dq_ds_f32_kernel(const BwdArgs a) {
  using Tile = DqDsF32<D>;
  constexpr int DT = D / 32;
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
  const int nqt = a.T / Tile::TILE, nqb = (nqt + Tile::TILES - 1) / Tile::TILES;
  int qb, b, h;
  decode_block(blockIdx.x, nqb, a.B, a.Hq, a.Hkv, 32, qb, b, h);
  const int G = a.Hq / a.Hkv, hk = h / G;
  // Query tile of this wavefront (none past the end) and the key tiles [first, last] it has dS for: those of
  // which it sees a key.  The workgroup walks from its first wavefront's first to its last one's last.
  const int t_q = qb * Tile::TILES + wave;
  auto first_key_tile = [&](int t) __attribute__((always_inline)) {
    return a.mask_kind == AXL_MASK_SLIDING_WINDOW ? max(0, (int)(((int64_t)32 * t - a.window) / 32)) : 0;
  };
  const int first = first_key_tile(t_q), last = t_q < nqt ? t_q : -1;
  const int t_begin = first_key_tile(qb * Tile::TILES), t_end = min(nqt, (qb + 1) * Tile::TILES);

  TileReadOffsets<D> off;
  off.init(lane);
  floatx16 acc[DT];
#pragma unroll
  for (int i = 0; i < DT; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[i][r] = 0.f;

  const int st_row = tid / (D / 4), st_c4 = tid % (D / 4);
  constexpr int ROW_STEP = Tile::NT / (D / 4);
  const float* const k_thread = (const float*)a.k + b * a.ks.b + hk * a.ks.h + (int64_t)st_row * a.ks.s + st_c4 * 4;
  const float* const ds_lane = (const float*)a.ds + 4 * lane +
      ds32_run_start((int64_t)b * a.Hkv + hk, a.T, G, min(t_q, nqt - 1), h - hk * G) * kDs32BlockElems;
  float* const ds_own = (float*)(smem + Tile::DS_BASE) + wave * kDs32BlockElems;
  // Element (query q, key k) of a block: quad i = 2 (q / 16) + q % 8 / 4 of lane (k, q / 8 % 2), element q % 4.
  const int qq = 2 * (l32 >> 4) + ((l32 >> 2) & 1), qg = (l32 >> 3) & 1;
  const float* const ds_q = ds_own + 4 * (64 * qq + 32 * qg) + (l32 & 3);
  const int ds_xor = 2 * qq + qg;

  float4 kx[Tile::LD4];
  floatx4 dsx[4];
  auto request = [&](int t) __attribute__((always_inline)) {
    const float* kp = k_thread + (int64_t)t * Tile::TILE * a.ks.s;
#pragma unroll
    for (int i = 0; i < Tile::LD4; i++) kx[i] = *(const float4*)(kp + i * ROW_STEP * a.ks.s);
    if (t >= first && t <= last) {
#pragma unroll
      for (int i = 0; i < 4; i++)
        dsx[i] = __builtin_nontemporal_load((const floatx4*)(ds_lane + (int64_t)t * kDs32BlockElems + 256 * i));
    }
  };
  auto deposit = [&](int t) __attribute__((always_inline)) {
    tile_deposit_split<D, Tile::NT>(smem + (t & 1) * Tile::TENSOR, kx, tid);
    if (t >= first && t <= last) {
#pragma unroll
      for (int i = 0; i < 4; i++) *(floatx4*)(ds_own + 4 * lane + 256 * i) = dsx[i];
    }
  };
  request(t_begin);
  deposit(t_begin);
  if (t_begin + 1 < t_end) request(t_begin + 1);
  __syncthreads();
  for (int t = t_begin; t < t_end; t++) {
    const bool mine = t >= first && t <= last, more = t + 1 < t_end;
    floatx16 x;                // register 8 kk + j: key 16 kk + 8 g + j
    if (mine) {
#pragma unroll
      for (int r = 0; r < 16; r++) x[r] = ds_q[4 * ((16 * (r / 8) + 8 * g + (r % 8)) ^ ds_xor)];
    }
    // Tile t + 1 from registers into LDS (the other K buffer was last read a tile ago; the dS block is the
    // wavefront's own and has just been read), tile t + 2 on its way: of the two wavefronts of a SIMD one does it
    // ahead of its MFMAs and the other behind them, so that it falls on the other one's MFMAs.
    auto advance = [&]() __attribute__((always_inline)) {
      if (more) deposit(t + 1);
      if (t + 2 < t_end) request(t + 2);
    };
    if (wave >= 4) advance();
    if (mine) multiply_columns<D>(acc, smem + (t & 1) * Tile::TENSOR, off, x);
    if (wave < 4) advance();
    __syncthreads();
  }

  if (t_q < nqt) {
    float* dqp = (float*)a.dq + b * a.dqs.b + (int64_t)(t_q * Tile::TILE + l32) * a.dqs.s + h * a.dqs.h;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int rq = 0; rq < 4; rq++) {
        float4 w = {acc[dt][4 * rq + 0] * a.scale, acc[dt][4 * rq + 1] * a.scale, acc[dt][4 * rq + 2] * a.scale,
                    acc[dt][4 * rq + 3] * a.scale};
        *(float4*)(dqp + 32 * dt + 8 * rq + 4 * g) = w;
      }
  }
}

// The 32 x D tiles of Q (times scale * log2(e), the forward's own product, so that both round alike) and dO as three bf16 planes each, as the dK/dV kernel keeps them in LDS (its loads are
// then plain copies that need neither registers nor arithmetic; every tile is read by all workgroups of a
// pair).  [B, Hq, T / 32] tiles; one workgroup per tile and tensor.  Bound by HBM: 10 bytes per
// element; 0.11 ms for 2 x 134 MB of fp32.
template <int D>
__global__ __launch_bounds__(256) void split_planes_kernel(const BwdArgs a) {
  using Tile = TileF32x<D>;
  const int nqt = a.T / Tile::TILE;
  const int64_t tile = blockIdx.x;                         // (b Hq + h) nqt + t
  const int t = (int)(tile % nqt);
  const int64_t bh = tile / nqt;
  const int h = (int)(bh % a.Hq), b = (int)(bh / a.Hq);
  const bool is_q = blockIdx.y == 0;
  const Strides3 st = is_q ? a.qs : a.dos;
  const float* src = (const float*)(is_q ? a.q : a.dout) + b * st.b + h * st.h + (int64_t)t * Tile::TILE * st.s;
  const float mult = is_q ? a.scale * kLog2e : 1.f;
  char* dst = const_cast<char*>(is_q ? a.q_planes : a.do_planes) + tile * Tile::TENSOR;
#pragma unroll
  for (int i = 0; i < Tile::TILE * (D / 8) / 256; i++) {
    const int e = threadIdx.x + 256 * i, row = e / (D / 8), c = e % (D / 8);
    const float4 lo = *(const float4*)(src + row * st.s + c * 8), hi = *(const float4*)(src + row * st.s + c * 8 + 4);
    const float x[8] = {lo.x * mult, lo.y * mult, lo.z * mult, lo.w * mult,
                        hi.x * mult, hi.y * mult, hi.z * mult, hi.w * mult};
    Split3x8 sp;
    split3x8(x, sp);
#pragma unroll
    for (int p = 0; p < 3; p++)
      *(bf16x8*)(dst + p * Tile::PLANE + row * Tile::STRIDE + ((c ^ tile_swizzle<D>(row)) << 4)) = sp.part[p].v;
  }
}

template <int D>
static hipError_t launch_split(const BwdArgs& a, hipStream_t stream) {
  hipLaunchKernelGGL(split_planes_kernel<D>, dim3(a.B * a.Hq * (a.T / TileF32x<D>::TILE), 2), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_bwd_split_f32x(const BwdArgs& a, int head_dim, hipStream_t stream) {
  return head_dim == 128 ? launch_split<128>(a, stream) : launch_split<64>(a, stream);
}

template <int D>
static hipError_t launch_dkdv(const BwdArgs& a, hipStream_t stream) {
  using Tile = DkdvF32x<D>;
  const bool aux = a.aux.bias || a.aux.drop;
  auto kernel = a.ds ? (aux ? flash_bwd_dkdv_f32x_kernel<D, true, true> : flash_bwd_dkdv_f32x_kernel<D, true, false>)
                     : (aux ? flash_bwd_dkdv_f32x_kernel<D, false, true> : flash_bwd_dkdv_f32x_kernel<D, false, false>);
  const hipError_t err = allow_dynamic_lds((const void*)kernel, Tile::LDS_BYTES);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(kernel, dim3((a.S / Tile::ROWS) * a.B * a.Hkv / a.kb_per_wg), dim3(Tile::NT), Tile::LDS_BYTES, stream, a);
  return hipGetLastError();
}

hipError_t launch_bwd_dkdv_f32x(const BwdArgs& a, int head_dim, hipStream_t stream) {
  return head_dim == 128 ? launch_dkdv<128>(a, stream) : launch_dkdv<64>(a, stream);
}

template <int D>
static hipError_t launch_dq_ds(const BwdArgs& a, hipStream_t stream) {
  using Tile = DqDsF32<D>;
  auto kernel = flash_bwd_dq_ds_f32_kernel<D>;
  const hipError_t err = allow_dynamic_lds((const void*)kernel, Tile::LDS_BYTES);
  if (err != hipSuccess) return err;
  const int nqb = (a.T / Tile::TILE + Tile::TILES - 1) / Tile::TILES;
  hipLaunchKernelGGL(kernel, dim3(nqb * a.B * a.Hq), dim3(Tile::NT), Tile::LDS_BYTES, stream, a);
  return hipGetLastError();
}

hipError_t launch_bwd_dq_ds_f32(const BwdArgs& a, int head_dim, hipStream_t stream) {
  return head_dim == 128 ? launch_dq_ds<128>(a, stream) : launch_dq_ds<64>(a, stream);
}

}  // namespace axl
