// MoBA prefill backward on gfx950 (deterministic, no atomics).
//
// Replaces OptMixedAttention.backward (src/moba_opt/mixed_attention.py:141-225):
// the self-branch and remote-branch flash-attention backwards, both evaluated
// with the GLOBAL output O and GLOBAL LSE of the merged forward
// (docs/semantics.md section 7), plus the autograd scatter of the packed
// remote dq/dkv back into q/k/v (grouped_attention.py:81-89), which is where
// GQA gradients of the heads sharing a KV head are summed.
//
//   delta_kernel : Delta = rowsum(dO * O)                                  [T*Hq]
//   dq_kernel<REMOTE> (dq2_kernel above 128 dims, self above 192) : query-major.  S^T = K Q^T, dP^T = V dO^T,
//        P = exp(S*scale - LSE), dS = P (dP - Delta), dQ^T += K^T dS^T.
//        REMOTE tiles (expert rows) write dq partials into the row's slot;
//        SELF tiles (causal within the chunk) add the slots in ascending order.
//   dK / dV (attn_dkdv*.hip): key-major.  One workgroup owns a tile of one chunk's keys for
//        one KV head and walks every query row that attends them: the causal
//        rows of the chunk for all G heads of the group, then the expert rows
//        that selected the chunk.  dK, dV accumulate in registers and are
//        written once.
#include <type_traits>

#include "common.h"
#include "bwd_args.h"
#include "../../include/moba_hip.h"

using namespace moba;

namespace {


constexpr int kBN = 64;   // dq: keys per LDS tile

// ------------------------------------------------------------------ delta
// 16 lanes per row, `row` the same for the 16.
template <int DT>
__device__ __forceinline__ void delta_row(const uint16_t* __restrict__ o,
                                          const uint16_t* __restrict__ g,
                                          const float* __restrict__ lse, int64_t row, int64_t rows,
                                          int D, float* __restrict__ delta, float scale,
                                          float* __restrict__ lse_k) {
  const int sub = threadIdx.x & 15;
  float acc = 0.0f;
  if (row < rows) {
    for (int d = sub * 8; d < D; d += 128) {
      const u16x8_t x = ld8(o + row * D + d), y = ld8(g + row * D + d);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc += to_f32<DT>(x[e]) * to_f32<DT>(y[e]);
    }
  }
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 16);
  if (row < rows && sub == 0) {
    delta[row] = acc;
    lse_k[row] = lse[row] / scale;
  }
}

template <int DT>
__global__ __launch_bounds__(256) void delta_kernel(const uint16_t* __restrict__ o,
                                                    const uint16_t* __restrict__ g,
                                                    const float* __restrict__ lse, int64_t rows,
                                                    int D, float* __restrict__ delta,
                                                    float scale, float* __restrict__ lse_k) {
  delta_row<DT>(o, g, lse, (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4), rows, D, delta, scale,
                lse_k);
}

// --------------------------------------------------------------------- dq
// Epilogue of one row.  Remote: dQ partial of the row's slot.  Self: the slots
// are added in ascending order; one slot per iteration, its loads issued
// together: slots below R are in the row's allocation, columns past D are
// clamped (they reach only entries that are not stored), unselected slots
// (sel < 0) add zero.
template <int DT, int DP, bool REMOTE>
__device__ __forceinline__ void finish_row(const BwdArgs& a, f32x16_t (&acc)[DP / 32], int64_t row,
                                           int slot, int hh) {
  constexpr int NDB = DP / 32;
  const int D = a.D;
  if constexpr (REMOTE) {
    uint16_t* po = a.part_dq + (int64_t)slot * D;
#pragma unroll
    for (int db = 0; db < NDB; ++db) store_block<DT>(po, acc[db], a.scale, db, 8 * hh, D);
  } else {
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[db][r] *= a.scale;
    for (int jj = 0; jj < a.R; ++jj) {
      const int64_t sl = row * a.R + jj;
      const bool on = a.sel[sl] >= 0;
      const uint16_t* po = a.part_dq + sl * D;
      constexpr int NBL = NDB <= 4 ? NDB : 2;
#pragma unroll
      for (int d4 = 0; d4 < NDB; d4 += NBL) {
        u16x8_t o[NBL][2];
#pragma unroll
        for (int db = 0; db < NBL; ++db)
#pragma unroll
          for (int m = 0; m < 2; ++m) {
            const int d = (d4 + db) * 32 + 16 * m + 8 * hh;
            o[db][m] = ld8(po + (d < D ? d : 0));
          }
#pragma unroll
        for (int db = 0; db < NBL; ++db)
#pragma unroll
          for (int m = 0; m < 2; ++m) {
            float x[8];
            spread_piece<DT>(o[db][m], x);
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[d4 + db][8 * m + i] += on ? x[i] : 0.0f;
          }
      }
    }
    uint16_t* orow = a.dq + row * D;
#pragma unroll
    for (int db = 0; db < NDB; ++db) store_block<DT>(orow, acc[db], 1.0f, db, 8 * hh, D);
  }
}

// Head dims up to 128, and the self launch up to 192 (dq2_kernel has the others).
// Per wave QB blocks of 32 query rows; K/V tiles of 64 keys double-buffered in
// LDS (row-major).  S^T = K Q^T and dP^T = V dO^T take K / V rows as the A
// operand; dQ^T = K^T dS^T reads K^T with the transposed LDS read.
template <int DT, int DP, bool REMOTE, int QB>
__global__ __launch_bounds__(256, attn_occupancy<DP>()) void dq_kernel(BwdArgs a) {
  constexpr int NKS = DP / 16, NDB = DP / 32;
  constexpr int TILE = kBN * DP, NB = DP / 8, NDMA = kBN * NB / 256;
  static_assert(DP <= 128 || !REMOTE, "dq2_kernel has the remote launch of the wide heads");
  // Two stages of K and V tiles (swz<DP> layout) filled by buffer loads
  // straight into LDS, as in the forward kernel.
  __shared__ __attribute__((aligned(16))) uint16_t K0[TILE];
  __shared__ __attribute__((aligned(16))) uint16_t V0[TILE];
  __shared__ __attribute__((aligned(16))) uint16_t K1[TILE];
  __shared__ __attribute__((aligned(16))) uint16_t V1[TILE];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int qi = lane & 31, hh = lane >> 5;
  const int D = a.D;

  int s[QB], h[QB], slot[QB];
  int pidx[QB];  // packed index of an expert row (row_off order)
  int packed[QB];
  bool valid[QB];
  int kh, k_lo, k_hi, s_wave0 = 0;
  if constexpr (REMOTE) {
    const ExpertTile x = expert_tile<128 * QB>(a);
    if (x.rows == 0) return;
    kh = x.kh;
    k_lo = x.k_lo;
    k_hi = x.k_hi;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      const int local = wave * (32 * QB) + qb * 32 + qi;
      valid[qb] = local < x.rows;
      pidx[qb] = x.row0 + local;
      packed[qb] = a.rows[x.row0 + min(local, x.rows - 1)];  // (row << 3) | j
    }
  } else {
    // 1-D grid over (tile, q head within the kv group), tiles in the
    // host's order of 8 XCD runs: workgroup L runs on XCD L % 8 and takes
    // entry xcd_contiguous(L) / G, so each run's tiles share that XCD's L2.
    // Entries are (chunk, first row, kv head); chunk -1 pads a run.
    const int t = xcd_contiguous(blockIdx.x, a.n_self_wg);
    if (t < 0) return;
    const int e = t / a.G, g = t - e * a.G;
    const int c = a.self_tiles[3 * e];
    if (c < 0) return;
    const int row0 = a.self_tiles[3 * e + 1];
    kh = a.self_tiles[3 * e + 2];
    k_lo = a.cu_chunk[c];
    const int c_end = a.cu_chunk[c + 1];
    k_hi = min(c_end, k_lo + row0 + 128 * QB);
    s_wave0 = k_lo + row0 + wave * (32 * QB);
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      h[qb] = kh * a.G + g;
      slot[qb] = 0;
      s[qb] = s_wave0 + qb * 32 + qi;
      valid[qb] = s[qb] < c_end;
      if (!valid[qb]) s[qb] = k_hi - 1;
    }
  }
  const int wave_s = __builtin_amdgcn_readfirstlane(wave);
  // Lane l of wave w loads blocks j = (n * 4 + w) * 64 + l: row j / NB,
  // physical block j % NB.  The row advances by 256 / NB per n, a multiple of
  // 16 up to 128 dims, and the swizzle depends on the row mod 16 only, so every n
  // has the same column and its offset is the n = 0 offset plus a uniform step
  // (added per load, not held in NDMA registers).
  constexpr bool UNI = (256 / NB) % 16 == 0;
  uint32_t voff[UNI ? 1 : NDMA];
  bool vok[UNI ? 1 : NDMA];
#pragma unroll
  for (int n = 0; n < (UNI ? 1 : NDMA); ++n) {
    const int j = (n * 4 + wave_s) * 64 + lane, row = j / NB;
    const int col = swz<DP>(row, (j % NB) * 8) - row * DP;  // swizzle is an involution
    voff[n] = (uint32_t)(((row * a.Hkv + kh) * D + col) * 2);
    vok[n] = col < D;
  }
  const uint32_t vstep = (uint32_t)((256 / NB) * a.Hkv * D * 2);
  const int n_keys = k_hi - k_lo;
  const uint32_t nrec = (uint32_t)((((int64_t)(n_keys - 1) * a.Hkv + kh + 1) * D) * 2);
  const uint16_t* kbase = a.k + (int64_t)k_lo * a.Hkv * D;
  const uint16_t* vbase = a.v + (int64_t)k_lo * a.Hkv * D;
  const uint32_t tile_bytes = (uint32_t)(kBN * a.Hkv * D * 2);
  auto dma = [&](uint16_t* Kd, uint16_t* Vd, int it) {
    const uint32_t soff = (uint32_t)it * tile_bytes;
    const uint32_t v0 = opaque(voff[0]);
#pragma unroll
    for (int n = 0; n < NDMA; ++n) {
      if (vok[UNI ? 0 : n]) {
        const uint32_t vo = UNI ? v0 + n * vstep : voff[n];
        load_lds16(make_rsrc(kbase, nrec), Kd + (n * 4 + wave_s) * 64 * 8, vo, soff);
        load_lds16(make_rsrc(vbase, nrec), Vd + (n * 4 + wave_s) * 64 * 8, vo, soff);
      }
    }
  };
  if (D < DP) {  // column blocks past D stay zero
#pragma unroll
    for (int n = 0; n < NDMA; ++n) {
      const int j = (n * 4 + wave) * 64 + lane;
      st8(K0 + j * 8, zero8()); st8(V0 + j * 8, zero8());
      st8(K1 + j * 8, zero8()); st8(V1 + j * 8, zero8());
    }
    __syncthreads();
  }
  // The first K / V tile goes out before the query rows: an expert's rows
  // wait for their row list, the tile only for the workgroup's entry (above 128
  // dims the rows come first and each load is guarded: otherwise the kernel
  // spills 325 registers).  Rows past the tile's end load the last row's data
  // and are never written.
  constexpr bool TILE_FIRST = DP <= 128;
  if constexpr (TILE_FIRST) dma(K0, V0, 0);
  u16x8_t qf[QB][NKS], gf[QB][NKS];
  float lse2[QB], lk[QB], dl[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    if constexpr (REMOTE) {
      const int sh = packed[qb] >> 3;
      slot[qb] = sh * a.R + (packed[qb] & 7);
      s[qb] = sh / a.Hq;
      h[qb] = sh % a.Hq;
    }
    const int64_t row = (int64_t)s[qb] * a.Hq + h[qb];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const int d = ks * 16 + hh * 8, dc = d < D ? d : 0;
      if constexpr (TILE_FIRST) {
        const u16x8_t xq = ld8(a.q + row * D + dc), xg = ld8(a.dout + row * D + dc);
        qf[qb][ks] = d < D ? xq : zero8();
        gf[qb][ks] = d < D ? xg : zero8();
      } else {
        qf[qb][ks] = valid[qb] && d < D ? ld8(a.q + row * D + d) : zero8();
        gf[qb][ks] = valid[qb] && d < D ? ld8(a.dout + row * D + d) : zero8();
      }
    }
    const float lr = a.lse[row];
    lse2[qb] = lr * kLog2e;
    lk[qb] = lr / a.scale;
    dl[qb] = a.delta[row];
  }
  if constexpr (REMOTE) {
    // The key-major dK/dV kernel reads the expert rows packed contiguously in
    // row_off order; this kernel holds exactly those rows, so it writes the
    // packed q / dO / lse_k / delta (the values delta_kernel and the loads above
    // produce) instead of a separate gather pass.
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      if (!valid[qb]) continue;
      const int64_t m = pidx[qb];
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        const int d = ks * 16 + hh * 8;
        if (d < D) {
          st8(a.pack_q + m * D + d, qf[qb][ks]);
          st8(a.pack_g + m * D + d, gf[qb][ks]);
        }
      }
      if (hh == 0) {
        a.pack_lse_k[m] = lk[qb];
        a.pack_delta[m] = dl[qb];
      }
    }
  }

  if constexpr (!TILE_FIRST) dma(K0, V0, 0);
  const uint32_t kbase0 = swz_b128_base<DP>(lane);
  const uint32_t trb0 = swz_tr_base<DP>(lane, 0), trb1 = swz_tr_base<DP>(lane, 1);

  f32x16_t acc[QB][NDB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int db = 0; db < NDB; ++db) acc[qb][db] = zero16();
  const float c2 = a.scale_log2;

  const int ntiles = (n_keys + kBN - 1) / kBN;
  auto tile = [&](const uint16_t* Kb, const uint16_t* Vb, const int it, auto mask_tag) {
    constexpr bool MASK = decltype(mask_tag)::value;
    const int kt0 = k_lo + it * kBN;
    const uint32_t kq = opaque(kbase0), t0 = opaque(trb0), t1 = opaque(trb1);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      f32x16_t sa[QB], pa[QB];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) { sa[qb] = zero16(); pa[qb] = zero16(); }
      wave_prio<1>();
      if constexpr (REMOTE && DP > 64) {
        // the expert variant holds more per-row state: above D = 64 no room
        // for a ring (it spills); at D <= 64 it takes the ring path below
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
          const uint32_t o = kb * 32 * DP * 2 + swz_b128<DP>(kq, ks);
          const u16x8_t ka = lds8(Kb, o), va = lds8(Vb, o);
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) {
            sa[qb] = mfma32<DT>(ka, qf[qb][ks], sa[qb]);
            pa[qb] = mfma32<DT>(va, gf[qb][ks], pa[qb]);
          }
        }
      } else {
        // K / V operand reads run PF k-steps ahead of the MFMAs, in this
        // order (the scheduling fences keep the compiler from sinking them)
        constexpr int PF = 3;
        u16x8_t rk[PF], rv[PF];
#pragma unroll
        for (int i = 0; i < PF && i < NKS; ++i) {
          const uint32_t o = kb * 32 * DP * 2 + swz_b128<DP>(kq, i);
          rk[i] = lds8(Kb, o);
          rv[i] = lds8(Vb, o);
        }
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
          const u16x8_t ka = rk[ks % PF], va = rv[ks % PF];
          if (ks + PF < NKS) {
            const uint32_t o = kb * 32 * DP * 2 + swz_b128<DP>(kq, ks + PF);
            rk[ks % PF] = lds8(Kb, o);
            rv[ks % PF] = lds8(Vb, o);
          }
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) {
            sa[qb] = mfma32<DT>(ka, qf[qb][ks], sa[qb]);
            pa[qb] = mfma32<DT>(va, gf[qb][ks], pa[qb]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      wave_prio<0>();
      u16x8_t dsv[QB][2];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        float tmp[16];
        const float nl = -lse2[qb];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float p = fast_exp2(fmaf(sa[qb][r], c2, nl));
          if constexpr (MASK) {
            const int key = kt0 + kb * 32 + 8 * (r >> 2) + 4 * hh + (r & 3);
            p = (key < k_hi && (REMOTE || key <= s[qb])) ? p : 0.0f;
          }
          tmp[r] = p * (pa[qb][r] - dl[qb]);
        }
        dsv[qb][0] = pack8<DT>(tmp);
        dsv[qb][1] = pack8<DT>(tmp + 8);
      }
      wave_prio<1>();
      if constexpr (REMOTE && DP > 64) {
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const uint32_t ro = (kb * 32 + t * 16) * DP * 2;
            const u16x8_t kt = lds_tr8(Kb, ro + swz_tr<DP>(t0, db), ro + swz_tr<DP>(t1, db));
#pragma unroll
            for (int qb = 0; qb < QB; ++qb) acc[qb][db] = mfma32<DT>(kt, dsv[qb][t], acc[qb][db]);
          }
        // issue order for this 32-key block: LDS operand reads run at most
        // two MFMAs ahead, which bounds the registers they hold
        if constexpr (QB == 1) {
          __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
          for (int i = 0; i < NKS - 2; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
          }
          __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 200, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
          for (int i = 0; i < 2 * NDB - 2; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
          }
          __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        }
      } else {
        // K^T operand reads pipelined the same way; step i is d block i / 2
        // of 16-key half i % 2
        constexpr int N2 = 2 * NDB, PF = 4;
        u16x8_t ring[PF];
        auto rd = [&](int i) __attribute__((always_inline)) {
          const uint32_t ro = (kb * 32 + (i % 2) * 16) * DP * 2;
          return lds_tr8(Kb, ro + swz_tr<DP>(t0, i / 2), ro + swz_tr<DP>(t1, i / 2));
        };
#pragma unroll
        for (int i = 0; i < PF && i < N2; ++i) ring[i] = rd(i);
#pragma unroll
        for (int i = 0; i < N2; ++i) {
          const u16x8_t kt = ring[i % PF];
          if (i + PF < N2) ring[i % PF] = rd(i + PF);
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) acc[qb][i / 2] = mfma32<DT>(kt, dsv[qb][i % 2], acc[qb][i / 2]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto stage_sync = [&]() {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's tile loads landed
    __builtin_amdgcn_s_barrier();
  };
  auto run = [&](const uint16_t* Kb, const uint16_t* Vb, int it) {
    const int kt0 = k_lo + it * kBN;
    // a causal tile wholly above this wave's rows adds exact zeros: skip it
    // (the wave still joins the stage barriers)
    if (!REMOTE && kt0 > s_wave0 + 32 * QB - 1) return;
    const bool need_mask = (kt0 + kBN > k_hi) || (!REMOTE && kt0 + kBN - 1 > s_wave0);
    if (need_mask) tile(Kb, Vb, it, std::true_type{}); else tile(Kb, Vb, it, std::false_type{});
  };
  stage_sync();
  for (int it = 0; it < ntiles; it += 2) {
    if (it + 1 < ntiles) dma(K1, V1, it + 1);
    run(K0, V0, it);
    stage_sync();
    if (it + 1 >= ntiles) break;
    if (it + 2 < ntiles) dma(K0, V0, it + 2);
    run(K1, V1, it + 1);
    stage_sync();
  }

#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
    if (valid[qb])
      finish_row<DT, DP, REMOTE>(a, acc[qb], (int64_t)s[qb] * a.Hq + h[qb], slot[qb], hh);
}

// --------------------------------------------- dq, head dims 129..256
// The same work and tiles of 128 rows, by 4 wave pairs of 32 rows.  Here Q, dO
// and dQ of 32 rows take 256 registers: one wave that holds all three has them
// in both register files and moves operands between these for most MFMAs, alone
// on its SIMD.  So a pair shares a SIMD and splits the products, over blocks of
// 32 keys.  At step t:
//   role S (Q, dO):  S^T = K_t Q^T, dP^T = V_t dO^T, dS_t to LDS (the operand
//                    as its lane holds it: 2 KB per pair)
//   role G (dQ):     dQ^T += K_{t-1}^T dS_{t-1}
// Role S goes first (s_setprio): role G's MFMAs run under its element-wise
// work.  K has 4 stages and V 3 (t - 1, t, and two blocks of loads in flight);
// one barrier a step.  The sums are those of dq_kernel, in its order.
// T 8192, 16/4 heads, chunk 1024, top-3, D 256: remote 570 -> 425-454 us, the
// training step 1780 -> 1681 us; matrix units busy 39% of the cycles, LDS 22%
// with no bank conflicts.  The self launch (above 192 dims; matrix units
// 24%, LDS 14%) gains over one wave per 32 rows where a few long tiles decide and
// loses where many tiles fill the CUs: full causal attention, D 256, delta and
// dQ, us: 4096 tokens, 8 heads 185 -> 168, 32768, 4 heads 3713 -> 3560, 8192,
// 16/4 heads 873 -> 877, 8 x 1024 169.5 -> 172, 16 x 512 130 -> 134.  2 to 5
// (role S) or 4 to 8 (role G) operand reads in flight and no priority measure
// the same, role G first 8% slower; the element-wise work of block t - 1 between
// role S's MFMAs of block t (two S^T and dP^T in registers, five K stages) is
// 2% slower.
constexpr int kBK = 32;  // keys per block

template <int DT, int DP, bool REMOTE>
__global__ __launch_bounds__(512, 2) void dq2_kernel(BwdArgs a) {
  constexpr int NKS = DP / 16, NDB = DP / 32, NB = DP / 8;
  constexpr int TILE = kBK * DP, NDMA = kBK * NB / 512;
  constexpr int NSK = 4, NSV = 3;
  __shared__ __attribute__((aligned(16))) uint16_t Ks[NSK * TILE];
  __shared__ __attribute__((aligned(16))) uint16_t Vs[NSV * TILE];
  __shared__ __attribute__((aligned(16))) u16x8_t Ds[2][4][2][64];  // dS of block & 1, per pair

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pair = wave & 3, qi = lane & 31, hh = lane >> 5;
  const int D = a.D;
  int s, h, slot = 0, kh, k_lo, k_hi, s_wave0 = 0;
  bool valid;
  if constexpr (REMOTE) {
    const ExpertTile x = expert_tile<128>(a);
    if (x.rows == 0) return;
    kh = x.kh;
    k_lo = x.k_lo;
    k_hi = x.k_hi;
    const int local = pair * 32 + qi;
    valid = local < x.rows;
    const int packed = a.rows[x.row0 + min(local, x.rows - 1)];  // (row << 3) | j
    slot = (packed >> 3) * a.R + (packed & 7);
    s = (packed >> 3) / a.Hq;
    h = (packed >> 3) % a.Hq;
  } else {
    const int t = xcd_contiguous(blockIdx.x, a.n_self_wg);
    if (t < 0) return;
    const int e = t / a.G, g = t - e * a.G;
    const int c = a.self_tiles[3 * e];
    if (c < 0) return;
    const int row0 = a.self_tiles[3 * e + 1];
    kh = a.self_tiles[3 * e + 2];
    k_lo = a.cu_chunk[c];
    const int c_end = a.cu_chunk[c + 1];
    k_hi = min(c_end, k_lo + row0 + 128);
    s_wave0 = k_lo + row0 + pair * 32;
    h = kh * a.G + g;
    s = s_wave0 + qi;
    valid = s < c_end;
    if (!valid) s = k_hi - 1;
  }
  const int64_t row = (int64_t)s * a.Hq + h;

  // Thread t loads 16-byte blocks n * 512 + t of a tile.  Columns past D and
  // keys past the end read past num_records, i.e. zeros; a block past the last
  // loads zeros into a stage nobody reads, so every block is 2 * NDMA loads.
  const int n_keys = k_hi - k_lo, nblk = (n_keys + kBK - 1) / kBK;
  const uint32_t nrec = (uint32_t)((((int64_t)(n_keys - 1) * a.Hkv + kh + 1) * D) * 2);
  const __amdgpu_buffer_rsrc_t rk = make_rsrc(a.k + (int64_t)k_lo * a.Hkv * D, nrec);
  const __amdgpu_buffer_rsrc_t rv = make_rsrc(a.v + (int64_t)k_lo * a.Hkv * D, nrec);
  auto dma = [&](int t, int sk, int sv) __attribute__((always_inline)) {
    const int tid = (int)opaque(threadIdx.x);
#pragma unroll
    for (int n = 0; n < NDMA; ++n) {
      const int j = n * 512 + tid, r = j / NB, col = swz<DP>(r, (j % NB) * 8) - r * DP;
      const int key = t * kBK + r;
      const uint32_t off = (key < n_keys && col < D) ? (uint32_t)((key * a.Hkv + kh) * D + col) * 2 : nrec;
      const int jb = (n * 512 + wave * 64) * 8;
      dma_lds16(rk, Ks + sk * TILE + jb, off, 0);
      dma_lds16(rv, Vs + sv * TILE + jb, off, 0);
    }
  };
  // causal blocks wholly above the pair's rows add exact zeros
  auto skipped = [&](int t) __attribute__((always_inline)) {
    return t < 0 || t >= nblk || (!REMOTE && k_lo + t * kBK > s_wave0 + 31);
  };
  dma(0, 0, 0);
  dma(1, 1, 1);

  // One step per block and one more, so that role G finishes the last.  Loads
  // run two blocks ahead; at the step's end those of the next block have landed.
  auto steps = [&](auto&& work) __attribute__((always_inline)) {
    lds_barrier();
    int sv = 0;
    for (int t = 0; t <= nblk; ++t) {
      dma(t + 2, (t + 2) % NSK, sv == 0 ? 2 : sv - 1);
      __builtin_amdgcn_sched_barrier(0);
      work(t, sv);
      sv = sv == NSV - 1 ? 0 : sv + 1;
      wait_vmcnt<2 * NDMA>();
      lds_barrier();
    }
    wait_vmcnt<0>();  // no load may reach the LDS of the next workgroup
  };

  if (wave < 4) {
    u16x8_t qf[NKS], gf[NKS];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const int d = ks * 16 + hh * 8, dc = d < D ? d : 0;
      const u16x8_t xq = ld8(a.q + row * D + dc), xg = ld8(a.dout + row * D + dc);
      qf[ks] = d < D ? xq : zero8();
      gf[ks] = d < D ? xg : zero8();
    }
    const float nl = -a.lse[row] * kLog2e, dl = a.delta[row], c2 = a.scale_log2;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // rows and the first two blocks landed
    const uint32_t kq0 = swz_b128_base<DP>(lane);
    __builtin_amdgcn_s_setprio(1);
    steps([&](int t, int sv) __attribute__((always_inline)) {
      if (skipped(t)) return;
      const uint16_t* Kb = Ks + (t % NSK) * TILE;
      const uint16_t* Vb = Vs + sv * TILE;
      const uint32_t kq = opaque(kq0);
      f32x16_t sa = zero16(), pa = zero16();
      constexpr int PF = 3;  // operand reads ahead of their MFMAs
      u16x8_t ka[PF], va[PF];
      auto rd = [&](int i) __attribute__((always_inline)) {
        const uint32_t o = swz_b128<DP>(kq, i);
        ka[i % PF] = lds8(Kb, o);
        va[i % PF] = lds8(Vb, o);
      };
#pragma unroll
      for (int i = 0; i < PF; ++i) rd(i);
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        const u16x8_t xk = ka[ks % PF], xv = va[ks % PF];
        if (ks + PF < NKS) rd(ks + PF);
        sa = mfma32<DT>(xk, qf[ks], sa);
        pa = mfma32<DT>(xv, gf[ks], pa);
        __builtin_amdgcn_sched_barrier(0);
      }
      float p[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) p[r] = fast_exp2(fmaf(sa[r], c2, nl));
      const int kt0 = k_lo + t * kBK;
      if (kt0 + kBK > k_hi || (!REMOTE && kt0 + kBK - 1 > s_wave0)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = kt0 + 8 * (r >> 2) + 4 * hh + (r & 3);
          p[r] = (key < k_hi && (REMOTE || key <= s)) ? p[r] : 0.0f;
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) p[r] *= pa[r] - dl;
      Ds[t & 1][pair][0][lane] = pack8<DT>(p);
      Ds[t & 1][pair][1][lane] = pack8<DT>(p + 8);
    });
  } else {
    f32x16_t acc[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db) acc[db] = zero16();
    __builtin_amdgcn_s_waitcnt(0x0F70);
    const uint32_t trb0 = swz_tr_base<DP>(lane, 0), trb1 = swz_tr_base<DP>(lane, 1);
    steps([&](int t, int) __attribute__((always_inline)) {
      if (skipped(t - 1)) return;
      const uint16_t* Kb = Ks + ((t - 1) % NSK) * TILE;
      const uint32_t t0 = opaque(trb0), t1 = opaque(trb1);
      const u16x8_t ds[2] = {Ds[(t - 1) & 1][pair][0][lane], Ds[(t - 1) & 1][pair][1][lane]};
      constexpr int N2 = 2 * NDB, PF = 4;  // step i: d block i / 2, 16-key half i % 2
      u16x8_t ring[PF];
      auto rd = [&](int i) __attribute__((always_inline)) {
        const uint32_t ro = (i % 2) * 16 * DP * 2;
        return lds_tr8(Kb, ro + swz_tr<DP>(t0, i / 2), ro + swz_tr<DP>(t1, i / 2));
      };
#pragma unroll
      for (int i = 0; i < PF; ++i) ring[i] = rd(i);
#pragma unroll
      for (int i = 0; i < N2; ++i) {
        const u16x8_t kt = ring[i % PF];
        if (i + PF < N2) ring[i % PF] = rd(i + PF);
        acc[i / 2] = mfma32<DT>(kt, ds[i % 2], acc[i / 2]);
        __builtin_amdgcn_sched_barrier(0);
      }
    });
    if (valid) finish_row<DT, DP, REMOTE>(a, acc, row, slot, hh);
  }
}

// Up to 192 dims the causal launch is faster with one wave per 32 rows (64-key
// tiles, half the barriers): delta and dQ, full causal, 16/4 heads, dq2_kernel ->
// this, us: 16 x 512 tokens D 136 107 -> 98, D 160 111 -> 104, D 192 118.5 ->
// 113.5; 2 x 4096 D 192 392 -> 383; 4096 tokens, 8 heads, D 192 166 -> 167.  At
// 224 both are within 2.5% either way, at 256 see dq2_kernel.
template <int DT, int DP, bool REMOTE>
void launch_dq(const BwdArgs& a, unsigned grid, hipStream_t st) {
  if constexpr (DP <= 128 || !REMOTE) {
    if (DP <= 128 || a.D <= 192) {
      hipLaunchKernelGGL((dq_kernel<DT, DP, REMOTE, attn_qb<DP>()>), dim3(grid), dim3(256), 0, st, a);
      return;
    }
  }
  if constexpr (DP > 128)
    hipLaunchKernelGGL((dq2_kernel<DT, DP, REMOTE>), dim3(grid), dim3(512), 0, st, a);
}

// Row-split schedule of the key-major kernels, built on the device because
// the expert row counts live there.  Tile t costs n_t row tiles (its causal
// tiles for the G heads plus its expert's packed tiles, the count every
// key-major kernel derives).  The kernel picks the smallest segment length L
// with sum ceil(n_t / L) <= nwg, cuts each tile into that many equal
// segments, and deals the segments, in the XCD-grouped order of the host's
// list (its entries L % 8 == x, i.e. whole (chunk, kv head) groups per XCD),
// to the XCDs in contiguous runs: workgroup g runs on XCD g % 8, so a run of
// segments that share query rows stays in one L2.  One workgroup; a fixed
// function of the counts, so the sums below keep a fixed order.
constexpr int kSchedMaxTiles = 4096;

__device__ int block_sum_1024(int v, int* red) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  int t = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) t += red[i];
  return t;
}

template <int ROWS>
__device__ __forceinline__ void dkdv_schedule(const BwdArgs& a, int n_kv, int nwg, int* sched,
                                              int* seg) {
  __shared__ int work[kSchedMaxTiles];
  __shared__ int first[kSchedMaxTiles + 1];
  __shared__ int red[16];
  const int tid = threadIdx.x;
  const bool grouped = n_kv % 8 == 0;
  const int ni = n_kv / 8;
  auto tile_of = [&](int o) { return grouped ? (o % ni) * 8 + o / ni : o; };
  int wmax = 0, wsum = 0, nvalid = 0;
  for (int o = tid; o < n_kv; o += 1024) {
    const int* t = a.kv_tiles + 4 * tile_of(o);
    int n = 0;
    if (t[0] >= 0) {
      const int c = t[0], kt0 = t[1], f = t[2], kh = t[3];
      const int c_hi = a.cu_chunk[c + 1], key0 = a.cu_chunk[c] + kt0;
      const int n_self = (max(0, c_hi - key0) + ROWS - 1) / ROWS;
      const int n_rem = (f >= 0 && a.R > 0) ? a.counts[f * a.Hkv + kh] : 0;
      n = max(1, a.G * n_self + (n_rem + ROWS - 1) / ROWS);  // >= 1: its keys get written
    }
    work[o] = n;
    wmax = max(wmax, n);
    wsum += n;
    nvalid += n > 0;
  }
  // sum ceil(n_t / L) lies in [W / L, W / L + valid tiles]: the answer lies in
  // [ceil(W / nwg), ceil(W / (nwg - valid))], and max n_t always fits
  const int W = block_sum_1024(wsum, red), nv = block_sum_1024(nvalid, red);
  // block max through the sum helper's scratch (values are >= 0)
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) wmax = max(wmax, __shfl_xor(wmax, o, 64));
  __syncthreads();
  if ((tid & 63) == 0) red[tid >> 6] = wmax;
  __syncthreads();
  int hi = 1;
#pragma unroll
  for (int i = 0; i < 16; ++i) hi = max(hi, red[i]);
  if (nwg > nv) hi = min(hi, max(1, (W + (nwg - nv) - 1) / (nwg - nv)));
  int lo = min(hi, max(1, (W + nwg - 1) / nwg));
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    int cnt = 0;
    for (int o = tid; o < n_kv; o += 1024) cnt += (work[o] + mid - 1) / mid;
    if (block_sum_1024(cnt, red) <= nwg) hi = mid; else lo = mid + 1;
  }
  const int L = lo;
  // exclusive scan of the segment counts: thread tid owns a contiguous run
  const int per = (n_kv + 1023) / 1024;
  const int o0 = min(n_kv, tid * per), o1 = min(n_kv, o0 + per);
  int mine = 0;
  for (int o = o0; o < o1; ++o) mine += (work[o] + L - 1) / L;
  int inc = mine;  // inclusive scan over the wave, then over the waves
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(inc, o, 64);
    if ((tid & 63) >= o) inc += y;
  }
  __syncthreads();
  if ((tid & 63) == 63) red[tid >> 6] = inc;
  __syncthreads();
  int base = 0;
  for (int i = 0; i < (tid >> 6); ++i) base += red[i];
  int run = base + inc - mine;
  for (int o = o0; o < o1; ++o) {
    first[o] = run;
    run += (work[o] + L - 1) / L;
  }
  int S = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) S += red[i];
  if (tid == 0) first[n_kv] = S;
  __syncthreads();
  for (int o = tid; o < n_kv; o += 1024) {
    seg[2 * tile_of(o)] = first[o];
    seg[2 * tile_of(o) + 1] = first[o + 1] - first[o];
  }
  for (int g = tid; g < nwg; g += 1024) {
    int j = g;
    bool ok = g < S;
    if (grouped) {  // XCD x = g % 8 takes segments [ceil(x S / 8), ceil((x+1) S / 8))
      const int x = g % 8, s0 = (x * S + 7) / 8, s1 = ((x + 1) * S + 7) / 8;
      j = s0 + g / 8;
      ok = j < s1;
    }
    int4 w = {-1, 0, 0, -1};
    if (ok) {
      int l = 0, h = n_kv - 1;  // last o with first[o] <= j
      while (l < h) {
        const int m = (l + h + 1) >> 1;
        if (first[m] <= j) l = m; else h = m - 1;
      }
      const int ns = first[l + 1] - first[l], sidx = j - first[l], n = work[l];
      w = {tile_of(l), (int)((int64_t)n * sidx / ns), (int)((int64_t)n * (sidx + 1) / ns),
           ns > 1 ? j : -1};
    }
    reinterpret_cast<int4*>(sched)[g] = w;
  }
}

template <int ROWS>
__global__ __launch_bounds__(1024) void dkdv_sched_kernel(BwdArgs a, int n_kv, int nwg, int* sched,
                                                          int* seg) {
  dkdv_schedule<ROWS>(a, n_kv, nwg, sched, seg);
}

// The whole backward in one call: the schedule reads only the routing's counts,
// so workgroup 0 builds it while the others form delta, instead of a launch of
// one workgroup between dQ and dK/dV with the other CUs idle.  1024 threads per
// workgroup, 64 delta rows each: the schedule's 33 KB of LDS then still leaves
// a CU its 32 waves.  GQA 16K step 1333 -> 1321 us, fp16 ragged 727 -> 713 us.
template <int DT, int ROWS>
__global__ __launch_bounds__(1024) void delta_sched_kernel(BwdArgs a, int64_t rows, int n_kv,
                                                           int nwg, int* sched, int* seg) {
  if (blockIdx.x == 0) {
    dkdv_schedule<ROWS>(a, n_kv, nwg, sched, seg);
    return;
  }
  delta_row<DT>(a.out, a.dout, a.lse, (int64_t)(blockIdx.x - 1) * 64 + (threadIdx.x >> 4), rows,
                a.D, a.delta, a.scale, a.lse_k);
}

// dK / dV of the split tiles: workgroups (kv tile, y) share a tile's 16-byte
// elements, each summed over the tile's slots in slot order (tiles with one
// slot were written by the key-major kernel itself).
constexpr int kReduceSplit = 8;
template <int DT>
__global__ __launch_bounds__(256) void dkdv_reduce_kernel(BwdArgs a) {
  const int* t = a.kv_tiles + 4 * blockIdx.x;
  if (t[0] < 0) return;
  const int j0 = a.kv_seg[2 * blockIdx.x], ns = a.kv_seg[2 * blockIdx.x + 1];
  if (ns <= 1) return;
  const int c = t[0], kh = t[3], D = a.D;
  const int key0 = a.cu_chunk[c] + t[1];
  const int nk = min(kKvTileKeys, a.cu_chunk[c + 1] - key0);
  const int n4 = nk * D / 4;
  const int64_t slot4 = kv_slot_floats(D) / 4;
  const f32x4_t* part = reinterpret_cast<const f32x4_t*>(a.part_dkv) + j0 * slot4;
  for (int i = blockIdx.y * 256 + threadIdx.x; i < 2 * n4; i += 256 * kReduceSplit) {
    const int which = i >= n4;  // 0 = dK, 1 = dV
    const int jj = which ? i - n4 : i;
    const f32x4_t* src = part + which * (kKvTileKeys * D / 4) + jj;
    f32x4_t acc = src[0];
    int s = 1;
    for (; s + 4 <= ns; s += 4) {  // four loads in flight, added in slot order
      f32x4_t x[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] = src[(s + u) * slot4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += x[u][e];
    }
    for (; s < ns; ++s) {
      const f32x4_t x = src[s * slot4];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += x[e];
    }
    const float sc = which ? 1.0f : a.scale;
    u16x4_t r;
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = from_f32<DT>(acc[e] * sc);
    const int key = key0 + jj / (D / 4), d = (jj % (D / 4)) * 4;
    *reinterpret_cast<u16x4_t*>((which ? a.dv : a.dk) + ((int64_t)key * a.Hkv + kh) * D + d) = r;
  }
}

template <int DT, int DP>
int launch_bwd(const BwdArgs& a, int n_self, int n_kv, int max_remote, int parts, hipStream_t st) {
  const int64_t rows = (int64_t)a.T * a.Hq;
  const int n_wg = n_kv * a.kv_splits;
  int* const sched = const_cast<int*>(a.kv_sched);
  int* const seg = const_cast<int*>(a.kv_seg);
  const bool both = parts == 3 && n_kv > 0 && a.kv_splits > 1;
  if (both)
    hipLaunchKernelGGL((delta_sched_kernel<DT, kv_rows<DP>()>),
                       dim3((unsigned)((rows + 63) / 64 + 1)), dim3(1024), 0, st, a, rows, n_kv,
                       n_wg, sched, seg);
  if (parts & 1) {
    if (!both)
      hipLaunchKernelGGL(delta_kernel<DT>, dim3((unsigned)((rows + 15) / 16)), dim3(256), 0,
                         st, a.out, a.dout, a.lse, rows, a.D, a.delta, a.scale, a.lse_k);
    if (max_remote > 0 && a.R > 0)
      launch_dq<DT, DP, true>(a, (unsigned)((max_remote + 7) / 8 * 8), st);
    if (n_self > 0)
      launch_dq<DT, DP, false>(a, (unsigned)(((int64_t)n_self * a.G + 7) / 8 * 8), st);
  }
  if ((parts & 2) && n_kv > 0) {
    // kKvTileKeys keys per workgroup in every kernel; the host's key tiles match
    if (a.kv_splits > 1 && !both)
      hipLaunchKernelGGL(dkdv_sched_kernel<kv_rows<DP>()>, dim3(1), dim3(1024), 0, st, a, n_kv,
                         n_wg, sched, seg);
    if constexpr (DP <= 128) {
      if constexpr (DP <= 64) launch_dkdv1<DT, DP>(a, n_wg, st);
      else launch_dkdv2<DT, DP>(a, n_wg, st);
    } else {
      launch_dkdv4<DT, DP>(a, n_wg, st);
    }
    if (a.kv_splits > 1)
      hipLaunchKernelGGL(dkdv_reduce_kernel<DT>, dim3(n_kv, kReduceSplit), dim3(256), 0, st, a);
  }
  return moba_launch_status("prefill_bwd");
}

template <int DT>
int dispatch_bwd(const BwdArgs& a, int n_self, int n_kv, int max_remote, int parts, hipStream_t st) {
  if (a.D <= 32) return launch_bwd<DT, 32>(a, n_self, n_kv, max_remote, parts, st);
  if (a.D <= 64) return launch_bwd<DT, 64>(a, n_self, n_kv, max_remote, parts, st);
  if (a.D <= 128) return launch_bwd<DT, 128>(a, n_self, n_kv, max_remote, parts, st);
  return launch_bwd<DT, 256>(a, n_self, n_kv, max_remote, parts, st);
}

// Bytes of the schedule head of the row-split workspace (256-byte aligned).
int64_t dkdv_sched_bytes(int n_kv, int splits) {
  return ((int64_t)16 * n_kv * splits + (int64_t)8 * n_kv + 255) / 256 * 256;
}

}  // namespace

extern "C" int64_t moba_hip_prefill_bwd_work(int n_kv_tiles, int kv_splits, int D) {
  if (n_kv_tiles < 1 || kv_splits < 2 || kv_splits > 16 || D < 8 || D > 256) return 0;
  return dkdv_sched_bytes(n_kv_tiles, kv_splits) +
         (int64_t)n_kv_tiles * kv_splits * kv_slot_floats(D) * 4;
}

extern "C" int moba_hip_prefill_bwd_tiles(const void* q, const void* k, const void* v, const void* out,
                                    const void* dout, const float* lse, int dtype, int T, int Hq,
                                    int Hkv, int D, float scale, const int* cu_chunk,
                                    const int* self_tiles, int n_self_tiles, const int* kv_tiles,
                                    int n_kv_tiles, const int* sel, int R, const int* filtered,
                                    int E, const int* tile_off, const int* row_off,
                                    const int* counts, const int* rows, const int* tiles,
                                    int max_remote_tiles,
                                    float* delta, void* part_dq, void* dq, void* dk, void* dv,
                                    int parts, int kv_splits, float* part_dkv, void* pack,
                                    void* stream) {
  if (dtype != 0 && dtype != 1) { moba_set_error("prefill_bwd: dtype must be 0 (bf16) or 1 (fp16)"); return MOBA_ERR_ARG; }
  if (D < 8 || D > 256 || D % 8) { moba_set_error("prefill_bwd: head_dim must be a multiple of 8 in [8,256]"); return MOBA_ERR_ARG; }
  if (Hq < 1 || Hkv < 1 || Hq % Hkv) { moba_set_error("prefill_bwd: Hq must be a positive multiple of Hkv"); return MOBA_ERR_ARG; }
  if (R < 0 || R > 8) { moba_set_error("prefill_bwd: remote count must be in [0,8]"); return MOBA_ERR_ARG; }
  if (Hq > 65535 || (int64_t)n_self_tiles * (Hq / Hkv) > (1 << 30)) { moba_set_error("prefill_bwd: too many heads or self tiles"); return MOBA_ERR_ARG; }
  if (parts < 1 || parts > 3) { moba_set_error("prefill_bwd: parts must be 1 (dq), 2 (dk/dv) or 3 (both)"); return MOBA_ERR_ARG; }
  if ((int64_t)T * Hq * D * 2 >= ((int64_t)1 << 32)) { moba_set_error("prefill_bwd: q / dO must be smaller than 4 GiB (32-bit buffer offsets)"); return MOBA_ERR_ARG; }
  if (kv_splits < 1 || kv_splits > 16 || (kv_splits > 1 && part_dkv == nullptr)) { moba_set_error("prefill_bwd: kv_splits must be in [1,16], with a part_dkv workspace when > 1"); return MOBA_ERR_ARG; }
  if (kv_splits > 1 && n_kv_tiles > kSchedMaxTiles) { moba_set_error("prefill_bwd: kv_splits > 1 needs n_kv_tiles <= 4096"); return MOBA_ERR_ARG; }
  if ((int64_t)n_kv_tiles * kv_splits > 0x7fffffff / 4) { moba_set_error("prefill_bwd: too many kv workgroups"); return MOBA_ERR_ARG; }
  BwdArgs a;
  a.q = (const uint16_t*)q; a.k = (const uint16_t*)k; a.v = (const uint16_t*)v;
  a.out = (const uint16_t*)out; a.dout = (const uint16_t*)dout; a.lse = lse;
  a.T = T; a.Hq = Hq; a.Hkv = Hkv; a.D = D; a.G = Hq / Hkv;
  a.scale = scale; a.scale_log2 = scale * kLog2e;
  a.cu_chunk = cu_chunk; a.self_tiles = self_tiles; a.kv_tiles = kv_tiles;
  a.n_self_wg = n_self_tiles * (Hq / Hkv);
  a.sel = sel; a.R = R; a.filtered = filtered; a.E = E;
  a.tile_off = tile_off; a.row_off = row_off; a.counts = counts; a.rows = rows;
  a.tiles = (const int4*)tiles;
  a.delta = delta; a.part_dq = (uint16_t*)part_dq; a.kv_splits = kv_splits;
  a.kv_sched = a.kv_seg = nullptr; a.part_dkv = nullptr;
  if (kv_splits > 1) {  // workspace: schedule, tile slots, then the partial slots
    char* ws = (char*)part_dkv;
    a.kv_sched = (const int*)ws;
    a.kv_seg = a.kv_sched + 4 * (int64_t)n_kv_tiles * kv_splits;
    a.part_dkv = (float*)(ws + dkdv_sched_bytes(n_kv_tiles, kv_splits));
  }
  a.dq = (uint16_t*)dq; a.dk = (uint16_t*)dk; a.dv = (uint16_t*)dv;
  a.lse_k = delta + (int64_t)T * Hq;  // adjacent to delta (one load per row in the key-major kernels)
  a.pack_rows = (R > 0 && D <= 128) ? (int64_t)T * Hq * R : 0;
  a.pack_q = (uint16_t*)pack;
  a.pack_g = a.pack_q + a.pack_rows * D;
  a.pack_lse_k = (float*)(a.pack_g + a.pack_rows * D);
  a.pack_delta = a.pack_lse_k + a.pack_rows;
  if (a.pack_rows > 0 && pack == nullptr) { moba_set_error("prefill_bwd: the pack workspace is required when R > 0 and head_dim <= 128"); return MOBA_ERR_ARG; }
  if (a.pack_rows * D * 2 >= ((int64_t)1 << 32)) { moba_set_error("prefill_bwd: packed expert rows must be smaller than 4 GiB (32-bit buffer offsets)"); return MOBA_ERR_ARG; }
  hipStream_t st = (hipStream_t)stream;
  const int mr = R > 0 ? max_remote_tiles : 0;
  return dtype == 0 ? dispatch_bwd<0>(a, n_self_tiles, n_kv_tiles, mr, parts, st)
                    : dispatch_bwd<1>(a, n_self_tiles, n_kv_tiles, mr, parts, st);
}

extern "C" int moba_hip_prefill_bwd(const void* q, const void* k, const void* v, const void* out,
                                    const void* dout, const float* lse, int dtype, int T, int Hq,
                                    int Hkv, int D, float scale, const int* cu_chunk,
                                    const int* self_tiles, int n_self_tiles, const int* kv_tiles,
                                    int n_kv_tiles, const int* sel, int R, const int* filtered,
                                    int E, const int* tile_off, const int* row_off,
                                    const int* counts, const int* rows, int max_remote_tiles,
                                    float* delta, void* part_dq, void* dq, void* dk, void* dv,
                                    int parts, int kv_splits, float* part_dkv, void* pack,
                                    void* stream) {
  return moba_hip_prefill_bwd_tiles(q, k, v, out, dout, lse, dtype, T, Hq, Hkv, D, scale, cu_chunk,
                                    self_tiles, n_self_tiles, kv_tiles, n_kv_tiles, sel, R,
                                    filtered, E, tile_off, row_off, counts, rows, nullptr,
                                    max_remote_tiles, delta, part_dq, dq, dk, dv, parts, kv_splits,
                                    part_dkv, pack, stream);
}
