// Key-major dK / dV of the MoBA prefill backward for head dims 129..256: wave
// pairs with split roles, one product block per step and one body.
//
// Replaces the dk/dv halves of the two flash-attention backwards in
// OptMixedAttention.backward (src/moba_opt/mixed_attention.py:165-221) and the
// autograd scatter-add of the packed remote dk/dv into k/v
// (grouped_attention.py:81-89): every query row that attends a key -- the
// causal rows of the key's own chunk for all G heads of its KV group, then the
// expert rows that selected the chunk -- is visited by the one workgroup that
// owns the key, so dK / dV are summed in registers in a fixed order and
// written once (no atomics).
//
// A workgroup of 8 waves owns 128 keys of one chunk and one KV head as 4 wave
// pairs of 32 keys; the two waves of a pair share a SIMD and split the four
// products as in the kernel of the 65..128-wide heads (attn_dkdv2.hip), over
// 32-row tiles of (Q, dO).  At step t:
//   role P (-K, dV):   X_t = lse_k - Q_t K^T  interleaved with
//                      dV += P_{t-1}^T dO_{t-1};  P_t = exp2(-c X_t)
//   role D (-V, -dK):  -dS_{t-1} = P_{t-1} Y_{t-1}, then Y_t = delta - dO_t V^T
//                      interleaved with -dK += (-dS_{t-1})^T Q_{t-1}
// P passes through LDS in fp32 (from the rounded P, dK's error at 256 dims
// doubled).  The only synchronisation is one barrier per step, where the three
// stages rotate.
//
// What bounds it is registers: a 32-key operand (64) and a 32-key accumulator
// (128) leave 64 of a wave's 256, so
//  * there is one body: full tiles branch around the mask, and a product
//    that takes no part reads a tile of zeros (variants of the block made the
//    compiler copy the accumulators: 300 to 1000 spilled registers);
//  * the row list is loaded a step before the loads that need it and stays
//    untouched until then, so no wait for it drains the tile loads (it cost
//    0.12 ms);
//  * what can be recomputed from the thread index is (opaque()).
// LDS operands still arrive just in time, with one read in flight: about 2.6
// us per step where the MFMAs take 1.0.  T 8192, 16/4 heads, chunk 1024,
// top-3, D 256: 1313 -> 715-750 us (the two-stage kernel it replaces held one
// product at a time between two barriers per tile and spilled 77 registers).
// One product per wave (8 waves on 64 keys, nothing spilled, operands four
// reads ahead) took 866 us: its tiles feed half the keys, and loading them
// alone takes 596.
#include <type_traits>

#include "common.h"
#include "bwd_args.h"

namespace moba {
namespace {

constexpr int kPairKeys = 32;  // keys per wave pair

template <int DT, int DP>
__global__ __launch_bounds__(512, 2) void dkdv4_kernel(BwdArgs a) {
  constexpr int kRows = kv_rows<DP>();
  static_assert(kRows == 32, "one 32-row block per tile");
  constexpr int NKS = DP / 16, NDB = DP / 32, NB = DP / 8;
  constexpr int NDMA = kRows * NB / 512;        // 16-byte blocks per thread per operand
  constexpr int TILE = kRows * DP;
  constexpr int NST = 3;                        // stages: tiles t - 1, t and t + 1
  __shared__ __attribute__((aligned(16))) uint16_t Qs[NST * TILE];
  __shared__ __attribute__((aligned(16))) uint16_t Gs[NST * TILE];
  __shared__ __attribute__((aligned(16))) uint16_t Zs[TILE];
  __shared__ __attribute__((aligned(16))) float Ls[2][2 * kRows];  // lse_k, then delta
  __shared__ __attribute__((aligned(16))) f32x4_t Pf[2][4][4][64];  // P of tile & 1, per pair

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qi = lane & 31, hh = lane >> 5;
  const int pair = wave & 3;
  const bool role_p = wave < 4;
  const int D = a.D, G = a.G;
  int ti, s_lo, s_hi, slot;
  if (!kv_work(a, ti, s_lo, s_hi, slot)) return;
  const int* tile = a.kv_tiles + 4 * ti;
  const int c = tile[0], kt0 = tile[1], f = tile[2], kh = tile[3];
  if (c < 0) return;                            // padding entry of the XCD-ordered list
  const int c_hi = a.cu_chunk[c + 1];
  const int key0 = a.cu_chunk[c] + kt0;         // first key of the workgroup
  const int off0 = pair * kPairKeys;            // this pair's keys within it
  const int mykey = key0 + off0 + qi;           // this lane's key (B operand column)

  // Uninitialised LDS could hold NaN patterns that a zero probability would
  // not cancel; column blocks past D are never loaded and must read zero.
  for (int j = tid; j < TILE / 8; j += 512) st8(Zs + j * 8, zero8());
  for (int j = tid; j < NST * TILE / 8; j += 512) {
    st8(Qs + j * 8, zero8());
    st8(Gs + j * 8, zero8());
  }
  __syncthreads();

  // query tiles: G * n_self causal tiles (rows from key0 to the chunk end, for
  // every head of the group), then the expert's rows
  const int n_self = (c_hi - key0 + kRows - 1) / kRows;
  const int e = (f >= 0 && a.R > 0) ? f * a.Hkv + kh : -1;
  const int n_rem = e >= 0 ? a.counts[e] : 0;
  const int n_tiles = G * n_self + (n_rem + kRows - 1) / kRows;
  const int it_lo = s_lo, it_hi = min(s_hi, n_tiles);

  struct Cur { int it, g, s; };  // causal tile s of head g while g < G, else expert tile s
  auto next = [&](Cur t) __attribute__((always_inline)) {
    ++t.it; ++t.s;
    if (t.g < G && t.s == n_self) { t.s = 0; ++t.g; }
    return t;
  };
  const uint32_t qbytes = (uint32_t)((int64_t)a.T * a.Hq * D * 2);
  const uint32_t lbytes = (uint32_t)((int64_t)a.T * a.Hq * 4);
  const __amdgpu_buffer_rsrc_t rq = make_rsrc(a.q, qbytes), rg = make_rsrc(a.dout, qbytes);
  // delta and lse_k are adjacent arrays (delta first): wave 0's lanes 0..31
  // load lse_k of the tile's rows, lanes 32..63 their delta
  const __amdgpu_buffer_rsrc_t rl = make_rsrc(a.delta, 2 * lbytes);
  // Expert rows of this thread's blocks and, in the last entry, of its lane's
  // row terms, for the tile that is loaded next: the list's own values, loaded
  // unconditionally (any entry where there is no such row) and not touched
  // before the loads that need them, a step later.  A use, a branch or a copy
  // in between would wait for them, and so for the tile loads issued before.
  const int* list = e >= 0 && n_rem > 0 ? a.rows + a.row_off[e] : a.kv_tiles;
  const int last = max(n_rem, 1) - 1;
  int grow[NDMA + 1];
  auto fetch = [&](Cur t) __attribute__((always_inline)) {
    const int r0 = t.g < G ? 0 : t.s * kRows, tid = (int)opaque(threadIdx.x);
#pragma unroll
    for (int n = 0; n <= NDMA; ++n)
      grow[n] = list[min(r0 + (n < NDMA ? (n * 512 + tid) / NB : tid & 31), last)];
  };
  // Rows past the tile's end read past num_records, i.e. zeros: a zero Q and
  // dO row adds nothing.  A tile past the share loads nothing.
  auto dma = [&](Cur t, int st, int ls) __attribute__((always_inline)) {
    if (t.it >= it_hi) return;
    const bool is_self = t.g < G;
    const int s0 = key0 + t.s * kRows, tid = (int)opaque(threadIdx.x), lane = tid & 63;
    const int nvalid = is_self ? c_hi - s0 : n_rem - t.s * kRows;
    auto row = [&](int n, int q) { return is_self ? (s0 + q) * a.Hq + kh * G + t.g : grow[n] >> 3; };
#pragma unroll
    for (int n = 0; n < NDMA; ++n) {
      const int j = n * 512 + tid, q = j / NB, col = swz<DP>(q, (j % NB) * 8) - q * DP;
      const uint32_t off = (q < nvalid && col < D)
                               ? (uint32_t)(((int64_t)row(n, q) * D + col) * 2) : qbytes;
      const int jb = (n * 512 + wave * 64) * 8;
      dma_lds16(rq, Qs + st * TILE + jb, off, 0);
      dma_lds16(rg, Gs + st * TILE + jb, off, 0);
    }
    if (wave == 0) {
      const uint32_t off = (lane & 31) < nvalid
                               ? (lane < 32 ? lbytes : 0) + (uint32_t)row(NDMA, lane & 31) * 4 : 2 * lbytes;
      dma_lds4(rl, Ls[ls], off, 0);
    }
  };
  // causal rows that end before the pair's first key contribute nothing
  auto skipped = [&](Cur t) __attribute__((always_inline)) {
    return t.it >= it_hi || (t.g < G && t.s * kRows + kRows - 1 < off0);
  };

  const uint32_t kq0 = swz_b128_base<DP>(lane);
  const uint32_t trb0 = swz_tr_base<DP>(lane, 0);

  auto body = [&](auto role_tag) __attribute__((always_inline)) {
  constexpr bool ROLE_P = decltype(role_tag)::value;
  // -K (role P) or -V (role D) rows: B operands, column = key, k = d
  u16x8_t kv[NKS];
  const uint16_t* src = ROLE_P ? a.k : a.v;
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
    const int d = ks * 16 + hh * 8;
    const u16x8_t x = ld8(src + ((int64_t)min(mykey, c_hi - 1) * a.Hkv + kh) * D + (d < D ? d : 0));
    kv[ks] = mykey < c_hi && d < D ? neg8(x) : zero8();
  }
  // landed before the tile loads start (the compiler's own waits for them
  // would otherwise also drain the tile loads in flight)
  __builtin_amdgcn_s_waitcnt(0x0F70);
  f32x16_t acc[NDB], sp = zero16();  // dV or -dK; X of the tile, or Y
#pragma unroll
  for (int i = 0; i < NDB; ++i) acc[i] = zero16();
  u16x8_t op[2] = {zero8(), zero8()};  // P or -dS of the tile before, as A operand

  // Chain A: sp = row terms Li + (tile A rows) x kv.  Chain B: acc += op^T x
  // (tile B rows), read transposed.  Both are NKS = 2 NDB MFMAs long.
  static_assert(NKS == 2 * NDB, "chain lengths");
  auto block = [&](const uint16_t* A, const float* Li,
                   const uint16_t* B) __attribute__((always_inline)) {
    const uint32_t kq = opaque(kq0), t0 = opaque(trb0);
    auto rda = [&](int i) __attribute__((always_inline)) { return lds8(A, swz_b128<DP>(kq, i)); };
    auto rdb = [&](int i) __attribute__((always_inline)) {  // 16-row half i / NDB, d block i % NDB
      // rows 8 further down lie at the swizzle's neighbouring block
      const uint32_t ro = (i / NDB) * 16 * DP * 2, x = swz_tr<DP>(t0, i % NDB);
      return lds_tr8(B, ro + x, ro + (x ^ 16) + 8 * DP * 2);
    };
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // D layout: lane holds rows 8j + 4(lane / 32) + i
      const f32x4_t l4 = *reinterpret_cast<const f32x4_t*>(Li + 8 * j + 4 * (((int)opaque(threadIdx.x) >> 5) & 1));
#pragma unroll
      for (int i = 0; i < 4; ++i) sp[4 * j + i] = l4[i];
    }
    u16x8_t ra = rda(0), rb = rdb(0);
#pragma unroll
    for (int i = 0; i < NKS; ++i) {
      const u16x8_t xa = ra, xb = rb;
      if (i + 1 < NKS) ra = rda(i + 1);
      sp = mfma32<DT>(xa, kv[i], sp);
      if (i + 1 < NKS) rb = rdb(i + 1);
      acc[i % NDB] = mfma32<DT>(op[i / NDB], xb, acc[i % NDB]);
    }
    // issue order: an operand is read behind the MFMA before the one that
    // takes it (4 row-term reads; then 1 read of chain A, 2 of chain B a step)
    __builtin_amdgcn_sched_group_barrier(0x100, 7, 0);
#pragma unroll
    for (int i = 0; i < NKS - 1; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
  };
  // Both chains always run: a product that takes no part reads a tile of
  // zeros (chain B) or is not used (chain A).
  auto run_block = [&](bool prev, const uint16_t* A, const float* Li,
                       const uint16_t* B) __attribute__((always_inline)) {
    if (!prev) op[0] = op[1] = zero8();
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
    block(A, Li, prev ? B : Zs);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
  };

  Cur t = it_lo < G * n_self ? Cur{it_lo, it_lo / n_self, it_lo % n_self}
                             : Cur{it_lo, G, it_lo - G * n_self};
  fetch(t);
  dma(t, 0, 0);
  Cur tn = next(t);
  fetch(tn);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  lds_barrier();
  const float nc2 = -a.scale_log2;
  bool prev = false;                   // tile t - 1 takes part
  int st = 0, b = 0;                   // stage and parity of tile t
  // one step past it_hi, so both roles finish the last tile
  for (int it = it_lo; it <= it_hi; ++it) {
    const int sn = st == NST - 1 ? 0 : st + 1, sp1 = st == 0 ? NST - 1 : st - 1;
    dma(tn, sn, b ^ 1);
    const Cur tf = next(tn);
    fetch(tf);
    __builtin_amdgcn_sched_barrier(0);  // the next tile's loads go out first
    const bool cur = !skipped(t);
    if constexpr (ROLE_P) {
      run_block(prev, Qs + st * TILE, Ls[b], Gs + sp1 * TILE);
      if (cur) {
        const bool is_self = t.g < G;
        const int ln = (int)opaque(threadIdx.x) & 63;
        const int row0 = t.s * kRows;  // causal rows, from the workgroup's first key
        if (key0 + off0 + kPairKeys > c_hi || (is_self && row0 < off0 + kPairKeys - 1)) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {  // a masked pair's P becomes exp2(-inf) = 0
            const int row = row0 + 8 * (r >> 2) + 4 * (ln >> 5) + (r & 3), k = off0 + (ln & 31);
            sp[r] = (key0 + k < c_hi && (!is_self || k <= row)) ? sp[r] : INFINITY;
          }
        }
        uint32_t w[8];  // packed pairs (rows 8j + 4hh + 2m, + 1) at w[2j + m]
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          f32x4_t p;
#pragma unroll
          for (int i = 0; i < 4; ++i) p[i] = fast_exp2(sp[4 * j + i] * nc2);
          Pf[b][pair][j][ln] = p;
          w[2 * j] = pack2<DT>(p[0], p[1]);
          w[2 * j + 1] = pack2<DT>(p[2], p[3]);
        }
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2)
          op[h2] = __builtin_bit_cast(
              u16x8_t, (u32x4_t){w[4 * h2], w[4 * h2 + 1], w[4 * h2 + 2], w[4 * h2 + 3]});
      }
    } else {
      if (prev) {
        uint32_t w[8];
        const int ln = (int)opaque(threadIdx.x) & 63;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const f32x4_t p = Pf[b ^ 1][pair][j][ln];
          w[2 * j] = pack2<DT>(p[0] * sp[4 * j], p[1] * sp[4 * j + 1]);
          w[2 * j + 1] = pack2<DT>(p[2] * sp[4 * j + 2], p[3] * sp[4 * j + 3]);
        }
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2)
          op[h2] = __builtin_bit_cast(
              u16x8_t, (u32x4_t){w[4 * h2], w[4 * h2 + 1], w[4 * h2 + 2], w[4 * h2 + 3]});
      }
      run_block(prev, Gs + st * TILE, Ls[b] + kRows, Qs + sp1 * TILE);
    }
    prev = cur;
    t = tn; tn = tf;
    st = sn; b ^= 1;
    __builtin_amdgcn_s_waitcnt(0x0F70);
    lds_barrier();
  }
  const int ln = (int)opaque(threadIdx.x) & 63, qi = ln & 31, hh = ln >> 5;
  // D layout: lane holds column d = i*32 + qi, keys 8j + 4hh + r.  A row
  // split writes fp32 partials to its slot for the fixed-order reduction.
  float* pdst = a.part_dkv + (int64_t)max(slot, 0) * kv_slot_floats(D) +
                (ROLE_P ? kKvTileKeys * D : 0);
  uint16_t* dst = ROLE_P ? a.dv : a.dk;
  const float psc = ROLE_P ? 1.0f : -1.0f, osc = ROLE_P ? 1.0f : -a.scale;
#pragma unroll
  for (int i = 0; i < NDB; ++i) {
    const int d = i * 32 + qi;
    if (d >= D) continue;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int k = off0 + 8 * (r >> 2) + 4 * hh + (r & 3), key = key0 + k;
      if (key >= c_hi) continue;
      if (slot >= 0) pdst[k * D + d] = acc[i][r] * psc;
      else dst[((int64_t)key * a.Hkv + kh) * D + d] = from_f32<DT>(acc[i][r] * osc);
    }
  }
  };
  if (role_p) body(std::true_type{}); else body(std::false_type{});
}

}  // namespace

template <int DT, int DP> void launch_dkdv4(const BwdArgs& a, int n_wg, hipStream_t st) {
  hipLaunchKernelGGL((dkdv4_kernel<DT, DP>), dim3(n_wg), dim3(512), 0, st, a);
}

template void launch_dkdv4<0, 256>(const BwdArgs&, int, hipStream_t);
template void launch_dkdv4<1, 256>(const BwdArgs&, int, hipStream_t);

}  // namespace moba
