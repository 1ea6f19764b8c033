// Prefill routing: chunk-mean key pooling, FP32 gate scores, stable top-k, and
// the expert-major packing of the selected (query, head) rows.
//
// Replaces the torch routing ops of src/moba_opt/grouped_attention.py:48-94
// (stack/index_select, mean, einsum, mask, topk/argmax loop, nonzero packing).
// The arithmetic order is the canonical one of the CPU oracle, so the selected
// block sets are bit-identical to it:
//   mean  = canonical fp32 sum over the chunk's tokens (64 strided partial
//           sums + fixed pairwise tree), / C  (optionally rounded to the
//           input dtype: route_precision "upstream")
//   gate  = fma chain over d = 0..D-1 in fp32
//   top-k = descending gate, exact ties -> lowest chunk, -inf never chosen.
#include <type_traits>

#include "common.h"
#include "../../include/moba_hip.h"

using namespace moba;

namespace {

constexpr int kMaxRemote = 8;

// Pick bits of a block of 256 consecutive tokens of one head (thread = token),
// for the candidates [t0, t0 + kPickRows): word 4 r + w holds the tokens of
// wave w that picked candidate t0 + r.  A token's rank among the block's picks
// of a candidate is then a population count, and so is the block's number of
// picks.  The words are built by OR, which no order changes.  fs: the
// thread's picks (filtered indices, -1 for none).
constexpr int kPickRows = 256;

MOBA_DEV void pick_bits(uint64_t* bits, const int (&fs)[kMaxRemote], int t0) {
  const int tid = threadIdx.x;
  __syncthreads();  // the words of the tile before are consumed
#pragma unroll
  for (int w = 0; w < 4; ++w) bits[4 * tid + w] = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kMaxRemote; ++j) {
    const int r = fs[j] - t0;
    if (fs[j] >= 0 && r >= 0 && r < kPickRows)
      atomicOr(reinterpret_cast<unsigned long long*>(bits + 4 * r + (tid >> 6)),
               1ull << (tid & 63));
  }
  __syncthreads();
}

// One workgroup per (filtered chunk, kv head, dim slice of D / ds).  The mean of dim d is the
// canonical sum: 64 partial sums s_j over the tokens j, j+64, j+128, ... in
// increasing order, then the fixed tree canon_tree over j.  Work item
// (j, column block b) of 8 dims is p = j * nd8 + b, so a wave's loads cover
// whole rows (coalesced); thread t owns items t, t + 256, ...  The partials
// go through LDS to one wave per dim, lane j holding s_j, for the tree.
template <int DT, int NP>
__global__ __launch_bounds__(256) void chunk_means_kernel(const uint16_t* __restrict__ k, int Hkv,
                                                          int D, const int* __restrict__ chunk_start,
                                                          int C, int precision, int ds,
                                                          float* __restrict__ means) {
  extern __shared__ float part[];  // [64][D]
  const int nd8 = D / 8 / ds, np = 64 * nd8;  // this workgroup's 8-dim blocks
  const int sub = blockIdx.x % ds, fk = blockIdx.x / ds;
  const int kh = fk % Hkv, f = fk / Hkv;
  const int tid = threadIdx.x;
  const int64_t stride = (int64_t)Hkv * D;
  const uint16_t* base = k + ((int64_t)chunk_start[f] * Hkv + kh) * D;
  float acc[NP][8];
  int jj[NP], bb[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int p = tid + 256 * i;
    jj[i] = p < np ? p / nd8 : C;  // items past np load nothing
    bb[i] = sub * nd8 + p % nd8;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[i][e] = 0.0f;
  }
  // KU row groups of 64 tokens per pass: all their loads are issued before
  // the adds, which then run in token order (one load latency per pass, not
  // per group)
  constexpr int KU = NP <= 2 ? 8 : 4;
  for (int t0 = 0; t0 < C; t0 += 64 * KU) {
    u16x8_t x[KU][NP];
#pragma unroll
    for (int u = 0; u < KU; ++u)
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int t = t0 + 64 * u + jj[i];
        x[u][i] = t < C ? ld8(base + t * stride + bb[i] * 8) : zero8();
      }
#pragma unroll
    for (int u = 0; u < KU; ++u)
#pragma unroll
      for (int i = 0; i < NP; ++i)
        if (t0 + 64 * u + jj[i] < C) {
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[i][e] = acc[i][e] + to_f32<DT>(x[u][i][e]);
        }
  }
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int p = tid + 256 * i;
    if (p < np) {
#pragma unroll
      for (int e = 0; e < 8; ++e) part[jj[i] * D + bb[i] * 8 + e] = acc[i][e];
    }
  }
  __syncthreads();
  const int lane = tid & 63, w = tid >> 6;
  float* dst = means + ((int64_t)f * Hkv + kh) * D;
  for (int d = sub * nd8 * 8 + w; d < (sub + 1) * nd8 * 8; d += 4) {
    float m = canon_tree(part[lane * D + d]) / (float)C;
    if (precision == 0) m = to_f32<DT>(from_f32<DT>(m));
    if (lane == 0) dst[d] = m;
  }
}

// One thread per (token, q head): a workgroup takes 256 consecutive tokens of
// one head.  The means rows its tokens score (filtered indices [flo, fhi) of
// the head's kv head) go through LDS in tiles of kRouteTile rows; a wave walks
// the union of its lanes' candidate ranges, 16 or 8 candidates at a time, and
// lanes outside a candidate's range discard its score.
//
// The canonical gate is a sequential fma chain over d per (token, candidate):
// too long for the vector unit (each fma also needs the candidate's mean in
// every lane), but it is what v_mfma_f32_4x4x1_16b_f32 does: one fma per
// output, 16 blocks of 4 candidates x 4 tokens, so D of them in d order form
// the chains of 4 candidates for the wave's 64 tokens, bit for bit, at twice
// the rate of plain fmas.  Lane l supplies its token's q[d] and the mean of
// candidate l % 4, and receives its own token's four scores.  Rows of the LDS
// tile are padded by 16 bytes, so the four rows a read touches lie in
// different banks; the token's q row stays in the input type (half the
// registers, converted as it is used).  Against a chain of fmas with the mean
// in a DPP row broadcast (T 32768, 8 heads, D 128, 63 candidates: 138 -> 87
// us; 32 heads, 7 candidates: 116 -> 97; T 8192, 16 heads, D 256, 7
// candidates: 43 -> 24).  Eight candidates a pass instead of 16 took 101 us
// in the first case (the conversions), four 117.
constexpr int kRouteTile = 32;

// The four values of two packed words, converted where they are used: kept
// out of the compiler's sight, which would convert the whole row ahead of the
// loop and hold it in twice the registers.  The trailing s_nop covers the two
// wait states between a vector write and an MFMA that reads it (the compiler
// does not look inside the block).
template <int DT> MOBA_DEV f32x4_t late_f32x4(uint32_t w0, uint32_t w1) {
  float x0, x1, x2, x3;
  if constexpr (DT == 0) {
    asm volatile(
        "v_lshlrev_b32 %0, 16, %4\n"
        "v_and_b32 %1, 0xffff0000, %4\n"
        "v_lshlrev_b32 %2, 16, %5\n"
        "v_and_b32 %3, 0xffff0000, %5\n"
        "s_nop 1"
        : "=&v"(x0), "=&v"(x1), "=&v"(x2), "=&v"(x3) : "v"(w0), "v"(w1));
  } else {
    asm volatile(
        "v_cvt_f32_f16 %0, %4\n"
        "v_cvt_f32_f16_sdwa %1, %4 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:WORD_1\n"
        "v_cvt_f32_f16 %2, %5\n"
        "v_cvt_f32_f16_sdwa %3, %5 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:WORD_1\n"
        "s_nop 1"
        : "=&v"(x0), "=&v"(x1), "=&v"(x2), "=&v"(x3) : "v"(w0), "v"(w1));
  }
  return (f32x4_t){x0, x1, x2, x3};
}

// RM: the largest R the selection registers hold.
template <int DT, int DP, int RM>
__global__ __launch_bounds__(256) void route_kernel(const uint16_t* __restrict__ q, int T, int Hq,
                                                    int Hkv, int D,
                                                    const float* __restrict__ means,
                                                    const int* __restrict__ cu_chunk, int nchunk,
                                                    const int* __restrict__ chunk_batch,
                                                    const int* __restrict__ first_chunk, int R,
                                                    int F, int* __restrict__ sel,
                                                    float* __restrict__ gate,
                                                    int* __restrict__ blk_count) {
  constexpr int LD = DP + 4;  // floats per LDS row of the means tile
  // 256 tokens x 64 dims of q while it is loaded, then the means tiles
  constexpr int kStageFloats = 256 * 64 / 2;
  __shared__ __attribute__((aligned(16))) float mt[kRouteTile * LD > kStageFloats ? kRouteTile * LD : kStageFloats];
  __shared__ int red[2][4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int s = blockIdx.x * 256 + tid;
  const int h = blockIdx.y;
  const bool live = s < T;
  const int G = Hq / Hkv, kh = h / G;
  // The wave's q rows come in whole 128-byte lines, 8 lanes to a row of 64
  // dims, and reach their lanes through LDS (16-byte block x of row r at block
  // x ^ (r / 2 % 8): no bank conflicts either way).  Each lane loading its own
  // row took eight times the lines.
  const int64_t idx = (int64_t)s * Hq + h;
  constexpr int NQ = DP / 8;
  u16x8_t qv[NQ];
  {
    uint16_t* st = reinterpret_cast<uint16_t*>(mt) + (tid >> 6) * 64 * 64;
    const int s0 = blockIdx.x * 256 + (tid >> 6) * 64;
    u16x8_t x[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) {  // slice i / 8 of 64 dims, rows 8 (i % 8) ..
      const int r = (i % 8) * 8 + (lane >> 3), d = (i / 8) * 64 + (lane & 7) * 8;
      x[i] = ld8(q + ((int64_t)min(s0 + r, T - 1) * Hq + h) * D + (d < D ? d : 0));
      if (d >= D) x[i] = zero8();
    }
#pragma unroll
    for (int sl = 0; sl < NQ / 8; ++sl) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int r = i * 8 + (lane >> 3);
        st8(st + r * 64 + (((lane & 7) ^ ((r >> 1) & 7)) * 8), x[sl * 8 + i]);
      }
      wave_lds_sync();
#pragma unroll
      for (int i = 0; i < 8; ++i)
        qv[sl * 8 + i] = ld8(st + lane * 64 + ((i ^ ((lane >> 1) & 7)) * 8));
      wave_lds_sync();
    }
  }
  // chunk containing s (the last token's for the threads past T)
  const int sc = live ? s : T - 1;
  // search once per wave for its first token (uniform loads), then per lane
  // only when the wave straddles a chunk boundary
  const int sw = __builtin_amdgcn_readfirstlane(sc);
  int lo = 0, hi = nchunk - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (cu_chunk[mid] <= sw) lo = mid; else hi = mid - 1;
  }
  if (__ballot(sc >= cu_chunk[lo + 1]) != 0) {
    lo = 0; hi = nchunk - 1;
    while (lo < hi) {
      int mid = (lo + hi + 1) >> 1;
      if (cu_chunk[mid] <= sc) lo = mid; else hi = mid - 1;
    }
  }
  const int cs = lo, b = chunk_batch[cs], c0 = first_chunk[cs];
  // this thread's candidates are filtered rows [c0 - b, cs - b)
  const int f0 = c0 - b, f1 = cs - b;
  int mn = live && f1 > f0 ? f0 : 0x7fffffff, mx = live && f1 > f0 ? f1 : 0;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    mn = min(mn, __shfl_xor(mn, o, 64));
    mx = max(mx, __shfl_xor(mx, o, 64));
  }
  const int wlo = __builtin_amdgcn_readfirstlane(mn), whi = __builtin_amdgcn_readfirstlane(mx);
  if (lane == 0) { red[0][tid >> 6] = wlo; red[1][tid >> 6] = whi; }
  __syncthreads();
  const int flo = min(min(red[0][0], red[0][1]), min(red[0][2], red[0][3]));
  const int fhi = max(max(red[1][0], red[1][1]), max(red[1][2], red[1][3]));

  float val[RM];
  int ix[RM];
  int cnt = 0;
#pragma unroll
  for (int j = 0; j < RM; ++j) { val[j] = -INFINITY; ix[j] = -1; }

  // LDS tile: columns past D and rows past the tile's end zero (so are q's),
  // and fma(0, 0, acc) == acc keeps the chain exact over the padding
  constexpr int NST = (kRouteTile * DP / 4 + 255) / 256;
  for (int t0 = flo; t0 < fhi; t0 += kRouteTile) {
    const int nt = min(kRouteTile, fhi - t0);
    f32x4_t stg[NST];
#pragma unroll
    for (int i = 0; i < NST; ++i) {
      const int x = tid + 256 * i, r = x / (DP / 4), d = (x % (DP / 4)) * 4;
      stg[i] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
      if (r < nt && d < D)
        stg[i] = *reinterpret_cast<const f32x4_t*>(means + ((int64_t)(t0 + r) * Hkv + kh) * D + d);
    }
    __syncthreads();  // the previous tile is consumed
#pragma unroll
    for (int i = 0; i < NST; ++i) {
      const int x = tid + 256 * i;
      if (x < kRouteTile * DP / 4)
        *reinterpret_cast<f32x4_t*>(mt + (x / (DP / 4)) * LD + (x % (DP / 4)) * 4) = stg[i];
    }
    __syncthreads();
    const int fa = max(wlo, t0), fb = min(whi, t0 + nt);
    // 4 NC candidates from g on, NC independent chains per lane; rows past the
    // tile are read as its last and their scores discarded
    auto group = [&](int g, auto nc_tag) __attribute__((always_inline)) {
      constexpr int NC = decltype(nc_tag)::value;
      const float* row[NC];
      f32x4_t acc[NC];
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        row[k] = mt + min(g - t0 + 4 * k + (lane & 3), kRouteTile - 1) * LD;
        acc[k] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int d4 = 0; d4 < DP / 4; ++d4) {
        f32x4_t m[NC];
#pragma unroll
        for (int k = 0; k < NC; ++k) m[k] = *reinterpret_cast<const f32x4_t*>(row[k] + 4 * d4);
        const u32x4_t w = __builtin_bit_cast(u32x4_t, qv[d4 / 2]);
        const f32x4_t x = late_f32x4<DT>(w[(d4 % 2) * 2], w[(d4 % 2) * 2 + 1]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int k = 0; k < NC; ++k)
            acc[k] = __builtin_amdgcn_mfma_f32_4x4x1f32(m[k][e], x[e], acc[k], 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4 * NC; ++r) {
        const int f = g + r;
        const float score = acc[r / 4][r % 4];
        if (f >= fb || !(live && f >= f0 && f < f1)) continue;
        const int c = f + b;
        if (gate) gate[((int64_t)f * Hq + h) * T + s] = score;
        // stable insertion into the descending list: equal scores stay behind the
        // earlier (lower) chunk, so exact ties resolve to the lowest index.
        if (cnt == R && !(score > val[R - 1])) continue;
        int pos = 0;
#pragma unroll
        for (int j = 0; j < RM; ++j) pos += (j < cnt && val[j] >= score);
#pragma unroll
        for (int j = RM - 1; j >= 1; --j)
          if (j > pos && j < R) { val[j] = val[j - 1]; ix[j] = ix[j - 1]; }
#pragma unroll
        for (int j = 0; j < RM; ++j)
          if (j == pos) { val[j] = score; ix[j] = c; }
        if (cnt < R) cnt++;
      }
    };
    int g = fa;
    for (; fb - g > 8; g += 16) group(g, std::integral_constant<int, 4>{});
    for (; g < fb; g += 8) group(g, std::integral_constant<int, 2>{});
  }
  // ascending chunk order for the slot list (static sorting network)
#pragma unroll
  for (int pass = 0; pass < RM; ++pass) {
#pragma unroll
    for (int j = 0; j + 1 < RM; ++j) {
      if (j + 1 < cnt && ix[j] > ix[j + 1]) { int t = ix[j]; ix[j] = ix[j + 1]; ix[j + 1] = t; }
    }
  }
  if (live) {
    int* out = sel + idx * R;
    for (int j = 0; j < R; ++j) out[j] = j < cnt ? ix[j] : -1;
  }
  if (blk_count == nullptr) return;
  // this workgroup's count of every candidate, for the expert packing
  int fs[kMaxRemote];
#pragma unroll
  for (int j = 0; j < kMaxRemote; ++j) fs[j] = live && j < RM && j < cnt ? ix[j < RM ? j : 0] - b : -1;
  static_assert(sizeof(mt) >= kPickRows * 4 * 8, "the means tile holds the pick bits");
  uint64_t* bits = reinterpret_cast<uint64_t*>(mt);
  int* dst = blk_count + (int64_t)h * gridDim.x + blockIdx.x;
  const int64_t fstep = (int64_t)Hq * gridDim.x;
  for (int f = tid; f < F; f += 256)
    if (f < flo || f >= fhi) dst[f * fstep] = 0;
  for (int t0 = flo; t0 < fhi; t0 += kPickRows) {
    pick_bits(bits, fs, t0);
    const int f = t0 + tid;
    if (f < fhi) {
      const uint64_t* w = bits + 4 * tid;
      dst[f * fstep] = __popcll(w[0]) + __popcll(w[1]) + __popcll(w[2]) + __popcll(w[3]);
    }
  }
}

__global__ void fill_f32_kernel(float* p, int64_t n, float v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ---- expert packing ------------------------------------------------------
// Expert e = f*Hkv + kvh (reference order: (chunk, kv head)).  Its rows are
// the (g, s) that picked chunk f, g-major and s ascending, as the reference's
// nonzero over [F*Hkv, G*T] enumerates them (grouped_attention.py:78-80).
// Blocks of 256 consecutive tokens of one head are counted per candidate
// (blk_count[f][h][block]: an expert's blocks are contiguous and in the order
// of its rows), the counts become offsets within the expert, and each block
// places its picks: no pass reads more than the picks and the counts.
// Scanning every candidate row of every expert for its selection bit, in a
// count and in a fill pass, took 59 us at T 32768, 8 heads, 63 candidates (20
// here), and 25 us at T 8192, 12 heads, 15 candidates (13 here).  What is left
// is latency: selection, chunk, offset and row are four dependent accesses
// (all eight pick slots loaded without branches measured slower, 20 -> 23 us:
// three of them hold picks).

struct PackArgs {
  const int* sel;
  int T, Hq, Hkv, R;
  const int *cu_chunk, *chunk_batch, *cu_seqlens, *filtered;
  int F, block_rows;
  int *counts, *row_off, *tile_off, *rows, *blk;
  int4* tiles;   // remote tile of every workgroup (ExpertTile), or null
  int n_tiles;   // entries of tiles
};

// Filtered index of each pick of (s, h); -1 for none and for an entry that is
// not a candidate of the token (a later chunk, another sequence's).  With
// `at`, also the block's entry of the block counts for each pick; it is
// loaded beside what the check reads, not after it.
MOBA_DEV void load_picks(const PackArgs& a, int s, int h, int (&fs)[kMaxRemote],
                         int (*at)[kMaxRemote] = nullptr, int64_t blk = 0, int nblk = 0) {
  int c[kMaxRemote], b[kMaxRemote];
#pragma unroll
  for (int j = 0; j < kMaxRemote; ++j)
    c[j] = s < a.T && j < a.R ? a.sel[((int64_t)s * a.Hq + h) * a.R + j] : -1;
#pragma unroll
  for (int j = 0; j < kMaxRemote; ++j) b[j] = c[j] >= 0 ? a.chunk_batch[c[j]] : 0;
#pragma unroll
  for (int j = 0; j < kMaxRemote; ++j) {
    fs[j] = -1;
    const int f = c[j] - b[j];
    if (c[j] < 0 || f >= a.F) continue;
    const int n = at ? a.blk[((int64_t)f * a.Hq + h) * nblk + blk] : 0;
    const bool ok = a.filtered[f] == c[j] && s >= a.cu_chunk[c[j] + 1] &&
                    s < a.cu_seqlens[b[j] + 1];
    if (ok) fs[j] = f;
    if (at) (*at)[j] = n;
  }
}

// Block counts of an existing selection (the route kernel writes its own).
__global__ __launch_bounds__(256) void pick_count_kernel(PackArgs a) {
  __shared__ uint64_t bits[kPickRows * 4];
  const int tid = threadIdx.x, h = blockIdx.y;
  int fs[kMaxRemote];
  load_picks(a, blockIdx.x * 256 + tid, h, fs);
  for (int t0 = 0; t0 < a.F; t0 += kPickRows) {
    pick_bits(bits, fs, t0);
    const int f = t0 + tid;
    if (f < a.F) {
      const uint64_t* w = bits + 4 * tid;
      a.blk[((int64_t)f * a.Hq + h) * gridDim.x + blockIdx.x] =
          __popcll(w[0]) + __popcll(w[1]) + __popcll(w[2]) + __popcll(w[3]);
    }
  }
}

// Exclusive scan over the 256 threads of a workgroup; total: the sum.
template <typename I> MOBA_DEV I block_scan_256(I v, I& total, I* part) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  I inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const I y = __shfl_up(inc, o, 64);
    if (lane >= o) inc += y;
  }
  __syncthreads();  // part's earlier use is over
  if (lane == 63) part[w] = inc;
  __syncthreads();
  I before = 0;
  total = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i < w) before += part[i];
    total += part[i];
  }
  return before + inc - v;
}

// One workgroup per expert: its block counts become exclusive offsets, and
// their sum the expert's row count.
__global__ __launch_bounds__(256) void expert_blocks_kernel(int* __restrict__ blk_count, int nblk,
                                                            int Hq, int Hkv,
                                                            int* __restrict__ counts) {
  __shared__ int part[4];
  const int e = blockIdx.x, f = e / Hkv, kh = e % Hkv, G = Hq / Hkv;
  int* c = blk_count + ((int64_t)f * Hq + kh * G) * nblk;
  const int n = G * nblk;
  int run = 0;
  for (int i0 = 0; i0 < n; i0 += 256) {
    const int i = i0 + threadIdx.x;
    int total;
    const int before = block_scan_256(i < n ? c[i] : 0, total, part);
    if (i < n) c[i] = run + before;
    run += total;
  }
  if (threadIdx.x == 0) counts[e] = run;
}

// Exclusive scans of row counts and tile counts over the experts (one
// workgroup; for more experts than a fill workgroup scans by itself).
__global__ __launch_bounds__(256) void expert_scan_kernel(const int* __restrict__ counts, int E,
                                                          int block_rows,
                                                          int* __restrict__ row_off,
                                                          int* __restrict__ tile_off) {
  __shared__ int64_t part[4];
  int64_t run = 0;  // rows in the low half, tiles in the high half
  for (int e0 = 0; e0 < E; e0 += 256) {
    const int e = e0 + threadIdx.x;
    const int r = e < E ? counts[e] : 0;
    int64_t total;
    const int64_t x = run + block_scan_256(
        (int64_t)r | (int64_t)((r + block_rows - 1) / block_rows) << 32, total, part);
    if (e < E) { row_off[e] = (int)x; tile_off[e] = (int)(x >> 32); }
    run += total;
  }
  if (threadIdx.x == 0) { row_off[E] = (int)run; tile_off[E] = (int)(run >> 32); }
}

// The remote kernels' work, workgroup by workgroup: entry L is the tile that
// xcd_contiguous gives workgroup L, as {first key, keys, first row of the row
// list, kv head << 9 | rows}; 0 rows where there is none.  One 16-byte load
// then starts a workgroup that would otherwise search tile_off for its expert
// and follow the expert to its chunk (11 dependent loads at 504 experts): at
// T 32768, 8 heads, chunk 512 the remote dQ kernel went from 494 to 444 us and
// the remote forward from 325 to 317, with the first K / V tile on its way
// before the query rows.
// Workgroup w of nwg fills in the experts w, w + nwg, ... and its share of the
// empty entries.
MOBA_DEV void write_tiles(const PackArgs& a, int e, int row0, int tile0, int total) {
  const int per = (total + 7) >> 3, n = a.counts[e], c = a.filtered[e / a.Hkv];
  const int k_lo = a.cu_chunk[c], nk = a.cu_chunk[c + 1] - k_lo, kh = e % a.Hkv;
  for (int i = threadIdx.x; i * a.block_rows < n; i += 256) {
    const int t = tile0 + i, rows = min(a.block_rows, n - i * a.block_rows);
    const int4 v = {k_lo, nk, row0 + i * a.block_rows, kh << 9 | rows};
    const int L = (t % per) * 8 + t / per;
    if (L < a.n_tiles) a.tiles[L] = v;
  }
}
MOBA_DEV void clear_tiles(const PackArgs& a, int w, int nwg, int total) {
  const int per = (total + 7) >> 3;
  for (int L = w * 256 + threadIdx.x; L < a.n_tiles; L += nwg * 256)
    if ((L >> 3) >= per || (L & 7) * per + (L >> 3) >= total) a.tiles[L] = {0, 0, 0, 0};
}

// Ordered compaction: rows[row_off[e] + rank] = ((s*Hq + h) << 3) | j (R <= 8).
// Workgroup (block, h) places the picks of its 256 tokens.  With SCAN each
// workgroup scans the experts' counts by itself (E <= kScanExperts, 8 loads
// per thread at most) instead of waiting for a one-workgroup launch, and the
// first one writes row_off and tile_off.
constexpr int kScanExperts = 2048;

template <bool SCAN>
__global__ __launch_bounds__(256) void expert_fill_kernel(PackArgs a) {
  __shared__ uint64_t bits[kPickRows * 4];
  __shared__ int64_t off[SCAN ? kScanExperts : 1];  // rows in the low half, tiles in the high half
  __shared__ int64_t part[4];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int blk = blockIdx.x, h = blockIdx.y, nblk = gridDim.x;
  const int Hq = a.Hq, Hkv = a.Hkv, E = a.F * Hkv, block_rows = a.block_rows;
  const int s = blk * 256 + tid, kh = h / (Hq / Hkv);
  int fs[kMaxRemote];
  int at[kMaxRemote];  // the block's first position within each picked expert
  load_picks(a, s, h, fs, &at, blk, nblk);
  int64_t total = 0;
  if constexpr (SCAN) {
    constexpr int PT = kScanExperts / 256;  // consecutive experts per thread
    int n[PT];
    int64_t mine = 0;
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      n[i] = tid * PT + i < E ? a.counts[tid * PT + i] : 0;
      mine += (int64_t)n[i] | (int64_t)((n[i] + block_rows - 1) / block_rows) << 32;
    }
    int64_t x = block_scan_256(mine, total, part);
    const bool first = blk == 0 && h == 0;
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int e = tid * PT + i;
      if (e < E) {
        off[e] = x;
        if (first) { a.row_off[e] = (int)x; a.tile_off[e] = (int)(x >> 32); }
      }
      x += (int64_t)n[i] | (int64_t)((n[i] + block_rows - 1) / block_rows) << 32;
    }
    if (first && tid == 0) { a.row_off[E] = (int)total; a.tile_off[E] = (int)(total >> 32); }
  }
#pragma unroll
  for (int j = 0; j < kMaxRemote; ++j) {
    if (!SCAN && fs[j] >= 0) at[j] += a.row_off[fs[j] * Hkv + kh];
  }
  for (int t0 = 0; t0 < a.F; t0 += kPickRows) {
    pick_bits(bits, fs, t0);  // its barriers order the writes of off, too
#pragma unroll
    for (int j = 0; j < kMaxRemote; ++j) {
      const int r = fs[j] - t0;
      if (fs[j] < 0 || r < 0 || r >= kPickRows) continue;
      const uint64_t* b = bits + 4 * r;
      int rank = __popcll(b[w] & ((1ull << lane) - 1ull));
      for (int i = 0; i < w; ++i) rank += __popcll(b[i]);
      const int base = at[j] + (SCAN ? (int)off[fs[j] * Hkv + kh] : 0);
      a.rows[base + rank] = ((s * Hq + h) << 3) | j;
    }
  }
  if (a.tiles == nullptr) return;
  const int wg = h * nblk + blk, nwg = nblk * Hq;
  const int ntiles = SCAN ? (int)(total >> 32) : a.tile_off[E];
  for (int e = wg; e < E; e += nwg)
    write_tiles(a, e, SCAN ? (int)off[e] : a.row_off[e],
                SCAN ? (int)(off[e] >> 32) : a.tile_off[e], ntiles);
  clear_tiles(a, wg, nwg, ntiles);
}

int64_t pick_blocks(int T) { return ((int64_t)T + 255) / 256; }

// Offsets and rows from the block counts in a.blk.
void launch_pack(const PackArgs& a, hipStream_t st) {
  const int E = a.F * a.Hkv, nblk = (int)pick_blocks(a.T);
  hipLaunchKernelGGL(expert_blocks_kernel, dim3(E), dim3(256), 0, st, a.blk, nblk, a.Hq, a.Hkv,
                     a.counts);
  const dim3 grid(nblk, a.Hq);
  if (E <= kScanExperts) {
    hipLaunchKernelGGL(expert_fill_kernel<true>, grid, dim3(256), 0, st, a);
  } else {
    hipLaunchKernelGGL(expert_scan_kernel, dim3(1), dim3(256), 0, st, a.counts, E, a.block_rows,
                       a.row_off, a.tile_off);
    hipLaunchKernelGGL(expert_fill_kernel<false>, grid, dim3(256), 0, st, a);
  }
}

}  // namespace

extern "C" int moba_hip_chunk_means(const void* k, int dtype, int T, int Hkv, int D,
                                    const int* chunk_start, int F, int chunk, int precision,
                                    float* means, void* stream) {
  (void)T;
  if (F <= 0) return MOBA_OK;
  if (dtype != 0 && dtype != 1) { moba_set_error("chunk_means: dtype must be 0 (bf16) or 1 (fp16)"); return MOBA_ERR_ARG; }
  if (D < 8 || D % 8 || Hkv < 1 || chunk < 1) { moba_set_error("chunk_means: bad shape"); return MOBA_ERR_ARG; }
  if (D > 256) { moba_set_error("chunk_means: head_dim must be at most 256"); return MOBA_ERR_ARG; }
  // dim slices per (chunk, kv head), until the grid has about 512 workgroups,
  // each slice at least 128 bytes of a key row (whole 128-byte lines; 64 when
  // there are fewer than 64 (chunk, kv head) pairs)
  int ds = 1;
  const int64_t wgs = (int64_t)F * Hkv;
  while ((D / 8) % (2 * ds) == 0 && D / 8 / (2 * ds) >= (wgs < 64 ? 4 : 8) && wgs * ds < 512) ds *= 2;
  dim3 grid((unsigned)((int64_t)F * Hkv * ds)), block(256);
  const size_t lds = (size_t)64 * D * sizeof(float);
  hipStream_t st = (hipStream_t)stream;
  const uint16_t* kp = (const uint16_t*)k;
#define MOBA_MEANS(DT_, NP_) \
  hipLaunchKernelGGL((chunk_means_kernel<DT_, NP_>), grid, block, lds, st, kp, Hkv, D, chunk_start, \
                     chunk, precision, ds, means)
  const int nd8 = D / 8 / ds;
  if (dtype == 0) {
    if (nd8 <= 4) MOBA_MEANS(0, 1); else if (nd8 <= 8) MOBA_MEANS(0, 2);
    else if (nd8 <= 16) MOBA_MEANS(0, 4); else MOBA_MEANS(0, 8);
  } else {
    if (nd8 <= 4) MOBA_MEANS(1, 1); else if (nd8 <= 8) MOBA_MEANS(1, 2);
    else if (nd8 <= 16) MOBA_MEANS(1, 4); else MOBA_MEANS(1, 8);
  }
#undef MOBA_MEANS
  return moba_launch_status("chunk_means");
}

static int route_prefill(const void* q, int dtype, int T, int Hq, int Hkv, int D,
                         const float* means, const int* cu_chunk, int nchunk,
                         const int* chunk_batch, const int* first_chunk, int R, int F, int* sel,
                         float* gate, int* blk_count, hipStream_t st) {
  if (R < 1 || R > kMaxRemote) { moba_set_error("route_prefill: remote count must be in [1,8]"); return MOBA_ERR_ARG; }
  if (D % 8 || D < 8) { moba_set_error("route_prefill: head_dim must be a multiple of 8"); return MOBA_ERR_ARG; }
  if (Hq % Hkv) { moba_set_error("route_prefill: Hq must be a multiple of Hkv"); return MOBA_ERR_ARG; }
  if (gate) {
    const int64_t n = (int64_t)F * Hq * T;
    hipLaunchKernelGGL(fill_f32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, gate,
                       n, -INFINITY);
  }
  if (D > 256) { moba_set_error("route_prefill: head_dim must be at most 256"); return MOBA_ERR_ARG; }
  dim3 grid((unsigned)((T + 255) / 256), (unsigned)Hq), block(256);
  const uint16_t* qp = (const uint16_t*)q;
#define MOBA_ROUTE(DT_, DP_, RM_) \
  hipLaunchKernelGGL((route_kernel<DT_, DP_, RM_>), grid, block, 0, st, qp, T, Hq, Hkv, D, means, \
                     cu_chunk, nchunk, chunk_batch, first_chunk, R, F, sel, gate, blk_count)
#define MOBA_ROUTE_RM(DT_, DP_) \
  if (R <= 4) MOBA_ROUTE(DT_, DP_, 4); else MOBA_ROUTE(DT_, DP_, 8);
#define MOBA_ROUTE_DT(DT_) \
  if (D <= 64) { MOBA_ROUTE_RM(DT_, 64) } else if (D <= 128) { MOBA_ROUTE_RM(DT_, 128) } \
  else { MOBA_ROUTE_RM(DT_, 256) }
  if (dtype == 0) {
    MOBA_ROUTE_DT(0)
  } else {
    MOBA_ROUTE_DT(1)
  }
#undef MOBA_ROUTE_DT
#undef MOBA_ROUTE_RM
#undef MOBA_ROUTE
  return moba_launch_status("route_prefill");
}

extern "C" int moba_hip_route_prefill(const void* q, int dtype, int T, int Hq, int Hkv, int D,
                                      const float* means, const int* cu_chunk, int nchunk,
                                      const int* chunk_batch, const int* first_chunk, int R,
                                      int F, int* sel, float* gate, void* stream) {
  return route_prefill(q, dtype, T, Hq, Hkv, D, means, cu_chunk, nchunk, chunk_batch, first_chunk,
                       R, F, sel, gate, nullptr, (hipStream_t)stream);
}

// Work ints of the expert packing: the block counts of every (candidate, head).
extern "C" int64_t moba_hip_pack_experts_work(int T, int Hq, int Hkv, int F) {
  if (T < 0 || Hq < 1 || Hkv < 1 || Hq % Hkv || F < 0) return -1;
  return (int64_t)F * Hq * pick_blocks(T);
}

static int check_pack(int T, int Hq, int Hkv, int R, const int* work) {
  if ((int64_t)T * Hq * R >= (1ll << 31) || (int64_t)T * Hq >= (1ll << 28)) { moba_set_error("pack_experts: T*Hq*R exceeds int32 or T*Hq exceeds 2^28"); return MOBA_ERR_ARG; }
  if (R > 8) { moba_set_error("pack_experts: at most 8 remote chunks per query"); return MOBA_ERR_ARG; }
  if (Hkv < 1 || Hq % Hkv) { moba_set_error("pack_experts: Hq must be a multiple of Hkv"); return MOBA_ERR_ARG; }
  if (work == nullptr || ((uintptr_t)work & 7)) { moba_set_error("pack_experts: the work buffer (moba_hip_pack_experts_work ints, 8-byte aligned) is required"); return MOBA_ERR_ARG; }
  return MOBA_OK;
}

extern "C" int moba_hip_pack_experts(const int* sel, int T, int Hq, int Hkv, int R,
                                     const int* cu_chunk, const int* chunk_batch,
                                     const int* cu_seqlens, const int* filtered, int F,
                                     int block_rows, int* counts, int* row_off, int* tile_off,
                                     int* rows, int* work, void* stream) {
  if (F <= 0) return MOBA_OK;
  if (int rc = check_pack(T, Hq, Hkv, R, work)) return rc;
  if (T < 1) return MOBA_OK;
  hipStream_t st = (hipStream_t)stream;
  const PackArgs a = {sel, T, Hq, Hkv, R, cu_chunk, chunk_batch, cu_seqlens, filtered, F,
                      block_rows, counts, row_off, tile_off, rows, work, nullptr, 0};
  hipLaunchKernelGGL(pick_count_kernel, dim3((unsigned)pick_blocks(T), Hq), dim3(256), 0, st, a);
  launch_pack(a, st);
  return moba_launch_status("pack_experts");
}

extern "C" int moba_hip_prefill_route(const void* q, const void* k, int dtype, int T, int Hq,
                                      int Hkv, int D, const int* chunk_start, int chunk,
                                      int precision, const int* cu_chunk, int nchunk,
                                      const int* chunk_batch, const int* first_chunk,
                                      const int* cu_seqlens, const int* filtered, int R, int F,
                                      int block_rows, float* means, int* sel, float* gate,
                                      int* counts, int* row_off, int* tile_off, int* rows,
                                      int* tiles, int n_tiles, int* work, void* stream) {
  if (F <= 0) return MOBA_OK;
  if (tiles && (n_tiles < 1 || block_rows > 511 || ((uintptr_t)tiles & 15))) { moba_set_error("prefill_route: tiles must hold n_tiles 16-byte aligned entries of at most 511 rows"); return MOBA_ERR_ARG; }
  if (Hkv < 1 || Hq < 1) { moba_set_error("prefill_route: bad head counts"); return MOBA_ERR_ARG; }
  if (int rc = check_pack(T, Hq, Hkv, R, work)) return rc;
  if (int rc = moba_hip_chunk_means(k, dtype, T, Hkv, D, chunk_start, F, chunk, precision, means,
                                    stream)) return rc;
  hipStream_t st = (hipStream_t)stream;
  if (int rc = route_prefill(q, dtype, T, Hq, Hkv, D, means, cu_chunk, nchunk, chunk_batch,
                             first_chunk, R, F, sel, gate, work, st)) return rc;
  launch_pack({sel, T, Hq, Hkv, R, cu_chunk, chunk_batch, cu_seqlens, filtered, F, block_rows,
               counts, row_off, tile_off, rows, work, (int4*)tiles, n_tiles}, st);
  return moba_launch_status("prefill_route");
}
