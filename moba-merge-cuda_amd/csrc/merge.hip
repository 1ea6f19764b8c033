// Standalone deterministic global-softmax merge of caller-owned partials.
//
// Replaces merge_forward (src/moba_opt/ops/bindings.cpp:6-22,
// src/moba_opt/ops/merge.cu:187-288): row p of the output combines the self
// partial (self_out[p], self_lse[p]) with every remote partial j whose
// mapping[j] == p,
//     m = max(l_self, l_j),  w = exp(l - m),  z = sum_j w_j + w_self,
//     O = (w_self o_self + sum_j w_j o_j) / z,  L = m + log z,
// O in the input dtype, L fp32 natural log.  The reference builds per-row
// slot lists with atomic tickets (order depends on timing) and, in its
// deterministic mode, sorts each row's slots afterwards.  Here a row has kmax
// slots that hold its smallest remote indices in ascending order whatever
// order they arrive in: an index enters slot 0 by an integer minimum, the
// larger of it and what it met goes on to slot 1, and so on.  Every slot then
// sees each index that the slots before it did not keep, so slot i ends with
// the row's i-th smallest index.  No floating-point value passes through an
// atomic; the merge adds a row's partials in slot order.  Results are bitwise
// repeatable.
//
// Three launches on the stream (all sizes from the arguments; the host never
// waits): empty slots and status words, insertion (one thread per remote
// partial), merge.  status[0] = 1 when a mapping entry is outside [0, T*H)
// (such entries are ignored), status[1] = 1 when a row has more than kmax
// remote partials (only the first kmax, in j order, are used); the caller
// reads them after the stream reaches them.
//
// The work is bound by memory: every partial and every output once.  At T
// 16384, 14 heads, D 64, bf16, 344K remote partials (107 MB) the three
// launches take 2 + 20 + 20 us (the last at 5.4 TB/s); ordering the partials
// by a radix sort on the row (three digit passes of histogram, one-workgroup
// scan and scatter, 530 us) before a one-wave-per-row merge (85 us) took 620.
#include "common.h"
#include "../../include/moba_hip.h"

using namespace moba;

namespace {

constexpr int kEmpty = 0x7fffffff;  // slot without a partial: above every index

__global__ __launch_bounds__(256) void merge_init_kernel(int* slots, int64_t P, int kmax,
                                                         int* status) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i == 0) { status[0] = 0; status[1] = 0; }
  if (i >= P) return;
  for (int r = 0; r < kmax; ++r) slots[r * P + i] = kEmpty;
}

// One thread per remote partial.  A partial usually finds its row's first
// free slot in one or two minima (kmax bounds them), the rows of a launch
// rarely meet, and what bounds the kernel is the latency of those returns.
//
// Where rows do meet, minima on one address are served one by one, 11 ns each.
// So a wave's lanes of one row are found (each leaves its number at a hash of
// its row; a lane that reads another lane of its row there has company) and
// numbered: the lane of rank r has r smaller indices beside it, so it can start
// at slot r, and from rank kmax on it is not among the row's first kmax.  From
// four of them on they look before each minimum (fewer meet by chance, and a
// look is a memory latency): a slot only ever falls, so one that reads below x,
// be it stale, will not take x.
// Whole call, 344K partials, kmax 8, us, without -> with this (the radix sort
// took 590 in each case): one row 31247 -> 179, every other partial of one row
// 15654 -> 256, 16 rows in turn 2014 -> 342, 64 rows in turn (never two in a
// wave) 665 -> 665, sorted runs of eight 139 -> 67, spread 79 -> 79; T 16384, 14
// heads, kmax 2: 67.3 -> 67.4.
constexpr int kRowHash = 256;

template <typename MT>
__global__ __launch_bounds__(256) void merge_insert_kernel(const MT* __restrict__ mapping,
                                                           int64_t n, int64_t P, int kmax,
                                                           int* slots, int* status) {
  __shared__ uint8_t last[4][kRowHash];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t m = j < n ? (int64_t)mapping[j] : 0;
  const bool ok = j < n && m >= 0 && m < P;
  if (j < n && !ok) status[0] = 1;
  const int p = ok ? (int)m : -1;
  uint8_t* at = &last[w][(uint32_t)p * 2654435761u >> 24];
  if (ok) *at = (uint8_t)lane;
  wave_lds_sync();
  const int mate = ok ? *at : lane;
  const bool met = __shfl(p, mate, 64) == p && mate != lane;  // -1: its own lane
  int* row = slots + (int64_t)p * kmax;
  int x = (int)j, i = 0;
  uint64_t todo = __ballot(met);
  if (todo != 0) {  // uniform
    bool crowd = false;
    for (; todo != 0;) {
      const bool mine = p == __builtin_amdgcn_readlane(p, __ffsll((unsigned long long)todo) - 1);
      const uint64_t mates = __ballot(mine);
      if (mine) {
        i = __popcll(mates & ((1ull << lane) - 1ull));
        crowd = __popcll(mates) >= 4;
      }
      todo &= ~mates;
    }
    auto look = [&](int k) { return __hip_atomic_load(row + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    if (crowd) {
      if (i < kmax && look(kmax - 1) < x) i = kmax;
      for (; i < kmax; ++i) {
        if (look(i) < x) continue;
        const int old = atomicMin(row + i, x);
        x = max(old, x);
        if (x == kEmpty) return;
      }
      status[1] = 1;  // more than kmax: an index has no slot
      return;
    }
  }
  if (!ok) return;
  for (; i < kmax; ++i) {
    const int old = atomicMin(row + i, x);
    x = max(old, x);
    if (x == kEmpty) return;
  }
  status[1] = 1;
}

// 16 bytes of a row: 8 elements (16-bit types) or 4 (fp32).
template <int DT> constexpr int vec_elems() { return DT == 2 ? 4 : 8; }
template <int DT>
MOBA_DEV void load_vec(const void* base, int64_t off, float (&x)[vec_elems<DT>()]) {
  if constexpr (DT == 2) {
    const f32x4_t v = *reinterpret_cast<const f32x4_t*>(static_cast<const float*>(base) + off);
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = v[e];
  } else {
    const u16x8_t v = ld8(static_cast<const uint16_t*>(base) + off);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = to_f32<DT>(v[e]);
  }
}

// 2^lshift lanes per row, 16 bytes of the row each, so a wave covers several
// rows of a small head dim; every lane of a row holds the row's slots and
// weights.  All of a row's loads are issued together: a slot without a
// partial loads the self partial in its place (the address is always valid)
// and is left out of the sums by a select, never by a zero weight.
// K: slots loaded per row, kmax <= K.
template <int DT, int K>
__global__ __launch_bounds__(256) void merge_rows_kernel(
    const void* __restrict__ self_out, const float* __restrict__ self_lse,
    const void* __restrict__ remote_out, const float* __restrict__ remote_lse,
    const int* __restrict__ slots, int64_t P, int D, int lshift, int kmax,
    void* __restrict__ out, float* __restrict__ lse) {
  constexpr int V = vec_elems<DT>();
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t p = t >> lshift;
  const int d = ((int)t & ((1 << lshift) - 1)) * V;
  if (p >= P || d >= D) return;
  int idx[K];
#pragma unroll
  for (int i = 0; i < K; ++i) idx[i] = slots[p * kmax + min(i, kmax - 1)];
  const float l_self = self_lse[p];
  float l[K], x[K][V], acc[V];
  load_vec<DT>(self_out, p * D + d, acc);
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const bool on = i < kmax && idx[i] != kEmpty;
    l[i] = *(on ? remote_lse + idx[i] : self_lse + p);
    load_vec<DT>(on ? remote_out : self_out, (on ? (int64_t)idx[i] : p) * D + d, x[i]);
  }
  float m = l_self;
#pragma unroll
  for (int i = 0; i < K; ++i) m = fmaxf(m, l[i]);
  const float w_self = expf(l_self - m);
#pragma unroll
  for (int e = 0; e < V; ++e) acc[e] *= w_self;
  float z = 0.0f;  // remote weights in slot order, then self
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const bool on = i < kmax && idx[i] != kEmpty;
    const float w = expf(l[i] - m);
    z = on ? z + w : z;
#pragma unroll
    for (int e = 0; e < V; ++e) acc[e] = on ? acc[e] + w * x[i][e] : acc[e];
  }
  z += w_self;
  const float iz = 1.0f / z;
  if constexpr (DT == 2) {
    f32x4_t o;
#pragma unroll
    for (int e = 0; e < V; ++e) o[e] = acc[e] * iz;
    *reinterpret_cast<f32x4_t*>(static_cast<float*>(out) + p * D + d) = o;
  } else {
#pragma unroll
    for (int e = 0; e < V; ++e) acc[e] *= iz;
    st8(static_cast<uint16_t*>(out) + p * D + d, pack8<DT>(acc));
  }
  if (d == 0) lse[p] = m + logf(z);
}

struct MergeArgs {
  const void *self_out, *remote_out;
  const float *self_lse, *remote_lse;
  int* slots;
  int64_t P;
  int D, kmax;
  void* out;
  float* lse;
};

template <int DT>
void launch_rows(const MergeArgs& a, hipStream_t st) {
  int lshift = 0;
  while ((vec_elems<DT>() << lshift) < a.D) ++lshift;
  const dim3 grid((unsigned)(((a.P << lshift) + 255) / 256));
#define MOBA_MERGE(K_)                                                                           \
  hipLaunchKernelGGL((merge_rows_kernel<DT, K_>), grid, dim3(256), 0, st, a.self_out,            \
                     a.self_lse, a.remote_out, a.remote_lse, a.slots, a.P, a.D, lshift, a.kmax,  \
                     a.out, a.lse)
  if (a.kmax <= 1) MOBA_MERGE(1); else if (a.kmax <= 2) MOBA_MERGE(2);
  else if (a.kmax <= 4) MOBA_MERGE(4); else MOBA_MERGE(8);
#undef MOBA_MERGE
}

template <typename MT>
int merge(const void* self_out, const float* self_lse, const void* remote_out,
          const float* remote_lse, const MT* mapping, int dtype, int64_t T, int H, int D,
          int64_t M, int kmax, void* work, int* status, void* out, float* lse, void* stream) {
  if (dtype < 0 || dtype > 2) { moba_set_error("merge: dtype must be 0 (bf16), 1 (fp16) or 2 (fp32)"); return MOBA_ERR_ARG; }
  if (T < 1 || H < 1) { moba_set_error("merge: nonempty T,H required"); return MOBA_ERR_ARG; }
  if (D < 8 || D > 256 || D % 8) { moba_set_error("merge: head_dim must be a multiple of 8 in [8,256]"); return MOBA_ERR_ARG; }
  if (kmax < 1 || kmax > 8) { moba_set_error("merge: kmax must be in [1,8]"); return MOBA_ERR_ARG; }
  const int64_t P = T * H;
  if (P >= INT32_MAX || M < 0 || M >= INT32_MAX) { moba_set_error("merge: mapping exceeds int32 indexing capacity"); return MOBA_ERR_ARG; }
  if (!self_out || !self_lse || !out || !lse || !status || !work || (M > 0 && (!remote_out || !remote_lse || !mapping))) {
    moba_set_error("merge: null buffer");
    return MOBA_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  int* slots = static_cast<int*>(work);
  hipLaunchKernelGGL(merge_init_kernel, dim3((unsigned)((P + 255) / 256)), dim3(256), 0, st, slots, P,
                     kmax, status);
  if (M > 0)
    hipLaunchKernelGGL(merge_insert_kernel<MT>, dim3((unsigned)((M + 255) / 256)), dim3(256), 0,
                       st, mapping, M, P, kmax, slots, status);
  const MergeArgs a = {self_out, remote_out, self_lse, remote_lse, slots, P, D, kmax, out, lse};
  if (dtype == 0) launch_rows<0>(a, st);
  else if (dtype == 1) launch_rows<1>(a, st);
  else launch_rows<2>(a, st);
  return moba_launch_status("merge");
}

}  // namespace

extern "C" int64_t moba_hip_merge_work(int64_t P, int64_t M) {
  if (P < 1 || M < 0 || P >= INT32_MAX || M >= INT32_MAX) return -1;
  return P * 8 * (int64_t)sizeof(int);  // slots for the largest kmax
}

extern "C" int moba_hip_merge(const void* self_out, const float* self_lse, const void* remote_out,
                              const float* remote_lse, const int64_t* mapping, int dtype,
                              int64_t T, int H, int D, int64_t M, int kmax, void* work,
                              int* status, void* out, float* lse, void* stream) {
  return merge(self_out, self_lse, remote_out, remote_lse, mapping, dtype, T, H, D, M, kmax, work,
               status, out, lse, stream);
}

extern "C" int moba_hip_merge_i32(const void* self_out, const float* self_lse,
                                  const void* remote_out, const float* remote_lse,
                                  const int32_t* mapping, int dtype, int64_t T, int H, int D,
                                  int64_t M, int kmax, void* work, int* status, void* out,
                                  float* lse, void* stream) {
  return merge(self_out, self_lse, remote_out, remote_lse, mapping, dtype, T, H, D, M, kmax, work,
               status, out, lse, stream);
}
