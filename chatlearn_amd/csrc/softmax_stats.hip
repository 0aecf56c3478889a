// Softmax statistics (logprob, entropy, lse) from materialised logits and the
// matching d(logits), for call sites that already hold [R, V] logits.
// One block per row, 16 bytes per lane and four loads in flight per thread; the row is streamed once for the
// statistics (online max / sum / weighted sum, fp32).  The backward reads it once more and writes
// d(logits), taking lse / entropy from the forward when the caller kept them.  HBM-bound:
// V*sizeof(dtype) bytes per row read (+ the same written).  A row may start anywhere: what lies before its first
// and behind its last 16-byte boundary goes element by element, the rest in 16-byte pieces (519 rows of 32003 fp32,
// three quarters of them misaligned: 48 -> 16 us, gradients 73 -> 28 us; as bf16 47 -> 13 and 46 -> 17.5 us).
// 2048 rows of the 152k vocabulary, bf16: statistics 111 us = 5.6 TB/s, gradients 190 us = 6.5 TB/s (a part of it the last-level
// cache's, see kKeptBytes), where a copy of 1 GB reaches 5.0 TB/s on this card.
#include "common.hpp"

namespace clgrpo {

template <typename T> __device__ __forceinline__ float to_f32(T v);
template <> __device__ __forceinline__ float to_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ float to_f32<__bf16>(__bf16 v) { return (float)v; }

struct RowStats { float m, s, u; };

__device__ __forceinline__ void rs_merge(RowStats& a, const RowStats& b) {
  const float nm = fmaxf(a.m, b.m);
  const float fa = (a.m == nm) ? 1.f : expf(a.m - nm);
  const float fb = (b.m == nm) ? 1.f : expf(b.m - nm);
  a.s = a.s * fa + b.s * fb;
  a.u = a.u * fa + b.u * fb;
  a.m = nm;
}

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// 16 bytes of a row as floats.
template <typename T> struct Vec16 {
  static constexpr int N = 16 / (int)sizeof(T);
  __device__ static __forceinline__ void unpack(const u32x4_t& raw, float (&z)[N]) {
    const T* e = reinterpret_cast<const T*>(&raw);
#pragma unroll
    for (int k = 0; k < N; ++k) z[k] = to_f32<T>(e[k]);
  }
  __device__ static __forceinline__ u32x4_t pack(const float (&d)[N]) {
    alignas(16) T e[N];
#pragma unroll
    for (int k = 0; k < N; ++k) e[k] = (T)d[k];
    return *reinterpret_cast<const u32x4_t*>(e);
  }
};

// Online (max, sum e^{z-max}, sum e^{z-max} z) update with N new values: one rescale, then N exponentials
// against a fixed maximum (no per-element branch).
template <int N>
__device__ __forceinline__ void rs_update(RowStats& st, const float (&z)[N]) {
  float vmax = z[0];
#pragma unroll
  for (int k = 1; k < N; ++k) vmax = fmaxf(vmax, z[k]);
  constexpr float kLog2e = 1.4426950408889634f;
  if (vmax > st.m) {
    const float f = __builtin_amdgcn_exp2f((st.m - vmax) * kLog2e);   // st.m = -inf -> 0
    st.s *= f;
    st.u *= f;
    st.m = vmax;
  }
  // Only -inf so far: every term is 0, and so it is for what lies below -2e38 (entries masked with the type's lowest
  // value), where -m log2(e) overflows and an infinite sum would outlive the rescale to the first ordinary entry.
  const float nb = (st.m == -INFINITY) ? 0.f : -fmaxf(st.m, -2e38f) * kLog2e;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const float e = __builtin_amdgcn_exp2f(fmaf(z[k], kLog2e, nb));   // one hardware exp2 per element
    st.s += e;
    st.u = fmaf(e, z[k], st.u);
  }
}

// A row of V elements from `row`: elements before the first 16-byte boundary, whole pieces, the rest.
template <typename T>
struct RowSpan {
  static constexpr int N = Vec16<T>::N;
  int head, tail;
  int64_t pieces;
  const u32x4_t* vec;
  __device__ __forceinline__ RowSpan(const T* row, int64_t V) {
    head = (int)((16 - (reinterpret_cast<uintptr_t>(row) & 15)) & 15) / (int)sizeof(T);
    if (head > V) head = (int)V;
    pieces = (V - head) / N;
    tail = (int)(V - head - pieces * N);
    vec = reinterpret_cast<const u32x4_t*>(row + head);
  }
  // the element outside the pieces that thread `tid` takes, or -1 (head and tail have at most 7 each)
  __device__ __forceinline__ int64_t loose(int tid) const {
    if (tid < head) return tid;
    if (tid >= 32 && tid - 32 < tail) return head + pieces * N + (tid - 32);
    return -1;
  }
};

// What passes over logits leave in the last-level cache (256 MB), which allocates on loads and stores alike: with more logits than
// fit, each line that a pass brings in pushes one out that was written before and has to go to memory first.  Such passes
// go around the cache (kOnce) where nobody will find in it what they bring: the statistics for all rows but the last kKeptBytes; the
// gradients, which take the rows from the last one on, for their loads and for the stores in front of which another
// kKeptGradients follow.  Fewer logits are better off in the cache altogether.
//   logits just written -> statistics -> gradients -> a pass that reads the gradients, us:  2048 rows of the 152k vocabulary, bf16
//   566 -> 502, 800 235 -> 210, 600 175 -> 167, 4096 of 129280 913 -> 873, 1024 of 50257 fp32 184 -> 168; statistics alone 146 -> 111
//   for 2048 rows.  With all of it around the cache 300 rows of 152k (91 MB) 100 -> 107, 519 of 32003 fp32 76 -> 86; with all
//   gradients stored around it 514 and 179 for the 502 and 168.
constexpr int64_t kKeptBytes = 160 << 20, kKeptGradients = 128 << 20;

// Copies of a loop and not a condition inside it: the compiler makes one access of the two sides, without the hint.
template <bool kOnce>
__device__ __forceinline__ u32x4_t load16(const u32x4_t* p) {
  if constexpr (kOnce) return __builtin_nontemporal_load(p);
  else return *p;
}
template <bool kOnce>
__device__ __forceinline__ void store16(u32x4_t v, u32x4_t* p) {
  if constexpr (kOnce) __builtin_nontemporal_store(v, p);
  else *p = v;
}

template <typename T, int BLOCK, bool kOnce>
__device__ RowStats row_stats(const T* row, int64_t V) {
  constexpr int N = Vec16<T>::N;
  RowStats st{-INFINITY, 0.f, 0.f};
  const RowSpan<T> span(row, V);
  const u32x4_t* rv = span.vec;
  int64_t i = threadIdx.x;
  // two independent running states per thread (merged below): the update is a dependent chain; the next four pieces
  // are requested before the current four are worked on
  RowStats st2{-INFINITY, 0.f, 0.f};
  auto four = [&](const u32x4_t (&r)[4]) {
    float z[N], y[N];
    Vec16<T>::unpack(r[0], z); Vec16<T>::unpack(r[1], y);
    rs_update<N>(st, z); rs_update<N>(st2, y);
    Vec16<T>::unpack(r[2], z); Vec16<T>::unpack(r[3], y);
    rs_update<N>(st, z); rs_update<N>(st2, y);
  };
  if (i + 3 * BLOCK < span.pieces) {
    u32x4_t cur[4], nxt[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) cur[k] = load16<kOnce>(rv + i + k * BLOCK);
    for (i += 4 * BLOCK; i + 3 * BLOCK < span.pieces; i += 4 * BLOCK) {
#pragma unroll
      for (int k = 0; k < 4; ++k) nxt[k] = load16<kOnce>(rv + i + k * BLOCK);
      __builtin_amdgcn_sched_barrier(0);
      four(cur);
#pragma unroll
      for (int k = 0; k < 4; ++k) cur[k] = nxt[k];
    }
    four(cur);
  }
  for (; i < span.pieces; i += BLOCK) {
    float z[N];
    Vec16<T>::unpack(rv[i], z);
    rs_update<N>(st, z);
  }
  const int64_t loose = span.loose(threadIdx.x);
  if (loose >= 0) {
    const float z[1] = {to_f32<T>(row[loose])};
    rs_update<1>(st2, z);
  }
  rs_merge(st, st2);
  auto fold = [&](int from) {
    for (int off = from; off > 0; off >>= 1) {
      RowStats o{__shfl_xor(st.m, off), __shfl_xor(st.s, off), __shfl_xor(st.u, off)};
      rs_merge(st, o);
    }
  };
  fold(32);
  __shared__ RowStats sh[BLOCK / 64];
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = st;
  __syncthreads();
  st = sh[threadIdx.x % (BLOCK / 64)];     // every wave folds all waves' results
  fold(BLOCK / 128);
  return st;
}

template <typename T, int BLOCK>
__global__ __launch_bounds__(BLOCK) void softmax_stats_kernel(clgrpo_softmax_stats_args a) {
  const int64_t r = blockIdx.x;
  const T* row = static_cast<const T*>(a.logits) + r * a.ld;
  const bool once = (a.R - r) * a.ld * (int64_t)sizeof(T) > kKeptBytes;
  const RowStats st = once ? row_stats<T, BLOCK, true>(row, a.V) : row_stats<T, BLOCK, false>(row, a.V);
  if (threadIdx.x == 0) {
    const float lse = st.m + logf(st.s);
    if (a.lse) a.lse[r] = lse;
    if (a.entropy) a.entropy[r] = lse - st.u / st.s;
    if (a.logprob) {
      const int64_t y = a.labels[r];
      a.logprob[r] = (y >= 0 && y < a.V) ? to_f32<T>(row[y]) - lse : NAN;
    }
  }
}

// d(logits) of one row: with the row's lse (and entropy, when it carries a gradient) from the forward the
// row is read once and written once; without them the statistics are rebuilt by one more pass over it.
template <typename T, int BLOCK, bool kOnce>
__device__ __forceinline__ void row_gradients(const clgrpo_softmax_stats_bwd_args& a, int64_t r, float lse, float ent) {
  constexpr int N = Vec16<T>::N;
  const T* row = static_cast<const T*>(a.logits) + r * a.ld;
  T* out = static_cast<T*>(a.dlogits) + r * a.V;
  const float glp = a.g_logprob ? a.g_logprob[r] : 0.f;
  const float gen = a.g_entropy ? a.g_entropy[r] : 0.f;
  const int64_t y = a.g_logprob ? a.labels[r] : -1;
  auto dz = [&](float z, int64_t v) {
    const float logp = z - lse;
    const float p = __builtin_amdgcn_exp2f(logp * 1.4426950408889634f);
    float d = -p * (glp + gen * (logp + ent));
    if (v == y) d += glp;
    return d;
  };
  if (((reinterpret_cast<uintptr_t>(row) ^ reinterpret_cast<uintptr_t>(out)) & 15) == 0) {
    const RowSpan<T> span(row, a.V);
    const u32x4_t* rv = span.vec;
    u32x4_t* ov = reinterpret_cast<u32x4_t*>(out + span.head);
    auto one = [&](const u32x4_t& raw, int64_t i) {
      float z[N], d[N];
      Vec16<T>::unpack(raw, z);
#pragma unroll
      for (int k = 0; k < N; ++k) d[k] = dz(z[k], span.head + i * N + k);
      store16<kOnce>(Vec16<T>::pack(d), ov + i);
    };
    int64_t i = threadIdx.x;
    for (; i + 3 * BLOCK < span.pieces; i += 4 * BLOCK) {
      const u32x4_t r0 = load16<kOnce>(rv + i), r1 = load16<kOnce>(rv + i + BLOCK), r2 = load16<kOnce>(rv + i + 2 * BLOCK),
                    r3 = load16<kOnce>(rv + i + 3 * BLOCK);
      one(r0, i); one(r1, i + BLOCK); one(r2, i + 2 * BLOCK); one(r3, i + 3 * BLOCK);
    }
    for (; i < span.pieces; i += BLOCK) one(rv[i], i);
    const int64_t loose = span.loose(threadIdx.x);
    if (loose >= 0) out[loose] = (T)dz(to_f32<T>(row[loose]), loose);
  } else {
    // rows a stride apart that shifts them against the packed result
    for (int64_t v = threadIdx.x; v < a.V; v += BLOCK) out[v] = (T)dz(to_f32<T>(row[v]), v);
  }
}
template <typename T, int BLOCK>
__global__ __launch_bounds__(BLOCK) void softmax_stats_bwd_kernel(clgrpo_softmax_stats_bwd_args a) {
  const bool once = a.R * a.ld * (int64_t)sizeof(T) > kKeptBytes;
  const int64_t r = once ? (int64_t)gridDim.x - 1 - blockIdx.x : blockIdx.x;     // the cache has the last rows
  float lse, ent;
  if (a.lse != nullptr && (a.g_entropy == nullptr || a.entropy != nullptr)) {
    lse = a.lse[r];
    ent = a.g_entropy ? a.entropy[r] : 0.f;
  } else {
    const RowStats st = row_stats<T, BLOCK, false>(static_cast<const T*>(a.logits) + r * a.ld, a.V);
    lse = st.m + logf(st.s);
    ent = lse - st.u / st.s;
  }
  if (once && r * a.V * (int64_t)sizeof(T) > kKeptGradients) row_gradients<T, BLOCK, true>(a, r, lse, ent);
  else row_gradients<T, BLOCK, false>(a, r, lse, ent);
}

// Threads per row.  Measured with 256 / 512 / 1024 (us): statistics of 48 bf16 rows of the 152k vocabulary 15.6 / 13.9 /
// 14.5, of 600 42 / 46 / 60, of 2048 116 / 125 / 155 - a wider block waits longer for its slowest wave's reduction; gradients
// of 48 24 / 19 / 18, of 2048 249 / 239 / 237, of 519 fp32 rows of 32003 28.5 / 28.0 / 31.0.
constexpr int kStatsThreads = 256, kStatsBwdThreads = 512;

}  // namespace clgrpo

using namespace clgrpo;

extern "C" int clgrpo_softmax_stats(const clgrpo_softmax_stats_args* a, void* stream) {
  CLGRPO_REQUIRE_PTR(a, "args");
  if (a->dtype != CLGRPO_BF16 && a->dtype != CLGRPO_F32) return fail(CLGRPO_EDTYPE, "clgrpo_softmax_stats: dtype %d", a->dtype);
  if (a->R < 0 || a->V <= 0 || a->ld < a->V) return fail(CLGRPO_EINVAL, "clgrpo_softmax_stats: R=%lld V=%lld ld=%lld",
                                                         (long long)a->R, (long long)a->V, (long long)a->ld);
  if (a->R == 0) return CLGRPO_OK;
  CLGRPO_REQUIRE_PTR(a->logits, "logits");
  if (a->logprob) CLGRPO_REQUIRE_PTR(a->labels, "labels");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (a->dtype == CLGRPO_BF16) hipLaunchKernelGGL((softmax_stats_kernel<__bf16, kStatsThreads>), dim3((unsigned)a->R), dim3(kStatsThreads), 0, s, *a);
  else hipLaunchKernelGGL((softmax_stats_kernel<float, kStatsThreads>), dim3((unsigned)a->R), dim3(kStatsThreads), 0, s, *a);
  return check_launch("softmax_stats_kernel");
}

extern "C" int clgrpo_softmax_stats_bwd(const clgrpo_softmax_stats_bwd_args* a, void* stream) {
  CLGRPO_REQUIRE_PTR(a, "args");
  if (a->dtype != CLGRPO_BF16 && a->dtype != CLGRPO_F32) return fail(CLGRPO_EDTYPE, "clgrpo_softmax_stats_bwd: dtype %d", a->dtype);
  if (a->R < 0 || a->V <= 0 || a->ld < a->V) return fail(CLGRPO_EINVAL, "clgrpo_softmax_stats_bwd: bad sizes");
  if (a->R == 0) return CLGRPO_OK;
  CLGRPO_REQUIRE_PTR(a->logits, "logits");
  CLGRPO_REQUIRE_PTR(a->dlogits, "dlogits");
  if (a->g_logprob) CLGRPO_REQUIRE_PTR(a->labels, "labels");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (a->dtype == CLGRPO_BF16) hipLaunchKernelGGL((softmax_stats_bwd_kernel<__bf16, kStatsBwdThreads>), dim3((unsigned)a->R), dim3(kStatsBwdThreads), 0, s, *a);
  else hipLaunchKernelGGL((softmax_stats_bwd_kernel<float, kStatsBwdThreads>), dim3((unsigned)a->R), dim3(kStatsBwdThreads), 0, s, *a);
  return check_launch("softmax_stats_bwd_kernel");
}
