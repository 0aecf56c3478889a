// Backward of the fused lm_head + log-softmax statistics.
//
// Per chunk of tokens (the chunk length is set by the workspace the caller gives):
//   1. dz kernel: recompute a z^T tile [256 vocab x 256 tokens] on the matrix cores
//      exactly as the forward does, turn it into d(logits) with the stored lse,
//      and write it in both orientations, dz[token][vocab] and dzT[vocab][token].
//   2. dhidden[chunk] = dz * W        as an NT GEMM against WT = W^T (built once per call)
//   3. dW (+)= dzT * hidden[chunk]    as an NT GEMM against hidT = hidden[chunk]^T, fp32 out
// Every contraction runs through the same K-contiguous MFMA tile (gemm_core.hpp).
//
// Algorithmic work: 4*T*H*V flop (dhidden + dW); the z recomputation (2*T*H*V) is overhead.
#include "head_internal.hpp"
#include "gemm_core.hpp"

namespace clgrpo {

int validate_head_shape(const char* who, int64_t T, int64_t H, int64_t V, int32_t dtype);

constexpr float kLog2e = 1.4426950408889634f;

// VEC = 16 / sizeof(T) floats as one 16-byte piece of the operand dtype.
__device__ __forceinline__ u32x4 pack_vec(const float (&v)[4], float*) {
  const f32x4 x = {v[0], v[1], v[2], v[3]};
  return __builtin_bit_cast(u32x4, x);
}
__device__ __forceinline__ u32x4 pack_vec(const float (&v)[8], __bf16*) {
  bf16x8 x;
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (__bf16)v[e];
  return __builtin_bit_cast(u32x4, x);
}

struct DzParams {
  const void* hidden;   // chunk base: [Tc, H]
  const void* weight;   // [V, H]
  const int64_t* labels;  // chunk base
  int64_t label_offset;   // first vocabulary id of `weight` (0 unless this is a vocabulary shard)
  const float* lse;
  const float* entropy;   // or nullptr
  const float* g_lp;
  const float* g_ent;     // or nullptr
  int Tc;       // valid tokens in the chunk
  int ldt;      // K extent of dzT = Tc rounded up to 64
  int H, V;
  int ldv;      // K extent of dz = V rounded up to 64
  int n_tb, n_vt;
  float c, inv_temperature;
  void* dz;     // Tc x ldv, K-blocked (see blocked_index)
  void* dzT;    // V x ldt, K-blocked
};

template <typename T>
__global__ __launch_bounds__(kHeadThreads, 1) void lmhead_dz_kernel(DzParams p) {
  using Tile = LogitTile<T>;
  constexpr int MI = Tile::MI, NI = Tile::NI, VEC = Tile::VEC;
  extern __shared__ __align__(16) char lds[];

  const int item = xcd_remap(blockIdx.x, gridDim.x);
  if (item >= p.n_tb * p.n_vt) return;
  int vt, tb;
  grouped_tile(item, p.n_vt, p.n_tb, 4, vt, tb);

  const int la = Tile::wave_m() + Tile::lane_a0(), lb = Tile::wave_n() + Tile::lane_b0();
  const int t0 = tb * 256, v0 = vt * 256;
  const int b_rows = (p.Tc - t0) < 256 ? (p.Tc - t0) : 256;
  const int a_rows = (p.V - v0) < 256 ? (p.V - v0) : 256;
  const T* hidden = static_cast<const T*>(p.hidden) + (int64_t)t0 * p.H;
  const T* weight = static_cast<const T*>(p.weight) + (int64_t)v0 * p.H;

  // A token block whose upstream gradients are all zero (e.g. prompt-only rows) needs no GEMM.
  bool any_grad = false;
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int t = t0 + lb + Tile::b_block(j);
    if (t < p.Tc) any_grad |= (p.g_lp[t] != 0.f) | (p.g_ent != nullptr && p.g_ent[t] != 0.f);
  }
  // (the flags pass through the tile's own LDS: all of it is spoken for)
  int* live = reinterpret_cast<int*>(lds);
  const bool wave_live = __any(any_grad);
  if ((threadIdx.x & 63) == 0) live[threadIdx.x >> 6] = wave_live;
  __syncthreads();
  const bool block_live = (live[0] | live[1] | live[2] | live[3]) != 0;
  __syncthreads();

  typename Tile::Acc acc;
  Tile::zero(acc);
  if (block_live) {
    Tile core;
    const int nslab = p.H / Tile::kSlabK;
    core.start(Tile::Operand::row_major(weight, p.H, a_rows), Tile::Operand::row_major(hidden, p.H, b_rows), nslab, lds);
    core.run(acc, nslab);
    Tile::finish();
  }

  // Per-token coefficients.  Tokens past the chunk get zero gradient and a huge lse, so p = 0.
  int lab[NI];
  float lse[NI], glp[NI], gent[NI], ent[NI];
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int t = t0 + lb + Tile::b_block(j);
    const bool ok = t < p.Tc;
    lab[j] = -1;
    if (ok) {
      const int64_t rel = p.labels[t] - p.label_offset;   // a label outside these rows matches nothing
      if (rel >= 0 && rel < p.V) lab[j] = (int)rel;
    }
    lse[j] = ok ? p.lse[t] : 1e30f;
    glp[j] = ok ? p.g_lp[t] : 0.f;
    gent[j] = (ok && p.g_ent) ? p.g_ent[t] : 0.f;
    ent[j] = (ok && p.g_ent) ? p.entropy[t] : 0.f;
  }

  T* dz = static_cast<T*>(p.dz);
  T* dzT = static_cast<T*>(p.dzT);
  const float it = p.inv_temperature;
  constexpr int AG = VEC / 4;                 // blocks along A whose registers make up VEC consecutive vocabulary rows
#pragma unroll
  for (int i = 0; i < MI; i += AG) {
    float d[NI][VEC];
    const int v = v0 + la + Tile::a_block(i);
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        const float zraw = acc_get(acc[i + e / 4][j], e % 4);
        const float pr = __builtin_amdgcn_exp2f(fmaf(zraw, p.c, -lse[j] * kLog2e));
        const float logp = fmaf(zraw, it, -lse[j]);
        // dz = it * ( glp*(1[v==y] - p) - gent * p * (logp + ent) )
        float x = -it * pr * fmaf(gent[j], logp + ent[j], glp[j]);
        if (lab[j] == v + e) x += it * glp[j];
        if (v + e >= p.V || !block_live) x = 0.f;   // vocabulary padding columns / dead block
        d[j][e] = x;
      }
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int t = t0 + lb + Tile::b_block(j);
      if (t < p.Tc && v < p.ldv)
        *reinterpret_cast<u32x4*>(dz + blocked_index<T>(t, v, p.ldv / Tile::kSlabK)) = pack_vec(d[j], (T*)nullptr);
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e)
#pragma unroll
      for (int j = 0; j < NI; j += VEC) {
        float x[VEC];
#pragma unroll
        for (int k = 0; k < VEC; ++k) x[k] = d[j + k][e];
        const int t = t0 + lb + Tile::b_block(j);
        if (v + e < p.V && t < p.ldt)
          *reinterpret_cast<u32x4*>(dzT + blocked_index<T>(v + e, t, p.ldt / Tile::kSlabK)) = pack_vec(x, (T*)nullptr);
      }
  }
}

// d(logits) from kept logits, in place, plus its transpose.  A unit is 256 token rows x one 128-byte slab of
// vocabulary: 32 KB of the K-blocked kept logits, which become the same 32 KB of the K-blocked dz operand.
// A thread takes a square of VEC tokens x VEC vocabulary entries: VEC 16-byte pieces in, VEC pieces of
// dz back over them, VEC pieces of dzT, the transposition being a choice of registers (no LDS, no barrier
// between units).  Eight lanes cover a slab row, eight lane groups eight of its token groups, so every access
// of a wave is whole 128-byte lines.  HBM-bound: reads 1x, writes 2x the chunk.
struct DzFromZParams {
  void* z;            // Tc x ldv: in kept logits (KeptLogit<T>), out dz (T), K-blocked
  void* dzT;          // V rows, K-blocked: the slab of the chunk's first token
  const int64_t* labels;
  int64_t label_offset;
  const float* lse;
  const float* entropy;
  const float* g_lp;
  const float* g_ent;
  const int32_t* order;   // optional [Tc]: row n is token order[n] of the per-token arrays
  int Tc, ldt, V, ldv;    // ldt: tokens of dzT to write, Tc rounded up to 64
  int64_t t_slabs;        // slabs per row of dzT, of which these tokens are the first ldt / E
  float c, inv_temperature;
};

template <typename T>
__global__ __launch_bounds__(256) void dz_from_z_kernel(DzFromZParams p) {
  typedef typename KeptLogit<T>::type ZT;
  static_assert(sizeof(ZT) == sizeof(T), "d(logits) overwrites the kept logits in place");
  constexpr int E = Elem<T>::kSlabK;                // vocabulary entries of a unit (64 or 32)
  constexpr int VEC = 16 / (int)sizeof(T);          // elements per 16-byte piece
  constexpr int kPasses = kBlockRows / VEC / 32;    // a pass of 256 threads covers 32 token groups
  __shared__ float s_lse[kBlockRows], s_ent[kBlockRows], s_glp[kBlockRows], s_gen[kBlockRows];
  __shared__ int s_lab[kBlockRows];
  const int rb = blockIdx.x;
  const int64_t n_kslab = p.ldv / E;
  const float it = p.inv_temperature;
  {
    const int n = rb * kBlockRows + threadIdx.x;
    const bool ok = n < p.Tc;
    const int t = ok && p.order ? p.order[n] : n;
    s_glp[threadIdx.x] = ok ? p.g_lp[t] : 0.f;      // rows past the chunk and rows without a gradient give zeros
    s_gen[threadIdx.x] = (ok && p.g_ent) ? p.g_ent[t] : 0.f;
    s_lse[threadIdx.x] = ok ? p.lse[t] : 0.f;
    s_ent[threadIdx.x] = (ok && p.g_ent) ? p.entropy[t] : 0.f;
    int lab = -1;
    if (ok) {
      const int64_t rel = p.labels[t] - p.label_offset;
      if (rel >= 0 && rel < p.V) lab = (int)rel;
    }
    s_lab[threadIdx.x] = lab;
  }
  __syncthreads();
  const int q = threadIdx.x & 7, cg = threadIdx.x >> 3;   // piece within the slab row, token group
  T* dzT = static_cast<T*>(p.dzT);
  for (int ks = blockIdx.y; ks < (int)n_kslab; ks += gridDim.y) {
    char* unit = static_cast<char*>(p.z) + ((int64_t)rb * n_kslab + ks) * (kBlockRows * kRowBytes);
    const int v = ks * E + q * VEC;
#pragma unroll
    for (int pass = 0; pass < kPasses; ++pass) {
      const int R = (pass * 32 + cg) * VEC;         // first token row of this thread's square
      u32x4 raw[VEC];
#pragma unroll
      for (int k = 0; k < VEC; ++k) raw[k] = *reinterpret_cast<const u32x4*>(unit + (R + k) * kRowBytes + q * 16);
      float d[VEC][VEC];
#pragma unroll
      for (int k = 0; k < VEC; ++k) {
        const float glp = s_glp[R + k], gen = s_gen[R + k], lse = s_lse[R + k], ent = s_ent[R + k];
        const int lab = s_lab[R + k] - v;
        const bool live = glp != 0.f || gen != 0.f;
        const float lse2 = lse * kLog2e;
        const ZT* in = reinterpret_cast<const ZT*>(&raw[k]);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          const float zraw = (float)in[e];
          const float pr = __builtin_amdgcn_exp2f(fmaf(zraw, p.c, -lse2));
          const float logp = fmaf(zraw, it, -lse);
          float x = -it * pr * fmaf(gen, logp + ent, glp);
          if (lab == e) x += it * glp;
          d[k][e] = (live && v + e < p.V) ? x : 0.f;      // vocabulary padding columns give zeros
        }
      }
#pragma unroll
      for (int k = 0; k < VEC; ++k) *reinterpret_cast<u32x4*>(unit + (R + k) * kRowBytes + q * 16) = pack_vec(d[k], (T*)nullptr);
      const int tok = rb * kBlockRows + R;
      if (tok < p.ldt) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          float x[VEC];
#pragma unroll
          for (int k = 0; k < VEC; ++k) x[k] = d[k][e];
          if (v + e < p.V) *reinterpret_cast<u32x4*>(dzT + blocked_index<T>(v + e, tok, p.t_slabs)) = pack_vec(x, (T*)nullptr);
        }
      }
    }
  }
}

// C (+)= A B^T with A [M x K] and B [N x K] K-blocked, C row-major in one of two orientations; either way
// a lane's 16-byte pieces lie along C's rows and a store instruction covers runs of at least 64 bytes:
//   kMContig = false: C[m][n], ld = ldc, fp32 or 16-bit (dW: A = dz^T, B = hidden^T).  A lane holds 4 consecutive n of
//     a row (GemmTile with BV = 4), 16 lanes 256 contiguous bytes of each of 4 rows for fp32, 128 for 16-bit results.
//   kMContig = true:  C[n][m], ld = ldc (dhidden: A = W^T, B = dz).  A lane holds VEC consecutive m of a row, the 4
//     lane groups 64 contiguous bytes of each of 16 rows for 16-bit results.
template <typename T, bool kMContig> using OutTile = GemmTile<T, kMContig ? 16 / (int)sizeof(T) : 4>;

struct GemmParams {
  const void* A;      // M x K, K-blocked with a_kslabs slabs per row block
  const void* B;      // N x K, K-blocked with b_kslabs slabs per row block
  void* C;
  int64_t a_kslabs, b_kslabs, ldc;
  int M, N, K;
  int n_mt, n_nt;
  int accumulate;
  int k_split;        // > 1: work item = (tile, K range); fp32 partial tiles go to `partial`
  int k_per_split;    // K extent of one range, a multiple of the slab
  int n_walk;         // > 0: workgroups walk runs of tiles (see gemm_nt_kernel); needs k_split == 1
  float* partial;     // [k_split] copies of C's shape in fp32, densely packed (row stride N or M)
  const int32_t* order;   // kMContig, optional [N]: row n of the result is row order[n] of the `total` rows of C
  int64_t total;
};

// Addresses of a 256 x 256 output tile for the accumulator layout: a range-checked buffer descriptor over
// the tile's valid rows and one per-lane byte offset per group of BV (kMContig: per block) of the lane dimension.
// Along the lane dimension (n) elements outside the tile get a per-lane offset far outside the descriptor: loads
// of them give 0 and stores are dropped.  Along the register dimension (m) nothing relies on the range check:
// kMContig skips whole 32-row groups (its M extents are multiples of 32), and the other orientation tests
// every row against the tile's valid rows unless the tile is a full one.
template <typename T, typename OutT, bool kMContig>
struct TileAddr {
  using Tile = OutTile<T, kMContig>;
  static constexpr int ES = (int)sizeof(OutT);
  static constexpr int AG = Tile::VEC / 4;                  // blocks along m whose registers are consecutive
  static constexpr int kGroups = kMContig ? Tile::NI : Tile::NI / 4;
  __amdgpu_buffer_rsrc_t rsrc;
  int voff[kGroups];
  int row_bytes, a_rows, row_lim;   // row_lim: valid rows from this lane's first row on
  __device__ __forceinline__ TileAddr(OutT* base, int64_t ld, int m0, int n0, int a_rows_, int b_rows,
                                      const int32_t* order = nullptr, int64_t total = 0) {
    row_bytes = (int)(ld * (int64_t)ES);
    a_rows = a_rows_;
    const int m = Tile::wave_m() + Tile::lane_a0();
    row_lim = a_rows_ - m;
    const int rows = kMContig ? b_rows : a_rows_, cols = kMContig ? a_rows_ : b_rows;
    const bool ordered = kMContig && order != nullptr;
    const int bytes = ordered ? (int)(total * row_bytes) - m0 * ES : (rows > 0 ? (rows - 1) * row_bytes + cols * ES : 0);
    OutT* origin = kMContig ? base + (ordered ? 0 : (int64_t)n0 * ld) + m0 : base + (int64_t)m0 * ld + n0;
    rsrc = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<char*>(origin), 0, bytes, 0x00020000);
#pragma unroll
    for (int k = 0; k < kGroups; ++k) {
      const int n = Tile::wave_n() + Tile::lane_b0() + Tile::b_block(kMContig ? k : 4 * k);
      if (n >= b_rows) voff[k] = 0x7f000000;
      else if (kMContig) voff[k] = (ordered ? order[n0 + n] : n) * row_bytes + m * ES;
      else voff[k] = m * row_bytes + n * ES;
    }
  }
  // kMContig: blocks i .. i + AG - 1 lie inside the tile (uniform over the wave)
  __device__ __forceinline__ bool group_ok(int i) const { return Tile::wave_m() + (Tile::a_block(i) & ~31) < a_rows; }
  __device__ __forceinline__ bool full_rows() const { return a_rows == Tile::BM; }
};

// N consecutive elements of a row: 4 or 8 floats, or 8 (T = bf16) 16-bit values.
template <int N>
__device__ __forceinline__ void row_load(float (&x)[N], const __amdgpu_buffer_rsrc_t& rsrc, int voff, int soff, float*) {
#pragma unroll
  for (int k = 0; k < N; k += 4) {
    const f32x4 v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff + k * 4, soff, 0));
    x[k] = v[0]; x[k + 1] = v[1]; x[k + 2] = v[2]; x[k + 3] = v[3];
  }
}
__device__ __forceinline__ void row_load(float (&x)[8], const __amdgpu_buffer_rsrc_t& rsrc, int voff, int soff, __bf16*) {
  const bf16x8 v = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff, soff, 0));
#pragma unroll
  for (int k = 0; k < 8; ++k) x[k] = (float)v[k];
}
template <int N>
__device__ __forceinline__ void row_store(const float (&x)[N], const __amdgpu_buffer_rsrc_t& rsrc, int voff, int soff, float*) {
#pragma unroll
  for (int k = 0; k < N; k += 4) {
    const f32x4 v = {x[k], x[k + 1], x[k + 2], x[k + 3]};
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rsrc, voff + k * 4, soff, 0);
  }
}
__device__ __forceinline__ void row_store(const float (&x)[8], const __amdgpu_buffer_rsrc_t& rsrc, int voff, int soff, __bf16*) {
  __builtin_amdgcn_raw_buffer_store_b128(pack_vec(x, (__bf16*)nullptr), rsrc, voff, soff, 0);
}

__device__ __forceinline__ void row_store(const float (&x)[4], const __amdgpu_buffer_rsrc_t& rsrc, int voff, int soff, __bf16*) {
  typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  const bf16x4 v = {(__bf16)x[0], (__bf16)x[1], (__bf16)x[2], (__bf16)x[3]};
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), rsrc, voff, soff, 0);
}

// fn(values of one run of a row, per-lane offset, scalar offset), for every run of the tile that lies inside it;
// kLoad: the values go into the accumulators afterwards.
template <typename T, typename OutT, bool kMContig, bool kLoad, typename AccT, typename Fn>
__device__ __forceinline__ void for_rows(const TileAddr<T, OutT, kMContig>& at, AccT& acc, Fn fn) {
  using Tile = OutTile<T, kMContig>;
  if constexpr (kMContig) {
    constexpr int AG = TileAddr<T, OutT, kMContig>::AG, N = 4 * AG;
#pragma unroll
    for (int i = 0; i < Tile::MI; i += AG) {
      if (!at.group_ok(i)) continue;
#pragma unroll
      for (int j = 0; j < Tile::NI; ++j) {
        float x[N] = {};
#pragma unroll
        for (int k = 0; k < (kLoad ? 0 : N); ++k) x[k] = acc_get(acc[i + k / 4][j], k % 4);
        fn(x, at.voff[j] + Tile::a_block(i) * (int)sizeof(OutT), 0);
        if (kLoad) {
#pragma unroll
          for (int k = 0; k < N; k += 4) acc_set(acc[i + k / 4][j], x[k], x[k + 1], x[k + 2], x[k + 3]);
        }
      }
    }
  } else {
    const bool full = at.full_rows();   // uniform over the workgroup
#pragma unroll
    for (int i = 0; i < Tile::MI; ++i)
#pragma unroll
      for (int j = 0; j < Tile::NI; j += 4) {
        float x[4][4];                    // [register of the four blocks][block]
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int dm = Tile::a_block(i) + r;
#pragma unroll
          for (int k = 0; k < 4; ++k) x[r][k] = kLoad ? 0.f : acc_get(acc[i][j + k], r);
          if (full || dm < at.row_lim) fn(x[r], at.voff[j / 4], dm * at.row_bytes);
        }
        if (kLoad) {
#pragma unroll
          for (int k = 0; k < 4; ++k) acc_set(acc[i][j + k], x[0][k], x[1][k], x[2][k], x[3][k]);
        }
      }
  }
}

// Accumulators of output tile (m0, n0) before its K loop: zeros, or - when the GEMM adds to C and one
// workgroup owns the whole K range of the tile - the tile's current contents.  Reading C here instead of
// in the epilogue puts the loads' latency in front of the K loop, where the first operand slabs are in
// flight anyway, and leaves the epilogue a pure store.
template <typename T, typename OutT, bool kMContig>
__device__ __forceinline__ void gemm_init_tile(const GemmParams& p, typename OutTile<T, kMContig>::Acc& acc, int m0, int n0,
                                               int a_rows, int b_rows) {
  constexpr bool kAdds = !kMContig && sizeof(OutT) == 4;    // only an fp32 C is ever added to
  if (!kAdds || !p.accumulate || p.k_split > 1) OutTile<T, kMContig>::zero(acc);
  if constexpr (kAdds) {
    if (!p.accumulate || p.k_split > 1) return;
    const TileAddr<T, OutT, kMContig> at(static_cast<OutT*>(p.C), p.ldc, m0, n0, a_rows, b_rows);
    for_rows<T, OutT, kMContig, true>(at, acc, [&](auto& x, int voff, int soff) { row_load(x, at.rsrc, voff, soff, (OutT*)nullptr); });
  }
}

// Output tile from the accumulators: C = acc (the accumulators already hold C's previous contents
// when the GEMM adds to it, see gemm_init_tile), or the fp32 partial of K range `ks`.
template <typename T, typename OutT, bool kMContig>
__device__ __forceinline__ void gemm_store_tile(const GemmParams& p, typename OutTile<T, kMContig>::Acc& acc, int m0, int n0,
                                                int a_rows, int b_rows, int ks) {
  if (p.k_split > 1) {
    const TileAddr<T, float, kMContig> at(p.partial + (int64_t)ks * p.M * p.N, kMContig ? p.M : p.N, m0, n0, a_rows, b_rows);
    for_rows<T, float, kMContig, false>(at, acc, [&](auto& x, int voff, int soff) { row_store(x, at.rsrc, voff, soff, (float*)nullptr); });
    return;
  }
  const TileAddr<T, OutT, kMContig> at(static_cast<OutT*>(p.C), p.ldc, m0, n0, a_rows, b_rows, p.order, p.total);
  for_rows<T, OutT, kMContig, false>(at, acc, [&](auto& x, int voff, int soff) { row_store(x, at.rsrc, voff, soff, (OutT*)nullptr); });
}

// Work item = (walk, fixed tile) when n_walk > 0: the workgroup keeps one operand's tile (A's m tile
// when C is [n][m], B's n tile when C is [m][n]) and walks a contiguous run of tiles of the other, so the
// K loops stream into each other (the next tile's first slabs are requested while the current tile
// finishes and is stored).  Otherwise work item = (K range, m tile, n tile), one K loop per workgroup.
template <typename T, typename OutT, bool kMContig>
__global__ __launch_bounds__(kHeadThreads, 1) void gemm_nt_kernel(GemmParams p) {
  using Tile = OutTile<T, kMContig>;
  constexpr int64_t kSlabElems = (int64_t)kBlockRows * Tile::kSlabK;   // elements of one block's slab
  extern __shared__ __align__(16) char lds[];

  // this workgroup's tiles: (mt, nt) first, then `count - 1` steps along the walked operand; one K range
  int item = xcd_remap(blockIdx.x, gridDim.x), mt, nt, count = 1, ks = 0, k0 = 0, k_len = p.K;
  if (p.n_walk > 0) {
    const int n_fixed = kMContig ? p.n_mt : p.n_nt;       // tiles of the operand that stays
    const int n_moving = kMContig ? p.n_nt : p.n_mt;      // tiles of the operand that is walked
    if (item >= p.n_walk * n_fixed) return;
    int walk, ft;
    grouped_tile(item, p.n_walk, n_fixed, 4, walk, ft);
    const int begin = (int)((int64_t)walk * n_moving / p.n_walk);
    count = (int)((int64_t)(walk + 1) * n_moving / p.n_walk) - begin;
    mt = kMContig ? ft : begin;
    nt = kMContig ? begin : ft;
  } else {
    if (item >= p.n_mt * p.n_nt * p.k_split) return;
    ks = item / (p.n_mt * p.n_nt);
    item -= ks * (p.n_mt * p.n_nt);
    grouped_tile(item, p.n_mt, p.n_nt, 8, mt, nt);
    k0 = ks * p.k_per_split;
    k_len = (p.K - k0) < p.k_per_split ? (p.K - k0) : p.k_per_split;
  }

  const int nslab = k_len / Tile::kSlabK;
  const int64_t s0 = k0 / Tile::kSlabK;   // first slab of this K range
  const bool stream = Tile::can_stream(nslab);
  typename Tile::Acc acc;
  Tile core;
  for (int k = 0; k < count; ++k) {
    const int m0 = mt * 256, n0 = nt * 256;
    const int a_rows = (p.M - m0) < 256 ? (p.M - m0) : 256;
    const int b_rows = (p.N - n0) < 256 ? (p.N - n0) : 256;
    const auto op_a = Tile::Operand::blocked(static_cast<const T*>(p.A) + ((int64_t)mt * p.a_kslabs + s0) * kSlabElems, a_rows);
    const auto op_b = Tile::Operand::blocked(static_cast<const T*>(p.B) + ((int64_t)nt * p.b_kslabs + s0) * kSlabElems, b_rows);
    gemm_init_tile<T, OutT, kMContig>(p, acc, m0, n0, a_rows, b_rows);
    if (k == 0 || !stream) core.start(op_a, op_b, nslab, lds);
    core.next_a = Tile::hold(op_a, nslab);
    core.next_b = Tile::hold(op_b, nslab);
    if (stream && k + 1 < count) {
      const int left = (kMContig ? p.N - n0 : p.M - m0) - 256;
      const int next_rows = left < 256 ? left : 256;
      core.next_a = kMContig ? Tile::cursor(op_a, nslab)
                             : Tile::cursor(Tile::Operand::blocked(op_a.base + p.a_kslabs * kSlabElems, next_rows), nslab);
      core.next_b = kMContig ? Tile::cursor(Tile::Operand::blocked(op_b.base + p.b_kslabs * kSlabElems, next_rows), nslab)
                             : Tile::cursor(op_b, nslab);
    }
    core.run(acc, nslab);
    if (!stream || k + 1 == count) Tile::finish();
    gemm_store_tile<T, OutT, kMContig>(p, acc, m0, n0, a_rows, b_rows, ks);
    if (kMContig) ++nt; else ++mt;
  }
}

template <typename OutT> __device__ __forceinline__ OutT cvt_out(float v);
template <> __device__ __forceinline__ float cvt_out<float>(float v) { return v; }
template <> __device__ __forceinline__ __bf16 cvt_out<__bf16>(float v) { return (__bf16)v; }

// C (+)= sum over splits of partial[s], each a dense copy of C's shape with `cols` elements per row (a multiple of 32).
// A thread takes 4 consecutive columns of one row, a block's row is uniform.  HBM-bound: reads the partials once.
// 16 ranges of 1064 rows at H = 4096 (279 MB): 82.7 -> 57.4 us = 4.9 TB/s, 7 of 5428 at 2048 85.5 -> 54.8 us; with one element
// per thread the index arithmetic (a 64-bit division each) was what took the time.
template <typename OutT>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ partial, int k_split, int64_t MN, int cols,
                                                            OutT* C, int64_t ldc, int accumulate,
                                                            const int32_t* __restrict__ order) {
  const int64_t row = blockIdx.x;
  const int col = (int)(blockIdx.y * blockDim.x + threadIdx.x) * 4;
  if (col >= cols) return;
  const f32x4* src = reinterpret_cast<const f32x4*>(partial + row * cols + col);
  const int64_t step = MN / 4;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  int s = 0;
  for (; s + 4 <= k_split; s += 4) {          // four ranges in flight, added in their order
    const f32x4 x0 = src[s * step], x1 = src[(s + 1) * step], x2 = src[(s + 2) * step], x3 = src[(s + 3) * step];
    v += x0; v += x1; v += x2; v += x3;
  }
  for (; s < k_split; ++s) v += src[s * step];
  OutT* dst = C + (order ? order[row] : row) * ldc + col;
  struct alignas(4 * sizeof(OutT)) Four { OutT x[4]; };
  const bool aligned = (reinterpret_cast<uintptr_t>(dst) & (4 * sizeof(OutT) - 1)) == 0;   // the caller's result may start anywhere
  Four out;
  if (accumulate) {
    if (aligned) out = *reinterpret_cast<const Four*>(dst);
    else for (int k = 0; k < 4; ++k) out.x[k] = dst[k];
    for (int k = 0; k < 4; ++k) v[k] += (float)out.x[k];
  }
  for (int k = 0; k < 4; ++k) out.x[k] = cvt_out<OutT>(v[k]);
  if (aligned) *reinterpret_cast<Four*>(dst) = out;
  else for (int k = 0; k < 4; ++k) dst[k] = out.x[k];
}

// dst(c, r) = src[r][c] (src[order[r]][c] with an order) for r < R, c < C and 0 for R <= r < r_dst, where dst is the K-blocked
// operand with C rows and ld_dst K elements (see blocked_index), of which the first r_dst are written.  64x64 tiles, 16-byte accesses on
// both sides (C and ld_src are multiples of 32 elements here, so a 16-byte piece never straddles an edge).
template <typename T>
__global__ __launch_bounds__(256) void transpose_block_kernel(const T* __restrict__ src, int64_t ld_src,
                                                              T* __restrict__ dst, int64_t ld_dst, int64_t r_dst, int R, int C,
                                                              const int32_t* __restrict__ order) {
  constexpr int VEC = 16 / (int)sizeof(T);       // elements per 16-byte access
  constexpr int CPR = 64 / VEC;                  // accesses per 64-wide tile row
  constexpr int RPP = 256 / CPR;                 // tile rows covered per pass
  constexpr int kE = kRowBytes / (int)sizeof(T);
  __shared__ T tile[64][64 + VEC];               // [c][r], padded rows
  const int r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
  const int q = threadIdx.x % CPR, row = threadIdx.x / CPR;
  for (int rr = row; rr < 64; rr += RPP) {
    const int r = r0 + rr, c = c0 + q * VEC;
    alignas(16) T vals[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) vals[j] = (T)0.f;
    if (r < R && c < C) *reinterpret_cast<u32x4*>(vals) = *reinterpret_cast<const u32x4*>(src + (int64_t)(order ? order[r] : r) * ld_src + c);
#pragma unroll
    for (int j = 0; j < VEC; ++j) tile[q * VEC + j][rr] = vals[j];
  }
  __syncthreads();
  for (int cc = row; cc < 64; cc += RPP) {
    const int c = c0 + cc, r = r0 + q * VEC;
    if (c < C && r < r_dst)
      *reinterpret_cast<u32x4*>(dst + blocked_index<T>(c, r, ld_dst / kE)) = *reinterpret_cast<const u32x4*>(&tile[cc][q * VEC]);
  }
}

// K ranges per tile that fill `cus` CUs best (1 = no split): work items = tiles x ranges, and a launch
// takes ceil(items / cus) rounds.  At most kMaxKSplit ranges, each at least 8 slabs long and none empty,
// and at most what `partial_bytes` can hold of fp32 partial tiles.  Fewer tiles than cus / kMaxKSplit may use twice as
// many ranges: a range is a chain of slabs on one CU while most of the others stand idle (143 rows at H = 1024, V = 32000:
// 4 tiles, 16 -> 32 ranges 44.8 -> 29.9 us, the sum over the ranges 6 us either way).
constexpr int kMaxKSplit = 16;
static int pick_k_split(int tiles, int M, int N, int K, int slab, size_t partial_bytes, int cus) {
  int best = 1;
  double best_eff = 0.0;
  const int most = tiles * kMaxKSplit < cus ? 2 * kMaxKSplit : kMaxKSplit;
  for (int s = 1; s <= most; ++s) {
    if (s > 1) {
      if ((size_t)s * M * N * sizeof(float) > partial_bytes || K / s < 8 * slab) break;
      const int64_t per = round_up64((K + s - 1) / s, slab);
      if ((int64_t)(s - 1) * per >= K) continue;     // rounding the range up to whole slabs would leave the last one empty
    }
    const long units = (long)tiles * s;
    const double eff = (double)units / (double)(((units + cus - 1) / cus) * cus);
    if (eff > best_eff + 0.04) { best_eff = eff; best = s; }   // a split must buy more than 4 % to be worth its extra pass
  }
  return best;
}

// How the dhidden GEMM (C[n][m], M = H output columns, N = token rows, K = vocabulary) is launched.  Its tile
// count rarely fills whole rounds of one workgroup per CU; cutting K into ranges (fp32 partial tiles, summed
// by a second pass) repairs that at the price of the partials' traffic.  When the tiles exceed one round the
// cheaper repair is to cut the token rows instead: a bulk launch over whole rounds of tiles without any K
// split, and a second launch over the remaining rows with the K split those few tiles want.
struct DhPlan {
  int bulk_nt;       // n tiles (256 token rows each) of the bulk launch; 0: one launch over all rows
  int k_split;       // K ranges of the single launch, or of the tail launch when bulk_nt > 0
  size_t partial_bytes;
};

static DhPlan plan_dhidden(int64_t rows, int64_t H, int64_t K, int slab, int cus, size_t partial_cap) {
  DhPlan pl{0, 1, 0};
  if (rows <= 0) return pl;
  const int n_mt = (int)((H + 255) / 256), n_nt = (int)((rows + 255) / 256);
  const int tiles = n_mt * n_nt;
  const long k_slabs = (K + slab - 1) / slab;
  auto cost = [&](long items, int s) {        // rounds x slabs per range, plus 2 % for the partials' traffic
    const long rounds = (items * s + cus - 1) / cus;
    const double c = (double)rounds * (double)((k_slabs + s - 1) / s);
    return s > 1 ? c * 1.02 : c;
  };
  const int s_one = pick_k_split(tiles, (int)H, (int)rows, (int)K, slab, partial_cap, cus);
  pl.k_split = s_one;
  double best = cost(tiles, s_one);
  const int per_round_n = cus / n_mt;
  if (per_round_n >= 1 && n_nt > per_round_n && n_nt % per_round_n != 0) {
    const int bulk_nt = n_nt / per_round_n * per_round_n;
    const int64_t tail_rows = rows - (int64_t)bulk_nt * 256;
    const int tail_tiles = (n_nt - bulk_nt) * n_mt;
    const int s_tail = pick_k_split(tail_tiles, (int)H, (int)tail_rows, (int)K, slab, partial_cap, cus);
    const double two = cost((long)bulk_nt * n_mt, 1) + cost(tail_tiles, s_tail) + 0.01 * (double)k_slabs;
    if (two < 0.98 * best) {
      pl.bulk_nt = bulk_nt;
      pl.k_split = s_tail;
      pl.partial_bytes = s_tail > 1 ? (size_t)s_tail * tail_rows * H * sizeof(float) : 0;
      return pl;
    }
  }
  pl.partial_bytes = s_one > 1 ? (size_t)s_one * rows * H * sizeof(float) : 0;
  return pl;
}

// Bytes of fp32 split-K partials the dhidden GEMM of `rows` tokens wants (planned for a 256-CU device, so
// that the workspace size does not depend on the device in use; a launch takes fewer ranges if they do not fit).
static size_t dhidden_partial_bytes(int64_t rows, int64_t H, int64_t ldv, int slab) {
  return plan_dhidden(rows, H, ldv, slab, 256, (size_t)1 << 30).partial_bytes;
}

// How the dW GEMM (C[m][n], M = vocabulary rows, N = H, K = the chunk's tokens) is launched.  With many more tiles
// than CUs its workgroups keep one tile of hidden^T and walk runs of vocabulary tiles (see gemm_nt_kernel); the walks
// are as long as the longest run, so when the vocabulary tiles do not divide by the number of walks the last
// `n_mt % n_walk` of them keep a sixteenth of the chip busy for a whole tile period (594 tiles on 16 walks: runs of
// 37 and 38).  The repair is the one of the dhidden GEMM: a bulk launch whose walks are all equally long, and a second
// launch over the remaining vocabulary tiles cut into K ranges that fill the CUs (fp32 partial tiles, summed by a small
// pass).  The partials' traffic (written and read once) is priced in, in slab periods of one tile.
struct DwPlan {
  int n_walk;        // walks of the (bulk) launch; 0: one workgroup per tile, no bulk / tail split
  int bulk_mt;       // vocabulary tiles of the bulk launch; 0: one launch over all of them
  int k_split;       // K ranges of the tail launch
  size_t partial_bytes;
};

static DwPlan plan_dweight(int64_t V, int64_t H, int64_t K, int slab, int cus, size_t partial_cap) {
  DwPlan pl{0, 0, 1, 0};
  const int n_mt = (int)((V + 255) / 256), n_nt = (int)((H + 255) / 256);
  if (!(n_nt <= cus && (long)n_mt * n_nt >= 4L * cus && K >= 2 * slab)) return pl;
  int n_walk = cus / n_nt;
  if (n_walk > n_mt) n_walk = n_mt;
  const long walk_periods = (n_mt + n_walk - 1) / n_walk;
  const long plain_rounds = ((long)n_mt * n_nt + cus - 1) / cus;
  if (walk_periods * 100 > plain_rounds * 104) return pl;     // one workgroup per tile is the better launch
  pl.n_walk = n_walk;
  const int base = n_mt / n_walk, rem = n_mt % n_walk;
  if (rem == 0 || base == 0) return pl;
  const long k_slabs = (K + slab - 1) / slab;
  const int64_t tail_rows = V - (int64_t)(n_mt - rem) * 256;
  const long tail_tiles = (long)rem * n_nt;
  // one slab period of a tile is about 1.65 us; the partials move at about 4 TB/s: 6.6 MB per slab period
  int best_s = 0;
  double best = 0.0;
  for (int s = 1; s <= kMaxKSplit; ++s) {
    const size_t bytes = s > 1 ? (size_t)s * tail_rows * H * sizeof(float) : 0;
    if (s > 1) {
      if (bytes > partial_cap || K / s < 8 * slab) break;
      const int64_t per = round_up64((K + s - 1) / s, slab);
      if ((int64_t)(s - 1) * per >= K) continue;
    }
    const long rounds = (tail_tiles * s + cus - 1) / cus;
    const double c = (double)rounds * (double)((k_slabs + s - 1) / s) + 2.0 * (double)bytes / 6.6e6 + (s > 1 ? 0.02 : 0.01) * (double)k_slabs;
    if (best_s == 0 || c < best) { best = c; best_s = s; }
  }
  const double now = (double)(base + 1) * (double)k_slabs, two = (double)base * (double)k_slabs + best;
  if (best_s == 0 || two >= 0.99 * now) return pl;
  pl.bulk_mt = n_mt - rem;
  pl.k_split = best_s;
  pl.partial_bytes = best_s > 1 ? (size_t)best_s * tail_rows * H * sizeof(float) : 0;
  return pl;
}

static size_t dweight_partial_bytes(int64_t rows, int64_t H, int64_t V, int slab) {
  return rows > 0 ? plan_dweight(V, H, round_up64(rows, 64), slab, 256, (size_t)1 << 30).partial_bytes : 0;
}

// dhidden of few rows straight from W [V, H], without W^T.  Building W^T reads and writes the weight once each (V = 151936,
// H = 4096: 465 us), more than a contraction over a few hundred rows takes.  A wave owns 128 columns of H, 128 rows and
// a K range.  Lane 16 g + c reads 8 vocabulary rows (k = 8 g ..) x 8 columns (8 c ..) of W, 16 bytes per row, and
// transposes the square between registers: the result is its A fragment of 8 blocks of 16 columns each, block i
// holding columns 8 c + i.  B fragments are 16-byte pieces of the K-blocked dz.  No LDS and no barriers: the
// four waves of a workgroup (512 columns) meet in the L1 on the dz pieces.  Bound by reading W as long as one or
// two blocks of 128 rows share it; with more rows the matrix work takes over, at a lower rate than the tile of
// gemm_core.hpp (the limit and both sides' times: kFewRows).
struct FewRowsParams {
  const __bf16* dz;       // K-blocked, whole blocks of 256 rows
  const __bf16* weight;
  float* partial;         // [k_split][rows][H]
  int64_t n_kslab;
  int rows, H, V;
  int n_h, n_t, k_split, slabs_per_split;
};

__global__ __launch_bounds__(256, 1) void dhidden_few_rows_kernel(FewRowsParams p) {
  const int item = xcd_remap(blockIdx.x, gridDim.x);
  if (item >= p.n_h * p.n_t * p.k_split) return;
  const int tt = item % p.n_t, ks = item / p.n_t / p.n_h;
  const int h0 = ((item / p.n_t % p.n_h) * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)) * 128;
  if (h0 >= p.H) return;
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int s0 = ks * p.slabs_per_split;
  const int n_slab = p.n_kslab - s0 < p.slabs_per_split ? (int)(p.n_kslab - s0) : p.slabs_per_split;
  const int last = 2 * n_slab - 1;                                // steps of 32 vocabulary rows
  const int col = h0 + 8 * c < p.H ? h0 + 8 * c : p.H - 8;        // columns past H: any, they are not stored
  const __bf16* z = p.dz + (((int64_t)(tt >> 1) * p.n_kslab + s0) * kBlockRows + (tt & 1) * 128 + c) * 64 + 8 * g;

  // Range-checked loads from a descriptor over the step's valid rows: rows past V read as zero, and no branch stands
  // between a request and the matrix instructions it is to overlap.  What is checked is the per-lane offset, so the row
  // is part of it (a scalar offset is outside the check by the builtin's contract).
  const int row_bytes = p.H * 2, voff = 8 * g * row_bytes + col * 2;
  auto load_a = [&](u32x4 (&raw)[8], int n) __attribute__((always_inline)) {
    const int v0 = s0 * 64 + (n < last ? n : last) * 32;
    const int rows = p.V - v0 < 32 ? (p.V > v0 ? p.V - v0 : 0) : 32;
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<__bf16*>(p.weight) + (int64_t)v0 * p.H, 0, rows * row_bytes, 0x00020000);
#pragma unroll
    for (int e = 0; e < 8; ++e) raw[e] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff + e * row_bytes, 0, 0);
  };
  auto load_b = [&](u32x4 (&b)[8], int n) __attribute__((always_inline)) {
    const int m = n < last ? n : last;
    const __bf16* at = z + (int64_t)(m >> 1) * (kBlockRows * 64) + (m & 1) * 32;
#pragma unroll
    for (int j = 0; j < 8; ++j) b[j] = *reinterpret_cast<const u32x4*>(at + j * 16 * 64);
  };
  f32x4 acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc_set(acc[i][j], 0.f, 0.f, 0.f, 0.f);
  u32x4 raw0[8], raw1[8], b0[8], b1[8];
  // one step: the fragments of `raw`, the requests for the step after next into it, the products with `b`
  auto step = [&](u32x4 (&raw)[8], const u32x4 (&b)[8], int n) __attribute__((always_inline)) {
    u32x4 a[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        a[i][q] = __builtin_amdgcn_perm(raw[2 * q + 1][i / 2], raw[2 * q][i / 2], i % 2 ? 0x07060302u : 0x05040100u);
    __builtin_amdgcn_sched_barrier(0);
    load_a(raw, n + 2);
    GemmTile<__bf16, 8>::settle();     // vector results on their way into matrix instructions
    each<64>([&](auto m) __attribute__((always_inline)) { Mma<__bf16>::slot(acc, a, b, decltype(m)::value); });
    __builtin_amdgcn_sched_barrier(0);
  };
  load_a(raw0, 0);
  load_b(b0, 0);
  load_a(raw1, 1);
  for (int s = 0; s < n_slab; ++s) {
    load_b(b1, 2 * s + 1);
    step(raw0, b0, 2 * s);
    load_b(b0, 2 * s + 2);
    step(raw1, b1, 2 * s + 1);
  }
  GemmTile<__bf16, 8>::settle();
  // register r of block (i, j): column 8 (4 g + r) + i, row 16 j + c
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int t = tt * 128 + 16 * j + c;
    if (t >= p.rows) continue;
    float* row = p.partial + ((int64_t)ks * p.rows + t) * p.H;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int h = h0 + 8 * (4 * g + r);
      if (h >= p.H) continue;
      f32x4 lo, hi;
#pragma unroll
      for (int i = 0; i < 4; ++i) { lo[i] = acc_get(acc[i][j], r); hi[i] = acc_get(acc[4 + i][j], r); }
      *reinterpret_cast<f32x4*>(row + h) = lo;
      *reinterpret_cast<f32x4*>(row + h + 4) = hi;
    }
  }
}

// K ranges: one workgroup per CU, none empty, at least 8 slabs each; fewer the more rows their partial sums have (384
// rows at H = 1024, V = 32000: whole step 284 us with 32 ranges, 295 with 42).
// Up to three blocks of 128 rows: whole training steps with W^T / without it, us, V = 151936 (H = 7168: 129280):
//   H = 2048: 100 rows 1030 / 809, 200 1165 / 983, 384 1298 / 1183, 512 1368 / 1317, 700 1634 / 1682
//   H = 4096: 100 rows 1669 / 1235, 200 1875 / 1556, 384 2235 / 2021, 512 2385 / 2317, 700 2997 / 3036
//   H = 7168: 100 rows 2351 / 1704, 200 2629 / 2213, 384 3289 / 2867, 480 3505 / 3590
constexpr int64_t kFewRows = 384;
struct FewRowsPlan {
  int n_h, n_t, k_split, slabs_per_split;
  size_t partial_bytes;
};
static FewRowsPlan plan_few_rows(int64_t rows, int64_t H, int64_t ldv, int cus, size_t partial_cap) {
  FewRowsPlan pl;
  pl.n_h = (int)((H + 511) / 512);
  pl.n_t = (int)((rows + 127) / 128);
  const int64_t n_slab = ldv / 64;
  int64_t s = cus / (pl.n_h * pl.n_t);
  const int64_t most = (int64_t)(partial_cap / ((size_t)rows * H * sizeof(float)));
  if (s > 64) s = 64;
  if (s > 96 / pl.n_t) s = 96 / pl.n_t;
  if (s > n_slab / 8) s = n_slab / 8;
  if (s > most) s = most;
  if (s < 1) s = 1;
  pl.slabs_per_split = (int)((n_slab + s - 1) / s);
  pl.k_split = (int)((n_slab + pl.slabs_per_split - 1) / pl.slabs_per_split);
  pl.partial_bytes = (size_t)pl.k_split * rows * H * sizeof(float);
  return pl;
}
static bool few_rows(int64_t rows, int64_t T, size_t es, bool saved, bool own_wt) {
  return es == 2 && saved && own_wt && rows == T && rows <= kFewRows;
}

struct BwdPlan {
  int64_t ldv;        // K extent of dz / WT (V rounded up to 64)
  int64_t chunk;      // tokens per chunk (multiple of 256 unless >= T)
  int64_t ldt;        // K extent of dzT / hidT for a full chunk (tokens rounded up to 64)
  size_t off_wt, off_hidt, off_dz, off_dzt, off_part, part_bytes, total;
};

static BwdPlan bwd_plan(int64_t T, int64_t H, int64_t V, size_t es, int64_t chunk_tokens, bool saved = false,
                        bool own_wt = true, bool own_dw = true) {
  BwdPlan pl;
  pl.ldv = round_up64(V, 64);
  int64_t chunk = (chunk_tokens <= 0 || chunk_tokens >= T) ? T : round_up64(chunk_tokens, 256);
  if (chunk > T) chunk = T;
  pl.chunk = chunk;
  pl.ldt = round_up64(chunk, 64);
  size_t off = 0;
  // K-blocked operands: whole blocks of 256 rows
  const size_t Hb = (size_t)round_up64(H, 256), Cb = (size_t)round_up64(chunk, 256), Vb = (size_t)round_up64(V, 256);
  const bool few = few_rows(chunk, T, es, saved, own_wt);       // reads W itself
  pl.off_wt = off;   off += own_wt && !few ? align_up(Hb * pl.ldv * es, 256) : 0;
  pl.off_hidt = off; off += own_dw ? align_up(Hb * pl.ldt * es, 256) : 0;
  pl.off_dz = off;   off += saved ? 0 : align_up(Cb * pl.ldv * es, 256);
  pl.off_dzt = off;  off += own_dw ? align_up(Vb * pl.ldt * es, 256) : 0;
  // split-K partials of the dhidden GEMM and of the dW GEMM's tail (used one after the other): what a full chunk and
  // the shorter last chunk want
  const int slab = (int)(kRowBytes / es);
  size_t part = 0;
  for (size_t b : {dhidden_partial_bytes(chunk, H, pl.ldv, slab), dhidden_partial_bytes(T % chunk, H, pl.ldv, slab),
                   own_dw ? dweight_partial_bytes(chunk, H, V, slab) : 0, own_dw ? dweight_partial_bytes(T % chunk, H, V, slab) : 0})
    if (b > part) part = b;
  if (few) {
    const size_t b = plan_few_rows(chunk, H, pl.ldv, 256, (size_t)1 << 30).partial_bytes;
    if (b > part) part = b;
  }
  pl.part_bytes = align_up(part, 256);
  pl.off_part = off; off += pl.part_bytes;
  pl.total = off;
  return pl;
}

// Largest chunk (multiple of 256, or T itself) whose plan fits into `bytes`; 0 if none does.
static int64_t chunk_for_workspace(int64_t T, int64_t H, int64_t V, size_t es, size_t bytes, bool saved, bool own_wt, bool own_dw) {
  if (bwd_plan(T, H, V, es, T, saved, own_wt, own_dw).total <= bytes) return T;
  int64_t lo = 0, hi = T / 256;   // in units of 256 tokens
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) / 2;
    if (bwd_plan(T, H, V, es, mid * 256, saved, own_wt, own_dw).total <= bytes) lo = mid; else hi = mid - 1;
  }
  return lo * 256;
}

template <typename OutT>
static int launch_splitk_reduce(const float* partial, int k_split, int rows, int cols, OutT* C, int64_t ldc, int accumulate,
                                const int32_t* order, hipStream_t stream) {
  const int threads = cols / 4 >= 256 ? 256 : (cols / 4 + 63) / 64 * 64;
  hipLaunchKernelGGL(splitk_reduce_kernel<OutT>, dim3(rows, (cols / 4 + threads - 1) / threads), dim3(threads), 0, stream,
                     partial, k_split, (int64_t)rows * cols, cols, C, ldc, accumulate, order);
  return check_launch("splitk_reduce_kernel");
}

template <typename T, typename OutT, bool kMContig>
static int launch_gemm_one(const void* A, int64_t a_kslabs, int M, const void* B, int64_t b_kslabs, int N, int K, void* C,
                           int64_t ldc, int accumulate, hipStream_t stream, float* partial, size_t partial_bytes,
                           int k_split_wanted, const RowOrder& rows = RowOrder{nullptr, 0}) {
  using Tile = OutTile<T, kMContig>;
  int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(&gemm_nt_kernel<T, OutT, kMContig>), Tile::kLdsBytes, "gemm_nt_kernel");
  if (rc) return rc;
  GemmParams g;
  g.A = A; g.B = B; g.C = C; g.a_kslabs = a_kslabs; g.b_kslabs = b_kslabs; g.ldc = ldc;
  g.M = M; g.N = N; g.K = K;
  g.n_mt = (M + 255) / 256; g.n_nt = (N + 255) / 256;
  g.accumulate = accumulate;
  g.order = rows.order; g.total = rows.total;
  const int slab = Tile::kSlabK;
  const int cus = device_cu_count();
  g.k_split = (partial && partial_bytes) ? k_split_wanted : 1;
  auto fits = [&](int ks) {      // partials fit the buffer and no K range is empty after rounding to whole slabs
    if (ks <= 1) return true;
    if ((size_t)ks * M * N * sizeof(float) > partial_bytes) return false;
    return (int64_t)(ks - 1) * round_up64((K + ks - 1) / ks, slab) < K;
  };
  while (!fits(g.k_split)) --g.k_split;
  g.k_per_split = g.k_split > 1 ? (int)round_up64((K + g.k_split - 1) / g.k_split, slab) : K;
  g.partial = partial;
  // Many more tiles than CUs and no K split: let one workgroup per CU walk runs of tiles instead of
  // launching one workgroup per tile.
  const int n_fixed = kMContig ? g.n_mt : g.n_nt, n_moving = kMContig ? g.n_nt : g.n_mt;
  g.n_walk = 0;
  if (g.k_split == 1 && n_fixed <= cus && g.n_mt * g.n_nt >= 4 * cus && K >= 2 * slab) {
    g.n_walk = cus / n_fixed;
    if (g.n_walk > n_moving) g.n_walk = n_moving;
    // A walk is as long as its longest run; one workgroup per tile takes ceil(tiles / CUs) rounds.  Streaming the K
    // loops into each other is worth a few per cent, not a whole extra tile period (H = 7168: 28 x 64 tiles are 7
    // rounds exactly, while 9 walks over 64 tiles make runs of 7 and 8).
    const long walk_periods = (n_moving + g.n_walk - 1) / g.n_walk;
    const long plain_rounds = ((long)g.n_mt * g.n_nt + cus - 1) / cus;
    if (walk_periods * 100 > plain_rounds * 104) g.n_walk = 0;
  }
  int grid = ((g.n_walk > 0 ? g.n_walk * n_fixed : g.n_mt * g.n_nt * g.k_split) + 7) / 8 * 8;
  hipLaunchKernelGGL((gemm_nt_kernel<T, OutT, kMContig>), dim3(grid), dim3(Tile::kThreads), Tile::kLdsBytes, stream, g);
  rc = check_launch("gemm_nt_kernel");
  if (rc || g.k_split == 1) return rc;
  return launch_splitk_reduce<OutT>(partial, g.k_split, kMContig ? N : M, kMContig ? M : N, static_cast<OutT*>(C), ldc, accumulate,
                                    rows.order, stream);
}

// C (+)= A B^T under the launch plan of its orientation: plan_dhidden (C[n][m], with `partial`) or plan_dweight (C[m][n]).
template <typename T, typename OutT, bool kMContig>
static int launch_gemm(const void* A, int64_t a_kslabs, int M, const void* B, int64_t b_kslabs, int N, int K, void* C,
                       int64_t ldc, int accumulate, hipStream_t stream, float* partial = nullptr,
                       size_t partial_bytes = 0, const RowOrder& rows = RowOrder{nullptr, 0}) {
  using Tile = OutTile<T, kMContig>;
  constexpr int64_t kSlabElems = (int64_t)kBlockRows * Tile::kSlabK;
  if (!kMContig) {
    // dW: equally long walks over most vocabulary tiles, the rest cut into K ranges (plan_dweight)
    const DwPlan dw = plan_dweight(M, N, K, Tile::kSlabK, device_cu_count(), partial ? partial_bytes : 0);
    if (dw.bulk_mt == 0)
      return launch_gemm_one<T, OutT, kMContig>(A, a_kslabs, M, B, b_kslabs, N, K, C, ldc, accumulate, stream, nullptr, 0, 1);
    const int bulk_rows = dw.bulk_mt * 256;
    int rc = launch_gemm_one<T, OutT, kMContig>(A, a_kslabs, bulk_rows, B, b_kslabs, N, K, C, ldc, accumulate, stream, nullptr, 0, 1);
    if (rc) return rc;
    const T* a_tail = static_cast<const T*>(A) + (int64_t)dw.bulk_mt * a_kslabs * kSlabElems;
    OutT* c_tail = static_cast<OutT*>(C) + (int64_t)bulk_rows * ldc;
    return launch_gemm_one<T, OutT, kMContig>(a_tail, a_kslabs, M - bulk_rows, B, b_kslabs, N, K, c_tail, ldc, accumulate, stream,
                                              dw.k_split > 1 ? partial : nullptr, dw.k_split > 1 ? partial_bytes : 0, dw.k_split);
  }
  if (!(partial && partial_bytes))
    return launch_gemm_one<T, OutT, kMContig>(A, a_kslabs, M, B, b_kslabs, N, K, C, ldc, accumulate, stream, nullptr, 0, 1, rows);
  const DhPlan pl = plan_dhidden(N, M, K, Tile::kSlabK, device_cu_count(), partial_bytes);
  if (pl.bulk_nt == 0)
    return launch_gemm_one<T, OutT, kMContig>(A, a_kslabs, M, B, b_kslabs, N, K, C, ldc, accumulate, stream, partial,
                                              partial_bytes, pl.k_split, rows);
  const int bulk_rows = pl.bulk_nt * 256;
  int rc = launch_gemm_one<T, OutT, kMContig>(A, a_kslabs, M, B, b_kslabs, bulk_rows, K, C, ldc, accumulate, stream,
                                              nullptr, 0, 1, rows);
  if (rc) return rc;
  const T* b_tail = static_cast<const T*>(B) + (int64_t)pl.bulk_nt * b_kslabs * kSlabElems;
  OutT* c_tail = static_cast<OutT*>(C) + (rows.order ? 0 : (int64_t)bulk_rows * ldc);
  const RowOrder tail{rows.order ? rows.order + bulk_rows : nullptr, rows.total};
  return launch_gemm_one<T, OutT, kMContig>(A, a_kslabs, M, b_tail, b_kslabs, N - bulk_rows, K, c_tail, ldc, accumulate,
                                            stream, partial, partial_bytes, pl.k_split, tail);
}

template <typename T>
static int launch_transpose(const T* src, int64_t ld_src, T* dst, int64_t r_dst, int R, int C, hipStream_t stream,
                            const int32_t* order = nullptr, int64_t ld_dst = 0) {
  dim3 grid((C + 63) / 64, (int)((r_dst + 63) / 64));
  hipLaunchKernelGGL(transpose_block_kernel<T>, grid, dim3(256), 0, stream, src, ld_src, dst, ld_dst ? ld_dst : r_dst, r_dst, R, C, order);
  return check_launch("transpose_block_kernel");
}

template <typename T>
static int run_dweight(const T* dzt, const T* hidt, int64_t ld, int64_t k, int64_t V, int64_t H, void* dweight, bool to_bf16,
                       bool accumulate, void* partial, size_t partial_bytes, hipStream_t stream) {
  // dW[v][h] (+)= sum_t dzT(v, t) hidT(h, t)   (M = V, N = H, K = the first k of ld tokens, C[m][n])
  constexpr int slab = GemmTile<T, 4>::kSlabK;
  if constexpr (sizeof(T) == 2) {
    if (to_bf16)
      return launch_gemm<T, __bf16, false>(dzt, ld / slab, (int)V, hidt, ld / slab, (int)H, (int)k, dweight, H, 0, stream,
                                           static_cast<float*>(partial), partial_bytes);
  }
  return launch_gemm<T, float, false>(dzt, ld / slab, (int)V, hidt, ld / slab, (int)H, (int)k, dweight, H, accumulate ? 1 : 0, stream,
                                      static_cast<float*>(partial), partial_bytes);
}

template <typename T>
static int run_bwd(const clgrpo_lmhead_bwd_args* a, hipStream_t stream, int64_t label_offset, const RowOrder& rows,
                   const DwOperands* kept) {
  using Tile = LogitTile<T>;
  const int64_t T_ = a->T, H = a->H, V = a->V;
  const bool saved = a->saved_logits != nullptr;
  const bool own_wt = a->weight_t == nullptr;
  const bool own_dw = kept == nullptr;
  const int64_t chunk = chunk_for_workspace(T_, H, V, sizeof(T), a->workspace_bytes, saved, own_wt, own_dw);
  if (chunk <= 0)
    return fail(CLGRPO_EWORKSPACE, "clgrpo_lmhead_bwd: workspace %zu bytes cannot hold a 256-token chunk (%zu needed)",
                a->workspace_bytes, bwd_plan(T_, H, V, sizeof(T), 256, saved, own_wt, own_dw).total);
  if (a->dweight_bf16 && chunk < T_)
    return fail(CLGRPO_EWORKSPACE, "clgrpo_lmhead_bwd: a 16-bit dweight needs a workspace for all %lld tokens at once", (long long)T_);
  const BwdPlan pl = bwd_plan(T_, H, V, sizeof(T), chunk, saved, own_wt, own_dw);
  const int64_t ldz = saved ? a->ld_saved : pl.ldv;
  char* ws = static_cast<char*>(a->workspace);
  T* wt = a->weight_t ? static_cast<T*>(a->weight_t) : reinterpret_cast<T*>(ws + pl.off_wt);
  T* dz_ws = reinterpret_cast<T*>(ws + pl.off_dz);
  const T* hidden = static_cast<const T*>(a->hidden);
  const T* weight = static_cast<const T*>(a->weight);

  int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(&lmhead_dz_kernel<T>), Tile::kLdsBytes, "lmhead_dz_kernel");
  if (rc) return rc;
  const bool few = few_rows(chunk, T_, sizeof(T), saved, own_wt);
  if (a->dhidden && !few && !(a->weight_t && a->weight_t_ready)) {
    // WT(h, v) = W[v][h], zero for V <= v < ldv, K-blocked
    rc = launch_transpose<T>(weight, H, wt, pl.ldv, (int)V, (int)H, stream);
    if (rc) return rc;
  }
  for (int64_t c0 = 0; c0 < T_; c0 += chunk) {
    const int64_t tc = (T_ - c0) < chunk ? (T_ - c0) : chunk;
    const int64_t ldt = round_up64(tc, 64);
    // the operands of dW: this chunk's own, or its place among the ones that the caller contracts later
    constexpr int64_t kSlabElems = (int64_t)kBlockRows * Tile::kSlabK;
    const int64_t k0 = kept ? kept->k + c0 : 0, ld_dw = kept ? kept->ld : ldt;
    T* dzt = (kept ? static_cast<T*>(kept->dzt) : reinterpret_cast<T*>(ws + pl.off_dzt)) + k0 / Tile::kSlabK * kSlabElems;
    T* hidt = (kept ? static_cast<T*>(kept->hidt) : reinterpret_cast<T*>(ws + pl.off_hidt)) + k0 / Tile::kSlabK * kSlabElems;
    T* dz = saved ? static_cast<T*>(a->saved_logits) + c0 * ldz : dz_ws;
    // with an order the chunk's tokens are looked up from the start of the arrays, without they follow one another
    const int64_t t0 = rows.order ? 0 : c0;
    const int32_t* order = rows.order ? rows.order + c0 : nullptr;
    if (saved) {
      DzFromZParams q;
      q.z = dz;
      q.dzT = dzt;
      q.labels = a->labels + t0;
      q.label_offset = label_offset;
      q.lse = a->lse + t0;
      q.entropy = a->g_entropy ? a->entropy + t0 : nullptr;
      q.g_lp = a->g_logprob + t0;
      q.g_ent = a->g_entropy ? a->g_entropy + t0 : nullptr;
      q.order = order;
      q.Tc = (int)tc;
      q.ldt = (int)ldt;
      q.t_slabs = ld_dw / Tile::kSlabK;
      q.V = (int)V;
      q.ldv = (int)ldz;
      q.c = a->inv_temperature * kLog2e;
      q.inv_temperature = a->inv_temperature;
      // a workgroup walks units of one token block, so that its coefficients are fetched once; 16 workgroups per CU
      const int64_t n_tb = (tc + kBlockRows - 1) / kBlockRows, n_units = ldz / Elem<T>::kSlabK;
      int64_t per_tb = (16 * (int64_t)device_cu_count() + n_tb - 1) / n_tb;
      if (per_tb > n_units) per_tb = n_units;
      dim3 grid((unsigned)n_tb, (unsigned)per_tb);
      hipLaunchKernelGGL(dz_from_z_kernel<T>, grid, dim3(256), 0, stream, q);
      rc = check_launch("dz_from_z_kernel");
      if (rc) return rc;
    } else {
      DzParams d;
      d.hidden = hidden + c0 * H;
      d.weight = weight;
      d.labels = a->labels + c0;
      d.label_offset = label_offset;
      d.lse = a->lse + c0;
      d.entropy = a->g_entropy ? a->entropy + c0 : nullptr;
      d.g_lp = a->g_logprob + c0;
      d.g_ent = a->g_entropy ? a->g_entropy + c0 : nullptr;
      d.Tc = (int)tc;
      d.ldt = (int)ldt;
      d.H = (int)H;
      d.V = (int)V;
      d.ldv = (int)pl.ldv;
      d.n_tb = (int)((ldt + 255) / 256);
      d.n_vt = (int)((V + 255) / 256);
      d.c = a->inv_temperature * kLog2e;
      d.inv_temperature = a->inv_temperature;
      d.dz = dz;
      d.dzT = dzt;
      int grid = (d.n_tb * d.n_vt + 7) / 8 * 8;
      hipLaunchKernelGGL(lmhead_dz_kernel<T>, dim3(grid), dim3(Tile::kThreads), Tile::kLdsBytes, stream, d);
      rc = check_launch("lmhead_dz_kernel");
      if (rc) return rc;
    }
    if (a->dhidden && few) {
      const FewRowsPlan fp = plan_few_rows(tc, H, pl.ldv, device_cu_count(), pl.part_bytes);
      FewRowsParams q;
      q.dz = reinterpret_cast<const __bf16*>(dz);
      q.weight = reinterpret_cast<const __bf16*>(weight);
      q.partial = reinterpret_cast<float*>(ws + pl.off_part);
      q.n_kslab = ldz / 64;
      q.rows = (int)tc; q.H = (int)H; q.V = (int)V;
      q.n_h = fp.n_h; q.n_t = fp.n_t; q.k_split = fp.k_split; q.slabs_per_split = fp.slabs_per_split;
      hipLaunchKernelGGL(dhidden_few_rows_kernel, dim3((fp.n_h * fp.n_t * fp.k_split + 7) / 8 * 8), dim3(256), 0, stream, q);
      rc = check_launch("dhidden_few_rows_kernel");
      if (rc) return rc;
      rc = launch_splitk_reduce<T>(q.partial, fp.k_split, (int)tc, (int)H, static_cast<T*>(a->dhidden) + t0 * H, H, 0, order, stream);
      if (rc) return rc;
    } else if (a->dhidden) {
      // dhidden[chunk][h] = sum_v WT[h][v] dz[t][v]   (M = H, N = tokens, C[n][m])
      rc = launch_gemm<T, T, true>(wt, pl.ldv / Tile::kSlabK, (int)H, dz, ldz / Tile::kSlabK, (int)tc, (int)pl.ldv,
                             static_cast<T*>(a->dhidden) + t0 * H, H, 0, stream,
                             reinterpret_cast<float*>(ws + pl.off_part), pl.part_bytes, RowOrder{order, rows.total});
      if (rc) return rc;
    }
    if (a->dweight || kept) {
      // hidT(h, t) = hidden[c0 + t][h], zero for tc <= t < ldt, K-blocked
      rc = launch_transpose<T>(hidden + t0 * H, H, hidt, ldt, (int)tc, (int)H, stream, order, ld_dw);
      if (rc) return rc;
    }
    if (a->dweight && !kept) {
      rc = run_dweight<T>(dzt, hidt, ldt, ldt, V, H, a->dweight, a->dweight_bf16 != 0, a->accumulate_dweight || c0 > 0,
                          ws + pl.off_part, pl.part_bytes, stream);
      if (rc) return rc;
    }
  }
  return CLGRPO_OK;
}

}  // namespace clgrpo

using namespace clgrpo;

extern "C" size_t clgrpo_lmhead_bwd_workspace_bytes(int64_t T, int64_t H, int64_t V, int32_t dtype,
                                                    int64_t chunk_tokens, int32_t with_saved_logits) {
  if (T <= 0 || H <= 0 || V <= 0 || (dtype != CLGRPO_BF16 && dtype != CLGRPO_F32)) return 0;
  return bwd_plan(T, H, V, dtype_bytes(dtype), chunk_tokens, (with_saved_logits & 1) != 0, (with_saved_logits & 2) == 0,
                  (with_saved_logits & 4) == 0).total;
}

extern "C" int clgrpo_lmhead_bwd_dhidden_plan(int64_t rows, int64_t H, int64_t V, int32_t dtype, int32_t cus, int32_t* out) {
  if (rows <= 0 || H <= 0 || V <= 0 || out == nullptr || (dtype != CLGRPO_BF16 && dtype != CLGRPO_F32)) return CLGRPO_EINVAL;
  const int slab = (int)(kRowBytes / dtype_bytes(dtype));
  const DhPlan pl = plan_dhidden(rows, H, round_up64(V, 64), slab, cus > 0 ? cus : 256, (size_t)1 << 30);
  out[0] = pl.bulk_nt;
  out[1] = pl.k_split;
  return CLGRPO_OK;
}

extern "C" int clgrpo_lmhead_bwd_dweight_plan(int64_t rows, int64_t H, int64_t V, int32_t dtype, int32_t cus, int32_t* out) {
  if (rows <= 0 || H <= 0 || V <= 0 || out == nullptr || (dtype != CLGRPO_BF16 && dtype != CLGRPO_F32)) return CLGRPO_EINVAL;
  const int slab = (int)(kRowBytes / dtype_bytes(dtype));
  const DwPlan pl = plan_dweight(V, H, round_up64(rows, 64), slab, cus > 0 ? cus : 256, (size_t)1 << 30);
  out[0] = pl.n_walk;
  out[1] = pl.bulk_mt;
  out[2] = pl.k_split;
  return CLGRPO_OK;
}

extern "C" size_t clgrpo_dweight_workspace_bytes(int64_t k, int64_t H, int64_t V, int32_t dtype) {
  if (k <= 0 || H <= 0 || V <= 0 || (dtype != CLGRPO_BF16 && dtype != CLGRPO_F32)) return 0;
  return align_up(dweight_partial_bytes(k, H, V, (int)(kRowBytes / dtype_bytes(dtype))), 256);
}

extern "C" int clgrpo_dweight(const clgrpo_dweight_args* a, void* stream) {
  static const char* who = "clgrpo_dweight";
  CLGRPO_REQUIRE_PTR(a, "args");
  int rc = validate_head_shape(who, a->k, a->H, a->V, a->dtype);
  if (rc) return rc;
  if (a->k % 64 != 0 || a->ld % 64 != 0 || a->ld < a->k)
    return fail(CLGRPO_ESHAPE, "%s: k=%lld of ld=%lld must be multiples of 64", who, (long long)a->k, (long long)a->ld);
  CLGRPO_REQUIRE_PTR(a->dzt, "dzt");
  CLGRPO_REQUIRE_PTR(a->hidt, "hidt");
  CLGRPO_REQUIRE_PTR(a->dweight, "dweight");
  if (a->dweight_bf16 && (a->accumulate || a->dtype != CLGRPO_BF16))
    return fail(CLGRPO_EINVAL, "%s: a 16-bit dweight needs 16-bit operands and is not added to", who);
  const size_t need = clgrpo_dweight_workspace_bytes(a->k, a->H, a->V, a->dtype);
  if (need > 0) CLGRPO_REQUIRE_PTR(a->workspace, "workspace");
  if (a->workspace_bytes < need)
    return fail(CLGRPO_EWORKSPACE, "%s: workspace %zu < %zu bytes", who, a->workspace_bytes, need);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (a->dtype == CLGRPO_BF16)
    return run_dweight<__bf16>(static_cast<const __bf16*>(a->dzt), static_cast<const __bf16*>(a->hidt), a->ld, a->k, a->V, a->H,
                               a->dweight, a->dweight_bf16 != 0, a->accumulate != 0, a->workspace, a->workspace_bytes, s);
  return run_dweight<float>(static_cast<const float*>(a->dzt), static_cast<const float*>(a->hidt), a->ld, a->k, a->V, a->H,
                            a->dweight, false, a->accumulate != 0, a->workspace, a->workspace_bytes, s);
}

int clgrpo::head_backward(const char* who, const clgrpo_lmhead_bwd_args* a, int64_t vocab_begin, const RowOrder& rows,
                          hipStream_t s, const DwOperands* kept) {
  CLGRPO_REQUIRE_PTR(a, "args");
  int rc = validate_head_shape(who, a->T, a->H, a->V, a->dtype);
  if (rc) return rc;
  CLGRPO_REQUIRE_PTR(a->hidden, "hidden");
  CLGRPO_REQUIRE_PTR(a->weight, "weight");
  CLGRPO_REQUIRE_PTR(a->labels, "labels");
  CLGRPO_REQUIRE_PTR(a->lse, "lse");
  CLGRPO_REQUIRE_PTR(a->g_logprob, "g_logprob");
  if (a->g_entropy != nullptr) CLGRPO_REQUIRE_PTR(a->entropy, "entropy");
  if (a->dhidden == nullptr && a->dweight == nullptr && kept == nullptr)
    return fail(CLGRPO_ENULL, "%s: both dhidden and dweight are NULL", who);
  if (a->dweight_bf16 && (a->accumulate_dweight || a->dtype != CLGRPO_BF16))
    return fail(CLGRPO_EINVAL, "%s: a 16-bit dweight needs 16-bit operands and is not added to", who);
  if (kept != nullptr && (a->saved_logits == nullptr || kept->k < 0 || kept->k % 64 != 0 || kept->ld % 64 != 0 ||
                          kept->k + round_up64(a->T, 64) > kept->ld))
    return fail(CLGRPO_ESHAPE, "%s: %lld tokens do not fit behind the %lld of %lld kept for dweight", who, (long long)a->T,
                (long long)kept->k, (long long)kept->ld);
  if (vocab_begin < 0) return fail(CLGRPO_EINVAL, "%s: vocab_begin=%lld", who, (long long)vocab_begin);
  if (!(a->inv_temperature > 0.f)) return fail(CLGRPO_EINVAL, "%s: inv_temperature must be > 0", who);
  CLGRPO_REQUIRE_PTR(a->workspace, "workspace");
  if (a->saved_logits != nullptr && (a->ld_saved < round_up64(a->V, 64) || a->ld_saved % 64 != 0))
    return fail(CLGRPO_ESHAPE, "%s: ld_saved=%lld must be a multiple of 64 and >= %lld", who, (long long)a->ld_saved,
                (long long)round_up64(a->V, 64));
  if (a->saved_logits != nullptr && a->saved_rows < round_up64(a->T, 256))
    return fail(CLGRPO_ESHAPE, "%s: saved_rows=%lld, but the kept-logits buffer must hold %lld rows (T rounded up to 256)", who,
                (long long)a->saved_rows, (long long)round_up64(a->T, 256));
  if (rows.order != nullptr && (a->saved_logits == nullptr || rows.total < a->T ||
                                rows.total * a->H * (int64_t)dtype_bytes(a->dtype) > kMaxOrderedBytes))
    return fail(CLGRPO_ESHAPE, "%s: a row order needs kept logits and at most %lld bytes of hidden states", who,
                (long long)kMaxOrderedBytes);
  return a->dtype == CLGRPO_BF16 ? run_bwd<__bf16>(a, s, vocab_begin, rows, kept) : run_bwd<float>(a, s, vocab_begin, rows, kept);
}

extern "C" int clgrpo_lmhead_bwd(const clgrpo_lmhead_bwd_args* a, void* stream) {
  CLGRPO_REQUIRE_PTR(a, "args");
  return head_backward("clgrpo_lmhead_bwd", a, 0, RowOrder{nullptr, a->T}, static_cast<hipStream_t>(stream));
}

extern "C" int clgrpo_lmhead_bwd_shard(const clgrpo_lmhead_bwd_args* a, int64_t vocab_begin, void* stream) {
  CLGRPO_REQUIRE_PTR(a, "args");
  return head_backward("clgrpo_lmhead_bwd_shard", a, vocab_begin, RowOrder{nullptr, a->T}, static_cast<hipStream_t>(stream));
}
