// Backward of the fused lm_head + log-softmax statistics.
//
// Per chunk of tokens (the chunk length is set by the workspace the caller gives):
//   1. d(logits) in place of the chunk's kept logits, or by recomputing a z^T tile [256 vocab x 256 tokens] on the
//      matrix cores exactly as the forward does.
//   2. dhidden[chunk] = dz * W        K = vocabulary, which runs across the rows of W
//   3. dW (+)= dz^T * hidden[chunk]   K = tokens, which run across the rows of dz, against hidT = hidden[chunk]^T; fp32 out
// Both contractions run through the MFMA tile of gemm_core.hpp, which turns an operand that lies across on its way
// from LDS into the matrix cores (see Side): neither W^T nor dz^T is formed.  Measured against NT products of transposed
// copies: see Side.
//
// Algorithmic work: 4*T*H*V flop (dhidden + dW); the z recomputation (2*T*H*V) is overhead.
#include "head_internal.hpp"
#include "gemm_core.hpp"
#include <type_traits>

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
  int ldt;      // tokens of dz to write = Tc rounded up to 64 (zeros past Tc)
  int H, V;
  int ldv;      // vocabulary extent of dz = V rounded up to 64
  int n_tb, n_vt;
  float c, inv_temperature;
  void* dz;     // ldt x ldv, in units (see unit_index)
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
    const auto op_a = Tile::Operand::row_major(weight, p.H, a_rows), op_b = Tile::Operand::row_major(hidden, p.H, b_rows);
    core.start(op_a, op_b, nslab, lds);
    core.run(acc, nslab);
    if constexpr (Tile::kSplit) core.redo(acc, op_a, op_b, nslab, lds, [&] { Tile::zero(acc); });
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
  const float it = p.inv_temperature;
  constexpr int AG = VEC / 4;                 // blocks along A whose registers make up VEC consecutive vocabulary rows
#pragma unroll
  for (int i = 0; i < MI; i += AG) {
    const int v = v0 + la + Tile::a_block(i);
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      float d[VEC];
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        const float zraw = acc_get(acc[i + e / 4][j], e % 4);
        const float pr = __builtin_amdgcn_exp2f(fmaf(zraw, p.c, -lse[j] * kLog2e));
        const float logp = fmaf(zraw, it, -lse[j]);
        // dz = it * ( glp*(1[v==y] - p) - gent * p * (logp + ent) )
        float x = -it * pr * fmaf(gent[j], logp + ent[j], glp[j]);
        if (lab[j] == v + e) x += it * glp[j];
        if (v + e >= p.V || !block_live) x = 0.f;   // vocabulary padding columns / dead block
        d[e] = x;
      }
      const int t = t0 + lb + Tile::b_block(j);
      if (t < p.ldt && v < p.ldv)
        *reinterpret_cast<u32x4*>(dz + unit_index<T>(t, v, p.ldv / Tile::kSlabK)) = pack_vec(d, (T*)nullptr);
    }
  }
}

// dst(c, r) = src[r][c] (src[order[r]][c] with an order) for r < R, c < C and 0 for R <= r < r_dst, where dst is the K-blocked
// operand with C rows and ld_dst K elements (see blocked_index), of which the first r_dst are written.  64x64 tiles of 256
// threads, 16-byte accesses on both sides (C and ld_src are multiples of 32 elements here, so a 16-byte piece never
// straddles an edge).
template <typename T>
struct TransposeParams {
  const T* src;
  T* dst;
  int64_t ld_src, ld_dst, r_dst;
  int R, C;
  const int32_t* order;
};
template <typename T>
__device__ __forceinline__ void transpose_tile(const TransposeParams<T>& p, int r0, int c0) {
  constexpr int VEC = 16 / (int)sizeof(T);       // elements per 16-byte access
  constexpr int CPR = 64 / VEC;                  // accesses per 64-wide tile row
  constexpr int RPP = 256 / CPR;                 // tile rows covered per pass
  constexpr int kE = kRowBytes / (int)sizeof(T);
  __shared__ T tile[64][64 + VEC];               // [c][r], padded rows
  const int q = threadIdx.x % CPR, row = threadIdx.x / CPR;
  for (int rr = row; rr < 64; rr += RPP) {
    const int r = r0 + rr, c = c0 + q * VEC;
    alignas(16) T vals[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) vals[j] = (T)0.f;
    if (r < p.R && c < p.C)
      *reinterpret_cast<u32x4*>(vals) = *reinterpret_cast<const u32x4*>(p.src + (int64_t)(p.order ? p.order[r] : r) * p.ld_src + c);
#pragma unroll
    for (int j = 0; j < VEC; ++j) tile[q * VEC + j][rr] = vals[j];
  }
  __syncthreads();
  for (int cc = row; cc < 64; cc += RPP) {
    const int c = c0 + cc, r = r0 + q * VEC;
    if (c < p.C && r < p.r_dst)
      *reinterpret_cast<u32x4*>(p.dst + blocked_index<T>(c, r, p.ld_dst / kE)) = *reinterpret_cast<const u32x4*>(&tile[cc][q * VEC]);
  }
}
template <typename T>
__global__ __launch_bounds__(256) void transpose_block_kernel(TransposeParams<T> p) {
  transpose_tile<T>(p, blockIdx.y * 64, blockIdx.x * 64);
}

// d(logits) from kept logits: in place, or into the operands of dW that the caller keeps.  HBM-bound: reads and writes the
// chunk once.  A thread owns one 16-byte piece of one or two tokens in every unit that its workgroup walks: their
// coefficients stay in registers, the loads of kAhead units are in flight together, and a wave's access is one kilobyte.
// The units are walked from the vocabulary's end on, whose logits a forward of several rounds has written last, which the last-level
// cache still has, and dhidden, which begins at the other end, finds there what was written last here.  The pass and dhidden
// behind the forward, us: 143 rows at H = 1024, V = 32000 40.0 -> 38.4, 1064 at 2048, V = 151936 669 -> 661; loss dict of 6680 tokens
// at H = 2048 and its backward 8.78 -> 8.74 ms, a step of 200 tokens 148 -> 147 us.  Loads or stores around the cache: nothing.
// The last workgroups of the launch write hidden^T, dW's other operand, which took a launch of 5 to 12 us of its own.
// 12126 rows of the 152k vocabulary: 2.25 -> 1.49 ms, 32768 rows 5.92 -> 3.57 ms (5.6 TB/s), against a pass that also wrote the
// transpose.
struct DzTokens {
  const int64_t* labels;
  int64_t label_offset;
  const float* lse;
  const float* entropy;
  const float* g_lp;
  const float* g_ent;
  const int32_t* order;   // optional [Tc]: row n is token order[n] of the per-token arrays
  int Tc, V;
  float c, inv_temperature;
};
// d(logits) of a row from its raw logits z, tau = 1 / inv_temperature:  x = z c - lse log2(e);
// dz = tau^-1 (g_lp (1[v = y] - 2^x) - g_H 2^x (x ln 2 + H))  =  2^x (k1 + k2 x) + [v = y] top.
struct DzRow {
  float shift, k1, k2, top;   // shift = -lse log2(e)
  int label;                  // or -1
  bool live;                  // rows past the chunk and rows without a gradient give zeros
  template <bool kEntropy>
  __device__ __forceinline__ static DzRow of(const DzTokens& p, int n) {
    DzRow r;
    const bool ok = n < p.Tc;
    const int t = ok && p.order ? p.order[n] : n;
    const float glp = ok ? p.g_lp[t] : 0.f, gen = kEntropy && ok ? p.g_ent[t] : 0.f, ent = kEntropy && ok ? p.entropy[t] : 0.f;
    r.shift = ok ? -(p.lse[t] * kLog2e) : 0.f;
    r.top = p.inv_temperature * glp;
    r.k1 = kEntropy ? -p.inv_temperature * fmaf(gen, ent, glp) : -r.top;
    r.k2 = kEntropy ? -p.inv_temperature * gen * 0.6931471805599453f : 0.f;
    r.live = glp != 0.f || gen != 0.f;
    r.label = -1;
    if (ok) {
      const int64_t rel = p.labels[t] - p.label_offset;
      if (rel >= 0 && rel < p.V) r.label = (int)rel;
    }
    return r;
  }
};

template <typename T>
struct DzFromZParams {
  const void* z;      // kept logits (KeptLogit<T>): z_kslab units per row of units
  void* dz;           // d(logits) (T): dz_kslab units per row of units
  DzTokens t;
  int64_t z_kslab, dz_kslab;
  int n_units;        // units of dz per row of units
  int row0, row_units;   // rows of units to convert
  int n_step;            // workgroups per row of units
  int whole;             // units of such a row to convert
  int n_edge;            // rows of units, from the first on, of which the units from `whole` on are converted
  int turn_rows;         // workgroups behind those turn 64 x 64 hidden states each, this many of them along the tokens
  TransposeParams<T> turn;
};

template <typename T, bool kEntropy>
__global__ __launch_bounds__(256) void dz_from_z_kernel(DzFromZParams<T> p) {
  typedef typename KeptLogit<T>::type ZT;
  static_assert(sizeof(ZT) == sizeof(T), "d(logits) overwrites the kept logits in place");
  constexpr int E = Elem<T>::kSlabK;                // tokens and vocabulary entries of a unit (64 or 32)
  constexpr int VEC = 16 / (int)sizeof(T);          // elements per 16-byte piece
  constexpr int kRows = E / 32;                     // tokens per thread
  constexpr int kAhead = 4;                         // units in flight
  // the same for the whole workgroup: its row of units, its last unit and the least it may reach, or its square of hidden states
  int item = blockIdx.x, unit_row, unit, least = 0, step = p.n_step;
  if (item < p.row_units * p.n_step) {
    unit_row = p.row0 + item % p.row_units;
    unit = p.whole - 1 - item / p.row_units;
  } else if ((item -= p.row_units * p.n_step) < p.n_edge) {
    unit_row = item;
    unit = p.n_units - 1;
    least = p.whole;
    step = 1;
  } else {
    item -= p.n_edge;
    transpose_tile<T>(p.turn, item % p.turn_rows * 64, item / p.turn_rows * 64);
    return;
  }
  const int q = threadIdx.x & 7, row = threadIdx.x >> 3;
  DzRow r[kRows];
#pragma unroll
  for (int h = 0; h < kRows; ++h) r[h] = DzRow::of<kEntropy>(p.t, unit_row * E + h * 32 + row);
  const int at = row * kRowBytes + q * 16;          // byte of this thread's first piece within a unit
  const char* z = static_cast<const char*>(p.z) + (int64_t)unit_row * p.z_kslab * (E * kRowBytes) + at;
  char* dz = static_cast<char*>(p.dz) + (int64_t)unit_row * p.dz_kslab * (E * kRowBytes) + at;
  for (int k0 = unit; k0 >= least; k0 -= kAhead * step) {
    u32x4 raw[kAhead][kRows];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int ks = k0 - u * step >= least ? k0 - u * step : k0;
#pragma unroll
      for (int h = 0; h < kRows; ++h)
        raw[u][h] = *reinterpret_cast<const u32x4*>(z + (int64_t)ks * (E * kRowBytes) + h * 32 * kRowBytes);
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int ks = k0 - u * step;
      if (ks < least) break;
      const int v = ks * E + q * VEC;
#pragma unroll
      for (int h = 0; h < kRows; ++h) {
        const ZT* in = reinterpret_cast<const ZT*>(&raw[u][h]);
        float d[VEC];
        const bool here = (unsigned)(r[h].label - v) < (unsigned)VEC;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          const float x = fmaf((float)in[e], p.t.c, r[h].shift);
          d[e] = __builtin_amdgcn_exp2f(x) * (kEntropy ? fmaf(x, r[h].k2, r[h].k1) : r[h].k1);
        }
        if (here) {
#pragma unroll
          for (int e = 0; e < VEC; ++e)
            if (r[h].label - v == e) {
              const float x = fmaf((float)in[e], p.t.c, r[h].shift);
              d[e] = fmaf(__builtin_amdgcn_exp2f(x), kEntropy ? fmaf(x, r[h].k2, r[h].k1) : r[h].k1, r[h].top);
            }
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) d[e] = r[h].live ? d[e] : 0.f;
        if (v + VEC > p.t.V) {                      // vocabulary padding columns give zeros
#pragma unroll
          for (int e = 0; e < VEC; ++e)
            if (v + e >= p.t.V) d[e] = 0.f;
        }
        *reinterpret_cast<u32x4*>(dz + (int64_t)ks * (E * kRowBytes) + h * 32 * kRowBytes) = pack_vec(d, (T*)nullptr);
      }
    }
  }
}

// The same conversion, bit for bit, as a guest of dhidden's K loop (16-bit operands): while the matrix cores contract the rows of
// one launch, its workgroups convert the rows of the next.  The pass by itself is bound by HBM and leaves the matrix cores idle;
// the K loop leaves HBM idle, and covers two vector instructions per matrix instruction of which it uses one in two: a piece is about
// 60 of the 190 left in a slab (two where H < 3072 asks for them: 32768 rows of 2048, V = 151936, 15.85 -> 15.63 ms; 12288 of 4096
// 10.57 -> 10.70).  What it still costs is power (see plan_hosts).
// A workgroup takes a run of units of one row of units, a thread kRows pieces of 16 bytes of every slab: requested two slabs before
// they are looked at, written a slab later, all by range-checked accesses, so that what lies past the run is neither read nor
// written.  The accesses stand behind a half's operand loads: the wait in the middle of a slab leaves the youngest of them out.
template <bool kEntropy, int kRowsOf>
struct DzGuest {
  static constexpr bool kHosts = true;
  static constexpr int kRows = kRowsOf, kOps = 2 * kRows, kUnitBytes = 64 * kRowBytes;
  static_assert(kRows == 1 || kRows == 2, "rows 32 apart of a unit");
  struct Params {
    const char* z;      // of the first row of units to convert
    char* dz;
    DzTokens t;
    int64_t z_kslab, dz_kslab;
    int n0;             // its first row
    int runs, run_rows, n_units, per_run;   // runs per row of units x rows of units; units, units of a run
  };
  __amdgpu_buffer_rsrc_t rsrc_z, rsrc_dz;
  int load_at, store_at, store_next;
  int rel[kRows];                  // label - vocabulary entry of the piece that is finished
  float shift[kRows], k1[kRows], k2[kRows], top[kRows], c;
  uint32_t live[kRows];
  u32x4 raw[2][kRows], out[kRows];
  float x[kRows][8], pr[kRows][8];
  int pairs;                       // pairs of slabs that the run takes

  __device__ __forceinline__ static int pieces(const Params& p, int item) {
    const int row = item / p.runs, run = item % p.runs;
    const int left = p.n_units - run * p.per_run;
    return row < p.run_rows && left > 0 ? (left < p.per_run ? left : p.per_run) : 0;
  }
  __device__ __forceinline__ void place(const Params& p, int item) {
    constexpr int kParts = 2 / kRows;            // of a row of units
    const int n = pieces(p, item);
    pairs = (n + 2) / 2;                         // one slab more, to write the last piece in
    const int row = n > 0 ? item / p.runs : 0, run = n > 0 ? item % p.runs : 0;
    const int lane_row = (int)(threadIdx.x >> 3) + row % kParts * 32, q = threadIdx.x & 7;
    const int64_t first = (int64_t)run * p.per_run;
    rsrc_z = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.z + (row / kParts * p.z_kslab + first) * kUnitBytes), 0, n * kUnitBytes, 0x00020000);
    rsrc_dz = __builtin_amdgcn_make_buffer_rsrc(p.dz + (row / kParts * p.dz_kslab + first) * kUnitBytes, 0, n * kUnitBytes, 0x00020000);
    load_at = store_next = lane_row * kRowBytes + q * 16;
    store_at = 0x7f000000;                       // there is no piece before the first
    c = p.t.c;
#pragma unroll
    for (int h = 0; h < kRows; ++h) {
      const DzRow r = DzRow::of<kEntropy>(p.t, p.n0 + row / kParts * 64 + h * 32 + lane_row);
      rel[h] = r.label < 0 ? -0x40000000 : r.label - ((int)first - 1) * 64 - q * 8;
      shift[h] = r.shift; k1[h] = r.k1; k2[h] = r.k2; top[h] = r.top;
      live[h] = r.live ? 0xffffffffu : 0u;
      out[h] = u32x4{0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < 8; ++e) x[h][e] = pr[h][e] = 0.f;
    }
  }
  template <int par>
  __device__ __forceinline__ void request(int h) {
    raw[par][h] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_z, load_at + h * 32 * kRowBytes, 0, 0);
  }
  __device__ __forceinline__ void begin() {
    // what the rows need has arrived: not a wait in the K loop
#pragma unroll
    for (int h = 0; h < kRows; ++h)
      asm volatile("" : "+v"(shift[h]), "+v"(k1[h]), "+v"(k2[h]), "+v"(top[h]), "+v"(rel[h]), "+v"(live[h]));
#pragma unroll
    for (int h = 0; h < kRows; ++h) request<0>(h);
    load_at += kUnitBytes;
#pragma unroll
    for (int h = 0; h < kRows; ++h) request<1>(h);
    load_at += kUnitBytes;
  }
  template <int par>
  struct Turn {
    DzGuest& g;
    static constexpr int kOps = DzGuest::kOps;
    __device__ __forceinline__ static void fence() { __builtin_amdgcn_sched_barrier(0); }
    // second half of a slab: exponents and exponentials of its piece; the request two slabs ahead
    template <int m>
    __device__ __forceinline__ void second() {
      constexpr int kEvery = 2 / kRows, n = m / kEvery, h = n / 16, i = n % 16;
      // not looked at before the wait in front of this half: what does is volatile, as that is
      if constexpr (m == 0)
        for (int r = 0; r < kRows; ++r) asm volatile("" : "+v"(g.raw[par][r]));
      if constexpr (m % kEvery == 0 && n < 16 * kRows) {
        if constexpr (i < 8) g.x[h][i] = fmaf((float)reinterpret_cast<const _Float16*>(&g.raw[par][h])[i], g.c, g.shift[h]);
        else g.pr[h][i - 8] = __builtin_amdgcn_exp2f(g.x[h][i - 8]);
        fence();
      }
      if constexpr (m >= 60 && m < 60 + kRows) { g.template request<par>(m - 60); fence(); }
      if constexpr (m == 63) { g.load_at += kUnitBytes; fence(); }
    }
    // first half of the next one: its d(logits), and the store
    template <int m>
    __device__ __forceinline__ void first() {
      constexpr int kEvery = 4 / kRows, n = m / kEvery, h = n / 8, e = n % 8;
      if constexpr (n < 8 * kRows) {
        if constexpr (m % kEvery == 0) {
          if constexpr (kEntropy) g.x[h][e] = fmaf(g.x[h][e], g.k2[h], g.k1[h]);
          else g.x[h][e] = g.rel[h] == e ? g.top[h] : 0.f;
          fence();
        }
        if constexpr (m % kEvery == kEvery / 2) {
          const float k = kEntropy ? g.x[h][e] : g.k1[h];
          g.pr[h][e] = fmaf(g.pr[h][e], k, kEntropy ? (g.rel[h] == e ? g.top[h] : 0.f) : g.x[h][e]);
          fence();
        }
      }
      constexpr int w = m - 34;
      if constexpr (w >= 0 && w < 8 * kRows && w % 2 == 0) {
        constexpr int o = w / 2, hh = o / 4, k = o % 4;
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        const bf16x2 two = {(__bf16)g.pr[hh][2 * k], (__bf16)g.pr[hh][2 * k + 1]};
        g.out[hh][k] = __builtin_bit_cast(uint32_t, two) & g.live[hh];
        fence();
      }
      if constexpr (m >= 60 && m < 60 + kRows) {
        __builtin_amdgcn_raw_buffer_store_b128(g.out[m - 60], g.rsrc_dz, g.store_at + (m - 60) * 32 * kRowBytes, 0, 0);
        fence();
      }
      if constexpr (m == 63) {
        g.store_at = g.store_next;
        g.store_next += kUnitBytes;
        for (int i = 0; i < kRows; ++i) g.rel[i] -= 64;
        fence();
      }
    }
  };
  template <int par> __device__ __forceinline__ Turn<par> turn() { return Turn<par>{*this}; }
};
struct NoDz {
  static constexpr bool kHosts = false;
  struct Params {};
};

// C (+)= A B^T with A [M x K] and B [N x K], C row-major in one of two orientations; either way
// a lane's 16-byte pieces lie along C's rows and a store instruction covers runs of at least 64 bytes:
//   dW (side kLogits):  C[m][n], ld = ldc, fp32 or 16-bit, A = dz^T (dz in units), B = hidden^T (K-blocked).  A lane holds
//     4 consecutive n of a row (GemmTile with BV = 4), 16 lanes 256 contiguous bytes of each of 4 rows for fp32, 128 for
//     16-bit results.
//   dhidden (kMContig): C[n][m], ld = ldc, A = W^T (kWeight: W itself; kRows: the caller's K-blocked W^T), B = dz (in
//     units).  A lane holds VEC consecutive m of a row, the 4 lane groups 64 contiguous bytes of each of 16 rows for 16-bit results.
template <Side S> constexpr bool kMContig = S != Side::kLogits;
template <typename T, Side S, int NI = 8> using OutTile = typename TileOf<T, kMContig<S> ? NI : 4, S, kMContig<S>, NI>::type;

struct GemmParams {
  const void* A;
  const void* B;
  void* C;
  int64_t a_step, b_step;   // A: slabs per row block (kRows), row stride in elements (kWeight), units per row of units (kLogits);
                            // B: units per row of units (kMContig), slabs per row block
  int64_t ldc;
  int M, N, K;
  int k_valid;              // kWeight: rows of W; the rest of K reads as zero
  int n_mt, n_nt;
  int k_split;        // > 1: work item = (tile, K range); fp32 partial tiles go to `partial`
  int k_per_split;    // K extent of one range, a multiple of the slab
  int xcd_wgs;        // see work_item
  int n_walk;         // > 0: workgroups walk runs of tiles (see gemm_kernel); needs k_split == 1
  float* partial;     // [k_split] copies of C's shape in fp32, densely packed (row stride N or M)
  const int32_t* order;   // kMContig, optional [N]: row n of the result is row order[n] of the `total` rows of C
  int64_t total;
};

// Addresses of a 256 x 256 output tile for the accumulator layout: a range-checked buffer descriptor over
// the tile's valid rows and one per-lane byte offset per group of BV (kMContig: per block) of the lane dimension.
// Along the lane dimension (n) elements outside the tile get a per-lane offset far outside the descriptor: loads
// of them give 0 and stores are dropped.  Along the register dimension (m) nothing relies on the range check:
// kMContig skips whole 32-row groups (its M extents are multiples of 32), and in the other orientation a row past the
// tile's valid ones gets such an offset too.
template <typename T, typename OutT, Side S, int NI>
struct TileAddr {
  using Tile = OutTile<T, S, NI>;
  static constexpr bool kMContig = clgrpo::kMContig<S>;
  static constexpr int ES = (int)sizeof(OutT);
  static constexpr int kPieces = Tile::MI * 4 / Tile::VEC;  // kMContig: runs of VEC consecutive m per lane and block j
  static constexpr int kGroups = kMContig ? Tile::NI : Tile::NI / 4;
  // element k of piece n: its block and register
  static constexpr int block(int n, int k) { return Tile::kAcross ? n / 4 * Tile::VEC + k : n * (Tile::VEC / 4) + k / 4; }
  static constexpr int reg(int n, int k) { return Tile::kAcross ? n % 4 : k % 4; }
  static constexpr int piece_off(int n) { return Tile::a_off(block(n, 0), reg(n, 0)); }
  __amdgpu_buffer_rsrc_t rsrc;
  int voff[kGroups];
  int row_bytes, a_rows, row_lim;   // row_lim: valid rows from this lane's first row on
  __device__ __forceinline__ TileAddr(OutT* base, int64_t ld, int m0, int n0, int a_rows_, int b_rows,
                                      const int32_t* order = nullptr, int64_t total = 0) {
    row_bytes = (int)(ld * (int64_t)ES);
    a_rows = a_rows_;
    if constexpr (!kMContig) asm volatile("" : "+s"(row_bytes));   // its multiples are not kept in registers across the K loops
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
  // kMContig: piece n lies inside the tile (uniform over the wave)
  __device__ __forceinline__ bool piece_ok(int n) const { return Tile::wave_m() + (piece_off(n) & ~31) < a_rows; }
  // otherwise: offset of group g of the row dm rows below the lane's first
  __device__ __forceinline__ int row_voff(int dm, int g) const { return dm < row_lim ? voff[g] : 0x7f000000; }
};

// What a contraction does with the previous contents of C.  kAddsAround: the same as kAdds, loads and stores around the last-level
// cache (256 MB; the accesses' non-temporal bit), which otherwise gives up hidden^T and d(logits), read again by the workgroups of
// every column of tiles, for lines of dW that nobody reads before they are gone.  From 112 MB of dW on:
//   dW added to, us: 300 tokens at H = 4096, V = 151936 976 -> 925, 1024 1476 -> 1428, 3573 3656 -> 3586; 1200 at 1536, V = 65536 300 -> 274;
//   2000 at 2048, V = 32000 265 -> 252; 6000 at 5120, V = 102400 4478 -> 4436; below it 600 at 512, V = 50257 (103 MB) 65.2 -> 67.8,
//   500 at 1024, V = 32000 (131 MB) 70.5 -> 71.5 where dW was in the cache, 78 -> 69 where it was not.
// A dW that is only written is as fast either way.
enum Adds : int { kOverwrites, kAdds, kAddsAround };
constexpr int64_t kAddsAroundBytes = 112 << 20;
constexpr int kNonTemporal = 2;                  // of the buffer accesses' cache policy

// N consecutive elements of a row: 4 or 8 floats, or 4 or 8 (T = bf16) 16-bit values.
template <int kPolicy, int N>
__device__ __forceinline__ void row_store(const float (&x)[N], const __amdgpu_buffer_rsrc_t& rsrc, int voff, int soff, float*) {
#pragma unroll
  for (int k = 0; k < N; k += 4) {
    const f32x4 v = {x[k], x[k + 1], x[k + 2], x[k + 3]};
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rsrc, voff + k * 4, soff, kPolicy);
  }
}
template <int kPolicy>
__device__ __forceinline__ void row_store(const float (&x)[8], const __amdgpu_buffer_rsrc_t& rsrc, int voff, int soff, __bf16*) {
  __builtin_amdgcn_raw_buffer_store_b128(pack_vec(x, (__bf16*)nullptr), rsrc, voff, soff, kPolicy);
}
template <int kPolicy>
__device__ __forceinline__ void row_store(const float (&x)[4], const __amdgpu_buffer_rsrc_t& rsrc, int voff, int soff, __bf16*) {
  typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  const bf16x4 v = {(__bf16)x[0], (__bf16)x[1], (__bf16)x[2], (__bf16)x[3]};
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), rsrc, voff, soff, kPolicy);
}

// fn(values of one run of a row, per-lane offset, scalar offset), for every run of the tile that lies inside it; a
// dW row past the tile gets an offset outside the descriptor, as elements past a row do.
template <typename T, typename OutT, Side S, int NI, typename AccT, typename Fn>
__device__ __forceinline__ void for_rows(const TileAddr<T, OutT, S, NI>& at, AccT& acc, Fn fn) {
  using Tile = OutTile<T, S, NI>;
  using Addr = TileAddr<T, OutT, S, NI>;
  if constexpr (kMContig<S>) {
#pragma unroll
    for (int n = 0; n < Addr::kPieces; ++n) {
      if (!at.piece_ok(n)) continue;
#pragma unroll
      for (int j = 0; j < Tile::NI; ++j) {
        float x[Tile::VEC];
#pragma unroll
        for (int k = 0; k < Tile::VEC; ++k) x[k] = acc_get(acc[Addr::block(n, k)][j], Addr::reg(n, k));
        fn(x, at.voff[j] + Addr::piece_off(n) * (int)sizeof(OutT), 0);
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < Tile::MI; ++i)
#pragma unroll
      for (int j = 0; j < Tile::NI; j += 4)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float x[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) x[k] = acc_get(acc[i][j + k], r);
          const int dm = Tile::a_off(i, r);
          fn(x, at.row_voff(dm, j / 4), dm * at.row_bytes);
        }
  }
}

// The tile's contents into the accumulators (dW only).  The loads of kAhead block rows are in flight before the first is
// used, and they are requested before the stores of the tile before: with one wave per SIMD nothing else hides their
// latency (H = 4096 over 151936 entries, loads of half a block row at a time -> these: 256 tokens 1.24 -> 0.96 ms = 5.2 TB/s
// over reads and writes, 1024 tokens 1.76 -> 1.48, 3520 tokens 3.55 -> 3.33).  A fourth block row ahead does not fit
// the registers.
template <typename T, Side S, int NI, int kPolicy, int kAhead = 3>
struct RowLoads {
  using Tile = OutTile<T, S, NI>;
  static constexpr int kSlots = kAhead + 1;
  f32x4 x[kSlots][NI / 4][4];      // [block row][group of four blocks][register of the blocks]
  typedef TileAddr<T, float, S, NI> At;
  __device__ __forceinline__ void fetch(const At& at, int i) {
#pragma unroll
    for (int g = 0; g < NI / 4; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int dm = Tile::a_off(i, r);
        x[i % kSlots][g][r] =
            __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(at.rsrc, at.row_voff(dm, g), dm * at.row_bytes, kPolicy));
      }
    Tile::fence();
  }
  __device__ __forceinline__ void begin(const At& at) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) fetch(at, i);
  }
  template <typename AccT>
  __device__ __forceinline__ void finish(const At& at, AccT& acc) {
#pragma unroll
    for (int i = 0; i < Tile::MI; ++i) {
      if (i + kAhead < Tile::MI) fetch(at, i + kAhead);
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const auto& b = x[i % kSlots][j / 4];
        acc_set(acc[i][j], b[0][j % 4], b[1][j % 4], b[2][j % 4], b[3][j % 4]);
      }
      Tile::fence();
    }
  }
};

// Output tile from the accumulators: C = acc (the accumulators already hold C's previous contents
// when the GEMM adds to it, see gemm_init_tile), or the fp32 partial of K range `ks`.
template <typename T, typename OutT, Side S, int NI, int kPolicy>
__device__ __forceinline__ void gemm_store_tile(const GemmParams& p, typename OutTile<T, S, NI>::Acc& acc, int m0, int n0,
                                                int a_rows, int b_rows, int ks) {
  if (p.k_split > 1) {
    const TileAddr<T, float, S, NI> at(p.partial + (int64_t)ks * p.M * p.N, kMContig<S> ? p.M : p.N, m0, n0, a_rows, b_rows);
    for_rows<T, float, S, NI>(at, acc, [&](auto& x, int voff, int soff) { row_store<0>(x, at.rsrc, voff, soff, (float*)nullptr); });
    return;
  }
  const TileAddr<T, OutT, S, NI> at(static_cast<OutT*>(p.C), p.ldc, m0, n0, a_rows, b_rows, p.order, p.total);
  for_rows<T, OutT, S, NI>(at, acc, [&](auto& x, int voff, int soff) { row_store<kPolicy>(x, at.rsrc, voff, soff, (OutT*)nullptr); });
}

// Work item = (walk, fixed tile) when n_walk > 0: the workgroup keeps one operand's tile (A's m tile
// when C is [n][m], B's n tile when C is [m][n]) and walks a contiguous run of tiles of the other, so the
// K loops stream into each other (the next tile's first slabs are requested while the current tile
// finishes and is stored).  Otherwise work item = (K range, m tile, n tile), one K loop per workgroup.
// kC: whether C is added to (see Adds), where one workgroup owns the whole K range of a tile (an argument in its place had fp32 tiles
// spill 400 registers).
template <typename T, typename OutT, Side S, int NI, Adds kC, typename G>
__global__ __launch_bounds__(kHeadThreads, 1) void gemm_kernel(GemmParams p, typename G::Params guest_of) {
  using Tile = OutTile<T, S, NI>;
  constexpr bool kMC = kMContig<S>, kLoadsC = kC != kOverwrites;
  constexpr int kPolicy = kC == kAddsAround ? kNonTemporal : 0;
  constexpr int E = Tile::kSlabK;
  constexpr int64_t kSlabElems = (int64_t)kBlockRows * E;   // elements of a K-blocked block's slab, and of a 256-wide row of units
  extern __shared__ __align__(16) char lds[];

  // this workgroup's tiles: (mt, nt) first, then `count - 1` steps along the walked operand; one K range
  int item = work_item(p.xcd_wgs), mt, nt, count = 1, ks = 0, k0 = 0, k_len = p.K;
  const int whole_item = item;
  if (p.n_walk > 0) {
    const int n_fixed = kMC ? p.n_mt : p.n_nt;       // tiles of the operand that stays
    const int n_moving = kMC ? p.n_nt : p.n_mt;      // tiles of the operand that is walked
    if (item >= p.n_walk * n_fixed) return;
    int walk, ft;
    grouped_tile(item, p.n_walk, n_fixed, 4, walk, ft);
    const int begin = (int)((int64_t)walk * n_moving / p.n_walk);
    count = (int)((int64_t)(walk + 1) * n_moving / p.n_walk) - begin;
    mt = kMC ? ft : begin;
    nt = kMC ? begin : ft;
  } else {
    if (item >= p.n_mt * p.n_nt * p.k_split) return;
    ks = item / (p.n_mt * p.n_nt);
    item -= ks * (p.n_mt * p.n_nt);
    grouped_tile(item, p.n_mt, p.n_nt, 8, mt, nt);
    k0 = ks * p.k_per_split;
    k_len = (p.K - k0) < p.k_per_split ? (p.K - k0) : p.k_per_split;
  }

  const int nslab = k_len / E;
  const int64_t s0 = k0 / E;   // first slab of this K range
  const bool stream = Tile::can_stream(nslab);
  const T* A = static_cast<const T*>(p.A);
  const T* B = static_cast<const T*>(p.B);
  auto operand_a = [&](int m_tile, int rows) {
    if constexpr (S == Side::kRows) return Tile::Operand::blocked(A + ((int64_t)m_tile * p.a_step + s0) * kSlabElems, rows);
    else if constexpr (S == Side::kWeight)
      return Tile::Operand::across_weight(A + (int64_t)k0 * p.a_step + m_tile * 256, p.a_step, m_tile * 256, rows, p.k_valid - k0);
    else return Tile::Operand::across_units(A + s0 * p.a_step * (E * E) + m_tile * kSlabElems, p.a_step, rows);
  };
  auto operand_b = [&](int n_tile, int rows) {
    if constexpr (kMC) return Tile::Operand::units(B + (n_tile * (int64_t)(Tile::BN / E) * p.b_step + s0) * (E * E), p.b_step, rows);
    else return Tile::Operand::blocked(B + ((int64_t)n_tile * p.b_step + s0) * kSlabElems, rows);
  };
  auto rows_of = [](int total, int tile, int width) { const int left = total - tile * width; return left < width ? left : width; };
  // Accumulators before a tile's K loop: zeros, or - when the GEMM adds to C and one workgroup owns the whole K range of
  // the tile - the tile's current contents, which leaves the epilogue a pure store.
  static_assert(!kLoadsC || (!kMC && sizeof(OutT) == 4), "only an fp32 dW is ever added to");
  typedef RowLoads<T, S, NI, kPolicy, Tile::kSplit ? 1 : 3> Loads;
  auto c_tile = [&](int m_tile) {
    return typename Loads::At(static_cast<float*>(p.C), p.ldc, m_tile * 256, nt * Tile::BN, rows_of(p.M, m_tile, 256),
                              rows_of(p.N, nt, Tile::BN));
  };
  typename Tile::Acc acc;
  Loads loads;
  if constexpr (kLoadsC) loads.begin(c_tile(mt));
  Tile core;
  bool again = false;      // the tile before was computed twice: nothing of this one has been requested
  for (int k = 0; k < count; ++k) {
    const int m0 = mt * 256, n0 = nt * Tile::BN;
    const int a_rows = rows_of(p.M, mt, 256), b_rows = rows_of(p.N, nt, Tile::BN);
    const auto op_a = operand_a(mt, a_rows);
    const auto op_b = operand_b(nt, b_rows);
    if constexpr (kLoadsC) loads.finish(c_tile(mt), acc);
    else Tile::zero(acc);
    [[maybe_unused]] std::conditional_t<G::kHosts, G, int> guest;
    if constexpr (G::kHosts) guest.place(guest_of, whole_item);     // one tile per workgroup
    if (k == 0 || !stream || again) core.start(op_a, op_b, nslab, lds);
    if (stream && k + 1 < count)
      core.follow(op_a, op_b, nslab, Tile::cursor_a(kMC ? op_a : operand_a(mt + 1, rows_of(p.M, mt + 1, 256)), nslab),
                  Tile::cursor_b(kMC ? operand_b(nt + 1, rows_of(p.N, nt + 1, Tile::BN)) : op_b, nslab));
    else
      core.follow(op_a, op_b, nslab, Tile::hold_a(op_a, nslab), Tile::hold_b(op_b, nslab));
    if constexpr (G::kHosts) {
      guest.begin();
      core.run_with(acc, nslab, guest.pairs, guest);
    } else {
      core.run(acc, nslab);
    }
    if constexpr (Tile::kSplit) {
      again = core.redo(acc, op_a, op_b, nslab, lds, [&] {
        if constexpr (kLoadsC) {
          RowLoads<T, S, NI, kPolicy, 0> old;
          old.finish(c_tile(mt), acc);
        } else {
          Tile::zero(acc);
        }
      });
    }
    if (!stream || k + 1 == count) Tile::finish();
    if constexpr (kLoadsC) {
      if (k + 1 < count) loads.begin(c_tile(mt + 1));
    }
    gemm_store_tile<T, OutT, S, NI, kPolicy>(p, acc, m0, n0, a_rows, b_rows, ks);
    if (kMC) ++nt; else ++mt;
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
  int ni;            // the single launch's tiles are 32 * ni rows wide
};

// Time of a tile of 32 * ni rows against one of 256.  A step loads as many bytes of W and transposes as many of its fragments,
// whatever the width (launches of full rounds, H = 512 - 7168: 0.62 - 0.68 at 128 rows, 0.80 - 0.85 at 192).
static double dh_tile_time(int ni) { return ni == 4 ? 0.63 : ni == 6 ? 0.80 : 1.0; }

// Narrower row tiles (16-bit operands, a single launch): where 256-row ones would be padding or too few, as in the
// forward's fwd_plan; whole units of 64 rows, so 192 or 128.  Taken where the plan then costs 3.5 % less, the partials' traffic
// counted: 6.6 MB per slab period of a tile (see plan_dweight).
// dhidden and the d(logits) pass, us: H = 4096, V = 151936: 128 rows 267 -> 260, 320 469 -> 409, 384 478 -> 422; H = 2048: 320
// 260 -> 235; H = 1024, V = 32000: 32 rows 36 -> 28, 200 45 -> 37, 320 53 -> 49.
// Over 2398 sizes (H 512 - 7168, V 9000 - 151936, 32 - 4096 rows), each timed at all three widths: 6 % less time than 256-row tiles on
// average, 0.3 % more than the best width; 21 sizes more than 2 % slower than 256-row tiles, by at most 8.6 %.  (With the time of a
// tile as 0.54 and 0.78 and a flat 2 % for partials: 135 sizes, up to 80 %; 640 rows at H = 7168, V = 129280 in five tiles of 128
// rows 1312 us, in three of 256 1007.)
static DhPlan plan_dhidden(int64_t rows, int64_t H, int64_t K, int slab, int cus, size_t partial_cap) {
  DhPlan pl{0, 1, 0, 8};
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
  auto full_cost = [&](long items, int s, int ni) {
    const long rounds = (items * s + cus - 1) / cus;
    return dh_tile_time(ni) * (double)rounds * (double)((k_slabs + s - 1) / s) + (s > 1 ? 2.0 * (double)s * rows * H * sizeof(float) / 6.6e6 : 0.0);
  };
  best = 0.965 * full_cost(tiles, s_one, 8);
  for (int ni = 6; slab == 64 && ni >= 4; ni -= 2) {
    const int t = n_mt * (int)((rows + 32 * ni - 1) / (32 * ni));
    const int s = pick_k_split(t, (int)H, (int)rows, (int)K, slab, partial_cap, cus);
    const double c = full_cost(t, s, ni);
    if (c < best) { best = c; pl.ni = ni; pl.k_split = s; }
  }
  pl.partial_bytes = pl.k_split > 1 ? (size_t)pl.k_split * rows * H * sizeof(float) : 0;
  return pl;
}

// Bytes of fp32 split-K partials the dhidden GEMM of `rows` tokens wants (planned for a 256-CU device, so
// that the workspace size does not depend on the device in use; a launch takes fewer ranges if they do not fit).
static size_t dhidden_partial_bytes(int64_t rows, int64_t H, int64_t ldv, int slab) {
  return plan_dhidden(rows, H, ldv, slab, 256, (size_t)1 << 30).partial_bytes;
}

// How the dW GEMM (C[m][n], M = vocabulary rows, N = H, K = the chunk's tokens) is launched.  With many more tiles
// than CUs its workgroups keep one tile of hidden^T and walk runs of vocabulary tiles (see gemm_kernel); the walks
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

struct BwdPlan {
  int64_t ldv;        // vocabulary extent of dz (V rounded up to 64)
  int64_t chunk;      // tokens per chunk (multiple of 256 unless >= T)
  int64_t ldt;        // token extent of hidT for a full chunk (tokens rounded up to 64)
  size_t off_hidt, off_dz, off_part, part_bytes, total;
};

static BwdPlan bwd_plan(int64_t T, int64_t H, int64_t V, size_t es, int64_t chunk_tokens, bool saved = false,
                        bool own_dw = true) {
  BwdPlan pl;
  pl.ldv = round_up64(V, 64);
  int64_t chunk = (chunk_tokens <= 0 || chunk_tokens >= T) ? T : round_up64(chunk_tokens, 256);
  if (chunk > T) chunk = T;
  pl.chunk = chunk;
  pl.ldt = round_up64(chunk, 64);
  size_t off = 0;
  const size_t Hb = (size_t)round_up64(H, 256);                 // K-blocked: whole blocks of 256 rows
  pl.off_hidt = off; off += own_dw ? align_up(Hb * pl.ldt * es, 256) : 0;
  pl.off_dz = off;   off += saved ? 0 : align_up((size_t)pl.ldt * pl.ldv * es, 256);
  // split-K partials of the dhidden GEMM and of the dW GEMM's tail (used one after the other): what a full chunk and
  // the shorter last chunk want
  const int slab = (int)(kRowBytes / es);
  size_t part = 0;
  for (size_t b : {dhidden_partial_bytes(chunk, H, pl.ldv, slab), dhidden_partial_bytes(T % chunk, H, pl.ldv, slab),
                   own_dw ? dweight_partial_bytes(chunk, H, V, slab) : 0, own_dw ? dweight_partial_bytes(T % chunk, H, V, slab) : 0})
    if (b > part) part = b;
  pl.part_bytes = align_up(part, 256);
  pl.off_part = off; off += pl.part_bytes;
  pl.total = off;
  return pl;
}

// Largest chunk (multiple of 256, or T itself) whose plan fits into `bytes`; 0 if none does.
static int64_t chunk_for_workspace(int64_t T, int64_t H, int64_t V, size_t es, size_t bytes, bool saved, bool own_dw) {
  if (bwd_plan(T, H, V, es, T, saved, own_dw).total <= bytes) return T;
  int64_t lo = 0, hi = T / 256;   // in units of 256 tokens
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) / 2;
    if (bwd_plan(T, H, V, es, mid * 256, saved, own_dw).total <= bytes) lo = mid; else hi = mid - 1;
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

// Operands of a contraction as GemmParams names them.
struct GemmIn {
  const void *A, *B;
  int64_t a_step, b_step;
  int k_valid;
};

template <typename T, typename OutT, Side S, int NI = 8, typename G = NoDz>
static int launch_gemm_one(const GemmIn& in, int M, int N, int K, void* C, int64_t ldc, int accumulate, hipStream_t stream,
                           float* partial, size_t partial_bytes, int k_split_wanted, const RowOrder& rows = RowOrder{nullptr, 0},
                           const typename G::Params& guest = typename G::Params{}) {
  using Tile = OutTile<T, S, NI>;
  constexpr bool kMC = kMContig<S>;
  GemmParams g;
  g.A = in.A; g.B = in.B; g.C = C; g.a_step = in.a_step; g.b_step = in.b_step; g.ldc = ldc; g.k_valid = in.k_valid;
  g.M = M; g.N = N; g.K = K;
  g.n_mt = (M + 255) / 256; g.n_nt = (N + Tile::BN - 1) / Tile::BN;
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
  const int n_fixed = kMC ? g.n_mt : g.n_nt, n_moving = kMC ? g.n_nt : g.n_mt;
  g.n_walk = 0;
  if (!G::kHosts && g.k_split == 1 && n_fixed <= cus && g.n_mt * g.n_nt >= 4 * cus && K >= 2 * slab) {
    g.n_walk = cus / n_fixed;
    if (g.n_walk > n_moving) g.n_walk = n_moving;
    // A walk is as long as its longest run; one workgroup per tile takes ceil(tiles / CUs) rounds.  Streaming the K
    // loops into each other is worth a few per cent, not a whole extra tile period (H = 7168: 28 x 64 tiles are 7
    // rounds exactly, while 9 walks over 64 tiles make runs of 7 and 8).
    const long walk_periods = (n_moving + g.n_walk - 1) / g.n_walk;
    const long plain_rounds = ((long)g.n_mt * g.n_nt + cus - 1) / cus;
    if (walk_periods * 100 > plain_rounds * 104) g.n_walk = 0;
  }
  // One workgroup per tile in several rounds: each round's tiles go to all XCDs, so that they stream the same stretches of
  // the operands (dhidden of 32768 rows at H = 7168, 14 rounds: 42.4 -> 41.5 ms, of 16384 20.9 -> 20.4; dW of 8192 rows at H =
  // 5120 9.11 -> 8.56; two and three rounds at H = 4096: no change).  dW of some hundred rows writes more than it reads, and eight
  // XCDs writing one stretch of dW at a time are slower than each its own (V = 151936, plain -> rounds, us: H = 5120 412 rows
  // 925 -> 1010, 1024 1432 -> 1534, 2048 2382 -> 2380, 4096 4569 -> 4397; H = 1536 768 rows 458 -> 472, 4096 1676 -> 1634); up to 128
  // rows it is the reads of hidden^T and dz that count again (H = 4096, 64 rows 479 -> 457).  fp32 tiles take ten times as long
  // for the same bytes: no gain from it, up to 4 % lost (dW of 64 rows at H = 1536 356 -> 371).
  const bool rounds = g.k_split == 1 && sizeof(T) == 2 && (kMC || K >= 2048 || K <= 128);
  ItemGrid grid{(g.n_walk * n_fixed + 7) / 8 * 8, 0};
  if (g.n_walk == 0) grid = rounds ? item_grid(g.n_mt * g.n_nt, cus) : ItemGrid{(g.n_mt * g.n_nt * g.k_split + 7) / 8 * 8, 0};
  g.xcd_wgs = grid.xcd_wgs;
  auto launch = [&](auto kernel) {
    const int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), Tile::kLdsBytes, "gemm_kernel");
    if (rc) return rc;
    hipLaunchKernelGGL(kernel, dim3(grid.grid), dim3(Tile::kThreads), Tile::kLdsBytes, stream, g, guest);
    return check_launch("gemm_kernel");
  };
  int rc;
  if constexpr (!kMC && sizeof(OutT) == 4)
    rc = !accumulate || g.k_split > 1                                ? launch(&gemm_kernel<T, OutT, S, NI, kOverwrites, NoDz>)
         : (int64_t)M * N * (int64_t)sizeof(OutT) > kAddsAroundBytes ? launch(&gemm_kernel<T, OutT, S, NI, kAddsAround, NoDz>)
                                                                     : launch(&gemm_kernel<T, OutT, S, NI, kAdds, NoDz>);
  else
    rc = launch(&gemm_kernel<T, OutT, S, NI, kOverwrites, G>);
  if (rc || g.k_split == 1) return rc;
  return launch_splitk_reduce<OutT>(partial, g.k_split, kMC ? N : M, kMC ? M : N, static_cast<OutT*>(C), ldc, accumulate,
                                    rows.order, stream);
}

// dhidden[n][m] = sum over K of A(m, k) dz(n, k) under plan_dhidden, with what `partial` has room for (nothing, where neither
// contraction of the chunk is planned with partial sums: the row tiles are the plan's all the same.  256-row tiles in that case:
// with the d(logits) pass, 1600 rows at H = 7168, V = 129280 2550 us for 2372, 3400 rows at H = 3584, V = 151936 3250 for 2960).
template <typename T, Side S>
static int launch_dhidden(const GemmIn& in, int M, int N, int K, void* C, int64_t ldc, hipStream_t stream, float* partial,
                          size_t partial_bytes, const RowOrder& rows) {
  constexpr int E = Elem<T>::kSlabK;
  const DhPlan pl = plan_dhidden(N, M, K, E, device_cu_count(), partial_bytes);
  if constexpr (sizeof(T) == 2) {
    if (pl.ni == 6) return launch_gemm_one<T, T, S, 6>(in, M, N, K, C, ldc, 0, stream, partial, partial_bytes, pl.k_split, rows);
    if (pl.ni == 4) return launch_gemm_one<T, T, S, 4>(in, M, N, K, C, ldc, 0, stream, partial, partial_bytes, pl.k_split, rows);
  }
  if (pl.bulk_nt == 0) return launch_gemm_one<T, T, S>(in, M, N, K, C, ldc, 0, stream, partial, partial_bytes, pl.k_split, rows);
  const int bulk_rows = pl.bulk_nt * 256;
  int rc = launch_gemm_one<T, T, S>(in, M, bulk_rows, K, C, ldc, 0, stream, nullptr, 0, 1, rows);
  if (rc) return rc;
  GemmIn tail = in;
  tail.B = static_cast<const T*>(in.B) + (int64_t)bulk_rows / E * in.b_step * (E * E);
  T* c_tail = static_cast<T*>(C) + (rows.order ? 0 : (int64_t)bulk_rows * ldc);
  const RowOrder tail_rows{rows.order ? rows.order + bulk_rows : nullptr, rows.total};
  return launch_gemm_one<T, T, S>(tail, M, N - bulk_rows, K, c_tail, ldc, 0, stream, partial, partial_bytes, pl.k_split, tail_rows);
}

// dW[m][n] (+)= sum over K of dz(k, m) hidT(n, k): equally long walks over most vocabulary tiles, the rest cut into K
// ranges (plan_dweight).
template <typename T, typename OutT>
static int launch_dweight(const GemmIn& in, int M, int N, int K, void* C, int64_t ldc, int accumulate, hipStream_t stream,
                          float* partial, size_t partial_bytes) {
  constexpr int E = Elem<T>::kSlabK;
  const DwPlan dw = plan_dweight(M, N, K, E, device_cu_count(), partial ? partial_bytes : 0);
  if (dw.bulk_mt == 0) return launch_gemm_one<T, OutT, Side::kLogits>(in, M, N, K, C, ldc, accumulate, stream, nullptr, 0, 1);
  const int bulk_rows = dw.bulk_mt * 256;
  int rc = launch_gemm_one<T, OutT, Side::kLogits>(in, bulk_rows, N, K, C, ldc, accumulate, stream, nullptr, 0, 1);
  if (rc) return rc;
  GemmIn tail = in;
  tail.A = static_cast<const T*>(in.A) + (int64_t)bulk_rows * E;
  OutT* c_tail = static_cast<OutT*>(C) + (int64_t)bulk_rows * ldc;
  return launch_gemm_one<T, OutT, Side::kLogits>(tail, M - bulk_rows, N, K, c_tail, ldc, accumulate, stream,
                                                 dw.k_split > 1 ? partial : nullptr, dw.k_split > 1 ? partial_bytes : 0, dw.k_split);
}

template <typename T>
static int launch_transpose(const TransposeParams<T>& p, hipStream_t stream) {
  dim3 grid((p.C + 63) / 64, (int)((p.r_dst + 63) / 64));
  hipLaunchKernelGGL(transpose_block_kernel<T>, grid, dim3(256), 0, stream, p);
  return check_launch("transpose_block_kernel");
}

// d(logits): the first `whole` units of `row_units` rows of units from row0 on, the others of the first n_edge rows; with `turn` hidden^T.
template <typename T>
static int launch_dz(DzFromZParams<T>& q, int row0, int row_units, int whole, int n_edge, bool turn, hipStream_t stream) {
  q.whole = whole;
  q.row0 = row0;
  q.row_units = row_units;
  q.n_edge = n_edge;
  // a workgroup walks units of one row of units, so that its coefficients are fetched once; 16 workgroups per CU
  int64_t per_row = row_units > 0 ? (16 * (int64_t)device_cu_count() + row_units - 1) / row_units : 0;
  if (per_row > whole) per_row = whole;
  q.n_step = (int)per_row;
  q.turn_rows = (int)((q.turn.r_dst + 63) / 64);
  const int64_t grid = (int64_t)row_units * per_row + n_edge + (turn ? (int64_t)q.turn_rows * ((q.turn.C + 63) / 64) : 0);
  if (grid == 0) return CLGRPO_OK;
  if (q.t.g_ent) hipLaunchKernelGGL((dz_from_z_kernel<T, true>), dim3((unsigned)grid), dim3(256), 0, stream, q);
  else hipLaunchKernelGGL((dz_from_z_kernel<T, false>), dim3((unsigned)grid), dim3(256), 0, stream, q);
  return check_launch("dz_from_z_kernel");
}

// Row tiles (of 256) of the launches in which dhidden's workgroups convert the next launch's d(logits): as many as fill one round
// of the CUs, the first launch what is left over (K ranges fill it).  0: dhidden and the conversion apart.
struct HostPlan {
  int first_nt, first_split, per_nt;
};
// Taken where it is the cheaper one, in periods of a tile's slab: rounds x slabs of the launches, 6.6 MB of a partial sum's traffic or
// 7.15 MB of the conversion's (5 TB/s) per period, of what guests convert the 0.35 that it still costs (12288 rows at H = 4096 in
// three launches: 1.0 ms less to convert in front of them, 0.66 ms gained).  What it loses is a round that whole row tiles do not fill
// (12836 rows at H = 2560, V = 32000: 510 tiles are two rounds of 256, not of 250), or a first launch without room for K ranges.
//   dhidden and d(logits), apart -> hosted, ms: H = 4096, V = 151936: 12288 rows 11.23 -> 10.57, 13397 12.45 -> 11.63; H = 2048: 10139
//   5.35 -> 4.97, 32768 16.9 -> 15.6; H = 7168, V = 129280: 32768 43.3 -> 41.1; H = 2560, V = 32000: 18657 2.74 -> 2.42
static HostPlan plan_hosts(int64_t rows, int64_t H, int64_t V, int cus, size_t partial_cap) {
  HostPlan hp{0, 1, 0};
  const int n_mt = (int)((H + 255) / 256), n_nt = (int)((rows + 255) / 256), per = cus / n_mt;
  if (per < 1 || n_nt <= per || V > (1 << 22)) return hp;     // a guest's run of units is within 32-bit offsets
  const int64_t K = round_up64(V, 64);
  const long slabs = (long)(K / 64);
  auto launch = [&](long tiles, int split, int64_t launch_rows) {
    const double partial = split > 1 ? 2.0 * split * (double)launch_rows * H * sizeof(float) / 6.6e6 : 0.0;
    return (double)((tiles * split + cus - 1) / cus) * (double)((slabs + split - 1) / split) + partial;
  };
  const double convert = 4.0 * (double)K / 7.15e6;      // per row
  const DhPlan dh = plan_dhidden(rows, H, K, 64, cus, partial_cap);
  double apart = rows * convert;
  if (dh.bulk_nt > 0) {
    const int64_t tail = rows - (int64_t)dh.bulk_nt * 256;
    apart += launch((long)dh.bulk_nt * n_mt, 1, 0) + launch((long)(n_nt - dh.bulk_nt) * n_mt, dh.k_split, tail);
  } else {
    apart += dh_tile_time(dh.ni) * launch((long)n_mt * ((rows + 32 * dh.ni - 1) / (32 * dh.ni)), dh.k_split, rows);
  }
  const int first = n_nt % per ? n_nt % per : per;
  const int split = pick_k_split(first * n_mt, (int)H, first * 256, (int)K, 64, partial_cap, cus);
  const double hosted = launch((long)first * n_mt, split, first * 256) + (double)((n_nt - first) / per) * slabs +
                        convert * (first * 256 + 0.35 * (rows - first * 256));
  if (hosted < 0.99 * apart) hp = HostPlan{first, split, per};
  return hp;
}

// d(logits) and dhidden of a chunk by plan_hosts, with G for a guest; with `turn` hidden^T as well.
template <typename T, typename G>
static int launch_hosted(const HostPlan& hp, DzFromZParams<T>& q, int n_rows, bool turn, const T* weight, int64_t H, T* out,
                         float* partial, size_t partial_bytes, const RowOrder& rows, hipStream_t stream) {
  constexpr int E = Elem<T>::kSlabK, kTileUnits = 256 / E, kParts = 2 / G::kRows;
  const int n_mt = (int)((H + 255) / 256), n_nt = (q.t.Tc + 255) / 256, slabs = q.n_units;
  const int whole = q.t.V / E;                          // units of a row that guests convert: the last one may end inside the vocabulary
  auto units_of = [&](int nt) { return nt * kTileUnits < n_rows ? nt * kTileUnits : n_rows; };    // rows of units of the first nt tiles
  int done = units_of(hp.first_nt);                     // of them are converted
  int rc = launch_dz(q, 0, done, whole, whole < q.n_units ? n_rows : 0, turn, stream);
  for (int nt = 0, width = hp.first_nt; rc == CLGRPO_OK && nt < n_nt; nt += width, width = hp.per_nt) {
    const int split = nt == 0 ? hp.first_split : 1;
    const int upto = units_of(nt + width + hp.per_nt);
    // Guests: as many of the next launch's rows as the workgroups have slabs for, all but one pair of theirs (see run_with).  The
    // last K range, if it is much the shortest, goes without.
    typename G::Params g{};
    const int per = (slabs + split - 1) / split, last = slabs - (split - 1) * per;
    const bool use_last = last * 10 >= per * 9;
    const int items = width * n_mt * (use_last ? split : split - 1), most = ((use_last ? last : per) - 1) / 2 * 2 - 1;
    int left = upto - done;
    if (left > 0 && most > 0 && last >= 3) {
      const int fit = items / (kParts * ((whole + most - 1) / most)), take = left < fit ? left : fit;
      if (take > 0) {
        const int row0 = upto - take;
        g.runs = items / (kParts * take);
        g.per_run = (whole + g.runs - 1) / g.runs;
        g.run_rows = kParts * take;
        g.n_units = whole;
        g.t = q.t;
        g.n0 = row0 * E;
        g.z_kslab = q.z_kslab;
        g.dz_kslab = q.dz_kslab;
        g.z = static_cast<const char*>(q.z) + (int64_t)row0 * q.z_kslab * G::kUnitBytes;
        g.dz = static_cast<char*>(q.dz) + (int64_t)row0 * q.dz_kslab * G::kUnitBytes;
        left -= take;
      }
    }
    const int r0 = nt * 256, r1 = (nt + width) * 256 < q.t.Tc ? (nt + width) * 256 : q.t.Tc;
    const GemmIn in{weight, static_cast<const T*>(q.dz) + (int64_t)r0 / E * q.dz_kslab * (E * E), H, q.dz_kslab, q.t.V};
    T* c = out + (rows.order ? 0 : (int64_t)r0 * H);
    float* part = split > 1 ? partial : nullptr;
    const size_t part_bytes = split > 1 ? partial_bytes : 0;
    const RowOrder c_rows{rows.order ? rows.order + r0 : nullptr, rows.total};
    rc = g.run_rows > 0
             ? launch_gemm_one<T, T, Side::kWeight, 8, G>(in, (int)H, r1 - r0, slabs * E, c, H, 0, stream, part, part_bytes, split, c_rows, g)
             : launch_gemm_one<T, T, Side::kWeight>(in, (int)H, r1 - r0, slabs * E, c, H, 0, stream, part, part_bytes, split, c_rows);
    if (rc == CLGRPO_OK && left > 0) rc = launch_dz(q, done, left, whole, 0, false, stream);
    done = upto;
  }
  return rc;
}

// dW[v][h] (+)= sum_t dz(t, v) hidT(h, t) over k tokens of dz (n_kslab units per row of units) and hidT (ld tokens).
template <typename T>
static int run_dweight(const T* dz, int64_t n_kslab, const T* hidt, int64_t ld, int64_t k, int64_t V, int64_t H, void* dweight,
                       bool to_bf16, bool accumulate, void* partial, size_t partial_bytes, hipStream_t stream) {
  const GemmIn in{dz, hidt, n_kslab, ld / Elem<T>::kSlabK, 0};
  float* part = static_cast<float*>(partial);
  if constexpr (sizeof(T) == 2) {
    if (to_bf16) return launch_dweight<T, __bf16>(in, (int)V, (int)H, (int)k, dweight, H, 0, stream, part, partial_bytes);
  }
  return launch_dweight<T, float>(in, (int)V, (int)H, (int)k, dweight, H, accumulate ? 1 : 0, stream, part, partial_bytes);
}

template <typename T>
static int run_bwd(const clgrpo_lmhead_bwd_args* a, hipStream_t stream, int64_t label_offset, const RowOrder& rows,
                   const DwOperands* kept) {
  using Tile = LogitTile<T>;
  const int64_t T_ = a->T, H = a->H, V = a->V;
  const bool saved = a->saved_logits != nullptr;
  const bool own_dw = kept == nullptr;
  const int64_t chunk = chunk_for_workspace(T_, H, V, sizeof(T), a->workspace_bytes, saved, own_dw);
  if (chunk <= 0)
    return fail(CLGRPO_EWORKSPACE, "clgrpo_lmhead_bwd: workspace %zu bytes cannot hold a 256-token chunk (%zu needed)",
                a->workspace_bytes, bwd_plan(T_, H, V, sizeof(T), 256, saved, own_dw).total);
  if (a->dweight_bf16 && chunk < T_)
    return fail(CLGRPO_EWORKSPACE, "clgrpo_lmhead_bwd: a 16-bit dweight needs a workspace for all %lld tokens at once", (long long)T_);
  const BwdPlan pl = bwd_plan(T_, H, V, sizeof(T), chunk, saved, own_dw);
  const int64_t ldz = saved ? a->ld_saved : pl.ldv;
  char* ws = static_cast<char*>(a->workspace);
  T* wt = static_cast<T*>(a->weight_t);
  T* dz_ws = reinterpret_cast<T*>(ws + pl.off_dz);
  const T* hidden = static_cast<const T*>(a->hidden);
  const T* weight = static_cast<const T*>(a->weight);

  int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(&lmhead_dz_kernel<T>), Tile::kLdsBytes, "lmhead_dz_kernel");
  if (rc) return rc;
  if (a->dhidden && wt && !a->weight_t_ready) {
    // the caller keeps W^T: WT(h, v) = W[v][h], zero for V <= v < ldv, K-blocked
    rc = launch_transpose(TransposeParams<T>{weight, wt, H, pl.ldv, pl.ldv, (int)V, (int)H, nullptr}, stream);
    if (rc) return rc;
  }
  for (int64_t c0 = 0; c0 < T_; c0 += chunk) {
    const int64_t tc = (T_ - c0) < chunk ? (T_ - c0) : chunk;
    const int64_t ldt = round_up64(tc, 64);
    // d(logits): in place of the kept logits, in the workspace, or in its place among the operands of dW that the caller
    // contracts later
    constexpr int E = Tile::kSlabK;
    constexpr int64_t kSlabElems = (int64_t)kBlockRows * E;
    const int64_t k0 = kept ? kept->k + c0 : 0, ld_dw = kept ? kept->ld : ldt;
    T* hidt = (kept ? static_cast<T*>(kept->hidt) : reinterpret_cast<T*>(ws + pl.off_hidt)) + k0 / E * kSlabElems;
    T* z = saved ? static_cast<T*>(a->saved_logits) + c0 * ldz : nullptr;
    T* dz = kept ? static_cast<T*>(kept->dzt) + k0 * pl.ldv : (saved ? z : dz_ws);
    const int64_t dz_kslab = (kept ? pl.ldv : ldz) / E;
    // with an order the chunk's tokens are looked up from the start of the arrays, without they follow one another
    const int64_t t0 = rows.order ? 0 : c0;
    const int32_t* order = rows.order ? rows.order + c0 : nullptr;
    // hidT(h, t) = hidden[c0 + t][h], zero for tc <= t < ldt, K-blocked
    const bool want_dw = a->dweight || kept;
    const TransposeParams<T> turn{hidden + t0 * H, hidt, H, ld_dw, ldt, (int)tc, (int)H, order};
    DzFromZParams<T> q;
    bool dhidden_done = false;
    if (saved) {
      q.z = z;
      q.dz = dz;
      q.t.labels = a->labels + t0;
      q.t.label_offset = label_offset;
      q.t.lse = a->lse + t0;
      q.t.entropy = a->g_entropy ? a->entropy + t0 : nullptr;
      q.t.g_lp = a->g_logprob + t0;
      q.t.g_ent = a->g_entropy ? a->g_entropy + t0 : nullptr;
      q.t.order = order;
      q.t.Tc = (int)tc;
      q.t.V = (int)V;
      q.t.c = a->inv_temperature * kLog2e;
      q.t.inv_temperature = a->inv_temperature;
      q.z_kslab = ldz / E;
      q.dz_kslab = dz_kslab;
      q.n_units = (int)(pl.ldv / E);
      q.turn = turn;
      if constexpr (sizeof(T) == 2) {
        if (a->dhidden && !wt) {
          // a launch's d(logits) while the one before it is contracted
          const HostPlan hp = plan_hosts(tc, H, V, device_cu_count(), pl.part_bytes);
          if (hp.first_nt > 0) {
            auto hosted = [&](auto guest) {
              return launch_hosted<T, decltype(guest)>(hp, q, (int)(ldt / E), want_dw, weight, H, static_cast<T*>(a->dhidden) + t0 * H,
                                                       reinterpret_cast<float*>(ws + pl.off_part), pl.part_bytes,
                                                       RowOrder{order, rows.total}, stream);
            };
            // a guest's two pieces per slab, where one would take more slabs than there are (the rows of a launch have 2048 / H of them)
            rc = q.t.g_ent ? hosted(DzGuest<true, 1>{}) : H < 3072 ? hosted(DzGuest<false, 2>{}) : hosted(DzGuest<false, 1>{});
            if (rc) return rc;
            dhidden_done = true;
          }
        }
      }
      if (!dhidden_done) {
        rc = launch_dz(q, 0, (int)(ldt / E), q.n_units, 0, want_dw, stream);
        if (rc) return rc;
      }
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
      int grid = (d.n_tb * d.n_vt + 7) / 8 * 8;
      hipLaunchKernelGGL(lmhead_dz_kernel<T>, dim3(grid), dim3(Tile::kThreads), Tile::kLdsBytes, stream, d);
      rc = check_launch("lmhead_dz_kernel");
      if (rc == 0 && want_dw) rc = launch_transpose(turn, stream);
      if (rc) return rc;
    }
    if (a->dhidden && !dhidden_done) {
      // dhidden[chunk][h] = sum_v W[v][h] dz[t][v]   (M = H, N = tokens, C[n][m])
      void* out = static_cast<T*>(a->dhidden) + t0 * H;
      float* part = reinterpret_cast<float*>(ws + pl.off_part);
      const RowOrder out_rows{order, rows.total};
      rc = wt ? launch_dhidden<T, Side::kRows>(GemmIn{wt, dz, pl.ldv / E, dz_kslab, 0}, (int)H, (int)tc, (int)pl.ldv, out, H,
                                               stream, part, pl.part_bytes, out_rows)
              : launch_dhidden<T, Side::kWeight>(GemmIn{weight, dz, H, dz_kslab, (int)V}, (int)H, (int)tc, (int)pl.ldv, out, H,
                                                 stream, part, pl.part_bytes, out_rows);
      if (rc) return rc;
    }
    if (a->dweight && !kept) {
      rc = run_dweight<T>(dz, dz_kslab, hidt, ldt, ldt, V, H, a->dweight, a->dweight_bf16 != 0, a->accumulate_dweight || c0 > 0,
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
  return bwd_plan(T, H, V, dtype_bytes(dtype), chunk_tokens, (with_saved_logits & 1) != 0, (with_saved_logits & 4) == 0).total;
}

extern "C" int clgrpo_lmhead_bwd_dhidden_plan(int64_t rows, int64_t H, int64_t V, int32_t dtype, int32_t cus, int32_t* out) {
  if (rows <= 0 || H <= 0 || V <= 0 || out == nullptr || (dtype != CLGRPO_BF16 && dtype != CLGRPO_F32)) return CLGRPO_EINVAL;
  const int slab = (int)(kRowBytes / dtype_bytes(dtype));
  const DhPlan pl = plan_dhidden(rows, H, round_up64(V, 64), slab, cus > 0 ? cus : 256, (size_t)1 << 30);
  out[0] = pl.bulk_nt;
  out[1] = pl.k_split;
  return CLGRPO_OK;
}

extern "C" int clgrpo_lmhead_bwd_dhidden_tile_plan(int64_t rows, int64_t H, int64_t V, int32_t dtype, int32_t cus,
                                                   int64_t partial_bytes, int32_t* out) {
  if (rows <= 0 || H <= 0 || V <= 0 || out == nullptr || (dtype != CLGRPO_BF16 && dtype != CLGRPO_F32)) return CLGRPO_EINVAL;
  const DhPlan pl = plan_dhidden(rows, H, round_up64(V, 64), (int)(kRowBytes / dtype_bytes(dtype)), cus > 0 ? cus : 256,
                                 partial_bytes < 0 ? (size_t)1 << 30 : (size_t)partial_bytes);
  out[0] = pl.bulk_nt;
  out[1] = pl.k_split;
  out[2] = 32 * pl.ni;
  out[3] = (int32_t)(1000.0 * dh_tile_time(pl.ni) + 0.5);
  return CLGRPO_OK;
}

extern "C" int clgrpo_lmhead_bwd_guest_plan(int64_t rows, int64_t H, int64_t V, int32_t cus, int64_t partial_bytes, int32_t* out) {
  if (rows <= 0 || H <= 0 || V <= 0 || out == nullptr) return CLGRPO_EINVAL;
  const HostPlan hp = plan_hosts(rows, H, V, cus > 0 ? cus : 256, partial_bytes < 0 ? (size_t)1 << 30 : (size_t)partial_bytes);
  out[0] = hp.first_nt;
  out[1] = hp.first_split;
  out[2] = hp.per_nt;
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
    return run_dweight<__bf16>(static_cast<const __bf16*>(a->dzt), round_up64(a->V, 64) / Elem<__bf16>::kSlabK,
                               static_cast<const __bf16*>(a->hidt), a->ld, a->k, a->V, a->H, a->dweight, a->dweight_bf16 != 0, a->accumulate != 0, a->workspace, a->workspace_bytes, s);
  return run_dweight<float>(static_cast<const float*>(a->dzt), round_up64(a->V, 64) / Elem<float>::kSlabK,
                            static_cast<const float*>(a->hidt), a->ld, a->k, a->V, a->H, a->dweight, false, a->accumulate != 0, a->workspace, a->workspace_bytes, s);
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
