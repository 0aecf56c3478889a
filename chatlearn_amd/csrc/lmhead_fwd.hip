// Fused lm_head projection + online log-softmax statistics (forward).
//
// z^T tile [256 vocab x block of tokens] = W tile * hidden tile^T on the matrix cores;
// the vocabulary runs along the accumulator registers, the tokens along the
// lanes, so each lane keeps a running (max, sum e^{z-max}, sum e^{z-max} z,
// target logit) for its own tokens across all vocabulary tiles of its split.
// A workgroup owns one block of 256 tokens (or fewer, see fwd_plan) and one contiguous range of
// vocabulary tiles ("split"); a second small kernel merges the splits with an
// exact rescale and writes logprob / entropy / rowmax / lse.  Logits go to
// memory only when the caller asks for a chunk's raw logits to be kept for the
// backward; they then leave straight from the accumulators, 16 bytes per lane,
// in the layout of the backward's operand (see KeptLogit).
//
// Algorithmic work: 2*T*H*V flop; bytes 2*T*H + 2*V*H (bf16) + 16*T.
#include "head_internal.hpp"
#include "gemm_core.hpp"

namespace clgrpo {

constexpr int kFwdBM = 256, kFwdBN = 256;   // kFwdBN: the widest token block, see fwd_plan
constexpr float kLog2e = 1.4426950408889634f;
// Most vocabulary splits a forward launch of n_tb token blocks uses: 4096 workgroups in all, 64 splits at least
// (the partial records of up to 16384 tokens then stay below 17 MB).  A few token blocks need many splits to reach all
// CUs: with 64 at most, one block of a 152k vocabulary ran on 60 of 256 CUs, three blocks on 180.
inline int max_fwd_splits(int64_t n_tb) { return n_tb >= 64 ? 64 : (int)(4096 / n_tb); }
constexpr float kNoLogit = -3.0e38f;   // stands for a vocabulary row past V: finite, so that 0 * kNoLogit is 0

struct FwdParams {
  const void* hidden;
  const void* weight;
  const int64_t* labels;
  int64_t label_offset;  // first vocabulary id of `weight` (0 unless this is a vocabulary shard)
  int T, H, V;
  int n_tb, n_split, tiles_per_split, n_vt;
  float c;  // inv_temperature * log2(e)
  void* z_out;   // optional raw logits in units (see unit_index): rows x ldz entries of KeptLogit<T>
  int64_t ldz;
  const int32_t* z_row_map;  // optional [T]: destination row per token, < 0: not stored
  int z_rows;                // rows of z_out; mapped rows outside [0, z_rows) are not stored
  float4* part;  // [n_split][T]: (max raw, sum 2^{(z-max) c}, sum 2^{(z-max) c} z raw, target raw)
  int xcd_wgs;   // > 0: launch of several rounds, see xcd_round_remap
  const int32_t* order;   // optional [T]: row n is token order[n] of `total` (see RowOrder); kept logits go by n
  int total;
};

// 16 bytes of kept logits: consecutive vocabulary entries of one token.
__device__ __forceinline__ u32x4 pack_kept(const float (&v)[4], float*) {
  const f32x4 x = {v[0], v[1], v[2], v[3]};
  return __builtin_bit_cast(u32x4, x);
}
__device__ __forceinline__ u32x4 pack_kept(const float (&v)[8], _Float16*) {
  typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
  f16x8 x;
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (_Float16)v[e];     // round to nearest even
  return __builtin_bit_cast(u32x4, x);
}

__device__ __forceinline__ void merge_state(float& m, float& s, float& u, float om, float os,
                                            float ou, float c) {
  const float nm = fmaxf(m, om);
  const float a = (m == nm) ? 1.f : exp2f((m - nm) * c);
  const float b = (om == nm) ? 1.f : exp2f((om - nm) * c);
  s = s * a + os * b;
  u = u * a + ou * b;
  m = nm;
}

template <typename T, bool STORE_Z, int kNI>
__global__ __launch_bounds__(kHeadThreads, 1) void lmhead_fwd_kernel(FwdParams p) {
  using Tile = LogitTile<T, kNI>;
  constexpr int MI = Tile::MI, NI = Tile::NI, VEC = Tile::VEC;
  extern __shared__ __align__(16) char lds[];

  const int item = work_item(p.xcd_wgs);
  if (item >= p.n_tb * p.n_split) return;
  int vs, tb;
  grouped_tile(item, p.n_split, p.n_tb, 4, vs, tb);
  if (STORE_Z && sizeof(typename KeptLogit<T>::type) == 2) {
    // Kept logits are IEEE half: a raw logit beyond the half range must stay finite (the largest half),
    // or the softmax the backward rebuilds from it would be inf/NaN.  The wave's FP16_OVFL mode bit
    // (MODE register, bit 23) makes every conversion to half clamp instead of overflowing to infinity.
    __builtin_amdgcn_s_setreg(1 | (23 << 6) | (0 << 11), 1);
  }

  const int lane = threadIdx.x & 63;
  const int wm = Tile::wave_m(), wn = Tile::wave_n();
  const int wm_u = __builtin_amdgcn_readfirstlane(wm);
  const int la = wm + Tile::lane_a0();               // this lane's first vocabulary row / token of the tile
  const int lb = wn + Tile::lane_b0();
  const int t0 = tb * Tile::BN;
  const int b_rows = (p.T - t0) < Tile::BN ? (p.T - t0) : Tile::BN;
  const T* weight = static_cast<const T*>(p.weight);
  const float c = p.c;

  int lab[NI], zrow[NI];
  float m[NI], s[NI], u[NI], zt[NI];
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int tok = t0 + lb + Tile::b_block(j);
    lab[j] = -1;
    if (p.labels != nullptr && tok < p.T) {
      const int64_t rel = p.labels[p.order ? p.order[tok] : tok] - p.label_offset;   // a label outside these rows matches nothing
      if (rel >= 0 && rel < p.V) lab[j] = (int)rel - la;
      else lab[j] = -0x40000000;
    } else {
      lab[j] = -0x40000000;
    }
    zrow[j] = (STORE_Z && tok < p.T) ? (p.z_row_map ? p.z_row_map[tok] : tok) : -1;
    if (zrow[j] >= p.z_rows) zrow[j] = -1;
    m[j] = -INFINITY;
    s[j] = 0.f;
    u[j] = 0.f;
    zt[j] = 0.f;
  }

  Tile core;
  const int nslab = p.H / Tile::kSlabK;
  const bool stream = Tile::can_stream(nslab);
  const int32_t* order = p.order ? p.order + t0 : nullptr;
  const auto op_b = Tile::Operand::row_major(static_cast<const T*>(p.hidden) + (order ? 0 : (int64_t)t0 * p.H), p.H,
                                             order ? p.total : b_rows);
  const int vt_begin = vs * p.tiles_per_split;
  const int vt_end = (vt_begin + p.tiles_per_split) < p.n_vt ? (vt_begin + p.tiles_per_split) : p.n_vt;
  bool again = false;      // the tile before was computed twice: nothing of this one has been requested
  typename Tile::Acc acc;
  Tile::zero(acc);
  for (int vt = vt_begin; vt < vt_end; ++vt) {
    const int v0 = vt * kFwdBM;
    const int a_rows = (p.V - v0) < kFwdBM ? (p.V - v0) : kFwdBM;
    const auto op_a = Tile::Operand::row_major(weight + (int64_t)v0 * p.H, p.H, a_rows);
    if constexpr (Tile::kSplit) Tile::zero(acc);
    if (vt == vt_begin || !stream || again) core.start(op_a, op_b, nslab, lds, order, b_rows);
    if (stream && vt + 1 < vt_end) {
      const int v1 = v0 + kFwdBM;
      const int next_rows = (p.V - v1) < kFwdBM ? (p.V - v1) : kFwdBM;
      core.follow(op_a, op_b, nslab, Tile::cursor_a(Tile::Operand::row_major(weight + (int64_t)v1 * p.H, p.H, next_rows), nslab),
                  Tile::cursor_b(op_b, nslab));
    } else {
      core.follow(op_a, op_b, nslab, Tile::hold_a(op_a, nslab), Tile::hold_b(op_b, nslab));
    }
    if constexpr (Tile::kSplit) core.run(acc, nslab);
    else core.run_fresh(acc, nslab);
    if constexpr (Tile::kSplit) again = core.redo(acc, op_a, op_b, nslab, lds, [&] { Tile::zero(acc); }, order, b_rows);
    if (!stream) Tile::finish();

    const bool full = a_rows == kFwdBM;
    // this wave's first unit of the tile, and this lane's piece in it
    char* z_tile = static_cast<char*>(p.z_out) + (int64_t)((v0 + wm_u) / Tile::kSlabK) * Tile::kUnitBytes;
    const int z_lane = Tile::lane_a0() * (int)sizeof(typename KeptLogit<T>::type);
    const uint32_t n_units = (uint32_t)(p.ldz / Tile::kSlabK);
    // Raw logits for the backward: VEC consecutive vocabulary entries of a token are one 16-byte piece of
    // its unit.  Vocabulary rows past V hold zeros already (the operand loads are range-checked), and the backward
    // ignores whatever the padding columns hold.
    auto keep = [&](int j, const float (&x)[MI * 4], auto whole) __attribute__((always_inline)) {
      typedef typename KeptLogit<T>::type ZT;
      constexpr int AG = VEC / 4;                     // blocks whose registers make up one piece
      // The row is the same for every vocabulary tile, so the compiler would keep the 64-bit addresses it
      // forms from it alive across the K loops, where registers are scarcest, spill them, and reload them
      // between the stores (a reload waits for the stores issued before it).  Re-deriving one from the 32-bit row
      // costs a handful of instructions per tile; the pieces lie at constants from it (with an address of its own
      // per piece, some 20 instructions each, 16384 tokens at H = 2048 took 7.55 ms for 7.44).
      int row = zrow[j];
      asm volatile("" : "+v"(row));
      if (row >= 0) {
        char* z_row = z_tile + ((uint64_t)(uint32_t)(row / Tile::kSlabK) * n_units) * Tile::kUnitBytes +
                      (uint32_t)(row % Tile::kSlabK * kRowBytes + z_lane);
#pragma unroll
        for (int i = 0; i < MI; i += AG) {
          if (!decltype(whole)::value && v0 + wm_u + Tile::a_block(i) / 32 * 32 >= p.ldz) continue;     // the same for all lanes
          float piece[VEC];
#pragma unroll
          for (int e = 0; e < VEC; ++e) piece[e] = x[i * 4 + e];
          *reinterpret_cast<u32x4*>(z_row + Tile::a_block(i) / Tile::kSlabK * Tile::kUnitBytes +
                                    Tile::a_block(i) % Tile::kSlabK * (int)sizeof(ZT)) = pack_kept(piece, (ZT*)nullptr);
        }
      }
    };
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      // this token's logits of the lane's vocabulary rows
      float x[MI * 4];
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) x[i * 4 + r] = acc_get(acc[i][j], r);

      if (STORE_Z && full) keep(j, x, Const<1>{});

      // Target logit: only a lane whose rows of this tile hold the label looks for it.
      const int rel = lab[j] - v0;
      if (__builtin_expect(__any((unsigned)rel < (unsigned)Tile::WM), 0)) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (rel == Tile::a_block(i) + r) zt[j] = x[i * 4 + r];
      }

      if (__builtin_expect(!full, 0)) {
        // last, partial vocabulary tile: the zeros of rows past V must not count
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (la + Tile::a_block(i) + r >= a_rows) x[i * 4 + r] = kNoLogit;
      }
      float tmax = x[0];
#pragma unroll
      for (int k = 1; k < MI * 4; ++k) tmax = fmaxf(tmax, x[k]);
      if (!full && tmax == kNoLogit && m[j] == -INFINITY) continue;   // this lane has seen no valid row yet
      const float nm = fmaxf(m[j], tmax);
      const float scale = exp2f((m[j] - nm) * c);  // m = -inf on the first tile -> 0
      const float nb = -nm * c;
      float ls = 0.f, lu = 0.f;
#pragma unroll
      for (int k = 0; k < MI * 4; ++k) {
        const float e = __builtin_amdgcn_exp2f(fmaf(x[k], c, nb));
        ls += e;
        lu = fmaf(e, x[k], lu);
      }
      s[j] = fmaf(s[j], scale, ls);
      u[j] = fmaf(u[j], scale, lu);
      m[j] = nm;
    }
    // A tile that ends inside the vocabulary keeps its logits apart: the test per piece, mixed into the loop above, put every
    // store of every tile out of line, two jumps away (7.34 ms against 7.26 at 16384 tokens of 2048).
    if (STORE_Z && !full) {
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        float x[MI * 4];
#pragma unroll
        for (int k = 0; k < MI * 4; ++k) x[k] = acc_get(acc[k / 4][j], k % 4);
        keep(j, x, Const<0>{});
      }
    }
  }
  if (stream) Tile::finish();

  // Merge the four lanes that hold the same token's other vocabulary rows.
#pragma unroll
  for (int j = 0; j < NI; ++j) {
#pragma unroll
    for (int off = 16; off < 64; off <<= 1) {
      const float om = __shfl_xor(m[j], off);
      const float os = __shfl_xor(s[j], off);
      const float ou = __shfl_xor(u[j], off);
      const float oz = __shfl_xor(zt[j], off);
      merge_state(m[j], s[j], u[j], om, os, ou, c);
      zt[j] += oz;
    }
  }
  // Merge the two waves that share these tokens through LDS.
  float4* xch = reinterpret_cast<float4*>(lds);
  if (wm != 0 && lane < 16) {
#pragma unroll
    for (int j = 0; j < NI; ++j) xch[lb + Tile::b_block(j)] = make_float4(m[j], s[j], u[j], zt[j]);
  }
  __syncthreads();
  if (wm == 0 && lane < 16) {
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const float4 o = xch[lb + Tile::b_block(j)];
      merge_state(m[j], s[j], u[j], o.x, o.y, o.z, c);
      zt[j] += o.w;
      const int tok = t0 + lb + Tile::b_block(j);
      if (tok < p.T) p.part[(int64_t)vs * p.T + tok] = make_float4(m[j], s[j], u[j], zt[j]);
    }
  }
}

struct FinalizeParams {
  const float4* part;
  const int64_t* labels;
  int T, V, n_split;
  float c, inv_temperature;
  float* logprob;
  float* entropy;
  float* rowmax;
  float* lse;
  float4* record;   // non-null: only the merged (max, sum, sum*z, target) record is written
  const int32_t* order;   // optional: row n writes to and takes its label from token order[n]
};

// G threads per token, each merging every G-th split, then each other through LDS; a block is 256 / G consecutive
// tokens wide.  The loop over splits is a chain of merges behind loads: with one thread per token 60 splits
// took 21 us whatever the number of tokens (four loads are in flight per thread now, and G = 8 cuts the chain).
constexpr int kFinalizeThreads = 256;
template <int G>
__global__ __launch_bounds__(kFinalizeThreads) void lmhead_fwd_finalize_kernel(FinalizeParams p) {
  constexpr int kTok = kFinalizeThreads / G;
  const int g = threadIdx.x / kTok, t = blockIdx.x * kTok + threadIdx.x % kTok;
  float m = -INFINITY, s = 0.f, u = 0.f, zt = 0.f;
  if (t < p.T) {
    const float4* part = p.part + t;
    int k = g;
    for (; k + 3 * G < p.n_split; k += 4 * G) {
      float4 o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = part[(int64_t)(k + e * G) * p.T];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        merge_state(m, s, u, o[e].x, o[e].y, o[e].z, p.c);
        zt += o[e].w;
      }
    }
    for (; k < p.n_split; k += G) {
      const float4 o = part[(int64_t)k * p.T];
      merge_state(m, s, u, o.x, o.y, o.z, p.c);
      zt += o.w;
    }
  }
  if (G > 1) {
    __shared__ float4 sh[kFinalizeThreads];
    sh[threadIdx.x] = make_float4(m, s, u, zt);
    __syncthreads();
    if (g != 0) return;
#pragma unroll
    for (int e = 1; e < G; ++e) {
      const float4 o = sh[e * kTok + threadIdx.x];
      merge_state(m, s, u, o.x, o.y, o.z, p.c);
      zt += o.w;
    }
  }
  if (t >= p.T) return;
  if (p.record) {
    p.record[t] = make_float4(m, s, u, zt);
    return;
  }
  const int tok = p.order ? p.order[t] : t;
  const float mx = m * p.inv_temperature;
  const float lse = mx + logf(s);
  p.lse[tok] = lse;
  if (p.rowmax) p.rowmax[tok] = mx;
  if (p.entropy) p.entropy[tok] = lse - p.inv_temperature * u / s;
  if (p.logprob) {
    const int64_t lab = p.labels[tok];
    // A label outside [0, V) has no logit; NaN marks it instead of a silent wrong number.
    p.logprob[tok] = (lab >= 0 && lab < p.V) ? (zt * p.inv_temperature - lse) : NAN;
  }
}

static int launch_finalize(const FinalizeParams& f, hipStream_t stream) {
  if (f.n_split >= 16)
    hipLaunchKernelGGL(lmhead_fwd_finalize_kernel<8>, dim3((f.T + 31) / 32), dim3(kFinalizeThreads), 0, stream, f);
  else
    hipLaunchKernelGGL(lmhead_fwd_finalize_kernel<1>, dim3((f.T + 255) / 256), dim3(kFinalizeThreads), 0, stream, f);
  return check_launch("lmhead_fwd_finalize_kernel");
}

// Split of the vocabulary tiles over workgroups.  A workgroup walks ceil(n_vt / n_split) tiles for
// one block of 256 tokens; with each CU holding one workgroup a launch takes
// ceil(n_tb * n_split / CUs) rounds, so its cost in tile periods is rounds * tiles-per-workgroup.
// Many splits and several rounds are fine (65 token blocks: 35 splits of 17 tiles, 9 rounds = 153 tile
// periods against the ideal 151), so the plan stays within a few per cent of n_tb * n_vt / CUs tile periods
// from about 7 token blocks on.  Two smaller terms, both measured on launches of equal tile periods, with a core of eight
// waves per tile that the present one has replaced (not measured again since):
//  - the splits are handed out in groups of 4 (the workgroups of an XCD then form a block of 4 splits x
//    CUs/32 token blocks that shares operand slabs in the XCD's L2: 4 + 8 = 12 slabs per step for 32 tiles).
//    A last group of w < 4 splits makes blocks of w x 32/w, w + 32/w slabs per step; the time grows by about
//    0.11 of that excess (65536 tokens at H = 4096: 5 splits 63.4 ms, 2 splits 64.2 ms, 6 splits 61.3 ms
//    against 60.6 ms with 4 or 60.9 ms with 8);
//  - every run of tiles starts with a K loop whose first slabs nothing has requested in advance and ends
//    with its partial record: 0.3 tile periods (32768 tokens at H = 7168: 22 splits x 23 tiles 45.2 ms, 4
//    x 127 or 8 x 64 tiles 44.3 - 44.6 ms).
// Returns the launch's cost in sixteenths of a tile period.  `cus` <= 0 plans for a 256-CU device.
static double fwd_single_cost(int n_tb, int n_vt, int cus, int& n_split, int& tiles_per_split) {
  if (cus <= 0) cus = 256;
  const double xcd_wgs = cus / 8.0, full_block = 4.0 + xcd_wgs / 4.0;
  int best = 1;
  double best_cost = -1.0;
  const int most = max_fwd_splits(n_tb) < n_vt ? max_fwd_splits(n_tb) : n_vt;
  for (int sp = 1; sp <= most; ++sp) {
    const int tps = (n_vt + sp - 1) / sp;
    const int eff_sp = (n_vt + tps - 1) / tps;
    const long rounds = ((long)n_tb * eff_sp + cus - 1) / cus;
    const int rem = eff_sp % 4;
    const double excess = rem ? (double)rem / eff_sp * ((rem + xcd_wgs / rem) / full_block - 1.0) : 0.0;
    const double cost = (double)rounds * (tps + 0.3) * 16.0 * (1.0 + 0.11 * excess) + eff_sp * 0.01;
    if (best_cost < 0 || cost < best_cost) { best_cost = cost; best = sp; }
  }
  tiles_per_split = (n_vt + best - 1) / best;
  n_split = (n_vt + tiles_per_split - 1) / tiles_per_split;
  return best_cost;
}

// A tile of 32 * ni tokens against one of 256: its time.  A step of its K loop loads as many bytes of W and reads as many of its
// fragments, whatever the width, so the narrower tile takes more than ni / 8 of the time: 0.59 - 0.65 at ni = 4 from H = 2048 on
// (V = 151936, launches of full rounds).  What a tile takes besides its K loop is nearer to ni / 8 and weighs more the shorter
// the loop is: 0.56 - 0.58 at H = 512 and 1024.
static double fwd_tile_time(int ni, int64_t H) {
  static constexpr double kLong[9] = {0, 0, 0, 0, 0.63, 0.70, 0.81, 0.88, 1.0};
  const double w = H <= 1024 ? 0.0 : H >= 2048 ? 1.0 : (H - 1024) / 1024.0;
  return (1.0 - w) * ni / 8.0 * (1.0 + 0.02 * (8 - ni)) + w * kLong[ni];
}

// Width of the token blocks: 32 * ni tokens.  The last block of 256 is padding for the most part where T is a little over a
// multiple of 256, and a launch of fewer items than CUs leaves the rest idle.  A narrower tile is taken where the plan then
// costs 4 % less; 16-bit inputs only.  Up to two wide blocks that fill the CUs are bound by reading W, so they are
// not made into more blocks (256 tokens, V = 151936, as two blocks of 128 for one of 256: H = 7168 577 us for 522, 4096 315 for 285,
// 2048 179 for 171, 1024 95 for 92; at H = 512 the two would take 52 for 58).
//   H = 4096, V = 151936, us: 128 tokens 269 -> 228, 260 428 -> 333, 400 463 -> 426, 588 638 -> 579, 900 882 -> 848, 1100 1062 -> 968
//   H = 2048:                 128 tokens 161 -> 148, 260 229 -> 188, 588 340 -> 311, 1100 555 -> 510
//   H = 1024, V = 32000:      200 tokens  38 ->  28, 300  40 ->  31, 588  60 ->  45, 1100  84 ->  69
// Over 2408 sizes (H 512 - 7168, V 9000 - 151936, 32 - 4096 tokens), each timed at all five widths: 9 % less time than 256-wide blocks
// on average, 0.4 % more than the best width; 5 sizes more than 2 % slower than 256-wide blocks, none by more than 3.6 %.  (With the
// time of a tile as 0.54 at ni = 4 for every H: 97 sizes, up to 33 %; 512 tokens at H = 7168, V = 32000 169 -> 211 us.)
struct FwdPlan {
  int ni, n_tb, n_split, tiles_per_split;
};
static FwdPlan fwd_plan(int64_t T, int64_t H, int n_vt, int cus, bool narrow) {
  if (cus <= 0) cus = 256;
  const int wide_tb = (int)((T + kFwdBN - 1) / kFwdBN);
  FwdPlan best{8, wide_tb, 0, 0};
  double best_cost = 0.96 * fwd_single_cost(best.n_tb, n_vt, cus, best.n_split, best.tiles_per_split);
  for (int ni = 7; narrow && ni >= 4; --ni) {
    FwdPlan pl{ni, (int)((T + 32 * ni - 1) / (32 * ni)), 0, 0};
    if (pl.n_tb > wide_tb && wide_tb <= 2 && wide_tb * n_vt > cus) continue;
    const double c = fwd_tile_time(ni, H) * fwd_single_cost(pl.n_tb, n_vt, cus, pl.n_split, pl.tiles_per_split);
    if (c < best_cost) { best_cost = c; best = pl; }
  }
  return best;
}

template <typename T, bool STORE_Z, int NI>
static int launch_fwd_kernel(const FwdParams& p, const ItemGrid& ig, hipStream_t stream) {
  using Tile = LogitTile<T, NI>;
  const int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(&lmhead_fwd_kernel<T, STORE_Z, NI>), Tile::kLdsBytes, "lmhead_fwd_kernel");
  if (rc) return rc;
  hipLaunchKernelGGL((lmhead_fwd_kernel<T, STORE_Z, NI>), dim3(ig.grid), dim3(Tile::kThreads), Tile::kLdsBytes, stream, p);
  return check_launch("lmhead_fwd_kernel");
}

template <typename T, bool STORE_Z>
static int launch_fwd(const clgrpo_lmhead_fwd_args* a, hipStream_t stream, int64_t label_offset, float4* record,
                      const RowOrder& rows) {
  constexpr bool kNarrow = sizeof(T) == 2;
  FwdParams p;
  p.hidden = a->hidden;
  p.weight = a->weight;
  p.labels = a->labels;
  p.label_offset = label_offset;
  p.T = (int)a->T;
  p.H = (int)a->H;
  p.V = (int)a->V;
  p.n_vt = (int)((a->V + kFwdBM - 1) / kFwdBM);
  const FwdPlan pl = fwd_plan(a->T, a->H, p.n_vt, device_cu_count(), kNarrow);
  p.n_tb = pl.n_tb; p.n_split = pl.n_split; p.tiles_per_split = pl.tiles_per_split;
  p.c = a->inv_temperature * kLog2e;
  p.part = static_cast<float4*>(a->workspace);
  p.z_out = a->saved_logits;
  p.ldz = a->ld_saved;
  p.z_row_map = a->saved_row_map;
  p.z_rows = (int)a->saved_rows;
  p.order = rows.order;
  p.total = (int)rows.total;
  const ItemGrid ig = item_grid(p.n_tb * p.n_split, device_cu_count());
  p.xcd_wgs = ig.xcd_wgs;
  int rc;
  if constexpr (kNarrow) {
    rc = pl.ni == 4 ? launch_fwd_kernel<T, STORE_Z, 4>(p, ig, stream) : pl.ni == 5 ? launch_fwd_kernel<T, STORE_Z, 5>(p, ig, stream)
       : pl.ni == 6 ? launch_fwd_kernel<T, STORE_Z, 6>(p, ig, stream) : pl.ni == 7 ? launch_fwd_kernel<T, STORE_Z, 7>(p, ig, stream)
                    : launch_fwd_kernel<T, STORE_Z, 8>(p, ig, stream);
  } else {
    rc = launch_fwd_kernel<T, STORE_Z, 8>(p, ig, stream);
  }
  if (rc) return rc;
  FinalizeParams f;
  f.part = p.part;
  f.labels = a->labels;
  f.T = p.T;
  f.V = p.V;
  f.n_split = p.n_split;
  f.c = p.c;
  f.inv_temperature = a->inv_temperature;
  f.logprob = a->labels ? a->logprob : nullptr;
  f.entropy = a->entropy;
  f.rowmax = a->rowmax;
  f.lse = a->lse;
  f.record = record;
  f.order = rows.order;
  return launch_finalize(f, stream);
}

int validate_head_shape(const char* who, int64_t T, int64_t H, int64_t V, int32_t dtype) {
  if (dtype != CLGRPO_BF16 && dtype != CLGRPO_F32) return fail(CLGRPO_EDTYPE, "%s: dtype %d unsupported", who, dtype);
  if (T <= 0 || H <= 0 || V <= 0) return fail(CLGRPO_EINVAL, "%s: T, H, V must be positive (got %lld, %lld, %lld)", who,
                                             (long long)T, (long long)H, (long long)V);
  const int slab = dtype == CLGRPO_BF16 ? 64 : 32;
  if (H % slab != 0) return fail(CLGRPO_ESHAPE, "%s: H=%lld must be a multiple of %d", who, (long long)H, slab);
  // 256 rows of H elements must stay below 2^31 bytes (32-bit offsets of the buffer loads)
  if (T >= (1LL << 30) || V >= (1LL << 30) || H > (1LL << 20)) return fail(CLGRPO_ESHAPE, "%s: size too large", who);
  return CLGRPO_OK;
}

}  // namespace clgrpo

using namespace clgrpo;

extern "C" int64_t clgrpo_saved_logits_ld(int64_t V) { return V <= 0 ? 0 : round_up64(V, 64); }

extern "C" int clgrpo_lmhead_fwd_launch_plan(int64_t T, int64_t V, int32_t cus, int32_t* out) {
  if (T <= 0 || V <= 0 || out == nullptr) return CLGRPO_EINVAL;
  const FwdPlan pl = fwd_plan(T, 4096, (int)((V + kFwdBM - 1) / kFwdBM), cus, true);
  out[0] = pl.n_tb;
  out[1] = pl.n_split;
  out[2] = pl.tiles_per_split;
  return CLGRPO_OK;
}

extern "C" int clgrpo_lmhead_fwd_tile_plan(int64_t T, int64_t H, int64_t V, int32_t dtype, int32_t cus, int32_t* out) {
  if (T <= 0 || H <= 0 || V <= 0 || out == nullptr || (dtype != CLGRPO_BF16 && dtype != CLGRPO_F32)) return CLGRPO_EINVAL;
  const FwdPlan pl = fwd_plan(T, H, (int)((V + kFwdBM - 1) / kFwdBM), cus, dtype == CLGRPO_BF16);
  out[0] = pl.n_tb;
  out[1] = pl.n_split;
  out[2] = pl.tiles_per_split;
  out[3] = 32 * pl.ni;
  out[4] = (int32_t)(1000.0 * fwd_tile_time(pl.ni, H) + 0.5);
  return CLGRPO_OK;
}

extern "C" size_t clgrpo_lmhead_fwd_workspace_bytes(int64_t T, int64_t H, int64_t V, int32_t dtype) {
  (void)H;
  (void)dtype;
  if (T <= 0 || V <= 0) return 0;
  // One record per token and vocabulary split; the split count depends on the device's CU count and never
  // exceeds max_fwd_splits, so this bound holds on any device.  Fewer tokens may take more splits (2200 tokens 455,
  // 2600 372), so it is the largest over all launches of up to T tokens: below 64 blocks of 256, splits x tokens is at
  // most 4096 x 256.  A caller may size scratch memory for its longest call and use it for any shorter one.
  const int64_t n_vt = (V + kFwdBM - 1) / kFwdBM;
  const int64_t few_blocks = n_vt * T < 4096 * kFwdBN ? n_vt * T : 4096 * kFwdBN, many_blocks = (n_vt < 64 ? n_vt : 64) * T;
  return (size_t)(few_blocks > many_blocks ? few_blocks : many_blocks) * sizeof(float4);
}

// Shared by the whole-vocabulary entry point (record == nullptr), the shard one and the whole step.
int clgrpo::head_forward(const char* who, const clgrpo_lmhead_fwd_args* a, int64_t vocab_begin, void* record_ptr,
                         const RowOrder& rows, hipStream_t s) {
  float4* record = static_cast<float4*>(record_ptr);
  CLGRPO_REQUIRE_PTR(a, "args");
  int rc = validate_head_shape(who, a->T, a->H, a->V, a->dtype);
  if (rc) return rc;
  CLGRPO_REQUIRE_PTR(a->hidden, "hidden");
  CLGRPO_REQUIRE_PTR(a->weight, "weight");
  if (record == nullptr) {
    CLGRPO_REQUIRE_PTR(a->lse, "lse");
    if (a->labels != nullptr) CLGRPO_REQUIRE_PTR(a->logprob, "logprob");
  }
  if (vocab_begin < 0) return fail(CLGRPO_EINVAL, "%s: vocab_begin=%lld", who, (long long)vocab_begin);
  if (!(a->inv_temperature > 0.f)) return fail(CLGRPO_EINVAL, "%s: inv_temperature must be > 0", who);
  CLGRPO_REQUIRE_PTR(a->workspace, "workspace");
  const size_t need = clgrpo_lmhead_fwd_workspace_bytes(a->T, a->H, a->V, a->dtype);
  if (a->workspace_bytes < need)
    return fail(CLGRPO_EWORKSPACE, "%s: workspace %zu < %zu bytes", who, a->workspace_bytes, need);
  if (a->saved_logits != nullptr && (a->ld_saved < clgrpo_saved_logits_ld(a->V) || a->ld_saved % 64 != 0))
    return fail(CLGRPO_ESHAPE, "%s: ld_saved=%lld must be a multiple of 64 and >= %lld", who,
                (long long)a->ld_saved, (long long)clgrpo_saved_logits_ld(a->V));
  if (a->saved_logits != nullptr && (a->saved_rows <= 0 || a->saved_rows >= (1LL << 31)))
    return fail(CLGRPO_EINVAL, "%s: saved_rows=%lld", who, (long long)a->saved_rows);
  if (rows.order != nullptr && (rows.total < a->T || rows.total * a->H * (int64_t)dtype_bytes(a->dtype) > kMaxOrderedBytes))
    return fail(CLGRPO_ESHAPE, "%s: %lld rows of %lld elements are too large for a row order", who, (long long)rows.total,
                (long long)a->H);
  if (a->saved_logits != nullptr)
    return a->dtype == CLGRPO_BF16 ? launch_fwd<__bf16, true>(a, s, vocab_begin, record, rows)
                                   : launch_fwd<float, true>(a, s, vocab_begin, record, rows);
  return a->dtype == CLGRPO_BF16 ? launch_fwd<__bf16, false>(a, s, vocab_begin, record, rows)
                                 : launch_fwd<float, false>(a, s, vocab_begin, record, rows);
}

extern "C" int clgrpo_lmhead_fwd(const clgrpo_lmhead_fwd_args* a, void* stream) {
  CLGRPO_REQUIRE_PTR(a, "args");
  return head_forward("clgrpo_lmhead_fwd", a, 0, nullptr, RowOrder{nullptr, a->T}, static_cast<hipStream_t>(stream));
}

extern "C" int clgrpo_lmhead_fwd_shard(const clgrpo_lmhead_fwd_args* a, int64_t vocab_begin, void* record,
                                       void* stream) {
  CLGRPO_REQUIRE_PTR(record, "record");
  CLGRPO_REQUIRE_PTR(a, "args");
  return head_forward("clgrpo_lmhead_fwd_shard", a, vocab_begin, record, RowOrder{nullptr, a->T}, static_cast<hipStream_t>(stream));
}

extern "C" int clgrpo_lmhead_merge_shards(const void* records, int64_t n_shards, int64_t T, const int64_t* labels,
                                          int64_t V_total, float inv_temperature, float* logprob, float* entropy,
                                          float* rowmax, float* lse, void* stream) {
  CLGRPO_REQUIRE_PTR(records, "records");
  CLGRPO_REQUIRE_PTR(lse, "lse");
  if (labels != nullptr) CLGRPO_REQUIRE_PTR(logprob, "logprob");
  if (n_shards <= 0 || n_shards > 4096 || T <= 0 || T >= (1LL << 30) || V_total <= 0)
    return fail(CLGRPO_EINVAL, "clgrpo_lmhead_merge_shards: n_shards=%lld T=%lld V_total=%lld", (long long)n_shards,
                (long long)T, (long long)V_total);
  if (!(inv_temperature > 0.f)) return fail(CLGRPO_EINVAL, "clgrpo_lmhead_merge_shards: inv_temperature must be > 0");
  FinalizeParams f;
  f.part = static_cast<const float4*>(records);
  f.labels = labels;
  f.T = (int)T;
  f.V = (int)(V_total < (1LL << 31) - 1 ? V_total : (1LL << 31) - 1);
  f.n_split = (int)n_shards;
  f.c = inv_temperature * kLog2e;
  f.inv_temperature = inv_temperature;
  f.logprob = labels ? logprob : nullptr;
  f.entropy = entropy;
  f.rowmax = rowmax;
  f.lse = lse;
  f.record = nullptr;
  f.order = nullptr;
  return launch_finalize(f, static_cast<hipStream_t>(stream));
}
