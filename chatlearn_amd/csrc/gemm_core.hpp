// GEMM workgroup tile for gfx950 (CDNA4): C^[256 x 256] = A[256 x K] * B[256 x K]^T, B K-contiguous in memory, A either
// way round, fp32 accumulation on the matrix cores.
//
// One workgroup of 2 x 2 wavefronts (64 lanes each, one per SIMD of a CU) owns a 256 x 256 tile; a wave
// owns 128 x 128 of it as 8 x 8 blocks of 16 x 16 (narrower along B: 8 x kNI).  K is walked in slabs of 128 bytes per row (64 bf16 or 32
// fp32 elements), each slab in two halves of 64 bytes.
//
// What bounds it: on random operands the chip runs at its power limit (the shader clock settles at 1.5 -
// 1.6 GHz), so the rate is what is left after data movement and idle issue slots have taken their energy.
//  - 128 x 128 per wave reads 16 fragments per 64 matrix instructions; the 128 x 64 of eight waves read 12 per 32.
//  - v_mfma 16x16x32 against 32x32x16 on the same operands: 2 % more rate out of registers (1870 against 1827
//    TFLOP/s), 6 % in this loop.
//  - every instruction's place is fixed in the source (see the schedule): with one wave per SIMD nothing else would
//    fill a gap.
// 12126 rows, H = 4096, V = 151936 (bf16): 1.46 - 1.54 PFLOP/s for either contraction of the backward, by the machine; under the
// counters matrix cores busy 0.85 of the cycles at 1.61 GHz (profiles/head_gemm_kernels_c2_sq_counters.txt).  With the barriers
// and load waits left out (wrong results) they were busy 1.5 % of the cycles more and the clock fell: 0.5 % less time.  The
// eight-wave 32x32x16 form of this tile with two 64 KB stages ran 13 % slower.
//
// Operand slabs travel HBM/L2 -> LDS directly (buffer loads with an LDS destination; no registers, no LDS
// store instructions) into two rings of 32 KB slots, three for A and two for B: all 160 KB.  While the matrix
// cores work on slab s, B(s+1) and A(s+1), A(s+2) land; a slot is requested again right after the barrier
// behind its last fragment read.  The third A slot is what makes the loads of a slab early enough: with two
// 64 KB stages (same loop) the rate was 6 % lower.  One barrier per slab, preceded by an explicit
// wait for this wave's own loads, because a barrier alone does not wait for loads whose destination is LDS; the
// youngest eight (the A slab after next) stay outstanding.
//
// A load fills LDS in lane order, so rows are 128 bytes apart with no padding; bank conflicts are
// avoided by which 16-byte chunk and row a lane fetches, undone by the fragment reads (0 conflict cycles, see Bank conflicts).
//
// Operands are row-major (the caller's hidden states and weight), K-blocked (hidden^T, a caller's W^T: per tile and
// slab one contiguous 32 KB piece, see Operand) or kept logits / d(logits) (units, see unit_index).  A may also lie the
// other way round, with the contracted dimension along its rows (see Side): d(logits) has tokens as rows and
// serves both contractions of the backward, and W is read as it is for dhidden.  Neither has a transposed copy.
// Consecutive tiles of a workgroup stream into each other: requests that run past a tile's last slab continue
// with the next tile's first ones, whose first fragments are in registers when the tile ends.
//
// Accumulators (v_mfma_f32_16x16x*): lane l = 16 g + c holds, in register r of block (i, j), the product of
//     A row lane_a0() + a_off(i, r)   and   B row lane_b0() + b_block(j)   of the wave's 128.
// Which rows of the wave's 128 make up a block is free, because it only decides where a fragment is read
// from.  a_off gives a lane VEC = 16 / sizeof(T) consecutive A rows (bf16: over a pair of blocks), b_block BV
// consecutive B rows over BV blocks, so that 16-byte pieces of either orientation of the result are in one
// lane and leave without a shuffle.  The callers put the dimension they reduce over (vocabulary, for the
// softmax statistics) on A, which makes that reduction mostly lane-local.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <utility>

namespace clgrpo {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kRowBytes = 128;    // K-slab bytes per tile row
constexpr int kChunksPerRow = 8;  // 16-byte chunks per slab row
constexpr int kBlockRows = 256;   // rows per block of a K-blocked operand

template <typename T> struct Elem;
template <> struct Elem<__bf16> { static constexpr int kSlabK = 64; };
template <> struct Elem<float> { static constexpr int kSlabK = 32; };

// Element (row, k) of a K-blocked operand with `n_kslab` slabs per row: blocks of 256 rows, each
// block holding its slabs one after another, each slab 256 rows of 128 bytes.
template <typename T>
__host__ __device__ __forceinline__ int64_t blocked_index(int64_t row, int64_t k, int64_t n_kslab) {
  constexpr int E = kRowBytes / (int)sizeof(T);
  return (((row / kBlockRows) * n_kslab + k / E) * kBlockRows + (row % kBlockRows)) * E + (k % E);
}

// Element (token, v) of kept logits and of d(logits) with `n_kslab` slabs per token: units of one slab's 128 bytes of
// vocabulary by as many tokens as a slab has elements (64 x 64 of 16 bits, 32 x 32 of fp32), the units of a row of units one
// after another.  A 256-wide tile of either orientation and one slab of the other dimension are then whole units: 256 / E
// pieces of E * 128 bytes, one 32 KB run where the tile lies along the vocabulary.
template <typename T>
__host__ __device__ __forceinline__ int64_t unit_index(int64_t token, int64_t v, int64_t n_kslab) {
  constexpr int E = kRowBytes / (int)sizeof(T);
  return ((token / E * n_kslab + v / E) * E + token % E) * E + v % E;
}

// Kept logits: the forward leaves a chunk's raw logits for the backward in the layout (see unit_index) that the
// d(logits) operand will have, so that the kernel that turns one into the other works in place.  16-bit inputs keep their logits as IEEE half (10 mantissa bits against bf16's 7: the
// softmax the backward rebuilds from them is 8x closer to the fp32 one), fp32 inputs as fp32.
template <typename T> struct KeptLogit;
template <> struct KeptLogit<__bf16> { typedef _Float16 type; };
template <> struct KeptLogit<float> { typedef float type; };

// Matrix instructions of slot m of a slab half: 64 bytes of K of block (i, j) = (m / NI, m % NI), odd
// rows walked backwards so that neighbours share an operand.  Written as assembly because that is what ties the
// accumulators to the accumulation registers: left to itself the compiler moves all 256 of them between the
// register files around every loop, and spills what is in their way.  The compiler does not see the
// instruction's latency either: see settle().  Everything else that touches an accumulator goes through
// acc_get / acc_set for the same reason.
template <typename T> struct Mma;
template <> struct Mma<__bf16> {
  template <bool kAcross, bool kFresh, int NI>
  __device__ static __forceinline__ void slot(f32x4 (&acc)[8][NI], const u32x4 (&a)[8], const u32x4 (&b)[NI], int m) {
    const int i = m / NI, j = (i & 1) ? NI - 1 - m % NI : m % NI;
    // kFresh: the product alone.  The accumulator stays an operand that is read, for the compiler: as a plain result it is given other
    // registers, and hundreds are spilled.
    if constexpr (kFresh) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "+a"(acc[i][j]) : "v"(a[i]), "v"(b[j]));
    else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(a[i]), "v"(b[j]));
  }
};
template <> struct Mma<float> {
  // 16 bytes hold four K=4 steps: lane group g, element e stands for k = 4g + e in both operands.  A slot takes
  // step m % 8 / 2 of four blocks of row i, so that an accumulator comes up again eight instructions later.
  // kAcross: a[4 q + e] holds k = 4g + e of the four blocks 4 q .. 4 q + 3 (an A with K along its rows): the
  // transposition of a 4 x 4 square of single registers is a choice of registers.
  template <bool kAcross, bool kFresh, int NI>
  __device__ static __forceinline__ void slot(f32x4 (&acc)[8][NI], const u32x4 (&a)[8], const u32x4 (&b)[NI], int m) {
    static_assert(!kFresh, "sixteen bits only");
    static_assert(NI == 8, "four blocks of a row per slot");
    const int i = m / 8, e = m % 8 / 2;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int j = (m % 2) * 4 + k;
      const uint32_t av = kAcross ? a[i / 4 * 4 + e][i % 4] : a[i][e];
      asm volatile("v_mfma_f32_16x16x4_f32 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(av), "v"(b[j][e]));
    }
  }
};

__device__ __forceinline__ float acc_get(const f32x4& acc, int r) {
  float v;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(acc[r]));
  return v;
}
__device__ __forceinline__ void acc_set(f32x4& acc, float v0, float v1, float v2, float v3) {
  float a0, a1, a2, a3;
  asm volatile("v_accvgpr_write_b32 %0, %1" : "=a"(a0) : "v"(v0));
  asm volatile("v_accvgpr_write_b32 %0, %1" : "=a"(a1) : "v"(v1));
  asm volatile("v_accvgpr_write_b32 %0, %1" : "=a"(a2) : "v"(v2));
  asm volatile("v_accvgpr_write_b32 %0, %1" : "=a"(a3) : "v"(v3));
  acc = f32x4{a0, a1, a2, a3};
}

// fn(constant 0), ..., fn(constant N - 1), spelled out: an unrolled loop of this many instructions is over the
// compiler's limit, and what is left rolled up would index registers in memory.
template <int N> struct Const { static constexpr int value = N; };
template <typename Fn, int... M>
__device__ __forceinline__ void each(Fn fn, std::integer_sequence<int, M...>) { (fn(Const<M>{}), ...); }
template <int N, typename Fn>
__device__ __forceinline__ void each(Fn fn) { each(fn, std::make_integer_sequence<int, N>{}); }

// Where the contracted dimension K of operand A lies.
//   kRows:    along the rows of memory (row-major or K-blocked, see Operand): a fragment is 16 bytes of an A row.
//   kWeight:  across them, in a row-major matrix [K][M] (W for dhidden: K = vocabulary, M = H).
//   kLogits:  across them, in units (d(logits) for dW: K = tokens, M = vocabulary).
// Across: a slab is kSlabK rows of 256 columns, in LDS kSub pieces of kSlabK rows x 128 bytes.  A lane reads VEC
// rows (k = VEC g ..) of 16 bytes and transposes that square between registers.  bf16: 32 v_perm_b32 for the 8
// fragments of a half, half of a 4-cycle instruction per matrix instruction of 16 cycles, no LDS access more than
// reading rows takes; fp32: a choice of registers.  It costs 1.5 - 2 % of a contraction (12288 tokens, H = 4096, V = 151936:
// dhidden 9.9 -> 10.05 ms, dW the same within the runs); the transposed copies cost more: W^T 0.46 ms, dz^T 0.75 - 1.1 ms of
// the d(logits) pass and as much memory as the logits.  16384 tokens at H = 4096, whole step: 38.6 -> 37.3 ms, 32768 at
// 2048: 46.9 -> 45.2, 6400 at 2048: 10.0 -> 9.4.  ds_read_b64_tr_b16 in its place needs twice the LDS reads (dW 14 % slower).
// Up to 384 rows a kernel without LDS read W directly; this tile is faster from the first row on (dhidden and the
// d(logits) pass, 256 rows at H = 4096: 471 -> 312 us, 32 rows 271 -> 242).
enum class Side { kRows, kWeight, kLogits };

// BV: consecutive B rows a lane holds (see above).  kUnitsB: B is d(logits) in units (see unit_index).  kNI: 16 x 16 blocks per
// wave along B, so a tile is 32 kNI rows of B wide: 256, or less where whole tiles of 256 would be mostly padding.
template <typename T, int BV, Side kSideA = Side::kRows, bool kUnitsB = false, int kNI = 8>
struct GemmTile {
  static constexpr int MI = 8, NI = kNI;               // 16 x 16 blocks per wave along A / B
  static constexpr int BM = 256, BN = 32 * NI, WM = 128, WN = 16 * NI;
  static constexpr int kSlots = MI * NI;               // matrix instructions of half a slab
  static constexpr int kThreads = 256;
  static constexpr int kSlotBytes = 256 * kRowBytes;   // one operand's slab
  static constexpr int kASlots = 3, kBSlots = 2;
  static constexpr int kLdsBytes = (kASlots + kBSlots) * kSlotBytes;
  static constexpr int kSlabK = Elem<T>::kSlabK;
  static constexpr int VEC = 16 / (int)sizeof(T);      // elements per 16-byte piece
  static constexpr int kBB = kASlots * kSlotBytes;     // LDS offset of the B ring
  static constexpr bool kAcross = kSideA != Side::kRows;
  static constexpr bool kSplit = false;                     // see SplitTile
  static constexpr bool kPerm = kAcross && VEC == 8;   // fragments are made from what is read
  static constexpr int kUnitBytes = kSlabK * kRowBytes;     // a unit of d(logits); a piece of a slab read across
  static constexpr int kSub = 256 / kSlabK;                 // of them per 256-wide slab
  static constexpr uint32_t kHalf = kAcross ? (uint32_t)kUnitBytes / 2 : 64u;   // from a slab's first half to its second in LDS
  static_assert(NI % BV == 0 && NI >= 4 && NI <= 8, "B rows per lane");
  static_assert(!kUnitsB || BN % 64 == 0, "a tile of d(logits) is whole units");

  typedef f32x4 Acc[MI][NI];
  typedef __attribute__((address_space(3))) char lds_char;
  typedef __attribute__((address_space(3))) const u32x4 lds_vec;

  // This lane's rows within the wave's 128: lane_a0() + a_off(i, r) for register r of blocks i, lane_b0() + b_block(j)
  // of blocks j.
  __device__ static __forceinline__ constexpr int a_block(int i) {
    return VEC == 8 ? (i >> 1) * 32 + (i & 1) * 4 : i * 16;
  }
  __device__ static __forceinline__ constexpr int a_off(int i, int r) {
    return kAcross ? i / VEC * 16 * VEC + 4 * VEC * r + i % VEC : a_block(i) + r;
  }
  __device__ static __forceinline__ int a_lane(int rho) { return VEC == 8 ? (rho >> 2) * 8 + (rho & 3) : rho; }
  __device__ static __forceinline__ constexpr int b_block(int j) { return (j / BV) * 16 * BV + j % BV; }
  __device__ static __forceinline__ int lane_a0() {     // first A row of this lane (block 0, register 0)
    const int g = (threadIdx.x & 63) >> 4;
    return VEC * g;
  }
  __device__ static __forceinline__ int lane_b0() { return (threadIdx.x & 15) * BV; }
  __device__ static __forceinline__ int wave_m() { return ((threadIdx.x >> 6) & 1) * WM; }
  __device__ static __forceinline__ int wave_n() { return (threadIdx.x >> 7) * WN; }

  // Bank conflicts.  LDS has 64 banks of 4 bytes, two rows of a slab wide; a wave's 16-byte read takes lanes 0-3, 12-15,
  // 20-27 in one cycle, 4-11, 16-19, 28-31 in the next, and so on 32 lanes further (counted with pairs of lanes on
  // one bank).  In lanes (c, g): eight c's of lane group g and the other eight of g + 1.  These sixteen must fall on
  // eight chunks of either parity of rows.
  //   A rows: the swizzle of a row's chunks is enough, its rows differ in parity.
  //   B rows (row BV c + j): all of one parity (BV even), so rows are exchanged in pairs where c is odd (b_row), and the chunks
  //     are swizzled by the rest of c.  Without the exchange every B read took 4 cycles more (half of SQ_LDS_BANK_CONFLICT per read).
  //   A across: chunks of one row over two pieces of a slab; the odd pieces have their rows exchanged in pairs.
  // A lane reads an exchanged row at the other address of its pair: odd rows go by addresses of their own (odd_a, odd_b).
  __device__ static __forceinline__ int a_swz(int row) { return VEC == 8 ? (row & 3) | ((row >> 3) & 1) << 2 : row & 7; }
  __device__ static __forceinline__ int b_swz(int row) { return row / (2 * BV) & 7; }
  static constexpr int kPairs = BV % 2 == 0;           // an odd BV gives its rows both parities by itself
  __device__ static __forceinline__ int b_row(int row) { return row ^ (row / BV & kPairs); }     // its own inverse

  // Where an operand's tile lives in memory: `rows` valid rows starting at `base`, consecutive
  // rows `row_bytes` apart, consecutive 128-byte K slabs of a row `slab_bytes` apart.
  //   row-major [rows][ld]:                  row_bytes = ld * sizeof(T), slab_bytes = 128
  //   K-blocked [row block][K slab][256][128 B]: row_bytes = 128, slab_bytes = 256 * 128 (one
  //   contiguous 32 KB piece per tile and slab)
  //   units (as B): row_bytes = 128, slab_bytes = one unit, rows of units `unit_row` bytes apart
  // Across (as A) `rows` counts the valid columns of the tile, and `k_left` the valid rows from the K range's first on:
  //   kWeight: row_bytes = ld * sizeof(T), slab_bytes = kSlabK rows, sub_bytes = 128, front = bytes in front of base in its row
  //   kLogits: row_bytes = 128, slab_bytes = a row of units, sub_bytes = one unit
  struct Operand {
    const T* base;
    int row_bytes;
    int64_t slab_bytes;
    int rows;
    int sub_bytes;
    int k_left;
    int front;
    int64_t unit_row;
    __device__ static __forceinline__ Operand row_major(const T* base, int64_t ld, int rows) {
      return Operand{base, (int)(ld * (int64_t)sizeof(T)), kRowBytes, rows, 0, 0, 0, 0};
    }
    __device__ static __forceinline__ Operand blocked(const T* block_base, int rows) {
      return Operand{block_base, kRowBytes, kBlockRows * kRowBytes, rows, 0, 0, 0, 0};
    }
    __device__ static __forceinline__ Operand units(const T* base, int64_t n_kslab, int rows) {
      return Operand{base, kRowBytes, kUnitBytes, rows, 0, 0, 0, n_kslab * kUnitBytes};
    }
    __device__ static __forceinline__ Operand across_weight(const T* base, int64_t ld, int col0, int cols, int k_left) {
      const int row = (int)(ld * (int64_t)sizeof(T));
      return Operand{base, row, (int64_t)kSlabK * row, cols, kRowBytes, k_left, col0 * (int)sizeof(T), 0};
    }
    __device__ static __forceinline__ Operand across_units(const T* base, int64_t n_kslab, int cols) {
      return Operand{base, kRowBytes, n_kslab * kUnitBytes, cols, kUnitBytes, 0, 0, 0};
    }
  };

  // The next slab to request of one operand.  Loads go through range-checked buffer descriptors that cover
  // exactly the valid rows, so rows past them read as zero and nothing outside the operands is touched: the
  // row offset is in the per-lane part, which is what the hardware checks, the K-slab offset in the base
  // address, and the size is what is left of the valid rows from there.
  //   kWeight: `bytes` covers the slab's valid rows of `k_left`; columns past the tile's get an offset outside of it
  //   kLogits: `bytes` covers the units of the tile that exist
  //   kUnitsB: `bytes` counts the tile's rows of units that hold any valid row; the others read as zero
  struct Cursor {
    const char* p;
    int bytes;
    int left;       // slabs of this tile from here on
    int k_left;
    int64_t step;
  };

  int64_t slab_a, slab_b;                     // address step per slab
  int shrink_a, shrink_b;                     // size step per slab
  int64_t jump_a, jump_b;                     // address step behind a tile's last slab
  int pass_a;                                 // bytes between the rows of two loads of a slab
  int row_a, front_a;
  int64_t unit_row_b;
  Cursor a, b, next_a, next_b;
  __amdgpu_buffer_rsrc_t rsrc_a, rsrc_b;
  const char* unit_b;                         // this slab's unit of the next load
  int voff_a[8], voff_b[NI];
  u32x4 raw[8];                               // kPerm: a half of A as it is read
  u32x4 af[2][MI], bf[2][NI];
  uint32_t a0, b0;                            // this lane's fragment addresses in slot 0 of either ring, first half of a slab
  uint32_t odd_a, odd_b;                      // added to them for odd rows
  uint32_t sa, sb;                            // slots of the slab that is read (bytes); B's other slot is sb ^ kSlotBytes
  uint32_t sa1;                               // A's slot after sa
  uint32_t da;                                // slot of the A slab that is requested
  uint32_t w0;                                // this wave's place in a load

  __device__ static __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }
  __device__ __forceinline__ void make_a() {
    rsrc_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a.p), 0, a.bytes, 0x00020000);
  }
  __device__ __forceinline__ void make_b() {
    if constexpr (kUnitsB) { next_unit(0, 0); next_unit(1, 0); }
    else rsrc_b = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(b.p), 0, b.bytes, 0x00020000);
  }
  // Load p (0 .. 7, of B 0 .. NI - 1) of the slab at the cursor: 8 rows per wave, 32 per workgroup (across: 8 rows of one piece).
  __device__ __forceinline__ void load_a(int p) {
    if constexpr (kAcross)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_char*)(uintptr_t)(w0 + da + p * 4096), 16, voff_a[p], 0, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_char*)(uintptr_t)(w0 + da + p * 4096), 16, voff_a[0] + p * pass_a, 0, 0, 0);
  }
  static constexpr int kUnitLoads = kSlabK / 32;       // loads per unit
  __device__ __forceinline__ void next_unit(int part, int u) {     // the descriptor of the slab's unit u
    if (part == 0) unit_b = u == 0 ? b.p : unit_b + unit_row_b;
    else rsrc_b = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(unit_b), 0, u < b.bytes ? kUnitBytes : 0, 0x00020000);
  }
  __device__ __forceinline__ void load_b(int p, uint32_t slot) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (lds_char*)(uintptr_t)(w0 + kBB + slot + p * 4096), 16, voff_b[p], 0, 0, 0);
  }
  __device__ __forceinline__ void load_slab_b(uint32_t slot) {
#pragma unroll
    for (int p = 0; p < NI; ++p) {
      if (kUnitsB && p > 0 && p % kUnitLoads == 0) { next_unit(0, p / kUnitLoads); next_unit(1, p / kUnitLoads); }
      load_b(p, slot);
    }
  }
  // left == 0 ? x : y of scalar values.  As assembly, because the compiler may make a branch of it, and a branch in the slab
  // loop ends the schedule: dW of 12288 tokens at H = 4096 then takes 11.9 ms for 10.3.
  __device__ static __forceinline__ int if_zero(int left, int x, int y) {
    int r;
    asm("s_cmp_eq_u32 %1, 0\n\ts_cselect_b32 %0, %2, %3" : "=s"(r) : "s"(left), "s"(x), "s"(y) : "scc");
    return r;
  }
  __device__ static __forceinline__ int64_t if_zero(int left, int64_t x, int64_t y) {
    int64_t r;
    asm("s_cmp_eq_u32 %1, 0\n\ts_cselect_b64 %0, %2, %3" : "=s"(r) : "s"(left), "s"(x), "s"(y) : "scc");
    return r;
  }
  // The cursors' step to the next slab, in pieces of at most three scalar instructions: what a matrix instruction covers.
  static constexpr int kSteps = 6;
  __device__ static __forceinline__ void advance(int n, Cursor& c, const Cursor& next, int64_t slab, int64_t jump, int shrink) {
    if (n == 0) c.left -= 1;
    if (n == 1) c.step = if_zero(c.left, jump, slab);
    if (n == 2) c.p += c.step;
    if (n == 3) c.bytes = if_zero(c.left, next.bytes, c.bytes - shrink);
    if (n == 4) c.left = if_zero(c.left, next.left, c.left);
  }
  __device__ __forceinline__ void step_a(int n) {
    if constexpr (kSideA == Side::kWeight) {
      if (n == 3) a.k_left = if_zero(a.left, next_a.k_left, a.k_left - kSlabK);
      else advance(n, a, next_a, slab_a, jump_a, 0);
      if (n == 5) a.bytes = weight_bytes(a.k_left, row_a, front_a);
    } else {
      advance(n, a, next_a, slab_a, jump_a, shrink_a);
    }
  }
  __device__ __forceinline__ void step_b(int n) { advance(n, b, next_b, slab_b, jump_b, shrink_b); }
  __device__ __forceinline__ void step_a() { for (int n = 0; n < kSteps; ++n) step_a(n); }
  __device__ __forceinline__ void step_b() { for (int n = 0; n < kSteps; ++n) step_b(n); }
  __device__ static __forceinline__ uint32_t next_slot(uint32_t slot) { return slot == (kASlots - 1) * kSlotBytes ? 0 : slot + kSlotBytes; }
  __device__ __forceinline__ void read_b(int set, uint32_t pb, int j) {
    bf[set][j] = *(lds_vec*)(uintptr_t)((j % 2 ? pb + odd_b : pb) + b_block(j) * kRowBytes);
  }
  // Fragment read n (0 .. MI + NI - 1) of a half: the first A fragment, all of B, the rest of A; across: all of A, all of B.
  __device__ __forceinline__ void read(int set, uint32_t pa, uint32_t pb, int n) {
    if constexpr (kAcross) {
      if (n >= MI) read_b(set, pb, n - MI);
      else if constexpr (kPerm) raw[n] = *(lds_vec*)(uintptr_t)((n % 2 ? pa + odd_a : pa) + n * kRowBytes);
      else af[set][n] = *(lds_vec*)(uintptr_t)((n % 2 ? pa + odd_a : pa) + n / VEC * 2 * kUnitBytes + n % VEC * kRowBytes);
    } else {
      if (n == 0) af[set][0] = *(lds_vec*)(uintptr_t)(pa);
      else if (n <= NI) read_b(set, pb, n - 1);
      else af[set][n - NI] = *(lds_vec*)(uintptr_t)(pa + a_block(n - NI) * kRowBytes);
    }
  }
  // Register n (0 .. 31) of a half's fragments: rows 2 q, 2 q + 1 of column i of the square.
  __device__ __forceinline__ void perm(int set, int n) {
    const int i = n / 4, q = n % 4;
    af[set][i][q] = __builtin_amdgcn_perm(raw[2 * q + 1][i / 2], raw[2 * q][i / 2],
                                          i % 2 ? 0x07060302u : 0x05040100u);
  }

  // Bytes of a kWeight slab of which k_left rows are valid, from the tile's first column on.
  __device__ static __forceinline__ int weight_bytes(int k_left, int row, int front) {
    const int rows = k_left < kSlabK ? k_left : kSlabK;
    const int bytes = rows * row - front;
    return bytes > 0 ? bytes : 0;
  }
  __device__ static __forceinline__ Cursor cursor(const Operand& o, int nslab) {
    return Cursor{reinterpret_cast<const char*>(o.base), o.rows * o.row_bytes, nslab, 0, 0};
  }
  __device__ static __forceinline__ Cursor cursor_a(const Operand& o, int nslab) {
    if constexpr (kSideA == Side::kRows) return cursor(o, nslab);
    const int bytes = kSideA == Side::kWeight ? weight_bytes(o.k_left, o.row_bytes, o.front)
                                              : (o.rows + kSlabK - 1) / kSlabK * kUnitBytes;
    return Cursor{reinterpret_cast<const char*>(o.base), bytes, nslab, o.k_left, 0};
  }
  __device__ static __forceinline__ Cursor cursor_b(const Operand& o, int nslab) {
    if constexpr (!kUnitsB) return cursor(o, nslab);
    return Cursor{reinterpret_cast<const char*>(o.base), (o.rows + kSlabK - 1) / kSlabK, nslab, 0, 0};
  }
  // What the cursor does behind the last slab of the last tile: request that slab again.
  __device__ static __forceinline__ Cursor held(Cursor c, const Operand& o, int nslab, int shrink) {
    c.p += (int64_t)(nslab - 1) * o.slab_bytes;
    c.bytes -= (nslab - 1) * shrink;
    c.left = 1;
    return c;
  }
  __device__ static __forceinline__ Cursor hold_a(const Operand& o, int nslab) {
    Cursor c = held(cursor_a(o, nslab), o, nslab, shrink(o));
    if constexpr (kSideA == Side::kWeight) {
      c.k_left -= (nslab - 1) * kSlabK;
      c.bytes = weight_bytes(c.k_left, o.row_bytes, o.front);
    }
    return c;
  }
  __device__ static __forceinline__ Cursor hold_b(const Operand& o, int nslab) { return held(cursor_b(o, nslab), o, nslab, shrink(o)); }
  __device__ static __forceinline__ int shrink(const Operand& o) { return o.slab_bytes == kRowBytes ? kRowBytes : 0; }
  // What follows the tile whose operands are A and B: a call per tile, behind start().
  __device__ __forceinline__ void follow(const Operand& A, const Operand& B, int nslab, const Cursor& na, const Cursor& nb) {
    next_a = na; next_b = nb;
    jump_a = na.p - (reinterpret_cast<const char*>(A.base) + (int64_t)(nslab - 1) * A.slab_bytes);
    jump_b = nb.p - (reinterpret_cast<const char*>(B.base) + (int64_t)(nslab - 1) * B.slab_bytes);
  }

  // b_order: row r of the B tile is row b_order[r] of B.base (B.rows: rows of the whole array; b_rows of them used).
  __device__ __forceinline__ void place(const Operand& A, const Operand& B, int nslab, char* shared,
                                        const int32_t* b_order = nullptr, int b_rows = 0) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t lds = (uint32_t)(uintptr_t)(lds_char*)shared;
    slab_a = A.slab_bytes; slab_b = B.slab_bytes;
    shrink_a = kAcross ? 0 : shrink(A);
    shrink_b = shrink(B);
    pass_a = 32 * A.row_bytes;
    row_a = A.row_bytes; front_a = A.front;
    unit_row_b = B.unit_row;
    w0 = lds + __builtin_amdgcn_readfirstlane(wave) * 1024;
    // A wave's load fills 1 KB of LDS in lane order: 8 rows x 8 chunks.  The lane that lands on (row, slot)
    // fetches chunk slot ^ swz(row); load p of a slab starts 32 p rows further down, which leaves a_swz as it is.
    const int row = wave * 8 + (lane >> 3), chunk = lane & 7;
    if constexpr (kAcross) {
#pragma unroll
      for (int p = 0; p < 8; ++p) {
        const int sub = p * 32 / kSlabK, k = (p * 32 % kSlabK + row) ^ (sub & 1);
        const bool valid = kSideA == Side::kLogits || sub * kSlabK < A.rows;
        voff_a[p] = valid ? sub * A.sub_bytes + k * A.row_bytes + chunk * 16 : 0x7fffff00;
      }
    } else {
      voff_a[0] = row * A.row_bytes + (chunk ^ a_swz(row)) * 16;
    }
#pragma unroll
    for (int p = 0; p < NI; ++p) {
      const int r = b_row(row + 32 * p);
      const int off = kUnitsB ? r % kSlabK * kRowBytes
                              : (b_order == nullptr ? r * B.row_bytes : (r < b_rows ? b_order[r] * B.row_bytes : 0x7fffff00));
      voff_b[p] = off + (chunk ^ b_swz(r)) * 16;
    }
    const int g = lane >> 4, c = lane & 15;
    const int fa = a_lane(c), fb = c * BV;
    if constexpr (kAcross) {
      const int pc = (c & 3) * 4 + (c >> 2), sub = wave_m() / kSlabK + (pc >> 3);    // chunk of the wave's first 16
      a0 = lds + sub * kUnitBytes + (VEC * g + (sub & 1)) * kRowBytes + (pc & 7) * 16;
      odd_a = -2 * (sub & 1) * kRowBytes;
    } else {
      a0 = lds + (wave_m() + fa) * kRowBytes + (g ^ a_swz(fa)) * 16;
    }
    b0 = lds + kBB + (wave_n() + fb + (c & kPairs)) * kRowBytes + (g ^ b_swz(fb)) * 16;
    odd_b = -2 * (c & kPairs) * kRowBytes;
    a = cursor_a(A, nslab); b = cursor_b(B, nslab);
    follow(A, B, nslab, hold_a(A, nslab), hold_b(B, nslab));
    make_a(); make_b();
    da = sa = sb = 0;
  }
  __device__ __forceinline__ void load_slab_a() {
#pragma unroll
    for (int p = 0; p < 8; ++p) load_a(p);
  }

  // First tile of a workgroup (or of a run that does not stream): nothing is in flight, LDS is free.
  __device__ __forceinline__ void start(const Operand& A, const Operand& B, int nslab, char* shared,
                                        const int32_t* b_order = nullptr, int b_rows = 0) {
    place(A, B, nslab, shared, b_order, b_rows);
    load_slab_a();
    load_slab_b(0);
    step_a(); step_b(); make_a(); make_b(); da = kSlotBytes;
    load_slab_a();
    step_a(); make_a(); da = 2 * kSlotBytes;
    __builtin_amdgcn_s_waitcnt(0x0F78);    // all but the youngest eight loads
    __syncthreads();
#pragma unroll
    for (int n = 0; n < MI + NI; ++n) read(0, a0, b0, n);
    if constexpr (kPerm) {
#pragma unroll
      for (int n = 0; n < 4 * MI; ++n) perm(0, n);
    }
    load_slab_b(kSlotBytes);
  }

  // The schedule of a half of a slab: 64 slots of one matrix instruction (fp32: four) each.  It takes 16 cycles and its issue 4, so
  // three more instructions fit behind it, and every one beyond that is a gap in the matrix cores' work: the same
  // instructions with up to nine scalar ones in a slot were 5 % slower in the contraction that has the most of them.  Fragment
  // reads take even slots of the first 32, a load every eighth (three instructions by itself, its LDS address goes through
  // m0), scalar steps the odd slots left over, the second 32 slots the transposition.  Loads every 4 or 6 slots: no faster.
  // (Narrower tiles keep the same order in fewer slots; A's loads then come every NI.)
  static constexpr int load_a_at(int m) { return m % NI == 1 ? m / NI : -1; }
  static constexpr int load_b_at(int m) { return m % 8 == 1 ? m / 8 : -1; }
  static constexpr int unit_at(int m) {                // unit that begins with slot m's load of B
    return kUnitsB && load_b_at(m) > 0 && load_b_at(m) < NI && load_b_at(m) % kUnitLoads == 0 ? load_b_at(m) / kUnitLoads : -1;
  }
  static constexpr bool spare(int h, int m) {          // odd, without a load; a unit's descriptor is made in the two slots before its load
    return m % 2 == 1 && (h == 0 ? load_a_at(m) < 0 : load_b_at(m) < 0 && unit_at(m + 2) <= 0);
  }
  static constexpr int step_at(int h, int m) {         // scalar step of slot m
    if (!spare(h, m)) return -1;
    int n = 0;
    for (int k = 1; k < m; k += 2) n += spare(h, k);
    return n;
  }
  static constexpr int perm_from(int h, int m) {       // registers transposed in front of slot m: none behind a load, two in the first slots
    constexpr int first = NI == 8 ? 32 : NI == 6 ? 24 : 18;
    if (m <= first) return 0;
    if (NI < 8) return 4 * MI * (m - first) / (kSlots - first);
    int n = 0, twice = 4;
    for (int k = first; k < m; ++k)
      if ((h == 0 ? load_a_at(k) : load_b_at(k)) < 0) n += twice > 0 ? (--twice, 2) : 1;
    return n;
  }

  // A slab, and what a guest does beside it: guest.first<m>() and guest.second<m>() stand behind matrix instruction m of
  // either half, and have issued Guest::kOps vector memory accesses between one half's loads and the next one's.
  struct NoGuest {
    static constexpr int kOps = 0;
    template <int m> __device__ __forceinline__ void first() {}
    template <int m> __device__ __forceinline__ void second() {}
  };
  template <bool kFresh = false, typename Guest>
  __device__ __forceinline__ void slab(Acc& acc, Guest& guest) {
#ifdef __HIP_DEVICE_COMPILE__      // the host's pass drops kernels whose body holds this many lambdas, without a word
    each<kSlots>([&](auto c) __attribute__((always_inline)) {            // first half of the slab
      constexpr int m = decltype(c)::value, n = step_at(0, m);
      Mma<T>::template slot<kAcross, kFresh, NI>(acc, af[0], bf[0], m);
      fence();
      if constexpr (m % 2 == 0 && m < 2 * (MI + NI)) { read(1, half_a() + sa, (b0 ^ 64) + sb, m / 2); fence(); }
      if constexpr (load_a_at(m) >= 0) { load_a(load_a_at(m)); fence(); }
      if constexpr (n >= 0 && n < kSteps) { step_b(n); fence(); }
      if constexpr (n == kSteps) { make_b(); fence(); }
      if constexpr (n == kSteps + 1) { sa1 = next_slot(sa); fence(); }
      if constexpr (kPerm) {
#pragma unroll
        for (int k = perm_from(0, m); k < perm_from(0, m + 1); ++k) { perm(1, k); fence(); }
      }
      guest.template first<m>();
    });
    fence();
    // every wave has the last fragments of this slab, and the next one's loads have landed: all but the youngest eight, A of the slab
    // after it, and what the guest has issued around them
    __builtin_amdgcn_s_waitcnt(0x0070 + 8 + Guest::kOps);
    static_assert(8 + Guest::kOps < 16, "the wait's upper bits are elsewhere");
    __builtin_amdgcn_s_barrier();
    fence();
    each<kSlots>([&](auto c) __attribute__((always_inline)) {            // second half, while the next slab's first fragments come in
      constexpr int m = decltype(c)::value, n = step_at(1, m);
      Mma<T>::template slot<kAcross, false, NI>(acc, af[1], bf[1], m);
      fence();
      if constexpr (m % 2 == 0 && m < 2 * (MI + NI)) { read(0, a0 + sa1, b0 + (sb ^ kSlotBytes), m / 2); fence(); }
      if constexpr (load_b_at(m) >= 0) { load_b(load_b_at(m), sb); fence(); }
      if constexpr (unit_at(m + 2) > 0) { next_unit(0, unit_at(m + 2)); fence(); }
      if constexpr (unit_at(m + 1) > 0) { next_unit(1, unit_at(m + 1)); fence(); }
      if constexpr (n >= 0 && n < kSteps) { step_a(n); fence(); }
      if constexpr (n == kSteps) { make_a(); fence(); }
      if constexpr (n == kSteps + 1) { da = next_slot(da); fence(); }
      if constexpr (kPerm) {
#pragma unroll
        for (int k = perm_from(1, m); k < perm_from(1, m + 1); ++k) { perm(0, k); fence(); }
      }
      guest.template second<m>();
    });
    sa = sa1; sb ^= kSlotBytes;
#endif
  }

  // One tile's K loop of `nslab` slabs; acc must be initialised by the caller.  Between tiles of a
  // streaming workgroup LDS stays in use; after the last one call finish() before touching it.
  __device__ __forceinline__ void run(Acc& acc, int nslab) {
    settle();
    NoGuest none;
    for (int s = 0; s < nslab; ++s) slab(acc, none);
    settle();
  }
  // The same over accumulators that hold anything.  Clearing them takes 256 instructions per tile that no matrix instruction covers
  // (forward, V = 151936: 16384 tokens of 2048 7.32 -> 7.28 ms, of 4096 without kept logits 13.11 -> 13.03, 588 tokens 602 -> 598 us; 8192
  // of 1024, V = 102400 1.424 -> 1.408 ms; with H = 7168, and up to a few tiles per workgroup, no difference).
  __device__ __forceinline__ void run_fresh(Acc& acc, int nslab) {
    settle();
    NoGuest none;
    slab<true>(acc, none);
    for (int s = 1; s < nslab; ++s) slab(acc, none);
    settle();
  }
  // The same as run() with a guest in the first 2 `pairs` slabs; at least one pair and one slab more.  (A loop that may not run at all, between
  // the accumulators' clearing and another one, had them moved and 200 registers spilled.)
  template <typename Guest>
  __device__ __forceinline__ void run_with(Acc& acc, int nslab, int pairs, Guest& guest) {
    settle();
    int s = 0;
    do {
      auto even = guest.template turn<0>();
      slab(acc, even);
      auto odd = guest.template turn<1>();
      slab(acc, odd);
    } while (++s < pairs);
    NoGuest none;
    s = 2 * pairs;
    do slab(acc, none); while (++s < nslab);
    settle();
  }

  __device__ __forceinline__ uint32_t half_a() const { return kAcross ? a0 + kUnitBytes / 2 : a0 ^ 64; }

  // Wait states between matrix instructions and other accesses to the accumulators, in either direction: at most
  // 19 (result of a 16-pass instruction read by the vector unit).
  __device__ static __forceinline__ void settle() {
    fence();
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    fence();
  }

  // All loads have landed and every wave is past its last fragment read: LDS is free.
  __device__ static __forceinline__ void finish() {
    __builtin_amdgcn_s_waitcnt(0x0070);
    __syncthreads();
  }

  // Whether a workgroup's tiles of `nslab` slabs can stream: A is requested three slabs ahead, which must not
  // reach beyond the next tile.
  __device__ static __forceinline__ bool can_stream(int nslab) { return nslab >= kASlots; }

  __device__ static __forceinline__ void zero(Acc& acc) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) acc_set(acc[i][j], 0.f, 0.f, 0.f, 0.f);
  }
};

// The tile of fp32 operands, on the 16-bit matrix cores.
//
// An operand element is the sum of three 16-bit floats: x0 = x rounded to 8 bits of mantissa, x1 the rest rounded, x2 what is
// left (24 bits in all: of 4 M random values none had a remainder; below 2^-108 the last parts lose bits to the smallest exponent).  A
// product takes the six of the nine partial products that are above 2^-26 of it, into the same fp32 accumulators: six v_mfma 16x16x32
// of 16 cycles in the place of eight v_mfma 16x16x4_f32 of 32, and six additions to an accumulator in the place of 32.
//   1536 tokens, H = 1024, V = 151936, us: forward 3270 -> 2020, dhidden 3360 -> 1915, dW 3220 -> 1870
//   error against 64 bits there (2-norm): logprob 6.5e-8 -> 6.1e-8, dhidden 2.2e-6 -> 1.2e-6, dW 6.8e-7 -> 3.3e-7; the same or better
//   over eight sizes of 96 - 4096 tokens, H 512 - 2048, V 32000 - 151936
// What bounds it: issue beside the matrix cores and their power (busy 0.68 - 0.75 of the cycles at 1.9 GHz, where the fp32
// instructions were busy 0.86 - 0.93 at 2.4).
//
// The operands stay fp32 in memory and in LDS.  A wave splits the fragments it has read, 44 instructions for the eight elements
// that a lane has of a block, 704 beside the 384 matrix instructions of a slab, each of which covers two (a third costs 5
// cycles).  v_dot2_f32_bf16 with (-1, 0), which leaves the rest of an element in one instruction, holds up the matrix cores: 34 cycles
// per matrix instruction with one of them beside each.
// Registers decide the order: the parts of all eight B blocks are kept (96), those of A are made a pair of blocks ahead (2 x 24).
// A slab is four pairs q of A blocks, a pair eight steps j of B blocks, a step twelve matrix instructions.  Beside them
//   steps 1 - 7 of a pair            split the next pair of A blocks;
//   steps 1 - 7 of the last pair     split B blocks 0 - 3 of the next slab, into the registers of this one's, which are used up;
//   steps 0 - 6 of the first pair    split B blocks 4 - 7, each before its first use;
//   the last / the first pair        request A of the slab after next / B of the next slab.
// One barrier per slab, behind the third pair: the next slab has landed, and what is left of this one is in registers.  Two slots
// per operand are enough, as a slab takes three times as long as one of 16-bit elements.
//
// What is not finite has no such parts (inf - inf): a tile with a NaN among its sums is computed again by the fp32
// instructions (see redo), whose result stands.
template <int BV, Side kSideA = Side::kRows, bool kUnitsB = false>
struct SplitTile : GemmTile<float, BV, kSideA, kUnitsB> {
  using Whole = GemmTile<float, BV, kSideA, kUnitsB>;
  using typename Whole::Acc;
  using typename Whole::Operand;
  using typename Whole::lds_vec;
  static constexpr bool kSplit = true, kAcross = Whole::kAcross;
  static constexpr int kSlotBytes = Whole::kSlotBytes, kUnitBytes = Whole::kUnitBytes, kVec = Whole::VEC;

  u32x4 xa[kAcross ? 8 : 4];      // A as it is read: two halves of two blocks, or (across, where a read covers four) eight k of four
  u32x4 xb[2][2];                 // B as it is read: a block's two halves
  u32x4 pa[2][2][3], pb[8][3];    // parts: [set][block of the pair][part], [block][part]
  uint32_t ra[8], rb[8], wa, wb;  // what is left of the elements being split, a part of one

  // Instruction n (0 .. 43) of splitting eight elements x(0) .. x(7): round two of them, widen one, subtract it.
  static constexpr int kSplitOps = 44;
  template <int n, typename X>
  __device__ static __forceinline__ void split(u32x4 (&part)[3], uint32_t (&rest)[8], uint32_t& wide, X x) {
    constexpr int t = n / 20, k = n % 20, e = (k - 4) / 2;
    auto left = [&](int i) { return t == 0 ? x(i) : rest[i]; };
    if constexpr (k < 4) {
      uint32_t r;
      asm volatile("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(left(2 * k)), "v"(left(2 * k + 1)));
      part[t][k] = r;
    } else if constexpr (k % 2 == 0) {
      wide = e % 2 ? part[t][e / 2] & 0xffff0000u : part[t][e / 2] << 16;
    } else {
      rest[e] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(float, left(e)) - __builtin_bit_cast(float, wide));
    }
    Whole::fence();
  }
  // of block b of the pair q of A, of block j of B
  template <int n, int b, int q>
  __device__ __forceinline__ void split_a() {
    split<n>(pa[q % 2][b], ra, wa, [&](int e) { return kAcross ? xa[e][(2 * q + b) % 4] : xa[2 * b + e / 4][e % 4]; });
  }
  template <int n, int j>
  __device__ __forceinline__ void split_b() {
    split<n>(pb[j], rb, wb, [&](int e) { return xb[j % 2][e / 4][e % 4]; });
  }
  // Reads of the pair q of A (across: of the four blocks it begins) and of block j of B in the slot at `slot`.
  static constexpr int kReadsA = kAcross ? 8 : 4;
  template <int n, int q>
  __device__ __forceinline__ void read_a(uint32_t slot) {
    if constexpr (kAcross) {
      const uint32_t at = this->a0 + slot + n / 4 * (kUnitBytes / 2);
      xa[n] = *(lds_vec*)(uintptr_t)((n % 2 ? at + this->odd_a : at) + q / 2 * 2 * kUnitBytes + n % 4 * kRowBytes);
    } else {
      xa[n] = *(lds_vec*)(uintptr_t)((n % 2 ? this->a0 ^ 64 : this->a0) + slot + Whole::a_block(2 * q + n / 2) * kRowBytes);
    }
    Whole::fence();
  }
  template <int n, int j>
  __device__ __forceinline__ void read_b(uint32_t slot) {
    const uint32_t at = (n ? this->b0 ^ 64 : this->b0) + slot;
    xb[j % 2][n] = *(lds_vec*)(uintptr_t)((j % 2 ? at + this->odd_b : at) + Whole::b_block(j) * kRowBytes);
    Whole::fence();
  }

  __device__ __forceinline__ void start(const Operand& A, const Operand& B, int nslab, char* shared,
                                        const int32_t* b_order = nullptr, int b_rows = 0) {
    this->place(A, B, nslab, shared, b_order, b_rows);
    this->load_slab_a();
    this->load_slab_b(0);
    this->step_a(); this->step_b(); this->make_a(); this->make_b();
    this->da = kSlotBytes;
    this->load_slab_a();
    __builtin_amdgcn_s_waitcnt(0x0F78);    // all but the youngest eight loads
    __syncthreads();
  }

  // The parts a slab's first pair begins with, for a tile's first slab.
  __device__ __forceinline__ void prime() {
    each<kReadsA>([&](auto n) __attribute__((always_inline)) { read_a<decltype(n)::value, 0>(this->sa); });
    each<2>([&](auto b) __attribute__((always_inline)) {
      each<kSplitOps>([&](auto n) __attribute__((always_inline)) { split_a<decltype(n)::value, decltype(b)::value, 0>(); });
    });
    each<5>([&](auto c) __attribute__((always_inline)) {
      constexpr int j = decltype(c)::value;
      read_b<0, j>(this->sa);
      read_b<1, j>(this->sa);
      if constexpr (j > 0) each<kSplitOps>([&](auto n) __attribute__((always_inline)) { split_b<decltype(n)::value, j - 1>(); });
    });
  }

  // The B blocks are split one after another from the second step of a slab's last pair on.  The block that a step reads: each
  // before its first instruction, in the registers of the one before the last, which is through.
  static constexpr int b_step(int q, int j) { return q == 3 ? j : q == 0 ? 8 + j : -1; }
  static constexpr int b_read(int step) {
    return step == 0 ? 0 : step == 2 ? 1 : step == 3 ? 2 : step == 5 ? 3 : step == 7 ? 4 : step == 8 ? 5 : step == 10 ? 6 : step == 12 ? 7 : -1;
  }
  static constexpr int kStepSlots = 12;
  // Instructions of splitting `blocks` blocks over `steps` steps that stand in front of slot m of them.
  static constexpr int at(int m, int steps, int blocks) { return blocks * kSplitOps * m / (steps * kStepSlots); }

  // What stands behind matrix instruction m of step j of pair q.
  template <int q, int j, int m>
  __device__ __forceinline__ void beside() {
    constexpr int step = b_step(q, j), next = (q + 1) % 4;
    const uint32_t other = this->sa ^ kSlotBytes;
    if constexpr (b_read(step) >= 0 && m < 2) read_b<m, b_read(step)>(q == 3 ? other : this->sa);
    if constexpr (j == 0 && m >= 2 && m < 2 + kReadsA && (!kAcross || next % 2 == 0)) read_a<m - 2, next>(q == 3 ? other : this->sa);
    if constexpr (step >= 1 && step <= 14) {
      constexpr int from = at((step - 1) * kStepSlots + m, 14, 8), to = at((step - 1) * kStepSlots + m + 1, 14, 8);
      each<to - from>([&](auto c) __attribute__((always_inline)) {
        constexpr int n = from + decltype(c)::value;
        split_b<n % kSplitOps, n / kSplitOps>();
      });
    }
    if constexpr (j >= 1) {
      constexpr int from = at((j - 1) * kStepSlots + m, 7, 2), to = at((j - 1) * kStepSlots + m + 1, 7, 2);
      each<to - from>([&](auto c) __attribute__((always_inline)) {
        constexpr int n = from + decltype(c)::value;
        split_a<n % kSplitOps, n / kSplitOps, next>();
      });
    }
    if constexpr (q == 3 && m == 6) { this->load_a(j); Whole::fence(); }
    if constexpr (q == 0 && kUnitsB && j > 0 && (m == 3 || m == 4)) { this->next_unit(m - 3, j); Whole::fence(); }
    if constexpr (q == 0 && m == 6) { this->load_b(j, other); Whole::fence(); }
    if constexpr (q == 1 && m == 10) {
      if constexpr (j < Whole::kSteps) this->step_a(j);
      if constexpr (j == Whole::kSteps) this->make_a();
      if constexpr (j == Whole::kSteps + 1) this->da = this->sa;
      Whole::fence();
    }
    if constexpr (q == 2 && m == 10) {
      if constexpr (j < Whole::kSteps) this->step_b(j);
      if constexpr (j == Whole::kSteps) this->make_b();
      Whole::fence();
    }
  }

  __device__ __forceinline__ void run(Acc& acc, int nslab) {
#ifdef __HIP_DEVICE_COMPILE__
    Whole::settle();
    prime();
    for (int s = 0; s < nslab; ++s) {
      each<4>([&](auto cq) __attribute__((always_inline)) {
        each<8>([&](auto cj) __attribute__((always_inline)) {
          each<kStepSlots>([&](auto cm) __attribute__((always_inline)) {
            constexpr int q = decltype(cq)::value, j = decltype(cj)::value, m = decltype(cm)::value;
            constexpr int of_a[6] = {0, 0, 1, 1, 0, 2}, of_b[6] = {2, 1, 1, 0, 0, 0};
            asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                         : "+a"(acc[2 * q + m % 2][j]) : "v"(pa[q % 2][m % 2][of_a[m / 2]]), "v"(pb[j][of_b[m / 2]]));
            Whole::fence();
            beside<q, j, m>();
          });
        });
        if constexpr (decltype(cq)::value == 2) {
          __builtin_amdgcn_s_waitcnt(0x0070);      // the next slab has landed, this one's reads are through
          __builtin_amdgcn_s_barrier();
          Whole::fence();
        }
      });
      this->sa ^= kSlotBytes;
    }
    Whole::settle();
#endif
  }

  // Behind run(): whether the tile had to be computed again.  An operand element that is not finite makes every sum of its row NaN
  // (its parts are, and 0 * NaN is), so a sum of every row and one of every column tell.  `init` sets the accumulators as they were
  // before run().  LDS is free then, and the next tile begins with start().
  template <typename Init>
  __device__ __forceinline__ bool redo(Acc& acc, const Operand& A, const Operand& B, int nslab, char* shared, Init init,
                                       const int32_t* b_order = nullptr, int b_rows = 0) {
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < Whole::MI; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) sum += acc_get(acc[i][0], r);
#pragma unroll
    for (int j = 1; j < Whole::NI; ++j) sum += acc_get(acc[0][j], 0);
    // the flags are in the third slot of A, which this tile does not use
    typedef __attribute__((address_space(3))) volatile uint32_t lds_flag;
    lds_flag* flag = (lds_flag*)(uintptr_t)((uint32_t)(uintptr_t)(typename Whole::lds_char*)shared + 2 * kSlotBytes);
    const bool bad = __any(sum != sum);
    if ((threadIdx.x & 63) == 0) flag[threadIdx.x >> 6] = bad;
    __builtin_amdgcn_s_waitcnt(0xC07F);      // this wave's flag is written (loads stay outstanding)
    __builtin_amdgcn_s_barrier();
    const uint32_t any = flag[0] | flag[1] | flag[2] | flag[3];
    if (__builtin_expect(__builtin_amdgcn_readfirstlane(any) == 0, 1)) return false;
    Whole::finish();
    init();
    Whole whole;
    whole.start(A, B, nslab, shared, b_order, b_rows);
    whole.run(acc, nslab);
    Whole::finish();
    return true;
  }
};

// The tile for operands of type T.
template <typename T, int BV, Side S = Side::kRows, bool kUnitsB = false, int NI = 8>
struct TileOf { typedef GemmTile<T, BV, S, kUnitsB, NI> type; };
template <int BV, Side S, bool kUnitsB>
struct TileOf<float, BV, S, kUnitsB, 8> { typedef SplitTile<BV, S, kUnitsB> type; };

constexpr int kHeadThreads = 256;
// The tile of the kernels that hold logits (A = vocabulary, B = tokens).  Its results leave along A only, so neighbouring lanes may
// hold neighbouring tokens: a store covers 64 bytes of sixteen rows that follow one another, and labels and records are read in runs.  With
// eight consecutive tokens per lane, as the tiles of the backward have them, forward without kept logits, 16384 tokens of 2048:
// 6.87 -> 6.79 ms, 8192 of 4096 6.59 -> 6.54; with them 7.18 -> 7.16, 6.76 -> 6.73; 200 tokens of 1024, V = 32000 28.4 -> 28.0 us.
// The widths between are no faster with it (320 tokens of 2048, V = 32000 42.6 -> 43.0 us, 588 of 4096 580 -> 586).
template <typename T, int NI = 8> using LogitTile = typename TileOf<T, NI % 4 == 0 ? 1 : NI, Side::kRows, false, NI>::type;

// Workgroup id -> logical work item so that the workgroups resident on one XCD
// (hardware deals consecutive ids round-robin over the 8 XCDs) own a contiguous
// range of logical items and therefore share operand tiles in that XCD's L2.
// grid must be padded to a multiple of 8; items >= n_items return -1.
__device__ __forceinline__ int xcd_remap(int bid, int grid) {
  const int per_xcd = grid >> 3;
  return (bid & 7) * per_xcd + (bid >> 3);
}

// The same for launches of several rounds (more items than the CUs hold at once; xcd_wgs = workgroups
// resident per XCD = CUs / 8, grid padded to a multiple of 8 * xcd_wgs): the hardware starts workgroups in
// id order, so the k-th batch of xcd_wgs workgroups of every XCD runs at about the same time.  Those 8
// batches get 8 consecutive blocks of the logical order: at any time all XCDs work inside one stretch of
// 8 * xcd_wgs consecutive items - the same few operand tiles of the slow dimension of grouped_tile, which
// the last-level cache then serves to all of them from one HBM read - instead of eight stretches a
// eighth of the launch apart.  Bit-identical results; measured on the forward, with a core of eight waves: 32768 tokens at H = 7168
// (22 vocabulary splits, 11 rounds) 48.1 -> 45.2 ms, 16640 tokens at H = 4096 (35 splits, 9 rounds) 16.1 ->
// 15.4 ms, no change for launches of one or two rounds.  Used by the forward and by plain launches of
// the backward's products (see launch_gemm_one); the kernel that recomputes d(logits) tile by tile got 6 % slower with it.
__device__ __forceinline__ int xcd_round_remap(int bid, int xcd_wgs) {
  const int x = bid & 7, slot = bid >> 3;
  return ((slot / xcd_wgs) * 8 + x) * xcd_wgs + slot % xcd_wgs;
}

// Work item of this workgroup: xcd_wgs > 0 selects the mapping for launches of several rounds.
__device__ __forceinline__ int work_item(int xcd_wgs) {
  return xcd_wgs > 0 ? xcd_round_remap(blockIdx.x, xcd_wgs) : xcd_remap(blockIdx.x, gridDim.x);
}

// Host side: grid size for n_items work items on a device with `cus` CUs, and the xcd_wgs to hand to the
// kernel (0: one round or less, plain xcd_remap on a grid padded to a multiple of 8).
struct ItemGrid {
  int grid, xcd_wgs;
};
inline ItemGrid item_grid(int n_items, int cus) {
  const int xw = cus / 8;
  if (xw > 0 && n_items > 8 * xw) return ItemGrid{(n_items + 8 * xw - 1) / (8 * xw) * (8 * xw), xw};
  return ItemGrid{(n_items + 7) / 8 * 8, 0};
}

// Logical item -> (m tile, n tile), walking groups of `gm` m-tiles across all n
// tiles so neighbours in the logical order share A rows or B rows.
__device__ __forceinline__ void grouped_tile(int item, int n_m, int n_n, int gm, int& mt, int& nt) {
  const int per_group = gm * n_n;
  const int g = item / per_group;
  const int first_m = g * gm;
  const int rows = (n_m - first_m) < gm ? (n_m - first_m) : gm;
  const int in_g = item - g * per_group;
  mt = first_m + in_g % rows;
  nt = in_g / rows;
}

}  // namespace clgrpo
