// NT-GEMM workgroup tile for gfx950 (CDNA4): C^[256 x 256] = A[256 x K] * B[256 x K]^T,
// both operands K-contiguous in memory, fp32 accumulation on the matrix cores.
//
// One workgroup of 2 x 2 wavefronts (64 lanes each, one per SIMD of a CU) owns a 256 x 256 tile; a wave
// owns 128 x 128 of it as 8 x 8 blocks of 16 x 16.  K is walked in slabs of 128 bytes per row (64 bf16 or 32
// fp32 elements), each slab in two halves of 64 bytes.
//
// What bounds it: on random operands the chip runs at its power limit (the shader clock settles at 1.5 -
// 1.6 GHz), so the rate is what is left after data movement and idle issue slots have taken their energy.
//  - 128 x 128 per wave reads 16 fragments per 64 matrix instructions; the 128 x 64 of eight waves read 12 per 32.
//  - v_mfma 16x16x32 against 32x32x16 on the same operands: 2 % more rate out of registers (1870 against 1827
//    TFLOP/s), 6 % in this loop.
//  - every instruction's place is fixed in the source: a fragment read of the next half after every second
//    matrix instruction, an operand load after every eighth (more often and the loads back up behind the
//    vector memory path, which takes a wave's kilobyte per 16 cycles, and the wave with them), scalar address
//    work one piece at a time in between.  With one wave per SIMD nothing else would fill a gap.
// Measured on operands of M = 4096, N = 12288, K = 32768 (bf16): 1493 TFLOP/s row-major, 1505 K-blocked; the
// eight-wave 32x32x16 form of this tile with two 64 KB stages ran 1310.
//
// Operand slabs travel HBM/L2 -> LDS directly (buffer loads with an LDS destination; no registers, no LDS
// store instructions) into two rings of 32 KB slots, three for A and two for B: all 160 KB.  While the matrix
// cores work on slab s, B(s+1) and A(s+1), A(s+2) land; a slot is requested again right after the barrier
// behind its last fragment read.  The third A slot is what makes the loads of a slab early enough: with two
// 64 KB stages (same loop) the row-major rate is 1398.  One barrier per slab, preceded by an explicit
// wait for this wave's own loads, because a barrier alone does not wait for loads whose destination is LDS; the
// youngest eight (the A slab after next) stay outstanding.
//
// A load fills LDS in lane order, so rows are 128 bytes apart with no padding; bank conflicts are
// avoided by an XOR swizzle of the 16-byte K-chunks within a row, applied on the global side of the load and
// undone by the fragment reads (0 conflict cycles).
//
// Operands are either row-major (the caller's hidden states and weight) or K-blocked (the library's own
// intermediates: per tile and slab one contiguous 32 KB piece, see Operand).  Consecutive tiles of a
// workgroup stream into each other: requests that run past a tile's last slab continue with the next
// tile's first ones, whose first fragments are in registers when the tile ends.
//
// Accumulators (v_mfma_f32_16x16x*): lane l = 16 g + c holds, in register r of block (i, j), the product of
//     A row a_row(i, 4 g + r)   and   B row b_row(j, c).
// Which rows of the wave's 128 make up a block is free, because it only decides where a fragment is read
// from.  a_row gives a lane VEC = 16 / sizeof(T) consecutive A rows (bf16: over a pair of blocks), b_row BV
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

// Kept logits: the forward leaves a chunk's raw logits for the backward in the K-blocked layout (rows =
// tokens, K = vocabulary) that the d(logits) operand will have, so that the kernel that turns one into the
// other works in place.  16-bit inputs keep their logits as IEEE half (10 mantissa bits against bf16's 7: the
// softmax the backward rebuilds from them is 8x closer to the fp32 one), fp32 inputs as fp32.
template <typename T> struct KeptLogit;
template <> struct KeptLogit<__bf16> { typedef _Float16 type; };
template <> struct KeptLogit<float> { typedef float type; };

// Matrix instructions of slot m (0 .. 63) of a slab half: 64 bytes of K of block (i, j) = (m / 8, m % 8), odd
// rows walked backwards so that neighbours share an operand.  Written as assembly because that is what ties the
// accumulators to the accumulation registers: left to itself the compiler moves all 256 of them between the
// register files around every loop, and spills what is in their way.  The compiler does not see the
// instruction's latency either: see settle().  Everything else that touches an accumulator goes through
// acc_get / acc_set for the same reason.
template <typename T> struct Mma;
template <> struct Mma<__bf16> {
  __device__ static __forceinline__ void slot(f32x4 (&acc)[8][8], const u32x4 (&a)[8], const u32x4 (&b)[8], int m) {
    const int i = m / 8, j = (i & 1) ? 7 - m % 8 : m % 8;
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(a[i]), "v"(b[j]));
  }
};
template <> struct Mma<float> {
  // 16 bytes hold four K=4 steps: lane group g, element e stands for k = 4g + e in both operands.  A slot takes
  // step m % 8 / 2 of four blocks of row i, so that an accumulator comes up again eight instructions later.
  __device__ static __forceinline__ void slot(f32x4 (&acc)[8][8], const u32x4 (&a)[8], const u32x4 (&b)[8], int m) {
    const int i = m / 8, e = m % 8 / 2;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int j = (m % 2) * 4 + k;
      asm volatile("v_mfma_f32_16x16x4_f32 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(a[i][e]), "v"(b[j][e]));
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

// BV: consecutive B rows a lane holds (see above), 8 or 4.
template <typename T, int BV>
struct GemmTile {
  static constexpr int BM = 256, BN = 256, WM = 128, WN = 128;
  static constexpr int MI = 8, NI = 8;                 // 16 x 16 blocks per wave along A / B
  static constexpr int kThreads = 256;
  static constexpr int kSlotBytes = 256 * kRowBytes;   // one operand's slab
  static constexpr int kASlots = 3, kBSlots = 2;
  static constexpr int kLdsBytes = (kASlots + kBSlots) * kSlotBytes;
  static constexpr int kSlabK = Elem<T>::kSlabK;
  static constexpr int VEC = 16 / (int)sizeof(T);      // elements per 16-byte piece
  static constexpr int kBB = kASlots * kSlotBytes;     // LDS offset of the B ring
  static_assert(BV == 8 || BV == 4, "B rows per lane");

  typedef f32x4 Acc[MI][NI];
  typedef __attribute__((address_space(3))) char lds_char;
  typedef __attribute__((address_space(3))) const u32x4 lds_vec;

  // This lane's rows within the wave's 128: a_row(i, r) of register r of blocks i, b_row(j) of blocks j.
  __device__ static __forceinline__ constexpr int a_block(int i) {
    return VEC == 8 ? (i >> 1) * 32 + (i & 1) * 4 : i * 16;
  }
  __device__ static __forceinline__ int a_lane(int rho) { return VEC == 8 ? (rho >> 2) * 8 + (rho & 3) : rho; }
  __device__ static __forceinline__ constexpr int b_block(int j) { return (j / BV) * 16 * BV + j % BV; }
  __device__ static __forceinline__ int lane_a0() {     // first A row of this lane (block 0, register 0)
    const int g = (threadIdx.x & 63) >> 4;
    return VEC == 8 ? g * 8 : g * 4;
  }
  __device__ static __forceinline__ int lane_b0() { return (threadIdx.x & 15) * BV; }
  __device__ static __forceinline__ int wave_m() { return ((threadIdx.x >> 6) & 1) * WM; }
  __device__ static __forceinline__ int wave_n() { return (threadIdx.x >> 7) * WN; }

  // Swizzle of LDS row R's chunks: eight rows that one fragment read takes together get eight values.
  __device__ static __forceinline__ int a_swz(int row) { return VEC == 8 ? (row & 3) | ((row >> 3) & 1) << 2 : row & 7; }
  __device__ static __forceinline__ int b_swz(int row) { return (BV == 8 ? row >> 3 : row >> 2) & 7; }

  // Where an operand's tile lives in memory: `rows` valid rows starting at `base`, consecutive
  // rows `row_bytes` apart, consecutive 128-byte K slabs of a row `slab_bytes` apart.
  //   row-major [rows][ld]:                  row_bytes = ld * sizeof(T), slab_bytes = 128
  //   K-blocked [row block][K slab][256][128 B]: row_bytes = 128, slab_bytes = 256 * 128 (one
  //   contiguous 32 KB piece per tile and slab)
  struct Operand {
    const T* base;
    int row_bytes;
    int slab_bytes;
    int rows;
    __device__ static __forceinline__ Operand row_major(const T* base, int64_t ld, int rows) {
      return Operand{base, (int)(ld * (int64_t)sizeof(T)), kRowBytes, rows};
    }
    __device__ static __forceinline__ Operand blocked(const T* block_base, int rows) {
      return Operand{block_base, kRowBytes, kBlockRows * kRowBytes, rows};
    }
  };

  // The next slab to request of one operand.  Loads go through range-checked buffer descriptors that cover
  // exactly the valid rows, so rows past them read as zero and nothing outside the operands is touched: the
  // row offset is in the per-lane part, which is what the hardware checks, the K-slab offset in the base
  // address, and the size is what is left of the valid rows from there.
  struct Cursor {
    const char* p;
    int bytes;
    int left;       // slabs of this tile from here on
  };

  int slab_a, slab_b, shrink_a, shrink_b;     // address step and size step per slab
  int pass_a;                                 // bytes between the rows of two loads of a slab
  Cursor a, b, next_a, next_b;
  lds_char* lds;
  __amdgpu_buffer_rsrc_t rsrc_a, rsrc_b;
  int voff_a, voff_b[8];
  u32x4 af[2][MI], bf[2][NI];
  uint32_t a0, b0;                            // this lane's fragment address in slot 0 of either ring
  uint32_t ra, rb, na, nb;                    // the same in the slab being read and in the one after it
  uint32_t da, db;                            // where the next requested slab goes
  uint32_t w0;

  __device__ static __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }
  __device__ __forceinline__ void make_a() {
    rsrc_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a.p), 0, a.bytes, 0x00020000);
  }
  __device__ __forceinline__ void make_b() {
    rsrc_b = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(b.p), 0, b.bytes, 0x00020000);
  }
  // Load p (0 .. 7) of the slab at the cursor: 8 rows per wave, 32 per workgroup.
  __device__ __forceinline__ void load_a(int p) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, lds + da + p * 4096, 16, voff_a + p * pass_a, 0, 0, 0);
  }
  __device__ __forceinline__ void load_b(int p) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, lds + db + p * 4096, 16, voff_b[p], 0, 0, 0);
  }
  __device__ __forceinline__ void step_a() { step_a1(); step_a2(); step_a3(); }
  // in pieces, to be placed between matrix instructions; masks, because a select would become a branch
  __device__ __forceinline__ void step_a1() { a.left -= 1; }
  __device__ __forceinline__ void step_a2() {
    const int64_t sw = -(int64_t)(a.left == 0);
    a.p += ((next_a.p - a.p) & sw) | (slab_a & ~sw);
  }
  __device__ __forceinline__ void step_a3() {
    const int sw = -(int)(a.left == 0);
    a.bytes += ((next_a.bytes - a.bytes) & sw) | (-shrink_a & ~sw);
    a.left |= next_a.left & sw;
  }
  __device__ __forceinline__ void step_b() { step_b1(); step_b2(); step_b3(); }
  // in pieces, to be placed between matrix instructions; masks, because a select would become a branch
  __device__ __forceinline__ void step_b1() { b.left -= 1; }
  __device__ __forceinline__ void step_b2() {
    const int64_t sw = -(int64_t)(b.left == 0);
    b.p += ((next_b.p - b.p) & sw) | (slab_b & ~sw);
  }
  __device__ __forceinline__ void step_b3() {
    const int sw = -(int)(b.left == 0);
    b.bytes += ((next_b.bytes - b.bytes) & sw) | (-shrink_b & ~sw);
    b.left |= next_b.left & sw;
  }
  __device__ __forceinline__ void slot_a() { const uint32_t t = da + kSlotBytes; da = t >= (uint32_t)kBB ? t - kBB : t; }
  __device__ __forceinline__ void slot_b() { db = 2 * (kBB + w0) + kSlotBytes - db; }
  // Fragment read n (0 .. 15) of a half: the first A fragment, all of B, the rest of A.
  __device__ __forceinline__ void read(int set, uint32_t pa, uint32_t pb, int n) {
    if (n == 0) af[set][0] = *(lds_vec*)(lds + pa);
    else if (n <= NI) bf[set][n - 1] = *(lds_vec*)(lds + pb + b_block(n - 1) * kRowBytes);
    else af[set][n - NI] = *(lds_vec*)(lds + pa + a_block(n - NI) * kRowBytes);
  }

  __device__ static __forceinline__ Cursor cursor(const Operand& o, int nslab) {
    return Cursor{reinterpret_cast<const char*>(o.base), o.rows * o.row_bytes, nslab};
  }
  // What the cursor does behind the last slab of the last tile: request that slab again.
  __device__ static __forceinline__ Cursor hold(const Operand& o, int nslab) {
    const int shrink = o.slab_bytes == kRowBytes ? kRowBytes : 0;
    return Cursor{reinterpret_cast<const char*>(o.base) + (int64_t)(nslab - 1) * o.slab_bytes,
                  o.rows * o.row_bytes - (nslab - 1) * shrink, 1};
  }

  // First tile of a workgroup (or of a run that does not stream): nothing is in flight, LDS is free.
  // b_order: row r of the B tile is row b_order[r] of B.base (B.rows: rows of the whole array; b_rows of them used).
  __device__ __forceinline__ void start(const Operand& A, const Operand& B, int nslab, char* shared,
                                        const int32_t* b_order = nullptr, int b_rows = 0) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    lds = (lds_char*)shared;
    slab_a = A.slab_bytes; slab_b = B.slab_bytes;
    shrink_a = A.slab_bytes == kRowBytes ? kRowBytes : 0;
    shrink_b = B.slab_bytes == kRowBytes ? kRowBytes : 0;
    pass_a = 32 * A.row_bytes;
    w0 = __builtin_amdgcn_readfirstlane(wave) * 1024;
    // A wave's load fills 1 KB of LDS in lane order: 8 rows x 8 chunks.  The lane that lands on (row, slot)
    // fetches chunk slot ^ swz(row); load p of a slab starts 32 p rows further down, which leaves a_swz as it is.
    const int row = wave * 8 + (lane >> 3), chunk = lane & 7;
    voff_a = row * A.row_bytes + (chunk ^ a_swz(row)) * 16;
#pragma unroll
    for (int p = 0; p < 8; ++p) {
      const int r = row + 32 * p;
      const int off = b_order == nullptr ? r * B.row_bytes : (r < b_rows ? b_order[r] * B.row_bytes : 0x7fffff00);
      voff_b[p] = off + (chunk ^ b_swz(r)) * 16;
    }
    const int g = lane >> 4, c = lane & 15;
    const int fa = a_lane(c), fb = c * BV;
    a0 = (wave_m() + fa) * kRowBytes + (g ^ a_swz(fa)) * 16;
    b0 = kBB + (wave_n() + fb) * kRowBytes + (g ^ b_swz(fb)) * 16;
    a = cursor(A, nslab); b = cursor(B, nslab);
    next_a = hold(A, nslab); next_b = hold(B, nslab);
    make_a(); make_b();
    da = w0; db = kBB + w0;
#pragma unroll
    for (int p = 0; p < 8; ++p) load_a(p);
#pragma unroll
    for (int p = 0; p < 8; ++p) load_b(p);
    step_a(); step_b(); make_a(); make_b(); slot_a(); slot_b();
#pragma unroll
    for (int p = 0; p < 8; ++p) load_a(p);
    step_a(); make_a(); slot_a();
    __builtin_amdgcn_s_waitcnt(0x0F78);    // all but the youngest eight loads
    __syncthreads();
    ra = a0; rb = b0; na = a0 + kSlotBytes; nb = b0 + kSlotBytes;
#pragma unroll
    for (int n = 0; n < 16; ++n) read(0, ra, rb, n);
#pragma unroll
    for (int p = 0; p < 8; ++p) load_b(p);
  }

  // One tile's K loop of `nslab` slabs; acc must be initialised by the caller.  Between tiles of a
  // streaming workgroup LDS stays in use; after the last one call finish() before touching it.
  __device__ __forceinline__ void run(Acc& acc, int nslab) {
    settle();
    for (int s = 0; s < nslab; ++s) {
      each<MI * NI>([&](auto c) __attribute__((always_inline)) {            // first half of the slab
        constexpr int m = decltype(c)::value;
        Mma<T>::slot(acc, af[0], bf[0], m);
        fence();
        if constexpr (m % 2 == 0 && m < 32) { read(1, ra ^ 64, rb ^ 64, m / 2); fence(); }
        if constexpr (m % 8 == 1) { load_a(m / 8); fence(); }
        if constexpr (m == 35) { step_b1(); fence(); }
        if constexpr (m == 37) { step_b2(); fence(); }
        if constexpr (m == 43) { step_b3(); fence(); }
        if constexpr (m == 45) { make_b(); fence(); }
        if constexpr (m == 47) { slot_b(); fence(); }
      });
      fence();
      // every wave has the last fragments of this slab, and the next one's loads have landed
      __builtin_amdgcn_s_waitcnt(0x0078);
      __builtin_amdgcn_s_barrier();
      fence();
      each<MI * NI>([&](auto c) __attribute__((always_inline)) {            // second half, while the next slab's first fragments come in
        constexpr int m = decltype(c)::value;
        Mma<T>::slot(acc, af[1], bf[1], m);
        fence();
        if constexpr (m % 2 == 0 && m < 32) { read(0, na, nb, m / 2); fence(); }
        if constexpr (m % 8 == 1) { load_b(m / 8); fence(); }
        if constexpr (m == 35) { step_a1(); fence(); }
        if constexpr (m == 37) { step_a2(); fence(); }
        if constexpr (m == 43) { step_a3(); fence(); }
        if constexpr (m == 45) { make_a(); fence(); }
        if constexpr (m == 47) { slot_a(); fence(); }
        if constexpr (m == 51) { ra = na; rb = nb; fence(); }
        if constexpr (m == 53) { const uint32_t t = na + kSlotBytes; na = t >= (uint32_t)kBB ? t - kBB : t; fence(); }
        if constexpr (m == 55) { nb = 2 * b0 + kSlotBytes - nb; fence(); }
      });
    }
    settle();
  }

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

constexpr int kHeadThreads = 256;
// The tile of the kernels that hold logits (A = vocabulary, B = tokens): a lane's 16-byte pieces run along either.
template <typename T> using LogitTile = GemmTile<T, 16 / (int)sizeof(T)>;

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
// 15.4 ms, no change for launches of one or two rounds.  Used by the forward only: the kernel that recomputes
// d(logits) tile by tile got 6 % slower with it, the plain GEMM launches moved by less than 1 % either way.
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
