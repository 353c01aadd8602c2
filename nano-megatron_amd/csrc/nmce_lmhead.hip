// Fused LM head + vocabulary-parallel cross entropy for gfx950.
//
// Replaces ParallelLMHead's projection Z = X @ W^T (nano_megatron/model.py:192,
// run in bf16 under autocast, model.py:255-257) followed by the loss of
// nano_megatron/cross_entropy.py:16-65, without ever storing Z: at most one
// chunk of tokens' bf16 exponentials (the caller's choice of chunk, up to every
// token), or one vocabulary chunk's gradient, at a time.
//
// Every product is one bf16 GEMM core, C[m, n] = sum_k A[m, k] * B[n, k] on
// v_mfma_f32_16x16x32_bf16, each operand K-contiguous or MN-contiguous
// (gemm_mainloop):
//
//   forward   Z^T = W X^T    (M = vocab, N = tokens, K = hidden). The epilogue
//             reduces each 128-row vocabulary block of a token's column to a
//             partial (max, sum exp, target logit); this statistics-only form
//             stores nothing of Z.
//   backward  per vocabulary chunk of Vc rows:
//             dZ^T_c = recompute(W_c X^T) -> (softmax - onehot) * g, bf16 [Vc,
//                      tokens] (and [tokens, Vc] for callers that form the
//                      products themselves)
//             dW_c   = dZ^T_c X      (M = Vc, N = hidden, K = tokens; B = X^T)
//             dX    += dZ_c W_c      (M = tokens, N = hidden, K = Vc; both read
//                                     vocabulary-row major, split over K when
//                                     the tiles are few)
//
// The one-pass path (the drop-in's default) computes Z once, per chunk of
// tokens (the caller's choice; the drop-in takes a quarter of the tokens, or all
// of them where that whole workspace is no larger):
//             P^T  = exp(W X^T - block max), bf16, with the partial statistics
//             dZ^T = P^T * exp(block max - M) * g / S - onehot, in place
//                    (once the statistics are combined)
//             dX   = dZ W            (K = vocab; dZ^T and W both read
//                                     vocabulary-row major, as they lie; split
//                                     over K when the chunk's tiles are few)
//             dW  += dZ^T X          (K = the chunk's tokens; both operands
//                                     K-contiguous: X_c^T, the chunk's hidden
//                                     rows transposed, H x chunk bf16, tens of
//                                     MB; fp32 across chunks only when there
//                                     are several)
// so 6 N V H flops in all, against 8 N V H for the recomputing backward, and
// no copy of anything the size of the logits or the weight.
//
// Tokens are the MFMA N dimension in the loss GEMMs: the 16x16 accumulators
// give each lane 32 vocabulary rows of each of 8 tokens, so the per-token
// reductions are mostly in-register, with one merge over four lane groups.
//
// Main loop: a 256x256 output tile per 256-lane workgroup (four waves, 2x2,
// one per SIMD, each 128x128 = 64 accumulators of 16x16 held in AGPRs), K in
// steps of 64. Each wave reads its next fragments from LDS under the MFMAs of
// the current ones (two register sets), and the reads and the next stages'
// loads have fixed places between the MFMAs. Operand tiles move HBM/L2 -> LDS
// with 16-byte direct-to-LDS loads (MUBUF buffer_load_dwordx4 ... lds, no VGPR
// staging), A triple- and B double-buffered. A K-contiguous operand sits in
// rows of 128 bytes with the 16-byte chunks XOR-swizzled by ((row >> 1) & 7).
// gfx950's LDS has 64 banks, so a ds_read_b128 serves 16 lanes (16 consecutive
// rows of a fragment) per cycle; this swizzle puts those 16 rows on 16 distinct
// 16-byte bank groups (row parity picks the half of the banks, the swizzled
// chunk the group). An MN-contiguous operand sits in 64 k-rows of 512 bytes
// and its fragments come from gfx950's transposing LDS read,
// ds_read_b64_tr_b16, with the same fragments, so the two layouts give the
// same bits. Workgroups are mapped to tiles so that each XCD (one L2) owns a
// contiguous band of tiles walked in groups that share operands.
//
// The dZ epilogue stages the bf16 tile in the freed LDS with the token index
// XOR-swizzled by the vocabulary pair, so that both output layouts leave as
// coalesced 512-byte row segments.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <type_traits>

#include "nmce.h"
#include "nmce_device.h"

namespace nmce {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void_t;

constexpr int kBM = 256;          // tile rows (GEMM M)
constexpr int kBN = 256;          // tile columns (GEMM N)
constexpr int kBK = 64;           // K per stage (128 bytes of bf16 per row)
// Four waves, one per SIMD, each 128 x 128 of the tile (2 x 2). Against eight
// waves of 128 x 64 (two per SIMD) a wave reads a third less from LDS per
// product, and that and the smaller MFMA (below) are what a chip at its power
// cap turns into clock: 1190 -> 1525 TFLOP/s on 16384 x 16384 x 8192, 1175 ->
// 1538 on 4096 x 4096 x 65536.
constexpr int kWavesM = 2;
constexpr int kWavesN = 2;
constexpr int kWaves = kWavesM * kWavesN;
constexpr int kThreads = 64 * kWaves;
constexpr int kWaveM = kBM / kWavesM;  // 128
constexpr int kWaveN = kBN / kWavesN;  // 128
constexpr int kF = kWaveM / 16;        // 8 fragments of 16 rows (columns) a side
static_assert(kWaveM == kWaveN, "a wave's tile is square");
constexpr int kStage = kBM * kBK * 2;  // bytes of one operand's stage: 32 KiB
static_assert(kBM == kBN, "the operands' stages have one size");
// A's stages in three buffers, B's in two: all of a compute unit's LDS. A
// stage's A loads are then issued before the barrier that frees B's buffer,
// which spreads a stage's loads over the whole K step (gemm_mainloop).
constexpr int kBufsA = 3;
constexpr int kBufsB = 2;
constexpr int kLdsBytes = (kBufsA + kBufsB) * kStage;  // dynamic LDS: 160 KiB
static_assert(kLdsBytes <= 160 * 1024, "the stages fit a compute unit's LDS");
// 1 KiB LDS blocks per stage and operand, and per wave of them.
constexpr int kBlocks = kStage / 1024;
constexpr int kBlocksPerWave = kBlocks / kWaves;
// Tile rows per raster group inside an XCD band: 4 of 2, 4 and 8 is the
// fastest for the products of many tiles (16384 x 16384 x 8192: 1545 TFLOP/s
// against 1476 with 8; the [16384, 4096] x [128256, 4096] step 39.3 ms against
// 39.6 with 8 and 39.9 with 2) and no slower than 1.5% elsewhere.
constexpr int kGroupM = 4;
constexpr int kXcds = 8;
constexpr float kMaxFloorL = -1.0e38f;

// Partial statistics cover this many vocabulary rows (one wave's rows).
constexpr int kPartialRows = kWaveM;

// A wave's 128 x 128 results: c[i][j] is the 16 x 16 block of rows 16 i and
// columns 16 j; lane l holds column l % 16, rows 4 (l / 16) + e of it, or,
// from a main loop with kRows, row l % 16, columns 4 (l / 16) + e.
struct Acc {
  f32x4_t c[kF][kF];
};

// acc += A B^T of one 16 x 16 block, K = 32, as an instruction that updates
// its accumulator registers in place. With the builtin the compiler gives 64
// accumulators results in other registers than their inputs and moves them
// back (360 moves per K step, 1055-1200 instead of 1440 TFLOP/s). The 16 x 16
// form moves half the accumulator bytes per product that the 32 x 32 x 16 form
// does, with the same sums: 1440 against 1240 TFLOP/s in the same loop.
// The compiler puts no wait states around an instruction that it does not know
// for an MFMA: its fragments come from LDS reads, whose waits it counts, and
// nothing else touches the accumulators within the loop (gemm_mainloop waits
// before the first and after the last; a test looks at the generated code).
__device__ __forceinline__ void mfma_16x16x32(f32x4_t& c, const bf16x8_t& a, const bf16x8_t& b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

// Tile index for workgroup b. The dispatcher deals workgroups to the 8 XCDs
// round-robin (block b runs on XCD b % 8); give each XCD a contiguous band of
// tile ids, and inside the band walk groups of kGroupM tile rows column by
// column, so the tiles that run together on one L2 share A and B stripes.
__device__ __forceinline__ void tile_coords(int b, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int total = tiles_m * tiles_n;
  const int xcd = b % kXcds;
  const int q = total / kXcds, r = total % kXcds;
  const int tid = xcd * q + (xcd < r ? xcd : r) + b / kXcds;
  const int group = kGroupM * tiles_n;
  const int g = tid / group;
  const int first_m = g * kGroupM;
  const int gm = (tiles_m - first_m) < kGroupM ? (tiles_m - first_m) : kGroupM;
  const int in_g = tid - g * group;
  tm = first_m + in_g % gm;
  tn = in_g / gm;
}

// The loads of one operand's stages (64 k each) into LDS by this wave: 1 KiB
// blocks blk0 .. blk0 + 7, one MUBUF direct-to-LDS load each.
//
// K-contiguous (kMN = false): a block is 8 rows of 128 bytes; lane p writes
// row p / 8, physical chunk p % 8, which holds logical chunk
// (p % 8) ^ ((row >> 1) & 7). The K position goes in the scalar offset, so a
// stage needs no per-lane arithmetic. MN-contiguous: a block is k-rows 2 b and
// 2 b + 1 of 512 bytes; lane p writes row 2 b + p / 32, physical chunk p % 32,
// which holds logical chunk (p % 32) ^ 4 (row & 3) ^ 2 ((row >> 3) & 1). The
// resource's base moves by 64 rows per stage (the offset would pass 32 bits).
//
// The buffer resource has no stride and no range limit (every offset is
// clamped in bounds) and gfx9's data format word.
template <bool kMN>
struct StageLoads {
  i32x4_t rsrc;
  const char* base;
  int64_t row_bytes, krows;
  uint32_t off[kBlocksPerWave];
  int row0, last_chunk, lane, soff;

  __device__ __forceinline__ void set_base(const char* p) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    rsrc[0] = __builtin_amdgcn_readfirstlane(static_cast<int>(a & 0xffffffffu));
    rsrc[1] = __builtin_amdgcn_readfirstlane(static_cast<int>(a >> 32));
  }
  __device__ __forceinline__ int krow(int j) const { return row0 + 2 * j; }
  __device__ __forceinline__ int chunk_bytes(int j) const {
    int chunk = (lane & 31) ^ (4 * (krow(j) & 3)) ^ (2 * ((krow(j) >> 3) & 1));
    if (chunk > last_chunk) chunk = last_chunk;
    return chunk * 16;
  }
  // first: the operand's element at the tile's first row (column), k = 0;
  // rows: the operand's rows (columns) from there on; krows_: its k-rows (kMN).
  __device__ __forceinline__ void init(const uint16_t* first, int64_t ld, int64_t rows,
                                       int64_t krows_, int wave, int lane_) {
    lane = lane_;
    base = reinterpret_cast<const char*>(first);
    row_bytes = ld * 2;
    krows = krows_;
    soff = 0;
    const int blk0 = wave * kBlocksPerWave;
    if constexpr (kMN) {
      row0 = 2 * blk0 + (lane >> 5);
      const int64_t last = (rows + 7) / 8 - 1;  // >= 0
      last_chunk = static_cast<int>(last < 31 ? last : 31);
#pragma unroll
      for (int j = 0; j < kBlocksPerWave; ++j)
        off[j] = static_cast<uint32_t>(krow(j) * row_bytes + chunk_bytes(j));
    } else {
#pragma unroll
      for (int j = 0; j < kBlocksPerWave; ++j) {
        const int tile_row = (blk0 + j) * 8 + (lane >> 3);
        const int chunk = (lane & 7) ^ ((tile_row >> 1) & 7);
        const int64_t r = tile_row < rows ? tile_row : rows - 1;
        off[j] = static_cast<uint32_t>(r * row_bytes + chunk * 16);
      }
    }
    set_base(base);
    rsrc[2] = -1;
    rsrc[3] = 0x00020000;
  }
  // The number of leading stages whose k-rows all exist.
  __device__ __forceinline__ int full_stages(int stages) const {
    if constexpr (!kMN) return stages;
    const int64_t f = krows / kBK;
    return f < stages ? static_cast<int>(f) : stages;
  }
  // Stage kt (all of its k-rows exist) is the next one to be loaded.
  __device__ __forceinline__ void at(int kt) {
    if constexpr (kMN)
      set_base(base + kt * (kBK * row_bytes));
    else
      soff = __builtin_amdgcn_readfirstlane(kt * (kBK * 2));
  }
  __device__ __forceinline__ void load(char* dst, int j) const {
    raw_buffer_load_lds(rsrc, (lds_void_t*)(dst + j * 1024), 16, static_cast<int>(off[j]), soff, 0,
                        0);
  }
  // A whole stage at once, whose k-rows may end before it does (kMN): those
  // past the last are read as the last.
  __device__ __forceinline__ void stage(char* dst, int kt) {
    const int64_t k0 = static_cast<int64_t>(kt) * kBK;
    if (kMN && k0 + kBK > krows) {
      const int64_t b0 = k0 < krows ? k0 : krows - 1;
      set_base(base + b0 * row_bytes);
#pragma unroll
      for (int j = 0; j < kBlocksPerWave; ++j) {
        int64_t row = k0 + krow(j);
        if (row > krows - 1) row = krows - 1;
        raw_buffer_load_lds(rsrc, (lds_void_t*)(dst + j * 1024), 16,
                            static_cast<int>((row - b0) * row_bytes) + chunk_bytes(j), 0, 0, 0);
      }
      return;
    }
    at(kt);
#pragma unroll
    for (int j = 0; j < kBlocksPerWave; ++j) load(dst, j);
  }
};

// One operand's fragments of 16 rows (columns) and 32 k from its stage: lane l
// gets row l % 16, k 8 (l / 16) .. + 7. K-contiguous: one ds_read_b128 of the
// row's logical chunk 4 s + l / 16 (sub-step s); 16 consecutive rows of one
// chunk are on distinct 16-byte bank groups. MN-contiguous: two
// ds_read_b64_tr_b16, each giving a lane 4 consecutive k of its column (in a
// group of 16 lanes, lanes 4 r .. 4 r + 3 read the 16 columns of k-row r and
// lane j receives column j of the 4 rows). Lane 16 g + 4 r + u reads k-row
// 8 g + r (+ 4 for the second, + 32 s), columns 4 u .. 4 u + 3 of the
// fragment; the swizzle puts the 8 k-rows that half of the lanes read (rows
// 0-3 and 8-11) on distinct 32 bytes of the 256 that the banks span.
template <bool kMN>
struct Frags {
  int off0, off1;  // K-contiguous: the lane's byte offset in sub-step 0 and 1
  int lane;
  int col0;        // first row (column) of the wave's 128

  __device__ __forceinline__ void init(int first, int lane_) {
    lane = lane_;
    col0 = first;
    const int r = lane & 15, q = lane >> 4;
    off0 = (first + r) * 128 + ((q ^ ((r >> 1) & 7)) << 4);
    off1 = (first + r) * 128 + (((4 + q) ^ ((r >> 1) & 7)) << 4);
  }
  // K-contiguous: the whole fragment f of sub-step s.
  __device__ __forceinline__ bf16x8_t read(const char* st, int s, int f) const {
    return *reinterpret_cast<const bf16x8_t*>(st + (s ? off1 : off0) + f * 16 * 128);
  }
  // MN-contiguous: its half h (k 4 h .. 4 h + 3 of the lane's eight).
  __device__ __forceinline__ s16x4_t read_half(const char* st, int s, int f, int h) const {
    const int g = lane >> 4, r = (lane >> 2) & 3, u = lane & 3;
    // k-rows 8 g + r and 8 g + 4 + r share the swizzle (row & 3 = r,
    // (row >> 3) & 1 = g & 1); 32 s does not change it either.
    const int chunk = (((col0 + 16 * f) >> 3) + (u >> 1)) ^ (4 * r) ^ (2 * (g & 1));
    const char* p = st + (8 * g + r) * 512 + chunk * 16 + 8 * (u & 1) + s * (32 * 512);
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4_t*)(p + h * (4 * 512)));
  }
  static __device__ __forceinline__ bf16x8_t join(const s16x4_t& lo, const s16x4_t& hi) {
    typedef short s16x8_t __attribute__((ext_vector_type(8)));
    const s16x8_t v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8_t, v);
  }
};

// The main loop: acc = A[m0:m0+256, 0:K] * B[n0:n0+256, 0:K]^T, each operand
// K-contiguous (A[m, k] at A + m * lda + k; kAMN = false) or MN-contiguous
// (A[m, k] at A + k * lda + m; kAMN = true), and B likewise.
// K-contiguous operands: rows >= M (N) are read from the last valid row; their
// results are masked by the epilogues. MN-contiguous operands: columns are
// read in 8-element chunks up to the one holding column M - 1 (N - 1), so the
// rows must be allocated to a multiple of 8 elements past it; later chunks
// repeat that one. An MN-contiguous operand may hold fewer k-rows than K
// (ka_rows, kb_rows): k-rows past its last are read as its last, so the other
// operand must hold zeros there. Requires K % 64 == 0, lda and ldb multiples of 8 elements,
// 16-byte aligned A and B, and 256 * ld * 2 < 2^32 bytes (K-contiguous) or
// 64 * ld * 2 < 2^32 bytes (MN-contiguous).
//
// A K step is two sub-steps of 32 k, 64 MFMAs each. One wave per SIMD has
// nothing else to hide a wait, so the stream is fixed: after every third MFMA
// one fragment of the next sub-step is read from LDS (the 16 reads are done
// by the 48th of 64 MFMAs, so none is waited for), and after every sixth one
// of the stage's 16 loads is issued (issued together they fill the address
// unit's queue and the wave stalls: 1370 against 1450 TFLOP/s with one every
// second MFMA, 1525 spread over both sub-steps, on 16384 x 16384 x 8192).
// Stage kt + 2's A goes into the buffer that stage kt - 1 had, during the first
// sub-step of kt; its B into stage kt's buffer, after the barrier at which every
// wave has read the last of stage kt. That barrier waits for all but the wave's
// newest eight loads (stage kt + 2's A).
//
// kRows hands the MFMA its operands the other way round, which gives the lane
// four columns of one row instead of four rows of one column (the same sums):
// what an epilogue wants that stores rows.
template <bool kAMN, bool kBMN, bool kRows = false>
__device__ __forceinline__ void gemm_mainloop(const uint16_t* __restrict__ A, int64_t lda,
                                              int64_t M, const uint16_t* __restrict__ B,
                                              int64_t ldb, int64_t N, int64_t K, int64_t m0,
                                              int64_t n0, char* lds, Acc& acc,
                                              int64_t ka_rows = 0, int64_t kb_rows = 0) {
  const int lane = threadIdx.x & 63;
  // The wave index is uniform across the wave; say so, so that the load
  // bases and LDS destinations below live in scalar registers.
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / kWavesN, wn = wave % kWavesN;

  StageLoads<kAMN> la;
  StageLoads<kBMN> lb;
  la.init(kAMN ? A + m0 : A + m0 * lda, lda, M - m0, ka_rows, wave, lane);
  lb.init(kBMN ? B + n0 : B + n0 * ldb, ldb, N - n0, kb_rows, wave, lane);
  Frags<kAMN> fa;
  Frags<kBMN> fb;
  fa.init(wm * kWaveM, lane);
  fb.init(wn * kWaveN, lane);

  char* const lds_b = lds + kBufsA * kStage;
  const int lds_w = wave * (kBlocksPerWave * 1024);
  const int kt_n = static_cast<int>(K / kBK);

  la.stage(lds + lds_w, 0);
  lb.stage(lds_b + lds_w, 0);
  if (kt_n > 1) {
    la.stage(lds + kStage + lds_w, 1);
    lb.stage(lds_b + kStage + lds_w, 1);
  }
#pragma unroll
  for (int i = 0; i < kF; ++i)
#pragma unroll
    for (int j = 0; j < kF; ++j) acc.c[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  // The compiler does not know that mfma_16x16x32 reads them as an MFMA does:
  // the zeros are written, and have settled, before the first one.
#pragma unroll
  for (int i = 0; i < kF; ++i)
#pragma unroll
    for (int j = 0; j < kF; ++j) asm volatile("" : "+a"(acc.c[i][j]));
  asm volatile("s_nop 7" ::: "memory");
  // Stage 0 is what the first reads need; the compiler puts a wait for nearly
  // all loads in flight before the barrier of its own accord, stage 1's among
  // them.
  if (kt_n > 1)
    asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
  else
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  struct Set {
    bf16x8_t a[kF], b[kF];
  };
  // Fragment q of a sub-step in the order the MFMAs first use them, b0 a0 b1
  // a1 ...: part 1 completes it, part 0 reads a transposed one's first half.
  s16x4_t half;
  auto read = [&](const char* pa, const char* pb, int s, Set& f, int q, int part) {
    if (q & 1) {
      if constexpr (!kAMN) {
        if (part == 1) f.a[q >> 1] = fa.read(pa, s, q >> 1);
      } else if (part == 0) {
        half = fa.read_half(pa, s, q >> 1, 0);
      } else {
        f.a[q >> 1] = fa.join(half, fa.read_half(pa, s, q >> 1, 1));
      }
    } else {
      if constexpr (!kBMN) {
        if (part == 1) f.b[q >> 1] = fb.read(pb, s, q >> 1);
      } else if (part == 0) {
        half = fb.read_half(pb, s, q >> 1, 0);
      } else {
        f.b[q >> 1] = fb.join(half, fb.read_half(pb, s, q >> 1, 1));
      }
    }
  };
  // One sub-step: the 64 MFMAs of `cur`, the 16 fragment reads of the next
  // sub-step after every third of them (a transposed fragment's two halves
  // after the second and the third), and kLoads loads, six MFMAs apart, after
  // MFMAs that no read follows: an MFMA's 16 cycles hide about three other
  // instructions.
  constexpr int kLoadGap = 6;
  auto mma = [&](int i, int j, const Set& f) {
    if constexpr (kRows)
      mfma_16x16x32(acc.c[i][j], f.b[j], f.a[i]);
    else
      mfma_16x16x32(acc.c[i][j], f.a[i], f.b[j]);
  };
  auto step = [&](const char* pa, const char* pb, int s, Set& next, const Set& cur, auto loads,
                  auto&& load) {
    constexpr int kLoads = decltype(loads)::value;
#pragma unroll
    for (int x = 0; x < kF * kF; ++x) {
      const int i = x / kF, j = (i & 1) ? kF - 1 - x % kF : x % kF;
      mma(i, j, cur);
      if (x % 3 != 0 && x / 3 < 2 * kF) read(pa, pb, s, next, x / 3, x % 3 - 1);
      if (x % kLoadGap == 0 && x / kLoadGap < kLoads) load(x / kLoadGap);
      if (kAMN || kBMN || x % 3 == 2) __builtin_amdgcn_sched_barrier(0);
    }
  };
  using NoLoads = std::integral_constant<int, 0>;
  using Loads = std::integral_constant<int, kBlocksPerWave>;
  auto none = [](int) {};

  Set f0, f1;
#pragma unroll
  for (int q = 0; q < 2 * kF; ++q) {
    read(lds, lds_b, 0, f0, q, 0);
    read(lds, lds_b, 0, f0, q, 1);
  }
  int a_cur = 0;               // byte offset of stage kt's A buffer
  auto next_a = [](int o) { return o == (kBufsA - 1) * kStage ? 0 : o + kStage; };
  auto prev_a = [](int o) { return o == 0 ? (kBufsA - 1) * kStage : o - kStage; };
  // Stages [0, full) have all their k-rows: their loads run inside the
  // sub-steps. The last one or two steps load with clamped rows, or nothing.
  const int full_a = la.full_stages(kt_n), full_b = lb.full_stages(kt_n);
  const int full = full_a < full_b ? full_a : full_b;
  int kt = 0;
  for (; kt + 2 < full; ++kt) {
    const int a_nxt = next_a(a_cur);
    const int b_cur = (kt & 1) * kStage;
    char* da = lds + prev_a(a_cur) + lds_w;
    la.at(kt + 2);
    step(lds + a_cur, lds_b + b_cur, 1, f1, f0, Loads{}, [&](int l) { la.load(da, l); });
    asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    char* db = lds_b + b_cur + lds_w;
    lb.at(kt + 2);
    step(lds + a_nxt, lds_b + (kStage - b_cur), 0, f0, f1, Loads{},
         [&](int l) { lb.load(db, l); });
    a_cur = a_nxt;
  }
  static_assert(kBlocksPerWave == 8, "the loop's wait leaves one stage's A loads in flight");
  for (; kt + 1 < kt_n; ++kt) {
    const int a_nxt = next_a(a_cur);
    const int b_cur = (kt & 1) * kStage;
    if (kt + 2 < kt_n) la.stage(lds + prev_a(a_cur) + lds_w, kt + 2);
    step(lds + a_cur, lds_b + b_cur, 1, f1, f0, NoLoads{}, none);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (kt + 2 < kt_n) lb.stage(lds_b + b_cur + lds_w, kt + 2);
    step(lds + a_nxt, lds_b + (kStage - b_cur), 0, f0, f1, NoLoads{}, none);
    a_cur = a_nxt;
  }
  step(lds + a_cur, lds_b + (kt & 1) * kStage, 1, f1, f0, NoLoads{}, none);
#pragma unroll
  for (int x = 0; x < kF * kF; ++x) mma(x / kF, x % kF, f1);
  // The compiler does not know the MFMAs' latency: let the last ones finish
  // before anything reads the accumulators.
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int i = 0; i < kF; ++i)
#pragma unroll
    for (int j = 0; j < kF; ++j) asm volatile("" : "+a"(acc.c[i][j]));
}

// Row (within the wave's 128 rows) of accumulator row block i, element e, for
// a lane in 16-lane group g: the 16x16 result gives lane l column l % 16 and
// rows 4 (l / 16) + e.
__device__ __forceinline__ int acc_row(int i, int e, int g) { return 16 * i + 4 * g + e; }

// The epilogues stage a 256 x 256 bf16 tile in LDS as words of two rows: word
// (vp, c) at vp * kBN + (c ^ stage_swz(vp)) holds rows 2 vp and 2 vp + 1 of
// column c. The swizzle keeps groups of 4 columns together (16-byte reads).
// Its bits 4 and 5 take vp's bits 1 and 2, so that the four row groups of a
// 16x16 block (lanes 16 g ..: vp = 8 i + 2 g) are written to the four 16-bank
// groups; bits 2, 3 and (again) 4 take vp's bits 3, 4 and 5, so that one
// column read at every fourth vp (lmhead_dz_kernel) spreads over 16 of the 64
// banks, two rows to a bank.
__device__ __forceinline__ int stage_swz(int vp) {
  return ((((vp >> 1) ^ (vp >> 5)) & 1) << 4) | (((vp >> 2) & 1) << 5) | (((vp >> 3) & 3) << 2);
}

// Word of rows 16 i + 4 g + 2 h, + 1 (of wave row wm) and tile column c.
__device__ __forceinline__ uint32_t* stage_word(uint32_t* P, int wm, int i, int g, int h, int c) {
  // stage_swz(64 wm + 8 i + 2 g + h), the lane's part and the block's apart.
  const int lane_swz = ((g & 1) << 4) | ((g >> 1) << 5);
  const int block_swz = ((i & 3) << 2) | ((i >> 2) << 4);
  return P + (wm * (kWaveM / 2) + 2 * g) * kBN + (8 * i + h) * kBN + ((c ^ lane_swz) ^ block_swz);
}

// 8 columns t0 .. t0 + 7 of staged rows 2 vp (lo) and 2 vp + 1 (hi), bf16.
__device__ __forceinline__ void staged_rows(const uint32_t* P, int vp, int t0, u32x4& lo,
                                            u32x4& hi) {
  const int swz = stage_swz(vp);
  const u32x4 a = *reinterpret_cast<const u32x4*>(P + vp * kBN + (t0 ^ swz));
  const u32x4 b = *reinterpret_cast<const u32x4*>(P + vp * kBN + ((t0 + 4) ^ swz));
  lo = u32x4{(a.x & 0xffffu) | (a.y << 16), (a.z & 0xffffu) | (a.w << 16),
             (b.x & 0xffffu) | (b.y << 16), (b.z & 0xffffu) | (b.w << 16)};
  hi = u32x4{(a.x >> 16) | (a.y & 0xffff0000u), (a.z >> 16) | (a.w & 0xffff0000u),
             (b.x >> 16) | (b.y & 0xffff0000u), (b.z >> 16) | (b.w & 0xffff0000u)};
}
// The staged tile leaves 32 lanes to a pair of rows, 8 columns a lane.
constexpr int kStagedIters = (kBM / 2) * (kBN / 8) / kThreads;

// max(a, b, c) as one v_max3_f32 (two IEEE maxNum steps: a quiet NaN operand
// is ignored). fmaxf gives the same value, but the compiler quiets every
// operand it cannot prove canonical with a v_max_f32 x, x first, which for
// MFMA results (never signalling NaNs) only costs issue slots.
__device__ __forceinline__ float max3_hw(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// mask ? a : b, bit by bit, as one v_bfi_b32. Kept opaque: written as a
// select between two accumulator elements, the compiler turns it into a load
// at a computed index, which puts the accumulators in scratch memory.
__device__ __forceinline__ float bit_select(uint32_t mask, float a, float b) {
  float r;
  asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(r) : "v"(mask), "v"(a), "v"(b));
  return r;
}

// Merge of a value over the four 16-lane groups of a wave (the lanes that hold
// one column's rows), every lane getting the result: lanes 16-31 against 0-15
// and 48-63 against 32-47, then the halves, by gfx950's row and half swaps.
template <typename Op>
__device__ __forceinline__ float merge_groups(float v, Op op) {
  typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
  const uint32_t w = __float_as_uint(v);
  const auto r16 = __builtin_amdgcn_permlane16_swap(w, w, false, false);
  const float x = op(__uint_as_float(r16[0]), __uint_as_float(r16[1]));
  const uint32_t u = __float_as_uint(x);
  const auto r32 = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return op(__uint_as_float(r32[0]), __uint_as_float(r32[1]));
}
__device__ __forceinline__ float max_op(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ float add_op(float a, float b) { return a + b; }

// One column's statistics over the wave's 128 rows.
struct ColumnStats {
  float max, sum_m1, pick;
};

// The per-token statistics of kCols columns j0 .. of the wave's results
// (Z^T: rows are vocabulary rows, columns tokens): maximum, sum exp(z - max)
// - 1 and the target row's z (0 when tl[.] < 0, the target row within the
// wave's rows otherwise), over the rows < valid_rows (kFull: all 128). The
// terms of the sum that equal 1 (the maximum and its ties) are counted apart:
// fract zeroes exactly those, so the maximum's 1 never enters a rounded sum
// with the small terms. `keep(jj, i, p)` gets the four exponentials of row
// block i of column j0 + jj (0 for rows past valid_rows).
//
// VALU work with the MFMA pipe idle, at every tile, so full tiles drop the
// per-element row masks, take the maximum two values per v_max3_f32, and find
// the target's element by a select tree on its row, only where a lane of the
// wave has one (the wave's 128 rows of V hold few of its tokens' targets).
// Both forms give the same bits. The columns go together so that their
// merges' latencies overlap.
template <int kCols, bool kFull, typename Keep>
__device__ __forceinline__ void column_stats(const Acc& acc, int j0, int g, int valid_rows,
                                             const int* tl, ColumnStats* out, Keep&& keep) {
  float mx[kCols];
#pragma unroll
  for (int jj = 0; jj < kCols; ++jj) {
    mx[jj] = kMaxFloorL;
#pragma unroll
    for (int i = 0; i < kF; ++i) {
      const f32x4_t z = acc.c[i][j0 + jj];
      if constexpr (kFull) {
        mx[jj] = max3_hw(max3_hw(mx[jj], z[0], z[1]), z[2], z[3]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (acc_row(i, e, g) < valid_rows) mx[jj] = fmaxf(mx[jj], z[e]);
      }
    }
  }
#pragma unroll
  for (int jj = 0; jj < kCols; ++jj) mx[jj] = merge_groups(mx[jj], max_op);
#pragma unroll
  for (int jj = 0; jj < kCols; ++jj) {
    float pick = 0.0f;
    if (__builtin_amdgcn_ballot_w64(tl[jj] >= 0)) {
      // Element (i, e) of row 16 i + 4 g + e: a tree on the row's bits 0, 1,
      // 4, 5 and 6, then the lane group that holds bits 2 and 3.
      const int row = tl[jj];
      const uint32_t m0 = 0u - (row & 1), m1 = 0u - ((row >> 1) & 1);
      const uint32_t m4 = 0u - ((row >> 4) & 1), m5 = 0u - ((row >> 5) & 1);
      const uint32_t m6 = 0u - ((row >> 6) & 1);
      float b[kF];
#pragma unroll
      for (int i = 0; i < kF; ++i) {
        const f32x4_t z = acc.c[i][j0 + jj];
        b[i] = bit_select(m1, bit_select(m0, z[3], z[2]), bit_select(m0, z[1], z[0]));
      }
      const float c0 = bit_select(m4, b[1], b[0]), c1 = bit_select(m4, b[3], b[2]);
      const float c2 = bit_select(m4, b[5], b[4]), c3 = bit_select(m4, b[7], b[6]);
      const float z = bit_select(m6, bit_select(m5, c3, c2), bit_select(m5, c1, c0));
      pick = merge_groups((row >= 0 && ((row >> 2) & 3) == g) ? z : 0.0f, add_op);
    }
    out[jj].pick = pick;
  }
  float se[kCols], sr[kCols];
#pragma unroll
  for (int jj = 0; jj < kCols; ++jj) {
    se[jj] = sr[jj] = 0.0f;
#pragma unroll
    for (int i = 0; i < kF; ++i) {
      const f32x4_t z = acc.c[i][j0 + jj];
      float p[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        p[e] = (kFull || acc_row(i, e, g) < valid_rows) ? exp_shift(z[e], mx[jj]) : 0.0f;
        se[jj] += p[e];
        sr[jj] += __builtin_amdgcn_fractf(p[e]);
      }
      keep(jj, i, p);
    }
  }
#pragma unroll
  for (int jj = 0; jj < kCols; ++jj) {
    const float e = merge_groups(se[jj], add_op), r = merge_groups(sr[jj], add_op);
    const float ones = rintf(e - r);  // at least the maximum's own 1
    out[jj].max = mx[jj];
    out[jj].sum_m1 = (ones - 1.0f) + r;
  }
}

// Columns whose statistics are formed together: two columns' 64 values and
// their exponentials beside the 256 accumulators take all 512 registers, and the
// compiler spills one or two more (8 bytes of scratch a lane in lmhead_p_kernel,
// 12 in lmhead_stats_kernel).
constexpr int kStatCols = 2;

// The partial statistics of the wave's 128 rows x 128 tokens, written for the
// rows' 128-row block: pmax[blk * N + t], psum1[blk * N + t] and ptgt[blk * N +
// t]. `keep(j, i, p)` as in column_stats, with the column block's index.
template <typename Keep>
__device__ __forceinline__ void wave_stats(const Acc& acc, int64_t vrow0, int64_t V, int64_t tok0,
                                           int64_t N, const int64_t* __restrict__ target,
                                           int64_t vstart, float* __restrict__ pmax,
                                           float* __restrict__ psum1, float* __restrict__ ptgt,
                                           int lane, Keep&& keep) {
  const int g = lane >> 4;
  const int64_t blk = vrow0 / kPartialRows;
  const int64_t vr = V - vrow0;
  // rows >= valid_rows of this wave's 128 are padding (possibly all of them)
  const int valid_rows = static_cast<int>(vr < 0 ? 0 : (vr < kWaveM ? vr : kWaveM));
  auto columns = [&](auto full_tag, int j0) {
    constexpr bool kFull = decltype(full_tag)::value;
    int tl[kStatCols];
    ColumnStats st[kStatCols];
#pragma unroll
    for (int jj = 0; jj < kStatCols; ++jj) {
      const int64_t tok = tok0 + 16 * (j0 + jj) + (lane & 15);
      tl[jj] = -1;  // target row within this wave's valid rows, or -1
      if (kFull || tok < N) {
        // Rows past the shard's end pad the last block (they repeat its last
        // row); a target there belongs to the next shard and picks nothing.
        const int64_t t = target[tok] - vstart - vrow0;
        tl[jj] = (t >= 0 && t < valid_rows) ? static_cast<int>(t) : -1;
      }
    }
    column_stats<kStatCols, kFull>(acc, j0, g, valid_rows, tl, st, [&](int jj, int i, float* p) {
      if (!kFull && tok0 + 16 * (j0 + jj) + (lane & 15) >= N) p[0] = p[1] = p[2] = p[3] = 0.0f;
      keep(j0 + jj, i, p);
    });
#pragma unroll
    for (int jj = 0; jj < kStatCols; ++jj) {
      const int64_t tok = tok0 + 16 * (j0 + jj) + (lane & 15);
      if (g == 0 && (kFull || tok < N) && valid_rows > 0) {
        pmax[blk * N + tok] = st[jj].max;
        psum1[blk * N + tok] = st[jj].sum_m1;
        ptgt[blk * N + tok] = st[jj].pick;
      }
    }
  };
  if (valid_rows == kWaveM && tok0 + kWaveN <= N) {
#pragma unroll
    for (int j0 = 0; j0 < kF; j0 += kStatCols) {
      columns(std::true_type{}, j0);
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
#pragma unroll
    for (int j0 = 0; j0 < kF; j0 += kStatCols) {
      columns(std::false_type{}, j0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// ---------------------------------------------------------------------------
// Forward: Z^T tile -> per (128-row vocabulary block, token) partial stats.
//   pmax[b*N + t], psum1[b*N + t] = max and sum exp(z - max) - 1 over the
//   block's valid rows; ptgt[b*N + t] = z of the target row if it lies in the
//   block, else 0. (cross_entropy.py:21, :28-36, :40-41 restricted to the block.)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads, 1) void lmhead_stats_kernel(
    const uint16_t* __restrict__ W, const uint16_t* __restrict__ X, int64_t V, int64_t N,
    int64_t H, const int64_t* __restrict__ target, int64_t vstart, float* __restrict__ pmax,
    float* __restrict__ psum1, float* __restrict__ ptgt) {
  extern __shared__ __align__(16) char lds[];
  const int tiles_m = static_cast<int>((V + kBM - 1) / kBM);
  const int tiles_n = static_cast<int>((N + kBN - 1) / kBN);
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int64_t m0 = static_cast<int64_t>(tm) * kBM, n0 = static_cast<int64_t>(tn) * kBN;
  Acc acc;
  gemm_mainloop<false, false>(W, H, V, X, H, N, H, m0, n0, lds, acc);

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave / kWavesN, wn = wave % kWavesN;
  const int64_t vrow0 = m0 + wm * kWaveM;  // first vocabulary row of this wave
  if (vrow0 >= V) return;
  wave_stats(acc, vrow0, V, n0 + wn * kWaveN, N, target, vstart, pmax, psum1, ptgt, lane,
             [](int, int, const float*) {});
}

// Merge the partial statistics of nb vocabulary blocks into shard statistics:
// max, sum exp relative to it minus one, and the target logit (0 when not in
// the shard). A workgroup takes 16 tokens; 16 slices of its threads stride
// over the blocks with a running (max, sum - 1) each, then merge through LDS.
// kWhole: the shard is the whole vocabulary, so the merged statistics are the
// final ones and the loss is formed here (ce_combine_kernel's expression for
// one shard), where a combine launch would read them back; assumed (unless
// NULL) gets the upstream value the gradients are written for
// (hint_assume_kernel's). Each of those launches took 5 and 2 us of a small
// batch's 200.
constexpr int kRedTokens = 16;
constexpr int kRedSlices = 16;

template <bool kWhole>
__global__ __launch_bounds__(kRedTokens * kRedSlices) void lmhead_reduce_partials_kernel(
    const float* __restrict__ pmax, const float* __restrict__ psum1,
    const float* __restrict__ ptgt, int64_t nb, int64_t N, float* __restrict__ row_max,
    float* __restrict__ row_sumexp_m1, float* __restrict__ target_logit,
    float* __restrict__ loss, const float* __restrict__ hint, float* __restrict__ assumed) {
  if constexpr (kWhole) {
    if (assumed && blockIdx.x == 0 && threadIdx.x == 0) assumed[0] = usable_hint(hint[0]);
  }
  __shared__ float sm[kRedSlices][kRedTokens], ss[kRedSlices][kRedTokens],
      st[kRedSlices][kRedTokens];
  const int tl = threadIdx.x % kRedTokens;
  const int slice = threadIdx.x / kRedTokens;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * kRedTokens + tl;
  float m = kMaxFloorL, sum1 = -1.0f, tg = 0.0f;
  if (t < N) {
    // Eight blocks' loads in flight before they are merged, in block order
    // as one at a time would (the same bits): a slice's walk was one L2 round
    // trip per block.
    constexpr int kAhead = 8;
    int64_t b = slice;
    for (; b + (kAhead - 1) * kRedSlices < nb; b += kAhead * kRedSlices) {
      float xm[kAhead], xs[kAhead], xt[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int64_t o = (b + u * kRedSlices) * N + t;
        xm[u] = pmax[o];
        xs[u] = psum1[o];
        xt[u] = ptgt[o];
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        merge_excess(m, sum1, xm[u], xs[u]);
        tg += xt[u];
      }
    }
    for (; b < nb; b += kRedSlices) {
      merge_excess(m, sum1, pmax[b * N + t], psum1[b * N + t]);
      tg += ptgt[b * N + t];
    }
  }
  sm[slice][tl] = m;
  ss[slice][tl] = sum1;
  st[slice][tl] = tg;
  __syncthreads();
  if (slice == 0 && t < N) {
    float gm = sm[0][tl], gs = ss[0][tl], gt = st[0][tl];
    for (int k = 1; k < kRedSlices; ++k) {
      merge_excess(gm, gs, sm[k][tl], ss[k][tl]);
      gt += st[k][tl];
    }
    row_max[t] = gm;
    row_sumexp_m1[t] = gs;
    target_logit[t] = gt;
    if constexpr (kWhole) loss[t] = log1pf(gs) - (gt - gm);
  }
}

// ---------------------------------------------------------------------------
// Backward, step 1: recompute a chunk of Z^T and write
//   dZ[v, t] = (exp(z - gmax[t]) / (1 + gsum1[t]) - [v == target[t]]) * g[t]
// (cross_entropy.py:53-65) as bf16 into dzt[v * ldt + t] and dz[t * ldz + v].
// Rows v >= Mvalid and tokens t >= N are written as 0 (they pad the K extents
// of the two GEMMs that follow). The tile goes through LDS so that both
// layouts leave as coalesced 16-byte stores. kBoth = false writes dzt only.
// ---------------------------------------------------------------------------
template <bool kBoth>
__global__ __launch_bounds__(kThreads, 1) void lmhead_dz_kernel(
    const uint16_t* __restrict__ Wc, const uint16_t* __restrict__ X, int64_t Mvalid,
    int64_t Mpad, int64_t N, int64_t H, const int64_t* __restrict__ target, int64_t vfirst,
    const float* __restrict__ gmax, const float* __restrict__ gsum1,
    const float* __restrict__ gout, int64_t gout_stride, uint16_t* __restrict__ dzt,
    int64_t ldt, uint16_t* __restrict__ dz, int64_t ldz) {
  extern __shared__ __align__(16) char lds[];
  const int tiles_m = static_cast<int>(Mpad / kBM);
  const int tiles_n = static_cast<int>((ldt + kBN - 1) / kBN);
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int64_t m0 = static_cast<int64_t>(tm) * kBM, n0 = static_cast<int64_t>(tn) * kBN;
  Acc acc;
  gemm_mainloop<false, false>(Wc, H, Mvalid, X, H, N, H, m0, n0, lds, acc);

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave / kWavesN, wn = wave % kWavesN;
  const int g4 = lane >> 4;
  const int64_t vrow0 = m0 + wm * kWaveM;
  const int64_t vr = Mvalid - vrow0;
  const int valid_rows = static_cast<int>(vr < 0 ? 0 : (vr < kWaveM ? vr : kWaveM));
  // The operand buffers are free once every wave is done with its last
  // fragments; the 256x256 bf16 tile of dZ (128 KiB) is staged there.
  __syncthreads();
  uint32_t* P = reinterpret_cast<uint32_t*>(lds);
#pragma unroll
  for (int j = 0; j < kF; ++j) {
    const int tloc = wn * kWaveN + 16 * j + (lane & 15);
    const int64_t tok = n0 + tloc;
    const bool tok_ok = tok < N;
    float M = 0.0f, scale = 0.0f, g = 0.0f, T1 = 0.0f;
    int tl = -1;  // target row within this wave's rows, or -1
    if (tok_ok) {
      g = gout[tok * gout_stride];
      T1 = gsum1[tok];
      M = gmax[tok];
      scale = g / (1.0f + T1);
      const int64_t t = target[tok] - vfirst - vrow0;
      tl = (t >= 0 && t < valid_rows) ? static_cast<int>(t) : -1;
    }
    // The target row, (softmax - 1) * g (cross_entropy.py:58-64): when the
    // target is the maximum, -T1 / (1 + T1) * g from T1 itself (no
    // cancellation for a confident token, exactly 0 when T1 = 0); otherwise
    // its softmax is at most 1/2 and the plain form loses nothing.
    float zt = 0.0f;
#pragma unroll
    for (int i = 0; i < kF; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) zt = (acc_row(i, e, g4) == tl) ? acc.c[i][j][e] : zt;
    const float dt = zt == M ? -T1 / (1.0f + T1) * g : (exp_shift(zt, M) / (1.0f + T1) - 1.0f) * g;
#pragma unroll
    for (int i = 0; i < kF; ++i) {
      float d[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = acc_row(i, e, g4);
        float p = exp_shift(acc.c[i][j][e], M) * scale;
        p = (r == tl) ? dt : p;
        d[e] = (tok_ok && r < valid_rows) ? p : 0.0f;
      }
      // Into the LDS tile as (even, odd) vocabulary-row pairs of one token.
      *stage_word(P, wm, i, g4, 0, tloc) = pack_bf16x2(d[0], d[1]);
      *stage_word(P, wm, i, g4, 1, tloc) = pack_bf16x2(d[2], d[3]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();
  // dz [N, ldz]: 32 lanes per token row, each 8 consecutive vocabulary rows
  // (16 bytes), so one store instruction writes two 512-byte row segments.
#pragma unroll 4
  for (int it = 0; kBoth && it < kBN * (kBM / 8) / kThreads; ++it) {
    const int lin = it * kThreads + static_cast<int>(threadIdx.x);
    const int t = lin / (kBM / 8);
    const int L = lin % (kBM / 8);  // vocabulary rows 8L .. 8L+7, pairs 4L .. 4L+3
    const int64_t tok = n0 + t;
    uint32_t c4[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) c4[u] = P[(4 * L + u) * kBN + (t ^ stage_swz(4 * L + u))];
    const u32x4 w = {c4[0], c4[1], c4[2], c4[3]};
    if (tok < N) *reinterpret_cast<u32x4*>(dz + tok * ldz + m0 + 8 * L) = w;
  }
  // dz^T [Vc, ldt]: 32 lanes cover one pair of vocabulary rows (256 tokens);
  // each reads 8 words (8 tokens of both rows) and writes 16 bytes to each row.
#pragma unroll 2
  for (int it = 0; it < kStagedIters; ++it) {
    const int lin = it * kThreads + static_cast<int>(threadIdx.x);
    const int vp = lin / (kBN / 8);
    const int t0 = 8 * (lin % (kBN / 8));
    u32x4 lo, hi;
    staged_rows(P, vp, t0, lo, hi);
    const int64_t tok0 = n0 + t0;
    if (tok0 < ldt) {
      *reinterpret_cast<u32x4*>(dzt + (m0 + 2 * vp) * ldt + tok0) = lo;
      *reinterpret_cast<u32x4*>(dzt + (m0 + 2 * vp + 1) * ldt + tok0) = hi;
    }
  }
}

// The stored products' epilogues take the results row by row (kRows): lane l
// holds, of each 16x16 block, row l % 16 and columns 4 g .. 4 g + 3 (g = l /
// 16), and stages them through the freed LDS, so that whole row segments of
// 512 bytes (bf16) or 1 KiB (fp32) leave. Stored straight from the registers
// they are segments of 64 bytes: 1358 against 1415 TFLOP/s with fp32 out on
// 128256 x 4096 x 4096, 1457 against 1485 with bf16.
//
// The fp32 epilogues (modes 1-3 of gemm_store_kernel). The 256x256 fp32 tile
// goes through the freed LDS in two passes of 128 rows: pass q takes row
// blocks i = 4q .. 4q + 3 of every wave, i.e. tile rows 64 q .. 64 q + 63
// and 128 + 64 q .. 128 + 64 q + 63, so each pass reads its own half of the
// accumulator registers. Staged row r (1 KiB) is tile row
// 128 (r >> 6) + 64 q + (r & 63); its 16-byte chunk c sits at c ^ (r & 15),
// which puts the 16 rows that 16 lanes write on distinct 16-byte bank groups
// (the lane's four columns of a block are one chunk). Every thread then moves
// 32 chunks:
// staged row 4 p + wave, chunk lane, so a wave's access is one 1 KiB row
// segment of Cf (or 512 bytes of C).
// kVec (N % 4 == 0, ldc % 4 == 0, Cf 16-byte and C 8-byte aligned, 512 rows
// within 32-bit offsets): buffer resources on the wave's first row, the
// lane's column in the one offset register and the row step in the scalar
// offset of the loads (the 16-byte stores take it in the per-lane offset:
// buffer_store_b128). The hardware range check covers the per-lane offset
// only, so rows past M (passes p >= np, uniform) are skipped explicitly, and
// a lane whose columns lie past N gets the offset 2^31, more than a resource's
// size and no row step takes it past 32 bits: its accesses are out of range (no
// memory access, a load reads 0, a store is dropped) whether or not the row
// step takes part in the check. (As a product of the row stride it made the
// compiler carry the stride in a lane register and loop over its values at
// every load.) Every access left is inside the matrix. In modes 2 and 3 the 32 loads of Cf are
// issued before the pass is staged, so that their latency runs under the
// staging and 128 KiB are in flight. Cf is streamed (non-temporal) both ways.
// Without kVec the pass leaves element by element.
// kFull: all of the tile's rows exist, nothing is tested. Behind a branch the
// compiler cannot count what is in flight and waits for everything, which with
// each row's load issued behind an earlier row's store was a memory round trip
// a row. Accumulating launches, us: K = 512 on [16348, 2368] 138 -> 95, on
// [128256, 4096] 1383 -> 924; K = 4096 on [128256, 4096] 3531 -> 3255 (mode 2),
// 3469 -> 3121 (mode 3). With the loads in flight, reading the tile's lines
// ahead under the last K steps only costs: 3348 and 3197.
//   kMode 1: Cf = acc;  kMode 2: Cf += acc;  kMode 3: C = bf16(Cf + acc)
template <int kMode, bool kVec, bool kFull>
__device__ __forceinline__ void store_f32_pass(const Acc& acc, int q, char* lds,
                                               float* __restrict__ Cf, uint16_t* __restrict__ C,
                                               int64_t ldc, int64_t M, int64_t N, int64_t m0,
                                               int64_t n0) {
  static_assert(kMode >= 1 && kMode <= 3, "fp32 epilogue modes");
  static_assert(kBN == 256 && kWavesM == 2 && kF == 8 && 128 * kBN * 4 <= kLdsBytes,
                "two passes of 128 rows fit the stages");
  constexpr int kRowsPerPass = kThreads / 64;  // 4
  constexpr int kPasses = 128 / kRowsPerPass;  // 32
  constexpr int kNt = 2;                       // cache policy: non-temporal
  constexpr uint32_t kPast = 1u << 31;         // a lane past N: beyond every resource here
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / kWavesN, wn = wave % kWavesN;
  const int g = lane >> 4;
  float* S = reinterpret_cast<float*>(lds);
  const bool col_ok = n0 + 4 * lane < N;
  // Tile rows of staged rows 4 p + wave, relative to the pass's first row.
  auto row_off = [](int p) { return 4 * p + 64 * (p >> 4); };
  const int64_t row0 = m0 + 64 * q + wave;  // tile row of staged row `wave`
  // valid passes: a prefix, rows increase with p
  int np = kPasses;
  if constexpr (!kFull) {
    np = 0;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) np += (row0 + row_off(p) < M) ? 1 : 0;
    np = __builtin_amdgcn_readfirstlane(np);
  }
  const int64_t lim = np == 0 ? 0 : (np < kPasses ? row_off(np) : row_off(kPasses - 1) + 1);
  const uint32_t vf = col_ok ? static_cast<uint32_t>(lane) * 16u : kPast;
  float* cf_base = Cf + (np > 0 ? row0 : 0) * ldc + n0;
  u32x4 old[kPasses];
  __amdgpu_buffer_rsrc_t rf;
  if constexpr (kVec) {
    rf = __builtin_amdgcn_make_buffer_rsrc(cf_base, 0, static_cast<int>(lim * ldc * 4), 0x00020000);
    if constexpr (kMode >= 2) {
#pragma unroll
      for (int p = 0; p < kPasses; ++p) {
        if (kFull || p < np)
          old[p] = __builtin_amdgcn_raw_buffer_load_b128(
              rf, vf, static_cast<uint32_t>(row_off(p) * ldc * 4), kNt);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < kF; ++j)
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const int r = wm * 64 + 16 * f + (lane & 15);
      const int c = (wn * (kWaveN / 4) + 4 * j + g) ^ (lane & 15);
      *reinterpret_cast<f32x4_t*>(S + r * kBN + 4 * c) = acc.c[4 * q + f][j];
    }
  __syncthreads();
#pragma unroll
  for (int p = 0; p < kPasses; ++p) {
    const int r = p * kRowsPerPass + wave;
    const u32x4 sv =
        *reinterpret_cast<const u32x4*>(S + r * kBN + ((lane ^ ((4 * p + wave) & 15)) << 2));
    if constexpr (!kVec) {
      const int64_t row = row0 + row_off(p);
      const float sf[4] = {__uint_as_float(sv.x), __uint_as_float(sv.y), __uint_as_float(sv.z),
                           __uint_as_float(sv.w)};
      for (int j = 0; j < 4; ++j) {
        const int64_t col = n0 + 4 * lane + j;
        if (row >= M || col >= N) continue;
        const int64_t o = row * ldc + col;
        if constexpr (kMode == 1) Cf[o] = sf[j];
        if constexpr (kMode == 2) Cf[o] += sf[j];
        if constexpr (kMode == 3) C[o] = f32_to_bf16(Cf[o] + sf[j]);
      }
    } else {
      if (!kFull && p >= np) continue;
      const uint32_t so = static_cast<uint32_t>(row_off(p) * ldc * 4);
      if constexpr (kMode == 1) {
        buffer_store_b128<kNt>(sv, rf, vf + so);
      } else {
        const u32x4 o = old[p];
        const float v0 = __uint_as_float(sv.x) + __uint_as_float(o.x);
        const float v1 = __uint_as_float(sv.y) + __uint_as_float(o.y);
        const float v2 = __uint_as_float(sv.z) + __uint_as_float(o.z);
        const float v3 = __uint_as_float(sv.w) + __uint_as_float(o.w);
        if constexpr (kMode == 2) {
          buffer_store_b128<kNt>(
              u32x4{__float_as_uint(v0), __float_as_uint(v1), __float_as_uint(v2),
                    __float_as_uint(v3)},
              rf, vf + so);
        } else {
          typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
          const auto rh = __builtin_amdgcn_make_buffer_rsrc(
              C + (np > 0 ? row0 : 0) * ldc + n0, 0, static_cast<int>(lim * ldc * 2), 0x00020000);
          __builtin_amdgcn_raw_buffer_store_b64(
              u32x2{pack_bf16x2(v0, v1), pack_bf16x2(v2, v3)}, rh,
              col_ok ? static_cast<uint32_t>(lane) * 8u : kPast,
              static_cast<uint32_t>(row_off(p) * ldc * 2), 0);
        }
      }
    }
  }
  __syncthreads();  // the next pass reuses S
}

template <int kMode, bool kVec>
__device__ __forceinline__ void store_f32_tile(const Acc& acc, char* lds, float* __restrict__ Cf,
                                               uint16_t* __restrict__ C, int64_t ldc, int64_t M,
                                               int64_t N, int64_t m0, int64_t n0) {
  __syncthreads();  // every wave is done with the operand buffers
  if (kVec && m0 + kBM <= M) {
    store_f32_pass<kMode, kVec, true>(acc, 0, lds, Cf, C, ldc, M, N, m0, n0);
    store_f32_pass<kMode, kVec, true>(acc, 1, lds, Cf, C, ldc, M, N, m0, n0);
  } else {
    store_f32_pass<kMode, kVec, false>(acc, 0, lds, Cf, C, ldc, M, N, m0, n0);
    store_f32_pass<kMode, kVec, false>(acc, 1, lds, Cf, C, ldc, M, N, m0, n0);
  }
}

// bf16 out: rows of 512 bytes whose 16-byte chunk c sits at c ^ (row & 15):
// the 16 rows of a block that 32 lanes write 8 bytes of each are on distinct
// 16-byte bank groups. The stores are non-temporal: the product is read by a
// later kernel, if at all, and its lines would take L2 from the next tiles'
// operands. Against words of two rows, unscrambled on the way out, and cached
// stores: K = 512 875 -> 1030 TFLOP/s, K = 1600 1166 -> 1247, K = 4096 1445 ->
// 1459. Tiles that reach past M or N, and outputs that are not 16-byte
// aligned, test every row and column.
__device__ __forceinline__ void store_bf16_tile(const Acc& acc, char* lds,
                                                uint16_t* __restrict__ C, int64_t ldc, int64_t M,
                                                int64_t N, int64_t m0, int64_t n0) {
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave / kWavesN, wn = wave % kWavesN;
  const int g = lane >> 4, c = lane & 15;
  const bool vec_ok = (ldc & 7) == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
  __syncthreads();  // every wave is done with the operand buffers
  char* row = lds + (wm * kWaveM + c) * (kBN * 2) + 8 * (g & 1);
#pragma unroll
  for (int j = 0; j < kF; ++j) {
    char* at = row + (((wn * (kWaveN / 8) + 2 * j + (g >> 1)) ^ c) << 4);
#pragma unroll
    for (int i = 0; i < kF; ++i)
      *reinterpret_cast<u32x2*>(at + i * (16 * kBN * 2)) =
          u32x2{pack_bf16x2(acc.c[i][j][0], acc.c[i][j][1]),
                pack_bf16x2(acc.c[i][j][2], acc.c[i][j][3])};
  }
  __syncthreads();
  constexpr int kRowStep = kThreads / (kBN / 8);  // 8 rows of 32 chunks at a time
  constexpr int kIters = kBM / kRowStep;
  const int r0 = static_cast<int>(threadIdx.x) / (kBN / 8);
  const int q = static_cast<int>(threadIdx.x) % (kBN / 8);
  auto staged = [&](int it) {
    const int r = r0 + it * kRowStep;
    return *reinterpret_cast<const u32x4*>(lds + r * (kBN * 2) + ((q ^ (r & 15)) << 4));
  };
  if (vec_ok && m0 + kBM <= M && n0 + kBN <= N) {  // every store in bounds: no tests
    uint16_t* dst = C + (m0 + r0) * ldc + n0 + 8 * q;
#pragma unroll 8
    for (int it = 0; it < kIters; ++it) {
      store_stream(reinterpret_cast<u32x4*>(dst), staged(it));
      dst += kRowStep * ldc;
    }
    return;
  }
  const int64_t col = n0 + 8 * q;
#pragma unroll 2
  for (int it = 0; it < kIters; ++it) {
    const u32x4 w = staged(it);
    const int64_t r = m0 + r0 + it * kRowStep;
    if (r >= M || col >= N) continue;
    uint16_t* dst = C + r * ldc + col;
    if (vec_ok && col + 8 <= N) {
      store_stream(reinterpret_cast<u32x4*>(dst), w);
    } else {
      const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
      for (int e = 0; e < 8 && col + e < N; ++e)
        dst[e] = static_cast<uint16_t>(e & 1 ? ws[e >> 1] >> 16 : ws[e >> 1] & 0xffffu);
    }
  }
}

// ---------------------------------------------------------------------------
// Plain GEMM with a stored result: C[m, n] (ldc) for m < M, n < N.
//   kMode 0: C = acc as bf16
//   kMode 1: Cf = acc (fp32)
//   kMode 2: Cf += acc (fp32)
//   kMode 3: C = bf16(Cf + acc)
// Split K (splits > 1, mode 1 only): the grid holds `splits` copies of the
// tile grid; copy s takes k in [s ks, min((s + 1) ks, K)) and writes its
// partial product to Cf + s * split_stride. Copies are numbered as extra tile
// rows (split-major), so the XCD bands keep tiles of one K range together.
// kVec (modes 1-3): the output meets store_f32_tile's conditions for 16-byte
// accesses (the host checks them); otherwise it leaves element by element.
// ---------------------------------------------------------------------------
template <int kMode, bool kAMN, bool kBMN, bool kVec>
__device__ __forceinline__ void gemm_store_tile(
    int block, char* lds, const uint16_t* __restrict__ A, int64_t lda, int64_t M,
    const uint16_t* __restrict__ B, int64_t ldb, int64_t N, int64_t K, uint16_t* __restrict__ C,
    float* __restrict__ Cf, int64_t ldc, int64_t ka_rows, int64_t kb_rows, int splits, int64_t ks,
    int64_t split_stride) {
  const int tiles_m = static_cast<int>((M + kBM - 1) / kBM);
  const int tiles_n = static_cast<int>((N + kBN - 1) / kBN);
  int tmv, tn;
  tile_coords(block, tiles_m * splits, tiles_n, tmv, tn);
  const int split = tmv / tiles_m;
  const int tm = tmv - split * tiles_m;
  const int64_t m0 = static_cast<int64_t>(tm) * kBM, n0 = static_cast<int64_t>(tn) * kBN;
  // This copy's K range: the operands start at its first k (a k-column of a
  // K-contiguous operand, a k-row of an MN-contiguous one).
  const int64_t k0 = split * ks;
  const int64_t kl = (K - k0) < ks ? (K - k0) : ks;
  const uint16_t* As = kAMN ? A + k0 * lda : A + k0;
  const uint16_t* Bs = kBMN ? B + k0 * ldb : B + k0;
  Cf += split * split_stride;
  Acc acc;
  gemm_mainloop<kAMN, kBMN, /*kRows=*/true>(As, lda, M, Bs, ldb, N, kl, m0, n0, lds, acc,
                                            ka_rows - k0, kb_rows - k0);
  if constexpr (kMode != 0)
    store_f32_tile<kMode, kVec>(acc, lds, Cf, C, ldc, M, N, m0, n0);
  else
    store_bf16_tile(acc, lds, C, ldc, M, N, m0, n0);
}

template <int kMode, bool kAMN = false, bool kBMN = false, bool kVec = true>
__global__ __launch_bounds__(kThreads, 1) void gemm_store_kernel(
    const uint16_t* __restrict__ A, int64_t lda, int64_t M, const uint16_t* __restrict__ B,
    int64_t ldb, int64_t N, int64_t K, uint16_t* __restrict__ C, float* __restrict__ Cf,
    int64_t ldc, int64_t ka_rows, int64_t kb_rows, int splits, int64_t ks,
    int64_t split_stride) {
  extern __shared__ __align__(16) char lds[];
  gemm_store_tile<kMode, kAMN, kBMN, kVec>(blockIdx.x, lds, A, lda, M, B, ldb, N, K, C, Cf, ldc,
                                           ka_rows, kb_rows, splits, ks, split_stride);
}

// One chunk's two backward products in one grid: dX = dZ W (kSplit: K ranges'
// fp32 partials; else bf16) by the first x_blocks workgroups, then dW = dZ^T X
// in bf16. dX's tiles are few and long, dW's many and short, so dW's fill the
// compute units that dX's one round leaves idle or frees early, and one last
// round is left partly empty instead of two. Steps: [512, 768] x [50304, 768]
// 225 -> 204 us, [135, 960] x [111313, 960] 269 -> 256, [1548, 3904] x [256000,
// 3904] 8.23 -> 8.06 ms; where dW alone has tens of rounds there is no
// difference ([4096, 4096] x [128256, 4096] 9.48 ms either way). Chunks that
// accumulate dW in fp32 keep two launches: their dW is long, and its epilogue
// another.
struct PairArgs {
  const uint16_t* dzt;  // [vpad, ldt]
  int64_t ldt, vpad;
  const uint16_t* W;    // [V, H]
  int64_t V, H;
  const uint16_t* xt;   // [H, ldt]
  int64_t n;            // tokens
  uint16_t* dx;         // [n, H]
  float* part;          // [splits][n][H]
  uint16_t* dw;         // [V, H]
  int64_t ks;
  int splits, x_blocks;
};
template <bool kSplit>
__global__ __launch_bounds__(kThreads, 1) void gemm_pair_kernel(PairArgs p) {
  extern __shared__ __align__(16) char lds[];
  const int b = blockIdx.x;
  if (b < p.x_blocks)
    gemm_store_tile<kSplit ? 1 : 0, true, true, true>(b, lds, p.dzt, p.ldt, p.n, p.W, p.H, p.H,
                                                      p.vpad, p.dx, p.part, p.H, p.vpad, p.V,
                                                      p.splits, p.ks, p.n * p.H);
  else
    gemm_store_tile<0, false, false, true>(b - p.x_blocks, lds, p.dzt, p.ldt, p.V, p.xt, p.ldt,
                                           p.H, p.ldt, p.dw, nullptr, p.H, 0, 0, 1, p.ldt, 0);
}

// ---------------------------------------------------------------------------
// One-pass fused loss, step 1 (per chunk of tokens): the statistics GEMM of
// lmhead_stats_kernel whose epilogue also keeps the exponentials it forms,
//   pt[v * ldt + t] = bf16(exp(z[v, t] - pmax[b * N + t]))   (b = v / 128)
// for v < V and t < N, and 0 for the padding of the tile grid (rows up to the
// next multiple of 256, tokens up to ldt). Once the row statistics are known,
// dZ is pt times one factor per (block, token) (lmhead_dz_rescale_kernel), so
// the logits never need to be recomputed. pt leaves through LDS as 512-byte
// row segments, as in lmhead_dz_kernel.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads, 1) void lmhead_p_kernel(
    const uint16_t* __restrict__ W, const uint16_t* __restrict__ X, int64_t V, int64_t N,
    int64_t H, const int64_t* __restrict__ target, int64_t vstart, float* __restrict__ pmax,
    float* __restrict__ psum1, float* __restrict__ ptgt, uint16_t* __restrict__ pt,
    int64_t ldt) {
  extern __shared__ __align__(16) char lds[];
  const int tiles_m = static_cast<int>((V + kBM - 1) / kBM);
  const int tiles_n = static_cast<int>((N + kBN - 1) / kBN);
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int64_t m0 = static_cast<int64_t>(tm) * kBM, n0 = static_cast<int64_t>(tn) * kBN;
  Acc acc;
  gemm_mainloop<false, false>(W, H, V, X, H, N, H, m0, n0, lds, acc);

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave / kWavesN, wn = wave % kWavesN;
  const int g = lane >> 4;
  __syncthreads();  // every wave is done with the operand buffers
  uint32_t* P = reinterpret_cast<uint32_t*>(lds);
  wave_stats(acc, m0 + wm * kWaveM, V, n0 + wn * kWaveN, N, target, vstart, pmax, psum1, ptgt,
             lane, [&](int j, int i, const float* p) {
               const int c = wn * kWaveN + 16 * j + (lane & 15);
               *stage_word(P, wm, i, g, 0, c) = pack_bf16x2(p[0], p[1]);
               *stage_word(P, wm, i, g, 1, c) = pack_bf16x2(p[2], p[3]);
             });
  __syncthreads();
  // pt [Mpad, ldt]: 32 lanes cover one pair of vocabulary rows (256 tokens).
  // Non-temporal stores: pt (N V bf16, gigabytes) is read back only by the
  // rescale kernel, so it should not take L2 lines from the operand stripes
  // the next tiles of this XCD read (measured: the kernel 2% faster).
#pragma unroll 2
  for (int it = 0; it < kStagedIters; ++it) {
    const int lin = it * kThreads + static_cast<int>(threadIdx.x);
    const int vp = lin / (kBN / 8);
    const int t0 = 8 * (lin % (kBN / 8));
    u32x4 lo, hi;
    staged_rows(P, vp, t0, lo, hi);
    const int64_t tok0 = n0 + t0;
    if (tok0 < ldt) {
      store_stream(reinterpret_cast<u32x4*>(pt + (m0 + 2 * vp) * ldt + tok0), lo);
      store_stream(reinterpret_cast<u32x4*>(pt + (m0 + 2 * vp + 1) * ldt + tok0), hi);
    }
  }
}

// ---------------------------------------------------------------------------
// One-pass fused loss, step 2: dZ from the kept exponentials, once the row
// statistics (M, T1) are combined (cross_entropy.py:53-65):
//   dZ[t, v] = exp(z - M) / (1 + T1) * g = pt[v, t] * exp(pmax[b, t] - M) * g / (1 + T1)
// and, on the target row, (softmax - 1) * g from the fp32 target logit
// (target_grad), written in place into pt, which both backward products then
// read as it lies (vocabulary-major). A workgroup takes one 128-row block of
// partial statistics and 256 tokens; the factor of each (block, token) is
// formed once. Rows past V and blocks past nb come out 0 (pt holds 0 there).
// blockIdx.x walks the token tiles, so consecutive workgroups cover whole
// rows of pt (measured 2.5% faster than walking the row blocks first).
//
// The grid's rows past row_blocks transpose the chunk's hidden rows for the dW
// product (X_c [N, H] to xt [H, ldt], zero past N): work of its own that a
// launch by itself took 5 us for at [512, 768] and 14 at [4096, 4096], nearly
// all of it the launch.
// ---------------------------------------------------------------------------
constexpr int kRsRows = kPartialRows;  // 128: one block of partial statistics
constexpr int kRsToks = 256;
constexpr int kTrTile = 64;            // transpose tiles: 64 x 64

// bf16 transpose with zero padding, the 64 x 64 tile at rows r0 and columns c0
// of `in`: out[c * ldo + r] = in[r * ldi + c] for r < R, c < C; out[c * ldo +
// r] = 0 for R <= r < ldo. Through LDS; interior tiles move 16 bytes per load
// and per store (vec_ok: ldi, ldo and the base pointers 16-byte aligned), edge
// tiles go element by element. 256 lanes.
__device__ __forceinline__ void transpose_tile(uint16_t (*t)[kTrTile + 2],
                                               const uint16_t* __restrict__ in, int64_t R,
                                               int64_t C, int64_t ldi, uint16_t* __restrict__ out,
                                               int64_t ldo, bool vec_ok, int64_t r0, int64_t c0) {
  const int tid = threadIdx.x;
  const bool interior = vec_ok && r0 + 64 <= R && c0 + 64 <= C && r0 + 64 <= ldo;
  if (interior) {
    // in: 64 rows x 8 vectors of 8 elements
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = tid / 8 + 32 * i;
      const int cv = (tid % 8) * 8;
      const u32x4 v = *reinterpret_cast<const u32x4*>(in + (r0 + row) * ldi + c0 + cv);
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        t[row][cv + 2 * e] = static_cast<uint16_t>(w[e] & 0xffffu);
        t[row][cv + 2 * e + 1] = static_cast<uint16_t>(w[e] >> 16);
      }
    }
    __syncthreads();
    // out: 64 rows (c) x 8 vectors of 8 elements (r)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int col = tid / 8 + 32 * i;
      const int rv = (tid % 8) * 8;
      uint32_t w[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        w[e] = static_cast<uint32_t>(t[rv + 2 * e][col]) |
               (static_cast<uint32_t>(t[rv + 2 * e + 1][col]) << 16);
      *reinterpret_cast<u32x4*>(out + (c0 + col) * ldo + r0 + rv) = u32x4{w[0], w[1], w[2], w[3]};
    }
    return;
  }
  const int tx = tid & 63, ty = tid >> 6;
  for (int i = ty; i < 64; i += 4) {
    const int64_t r = r0 + i, c = c0 + tx;
    t[i][tx] = (r < R && c < C) ? in[r * ldi + c] : static_cast<uint16_t>(0);
  }
  __syncthreads();
  for (int i = ty; i < 64; i += 4) {
    const int64_t c = c0 + i, r = r0 + tx;
    if (c < C && r < ldo) out[c * ldo + r] = t[tx][i];
  }
}

__global__ __launch_bounds__(256) void lmhead_dz_rescale_kernel(
    uint16_t* __restrict__ pt, int64_t ldt, int64_t V, int64_t N, const float* __restrict__ pmax,
    int64_t nb, const float* __restrict__ gmax, const float* __restrict__ gsum1,
    const float* __restrict__ tlogit, const int64_t* __restrict__ target, int64_t vstart,
    const float* __restrict__ gout, int64_t gstride, float gdiv, int row_blocks,
    const uint16_t* __restrict__ x, int64_t H, uint16_t* __restrict__ xt) {
  if (static_cast<int>(blockIdx.y) >= row_blocks) {
    __shared__ uint16_t tile[kTrTile][kTrTile + 2];
    const int64_t id = static_cast<int64_t>(blockIdx.y - row_blocks) * gridDim.x + blockIdx.x;
    const int64_t across = (H + kTrTile - 1) / kTrTile;
    const int64_t r0 = id / across * kTrTile;
    if (r0 >= ldt) return;
    transpose_tile(tile, x, N, H, H, xt, ldt, true, r0, id % across * kTrTile);
    return;
  }
  __shared__ float s_scale[kRsToks];
  __shared__ float s_dt[kRsToks];
  __shared__ int s_tv[kRsToks];
  const int64_t blk = blockIdx.y;
  const int64_t v0 = blk * kRsRows;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kRsToks;
  const int tid = threadIdx.x;
  if (tid < kRsToks) {
    const int64_t t = t0 + tid;
    float c = 0.0f, dt = 0.0f;
    int tv = -1;
    if (t < N && blk < nb) {
      const float M = gmax[t], T1 = gsum1[t];
      const float g = gout[t * gstride] / gdiv;
      c = exp_shift(pmax[blk * N + t], M) * (g / (1.0f + T1));
      const int64_t lt = target[t] - vstart - v0;
      if (lt >= 0 && lt < kRsRows && v0 + lt < V) {
        tv = static_cast<int>(lt);
        dt = target_grad(tlogit[t], M, T1, g);
      }
    }
    s_scale[tid] = c;
    s_dt[tid] = dt;
    s_tv[tid] = tv;
  }
  __syncthreads();
  const int lane = tid & 63;
  const int wave = tid >> 6;
  // A lane takes tokens 8s .. 8s + 7 of two adjacent rows per iteration; a
  // wave's load covers two rows' 512-byte segments. The last tile of a row
  // may stop at ldt (a multiple of 64) partway.
  const int sg = lane & 31;
  const int tg = 8 * sg;
  const bool tok_ok = t0 + tg < ldt;
  auto fix = [&](float* f, int r) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      // A zero factor (padding, or an exponential that underflows) writes 0
      // whatever the buffer held: the padding columns past a short last
      // chunk's tiles were never written.
      const float c = s_scale[tg + k];
      f[k] = c == 0.0f ? 0.0f : f[k] * c;
      f[k] = (s_tv[tg + k] == r) ? s_dt[tg + k] : f[k];
    }
  };
  if (!tok_ok) return;
#pragma unroll 4
  for (int it = 0; it < kRsRows / 2 / 8; ++it) {
    const int r = 2 * ((lane >> 5) + 2 * (wave + 4 * it));  // even row of the pair
    u32x4* p0 = reinterpret_cast<u32x4*>(pt + (v0 + r) * ldt + t0 + tg);
    u32x4* p1 = reinterpret_cast<u32x4*>(pt + (v0 + r + 1) * ldt + t0 + tg);
    // Cached both ways: what of the chunk the caches still hold (the last of
    // P^T when this starts, the last of dZ^T for the products that follow) is
    // not fetched again, and a chunk that fits them never leaves: [512] x 50304
    // 23 -> 19 us, [2103] x 50257 82 -> 70, [4096] x 128256 374 -> 360 against
    // non-temporal accesses.
    const u32x4 a = *p0;
    const u32x4 b = *p1;
    float fa[8], fb[8];
    Elem<uint16_t>::unpack(a, fa);
    Elem<uint16_t>::unpack(b, fb);
    fix(fa, r);
    fix(fb, r + 1);
    *p0 = Elem<uint16_t>::pack(fa);
    *p1 = Elem<uint16_t>::pack(fb);
  }
}

// A product split over K (gemm_store_kernel, splits > 1) summed into bf16:
// out[r * ldo + c] = bf16(sum_s part[s][r][c]) for r < M, c < N (N, ldo % 4 == 0),
// with the partials [splits][M][N] fp32 contiguous. The splits are added in
// order, so the result does not depend on how the GEMM was scheduled; eight
// ranges' loads are in flight at a time. One token chunk has at most one round
// of ranges (256); the recomputing backward sums those of all its vocabulary
// chunks, a thousand and more where a caller asks for small ones.
__global__ __launch_bounds__(256) void split_sum_bf16_kernel(const float* __restrict__ part,
                                                             int splits, int64_t M, int64_t N,
                                                             uint16_t* __restrict__ out,
                                                             int64_t ldo) {
  const int64_t total = M * N;
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i >= total) return;
  float a[4];
  Elem<float>::unpack(load_stream(reinterpret_cast<const u32x4*>(part + i)), a);
#pragma unroll 8
  for (int sp = 1; sp < splits; ++sp) {
    float b[4];
    Elem<float>::unpack(load_stream(reinterpret_cast<const u32x4*>(part + sp * total + i)), b);
#pragma unroll
    for (int k = 0; k < 4; ++k) a[k] += b[k];
  }
  const int64_t r = i / N, c = i - r * N;
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  uint16_t* dst = out + r * ldo + c;
  if ((reinterpret_cast<uintptr_t>(out) & 7) == 0) {
    *reinterpret_cast<u32x2*>(dst) = u32x2{pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3])};
  } else {  // gradients need be aligned to their element only
#pragma unroll
    for (int k = 0; k < 4; ++k) dst[k] = f32_to_bf16(a[k]);
  }
}

// The transpose of transpose_tile by itself.
__global__ __launch_bounds__(256) void transpose_bf16_kernel(const uint16_t* __restrict__ in,
                                                             int64_t R, int64_t C, int64_t ldi,
                                                             uint16_t* __restrict__ out,
                                                             int64_t ldo, int vec_ok) {
  __shared__ uint16_t t[kTrTile][kTrTile + 2];
  transpose_tile(t, in, R, C, ldi, out, ldo, vec_ok != 0,
                 static_cast<int64_t>(blockIdx.y) * kTrTile,  // over ldo (padded R)
                 static_cast<int64_t>(blockIdx.x) * kTrTile);
}

inline int launch_status() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? NMCE_OK : static_cast<int>(e);
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

inline int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

int configure_lds() {
  static std::atomic<bool> done[4];
  const void* kernels[] = {
      reinterpret_cast<const void*>(&lmhead_stats_kernel),
      reinterpret_cast<const void*>(&lmhead_dz_kernel<true>),
      reinterpret_cast<const void*>(&lmhead_dz_kernel<false>),
      reinterpret_cast<const void*>(&lmhead_p_kernel),
  };
  for (int i = 0; i < 4; ++i)
    if (const int rc = allow_lds(kernels[i], kLdsBytes, done[i])) return rc;
  return NMCE_OK;
}

// A GEMM operand is usable when its base is 16-byte aligned, its row stride is
// a whole number of 16-byte chunks, and one 256-row tile spans < 4 GiB.
inline bool operand_ok(const void* p, int64_t ld) {
  return p != nullptr && aligned16(p) && ld % 8 == 0 && ld > 0 && ld < (int64_t{1} << 22);
}

// The product kernels by output mode and operand layout: K-contiguous A, and
// B K-contiguous (b_mn = false) or MN-contiguous with kb_rows k-rows (b_mn,
// in mode 0; with A MN-contiguous too, a_mn, in modes 0 and 1).
template <int kMode, bool kAMN, bool kBMN, bool kVec>
int launch_store(dim3 grid, hipStream_t stream, const uint16_t* A, int64_t lda, int64_t M,
                 const uint16_t* B, int64_t ldb, int64_t N, int64_t K, uint16_t* C, float* Cf,
                 int64_t ldc, int64_t ka_rows, int64_t kb_rows, int splits,
                 int64_t ks, int64_t split_stride) {
  static std::atomic<bool> lds_set{false};
  if (const int rc =
          allow_lds(reinterpret_cast<const void*>(&gemm_store_kernel<kMode, kAMN, kBMN, kVec>),
                    kLdsBytes, lds_set))
    return rc;
  hipLaunchKernelGGL((gemm_store_kernel<kMode, kAMN, kBMN, kVec>), grid, dim3(kThreads),
                     kLdsBytes, stream, A, lda, M, B, ldb, N, K, C, Cf, ldc, ka_rows, kb_rows,
                     splits, ks, split_stride);
  return NMCE_OK;
}

// splits > 1 (mode 1 only): K in `splits` ranges of ks (a multiple of kBK;
// the last one may be shorter), partial products at Cf + s * split_stride.
int launch_gemm_store(int mode, const uint16_t* A, int64_t lda, int64_t M, const uint16_t* B,
                      int64_t ldb, int64_t N, int64_t K, uint16_t* C, float* Cf, int64_t ldc,
                      hipStream_t stream, bool a_mn = false,
                      bool b_mn = false, int64_t ka_rows = 0, int64_t kb_rows = 0,
                      int splits = 1, int64_t ks = 0, int64_t split_stride = 0) {
  if (splits < 1 || (splits > 1 && (mode != 1 || ks <= 0 || ks % kBK != 0 ||
                                    (splits - 1) * ks >= K)))
    return NMCE_EINVAL_SHAPE;
  if (splits == 1) ks = K;
  const int64_t tiles = ((M + kBM - 1) / kBM) * ((N + kBN - 1) / kBN) * splits;
  const dim3 grid(static_cast<unsigned>(tiles));
  if ((a_mn && (!b_mn || mode > 1)) || (b_mn && !a_mn && mode > 0)) return NMCE_EINVAL_SHAPE;
  // The fp32 epilogues' 16-byte form: whole 16-byte chunks, aligned outputs,
  // and every offset (a pass's 189 rows, plus as much again for a lane past
  // N) within 32 bits.
  const bool vec = (N & 3) == 0 && (ldc & 3) == 0 && (reinterpret_cast<uintptr_t>(Cf) & 15) == 0 &&
                   (mode != 3 || (reinterpret_cast<uintptr_t>(C) & 7) == 0) &&
                   ldc * 4 * 512 < (int64_t{1} << 32);
  int st = NMCE_OK;
  // (mode 0 has one form: its epilogue tests its own alignment)
#define NMCE_STORE(MODE, AMN, BMN)                                                                \
  st = vec ? launch_store<MODE, AMN, BMN, true>(grid, stream, A, lda, M, B, ldb, N, K, C, Cf,      \
                                                ldc, ka_rows, kb_rows, splits, ks, split_stride)   \
           : launch_store<MODE, AMN, BMN, MODE == 0>(grid, stream, A, lda, M, B, ldb, N, K, C, Cf, \
                                                     ldc, ka_rows, kb_rows, splits, ks,            \
                                                     split_stride)
  if (a_mn) {
    if (mode == 0) NMCE_STORE(0, true, true);
    else NMCE_STORE(1, true, true);
  } else if (b_mn) {
    NMCE_STORE(0, false, true);
  } else {
    switch (mode) {
      case 0: NMCE_STORE(0, false, false); break;
      case 1: NMCE_STORE(1, false, false); break;
      case 2: NMCE_STORE(2, false, false); break;
      default: NMCE_STORE(3, false, false); break;
    }
  }
#undef NMCE_STORE
  if (st) return st;
  return launch_status();
}

// Both products write 16-byte vectors at 32-bit offsets (launch_gemm_store's
// `vec`, for row strides of H, a multiple of 64).
inline bool pair_ok(int64_t h) { return h * 4 * 512 < (int64_t{1} << 32); }

template <bool kSplit>
int launch_pair_as(const PairArgs& p, int64_t blocks, hipStream_t s) {
  static std::atomic<bool> lds_set{false};
  if (const int rc = allow_lds(reinterpret_cast<const void*>(&gemm_pair_kernel<kSplit>), kLdsBytes,
                               lds_set))
    return rc;
  hipLaunchKernelGGL(gemm_pair_kernel<kSplit>, dim3(static_cast<unsigned>(blocks)),
                     dim3(kThreads), kLdsBytes, s, p);
  return launch_status();
}

// Fills in x_blocks.
int launch_pair(PairArgs p, bool split, hipStream_t s) {
  const int64_t h_tiles = (p.H + kBN - 1) / kBN;
  const int64_t x_blocks = ((p.n + kBM - 1) / kBM) * h_tiles * p.splits;
  p.x_blocks = static_cast<int>(x_blocks);
  const int64_t blocks = x_blocks + ((p.V + kBM - 1) / kBM) * h_tiles;
  return split ? launch_pair_as<true>(p, blocks, s) : launch_pair_as<false>(p, blocks, s);
}

int launch_transpose(const uint16_t* in, int64_t R, int64_t C, int64_t ldi, uint16_t* out,
                     int64_t ldo, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>((C + 63) / 64), static_cast<unsigned>((ldo + 63) / 64));
  const int vec_ok = aligned16(in) && aligned16(out) && ldi % 8 == 0 && ldo % 8 == 0;
  hipLaunchKernelGGL(transpose_bf16_kernel, grid, dim3(256), 0, stream, in, R, C, ldi, out, ldo,
                     vec_ok);
  return launch_status();
}

// Workspace carve-up of the backward (all offsets 256-byte aligned).
struct BwdLayout {
  int64_t ldt;    // tokens padded to 64 (K of the dW GEMM)
  int64_t vpad;   // vocabulary padded to 256 (columns of W^T)
  int64_t chunk;  // vocabulary rows per chunk (multiple of 256)
  int64_t n_chunks;
  int64_t off_xt, off_wt, off_dzt, off_dz, off_acc, total;
};

inline int64_t align256(int64_t x) { return round_up(x, 256); }

BwdLayout bwd_layout(int64_t n, int64_t h, int64_t v, int64_t chunk) {
  BwdLayout L{};
  L.ldt = round_up(n, 64);
  L.vpad = round_up(v, kBM);
  L.chunk = chunk <= 0 ? L.vpad : round_up(chunk, kBM);
  if (L.chunk > L.vpad) L.chunk = L.vpad;
  L.n_chunks = (L.vpad + L.chunk - 1) / L.chunk;
  int64_t off = 0;
  L.off_xt = off; off += align256(h * L.ldt * 2);
  L.off_wt = off; off += align256(h * L.vpad * 2);
  L.off_dzt = off; off += align256(L.chunk * L.ldt * 2);
  L.off_dz = off; off += align256(n * L.chunk * 2);
  L.off_acc = off; off += L.n_chunks > 1 ? align256(n * h * 4) : 0;
  L.total = off;
  return L;
}

// The carve-up of the same bytes by a backward whose dX product reads dZ^T and
// the weight as they lie (bwd_direct): X^T stays where BwdLayout has it, dZ^T of
// one chunk follows, and what W^T, dZ and the accumulator would take holds fp32
// partials of dX, [n, h] each, one per K range of every chunk.
struct DirectLayout {
  int64_t off_dzt, off_part;
  int64_t splits;  // K ranges of a chunk's dX product; 0: the partials do not fit
  int64_t ks;      // their length
};

int64_t fwd_partial_blocks(int64_t v) { return (v + kPartialRows - 1) / kPartialRows; }

// K ranges for a product of `tiles` output tiles over K (a multiple of kBK)
// on `cus` compute units, one 256x256 tile per compute unit at a time: the
// fewest ranges (at most 8, each at least 2048 long, each holding some of the
// first `k_valid` k) whose rounds of tiles leave at most 5% of the compute
// units idle, else the fewest with the least idle share. ks gets the range
// length (a multiple of kBK). The product is counted by itself,
// also where gemm_pair_kernel's other tiles would fill the idle units: fewer
// ranges may do there, which has not been measured.
//
// Where even 8 ranges leave part of one round idle (fewer than 32 tiles on
// 256 compute units: small batches, whose K is the whole vocabulary), the
// product is one round of long serial K walks, and more ranges (up to one
// round, each at least 1024 long) shorten them: a range costs kStageUs per
// stage of its K, and the `out` partial values of each range a write and a
// read at kPartialBytesPerUs. [512, 768] x [50304, 768] (6 tiles, K = 50432):
// 126 + 5.6 us (product + sum) at 8 ranges, 43 + 9.4 at the model's 33.
int choose_splits(int64_t tiles, int64_t out, int64_t K, int64_t k_valid, int cus, int64_t* ks) {
  constexpr double kStageUs = 1.25;
  constexpr double kPartialBytesPerUs = 4e6;
  const auto valid = [&](int s, int64_t least) {
    const int64_t len = round_up((K + s - 1) / s, kBK);
    return s == 1 || (K / s >= least && (s - 1) * len < K && (s - 1) * len < k_valid);
  };
  int best = 1;
  int more = 1;
  double best_idle = 1e30;
  for (int s = 1; s <= 8; ++s) {
    if (!valid(s, 2048)) break;
    const int64_t t = tiles * s;
    const int64_t rounds = (t + cus - 1) / cus;
    const double idle = static_cast<double>(rounds * cus) / static_cast<double>(t);
    if (idle <= 1.05) {
      best = s;
      break;
    }
    if (idle < best_idle - 1e-9) {
      best_idle = idle;
      best = s;
    }
  }
  if (tiles * 8 < cus) {
    double best_us = 1e30;
    for (int s = best; s <= cus / tiles && (s == best || valid(s, 1024)); ++s) {
      const double us = kStageUs * static_cast<double>((K + s - 1) / s) / kBK +
                        8.0 * static_cast<double>(out) * s / kPartialBytesPerUs;
      if (us < best_us) {
        best_us = us;
        more = s;
      }
    }
    best = more;
  }
  *ks = best == 1 ? K : round_up((K + best - 1) / best, kBK);
  return best;
}

// The K ranges are choose_splits' for a whole chunk, and no more than fit. One
// range a chunk is enough to run (the chunks' partials take the accumulator's
// place); where even that does not fit (many tokens in many small chunks), the
// accumulating products on W^T remain.
DirectLayout direct_layout(const BwdLayout& L, int64_t n, int64_t h, int cus) {
  DirectLayout D{};
  D.off_dzt = L.off_wt;
  D.off_part = D.off_dzt + align256(L.chunk * L.ldt * 2);
  const int64_t fit = (L.total - D.off_part) / (n * h * 4) / L.n_chunks;
  if (fit < 1 || !pair_ok(h)) return D;
  const int64_t tiles = ((n + kBM - 1) / kBM) * ((h + kBN - 1) / kBN);
  D.splits = choose_splits(tiles, n * h, L.chunk, L.chunk, cus, &D.ks);
  if (D.splits > fit) {
    D.splits = fit;
    D.ks = round_up((L.chunk + fit - 1) / fit, kBK);
  }
  return D;
}

// Workspace of the one-pass fused loss (all offsets 256-byte aligned).
struct FusedLayout {
  int64_t chunk;     // tokens per chunk (the last one may hold fewer)
  int64_t n_chunks;
  int64_t ldt;       // chunk tokens padded to 64: row stride of P^T, K of the dW GEMM
  int64_t vpad;      // vocabulary padded to 256: rows of P^T, K of the dX GEMM
  int64_t nb;        // 128-row blocks of partial statistics
  int64_t off_pt, off_part, off_acc, total;
  int64_t dx_splits;  // K ranges of a chunk's dX product (split K when its tiles are few)
  int64_t dx_ks;      // their length
  int64_t off_dxp;    // their fp32 partials [dx_splits][chunk][h] (dx_splits > 1)
  int64_t off_xt;     // the chunk's hidden rows transposed, X_c^T [h, ldt] bf16
};

FusedLayout fused_layout(int64_t n, int64_t h, int64_t v, int64_t token_chunk, int cus) {
  FusedLayout L{};
  L.chunk = (token_chunk <= 0 || token_chunk >= n) ? n : round_up(token_chunk, kBN);
  if (L.chunk > n) L.chunk = n;
  L.n_chunks = (n + L.chunk - 1) / L.chunk;
  L.ldt = round_up(L.chunk, 64);
  L.vpad = round_up(v, kBM);
  L.nb = fwd_partial_blocks(v);
  const int64_t dx_tiles = ((L.chunk + kBM - 1) / kBM) * ((h + kBN - 1) / kBN);
  L.dx_splits = choose_splits(dx_tiles, L.chunk * h, L.vpad, v, cus, &L.dx_ks);
  int64_t off = 0;
  L.off_pt = off; off += align256(L.vpad * L.ldt * 2);
  L.off_part = off; off += align256(3 * L.nb * L.chunk * 4);
  L.off_acc = off; off += L.n_chunks > 1 ? align256(v * h * 4) : 0;
  L.off_dxp = off; off += L.dx_splits > 1 ? align256(L.dx_splits * L.chunk * h * 4) : 0;
  L.off_xt = off; off += align256(h * L.ldt * 2);
  L.total = off;
  return L;
}

int check_fwd_args(const void* hidden, const void* weight, int dtype, int64_t n_rows,
                   int64_t hidden_size, int64_t vocab_local, const int64_t* target,
                   const float* row_max, const float* row_sumexp_m1, const float* target_logit) {
  if (dtype != NMCE_BF16) return NMCE_EINVAL_DTYPE;
  if (n_rows < 0 || vocab_local < 1 || hidden_size < kBK || hidden_size % kBK != 0)
    return NMCE_EINVAL_SHAPE;
  if (n_rows == 0) return NMCE_OK;
  if (!operand_ok(hidden, hidden_size) || !operand_ok(weight, hidden_size))
    return NMCE_EINVAL_ALIGN;
  if (!target || !row_max || !row_sumexp_m1 || !target_logit) return NMCE_EINVAL_PTR;
  if (n_rows > (int64_t{1} << 30) || vocab_local > (int64_t{1} << 30)) return NMCE_EINVAL_SHAPE;
  return NMCE_OK;
}

// The statistics GEMM over n tokens and its reduction, with the
// [3, fwd_partial_blocks(V), n] fp32 partials at `partials`.
int launch_fwd_stats(const uint16_t* X, const uint16_t* W, int64_t n, int64_t H, int64_t V,
                     const int64_t* target, int64_t vstart, float* row_max, float* row_sumexp_m1,
                     float* target_logit, float* partials, hipStream_t s) {
  const int64_t nb = fwd_partial_blocks(V);
  float* pmax = partials;
  float* psum1 = pmax + nb * n;
  float* ptgt = psum1 + nb * n;
  const int64_t tiles = ((V + kBM - 1) / kBM) * ((n + kBN - 1) / kBN);
  hipLaunchKernelGGL(lmhead_stats_kernel, dim3(static_cast<unsigned>(tiles)), dim3(kThreads),
                     kLdsBytes, s, W, X, V, n, H, target, vstart, pmax, psum1, ptgt);
  int st = launch_status();
  if (st) return st;
  hipLaunchKernelGGL(lmhead_reduce_partials_kernel<false>,
                     dim3(static_cast<unsigned>((n + kRedTokens - 1) / kRedTokens)),
                     dim3(kRedTokens * kRedSlices), 0, s, pmax, psum1, ptgt, nb, n, row_max,
                     row_sumexp_m1, target_logit, nullptr, nullptr, nullptr);
  return launch_status();
}

// ---- the allocation-free forward's scratch ----------------------------------
// The partial statistics of nmce_lmhead_ce_fwd_stats_noalloc live in this
// fixed device array (one copy per GPU, held until the process ends) instead
// of a caller workspace. In host code `scratch` only names the array: its
// device address on the current GPU comes from hipGetSymbolAddress, taken once
// per device and kept in scratch_ptr.
constexpr int64_t kScratchBytes = int64_t{64} << 20;
constexpr int64_t kScratchFloats = kScratchBytes / 4;
static __device__ __align__(256) float scratch[kScratchFloats];

constexpr int kMaxDevices = 64;
std::mutex scratch_mu;
float* scratch_ptr[kMaxDevices] = {};

int scratch_on_current_device(float** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return static_cast<int>(e);
  if (dev < 0 || dev >= kMaxDevices) return NMCE_EINVAL_SCRATCH;
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (!scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return static_cast<int>(e);
    if (!p) return NMCE_EINVAL_SCRATCH;
    scratch_ptr[dev] = static_cast<float*>(p);
  }
  *out = scratch_ptr[dev];
  return NMCE_OK;
}

}  // namespace
}  // namespace nmce

using namespace nmce;

extern "C" {

int64_t nmce_lmhead_ce_fwd_workspace_bytes(int64_t n_rows, int64_t hidden, int64_t vocab_local) {
  (void)hidden;
  if (n_rows < 0 || vocab_local < 0) return -1;
  return align256(3 * fwd_partial_blocks(vocab_local) * n_rows * 4);
}

int64_t nmce_lmhead_ce_bwd_workspace_bytes(int64_t n_rows, int64_t hidden, int64_t vocab_local,
                                           int64_t vocab_chunk) {
  if (n_rows < 0 || hidden < 0 || vocab_local < 0) return -1;
  return bwd_layout(n_rows, hidden, vocab_local, vocab_chunk).total;
}

int nmce_lmhead_ce_fwd_stats(const void* hidden, const void* weight, int dtype, int64_t n_rows,
                             int64_t hidden_size, int64_t vocab_local, const int64_t* target,
                             int64_t vocab_start, float* row_max, float* row_sumexp_m1,
                             float* target_logit, void* workspace, int64_t workspace_bytes,
                             void* stream) {
  int st = check_fwd_args(hidden, weight, dtype, n_rows, hidden_size, vocab_local, target, row_max,
                          row_sumexp_m1, target_logit);
  if (st != NMCE_OK || n_rows == 0) return st;
  const int64_t need = nmce_lmhead_ce_fwd_workspace_bytes(n_rows, hidden_size, vocab_local);
  if (!workspace || workspace_bytes < need || !aligned16(workspace)) return NMCE_EINVAL_WORKSPACE;
  if ((st = configure_lds())) return st;
  return launch_fwd_stats(static_cast<const uint16_t*>(hidden), static_cast<const uint16_t*>(weight),
                          n_rows, hidden_size, vocab_local, target, vocab_start, row_max,
                          row_sumexp_m1, target_logit, static_cast<float*>(workspace),
                          static_cast<hipStream_t>(stream));
}

int nmce_lmhead_ce_fwd_stats_noalloc(const void* hidden, const void* weight, int dtype,
                                     int64_t n_rows, int64_t hidden_size, int64_t vocab_local,
                                     const int64_t* target, int64_t vocab_start, float* row_max,
                                     float* row_sumexp_m1, float* target_logit, void* stream) {
  int st = check_fwd_args(hidden, weight, dtype, n_rows, hidden_size, vocab_local, target, row_max,
                          row_sumexp_m1, target_logit);
  if (st != NMCE_OK || n_rows == 0) return st;
  // Tokens per launch: as many as the scratch holds the partials of, in
  // whole 256-token tile columns when that is at least one column.
  const int64_t per_token = 3 * fwd_partial_blocks(vocab_local);  // floats
  if (per_token > kScratchFloats) return NMCE_EINVAL_SCRATCH;
  int64_t chunk = kScratchFloats / per_token;
  if (chunk >= kBN) chunk = chunk / kBN * kBN;
  float* partials = nullptr;
  if ((st = scratch_on_current_device(&partials))) return st;
  if ((st = configure_lds())) return st;
  const auto* X = static_cast<const uint16_t*>(hidden);
  for (int64_t t0 = 0; t0 < n_rows; t0 += chunk) {
    const int64_t m = (n_rows - t0) < chunk ? (n_rows - t0) : chunk;
    st = launch_fwd_stats(X + t0 * hidden_size, static_cast<const uint16_t*>(weight), m,
                          hidden_size, vocab_local, target + t0, vocab_start, row_max + t0,
                          row_sumexp_m1 + t0, target_logit + t0, partials,
                          static_cast<hipStream_t>(stream));
    if (st) return st;
  }
  return NMCE_OK;
}

}  // extern "C"

namespace nmce {
namespace {

// Shared argument checks of the backward entry points; fills the layout.
int check_bwd_args(const void* hidden, const void* weight, int dtype, int64_t n_rows,
                   int64_t hidden_size, int64_t vocab_local, int64_t vocab_chunk,
                   const void* workspace, int64_t workspace_bytes, BwdLayout& L) {
  if (dtype != NMCE_BF16) return NMCE_EINVAL_DTYPE;
  if (n_rows < 1 || vocab_local < 1 || hidden_size < kBK || hidden_size % kBK != 0)
    return NMCE_EINVAL_SHAPE;
  if (!operand_ok(hidden, hidden_size) || !operand_ok(weight, hidden_size))
    return NMCE_EINVAL_ALIGN;
  if (n_rows > (int64_t{1} << 30) || vocab_local > (int64_t{1} << 30)) return NMCE_EINVAL_SHAPE;
  L = bwd_layout(n_rows, hidden_size, vocab_local, vocab_chunk);
  if (L.ldt >= (int64_t{1} << 22) || L.vpad >= (int64_t{1} << 22) || L.chunk >= (int64_t{1} << 22))
    return NMCE_EINVAL_SHAPE;
  if (!workspace || workspace_bytes < L.total || !aligned16(workspace))
    return NMCE_EINVAL_WORKSPACE;
  return NMCE_OK;
}

int bwd_prepare(const uint16_t* X, const uint16_t* W, int64_t n_rows, int64_t H, int64_t V,
                const BwdLayout& L, char* ws, hipStream_t s) {
  // X^T [H, ldt] and W^T [H, vpad], zero-padded along the token / vocab axis.
  int st = launch_transpose(X, n_rows, H, H, reinterpret_cast<uint16_t*>(ws + L.off_xt), L.ldt, s);
  if (st) return st;
  return launch_transpose(W, V, H, H, reinterpret_cast<uint16_t*>(ws + L.off_wt), L.vpad, s);
}

int bwd_dz(const uint16_t* X, const uint16_t* W, int64_t n_rows, int64_t H, int64_t V,
           const int64_t* target, int64_t vocab_start, const float* g_max,
           const float* g_sumexp_m1, const float* grad_output, int64_t gout_stride, int64_t c,
           const BwdLayout& L, uint16_t* dzt, uint16_t* dz, hipStream_t s) {
  const int64_t v0 = c * L.chunk;
  const int64_t mvalid = (V - v0) < L.chunk ? (V - v0) : L.chunk;
  const int64_t mpad = round_up(mvalid, kBM);
  const int64_t tiles = (mpad / kBM) * ((L.ldt + kBN - 1) / kBN);
  hipLaunchKernelGGL(dz ? lmhead_dz_kernel<true> : lmhead_dz_kernel<false>,
                     dim3(static_cast<unsigned>(tiles)), dim3(kThreads),
                     kLdsBytes, s, W + v0 * H, X, mvalid, mpad, n_rows, H, target,
                     vocab_start + v0, g_max, g_sumexp_m1, grad_output, gout_stride, dzt, L.ldt,
                     dz, L.chunk);
  return launch_status();
}

// The backward's products with nothing transposed but X: dX = dZ W of each
// chunk reads dZ^T and W vocabulary-row major, as they lie, in K ranges where
// its tiles leave compute units idle, and the ranges' partials of all chunks
// are summed at the end. Against both layouts of dZ, a W^T and an fp32
// accumulator (BwdLayout), in the same workspace: no transpose of the weight
// and half of dZ's stores, and the few tiles of a small batch no longer walk
// the whole chunk serially. Forward and backward: [64, 1024] x
// [50304, 1024] 994 -> 257 us, [660, 1536] x [151936, 1536] 3.83 -> 1.44 ms,
// [2048, 2048] x [32000, 2048] 1.26 -> 0.86, [4564, 3456] x [64128, 3456] 6.06
// -> 5.82, [12288, 4096] x [128256, 4096] 35.9 -> 35.0.
int bwd_direct(const uint16_t* X, const uint16_t* W, int64_t n_rows, int64_t H, int64_t V,
               const int64_t* target, int64_t vocab_start, const float* g_max,
               const float* g_sumexp_m1, const float* grad_output, int64_t gout_stride,
               const BwdLayout& L, const DirectLayout& D, char* ws, uint16_t* dX, uint16_t* dW,
               hipStream_t s) {
  auto* xt = reinterpret_cast<uint16_t*>(ws + L.off_xt);
  auto* dzt = reinterpret_cast<uint16_t*>(ws + D.off_dzt);
  auto* part = reinterpret_cast<float*>(ws + D.off_part);
  int st = launch_transpose(X, n_rows, H, H, xt, L.ldt, s);
  if (st) return st;
  int parts = 0;
  for (int64_t c = 0; c < L.n_chunks; ++c) {
    const int64_t v0 = c * L.chunk;
    const int64_t mvalid = (V - v0) < L.chunk ? (V - v0) : L.chunk;
    const int64_t mpad = round_up(mvalid, kBM);
    if ((st = bwd_dz(X, W, n_rows, H, V, target, vocab_start, g_max, g_sumexp_m1, grad_output,
                     gout_stride, c, L, dzt, nullptr, s)))
      return st;
    // Ranges that begin inside the shard; a last chunk may have fewer.
    const int ranges = D.splits == 1 ? 1 : static_cast<int>((mvalid + D.ks - 1) / D.ks);
    const bool split = L.n_chunks > 1 || D.splits > 1;
    const PairArgs p{dzt, L.ldt, mpad, W + v0 * H, mvalid, H, xt, n_rows, dX,
                     part + parts * n_rows * H, dW + v0 * H, ranges == 1 ? mpad : D.ks, ranges, 0};
    if ((st = launch_pair(p, split, s)) || !split) return st;
    parts += ranges;
  }
  const int64_t quads = n_rows * H / 4;
  hipLaunchKernelGGL(split_sum_bf16_kernel, dim3(static_cast<unsigned>((quads + 255) / 256)),
                     dim3(256), 0, s, part, parts, n_rows, H, dX, H);
  return launch_status();
}

}  // namespace
}  // namespace nmce

extern "C" {

int nmce_lmhead_ce_bwd_layout(int64_t n_rows, int64_t hidden_size, int64_t vocab_local,
                              int64_t vocab_chunk, int64_t* layout) {
  if (!layout) return NMCE_EINVAL_PTR;
  if (n_rows < 1 || hidden_size < 1 || vocab_local < 1) return NMCE_EINVAL_SHAPE;
  const BwdLayout L = bwd_layout(n_rows, hidden_size, vocab_local, vocab_chunk);
  const int64_t v[NMCE_LMHEAD_LAYOUT_FIELDS] = {L.total,  L.ldt,    L.vpad,   L.chunk, L.n_chunks,
                                                L.off_xt, L.off_wt, L.off_dzt, L.off_dz, L.off_acc};
  for (int i = 0; i < NMCE_LMHEAD_LAYOUT_FIELDS; ++i) layout[i] = v[i];
  return NMCE_OK;
}

int nmce_lmhead_ce_bwd_prepare(const void* hidden, const void* weight, int dtype, int64_t n_rows,
                               int64_t hidden_size, int64_t vocab_local, int64_t vocab_chunk,
                               void* workspace, int64_t workspace_bytes, void* stream) {
  BwdLayout L;
  int st = check_bwd_args(hidden, weight, dtype, n_rows, hidden_size, vocab_local, vocab_chunk,
                          workspace, workspace_bytes, L);
  if (st) return st;
  if ((st = configure_lds())) return st;
  return bwd_prepare(static_cast<const uint16_t*>(hidden), static_cast<const uint16_t*>(weight),
                     n_rows, hidden_size, vocab_local, L, static_cast<char*>(workspace),
                     static_cast<hipStream_t>(stream));
}

int nmce_lmhead_ce_bwd_dz(const void* hidden, const void* weight, int dtype, int64_t n_rows,
                          int64_t hidden_size, int64_t vocab_local, const int64_t* target,
                          int64_t vocab_start, const float* g_max, const float* g_sumexp_m1,
                          const float* grad_output, int64_t gout_stride, int64_t vocab_chunk,
                          int64_t chunk_index, void* workspace, int64_t workspace_bytes,
                          void* stream) {
  BwdLayout L;
  int st = check_bwd_args(hidden, weight, dtype, n_rows, hidden_size, vocab_local, vocab_chunk,
                          workspace, workspace_bytes, L);
  if (st) return st;
  if (!target || !g_max || !g_sumexp_m1 || !grad_output) return NMCE_EINVAL_PTR;
  if (gout_stride < 0 || chunk_index < 0 || chunk_index >= L.n_chunks) return NMCE_EINVAL_SHAPE;
  if ((st = configure_lds())) return st;
  char* ws = static_cast<char*>(workspace);
  return bwd_dz(static_cast<const uint16_t*>(hidden), static_cast<const uint16_t*>(weight), n_rows,
                hidden_size, vocab_local, target, vocab_start, g_max, g_sumexp_m1, grad_output,
                gout_stride, chunk_index, L, reinterpret_cast<uint16_t*>(ws + L.off_dzt),
                reinterpret_cast<uint16_t*>(ws + L.off_dz), static_cast<hipStream_t>(stream));
}

int nmce_lmhead_ce_bwd(const void* hidden, const void* weight, int dtype, int64_t n_rows,
                       int64_t hidden_size, int64_t vocab_local, const int64_t* target,
                       int64_t vocab_start, const float* g_max, const float* g_sumexp_m1,
                       const float* grad_output, int64_t gout_stride, void* grad_hidden,
                       void* grad_weight, int64_t vocab_chunk, void* workspace,
                       int64_t workspace_bytes, void* stream) {
  if (n_rows == 0 && dtype == NMCE_BF16) return NMCE_OK;
  BwdLayout L;
  int st = check_bwd_args(hidden, weight, dtype, n_rows, hidden_size, vocab_local, vocab_chunk,
                          workspace, workspace_bytes, L);
  if (st) return st;
  if (!target || !g_max || !g_sumexp_m1 || !grad_output || !grad_hidden || !grad_weight)
    return NMCE_EINVAL_PTR;
  if (gout_stride < 0) return NMCE_EINVAL_SHAPE;
  if ((st = configure_lds())) return st;
  auto s = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  const uint16_t* xt = reinterpret_cast<const uint16_t*>(ws + L.off_xt);
  const uint16_t* wt = reinterpret_cast<const uint16_t*>(ws + L.off_wt);
  uint16_t* dzt = reinterpret_cast<uint16_t*>(ws + L.off_dzt);
  uint16_t* dz = reinterpret_cast<uint16_t*>(ws + L.off_dz);
  float* acc = reinterpret_cast<float*>(ws + L.off_acc);
  const auto* X = static_cast<const uint16_t*>(hidden);
  const auto* W = static_cast<const uint16_t*>(weight);
  auto* dX = static_cast<uint16_t*>(grad_hidden);
  auto* dW = static_cast<uint16_t*>(grad_weight);
  const int64_t H = hidden_size;

  const DirectLayout D = direct_layout(L, n_rows, H, device_cus());
  if (D.splits > 0)
    return bwd_direct(X, W, n_rows, H, vocab_local, target, vocab_start, g_max, g_sumexp_m1,
                      grad_output, gout_stride, L, D, ws, dX, dW, s);
  if ((st = bwd_prepare(X, W, n_rows, H, vocab_local, L, ws, s))) return st;
  for (int64_t c = 0; c < L.n_chunks; ++c) {
    const int64_t v0 = c * L.chunk;
    const int64_t mvalid = (vocab_local - v0) < L.chunk ? (vocab_local - v0) : L.chunk;
    const int64_t mpad = round_up(mvalid, kBM);
    // dZ of this chunk, both layouts.
    if ((st = bwd_dz(X, W, n_rows, H, vocab_local, target, vocab_start, g_max, g_sumexp_m1,
                     grad_output, gout_stride, c, L, dzt, dz, s)))
      return st;
    // dW rows [v0, v0 + mvalid) = dZ^T_c X  (K = tokens, padded with zeros).
    if ((st = launch_gemm_store(0, dzt, L.ldt, mvalid, xt, L.ldt, H, L.ldt, dW + v0 * H, nullptr, H,
                                s)))
      return st;
    // dX (+)= dZ_c W_c  (K = the chunk's padded vocabulary rows).
    int mode;
    if (L.n_chunks == 1) mode = 0;
    else if (c == 0) mode = 1;
    else if (c + 1 < L.n_chunks) mode = 2;
    else mode = 3;
    if ((st = launch_gemm_store(mode, dz, L.chunk, n_rows, wt + v0, L.vpad, H, mpad, dX, acc, H, s)))
      return st;
  }
  return NMCE_OK;
}

}  // extern "C"

namespace nmce {
namespace {

__global__ void hint_assume_kernel(const float* __restrict__ hint, float* __restrict__ assumed) {
  if (threadIdx.x == 0) assumed[0] = usable_hint(hint[0]);
}

int check_fused_args(const void* hidden, const void* weight, int dtype, int64_t n_rows,
                     int64_t hidden_size, int64_t vocab_local, int64_t token_chunk,
                     const void* workspace, int64_t workspace_bytes, FusedLayout& L) {
  if (dtype != NMCE_BF16) return NMCE_EINVAL_DTYPE;
  if (n_rows < 1 || vocab_local < 1 || hidden_size < kBK || hidden_size % kBK != 0)
    return NMCE_EINVAL_SHAPE;
  if (n_rows > (int64_t{1} << 30) || vocab_local > (int64_t{1} << 30)) return NMCE_EINVAL_SHAPE;
  if (!operand_ok(hidden, hidden_size) || !operand_ok(weight, hidden_size))
    return NMCE_EINVAL_ALIGN;
  L = fused_layout(n_rows, hidden_size, vocab_local, token_chunk, device_cus());
  // Per-lane offsets are 32-bit: 256 rows of P^T (dW's K-contiguous A) and 64
  // k-rows of P^T, W and X (MN-contiguous operands) must stay below 2 GiB;
  // ldt < 2^22 covers P^T, and operand_ok above bounds H.
  if (L.ldt >= (int64_t{1} << 22)) return NMCE_EINVAL_SHAPE;
  // The dZ rescale's grid walks the 128-row blocks in its second dimension.
  if (L.vpad / kRsRows > 65535) return NMCE_EINVAL_SHAPE;
  if (!workspace || workspace_bytes < L.total || !aligned16(workspace))
    return NMCE_EINVAL_WORKSPACE;
  return NMCE_OK;
}

}  // namespace
}  // namespace nmce

extern "C" {

int nmce_lmhead_ce_fused_layout(int64_t n_rows, int64_t hidden_size, int64_t vocab_local,
                                int64_t token_chunk, int64_t* layout) {
  if (!layout) return NMCE_EINVAL_PTR;
  if (n_rows < 1 || hidden_size < 1 || vocab_local < 1) return NMCE_EINVAL_SHAPE;
  const FusedLayout L = fused_layout(n_rows, hidden_size, vocab_local, token_chunk, device_cus());
  const int64_t v[NMCE_LMHEAD_FUSED_LAYOUT_FIELDS] = {
      L.total,  L.chunk,    L.n_chunks, L.ldt,     L.vpad,      L.nb,
      L.off_pt, L.off_part, L.off_acc,  L.off_dxp, L.dx_splits, L.off_xt};
  for (int i = 0; i < NMCE_LMHEAD_FUSED_LAYOUT_FIELDS; ++i) layout[i] = v[i];
  return NMCE_OK;
}

int64_t nmce_lmhead_ce_fused_workspace_bytes(int64_t n_rows, int64_t hidden_size,
                                             int64_t vocab_local, int64_t token_chunk,
                                             int compute_units) {
  if (n_rows < 1 || hidden_size < 1 || vocab_local < 1 || compute_units < 0) return -1;
  return fused_layout(n_rows, hidden_size, vocab_local, token_chunk,
                      compute_units > 0 ? compute_units : device_cus()).total;
}

int nmce_hint_assume(const float* hint, float* assumed, void* stream) {
  if (!hint || !assumed) return NMCE_EINVAL_PTR;
  hipLaunchKernelGGL(hint_assume_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream),
                     hint, assumed);
  return launch_status();
}

}  // extern "C"

namespace nmce {
namespace {

// A chunk's statistics; with `loss` the shard is the whole vocabulary and
// they are final.
int fused_chunk_stats(const void* hidden, const void* weight, int dtype, int64_t n_rows,
                      int64_t hidden_size, int64_t vocab_local, const int64_t* target,
                      int64_t vocab_start, int64_t token_chunk, int64_t chunk_index, float* loss,
                      float* row_max, float* row_sumexp_m1, float* target_logit,
                      const float* hint, float* assumed, void* workspace,
                      int64_t workspace_bytes, void* stream) {
  FusedLayout L;
  int st = check_fused_args(hidden, weight, dtype, n_rows, hidden_size, vocab_local, token_chunk,
                            workspace, workspace_bytes, L);
  if (st) return st;
  if (!target || !row_max || !row_sumexp_m1 || !target_logit) return NMCE_EINVAL_PTR;
  if (chunk_index < 0 || chunk_index >= L.n_chunks) return NMCE_EINVAL_SHAPE;
  if ((st = configure_lds())) return st;
  auto s = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  const int64_t t0 = chunk_index * L.chunk;
  const int64_t nc = (n_rows - t0) < L.chunk ? (n_rows - t0) : L.chunk;
  const int64_t H = hidden_size, V = vocab_local;
  float* pmax = reinterpret_cast<float*>(ws + L.off_part);
  float* psum1 = pmax + L.nb * nc;
  float* ptgt = psum1 + L.nb * nc;
  const int64_t tiles = (L.vpad / kBM) * ((nc + kBN - 1) / kBN);
  hipLaunchKernelGGL(lmhead_p_kernel, dim3(static_cast<unsigned>(tiles)), dim3(kThreads),
                     kLdsBytes, s, static_cast<const uint16_t*>(weight),
                     static_cast<const uint16_t*>(hidden) + t0 * H, V, nc, H, target + t0,
                     vocab_start, pmax, psum1, ptgt, reinterpret_cast<uint16_t*>(ws + L.off_pt),
                     L.ldt);
  if ((st = launch_status())) return st;
  const dim3 grid(static_cast<unsigned>((nc + kRedTokens - 1) / kRedTokens));
  const dim3 block(kRedTokens * kRedSlices);
  if (loss)
    hipLaunchKernelGGL(lmhead_reduce_partials_kernel<true>, grid, block, 0, s, pmax, psum1, ptgt,
                       L.nb, nc, row_max + t0, row_sumexp_m1 + t0, target_logit + t0, loss + t0,
                       hint, assumed);
  else
    hipLaunchKernelGGL(lmhead_reduce_partials_kernel<false>, grid, block, 0, s, pmax, psum1, ptgt,
                       L.nb, nc, row_max + t0, row_sumexp_m1 + t0, target_logit + t0, nullptr,
                       nullptr, nullptr);
  return launch_status();
}

}  // namespace
}  // namespace nmce

extern "C" {

int nmce_lmhead_ce_fused_chunk_stats(const void* hidden, const void* weight, int dtype,
                                     int64_t n_rows, int64_t hidden_size, int64_t vocab_local,
                                     const int64_t* target, int64_t vocab_start,
                                     int64_t token_chunk, int64_t chunk_index, float* row_max,
                                     float* row_sumexp_m1, float* target_logit, void* workspace,
                                     int64_t workspace_bytes, void* stream) {
  return fused_chunk_stats(hidden, weight, dtype, n_rows, hidden_size, vocab_local, target,
                           vocab_start, token_chunk, chunk_index, nullptr, row_max, row_sumexp_m1,
                           target_logit, nullptr, nullptr, workspace, workspace_bytes, stream);
}

int nmce_lmhead_ce_fused_chunk_loss(const void* hidden, const void* weight, int dtype,
                                    int64_t n_rows, int64_t hidden_size, int64_t vocab,
                                    const int64_t* target, int64_t token_chunk,
                                    int64_t chunk_index, float* loss, float* g_max,
                                    float* g_sumexp_m1, float* target_logit, const float* hint,
                                    float* assumed, void* workspace, int64_t workspace_bytes,
                                    void* stream) {
  if (n_rows > 0 && (!loss || (assumed && !hint))) return NMCE_EINVAL_PTR;
  return fused_chunk_stats(hidden, weight, dtype, n_rows, hidden_size, vocab, target, 0,
                           token_chunk, chunk_index, loss, g_max, g_sumexp_m1, target_logit, hint,
                           assumed, workspace, workspace_bytes, stream);
}

int nmce_lmhead_ce_fused_chunk_grads(const void* hidden, const void* weight, int dtype,
                                     int64_t n_rows, int64_t hidden_size, int64_t vocab_local,
                                     const int64_t* target, int64_t vocab_start,
                                     int64_t token_chunk, int64_t chunk_index, const float* g_max,
                                     const float* g_sumexp_m1, const float* target_logit,
                                     const float* grad_output, int64_t gout_stride,
                                     float gout_div, void* grad_hidden, void* grad_weight,
                                     void* workspace, int64_t workspace_bytes, void* stream) {
  FusedLayout L;
  int st = check_fused_args(hidden, weight, dtype, n_rows, hidden_size, vocab_local, token_chunk,
                            workspace, workspace_bytes, L);
  if (st) return st;
  if (!target || !g_max || !g_sumexp_m1 || !target_logit || !grad_output || !grad_hidden ||
      !grad_weight)
    return NMCE_EINVAL_PTR;
  if (chunk_index < 0 || chunk_index >= L.n_chunks || gout_stride < 0 || !(gout_div > 0.0f))
    return NMCE_EINVAL_SHAPE;
  if ((st = configure_lds())) return st;
  auto s = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  const int64_t t0 = chunk_index * L.chunk;
  const int64_t nc = (n_rows - t0) < L.chunk ? (n_rows - t0) : L.chunk;
  const int64_t H = hidden_size, V = vocab_local;
  const auto* X = static_cast<const uint16_t*>(hidden);
  const auto* W = static_cast<const uint16_t*>(weight);
  auto* pt = reinterpret_cast<uint16_t*>(ws + L.off_pt);
  const float* pmax = reinterpret_cast<const float*>(ws + L.off_part);
  // dZ^T of the chunk, in place of P^T, and X_c^T beside it (by itself where
  // the grid has no rows left for it).
  auto* xt = reinterpret_cast<uint16_t*>(ws + L.off_xt);
  const int64_t across = (L.ldt + kRsToks - 1) / kRsToks;
  const int64_t row_blocks = L.vpad / kRsRows;
  const int64_t tr_tiles = (L.ldt / kTrTile) * ((H + kTrTile - 1) / kTrTile);
  int64_t tr_rows = (tr_tiles + across - 1) / across;
  if (row_blocks + tr_rows > 65535) {
    if ((st = launch_transpose(X + t0 * H, nc, H, H, xt, L.ldt, s))) return st;
    tr_rows = 0;
  }
  hipLaunchKernelGGL(lmhead_dz_rescale_kernel,
                     dim3(static_cast<unsigned>(across),
                          static_cast<unsigned>(row_blocks + tr_rows)),
                     dim3(256), 0, s, pt, L.ldt, V, nc, pmax, L.nb, g_max + t0, g_sumexp_m1 + t0,
                     target_logit + t0, target + t0, vocab_start, grad_output + t0 * gout_stride,
                     gout_stride, gout_div, static_cast<int>(row_blocks), X + t0 * H, H, xt);
  if ((st = launch_status())) return st;
  // dX rows of the chunk = dZ_c W: both operands read as they lie, k-row
  // (vocabulary) major: dZ^T [vpad, ldt] and W [V, H] (K = the padded
  // vocabulary; dZ^T is zero past V, so W's k-rows stop at V). A chunk with
  // too few tiles to fill the device splits K and sums the fp32 partials.
  uint16_t* dx_rows = static_cast<uint16_t*>(grad_hidden) + t0 * H;
  if (L.n_chunks == 1 && pair_ok(H)) {
    const PairArgs p{pt, L.ldt, L.vpad, W, V, H, xt, nc, dx_rows,
                     reinterpret_cast<float*>(ws + L.off_dxp),
                     static_cast<uint16_t*>(grad_weight),
                     L.dx_splits == 1 ? L.vpad : L.dx_ks, static_cast<int>(L.dx_splits), 0};
    if ((st = launch_pair(p, L.dx_splits > 1, s)) || L.dx_splits == 1) return st;
    const int64_t quads = nc * H / 4;
    hipLaunchKernelGGL(split_sum_bf16_kernel, dim3(static_cast<unsigned>((quads + 255) / 256)),
                       dim3(256), 0, s, p.part, p.splits, nc, H, dx_rows, H);
    return launch_status();
  }
  if (L.dx_splits == 1) {
    if ((st = launch_gemm_store(0, pt, L.ldt, nc, W, H, H, L.vpad, dx_rows, nullptr, H, s,
                                true, true, L.vpad, V)))
      return st;
  } else {
    float* part = reinterpret_cast<float*>(ws + L.off_dxp);
    if ((st = launch_gemm_store(1, pt, L.ldt, nc, W, H, H, L.vpad, nullptr, part, H, s,
                                true, true, L.vpad, V,
                                static_cast<int>(L.dx_splits), L.dx_ks, nc * H)))
      return st;
    const int64_t quads = nc * H / 4;
    hipLaunchKernelGGL(split_sum_bf16_kernel, dim3(static_cast<unsigned>((quads + 255) / 256)),
                       dim3(256), 0, s, part, static_cast<int>(L.dx_splits), nc, H, dx_rows, H);
    if ((st = launch_status())) return st;
  }
  // dW (+)= dZ_c^T X_c: A = dZ^T (K = the chunk's padded tokens contiguous),
  // B = X_c^T [H, ldt], the chunk's hidden rows transposed above (zero past
  // the chunk's tokens), so that both operands are K-contiguous: measured
  // 0.14 ms faster per chunk of 4096 tokens at H = 4096 than reading X as it
  // lies (MN-contiguous), for a transpose of 32 MB. The same products, bit
  // for bit. Accumulated in fp32 across chunks and rounded to bf16 by the
  // last.
  int mode;
  if (L.n_chunks == 1) mode = 0;
  else if (chunk_index == 0) mode = 1;
  else if (chunk_index + 1 < L.n_chunks) mode = 2;
  else mode = 3;
  return launch_gemm_store(mode, pt, L.ldt, V, xt, L.ldt, H, L.ldt,
                           static_cast<uint16_t*>(grad_weight),
                           reinterpret_cast<float*>(ws + L.off_acc), H, s);
}

}  // extern "C"

extern "C" int nmce_gemm_nt_bf16(const void* a, int64_t lda, const void* b, int64_t ldb,
                                 int64_t m, int64_t n, int64_t k, void* c, int c_dtype,
                                 int64_t ldc, void* stream) {
  if (m < 0 || n < 0 || k < 0 || k % kBK != 0) return NMCE_EINVAL_SHAPE;
  if (c_dtype != NMCE_BF16 && c_dtype != NMCE_F32) return NMCE_EINVAL_DTYPE;
  if (m == 0 || n == 0) return NMCE_OK;
  if (!operand_ok(a, lda) || !operand_ok(b, ldb) || lda < k || ldb < k) return NMCE_EINVAL_ALIGN;
  if (!c || ldc < n) return NMCE_EINVAL_PTR;
  if (m > (int64_t{1} << 30) || n > (int64_t{1} << 30)) return NMCE_EINVAL_SHAPE;
  if (k == 0) return NMCE_EINVAL_SHAPE;
  int st = configure_lds();
  if (st) return st;
  return launch_gemm_store(c_dtype == NMCE_BF16 ? 0 : 1, static_cast<const uint16_t*>(a), lda, m,
                           static_cast<const uint16_t*>(b), ldb, n, k,
                           static_cast<uint16_t*>(c), static_cast<float*>(c), ldc,
                           static_cast<hipStream_t>(stream));
}

extern "C" int nmce_gemm_mn_bf16(int a_mn, const void* a, int64_t lda, const void* b,
                                 int64_t ldb, int64_t m, int64_t n, int64_t k, void* c,
                                 int64_t ldc, void* stream) {
  if (m < 0 || n < 0 || k <= 0 || k % kBK != 0) return NMCE_EINVAL_SHAPE;
  if (m == 0 || n == 0) return NMCE_OK;
  const bool a_ok = a_mn ? lda >= (m + 7) / 8 * 8 && 64 * lda < (int64_t{1} << 31) : lda >= k;
  if (!operand_ok(a, lda) || !operand_ok(b, ldb) || !a_ok || ldb < (n + 7) / 8 * 8 ||
      64 * ldb >= (int64_t{1} << 31))
    return NMCE_EINVAL_ALIGN;
  if (!c || ldc < n) return NMCE_EINVAL_PTR;
  if (m > (int64_t{1} << 30) || n > (int64_t{1} << 30)) return NMCE_EINVAL_SHAPE;
  int st = configure_lds();
  if (st) return st;
  return launch_gemm_store(0, static_cast<const uint16_t*>(a), lda, m,
                           static_cast<const uint16_t*>(b), ldb, n, k, static_cast<uint16_t*>(c),
                           nullptr, ldc, static_cast<hipStream_t>(stream), a_mn != 0,
                           true, k, k);
}
