// lm_head projection fused with log-prob / entropy: logits = hidden[T,H] . W[V,H]^T are produced tile by tile on
// the matrix cores and consumed in the epilogue; no [T, V] tensor is needed (the forward may park its tiles for the
// backward, see below).
//
// Replaces FusedLinearForPPO (siirl/utils/experimental/torch_functional.py:20-211) and linear_cross_entropy
// (siirl/utils/kernel/linear_cross_entropy.py:40-117 -> siirl/utils/kernel/kernels.py:507-696,1378-1586); the
// per-tile online-softmax state (max, sum exp, sum x*exp) is the one of kernels.py:254-266,343-350.
//
// One GEMM core, C[M,N] = A[M,K] . B[N,K]^T, 16-bit operands, fp32 accumulation, 128 x 256 x 64 workgroup tile,
// 4 waves of 128 x 64 (8 x 4 MFMA 16x16x32 tiles, 128 accumulator registers each), two workgroups per CU.  The 16x16x32 shape moves
// half the accumulator data per flop of the 32x32x16 one; with random operand bits the matrix cores then sustain
// 1.79 instead of 1.62 PFLOP/s in an LDS-fed loop at this part's power limit, which is what sets these kernels' time.
//   * A (K-major rows) goes global -> LDS by DMA (global_load_lds_dwordx4, no staging registers, no ds_write)
//     into a ring of four 16 KB stages.  Rows are unpadded; 16-byte chunks are XOR-swizzled by (row / 2) % 8 so
//     that the ds_read_b128 fragment reads are conflict-free.  A stage is issued three K-steps before it is read
//     and published (barrier) one step before, so the first fragments of the next step are read ahead of the
//     barrier and the matrix cores do not drain at it.
//   * B never touches the LDS: it is prepared once per call in the MFMA operand's lane order ("fragment-packed")
//     and each lane loads its 16-byte operands straight into registers, one K-step ahead.
//   * all loads of the main loop are inline asm with hand-placed s_waitcnt vmcnt: the compiler's own tracking
//     would wait for every outstanding DMA before each LDS read.
// Four epilogues: softmax partials (forward), packed dlogits (backward), fp32 sums (d hidden), a store in the operands'
// type (d weight).  The backward walks the vocabulary in groups of columns: recompute the group's logits into
// dlogits[T, group], then dH += dlogits . W_group and dW_group = dlogits^T . hidden as two more runs of the same core.
// dlogits are written fragment-packed, once, and serve both: as d hidden's B operand (its A is W as it lies in memory,
// given by K-rows) and as d weight's A operand (its B a packed transposed copy of hidden).  A transposed copy of W, which
// d hidden took as its B operand, cost 350 us a call at H=3584, V=152064 whatever the token count, and dlogits row by
// row, as its A operand, 128 bytes of each of 256 rows per K-step: T=1500, H=2048, V=50257 503 -> 300 us.
// Optionally the forward also parks the fp32 accumulator tiles in memory (4 bytes per logit, in the accumulator's
// own lane order, so stores and loads are whole 1 KB wave accesses); the backward then replays the tiles through
// the same dlogits epilogue instead of recomputing the GEMM: a third of the backward's matrix work is traded for
// one streaming pass.
#include "common.hpp"

#include <type_traits>

namespace siirl {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// Workgroup tile 128 x 256 x 64, 4 waves along N, one per SIMD; two workgroups per CU (the LDS rings), which run through
// their prologues and epilogues at different times.  Against tiles of 256 x 256 with 8 waves and one workgroup per CU, us:
// forward T=200 345 -> 297, T=3001 (H=2048, fp16) 1710 -> 1660, T=16384 12990 -> 12540; recompute T=200 334 -> 289, 8192
// columns at T=16384 717 -> 684; d weight T=200 542 -> 488, T=16384 the same (H=3584, V=152064 bf16 where not said).
constexpr int BM = 128, BN = 256, BK = 64;
constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kWavesPerSimd = 2;
constexpr int MI = BM / 16, NJ = BN / (kWaves * 16);  // 16x16 MFMA tiles per wave: 8 x 4
constexpr int KS = BK / 32;                           // K = 32 slices per K-step
static_assert(MI == 8 && NJ == 4 && KS == 2, "the K-step schedule is written for 8 x 4 tiles and two K slices");
constexpr int kRowBytes = BK * 2;          // unpadded rows, 16-byte chunks XOR-swizzled by (row / 2) % 8
constexpr int kStageBytes = BM * kRowBytes;  // 16 KB of A: B goes global -> registers
constexpr int kStages = 4;
constexpr int kSmemBytes = kStages * kStageBytes;
constexpr int kDmaPerWave = kStageBytes / 1024 / kWaves;  // 1 KB per wave instruction
// The backward walks the vocabulary in groups: the group's logits are recomputed into dlogits, then d hidden and
// d weight are updated from them.  A group is 65536 columns at 16384 tokens and above (512 x 64 tiles of dlogits and
// 512 x 14 of d weight at H = 3584 fill whole rounds of the 256 CUs, two workgroups each; 4 / 8 / 19 times 8192 columns measured 34.4 / 33.7
// / 33.2 ms per backward at T=16384, V=152064), and as many times more with fewer tokens as keep the same bytes of
// dlogits: at T=200, V=152064 one group instead of three.
constexpr int64_t kGroupCols = 65536, kGroupTokens = 16384;
constexpr int kPadBlocks = 2;  // extra 1 KB blocks per 16 tokens of D: keeps the token blocks of a stage off a power-of-two
                               // stride, which would put them all in one memory channel

struct GemmArgs {
  const uint16_t* A;
  int64_t lda;
  const u32x4* Bp;  // fragment-packed B (see pack layout), already offset to the first K block of this GEMM
  int64_t kb_total; // 32-wide K blocks per 16-row block of the packed buffer
  int M, N, K;  // K is a multiple of BK; rows beyond M are clamped on load and masked by the epilogue
  int tiles_m, tiles_n;
  int splits;  // K is cut into `splits` runs of K-steps; run s is tile column tn + s * tiles_n of the raster
  int blk_m;   // tiles along M of an XCD's block of 32 tiles
  int chunk;   // tile places per XCD, or 0: whole blocks in turn
  // A_KROWS: a last K-step that A does not fill is read from a copy of its rows, padded with zeros to BK of them
  const uint16_t* A_tail;
  int kt_tail;  // its index (the last step), or past it
};
// How the A operand lies in memory: [M][K] with K contiguous; [K][M] with M contiguous; or fragment-packed as the B
// operand of a GEMM whose N is this one's K and whose K is this one's M (16-row blocks along K, 32-wide blocks along M).
enum { A_ROWS = 0, A_KROWS = 1, A_PACKED = 2 };

struct TileCoord {
  int tm, tn;
  bool valid;
};
// XCD-aware rasterisation.  Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2, so
// workgroup id runs on XCD id % 8 as that XCD's (id / 8)-th workgroup.  The tile grid is cut into blocks of
// blk_m x blk_n tiles (32 tiles: half of one XCD's resident set; blk_m is the launch's choice among the powers of two); block b
// goes to XCD b % 8 and its tiles to 32 consecutive workgroups of that XCD, so the workgroups sharing an L2 at any
// time share blk_m A-tiles and blk_n B-tiles instead of streaming 32 different A-tiles.  Blocks sweep M fastest
// inside a strip of blk_n N-tiles, which keeps a strip's B-tiles hot across the 8 XCDs.  (Sweeping N fastest instead, which would stream the big
// operand from memory once rather than once per strip, measured 4 % slower forward and 8-17 % slower backward GEMMs
// at T=16384, H=3584, V=152064: the L2 reuse inside a strip matters more than the bytes from memory.)
constexpr int kXcd = 8, kBlkTiles = 32;
// With few blocks that hand-out is uneven (9 or 10 blocks leave one or two XCDs a second round while the others stop): up
// to kChunkBlocks of them, an XCD takes an eighth of all their tiles instead, consecutive in the same order (`chunk` tile
// places).  d hidden at T=200, H=3584, V=152064 (28 x 18 tiles): 391 us in blocks of 8 x 4 in turn, 290 us as 32 x 1, chunked.
constexpr int64_t kChunkBlocks = 64;
inline int64_t raster_grid(GemmArgs& g) {
  const int blk_n = kBlkTiles / g.blk_m;
  const int64_t blocks = (int64_t)((g.tiles_m + g.blk_m - 1) / g.blk_m) * (((int64_t)g.tiles_n * g.splits + blk_n - 1) / blk_n);
  g.chunk = blocks <= kChunkBlocks ? (int)((blocks * kBlkTiles + kXcd - 1) / kXcd) : 0;
  return g.chunk ? (int64_t)g.chunk * kXcd : (blocks + kXcd - 1) / kXcd * kXcd * kBlkTiles;
}
__device__ __forceinline__ TileCoord tile_of(const GemmArgs& g, int id) {
  const int blk_m = g.blk_m, blk_n = kBlkTiles / blk_m;
  const int xcd = id % kXcd, l = id / kXcd;
  const int at = g.chunk ? xcd * g.chunk + l : ((l / kBlkTiles) * kXcd + xcd) * kBlkTiles + l % kBlkTiles;
  const int blk = at / kBlkTiles, j = at % kBlkTiles;
  const int mb = (g.tiles_m + blk_m - 1) / blk_m;
  const int tm = (blk % mb) * blk_m + j % blk_m;
  const int tn = (blk / mb) * blk_n + j / blk_m;
  return {tm, tn, tm < g.tiles_m && tn < g.tiles_n * g.splits};
}

// Accumulator coordinates of lane `lane` in wave wn: element r (0..3) of acc[i][j] is
//   row = i*16 + (lane/16)*4 + r ,  col = wn*64 + j*16 + lane%16   (tile-relative)
__device__ __forceinline__ int acc_row(int i, int r, int lane) {
  return i * 16 + (lane >> 4) * 4 + r;
}
__device__ __forceinline__ int acc_col(int wn, int j, int lane) { return wn * (NJ * 16) + j * 16 + (lane & 15); }
// An epilogue with kRowsPerLane takes the accumulator the other way round (the MFMA's operands are swapped): a lane owns
// the rows row_of_lane(i) and, with B packed in the column order of transpose_pack_b_kernel, 8 consecutive columns from
// col_of_lane(j) on of each pair j, j + 1 (j even) of N-tiles: element r of acc[i][j] is column col_of_lane(j) + r.
__device__ __forceinline__ int row_of_lane(int i, int lane) { return i * 16 + (lane & 15); }
__device__ __forceinline__ int col_of_lane(int wn, int j, int lane) {
  return wn * (NJ * 16) + (j >> 1) * 32 + (lane >> 4) * 8 + (j & 1) * 4;
}

// m0 (the DMA's LDS base) is a reserved register: naming it in a clobber list is right but draws a warning
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// F16: the 16-bit operands are IEEE half instead of bf16 (the same data movement, the other MFMA)
// A_ONCE (gemm_once_kernel): one token tile, so that W is read once, and W larger than the memory-side cache: its loads are non-temporal, or
// what they bring in would push out what every workgroup reads, the B operand, and itself before anyone asks for it again.
// Forward / recompute / d hidden (us): T=200, H=3584, V=152064 297 / 281 / 280 -> 256 / 278 / 292 (the ordinary loads find the
// end of W that the product before left in the cache: alone they take 317), T=256, H=2048, V=151936 fp16 200 / 226 / 170 ->
// 155 / 175 / 172, T=50, H=2048, V=100000 175 / 125 / 94 -> 114 / 123 / 112.  A smaller W stays in the cache from one product
// to the next: T=64, H=2048, V=50257 79 / 45 / 47 -> 60 / 64 / 55.  With more token tiles W comes from the L2 to all but the
// first of them: T=400 437 / 454 / 618 -> 479 / 514 / 702.
template <class Epi, int AL, bool F16, bool A_ONCE>
__device__ __forceinline__ void gemm_nt_tile(GemmArgs g, Epi epi) {
  static_assert(!(F16 && Epi::kRowsPerLane), "the gradient GEMMs multiply bf16");
  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wn = tid >> 6;
  TileCoord tc = tile_of(g, blockIdx.x);
  if (!tc.valid) return;
  // (integer divisions leave their results in vector registers; these are the same in every lane)
  tc.tm = __builtin_amdgcn_readfirstlane(tc.tm);
  tc.tn = __builtin_amdgcn_readfirstlane(tc.tn);
  const int split = __builtin_amdgcn_readfirstlane(tc.tn / g.tiles_n);
  const int m0 = tc.tm * BM, n0 = (tc.tn - split * g.tiles_n) * BN;
  // this workgroup's run of K-steps (the host keeps every run non-empty)
  const int kt_per = __builtin_amdgcn_readfirstlane((g.K / BK + g.splits - 1) / g.splits);
  const int kt_first = split * kt_per;
  const int KT = (g.K / BK - kt_first < kt_per) ? g.K / BK - kt_first : kt_per;

  // A: global -> LDS by DMA (global_load_lds_dwordx4): wave instruction I = w * kDmaPerWave + i fills the 1 KB
  // [I * 1024, I * 1024 + 1024) of the stage.
  //   A[M][K] (A_ROWS): 16-byte slot sl = I * 64 + lane holds row sl / 8, chunk (sl % 8) ^ ((row / 2) % 8).  Rows
  //     past the matrix edge are clamped to the last row.
  //   A[K][M] (A_KROWS): the stage is 64 K-rows of BM * 2 bytes; with c = BM / 8 chunks a row, slot sl holds
  //     K-row sl / c, chunk (sl % c) ^ 2 * (row % 4), i.e. the 32-byte segments of a row are XOR-swizzled by the row so
  //     that the four K-rows a transposing fragment read touches lie in different banks.  A chunk past M (a multiple of
  //     64) is read as the tile's first one and only reaches output rows that the epilogue masks.
  //   A_PACKED: the stage is 4 x BM / 32 packed blocks of 1 KB, one per wave instruction.  Slot 16 q + t of a block
  //     holds the 8 M-entries from 8 q on of K-row t ^ 4 * (q % 2): the two chunks of a transposing fragment read that
  //     are 256 bytes apart then lie in different banks.  Blocks past M are inside the buffer (its pitch covers tiles).
  const int wu = __builtin_amdgcn_readfirstlane(wn);
  const char* gA;
  int64_t a_step;  // bytes from one K-step to the next
  if constexpr (AL == A_ROWS) {
    gA = reinterpret_cast<const char*>(g.A + (int64_t)m0 * g.lda + (int64_t)kt_first * BK);
    a_step = (int64_t)BK * 2;
  } else if constexpr (AL == A_KROWS) {
    gA = reinterpret_cast<const char*>(g.A + (int64_t)kt_first * BK * g.lda + m0);
    a_step = (int64_t)BK * g.lda * 2;
  } else {  // lda: 32-wide blocks from one 16-row block to the next
    gA = reinterpret_cast<const char*>(g.A) + ((int64_t)kt_first * (BK / 16) * g.lda + (m0 >> 5)) * 1024;
    a_step = (int64_t)(BK / 16) * g.lda * 1024;
  }
  uint32_t offA[kDmaPerWave];
#pragma unroll
  for (int i = 0; i < kDmaPerWave; ++i) {
    const int I = wu * kDmaPerWave + i, sl = I * 64 + lane;
    if constexpr (AL == A_KROWS) {
      constexpr int kRowChunks = BM / 8;
      const int row = sl / kRowChunks;
      int ch = (sl % kRowChunks) ^ ((row & 3) << 1);
      if (m0 + ch * 8 >= g.M) ch = 0;
      offA[i] = (uint32_t)row * (uint32_t)g.lda * 2u + ch * 16;
    } else if constexpr (AL == A_PACKED) {
      constexpr int kBlocks = BM / 32;
      offA[i] = ((uint32_t)(I / kBlocks) * (uint32_t)g.lda + I % kBlocks) * 1024u + (lane ^ ((lane >> 2) & 4)) * 16;
    } else {
      int row = sl >> 3;
      const int ch = (sl & 7) ^ ((row >> 1) & 7);
      row = (m0 + row < g.M) ? row : g.M - 1 - m0;
      offA[i] = (uint32_t)row * (uint32_t)g.lda * 2u + ch * 16;
    }
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  // B: fragment-packed, one 16-byte load per lane per MFMA operand, no LDS.  N-tile j of the wave, K slice s of the
  // K-step: chunk ((n0 / 16 + wn * NJ + j) * kb_total + kt * KS + s) * 64 + lane.
  const char* gB =
      reinterpret_cast<const char*>(g.Bp + ((int64_t)(n0 >> 4) * g.kb_total + (int64_t)kt_first * KS) * 64);
  uint32_t offB[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) offB[j] = (uint32_t)(((wn * NJ + j) * g.kb_total * 64 + lane) * 16);

  floatx4 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

  u32x4 b0[NJ][KS], b1[NJ][KS];
  const int kt_tail = g.kt_tail - kt_first;
  const int64_t to_tail = reinterpret_cast<const char*>(g.A_tail + m0) - (gA + (int64_t)kt_tail * a_step);  // (kt_tail is the last step)
  auto dma = [&](int stage, int kt, int i0 = 0, int i1 = kDmaPerWave) {
    // (No branch around the loads, and no register to spare: where the compiler copies or spills the B registers it does
    // so before their wait.  The build reads its own listing for that, siirl_amd/asm_check.py, and refuses it.)
    const char* base = gA + (int64_t)kt * a_step;
    if (AL == A_KROWS) base += to_tail & (int64_t)__builtin_amdgcn_readfirstlane((kt - kt_tail) >> 31 ^ -1);
#pragma unroll
    for (int i = i0; i < i1; ++i) {
      const uint32_t dst = lds0 + stage * kStageBytes + (wu * kDmaPerWave + i) * 1024;
      if constexpr (A_ONCE)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(dst), "v"(offA[i]), "s"(base) : "m0", "memory");
      else
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(offA[i]), "s"(base) : "m0", "memory");
    }
  };
  auto bload = [&](u32x4 (&b)[NJ][KS], int kt, int j) {
    const char* base = gB + (int64_t)kt * (KS * 1024);
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(b[j][0]) : "v"(offB[j]), "s"(base));
    asm volatile("global_load_dwordx4 %0, %1, %2 offset:1024" : "=v"(b[j][1]) : "v"(offB[j]), "s"(base));
  };
  // waits until only this wave's last N loads are in flight (N = kDmaPerWave: one stage of DMA) and ties the B
  // registers to the wait
  static_assert(NJ * KS == 8 && kDmaPerWave % 2 == 0, "see the load schedule of a K-step");
  auto bwait = [&](u32x4 (&b)[NJ][KS], auto in_flight) {
    asm volatile("s_waitcnt vmcnt(%[n])"
                 : "+v"(b[0][0]), "+v"(b[0][1]), "+v"(b[1][0]), "+v"(b[1][1]), "+v"(b[2][0]), "+v"(b[2][1]),
                   "+v"(b[3][0]), "+v"(b[3][1])
                 : [n] "n"(decltype(in_flight)::value)
                 : "memory");
  };
  using OneStage = std::integral_constant<int, kDmaPerWave>;
  using Nothing = std::integral_constant<int, 0>;

#pragma unroll
  for (int j = 0; j < NJ; ++j) bload(b0, 0, j);
  dma(0, 0);
  dma(1, KT > 1 ? 1 : 0);
  dma(2, KT > 2 ? 2 : 0);
  bwait(b0, OneStage{});
  __syncthreads();

  // A fragments of MFMA group gq = 2 * s + hf: K slice s (32 columns), row blocks hf * 4 .. hf * 4 + 3 of the wave's
  // eight 16-row blocks.  A_ROWS: lane (m = lane % 16, 8-column chunk lane / 16 of the slice) reads its 8
  // consecutive K entries as one 16-byte chunk of row m.  Otherwise the stage holds K-rows, so the 8 entries come
  // from two transposing reads (ds_read_b64_tr_b16): in each block of 16 lanes, lane 4 e + c addresses the 8 bytes of
  // K-row e, M-chunk c, and receives the entries of K-rows 0..3 at M = its own index in the block; block lane / 16
  // takes the 8 K-rows lane / 16 * 8 .. + 7 of the slice.
  const int m15 = lane & 15, kq = lane >> 4, sw = m15 >> 1;
  const int frag_row = m15 * kRowBytes;
  int xk[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) xk[s] = frag_row + (((s * 4 + kq) ^ sw) << 4);
  const int tq = m15 >> 2;
  const int xt0 = (kq * 8 + tq) * (BM * 2) + (lane & 3) * 8 + (tq << 5);  // row block ii: xt0 ^ (ii << 5)
  // A_PACKED: K-row t = (kq % 2) * 8 + tq of the 16-row block kq / 2 of the slice, the M-chunk's 8 bytes of its 16
  const int mc = lane & 3;
  const int xp0 = (kq >> 1) * (BM * 32) + ((kq & 1) * 8 + (mc & 2) * 2 + tq) * 16 + (mc >> 1) * 256 + (mc & 1) * 8;

  // step kt: stage kt % 4 is read; B(kt + 1) and DMA(kt + 3) are issued; the barrier at the end publishes stage
  // (kt + 2) % 4, whose DMA was issued one step earlier, and frees stage kt % 4 for DMA(kt + 4).  The last three steps
  // have nothing left to fetch by DMA and wait for all loads instead; the last one fetches and publishes nothing.
  // A fragments are read one MFMA group ahead; the group after the last one of a step is the first of the next
  // step, whose stage was published by the previous barrier, so the reads cross the barrier.
  bf16x8 afa[4], afb[4];
  auto fread = [&](bf16x8 (&af)[4], int stage, int gq) {
    const char* cur = smem + stage * kStageBytes;
    const int s = gq >> 1, hf = gq & 1;
    if constexpr (AL != A_ROWS) {
      typedef short s16x4 __attribute__((ext_vector_type(4)));
      typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        // K-rows 0 .. 3 and 4 .. 7 of the lane's eight
        const int in_stage = s * (32 * BM * 2) + (AL == A_KROWS ? hf * 128 : (hf * 4 + ii) * 512);
        const char* at = cur + in_stage + (AL == A_KROWS ? xt0 ^ (ii << 5) : xp0);
        const char* at4 = AL == A_KROWS ? at + 4 * BM * 2 : cur + in_stage + (xp0 ^ 64);
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at4));
        af[ii] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    } else {
#pragma unroll
      for (int ii = 0; ii < 4; ++ii)
        af[ii] = *reinterpret_cast<const bf16x8*>(cur + xk[s] + (hf * 4 + ii) * 16 * kRowBytes);
    }
  };
  auto mma = [&](bf16x8 (&af)[4], u32x4 (&bc)[NJ][KS], int gq) {
    const int s = gq >> 1, hf = gq & 1;
#pragma unroll
    for (int ii = 0; ii < 4; ++ii)
#pragma unroll
      for (int jj = 0; jj < NJ; ++jj) {
        // boustrophedon over the N-tiles: consecutive MFMAs always share one operand (0.5-0.8 % faster at T=16384,
        // H=3584, V=152064 than restarting at N-tile 0 for every row block: fewer operand wires toggle)
        const int j = (ii & 1) ? NJ - 1 - jj : jj;
        floatx4& c = acc[hf * 4 + ii][j];
        if constexpr (F16)
          c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, af[ii]), __builtin_bit_cast(f16x8, bc[j][s]), c, 0, 0, 0);
        else if constexpr (Epi::kRowsPerLane)
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, bc[j][s]), af[ii], c, 0, 0, 0);
        else
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[ii], __builtin_bit_cast(bf16x8, bc[j][s]), c, 0, 0, 0);
      }
  };
  fread(afa, 0, 0);
  // One K-step: four groups of 16 MFMAs.  The 12 vector-memory instructions are spread over the step (B for two
  // N-tiles before each of the first two groups, half of the DMA before each of the last two) instead of being issued
  // in one burst, and the wave raises its priority while it issues MFMAs so that its SIMD partner's loads do not
  // delay them.
  auto mma_prio = [&](bf16x8 (&af)[4], u32x4 (&bc)[NJ][KS], int gq) {
    __builtin_amdgcn_s_setprio(1);
    mma(af, bc, gq);
    __builtin_amdgcn_s_setprio(0);
  };
  enum { STEP_MAIN, STEP_TAIL, STEP_LAST };
  auto step = [&](auto kind, int kt, u32x4 (&bc)[NJ][KS], u32x4 (&bn)[NJ][KS]) {
    constexpr int kKind = decltype(kind)::value;
    const int stage = kt & 3;
    if constexpr (kKind != STEP_LAST)
#pragma unroll
      for (int j = 0; j < NJ / 2; ++j) bload(bn, kt + 1, j);
    fread(afb, stage, 1);
    mma_prio(afa, bc, 0);
    if constexpr (kKind != STEP_LAST)
#pragma unroll
      for (int j = NJ / 2; j < NJ; ++j) bload(bn, kt + 1, j);
    fread(afa, stage, 2);
    mma_prio(afb, bc, 1);
    if constexpr (kKind == STEP_MAIN) dma((stage + 3) & 3, kt + 3, 0, kDmaPerWave / 2);
    fread(afb, stage, 3);
    mma_prio(afa, bc, 2);
    if constexpr (kKind == STEP_MAIN) dma((stage + 3) & 3, kt + 3, kDmaPerWave / 2, kDmaPerWave);
    if constexpr (kKind != STEP_LAST) fread(afa, (stage + 1) & 3, 0);
    mma_prio(afb, bc, 3);
    if constexpr (kKind == STEP_MAIN) bwait(bn, OneStage{});
    if constexpr (kKind == STEP_TAIL) bwait(bn, Nothing{});
    if constexpr (kKind != STEP_LAST) __syncthreads();
  };
  using Main = std::integral_constant<int, STEP_MAIN>;
  using Tail = std::integral_constant<int, STEP_TAIL>;
  using Last = std::integral_constant<int, STEP_LAST>;
  // The pairs of main steps swap the two B register sets by name.  What follows them moves the 32 registers instead: with
  // a copy of the tail for each parity the compiler loses the accumulators' places where the copies join (1773 spills).
  auto take_over = [&]() {
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int s = 0; s < KS; ++s) b0[j][s] = b1[j][s];
  };
  int kt = 0;
  for (; kt + 5 <= KT; kt += 2) {
    step(Main{}, kt, b0, b1);
    step(Main{}, kt + 1, b1, b0);
  }
  if (kt + 4 <= KT) {
    step(Main{}, kt++, b0, b1);
    take_over();
  }
  if (KT >= 3) {
    step(Tail{}, kt++, b0, b1);
    take_over();
  }
  if (KT >= 2) {
    step(Tail{}, kt++, b0, b1);
    take_over();
  }
  step(Last{}, kt, b0, b1);
  // nothing is in flight here but, with fewer than three K-steps, the spare DMA of the prologue; the epilogue reuses
  // the LDS
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  int em0 = m0, en0 = n0, el = lane;
  asm volatile("" : "+s"(em0), "+s"(en0), "+v"(el));  // (no address of the epilogue is computed before the main loop)
  epi(acc, em0, en0, tc.tm, split, wn, el, tid, smem);
}

template <class Epi, int AL = A_ROWS, bool F16 = false>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kWavesPerSimd, kWavesPerSimd))) void gemm_nt_kernel(GemmArgs g, Epi epi) {
  gemm_nt_tile<Epi, AL, F16, false>(g, epi);
}

template <class Epi, int AL = A_ROWS, bool F16 = false>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kWavesPerSimd, kWavesPerSimd))) void gemm_once_kernel(GemmArgs g, Epi epi) {
  gemm_nt_tile<Epi, AL, F16, true>(g, epi);
}
#pragma clang diagnostic pop

// The same product for a K of at most four K-steps and a packed A (d weight at up to 256 tokens).  A tile of it is one to
// four K-steps of matrix work between a fetch and a store of 64 KB, and gemm_nt_kernel starts a workgroup for each: at
// T=200, H=3584, V=152064 it wrote d weight at 2.2 TB/s.  Here the four stages of the ring hold a row tile's whole K, and
// the workgroup walks n_per tiles along N with it: no barrier after the first, so that its waves, and the CU's other
// workgroup, multiply while some of them store.  What remains is matrix work
// (200 us at the rate of the large GEMMs) and the store of C (180 us) hardly overlapping.  d weight, us: T=200 485 -> 440, and
// 43 at T=64, H=2048, V=50257 (4.8 TB/s).  Fetching B two steps ahead with branch-free stores, so that no fetch waits behind a
// store, measured the same (439); non-temporal stores 454, and 129 at T=64.
constexpr int kShortSteps = kStages;
template <class Epi>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kWavesPerSimd, kWavesPerSimd))) void gemm_short_k_kernel(
    GemmArgs g, int n_per, Epi epi) {
  static_assert(Epi::kRowsPerLane, "the MFMA operands are swapped");
  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wn = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tm = blockIdx.x % g.tiles_m, tn0 = (int)(blockIdx.x / g.tiles_m) * n_per;
  const int tn1 = tn0 + n_per < g.tiles_n ? tn0 + n_per : g.tiles_n;
  const int m0 = tm * BM, KT = g.K / BK;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const char* gA = reinterpret_cast<const char*>(g.A) + (int64_t)(m0 >> 5) * 1024;
  for (int kt = 0; kt < KT; ++kt)
#pragma unroll
    for (int i = 0; i < kDmaPerWave; ++i) {  // slots as in gemm_nt_kernel, A_PACKED
      constexpr int kBlocks = BM / 32;
      const int I = wn * kDmaPerWave + i;
      const char* base = gA + ((int64_t)(kt * (BK / 16) + I / kBlocks) * g.lda + I % kBlocks) * 1024;
      const uint32_t dst = lds0 + kt * kStageBytes + I * 1024, off = (lane ^ ((lane >> 2) & 4)) * 16;
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off), "s"(base) : "m0", "memory");
    }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  const int kq = lane >> 4, mc = lane & 3, tq = (lane & 15) >> 2;
  const char* frag = smem + (kq >> 1) * (BM * 32) + ((kq & 1) * 8 + (mc & 2) * 2 + tq) * 16 + (mc >> 1) * 256 + (mc & 1) * 8;
  const char* frag4 = smem + ((uint32_t)(frag - smem) ^ 64u);
  auto fetch = [&](u32x4 (&b)[NJ][KS], int tn, int kt) {
    const u32x4* p = g.Bp + ((int64_t)(tn * (BN / 16) + wn * NJ) * g.kb_total + kt * KS) * 64 + lane;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int s = 0; s < KS; ++s) b[j][s] = p[(int64_t)j * g.kb_total * 64 + s * 64];
  };
  u32x4 b[NJ][KS], bn[NJ][KS];
  fetch(b, tn0, 0);
  for (int tn = tn0; tn < tn1; ++tn) {
    floatx4 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int kt = 0; kt < KT; ++kt) {
      // the next step's B, of this tile or the next one (past the end: of the last step again)
      const bool same = kt + 1 < KT, more = same || tn + 1 < tn1;
      fetch(bn, more && !same ? tn + 1 : tn, same ? kt + 1 : (more ? 0 : kt));
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          typedef short s16x4 __attribute__((ext_vector_type(4)));
          typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
          const int at = kt * kStageBytes + s * (32 * BM * 2) + i * 512;
          const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(frag + at));
          const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(frag4 + at));
          const bf16x8 af = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
          for (int j = 0; j < NJ; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b[j][s]), af, acc[i][j], 0, 0, 0);
        }
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int s = 0; s < KS; ++s) b[j][s] = bn[j][s];
    }
    epi(acc, m0, tn * BN, tm, 0, wn, lane, tid, smem);
  }
}

// ------------------------------------------------------------------------------ parked accumulator tiles

// Tile (tm, tn) of the forward GEMM occupies kQuads * kThreads 16-byte slots; slot c * kThreads + tid holds thread
// tid's acc[i][j] (four registers), c = i * NJ + j.  A wave instruction therefore moves one contiguous KB, and the
// tile can be handed to any epilogue exactly as the main loop would have left it.
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kQuads = MI * NJ;
constexpr int64_t kSavedTileBytes = (int64_t)kQuads * kThreads * 16;  // BM * BN * 4
__device__ __forceinline__ f32x4* saved_tile(float* base, int tm, int tn, int tiles_n) {
  return reinterpret_cast<f32x4*>(base) + ((int64_t)tm * tiles_n + tn) * (kQuads * kThreads);
}

// Runs an epilogue over parked tiles: workgroup b takes tile (tm_first + b / tiles_n, b % tiles_n) and calls the
// epilogue with vocabulary row m0 counted from the first tile row of the launch.
template <class Epi>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kWavesPerSimd, kWavesPerSimd))) void replay_tiles_kernel(
    const float* __restrict__ saved, int tiles_n, int tm_first, Epi epi) {
  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wn = tid >> 6;
  const int tml = blockIdx.x / tiles_n, tn = blockIdx.x - tml * tiles_n;
  const f32x4* src = saved_tile(const_cast<float*>(saved), tm_first + tml, tn, tiles_n) + tid;
  floatx4 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_nontemporal_load(src + (i * NJ + j) * kThreads);
  epi(acc, tml * BM, tn * BN, tml, 0, wn, lane, tid, smem);
}

// ------------------------------------------------------------------------------ epilogue: softmax partials

// The two fused GEMMs run "transposed": M is the vocabulary (A = W), N the tokens (B = hidden).  In the MFMA
// accumulator layout a lane then owns one token (column) and its registers run over vocabulary rows, so the
// softmax reductions over the vocabulary are in-register, followed by two exchanges between the four lanes that
// share a token -- no 16-lane butterfly per row.
//
// Per token of the tile: mx = max_v z, s = sum exp(z - mx), t = sum z * exp(z - mx) over the tile's 128
// vocabulary rows, z = acc * inv_T; one (mx, s, t) per token is written to part[tm][.][token].
struct SoftmaxPartialsEpi {
  static constexpr bool kRowsPerLane = false;
  float inv_T;
  int T, V;
  float* part;  // [tiles_m][3][T]
  float* save;  // null, or the parked accumulator tiles (see saved_tile)
  int tiles_n;
  // The (mx, s, t) of each of the wave's tokens.  Works on the raw accumulator a (z = a * inv_T):
  // a maximum, one fused multiply-add, one exp2 and two accumulations per logit; no matrix work runs beside this, so
  // its length counts in full (FULL: no vocabulary row of the tile is past the end, nothing is compared or selected).
  template <bool FULL>
  __device__ __forceinline__ void reduce(floatx4 (&acc)[MI][NJ], int m0, int n0, int wn, int lane, float* o) const {
    const float ninf = -__builtin_inff();
    const float ek = inv_T * kLog2e;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      float mx = ninf;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (FULL || m0 + acc_row(i, r, lane) < V) mx = fmaxf(mx, acc[i][j][r]);
      mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
      mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
      float s = 0.f, t = 0.f;
      if (mx > ninf) {
        const float nmk = -mx * ek;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if (!FULL && m0 + acc_row(i, r, lane) >= V) continue;
            const float e = fast_exp2(fmaf(acc[i][j][r], ek, nmk));
            s += e;
            t = fmaf(acc[i][j][r], e, t);
          }
      }
      s += __shfl_xor(s, 16, kWave);
      t += __shfl_xor(t, 16, kWave);
      s += __shfl_xor(s, 32, kWave);
      t += __shfl_xor(t, 32, kWave);
      const int tok = n0 + acc_col(wn, j, lane);
      if (lane < 16 && tok < T) {
        o[tok] = mx * inv_T;
        o[(int64_t)T + tok] = s;
        o[2 * (int64_t)T + tok] = t * inv_T;
      }
    }
  }
  __device__ __forceinline__ void operator()(floatx4 (&acc)[MI][NJ], int m0, int n0, int tm, int split, int wn, int lane,
                                             int tid, char* smem) const {
    // Parking takes the forward at T=16384, H=3584, V=152064 from 12.6 to 13.9 ms for 9.97 GB.
    if (save) {
      f32x4* dst = saved_tile(save, tm, n0 / BN, tiles_n) + tid;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) dst[(i * NJ + j) * kThreads] = acc[i][j];
    }
    float* o = part + (int64_t)tm * 3 * T;
    if (m0 + BM <= V)
      reduce<true>(acc, m0, n0, wn, lane, o);
    else
      reduce<false>(acc, m0, n0, wn, lane, o);
  }
};

// ------------------------------------------------------------------------------ epilogue: dlogits

// d raw_logit = inv_T * ( g_lp * (1[v == y] - p) - g_h * p * (z - ex) ),  p = exp(z - lse), z = acc * inv_T,
// written as bf16, fragment-packed like a B operand B[n = token][k = v]: block (token / 16, v / 32) is the 1 KB
// D + ((token / 16) * kb_total + v / 32) * 1 KB.  v is group-relative and is the M dimension of this GEMM.  Rows v in
// [Vs, Vpad) are written as zeros: they are K-padding of the d-hidden GEMM that consumes D; so are the tokens in
// [T, Tpad) for d weight.  A lane owns one token, so the per-token coefficients are loaded once per lane, and a wave
// writes D in runs of 512 bytes.  The one layout serves both consumers: d hidden takes it as its B operand, d weight
// as an A operand given by packed K-rows.
struct DlogitsEpi {
  static constexpr bool kRowsPerLane = false;
  float inv_T;
  int T, Tpad, Vs, Vpad;
  int64_t v0;  // first vocabulary column of the group
  const float* lse;
  const float* ex;
  const float* g_lp;  // may be null
  const float* g_h;   // may be null
  const int64_t* labels;
  char* D;
  int64_t kb_total;
  // One lane's part of the tile.  With a = raw accumulator (z = a * inv_T) the gradient is
  //   d = p * (c0 + c1 * a) + [v == y] * cy,   p = exp2(a * ek + nl),
  // ek = inv_T * log2(e), nl = -lse * log2(e), c1 = -g_h * inv_T^2, c0 = inv_T * (g_h * ex - g_lp), cy = g_lp * inv_T:
  // two fused multiply-adds, one exp2 and one multiply per logit.  FULL: every vocabulary row of the tile is inside
  // the group.
  template <bool FULL>
  __device__ __forceinline__ void tile(floatx4 (&acc)[MI][NJ], int m0, int n0, int wn, int lane) const {
    const float ek = inv_T * kLog2e;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int tok = n0 + acc_col(wn, j, lane);
      if (tok >= Tpad) continue;
      // chunk (token % 16) + 16 * (v % 32 / 8) of the block; the lane's four rows are half a chunk
      char* dblk = D + ((int64_t)(tok >> 4) * kb_total + (m0 >> 5)) * 1024 + (lane & 15) * 16 +
                   (lane >> 5) * 256 + ((lane >> 4) & 1) * 8;
      if (tok >= T) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
          if (FULL || m0 + acc_row(i, 0, lane) < Vpad) *reinterpret_cast<uint2*>(dblk + i * 512) = make_uint2(0u, 0u);
        continue;
      }
      const float g1 = g_lp ? g_lp[tok] : 0.f;
      const float g2 = g_h ? g_h[tok] : 0.f;
      const float nl = -lse[tok] * kLog2e;
      const float exv = g_h ? ex[tok] : 0.f;
      const float c1 = -g2 * inv_T * inv_T, c0 = inv_T * (g2 * exv - g1), cy = g1 * inv_T;
      int y = -1;
      if (g_lp) {
        const int64_t yl = labels[tok] - v0;
        if (yl >= 0 && yl < Vs) y = (int)yl;
      }
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const int v = m0 + acc_row(i, 0, lane);  // 4 consecutive vocabulary rows of the group
        float d[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float a = acc[i][j][e];
          const float p = fast_exp2(fmaf(a, ek, nl));
          float g = p * fmaf(a, c1, c0);
          if (v + e == y) g += cy;
          d[e] = (FULL || v + e < Vs) ? g : 0.f;
        }
        if (FULL || v < Vpad)
          *reinterpret_cast<uint2*>(dblk + i * 512) = make_uint2(pack_bf16(d[0], d[1]), pack_bf16(d[2], d[3]));
      }
    }
  }
  __device__ __forceinline__ void operator()(floatx4 (&acc)[MI][NJ], int m0, int n0, int tm, int split, int wn,
                                             int lane, int tid, char* smem) const {
    if (m0 + BM <= Vs)
      tile<true>(acc, m0, n0, wn, lane);
    else
      tile<false>(acc, m0, n0, wn, lane);
  }
};

// ------------------------------------------------------------------------------ epilogues: plain stores

// d hidden: C_s[token][h] = (beta ? C_s : 0) + acc, one fp32 buffer C_s = C + s * split_stride per K run.  M is the hidden
// index, N the token: the four lanes of a token hold 16 consecutive columns of its row.
struct AccumF32Epi {
  static constexpr bool kRowsPerLane = false;
  float* C;
  int64_t ldc, split_stride;
  int M, N, beta;
  __device__ __forceinline__ void operator()(floatx4 (&acc)[MI][NJ], int m0, int n0, int tm, int split, int wn, int lane, int tid,
                             char* smem) const {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int tok = n0 + acc_col(wn, j, lane);
      if (tok >= N) continue;
      float* p = C + split * split_stride + (int64_t)tok * ldc;
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const int h = m0 + acc_row(i, 0, lane);
        if (h >= M) continue;
        f32x4* q = reinterpret_cast<f32x4*>(p + h);
        *q = beta ? *q + acc[i][j] : acc[i][j];
      }
    }
  }
};

// one value rounded to SIIRL_BF16, SIIRL_F16 or SIIRL_F32 and stored as element `at` of `out`
__device__ __forceinline__ void store_one(void* out, int64_t at, float v, int out_dtype) {
  if (out_dtype == SIIRL_BF16)
    reinterpret_cast<uint16_t*>(out)[at] = (uint16_t)(pack_bf16(v, 0.f) & 0xffffu);
  else if (out_dtype == SIIRL_F16)
    reinterpret_cast<uint16_t*>(out)[at] = (uint16_t)(pack_f16(v, 0.f) & 0xffffu);
  else
    reinterpret_cast<float*>(out)[at] = v;
}
__device__ __forceinline__ uint2 pack4(floatx4 v, int out_dtype) {
  return out_dtype == SIIRL_BF16 ? make_uint2(pack_bf16(v.x, v.y), pack_bf16(v.z, v.w))
                                 : make_uint2(pack_f16(v.x, v.y), pack_f16(v.z, v.w));
}

// C[row][col] = acc, rounded to the output type (out_dtype: SIIRL_BF16, SIIRL_F16 or SIIRL_F32).  Takes the accumulator
// by rows: the four lanes of a row write 64 consecutive bytes per instruction (16-bit types).  With 16 columns a lane an
// instruction wrote 16 bytes of every 32, and the L2 had to hold the half-written lines until their other half came:
// T=16384, H=3584,
// V=152064 forward + backward 54.2 -> 53.2 ms, d weight at T=64, H=2048, V=50257 47 -> 43 us.  N is a multiple of 64, so a wave's columns are all inside the matrix or all outside.
struct StoreEpi {
  static constexpr bool kRowsPerLane = true;
  void* C;
  int64_t ldc;
  int M, N, out_dtype;
  __device__ __forceinline__ void operator()(floatx4 (&acc)[MI][NJ], int m0, int n0, int tm, int split, int wn, int lane, int tid,
                             char* smem) const {
    if (n0 + col_of_lane(wn, 0, lane) >= N) return;
    const bool aligned = ((uintptr_t)C & 15) == 0;  // (a caller's buffer need not be; ldc and a pair's columns are multiples of 8)
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int row = m0 + row_of_lane(i, lane);
      if (row >= M) continue;
      const int64_t at = (int64_t)row * ldc + n0;
      if (!aligned) {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) store_one(C, at + col_of_lane(wn, j, lane) + r, acc[i][j][r], out_dtype);
      } else if (out_dtype == SIIRL_F32) {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(C) + at + col_of_lane(wn, j, lane)) = acc[i][j];
      } else {
#pragma unroll
        for (int j = 0; j < NJ; j += 2) {
          const uint2 a = pack4(acc[i][j], out_dtype), b = pack4(acc[i][j + 1], out_dtype);
          *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(C) + at + col_of_lane(wn, j, lane)) = u32x4{a.x, a.y, b.x, b.y};
        }
      }
    }
  }
};

// ------------------------------------------------------------------------------ small kernels

// Fragment-packed B operand.  For a K-major matrix B[n][k] the packed buffer holds, for each block of 16 rows nb
// and each block of 32 columns kb, the 64 x 16 bytes that one 16x16x32 MFMA takes as its B operand, in lane order:
//   chunk index ((nb * KB + kb) * 64 + l),  l = (n % 16) + 16 * ((k % 32) / 8),  8 consecutive k per chunk.
// Rows n >= N and columns k >= K are zero.  One thread per chunk.
__global__ __launch_bounds__(256) void pack_b_kernel(const uint16_t* __restrict__ in, int64_t ld_in, int N, int K,
                                                     u32x4* __restrict__ out, int64_t KB, int64_t chunks) {
  const int64_t ch = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (ch >= chunks) return;
  const int l = (int)(ch & 63);
  const int64_t blk = ch >> 6, kb = blk % KB, nb = blk / KB;
  const int64_t n = nb * 16 + (l & 15), k = kb * 32 + (l >> 4) * 8;
  u32x4 v = {0u, 0u, 0u, 0u};
  if (n < N && k < K) v = *reinterpret_cast<const u32x4*>(in + n * ld_in + k);  // K % 8 == 0
  out[ch] = v;
}

// The same packing of the transpose: B[n][k] = in[k][n] with in of shape [R = K][C = N].  A workgroup stages a
// 64 x 64 tile through LDS and emits its 512 chunks.  Within each 64 columns, column n = 32 h + 8 q + 4 e + r takes the place
// of row 4 q + r of 16-row block 2 h + e, so that an epilogue with kRowsPerLane finds 8 consecutive columns in a lane.
// from_f16: the input holds IEEE halves, the packed output bf16 (round to nearest even).
__device__ __forceinline__ uint32_t half2_to_bf16x2(uint32_t w) { return pack_bf16(f16_lo(w), f16_hi(w)); }
__global__ __launch_bounds__(256) void transpose_pack_b_kernel(const uint16_t* __restrict__ in, int64_t ld_in, int R,
                                                               int C, u32x4* __restrict__ out, int64_t KB, int from_f16) {
  __shared__ __align__(16) uint16_t tile[64][72];  // 144-byte rows: 16-byte aligned, 36 dwords (column reads spread)
  const int r0 = blockIdx.x * 64, c0 = blockIdx.y * 64;  // r = k, c = n
  // 16 bytes (8 columns) per thread and pass, 8 threads per row, 32 rows per pass; ld_in and c0 are multiples of 8
  for (int q = threadIdx.x; q < 512; q += 256) {
    const int rr = q >> 3, cc = (q & 7) * 8;
    const int r = r0 + rr, c = c0 + cc;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (r < R) {
      if (c + 8 <= C) {
        v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(in + (int64_t)r * ld_in + c));
      } else if (c < C) {
        uint16_t t[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = c + e < C ? in[(int64_t)r * ld_in + c + e] : (uint16_t)0;
        v = u32x4{(uint32_t)t[0] | ((uint32_t)t[1] << 16), (uint32_t)t[2] | ((uint32_t)t[3] << 16),
                  (uint32_t)t[4] | ((uint32_t)t[5] << 16), (uint32_t)t[6] | ((uint32_t)t[7] << 16)};
      }
    }
    if (from_f16) v = u32x4{half2_to_bf16x2(v.x), half2_to_bf16x2(v.y), half2_to_bf16x2(v.z), half2_to_bf16x2(v.w)};
    *reinterpret_cast<u32x4*>(&tile[rr][cc]) = v;
  }
  __syncthreads();
  for (int q = threadIdx.x; q < 512; q += 256) {
    const int nl = q & 63, kc = q >> 6;  // local n, local chunk of 8 k
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = (uint32_t)tile[kc * 8 + 2 * e][nl] | ((uint32_t)tile[kc * 8 + 2 * e + 1][nl] << 16);
    const int64_t n = c0 + nl, k = r0 + kc * 8;
    const int64_t nb = (n >> 6) * 4 + ((n >> 5) & 1) * 2 + ((n >> 2) & 1);  // 16-row block
    const int nr = (int)(((n >> 3) & 3) * 4 + (n & 3));                     // row in it
    const int64_t ch = (nb * KB + (k >> 5)) * 64 + nr + 16 * ((k >> 3) & 3);
    out[ch] = u32x4{w[0], w[1], w[2], w[3]};
  }
}

// out = in rounded from IEEE half to bf16; eight elements per thread and pass
__global__ __launch_bounds__(256) void f16_to_bf16_kernel(const u32x4* __restrict__ in, u32x4* __restrict__ out, int64_t n8) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += (int64_t)gridDim.x * 256) {
    const u32x4 v = __builtin_nontemporal_load(in + i);
    out[i] = u32x4{half2_to_bf16x2(v.x), half2_to_bf16x2(v.y), half2_to_bf16x2(v.z), half2_to_bf16x2(v.w)};
  }
}

// 16-byte pieces: the first `have` of them copied, the others zero
__global__ __launch_bounds__(256) void copy_padded_kernel(const u32x4* __restrict__ in, int64_t have, u32x4* __restrict__ out,
                                                          int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = i < have ? in[i] : u32x4{0u, 0u, 0u, 0u};
}

// label_logit[row] = inv_T * <hidden[row], W[labels[row]]>, one wave per row (NaN for a label outside [0, V))
__global__ __launch_bounds__(256) void label_logit_kernel(const uint16_t* __restrict__ hidden,
                                                          const uint16_t* __restrict__ W,
                                                          const int64_t* __restrict__ labels, int T, int H, int64_t V,
                                                          float inv_T, float* __restrict__ out, int f16) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= T) return;
  const int64_t y = labels[row];
  if (y < 0 || y >= V) {
    if (lane == 0) out[row] = __builtin_nanf("");
    return;
  }
  const u32x4* a = reinterpret_cast<const u32x4*>(hidden + (int64_t)row * H);
  const u32x4* b = reinterpret_cast<const u32x4*>(W + y * (int64_t)H);
  float s = 0.f;
  for (int i = lane; i < H / 8; i += kWave) {
    const u32x4 u = a[i], v = b[i];
    if (f16)
      s += f16_lo(u.x) * f16_lo(v.x) + f16_hi(u.x) * f16_hi(v.x) + f16_lo(u.y) * f16_lo(v.y) + f16_hi(u.y) * f16_hi(v.y) +
           f16_lo(u.z) * f16_lo(v.z) + f16_hi(u.z) * f16_hi(v.z) + f16_lo(u.w) * f16_lo(v.w) + f16_hi(u.w) * f16_hi(v.w);
    else
      s += bf16_lo(u.x) * bf16_lo(v.x) + bf16_hi(u.x) * bf16_hi(v.x) + bf16_lo(u.y) * bf16_lo(v.y) +
           bf16_hi(u.y) * bf16_hi(v.y) + bf16_lo(u.z) * bf16_lo(v.z) + bf16_hi(u.z) * bf16_hi(v.z) +
           bf16_lo(u.w) * bf16_lo(v.w) + bf16_hi(u.w) * bf16_hi(v.w);
  }
  s = wave_sum(s);
  if (lane == 0) out[row] = s * inv_T;
}

// folds the per-tile partials of each token: lse, ex, entropy, logprob.  A workgroup handles kMergeTok tokens;
// kMergeGrp thread groups each merge every kMergeGrp-th tile online, then the states are merged through LDS.
// Bound by the latency of its loads at few tokens (13 workgroups at T=200) and by the read of the partials at many: 64
// groups, whose loads do not depend on each other, four tiles at a time.  1188 tiles: T=200 68 -> 13 us, T=16384
// 95 -> 78 us against 16 groups that waited for a tile's maximum before they read its sums.
constexpr int kMergeTok = 16, kMergeGrp = 64, kMergeThreads = kMergeTok * kMergeGrp, kMergeFold = 8, kMergeAhead = 4;
__global__ __launch_bounds__(kMergeThreads) void merge_partials_kernel(const float* __restrict__ part, int nparts, int T,
                                                                       const float* __restrict__ label_logit,
                                                                       float* __restrict__ logprob,
                                                                       float* __restrict__ entropy,
                                                                       float* __restrict__ lse_out,
                                                                       float* __restrict__ ex_out) {
  __shared__ float sh[kMergeGrp][kMergeTok][3];
  __shared__ double shd[kMergeFold][kMergeTok][2];
  const float ninf = -__builtin_inff();
  const int tl = threadIdx.x % kMergeTok, grp = threadIdx.x / kMergeTok;
  const int row = blockIdx.x * kMergeTok + tl;
  float M = ninf, s = 0.f, t = 0.f;
  if (row < T) {
    for (int p0 = grp; p0 < nparts; p0 += kMergeAhead * kMergeGrp) {
      float m[kMergeAhead], ps[kMergeAhead], pt[kMergeAhead], Mn = M;
#pragma unroll
      for (int k = 0; k < kMergeAhead; ++k) {
        const int p = p0 + k * kMergeGrp;
        const float* q = part + (int64_t)(p < nparts ? p : p0) * 3 * T + row;
        m[k] = q[0];
        ps[k] = q[T];
        pt[k] = q[2 * (int64_t)T];
        if (p >= nparts) m[k] = ninf;
      }
#pragma unroll
      for (int k = 0; k < kMergeAhead; ++k) Mn = fmaxf(Mn, m[k]);
      if (Mn > ninf) {
        const float fo = fast_exp2((M - Mn) * kLog2e);
        s *= fo;
        t *= fo;
#pragma unroll
        for (int k = 0; k < kMergeAhead; ++k) {
          if (!(m[k] > ninf)) continue;
          const float fn = fast_exp2((m[k] - Mn) * kLog2e);
          s += ps[k] * fn;
          t += pt[k] * fn;
        }
        M = Mn;
      }
    }
  }
  sh[grp][tl][0] = M;
  sh[grp][tl][1] = s;
  sh[grp][tl][2] = t;
  __syncthreads();
  float Mx = ninf;
  double ss = 0.0, tt = 0.0;
  if (grp < kMergeFold) {
#pragma unroll
    for (int g = 0; g < kMergeGrp; ++g) Mx = fmaxf(Mx, sh[g][tl][0]);
#pragma unroll
    for (int g = 0; g < kMergeGrp / kMergeFold; ++g) {
      const float* a = sh[grp * (kMergeGrp / kMergeFold) + g][tl];
      if (a[0] > ninf) {
        const float f = fast_exp2((a[0] - Mx) * kLog2e);
        ss += (double)(a[1] * f);
        tt += (double)(a[2] * f);
      }
    }
    shd[grp][tl][0] = ss;
    shd[grp][tl][1] = tt;
  }
  __syncthreads();
  if (grp != 0 || row >= T) return;
#pragma unroll
  for (int g = 1; g < kMergeFold; ++g) {
    ss += shd[g][tl][0];
    tt += shd[g][tl][1];
  }
  const float lse = Mx + logf((float)ss);
  const float exv = (float)(tt / ss);
  lse_out[row] = lse;
  if (ex_out) ex_out[row] = exv;
  if (entropy) entropy[row] = lse - exv;
  if (logprob) logprob[row] = label_logit[row] - lse;
}

// out = the sum of `splits` buffers, `stride` four-element vectors apart, rounded to out_dtype (SIIRL_BF16, SIIRL_F16 or
// SIIRL_F32).  A pure stream: 16-byte loads, the buffers added in their order.
__global__ __launch_bounds__(256) void sum_convert_kernel(const f32x4* __restrict__ in, int64_t stride, int splits,
                                                          void* __restrict__ out, int64_t n4, int out_dtype) {
  const bool aligned = ((uintptr_t)out & 15) == 0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (int64_t)gridDim.x * 256) {
    f32x4 v = in[i];
    for (int s = 1; s < splits; ++s) v += in[s * stride + i];
    if (!aligned) {
#pragma unroll
      for (int r = 0; r < 4; ++r) store_one(out, i * 4 + r, v[r], out_dtype);
    } else if (out_dtype == SIIRL_F32) {
      reinterpret_cast<f32x4*>(out)[i] = v;
    } else {
      reinterpret_cast<uint2*>(out)[i] = pack4(v, out_dtype);
    }
  }
}

// fp32 operands are staged as three bf16 terms per element so that the bf16 matrix cores reproduce the product to
// 2^-16: x = hi + lo + O(2^-16 x) with hi = bf16(x), lo = bf16(x - hi), and
//   a . b ~ a_hi . b_hi + a_hi . b_lo + a_lo . b_hi .
// A row of K floats becomes a row of 3 K bf16: [hi | hi | lo] for the A operand (role 0), [hi | lo | hi] for the B
// operand (role 1); the GEMM then simply runs over K' = 3 K.  The first K columns are bf16(x): what the two gradient
// GEMMs use.  Four elements per thread.
__global__ __launch_bounds__(256) void split3_kernel(const float* __restrict__ in, int64_t rows, int64_t K,
                                                     uint16_t* __restrict__ out, int role) {
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;  // quad index
  const int64_t kq = K / 4;
  if (q >= rows * kq) return;
  const int64_t r = q / kq, k = (q - r * kq) * 4;
  const float4 x = *reinterpret_cast<const float4*>(in + r * K + k);
  const uint32_t h01 = pack_bf16(x.x, x.y), h23 = pack_bf16(x.z, x.w);
  const uint32_t l01 = pack_bf16(x.x - bf16_lo(h01), x.y - bf16_hi(h01));
  const uint32_t l23 = pack_bf16(x.z - bf16_lo(h23), x.w - bf16_hi(h23));
  uint16_t* o = out + r * 3 * K + k;
  *reinterpret_cast<uint2*>(o) = make_uint2(h01, h23);
  *reinterpret_cast<uint2*>(o + K) = role == 0 ? make_uint2(h01, h23) : make_uint2(l01, l23);
  *reinterpret_cast<uint2*>(o + 2 * K) = role == 0 ? make_uint2(l01, l23) : make_uint2(h01, h23);
}

// ------------------------------------------------------------------------------ host

inline int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

// Shape of an XCD's block: `blk_m` tiles along M where the grid has room for it.  A grid narrower than the block in one
// direction would leave most of the block's workgroup ids without a tile (a token count of one tile in blocks of 4 x 8:
// 7 of 8 ids start and leave, each holding the CU's LDS meanwhile), so the block is made longer in the other one.
inline int fit_blk_m(int blk_m, int64_t tiles_m, int64_t tiles_n) {
  while (blk_m > 1 && blk_m / 2 >= tiles_m) blk_m /= 2;
  while (blk_m < kBlkTiles && kBlkTiles / blk_m / 2 >= tiles_n) blk_m *= 2;
  return blk_m;
}

template <class Epi, int AL = A_ROWS, bool F16 = false>
int launch_gemm(const uint16_t* A, int64_t lda, const u32x4* Bp, int64_t kb_total, int M, int N, int K, const Epi& epi,
                hipStream_t st, const char* what, int splits = 1, int blk_m = 8, const uint16_t* A_tail = nullptr) {
  GemmArgs g{A, lda, Bp, kb_total, M, N, K, (M + BM - 1) / BM, (N + BN - 1) / BN, splits, blk_m, 0,
             A_tail, A_tail ? K / BK - 1 : K / BK};
  g.blk_m = fit_blk_m(blk_m, g.tiles_m, (int64_t)g.tiles_n * splits);
  if (AL == A_PACKED && lda * 32 < (int64_t)g.tiles_m * BM) return fail(SIIRL_ERR_INVALID_ARGUMENT, "%s: row pitch %lld is shorter than %d tiles", what, (long long)lda, g.tiles_m);
  const int64_t grid = raster_grid(g);
  auto launch = [&](void (*kernel)(GemmArgs, Epi)) -> int {
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kSmemBytes)) return rc;
    kernel<<<dim3((unsigned)grid), dim3(kThreads), kSmemBytes, st>>>(g, epi);
    return SIIRL_OK;
  };
  if constexpr (AL != A_PACKED) {  // (the packed A of d weight is small and read by every column tile)
    if (g.tiles_n == 1 && streams_past_cache(2.0 * (double)M * (double)K)) {
      if (int rc = launch(&gemm_once_kernel<Epi, AL, F16>)) return rc;
      SIIRL_LAUNCH_CHECK(what);
      return SIIRL_OK;
    }
  }
  if (int rc = launch(&gemm_nt_kernel<Epi, AL, F16>)) return rc;
  SIIRL_LAUNCH_CHECK(what);
  return SIIRL_OK;
}

// C = A . B^T with a packed A and K of at most kShortSteps K-steps.  The tiles along N are cut into as many equal runs as
// make four rounds of the CUs' 512 workgroups, or less where N has fewer tiles.
template <class Epi>
int launch_short_k(const uint16_t* A, int64_t lda, const u32x4* Bp, int64_t kb_total, int M, int N, int K, const Epi& epi,
                   hipStream_t st, const char* what) {
  if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(&gemm_short_k_kernel<Epi>), kSmemBytes)) return rc;
  const GemmArgs g{A, lda, Bp, kb_total, M, N, K, (M + BM - 1) / BM, (N + BN - 1) / BN, 1, 1, 0, nullptr, K / BK};
  if (K > kShortSteps * BK || lda * 32 < (int64_t)g.tiles_m * BM)
    return fail(SIIRL_ERR_INVALID_ARGUMENT, "%s: K=%d or row pitch %lld does not fit %d tiles", what, K, (long long)lda, g.tiles_m);
  const int64_t want = (4 * 512 + g.tiles_m - 1) / g.tiles_m;  // runs along N
  const int runs = (int)(want < g.tiles_n ? want : g.tiles_n), n_per = (g.tiles_n + runs - 1) / runs;
  const int64_t grid = (int64_t)g.tiles_m * ((g.tiles_n + n_per - 1) / n_per);
  gemm_short_k_kernel<Epi><<<dim3((unsigned)grid), dim3(kThreads), kSmemBytes, st>>>(g, n_per, epi);
  SIIRL_LAUNCH_CHECK(what);
  return SIIRL_OK;
}

// Tiles along M of an XCD's block, per GEMM of the fused path.  Measured at T=16384, H=3584, V=152064 (ms per step for
// blocks of 2 x 16 / 4 x 8 / 8 x 4 / 16 x 2 tiles): forward 12.77 / 12.54 / 12.81 / 13.74; recompute + dlogits 13.35 / 12.97 /
// 13.31 / 13.65; d hidden 15.33 / 13.44 / 14.68 / 15.09; d weight 15.46 / 12.86 / 12.74 / 13.92.  The A operand
// of the first two is W, streamed from memory once per strip of blk_n token tiles: wider strips read it less often.
// Recompute at fewer tokens, 2 x 16 / 4 x 8 (us, with d weight): H=2048, V=50257 T=3001 1005 / 1026, T=4096 1347 / 1319; H=1024,
// V=32000 T=2048 227 / 231, T=8192 909 / 870: the wide blocks below 16 token tiles.
// With one token tile the tiles of a d hidden K run share nothing but its dlogits, so they go to one XCD: 649 / 437 / 410 /
// 304 / 300 us for 2 x 16 .. 32 x 1 at T=200.
constexpr int kBlkFwd = 4, kBlkDHidden = 4, kBlkDWeight = 8;
inline int blk_recompute(int tiles_t) { return tiles_t < 16 ? 2 : 4; }

// Number of K runs of the d-hidden GEMM, each with an fp32 buffer of its own that sum_convert_kernel adds up.  The
// tiles of [T, H] alone rarely fill the 256 CUs, two each: 1792 tiles at T=16384, H=3584 are 3.5 rounds (two runs: 7), 28
// tiles at T=200 a fraction of one (18 runs: 504 workgroups).  The run count is the one with the least time by
// the kernel's measured 1.2 us per K-step of the two tiles on a CU and about 12 us per tile besides, plus the buffers' write and read at 5 TB/s.
constexpr int kMaxSplits = 64;
constexpr double kSplitBytes = 512.0 * 1048576.0;  // bound on the buffers of more than two runs
// Up to 1024 tokens the choice does not look at T (it is the one for a single token tile; at T=1024, H=3584, K=152064
// 18 runs model as 786 us against 710 us for the best 9), so that a row of d hidden keeps its bits whatever other rows
// a small batch holds.  The bound is then that of the 1024.
constexpr int64_t kSplitSameTokens = 1024;
inline int pick_splits(int64_t T, int64_t H, int64_t K) {
  const int64_t most = T <= kSplitSameTokens ? kSplitSameTokens : T;
  if (T <= kSplitSameTokens) T = BN;
  const int64_t tiles = ((T + BN - 1) / BN) * ((H + BM - 1) / BM), KT = K / BK;
  int best = 1;
  double best_us = 0.;
  for (int s = 1; s <= kMaxSplits && s <= KT; ++s) {
    const double bytes = 4.0 * (double)T * (double)H * s;
    if (s > 2 && 4.0 * (double)most * (double)H * s > kSplitBytes) break;
    const int64_t per = (KT + s - 1) / s;
    if ((s - 1) * per >= KT) continue;  // the last run would be empty
    const double us = (double)((tiles * s + 511) / 512) * (1.2 * (double)per + 12.0) + 2.0 * bytes / 5e6;
    if (s == 1 || us < best_us) best_us = us, best = s;
  }
  return best;
}

// K of the logits GEMM for operands of `dtype`: the hidden size, or three bf16 terms per fp32 element (split3_kernel)
inline int64_t logits_k(int dtype, int64_t H) { return dtype == SIIRL_F32 ? 3 * H : H; }

int check_fused(const void* hidden, const void* weight, int64_t T, int64_t H, int64_t V, float inv_T, int dtype) {
  SIIRL_REQUIRE(dtype == SIIRL_BF16 || dtype == SIIRL_F16 || dtype == SIIRL_F32,
                "fused lm_head path takes bf16, fp16 or fp32 operands (dtype %d given)", dtype);
  // 32-bit byte offsets inside a tile bound the row pitch of every A operand (W: 128 rows of K or 64 K-rows; D: four
  // 16-token rows of blocks)
  SIIRL_REQUIRE(T >= 1 && T < (1LL << 22) && V >= 1 && V < (1LL << 30), "T=%lld (< 4194304) V=%lld out of range",
                (long long)T, (long long)V);
  SIIRL_REQUIRE(H >= BK && H % BK == 0 && logits_k(dtype, H) < (1 << 22),
                "hidden size %lld must be a positive multiple of %d (below %d)", (long long)H, BK,
                (1 << 22) / (dtype == SIIRL_F32 ? 3 : 1));
  SIIRL_REQUIRE(hidden && weight, "NULL operand");
  SIIRL_REQUIRE(((uintptr_t)hidden & 15) == 0 && ((uintptr_t)weight & 15) == 0, "operands must be 16-byte aligned");
  SIIRL_REQUIRE(inv_T > 0.f && inv_T < 1e30f, "inv_temperature must be positive and finite");
  return SIIRL_OK;
}
int check_ws_align(const void* ws) {
  SIIRL_REQUIRE(((uintptr_t)ws & 255) == 0, "workspace must be 256-byte aligned");
  return SIIRL_OK;
}

// hs / wsp: the three-term bf16 copies of fp32 operands ([T][3 H], [V][3 H]); absent for 16-bit operands
struct FwdWs {
  size_t part, label, hp, hs, wsp, total;
};
FwdWs fwd_ws(int64_t T, int64_t H, int64_t V, int dtype) {
  FwdWs w;
  const int64_t tiles_v = (V + BM - 1) / BM, Kc = logits_k(dtype, H);
  size_t off = 0;
  w.part = off; off += round_up((size_t)tiles_v * 3 * T * 4, 256);
  w.label = off; off += round_up((size_t)T * 4, 256);
  w.hp = off; off += (size_t)round_up(T, BN) * Kc * 2;
  w.hs = off; off += dtype == SIIRL_F32 ? round_up((size_t)T * Kc * 2, 256) : 0;
  w.wsp = off; off += dtype == SIIRL_F32 ? round_up((size_t)V * Kc * 2, 256) : 0;
  w.total = off;
  return w;
}

struct BwdWs {
  size_t hp, w16, wtail, htp, d, dh32, hs, wsp, total;
  int64_t ldt, hpad, group, kb_d;  // ldt: token count padded to BK (the K of the d-weight GEMM); group: columns of a
                                   // vocabulary group; kb_d: 1 KB blocks of D per 16 tokens
  int dh_splits;                            // K runs of the first (largest) group's d-hidden GEMM
};
BwdWs bwd_ws(int64_t T, int64_t H, int64_t V, bool want_dh, bool want_dw, int dtype) {
  BwdWs w;
  const int64_t Kc = logits_k(dtype, H);
  w.ldt = round_up(T, BK);
  int64_t n = kGroupTokens / w.ldt;  // at most 64: a tile's byte offsets into D have 32 bits
  n = n < 1 ? 1 : (n > 64 ? 64 : n);
  w.group = n * kGroupCols < V ? n * kGroupCols : round_up(V, 256);
  w.kb_d = w.group / 32 + kPadBlocks;
  w.dh_splits = pick_splits(T, H, w.group < V ? w.group : round_up(V, BK));
  w.hpad = round_up(H, BN);
  size_t off = 0;
  w.hp = off; off += (size_t)round_up(T, BN) * Kc * 2;
  w.w16 = off; off += want_dh && dtype == SIIRL_F16 ? round_up((size_t)V * H * 2, 256) : 0;
  w.wtail = off; off += want_dh && V % BK ? round_up((size_t)BK * Kc * 2, 256) : 0;
  w.htp = off; off += want_dw ? (size_t)w.hpad * w.ldt * 2 : 0;
  w.d = off; off += (size_t)(round_up(T, BN) / 16) * w.kb_d * 1024;  // tokens [T, ldt) are K-padding of d weight: zeros
  w.dh32 = off; off += want_dh ? w.dh_splits * round_up((size_t)T * H * 4, 256) : 0;  // one buffer per K run
  w.hs = off; off += dtype == SIIRL_F32 ? round_up((size_t)T * Kc * 2, 256) : 0;
  w.wsp = off; off += dtype == SIIRL_F32 ? round_up((size_t)V * Kc * 2, 256) : 0;
  w.total = off;
  return w;
}

// fp32 operands -> their three-term bf16 copies (hidden in the B role, weight in the A role)
int stage_f32(const void* hidden, const void* weight, int64_t T, int64_t H, int64_t V, uint16_t* hs, uint16_t* wsp,
              hipStream_t st) {
  const int64_t qh = T * (H / 4), qw = V * (H / 4);
  split3_kernel<<<dim3((unsigned)((qh + 255) / 256)), dim3(256), 0, st>>>((const float*)hidden, T, H, hs, 1);
  SIIRL_LAUNCH_CHECK("split3_kernel(hidden)");
  split3_kernel<<<dim3((unsigned)((qw + 255) / 256)), dim3(256), 0, st>>>((const float*)weight, V, H, wsp, 0);
  SIIRL_LAUNCH_CHECK("split3_kernel(weight)");
  return SIIRL_OK;
}

int pack_hidden(const uint16_t* h, int64_t T, int64_t H, u32x4* out, hipStream_t st) {
  const int64_t chunks = round_up(T, BN) * H / 8;
  pack_b_kernel<<<dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, st>>>(h, H, (int)T, (int)H, out, H / 32, chunks);
  SIIRL_LAUNCH_CHECK("pack_b_kernel");
  return SIIRL_OK;
}

// The per-token operands of the backward for the listed token rows only (a row index outside [0, T) yields zero
// gradients: the row then contributes nothing).
__global__ __launch_bounds__(256) void gather_token_operands_kernel(const int64_t* __restrict__ rows, int64_t n, int64_t T,
                                                                    const int64_t* __restrict__ labels,
                                                                    const float* __restrict__ lse,
                                                                    const float* __restrict__ ex,
                                                                    const float* __restrict__ g_lp,
                                                                    const float* __restrict__ g_ent,
                                                                    int64_t* __restrict__ labels_c, float* __restrict__ lse_c,
                                                                    float* __restrict__ ex_c, float* __restrict__ g_lp_c,
                                                                    float* __restrict__ g_ent_c) {
  const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (j >= n) return;
  const int64_t r = rows[j];
  const bool ok = r >= 0 && r < T;
  labels_c[j] = ok && labels ? labels[r] : -1;
  lse_c[j] = ok ? lse[r] : 0.f;
  ex_c[j] = ok && ex ? ex[r] : 0.f;
  g_lp_c[j] = ok && g_lp ? g_lp[r] : 0.f;
  g_ent_c[j] = ok && g_ent ? g_ent[r] : 0.f;
}

struct RowsWs {
  size_t hidden, labels, lse, ex, g_lp, g_ent, dh, inner, inner_bytes, total;
};
RowsWs rows_ws(int64_t n, int64_t H, int64_t V, bool want_dh, bool want_dw, int dtype) {
  const size_t es = dtype_size(dtype);
  RowsWs w;
  size_t off = 0;
  auto take = [&off](size_t bytes) {
    const size_t at = off;
    off += round_up(bytes, 256);
    return at;
  };
  w.hidden = take((size_t)n * H * es);
  w.labels = take((size_t)n * 8);
  w.lse = take((size_t)n * 4);
  w.ex = take((size_t)n * 4);
  w.g_lp = take((size_t)n * 4);
  w.g_ent = take((size_t)n * 4);
  w.dh = take(want_dh ? (size_t)n * H * es : 0);
  w.inner = off;
  w.inner_bytes = n > 0 ? bwd_ws(n, H, V, want_dh, want_dw, dtype).total : 0;
  w.total = off + w.inner_bytes;
  return w;
}

}  // namespace
}  // namespace siirl

using namespace siirl;

extern "C" size_t siirl_fused_linear_fwd_workspace_bytes_dtype(int dtype, int64_t T, int64_t H, int64_t V) {
  if (T < 1 || V < 1 || H < 1 || dtype_size(dtype) == 0) return 0;
  return fwd_ws(T, H, V, dtype).total;
}
extern "C" size_t siirl_fused_linear_fwd_workspace_bytes(int64_t T, int64_t H, int64_t V) {
  return siirl_fused_linear_fwd_workspace_bytes_dtype(SIIRL_BF16, T, H, V);
}

extern "C" size_t siirl_fused_linear_bwd_workspace_bytes_dtype(int dtype, int64_t T, int64_t H, int64_t V,
                                                               int want_d_hidden, int want_d_weight) {
  if (T < 1 || V < 1 || H < 1 || dtype_size(dtype) == 0) return 0;
  return bwd_ws(T, H, V, want_d_hidden != 0, want_d_weight != 0, dtype).total;
}
extern "C" size_t siirl_fused_linear_bwd_workspace_bytes(int64_t T, int64_t H, int64_t V, int want_d_hidden,
                                                         int want_d_weight) {
  return siirl_fused_linear_bwd_workspace_bytes_dtype(SIIRL_BF16, T, H, V, want_d_hidden, want_d_weight);
}

extern "C" size_t siirl_fused_linear_saved_logits_bytes(int64_t T, int64_t V) {
  if (T < 1 || V < 1) return 0;
  return (size_t)(((V + BM - 1) / BM) * ((T + BN - 1) / BN) * kSavedTileBytes);
}

extern "C" int siirl_fused_linear_logprob_entropy_fwd(const void* hidden, const void* weight, int dtype,
                                                      const int64_t* labels, int64_t T, int64_t H, int64_t V,
                                                      float inv_temperature, float* logprob, float* entropy, float* lse,
                                                      float* ex, float* saved_logits, void* workspace,
                                                      size_t workspace_bytes, siirl_stream_t stream) {
  if (int rc = check_fused(hidden, weight, T, H, V, inv_temperature, dtype)) return rc;
  SIIRL_REQUIRE(lse != nullptr, "lse is NULL");
  SIIRL_REQUIRE(((uintptr_t)saved_logits & 15) == 0, "saved_logits must be 16-byte aligned");
  SIIRL_REQUIRE((logprob == nullptr) == (labels == nullptr), "labels and logprob must be given together");
  SIIRL_REQUIRE(entropy == nullptr || ex != nullptr, "ex is required when entropy is requested");
  const FwdWs ws = fwd_ws(T, H, V, dtype);
  if (workspace == nullptr || workspace_bytes < ws.total)
    return fail(SIIRL_ERR_WORKSPACE, "workspace of %zu bytes is smaller than the %zu needed", workspace_bytes, ws.total);
  if (int rc = check_ws_align(workspace)) return rc;
  hipStream_t st = (hipStream_t)stream;
  float* part = reinterpret_cast<float*>((char*)workspace + ws.part);
  float* label_logit = reinterpret_cast<float*>((char*)workspace + ws.label);
  const uint16_t* h = (const uint16_t*)hidden;
  const uint16_t* w = (const uint16_t*)weight;
  const int64_t Kc = logits_k(dtype, H);
  const bool f16 = dtype == SIIRL_F16;
  if (dtype == SIIRL_F32) {
    uint16_t* hs = (uint16_t*)((char*)workspace + ws.hs);
    uint16_t* wsp = (uint16_t*)((char*)workspace + ws.wsp);
    if (int rc = stage_f32(hidden, weight, T, H, V, hs, wsp, st)) return rc;
    h = hs;
    w = wsp;
  }
  if (labels) {
    label_logit_kernel<<<dim3((unsigned)((T + 3) / 4)), dim3(256), 0, st>>>(h, w, labels, (int)T, (int)Kc, V,
                                                                          inv_temperature, label_logit, (int)f16);
    SIIRL_LAUNCH_CHECK("label_logit_kernel");
  }
  u32x4* hp = reinterpret_cast<u32x4*>((char*)workspace + ws.hp);
  if (int rc = pack_hidden(h, T, Kc, hp, st)) return rc;
  SoftmaxPartialsEpi epi{inv_temperature, (int)T, (int)V, part, saved_logits, (int)((T + BN - 1) / BN)};
  if (int rc = f16 ? launch_gemm<SoftmaxPartialsEpi, A_ROWS, true>(w, Kc, hp, Kc / 32, (int)V, (int)T, (int)Kc, epi, st,
                                                                  "gemm_nt_kernel<SoftmaxPartialsEpi, f16>", 1, kBlkFwd)
                   : launch_gemm(w, Kc, hp, Kc / 32, (int)V, (int)T, (int)Kc, epi, st, "gemm_nt_kernel<SoftmaxPartialsEpi>", 1,
                                 kBlkFwd))
    return rc;
  const int tiles_v = (int)((V + BM - 1) / BM);
  merge_partials_kernel<<<dim3((unsigned)((T + kMergeTok - 1) / kMergeTok)), dim3(kMergeThreads), 0, st>>>(part, tiles_v, (int)T, label_logit,
                                                                               logprob, entropy, lse, ex);
  SIIRL_LAUNCH_CHECK("merge_partials_kernel");
  return SIIRL_OK;
}

extern "C" int siirl_fused_linear_logprob_entropy_bwd(const void* hidden, const void* weight, int dtype,
                                                      const int64_t* labels, int64_t T, int64_t H, int64_t V,
                                                      float inv_temperature, const float* lse, const float* ex,
                                                      const float* saved_logits, const float* g_logprob,
                                                      const float* g_entropy, void* d_hidden, void* d_weight,
                                                      void* workspace, size_t workspace_bytes, siirl_stream_t stream) {
  if (int rc = check_fused(hidden, weight, T, H, V, inv_temperature, dtype)) return rc;
  SIIRL_REQUIRE(lse != nullptr, "lse is NULL");
  SIIRL_REQUIRE(((uintptr_t)saved_logits & 15) == 0, "saved_logits must be 16-byte aligned");
  SIIRL_REQUIRE(g_logprob != nullptr || g_entropy != nullptr, "no upstream gradient given");
  SIIRL_REQUIRE(g_logprob == nullptr || labels != nullptr, "labels is required with g_logprob");
  SIIRL_REQUIRE(g_entropy == nullptr || ex != nullptr, "ex is required with g_entropy");
  SIIRL_REQUIRE(d_hidden != nullptr || d_weight != nullptr, "neither d_hidden nor d_weight requested");
  const bool want_dh = d_hidden != nullptr, want_dw = d_weight != nullptr;
  const BwdWs ws = bwd_ws(T, H, V, want_dh, want_dw, dtype);
  if (workspace == nullptr || workspace_bytes < ws.total)
    return fail(SIIRL_ERR_WORKSPACE, "workspace of %zu bytes is smaller than the %zu needed", workspace_bytes, ws.total);
  if (int rc = check_ws_align(workspace)) return rc;
  hipStream_t st = (hipStream_t)stream;
  char* base = (char*)workspace;
  u32x4* hp = (u32x4*)(base + ws.hp);          // packed hidden: B[n = token][k = K of the logits GEMM]
  u32x4* W16 = (u32x4*)(base + ws.w16);        // fp16 operands: bf16 copy of W
  u32x4* Htp = (u32x4*)(base + ws.htp);        // packed hidden^T: B[n = H][k = token]
  char* D = base + ws.d;                       // packed dlogits of one vocabulary group
  float* dH32 = (float*)(base + ws.dh32);      // [T][H]
  const uint16_t* h = (const uint16_t*)hidden;
  const uint16_t* w = (const uint16_t*)weight;
  // The logits are recomputed from the operands as given (fp16: the half MFMA; fp32: three bf16 terms per element,
  // K = 3 H).  The two gradient GEMMs multiply the bf16 dlogits with hidden and W in bf16 and write their fp32 sums in the
  // operands' dtype.  hidden is packed transposed (fp16: rounded on the way); W is read by K-rows where it lies (bf16), from
  // a plain bf16 copy (fp16; 365 us a call at H=3584, V=152064) or from the first term of the staged rows (fp32).
  const int64_t Kc = logits_k(dtype, H);
  const bool f16 = dtype == SIIRL_F16;
  if (dtype == SIIRL_F32) {
    uint16_t* hs = (uint16_t*)(base + ws.hs);
    uint16_t* wsp = (uint16_t*)(base + ws.wsp);
    if (int rc = stage_f32(hidden, weight, T, H, V, hs, wsp, st)) return rc;
    h = hs;
    w = wsp;
  }

  if (!saved_logits)
    if (int rc = pack_hidden(h, T, Kc, hp, st)) return rc;
  uint16_t* Wtail = (uint16_t*)(base + ws.wtail);  // the last V % BK rows of W and zeros
  const uint16_t* wg = w;  // W as the gradient GEMM reads it: bf16 rows of pitch Kc, H of them used
  if (want_dh && f16) {
    const int64_t n8 = V * H / 8;
    f16_to_bf16_kernel<<<dim3((unsigned)((n8 + 255) / 256 < 65536 ? (n8 + 255) / 256 : 65536)), dim3(256), 0, st>>>(
        reinterpret_cast<const u32x4*>(w), W16, n8);
    SIIRL_LAUNCH_CHECK("f16_to_bf16_kernel");
    wg = reinterpret_cast<const uint16_t*>(W16);
  }
  if (want_dh && V % BK) {
    const int64_t n8 = BK * Kc / 8, have8 = V % BK * Kc / 8;  // (Kc is a multiple of BK)
    copy_padded_kernel<<<dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, st>>>(
        reinterpret_cast<const u32x4*>(wg + V / BK * BK * Kc), have8, reinterpret_cast<u32x4*>(Wtail), n8);
    SIIRL_LAUNCH_CHECK("copy_padded_kernel");
  }
  if (want_dw) {
    transpose_pack_b_kernel<<<dim3((unsigned)(ws.ldt / 64), (unsigned)(ws.hpad / 64)), dim3(256), 0, st>>>(
        h, Kc, (int)T, (int)H, Htp, ws.ldt / 32, (int)f16);
    SIIRL_LAUNCH_CHECK("transpose_pack_b_kernel(hidden)");
  }
  const int64_t dh32_stride = (int64_t)(round_up((size_t)T * H * 4, 256) / 4);
  const int tiles_t = (int)((T + BN - 1) / BN);
  // The recompute goes in launches of about 4096 workgroups (8192 columns at 16384 tokens, whose 59 MB of W stay in the
  // memory-side cache while the token tiles pass over them: 0.4 % of the whole step faster than one launch per group).  At
  // T=200 that is one launch of 1188 workgroups; 19 launches of 8192 columns had 32 each (1766 against 330 us).
  const int slab = 8192 * (tiles_t < 64 ? 64 / tiles_t : 1);
  for (int64_t v0 = 0; v0 < V; v0 += ws.group) {
    const int N = (int)(V - v0 < ws.group ? V - v0 : ws.group);
    const int Npad = (int)round_up(N, BK);
    if (!saved_logits) {
      for (int s0 = 0; s0 < N; s0 += slab) {
        const int Ns = N - s0 < slab ? N - s0 : slab;
        const DlogitsEpi epi{inv_temperature, (int)T, (int)ws.ldt, Ns, (int)round_up(Ns, BK), v0 + s0, lse, ex, g_logprob,
                             g_entropy, labels, D + (s0 >> 5) * 1024, ws.kb_d};
        const uint16_t* ws0 = w + (v0 + s0) * Kc;
        if (int rc = f16 ? launch_gemm<DlogitsEpi, A_ROWS, true>(ws0, Kc, hp, Kc / 32, Ns, (int)T, (int)Kc, epi, st,
                                                                "gemm_nt_kernel<DlogitsEpi, f16>", 1, blk_recompute(tiles_t))
                         : launch_gemm(ws0, Kc, hp, Kc / 32, Ns, (int)T, (int)Kc, epi, st, "gemm_nt_kernel<DlogitsEpi>", 1,
                                       blk_recompute(tiles_t)))
          return rc;
      }
    } else {
      // the group's dlogits in one pass over the tiles the forward parked
      const DlogitsEpi epi{inv_temperature, (int)T, (int)ws.ldt, N, Npad, v0, lse, ex, g_logprob, g_entropy, labels, D, ws.kb_d};
      const void* fn = reinterpret_cast<const void*>(&replay_tiles_kernel<DlogitsEpi>);
      if (int rc = allow_dynamic_lds(fn, kSmemBytes)) return rc;
      const int64_t wgs = (int64_t)((N + BM - 1) / BM) * tiles_t;
      replay_tiles_kernel<DlogitsEpi><<<dim3((unsigned)wgs), dim3(kThreads), kSmemBytes, st>>>(
          saved_logits, tiles_t, (int)(v0 / BM), epi);
      SIIRL_LAUNCH_CHECK("replay_tiles_kernel<DlogitsEpi>");
    }
    if (want_dh) {
      // dH[T, H] += D[T, K] . W[v0 : v0 + K, H] over the group's columns, as its transpose: W is the A operand given by its
      // K-rows, as it lies in memory, the packed D the B operand.  A shallower last group may take fewer runs than the
      // first one: it then adds to the first buffers only.
      int splits = ws.dh_splits;
      if (v0 > 0) {
        const int fit = pick_splits(T, H, Npad);
        splits = fit < splits ? fit : splits;
        const int KT = Npad / BK, per = (KT + splits - 1) / splits;
        splits = (KT + per - 1) / per;  // no run is empty
      }
      AccumF32Epi acc{dH32, H, dh32_stride, (int)H, (int)T, v0 > 0 ? 1 : 0};
      if (int rc = launch_gemm<AccumF32Epi, A_KROWS>(wg + v0 * Kc, Kc, reinterpret_cast<const u32x4*>(D), ws.kb_d, (int)H,
                                                     (int)T, Npad, acc, st, "gemm_nt_kernel<AccumF32Epi, A by K-rows>",
                                                     splits, T <= BN ? kBlkTiles : kBlkDHidden, N < Npad ? Wtail : nullptr))
        return rc;
    }
    if (want_dw) {
      // dW[v0 : v0 + N, H] = D[ldt, N]^T . Ht[H, ldt]^T over the group's vocabulary rows: D is the A operand given by its
      // packed K-rows (tokens)
      StoreEpi sto{(char*)d_weight + v0 * H * (int64_t)dtype_size(dtype), H, N, (int)H, dtype};
      const uint16_t* Da = reinterpret_cast<const uint16_t*>(D);
      if (int rc = ws.ldt <= kShortSteps * BK
                       ? launch_short_k(Da, ws.kb_d, Htp, ws.ldt / 32, N, (int)H, (int)ws.ldt, sto, st,
                                        "gemm_short_k_kernel<StoreEpi>")
                       : launch_gemm<StoreEpi, A_PACKED>(Da, ws.kb_d, Htp, ws.ldt / 32, N, (int)H, (int)ws.ldt, sto, st,
                                                         "gemm_nt_kernel<StoreEpi, packed A>", 1, kBlkDWeight))
        return rc;
    }
  }
  if (want_dh) {
    const int64_t n4 = T * H / 4;  // H is a multiple of BK
    const unsigned blocks = (unsigned)((n4 + 255) / 256 < 16384 ? (n4 + 255) / 256 : 16384);
    sum_convert_kernel<<<dim3(blocks), dim3(256), 0, st>>>(reinterpret_cast<const f32x4*>(dH32), dh32_stride / 4, ws.dh_splits,
                                                           d_hidden, n4, dtype);
    SIIRL_LAUNCH_CHECK("sum_convert_kernel");
  }
  return SIIRL_OK;
}

extern "C" size_t siirl_fused_linear_bwd_rows_workspace_bytes_dtype(int dtype, int64_t n_rows, int64_t H, int64_t V,
                                                                    int want_d_hidden, int want_d_weight) {
  if (n_rows < 0 || H <= 0 || V <= 0 || dtype_size(dtype) == 0) return 0;
  return rows_ws(n_rows, H, V, want_d_hidden != 0, want_d_weight != 0, dtype).total;
}
extern "C" size_t siirl_fused_linear_bwd_rows_workspace_bytes(int64_t n_rows, int64_t H, int64_t V, int want_d_hidden,
                                                              int want_d_weight) {
  return siirl_fused_linear_bwd_rows_workspace_bytes_dtype(SIIRL_BF16, n_rows, H, V, want_d_hidden, want_d_weight);
}

extern "C" int siirl_fused_linear_logprob_entropy_bwd_rows(const void* hidden, const void* weight, int dtype,
                                                           const int64_t* labels, int64_t T, int64_t H, int64_t V,
                                                           float inv_temperature, const float* lse, const float* ex,
                                                           const float* g_logprob, const float* g_entropy,
                                                           const int64_t* rows, int64_t n_rows, void* d_hidden,
                                                           void* d_weight, void* workspace, size_t workspace_bytes,
                                                           siirl_stream_t stream) {
  if (int rc = check_fused(hidden, weight, T, H, V, inv_temperature, dtype)) return rc;
  SIIRL_REQUIRE(n_rows >= 0 && n_rows <= T, "n_rows=%lld must lie in [0, T=%lld]", (long long)n_rows, (long long)T);
  SIIRL_REQUIRE(n_rows == 0 || rows != nullptr, "rows is NULL");
  SIIRL_REQUIRE(lse != nullptr, "lse is NULL");
  SIIRL_REQUIRE(g_logprob != nullptr || g_entropy != nullptr, "no upstream gradient given");
  SIIRL_REQUIRE(g_logprob == nullptr || labels != nullptr, "labels is required with g_logprob");
  SIIRL_REQUIRE(g_entropy == nullptr || ex != nullptr, "ex is required with g_entropy");
  SIIRL_REQUIRE(d_hidden != nullptr || d_weight != nullptr, "neither d_hidden nor d_weight requested");
  const bool want_dh = d_hidden != nullptr, want_dw = d_weight != nullptr;
  if (n_rows == 0) {  // no row carries a gradient: both results are zero
    if (want_dh)
      if (int rc = siirl_scatter_rows(nullptr, nullptr, 0, H * (int64_t)dtype_size(dtype), T, d_hidden, stream)) return rc;
    if (want_dw)
      if (int rc = siirl_scatter_rows(nullptr, nullptr, 0, H * (int64_t)dtype_size(dtype), V, d_weight, stream)) return rc;
    return SIIRL_OK;
  }
  const RowsWs ws = rows_ws(n_rows, H, V, want_dh, want_dw, dtype);
  const int64_t row_bytes = H * (int64_t)dtype_size(dtype);
  if (workspace == nullptr || workspace_bytes < ws.total)
    return fail(SIIRL_ERR_WORKSPACE, "workspace of %zu bytes is smaller than the %zu needed", workspace_bytes, ws.total);
  if (int rc = check_ws_align(workspace)) return rc;
  hipStream_t st = (hipStream_t)stream;
  char* base = (char*)workspace;
  void* hidden_c = base + ws.hidden;
  int64_t* labels_c = (int64_t*)(base + ws.labels);
  float* lse_c = (float*)(base + ws.lse);
  float* ex_c = (float*)(base + ws.ex);
  float* g_lp_c = (float*)(base + ws.g_lp);
  float* g_ent_c = (float*)(base + ws.g_ent);
  void* dh_c = base + ws.dh;
  if (int rc = siirl_gather_rows(hidden, rows, n_rows, row_bytes, T, hidden_c, stream)) return rc;
  gather_token_operands_kernel<<<dim3((unsigned)((n_rows + 255) / 256)), dim3(256), 0, st>>>(
      rows, n_rows, T, labels, lse, ex, g_logprob, g_entropy, labels_c, lse_c, ex_c, g_lp_c, g_ent_c);
  SIIRL_LAUNCH_CHECK("gather_token_operands_kernel");
  if (int rc = siirl_fused_linear_logprob_entropy_bwd(hidden_c, weight, dtype, labels_c, n_rows, H, V, inv_temperature,
                                                      lse_c, ex_c, nullptr, g_logprob ? g_lp_c : nullptr,
                                                      g_entropy ? g_ent_c : nullptr, want_dh ? dh_c : nullptr, d_weight,
                                                      base + ws.inner, ws.inner_bytes, stream))
    return rc;
  if (want_dh)
    if (int rc = siirl_scatter_rows(dh_c, rows, n_rows, row_bytes, T, d_hidden, stream)) return rc;
  return SIIRL_OK;
}
