// GEMM C = A * B for f16/bf16 A [M, K] and B [K, N], each stored row-major or transposed,
// float32 accumulation: the fast path behind tk_gemm (src/tklab/kernels/matmul.py:72-164
// computes the same product with a Triton tile loop).
//
// Block tile 256 x 256, K step 32, 512 threads = 8 wave64s in a 2 (M) x 4 (N) grid, two
// waves per SIMD; each wave owns 128 x 64 of C as 8 x 4 tiles of v_mfma_f32_16x16x32
// (128 accumulators). With two waves per SIMD, one wave's LDS reads, DMA issue and
// barrier waits are covered by the other wave's MFMAs. 16x16x32 rather than 32x32x16:
// the clock is power-limited under dense MFMA load, and the 16x16 shape sustains more
// FLOP/s (MFMA-only with random operands 1.90 vs 1.78 PFLOP/s bf16; this GEMM 1.39 vs
// 1.29 PFLOP/s at 8192^3 with the same tiles and LDS traffic). The MFMAs compute C^T
// tiles (the B fragment as the first operand), so a lane's four accumulator registers
// are four consecutive columns of one row (8 bytes once rounded). The epilogue stages the
// rounded tile in the idle rings and writes whole rows from there.
//
// Operands reach LDS by buffer->LDS DMA (buffer_load_dwordx4 ... lds): no VGPR staging.
// A and B have rings of their own: A in 64-wide K tiles (three stages of 256 rows x 128 B),
// B in 32-wide K tiles (four stages of 32 k-rows x 512 B), 160 KiB in all. Each DMA request
// then covers a whole 128-byte line: with 32-wide A tiles every A row was a 64-byte half
// line, and the vector memory path (texture data unit 95 % busy, two thirds of it waiting
// on L1, L1 waiting on L2 two thirds of the time) moved a third more requests than bytes
// needed. The loop runs 32-wide steps with one barrier each, placed between the wave's
// row tiles 0-3 and 4-7: rows 0-3 run while rows 4-7 of the same step are read and the
// step's DMA is issued; rows 4-7 run while the next step's rows 0-3 and B fragments (a
// second register set) are read.
//
// Stage layout (bytes), chosen so every LDS read phase touches 64 distinct banks:
//   A: 256 rows x 128 B; the 16-byte chunk c (k = 8c .. 8c+7 of the 64-wide tile) of row r
//      sits at chunk c ^ a_swz(r), a_swz(r) = (r >> 1) & 7. A fragment (16 rows, lane
//      group g taking k = 8g .. 8g+7 of the step's 32-wide half) is one ds_read_b128.
//   B: 32 k-rows x 512 B, row-major in n; the 32-byte granule g (n = 16g .. 16g+15) of
//      k-row k sits at granule g ^ (2 * (k & 3) + ((k >> 3) & 1)). Fragments are read
//      with ds_read_b64_tr_b16, which transposes 4 k x 16 n blocks into the MFMA B
//      layout: two reads give one lane its 8 consecutive k of one column. One read phase
//      (32 lanes) covers two lane groups on k-rows 8 apart; the (k >> 3) term puts their
//      8 granules on distinct banks.
// A DMA instruction moves 64 lanes x 16 B into 1 KiB of contiguous LDS at M0, so the
// swizzle is applied on the global side: each lane fetches the chunk that belongs at its
// LDS slot.
//
// The compiler inserts vmcnt(0) before any LDS read that may alias an LDS DMA, which
// would drain the prefetch ring every step; fragment reads are therefore inline asm
// ordered by explicit s_waitcnt, with the MFMA/LDS/DMA interleave pinned by
// sched_barrier.
//
// Tile order: workgroup w runs on XCD w % 8; tiles are renumbered so each XCD walks a
// contiguous range in groups of 4 M-tiles, sharing A and B panels in that XCD's L2.
//
// Transposed operands (a linear layer's gradients dy * w^T and x^T * dy) keep the tiles, the
// steps and the order of every sum; only what a stage holds and how its fragments are read
// changes. A [K][M] comes in 32-wide k-row tiles like B and is read transposed (TN); B [N][K]
// comes in 64-wide tiles like A and is read as rows (NT). Loading them element by element
// through registers (the general kernel in gemm.hip) ran 8192 x 4096 x 4096 in 4.1 ms each
// way, bound by its 2-byte loads; these run dy * w^T and x^T * dy at the row-major product's
// speed (all three products: 8.41 -> 0.584 ms, 1.41 PFLOP/s bf16).
//
// Row-scaled variant (kRowScale): C[m, :] = round(s[m] * acc),
// one float32 multiply before the rounding. With s = rstd of a normalization whose
// weight is folded into B, this is the normalized GEMM rms_norm(a) * B' without the
// normalized activations ever being written.
//
// SwiGLU variant (kSwiGLU): Y = swiglu(value = A*B_up, gate = A*B_gate) for two weights
// [K, N]. A block computes 256 x 128 of Y from a 256-column B tile holding the gate
// columns n0..n0+127 then the same up columns, laid out in LDS as two 128-column blocks
// (256-byte k-rows, same granule swizzle: still 64 distinct banks per read phase), so
// every B DMA instruction reads one weight. Wave (wm, wq) takes gate columns 32wq ..
// 32wq+31 as its N tiles 0, 1 and the same up columns as N tiles 2, 3, and
// the epilogue rounds both to the storage type (as the unfused GEMMs store them) and
// writes value * gate * sigmoid(gate): the two M x N intermediates never reach HBM and
// the result is bitwise that of the two GEMMs followed by the SwiGLU kernel.
#include "gemm_device.hpp"
#include "gemm_tile.hpp"

#include <algorithm>

#pragma clang fp contract(off)

namespace {

using namespace tk::gemm_dma;

constexpr int BM = 256, BN = 256, BK = 32;
constexpr int kThreads = 512;  // 8 waves
constexpr int kGroupM = 4;
// K-contiguous operands come in 64-wide K tiles (256 rows x 128 B), the others in 32-wide K
// tiles (32 k-rows x 512 B). NN: three 64-wide A stages and four 32-wide B stages; NT: three
// 64-wide A and two 64-wide B stages; TN: four 32-wide stages of each. At most 160 KiB: all
// of the CU's LDS.
constexpr int kAStages = 3, kBStages = 4;
constexpr int kABytes = 256 * 64 * 2;        // 32 KiB per 64-wide stage
constexpr int kOperandBytes = 256 * BK * 2;  // 16 KiB per 32-wide stage
constexpr int kLdsBytes = kAStages * kABytes + kBStages * kOperandBytes;
// Epilogue: the C tile is staged in the ring's LDS (at most 256 rows of 528 bytes), the row
// scales of the row-scaled variant after it.
constexpr int kScaleOff = 256 * 528;
static_assert(kScaleOff + 256 * 4 <= kLdsBytes, "row scales past the LDS block");

// Sources of the DMA instructions a wave issues per tile: src for full tiles, last for the
// operand's last tile, of which kv K columns (or k-rows) lie inside K. What lies past K in a
// K-contiguous operand is the next row, inside the buffer, so lanes past kv must read nothing
// (kOob) on their own; k-rows past K are past the buffer's end (the range check covers soffset,
// which carries a tile's offset) and follow the same rule. K % 8 == 0 wherever K is contiguous, so
// a lane's chunk is wholly inside or outside.
//
// 64-wide tile of a K-contiguous operand, instruction x (0..3): rows 8 (4 wave + x) .. +7,
// eight lanes per 128-byte row; each lane fetches the chunk that belongs at its LDS slot.
__device__ __forceinline__ void wide_source(int x, int wave, int lane, int row0, int rows, int ld,
                                            int kv, uint32_t& src, uint32_t& last) {
  const int r = (wave * 4 + x) * 8 + (lane >> 3);
  const int c = (lane & 7) ^ a_swz(r);
  src = (row0 + r < rows) ? uint32_t((row0 + r) * ld + c * 8) * 2u : kOob;
  last = c * 8 < kv ? src : kOob;
}

// 32-wide tile of an operand stored by k-rows, instruction i (0, 1): two k-rows of 512 B.
__device__ __forceinline__ void krow_source(int i, int wave, int lane, int col0, int cols, int ld,
                                            int kv, uint32_t& src, uint32_t& last) {
  const int kr = (wave * 2 + i) * 2 + (lane >> 5);
  const int slot = lane & 31;
  const int chunk = (((slot >> 1) ^ b_swz(kr)) << 1) | (slot & 1);
  src = (col0 + chunk * 8 < cols) ? uint32_t(kr * ld + col0 + chunk * 8) * 2u : kOob;
  last = kr < kv ? src : kOob;
}

// One 256 x 256 tile (256 x 128 of Y with kSwiGLU). kKTail: K need not be a multiple of 32.
template <typename T, Layout kLayout, bool kKTail, bool kSwiGLU, bool kRowScale>
__device__ __forceinline__ void gemm_tile_256(const T* __restrict__ A, const T* __restrict__ B,
                                              const T* __restrict__ B2, T* __restrict__ C,
                                              const Problem& p) {
  constexpr bool kARows = kLayout == Layout::TN;  // A stored by k-rows [K][M]
  constexpr bool kBWide = kLayout == Layout::NT;  // B stored K-contiguous [N][K]
  constexpr int kBRing = kARows ? kBStages * kOperandBytes : kAStages * kABytes;
  constexpr int kTileN = kSwiGLU ? 128 : BN;
  constexpr int kRowB = kSwiGLU ? 256 : 512;
  __shared__ __attribute__((aligned(1024))) char lds[kLdsBytes];

  const int total = p.tiles_m * p.tiles_n;
  int w = blockIdx.x;
  if (total % kXcds == 0) w = (w % kXcds) * (total / kXcds) + w / kXcds;
  const int per_group = kGroupM * p.tiles_n;
  const int first_m = (w / per_group) * kGroupM;
  const int group_m = min(p.tiles_m - first_m, kGroupM);
  const int tile_m = first_m + (w % per_group) % group_m;
  const int tile_n = (w % per_group) / group_m;
  const int m0 = tile_m * BM, n0 = tile_n * kTileN;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = (wave >> 2) * 128, wn = (wave & 3) * 64;
  const int l16 = lane & 15, lg = lane >> 4;
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc((void*)A, (short)0, p.a_bytes, 0x00020000);
  const bool up_half = kSwiGLU && wave >= 4;
  const __amdgpu_buffer_rsrc_t rb =
      up_half ? __builtin_amdgcn_make_buffer_rsrc((void*)B2, (short)0, p.b2_bytes, 0x00020000)
              : __builtin_amdgcn_make_buffer_rsrc((void*)B, (short)0, p.b_bytes, 0x00020000);
  const int ldb = up_half ? p.ldb2 : p.ldb;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_void*)lds;

  const int kt = (p.k + BK - 1) / BK;  // 32-wide K tiles
  const int kt64 = (kt + 1) / 2;       // 64-wide K tiles (the last one half used when kt is odd)
  const int kv64 = p.k - (kt64 - 1) * 64, kv32 = p.k - (kt - 1) * 32;
  constexpr int kADma = kARows ? 2 : 4, kBDma = kBWide ? 4 : 2;
  uint32_t a_src[kADma], a_last[kADma], b_src[kBDma], b_last[kBDma];
#pragma unroll
  for (int x = 0; x < kADma; ++x) {
    if constexpr (kARows)
      krow_source(x, wave, lane, m0, p.m, p.lda, kv32, a_src[x], a_last[x]);
    else
      wide_source(x, wave, lane, m0, p.m, p.lda, kv64, a_src[x], a_last[x]);
  }
#pragma unroll
  for (int i = 0; i < kBDma; ++i) {
    if constexpr (kSwiGLU) {
      const int L = wave * 2 + i;
      const int kr = 4 * (L & 7) + (lane >> 4);
      const int slot = lane & 15;
      const int chunk = (((slot >> 1) ^ b_swz(kr)) << 1) | (slot & 1);
      b_src[i] = (n0 + chunk * 8 < p.n) ? uint32_t(kr * ldb + n0 + chunk * 8) * 2u : kOob;
    } else if constexpr (kBWide) {
      wide_source(i, wave, lane, n0, p.n, ldb, kv64, b_src[i], b_last[i]);
    } else {
      krow_source(i, wave, lane, n0, p.n, ldb, kv32, b_src[i], b_last[i]);
    }
  }
  const uint32_t a_tile_bytes = kARows ? uint32_t(BK * p.lda) * 2u : 128u;
  const uint32_t b_tile_bytes = kBWide ? 128u : uint32_t(BK * ldb) * 2u;

  float row_scale = 0.f;
  if constexpr (kRowScale)
    if (threadIdx.x < BM) row_scale = p.row_scale[min(m0 + (int)threadIdx.x, p.m - 1)];

  // Tiles past the end reload the last one into a stage that is never read, keeping every
  // step's DMA count constant. `stage`: the stage's byte offset in the operand's ring.
  auto dma_a = [&](int x, int tile, int stage) {
    const int end = (kARows ? kt : kt64) - 1;
    tile = min(tile, end);
    const bool last = tile == end && (!kARows || kKTail);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        ra, (lds_void*)(lds + stage + (wave * kADma + x) * 1024), 16,
        last ? a_last[x] : a_src[x], tile * a_tile_bytes, 0, 0);
  };
  auto dma_b = [&](int x, int tile, int stage) {
    const int end = (kBWide ? kt64 : kt) - 1;
    tile = min(tile, end);
    const bool last = tile == end && (kBWide || kKTail);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rb, (lds_void*)(lds + kBRing + stage + (wave * kBDma + x) * 1024), 16,
        last ? b_last[x] : b_src[x], tile * b_tile_bytes, 0, 0);
  };

  // A: row wm + l16 (+16 per row tile), chunk lg (first 32-wide half of the 64-wide tile)
  // or 4 + lg (second half), swizzled (a_swz reads only the row's low four bits, the same
  // for every row tile). B: k-rows 8 lg + (l16 >> 2) (+4), columns of N tile j starting at
  // 4 (l16 & 3). A by k-rows is read like B, a wide B like A.
  uint32_t a_addr0, a_addr1, b_addr[4];
  {
    const int jj = l16 >> 2, q = l16 & 3;
    const int kr = 8 * lg + jj;
    const int sw = b_swz(kr);
    if constexpr (kARows) {
      // Row tile I's granule is (wm / 16 + I) ^ sw; wm / 16 is a multiple of 8, so I flips
      // address bits 5..7 (read_a_frag).
      a_addr0 = a_addr1 = kr * 512 + (((wm / 16) ^ sw) * 32) + q * 8;
    } else {
      a_addr0 = (wm + l16) * 128 + ((lg ^ a_swz(l16)) * 16);
      a_addr1 = (wm + l16) * 128 + (((4 + lg) ^ a_swz(l16)) * 16);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (kSwiGLU) {
        // N tiles 0, 1: gate columns 32 (wave & 3) + 16 j; tiles 2, 3: the same up columns.
        const int g = 2 * (wave & 3) + (j & 1);
        b_addr[j] = (j >> 1) * 8192 + kr * 256 + ((g ^ sw) * 32) + q * 8;
      } else if constexpr (kBWide) {
        b_addr[j] = (wn + l16) * 128 + ((((j & 1) * 4 + lg) ^ a_swz(l16)) * 16);  // [half]
      } else {
        const int g = wn / 16 + j;
        b_addr[j] = kr * 512 + ((g ^ sw) * 32) + q * 8;
      }
    }
  }
  // Where the reads of half H of the A stage at LDS offset `stage` start, and row tile I's
  // fragment from there. The start is formed ahead of the pinned MFMA sequence.
  auto a_base = [&](auto half, uint32_t stage) {
    return lds_base + stage + (kARows ? 0 : decltype(half)::value ? a_addr1 : a_addr0);
  };
  auto read_a_frag = [&](auto tile, uint32_t base) {
    constexpr int I = decltype(tile)::value;
    if constexpr (kARows)
      return read_b<512>(base + (a_addr0 ^ (I << 5)));
    else
      return read_a<I>(base);
  };
  // N tile J's fragment of the B stage at `base` (64-wide half H of a wide B).
  auto read_b_frag = [&](auto tile, auto half, uint32_t base) {
    constexpr int J = decltype(tile)::value;
    if constexpr (kBWide)
      return read_a<J>(base + b_addr[decltype(half)::value]);
    else
      return read_b<kRowB>(base + b_addr[J]);
  };

  f32x4 acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // DMA schedule (NN). 32-wide step t issues B tile t + 3 (two instructions per wave) into B
  // stage (t + 3) % 4 and, when t is odd, the 64-wide A tile (t + 3) / 2 (four per wave)
  // into A stage ((t + 3) / 2) % 3. A stage reuse: A tile v's last fragments (rows 4-7 of
  // step 2v + 1) are read in the first half of step 2v + 1 and waited for after that step's
  // barrier, so every wave is done with them at the barrier of step 2v + 2; tile v + 3
  // refills the stage from step 2v + 3 on. B stage reuse: B tile t's fragments are read in
  // the second half of step t - 1 and waited for at the start of step t; tile t + 4 refills
  // the stage in step t + 1. Step t's barrier needs 32-wide tile t + 1 landed, issued in
  // step t - 2 or earlier, so each wave waits until at most the 8 instructions of steps
  // t - 1 and t are in flight. The prologue is steps -3 .. -1 of the same schedule.
  //
  // TN. A comes by k-rows in a ring like B's. Its tile t's last fragments (rows 4-7) are
  // waited for after the barrier of step t, so the refill of that stage (tile t + 4) is
  // issued in the second half of step t + 1, after the next barrier. At the barrier of step
  // t, tile t + 1 of both must have landed: A's was issued in the second half of step t - 2,
  // and B t + 2, A t + 2 and B t + 3 (6 instructions) came after it.
  //
  // NT. B comes in 64-wide tiles, two stages. Tile v's last fragments (step 2v + 1's, read in
  // the second half of step 2v) are waited for at the start of step 2v + 1, so tile v + 2
  // refills the stage in the second half of step 2v + 1, two steps before the barrier that
  // publishes it (step 2v + 3's, where only A tile v + 3's 4 instructions may be in flight).
  constexpr int kAStage = kARows ? kOperandBytes : kABytes;
  constexpr int kBStage = kBWide ? kABytes : kOperandBytes;
  auto tile_a = [&](int tile) {
#pragma unroll
    for (int x = 0; x < kADma; ++x) dma_a(x, tile, tile * kAStage);
  };
  auto tile_b = [&](int tile) {
#pragma unroll
    for (int x = 0; x < kBDma; ++x) dma_b(x, tile, tile * kBStage);
  };
  if constexpr (kARows) {
    tile_b(0); tile_a(0); tile_b(1); tile_a(1); tile_b(2); tile_a(2);
  } else if constexpr (kBWide) {
    tile_a(0); tile_b(0); tile_a(1); tile_b(1);
  } else {
    tile_a(0); tile_b(0); tile_b(1); tile_a(1); tile_b(2);
  }
  wait_vmcnt<8>();
  barrier_no_fence();

  using Half0 = std::integral_constant<int, 0>;
  using Half1 = std::integral_constant<int, 1>;
  i32x4 a_lo[4], a_hi[4], b0[4], b1[4];
  unroll4([&](auto i) {
    constexpr int x = decltype(i)::value;
    a_lo[x] = read_a_frag(i, a_base(Half0{}, 0));
    b0[x] = read_b_frag(i, Half0{}, lds_base + kBRing);
  });

  // One 32-wide step t, half H of 64-wide K tile u = t / 2. `ao` is the tile's stage in a
  // 64-wide A ring, `ao_next` the next tile's, `ao_fill` the third one; `bo` is the stage of
  // step 2u in a 32-wide ring (0 or 2 stages in, so the others are XORs away) or of tile u in
  // the two-stage 64-wide B ring. All are byte offsets. Bc holds this step's B fragments, Bn
  // receives the next step's.
  auto step = [&](auto half, int t, int ao, int ao_next, int ao_fill, int bo, i32x4 (&Bc)[4],
                  i32x4 (&Bn)[4]) {
    constexpr int H = decltype(half)::value;
    using Next = std::integral_constant<int, 1 - H>;
    const int rows_cur = H ? bo ^ kOperandBytes : bo;
    const int rows_next = H ? bo ^ 2 * kOperandBytes : bo ^ kOperandBytes;
    const int rows_fill = H ? bo : bo ^ 3 * kOperandBytes;  // stage (t + 3) % 4
    const int wide_next = H ? bo ^ kABytes : bo;
    const uint32_t a_cur = a_base(half, kARows ? rows_cur : ao);
    const uint32_t a_next = a_base(Next{}, kARows ? rows_next : H ? ao_next : ao);
    const uint32_t b_next = lds_base + kBRing + (kBWide ? wide_next : rows_next);
    wait_lgkm_pin(a_lo);
    wait_lgkm_pin(Bc);
    sched_fence();
    // Rows 0-3; read rows 4-7 of this step, issue the DMA.
    unroll4([&](auto row) {
      unroll4([&](auto col) {
        constexpr int i = decltype(row)::value, j = decltype(col)::value;
        acc[i][j] = Mfma<T>::run(Bc[j], a_lo[i], acc[i][j]);
        sched_fence();
        if constexpr (j == 0)
          a_hi[i] = read_a_frag(std::integral_constant<int, 4 + i>{}, a_cur);
        if constexpr (!kARows && H == 1 && j == 1) dma_a(i, (t + 3) >> 1, ao_fill);
        if constexpr (!kBWide && j == 3 && (i & 1) == 0) dma_b(i >> 1, t + 3, rows_fill);
        sched_fence();
      });
    });
    wait_vmcnt<kARows ? 6 : kBWide && H == 1 ? 4 : 8>();
    barrier_no_fence();
    wait_lgkm_pin(a_hi);
    sched_fence();
    // Rows 4-7; read rows 0-3 and B of step t + 1.
    unroll4([&](auto row) {
      unroll4([&](auto col) {
        constexpr int i = decltype(row)::value, j = decltype(col)::value;
        acc[4 + i][j] = Mfma<T>::run(Bc[j], a_hi[i], acc[4 + i][j]);
        sched_fence();
        if constexpr (j == 0) a_lo[i] = read_a_frag(row, a_next);
        if constexpr (kARows && j == 1 && (i & 1) == 0) dma_a(i >> 1, t + 3, rows_fill);
        if constexpr (j == 2) Bn[i] = read_b_frag(row, Next{}, b_next);
        if constexpr (kBWide && H == 1 && j == 3) dma_b(i, (t + 3) >> 1, bo);
        sched_fence();
      });
    });
  };

  int ao = 0, bo = 0;
  for (int u = 0; 2 * u < kt; ++u) {
    const int ao_next = ao == (kAStages - 1) * kABytes ? 0 : ao + kABytes;
    const int ao_fill = 3 * kABytes - ao - ao_next;
    step(Half0{}, 2 * u, ao, ao_next, ao_fill, bo, b0, b1);
    if (2 * u + 1 < kt) step(Half1{}, 2 * u + 1, ao, ao_next, ao_fill, bo, b1, b0);
    ao = ao_next;
    bo ^= kBWide ? kABytes : 2 * kOperandBytes;
  }
  wait_vmcnt<0>();
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");

  // acc[i][j] holds C^T: register r of lane l is C[m][n] with m = m0 + wm + 16 i + l % 16 and
  // n = n0 + (N tile j's first column) + 4 (l / 16) + r: four consecutive columns of one row.
  // The rings are idle once every wave is here.
  __syncthreads();
  const float* scales = reinterpret_cast<const float*>(lds + kScaleOff);
  if constexpr (kRowScale) {
    if (threadIdx.x < BM) reinterpret_cast<float*>(lds + kScaleOff)[threadIdx.x] = row_scale;
    __syncthreads();
  }
  // The tile's outputs as (row within the tile, column within the tile, four values).
  auto for_each_out = [&](auto&& emit) {
    if constexpr (kSwiGLU) {
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r)
            v[r] = static_cast<float>(swiglu_out<T>(acc[i][jj][r], acc[i][jj + 2][r]));
          emit(wm + i * 16 + l16, (wave & 3) * 32 + jj * 16 + lg * 4, v);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float sc = kRowScale ? scales[wm + i * 16 + l16] : 1.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = kRowScale ? acc[i][j][r] * sc : acc[i][j][r];
          emit(wm + i * 16 + l16, wn + j * 16 + lg * 4, v);
        }
      }
    }
  };
  static_assert(BM * stage_stride(kTileN) <= kScaleOff, "staged tile overlaps the row scales");
  store_tile<T, BM, kTileN, kThreads>(C, p, m0, n0, lds, for_each_out);
}


// Row-major operands with K % 32 == 0 (NN), and the fused variants.
template <typename T, bool kSwiGLU, bool kRowScale>
__global__ __attribute__((amdgpu_flat_work_group_size(kThreads, kThreads),
                          amdgpu_waves_per_eu(2, 2))) void
gemm_dma_kernel(const T* __restrict__ A, const T* __restrict__ B, const T* __restrict__ B2,
                T* __restrict__ C, Problem p) {
  gemm_tile_256<T, Layout::NN, false, kSwiGLU, kRowScale>(A, B, B2, C, p);
}

// Transposed operands and K % 32 != 0.
template <typename T, Layout kLayout>
__global__ __attribute__((amdgpu_flat_work_group_size(kThreads, kThreads),
                          amdgpu_waves_per_eu(2, 2))) void
gemm_kernel(const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C, Problem p) {
  gemm_tile_256<T, kLayout, true, false, false>(A, B, B, C, p);
}

}  // namespace

namespace tk {

namespace gemm_dma {

bool plan(const void* a, const void* b, int64_t m, int64_t n, int64_t k, int64_t stride_am,
          int64_t stride_ak, int64_t stride_bk, int64_t stride_bn, Plan* plan) {
  // Buffer offsets are 32-bit with kOob (2^31) reserved as "outside"; strides are positive (the
  // offsets are unsigned). An operand is stored as `rows` rows of `cols` contiguous values.
  if (m <= 0 || n <= 0 || k <= 0 || stride_am <= 0 || stride_ak <= 0 || stride_bk <= 0 ||
      stride_bn <= 0)
    return false;
  auto stored = [](const void* p, int64_t rows, int64_t cols, int64_t row_stride,
                   int64_t col_stride) {
    return col_stride == 1 && cols % 8 == 0 && row_stride % 8 == 0 && aligned16(p) &&
           (extent(rows, row_stride, 1, 0) + cols) * 2 < int64_t(kOob);
  };
  const bool a_k = stored(a, m, k, stride_am, stride_ak);  // [M][K]
  const bool a_m = stored(a, k, m, stride_ak, stride_am);  // [K][M]
  const bool b_n = stored(b, k, n, stride_bk, stride_bn);  // [K][N]
  const bool b_k = stored(b, n, k, stride_bn, stride_bk);  // [N][K]
  if (a_k && b_n)
    *plan = {Layout::NN, false, k % BK != 0, stride_am, stride_bk};
  else if (a_k && b_k)
    *plan = {Layout::NT, false, true, stride_am, stride_bn};
  else if (a_m && b_n)
    *plan = {Layout::TN, false, true, stride_ak, stride_bk};
  else if (a_m && b_k)  // C^T = B^T A^T, both row-major
    *plan = {Layout::NN, true, true, stride_bn, stride_ak};
  else
    return false;
  return true;
}

// A launch takes about (tiles a CU gets) x (operand lines per tile): see gemm_tile_kernels.hpp.
// The constants are cycles: kPerLine for each 128-byte line of a 64-wide K tile (one tile row
// or column; rows past the problem's edge count, their DMA slots carry nothing else), kPerTile
// for a tile's first loads and its epilogue. Against every tile of kTiles on 30 problems from
// 1x4096x4096 to 5000x5000x2048 (three layouts, SwiGLU) the choice is the fastest or within 6 %
// of it. 256 x 256 against the chosen tile, bf16: 1024^3 22.3 -> 11.3 us (64 x 64; 11 us is the
// host's time per call), 2048^3 39.0 -> 20.0 (128 x 128), 1000x6144x4096 74.9 -> 49.0 (128 x
// 192), 3000^3 61.5 -> 53.0 (192 x 192), 8192x1024x4096 71.5 -> 59.6 (128 x 256), 16x4096x4096
// 66.5 -> 15.3 (64 x 64); 4096^3 100 (256 x 256) against 121 (256 x 128).
int pick_tile(const Tile* tiles, int count, int64_t m, int64_t n, int64_t k, Variant variant) {
  constexpr double kPerLine = 6.1, kPerTile = 4000.0;
  constexpr int64_t kCus = 256;
  int best = 0;
  double best_cost = 0;
  for (int i = 0; i < count; ++i) {
    const Tile& t = tiles[i];
    if (variant == Variant::kSwiGLU && t.n % 128 != 0) continue;
    const int64_t out_n = variant == Variant::kSwiGLU ? t.n / 2 : t.n;
    const int64_t rounds = cdiv(cdiv(m, t.m) * cdiv(n, out_n), kCus);
    const double cost = double(rounds) * (kPerTile + kPerLine * (t.m + t.n) * double(cdiv(k, 64)));
    if (i == 0 || cost < best_cost) {
      best = i;
      best_cost = cost;
    }
  }
  return best;
}

}  // namespace gemm_dma

bool gemm_dma_applies(const void* a, const void* b, int64_t m, int64_t n, int64_t k,
                      int64_t stride_am, int64_t stride_ak, int64_t stride_bk,
                      int64_t stride_bn) {
  gemm_dma::Plan p;
  return gemm_dma::plan(a, b, m, n, k, stride_am, stride_ak, stride_bk, stride_bn, &p) &&
         p.layout == gemm_dma::Layout::NN && !p.swap && !p.k_tail;
}

namespace {

template <typename T>
void launch_256(const gemm_dma::Plan& plan, const void* a, const void* b, void* c,
                const Problem& p, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(p.tiles_m * p.tiles_n)), block(kThreads);
  const T* pa = static_cast<const T*>(a);
  const T* pb = static_cast<const T*>(b);
  T* pc = static_cast<T*>(c);
  if (p.row_scale != nullptr)
    hipLaunchKernelGGL((gemm_dma_kernel<T, false, true>), grid, block, 0, stream, pa, pb, pb, pc, p);
  else if (plan.layout == Layout::NN && !plan.k_tail)
    hipLaunchKernelGGL((gemm_dma_kernel<T, false, false>), grid, block, 0, stream, pa, pb, pb, pc, p);
  else if (plan.layout == Layout::NN)
    hipLaunchKernelGGL((gemm_kernel<T, Layout::NN>), grid, block, 0, stream, pa, pb, pc, p);
  else if (plan.layout == Layout::NT)
    hipLaunchKernelGGL((gemm_kernel<T, Layout::NT>), grid, block, 0, stream, pa, pb, pc, p);
  else
    hipLaunchKernelGGL((gemm_kernel<T, Layout::TN>), grid, block, 0, stream, pa, pb, pc, p);
}

}  // namespace

void gemm_dma_launch(const gemm_dma::Plan& plan, int dtype, const void* a, const void* b, void* c,
                     int64_t m, int64_t n, int64_t k, int64_t stride_cm, int64_t stride_cn,
                     hipStream_t stream, const float* row_scale) {
  if (plan.swap) {
    std::swap(a, b);
    std::swap(m, n);
    std::swap(stride_cm, stride_cn);
  }
  const Variant variant = row_scale != nullptr ? Variant::kRowScale : Variant::kPlain;
  const int tile = pick_tile(kTiles, kTileCount, m, n, k, variant);
  const int64_t a_rows = plan.layout == Layout::TN ? k : m, a_cols = plan.layout == Layout::TN ? m : k;
  const int64_t b_rows = plan.layout == Layout::NT ? n : k, b_cols = plan.layout == Layout::NT ? k : n;
  const uint32_t b_bytes = (uint32_t)(((b_rows - 1) * plan.ldb + b_cols) * 2);
  Problem p{(int)m,
            (int)n,
            (int)k,
            (int)plan.lda,
            (int)plan.ldb,
            (int)plan.ldb,
            stride_cm,
            stride_cn,
            (int)cdiv(m, kTiles[tile].m),
            (int)cdiv(n, kTiles[tile].n),
            (uint32_t)(((a_rows - 1) * plan.lda + a_cols) * 2),
            b_bytes,
            b_bytes,
            row_scale};
  if (tile != 0) {
    if (dtype == TK_DTYPE_F16)
      launch_tile<_Float16>(tile, variant, plan, a, b, b, c, p, stream);
    else
      launch_tile<__bf16>(tile, variant, plan, a, b, b, c, p, stream);
  } else if (dtype == TK_DTYPE_F16) {
    launch_256<_Float16>(plan, a, b, c, p, stream);
  } else {
    launch_256<__bf16>(plan, a, b, c, p, stream);
  }
}

bool gemm_split_launch(int dtype, const void* a, const void* b, const void* b_up,
                       const float* row_scale, void* c, float* partial, int64_t m, int64_t n,
                       int64_t k, int64_t splits, const int64_t* strides, hipStream_t stream) {
  const int64_t sam = strides[0], sak = strides[1], sbk = strides[2], sbn = strides[3];
  const int64_t suk = strides[4], sun = strides[5];
  int64_t scm = strides[6], scn = strides[7];
  gemm_dma::Plan plan;
  if (!gemm_dma::plan(a, b, m, n, k, sam, sak, sbk, sbn, &plan)) return false;
  const Variant variant = b_up != nullptr        ? Variant::kSwiGLU
                          : row_scale != nullptr ? Variant::kRowScale
                                                 : Variant::kPlain;
  if (variant != Variant::kPlain &&
      (!gemm_dma_applies(a, b, m, n, k, sam, sak, sbk, sbn) ||
       (b_up != nullptr && !gemm_dma_applies(a, b_up, m, n, k, sam, sak, suk, sun))))
    return false;
  if (plan.swap) {
    std::swap(a, b);
    std::swap(m, n);
    std::swap(scm, scn);
  }
  const bool a_rows = plan.layout == Layout::TN, b_wide = plan.layout == Layout::NT;
  auto bytes = [](int64_t rows, int64_t ld, int64_t cols) {
    return (uint32_t)(((rows - 1) * ld + cols) * 2);
  };
  const int64_t kt = cdiv(k, 64), per = cdiv(kt, splits);
  Problem p{(int)m,
            (int)n,
            (int)k,
            (int)plan.lda,
            (int)plan.ldb,
            (int)(b_up != nullptr ? suk : plan.ldb),
            scm,
            scn,
            (int)cdiv(m, 64),
            (int)cdiv(n, 64),
            bytes(a_rows ? k : m, plan.lda, a_rows ? m : k),
            bytes(b_wide ? n : k, plan.ldb, b_wide ? k : n),
            b_up != nullptr ? bytes(k, suk, n) : 0u,
            row_scale,
            partial,
            (int)per};
  const int runs = (int)cdiv(kt, per);  // no run is empty
  if (dtype == TK_DTYPE_F16)
    launch_split<_Float16>(variant, plan, a, b, b_up, c, p, runs, stream);
  else
    launch_split<__bf16>(variant, plan, a, b, b_up, c, p, runs, stream);
  return true;
}

void gemm_swiglu_dma_launch(int dtype, const void* a, const void* b_gate, const void* b_up,
                            void* y, int64_t m, int64_t n, int64_t k, int64_t stride_am,
                            int64_t stride_gk, int64_t stride_uk, int64_t stride_ym,
                            int64_t stride_yn, hipStream_t stream) {
  const int tile = pick_tile(kTiles, kTileCount, m, n, k, Variant::kSwiGLU);
  Problem p{(int)m,
            (int)n,
            (int)k,
            (int)stride_am,
            (int)stride_gk,
            (int)stride_uk,
            stride_ym,
            stride_yn,
            (int)cdiv(m, kTiles[tile].m),
            (int)cdiv(n, kTiles[tile].n / 2),
            (uint32_t)(((m - 1) * stride_am + k) * 2),
            (uint32_t)(((k - 1) * stride_gk + n) * 2),
            (uint32_t)(((k - 1) * stride_uk + n) * 2),
            nullptr};
  const dim3 grid(static_cast<unsigned>(p.tiles_m * p.tiles_n));
  const gemm_dma::Plan plan{Layout::NN, false, false, stride_am, stride_gk};
  if (tile != 0) {
    if (dtype == TK_DTYPE_F16)
      launch_tile<_Float16>(tile, Variant::kSwiGLU, plan, a, b_gate, b_up, y, p, stream);
    else
      launch_tile<__bf16>(tile, Variant::kSwiGLU, plan, a, b_gate, b_up, y, p, stream);
    return;
  }
  if (dtype == TK_DTYPE_F16)
    hipLaunchKernelGGL((gemm_dma_kernel<_Float16, true, false>), grid, dim3(kThreads), 0, stream,
                       static_cast<const _Float16*>(a), static_cast<const _Float16*>(b_gate),
                       static_cast<const _Float16*>(b_up), static_cast<_Float16*>(y), p);
  else
    hipLaunchKernelGGL((gemm_dma_kernel<__bf16, true, false>), grid, dim3(kThreads), 0, stream,
                       static_cast<const __bf16*>(a), static_cast<const __bf16*>(b_gate),
                       static_cast<const __bf16*>(b_up), static_cast<__bf16*>(y), p);
}

}  // namespace tk
