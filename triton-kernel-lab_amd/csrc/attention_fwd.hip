// Flash attention forward for head_dim 64/128 (f16/bf16) on CDNA4 MFMA: the path behind
// tk_attn_fwd (src/tklab/kernels/flash_attention.py:124-264 is the Triton kernel it
// replaces: base-2 online softmax on scores * scale * log2(e) in _attention_inner
// (:55-121), O = acc / l and log-sum-exp m + log2(l) (:248-264)).
//
// Workgroup: 256 queries, 8 wave64s of 32 queries (two 16-query tiles), two waves per SIMD.
// Key/value blocks of 64 (four 16-key tiles). All products are v_mfma_f32_16x16x32.
//
// Per wave and key block j:
//   S^T = K Q^T     4 key tiles x 2 query tiles over D/32 k-steps: lane l holds query
//                   16 qt + l % 16 and keys 16 kt + 4 (l / 16) + {0..3}, so a query's
//                   maximum and sum span the four lanes l % 16 + 16 {0..3} (permlane32 and
//                   permlane16 swaps).
//   softmax         masked only on diagonal / ragged blocks. The reference maximum only
//                   moves when a block's maximum exceeds it by more than 2^8 (exponentials
//                   stay <= 256), so O is rescaled in a few blocks rather than most, and
//                   the cross-lane maximum is only formed when some lane's own maximum
//                   would move it.
//   O^T += V^T P^T  D/16 feature tiles x 2 query tiles over two 32-key steps; P^T comes
//                   straight from the S^T registers (key tiles 2s and 2s + 1 give k-index
//                   0..3 and 4..7 of lane group l / 16), and V^T fragments are read with
//                   ds_read_b64_tr_b16 from row-major V rows in exactly that key order.
// Q fragments stay in registers for the whole key loop.
//
// Ping-pong: the barrier-separated phases alternate an MFMA phase M(j) (O^T += V_{j-1}^T
// P_{j-1}^T, then S^T_j) and a softmax phase V(j); the two waves of each SIMD (found from
// the hardware SIMD id) run opposite phases, so one wave's exponentials overlap the other's
// MFMAs. Each phase's register results are pinned before its barrier so the compiler
// cannot sink them into the next phase.
//
// K and V blocks reach LDS by buffer->LDS DMA (no VGPR staging) into a 4-stage ring; block
// j is read in phases 2j .. 2j+3 and its stage is refilled from phase 2j+4 on: each wave
// issues its share of block m + 2 spread over the read units of its MFMA phase of block m
// (issued as one burst after a barrier, the DMA instructions held the issuing waves ~300
// cycles per block; causal D128 1.91 -> 1.83 ms). LDS layouts keep every read phase on 64
// distinct banks:
//   K [64 keys][D]: 16-byte chunk c of row r at slot c ^ kswz(r) (ds_read_b128, 16 lanes
//                   per phase read one chunk of 16 rows);
//   V [64 keys][D]: 32-byte granule g of row r at granule g ^ vswz(r) (ds_read_b64_tr_b16,
//                   32 lanes per phase read one granule of 8 rows).
// The DMA writes 1 KiB contiguous per instruction, so the swizzle is applied on the global
// side (each lane fetches the chunk that belongs in its LDS slot). LDS reads are inline
// asm ordered by explicit waits: the compiler would otherwise wait for every outstanding
// DMA before each read.
#include "attention.hpp"
#include "attention_dma.hpp"

#include <cmath>
#include <type_traits>

namespace {

using namespace tk_attn;

constexpr int kThreads = 512;
constexpr float kLazyRescale = 8.f;

struct Shape {
  int heads, seq;  // seq: the sequence length (varlen: the longest sequence)
  int group;  // query heads per KV head: K/V of head h are those of KV head h / group
  // Variable-length batches (null for equal lengths): sequence b is the rows
  // cu[b] .. cu[b+1] of a packed [total][head][dim] layout (the batch strides are 0),
  // and the LSE is [head][total].
  const int32_t* cu;
  int total, batch;
  int64_t q[3], k[3], v[3], o[3];  // batch, head, sequence strides (elements)
  float scale_log2;
  int q_blocks, tiles;
  uint32_t k_bytes, v_bytes;  // per-head buffer extents
  // RoPE applied to Q in the prologue (null: none): position-indexed tables [pos][D/2]
  // of T with row stride rope_stride; query i uses row i.
  const void* rope_cos;
  const void* rope_sin;
  int64_t rope_stride;
};

// Arguments of the forward kernel, passed as its only parameter (read through kernel_args
// in its tile loop).
template <typename T>
struct FwdArgs {
  const T* Q;
  const T* K;
  const T* V;
  T* O;
  float* lse;
  Shape s;
};

// Rotate-half RoPE of one 16-byte Q fragment pair: x1 holds features f .. f+7 and x2
// features f + D/2 .. f + D/2 + 7 (f < D/2); c and s hold cos/sin of f .. f+7. The
// arithmetic is the RoPE kernel's: products rounded separately (no contraction), then
// each result rounded to T, so the rotated Q is bitwise the one tk_rope_fwd stores.
template <typename T>
__device__ __forceinline__ void rope_fragment(i32x4& x1, i32x4& x2, i32x4 c, i32x4 s) {
#pragma clang fp contract(off)
  typedef T t8 __attribute__((ext_vector_type(8)));
  const t8 a = __builtin_bit_cast(t8, x1), b = __builtin_bit_cast(t8, x2);
  const t8 cv = __builtin_bit_cast(t8, c), sv = __builtin_bit_cast(t8, s);
  t8 y1, y2;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float xa = static_cast<float>(a[e]), xb = static_cast<float>(b[e]);
    const float ce = static_cast<float>(cv[e]), se = static_cast<float>(sv[e]);
    y1[e] = tk::from_f32<T>(xa * ce - xb * se);
    y2[e] = tk::from_f32<T>(xb * ce + xa * se);
  }
  x1 = __builtin_bit_cast(i32x4, y1);
  x2 = __builtin_bit_cast(i32x4, y2);
}

template <int D>
struct Geo {
  static constexpr int BM = 256, BN = 64, WAVES = 8, QW = 32;
  static constexpr int KS = D / 32;             // k-steps of S^T (32 features each)
  static constexpr int KH = KS / 2;             // k-steps per half of the feature range
  static constexpr int FT = D / 16;             // 16-feature tiles of O^T
  static constexpr int RB = D * 2;              // bytes per K/V row
  static constexpr int OPB = BN * RB;           // bytes per operand per stage
  static constexpr int STB = 2 * OPB;           // stage: K tile then V tile
  static constexpr int STAGES = 4;
  static constexpr int ROWS_PER_DMA = 1024 / RB;
  static constexpr int DMA_PER_OP = OPB / 1024 / WAVES;  // per wave, per operand
  static constexpr int DMA_PER_BLOCK = 2 * DMA_PER_OP;
  static constexpr int SLOTS = RB / 16;         // 16-byte slots per row
  // K: 16-byte chunk c of row r at slot c ^ kswz(r). A read phase (16 lanes) takes one
  // chunk of 16 consecutive rows.
  static __device__ __forceinline__ int kswz(int r) { return D == 128 ? (r & 15) : ((r >> 1) & 7); }
  // V: 32-byte granule g of row r at granule g ^ vswz(r). A transposed read phase (32
  // lanes) takes one granule of 8 consecutive rows.
  static __device__ __forceinline__ int vswz(int r) { return D == 128 ? (r & 7) : ((r >> 1) & 3); }
  // O staging: 16-byte granule q of staged row r at q ^ oswz(r). An 8-byte write phase (16
  // rows x 2 lane groups) and a 16-byte read phase then fall on distinct banks.
  static __device__ __forceinline__ int oswz(int r) { return D == 128 ? (r & 15) : ((r >> 1) & 7); }
};

// DMA of key/value block `blk` into its ring stage (clamped to `last`: blocks past the end
// reload the last one into a stage that is never read, keeping the per-phase load count
// constant).
template <int D>
__device__ __forceinline__ void dma_block(__amdgpu_buffer_rsrc_t rk, __amdgpu_buffer_rsrc_t rv,
                                          char* lds, const uint32_t* k_src,
                                          const uint32_t* v_src, int blk, int last,
                                          uint32_t k_blk, uint32_t v_blk, int wave) {
  using G = Geo<D>;
  char* stage = lds + (blk % G::STAGES) * G::STB;
  blk = min(blk, last);
#pragma unroll
  for (int x = 0; x < G::DMA_PER_OP; ++x) {
    const int id = wave * G::DMA_PER_OP + x;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (lds_void*)(stage + id * 1024), 16, k_src[x],
                                             blk * k_blk, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (lds_void*)(stage + G::OPB + id * 1024), 16,
                                             v_src[x], blk * v_blk, 0, 0);
  }
}

// DMA instruction i (0 .. DMA_PER_BLOCK - 1) of this wave's share of block `blk`: K chunks
// first, then V.
template <int D>
__device__ __forceinline__ void dma_one(__amdgpu_buffer_rsrc_t rk, __amdgpu_buffer_rsrc_t rv,
                                        char* lds, const uint32_t* k_src, const uint32_t* v_src,
                                        int blk, int last, uint32_t k_blk, uint32_t v_blk,
                                        int wave, int i) {
  using G = Geo<D>;
  char* stage = lds + (blk % G::STAGES) * G::STB;
  blk = min(blk, last);
  const int x = i % G::DMA_PER_OP;
  const int id = wave * G::DMA_PER_OP + x;
  if (i < G::DMA_PER_OP)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (lds_void*)(stage + id * 1024), 16, k_src[x],
                                             blk * k_blk, 0, 0);
  else
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (lds_void*)(stage + G::OPB + id * 1024), 16,
                                             v_src[x], blk * v_blk, 0, 0);
}

// The MFMA phase as a pipeline of read units of four LDS instructions each: V units
// (u < NV) hold 32-key step s = u / (FT/2) of feature tiles 2p and 2p+1 (p = u % (FT/2)),
// K units (u >= NV) k-step kk = u - NV of the four key tiles. Unit u's MFMAs run while
// units u+1 .. u+DEPTH-1 are in flight.
template <int D>
struct Units {
  static constexpr int FP = Geo<D>::FT / 2;  // feature-tile pairs per 32-key step
  static constexpr int NV = 2 * FP;          // V units of a block
  // Units in flight, and V units issued at the end of the softmax phase (at most 15 LDS
  // reads may be in flight before a wave's issue stalls). head_dim 64 keeps fewer in
  // flight to stay within 128 registers.
  static constexpr int DEPTH = D == 64 ? 3 : 4;
  static constexpr int PREFETCH = D == 64 ? 2 : 3;
};

// Issues V unit u of the V tile at vb into vu[u].
template <int D>
__device__ __forceinline__ void read_v_unit(i32x4 (&vu)[Units<D>::NV][2], uint32_t vb,
                                            const uint32_t (&va)[Geo<D>::FT], int u) {
  constexpr int FP = Units<D>::FP, RB = Geo<D>::RB;
  const int s = u / FP, p = u % FP;
#pragma unroll
  for (int i = 0; i < 2; ++i)
    vu[u][i] = s == 0 ? read_v16<0, RB>(vb + va[2 * p + i]) : read_v16<32, RB>(vb + va[2 * p + i]);
}

// The MFMA phase of one wave: O^T += V_{j-1}^T P^T from the previous softmax phase's pf
// (DO_PV; P^T is dead before S^T is produced), then S^T(j) = K_j Q^T into st (DO_S).
// kb / vb: LDS addresses of the K tile of block j and the V tile of block j-1. With DO_PV
// the first PREFETCH V units were issued by the preceding softmax phase.
template <typename T, int D, bool DO_S, bool DO_PV, typename Hook>
__device__ __forceinline__ void mfma_phase(Hook&& hook, uint32_t kb, uint32_t vb, const uint32_t (&ka)[Geo<D>::KS],
                                           const uint32_t (&va)[Geo<D>::FT],
                                           const i32x4 (&qf)[2][Geo<D>::KS], f32x4 (&st)[2][4],
                                           const i32x4 (&pf)[2][2], f32x4 (&acc)[Geo<D>::FT][2],
                                           i32x4 (&vu)[Units<D>::NV][2]) {
  using G = Geo<D>;
  constexpr int KS = G::KS, RB = G::RB, FP = Units<D>::FP;
  constexpr int NV = DO_PV ? Units<D>::NV : 0, NU = NV + (DO_S ? KS : 0);
  constexpr int DEPTH = Units<D>::DEPTH;
  constexpr int PRE = DO_PV ? Units<D>::PREFETCH : 0;  // units issued before the phase
  static_assert(!DO_PV || Units<D>::NV >= PRE, "the prefetched units are V units");
  i32x4 kf[KS][4];
  auto issue = [&](int u) {
    if (u < NV) {
      read_v_unit<D>(vu, vb, va, u);
    } else {
      const int kk = u - NV;
      const uint32_t a = kb + ka[kk];
      kf[kk][0] = lds_read_b128<0>(a);
      kf[kk][1] = lds_read_b128<16 * RB>(a);
      kf[kk][2] = lds_read_b128<32 * RB>(a);
      kf[kk][3] = lds_read_b128<48 * RB>(a);
    }
  };
#pragma unroll
  for (int u = PRE; u < DEPTH && u < NU; ++u) issue(u);
  sched_fence();
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    // Units u+1 .. min(u+DEPTH, NU)-1 may still be in flight (four instructions each).
    const int after = (u + DEPTH < NU ? u + DEPTH : NU) - (u + 1);
    if (after >= 3)
      wait_lgkm<12>();
    else if (after == 2)
      wait_lgkm<8>();
    else if (after == 1)
      wait_lgkm<4>();
    else
      wait_lgkm<0>();
    if (u < NV) {
      const int s = u / FP, p = u % FP;
      pin(vu[u][0]);
      pin(vu[u][1]);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int qt = 0; qt < 2; ++qt)
          acc[2 * p + i][qt] = Mma16<T>::run(vu[u][i], pf[qt][s], acc[2 * p + i][qt]);
    } else {
      const int kk = u - NV;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) pin(kf[kk][kt]);
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int qt = 0; qt < 2; ++qt)
          st[qt][kt] = Mma16<T>::run(kf[kk][kt], qf[qt][kk],
                                     kk == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : st[qt][kt]);
    }
    if (u + DEPTH < NU) issue(u + DEPTH);
    hook(u, NU);
    sched_fence();
  }
}

// head_dim 64 uses 64 KiB of LDS per workgroup: held to 128 registers, two workgroups
// share a CU (four waves per SIMD).
// Equal lengths at head_dim 128: one workgroup per causal pair of query blocks
// (paired_tile). Not at head_dim 64: at 128 registers the two-block loop spills inside the
// key loop (causal B4 H32 N8192 1.22 -> 1.42 ms).
template <int D>
constexpr bool kPaired = D == 128;

template <typename T, int D, bool CAUSAL>
__global__ __attribute__((amdgpu_flat_work_group_size(kThreads, kThreads),
                          amdgpu_waves_per_eu(D == 64 ? 4 : 2))) void
attn_fwd_dma_kernel(FwdArgs<T> kernel_arg) {
  using G = Geo<D>;
  constexpr int BM = G::BM, BN = G::BN, KS = G::KS, FT = G::FT, RB = G::RB, OPB = G::OPB,
                STB = G::STB, STAGES = G::STAGES, DPB = G::DMA_PER_BLOCK;
  __shared__ __attribute__((aligned(1024))) char lds[STAGES * STB];
  // O staging: 16 rows of D values per wave (one query tile at a time), 32 KiB at head_dim
  // 128 and 16 KiB at 64, so the ring and the staging fill the CU's 160 KiB (one workgroup
  // at 128, two at 64). Until the first epilogue it holds each wave's SIMD id.
  __shared__ __attribute__((aligned(16))) char ostage[G::WAVES * 16 * RB];

  const int wave0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_void*)lds;
  // Ping-pong partner: the two waves that share a SIMD (hardware SIMD id from HW_ID) take
  // opposite phases; grp is the wave's rank (0 or 1) among them.
  int grp = 0;
  {
    int* simd_of = reinterpret_cast<int*>(ostage);
    if ((threadIdx.x & 63) == 0) simd_of[wave0] = simd_id();
    __syncthreads();
#pragma unroll
    for (int w = 0; w < G::WAVES; ++w)
      grp += (w < wave0 && simd_of[w] == simd_of[wave0]) ? 1 : 0;
    grp = __builtin_amdgcn_readfirstlane(grp) & 1;
  }

  // Causal, equal lengths, head_dim 128: the two query blocks paired_tile deals this
  // workgroup (blocks i and QB-1-i of one head). Otherwise one query block per workgroup;
  // varlen: the heavy-first schedule over every sequence's query blocks (level = query
  // block), heads interleaved over the XCDs.
  for (int it = 0; (kPaired<D> && CAUSAL) || it == 0; ++it) {
    const FwdArgs<T>& args = kernel_args<FwdArgs<T>>();
    const Shape& s = args.s;
    const T* __restrict__ Q = args.Q;
    const T* __restrict__ K = args.K;
    const T* __restrict__ V = args.V;
    int b, h, qb, start = 0, N = s.seq;
    uint32_t k_bytes = s.k_bytes, v_bytes = s.v_bytes;
    if (s.cu != nullptr) {
      if (it > 0) break;
      h = varlen_head(blockIdx.x, s.heads);
      VarlenTile vt;
      if (!varlen_tile(s.cu, s.batch, s.total, s.seq, BM, blockIdx.x / s.heads, vt)) break;
      b = vt.b;
      qb = vt.level;
      const VarlenRows rows = varlen_rows(s.cu, b, s.total, s.seq);
      start = rows.start;
      N = rows.n;
      if (qb * BM >= N) break;  // uniform: the whole workgroup leaves
      k_bytes = uint32_t(((N - 1) * s.k[2] + D) * 2);
      v_bytes = uint32_t(((N - 1) * s.v[2] + D) * 2);
    } else if constexpr (kPaired<D> && CAUSAL) {
      int bh, rank;
      if (!paired_tile(it, s.tiles / s.q_blocks, s.q_blocks, bh, rank)) break;
      qb = s.q_blocks - 1 - rank;
      b = bh / s.heads;
      h = bh % s.heads;
    } else {
      // One tile per workgroup: XCD-contiguous ranges so a head's blocks share one L2;
      // causal: the heaviest (last) query block of a head first.
      if (it > 0) break;
      int w = blockIdx.x;
      if (s.tiles % 8 == 0) w = (w % 8) * (s.tiles / 8) + w / 8;
      const int bh = w / s.q_blocks;
      qb = CAUSAL ? s.q_blocks - 1 - w % s.q_blocks : w % s.q_blocks;
      b = bh / s.heads;
      h = bh % s.heads;
    }
    // After the first tile: every wave has left the previous tile (its last LDS reads
    // are not followed by a barrier) before this tile's DMA refills the ring.
    if (it > 0) barrier_no_fence();
    // The lane and wave indices pass through an empty asm once per tile, so the addresses
    // derived from them are formed inside the tile rather than hoisted and held across the
    // loop.
    int lane = threadIdx.x & 63;
    int wave = wave0;
    if constexpr (kPaired<D> && CAUSAL) asm volatile("" : "+v"(lane), "+s"(wave));
    const int c = lane & 15, g = lane >> 4;
    const int kvh = h / s.group;
    const T* Qh = Q + b * s.q[0] + h * s.q[1] + int64_t(start) * s.q[2];
    const T* Kh = K + b * s.k[0] + kvh * s.k[1] + int64_t(start) * s.k[2];
    const T* Vh = V + b * s.v[0] + kvh * s.v[1] + int64_t(start) * s.v[2];

    const int q0 = qb * BM;
    const int wq0 = q0 + wave * G::QW;

    const __amdgpu_buffer_rsrc_t rk =
        __builtin_amdgcn_make_buffer_rsrc((void*)Kh, (short)0, k_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv =
        __builtin_amdgcn_make_buffer_rsrc((void*)Vh, (short)0, v_bytes, 0x00020000);

    // DMA sources (bytes from the head's base, block-relative row). Rows past the sequence
    // end are past the buffer extent and read as zero: the range check is on voffset plus
    // soffset, which carries the block's offset.
    uint32_t k_src[G::DMA_PER_OP], v_src[G::DMA_PER_OP];
#pragma unroll
    for (int x = 0; x < G::DMA_PER_OP; ++x) {
      const int id = wave * G::DMA_PER_OP + x;
      const int row = id * G::ROWS_PER_DMA + lane / G::SLOTS;
      const int slot = lane % G::SLOTS;
      k_src[x] = uint32_t(row * s.k[2] + (slot ^ G::kswz(row)) * 8) * 2u;
      const int granule = (slot >> 1) ^ G::vswz(row);
      v_src[x] = uint32_t(row * s.v[2] + granule * 16 + (slot & 1) * 8) * 2u;
    }
    const int kv_end = CAUSAL ? min(N, q0 + BM) : N;
    const int kv_blocks = (kv_end + BN - 1) / BN;
    const int last = kv_blocks - 1;
    const uint32_t k_blk = uint32_t(BN * s.k[2]) * 2u, v_blk = uint32_t(BN * s.v[2]) * 2u;
    // The first STAGES - 1 blocks are fetched before anything else.
#pragma unroll
    for (int blk = 0; blk < STAGES - 1; ++blk)
      dma_block<D>(rk, rv, lds, k_src, v_src, blk, last, k_blk, v_blk, wave);

    // Q fragments (B operand of S^T): query tile qt holds query wq0 + 16 qt + c, k-step kk
    // features 32 kk + 8 g .. +7.
    i32x4 qf[2][KS];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      const int query = wq0 + 16 * qt + c;
#pragma unroll
      for (int kk = 0; kk < KS; ++kk)
        qf[qt][kk] = query < N
                         ? *reinterpret_cast<const i32x4*>(Qh + query * s.q[2] + kk * 32 + g * 8)
                         : i32x4{0, 0, 0, 0};
    }
    // RoPE: fragments kk and kk + KS/2 hold features 32 kk + 8 g .. +7 and the same + D/2,
    // so the rotate-half pairs sit in one lane. Queries past the end keep zero tables (their
    // Q is 0).
    if (s.rope_cos != nullptr) {
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        const int query = wq0 + 16 * qt + c;
        const int64_t at = int64_t(query) * s.rope_stride + g * 8;
        const T* cr = static_cast<const T*>(s.rope_cos) + at;
        const T* sr = static_cast<const T*>(s.rope_sin) + at;
#pragma unroll
        for (int kk = 0; kk < KS / 2; ++kk) {
          const i32x4 cv = query < N ? *reinterpret_cast<const i32x4*>(cr + kk * 32) : i32x4{0, 0, 0, 0};
          const i32x4 sv = query < N ? *reinterpret_cast<const i32x4*>(sr + kk * 32) : i32x4{0, 0, 0, 0};
          rope_fragment<T>(qf[qt][kk], qf[qt][kk + KS / 2], cv, sv);
        }
      }
    }
    // Lane read addresses inside a stage: K row c of key tile kt (+16 kt rows), chunk
    // 4 kk + g; V rows 4 g + j (+32 per key step, +16 for k-index 4..7), features
    // 16 ft + 4 q .. +3, with j = c / 4, q = c % 4.
    uint32_t ka[KS], va[FT];
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) ka[kk] = c * RB + (((4 * kk + g) ^ G::kswz(c)) * 16);
    {
      const int row = 4 * g + (c >> 2), q = c & 3;
#pragma unroll
      for (int ft = 0; ft < FT; ++ft) va[ft] = OPB + row * RB + ((ft ^ G::vswz(row)) * 32) + q * 8;
    }

    // O^T accumulators: acc[ft][qt] register r is feature 16 ft + 4 g + r of query
    // wq0 + 16 qt + c. st[qt][kt] register r: score of key n0 + 16 kt + 4 g + r.
    f32x4 acc[FT][2], st[2][4];
    i32x4 pf[2][2], vu[Units<D>::NV][2];
#pragma unroll
    for (int ft = 0; ft < FT; ++ft)
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) acc[ft][qt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run[2] = {kNegInf, kNegInf}, l_part[2] = {0.f, 0.f};
    const float sl2 = s.scale_log2;

    // Block 0 landed.
    wait_lgkm<0>();
    wait_vmcnt<(STAGES - 2) * DPB>();
    barrier_no_fence();
    // Ping-pong: the two waves that share a SIMD take opposite phases. The workgroup runs
    // phases t = 0, 1, ... separated by barriers; a wave alternates an MFMA phase M(j)
    // (S^T of block j, O^T += V^T P^T of block j-1) and a softmax phase V(j), the second
    // wave of each SIMD one phase behind the first, so one wave's exponentials run while
    // the other's MFMAs occupy the matrix pipe. Block j is read in phases 2j .. 2j+3; at
    // the start of phase 2m (m >= 1) its stage's next block m + STAGES - 2 is fetched,
    // and block m must have landed before phase 2m begins.
    const int phases = 2 * kv_blocks + 2;
    int t = 0;
    // Block m + STAGES - 2 (m >= 1) is fetched during this wave's MFMA phase of block m
    // (phase 2m + grp), its DMA_PER_BLOCK instructions spread over the phase's read units;
    // after the wave's last MFMA phase, at the start of phase 2m + grp (tail mode). Block m+1
    // was issued by every wave before the end of phase 2m + 1 (grp 0 in phase 2m - 2, grp 1
    // in 2m - 1), so the wait at the end of each odd phase, which leaves one block's
    // instructions in flight, still covers it.
    bool tail = false;
    int tail_m = 0;
    auto end_phase = [&]() {
      if (t & 1) wait_vmcnt<(STAGES - 3) * DPB>();
      barrier_no_fence();
      ++t;
      if (tail && tail_m <= kv_blocks && t == 2 * tail_m + grp) {
        dma_block<D>(rk, rv, lds, k_src, v_src, tail_m + STAGES - 2, last, k_blk, v_blk, wave);
        ++tail_m;
      }
    };
    // Hook of the MFMA phase of block m: after unit u of nu, the DMA instructions whose
    // share of the phase ends there (DMA_PER_BLOCK of them over the nu units).
    auto dma_hook = [&](int m) {
      return [&, m](int u, int nu) {
        const int a = (u * DPB) / nu, b2 = ((u + 1) * DPB) / nu;
        if (b2 != a)
          dma_one<D>(rk, rv, lds, k_src, v_src, m + STAGES - 2, last, k_blk, v_blk, wave, b2 - 1);
      };
    };
    auto no_hook = [](int, int) {};
    auto kbase = [&](int j) { return lds_base + (j % STAGES) * STB; };

    // Softmax phase of block j: P = exp2(S * scale * log2(e) - m) into pf, the running
    // statistics updated. The reference maximum m_run only moves when the block's maximum
    // exceeds it by more than kLazyRescale (log2 units): exponentials stay
    // <= 2^kLazyRescale, and O and l are rescaled in few blocks instead of whenever one of
    // the wave's 32 maxima grows. O = acc / l and the log-sum-exp m_run + log2(l) do not
    // depend on which reference is used.
    auto softmax_phase = [&](int j) {
      const int n0 = j * BN;
      const bool need_mask = n0 + BN > N || (CAUSAL && n0 + BN - 1 > wq0);
      if (__builtin_expect(need_mask, 0)) {
#pragma unroll
        for (int qt = 0; qt < 2; ++qt)
#pragma unroll
          for (int kt = 0; kt < 4; ++kt) {
            const int k0 = n0 + 16 * kt + 4 * g;  // the lane's first key of this tile
            int lim = N - 1 - k0;                 // last valid offset from k0
            if (CAUSAL) lim = min(lim, wq0 + 16 * qt + c - k0);
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (r > lim) st[qt][kt][r] = kNegInf;
          }
      }
      if constexpr (D == 128) {
        // Exponentials against the current reference first. A lane whose 16 exponentials of a
        // query sum to at most 2^kLazyRescale has none above it, so when no lane of the wave
        // exceeds that sum no reference moves and no maximum is needed. Otherwise the column
        // maxima are formed from the scores, which are still intact, and the queries whose
        // reference moves are recomputed.
        f32x4 p[2][4];
        float sum[2];
        auto exps = [&](int qt) {
          const float neg = -m_run[qt];
    #pragma unroll
          for (int kt = 0; kt < 4; ++kt)
    #pragma unroll
            for (int r = 0; r < 4; ++r)
              p[qt][kt][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(st[qt][kt][r], sl2, neg));
          float s0 = p[qt][0][0];
    #pragma unroll
          for (int i = 1; i < 16; ++i) s0 += p[qt][i / 4][i % 4];
          sum[qt] = s0;
        };
        exps(0);
        exps(1);
        constexpr float kLazyLimit = 256.f;  // 2^kLazyRescale
        if (__builtin_expect(
                __builtin_amdgcn_ballot_w64(!(sum[0] <= kLazyLimit) || !(sum[1] <= kLazyLimit)) != 0,
                0)) {
    #pragma unroll
          for (int qt = 0; qt < 2; ++qt) {
            float mx = kNegInf;
    #pragma unroll
            for (int kt = 0; kt < 4; ++kt)
    #pragma unroll
              for (int r = 0; r < 4; ++r) mx = fmaxf(mx, st[qt][kt][r]);
            const float bm = max_over_column(mx) * sl2;
            const bool move = bm > m_run[qt] + kLazyRescale;
            if (__builtin_amdgcn_ballot_w64(move)) {
              const float m_new = move ? bm : m_run[qt];
              const float alpha = move ? __builtin_amdgcn_exp2f(m_run[qt] - m_new) : 1.f;
              l_part[qt] *= alpha;
    #pragma unroll
              for (int ft = 0; ft < FT; ++ft) acc[ft][qt] *= alpha;
              m_run[qt] = m_new;
              exps(qt);
            }
          }
        }
    #pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
          l_part[qt] += sum[qt];
          pf[qt][0] = acc_frag2<T>(p[qt][0], p[qt][1]);
          pf[qt][1] = acc_frag2<T>(p[qt][2], p[qt][3]);
        }
      } else {
        // head_dim 64 (128 registers): the exponentials overwrite the scores, so the maximum
        // comes first. A column's maximum exceeds the threshold only if one of its four
        // lanes' does: the cross-lane reduction runs only when some lane of the wave sees
        // such a maximum.
        float mx[2], m_new[2];
        bool move[2];
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
          mx[qt] = kNegInf;
#pragma unroll
          for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) mx[qt] = fmaxf(mx[qt], st[qt][kt][r]);
          move[qt] = mx[qt] * sl2 > m_run[qt] + kLazyRescale;
          m_new[qt] = m_run[qt];
        }
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(move[0] || move[1]) != 0, 0)) {
#pragma unroll
          for (int qt = 0; qt < 2; ++qt) {
            const float bm = max_over_column(mx[qt]) * sl2;
            move[qt] = bm > m_run[qt] + kLazyRescale;
            m_new[qt] = move[qt] ? bm : m_run[qt];
          }
        }
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
          const float neg = -m_new[qt];
          float sum = 0.f;
#pragma unroll
          for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(st[qt][kt][r], sl2, neg));
              st[qt][kt][r] = pv;
              sum += pv;
            }
          if (__builtin_amdgcn_ballot_w64(move[qt])) {
            const float alpha = move[qt] ? __builtin_amdgcn_exp2f(m_run[qt] - m_new[qt]) : 1.f;
            l_part[qt] *= alpha;
#pragma unroll
            for (int ft = 0; ft < FT; ++ft) acc[ft][qt] *= alpha;
          }
          l_part[qt] += sum;
          m_run[qt] = m_new[qt];
          pf[qt][0] = acc_frag2<T>(st[qt][0], st[qt][1]);
          pf[qt][1] = acc_frag2<T>(st[qt][2], st[qt][3]);
        }
      }
    };

    // This wave multiplies a prefix of the workgroup's blocks (causal: those starting at or
    // before its last query); every wave takes part in every phase's barrier and loads.
    const int n = CAUSAL ? min(kv_blocks, (wq0 + G::QW - 1) / BN + 1) : kv_blocks;
    // The loop is entered after M(0) and leaves before V(n-1) (with the softmax phase first
    // in the body the compiler keeps one copy of the O accumulators across the back edge).
    // A phase's results are pinned before its closing barrier: the barrier orders memory
    // only, and the compiler would otherwise sink register work (the exponentials, the
    // MFMA chains) into the next phase, where it runs beside the partner wave's same kind
    // of work.
    auto pin_mfma = [&]() {
#pragma unroll
      for (int qt = 0; qt < 2; ++qt)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) pin(st[qt][kt]);
#pragma unroll
      for (int ft = 0; ft < FT; ++ft)
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) pin(acc[ft][qt]);
    };
    // The softmax phase ends by issuing the first PREFETCH V units of the next MFMA phase
    // (block j's V tile has landed since phase 2j).
    auto pin_softmax = [&](int j) {
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        pin(pf[qt][0]);
        pin(pf[qt][1]);
        asm volatile("" : "+v"(l_part[qt]), "+v"(m_run[qt]));
      }
#pragma unroll
      for (int u = 0; u < Units<D>::PREFETCH; ++u) read_v_unit<D>(vu, kbase(j), va, u);
    };
    if (grp) end_phase();
    mfma_phase<T, D, true, false>(no_hook, kbase(0), 0, ka, va, qf, st, pf, acc, vu);
    pin_mfma();
    end_phase();
    for (int j = 1; j < n; ++j) {
      softmax_phase(j - 1);
      pin_softmax(j - 1);
      end_phase();
      mfma_phase<T, D, true, true>(dma_hook(j), kbase(j), kbase(j - 1), ka, va, qf, st, pf, acc, vu);
      pin_mfma();
      end_phase();
    }
    softmax_phase(n - 1);
    pin_softmax(n - 1);
    end_phase();
    mfma_phase<T, D, false, true>(dma_hook(n), 0, kbase(n - 1), ka, va, qf, st, pf, acc, vu);
    tail = true;
    tail_m = n + 1;
    while (t < phases - 1) end_phase();
    // No DMA may still be writing when the workgroup's LDS is released.
    wait_vmcnt<0>();

    // O = O^T / l: acc[ft][qt] register r is feature 16 ft + 4 g + r of query
    // wq0 + 16 qt + c, 8 bytes once rounded. Each query tile goes through the wave's own
    // staging rows and leaves as whole rows, 16 bytes per lane and full 128-byte lines, with
    // non-temporal stores (the per-lane 8-byte stores wrote 32-byte pieces of lines); the
    // entry points accept only 16-byte aligned tensors and strides that are multiples of 8
    // elements, so every O row is 16-byte aligned. The staging rows belong to one wave: no
    // barrier. The output pointer, strides and lane indices are formed here afresh rather
    // than held across the key loop (at head_dim 64 that spilled registers).
    const FwdArgs<T>& ea = kernel_args<FwdArgs<T>>();
    int el = threadIdx.x & 63;
    asm volatile("" : "+v"(el));
    const int ec = el & 15, eg = el >> 4;
    const int64_t o_row = ea.s.o[2];
    T* const Oe = ea.O + b * ea.s.o[0] + h * ea.s.o[1] + int64_t(start) * o_row;
    char* const orows = ostage + wave * (16 * RB);
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      const float l = sum_over_column(l_part[qt]);
      const float inv = 1.0f / l;
#pragma unroll
      for (int ft = 0; ft < FT; ++ft) {
        uint2 u;
        u.x = pack2<T>(acc[ft][qt][0] * inv, acc[ft][qt][1] * inv);
        u.y = pack2<T>(acc[ft][qt][2] * inv, acc[ft][qt][3] * inv);
        *reinterpret_cast<uint2*>(orows + ec * RB + (((2 * ft + (eg >> 1)) ^ G::oswz(ec)) * 16) +
                                  (eg & 1) * 8) = u;
      }
      constexpr int LPR = RB / 16, RPI = 64 / LPR;  // lanes per row, rows per instruction
#pragma unroll
      for (int p = 0; p < 16 / RPI; ++p) {
        const int r = p * RPI + el / LPR, q = el % LPR;
        const i32x4 v = *reinterpret_cast<const i32x4*>(orows + r * RB + ((q ^ G::oswz(r)) * 16));
        const int row_query = wq0 + 16 * qt + r;
        if (row_query < N)
          __builtin_nontemporal_store(v, reinterpret_cast<i32x4*>(Oe + row_query * o_row + q * 8));
      }
      const int query = wq0 + 16 * qt + ec;
      if (query < N && ea.lse != nullptr && eg == 0) {
        const int64_t at = ea.s.cu != nullptr ? int64_t(h) * ea.s.total + start + query
                                              : (int64_t(b) * ea.s.heads + h) * N + query;
        ea.lse[at] = m_run[qt] + __log2f(l);
      }
    }
  }  // tiles
}

// ------------------------------------------------------------------ small workgroups
//
// The same forward for problems whose 256-query workgroups leave CUs idle, where the time is one
// workgroup's serial walk over its key blocks: a block costs a wave its MFMAs plus its
// exponentials, one after the other. Here a wave owns 16 QT queries (QT 1 or 2) and a workgroup
// has four waves, several workgroups per CU. QT = 1: four times as many workgroups walk
// blocks half as long; twice the LDS reads per MFMA make it the slower kernel once the chip is
// full. QT = 2 reads as much per MFMA as the 256-query kernel; workgroups that are not in step
// with each other take the place of its ping-pong, and their prologues and epilogues overlap,
// which pays wherever workgroups are short (ragged batches, causal head_dim 64). Each wave
// reads K, forms S, takes its softmax while the V fragments of the block's first half arrive,
// and multiplies.
//
// Every query sees the same operations in the same order as in the 256-query kernel, so the
// results are bitwise the same.
template <int D, int QT>
struct SmallGeo {
  using G = Geo<D>;
  static constexpr int QW = 16 * QT;  // queries per wave
  static constexpr int BM = 4 * QW, WAVES = 4, THREADS = 256;
  // 48 KiB at head_dim 64 (three workgroups per CU; four stages and two workgroups ran causal
  // H32 N2048 in 31.8 us against 29.2), 64 KiB at 128 (two).
  static constexpr int STAGES = D == 64 ? 3 : 2;
  static constexpr int DMA_PER_OP = G::OPB / 1024 / WAVES;
  static constexpr int DPB = 2 * DMA_PER_OP;
};

// A wave's share of the DMA of one key/value block, into its part `at` of the stage.
template <int D>
__device__ __forceinline__ void small_dma(__amdgpu_buffer_rsrc_t rk, __amdgpu_buffer_rsrc_t rv,
                                          char* at, const uint32_t* k_src, const uint32_t* v_src,
                                          uint32_t k_off, uint32_t v_off) {
#pragma unroll
  for (int x = 0; x < SmallGeo<D, 1>::DMA_PER_OP; ++x) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (lds_void*)(at + x * 1024), 16, k_src[x], k_off,
                                             0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (lds_void*)(at + Geo<D>::OPB + x * 1024), 16,
                                             v_src[x], v_off, 0, 0);
  }
}

template <typename T, int D, int QT, bool CAUSAL>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(D == 64 ? 3 : 2))) void
attn_fwd_small_kernel(FwdArgs<T> args) {
  using G = Geo<D>;
  using S = SmallGeo<D, QT>;
  constexpr int BN = G::BN, KS = G::KS, FT = G::FT, RB = G::RB, OPB = G::OPB, STB = G::STB,
                STAGES = S::STAGES;
  __shared__ __attribute__((aligned(1024))) char lds[STAGES * STB];
  const Shape& s = args.s;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_void*)lds;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;

  // Tiles: heaviest (last) query blocks first over all heads; with heads a multiple of 8 each
  // XCD keeps its own heads. Varlen: the heavy-first schedule over every sequence's blocks.
  int b, h, qb, start = 0, N = s.seq;
  uint32_t k_bytes = s.k_bytes, v_bytes = s.v_bytes;
  if (s.cu != nullptr) {
    h = varlen_head(blockIdx.x, s.heads);
    VarlenTile vt;
    if (!varlen_tile(s.cu, s.batch, s.total, s.seq, S::BM, blockIdx.x / s.heads, vt)) return;
    b = vt.b;
    qb = vt.level;
    const VarlenRows rows = varlen_rows(s.cu, b, s.total, s.seq);
    start = rows.start;
    N = rows.n;
    if (qb * S::BM >= N) return;
    k_bytes = uint32_t(((N - 1) * s.k[2] + D) * 2);
    v_bytes = uint32_t(((N - 1) * s.v[2] + D) * 2);
  } else {
    const int heads = s.tiles / s.q_blocks;
    int bh, rank;
    if (heads % 8 == 0) {
      const int per = heads / 8, i = blockIdx.x / 8;
      bh = (blockIdx.x % 8) * per + i % per;
      rank = i / per;
    } else {
      bh = blockIdx.x % heads;
      rank = blockIdx.x / heads;
    }
    qb = s.q_blocks - 1 - rank;
    b = bh / s.heads;
    h = bh % s.heads;
  }
  const int kvh = h / s.group;
  const T* Qh = args.Q + b * s.q[0] + h * s.q[1] + int64_t(start) * s.q[2];
  const T* Kh = args.K + b * s.k[0] + kvh * s.k[1] + int64_t(start) * s.k[2];
  const T* Vh = args.V + b * s.v[0] + kvh * s.v[1] + int64_t(start) * s.v[2];
  const int q0 = qb * S::BM;
  const int wq0 = q0 + wave * S::QW;
  const __amdgpu_buffer_rsrc_t rk =
      __builtin_amdgcn_make_buffer_rsrc((void*)Kh, (short)0, k_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rv =
      __builtin_amdgcn_make_buffer_rsrc((void*)Vh, (short)0, v_bytes, 0x00020000);
  uint32_t k_src[S::DMA_PER_OP], v_src[S::DMA_PER_OP];
#pragma unroll
  for (int x = 0; x < S::DMA_PER_OP; ++x) {
    const int row = (wave * S::DMA_PER_OP + x) * G::ROWS_PER_DMA + lane / G::SLOTS;
    const int slot = lane % G::SLOTS;
    k_src[x] = uint32_t(row * s.k[2] + (slot ^ G::kswz(row)) * 8) * 2u;
    v_src[x] = uint32_t(row * s.v[2] + ((slot >> 1) ^ G::vswz(row)) * 16 + (slot & 1) * 8) * 2u;
  }
  const int kv_end = CAUSAL ? min(N, q0 + S::BM) : N;
  const int blocks = (kv_end + BN - 1) / BN;
  const uint32_t k_blk = uint32_t(BN * s.k[2]) * 2u, v_blk = uint32_t(BN * s.v[2]) * 2u;
  // Rows past the sequence end read as zero, as in the 256-query kernel. Blocks past the end reload the last one into a stage that is never read.
  auto load = [&](int blk, int stage) {
    blk = min(blk, blocks - 1);
    small_dma<D>(rk, rv, lds + stage * STB + wave * S::DMA_PER_OP * 1024, k_src, v_src,
                 blk * k_blk, blk * v_blk);
  };
#pragma unroll
  for (int blk = 0; blk < STAGES - 1; ++blk) load(blk, blk);

  // Q fragments, rotated if asked, as in the 256-query kernel.
  i32x4 qf[QT][KS];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int query = wq0 + 16 * qt + c;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk)
      qf[qt][kk] = query < N
                       ? *reinterpret_cast<const i32x4*>(Qh + query * s.q[2] + kk * 32 + g * 8)
                       : i32x4{0, 0, 0, 0};
    if (s.rope_cos != nullptr) {
      const int64_t at = int64_t(query) * s.rope_stride + g * 8;
      const T* cr = static_cast<const T*>(s.rope_cos) + at;
      const T* sr = static_cast<const T*>(s.rope_sin) + at;
#pragma unroll
      for (int kk = 0; kk < KS / 2; ++kk) {
        const i32x4 cv = query < N ? *reinterpret_cast<const i32x4*>(cr + kk * 32) : i32x4{0, 0, 0, 0};
        const i32x4 sv = query < N ? *reinterpret_cast<const i32x4*>(sr + kk * 32) : i32x4{0, 0, 0, 0};
        rope_fragment<T>(qf[qt][kk], qf[qt][kk + KS / 2], cv, sv);
      }
    }
  }
  uint32_t ka[KS], va[FT];
#pragma unroll
  for (int kk = 0; kk < KS; ++kk) ka[kk] = c * RB + (((4 * kk + g) ^ G::kswz(c)) * 16);
  {
    const int row = 4 * g + (c >> 2), q = c & 3;
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) va[ft] = OPB + row * RB + ((ft ^ G::vswz(row)) * 32) + q * 8;
  }

  f32x4 acc[FT][QT];
#pragma unroll
  for (int ft = 0; ft < FT; ++ft)
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) acc[ft][qt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run[QT], l_part[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    m_run[qt] = kNegInf;
    l_part[qt] = 0.f;
  }
  const float sl2 = s.scale_log2;
  int stage = 0, fill = STAGES - 1;
  // Blocks this wave needs (causal: those that start at or before its last query).
  const int mine = CAUSAL && QT > 1 ? min(blocks, (wq0 + S::QW - 1) / BN + 1) : blocks;
  for (int j = 0; j < mine; ++j) {
    // Block j has landed in every wave's share, and every wave has read block j - 1, whose stage
    // takes block j + STAGES - 1.
    wait_vmcnt<(STAGES - 2) * S::DPB>();
    barrier_no_fence();
    const uint32_t base = lds_base + stage * STB;
    i32x4 kf[KS][4];
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      kf[kk][0] = lds_read_b128<0>(base + ka[kk]);
      kf[kk][1] = lds_read_b128<16 * RB>(base + ka[kk]);
      kf[kk][2] = lds_read_b128<32 * RB>(base + ka[kk]);
      kf[kk][3] = lds_read_b128<48 * RB>(base + ka[kk]);
    }
    load(j + STAGES - 1, fill);
    f32x4 st[QT][4];
    auto score = [&](auto step) {
      constexpr int kk = decltype(step)::value;
      wait_lgkm<4 * (KS - 1 - kk) < 15 ? 4 * (KS - 1 - kk) : 15>();
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) pin(kf[kk][kt]);
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
          st[qt][kt] = Mma16<T>::run(kf[kk][kt], qf[qt][kk],
                                     kk == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : st[qt][kt]);
    };
    score(std::integral_constant<int, 0>{});
    score(std::integral_constant<int, 1>{});
    if constexpr (KS == 4) {
      score(std::integral_constant<int, 2>{});
      score(std::integral_constant<int, 3>{});
    }
    // The first 32 keys' V fragments arrive during the softmax.
    i32x4 v0[FT], v1[FT];
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) v0[ft] = read_v16<0, RB>(base + va[ft]);

    const int n0 = j * BN;
    if (n0 + BN > N || (CAUSAL && n0 + BN - 1 > wq0)) {
#pragma unroll
      for (int qt = 0; qt < QT; ++qt)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
          const int k0 = n0 + 16 * kt + 4 * g;
          int lim = N - 1 - k0;
          if (CAUSAL) lim = min(lim, wq0 + 16 * qt + c - k0);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (r > lim) st[qt][kt][r] = kNegInf;
        }
    }
    i32x4 pf[QT][2];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      if constexpr (D == 128) {
        f32x4 p[4];
        float sum;
        auto exps = [&]() {
#pragma unroll
          for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              p[kt][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(st[qt][kt][r], sl2, -m_run[qt]));
          sum = p[0][0];
#pragma unroll
          for (int i = 1; i < 16; ++i) sum += p[i / 4][i % 4];
        };
        exps();
        constexpr float kLazyLimit = 256.f;  // 2^kLazyRescale
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(sum <= kLazyLimit)) != 0, 0)) {
          float mx = kNegInf;
#pragma unroll
          for (int i = 0; i < 16; ++i) mx = fmaxf(mx, st[qt][i / 4][i % 4]);
          const float bm = max_over_column(mx) * sl2;
          const bool move = bm > m_run[qt] + kLazyRescale;
          if (__builtin_amdgcn_ballot_w64(move)) {
            const float m_new = move ? bm : m_run[qt];
            const float alpha = move ? __builtin_amdgcn_exp2f(m_run[qt] - m_new) : 1.f;
            l_part[qt] *= alpha;
#pragma unroll
            for (int ft = 0; ft < FT; ++ft) acc[ft][qt] *= alpha;
            m_run[qt] = m_new;
            exps();
          }
        }
        l_part[qt] += sum;
        pf[qt][0] = acc_frag2<T>(p[0], p[1]);
        pf[qt][1] = acc_frag2<T>(p[2], p[3]);
      } else {
        float mx = kNegInf;
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, st[qt][i / 4][i % 4]);
        bool move = mx * sl2 > m_run[qt] + kLazyRescale;
        float m_new = m_run[qt];
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(move) != 0, 0)) {
          const float bm = max_over_column(mx) * sl2;
          move = bm > m_run[qt] + kLazyRescale;
          m_new = move ? bm : m_run[qt];
        }
        float sum = 0.f;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(st[qt][kt][r], sl2, -m_new));
            st[qt][kt][r] = pv;
            sum += pv;
          }
        if (__builtin_amdgcn_ballot_w64(move)) {
          const float alpha = move ? __builtin_amdgcn_exp2f(m_run[qt] - m_new) : 1.f;
          l_part[qt] *= alpha;
#pragma unroll
          for (int ft = 0; ft < FT; ++ft) acc[ft][qt] *= alpha;
        }
        l_part[qt] += sum;
        m_run[qt] = m_new;
        pf[qt][0] = acc_frag2<T>(st[qt][0], st[qt][1]);
        pf[qt][1] = acc_frag2<T>(st[qt][2], st[qt][3]);
      }
    }
    wait_lgkm<0>();
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) pin(v0[ft]);
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) v1[ft] = read_v16<32, RB>(base + va[ft]);
#pragma unroll
    for (int ft = 0; ft < FT; ++ft)
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) acc[ft][qt] = Mma16<T>::run(v0[ft], pf[qt][0], acc[ft][qt]);
    wait_lgkm<0>();
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) pin(v1[ft]);
#pragma unroll
    for (int ft = 0; ft < FT; ++ft)
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) acc[ft][qt] = Mma16<T>::run(v1[ft], pf[qt][1], acc[ft][qt]);
    fill = stage;
    stage = stage == STAGES - 1 ? 0 : stage + 1;
  }
  // The barriers and loads of the blocks that only later waves need.
  for (int j = mine; j < blocks; ++j) {
    wait_vmcnt<(STAGES - 2) * S::DPB>();
    barrier_no_fence();
    load(j + STAGES - 1, fill);
    fill = stage;
    stage = stage == STAGES - 1 ? 0 : stage + 1;
  }
  // No DMA may still write the ring, which stages the O rows (16 per wave) now.
  wait_vmcnt<0>();
  __syncthreads();

  char* const orows = lds + wave * (16 * RB);
  T* const Oh = args.O + b * s.o[0] + h * s.o[1] + int64_t(start) * s.o[2];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const float l = sum_over_column(l_part[qt]);
    const float inv = 1.0f / l;
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) {
      uint2 u;
      u.x = pack2<T>(acc[ft][qt][0] * inv, acc[ft][qt][1] * inv);
      u.y = pack2<T>(acc[ft][qt][2] * inv, acc[ft][qt][3] * inv);
      *reinterpret_cast<uint2*>(orows + c * RB + (((2 * ft + (g >> 1)) ^ G::oswz(c)) * 16) +
                                (g & 1) * 8) = u;
    }
    constexpr int LPR = RB / 16, RPI = 64 / LPR;  // lanes per row, rows per instruction
#pragma unroll
    for (int p = 0; p < 16 / RPI; ++p) {
      const int r = p * RPI + lane / LPR, q = lane % LPR;
      const i32x4 v = *reinterpret_cast<const i32x4*>(orows + r * RB + ((q ^ G::oswz(r)) * 16));
      const int row_query = wq0 + 16 * qt + r;
      if (row_query < N)
        __builtin_nontemporal_store(v, reinterpret_cast<i32x4*>(Oh + row_query * s.o[2] + q * 8));
    }
    const int query = wq0 + 16 * qt + c;
    if (query < N && args.lse != nullptr && g == 0) {
      const int64_t at = s.cu != nullptr ? int64_t(h) * s.total + start + query
                                         : (int64_t(b) * s.heads + h) * N + query;
      args.lse[at] = m_run[qt] + __log2f(l);
    }
  }
}

// Workgroups of `rows` queries a launch has (`total` > 0: a packed batch, where the lengths are on
// the device and this is an upper bound).
int64_t fwd_tiles(int64_t batch, int64_t heads, int64_t seq, int64_t total, int64_t rows) {
  return (total > 0 ? varlen_tiles(batch, total, seq, rows) : batch * tk::cdiv(seq, rows)) * heads;
}

// Queries that tiles of `rows` queries hold for a sequence of a packed batch: exactly where all have
// one length, half a tile of padding on the mean length otherwise (the lengths are on the device).
double packed_queries(int64_t batch, int64_t seq, int64_t total, int64_t rows) {
  return total == batch * seq ? double(rows * tk::cdiv(seq, rows))
                              : double(total) / double(batch) + double(rows) / 2;
}

// What 256-query tiles cost a packed batch over 128-query ones: (query, key) pairs of the whole
// blocks a sequence needs (causal: up to each tile's last query).
double packed_cost_of_256(int64_t batch, int64_t seq, int64_t total, bool causal) {
  auto cost = [&](int64_t rows) {
    const double queries = packed_queries(batch, seq, total, rows);
    return causal ? queries * (queries + double(rows)) : queries;
  };
  return cost(256) / cost(128);
}

// Rounds of one 256-query workgroup per CU that a packed batch takes, over the rounds it fills.
double packed_idle_of_256(int64_t batch, int64_t heads, int64_t seq, int64_t total) {
  const double rounds = double(batch * heads) * packed_queries(batch, seq, total, 256) / (256.0 * 256.0);
  return rounds > 1 ? std::ceil(rounds) / rounds : 1.0;
}

// Query tiles per wave of the small-workgroup kernel, or 0 for the 256-query kernel. A problem
// has `tiles` 64-query tiles. 256-query / QT 1 / QT 2 in us, bf16, one sequence of N for H heads:
//   causal D64:  H16 N1024 (256 tiles) 23.2/11.6/16.6, H16 N4096 (1024) 75/49/55,
//                H16 N8192 (2048) 245/173/158, H64 N8192 (8192) 635/700/587,
//                H128 N8192 (16384) 1176/-/1211
//   causal D128: H32 N1024 (512) 39.6/17.3/22.0, H8 N8192 (1024) 180/167/158,
//                H256 N512 (2048) 39.9/39.8/34.1, H64 N2048 (2048) 67.9/87.8/74.1,
//                H128 N1000 (2048) 44.1/-/43.9, H124 N1000 46.8/-/50.3, H108 N1000 43.9/-/42.2,
//                H113 N900 (1695) 44.8/-/50.2, H102 N923 (1530) 43.4/56.2/43.4
//   full D64:    H32 N1024 (512) 22.9/14.8/17.3, H64 N1024 (1024) 25.1/27.4/26.3
//   full D128:   H16 N1024 (256) 27.5/15.8/21.5, H7 N2048 (224) 47/27/38, H48 N512 (384)
//                17.6/13.0/13.4, H28 N1024 (448) 27.5/22.3/22.1, H14 N2048 (448) 47.6/40.1/38.5,
//                H4 N8192 (512) 168/155/138, H64 N1024 (1024) 32.5/45.0/35.9
// Packed batches: the small workgroups save padding and, with the chip full, read K and V from the
// caches twice as often. Query heads that share a KV head (`group` of them) share those reads.
// 256-query / QT 2 in us, H query heads over G KV heads, with packed_cost_of_256:
//   causal D128 H32 G8:  15 sequences in 12000 (1.28) 185/168, 32 x 1000 (1.11) 401/384,
//                        16 x 2048 (1.06) 613/633, 8 x 4096 (1.03) 1014/1095
//   causal D128 H16 G16: 60 of 400 .. 1500 (1.28) 377/357, 40 x 768 (1.14) 190/198, 32 x 1000
//                        222/247; H32 G32: 60 of 400 .. 1500 766/889, 40 x 768 413/473,
//                        100 x 300 (1.67) 372/292; H32 G16 27 x 386 (1.20) 120/100; few tiles: H8 G8
//                        15 of 300 .. 2000 63/53
//   causal D64  H16 G16: 15 of 300 .. 2000 (1.25) 65/59, 40 x 700 (1.14) 86/96; H8 G8 64 x 1024
//                        (1.11) 111/121; H32 G8 50 x 640 (1.33) 187/154; H4 G4 26 x 1898 73/67
//   full D128   H32 G8:  100 of 100 .. 1000 (1.13) 656/623, 15 to 1779 (1.13) 128/135, 40 x 768
//                        (1.00) 435/445; H32 G32 40 x 768 520/718, 100 x 256 268/289; H16 G16
//                        100 x 256 135/127; a last round of CUs half empty (packed_idle_of_256):
//                        H16 G16 12 x 500 (1.33) 45/39, 6 x 1000 (1.33) 65/58, H8 G4 19 x 532
//                        (1.12, cost 1.20) 46/39; none: H8 G8 12 x 500 23.1/24.4, 32 x 1000 146/174;
//                        H32 G32 3 of 1982 (1.73, cost 1.09) 42/36, 14 to 1056 (1.12, 1.11) 121/127
int small_query_tiles(int64_t batch, int64_t heads, int64_t kv_heads, int64_t seq, int64_t head_dim,
                      int64_t total, bool causal) {
  const int64_t tiles = fwd_tiles(batch, heads, seq, total, 64);
  const bool packed = total > 0, wide = head_dim == 128;
  if (tiles <= 512) return wide && !causal && seq >= 1024 && tiles > 384 ? 2 : 1;
  if (causal && !wide && tiles <= 1024) return 1;
  if (causal && wide && tiles <= 1024) return 2;
  if (!packed) {
    if (!causal) return 0;
    if (!wide) return tiles <= 8192 ? 2 : 0;
    // From four 256-query blocks per head on, heads that do not divide over the XCDs share their
    // L2s with others' keys, and the small workgroups read those twice as often.
    const int64_t bh = batch * heads;
    const int64_t most = seq <= 768 || bh % 8 == 0 ? 2048 : bh % 4 == 0 ? 1728 : 1500;
    return tiles <= most && seq <= 1024 ? 2 : 0;
  }
  const bool grouped = heads >= 4 * kv_heads, few_kv = kv_heads <= 16;
  const double cost = packed_cost_of_256(batch, seq, total, causal);
  if (causal) {
    if (wide ? tiles <= 2304 && seq <= 2048 : tiles <= 3328) return 2;
    return cost >= (grouped ? 1.1 : !few_kv ? 1.28 : wide ? 1.19 : 1.22) ? 2 : 0;
  }
  if (!wide) return 0;
  if (few_kv && seq <= 256) return 2;
  if (seq <= 1088 &&
      cost * packed_idle_of_256(batch, heads, seq, total) >= (few_kv ? 1.22 : 1.4))
    return 2;
  return cost >= (grouped && seq <= 1024 ? 1.12 : 1.22) ? 2 : 0;
}

// Causal head_dim 128, equal lengths: `items` workgroups (paired_items); otherwise one
// workgroup per query block.
template <typename T, int D>
void launch(int small, bool causal, int64_t items, hipStream_t st, const void* q, const void* k,
            const void* v, void* o, float* lse, const Shape& s) {
  if (small) {
    const dim3 grid(static_cast<unsigned>(s.tiles)), block(SmallGeo<D, 1>::THREADS);
    const FwdArgs<T> a{(const T*)q, (const T*)k, (const T*)v, (T*)o, lse, s};
    if (causal && small == 1)
      hipLaunchKernelGGL((attn_fwd_small_kernel<T, D, 1, true>), grid, block, 0, st, a);
    else if (causal)
      hipLaunchKernelGGL((attn_fwd_small_kernel<T, D, 2, true>), grid, block, 0, st, a);
    else if (small == 1)
      hipLaunchKernelGGL((attn_fwd_small_kernel<T, D, 1, false>), grid, block, 0, st, a);
    else if constexpr (D == 128)  // small_query_tiles gives head_dim 64 no other
      hipLaunchKernelGGL((attn_fwd_small_kernel<T, D, 2, false>), grid, block, 0, st, a);
    return;
  }
  const int64_t n = kPaired<D> && causal && s.cu == nullptr ? items : int64_t(s.tiles);
  const dim3 grid(static_cast<unsigned>(n));
  const FwdArgs<T> a{(const T*)q, (const T*)k, (const T*)v, (T*)o, lse, s};
  if (causal)
    hipLaunchKernelGGL((attn_fwd_dma_kernel<T, D, true>), grid, dim3(kThreads), 0, st, a);
  else
    hipLaunchKernelGGL((attn_fwd_dma_kernel<T, D, false>), grid, dim3(kThreads), 0, st, a);
}

int64_t head_extent_bytes(int64_t seq, int64_t head_dim, int64_t seq_stride) {
  return ((seq - 1) * seq_stride + head_dim) * 2;
}

}  // namespace

namespace tk {

bool attn_fwd_dma_applies(int64_t seq, int64_t head_dim, const int64_t* k_strides,
                          const int64_t* v_strides) {
  // Buffer offsets are 32-bit: each head's K and V rows must span less than 2 GiB.
  const int64_t lim = int64_t(1) << 31;
  return head_extent_bytes(seq, head_dim, k_strides[2]) < lim &&
         head_extent_bytes(seq, head_dim, v_strides[2]) < lim;
}

void attn_fwd_dma_launch(int dtype, const void* q, const void* k, const void* v, void* o,
                         float* lse, int64_t batch, int64_t heads, int64_t kv_heads, int64_t seq,
                         int64_t head_dim, const int64_t* q_strides, const int64_t* k_strides,
                         const int64_t* v_strides, const int64_t* o_strides, float sm_scale,
                         bool causal, hipStream_t stream, const int32_t* cu_seqlens,
                         int64_t total, const void* rope_cos, const void* rope_sin,
                         int64_t rope_stride) {
  Shape s{};
  s.rope_cos = rope_cos;
  s.rope_sin = rope_sin;
  s.rope_stride = rope_stride;
  s.heads = (int)heads;
  s.seq = (int)seq;
  s.group = (int)(heads / kv_heads);
  s.cu = cu_seqlens;
  s.total = (int)total;
  for (int i = 0; i < 3; ++i) {
    s.q[i] = q_strides[i];
    s.k[i] = k_strides[i];
    s.v[i] = v_strides[i];
    s.o[i] = o_strides[i];
  }
  s.scale_log2 = sm_scale * 1.4426950408889634f;
  s.batch = (int)batch;
  const int64_t packed = cu_seqlens != nullptr ? total : 0;
  const int small = small_query_tiles(batch, heads, kv_heads, seq, head_dim, packed, causal);
  const int64_t rows = small ? 64 * small : 256;
  s.q_blocks = (int)cdiv(seq, rows);
  s.tiles = (int)fwd_tiles(batch, heads, seq, packed, rows);
  s.k_bytes = (uint32_t)head_extent_bytes(seq, head_dim, k_strides[2]);
  s.v_bytes = (uint32_t)head_extent_bytes(seq, head_dim, v_strides[2]);
  const int64_t items = cu_seqlens == nullptr ? paired_items(batch * heads, s.q_blocks)
                                              : int64_t(s.tiles);
  if (dtype == TK_DTYPE_F16) {
    if (head_dim == 64) launch<_Float16, 64>(small, causal, items, stream, q, k, v, o, lse, s);
    else launch<_Float16, 128>(small, causal, items, stream, q, k, v, o, lse, s);
  } else {
    if (head_dim == 64) launch<__bf16, 64>(small, causal, items, stream, q, k, v, o, lse, s);
    else launch<__bf16, 128>(small, causal, items, stream, q, k, v, o, lse, s);
  }
}

}  // namespace tk

extern "C" int tk_attn_fwd_rows(int64_t batch, int64_t heads, int64_t kv_heads, int64_t seq,
                                int64_t head_dim, int64_t total, int causal) {
  if (batch <= 0 || kv_heads <= 0 || heads % kv_heads != 0 || heads <= 0 || seq <= 0 || total < 0 ||
      (head_dim != 64 && head_dim != 128))
    return 0;
  const int small = small_query_tiles(batch, heads, kv_heads, seq, head_dim, total, causal != 0);
  return small ? 64 * small : 256;
}
