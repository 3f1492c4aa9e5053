// GEMM entry points, C = A * B on CDNA4 MFMA: f16/bf16 inputs, float32 accumulation, f16/bf16
// output (src/tklab/kernels/matmul.py:72-164 computes the same product; here the tiling is
// MI355X's own), and the kernels for operands the DMA cannot load.
//
// tk_gemm sends operands stored by aligned rows (row-major or transposed) to the buffer->LDS
// DMA kernels (gemm_dma.hip, gemm_tile_kernels.hpp). This file's register-staged kernel takes
// everything else: odd row lengths and row strides, unaligned bases, two non-unit strides,
// operands of 2 GiB and more.
//
// It keeps the DMA tile kernel's block tiles, wave grid, LDS stage layout and fragment reads;
// only how a stage is filled differs. Each thread loads the 16-byte chunks that the DMA would
// have put at its LDS slots into registers, two K tiles ahead, and writes them to LDS one tile
// ahead: two register sets, two LDS stages, one barrier per 64-wide K tile. A chunk starts at
// any element: with one unit stride it is one 16-byte load at 2-byte alignment, strided operands
// load element by element. The loads have no branches (with them every load waited for the one
// before: 125 us below), and what lies past K is zeroed on the way to LDS.
// What bounds it is the vector memory path: an unaligned 128-byte row piece touches two lines.
// bf16 1500x1500x6000: 1651 us with the per-element loads of a 256 x 256 x 64 kernel -> 67 us
// (406 TFLOP/s; 64-bit offsets per load 72 us); fp16 4097^3 3150 -> 262 us; bf16 7x4001x4100
// 598 -> 28 us; a linear layer's three products at 1111x4099x2050 2467 -> 166 us.
#include "gemm_tile_kernels.hpp"

#include <algorithm>
#include <utility>

#pragma clang fp contract(off)

namespace {

using namespace tk::gemm_dma;

constexpr Tile kStagedTiles[] = {{256, 128}, {128, 128}, {64, 64}};
constexpr int kStagedTileCount = sizeof(kStagedTiles) / sizeof(kStagedTiles[0]);
constexpr int kFirstStrided = 1;  // element loads of a 256 x 128 tile do not fit the registers

// An operand: element (row, k) of a K-contiguous one at row * ld + k * inner, element (k, col)
// of one stored by k-rows at k * ld + col * inner. Element offsets of the problem fit 31 bits;
// 32-bit arithmetic may wrap for elements outside it.
struct Operand {
  uint32_t ld, inner;
  uint32_t extent;  // elements from the base to the last one, inclusive
};

struct StagedProblem {
  Problem p;
  Operand a, b;
};

// The element at offset `off` (below 2^31), as a scalar base plus a 32-bit byte offset.
template <typename V>
__device__ __forceinline__ const V* at(const uint16_t* base, uint32_t off) {
  return reinterpret_cast<const V*>(reinterpret_cast<const char*>(base) + off * 2u);
}

// Eight elements off, off + inner, ...; no branch, so that a tile's loads are all in flight at
// once. Offsets past the operand's end are moved back inside it: fix_chunk undoes that.
template <bool kUnit>
__device__ __forceinline__ i32x4 load_chunk(const uint16_t* __restrict__ base, const Operand& o,
                                            uint32_t off) {
  if constexpr (kUnit) {
    return at<Unaligned16>(base, min(off, o.extent - 8))->v;
  } else {
    typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
    u16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = *at<uint16_t>(base, min(off + e * o.inner, o.extent - 1));
    return __builtin_bit_cast(i32x4, v);
  }
}

// The chunk loaded for `off` as its first `valid` elements followed by zeros.
template <bool kUnit>
__device__ __forceinline__ i32x4 fix_chunk(i32x4 v, const Operand& o, uint32_t off, int valid) {
  if constexpr (kUnit) {
    const uint32_t shift = off > o.extent - 8 ? off - (o.extent - 8) : 0u;
    if (shift & 4) v = i32x4{v[2], v[3], 0, 0};
    if (shift & 2) v = i32x4{v[1], v[2], v[3], 0};
    if (shift & 1)
#pragma unroll
      for (int d = 0; d < 4; ++d)
        v[d] = int((uint32_t(v[d]) >> 16) | (d < 3 ? uint32_t(v[d + 1]) << 16 : 0u));
  }
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const int left = valid - 2 * d;
    v[d] = left >= 2 ? v[d] : left == 1 ? v[d] & 0xffff : 0;
  }
  return v;
}

template <typename T, int BM, int BN, Layout kLayout, bool kUnit>
__global__ __launch_bounds__(kTileThreads) void gemm_kernel(const T* __restrict__ A,
                                                            const T* __restrict__ B,
                                                            T* __restrict__ C, StagedProblem sp) {
  constexpr bool kARows = kLayout == Layout::TN, kBRows = kLayout != Layout::NT;
  constexpr int WM = Grid<BM, BN>::WM, WN = Grid<BM, BN>::WN;
  constexpr int MT = BM / WM / 16, NT = BN / WN / 16;
  constexpr int kStageBytes = (BM + BN) * 128;
  constexpr int kA = BM / 64, kB = BN / 64;  // chunks per thread and K tile
  constexpr int kStaged = BM * stage_stride(BN);
  __shared__ __attribute__((aligned(1024))) char lds[2 * kStageBytes > kStaged ? 2 * kStageBytes : kStaged];
  const Problem& p = sp.p;

  int m0, n0;
  tile_origin<BM, BN, BN>(p, m0, n0);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = (wave / WN) * (BM / WM), wn = (wave % WN) * (BN / WN);
  const int l16 = lane & 15, lg = lane >> 4;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_void*)lds;
  const int kt = (p.k + kTileK - 1) / kTileK;

  // Chunk x of this thread is the one at byte x * 8192 + wave * 1024 + lane * 16 of the
  // operand's stage (tile_source's placement). Rows and columns past the operand's edge load
  // the last one's values, which only reach outputs that are not stored; k past the edge must
  // read as zero (`valid` of a chunk's elements lie inside K).
  uint32_t a_off[kA], b_off[kB];  // of K tile 0
  int a_k[kA], b_k[kB];
  auto place = [&](auto rows, const Operand& o, int x, int first, int count, uint32_t& off, int& k) {
    const int i = x * 8 + wave, slot = lane & 7;
    if constexpr (decltype(rows)::value) {
      k = (i & 7) * 8 + (lane >> 3);
      const int col = first + (i >> 3) * 64 + ((((slot >> 1) ^ row_swz(k)) << 1) | (slot & 1)) * 8;
      off = k * o.ld + min(col, count - 1) * o.inner;
    } else {
      const int r = i * 8 + (lane >> 3);
      k = (slot ^ a_swz(r)) * 8;
      off = min(first + r, count - 1) * o.ld + k * o.inner;
    }
  };
  using ARows = std::integral_constant<bool, kARows>;
  using BRows = std::integral_constant<bool, kBRows>;
#pragma unroll
  for (int x = 0; x < kA; ++x) place(ARows{}, sp.a, x, m0, p.m, a_off[x], a_k[x]);
#pragma unroll
  for (int x = 0; x < kB; ++x) place(BRows{}, sp.b, x, n0, p.n, b_off[x], b_k[x]);
  const uint32_t a_step = kTileK * (kARows ? sp.a.ld : sp.a.inner);
  const uint32_t b_step = kTileK * (kBRows ? sp.b.ld : sp.b.inner);
  auto valid = [&](bool rows, int k) { return rows ? (k < p.k ? 8 : 0) : max(0, min(8, p.k - k)); };
  const uint16_t* a_base = reinterpret_cast<const uint16_t*>(A);
  const uint16_t* b_base = reinterpret_cast<const uint16_t*>(B);
  auto load = [&](int tile, i32x4 (&va)[kA], i32x4 (&vb)[kB]) {
#pragma unroll
    for (int x = 0; x < kA; ++x) va[x] = load_chunk<kUnit>(a_base, sp.a, a_off[x] + tile * a_step);
#pragma unroll
    for (int x = 0; x < kB; ++x) vb[x] = load_chunk<kUnit>(b_base, sp.b, b_off[x] + tile * b_step);
  };
  // Only a chunk within 8 rows of K's end can be cut short or moved (a row may be shorter than
  // a chunk).
  auto store = [&](int tile, i32x4 (&va)[kA], i32x4 (&vb)[kB]) {
    if ((tile + 1) * kTileK + 8 > p.k) {
#pragma unroll
      for (int x = 0; x < kA; ++x)
        va[x] = fix_chunk<kUnit>(va[x], sp.a, a_off[x] + tile * a_step,
                                 valid(kARows, tile * kTileK + a_k[x]));
#pragma unroll
      for (int x = 0; x < kB; ++x)
        vb[x] = fix_chunk<kUnit>(vb[x], sp.b, b_off[x] + tile * b_step,
                                 valid(kBRows, tile * kTileK + b_k[x]));
    }
    char* dst = lds + (tile & 1) * kStageBytes + wave * 1024 + lane * 16;
#pragma unroll
    for (int x = 0; x < kA; ++x) *reinterpret_cast<i32x4*>(dst + x * 8192) = va[x];
#pragma unroll
    for (int x = 0; x < kB; ++x) *reinterpret_cast<i32x4*>(dst + BM * 128 + x * 8192) = vb[x];
  };

  const Fragments<kARows, MT> fa(wm, l16, lg);
  const Fragments<kBRows, NT> fb(wn, l16, lg);
  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Tile t: the barrier says that every wave's part of stage t % 2 is written and that stage
  // (t + 1) % 2, which takes tile t + 1 below, has been read (tile t - 1).
  auto step = [&](int t, i32x4 (&ahead_a)[kA], i32x4 (&ahead_b)[kB], i32x4 (&next_a)[kA],
                  i32x4 (&next_b)[kB]) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    load(t + 2, ahead_a, ahead_b);
    const uint32_t base = lds_base + (t & 1) * kStageBytes;
    unroll<0, 2>([&](auto half) {
      constexpr int H = decltype(half)::value;
      i32x4 a[MT], b[NT];
      unroll<0, MT>([&](auto i) { a[decltype(i)::value] = fa.template read<decltype(i)::value, H>(base); });
      unroll<0, NT>([&](auto j) { b[decltype(j)::value] = fb.template read<decltype(j)::value, H>(base + BM * 128); });
      wait_lgkm_pin(a);
      wait_lgkm_pin(b);
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = Mfma<T>::run(b[j], a[i], acc[i][j]);
    });
    store(t + 1, next_a, next_b);
  };
  i32x4 a0[kA], b0[kB], a1[kA], b1[kB];
  load(0, a0, b0);
  load(1, a1, b1);
  store(0, a0, b0);
  for (int t = 0; t < kt; t += 2) {
    step(t, a0, b0, a1, b1);
    if (t + 1 < kt) step(t + 1, a1, b1, a0, b0);
  }
  __syncthreads();

  store_tile<T, BM, BN, kTileThreads>(C, p, m0, n0, lds, [&](auto&& emit) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
        emit(wm + i * 16 + l16, wn + j * 16 + lg * 4, v);
      }
  });
}

template <typename T, int BM, int BN>
void launch_staged(Layout layout, bool unit, const T* a, const T* b, T* c, const StagedProblem& sp,
                   hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(sp.p.tiles_m * sp.p.tiles_n)), block(kTileThreads);
  if (!unit) {
    if constexpr (BM < kStagedTiles[0].m)
      hipLaunchKernelGGL((gemm_kernel<T, BM, BN, Layout::NN, false>), grid, block, 0, stream, a, b, c, sp);
  } else if (layout == Layout::NN) {
    hipLaunchKernelGGL((gemm_kernel<T, BM, BN, Layout::NN, true>), grid, block, 0, stream, a, b, c, sp);
  } else if (layout == Layout::NT) {
    hipLaunchKernelGGL((gemm_kernel<T, BM, BN, Layout::NT, true>), grid, block, 0, stream, a, b, c, sp);
  } else {
    hipLaunchKernelGGL((gemm_kernel<T, BM, BN, Layout::TN, true>), grid, block, 0, stream, a, b, c, sp);
  }
}

// How the register-staged kernel takes a problem; `swap`: as C^T = B^T A^T, both row-major, where
// both operands are transposed (the other fields are after the swap).
struct StagedPlan {
  bool swap, unit;
  Layout layout;
  int tile;
  int64_t a_extent, b_extent;
};

StagedPlan staged_plan(int64_t m, int64_t n, int64_t k, int64_t stride_am, int64_t stride_ak,
                       int64_t stride_bk, int64_t stride_bn) {
  StagedPlan plan{};
  plan.swap = stride_ak != 1 && stride_am == 1 && stride_bn != 1 && stride_bk == 1;
  if (plan.swap) {
    std::swap(m, n);
    std::swap(stride_am, stride_bn);
    std::swap(stride_ak, stride_bk);
  }
  const bool a_rows = stride_ak != 1 && stride_am == 1, b_wide = stride_bn != 1 && stride_bk == 1;
  plan.a_extent = (m - 1) * stride_am + (k - 1) * stride_ak + 1;
  plan.b_extent = (k - 1) * stride_bk + (n - 1) * stride_bn + 1;
  // Wide loads need eight elements to load from.
  plan.unit = (stride_ak == 1 || a_rows) && (stride_bn == 1 || b_wide) && plan.a_extent >= 8 &&
              plan.b_extent >= 8;
  plan.layout = plan.unit && a_rows ? Layout::TN : plan.unit && b_wide ? Layout::NT : Layout::NN;
  const int first = plan.unit ? 0 : kFirstStrided;
  plan.tile = first + pick_tile(kStagedTiles + first, kStagedTileCount - first, m, n, k,
                                Variant::kPlain);
  return plan;
}

template <typename T>
void gemm_staged(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k,
                 int64_t stride_am, int64_t stride_ak, int64_t stride_bk, int64_t stride_bn,
                 int64_t stride_cm, int64_t stride_cn, hipStream_t stream) {
  const StagedPlan plan = staged_plan(m, n, k, stride_am, stride_ak, stride_bk, stride_bn);
  if (plan.swap) {
    std::swap(a, b);
    std::swap(m, n);
    std::swap(stride_am, stride_bn);
    std::swap(stride_ak, stride_bk);
    std::swap(stride_cm, stride_cn);
  }
  const Layout layout = plan.layout;
  const int tile = plan.tile;
  StagedProblem sp{};
  sp.p.m = (int)m;
  sp.p.n = (int)n;
  sp.p.k = (int)k;
  sp.p.scm = stride_cm;
  sp.p.scn = stride_cn;
  sp.p.tiles_m = (int)tk::cdiv(m, kStagedTiles[tile].m);
  sp.p.tiles_n = (int)tk::cdiv(n, kStagedTiles[tile].n);
  auto operand = [](int64_t ld, int64_t inner, int64_t extent) {
    return Operand{(uint32_t)ld, (uint32_t)inner, (uint32_t)extent};
  };
  sp.a = layout == Layout::TN ? operand(stride_ak, 1, plan.a_extent) : operand(stride_am, stride_ak, plan.a_extent);
  sp.b = layout == Layout::NT ? operand(stride_bn, 1, plan.b_extent) : operand(stride_bk, stride_bn, plan.b_extent);
  const T* pa = static_cast<const T*>(a);
  const T* pb = static_cast<const T*>(b);
  T* pc = static_cast<T*>(c);
  if (tile == 0)
    launch_staged<T, 256, 128>(layout, plan.unit, pa, pb, pc, sp, stream);
  else if (tile == 1)
    launch_staged<T, 128, 128>(layout, plan.unit, pa, pb, pc, sp, stream);
  else
    launch_staged<T, 64, 64>(layout, plan.unit, pa, pb, pc, sp, stream);
}

}  // namespace

extern "C" int tk_gemm_tile(const void* a, const void* b, int64_t m, int64_t n, int64_t k,
                            int64_t stride_am, int64_t stride_ak, int64_t stride_bk,
                            int64_t stride_bn) {
  const int64_t lim = INT32_MAX;
  for (int64_t s : {stride_am, stride_ak, stride_bk, stride_bn})
    if (s <= 0) return 0;
  if (m <= 0 || n <= 0 || k <= 0 || m > lim || n > lim || k > lim ||
      tk::extent(m, stride_am, k, stride_ak) > lim || tk::extent(k, stride_bk, n, stride_bn) > lim)
    return 0;
  auto pack = [](int kernel, Tile t) { return kernel << 20 | t.m << 10 | t.n; };
  Plan plan;
  if (tk::gemm_dma::plan(a, b, m, n, k, stride_am, stride_ak, stride_bk, stride_bn, &plan)) {
    const bool plain = plan.layout == Layout::NN && !plan.swap && !plan.k_tail;
    const int tile = plan.swap ? pick_tile(kTiles, kTileCount, n, m, k, Variant::kPlain)
                               : pick_tile(kTiles, kTileCount, m, n, k, Variant::kPlain);
    return pack(plain ? 1 : 2, kTiles[tile]);
  }
  return pack(3, kStagedTiles[staged_plan(m, n, k, stride_am, stride_ak, stride_bk, stride_bn).tile]);
}

extern "C" int tk_gemm(int dtype, const void* a, const void* b, void* c, int64_t m, int64_t n,
                       int64_t k, int64_t stride_am, int64_t stride_ak, int64_t stride_bk,
                       int64_t stride_bn, int64_t stride_cm, int64_t stride_cn, int acc_fp16,
                       void* stream) {
  (void)acc_fp16;  // MFMA accumulates f16/bf16 products in float32 only.
  if (dtype != TK_DTYPE_F16 && dtype != TK_DTYPE_BF16)
    return tk::fail("gemm: dtype must be float16 or bfloat16");
  if (a == nullptr || b == nullptr || c == nullptr) return tk::fail("gemm: null pointer");
  if (m <= 0 || n <= 0 || k <= 0) return tk::fail("gemm: empty problem");
  if (stride_am <= 0 || stride_ak <= 0 || stride_bk <= 0 || stride_bn <= 0 || stride_cm <= 0 ||
      stride_cn <= 0)
    return tk::fail("gemm: strides must be positive");
  // 32-bit element offsets inside the kernel.
  const int64_t lim = INT32_MAX;
  if (m > lim || n > lim || k > lim || tk::extent(m, stride_am, k, stride_ak) > lim ||
      tk::extent(k, stride_bk, n, stride_bn) > lim || tk::extent(m, stride_cm, n, stride_cn) > lim)
    return tk::fail("gemm: operand exceeds the int32 offset range");
  if (tk::cdiv(m, 64) * tk::cdiv(n, 64) > INT32_MAX) return tk::fail("gemm: too many tiles");
  hipStream_t s = tk::as_stream(stream);
  tk::gemm_dma::Plan plan;
  if (tk::gemm_dma::plan(a, b, m, n, k, stride_am, stride_ak, stride_bk, stride_bn, &plan)) {
    tk::gemm_dma_launch(plan, dtype, a, b, c, m, n, k, stride_cm, stride_cn, s);
    return tk::check_launch("gemm");
  }
  if (dtype == TK_DTYPE_F16)
    gemm_staged<_Float16>(a, b, c, m, n, k, stride_am, stride_ak, stride_bk, stride_bn, stride_cm,
                          stride_cn, s);
  else
    gemm_staged<__bf16>(a, b, c, m, n, k, stride_am, stride_ak, stride_bk, stride_bn, stride_cm,
                        stride_cn, s);
  return tk::check_launch("gemm");
}

extern "C" int tk_gemm_splitk(int dtype, const void* a, const void* b, const void* b_up,
                              const float* row_scale, void* c, float* workspace, int64_t m,
                              int64_t n, int64_t k, int64_t splits, int64_t stride_am,
                              int64_t stride_ak, int64_t stride_bk, int64_t stride_bn,
                              int64_t stride_uk, int64_t stride_un, int64_t stride_cm,
                              int64_t stride_cn, void* stream) {
  if (dtype != TK_DTYPE_F16 && dtype != TK_DTYPE_BF16)
    return tk::fail("gemm_splitk: dtype must be float16 or bfloat16");
  if (a == nullptr || b == nullptr || c == nullptr || workspace == nullptr)
    return tk::fail("gemm_splitk: null pointer");
  const int64_t strides[8] = {stride_am, stride_ak, stride_bk, stride_bn,
                              b_up != nullptr ? stride_uk : 1, b_up != nullptr ? stride_un : 1,
                              stride_cm, stride_cn};
  for (int64_t s : strides)
    if (s <= 0) return tk::fail("gemm_splitk: strides must be positive");
  if (b_up != nullptr && row_scale != nullptr)
    return tk::fail("gemm_splitk: either a second weight or row scales");
  if (m <= 0 || n <= 0 || k <= 0) return tk::fail("gemm_splitk: empty problem");
  const int64_t kt = tk::cdiv(k, 64);
  if (splits <= 0 || splits > kt || splits > 65535)
    return tk::fail("gemm_splitk: splits must be between 1 and the 64-wide tiles of K");
  const int64_t lim = INT32_MAX;
  if (m > lim || n > lim || k > lim || tk::extent(m, stride_cm, n, stride_cn) > lim)
    return tk::fail("gemm_splitk: operand exceeds the int32 offset range");
  if ((reinterpret_cast<uintptr_t>(workspace) & 15) != 0)
    return tk::fail("gemm_splitk: workspace must be 16-byte aligned");
  if (tk::cdiv(m, 64) * tk::cdiv(n, 64) > INT32_MAX || tk::cdiv(m * tk::cdiv(n, 4), 256) > INT32_MAX)
    return tk::fail("gemm_splitk: too many tiles");
  // Layouts the DMA kernels do not take run unsplit.
  if (!tk::gemm_split_launch(dtype, a, b, b_up, row_scale, c, workspace, m, n, k, splits, strides,
                             tk::as_stream(stream))) {
    if (b_up != nullptr)
      return tk_gemm_swiglu(dtype, a, b, b_up, c, m, n, k, stride_am, stride_ak, stride_bk,
                            stride_bn, stride_uk, stride_un, stride_cm, stride_cn, stream);
    if (row_scale != nullptr)
      return tk_gemm_rowscale(dtype, a, b, row_scale, c, m, n, k, stride_am, stride_ak, stride_bk,
                              stride_bn, stride_cm, stride_cn, stream);
    return tk_gemm(dtype, a, b, c, m, n, k, stride_am, stride_ak, stride_bk, stride_bn, stride_cm,
                   stride_cn, 0, stream);
  }
  return tk::check_launch("gemm_splitk");
}

extern "C" int tk_gemm_swiglu(int dtype, const void* a, const void* b_gate, const void* b_up,
                              void* y, int64_t m, int64_t n, int64_t k, int64_t stride_am,
                              int64_t stride_ak, int64_t stride_gk, int64_t stride_gn,
                              int64_t stride_uk, int64_t stride_un, int64_t stride_ym,
                              int64_t stride_yn, void* stream) {
  if (dtype != TK_DTYPE_F16 && dtype != TK_DTYPE_BF16)
    return tk::fail("gemm_swiglu: dtype must be float16 or bfloat16");
  if (a == nullptr || b_gate == nullptr || b_up == nullptr || y == nullptr)
    return tk::fail("gemm_swiglu: null pointer");
  if (m <= 0 || n <= 0 || k <= 0) return tk::fail("gemm_swiglu: empty problem");
  if (stride_ym <= 0 || stride_yn <= 0) return tk::fail("gemm_swiglu: strides must be positive");
  const int64_t lim = INT32_MAX;
  if (m > lim || n > lim || k > lim || tk::extent(m, stride_ym, n, stride_yn) > lim)
    return tk::fail("gemm_swiglu: operand exceeds the int32 offset range");
  if (!tk::gemm_dma_applies(a, b_gate, m, n, k, stride_am, stride_ak, stride_gk, stride_gn) ||
      !tk::gemm_dma_applies(a, b_up, m, n, k, stride_am, stride_ak, stride_uk, stride_un))
    return tk::fail("gemm_swiglu: needs unit inner strides, 16-byte aligned rows, k %% 32 == 0, "
                    "n %% 8 == 0 and operands below 2 GiB");
  if (tk::cdiv(m, 64) * tk::cdiv(n, 64) > INT32_MAX) return tk::fail("gemm_swiglu: too many tiles");
  tk::gemm_swiglu_dma_launch(dtype, a, b_gate, b_up, y, m, n, k, stride_am, stride_gk, stride_uk,
                             stride_ym, stride_yn, tk::as_stream(stream));
  return tk::check_launch("gemm_swiglu");
}

extern "C" int tk_gemm_rowscale(int dtype, const void* a, const void* b, const float* row_scale,
                                void* c, int64_t m, int64_t n, int64_t k, int64_t stride_am,
                                int64_t stride_ak, int64_t stride_bk, int64_t stride_bn,
                                int64_t stride_cm, int64_t stride_cn, void* stream) {
  if (dtype != TK_DTYPE_F16 && dtype != TK_DTYPE_BF16)
    return tk::fail("gemm_rowscale: dtype must be float16 or bfloat16");
  if (a == nullptr || b == nullptr || row_scale == nullptr || c == nullptr)
    return tk::fail("gemm_rowscale: null pointer");
  if (m <= 0 || n <= 0 || k <= 0) return tk::fail("gemm_rowscale: empty problem");
  if (stride_cm <= 0 || stride_cn <= 0) return tk::fail("gemm_rowscale: strides must be positive");
  const int64_t lim = INT32_MAX;
  if (m > lim || n > lim || k > lim || tk::extent(m, stride_cm, n, stride_cn) > lim)
    return tk::fail("gemm_rowscale: operand exceeds the int32 offset range");
  if (!tk::gemm_dma_applies(a, b, m, n, k, stride_am, stride_ak, stride_bk, stride_bn))
    return tk::fail("gemm_rowscale: needs unit inner strides, 16-byte aligned rows, k %% 32 == 0, "
                    "n %% 8 == 0 and operands below 2 GiB");
  if (tk::cdiv(m, 64) * tk::cdiv(n, 64) > INT32_MAX) return tk::fail("gemm_rowscale: too many tiles");
  const tk::gemm_dma::Plan plan{tk::gemm_dma::Layout::NN, false, false, stride_am, stride_bk};
  tk::gemm_dma_launch(plan, dtype, a, b, c, m, n, k, stride_cm, stride_cn, tk::as_stream(stream),
                      row_scale);
  return tk::check_launch("gemm_rowscale");
}
