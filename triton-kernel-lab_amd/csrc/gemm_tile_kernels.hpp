// DMA GEMM on tiles smaller than 256 x 256, for problems whose 256 x 256 tiles leave CUs idle.
//
// What bounds a tile is the operand bytes one CU can pull through its vector memory path (~21
// B/clock measured in the 256 x 256 kernel, against 32 B/clock its MFMAs could take), so a launch
// takes about (tiles per CU) x (tile rows + tile columns) x K: small tiles move more bytes per
// FLOP, but a problem of few large tiles leaves most CUs without any. pick_tile weighs the two.
//
// Block tile BM x BN, K step 64, 8 wave64s in a WM x WN grid of (BM / WM) x (BN / WN) wave tiles of
// v_mfma_f32_16x16x32, C^T orientation (gemm_dma.hip). A ring of kStages K tiles, one barrier
// per tile: the barrier of tile t says that tile t has landed (each wave waited for its own DMA
// instructions) and that every wave has read tile t - 1, whose stage then takes tile t +
// kStages - 1. Tiles of at most 192 rows and columns run two workgroups per CU where the grid has
// them.
//
// LDS stage: A then B, 128 bytes per tile row or column.
//   A K-contiguous operand: rows of 64 k; the 16-byte chunk c of row r sits at c ^ a_swz(r).
//   An operand stored by k-rows: blocks of 64 columns, 64 k-rows x 128 B; the 32-byte granule
//   g (16 columns) of k-row k sits at g ^ ((k >> 1 & 1) + 2 (k >> 3 & 1)). A transposed read
//   phase covers k-rows {0..3} + 8 {0, 1}: odd and even rows fall in opposite halves of the
//   banks and the swizzle separates the four rows of each half.
// Either way one DMA instruction moves eight 128-byte rows, one whole line each.
#pragma once
#include "gemm_tile.hpp"

#pragma clang fp contract(off)

namespace tk {
namespace gemm_dma {
namespace {

constexpr int kTileThreads = 512;
constexpr int kTileK = 64;

// Waves of a tile: WM x WN. SwiGLU needs an even number of N tiles per wave.
template <int BM, int BN>
struct Grid {
  static constexpr int WM = BN >= 2 * BM || (BM == BN && BM == 128) ? 2 : 4, WN = 8 / WM;
};

__device__ __forceinline__ int row_swz(int k) { return ((k >> 1) & 1) | (((k >> 3) & 1) << 1); }

// Source of DMA instruction i of an operand tile (eight 128-byte rows of the stage); `last` for
// the last K tile, of which kv columns (or k-rows) lie inside K.
template <bool kRows>
__device__ __forceinline__ void tile_source(int i, int lane, int first, int count, int ld, int kv,
                                            uint32_t& src, uint32_t& last) {
  const int slot = lane & 7;
  if constexpr (kRows) {
    const int kr = (i & 7) * 8 + (lane >> 3);
    const int chunk = (((slot >> 1) ^ row_swz(kr)) << 1) | (slot & 1);
    const int col = first + (i >> 3) * 64 + chunk * 8;
    src = col < count ? uint32_t(kr * ld + col) * 2u : kOob;
    last = kr < kv ? src : kOob;
  } else {
    const int r = i * 8 + (lane >> 3);
    const int chunk = slot ^ a_swz(r);
    src = first + r < count ? uint32_t((first + r) * ld + chunk * 8) * 2u : kOob;
    last = chunk * 8 < kv ? src : kOob;
  }
}

// Fragment reads of an operand: tile row (or column) `first` + 16 I + lane % 16.
template <bool kRows, int N>
struct Fragments {
  uint32_t addr[kRows ? N : 2];  // k-rows: per 16 columns; K-contiguous: per 32-wide half
  __device__ __forceinline__ Fragments(int first, int l16, int lg) {
    if constexpr (kRows) {
      const int kr = 8 * lg + (l16 >> 2), q = l16 & 3;
#pragma unroll
      for (int i = 0; i < N; ++i) set(i, first / 16 + i, kr, q);
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        addr[h] = (first + l16) * 128 + (((4 * h + lg) ^ a_swz(l16)) * 16);
    }
  }
  __device__ __forceinline__ void set(int i, int granule, int kr, int q) {
    addr[i] = (granule >> 2) * 8192 + kr * 128 + (((granule & 3) ^ row_swz(kr)) * 32) + q * 8;
  }
  template <int I, int H>
  __device__ __forceinline__ i32x4 read(uint32_t base) const {
    if constexpr (kRows) {
      const i32x2 lo = lds_read_tr16<H * 4096>(base + addr[I]);
      const i32x2 hi = lds_read_tr16<H * 4096 + 512>(base + addr[I]);
      return i32x4{lo[0], lo[1], hi[0], hi[1]};
    } else {
      return lds_read_b128<I * 2048>(base + addr[H]);
    }
  }
};

// First row and column of this workgroup's tile: workgroup w runs on XCD w % 8; each XCD walks a
// contiguous range of tiles in groups of kGroup M-tiles, sharing A and B panels in its L2.
template <int BM, int BN, int kOutN>
__device__ __forceinline__ void tile_origin(const Problem& p, int& m0, int& n0) {
  constexpr int kGroup = BN > BM ? 8 : 4;
  const int total = p.tiles_m * p.tiles_n;
  const int xcd = blockIdx.x % kXcds;
  const int w = xcd * (total / kXcds) + min(xcd, total % kXcds) + blockIdx.x / kXcds;
  const int per_group = kGroup * p.tiles_n;
  const int first_m = (w / per_group) * kGroup;
  const int group_m = min(p.tiles_m - first_m, kGroup);
  m0 = (first_m + (w % per_group) % group_m) * BM;
  n0 = ((w % per_group) / group_m) * kOutN;
}

template <int I, int N, typename F>
__device__ __forceinline__ void unroll(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    unroll<I + 1, N>(f);
  }
}

// kAnyK: K need not be a multiple of 32. kSplit: workgroup (x, y) sums the y-th run of
// p.split_tiles K tiles into p.partial (gemm_split_kernel).
template <typename T, int BM, int BN, int kStages, Layout kLayout, bool kAnyK, Variant kVariant,
          bool kSplit = false>
__device__ __forceinline__ void gemm_tile(const T* __restrict__ A, const T* __restrict__ B,
                                          const T* __restrict__ B2, T* __restrict__ C,
                                          const Problem& p) {
  constexpr bool kARows = kLayout == Layout::TN, kBRows = kLayout != Layout::NT;
  constexpr bool kSwiGLU = kVariant == Variant::kSwiGLU;
  constexpr bool kRowScale = kVariant == Variant::kRowScale;
  constexpr int WM = Grid<BM, BN>::WM, WN = Grid<BM, BN>::WN;
  constexpr int MT = BM / WM / 16, NT = BN / WN / 16;  // 16 x 16 tiles per wave
  constexpr int kStageBytes = (BM + BN) * 128;
  constexpr int kADma = BM / 64, kBDma = BN / 64;  // DMA instructions per wave and K tile
  constexpr int kOutN = kSwiGLU ? BN / 2 : BN;
  constexpr int kStaged = BM * stage_stride(kOutN);
  constexpr int kLds = kStages * kStageBytes > kStaged + BM * 4 ? kStages * kStageBytes
                                                                : kStaged + BM * 4;
  static_assert(!kSwiGLU || (NT % 2 == 0 && BN % 128 == 0), "gate and up columns per wave and block");
  __shared__ __attribute__((aligned(1024))) char lds[kLds];

  int m0, n0;
  tile_origin<BM, BN, kOutN>(p, m0, n0);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = (wave / WN) * (BM / WM), wq = wave % WN;
  const int l16 = lane & 15, lg = lane >> 4;
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc((void*)A, (short)0, p.a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb =
      __builtin_amdgcn_make_buffer_rsrc((void*)B, (short)0, p.b_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb2 =
      __builtin_amdgcn_make_buffer_rsrc((void*)B2, (short)0, p.b2_bytes, 0x00020000);
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_void*)lds;

  if constexpr (!kAnyK) __builtin_assume(p.k % 32 == 0);
  const int kt = (p.k + kTileK - 1) / kTileK;
  const int kv = p.k - (kt - 1) * kTileK;
  const int first = kSplit ? int(blockIdx.y) * p.split_tiles : 0;  // K tiles first .. end - 1
  const int end = kSplit ? min(kt, first + p.split_tiles) : kt;
  // Instruction x of wave w is instruction x * 8 + w of the operand's tile; with SwiGLU the
  // first half of them reads the gate weight.
  uint32_t a_src[kADma], a_last[kADma], b_src[kBDma], b_last[kBDma];
#pragma unroll
  for (int x = 0; x < kADma; ++x)
    tile_source<kARows>(x * 8 + wave, lane, m0, p.m, p.lda, kv, a_src[x], a_last[x]);
#pragma unroll
  for (int x = 0; x < kBDma; ++x) {
    const bool up = kSwiGLU && x >= kBDma / 2;
    tile_source<kBRows>((up ? x - kBDma / 2 : x) * 8 + wave, lane, n0, p.n, up ? p.ldb2 : p.ldb, kv,
                        b_src[x], b_last[x]);
  }
  const uint32_t a_step = kARows ? uint32_t(kTileK * p.lda) * 2u : 128u;
  const uint32_t b_step = kBRows ? uint32_t(kTileK * p.ldb) * 2u : 128u;
  const uint32_t b2_step = uint32_t(kTileK * p.ldb2) * 2u;

  float row_scale = 0.f;
  if constexpr (kRowScale)
    if (threadIdx.x < BM) row_scale = p.row_scale[min(m0 + (int)threadIdx.x, p.m - 1)];

  // Tiles past the end reload the last one into a stage that is never read, keeping every
  // tile's DMA count constant.
  auto load = [&](int tile, int stage) {
    tile = min(tile, end - 1);
    const bool last = tile == kt - 1;
    char* at = lds + stage * kStageBytes + wave * 1024;
#pragma unroll
    for (int x = 0; x < kADma; ++x)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void*)(at + x * 8192), 16,
                                               last ? a_last[x] : a_src[x], tile * a_step, 0, 0);
    at += BM * 128;
#pragma unroll
    for (int x = 0; x < kBDma; ++x) {
      const bool up = kSwiGLU && x >= kBDma / 2;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(up ? rb2 : rb, (lds_void*)(at + x * 8192), 16,
                                               last ? b_last[x] : b_src[x],
                                               tile * (up ? b2_step : b_step), 0, 0);
    }
  };

  const Fragments<kARows, MT> fa(wm, l16, lg);
  Fragments<kBRows, NT> fb(wq * (BN / WN), l16, lg);
  if constexpr (kSwiGLU) {
    // N tiles 0 .. NT/2 - 1: gate columns; the rest: the same up columns.
#pragma unroll
    for (int j = 0; j < NT; ++j)
      fb.set(j, (j < NT / 2 ? 0 : BN / 32) + wq * (NT / 2) + j % (NT / 2), 8 * lg + (l16 >> 2),
             l16 & 3);
  }

  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int t = 0; t < kStages - 1; ++t) load(first + t, t);

  i32x4 a0[MT], b0[NT], a1[MT], b1[NT];
  int stage = 0, fill = kStages - 1;
  for (int t = first; t < end; ++t) {
    wait_vmcnt<(kStages - 2) * (kADma + kBDma)>();
    barrier_no_fence();
    const uint32_t base = lds_base + stage * kStageBytes;
    unroll<0, MT>([&](auto i) { a0[i] = fa.template read<decltype(i)::value, 0>(base); });
    unroll<0, NT>([&](auto j) { b0[j] = fb.template read<decltype(j)::value, 0>(base + BM * 128); });
    load(t + kStages - 1, fill);
    wait_lgkm_pin(a0);
    wait_lgkm_pin(b0);
    unroll<0, MT>([&](auto i) { a1[i] = fa.template read<decltype(i)::value, 1>(base); });
    unroll<0, NT>([&](auto j) { b1[j] = fb.template read<decltype(j)::value, 1>(base + BM * 128); });
    sched_fence();
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = Mfma<T>::run(b0[j], a0[i], acc[i][j]);
    sched_fence();
    wait_lgkm_pin(a1);
    wait_lgkm_pin(b1);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = Mfma<T>::run(b1[j], a1[i], acc[i][j]);
    fill = stage;
    stage = stage == kStages - 1 ? 0 : stage + 1;
  }
  wait_vmcnt<0>();
  if constexpr (kSplit) {
    // [split][gate, up][m][n] float32; a lane's four values are consecutive columns.
    const int64_t plane = int64_t(p.m) * p.n;
    constexpr int kPlanes = kSwiGLU ? 2 : 1, kTiles = NT / kPlanes;
    float* out = p.partial + blockIdx.y * kPlanes * plane;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int m = m0 + wm + i * 16 + l16;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int n = n0 + wq * (kOutN / WN) + (j % kTiles) * 16 + lg * 4;
        float* at = out + (j / kTiles) * plane + int64_t(m) * p.n + n;
        if (m >= p.m || n >= p.n) continue;
        if ((p.n & 3) == 0) {
          *reinterpret_cast<f32x4*>(at) = acc[i][j];
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < p.n) at[e] = acc[i][j][e];
        }
      }
    }
    return;
  }
  __syncthreads();

  float* scales = reinterpret_cast<float*>(lds + kStaged);
  if constexpr (kRowScale) {
    if (threadIdx.x < BM) scales[threadIdx.x] = row_scale;
    __syncthreads();
  }
  store_tile<T, BM, kOutN, kTileThreads>(C, p, m0, n0, lds, [&](auto&& emit) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int r = wm + i * 16 + l16;
      const float sc = kRowScale ? scales[r] : 1.f;
#pragma unroll
      for (int j = 0; j < (kSwiGLU ? NT / 2 : NT); ++j) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (kSwiGLU)
            v[e] = static_cast<float>(swiglu_out<T>(acc[i][j][e], acc[i][j + NT / 2][e]));
          else
            v[e] = kRowScale ? acc[i][j][e] * sc : acc[i][j][e];
        }
        emit(r, wq * (kOutN / WN) + j * 16 + lg * 4, v);
      }
    }
  });
}

// Ring depth: as many K tiles as fit half a CU's LDS for the tiles that run two workgroups per
// CU, all of it for the larger ones.
constexpr int tile_stages(int bm, int bn) {
  const int bytes = (bm + bn) * 128;
  return bm + bn <= 192 ? 81920 / bytes : 163840 / bytes > 5 ? 5 : 163840 / bytes;
}

// Row-major operands with K % 32 == 0 (NN), and the fused variants.
template <typename T, int BM, int BN, Variant kVariant>
__global__ __launch_bounds__(kTileThreads) void gemm_dma_kernel(const T* __restrict__ A,
                                                                const T* __restrict__ B,
                                                                const T* __restrict__ B2,
                                                                T* __restrict__ C, Problem p) {
  gemm_tile<T, BM, BN, tile_stages(BM, BN), Layout::NN, false, kVariant>(A, B, B2, C, p);
}

// Transposed operands and K % 32 != 0.
template <typename T, int BM, int BN, Layout kLayout>
__global__ __launch_bounds__(kTileThreads) void gemm_kernel(const T* __restrict__ A,
                                                            const T* __restrict__ B,
                                                            T* __restrict__ C, Problem p) {
  gemm_tile<T, BM, BN, tile_stages(BM, BN), kLayout, true, Variant::kPlain>(A, B, B, C, p);
}

// Split K. A problem of few 64 x 64 tiles and a long K leaves most CUs idle while one workgroup
// walks K at what one CU pulls: unsplit, the five problems below request 29 to 48 GB/s per CU over
// the whole launch (64x4096x14336 43, 16x512x8192 48; deeper rings, two K tiles per barrier and nt
// loads changed nothing). Its K is cut into runs of whole K tiles, one workgroup each,
// whose float32 sums the second kernel adds in order of K and rounds as the unsplit epilogues
// do. bf16, unsplit -> split, both kernels: 64x4096x14336 84.6 -> 31.9 us (4 runs, 117 MB: 3.8
// TB/s), 16x2048x8192 37.1 -> 14.4 (8), 16x6144x4096 22.7 -> 16.7 (2), 16x512x8192 27.4 -> 10.6
// (8), SwiGLU 64x2048x8192 75.5 -> 25.8 (8). The wide tiles stay unsplit: SwiGLU 16x14336x4096
// 45.8, 2 runs 53.6.
template <typename T, int BM, int BN, Layout kLayout, Variant kVariant>
__global__ __launch_bounds__(kTileThreads) void gemm_split_kernel(const T* __restrict__ A,
                                                                  const T* __restrict__ B,
                                                                  const T* __restrict__ B2,
                                                                  Problem p) {
  gemm_tile<T, BM, BN, tile_stages(BM, BN), kLayout, true, kVariant, true>(A, B, B2, nullptr, p);
}

// C from the partial sums: one thread per four columns, splits added in order.
template <typename T, Variant kVariant>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(T* __restrict__ C, Problem p, int splits) {
  constexpr int kPlanes = kVariant == Variant::kSwiGLU ? 2 : 1;
  const int groups = (p.n + 3) / 4;
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= int64_t(p.m) * groups) return;
  const int m = int(i / groups), n = int(i % groups) * 4;
  const int64_t plane = int64_t(p.m) * p.n;
  const int count = min(4, p.n - n);
  float sum[kPlanes][4];
#pragma unroll
  for (int h = 0; h < kPlanes; ++h) {
#pragma unroll
    for (int e = 0; e < 4; ++e) sum[h][e] = 0.f;
    const float* at = p.partial + h * plane + int64_t(m) * p.n + n;
#pragma unroll 4
    for (int s = 0; s < splits; ++s, at += kPlanes * plane) {
      if ((p.n & 3) == 0) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(at);
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[h][e] += v[e];
      } else {
        for (int e = 0; e < count; ++e) sum[h][e] += at[e];
      }
    }
  }
  const float scale = kVariant == Variant::kRowScale ? p.row_scale[m] : 1.f;
  T* dst = C + m * p.scm + n * p.scn;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (e >= count) break;
    T v;
    if constexpr (kVariant == Variant::kSwiGLU)
      v = swiglu_out<T>(sum[0][e], sum[1][e]);
    else if constexpr (kVariant == Variant::kRowScale)
      v = tk::from_f32<T>(sum[0][e] * scale);
    else
      v = tk::from_f32<T>(sum[0][e]);
    dst[e * p.scn] = v;
  }
}

template <typename T, int BM, int BN>
void launch_one(Variant variant, const Plan& plan, const T* a, const T* b, const T* b2, T* c,
                const Problem& p, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(p.tiles_m * p.tiles_n)), block(kTileThreads);
  if (variant == Variant::kSwiGLU) {
    if constexpr (BN % 128 == 0 && (BN / Grid<BM, BN>::WN / 16) % 2 == 0)
      hipLaunchKernelGGL((gemm_dma_kernel<T, BM, BN, Variant::kSwiGLU>), grid, block, 0, stream, a,
                         b, b2, c, p);
  } else if (variant == Variant::kRowScale) {
    hipLaunchKernelGGL((gemm_dma_kernel<T, BM, BN, Variant::kRowScale>), grid, block, 0, stream, a,
                       b, b, c, p);
  } else if (plan.layout == Layout::NN && !plan.k_tail) {
    hipLaunchKernelGGL((gemm_dma_kernel<T, BM, BN, Variant::kPlain>), grid, block, 0, stream, a, b,
                       b, c, p);
  } else if (plan.layout == Layout::NN) {
    hipLaunchKernelGGL((gemm_kernel<T, BM, BN, Layout::NN>), grid, block, 0, stream, a, b, c, p);
  } else if (plan.layout == Layout::NT) {
    hipLaunchKernelGGL((gemm_kernel<T, BM, BN, Layout::NT>), grid, block, 0, stream, a, b, c, p);
  } else {
    hipLaunchKernelGGL((gemm_kernel<T, BM, BN, Layout::TN>), grid, block, 0, stream, a, b, c, p);
  }
}

template <typename T, int I>
void launch_index(int tile, Variant variant, const Plan& plan, const T* a, const T* b, const T* b2,
                  T* c, const Problem& p, hipStream_t stream) {
  if constexpr (I < kTileCount) {
    if (tile == I)
      launch_one<T, kTiles[I].m, kTiles[I].n>(variant, plan, a, b, b2, c, p, stream);
    else
      launch_index<T, I + 1>(tile, variant, plan, a, b, b2, c, p, stream);
  }
}

}  // namespace

template <typename T>
void launch_tile(int tile, Variant variant, const Plan& plan, const void* a, const void* b,
                 const void* b2, void* c, const Problem& p, hipStream_t stream) {
  launch_index<T, 1>(tile, variant, plan, static_cast<const T*>(a), static_cast<const T*>(b),
                     static_cast<const T*>(b2), static_cast<T*>(c), p, stream);
}

template <typename T>
void launch_split(Variant variant, const Plan& plan, const void* a, const void* b, const void* b2,
                  void* c, const Problem& p, int splits, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(p.tiles_m * p.tiles_n), static_cast<unsigned>(splits));
  const dim3 block(kTileThreads);
  const dim3 reduce(static_cast<unsigned>(cdiv(int64_t(p.m) * cdiv(p.n, 4), 256)));
  const T* pa = static_cast<const T*>(a);
  const T* pb = static_cast<const T*>(b);
  const T* pb2 = static_cast<const T*>(b2);
  T* pc = static_cast<T*>(c);
  if (variant == Variant::kSwiGLU)
    hipLaunchKernelGGL((gemm_split_kernel<T, 64, 128, Layout::NN, Variant::kSwiGLU>), grid, block,
                       0, stream, pa, pb, pb2, p);
  else if (plan.layout == Layout::NN)
    hipLaunchKernelGGL((gemm_split_kernel<T, 64, 64, Layout::NN, Variant::kPlain>), grid, block, 0,
                       stream, pa, pb, pb, p);
  else if (plan.layout == Layout::NT)
    hipLaunchKernelGGL((gemm_split_kernel<T, 64, 64, Layout::NT, Variant::kPlain>), grid, block, 0,
                       stream, pa, pb, pb, p);
  else
    hipLaunchKernelGGL((gemm_split_kernel<T, 64, 64, Layout::TN, Variant::kPlain>), grid, block, 0,
                       stream, pa, pb, pb, p);
  if (variant == Variant::kSwiGLU)
    hipLaunchKernelGGL((gemm_reduce_kernel<T, Variant::kSwiGLU>), reduce, dim3(256), 0, stream, pc,
                       p, splits);
  else if (variant == Variant::kRowScale)
    hipLaunchKernelGGL((gemm_reduce_kernel<T, Variant::kRowScale>), reduce, dim3(256), 0, stream,
                       pc, p, splits);
  else
    hipLaunchKernelGGL((gemm_reduce_kernel<T, Variant::kPlain>), reduce, dim3(256), 0, stream, pc,
                       p, splits);
}

}  // namespace gemm_dma
}  // namespace tk
