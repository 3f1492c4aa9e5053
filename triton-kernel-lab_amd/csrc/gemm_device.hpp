// Device code shared by the buffer->LDS DMA GEMM kernels (gemm_dma.hip, gemm_tile.hpp): the
// MFMA and LDS access wrappers, the LDS swizzles and the epilogue.
#pragma once
#include "gemm.hpp"
#include "tk_common.hpp"

#include <type_traits>
#include <utility>

// No floating-point contraction: the SwiGLU epilogue must round value * gate * sigmoid(gate)
// to float32 and then to the storage type, as the SwiGLU kernel and the reference do (a fused
// multiply-convert would round once).
#pragma clang fp contract(off)

namespace tk {
namespace gemm_dma {

constexpr int kXcds = 8;
constexpr uint32_t kOob = 0x80000000u;  // past every buffer's num_records: reads as zero

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void lds_void;


struct Problem {
  int m, n, k;
  int lda, ldb, ldb2;  // row strides of the stored matrices; ldb2: the up weight's k stride (SwiGLU variant)
  int64_t scm, scn;
  int tiles_m, tiles_n;
  uint32_t a_bytes, b_bytes, b2_bytes;
  const float* row_scale;  // kRowScale: C[m, :] = round(row_scale[m] * acc)
  // Split K: the float32 sums, and how many 64-wide K tiles a workgroup takes.
  float* partial = nullptr;
  int split_tiles = 0;
};

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  // s_waitcnt fields: vmcnt[3:0], expcnt[6:4] (7 = no wait), lgkmcnt[11:8] (15 = no wait),
  // vmcnt[5:4] at [15:14].
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// Workgroup barrier without the release/acquire fence __syncthreads() carries: the
// fence would wait for every outstanding DMA, while each caller has already waited
// for exactly the tile it is about to read.
__device__ __forceinline__ void barrier_no_fence() { asm volatile("s_barrier" ::: "memory"); }

__device__ __forceinline__ void sched_fence() { __builtin_amdgcn_sched_barrier(0); }

template <int OFF>
__device__ __forceinline__ i32x4 lds_read_b128(uint32_t addr) {
  i32x4 r;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "i"(OFF));
  return r;
}

template <int OFF>
__device__ __forceinline__ i32x2 lds_read_tr16(uint32_t addr) {
  i32x2 r;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "i"(OFF));
  return r;
}

// Y = value * gate * sigmoid(gate) on values already rounded to T, in the SwiGLU
// kernel's operation order (contraction off: each product rounded separately).
template <typename T>
__device__ __forceinline__ T swiglu_out(float gate_acc, float up_acc) {
  const float g = tk::round_to<T>(gate_acc);
  const float v = tk::round_to<T>(up_acc);
  return tk::from_f32<T>(v * g * tk::stable_sigmoid(g));
}

// v_mfma_f32_16x16x32: A lane l holds row l % 16, k = 8 (l / 16) .. +7; B lane l holds
// column l % 16, the same k; D lane l holds column l % 16, rows 4 (l / 16) .. +3.
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Mfma;
template <>
struct Mfma<_Float16> {
  static __device__ __forceinline__ f32x4 run(i32x4 a, i32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
template <>
struct Mfma<__bf16> {
  static __device__ __forceinline__ f32x4 run(i32x4 a, i32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};

// A row swizzle (128-byte rows): 16-byte chunk c of row r sits at c ^ a_swz(r). A fragment
// read phase takes one chunk of 16 consecutive rows: even and odd rows fall in opposite
// halves of a 256-byte bank row, and (r >> 1) & 7 puts the 8 rows of each half on distinct
// 16-byte slots.
__device__ __forceinline__ int a_swz(int r) { return (r >> 1) & 7; }

// B k-row swizzle: 32-byte granule g of k-row k sits at g ^ b_swz(k). A 16x16x32 B
// fragment read phase covers two 16-lane groups reading k-rows 8 apart, so the swizzle
// carries bit 3 of k besides the (k & 3) term that separates the 4 rows of one read.
__device__ __forceinline__ int b_swz(int k) { return 2 * (k & 3) + ((k >> 3) & 1); }

// A fragment of row tile I (16 rows = 2 KiB of the stage).
template <int I>
__device__ __forceinline__ i32x4 read_a(uint32_t addr) {
  return lds_read_b128<I * 2048>(addr);
}

// B fragment: k-rows +0..3 and +4..7 of this lane group (ROWB bytes per k-row).
template <int ROWB>
__device__ __forceinline__ i32x4 read_b(uint32_t addr) {
  const i32x2 lo = lds_read_tr16<0>(addr);
  const i32x2 hi = lds_read_tr16<4 * ROWB>(addr);
  return i32x4{lo[0], lo[1], hi[0], hi[1]};
}

// f(0) .. f(3) with compile-time indices.
template <typename F>
__device__ __forceinline__ void unroll4(F&& f) {
  f(std::integral_constant<int, 0>{});
  f(std::integral_constant<int, 1>{});
  f(std::integral_constant<int, 2>{});
  f(std::integral_constant<int, 3>{});
}

template <int N>
__device__ __forceinline__ void wait_lgkm_pin(i32x4 (&f)[N]) {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(f[i]));
}

// Four values rounded to T, packed in memory order.
template <typename T>
__device__ __forceinline__ uint2 pack4(const float (&v)[4]) {
  const uint32_t lo = uint32_t(__builtin_bit_cast(uint16_t, tk::from_f32<T>(v[0]))) |
                      (uint32_t(__builtin_bit_cast(uint16_t, tk::from_f32<T>(v[1]))) << 16);
  const uint32_t hi = uint32_t(__builtin_bit_cast(uint16_t, tk::from_f32<T>(v[2]))) |
                      (uint32_t(__builtin_bit_cast(uint16_t, tk::from_f32<T>(v[3]))) << 16);
  return uint2{lo, hi};
}

// LDS bytes per row of a staged tile of kCols outputs: 4 dwords past a multiple of the 64 banks
// (32 for 64 columns), so the 16 rows x 2 lane groups of an 8-byte write phase hit distinct
// banks.
constexpr int stage_stride(int cols) { return cols * 2 + 16; }

// 16 bytes at any element boundary (the compiler emits one dwordx4 access).
struct __attribute__((packed, aligned(2))) Unaligned16 {
  i32x4 v;
};

// Writes a kRows x kCols tile of C at (m0, n0). for_each(emit) calls emit(row, column, values)
// for every group of four consecutive columns this lane holds; the kThreads threads of the
// workgroup run it together and `lds` (kRows * stage_stride(kCols) bytes) is idle. With unit
// column stride the rounded tile is staged in LDS and written back as whole rows, 16 bytes per
// lane: non-temporal stores of full 128-byte lines when C rows are 16-byte aligned, stores at
// 2-byte alignment otherwise. Other layouts store element by element.
// Staged, the epilogue of fp16 4096^3 on 256 x 256 tiles took ~4 instead of ~8 us of a ~108 us
// launch (a timing-only copy without stores ran 102 us): 4096^3 108.1 -> 104.3 us, 8192^3 784
// -> 773 us, the row-scaled 16384x6144x4096 GEMM 675 -> 645 us. Staged with default-policy
// stores: 105.1, 773 and 654 us. Per-lane non-temporal stores write 32-byte segments of four
// lines and were 5-14 % slower than default-policy ones.
template <typename T, int kRows, int kCols, int kThreads, typename ForEach>
__device__ __forceinline__ void store_tile(T* __restrict__ C, const Problem& p, int m0, int n0,
                                           char* lds, ForEach&& for_each) {
  if (p.scn != 1) {
    for_each([&](int r, int c, const float (&v)[4]) {
      const int m = m0 + r, n = n0 + c;
      if (m >= p.m || n >= p.n) return;
      T* dst = C + m * p.scm + n * p.scn;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (n + q < p.n) dst[q * p.scn] = tk::from_f32<T>(v[q]);
    });
    return;
  }
  constexpr int kStride = stage_stride(kCols), kLanesPerRow = kCols / 8;
  for_each([&](int r, int c, const float (&v)[4]) {
    *reinterpret_cast<uint2*>(lds + r * kStride + c * 2) = pack4<T>(v);
  });
  __syncthreads();
  // Groups of 16 bytes, in order: kThreads / kLanesPerRow rows per pass where that is whole.
  constexpr bool kWhole = kThreads % kLanesPerRow == 0;
  constexpr int kRowStep = kWhole ? kThreads / kLanesPerRow : 1;
  static_assert(kRows * kLanesPerRow % kThreads == 0, "whole passes");
  auto each_group = [&](auto&& store) {
    int r = threadIdx.x / kLanesPerRow, c = (threadIdx.x % kLanesPerRow) * 8;
#pragma unroll 4
    for (int pass = 0; pass < kRows * kLanesPerRow / kThreads; ++pass) {
      if constexpr (!kWhole) {
        const int g = pass * kThreads + threadIdx.x;
        r = g / kLanesPerRow;
        c = (g % kLanesPerRow) * 8;
      }
      const int row = kWhole ? pass * kRowStep + r : r;
      const i32x4 v = *reinterpret_cast<const i32x4*>(lds + row * kStride + c * 2);
      if (m0 + row < p.m && n0 + c < p.n) store(C + (m0 + row) * p.scm + n0 + c, n0 + c, v);
    }
  };
  if ((p.n & 7) == 0 && (p.scm & 7) == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0) {
    // p.n % 8 == 0, so a 16-byte group is wholly inside or outside N.
    each_group([&](T* dst, int, i32x4 v) {
      __builtin_nontemporal_store(v, reinterpret_cast<i32x4*>(dst));
    });
  } else {
    each_group([&](T* dst, int n, i32x4 v) {
      if (n + 8 <= p.n) {
        reinterpret_cast<Unaligned16*>(dst)->v = v;
      } else {
#pragma unroll
        for (int q = 0; q < 7; ++q)
          if (n + q < p.n)
            reinterpret_cast<uint16_t*>(dst)[q] = uint16_t(uint32_t(v[q >> 1]) >> (16 * (q & 1)));
      }
    });
  }
}

}  // namespace gemm_dma
}  // namespace tk
