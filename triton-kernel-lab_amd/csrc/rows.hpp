// Row-per-group building blocks shared by the softmax and RMSNorm kernels.
//
// A row of `cols` elements is owned by a group of RT threads (RT = 64: one
// wave; RT = 256 or 1024: several waves meeting in LDS). Each thread holds
// VALS elements of the row in registers, as VALS/VEC vectors of VEC
// contiguous elements: vector i of thread `lane` covers columns
// [(i*RT + lane)*VEC, +VEC). With VEC = 16/sizeof(T) every access is one
// 128-bit load or store and a wave touches 1 KiB of contiguous row per
// vector index. Rows whose base or stride is not 16-byte aligned, or whose width is not a
// multiple of VEC, keep the vectors and access them at any element boundary (the *_any
// functions); VEC = 1 is left to rows narrower than one vector.
#pragma once

#include "tk_common.hpp"

namespace tk {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

// Cache-policy bits of gfx950 buffer loads and stores (the aux operand: sc0 = 1,
// nt = 2, sc1 = 16). Rows streamed once are loaded non-temporally so they do not
// displace reusable lines in L2 and the 256 MiB last-level cache; measured on the
// residual-RMSNorm step (bf16 16384 x 4096), non-temporal loads plus these store
// policies took the forward from 5.2 to 5.8 TB/s and the backward stage 1 from 4.9
// to 5.3 TB/s run alone, and the forward+backward step from 4.6 to 5.3 TB/s.
constexpr int kCpolDefault = 0;
constexpr int kCpolStream = 2;  // nt
constexpr int kCpolSc1 = 16;    // sc1

template <typename T, int VEC, int RT, int VALS>
__device__ __forceinline__ void load_row(const T* __restrict__ row, int cols, int lane, float* v,
                                         float fill) {
  constexpr int ITEMS = VALS / VEC;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int c = (i * RT + lane) * VEC;
    if (c < cols) {
      load_vec<T, VEC>(row + c, v + i * VEC);
    } else {
#pragma unroll
      for (int j = 0; j < VEC; ++j) v[i * VEC + j] = fill;
    }
  }
}

template <typename T, int VEC, int RT, int VALS>
__device__ __forceinline__ void store_row(T* __restrict__ row, int cols, int lane, const float* v) {
  constexpr int ITEMS = VALS / VEC;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int c = (i * RT + lane) * VEC;
    if (c < cols) store_vec<T, VEC>(row + c, v + i * VEC);
  }
}

// Branch-free 16-byte row access through a buffer resource spanning the row, with
// cache policy CPOL; columns at or past `cols` load as `fill` and are not stored.
// `row` must be wave-uniform (see RawRow::load_buf).
template <typename T, int VEC, int RT, int VALS, int CPOL>
__device__ __forceinline__ void load_row_buf(const T* row, int cols, int lane, float* v,
                                             float fill) {
  static_assert(VEC * sizeof(T) == 16, "16-byte vectors only");
  constexpr int ITEMS = VALS / VEC;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(row), (short)0, uint32_t(cols) * uint32_t(sizeof(T)), 0x00020000);
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int c = (i * RT + lane) * VEC;
    const Vec<T, VEC> r = __builtin_bit_cast(
        Vec<T, VEC>, __builtin_amdgcn_raw_buffer_load_b128(rs, uint32_t(c * int(sizeof(T))), 0, CPOL));
#pragma unroll
    for (int j = 0; j < VEC; ++j) v[i * VEC + j] = c < cols ? to_f32(r.v[j]) : fill;
  }
}

template <typename T, int VEC, int RT, int VALS, int CPOL>
__device__ __forceinline__ void store_row_buf(T* row, int cols, int lane, const float* v) {
  static_assert(VEC * sizeof(T) == 16, "16-byte vectors only");
  constexpr int ITEMS = VALS / VEC;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      row, (short)0, uint32_t(cols) * uint32_t(sizeof(T)), 0x00020000);
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int c = (i * RT + lane) * VEC;
    Vec<T, VEC> r;
#pragma unroll
    for (int j = 0; j < VEC; ++j) r.v[j] = from_f32<T>(v[i * VEC + j]);
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4, r), rs,
                                           uint32_t(c * int(sizeof(T))), 0, CPOL);
  }
}

// 16-byte access at any element boundary (one dwordx4 instruction). Neighbouring lanes share the
// lines, so loads keep the default policy (non-temporal ones: softmax fp16 16384 x 1001 12.0 ->
// 14.6 us, bf16 4096 x 8191 24.4 -> 28.0, bf16 512 x 65535 39.0 -> 35.7); stores are streamed.
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(2)));

__device__ __forceinline__ u32x4 load_any(const void* p) {
  return *static_cast<const u32x4_any*>(p);
}
__device__ __forceinline__ void store_any(void* p, u32x4 v) {
  __builtin_nontemporal_store(v, static_cast<u32x4_any*>(p));
}

// Elements s .. of a 16-byte vector moved to its front (0 <= s < its length; zeros behind).
template <int ES>
__device__ __forceinline__ u32x4 drop_elements(u32x4 v, int s) {
  const int words = s * ES / 4;
  if (words & 2) v = u32x4{v[2], v[3], 0u, 0u};
  if (words & 1) v = u32x4{v[1], v[2], v[3], 0u};
  if constexpr (ES == 2)
    if (s & 1)
      v = u32x4{(v[0] >> 16) | (v[1] << 16), (v[1] >> 16) | (v[2] << 16),
                (v[2] >> 16) | (v[3] << 16), v[3] >> 16};
  return v;
}

// Vector of columns c .. c+VEC-1 of a row of `cols` columns. Every load has its VEC elements in
// the row (near its end it starts at cols - VEC), with no branch around it, so all of a row's
// loads are in flight at once; any_fix then moves the elements to their places and sets what
// lies past the row to `fill` (the storage bits of one element). The row starts at least
// VEC - cols elements after the first one of its tensor.
template <typename T, int VEC>
__device__ __forceinline__ u32x4 any_load(const T* row, int cols, int c) {
  static_assert(VEC * sizeof(T) == 16, "16-byte vectors only");
  return load_any(row + min(c, cols - VEC));
}
// Columns of the vectors that a wave (WAVE) or the row's whole group loads together as its vector
// i. They are uniform, so vectors inside the row skip the work with a scalar branch; waves also
// skip the vectors past it (`end` of a wave: 4097 columns keep one of 16 waves busy with the row's
// end instead of all).
struct Span {
  int begin, end;
};
template <int VEC, int RT, bool WAVE>
__device__ __forceinline__ Span vector_span(int i, int lane) {
  if constexpr (WAVE && RT > 64) {
    const int begin = (i * RT + __builtin_amdgcn_readfirstlane(lane & ~63)) * VEC;
    return {begin, begin + 64 * VEC};
  }
  return {i * RT * VEC, (i + 1) * RT * VEC};
}
template <typename T, int VEC, bool WAVE>
__device__ __forceinline__ u32x4 any_fix(u32x4 v, int cols, int c, Span span, uint32_t fill) {
  if (WAVE && span.begin >= cols) {
    const uint32_t word = sizeof(T) == 4 ? fill : fill | (fill << 16);
    return u32x4{word, word, word, word};
  }
  if (span.end > cols) {
    v = drop_elements<int(sizeof(T))>(v, min(max(c - (cols - VEC), 0), VEC - 1));
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const bool in = c + j < cols;
      if constexpr (sizeof(T) == 4)
        v[j] = in ? v[j] : fill;
      else if (j % 2)
        v[j / 2] = in ? v[j / 2] : (v[j / 2] & 0xffffu) | (fill << 16);
      else
        v[j / 2] = in ? v[j / 2] : (v[j / 2] & 0xffff0000u) | fill;
    }
  }
  return v;
}
template <typename T, int VEC, bool WAVE>
__device__ __forceinline__ void any_store(T* row, int cols, int c, Span span, u32x4 v) {
  if (WAVE && span.begin >= cols) return;
  if (span.end <= cols || c + VEC <= cols) {
    tk::store_any(row + c, v);
  } else {
    const Vec<T, VEC> e = __builtin_bit_cast(Vec<T, VEC>, v);
#pragma unroll
    for (int j = 0; j < VEC - 1; ++j)
      if (c + j < cols) row[c + j] = e.v[j];
  }
}

// Rows at any element boundary through aligned vectors: the row is taken to start `shift`
// elements earlier, at the 16-byte boundary before it, and what lies outside it is set to `fill`
// on loading and not stored. The buffer ends with the dword that holds the row's last element.
// A group must cover cols + VEC - 1 columns (RT * VALS).
template <typename T>
__device__ __forceinline__ int row_shift(const T* row) {
  return static_cast<int>((reinterpret_cast<uintptr_t>(row) & 15) / sizeof(T));
}

template <typename T, int VEC, int RT, int VALS, int CPOL>
__device__ __forceinline__ void load_row_shift(const T* row, int shift, int cols, int lane,
                                               float* v, float fill) {
  static_assert(VEC * sizeof(T) == 16, "16-byte vectors only");
  constexpr int ITEMS = VALS / VEC;
  const int end = shift + cols;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(row - shift), (short)0, (uint32_t(end) * uint32_t(sizeof(T)) + 3) & ~3u,
      0x00020000);
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int c = (i * RT + lane) * VEC;
    const Vec<T, VEC> r = __builtin_bit_cast(
        Vec<T, VEC>, __builtin_amdgcn_raw_buffer_load_b128(rs, uint32_t(c * int(sizeof(T))), 0, CPOL));
#pragma unroll
    for (int j = 0; j < VEC; ++j) v[i * VEC + j] = to_f32(r.v[j]);
  }
  // Only the first vectors and those past the row's end hold anything else (uniform branches).
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    if (i > 0 && (i + 1) * RT * VEC <= end) continue;
    const int c = (i * RT + lane) * VEC;
#pragma unroll
    for (int j = 0; j < VEC; ++j)
      if (c + j < shift || c + j >= end) v[i * VEC + j] = fill;
  }
}

template <typename T, int VEC, int RT, int VALS, int CPOL>
__device__ __forceinline__ void store_row_shift(T* row, int shift, int cols, int lane,
                                                const float* v) {
  constexpr int ITEMS = VALS / VEC;
  const int end = shift + cols;
  T* base = row - shift;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      base, (short)0, uint32_t(end) * uint32_t(sizeof(T)), 0x00020000);
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int c = (i * RT + lane) * VEC;
    Vec<T, VEC> r;
#pragma unroll
    for (int j = 0; j < VEC; ++j) r.v[j] = from_f32<T>(v[i * VEC + j]);
    if ((i > 0 && (i + 1) * RT * VEC <= end) || (c >= shift && c + VEC <= end)) {
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4, r), rs,
                                             uint32_t(c * int(sizeof(T))), 0, CPOL);
    } else {
#pragma unroll
      for (int j = 0; j < VEC; ++j)
        if (c + j >= shift && c + j < end) base[c + j] = r.v[j];
    }
  }
}

// load_row and store_row with 16-byte vectors at any element boundary; fill is -inf or 0. The widest
// shape is never half empty, and its 16 vectors' checks delay a single row (f32 1 x 65535 10.2 -> 11.4 us).
template <int RT, int VALS>
constexpr bool kRowWaves = RT < 1024 || VALS < 64;

template <typename T, int VEC, int RT, int VALS>
__device__ __forceinline__ void load_row_any(const T* row, int cols, int lane, float* v,
                                             float fill) {
  constexpr int ITEMS = VALS / VEC;
  const T f = from_f32<T>(fill);
  uint32_t bits;
  if constexpr (sizeof(T) == 4)
    bits = __builtin_bit_cast(uint32_t, f);
  else
    bits = __builtin_bit_cast(uint16_t, f);
  u32x4 raw[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) raw[i] = any_load<T, VEC>(row, cols, (i * RT + lane) * VEC);
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const Vec<T, VEC> r = __builtin_bit_cast(
        Vec<T, VEC>, any_fix<T, VEC, kRowWaves<RT, VALS>>(
                          raw[i], cols, (i * RT + lane) * VEC,
                          vector_span<VEC, RT, kRowWaves<RT, VALS>>(i, lane), bits));
#pragma unroll
    for (int j = 0; j < VEC; ++j) v[i * VEC + j] = to_f32(r.v[j]);
  }
}

template <typename T, int VEC, int RT, int VALS>
__device__ __forceinline__ void store_row_any(T* row, int cols, int lane, const float* v) {
  constexpr int ITEMS = VALS / VEC;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    Vec<T, VEC> r;
#pragma unroll
    for (int j = 0; j < VEC; ++j) r.v[j] = from_f32<T>(v[i * VEC + j]);
    any_store<T, VEC, kRowWaves<RT, VALS>>(row, cols, (i * RT + lane) * VEC,
                                           vector_span<VEC, RT, kRowWaves<RT, VALS>>(i, lane),
                                           __builtin_bit_cast(u32x4, r));
  }
}

// Column of element e (0 <= e < VALS) held by thread `lane`.
template <int VEC, int RT>
__device__ __forceinline__ int row_column(int e, int lane) {
  return ((e / VEC) * RT + lane) * VEC + (e % VEC);
}

// Bits of one storage element <-> float32.
template <typename T>
__device__ __forceinline__ float bits_to_f32(uint32_t b);
template <>
__device__ __forceinline__ float bits_to_f32<float>(uint32_t b) { return __uint_as_float(b); }
template <>
__device__ __forceinline__ float bits_to_f32<__bf16>(uint32_t b) { return __uint_as_float(b << 16); }
template <>
__device__ __forceinline__ float bits_to_f32<_Float16>(uint32_t b) {
  return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(b)));
}
template <typename T>
__device__ __forceinline__ uint32_t f32_to_bits(float f) {
  if constexpr (sizeof(T) == 4) {
    return __float_as_uint(f);
  } else {
    return __builtin_bit_cast(uint16_t, from_f32<T>(f));
  }
}

// A row held in registers as packed storage words (no float copy): 16-bit
// rows take half the registers of their float32 values. Element e of thread
// `lane` is column row_column<VEC, RT>(e, lane).
template <typename T, int VEC, int RT, int VALS>
struct RawRow {
  static constexpr int ITEMS = VALS / VEC;
  static constexpr int PER_WORD = 4 / int(sizeof(T));  // elements per 32-bit word
  static constexpr int WORDS_PER_VEC = (VEC + PER_WORD - 1) / PER_WORD;
  uint32_t w[ITEMS * WORDS_PER_VEC];

  __device__ __forceinline__ void load(const T* __restrict__ row, int cols, int lane) {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const int c = (i * RT + lane) * VEC;
      uint32_t* dst = w + i * WORDS_PER_VEC;
      if constexpr (VEC * sizeof(T) == 16) {
        const uint4 u = c < cols ? *reinterpret_cast<const uint4*>(row + c) : make_uint4(0, 0, 0, 0);
        dst[0] = u.x;
        dst[1] = u.y;
        dst[2] = u.z;
        dst[3] = u.w;
      } else {
        static_assert(VEC == 1, "scalar fallback");
        dst[0] = c < cols ? f32_to_bits<T>(to_f32(row[c])) : 0u;
      }
    }
  }
  // Branch-free 16-byte variants through a buffer resource whose extent is the row
  // (columns past `cols` read as zero and are not written), with cache policy CPOL
  // (kCpol*). `row` must be the same for every lane of a wave: a divergent base
  // makes the compiler wrap each access in a readfirstlane loop.
  template <int CPOL>
  __device__ __forceinline__ void load_buf(const T* row, int cols, int lane) {
    static_assert(VEC * sizeof(T) == 16, "16-byte vectors only");
    const __amdgpu_buffer_rsrc_t rs = row_rsrc(row, cols);
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const u32x4 u = __builtin_bit_cast(
          u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, byte_offset(i, lane), 0, CPOL));
#pragma unroll
      for (int j = 0; j < 4; ++j) w[i * 4 + j] = u[j];
    }
  }
  template <int CPOL>
  __device__ __forceinline__ void store_buf(T* row, int cols, int lane) const {
    static_assert(VEC * sizeof(T) == 16, "16-byte vectors only");
    const __amdgpu_buffer_rsrc_t rs = row_rsrc(row, cols);
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const u32x4 u = {w[i * 4 + 0], w[i * 4 + 1], w[i * 4 + 2], w[i * 4 + 3]};
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4, u), rs, byte_offset(i, lane),
                                             0, CPOL);
    }
  }
  __device__ __forceinline__ static __amdgpu_buffer_rsrc_t row_rsrc(const T* row, int cols) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(row), (short)0,
                                             uint32_t(cols) * uint32_t(sizeof(T)), 0x00020000);
  }
  __device__ __forceinline__ static uint32_t byte_offset(int i, int lane) {
    return uint32_t((i * RT + lane) * VEC * int(sizeof(T)));
  }

  // 16-byte variants at any element boundary: load_any issues the loads (of any row with at
  // least VEC columns), fix_any puts the elements in place and zeroes what lies past the row.
  // SKIP: waves load no vectors past the row (a branch around each load, which costs a software
  // pipeline more than it saves).
  template <bool SKIP>
  __device__ __forceinline__ void load_any(const T* row, int cols, int lane) {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      u32x4 u = {0u, 0u, 0u, 0u};
      if (!SKIP || vector_span<VEC, RT, true>(i, lane).begin < cols)
        u = any_load<T, VEC>(row, cols, (i * RT + lane) * VEC);
#pragma unroll
      for (int j = 0; j < 4; ++j) w[i * 4 + j] = u[j];
    }
  }
  template <bool WAVE>
  __device__ __forceinline__ void fix_any(int cols, int lane) {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      u32x4 u = {w[i * 4 + 0], w[i * 4 + 1], w[i * 4 + 2], w[i * 4 + 3]};
      u = any_fix<T, VEC, WAVE>(u, cols, (i * RT + lane) * VEC, vector_span<VEC, RT, WAVE>(i, lane), 0u);
#pragma unroll
      for (int j = 0; j < 4; ++j) w[i * 4 + j] = u[j];
    }
  }
  template <bool WAVE>
  __device__ __forceinline__ void store_any(T* row, int cols, int lane) const {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const u32x4 u = {w[i * 4 + 0], w[i * 4 + 1], w[i * 4 + 2], w[i * 4 + 3]};
      any_store<T, VEC, WAVE>(row, cols, (i * RT + lane) * VEC, vector_span<VEC, RT, WAVE>(i, lane), u);
    }
  }

  __device__ __forceinline__ void store(T* __restrict__ row, int cols, int lane) const {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const int c = (i * RT + lane) * VEC;
      if (c >= cols) continue;
      const uint32_t* src = w + i * WORDS_PER_VEC;
      if constexpr (VEC * sizeof(T) == 16) {
        *reinterpret_cast<uint4*>(row + c) = make_uint4(src[0], src[1], src[2], src[3]);
      } else {
        row[c] = from_f32<T>(bits_to_f32<T>(src[0]));
      }
    }
  }
  __device__ __forceinline__ uint32_t bits(int e) const {
    if constexpr (VEC == 1 || PER_WORD == 1) {
      return w[e];
    } else {
      const uint32_t word = w[e / PER_WORD];
      return (e & 1) ? (word >> 16) : (word & 0xffffu);
    }
  }
  __device__ __forceinline__ float get(int e) const { return bits_to_f32<T>(bits(e)); }
  __device__ __forceinline__ void set(int e, float f) {
    const uint32_t b = f32_to_bits<T>(f);
    if constexpr (VEC == 1 || PER_WORD == 1) {
      w[e] = b;
    } else {
      uint32_t& word = w[e / PER_WORD];
      word = (e & 1) ? ((word & 0xffffu) | (b << 16)) : ((word & 0xffff0000u) | b);
    }
  }
};

// Launch shape for a row width: RT threads per row, VALS elements per thread.
struct RowShape {
  int rt;
  int vals;
};

// Smallest thread group (64, 256 or 1024 threads) that covers `cols` with at
// most `max_vals` register-resident elements per thread (VALS in {16, 32, 64}).
// Returns false when the row is wider than 1024 * max_vals.
inline bool pick_row_shape(int64_t cols, RowShape* shape, int max_vals = 64) {
  static const int kThreads[] = {64, 256, 1024};
  static const int kVals[] = {16, 32, 64};
  for (int rt : kThreads) {
    for (int vals : kVals) {
      if (vals <= max_vals && cols <= int64_t(rt) * vals) {
        *shape = {rt, vals};
        return true;
      }
    }
  }
  return false;
}

// How a row kernel accesses its rows.
enum class Access { kScalar, kAny, kShift, kAligned };

// 16-byte vectors wherever a row has one.
inline Access row_access(int dtype, int64_t cols, bool aligned) {
  return aligned                          ? Access::kAligned
         : cols >= 16 / elem_size(dtype) ? Access::kAny
                                          : Access::kScalar;
}

// Rows at any boundary that one vector per lane of a wave covers hold no more than that: with 16
// values per lane, whose other vectors are past the row, bf16 1M x 9 ran the norm in 491 us (now 263, one
// element per access 250), its backward in 1183 (692, 1575), softmax in 325 (189, 206).
inline void narrow_row_shape(int dtype, int64_t cols, Access access, RowShape* shape) {
  const int vec = 16 / elem_size(dtype);
  if (access == Access::kAny && cols <= 64 * vec) *shape = {64, vec};
}

}  // namespace tk

// Expands `__VA_ARGS__` with constexpr VEC and ACCESS bound to `access`.
#define TK_DISPATCH_ACCESS(T, access, ...)                                   \
  if ((access) == tk::Access::kScalar) {                                     \
    constexpr tk::Access ACCESS = tk::Access::kScalar;                       \
    constexpr int VEC = 1;                                                   \
    __VA_ARGS__;                                                             \
  } else if ((access) == tk::Access::kAny) {                                 \
    constexpr tk::Access ACCESS = tk::Access::kAny;                          \
    constexpr int VEC = 16 / int(sizeof(T));                                 \
    __VA_ARGS__;                                                             \
  } else {                                                                   \
    constexpr tk::Access ACCESS = tk::Access::kAligned;                      \
    constexpr int VEC = 16 / int(sizeof(T));                                 \
    __VA_ARGS__;                                                             \
  }

// Expands `__VA_ARGS__` with constexpr VEC, ACCESS, RT and VALS bound to `access` and `shape`
// (scalar rows are narrower than one vector: a single shape).
#define TK_DISPATCH_NORM_ROWS(T, access, shape, ...)                         \
  if ((access) == tk::Access::kScalar) {                                     \
    constexpr tk::Access ACCESS = tk::Access::kScalar;                       \
    constexpr int VEC = 1, RT = 64, VALS = 16;                               \
    __VA_ARGS__;                                                             \
  } else if ((access) == tk::Access::kAny) {                                 \
    constexpr tk::Access ACCESS = tk::Access::kAny;                          \
    constexpr int VEC = 16 / int(sizeof(T));                                 \
    if ((shape).vals < 16) {                                                 \
      constexpr int RT = 64, VALS = VEC;                                     \
      __VA_ARGS__;                                                           \
    } else {                                                                 \
      TK_DISPATCH_ROW_SHAPE(shape, __VA_ARGS__)                              \
    }                                                                        \
  } else {                                                                   \
    constexpr tk::Access ACCESS = tk::Access::kAligned;                      \
    constexpr int VEC = 16 / int(sizeof(T));                                 \
    TK_DISPATCH_ROW_SHAPE(shape, __VA_ARGS__)                                \
  }

// The same with shifted rows of 1024 threads.
#define TK_DISPATCH_ROWS(T, access, shape, ...)                              \
  if ((access) == tk::Access::kShift) {                                      \
    constexpr tk::Access ACCESS = tk::Access::kShift;                        \
    constexpr int VEC = 16 / int(sizeof(T)), RT = 1024;                      \
    if ((shape).vals == 16) { constexpr int VALS = 16; __VA_ARGS__; }        \
    else if ((shape).vals == 32) { constexpr int VALS = 32; __VA_ARGS__; }   \
    else { constexpr int VALS = 64; __VA_ARGS__; }                           \
  } else {                                                                   \
    TK_DISPATCH_NORM_ROWS(T, access, shape, __VA_ARGS__)                     \
  }

// Expands `__VA_ARGS__` with constexpr RT and VALS bound to `shape`.
#define TK_DISPATCH_ROW_SHAPE(shape, ...)                                \
  switch ((shape).rt * 100 + (shape).vals) {                             \
    case 6416: { constexpr int RT = 64, VALS = 16; __VA_ARGS__; break; }      \
    case 6432: { constexpr int RT = 64, VALS = 32; __VA_ARGS__; break; }      \
    case 6464: { constexpr int RT = 64, VALS = 64; __VA_ARGS__; break; }      \
    case 25616: { constexpr int RT = 256, VALS = 16; __VA_ARGS__; break; }    \
    case 25632: { constexpr int RT = 256, VALS = 32; __VA_ARGS__; break; }    \
    case 25664: { constexpr int RT = 256, VALS = 64; __VA_ARGS__; break; }    \
    case 102416: { constexpr int RT = 1024, VALS = 16; __VA_ARGS__; break; }  \
    case 102432: { constexpr int RT = 1024, VALS = 32; __VA_ARGS__; break; }  \
    case 102464: { constexpr int RT = 1024, VALS = 64; __VA_ARGS__; break; }  \
    default: return tk::fail("internal: no row kernel for shape %d/%d", (shape).rt, (shape).vals); \
  }

