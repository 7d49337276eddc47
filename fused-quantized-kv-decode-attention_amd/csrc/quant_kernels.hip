// gfx950 per-token KV quantizers: the on-GPU producers of the int8 / int4 KV
// formats the decode kernels read.
//
// Reference expressions (PyTorch, evaluated in the input's dtype):
//   int8: tests/test_kernels.py:32-34 -- s = max|x| / 127 clamped to >= 1e-8,
//         q = clamp(round(x / s), -127, 127), scales stored as fp16;
//   int4: nb:292-299 -- the same with 7, values packed two per byte, low
//         nibble = even element.
// The kernels reproduce those bytes exactly:
//   * the reference runs them on CUDA tensors, where PyTorch evaluates
//     a / qmax (tensor by Python scalar) as a * fp32(1/qmax), and x / s (tensor
//     by tensor) as a true division;
//   * fp32 input: s = max(a * fp32(1/qmax), 1e-8) and x / s in IEEE fp32
//     (correctly rounded division), round-half-even (v_rndne_f32), clamp,
//     scale = fp16(s);
//   * fp16 input: PyTorch evaluates each fp16 op in fp32 and rounds the result
//     to fp16, so s = fp16(a * fp32(1/qmax)) and every quotient is rounded to
//     fp16 before the round-half-even. A row whose fp16 scale underflows to 0 (max|x|
//     below ~4e-6) would divide by zero in the reference; here x = 0 maps to 0
//     and other x to +-qmax, the reference's clamp of +-inf.
//
// Layout: 16 lanes own one token row (D/16 consecutive elements each); a wave
// covers 4 rows per step, a 256-thread workgroup 16, grid-striding over rows.
// The append forms write a live cache's new K and V tokens in place, at host
// or device positions of contiguous caches, or at slots of paged caches.
// The row maximum is a DPP all-reduce within the 16-lane row. HBM-bound at
// bulk: reads 2 or 4 B per element, writes 1 or 0.5 B per element + 2 B per
// row. At a few microseconds per call the work per row shows: 64-bit divisions
// of the row index stood before each row (now multiply-shift), a row's load
// waited for its slot (now both are in flight), and int codes took a clamp of
// two, a round, a conversion and the shifts and ors of packing per element
// (now v_med3, one add, and byte gathers). K and V of 8190 x 8 bf16 rows, D
// 128, to int8 pages of 16: 14.1 -> 11.5 us (4.4 TB/s); 30000 x 8 fp16 rows to
// int4: 51.1 -> 38.5 us; 60000 x 8 bf16 rows, D 64, to int4: 74.5 -> 51.4 us;
// 800000 fp16 rows, D 128, contiguous int8: 57.4 -> 54.6 us (5.7 TB/s).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "kv_formats.h"
#include "launch.h"

namespace fqkv {

namespace {

template <int CTRL>
__device__ __forceinline__ float dpp_f(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}
// Max over each 16-lane row: quad_perm [1,0,3,2], quad_perm [2,3,0,1],
// row_half_mirror, row_mirror.
__device__ __forceinline__ float row16_max(float x) {
  x = fmaxf(x, dpp_f<0xB1>(x));
  x = fmaxf(x, dpp_f<0x4E>(x));
  x = fmaxf(x, dpp_f<0x141>(x));
  return fmaxf(x, dpp_f<0x140>(x));
}

// Source element types (the public header's FQKV_SRC_* values). bf16 rows
// widen exactly to fp32 and then follow the fp32 expressions.
enum { SRC_F16 = 0, SRC_F32 = 1, SRC_BF16 = 2 };
// the largest fp8 e4m3 value; as QMAX it selects the fp8 codes
constexpr int FP8_MAX = 448;

// A lane's D/16 consecutive elements of a row, as loaded.
template <int SRC, int D>
struct Slice {
  static constexpr int EPL = D / 16;
  static constexpr int WORDS = EPL * (SRC == SRC_F32 ? 4 : 2) / 4;
  uint32_t w[WORDS];

  __device__ __forceinline__ void load(const void* X, int64_t row, int i) {
    const uint8_t* p = (const uint8_t*)X + (row * 16 + i) * (4 * WORDS);
    if constexpr (WORDS == 2) {
      const u2_t v = *(const u2_t*)p;
      w[0] = v.x, w[1] = v.y;
    } else {
#pragma unroll
      for (int k = 0; k < WORDS / 4; ++k) {
        const u4_t v = *(const u4_t*)(p + 16 * k);
        w[4 * k] = v.x, w[4 * k + 1] = v.y, w[4 * k + 2] = v.z, w[4 * k + 3] = v.w;
      }
    }
  }
  __device__ __forceinline__ void values(float (&x)[EPL]) const {
    if constexpr (SRC == SRC_F32) {
#pragma unroll
      for (int e = 0; e < EPL; ++e) x[e] = __builtin_bit_cast(float, w[e]);
    } else {
#pragma unroll
      for (int k = 0; k < EPL / 2; ++k) {
        if constexpr (SRC == SRC_BF16) {
          x[2 * k] = __builtin_bit_cast(float, w[k] << 16);
          x[2 * k + 1] = __builtin_bit_cast(float, w[k] & 0xFFFF0000u);
        } else {
          x[2 * k] = (float)__builtin_bit_cast(_Float16, (uint16_t)w[k]);
          x[2 * k + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[k] >> 16));
        }
      }
    }
  }
};

// Byte 0 of a and byte 0 of b as bytes 0 and 1 (v_perm_b32).
__device__ __forceinline__ uint32_t low_bytes(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x0c0c0400u); }

// Quantize one row, whose 16 lanes hold it as x, into the destination row at
// qrow (D code bytes, or D/2 of packed int4) and its scale at *srow. The
// calling 16 lanes stay active together (the DPP reduction spans them); with
// live == false nothing is written (the pointers may be anything).
template <int SRC, int QMAX, int D>
__device__ __forceinline__ void quantize_row(const Slice<SRC, D>& src, uint8_t* __restrict__ qrow,
                                             _Float16* __restrict__ srow, bool live, int i) {
  // QMAX 448: fp8 e4m3 codes (no counterpart in the reference), always the
  // fp32 expressions: s = max(a * fp32(1/448), 1e-8), code = e4m3 round to
  // nearest even of clamp(x / s, +-448), scale stored as fp16(s)
  constexpr bool FP8 = QMAX == FP8_MAX;
  constexpr bool F16 = SRC == SRC_F16 && !FP8;  // fp16 rounding of the scale and the quotients
  constexpr int EPL = D / 16;  // elements per lane
  float x[EPL];
  src.values(x);
  float a = 0.0f;
#pragma unroll
  for (int e = 0; e < EPL; ++e) a = fmaxf(a, fabsf(x[e]));
  a = row16_max(a);

  float s;          // the divisor, as the reference holds it
  _Float16 s_out;   // the stored scale
  if constexpr (F16) {
    s_out = (_Float16)(a * (1.0f / (float)QMAX));  // fp16 op: fp32 result rounded to fp16
    s = (float)s_out;                      // clamp(min=1e-8) cannot lift an fp16 value
  } else {
    s = fmaxf(a * (1.0f / (float)QMAX), 1e-8f);
    s_out = (_Float16)s;
  }
  // x / s as a true division rounds it, from one division per row: with
  // y = RN(1/s), q = RN(x y) and the exact residual r = x - q s (one FMA),
  // RN(q + r y) = RN(x / s) (Markstein's correction step). Checked against
  // the division for every fp16 x and every fp16 s, and on 1.6e9 random fp32
  // pairs with quotients at and next to the rounding ties; only the sign of
  // a zero quotient can differ, which the integer codes drop.
  const float y = s != 0.0f ? 1.0f / s : 0.0f;
  float quot[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    const float q0 = x[e] * y;
    quot[e] = fmaf(fmaf(-q0, s, x[e]), y, q0);
    if constexpr (F16) quot[e] = (float)(_Float16)quot[e];
  }
  if constexpr (F16) {
    if (s == 0.0f) {
#pragma unroll
      for (int e = 0; e < EPL; ++e) quot[e] = x[e] == 0.0f ? 0.0f : copysignf((float)QMAX, x[e]);
    }
  }
  // the clamp as one v_med3_f32 (a NaN gives -QMAX, as max then min do)
#pragma unroll
  for (int e = 0; e < EPL; ++e) quot[e] = __builtin_amdgcn_fmed3f(quot[e], -(float)QMAX, (float)QMAX);
  if (!live) return;
  uint32_t w[EPL / 4];  // a byte per element
  if constexpr (FP8) {
    // v_cvt_pk_fp8_f32 rounds to nearest even (OCP e4m3; the clamp keeps it
    // in range); two codes per call, into the low or the high half
#pragma unroll
    for (int k = 0; k < EPL / 4; ++k) {
      const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(quot[4 * k], quot[4 * k + 1], 0, false);
      w[k] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(quot[4 * k + 2], quot[4 * k + 3], lo, true);
    }
  } else {
    // Round half to even by adding 1.5 * 2^23: the sum's unit is 1, and its
    // low bits are the integer's two's complement, of which v_perm_b32 gathers
    // the low bytes (rounding after the clamp gives the same integers, whose
    // bounds are integers).
    auto code = [&](int e) { return __builtin_bit_cast(uint32_t, quot[e] + 12582912.0f); };
#pragma unroll
    for (int k = 0; k < EPL / 4; ++k)
      w[k] = low_bytes(code(4 * k), code(4 * k + 1)) | low_bytes(code(4 * k + 2), code(4 * k + 3)) << 16;
  }
  if constexpr (QMAX == 7) {
    // nibbles of bytes 0, 1 and 2, 3 join in bytes 0 and 2
#pragma unroll
    for (int k = 0; k < EPL / 4; ++k) {
      w[k] &= 0x0F0F0F0Fu;
      w[k] |= w[k] >> 4;
    }
    uint8_t* out = qrow + (EPL / 2) * i;
    if constexpr (EPL == 8) {
      *(uint32_t*)out = __builtin_amdgcn_perm(w[1], w[0], 0x06040200u);
    } else {
      *(uint16_t*)out = (uint16_t)__builtin_amdgcn_perm(0u, w[0], 0x0c0c0200u);
    }
  } else {
    uint8_t* out = qrow + EPL * i;
    if constexpr (EPL == 8) {
      *(u2_t*)out = u2_t{w[0], w[1]};
    } else {
      *(uint32_t*)out = w[0];
    }
  }
  if (i == 0) *srow = s_out;
}

// Where the rows go: to(v, row, in, q, s) gives the code and scale address of
// row `row` of tensor v (0 K, 1 V) and returns whether it is written; `in`:
// the row exists.

// Contiguous [rows, D or D/2] codes and [rows] scales.
struct PlainDst {
  uint8_t* q;
  _Float16* s;
  template <int ROWB>
  __device__ __forceinline__ bool to(int, int64_t row, bool in, uint8_t*& qr, _Float16*& sr) const {
    qr = q + row * ROWB;
    sr = s + row;
    return in;
  }
};

// row / d for a wave-uniform choice of method: multiply-shift where every row
// index is below 2^31 (a 64-bit division costs some hundred cycles per row,
// which stood before each row's load or store).
struct RowDiv {
  int64_t d;
  FastDiv fast;
  bool small;
  RowDiv(int64_t rows, int64_t d_)
      : d(d_), fast(make_fastdiv((uint32_t)(d_ < (int64_t(1) << 31) ? d_ : 1))), small(rows < (int64_t(1) << 31)) {}
  // (d <= rows: a row index below 2^31 means a divisor below it)
  __device__ __forceinline__ int64_t operator()(int64_t row) const {
    return small ? (int64_t)fast_div((uint32_t)row, fast) : row / d;
  }
};

// A live cache: K and V rows of `rows` cache rows x n new tokens ([rows, n, D]
// each, contiguous) go to token positions pos .. pos+n-1 of caches laid out
// [rows, cap, D or D/2] with scales [rows, cap]. With pos_of set, the position
// of cache row r is pos_of[r / rows_per_pos] instead, read on the device (so a
// captured graph appends where the cache currently ends); rows whose tokens
// would not fit in [0, cap) are not written.
struct AppendDst {
  uint8_t* q[2];
  _Float16* s[2];
  int64_t n, cap, pos;
  const int32_t* pos_of;
  RowDiv div_n, div_pos;
  template <int ROWB>
  __device__ __forceinline__ bool to(int v, int64_t row, bool in, uint8_t*& qr, _Float16*& sr) const {
    const int64_t r = div_n(row);
    int64_t p = pos;
    bool fits = in;
    if (pos_of && in) {
      p = pos_of[div_pos(r)];
      fits = p >= 0 && p <= cap - n;
    }
    const int64_t dst = fits ? r * cap + p + (row - r * n) : 0;
    qr = q[v] + dst * ROWB;
    sr = s[v] + dst;
    return fits;
  }
};

// Paged serving caches: token t's K and V rows ([tokens, heads, D] each,
// contiguous) go to cache slot slots[t] = page * page_size + offset of paged
// caches addressed by strides (codes in bytes, scales in elements), so
// token-major (NHD) and head-major (HND) pages take the same kernel. A slot
// outside [0, nslots) (a padding token, marked -1) writes nothing.
struct PagedDst {
  uint8_t* q[2];      // K, V codes
  _Float16* s[2];     // K, V scales
  int64_t q_page, q_tok, q_head;  // bytes
  int64_t s_page, s_tok, s_head;  // elements
  int64_t nslots, heads;
  int page_log2;
  const int32_t* slots;
  RowDiv div_heads;
  template <int>
  __device__ __forceinline__ bool to(int v, int64_t row, bool in, uint8_t*& qr, _Float16*& sr) const {
    const int64_t t = div_heads(row);
    const int64_t h = row - t * heads;
    const int64_t slot = in ? (int64_t)slots[t] : -1;
    const bool live = slot >= 0 && slot < nslots;
    const int64_t pg = live ? slot >> page_log2 : 0;
    const int64_t off = live ? slot - (pg << page_log2) : 0;
    qr = q[v] + pg * q_page + off * q_tok + h * q_head;
    sr = s[v] + pg * s_page + off * s_tok + h * s_head;
    return live;
  }
};

// A 256-thread workgroup takes 16 R neighbouring rows of one tensor
// (blockIdx.y) at a time, a 16-lane group R of them 16 apart, whose loads and
// destinations (slots, positions) are all in flight before the first row is
// worked on.
template <int SRC, int QMAX, int D, int R, typename Dst>
__global__ void __launch_bounds__(256) quantize_rows_kernel(const void* __restrict__ Xk, const void* __restrict__ Xv,
                                                            int64_t rows, Dst dst) {
  const int i = threadIdx.x & 15;
  const int v = (int)blockIdx.y;
  const void* X = v ? Xv : Xk;
  for (int64_t base = (int64_t)blockIdx.x * (16 * R); base < rows; base += (int64_t)gridDim.x * (16 * R)) {
    const int64_t row = base + (threadIdx.x >> 4);
    Slice<SRC, D> x[R] = {};
    uint8_t* q[R];
    _Float16* s[R];
    bool live[R];
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (row + 16 * k < rows) x[k].load(X, row + 16 * k, i);
#pragma unroll
    for (int k = 0; k < R; ++k)
      live[k] = dst.template to<QMAX == 7 ? D / 2 : D>(v, row + 16 * k, row + 16 * k < rows, q[k], s[k]);
#pragma unroll
    for (int k = 0; k < R; ++k) quantize_row<SRC, QMAX, D>(x[k], q[k], s[k], live[k], i);
  }
}

template <int SRC, int QMAX, typename Dst>
hipError_t launch_rows(int D, const void* Xk, const void* Xv, int64_t rows, int tensors, const Dst& dst,
                       hipStream_t st) {
  // Rows of 128 bytes (8 per lane) go two at a time once that still gives every
  // CU of the card four workgroups; wider ones keep enough bytes in flight one
  // at a time, and their workgroups then overlap loads with stores better
  // (R = 1 / 2 / 4, us: K and V of 60000 x 8 bf16 rows, D 64, int4 60.8 / 51.4 /
  // 50.8; of 8190 x 8 bf16 rows, D 128, int8 11.5 / 12.7 / 15.2).
  const int R = D == 64 && SRC != SRC_F32 && rows * tensors >= 1024 * 32 ? 2 : 1;
  const int64_t want = (rows + 16 * R - 1) / (16 * R);
  const dim3 grid((unsigned)(want < (1 << 16) ? want : (1 << 16)), (unsigned)tensors);
  auto go = [&](auto d_c, auto r_c) {
    hipLaunchKernelGGL((quantize_rows_kernel<SRC, QMAX, decltype(d_c)::value, decltype(r_c)::value, Dst>), grid,
                       dim3(256), 0, st, Xk, Xv, rows, dst);
    return hipGetLastError();
  };
  using One = std::integral_constant<int, 1>;
  if (D == 128) return go(std::integral_constant<int, 128>(), One());
  if constexpr (SRC != SRC_F32) {
    if (R == 2) return go(std::integral_constant<int, 64>(), std::integral_constant<int, 2>());
  }
  return go(std::integral_constant<int, 64>(), One());
}

}  // namespace

// A launcher templated on <SRC, QMAX> for run-time source type and format.
template <typename Fn>
hipError_t by_src_fmt(int src, int fmt, Fn f) {
  auto q = [&](auto src_c) -> hipError_t {
    if (fmt == KV_I8) return f(src_c, std::integral_constant<int, 127>());
    if (fmt == KV_I4) return f(src_c, std::integral_constant<int, 7>());
    if (fmt == KV_FP8) return f(src_c, std::integral_constant<int, FP8_MAX>());
    return hipErrorInvalidValue;
  };
  switch (src) {
    case SRC_F16: return q(std::integral_constant<int, SRC_F16>());
    case SRC_F32: return q(std::integral_constant<int, SRC_F32>());
    case SRC_BF16: return q(std::integral_constant<int, SRC_BF16>());
  }
  return hipErrorInvalidValue;
}

hipError_t launch_quantize_append(int src, int fmt, int D, const void* Xk, const void* Xv, void* Qk, void* Qv,
                                  void* Sk, void* Sv, int64_t rows, int64_t n, int64_t cap, int64_t pos,
                                  const int32_t* pos_of, int64_t rows_per_pos, hipStream_t st) {
  if (rows < 1 || n < 1 || cap < 1 || n > cap || (D != 64 && D != 128)) return hipErrorInvalidValue;
  if (pos_of ? (rows_per_pos < 1 || rows % rows_per_pos != 0) : (pos < 0 || pos + n > cap))
    return hipErrorInvalidValue;
  const int64_t total = rows * n;
  const AppendDst d{{(uint8_t*)Qk, (uint8_t*)Qv},
                    {(_Float16*)Sk, (_Float16*)Sv},
                    n,
                    cap,
                    pos,
                    pos_of,
                    RowDiv(total, n),
                    RowDiv(rows, pos_of ? rows_per_pos : 1)};
  return by_src_fmt(src, fmt, [&](auto s_c, auto q_c) {
    return launch_rows<decltype(s_c)::value, decltype(q_c)::value>(D, Xk, Xv, total, 2, d, st);
  });
}

hipError_t launch_quantize_pages(int src, int fmt, int D, const void* Xk, const void* Xv, const int32_t* slots,
                                 int64_t tokens, int64_t heads, void* Qk, void* Qv, void* Sk, void* Sv,
                                 int64_t num_pages, int page_log2, int64_t q_page, int64_t q_tok, int64_t q_head,
                                 int64_t s_page, int64_t s_tok, int64_t s_head, hipStream_t st) {
  if (tokens < 1 || heads < 1 || num_pages < 1 || page_log2 < 0 || page_log2 > 30 || (D != 64 && D != 128))
    return hipErrorInvalidValue;
  const int64_t rows = tokens * heads;
  const PagedDst d{{(uint8_t*)Qk, (uint8_t*)Qv},
                   {(_Float16*)Sk, (_Float16*)Sv},
                   q_page,
                   q_tok,
                   q_head,
                   s_page,
                   s_tok,
                   s_head,
                   num_pages << page_log2,
                   heads,
                   page_log2,
                   slots,
                   RowDiv(rows, heads)};
  return by_src_fmt(src, fmt, [&](auto s_c, auto q_c) {
    return launch_rows<decltype(s_c)::value, decltype(q_c)::value>(D, Xk, Xv, rows, 2, d, st);
  });
}

hipError_t launch_quantize(int src, int fmt, int D, const void* X, void* Q, void* S, int64_t tokens,
                           hipStream_t st) {
  if (tokens < 1 || (D != 64 && D != 128)) return hipErrorInvalidValue;
  const PlainDst d{(uint8_t*)Q, (_Float16*)S};
  return by_src_fmt(src, fmt, [&](auto s_c, auto q_c) {
    return launch_rows<decltype(s_c)::value, decltype(q_c)::value>(D, X, nullptr, tokens, 1, d, st);
  });
}

}  // namespace fqkv
