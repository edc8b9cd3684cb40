// The standalone int4 packer and unpacker (pack_int4 / unpack_int4,
// core/quantization.py:31-45): signed codes [R, C] <-> bytes [R, ceil(C / 2)],
// element 2j in the low nibble of byte j.
//
// Bound by memory.  A thread turns 16 codes into 8 bytes or back, with one
// 16-byte access on the wide side (four for fp32 codes) at whatever alignment
// its row has: rows of an even number of codes that fill their bytes have no
// gaps, so the whole matrix is one run of codes; otherwise each row is cut by
// itself and its last piece goes code by code.  The byte-at-a-time kernels before
// spent their time on 64-bit divisions and one-byte accesses.  Measured at
// 11008 x 4096 (kernel trace): unpack 64.9 -> 11.9 us (68 MB, 5.7 TB/s); packing
// fp32 codes with the range check 31.8 us (203 MB, 6.4 TB/s), for which a packing
// kernel of 41 us and six torch passes (convert, compare twice, or, any, read)
// took 230 us.

#include "../../include/dscq.h"
#include "common.h"

namespace dscq {
namespace {

constexpr int kThreads = 256;
constexpr int kCodes = 16;  // per thread

typedef uint32_t u32x4_a1 __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t u32x2_a1 __attribute__((ext_vector_type(2), aligned(1)));

// Row and first code of thread i: pieces of kCodes codes, `per` of them a row.
struct Piece {
  int64_t row, c0;
};
__device__ __forceinline__ Piece piece_of(int64_t i, int64_t per, int64_t total) {
  Piece p;
  if (total <= 0xFFFFFFFFll) {  // uniform: a 32-bit division does
    const uint32_t r = (uint32_t)i / (uint32_t)per;
    p.row = r;
    p.c0 = (int64_t)((uint32_t)i - r * (uint32_t)per) * kCodes;
  } else {
    p.row = i / per;
    p.c0 = (i - p.row * per) * kCodes;
  }
  return p;
}

// One code as int8: fp32 codes convert as static_cast<int8_t> does here (to an
// integer, then its low byte).
__device__ __forceinline__ int code_of(const int8_t* p) { return *p; }
__device__ __forceinline__ int to_int8(float f) { return (int8_t)__float2int_rz(f); }
__device__ __forceinline__ int code_of(const float* p) { return to_int8(*p); }

template <typename T, bool CHECK>
__global__ __launch_bounds__(kThreads) void pack_int4_kernel(const T* codes, int64_t R, int64_t C,
                                                             int64_t per, uint8_t* packed,
                                                             int32_t* bad) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x, total = R * per;
  if (i >= total) return;
  const Piece p = piece_of(i, per, total);
  const T* src = codes + p.row * C + p.c0;
  uint8_t* dst = packed + p.row * ((C + 1) / 2) + p.c0 / 2;
  bool out = false;
  if (p.c0 + kCodes <= C) {
    uint32_t w[4];  // 16 int8 codes
    if constexpr (sizeof(T) == 1) {
      const u32x4_a1 v = *reinterpret_cast<const u32x4_a1*>(src);
      w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
      if (CHECK) {
#pragma unroll
        for (int k = 0; k < 4; ++k)  // byte + 8 outside [0, 15]
          out |= ((((w[k] & 0x7F7F7F7Fu) + 0x08080808u) ^ (w[k] & 0x80808080u)) & 0xF0F0F0F0u) != 0;
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const u32x4_a4 v = *reinterpret_cast<const u32x4_a4*>(src + 4 * k);
        const uint32_t f[4] = {v.x, v.y, v.z, v.w};
        w[k] = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const int c = to_int8(__uint_as_float(f[b]));
          if (CHECK) out |= (uint32_t)(c + 8) > 15u;
          w[k] |= (uint32_t)(c & 0xFF) << (8 * b);
        }
      }
    }
    u32x2_a1 o;
    uint32_t h[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint32_t ev = __builtin_amdgcn_perm(w[2 * k + 1], w[2 * k], 0x06040200u);
      const uint32_t od = __builtin_amdgcn_perm(w[2 * k + 1], w[2 * k], 0x07050301u);
      h[k] = (ev & 0x0F0F0F0Fu) | ((od & 0x0F0F0F0Fu) << 4);
    }
    o.x = h[0];
    o.y = h[1];
    *reinterpret_cast<u32x2_a1*>(dst) = o;
  } else {
    for (int64_t c = p.c0; c < C; c += 2) {
      const int lo = code_of(src + (c - p.c0));
      const int hi = c + 1 < C ? code_of(src + (c - p.c0) + 1) : 0;  // odd width: nibble 0
      if (CHECK) out |= (uint32_t)(lo + 8) > 15u || (uint32_t)(hi + 8) > 15u;
      dst[(c - p.c0) / 2] = (uint8_t)((lo & 15) | ((hi & 15) << 4));
    }
  }
  // Every writer stores the same 1.
  if (CHECK && out) *bad = 1;
}

// Four nibbles in the low halves of the bytes of v -> int8: bit 3 fills bits 4-7
// (8 * 32 - 8 * 2 = 0xF0; as one subtraction over the whole word).
__device__ __forceinline__ uint32_t sign_extend4(uint32_t v) {
  const uint32_t s = v & 0x08080808u;
  return v | ((s << 5) - (s << 1));
}

__global__ __launch_bounds__(kThreads) void unpack_int4_kernel(const uint8_t* packed, int64_t R,
                                                               int64_t CB, int64_t width,
                                                               int64_t per, int8_t* codes) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x, total = R * per;
  if (i >= total) return;
  const Piece p = piece_of(i, per, total);
  const uint8_t* src = packed + p.row * CB + p.c0 / 2;
  int8_t* dst = codes + p.row * width + p.c0;
  if (p.c0 + kCodes <= width) {
    const u32x2_a1 v = *reinterpret_cast<const u32x2_a1*>(src);
    const uint32_t w[2] = {v.x, v.y};
    uint32_t o[4];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint32_t lo = sign_extend4(w[k] & 0x0F0F0F0Fu);
      const uint32_t hi = sign_extend4((w[k] >> 4) & 0x0F0F0F0Fu);
      o[2 * k] = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
      o[2 * k + 1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
    }
    u32x4_a1 q;
    q.x = o[0]; q.y = o[1]; q.z = o[2]; q.w = o[3];
    *reinterpret_cast<u32x4_a1*>(dst) = q;
  } else {
    for (int64_t c = 0; p.c0 + c < width; ++c) {
      const int nib = (src[c / 2] >> ((c & 1) * 4)) & 15;
      dst[c] = (int8_t)(nib >= 8 ? nib - 16 : nib);
    }
  }
}

// Pieces a row, and the rows left after rows without gaps are joined into one.
int64_t pieces(int64_t& R, int64_t& C, bool joined, int64_t* per) {
  if (joined) {
    C *= R;
    R = 1;
  }
  *per = (C + kCodes - 1) / kCodes;
  return (R * *per + kThreads - 1) / kThreads;
}

}  // namespace

int pack_int4(const void* codes, bool f32, int64_t R, int64_t C, uint8_t* packed, int32_t* bad,
              hipStream_t stream) {
  if (R == 0 || C == 0) return DSCQ_OK;
  int64_t per;
  const int64_t blocks = pieces(R, C, C % 2 == 0, &per);
  if (blocks > 0x7FFFFFFF) return fail("pack_int4: grid too large");
  const dim3 grid((unsigned)blocks), block(kThreads);
  const int8_t* c8 = static_cast<const int8_t*>(codes);
  const float* cf = static_cast<const float*>(codes);
  if (f32) {
    if (bad)
      launch((pack_int4_kernel<float, true>), grid, block, stream, cf, R, C, per, packed, bad);
    else
      launch((pack_int4_kernel<float, false>), grid, block, stream, cf, R, C, per, packed, bad);
  } else {
    if (bad)
      launch((pack_int4_kernel<int8_t, true>), grid, block, stream, c8, R, C, per, packed, bad);
    else
      launch((pack_int4_kernel<int8_t, false>), grid, block, stream, c8, R, C, per, packed, bad);
  }
  return launch_status("pack_int4_kernel");
}

int unpack_int4(const uint8_t* packed, int64_t R, int64_t CB, int64_t width, int8_t* codes,
                hipStream_t stream) {
  if (R == 0 || width == 0) return DSCQ_OK;
  int64_t per;
  const bool joined = width == 2 * CB;
  const int64_t blocks = pieces(R, width, joined, &per);
  if (blocks > 0x7FFFFFFF) return fail("unpack_int4: grid too large");
  launch(unpack_int4_kernel, dim3((unsigned)blocks), dim3(kThreads), stream, packed, R, CB, width,
         per, codes);
  return launch_status("unpack_int4_kernel");
}

}  // namespace dscq
