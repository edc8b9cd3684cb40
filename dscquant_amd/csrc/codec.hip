// The standalone int4 packer and unpacker (pack_int4 / unpack_int4,
// core/quantization.py:31-45): signed codes [R, C] <-> bytes [R, ceil(C / 2)],
// element 2j in the low nibble of byte j.
//
// Bound by memory.  A thread turns 16 codes into 8 bytes or back, with one
// 16-byte access on the wide side (four for fp32 codes) at whatever alignment
// its row has: rows of an even number of codes that fill their bytes have no
// gaps, so the whole matrix is one run of codes; otherwise each row is cut by
// itself.  The byte-at-a-time kernels before spent their time on 64-bit divisions and one-byte accesses.  Measured at
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
__device__ __forceinline__ int to_int8(int8_t c) { return c; }
__device__ __forceinline__ int to_int8(float f) { return (int8_t)__float2int_rz(f); }

// The first `bytes` (1..8) of a 64-bit value at any address.
typedef uint32_t u32_a1 __attribute__((aligned(1)));
typedef uint16_t u16_a1 __attribute__((aligned(1)));
__device__ __forceinline__ void store_bytes(uint8_t* dst, uint32_t lo, uint32_t hi, int bytes) {
  if (bytes == 8) {
    u32x2_a1 o;
    o.x = lo;
    o.y = hi;
    *reinterpret_cast<u32x2_a1*>(dst) = o;
    return;
  }
  if (bytes & 4) {
    *reinterpret_cast<u32_a1*>(dst) = lo;
    dst += 4;
    lo = hi;
  }
  if (bytes & 2) {
    *reinterpret_cast<u16_a1*>(dst) = (uint16_t)lo;
    dst += 2;
    lo >>= 16;
  }
  if (bytes & 1) *dst = (uint8_t)lo;
}

// Mask of the first n codes' bytes in dword k of sixteen.
__device__ __forceinline__ uint32_t code_mask(int n, int k) {
  const int m = n - 4 * k;
  return m >= 4 ? ~0u : m <= 0 ? 0u : (1u << (8 * m)) - 1u;
}

// A row's last piece (n < 16 codes) reads on into the next row, in one access like any
// other, and drops what is not its own; only where sixteen would leave the matrix does it
// take its codes one by one.  Its bytes go out in halves.  Code by code, in a loop or
// unrolled, such rows were behind the byte-a-thread kernels: 7185 x 43 packed 2.33 us
// there, 3.25 in a loop, 2.43 so; unpacked 2.41 / 3.92 / 2.43; a million rows of 13
// 11.3 / 12.0 / 6.0 and 16.9 / 15.9 / 6.5.
template <typename T, bool CHECK>
__global__ __launch_bounds__(kThreads) void pack_int4_kernel(const T* codes, int64_t R, int64_t C,
                                                             int64_t per, uint8_t* packed,
                                                             int32_t* bad) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x, total = R * per;
  if (i >= total) return;
  const Piece p = piece_of(i, per, total);
  const int64_t at = p.row * C + p.c0;
  const T* src = codes + at;
  uint8_t* dst = packed + p.row * ((C + 1) / 2) + p.c0 / 2;
  const int n = (int)min((int64_t)kCodes, C - p.c0);
  uint32_t w[4];  // 16 int8 codes
  if (at + kCodes <= R * C) {
    if constexpr (sizeof(T) == 1) {
      const u32x4_a1 v = *reinterpret_cast<const u32x4_a1*>(src);
      w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const u32x4_a4 v = *reinterpret_cast<const u32x4_a4*>(src + 4 * k);
        const uint32_t f[4] = {v.x, v.y, v.z, v.w};
        w[k] = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b)
          w[k] |= (uint32_t)(to_int8(__uint_as_float(f[b])) & 0xFF) << (8 * b);
      }
    }
  } else {
    w[0] = w[1] = w[2] = w[3] = 0;
#pragma unroll
    for (int k = 0; k < kCodes; ++k)
      w[k / 4] |= (uint32_t)(to_int8(src[min(k, n - 1)]) & 0xFF) << (8 * (k % 4));
  }
  uint32_t out = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (n < kCodes) w[k] &= code_mask(n, k);  // zero codes: an odd width's last nibble is 0
    if (CHECK)                                // byte + 8 outside [0, 15]
      out |= (((w[k] & 0x7F7F7F7Fu) + 0x08080808u) ^ (w[k] & 0x80808080u)) & 0xF0F0F0F0u;
  }
  uint32_t h[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t ev = __builtin_amdgcn_perm(w[2 * k + 1], w[2 * k], 0x06040200u);
    const uint32_t od = __builtin_amdgcn_perm(w[2 * k + 1], w[2 * k], 0x07050301u);
    h[k] = (ev & 0x0F0F0F0Fu) | ((od & 0x0F0F0F0Fu) << 4);
  }
  store_bytes(dst, h[0], h[1], (n + 1) / 2);
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
  const int64_t at = p.row * CB + p.c0 / 2;
  const uint8_t* src = packed + at;
  uint8_t* dst = reinterpret_cast<uint8_t*>(codes + p.row * width + p.c0);
  const int n = (int)min((int64_t)kCodes, width - p.c0);
  uint32_t w[2];
  if (at + kCodes / 2 <= R * CB) {
    const u32x2_a1 v = *reinterpret_cast<const u32x2_a1*>(src);
    w[0] = v.x;
    w[1] = v.y;
  } else {
    w[0] = w[1] = 0;
#pragma unroll
    for (int k = 0; k < kCodes / 2; ++k)
      w[k / 4] |= (uint32_t)src[min(k, (n - 1) / 2)] << (8 * (k % 4));
  }
  uint32_t o[4];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t lo = sign_extend4(w[k] & 0x0F0F0F0Fu);
    const uint32_t hi = sign_extend4((w[k] >> 4) & 0x0F0F0F0Fu);
    o[2 * k] = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
    o[2 * k + 1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
  }
  if (n == kCodes) {
    u32x4_a1 q;
    q.x = o[0]; q.y = o[1]; q.z = o[2]; q.w = o[3];
    *reinterpret_cast<u32x4_a1*>(dst) = q;
  } else if (n >= 8) {
    store_bytes(dst, o[0], o[1], 8);
    if (n > 8) store_bytes(dst + 8, o[2], o[3], n - 8);
  } else {
    store_bytes(dst, o[0], o[1], n);
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
  if (joined) CB *= R;
  const int64_t blocks = pieces(R, width, joined, &per);
  if (blocks > 0x7FFFFFFF) return fail("unpack_int4: grid too large");
  launch(unpack_int4_kernel, dim3((unsigned)blocks), dim3(kThreads), stream, packed, R, CB, width,
         per, codes);
  return launch_status("unpack_int4_kernel");
}

}  // namespace dscq
