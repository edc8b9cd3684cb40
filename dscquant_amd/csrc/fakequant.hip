// Whole-row codes as floats and fake quantization, with no packing: the forms
// in which core/quantization.py hands codes to torch.
//   codes    weight_codes / activation_codes (core/quantization.py:7-21): float
//            codes [M, K], scales [M] and (activations) float zero-points [M];
//   dequant  quantize_weight / quantize_activation (:23-29): the row quantized
//            and put back on its scale, (code - zero) * scale in fp32 rounded to
//            the row's own type.
// Bit widths 2..8, fp16 / bf16 / fp32 rows, any K and any row alignment.
//
// Bound by memory: a row is read once and its result written once, where codes
// as bytes and torch passes over them (widen, slice copies, subtract, scale,
// narrow) went through memory five to nine times.  Thread t of a row takes the
// 8-element chunks t, t + threads, ... (one 16-byte load and store each for
// 16-bit types, contiguous over the wave); the row stays in registers between
// its reduction and its codes.  Rows of at most 2048 elements take one wave each
// (no barrier), up to 16384 a workgroup, longer ones are walked twice.
// Measured (bf16, 8 bits, kernel trace): weights 4096 x 4096 14.3 us (67 MB, 4.7 TB/s;
// a large copy runs at 5.1), activations 512 x 4096 5.4 us; QuantLinear at 8 bits,
// 512 x 4096 x 4096, 217 -> 72 us a call, of which its kernels (a 27 us dense product
// among them) are 49: the host's two calls and its read of the clips bound it.

#include <algorithm>

#include "../../include/dscq.h"
#include "common.h"
#include "mma_int4.h"
#include "rowquant.h"

namespace dscq {
namespace {

constexpr int kBlock = 256;

struct FakeArgs {
  const void* x;   // [M, K] T
  int64_t M;
  int K;
  float clip, qmax;
  void* out;       // DEQ: T [M, K]; else float codes [M, K]
  float* scales;   // [M] (codes form)
  float* zeros;    // [M] (codes form, activations) or null
};

// Eight results from element e0 of an output row: whole chunks as 16-byte
// stores at the element's alignment, the row's last chunk element by element.
template <typename O>
__device__ __forceinline__ void store_row8(O* row, int e0, int K, const float r[8]) {
  if (e0 + 8 <= K) {
    using u32x4 = u32x4_of<O>;
    u32x4* p = reinterpret_cast<u32x4*>(row + e0);
    if constexpr (sizeof(O) == 2) {
      u32x4 w;
      w.x = pack_pair<O>(r[0], r[1]);
      w.y = pack_pair<O>(r[2], r[3]);
      w.z = pack_pair<O>(r[4], r[5]);
      w.w = pack_pair<O>(r[6], r[7]);
      *p = w;
    } else {
      u32x4 a, b;
      a.x = __float_as_uint(r[0]); a.y = __float_as_uint(r[1]);
      a.z = __float_as_uint(r[2]); a.w = __float_as_uint(r[3]);
      b.x = __float_as_uint(r[4]); b.y = __float_as_uint(r[5]);
      b.z = __float_as_uint(r[6]); b.w = __float_as_uint(r[7]);
      p[0] = a;
      p[1] = b;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (e0 + i < K) row[e0 + i] = to_out<O>(r[i]);
  }
}

// One chunk (T in registers, zeros past the row) to its results.
template <int MODE, bool DEQ>
__device__ __forceinline__ void chunk_results(const float v[8], const RowScale& rs, float r[8]) {
  if constexpr (MODE == kAct) {
    uint32_t ev, od;
    float dmax = 0.0f;
    act_chunk_fast(v, rs, ev, od, dmax);
    if (dmax >= rs.thr) {
      asm volatile("" ::: "memory");  // keeps the divisions behind the branch
      act_chunk_exact(v, rs, 1.0f, ev, od);
    }
    const float zero = (float)(int)rs.zf;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float q = (float)((((i & 1) ? od : ev) >> (8 * (i >> 1))) & 0xFFu);
      r[i] = DEQ ? (q - zero) * rs.scale : q;
    }
  } else {
    wgt_levels(v, rs, rs.scale, r);
    const float z = rs.qmax + 1.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = DEQ ? (r[i] - z) * rs.scale : r[i] - z;
  }
}

template <typename T>
__device__ __forceinline__ void load_chunk(const T* row, int e0, int K, bool ragged, float v[8]) {
  Raw<T> raw = load_row8<T>(row, e0, K);
  if (ragged) load_row8_fix<T>(raw, e0, K);
  to_f32(raw, v);
}

template <int MODE>
__device__ __forceinline__ void chunk_minmax(const float v[8], float& mn, float& mx) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if (MODE == kAct) {
      mn = fminf(mn, v[i]);
      mx = fmaxf(mx, v[i]);
    } else {
      mx = fmaxf(mx, fabsf(v[i]));
    }
  }
}

// CH chunks per thread, WPR waves per row (1, or the workgroup's four); CH = 0:
// rows longer than the registers hold, walked twice.  SMALL: K < 8, element
// loads.
template <typename T, int MODE, bool DEQ, int CH, int WPR, bool SMALL = false>
__global__ __launch_bounds__(kBlock) void fake_quant_kernel(FakeArgs a) {
  constexpr int ROWS = 4 / WPR, TPR = 64 * WPR;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t row = (int64_t)blockIdx.x * ROWS + (WPR == 1 ? wave : 0);
  if (row >= a.M) return;  // WPR == 1 only: whole waves, no barrier below
  const int t = WPR == 1 ? (threadIdx.x & 63) : threadIdx.x;
  const T* x = static_cast<const T*>(a.x) + row * a.K;
  // Whether the last chunk of the wave in step c reaches past the row (uniform).
  auto ragged = [&](int c) { return (c * TPR + (WPR == 1 ? 0 : wave * 64) + 64) * 8 > a.K; };
  float v[CH > 0 ? CH : 1][8];
  float mn = 0.0f, mx = 0.0f;
  if constexpr (SMALL) {
    load_scalar<T>(x, t * 8, a.K, true, v[0]);
    chunk_minmax<MODE>(v[0], mn, mx);
  } else if constexpr (CH > 0) {
    Raw<T> raw[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) raw[c] = load_row8<T>(x, (c * TPR + t) * 8, a.K);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      if (ragged(c)) load_row8_fix<T>(raw[c], (c * TPR + t) * 8, a.K);
      to_f32(raw[c], v[c]);
      chunk_minmax<MODE>(v[c], mn, mx);
    }
  } else {
    for (int c = 0; c * TPR * 8 < a.K; ++c) {
      load_chunk<T>(x, (c * TPR + t) * 8, a.K, ragged(c), v[0]);
      chunk_minmax<MODE>(v[0], mn, mx);
    }
  }
  if (MODE == kAct) mn = wave_min(mn);
  mx = wave_max(mx);
  if constexpr (WPR > 1) {
    __shared__ float red[2][WPR];
    if ((threadIdx.x & 63) == 0) {
      red[0][wave] = mn;
      red[1][wave] = mx;
    }
    __syncthreads();
    mn = fminf(fminf(red[0][0], red[0][1]), fminf(red[0][2], red[0][3]));
    mx = fmaxf(fmaxf(red[1][0], red[1][1]), fmaxf(red[1][2], red[1][3]));
  }
  const RowScale rs = row_scale<MODE>(mn, mx, a.clip, a.qmax);
  using O = typename std::conditional<DEQ, T, float>::type;
  O* out = static_cast<O*>(a.out) + row * a.K;
  float r[8];
  if constexpr (CH > 0) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int e0 = (c * TPR + t) * 8;
      if (e0 >= a.K) continue;
      chunk_results<MODE, DEQ>(v[c], rs, r);
      store_row8<O>(out, e0, a.K, r);
    }
  } else {
    for (int c = 0; c * TPR * 8 < a.K; ++c) {
      const int e0 = (c * TPR + t) * 8;
      if (e0 >= a.K) continue;
      load_chunk<T>(x, e0, a.K, ragged(c), v[0]);
      chunk_results<MODE, DEQ>(v[0], rs, r);
      store_row8<O>(out, e0, a.K, r);
    }
  }
  if (!DEQ && t == 0) {
    a.scales[row] = rs.scale;
    if (MODE == kAct && a.zeros) a.zeros[row] = (float)(int)rs.zf;
  }
}

// Workgroups of one launch: a grid holds fewer than 2^32 threads, so more rows than 2^23
// workgroups of 256 take (8.4 M, four times as many up to 2048 elements each) run in
// several launches.
constexpr int64_t kMaxGrid = 1 << 23;

template <typename T, int MODE, bool DEQ>
int launch_fake_rows(const FakeArgs& a, hipStream_t stream) {
  // Waves per row: one while a row is at most four chunks per lane.
  const bool wide = a.K > 2048;
  const int64_t grid = wide ? a.M : (a.M + 3) / 4;
  const int ch = wide ? (a.K + 2047) / 2048 : (a.K + 511) / 512;
#define DSCQ_FAKE(CH, WPR, ...)                                                               \
  launch((fake_quant_kernel<T, MODE, DEQ, CH, WPR, ##__VA_ARGS__>), dim3((unsigned)grid),     \
         dim3(kBlock), stream, a)
  if (a.K < 8) {
    DSCQ_FAKE(1, 1, true);
  } else if (!wide) {
    if (ch == 1) DSCQ_FAKE(1, 1);
    else if (ch == 2) DSCQ_FAKE(2, 1);
    else DSCQ_FAKE(4, 1);
  } else {
    if (ch == 2) DSCQ_FAKE(2, 4);
    else if (ch <= 4) DSCQ_FAKE(4, 4);
    else if (ch <= 8) DSCQ_FAKE(8, 4);
    else DSCQ_FAKE(0, 4);
  }
#undef DSCQ_FAKE
  return launch_status("fake_quant_kernel");
}

template <typename T, int MODE, bool DEQ>
int launch_fake(const FakeArgs& a, hipStream_t stream) {
  const int64_t step = kMaxGrid * (a.K > 2048 ? 1 : 4);
  if (a.M <= step) return launch_fake_rows<T, MODE, DEQ>(a, stream);
  using O = typename std::conditional<DEQ, T, float>::type;
  // Timing events, if armed, span all the launches.
  const KernelEvents ev = take_kernel_events();
  for (int64_t r = 0; r < a.M; r += step) {
    FakeArgs p = a;
    p.M = std::min(step, a.M - r);
    p.x = static_cast<const T*>(a.x) + r * a.K;
    p.out = static_cast<O*>(a.out) + r * a.K;
    if (a.scales) p.scales = a.scales + r;
    if (a.zeros) p.zeros = a.zeros + r;
    arm_kernel_events({r == 0 ? ev.start : nullptr, r + step >= a.M ? ev.stop : nullptr});
    if (int rc = launch_fake_rows<T, MODE, DEQ>(p, stream)) return rc;
  }
  return DSCQ_OK;
}

template <typename T>
int launch_fake_typed(const FakeArgs& a, bool weight, bool dequant, hipStream_t stream) {
  if (weight)
    return dequant ? launch_fake<T, kWgt, true>(a, stream) : launch_fake<T, kWgt, false>(a, stream);
  return dequant ? launch_fake<T, kAct, true>(a, stream) : launch_fake<T, kAct, false>(a, stream);
}

}  // namespace

int fake_quant(const void* x, int dtype, int64_t M, int64_t K, float clip, float qmax, bool weight,
               bool dequant, void* out, float* scales, float* zeros, hipStream_t stream) {
  FakeArgs a;
  a.x = x;
  a.M = M;
  a.K = (int)K;
  a.clip = clip;
  a.qmax = qmax;
  a.out = out;
  a.scales = scales;
  a.zeros = zeros;
  if (dtype == DSCQ_F16) return launch_fake_typed<__half>(a, weight, dequant, stream);
  if (dtype == DSCQ_BF16) return launch_fake_typed<bf16>(a, weight, dequant, stream);
  return launch_fake_typed<float>(a, weight, dequant, stream);
}

}  // namespace dscq
