// extern "C" entry points of libdscq (declared in include/dscq.h): argument
// checks with the reference extension's messages (kernel/w4a4.cu:164-225),
// then asynchronous launches on the caller's stream.

#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstring>

#include "../../include/dscq.h"
#include "common.h"
#include "gemm_args.h"

namespace dscq {

int row_quant(const void* x, int dtype, int64_t M, int64_t K, int64_t MP, float clip,
              int mode, float qmax, int rotate_block, uint8_t* packed, uint8_t* codes,
              float* scales, int32_t* zeros, int32_t* sums, hipStream_t stream);
int pack_codes(const uint8_t* codes, uint8_t* packed, int64_t MP, int64_t KP,
               hipStream_t stream);
int silu_mul_quant(const void* gate, const void* up, int64_t ld, int64_t M, int64_t N,
                   int64_t MP, float clip, int rotate_block, uint8_t* packed, float* scales,
                   int32_t* zeros, void* hout, hipStream_t stream);
int pack_int4(const void* codes, bool f32, int64_t R, int64_t C, uint8_t* packed, int32_t* bad,
              hipStream_t stream);
int unpack_int4(const uint8_t* packed, int64_t R, int64_t CB, int64_t width,
                int8_t* codes, hipStream_t stream);
int w4a4_gemm(const uint8_t* a, const uint8_t* b, const float* sx, const int32_t* zx,
              const float* sw, const int32_t* sums, const void* bias, int64_t M,
              int64_t N, int64_t KP, bool decode, OutType out_type, void* out,
              int32_t* raw, hipStream_t stream, int32_t* ws = nullptr, int64_t ws_bytes = 0);
int64_t w4a4_gemm_workspace_bytes(int64_t M, int64_t N, int64_t KP, bool decode);
const char* gemm_kernel_name(int64_t M, int64_t N, int64_t KP, bool gated, bool decode, OutType out,
                             const void* out_ptr, const int32_t* raw, const void* ws,
                             int64_t ws_bytes);
bool gemm_silu_mul_fits(int64_t M, int64_t NH, int64_t KP, const void* h);
int w4a4_gemm_silu_mul(const uint8_t* a, const uint8_t* b_gu, const float* sx,
                       const int32_t* zx, const float* sw, const int32_t* sums,
                       const void* bias, int64_t M, int64_t NH, int64_t KP, void* h,
                       OutType out_type, hipStream_t stream);
int fake_quant(const void* x, int dtype, int64_t M, int64_t K, float clip, float qmax, bool weight,
               bool dequant, void* out, float* scales, float* zeros, hipStream_t stream);
bool linear_decode_fits(int64_t M, int64_t K);
bool gated_decode_fits(int64_t M, int64_t K);
int gated_decode(const void* x, int dtype, int64_t M, int64_t K, float clip, int rotate_block,
                 const uint8_t* b_gu, const float* sw, const int32_t* sums, const void* bias,
                 int64_t NH, void* h, hipStream_t stream);
int linear_decode(const void* x, int dtype, int64_t M, int64_t K, float clip, int rotate_block,
                  const uint8_t* b, const float* sw, const int32_t* sums, const void* bias,
                  int64_t N, OutType out_type, void* out, hipStream_t stream);

namespace {
thread_local char g_last_error[512] = "";
thread_local KernelEvents g_kernel_events = {nullptr, nullptr};
thread_local int g_gemm_kernel = 0;
}  // namespace

int gemm_kernel_preference() { return g_gemm_kernel; }

KernelEvents take_kernel_events() {
  const KernelEvents ev = g_kernel_events;
  g_kernel_events = {nullptr, nullptr};
  return ev;
}

void arm_kernel_events(KernelEvents ev) { g_kernel_events = ev; }

int cu_count() {
  // Per device, filled on first use; concurrent first calls store the same value.
  static std::atomic<int> cached[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n <= 0)
      n = 256;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

int fail(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
  va_end(ap);
  return DSCQ_EINVAL;
}

int launch_status(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) return DSCQ_OK;
  snprintf(g_last_error, sizeof(g_last_error), "%s launch failed: %s", what,
           hipGetErrorString(e));
  return (int)e;
}

namespace {

bool valid_dtype(int t) { return t == DSCQ_F16 || t == DSCQ_F32; }
OutType out_of(int out_fp32) { return out_fp32 ? OutType::kFloat : OutType::kHalf; }

int check_rotation(int rotate_block, int64_t K) {
  if (rotate_block != 0 && rotate_block != 128)
    return fail("rotate_block must be 0 or 128 (got %d)", rotate_block);
  if (rotate_block && K % rotate_block != 0)
    return fail("Rotation needs K to be a multiple of %d (got K=%lld)", rotate_block,
                (long long)K);
  return DSCQ_OK;
}

}  // namespace
}  // namespace dscq

using namespace dscq;

extern "C" {

const char* dscq_last_error(void) { return g_last_error; }

const char* dscq_version(void) { return "dscq 0.2.0 (gfx950)"; }

int dscq_time_next_kernel(void* start, void* stop) {
  g_kernel_events = {static_cast<hipEvent_t>(start), static_cast<hipEvent_t>(stop)};
  return DSCQ_OK;
}

int dscq_set_gemm_kernel(int which) {
  if (which < 0 || which > 4) return fail("set_gemm_kernel: 0 to 4 (got %d)", which);
  const int prev = g_gemm_kernel;
  g_gemm_kernel = which;
  return prev;
}

int dscq_device_supported(void) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return -(int)e;
  hipDeviceProp_t prop;
  e = hipGetDeviceProperties(&prop, dev);
  if (e != hipSuccess) return -(int)e;
  return strncmp(prop.gcnArchName, "gfx950", 6) == 0 ? 1 : 0;
}

int dscq_quantize(const void* x, int x_dtype, int64_t M, int64_t K, float clip, int fused,
                  int rotate_block, uint8_t* packed, float* scales, int32_t* zeros,
                  uint8_t* codes, void* stream) {
  DisarmOnExit disarm;
  // kernel/w4a4.cu:165-168
  if (!valid_dtype(x_dtype)) return fail("Only FP16 and FP32 inputs are supported");
  if (!(M > 0 && M <= 65535 && K > 0 && K <= 1048576))
    return fail("Require 1<=M<=65535 and 1<=K<=1048576");
  if (!(clip >= 0.5f && clip <= 1.0f)) return fail("Activation clip must be in [0.5,1]");
  if (int rc = check_rotation(rotate_block, K)) return rc;
  if (!x || !packed || !scales || !zeros) return fail("quantize: null buffer");
  if (!fused && !codes) return fail("quantize: the unfused path needs a codes buffer");
  const int64_t MP = ceil_to(M, 8), KP = ceil_to(K, 64);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (fused)
    return row_quant(x, x_dtype, M, K, MP, clip, 0, 15.0f, rotate_block, packed, nullptr,
                     scales, zeros, nullptr, s);
  // Two kernels: timing events, if armed, span both.
  const KernelEvents ev = take_kernel_events();
  arm_kernel_events({ev.start, nullptr});
  if (int rc = row_quant(x, x_dtype, M, K, MP, clip, 0, 15.0f, rotate_block, nullptr,
                         codes, scales, zeros, nullptr, s))
    return rc;
  arm_kernel_events({nullptr, ev.stop});
  return pack_codes(codes, packed, MP, KP, s);
}

int dscq_linear_decode(const void* x, int x_dtype, int64_t M, int64_t K, float clip,
                       int rotate_block, const uint8_t* b, const float* sw,
                       const int32_t* sums, const void* bias, int64_t N, int out_fp32,
                       void* out, void* stream) {
  DisarmOnExit disarm;
  if (!valid_dtype(x_dtype)) return fail("Only FP16 and FP32 inputs are supported");
  if (!linear_decode_fits(M, K))
    return fail("linear_decode: M=%lld, K=%lld exceed the fused decode kernel (quantize + "
                "matmul instead)", (long long)M, (long long)K);
  if (!(N > 0 && N <= 0x7FFFFFFFLL)) return fail("Invalid dimensions");
  if (!(clip >= 0.5f && clip <= 1.0f)) return fail("Activation clip must be in [0.5,1]");
  if (int rc = check_rotation(rotate_block, K)) return rc;
  if (!x || !b || !sw || !sums || !out) return fail("linear_decode: null buffer");
  if (reinterpret_cast<uintptr_t>(x) % 16 != 0)
    return fail("linear_decode: x must be 16-byte aligned");
  return linear_decode(x, x_dtype, M, K, clip, rotate_block, b, sw, sums, bias, N,
                       out_of(out_fp32), out, static_cast<hipStream_t>(stream));
}

int dscq_linear_decode_supported(int64_t M, int64_t K) { return linear_decode_fits(M, K) ? 1 : 0; }

int dscq_silu_mul_quantize(const void* gate, const void* up, int64_t ld, int64_t M,
                           int64_t N, float clip, int rotate_block, uint8_t* packed,
                           float* scales, int32_t* zeros, void* h, void* stream) {
  DisarmOnExit disarm;
  if (!(M > 0 && M <= 65535 && N > 0 && N <= 32768))
    return fail("silu_mul_quantize: require 1<=M<=65535 and 1<=N<=32768");
  if (ld < N) return fail("silu_mul_quantize: row stride %lld is below N=%lld", (long long)ld,
                          (long long)N);
  if (!(clip >= 0.5f && clip <= 1.0f)) return fail("Activation clip must be in [0.5,1]");
  if (int rc = check_rotation(rotate_block, N)) return rc;
  if (!gate || !up || !packed || !scales || !zeros) return fail("silu_mul_quantize: null buffer");
  return silu_mul_quant(gate, up, ld, M, N, ceil_to(M, 8), clip, rotate_block, packed, scales,
                        zeros, h, static_cast<hipStream_t>(stream));
}

int dscq_matmul_silu_mul(const uint8_t* a, const uint8_t* b_gu, const float* sx,
                         const int32_t* zx, const float* sw, const int32_t* sums,
                         const void* bias, int64_t M, int64_t N, int64_t KP, void* h,
                         void* stream) {
  DisarmOnExit disarm;
  if (!(M > 0 && M <= 65535)) return fail("matmul_silu_mul: require 1<=M<=65535");
  if (!a || !b_gu || !sx || !zx || !sw || !sums || !h) return fail("matmul_silu_mul: null buffer");
  if (!gemm_silu_mul_fits(M, N, KP, h))
    return fail("matmul_silu_mul: need N %% 64 == 0, KP %% 64 == 0, KP <= 65536, 16-byte "
                "aligned h (M=%lld, N=%lld, KP=%lld)", (long long)M, (long long)N,
                (long long)KP);
  return w4a4_gemm_silu_mul(a, b_gu, sx, zx, sw, sums, bias, M, N, KP, h, OutType::kHalf,
                            static_cast<hipStream_t>(stream));
}

int dscq_activation_codes(const void* x, int x_dtype, int64_t M, int64_t K, float clip,
                          int bits, int rotate_block, uint8_t* codes, float* scales,
                          int32_t* zeros, void* stream) {
  DisarmOnExit disarm;
  if (!valid_dtype(x_dtype)) return fail("Only FP16 and FP32 inputs are supported");
  if (!(M > 0 && M <= 65535 && K > 0 && K <= 1048576))
    return fail("Require 1<=M<=65535 and 1<=K<=1048576");
  if (!(clip > 0.0f && clip <= 1.0f)) return fail("Activation clip must be in (0,1]");
  if (bits < 2 || bits > 8) return fail("bits must be in [2,8] (got %d)", bits);
  if (int rc = check_rotation(rotate_block, K)) return rc;
  if (!x || !codes || !scales || !zeros) return fail("activation_codes: null buffer");
  const int64_t MP = ceil_to(M, 8);
  return row_quant(x, x_dtype, M, K, MP, clip, 0, (float)((1 << bits) - 1), rotate_block,
                   nullptr, codes, scales, zeros, nullptr, static_cast<hipStream_t>(stream));
}

int dscq_pack_weight(const void* w, int w_dtype, int64_t N, int64_t K, float clip,
                     int rotate_block, uint8_t* packed, float* sw, int32_t* sums,
                     int8_t* codes, void* stream) {
  DisarmOnExit disarm;
  if (!valid_dtype(w_dtype)) return fail("Only FP16 and FP32 inputs are supported");
  if (!(N > 0 && N <= 1048576 && K > 0 && K <= 1048576))
    return fail("Require 1<=N<=1048576 and 1<=K<=1048576");
  if (!(clip > 0.0f && clip <= 1.0f)) return fail("Weight clip must be in (0,1]");
  if (int rc = check_rotation(rotate_block, K)) return rc;
  if (!w || !packed || !sw || !sums) return fail("pack_weight: null buffer");
  return row_quant(w, w_dtype, N, K, ceil_to(N, 8), clip, 1, 7.0f, rotate_block, packed,
                   reinterpret_cast<uint8_t*>(codes), sw, nullptr, sums,
                   static_cast<hipStream_t>(stream));
}

int dscq_pack_weight_bf16(const void* w, int64_t N, int64_t K, float clip, int rotate_block,
                          uint8_t* packed, float* sw, int32_t* sums, int8_t* codes, void* stream) {
  DisarmOnExit disarm;
  if (!(N > 0 && N <= 1048576 && K > 0 && K <= 1048576))
    return fail("Require 1<=N<=1048576 and 1<=K<=1048576");
  if (!(clip > 0.0f && clip <= 1.0f)) return fail("Weight clip must be in (0,1]");
  if (int rc = check_rotation(rotate_block, K)) return rc;
  if (!w || !packed || !sw || !sums) return fail("pack_weight: null buffer");
  return row_quant(w, DSCQ_BF16, N, K, ceil_to(N, 8), clip, 1, 7.0f, rotate_block, packed,
                   reinterpret_cast<uint8_t*>(codes), sw, nullptr, sums,
                   static_cast<hipStream_t>(stream));
}

namespace {
// dscq_linear.  bf16 activations and results go through the kernels as they are:
// the layer in bf16 was the fp32 one between two conversions of torch (3001 x 8192
// x 8192 with a bias: 25 us widening, 20 quantize, 183 fp32 GEMM, 23 narrowing; 230
// us a call), now 14.6 + 155 us, 170 a call.
//
// Its workspace: the packed activations, their scales and zero points,
// then what the GEMM's K split takes, each at a 256-byte boundary.
struct LinearSpace {
  int64_t MP, KP, scales, zeros, split, bytes;
};
LinearSpace linear_space(int64_t M, int64_t K, int64_t N) {
  LinearSpace s;
  s.MP = ceil_to(M, 8);
  s.KP = ceil_to(K, 64);
  s.scales = ceil_to(s.MP * s.KP / 2, 256);
  s.zeros = s.scales + ceil_to(4 * s.MP, 256);
  s.split = s.zeros + ceil_to(4 * s.MP, 256);
  s.bytes = s.split + w4a4_gemm_workspace_bytes(M, N, s.KP, M < 8);
  return s;
}
bool linear_dims_ok(int64_t M, int64_t K, int64_t N) {
  return M > 0 && M <= 65535 && K > 0 && K <= 1048576 && N > 0 && N <= 0x7FFFFFFFLL;
}
}  // namespace

int64_t dscq_linear_workspace_bytes(int64_t M, int64_t K, int64_t N) {
  if (!linear_dims_ok(M, K, N)) return fail("Invalid dimensions");
  return linear_decode_fits(M, K) ? 0 : linear_space(M, K, N).bytes;
}

int dscq_linear(const void* x, int dtype, int64_t M, int64_t K, float clip, int rotate_block,
                const uint8_t* b, const float* sw, const int32_t* sums, const void* bias,
                int64_t N, void* out, void* workspace, int64_t workspace_bytes, void* stream) {
  DisarmOnExit disarm;
  if (!valid_dtype(dtype) && dtype != DSCQ_BF16)
    return fail("Only FP16, BF16 and FP32 inputs are supported");
  if (!linear_dims_ok(M, K, N)) return fail("Invalid dimensions");
  if (!(clip >= 0.5f && clip <= 1.0f)) return fail("Activation clip must be in [0.5,1]");
  if (int rc = check_rotation(rotate_block, K)) return rc;
  if (!x || !b || !sw || !sums || !out) return fail("linear: null buffer");
  const OutType ot = dtype == DSCQ_F16    ? OutType::kHalf
                     : dtype == DSCQ_BF16 ? OutType::kBf16
                                          : OutType::kFloat;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (linear_decode_fits(M, K))
    return linear_decode(x, dtype, M, K, clip, rotate_block, b, sw, sums, bias, N, ot, out, s);
  const LinearSpace w = linear_space(M, K, N);
  if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < w.bytes)
    return fail("linear: needs a 16-byte aligned workspace of %lld bytes", (long long)w.bytes);
  uint8_t* const base = static_cast<uint8_t*>(workspace);
  float* const sx = reinterpret_cast<float*>(base + w.scales);
  int32_t* const zx = reinterpret_cast<int32_t*>(base + w.zeros);
  // Two launches or more: timing events, if armed, span them all.
  const KernelEvents ev = take_kernel_events();
  arm_kernel_events({ev.start, nullptr});
  if (int rc = row_quant(x, dtype, M, K, w.MP, clip, 0, 15.0f, rotate_block, base, nullptr, sx, zx,
                         nullptr, s))
    return rc;
  arm_kernel_events({nullptr, ev.stop});
  const int64_t split = w.bytes - w.split;
  return w4a4_gemm(base, b, sx, zx, sw, sums, bias, M, N, w.KP, M < 8, ot, out, nullptr, s,
                   split ? reinterpret_cast<int32_t*>(base + w.split) : nullptr, split);
}

namespace {
// dscq_gated_mlp's workspace: the quantized input, h, and what the down projection
// takes as a linear of h (its packed rows, scales, zero points and K split).
struct MlpSpace {
  LinearSpace in, down;
  int64_t h, rest, bytes;
};
MlpSpace mlp_space(int64_t M, int64_t K, int64_t N, int64_t NO) {
  MlpSpace s;
  s.in = linear_space(M, K, 8);
  s.down = linear_space(M, N, NO);
  s.h = s.in.split;
  s.rest = s.h + ceil_to(2 * M * N, 256);
  s.bytes = s.rest + s.down.bytes;
  return s;
}
bool mlp_dims_ok(int64_t M, int64_t K, int64_t N, int64_t NO) {
  return linear_dims_ok(M, K, N) && linear_dims_ok(M, N, NO) &&
         gemm_silu_mul_fits(M, N, ceil_to(K, 64), nullptr);
}
// A few tokens: a product whose workgroups quantize its rows themselves takes one launch
// where quantize and the skinny-M GEMM take two (decode.hip), with the same result.  The
// saved ~4 us shrink with each round of workgroups that repeats the quantization, so
// from three rows it takes a grid of one workgroup (16 outputs) a CU, or a K whose weights
// outlast it.  The block, graph-replayed, weights from HBM, separate / fused gate and up /
// both products fused (us; M, K, N): 1, 4096, 11008 27.4 / - / 17.6; 2 27.4 / 23.7 / -;
// 3 27.5 / 25.1 / -; 4 27.4 / 25.2 / -; 1, 2048, 5632 15.7 / - / 9.8; 1, 4096, 14336 31.2 /
// 25.3 / -; 4 31.4 / 29.8 / -; 4, 4096, 4096 16.8 / - / 12.9 (the down product alone 14.9);
// 4, 1024, 4096 12.3 / - / 9.9 (11.0).  Not fused: 4, 2048, 5632 15.8 / 16.0; 8, 2048, 14336
// 26.4 / 27.8; 8, 1024, 4096 12.4 / 12.3.
bool mlp_fuses_gate_up(int64_t M, int64_t K, int64_t N) {
  return gated_decode_fits(M, K) && (M <= 2 || (M <= 4 && (N <= 16 * cu_count() || K >= 3072)));
}
}  // namespace

int64_t dscq_gated_mlp_workspace_bytes(int64_t M, int64_t K, int64_t N, int64_t NO) {
  if (!mlp_dims_ok(M, K, N, NO)) return fail("Invalid dimensions");
  return mlp_space(M, K, N, NO).bytes;
}

int dscq_gated_mlp(const void* x, int dtype, int64_t M, int64_t K, float clip, int rotate_block,
                   const uint8_t* b_gu, const float* sw_gu, const int32_t* sums_gu,
                   const void* bias_gu, int64_t N, float clip_down, int rotate_down,
                   const uint8_t* b_down, const float* sw_down, const int32_t* sums_down,
                   const void* bias_down, int64_t NO, void* out, void* workspace,
                   int64_t workspace_bytes, void* stream) {
  DisarmOnExit disarm;
  if (dtype != DSCQ_F16 && dtype != DSCQ_BF16)
    return fail("Only FP16 and BF16 inputs are supported");
  if (!mlp_dims_ok(M, K, N, NO)) return fail("Invalid dimensions");
  if (!(clip >= 0.5f && clip <= 1.0f && clip_down >= 0.5f && clip_down <= 1.0f))
    return fail("Activation clip must be in [0.5,1]");
  if (int rc = check_rotation(rotate_block, K)) return rc;
  if (int rc = check_rotation(rotate_down, N)) return rc;
  if (!x || !b_gu || !sw_gu || !sums_gu || !b_down || !sw_down || !sums_down || !out)
    return fail("gated_mlp: null buffer");
  const MlpSpace w = mlp_space(M, K, N, NO);
  if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < w.bytes)
    return fail("gated_mlp: needs a 16-byte aligned workspace of %lld bytes", (long long)w.bytes);
  const OutType ot = dtype == DSCQ_F16 ? OutType::kHalf : OutType::kBf16;
  hipStream_t s = static_cast<hipStream_t>(stream);
  uint8_t* const base = static_cast<uint8_t*>(workspace);
  float* const sx = reinterpret_cast<float*>(base + w.in.scales);
  int32_t* const zx = reinterpret_cast<int32_t*>(base + w.in.zeros);
  uint8_t* const ph = base + w.rest;
  float* const sh = reinterpret_cast<float*>(ph + w.down.scales);
  int32_t* const zh = reinterpret_cast<int32_t*>(ph + w.down.zeros);
  void* const h = base + w.h;
  const bool fuse_in = mlp_fuses_gate_up(M, K, N), fuse_down = M <= 4 && linear_decode_fits(M, N);
  // Two launches or more: timing events, if armed, span them all.
  const KernelEvents ev = take_kernel_events();
  arm_kernel_events({ev.start, nullptr});
  if (fuse_in) {
    if (int rc = gated_decode(x, dtype, M, K, clip, rotate_block, b_gu, sw_gu, sums_gu, bias_gu, N,
                              h, s))
      return rc;
  } else {
    if (int rc = row_quant(x, dtype, M, K, w.in.MP, clip, 0, 15.0f, rotate_block, base, nullptr, sx,
                           zx, nullptr, s))
      return rc;
    if (int rc = w4a4_gemm_silu_mul(base, b_gu, sx, zx, sw_gu, sums_gu, bias_gu, M, N, w.in.KP, h,
                                    ot, s))
      return rc;
  }
  if (fuse_down) {
    arm_kernel_events({nullptr, ev.stop});
    return linear_decode(h, dtype, M, N, clip_down, rotate_down, b_down, sw_down, sums_down,
                         bias_down, NO, ot, out, s);
  }
  if (int rc = row_quant(h, dtype, M, N, w.down.MP, clip_down, 0, 15.0f, rotate_down, ph, nullptr,
                         sh, zh, nullptr, s))
    return rc;
  arm_kernel_events({nullptr, ev.stop});
  const int64_t split = w.down.bytes - w.down.split;
  return w4a4_gemm(ph, b_down, sh, zh, sw_down, sums_down, bias_down, M, NO, w.down.KP, M < 8, ot,
                   out, nullptr, s, split ? reinterpret_cast<int32_t*>(ph + w.down.split) : nullptr,
                   split);
}

int dscq_weight_codes(const void* w, int w_dtype, int64_t N, int64_t K, float clip,
                      int bits, int rotate_block, int8_t* codes, float* scales,
                      void* stream) {
  DisarmOnExit disarm;
  if (!valid_dtype(w_dtype)) return fail("Only FP16 and FP32 inputs are supported");
  if (!(N > 0 && N <= 1048576 && K > 0 && K <= 1048576))
    return fail("Require 1<=N<=1048576 and 1<=K<=1048576");
  if (!(clip > 0.0f && clip <= 1.0f)) return fail("Weight clip must be in (0,1]");
  if (bits < 2 || bits > 8) return fail("bits must be in [2,8] (got %d)", bits);
  if (int rc = check_rotation(rotate_block, K)) return rc;
  if (!w || !codes || !scales) return fail("weight_codes: null buffer");
  return row_quant(w, w_dtype, N, K, ceil_to(N, 8), clip, 1,
                   (float)((1 << (bits - 1)) - 1), rotate_block, nullptr,
                   reinterpret_cast<uint8_t*>(codes), scales, nullptr, nullptr,
                   static_cast<hipStream_t>(stream));
}

namespace {
// Shared checks of dscq_fake_quant and dscq_float_codes: those of
// dscq_activation_codes / dscq_weight_codes, with bf16 rows and no row limit for
// activations.
int check_float_rows(int dtype, int64_t M, int64_t K, float clip, int bits, int weight) {
  if (!valid_dtype(dtype) && dtype != DSCQ_BF16)
    return fail("Only FP16, BF16 and FP32 inputs are supported");
  if (weight) {
    if (!(M > 0 && M <= 1048576 && K > 0 && K <= 1048576))
      return fail("Require 1<=N<=1048576 and 1<=K<=1048576");
    if (!(clip > 0.0f && clip <= 1.0f)) return fail("Weight clip must be in (0,1]");
  } else {
    if (!(M > 0 && K > 0 && K <= 1048576)) return fail("Require M>=1 and 1<=K<=1048576");
    if (!(clip > 0.0f && clip <= 1.0f)) return fail("Activation clip must be in (0,1]");
  }
  if (bits < 2 || bits > 8) return fail("bits must be in [2,8] (got %d)", bits);
  return DSCQ_OK;
}
float float_rows_qmax(int bits, int weight) {
  return (float)(weight ? (1 << (bits - 1)) - 1 : (1 << bits) - 1);
}
}  // namespace

int dscq_fake_quant(const void* x, int dtype, int64_t M, int64_t K, float clip, int bits,
                    int weight, void* out, void* stream) {
  DisarmOnExit disarm;
  if (int rc = check_float_rows(dtype, M, K, clip, bits, weight)) return rc;
  if (!x || !out) return fail("fake_quant: null buffer");
  return fake_quant(x, dtype, M, K, clip, float_rows_qmax(bits, weight), weight != 0, true, out,
                    nullptr, nullptr, static_cast<hipStream_t>(stream));
}

int dscq_float_codes(const void* x, int dtype, int64_t M, int64_t K, float clip, int bits,
                     int weight, float* codes, float* scales, float* zeros, void* stream) {
  DisarmOnExit disarm;
  if (int rc = check_float_rows(dtype, M, K, clip, bits, weight)) return rc;
  if (!x || !codes || !scales || (!weight && !zeros)) return fail("float_codes: null buffer");
  return fake_quant(x, dtype, M, K, clip, float_rows_qmax(bits, weight), weight != 0, false, codes,
                    scales, zeros, static_cast<hipStream_t>(stream));
}

int dscq_matmul(const uint8_t* a, const uint8_t* b, const float* sx, const int32_t* zx,
                const float* sw, const int32_t* sums, const void* bias, int64_t M,
                int64_t N, int64_t KP, int fused, int force_decode, int out_fp32,
                void* out, int32_t* raw, void* stream) {
  DisarmOnExit disarm;
  // kernel/w4a4.cu:197
  if (!(M > 0 && M <= 65535 && N > 0 && KP > 0 && KP <= 1048576 && KP % 64 == 0))
    return fail("Invalid dimensions");
  if (N > 0x7FFFFFFFLL) return fail("Invalid dimensions");
  if (!a || !b || !sx || !zx || !sw || !sums || !out) return fail("matmul: null buffer");
  if (!fused && !raw) return fail("matmul: the unfused path needs a raw buffer");
  // kernel/w4a4.cu:209: the skinny kernel for M < 8 or on request.
  const bool decode = force_decode != 0 || M < 8;
  return w4a4_gemm(a, b, sx, zx, sw, sums, bias, M, N, KP, decode, out_of(out_fp32), out,
                   fused ? nullptr : raw, static_cast<hipStream_t>(stream));
}

int64_t dscq_matmul_workspace_bytes(int64_t M, int64_t N, int64_t KP, int force_decode) {
  if (!(M > 0 && M <= 65535 && N > 0 && N <= 0x7FFFFFFFLL && KP > 0 && KP <= 1048576 &&
        KP % 64 == 0))
    return fail("Invalid dimensions");
  return w4a4_gemm_workspace_bytes(M, N, KP, force_decode != 0 || M < 8);
}

int dscq_matmul_ws(const uint8_t* a, const uint8_t* b, const float* sx, const int32_t* zx,
                   const float* sw, const int32_t* sums, const void* bias, int64_t M,
                   int64_t N, int64_t KP, int fused, int force_decode, int out_fp32,
                   void* out, int32_t* raw, void* workspace, int64_t workspace_bytes,
                   void* stream) {
  DisarmOnExit disarm;
  if (!(M > 0 && M <= 65535 && N > 0 && KP > 0 && KP <= 1048576 && KP % 64 == 0))
    return fail("Invalid dimensions");
  if (N > 0x7FFFFFFFLL) return fail("Invalid dimensions");
  if (!a || !b || !sx || !zx || !sw || !sums || !out) return fail("matmul: null buffer");
  if (!fused && !raw) return fail("matmul: the unfused path needs a raw buffer");
  if (workspace_bytes < 0) return fail("matmul: negative workspace size");
  const bool decode = force_decode != 0 || M < 8;
  return w4a4_gemm(a, b, sx, zx, sw, sums, bias, M, N, KP, decode, out_of(out_fp32), out,
                   fused ? nullptr : raw, static_cast<hipStream_t>(stream),
                   static_cast<int32_t*>(workspace), workspace_bytes);
}

const char* dscq_matmul_kernel(int64_t M, int64_t N, int64_t KP, int gated, int force_decode,
                               int out_dtype, const void* out, const int32_t* raw,
                               const void* workspace, int64_t workspace_bytes) {
  const bool ok = M > 0 && M <= 65535 && N > 0 && KP > 0 && KP <= 1048576 && KP % 64 == 0 &&
                  N <= 0x7FFFFFFFLL && (valid_dtype(out_dtype) || out_dtype == DSCQ_BF16);
  if (!ok || (gated && !gemm_silu_mul_fits(M, N, KP, out))) {
    fail("Invalid dimensions");
    return nullptr;
  }
  const OutType ot = out_dtype == DSCQ_F16    ? OutType::kHalf
                     : out_dtype == DSCQ_BF16 ? OutType::kBf16
                                              : OutType::kFloat;
  return gemm_kernel_name(M, N, KP, gated != 0, force_decode != 0 || M < 8, ot, out, raw, workspace,
                          workspace_bytes);
}

int dscq_pack_int4(const int8_t* codes, int64_t R, int64_t C, uint8_t* packed,
                   void* stream) {
  DisarmOnExit disarm;
  if (R < 0 || C < 0) return fail("pack_int4: negative shape");
  if ((R && C) && (!codes || !packed)) return fail("pack_int4: null buffer");
  return pack_int4(codes, false, R, C, packed, nullptr, static_cast<hipStream_t>(stream));
}

int dscq_pack_int4_checked(const void* codes, int codes_f32, int64_t R, int64_t C, uint8_t* packed,
                           int32_t* out_of_range, void* stream) {
  DisarmOnExit disarm;
  if (R < 0 || C < 0) return fail("pack_int4: negative shape");
  if ((R && C) && (!codes || !packed || !out_of_range)) return fail("pack_int4: null buffer");
  return pack_int4(codes, codes_f32 != 0, R, C, packed, out_of_range,
                   static_cast<hipStream_t>(stream));
}

int dscq_unpack_int4(const uint8_t* packed, int64_t R, int64_t CB, int64_t width,
                     int8_t* codes, void* stream) {
  DisarmOnExit disarm;
  if (R < 0 || CB < 0 || width < 0 || width > 2 * CB)
    return fail("unpack_int4: width must be in [0, 2 * packed columns]");
  if ((R && width) && (!codes || !packed)) return fail("unpack_int4: null buffer");
  return unpack_int4(packed, R, CB, width, codes, static_cast<hipStream_t>(stream));
}

}  // extern "C"
