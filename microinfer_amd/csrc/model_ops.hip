// Dense ops of the decoder layer around the paged attention path, for decode
// batches on gfx950 (entry points declared in include/mi_model.h).
//
//  * mi_rms_norm_residual: one wave per row, the row held in registers
//    between the sum of squares and the scaling.
//  * mi_silu_mul: one 16-byte vector of gate and of up per thread.
// The projections are in linear.hip.
#include "mi_common.h"
#include "mi_model.h"

namespace mi {
namespace {

// ---------------------------------------------------------------------------
// RMSNorm with the residual sum.
// ---------------------------------------------------------------------------
constexpr int kRowsPerBlock = 4;  // one wave per row
constexpr int kNormMaxDim = 8192;

struct NormArgs {
  const void* x;
  int64_t xs;
  const void* res;
  int64_t rs;
  const void* weight;
  void* out;
  int64_t os;
  void* res_out;
  int64_t ros;
  int32_t rows, dim;
  float eps;
};

// CPL: 8-element chunks per lane (dim <= 512 CPL).
template <typename E, int CPL>
__global__ __launch_bounds__(kRowsPerBlock * kWave) void rms_norm_residual_kernel(
    const NormArgs a) {
  using R = uint16_t;
  const int lane = threadIdx.x % kWave;
  const int row = blockIdx.x * kRowsPerBlock + threadIdx.x / kWave;
  if (row >= a.rows) return;
  const int chunks = a.dim / 8;
  const R* x = static_cast<const R*>(a.x) + row * a.xs;
  const R* res = a.res != nullptr ? static_cast<const R*>(a.res) + row * a.rs : nullptr;
  R* res_out = a.res_out != nullptr ? static_cast<R*>(a.res_out) + row * a.ros : nullptr;
  const R* wt = static_cast<const R*>(a.weight);
  // Every load of the row (x, residual, weight) is issued before the first
  // use, so the row costs one memory round trip.
  Pack<R, 8> s[CPL], w[CPL];
#pragma unroll
  for (int i = 0; i < CPL; ++i) {
    const int c = lane + i * kWave;
    if (c < chunks) w[i] = load_pack<R, 8>(wt + c * 8);
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < CPL; ++i) {
    const int c = lane + i * kWave;
    if (c < chunks) {
      s[i] = load_pack<R, 8>(x + c * 8);
      if (res != nullptr) {
        const Pack<R, 8> r = load_pack<R, 8>(res + c * 8);
#pragma unroll
        for (int j = 0; j < 8; ++j) s[i].v[j] = E::store(E::load(s[i].v[j]) + E::load(r.v[j]));
        if (res_out != nullptr) store_pack<R, 8>(res_out + c * 8, s[i]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float f = E::load(s[i].v[j]);
        ss = fmaf(f, f, ss);
      }
    }
  }
  ss = xor_sum<1, kWave>(ss);
  const float inv = rsqrtf(ss / static_cast<float>(a.dim) + a.eps);
  R* out = static_cast<R*>(a.out) + row * a.os;
#pragma unroll
  for (int i = 0; i < CPL; ++i) {
    const int c = lane + i * kWave;
    if (c < chunks) {
      Pack<R, 8> o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o.v[j] = norm_round<E>(s[i].v[j], inv, w[i].v[j]);
      store_pack<R, 8>(out + c * 8, o);
    }
  }
}

template <typename E>
int32_t launch_norm(const NormArgs& a, hipStream_t stream) {
  const dim3 grid(static_cast<uint32_t>((a.rows + kRowsPerBlock - 1) / kRowsPerBlock));
  const dim3 block(kRowsPerBlock * kWave);
  const int cpl = (a.dim / 8 + kWave - 1) / kWave;
  if (cpl <= 2)
    rms_norm_residual_kernel<E, 2><<<grid, block, 0, stream>>>(a);
  else if (cpl <= 4)
    rms_norm_residual_kernel<E, 4><<<grid, block, 0, stream>>>(a);
  else if (cpl <= 8)
    rms_norm_residual_kernel<E, 8><<<grid, block, 0, stream>>>(a);
  else
    rms_norm_residual_kernel<E, 16><<<grid, block, 0, stream>>>(a);
  return check_launch("mi_rms_norm_residual");
}

// ---------------------------------------------------------------------------
// SwiGLU gate.
// ---------------------------------------------------------------------------
constexpr int kSiluThreads = 256;

template <typename E>
__global__ __launch_bounds__(kSiluThreads) void silu_mul_kernel(const uint16_t* gu, int64_t gs,
                                                                uint16_t* out, int64_t os,
                                                                int32_t rows, int32_t inter) {
  using R = uint16_t;
  const int per_row = inter / 8;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * kSiluThreads + threadIdx.x;
  if (idx >= static_cast<int64_t>(rows) * per_row) return;
  const int r = static_cast<int>(idx / per_row);
  const int c = static_cast<int>(idx % per_row) * 8;
  const Pack<R, 8> g = load_pack<R, 8>(gu + r * gs + c);
  const Pack<R, 8> u = load_pack<R, 8>(gu + r * gs + inter + c);
  Pack<R, 8> o;
#pragma unroll
  for (int j = 0; j < 8; ++j) o.v[j] = silu_mul_round<E>(g.v[j], u.v[j]);
  store_pack<R, 8>(out + r * os + c, o);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
bool half_type(int32_t dtype) { return dtype == MI_DTYPE_BF16 || dtype == MI_DTYPE_F16; }

}  // namespace
}  // namespace mi

extern "C" int32_t mi_rms_norm_residual(const void* x, int64_t x_row_stride,
                                        const void* residual, int64_t residual_row_stride,
                                        const void* weight, float eps, void* out,
                                        int64_t out_row_stride, void* residual_out,
                                        int64_t residual_out_row_stride, int32_t rows,
                                        int32_t dim, int32_t dtype, void* stream) {
  using namespace mi;
  clear_error();
  if (!valid_dtype(dtype)) return fail(MI_ERR_INVALID_ARGUMENT, "mi_rms_norm_residual: bad dtype");
  if (rows < 0 || dim <= 0 || dim % 8)
    return fail(MI_ERR_INVALID_ARGUMENT,
                "mi_rms_norm_residual: need rows >= 0 and dim a positive multiple of 8");
  if (!half_type(dtype))
    return fail(MI_ERR_UNSUPPORTED, "mi_rms_norm_residual: 16-bit types only");
  if (dim > kNormMaxDim) return fail(MI_ERR_UNSUPPORTED, "mi_rms_norm_residual: dim above 8192");
  if (rows == 0) return MI_OK;
  if (!x || !weight || !out)
    return fail(MI_ERR_INVALID_ARGUMENT, "mi_rms_norm_residual: null pointer");
  if (x_row_stride < dim || out_row_stride < dim ||
      (residual && residual_row_stride < dim) ||
      (residual && residual_out && residual_out_row_stride < dim))
    return fail(MI_ERR_INVALID_ARGUMENT, "mi_rms_norm_residual: row strides below dim");
  if (!aligned16(x) || !aligned16(weight) || !aligned16(out) ||
      (residual && !aligned16(residual)) || (residual_out && !aligned16(residual_out)) ||
      x_row_stride % 8 || out_row_stride % 8 || (residual && residual_row_stride % 8) ||
      (residual_out && residual_out_row_stride % 8))
    return fail(MI_ERR_INVALID_ARGUMENT,
                "mi_rms_norm_residual: pointers and row strides must be 16-byte aligned");
  NormArgs a{};
  a.x = x;
  a.xs = x_row_stride;
  a.res = residual;
  a.rs = residual_row_stride;
  a.weight = weight;
  a.out = out;
  a.os = out_row_stride;
  a.res_out = residual ? residual_out : nullptr;
  a.ros = residual_out_row_stride;
  a.rows = rows;
  a.dim = dim;
  a.eps = eps;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == MI_DTYPE_BF16 ? launch_norm<BF16>(a, s) : launch_norm<F16>(a, s);
}

extern "C" int32_t mi_silu_mul(const void* gate_up, int64_t gate_up_row_stride, void* out,
                               int64_t out_row_stride, int32_t rows, int32_t inter,
                               int32_t dtype, void* stream) {
  using namespace mi;
  clear_error();
  if (!valid_dtype(dtype)) return fail(MI_ERR_INVALID_ARGUMENT, "mi_silu_mul: bad dtype");
  if (rows < 0 || inter <= 0 || inter % 8)
    return fail(MI_ERR_INVALID_ARGUMENT,
                "mi_silu_mul: need rows >= 0 and inter a positive multiple of 8");
  if (!half_type(dtype)) return fail(MI_ERR_UNSUPPORTED, "mi_silu_mul: 16-bit types only");
  if (rows == 0) return MI_OK;
  if (!gate_up || !out) return fail(MI_ERR_INVALID_ARGUMENT, "mi_silu_mul: null pointer");
  if (gate_up_row_stride < 2 * static_cast<int64_t>(inter) || out_row_stride < inter)
    return fail(MI_ERR_INVALID_ARGUMENT, "mi_silu_mul: row strides below the row lengths");
  if (!aligned16(gate_up) || !aligned16(out) || gate_up_row_stride % 8 || out_row_stride % 8)
    return fail(MI_ERR_INVALID_ARGUMENT,
                "mi_silu_mul: pointers and row strides must be 16-byte aligned");
  const int64_t threads = static_cast<int64_t>(rows) * (inter / 8);
  const int64_t blocks = (threads + kSiluThreads - 1) / kSiluThreads;
  if (blocks > 0x7fffffff) return fail(MI_ERR_UNSUPPORTED, "mi_silu_mul: too many rows");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const uint16_t* gu = static_cast<const uint16_t*>(gate_up);
  uint16_t* o = static_cast<uint16_t*>(out);
  if (dtype == MI_DTYPE_BF16)
    silu_mul_kernel<BF16><<<static_cast<uint32_t>(blocks), kSiluThreads, 0, s>>>(
        gu, gate_up_row_stride, o, out_row_stride, rows, inter);
  else
    silu_mul_kernel<F16><<<static_cast<uint32_t>(blocks), kSiluThreads, 0, s>>>(
        gu, gate_up_row_stride, o, out_row_stride, rows, inter);
  return check_launch("mi_silu_mul");
}
