// Row quantisation of an embedding table to int8 for MI355X (gfx950), as the reference's
// quantize_embedding_int8 (online_best/infer.py:895-901) evaluates on the device:
//   m = max_j |w[r, j]|                 (fp32; exact in any order)
//   s = max(m * RN32(1/127), 1e-8)      (torch divides a device tensor by a Python scalar as a
//                                        multiply by the scalar's fp32 reciprocal; then
//                                        torch.clamp(scale, min=1e-8))
//   q[r, j] = clamp(rint(w[r, j] / s), -128, 127)   (IEEE fp32 division, round half to even)
// Results are bit-identical to that expression for finite tables.
//
// A streaming pass: each element is read once and written once as a byte. Bound by HBM (2M rows of
// 128 bf16: 512 MB read, 264 MB written), so a lane group reads its row as 16-byte vectors, keeps
// it in registers between the maximum and the quantisation, and a wavefront has several rows in
// flight (quantize_rows_kernel). One wavefront per row with 2-byte loads, the row read twice and an
// IEEE division per element took 638 us on that table; this form takes 147 (5.3 TB/s).
#include <stdint.h>

#include "ebag_device.h"
#include "ebag_internal.h"

namespace cti {
namespace {

constexpr int kQuantThreads = 256;
constexpr int kQuantRowsPerBlock = kQuantThreads / kWave;  // wavefronts per workgroup
// Row sets a wavefront of the chunk form has in flight: 4 loads per lane.
constexpr int rows_in_flight(int chunks_per_lane) { return 4 / chunks_per_lane; }

// Any width and alignment: one wavefront per row, the row read twice.
template <typename T>
__global__ void __launch_bounds__(kQuantThreads) quantize_rows_loop_kernel(const char* w, int64_t rows, int64_t dim,
                                                                       int64_t row_stride, int8_t* q, float* scale) {
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kQuantRowsPerBlock + threadIdx.x / kWave;
  if (row >= rows) return;  // uniform over the wavefront
  const int lane = lane_id();
  const char* wr = w + row * row_stride * Elem<T>::kBytes;
  float m = 0.f;
  for (int64_t c = lane; c < dim; c += kWave) m = fmaxf(m, fabsf(Elem<T>::load(wr + c * Elem<T>::kBytes)));
#pragma unroll
  for (int k = 1; k < kWave; k <<= 1) m = fmaxf(m, shfl_xor_f32(m, k));
  float s = m * (1.0f / 127.0f);
  s = s < 1e-8f ? 1e-8f : s;
  if (lane == 0) scale[row] = s;
  int8_t* qr = q + row * dim;
  for (int64_t c = lane; c < dim; c += kWave) {
    float v = rintf(Elem<T>::load(wr + c * Elem<T>::kBytes) / s);
    v = v < -128.f ? -128.f : (v > 127.f ? 127.f : v);
    qr[c] = static_cast<int8_t>(v);
  }
}

// ---------------------------------------------------------------------------------------------
// Rows as chunks of C elements (one load of C * sizeof(T) bytes): a group of 1 << lg lanes holds a
// row, lane l chunks l, l + (1 << lg), ... (K of them); a wavefront quantises 64 >> lg rows side by
// side and kRows such sets at a time, all loads issued before the first is used.
// ---------------------------------------------------------------------------------------------
// C elements of T as loaded (C * sizeof(T) = 2, 4, 8 or 16 bytes).
template <int BYTES>
struct Chunk;
template <>
struct Chunk<2> { typedef uint16_t type; };
template <>
struct Chunk<4> { typedef uint32_t type; };
template <>
struct Chunk<8> { typedef u32x2 type; };
template <>
struct Chunk<16> { typedef u32x4 type; };

template <typename T, int C>
__device__ __forceinline__ void unpack_chunk(const typename Chunk<C * Elem<T>::kBytes>::type& raw, float* v) {
  constexpr int BYTES = C * Elem<T>::kBytes;
  uint4 w = make_uint4(0u, 0u, 0u, 0u);
  if constexpr (BYTES <= 4) w.x = raw;
  else if constexpr (BYTES == 8) w = make_uint4(raw.x, raw.y, 0u, 0u);
  else w = make_uint4(raw.x, raw.y, raw.z, raw.w);
  float t[16 / Elem<T>::kBytes];
  unpack16(w, t, T{});
#pragma unroll
  for (int e = 0; e < C; ++e) v[e] = t[e];
}

// Maximum over each aligned group of 1 << lg lanes, in every lane of the group (m >= 0): lane moves
// inside 16 lanes on the VALU (DPP), across them through LDS.
__device__ __forceinline__ float group_max(float m, int lg) {
  const auto dpp = [](float x, auto ctrl) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  if (lg > 0) m = fmaxf(m, dpp(m, std::integral_constant<int, 0xb1>{}));   // quad_perm: lane ^ 1
  if (lg > 1) m = fmaxf(m, dpp(m, std::integral_constant<int, 0x4e>{}));   // quad_perm: lane ^ 2
  if (lg > 2) m = fmaxf(m, dpp(m, std::integral_constant<int, 0x141>{}));  // row_half_mirror
  if (lg > 3) m = fmaxf(m, dpp(m, std::integral_constant<int, 0x140>{}));  // row_mirror
  if (lg > 4) m = fmaxf(m, shfl_xor_f32(m, 16));
  if (lg > 5) m = fmaxf(m, shfl_xor_f32(m, 32));
  return m;
}

// rint(RN32(v / s)) as a byte for C elements, given inv = RN32(1 / s). |v / s| < 128, so y = v * inv
// is within 128 * 2^-23 of v / s and RN32(v / s) within 128 * 2^-24: together below 2^-15. Where y is
// further than that from a rounding boundary (an integer + 1/2) both round to the same integer, which
// adding 1.5 * 2^23 leaves in the low byte; else (about one element in 16,000, and every NaN) the
// element takes the division.
template <int C>
__device__ __forceinline__ void quantize_chunk(const float* v, float s, float inv, uint32_t* q) {
  constexpr float kMagic = 12582912.f;
  bool sure = true;
#pragma unroll
  for (int e = 0; e < C; ++e) {
    const float y = v[e] * inv;
    const float t = y + kMagic;
    q[e] = __float_as_uint(t) & 0xffu;
    sure = sure && fabsf(y - (t - kMagic)) < 0.5f - 3.0517578125e-5f;  // false for NaN
  }
  if (__builtin_expect(!sure, 0)) {
#pragma unroll
    for (int e = 0; e < C; ++e) {
      float r = rintf(v[e] / s);
      r = r < -128.f ? -128.f : (r > 127.f ? 127.f : r);
      q[e] = static_cast<uint32_t>(static_cast<int32_t>(r)) & 0xffu;
    }
  }
}

template <typename T, int C, int K>
__global__ void __launch_bounds__(kQuantThreads) quantize_rows_kernel(const char* w, int64_t rows, int32_t chunks,
                                                                       int64_t row_bytes, int lg, int8_t* q,
                                                                       float* scale) {
  using V = typename Chunk<C * Elem<T>::kBytes>::type;
  constexpr int kRows = rows_in_flight(K);
  const int lane = lane_id();
  const int g = lane >> lg, sl = lane & ((1 << lg) - 1);
  const int R = kWave >> lg;
  const int64_t wave = static_cast<int64_t>(blockIdx.x) * kQuantRowsPerBlock + threadIdx.x / kWave;
  const int64_t r0 = wave * (R * kRows) + g;
  V raw[kRows][K];
#pragma unroll
  for (int u = 0; u < kRows; ++u) {
    const int64_t row = r0 + u * R;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = (k << lg) + sl;
      raw[u][k] = V{};
      if (row < rows && c < chunks) raw[u][k] = __builtin_nontemporal_load(reinterpret_cast<const V*>(w + row * row_bytes) + c);
    }
  }
#pragma unroll
  for (int u = 0; u < kRows; ++u) {
    const int64_t row = r0 + u * R;
    float v[K][C];
    float m = 0.f;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      unpack_chunk<T, C>(raw[u][k], v[k]);
#pragma unroll
      for (int e = 0; e < C; ++e) m = fmaxf(m, fabsf(v[k][e]));
    }
    m = group_max(m, lg);
    float s = m * (1.0f / 127.0f);
    s = s < 1e-8f ? 1e-8f : s;
    const float inv = 1.0f / s;
    if (row < rows && sl == 0) scale[row] = s;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = (k << lg) + sl;
      uint32_t b[C];
      quantize_chunk<C>(v[k], s, inv, b);
      if (row < rows && c < chunks) {
        int8_t* const dst = q + (row * chunks + c) * C;
        if constexpr (C == 1) {
          *dst = static_cast<int8_t>(b[0]);
        } else if constexpr (C == 2) {
          *reinterpret_cast<uint16_t*>(dst) = static_cast<uint16_t>(b[0] | (b[1] << 8));
        } else {
          uint32_t word[C / 4];
#pragma unroll
          for (int i = 0; i < C / 4; ++i)
            word[i] = b[4 * i] | (b[4 * i + 1] << 8) | (b[4 * i + 2] << 16) | (b[4 * i + 3] << 24);
          if constexpr (C == 4) __builtin_nontemporal_store(word[0], reinterpret_cast<uint32_t*>(dst));
          else __builtin_nontemporal_store(u32x2{word[0], word[1]}, reinterpret_cast<u32x2*>(dst));
        }
      }
    }
  }
}

// Chunks of C elements when the rows, the base pointers and the width allow loads of that size,
// and the row is at most 4 chunks per lane of a wavefront (single elements: 2; 200,000 rows of 129 /
// 191 / 255 bf16 took 62 / 68 / 82 us at 4, the loop kernel 59 / 64 / 79); false: not this form.
template <typename T, int C>
bool launch_chunks(const char* w, int64_t rows, int64_t dim, int64_t row_stride, int8_t* q, float* scale,
                   hipStream_t s) {
  constexpr int BYTES = C * Elem<T>::kBytes;
  if (dim % C != 0 || (row_stride * Elem<T>::kBytes) % BYTES != 0 || reinterpret_cast<uintptr_t>(w) % BYTES != 0 ||
      reinterpret_cast<uintptr_t>(q) % C != 0 || dim / C > (C == 1 ? 2 : 4) * kWave)
    return false;
  const int32_t chunks = static_cast<int32_t>(dim / C);
  const int K = chunks <= kWave ? 1 : (chunks <= 2 * kWave ? 2 : 4);
  int lg = 0;
  while ((K << lg) < chunks) ++lg;
  const int64_t per_block = static_cast<int64_t>(kQuantRowsPerBlock) * (kWave >> lg) * rows_in_flight(K);
  const dim3 grid(static_cast<unsigned>((rows + per_block - 1) / per_block)), block(kQuantThreads);
  const int64_t rb = row_stride * Elem<T>::kBytes;
  if (K == 1) hipLaunchKernelGGL((quantize_rows_kernel<T, C, 1>), grid, block, 0, s, w, rows, chunks, rb, lg, q, scale);
  if (K == 2) hipLaunchKernelGGL((quantize_rows_kernel<T, C, 2>), grid, block, 0, s, w, rows, chunks, rb, lg, q, scale);
  if constexpr (C > 1) {
    if (K == 4) hipLaunchKernelGGL((quantize_rows_kernel<T, C, 4>), grid, block, 0, s, w, rows, chunks, rb, lg, q, scale);
  }
  return true;
}

// The widest chunks that fit; wider rows than they cover take the loop kernel.
template <typename T>
void launch_quantize(const char* w, int64_t rows, int64_t dim, int64_t row_stride, int8_t* q, float* scale,
                     hipStream_t s) {
  constexpr int kMax = 16 / Elem<T>::kBytes;
  if (launch_chunks<T, kMax>(w, rows, dim, row_stride, q, scale, s)) return;
  if (launch_chunks<T, kMax / 2>(w, rows, dim, row_stride, q, scale, s)) return;
  if (launch_chunks<T, kMax / 4>(w, rows, dim, row_stride, q, scale, s)) return;
  if constexpr (kMax == 8) {
    if (launch_chunks<T, 1>(w, rows, dim, row_stride, q, scale, s)) return;
  }
  const dim3 grid(static_cast<unsigned>((rows + kQuantRowsPerBlock - 1) / kQuantRowsPerBlock)), block(kQuantThreads);
  hipLaunchKernelGGL((quantize_rows_loop_kernel<T>), grid, block, 0, s, w, rows, dim, row_stride, q, scale);
}

}  // namespace
}  // namespace cti

using namespace cti;

extern "C" int cti_ebag_quantize_int8(const void* weight, int32_t dtype, int64_t rows, int64_t dim,
                                      int64_t row_stride, int8_t* q, float* scale, void* stream) {
  clear_error();
  if (dtype != CTI_EBAG_F32 && dtype != CTI_EBAG_BF16 && dtype != CTI_EBAG_F16)
    return set_error(CTI_EBAG_EINVAL, "unknown dtype code %d", dtype);
  if (rows < 0) return set_error(CTI_EBAG_EINVAL, "rows must be >= 0 (got %lld)", (long long)rows);
  if (dim < 1) return set_error(CTI_EBAG_EINVAL, "dim must be >= 1 (got %lld)", (long long)dim);
  if (row_stride < dim) return set_error(CTI_EBAG_EINVAL, "row_stride %lld < dim %lld", (long long)row_stride, (long long)dim);
  if (rows == 0) return CTI_EBAG_OK;
  if (!weight || !q || !scale) return set_error(CTI_EBAG_EINVAL, "NULL device pointer among weight/q/scale");
  const int64_t blocks = (rows + kQuantRowsPerBlock - 1) / kQuantRowsPerBlock;
  if (blocks > INT32_MAX) return set_error(CTI_EBAG_EUNSUPPORTED, "too many rows (%lld)", (long long)rows);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const char* w = static_cast<const char*>(weight);
  switch (dtype) {
    case CTI_EBAG_F32: launch_quantize<float>(w, rows, dim, row_stride, q, scale, s); break;
    case CTI_EBAG_BF16: launch_quantize<bf16_t>(w, rows, dim, row_stride, q, scale, s); break;
    default: launch_quantize<f16_t>(w, rows, dim, row_stride, q, scale, s); break;
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(CTI_EBAG_EHIP, "quantize launch failed: %s", hipGetErrorString(e));
  return CTI_EBAG_OK;
}
