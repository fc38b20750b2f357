// The encoder's input LayerNorm followed by its Linear, on the matrix cores of gfx950 (MI355X).
//
// online_best/infer.py:1061-1085 normalises the pooled block [B, 28*D] (Triton kernel :829-858,
// output in the block's dtype) and maps it to d_model with nn.Linear (a library GEMM):
//   a[m, k] = bf16( ((x[m, k] - mean[m]) * rstd[m]) * gamma[k] + beta[k] )
//   y[m, n] = sum_k a[m, k] * w[n, k] + bias[n]              (fp32 accumulation, one rounding)
// Here both run in one kernel: the LayerNorm is applied while the pooled block's tiles are moved
// from HBM to LDS (each element normalised in fp32 as the LayerNorm kernel computes it and
// rounded to bf16 as that kernel stores it), so the normalised block never reaches HBM; the
// per-row mean and rstd come from the pooling or statistics pass (cti_ebag_layernorm with no
// output). Without statistics the kernel is the plain Linear.
//
// Three forms (the products on v_mfma_f32_16x16x32_bf16: lane l supplies A[l%16][8(l/16) .. +8)
// and B[8(l/16) .. +8)[l%16] and receives C[4(l/16) + r][l%16], r < 4), chosen by linear_plan:
//   ln_linear_band_kernel K a multiple of 128: bands of 128 rows by 256, 384 or 512 columns, the
//                         weight loaded straight to LDS;
//   ln_linear_big_kernel  K a multiple of 128: 128 x 256 or 128 x 128 tiles of 8 wavefronts, both
//                         operands through LDS (XOR-swizzled rows);
//   ln_linear_kernel      any K (a multiple of 8): 64 x 256 tiles of 4 wavefronts, each owning 64
//                         columns, x through LDS and the weight's fragments straight to registers.
// The last two walk K in steps of 64 with each step's loads issued two steps ahead into rotating
// register sets, x normalised on its way to LDS, two LDS buffers and one barrier per step, and
// number their workgroups so that the tiles of one row band run on one XCD, whose L2 then serves the
// band to each of them. When the tiles would leave CUs idle (few rows), K is split over several
// workgroups per tile: each writes its fp32 partial products to a caller's workspace and
// ln_linear_reduce_kernel adds the splits in split order, adds the bias and rounds once.
#include <stdint.h>

#include "ebag_device.h"
#include "ebag_internal.h"
#include "ebag_rules.h"

namespace cti {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kBK = kLinearStep;  // K per step
constexpr int kLds = kBK + 8;  // LDS row pitch in elements (144 bytes)
constexpr int kChunks = kBK / 8;  // 16-byte chunks per tile row
constexpr int kXcds = 8;
constexpr int kWaveCols = 64;  // output columns per wavefront

struct LinearParams {
  const char* x;      // [M, K] bf16
  const float* mean;  // [M], NULL: no LayerNorm
  const float* rstd;  // [M]
  const void* gamma;  // [K]
  const void* beta;   // [K]
  const char* w;      // [N, K] bf16
  const void* bias;   // [N] or NULL
  char* y;            // [M, N]
  int64_t M;
  int32_t N;
  int32_t K;
  int32_t tiles_m;
  int32_t tiles_n;
  float* part;          // split K: fp32 partial products [splits, M, N] (no bias), NULL: no split
  int32_t split_steps;  // split K: steps of kBK per split (even); split s is blockIdx.y
  int32_t bias_f32;     // bias is fp32 (else bf16)
  int32_t y_f32;        // y is fp32 (else bf16)
};

// One bf16 chunk (8 elements) normalised: ((x - mean) * rstd) * g + b, rounded to bf16.
__device__ __forceinline__ uint4 normalise8(const uint4& raw, float mean, float rstd, const float* g, const float* b) {
  float v[8];
  unpack16(raw, v, bf16_t{});
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = (v[e] - mean) * rstd * g[e] + b[e];
  return make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]),
                    pack_bf16x2(v[6], v[7]));
}

template <typename OT>
__device__ __forceinline__ void store_y(char* y, int64_t idx, float v) {
  if constexpr (std::is_same<OT, float>::value) reinterpret_cast<float*>(y)[idx] = v;
  else reinterpret_cast<uint16_t*>(y)[idx] = static_cast<uint16_t>(pack_bf16x2(v, 0.f));
}

template <int BM, int WAVES, int U, bool LN, typename PT, typename BT, typename OT>
__global__ void __launch_bounds__(WAVES * kWave) ln_linear_kernel(const LinearParams p) {
  constexpr int THREADS = WAVES * kWave;
  constexpr int BN = WAVES * kWaveCols;
  constexpr int MI = BM / 16, NI = kWaveCols / 16;  // 16 x 16 products per wavefront
  constexpr int PA = BM * kChunks / THREADS;        // x chunks per thread and step
  constexpr int kRowStep = THREADS / kChunks;
  static_assert(PA >= 1 && BM * kChunks % THREADS == 0, "tile shape");
  __shared__ __align__(16) uint16_t sA[2][BM * kLds];

  // XCD-contiguous numbering: dispatch position i runs on XCD i % 8; give each XCD a contiguous
  // range of tiles, column tiles fastest, so a row band's tiles share that XCD's L2.
  const int total = p.tiles_m * p.tiles_n;
  const int i = static_cast<int>(blockIdx.x);
  int tile = i;
  if (total % kXcds == 0) tile = (i % kXcds) * (total / kXcds) + i / kXcds;
  const int64_t m0 = static_cast<int64_t>(tile / p.tiles_n) * BM;
  const int n0 = (tile % p.tiles_n) * BN;

  const int t = static_cast<int>(threadIdx.x);
  const int lane = t & (kWave - 1);
  const int wave = t / kWave;
  const int kc = t % kChunks;  // this thread's chunk of each x row of a step (fixed over K)
  const int r0 = t / kChunks;  // its first row of the band; then every kRowStep rows
  const int fr = lane & 15;        // fragment row (A) / column (B)
  const int fk = (lane >> 4) * 8;  // fragment k offset

  // Every load below reads a valid address (rows past M or N and chunks past K read the last
  // row / chunk) and its value is replaced by zero afterwards: no branch around a load, so the
  // loads of a step issue back to back and retire in order.
  float mean[PA], rstd[PA];
  bool row_ok[PA];
  const char* xrow[PA];
#pragma unroll
  for (int q = 0; q < PA; ++q) {
    const int64_t m = m0 + r0 + q * kRowStep;
    row_ok[q] = m < p.M;
    const int64_t mc = row_ok[q] ? m : p.M - 1;
    mean[q] = 0.f;
    rstd[q] = 1.f;
    if constexpr (LN) {
      mean[q] = p.mean[mc];
      rstd[q] = p.rstd[mc];
    }
    xrow[q] = p.x + mc * p.K * 2;
  }
  // this lane's weight rows (one per 16-column fragment of the wavefront)
  const char* wrow[NI];
  bool col_ok[NI];
#pragma unroll
  for (int c = 0; c < NI; ++c) {
    const int n = n0 + wave * kWaveCols + c * 16 + fr;
    col_ok[c] = n < p.N;
    wrow[c] = p.w + static_cast<int64_t>(col_ok[c] ? n : p.N - 1) * p.K * 2;
  }

  const int nk = (p.K + kBK - 1) / kBK;
  constexpr int PV = LN ? 2 * Elem<PT>::kBytes / 2 : 0;  // 16-byte vectors of gamma + beta per chunk
  // register sets: step s's x chunks (with their gamma / beta) and weight fragments live in set
  // s % U from when they are issued (U steps ahead) until they are used
  uint4 ra[U][PA];
  uint4 rp[U][PV > 0 ? PV : 1];
  bf16x8 wb[U][2][NI];
  const uint4 zero4 = make_uint4(0u, 0u, 0u, 0u);
  auto issue_x = [&](int ks, uint4 (&a)[PA], uint4 (&pp)[PV > 0 ? PV : 1]) {
    const int k = ks * kBK + kc * 8;
    const int kq = k < p.K ? k : p.K - 8;  // steps and chunks past K read the last chunk
#pragma unroll
    for (int q = 0; q < PA; ++q) a[q] = load16(xrow[q] + static_cast<int64_t>(kq) * 2);
    if constexpr (LN) {
      constexpr int H = Elem<PT>::kBytes / 2;  // 16-byte vectors per 8 parameters
#pragma unroll
      for (int h = 0; h < H; ++h) {
        pp[h] = load16(static_cast<const char*>(p.gamma) + static_cast<int64_t>(kq) * Elem<PT>::kBytes + h * 16);
        pp[H + h] = load16(static_cast<const char*>(p.beta) + static_cast<int64_t>(kq) * Elem<PT>::kBytes + h * 16);
      }
    }
  };
  auto issue_w = [&](int ks, bf16x8 (&b)[2][NI]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = ks * kBK + h * 32 + fk;
      const int kq = k < p.K ? k : p.K - 8;
#pragma unroll
      for (int c = 0; c < NI; ++c) b[h][c] = __builtin_bit_cast(bf16x8, load16(wrow[c] + static_cast<int64_t>(kq) * 2));
    }
  };
  // zero the weight fragments past K or N (after their loads have been waited for)
  auto mask_w = [&](int ks, bf16x8 (&b)[2][NI]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bool kin = ks * kBK + h * 32 + fk < p.K;
#pragma unroll
      for (int c = 0; c < NI; ++c)
        if (!(kin && col_ok[c])) b[h][c] = __builtin_bit_cast(bf16x8, zero4);
    }
  };
  auto put_x = [&](int ks, int buf, const uint4 (&a)[PA], const uint4 (&pp)[PV > 0 ? PV : 1]) {
    const bool kin = ks * kBK + kc * 8 < p.K;
    float g[8], bt[8];
    if constexpr (LN) {
      constexpr int H = Elem<PT>::kBytes / 2;
#pragma unroll
      for (int h = 0; h < H; ++h) {
        unpack16(pp[h], g + h * (16 / Elem<PT>::kBytes), PT{});
        unpack16(pp[H + h], bt + h * (16 / Elem<PT>::kBytes), PT{});
      }
    }
#pragma unroll
    for (int q = 0; q < PA; ++q) {
      uint4 v = a[q];
      if constexpr (LN) v = normalise8(a[q], mean[q], rstd[q], g, bt);
      // rows past M and columns past K hold +0 (they must not add beta)
      if (!(row_ok[q] && kin)) v = zero4;
      *reinterpret_cast<uint4*>(&sA[buf][(r0 + q * kRowStep) * kLds + kc * 8]) = v;
    }
  };

  f32x4 acc[MI][NI];
#pragma unroll
  for (int a = 0; a < MI; ++a)
#pragma unroll
    for (int c = 0; c < NI; ++c) acc[a][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int buf, const bf16x8 (&b)[2][NI]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int a = 0; a < MI; ++a) {
        const bf16x8 fa = *reinterpret_cast<const bf16x8*>(&sA[buf][(a * 16 + fr) * kLds + h * 32 + fk]);
#pragma unroll
        for (int c = 0; c < NI; ++c) acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa, b[h][c], acc[a][c], 0, 0, 0);
      }
    }
  };

  // steps walked: nk rounded up to a multiple of U (the steps past nk load valid addresses and
  // multiply zeros), so that the unrolled body below holds no branch: the compiler then knows at
  // every use how many loads were issued after the one it waits for
  const int nks = (nk + U - 1) / U * U;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    issue_x(u, ra[u], rp[u]);
    issue_w(u, wb[u]);
  }
  put_x(0, 0, ra[0], rp[0]);
  issue_x(U, ra[0], rp[0]);
  __syncthreads();
  // iteration s writes step s + 1's x chunks (set (s + 1) % U) into the other LDS buffer and
  // refills that set with step s + 1 + U, multiplies step s (LDS buffer s % 2, weight set s % U)
  // and refills the weight set with step s + U; one barrier per step. The body is unrolled U
  // times so that every register set keeps its registers across the loop.
  for (int s0 = 0; s0 < nks; s0 += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u;
      put_x(s + 1, (s + 1) & 1, ra[(u + 1) % U], rp[(u + 1) % U]);
      issue_x(s + 1 + U, ra[(u + 1) % U], rp[(u + 1) % U]);
      mask_w(s, wb[u]);
      multiply(s & 1, wb[u]);
      issue_w(s + U, wb[u]);
      __syncthreads();
    }
  }

  // epilogue: + bias, one rounding to the output type
#pragma unroll
  for (int c = 0; c < NI; ++c) {
    const int n = n0 + wave * kWaveCols + c * 16 + fr;
    if (n >= p.N) continue;
    const float bn = p.bias ? Elem<BT>::load(static_cast<const char*>(p.bias) + static_cast<int64_t>(n) * Elem<BT>::kBytes)
                            : 0.f;
#pragma unroll
    for (int a = 0; a < MI; ++a) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t m = m0 + a * 16 + (lane >> 4) * 4 + r;
        if (m < p.M) store_y<OT>(p.y, m * p.N + n, acc[a][c][r] + bn);
      }
    }
  }
}

// Raw buffer over a whole array: byte offsets (voffset from the lane, soffset from the step).
typedef __amdgpu_buffer_rsrc_t Rsrc;
__device__ __forceinline__ Rsrc make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), static_cast<short>(0), static_cast<int>(bytes),
                                           0x00020000);  // raw buffer, 32-bit data format
}
__device__ __forceinline__ uint4 bload16(Rsrc r, uint32_t voff, uint32_t soff) {
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
  return make_uint4(v.x, v.y, v.z, v.w);
}

// 16 bytes per lane straight to LDS, lane l's to lds + 16 l (lds the same for every lane).
__device__ __forceinline__ void bload16_lds(Rsrc r, uint4* lds, uint32_t voff, uint32_t soff) {
#ifdef __HIP_DEVICE_COMPILE__  // the host pass has no 16-byte form
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, voff, soff, 0, 0);
#endif
}

// The large form (K a multiple of 128, byte offsets below 2^31): a workgroup of 8 wavefronts
// (2 x 4, each 64 x BN/4) owns a 128 x BN tile of y (BN = 256, or 128 when that leaves fewer
// than two tiles per CU); both
// operands pass through LDS, so each x element loaded feeds BN columns and each weight element
// 128 rows (the L2 -> CU traffic per product that the matrix cores can sustain). x chunks are
// normalised on their way to LDS, once per BN columns. Every load reads inside its array (rows
// past M or N read the last row: their products only reach accumulators that are not stored),
// buffer loads with the step in the scalar offset, U register sets rotating, two LDS buffers, one
// barrier per step, no branch in the loop.
template <int BN, int GN, int U, bool LN, typename PT, typename BT, typename OT>
__global__ void __launch_bounds__(2 * GN * kWave, GN == 2 ? 2 : 1) ln_linear_big_kernel(const LinearParams p) {
  constexpr int BM = 128, THREADS = 2 * GN * kWave;  // 2 x GN wavefronts
  constexpr int WN = BN / GN;                       // wavefront tile 64 x WN
  constexpr int MI = 4, NI = WN / 16;
  constexpr int PA = BM * kChunks / THREADS;        // x chunks per thread and step
  constexpr int PB = BN * kChunks / THREADS;        // weight chunks
  constexpr int kRowStep = THREADS / kChunks;
  constexpr int PV = LN ? Elem<PT>::kBytes : 0;     // 16-byte vectors of gamma + beta per chunk
  // LDS rows of 64 elements (128 bytes), no padding: chunk c of row r sits in slot c ^ (r & 7), so
  // the 16-byte chunk writes and the fragment reads meet no bank conflicts (2.75 M conflict cycles
  // per launch with rows padded to 72 elements)
  constexpr int kStageA = BM * kBK, kStageB = BN * kBK;
  __shared__ __align__(16) uint16_t sA[2][kStageA];
  __shared__ __align__(16) uint16_t sB[2][kStageB];

  const int total = p.tiles_m * p.tiles_n;
  const int i = static_cast<int>(blockIdx.x);
  int tile = i;
  if (total % kXcds == 0) tile = (i % kXcds) * (total / kXcds) + i / kXcds;
  const int64_t m0 = static_cast<int64_t>(tile / p.tiles_n) * BM;
  const int n0 = (tile % p.tiles_n) * BN;

  const int t = static_cast<int>(threadIdx.x);
  const int lane = t & (kWave - 1);
  const int wave = t / kWave;
  const int wm = wave / GN, wn = wave % GN;
  const int kc = t % kChunks, r0 = t / kChunks;
  const int fr = lane & 15, fk = (lane >> 4) * 8;

  const Rsrc xr = make_rsrc(p.x, static_cast<uint32_t>(p.M * p.K * 2));
  const Rsrc wr = make_rsrc(p.w, static_cast<uint32_t>(static_cast<int64_t>(p.N) * p.K * 2));
  const Rsrc gr = LN ? make_rsrc(p.gamma, static_cast<uint32_t>(p.K * Elem<PT>::kBytes)) : wr;
  const Rsrc br = LN ? make_rsrc(p.beta, static_cast<uint32_t>(p.K * Elem<PT>::kBytes)) : wr;
  const uint32_t poff = kc * 8 * Elem<PT>::kBytes;
  float mean[PA], rstd[PA];
  uint32_t xoff[PA], woff[PB];
#pragma unroll
  for (int q = 0; q < PA; ++q) {
    const int64_t m = m0 + r0 + q * kRowStep;
    const int64_t mc = m < p.M ? m : p.M - 1;
    mean[q] = 0.f;
    rstd[q] = 1.f;
    if constexpr (LN) {
      mean[q] = p.mean[mc];
      rstd[q] = p.rstd[mc];
    }
    xoff[q] = static_cast<uint32_t>((mc * p.K + kc * 8) * 2);
  }
#pragma unroll
  for (int q = 0; q < PB; ++q) {
    const int n = n0 + r0 + q * kRowStep;
    woff[q] = static_cast<uint32_t>((static_cast<int64_t>(n < p.N ? n : p.N - 1) * p.K + kc * 8) * 2);
  }

  // this workgroup's steps of K: all of them, or split blockIdx.y's range (an even count)
  const int nk_all = p.K / kBK;
  const int ks0 = p.part ? static_cast<int>(blockIdx.y) * p.split_steps : 0;
  const int nk = p.part ? (nk_all - ks0 < p.split_steps ? nk_all - ks0 : p.split_steps) : nk_all;
  uint4 ra[U][PA], rb[U][PB];
  uint4 rp[U][PV > 0 ? PV : 1];
  auto issue = [&](int ks, uint4 (&a)[PA], uint4 (&b)[PB], uint4 (&pp)[PV > 0 ? PV : 1]) {
    const uint32_t kq = static_cast<uint32_t>(ks0 + (ks < nk ? ks : nk - 1));  // later steps are never used
#pragma unroll
    for (int q = 0; q < PA; ++q) a[q] = bload16(xr, xoff[q], kq * kBK * 2);
    if constexpr (LN) {
      constexpr int HV = Elem<PT>::kBytes / 2;
#pragma unroll
      for (int h = 0; h < HV; ++h) {
        pp[h] = bload16(gr, poff + h * 16, kq * kBK * Elem<PT>::kBytes);
        pp[HV + h] = bload16(br, poff + h * 16, kq * kBK * Elem<PT>::kBytes);
      }
    }
#pragma unroll
    for (int q = 0; q < PB; ++q) b[q] = bload16(wr, woff[q], kq * kBK * 2);
  };
  auto put = [&](int buf, const uint4 (&a)[PA], const uint4 (&b)[PB], const uint4 (&pp)[PV > 0 ? PV : 1]) {
    float g[8], bt[8];
    if constexpr (LN) {
      constexpr int HV = Elem<PT>::kBytes / 2;
#pragma unroll
      for (int h = 0; h < HV; ++h) {
        unpack16(pp[h], g + h * (16 / Elem<PT>::kBytes), PT{});
        unpack16(pp[HV + h], bt + h * (16 / Elem<PT>::kBytes), PT{});
      }
    }
#pragma unroll
    for (int q = 0; q < PA; ++q) {
      uint4 v = a[q];
      if constexpr (LN) v = normalise8(a[q], mean[q], rstd[q], g, bt);
      *reinterpret_cast<uint4*>(&sA[buf][(r0 + q * kRowStep) * kBK + ((kc ^ (r0 & 7)) << 3)]) = v;
    }
#pragma unroll
    for (int q = 0; q < PB; ++q) *reinterpret_cast<uint4*>(&sB[buf][(r0 + q * kRowStep) * kBK + ((kc ^ (r0 & 7)) << 3)]) = b[q];
  };

  f32x4 acc[MI][NI];
#pragma unroll
  for (int a = 0; a < MI; ++a)
#pragma unroll
    for (int c = 0; c < NI; ++c) acc[a][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int buf) {
    // every fragment of the step is read first (16 LDS reads in flight), then the products; a
    // fragment row's r & 7 is fr & 7 (the other terms of the row are multiples of 8)
    bf16x8 fa[2][MI], fb[2][NI];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int c = 0; c < NI; ++c)
        fb[h][c] = *reinterpret_cast<const bf16x8*>(&sB[buf][(wn * WN + c * 16 + fr) * kBK + ((((h * 32 + fk) >> 3) ^ (fr & 7)) << 3)]);
#pragma unroll
      for (int a = 0; a < MI; ++a)
        fa[h][a] = *reinterpret_cast<const bf16x8*>(&sA[buf][(wm * 64 + a * 16 + fr) * kBK + ((((h * 32 + fk) >> 3) ^ (fr & 7)) << 3)]);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int a = 0; a < MI; ++a)
#pragma unroll
        for (int c = 0; c < NI; ++c)
          acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[h][a], fb[h][c], acc[a][c], 0, 0, 0);
  };

#pragma unroll
  for (int u = 0; u < U; ++u) issue(u, ra[u], rb[u], rp[u]);
  put(0, ra[0], rb[0], rp[0]);
  // kept after the write that reads set 0: hoisted above it, these loads would need registers
  // of their own, and the loop would begin with copies that wait for every load in flight
  __builtin_amdgcn_sched_barrier(0);
  issue(U, ra[0], rb[0], rp[0]);
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();
  // iteration s writes step s + 1 (set (s + 1) % U) into the other LDS buffer and refills that
  // set with step s + 1 + U, then multiplies step s; nk is a multiple of U, so the unrolled body
  // holds no branch and each register set keeps its registers across the loop (step nk's write
  // goes to a buffer that is not read again)
  for (int s0 = 0; s0 < nk; s0 += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u;
      put((s + 1) & 1, ra[(u + 1) % U], rb[(u + 1) % U], rp[(u + 1) % U]);
      // the scheduling barriers keep each phase where it is written: loads moved next to
      // their use would be waited for at once
      __builtin_amdgcn_sched_barrier(0);
      issue(s + 1 + U, ra[(u + 1) % U], rb[(u + 1) % U], rp[(u + 1) % U]);
      __builtin_amdgcn_sched_barrier(0);
      multiply(s & 1);
      __syncthreads();
    }
  }

  if (p.part) {  // split K: this split's fp32 partial products, added up by the reduction kernel
    float* const part = p.part + static_cast<int64_t>(blockIdx.y) * p.M * p.N;
#pragma unroll
    for (int c = 0; c < NI; ++c) {
      const int n = n0 + wn * WN + c * 16 + fr;
      if (n >= p.N) continue;
#pragma unroll
      for (int a = 0; a < MI; ++a) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int64_t m = m0 + wm * 64 + a * 16 + (lane >> 4) * 4 + r;
          if (m < p.M) part[m * p.N + n] = acc[a][c][r];
        }
      }
    }
    return;
  }
  // epilogue: + bias, one rounding to the output type
#pragma unroll
  for (int c = 0; c < NI; ++c) {
    const int n = n0 + wn * WN + c * 16 + fr;
    if (n >= p.N) continue;
    const float bn = p.bias ? Elem<BT>::load(static_cast<const char*>(p.bias) + static_cast<int64_t>(n) * Elem<BT>::kBytes)
                            : 0.f;
#pragma unroll
    for (int a = 0; a < MI; ++a) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t m = m0 + wm * 64 + a * 16 + (lane >> 4) * 4 + r;
        if (m < p.M) store_y<OT>(p.y, m * p.N + n, acc[a][c][r] + bn);
      }
    }
  }
}

// Workgroup barrier for what the wavefronts exchanged through ds_write / ds_read: loads in flight, those
// to LDS included, stay in flight (__syncthreads would wait for the latter).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // no instruction: keeps the compiler's order
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Vectors at any element's alignment: rows of y start at any multiple of its elements.
typedef f32x4 f32x4_any __attribute__((aligned(4)));
typedef u32x2 u32x2_any __attribute__((aligned(2)));

constexpr int kBandParams = kLinearBandParams;  // LDS for gamma and beta (160 KB in all)

// Waits until at most N of this wavefront's loads are in flight: all but the N newest have arrived, those to
// LDS included (the compiler does not follow every load to LDS around a loop).
template <int N>
__device__ __forceinline__ void wait_loads() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | (N >> 4 << 14));  // vmcnt(N)
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The band form (K a multiple of 128, byte offsets below 2^31, gamma and beta within kBandParams): a
// workgroup of 8 wavefronts owns 128 rows and 128 * NI columns of y, every wavefront all 128 rows of
// 16 * NI columns of its own. So x is normalised once per band (once per element when the columns
// cover N) on its way through registers to LDS, from where every wavefront reads it. The weight, which
// no two wavefronts of the workgroup share, is loaded straight to LDS without passing registers, half a
// step (32 of K) at a time into a wavefront's own two buffers, and needs no barrier: a half step first
// waits for its weight, reads its fragments, and, once its first products have waited for those, loads
// the next step's over them. x is loaded two steps ahead, after the step's weight loads (loads return
// in order, so the wait for a weight must not include the newest x). One barrier per pair of steps (two
// pairs of x buffers); fragments are read three groups of products ahead and the normalisation's vector
// instructions go between the products. The products are taken transposed (weight as the first
// operand), so a lane holds 4 consecutive columns of a row and stores them at once.
// Measured, M = 30000, K = 3584, N = 512, bf16 parameters: 110-126 us (870-1000 TFLOP/s; 128 x 128 tiles:
// 200 us). Weight fragments loaded from L2 to registers, each lane a row of its own, took 157 us (64 cache
// lines per load instruction), 32 x 32 products 150 us, one barrier per step 133 us.
template <int W, int NI, bool LN, typename PT>
__global__ void __launch_bounds__(W * kWave, 2) ln_linear_band_kernel(const LinearParams p) {
  constexpr int BM = 128, THREADS = W * kWave, BN = 16 * NI * W;
  constexpr int MI = BM / 16;
  constexpr int PA = BM * kChunks / THREADS;     // x chunks per thread and step
  constexpr int kRowStep = THREADS / kChunks;
  constexpr int HV = Elem<PT>::kBytes / 2;       // 16-byte vectors of 8 parameters
  constexpr int PV = LN ? 2 * HV : 1;
  static_assert(kRowStep % 8 == 0, "a thread's rows share their swizzle");
  // rows of 128 bytes, chunk c of row r in slot c ^ (r & 7) (no bank conflicts)
  __shared__ __align__(16) uint16_t sA[4][BM * kBK];  // two pairs of steps
  // the weight, half a step (32 of K) at a time, by wavefront: 64-byte rows, chunk c of row r in slot
  // c ^ (r >> 1 & 3)
  __shared__ __align__(16) uint4 sW0[W][NI][kWave];  // first halves
  __shared__ __align__(16) uint4 sW1[W][NI][kWave];  // second halves
  __shared__ uint4 s_par[LN ? kBandParams / 16 : 1];  // gamma and beta of this workgroup's steps

  const int tile = static_cast<int>(blockIdx.x);
  const int64_t m0 = static_cast<int64_t>(tile / p.tiles_n) * BM;
  const int n0 = (tile % p.tiles_n) * BN;
  const int t = static_cast<int>(threadIdx.x);
  const int lane = t & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int kc = t % kChunks, r0 = t / kChunks;
  const int fr = lane & 15, fq = lane >> 4;  // fragment row, 16-byte chunk of a 32-element half step

  const Rsrc xr = make_rsrc(p.x, static_cast<uint32_t>(p.M * p.K * 2));
  const Rsrc wr = make_rsrc(p.w, static_cast<uint32_t>(static_cast<int64_t>(p.N) * p.K * 2));
  // rows past M and columns past N read the last one: their products are not stored
  float mean[PA], rstd[PA];
  uint32_t xoff[PA], woff[NI];
#pragma unroll
  for (int q = 0; q < PA; ++q) {
    const int64_t m = m0 + r0 + q * kRowStep;
    const int64_t mc = m < p.M ? m : p.M - 1;
    mean[q] = 0.f;
    rstd[q] = 1.f;
    if constexpr (LN) {
      mean[q] = p.mean[mc];
      rstd[q] = p.rstd[mc];
    }
    xoff[q] = static_cast<uint32_t>((mc * p.K + kc * 8) * 2);
  }
  const int nw = n0 + wave * 16 * NI;  // the wavefront's first column
#pragma unroll
  for (int c = 0; c < NI; ++c) {  // lane l loads chunk (l & 3) ^ .. of row l / 4 of fragment c
    const int n = nw + c * 16 + (lane >> 2);
    const int chunk = (lane & 3) ^ (lane >> 3 & 3);
    woff[c] = static_cast<uint32_t>((static_cast<int64_t>(n < p.N ? n : p.N - 1) * p.K + chunk * 8) * 2);
  }

  // this workgroup's steps of K: all of them, or split blockIdx.y's range (an even count)
  const int nk_all = p.K / kBK;
  const int ks0 = p.part ? static_cast<int>(blockIdx.y) * p.split_steps : 0;
  const int nk = p.part ? (nk_all - ks0 < p.split_steps ? nk_all - ks0 : p.split_steps) : nk_all;

  uint4 ra[2][PA];   // x of steps s + 1 (set (s + 1) % 2) and s + 2
  // a step of this workgroup, the last one in place of those past it (which are never used)
  const auto step = [&](int ks) { return static_cast<uint32_t>(ks0 + (ks < nk ? ks : nk - 1)); };
  auto issue_x = [&](int ks, uint4 (&a)[PA]) {
#pragma unroll
    for (int q = 0; q < PA; ++q) a[q] = bload16(xr, xoff[q], step(ks) * kBK * 2);
  };
  // weight loads straight to LDS, lane l's 16 bytes to slot l
  auto issue_w = [&](int ks, auto half) {
    constexpr int h = decltype(half)::value;
#pragma unroll
    for (int c = 0; c < NI; ++c)
      bload16_lds(wr, h ? &sW1[wave][c][0] : &sW0[wave][c][0], woff[c], step(ks) * kBK * 2 + h * 64);
  };
  uint4 rp[PV];  // gamma and beta of the step being normalised
  auto read_p = [&](int ks) {
    if constexpr (LN) {
      const uint4* const pp = s_par + (static_cast<int>(step(ks) - ks0) * kChunks + kc) * PV;
#pragma unroll
      for (int h = 0; h < PV; ++h) rp[h] = pp[h];
    }
  };
  auto put_x = [&](uint16_t* to, const uint4 (&a)[PA], int q0, int q1) {
    float g[8], bt[8];
    if constexpr (LN) {
#pragma unroll
      for (int h = 0; h < HV; ++h) {
        unpack16(rp[h], g + h * (16 / Elem<PT>::kBytes), PT{});
        unpack16(rp[HV + h], bt + h * (16 / Elem<PT>::kBytes), PT{});
      }
    }
#pragma unroll
    for (int q = q0; q < q1; ++q) {
      uint4 v = a[q];
      if constexpr (LN) v = normalise8(a[q], mean[q], rstd[q], g, bt);
      *reinterpret_cast<uint4*>(to + q * kRowStep * kBK) = v;
    }
  };
  f32x4 acc[MI][NI];
#pragma unroll
  for (int a = 0; a < MI; ++a)
#pragma unroll
    for (int c = 0; c < NI; ++c) acc[a][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  // this thread's place in a step's x buffer: where it writes, and its fragments of either half
  constexpr int kPair = 2 * BM * kBK;
  uint16_t* const put_at = &sA[0][r0 * kBK + ((kc ^ (r0 & 7)) << 3)];
  const uint16_t* const frag_at0 = &sA[0][fr * kBK + ((fq ^ (fr & 7)) << 3)];
  const uint16_t* const frag_at1 = &sA[0][fr * kBK + (((4 + fq) ^ (fr & 7)) << 3)];
  const int wslot = fr * 4 + (fq ^ (fr >> 1 & 3));
  bf16x8 wb[2][NI];
  auto read_w = [&](auto half) {
    constexpr int h = decltype(half)::value;
#pragma unroll
    for (int c = 0; c < NI; ++c)
      wb[h][c] = __builtin_bit_cast(bf16x8, h ? sW1[wave][c][wslot] : sW0[wave][c][wslot]);
  };
  auto multiply = [&](int i, const bf16x8& fa) {
#pragma unroll
    for (int c = 0; c < NI; ++c)
      acc[i % MI][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[i / MI][c], fa, acc[i % MI][c], 0, 0, 0);
  };

  constexpr std::integral_constant<int, 0> first{};
  constexpr std::integral_constant<int, 1> second{};
  issue_x(0, ra[0]);
  issue_w(0, first);
  issue_w(0, second);
  issue_x(1, ra[1]);
  __builtin_amdgcn_sched_barrier(0);  // x of steps 2 and 3 is issued after all of these
  if constexpr (LN) {
    // gamma and beta of this workgroup's steps, 8 of each next to one another
    for (int i = t; i < nk * kChunks; i += THREADS) {
      const int64_t at = (static_cast<int64_t>(ks0) * kChunks + i) * HV;
#pragma unroll
      for (int h = 0; h < HV; ++h) {
        s_par[i * 2 * HV + h] = static_cast<const uint4*>(p.gamma)[at + h];
        s_par[i * 2 * HV + HV + h] = static_cast<const uint4*>(p.beta)[at + h];
      }
    }
    __syncthreads();
  }
  read_p(0);
  put_x(put_at, ra[0], 0, PA);
  issue_x(2, ra[0]);
  read_p(1);
  put_x(put_at + BM * kBK, ra[1], 0, PA);
  __builtin_amdgcn_sched_barrier(0);
  issue_x(3, ra[1]);
  // The first half steps' waits count on the order of loads that the loop keeps; here the compiler orders
  // them. So all but x of steps 2 and 3, the newest, have arrived before the loop, the weight in both
  // halves among them (no longer a wait than that for x of step 1, which they were issued before).
  wait_loads<2 * PA>();
  lds_barrier();
  constexpr int kAhead = 3;  // x fragments are read this many groups of products ahead
  // One half of step s: its fragments are read and the first products issued, which have then
  // waited for the weight's fragments; so the next step's half may be loaded over them. Then the
  // rest of the products, the normalisation's vector instructions between them.
  auto half_step = [&](int u, int s, int par, auto half) {
    constexpr int h = decltype(half)::value;
    const uint16_t* const from = (h ? frag_at1 : frag_at0) + par * kPair + u * BM * kBK;
    const auto frag = [&](int i) { return *reinterpret_cast<const bf16x8*>(from + i * 16 * kBK); };
    bf16x8 fa[MI];
    // loads issued since this half's weight: the other half's, and x (see the loop below)
    wait_loads<NI + PA>();
    read_w(half);
#pragma unroll
    for (int i = 0; i <= kAhead; ++i) fa[i] = frag(i);
    if (h == 0) read_p(s + 2);
    multiply(h * MI, fa[0]);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);  // the SIMD's other wavefront reads and waits meanwhile
    issue_w(s + 1, half);
#pragma unroll
    for (int i = kAhead + 1; i < MI; ++i) fa[i] = frag(i);
#pragma unroll
    for (int i = 1; i < MI; ++i) multiply(h * MI + i, fa[i]);
    put_x(put_at + (par ^ 1) * kPair + u * BM * kBK, ra[u], h ? PA / 2 : 0, h ? PA : PA / 2);
    __builtin_amdgcn_sched_group_barrier(0x20, NI, 0);
#pragma unroll
    for (int i = 1; i < MI; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x8, NI, 0);                        // products
      if (i + kAhead < MI) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
      if (LN) __builtin_amdgcn_sched_group_barrier(0x2, 12, 0);                // vector ALU
    }
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
  };
  // a pair of steps is multiplied while the next pair is normalised into the other two buffers, with
  // one barrier per pair; nk is even
  for (int s0 = 0, par = 0; s0 < nk; s0 += 2, par ^= 1) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      half_step(u, s0 + u, par, first);
      half_step(u, s0 + u, par, second);
      issue_x(s0 + u + 4, ra[u]);
      __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();
  }

  // lane l holds y[m0 + 16 a + l % 16][nw + 16 c + 4 (l / 16) + r]
  float* const part = p.part ? p.part + static_cast<int64_t>(blockIdx.y) * p.M * p.N : nullptr;
#pragma unroll
  for (int c = 0; c < NI; ++c) {
    const int n = nw + c * 16 + fq * 4;
    if (n >= p.N) continue;
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if (p.bias && !part) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int nr = n + r < p.N ? n + r : p.N - 1;
        bias[r] = p.bias_f32 ? static_cast<const float*>(p.bias)[nr]
                             : bf16_bits_to_f32(static_cast<const uint16_t*>(p.bias)[nr]);
      }
    }
#pragma unroll
    for (int a = 0; a < MI; ++a) {
      const int64_t m = m0 + a * 16 + fr;
      if (m >= p.M) continue;
      const int64_t at = m * p.N + n;
      f32x4 v = acc[a][c];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] += bias[r];
      const bool whole = n + 4 <= p.N;  // else the row's last 1 to 3 columns
      if (part || p.y_f32) {
        float* const y = (part ? part : reinterpret_cast<float*>(p.y)) + at;
        if (whole) {
          *reinterpret_cast<f32x4_any*>(y) = v;
        } else {
          for (int r = 0; r < 3 && n + r < p.N; ++r) y[r] = v[r];
        }
      } else {
        uint16_t* const y = reinterpret_cast<uint16_t*>(p.y) + at;
        if (whole) {
          *reinterpret_cast<u32x2_any*>(y) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        } else {
          for (int r = 0; r < 3 && n + r < p.N; ++r) y[r] = static_cast<uint16_t>(pack_bf16x2(v[r], 0.f));
        }
      }
    }
  }
}

// Split K: y[m, n] = (sum over splits, in split order, of the fp32 partials) + bias, one rounding.
// Four consecutive elements per thread (16-byte loads of each split's partials; M * N is a
// multiple of 4, so every split's block stays 16-byte aligned), the last thread taking the rest.
template <typename BT, typename OT>
__global__ void __launch_bounds__(256) ln_linear_reduce_kernel(const LinearParams p, int32_t splits) {
  const int64_t total = p.M * p.N;
  const int64_t i0 = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i0 >= total) return;
  float v[4];
  const int cnt = total - i0 < 4 ? static_cast<int>(total - i0) : 4;
  if (total % 4 == 0) {  // then cnt == 4
    const float4 q0 = *reinterpret_cast<const float4*>(p.part + i0);
    v[0] = q0.x;
    v[1] = q0.y;
    v[2] = q0.z;
    v[3] = q0.w;
    for (int sp = 1; sp < splits; ++sp) {
      const float4 q = *reinterpret_cast<const float4*>(p.part + static_cast<int64_t>(sp) * total + i0);
      v[0] += q.x;
      v[1] += q.y;
      v[2] += q.z;
      v[3] += q.w;
    }
  } else {
    for (int e = 0; e < cnt; ++e) v[e] = p.part[i0 + e];
    for (int sp = 1; sp < splits; ++sp)
      for (int e = 0; e < cnt; ++e) v[e] += p.part[static_cast<int64_t>(sp) * total + i0 + e];
  }
  for (int e = 0; e < cnt; ++e) {
    const int n = static_cast<int>((i0 + e) % p.N);
    const float bn = p.bias ? Elem<BT>::load(static_cast<const char*>(p.bias) + static_cast<int64_t>(n) * Elem<BT>::kBytes)
                            : 0.f;
    store_y<OT>(p.y, i0 + e, v[e] + bn);
  }
}

template <typename BT, typename OT>
void launch_reduce(const LinearParams& p, int splits, hipStream_t s) {
  const int64_t threads = (p.M * p.N + 3) / 4;
  hipLaunchKernelGGL((ln_linear_reduce_kernel<BT, OT>), dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0,
                     s, p, splits);
}

template <int NI, bool LN, typename PT, typename BT, typename OT>
hipError_t launch_band(LinearParams p, int splits, hipStream_t s) {
  constexpr int W = 8;
  p.tiles_m = static_cast<int32_t>((p.M + 127) / 128);
  p.tiles_n = (p.N + 16 * NI * W - 1) / (16 * NI * W);
  if (splits <= 1) p.part = nullptr;
  hipLaunchKernelGGL((ln_linear_band_kernel<W, NI, LN, PT>),
                     dim3(static_cast<unsigned>(p.tiles_m * p.tiles_n), static_cast<unsigned>(splits > 1 ? splits : 1)),
                     dim3(W * kWave), 0, s, p);
  if (splits > 1) launch_reduce<BT, OT>(p, splits, s);
  return hipGetLastError();
}

template <int BN, int GN, int U, bool LN, typename PT, typename BT, typename OT>
hipError_t launch_big(LinearParams p, int splits, hipStream_t s) {
  p.tiles_m = static_cast<int32_t>((p.M + 127) / 128);
  p.tiles_n = (p.N + BN - 1) / BN;
  const int64_t blocks = static_cast<int64_t>(p.tiles_m) * p.tiles_n;
  if (splits <= 1) p.part = nullptr;
  hipLaunchKernelGGL((ln_linear_big_kernel<BN, GN, U, LN, PT, BT, OT>),
                     dim3(static_cast<unsigned>(blocks), static_cast<unsigned>(splits > 1 ? splits : 1)),
                     dim3(2 * GN * kWave), 0, s, p);
  if (splits > 1) launch_reduce<BT, OT>(p, splits, s);
  return hipGetLastError();
}

template <int BM, int WAVES, int U, bool LN, typename PT, typename BT, typename OT>
hipError_t launch_tile(LinearParams p, hipStream_t s) {
  p.tiles_m = static_cast<int32_t>((p.M + BM - 1) / BM);
  p.tiles_n = (p.N + WAVES * kWaveCols - 1) / (WAVES * kWaveCols);
  const int64_t blocks = static_cast<int64_t>(p.tiles_m) * p.tiles_n;
  hipLaunchKernelGGL((ln_linear_kernel<BM, WAVES, U, LN, PT, BT, OT>), dim3(static_cast<unsigned>(blocks)),
                     dim3(WAVES * kWave), 0, s, p);
  return hipGetLastError();
}

// The form and the splits that linear_plan chooses for the shape and the workspace.
template <bool LN, typename PT, typename BT, typename OT>
hipError_t launch_linear(LinearParams p, int64_t ws_bytes, hipStream_t s) {
  const LinearPlan plan = linear_plan(p.M, p.N, p.K, LN ? Elem<PT>::kBytes : 0, p.part ? ws_bytes : 0);
  p.split_steps = plan.steps;
  switch (plan.form) {
    case kLinearBand:
      switch (linear_band_fragments(p.N)) {
        case 2: return launch_band<2, LN, PT, BT, OT>(p, plan.splits, s);
        case 3: return launch_band<3, LN, PT, BT, OT>(p, plan.splits, s);
        default: return launch_band<4, LN, PT, BT, OT>(p, plan.splits, s);
      }
    case kLinearTile256: return launch_big<256, 4, 2, LN, PT, BT, OT>(p, 1, s);
    case kLinearTile128: return launch_big<128, 4, 2, LN, PT, BT, OT>(p, plan.splits, s);
    default: return launch_tile<64, 4, 2, LN, PT, BT, OT>(p, s);
  }
}

template <bool LN, typename PT, typename BT>
hipError_t launch_out(int32_t odt, const LinearParams& p, int64_t ws, hipStream_t s) {
  return odt == CTI_EBAG_F32 ? launch_linear<LN, PT, BT, float>(p, ws, s) : launch_linear<LN, PT, BT, bf16_t>(p, ws, s);
}

template <bool LN, typename PT>
hipError_t launch_bias(int32_t bdt, int32_t odt, const LinearParams& p, int64_t ws, hipStream_t s) {
  return bdt == CTI_EBAG_F32 ? launch_out<LN, PT, float>(odt, p, ws, s) : launch_out<LN, PT, bf16_t>(odt, p, ws, s);
}

}  // namespace
}  // namespace cti

using namespace cti;

extern "C" int64_t cti_ebag_layernorm_linear_workspace_bytes(int64_t rows, int32_t cols, int32_t out_features) {
  if (rows < 1 || cols < 1 || out_features < 1) return 0;
  return linear_workspace_bytes(rows, out_features, cols);
}

extern "C" int cti_ebag_layernorm_linear(const void* x, int64_t rows, int32_t cols, const float* mean,
                                         const float* rstd, const void* gamma, const void* beta, int32_t param_dtype,
                                         const void* weight, int32_t out_features, const void* bias,
                                         int32_t bias_dtype, void* y, int32_t y_dtype, void* workspace,
                                         int64_t workspace_bytes, void* stream) {
  clear_error();
  if (rows < 0) return set_error(CTI_EBAG_EINVAL, "rows must be >= 0 (got %lld)", (long long)rows);
  if (cols < 1 || out_features < 1)
    return set_error(CTI_EBAG_EINVAL, "cols and out_features must be >= 1 (got %d, %d)", cols, out_features);
  if (cols % 8 != 0)
    return set_error(CTI_EBAG_EUNSUPPORTED, "cols must be a multiple of 8 (16-byte rows; got %d)", cols);
  const bool ln = mean != nullptr || rstd != nullptr || gamma != nullptr || beta != nullptr;
  if (ln && !(mean && rstd && gamma && beta))
    return set_error(CTI_EBAG_EINVAL, "mean, rstd, gamma and beta must be given together (or none of them)");
  if (ln && param_dtype != CTI_EBAG_F32 && param_dtype != CTI_EBAG_BF16)
    return set_error(CTI_EBAG_EINVAL, "gamma / beta must be fp32 or bf16 (dtype code %d)", param_dtype);
  if (bias && bias_dtype != CTI_EBAG_F32 && bias_dtype != CTI_EBAG_BF16)
    return set_error(CTI_EBAG_EINVAL, "bias must be fp32 or bf16 (dtype code %d)", bias_dtype);
  if (y_dtype != CTI_EBAG_F32 && y_dtype != CTI_EBAG_BF16)
    return set_error(CTI_EBAG_EINVAL, "the output must be fp32 or bf16 (dtype code %d)", y_dtype);
  if (rows == 0) return CTI_EBAG_OK;
  if (!x || !weight || !y) return set_error(CTI_EBAG_EINVAL, "NULL device pointer among x / weight / y");
  const auto a16 = [](const void* q) { return reinterpret_cast<uintptr_t>(q) % 16 == 0; };
  if (!a16(x) || !a16(weight) || (ln && (!a16(gamma) || !a16(beta))))
    return set_error(CTI_EBAG_EINVAL, "x, weight, gamma and beta must be 16-byte aligned");
  if (workspace_bytes < 0 || (workspace_bytes > 0 && !workspace))
    return set_error(CTI_EBAG_EINVAL, "workspace_bytes %lld without a workspace", (long long)workspace_bytes);
  if (workspace && !a16(workspace)) return set_error(CTI_EBAG_EINVAL, "the workspace must be 16-byte aligned");
  if (rows > (int64_t{INT32_MAX} / 2) * 64 || (rows + 63) / 64 * ((out_features + 255) / 256) > INT32_MAX)
    return set_error(CTI_EBAG_EUNSUPPORTED, "%lld rows x %d outputs need too many tiles", (long long)rows, out_features);
  LinearParams p{};
  p.x = static_cast<const char*>(x);
  p.mean = mean;
  p.rstd = rstd;
  p.gamma = gamma;
  p.beta = beta;
  p.w = static_cast<const char*>(weight);
  p.bias = bias;
  p.y = static_cast<char*>(y);
  p.M = rows;
  p.N = out_features;
  p.K = cols;
  p.bias_f32 = bias_dtype == CTI_EBAG_F32;
  p.y_f32 = y_dtype == CTI_EBAG_F32;
  p.part = workspace_bytes > 0 ? static_cast<float*>(workspace) : nullptr;
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipError_t e;
  const int32_t bdt = bias ? bias_dtype : CTI_EBAG_F32;
  const int64_t ws = p.part ? workspace_bytes : 0;
  if (!ln) e = launch_bias<false, float>(bdt, y_dtype, p, ws, s);
  else if (param_dtype == CTI_EBAG_F32) e = launch_bias<true, float>(bdt, y_dtype, p, ws, s);
  else e = launch_bias<true, bf16_t>(bdt, y_dtype, p, ws, s);
  if (e != hipSuccess) return set_error(CTI_EBAG_EHIP, "layernorm-linear launch failed: %s", hipGetErrorString(e));
  return CTI_EBAG_OK;
}
