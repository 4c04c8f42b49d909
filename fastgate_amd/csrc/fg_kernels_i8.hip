// int8- and int4-weight GEMV kernels, weights [N,K] row-major.
//
//  * w8a16 / w4a16: fp16 activations.  The integers reach v_dot2_f32_f16 or the MFMA as fp16
//    subnormals (a byte or nibble in the low mantissa bits under a zero exponent is that number
//    times 2^-24, exactly; see wq_m1_kernel), products and sums are fp32, and the per-output-channel
//    scale and the zero point are applied once per output.
//  * i8i8: int8 activations, v_dot4_i32_i8 or the int8 MFMA, exact int32 result.
//  * Two activation rows and more, where the activations fit LDS: the panel kernels (*_x_kernel).
//
// Replaces the device side of gemv_quantized_int8 (backend/cuda/hk/fastgemv.cuh:316-389,
// 8-byte loads, int8 -> fp32 convert, scalar FMAs) of the reference.
#include "fg_device.h"
#include "fg_internal.h"

#include <algorithm>
#include <type_traits>

namespace fg {

// Per-channel scale of the output a thread writes at the end, fetched ahead of the weight stream
// as raw bits.  Converting it at the point of the load would make the wave wait for this cold
// load before it issues anything else (measured: 0.3 us on the whole call at K = N = 8192);
// scale_value() keeps the conversion, and with it the wait, at the point of use.
__device__ __forceinline__ uint32_t scale_fetch(const half_t* scale, int n, bool mine) {
  uint32_t raw = 0x3c00u;  // 1.0
  if (scale != nullptr && mine) raw = reinterpret_cast<const uint16_t*>(scale)[n];
  return raw;
}
__device__ __forceinline__ float scale_value(uint32_t raw) {
  asm volatile("" : "+v"(raw));
  return f16_bits_to_f32((uint16_t)raw);
}

// The zero point (and the 128 that the subnormal form of int8 carries) leaves a dot product as one
// term, constant x Σx.  An activation row that holds an infinity or a NaN makes Σx non-finite, and
// that term would then turn every output of the row into NaN, where element-by-element arithmetic
// -- sum += x (float(w) - zp), backend/cuda/hk/fastgemv.cuh:344-363 -- gives ±inf when infinities
// of one sign meet weights on one side of the zero point.  Σx is non-finite for such rows only
// (finite halves cannot overflow an fp32 sum), so the thread that writes an output looks at it
// and, for such a row, computes its one output again the reference's way: K steps in one thread,
// paid only by input that is already broken.  BITS = 4: two nibbles a byte, the even k low.
__device__ __forceinline__ bool not_finite(float v) { return !(__builtin_fabsf(v) <= 3.4028234664e38f); }
template <int BITS>
__device__ float elementwise_dot(const uint8_t* __restrict__ wrow, const half_t* __restrict__ xrow, int K,
                                 float zero_point) {
  float s = 0.f;
  for (int k = 0; k < K; ++k) {
    int w;
    if (BITS == 8) {
      w = static_cast<int8_t>(wrow[k]);
    } else {
      const uint32_t b = wrow[k >> 1];
      w = (k & 1) ? b >> 4 : b & 15u;
    }
    s += static_cast<float>(xrow[k]) * (static_cast<float>(w) - zero_point);
  }
  return s;
}

// ---------------------------------------------------------------------------------------
// MR activation rows: one (the GEMV proper), and up to four where the launchers say so; int8 and int4
// weights.
//  * Lanes own 8 activations each, not 16 weight bytes: a chunk is UD 16-byte units of x a lane
//    (unit 64 d + lane, d < UD), so every x load is one contiguous KB per wave, and the weights
//    under a unit are 8 bytes (int8) or 4 bytes (int4) per row: UD 8- or 4-byte loads a row,
//    each contiguous over the wave.  With 16 weight bytes a lane, the lane's x is 32 or 64
//    bytes at that stride from its neighbour's: two or four loads that each touch every cache
//    line of the wave's span, which cost more than the weight loads themselves.
//  * The integers reach v_dot2_f32_f16 as fp16 subnormals: a byte or nibble in the low mantissa
//    bits of a half with a zero exponent field IS that number times 2^-24 (a nibble in bits 4-7:
//    times 2^-20), exactly.  Kernels keep fp16 subnormals (the compiler's default float mode
//    for gfx9), products and sums are fp32, and the power of two is put back once per output.
//    int8: 3 integer operations per 4 weights (sign flip to w + 128, two byte shuffles), the 128
//    taken out once per output as 128 Σx; int4: 5 per 8 weights (a shift, four masks) and no
//    constant at all -- against 5 and 7 with a bias to subtract in fp16.
//  * Waves of a workgroup interleave over the chunks of K; 16-lane sums by DPP, the rest through
//    LDS in a fixed order.
// K = N = 8192, one GPU, us per call: int4 9.5 -> 7.6 (a plain read of the 32 MiB: 6.1).  The x
// loads still cost 0.8 us of that (timed with x replaced by constants), for int8 too: 4 KB of x
// from L2 per 4 KB of weights from memory, whatever cache policy the weight loads carry; staging x
// in LDS once per 16-wave workgroup moves the cost into the wait before the first decode.
// Replaces the device side of gemv_quantized_int8 (backend/cuda/hk/fastgemv.cuh:316-389) and of
// gemv_quantized_int4 (:394-495, defined there but never launched) for one row.
// ---------------------------------------------------------------------------------------
template <int BITS, int RN, int NWV, int UD, int MR>
__global__ __launch_bounds__(64 * NWV) void wq_m1_kernel(const uint8_t* __restrict__ Wq,
                                                         const half_t* __restrict__ X,
                                                         const half_t* __restrict__ scale,
                                                         float scalar_scale, float zero_point,
                                                         half_t* __restrict__ Y, int N, int K) {
  constexpr int WB = BITS == 4 ? 4 : 8;  // weight bytes under one 16-byte unit of x
  typedef uint32_t wreg_t __attribute__((ext_vector_type(WB / 4)));
  constexpr int RC = RN + 1;             // columns of the reduction table per activation row: RN sums and Σx
  __shared__ float red[NWV * 4][MR * RC];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: addresses stay scalar
  const int n0 = blockIdx.x * RN;
  const size_t rowb = BITS == 4 ? (size_t)K >> 1 : (size_t)K;
  static_assert(MR * RN <= 64, "one output per thread of the first wave");
  const uint32_t scale_raw = scale_fetch(scale, n0 + (int)threadIdx.x % RN, threadIdx.x < MR * RN);
  // the constant that comes out with Σx: the zero point, and int8's + 128
  const float zp = BITS == 4 ? zero_point : zero_point + 128.f;
  const bool use_xsum = zp != 0.f;
  const uint8_t* Wt = Wq + (size_t)n0 * rowb;  // uniform; the lane's part is a 32-bit offset
  const uint32_t lane_w = lane * WB, lane_x = lane * 16;
  const half2_t ones = {static_cast<half_t>(1.f), static_cast<half_t>(1.f)};
  float acc0[MR][RN], acc1[MR][RN];
  float xsum[MR];
#pragma unroll
  for (int m = 0; m < MR; ++m) {
    xsum[m] = 0.f;
#pragma unroll
    for (int r = 0; r < RN; ++r) acc0[m][r] = acc1[m][r] = 0.f;
  }

  constexpr int kNonTemporal = 2;  // the nt bit of a buffer load's cache policy
  const __amdgpu_buffer_rsrc_t wrs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(Wt), 0, (int)(RN * rowb), 0x00020000);
  __amdgpu_buffer_rsrc_t xrs[MR];
#pragma unroll
  for (int m = 0; m < MR; ++m)
    xrs[m] = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(X + (size_t)m * K), 0, K * 2, 0x00020000);
  const int nunits = K >> 3;
  const int nchunks = (nunits + 64 * UD - 1) / (64 * UD);
  for (int ch = wave; ch < nchunks; ch += NWV) {
    wreg_t wr[RN][UD];
    u32x4 xv[MR][UD];
    // Buffer loads: a lane past the end of K gets zeros for x (the descriptor ends with the row), so
    // whatever its weight load returns -- the start of the next row, or zeros past the workgroup's
    // last row -- multiplies to zero: no predicate, no branch around any of the loads.
#pragma unroll
    for (int r = 0; r < RN; ++r)
#pragma unroll
      for (int d = 0; d < UD; ++d) {
        const int off = r * (int)rowb + (ch * (64 * UD) + 64 * d) * WB + (int)lane_w;
        if constexpr (WB == 4) wr[r][d][0] = __builtin_amdgcn_raw_buffer_load_b32(wrs, off, 0, kNonTemporal);
        else wr[r][d] = __builtin_bit_cast(wreg_t, __builtin_amdgcn_raw_buffer_load_b64(wrs, off, 0, kNonTemporal));
      }
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
      for (int d = 0; d < UD; ++d)
        xv[m][d] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                 xrs[m], (ch * (64 * UD) + 64 * d) * 16 + (int)lane_x, 0, 0));
    if (use_xsum) {
#pragma unroll
      for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int d = 0; d < UD; ++d)
#pragma unroll
          for (int i = 0; i < 4; ++i) xsum[m] = __builtin_amdgcn_fdot2(as_half2(xv[m][d][i]), ones, xsum[m], false);
    }
    if (BITS == 4) {  // (x_j, x_{j+4}): the halves that meet nibbles j and j + 4 of a register
#pragma unroll
      for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int d = 0; d < UD; ++d) {
          const u32x4 t = xv[m][d];
          xv[m][d].x = __builtin_amdgcn_perm(t.z, t.x, 0x05040100u);
          xv[m][d].y = __builtin_amdgcn_perm(t.z, t.x, 0x07060302u);
          xv[m][d].z = __builtin_amdgcn_perm(t.w, t.y, 0x05040100u);
          xv[m][d].w = __builtin_amdgcn_perm(t.w, t.y, 0x07060302u);
        }
    }
#pragma unroll
    for (int r = 0; r < RN; ++r)
#pragma unroll
      for (int d = 0; d < UD; ++d) {
        if constexpr (BITS == 4) {
          const uint32_t w = wr[r][d][0], w8 = w >> 8;  // nibbles 0,4 | 1,5 | 2,6 | 3,7
          const uint32_t n04 = w & 0x000F000Fu, n15 = w & 0x00F000F0u, n26 = w8 & 0x000F000Fu, n37 = w8 & 0x00F000F0u;
#pragma unroll
          for (int m = 0; m < MR; ++m) {
            acc0[m][r] = __builtin_amdgcn_fdot2(as_half2(n04), as_half2(xv[m][d].x), acc0[m][r], false);
            acc1[m][r] = __builtin_amdgcn_fdot2(as_half2(n15), as_half2(xv[m][d].y), acc1[m][r], false);
            acc0[m][r] = __builtin_amdgcn_fdot2(as_half2(n26), as_half2(xv[m][d].z), acc0[m][r], false);
            acc1[m][r] = __builtin_amdgcn_fdot2(as_half2(n37), as_half2(xv[m][d].w), acc1[m][r], false);
          }
        } else {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const uint32_t t = wr[r][d][h] ^ 0x80808080u;  // w + 128 as unsigned bytes
            const uint32_t b01 = __builtin_amdgcn_perm(0u, t, 0x04010400u);  // halves (b0, b1)
            const uint32_t b23 = __builtin_amdgcn_perm(0u, t, 0x04030402u);  // halves (b2, b3)
#pragma unroll
            for (int m = 0; m < MR; ++m) {
              acc0[m][r] = __builtin_amdgcn_fdot2(as_half2(b01), as_half2(xv[m][d][2 * h]), acc0[m][r], false);
              acc1[m][r] = __builtin_amdgcn_fdot2(as_half2(b23), as_half2(xv[m][d][2 * h + 1]), acc1[m][r], false);
            }
          }
        }
      }
  }

#pragma unroll
  for (int m = 0; m < MR; ++m) {
#pragma unroll
    for (int r = 0; r < RN; ++r) {
      // int4: acc1 holds the nibbles that sat 4 bits up
      const float a = BITS == 4 ? acc0[m][r] * 16777216.f + acc1[m][r] * 1048576.f
                                : (acc0[m][r] + acc1[m][r]) * 16777216.f;
      const float v = row16_allreduce(a);
      if ((lane & 15) == 0) red[wave * 4 + (lane >> 4)][m * RC + r] = v;
    }
    const float xs = row16_allreduce(xsum[m]);
    if ((lane & 15) == 0) red[wave * 4 + (lane >> 4)][m * RC + RN] = xs;
  }
  __syncthreads();
  if (threadIdx.x < MR * RN) {
    const int m = threadIdx.x / RN, r = threadIdx.x % RN;
    const float sum = lds_sum<NWV * 4>(&red[0][m * RC + r], MR * RC, NWV * 4);
    const float xs = lds_sum<NWV * 4>(&red[0][m * RC + RN], MR * RC, NWV * 4);
    float v = sum - zp * xs;
    if (not_finite(xs)) v = elementwise_dot<BITS>(Wt + (size_t)r * rowb, X + (size_t)m * K, K, zero_point);
    Y[(size_t)m * N + n0 + r] = static_cast<half_t>(v * (scalar_scale * scale_value(scale_raw)));
  }
}

template <int MB, int RN, int U>
__global__ __launch_bounds__(256) void i8i8_kernel(const int8_t* __restrict__ Wq,
                                                   const int8_t* __restrict__ Xq,
                                                   int32_t* __restrict__ out, int M, int N, int K) {
  __shared__ int red[16][RN * MB];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int nw = blockDim.x >> 6;
  const int n0 = blockIdx.x * RN;
  const int nq = K >> 4;

  int acc[RN][MB];
#pragma unroll
  for (int r = 0; r < RN; ++r)
#pragma unroll
    for (int m = 0; m < MB; ++m) acc[r][m] = 0;
  const int8_t* Wt = Wq + (size_t)n0 * K;
  const u32x4 zero = {0u, 0u, 0u, 0u};

  const int nsteps = (nq + nw * (64 * U) - 1) / (nw * (64 * U));
  int step = stagger_start(nsteps, 0);
  for (int it = 0; it < nsteps; ++it) {
    const int q0 = (step * nw + wave) * (64 * U);
    step = step + 1 == nsteps ? 0 : step + 1;
    u32x4 wr[U][RN];
    u32x4 xr[U][MB];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = q0 + u * 64 + lane;
      const bool ok = q < nq;
#pragma unroll
      for (int r = 0; r < RN; ++r)
        wr[u][r] = ok ? load16<true>(Wt + (size_t)r * K + (size_t)q * 16) : zero;
#pragma unroll
      for (int m = 0; m < MB; ++m)
        xr[u][m] = (ok && m < M) ? load16<false>(Xq + (size_t)m * K + (size_t)q * 16) : zero;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < RN; ++r)
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
          for (int c = 0; c < 4; ++c)
            acc[r][m] = __builtin_amdgcn_sdot4((int)wr[u][r][c], (int)xr[u][m][c], acc[r][m], false);
  }

#pragma unroll
  for (int r = 0; r < RN; ++r)
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const int v = row16_allreduce(acc[r][m]);
      if ((lane & 15) == 0) red[wave * 4 + (lane >> 4)][r * MB + m] = v;
    }
  __syncthreads();
  for (int t = threadIdx.x; t < RN * MB; t += blockDim.x) {
    const int m = t / RN, r = t % RN;
    const int sum = lds_sum_i32(&red[0][r * MB + m], RN * MB, nw * 4);
    if (m < M) out[(size_t)m * N + n0 + r] = sum;
  }
}

// Two to eight activation rows: as w4a16_x_kernel below, the activation panel in LDS, staged once a workgroup,
// which then walks over column tiles of 16; the weights of a tile go from memory through registers and two KB of
// wave-private LDS into the operand of v_mfma_i32_16x16x64_i8 (16 bytes = 16 k of row j a lane).  XR = rows of the
// panel, 4 or 8; its 16-byte pieces lie as [64 k][g][row], the rows of a group permuted by its number (the threads
// that stage it have consecutive k of one row).  Integer sums: exact in any order.  Launched with K <= KC.
// What bounds it: the weights at what memory gives (N = K = 8192 M=8 12.4 us, 5.4 TB/s, a plain read 11.9), on
// short calls launch, one memory latency for the panel and one for the weights (N=4096 K=2048 3.3).  Measured against
// a panel kernel with loads in operand order (18 instead of 64 bytes a clock a CU, see w4a16_x_kernel) and one tile a
// workgroup, us: M=8 N = K = 8192 15.9 / 12.4, N=14336 K=4096 16.6 / 11.3, N = K = 5120 11.4 / 6.8, N=4096 K=2048 3.7 /
// 3.3; M=4, the v_dot4 kernel, N = K = 8192 13.5 / 12.3, N=8192 K=4096 8.7 / 7.3, N = K = 5120 7.5 / 6.8.
template <int XR, int KC, int NW>
__global__ __launch_bounds__(64 * NW) void i8i8_x_kernel(const int8_t* __restrict__ Wq, const int8_t* __restrict__ Xq,
                                                         int32_t* __restrict__ out, int M, int N, int K) {
  typedef int int4_v __attribute__((ext_vector_type(4)));
  constexpr int PAIRS = KC / 128 / NW;                // 16 rows x 128 bytes of weights: two loads a wave
  // loads of 1 KB of an activation row a wave (fewer waves than rows: of several rows)
  constexpr int ROWS = NW < XR ? XR / NW : 1;
  constexpr int SEGS = ((KC + 1023) / 1024 * XR + NW - 1) / NW;
  static_assert(KC % (128 * NW) == 0, "whole pairs");
  constexpr int STRIP = 2048, RED = XR * 16;          // ints a wave hands over
  constexpr bool kOwnRed = XR * KC + NW * (STRIP + 8 * RED) <= 160 * 1024;
  __shared__ u32x4 panel[XR * KC / 16];
  __shared__ __attribute__((aligned(16))) unsigned char strips[NW * STRIP];
  __shared__ int own_red[kOwnRed ? 2 * NW * RED : 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, g = lane >> 4;             // operand order
  const int lr = lane >> 3, lp = lane & 7;            // load order: row, 16-byte piece of its 128
  constexpr int kNonTemporal = 2;
  constexpr int kBeyond = 0x7ffffff0;                 // past the descriptors: the load returns zeros
  // activations first: loads return in order, and the panel must not wait for the weights
  // waves that stage a row: NW / M
  int per_row = NW < XR ? 1 : NW / XR;
  if constexpr (XR == 4) per_row = M == 2 ? NW / 2 : (M == 3 ? NW / 3 : NW / 4);
  else if constexpr (NW == 16) per_row = M == 5 ? 3 : 2;
  const int xm = NW < XR ? wave * ROWS : wave / per_row, xs0 = wave - wave / per_row * per_row;
  u32x4 x[SEGS];
#pragma unroll
  for (int i = 0; i < SEGS; ++i) {
    const int row = xm + i % ROWS, seg = xs0 + per_row * (i / ROWS);
    const __amdgpu_buffer_rsrc_t xrs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(Xq + (size_t)row * K), 0, row < M ? K : 0, 0x00020000);
    x[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xrs, seg * 1024 + lane * 16, 0, 0));
  }
  __builtin_amdgcn_sched_barrier(0);
  u32x4 w[PAIRS][2];
  int w_off[PAIRS];
#pragma unroll
  for (int t = 0; t < PAIRS; ++t) {
    const int kb = (wave + NW * t) * 128 + lp * 16;
    w_off[t] = kb < K ? lr * K + kb : kBeyond;
  }
  const int tiles = N >> 4;
  auto load_pair = [&](int tile, int t) {
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(Wq + (size_t)tile * 16 * K), 0, tile < tiles ? 16 * K : 0, 0x00020000);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      w[t][h] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                              wrs, w_off[t] == kBeyond ? kBeyond : w_off[t] + 8 * h * K, 0, kNonTemporal));
  };
  int tile = blockIdx.x;
#pragma unroll
  for (int t = 0; t < PAIRS; ++t) {
    load_pair(tile, t);
    __builtin_amdgcn_sched_barrier(0);                // in this order: they are waited for one after the other
  }
#pragma unroll
  for (int i = 0; i < SEGS; ++i) {
    const int row = xm + i % ROWS, seg = xs0 + per_row * (i / ROWS);
    const int q = seg * 64 + lane;                    // 16-k piece
    asm volatile("" : "+v"(x[i]));                    // (or the load sinks below the weights', to its only use)
    if (row < M && q < KC / 16) panel[q * XR + (row ^ ((q >> 2) & (XR - 1)))] = x[i];
  }
  __syncthreads();

  unsigned char* const strip = strips + wave * STRIP;
  for (int parity = 0; tile < tiles; tile += gridDim.x, parity ^= 1) {
    int4_v acc = {0, 0, 0, 0};
    const int next = tile + (int)gridDim.x;
    auto walk = [&](auto more) {
#pragma unroll
      for (int t = 0; t < PAIRS; ++t) {
        const int pair = wave + NW * t;
        u32x4 xv[2];                                  // the panel's operands do not wait for the weights
#pragma unroll
        for (int u = 0; u < 2; ++u) xv[u] = panel[((pair * 2 + u) * 4 + g) * XR + ((j ^ (pair * 2 + u)) & (XR - 1))];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int h = 0; h < 2; ++h) *reinterpret_cast<u32x4*>(strip + h * 1024 + lr * 128 + 16 * (lp ^ lr)) = w[t][h];
        wave_lds_sync();
        if constexpr (more) load_pair(next, t);
#pragma unroll
        for (int u = 0; u < 2; ++u) {                 // (past the end of K: zero weights)
          const u32x4 wv = *reinterpret_cast<const u32x4*>(strip + j * 128 + 16 * ((4 * u + g) ^ (j & 7)));
          acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(int4_v, xv[u]), __builtin_bit_cast(int4_v, wv),
                                                      acc, 0, 0, 0);
        }
        wave_lds_sync();
      }
    };
    if (next < tiles) walk(std::true_type{});
    else walk(std::false_type{});
    // acc[r]: row 4g + r, column j
    int* const red = kOwnRed ? own_red + parity * NW * RED : reinterpret_cast<int*>(strips);
    constexpr int kRedStep = kOwnRed ? RED : STRIP / 4;
    if (4 * g < XR) {
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave * kRedStep + (4 * g + r) * 16 + j] = acc[r];
    }
    __syncthreads();
    if (tid < XR * 16) {
      int sum = 0;
#pragma unroll
      for (int v = 0; v < NW; ++v) sum += red[v * kRedStep + tid];
      if ((tid >> 4) < M) out[(size_t)(tid >> 4) * N + tile * 16 + (tid & 15)] = sum;
    }
    if (!kOwnRed) __syncthreads();
  }
}

__global__ __launch_bounds__(256) void dequant_i32_f16_kernel(const int32_t* __restrict__ acc,
                                                              const half_t* __restrict__ scale,
                                                              float x_scale, half_t* __restrict__ y,
                                                              int M, int N) {
  const size_t total = (size_t)M * N;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (size_t)gridDim.x * blockDim.x) {
    float s = x_scale;
    if (scale != nullptr) s *= static_cast<float>(scale[i % N]);
    y[i] = static_cast<half_t>(static_cast<float>(acc[i]) * s);
  }
}

// ---------------------------------------------------------------------------------------
// w8a16 with both operands staged through wave-private LDS (the int8 sibling of the fp16
// row-load kernel).  Per step a wave loads a 256-byte band (256 k) of the tile's 16 weight rows
// -- 4 rows x 256 B per instruction -- and the matching 512-byte band of the activation rows,
// parks them in LDS strips and reads them back in v_mfma_f32_16x16x32_f16 operand order: 8 bytes
// of one weight row per lane, converted to 8 fp16 there, against 16 bytes of one activation row.
// The activations are fetched once per 16 weight rows instead of once per 4, the dot products run
// on the matrix pipe, and the VALU only converts.  16-column tiles, 8 waves interleaving over K.
// XROWS = activation rows staged: 4, 8 or 16.  Serves what w8_panel leaves: rows too long for w8a16_x_kernel's panel, and
// long ones whose tiles come out even on the CUs without one.
// ---------------------------------------------------------------------------------------
template <int XROWS, int NW, int BW, int CB, int DEPTH = 2>
__global__ __launch_bounds__(64 * NW) void w8a16_r_kernel(const int8_t* __restrict__ Wq,
                                                          const half_t* __restrict__ X,
                                                          const half_t* __restrict__ scale,
                                                          float scalar_scale, float zero_point,
                                                          half_t* __restrict__ Y, int M, int N, int K) {
  // BW: weight bytes (= k) per row and band, 256 or 128.  CB: 16-column blocks per tile sharing the
  // staged activations (tile = 16 * CB columns).  BW = 128 with CB = 2 reads half the activation
  // bytes per weight byte of BW = 256 with CB = 1.
  constexpr int BX = 2 * BW;           // activation bytes per row and band
  constexpr int LPW = BW / 16;         // lanes per weight row piece
  constexpr int RPW = 64 / LPW;        // weight rows per load instruction
  constexpr int WI = 16 * CB / RPW;    // weight load instructions per step
  constexpr int LPX = BX / 16;         // lanes per activation row piece
  constexpr int RPX = 64 / LPX;        // activation rows per load instruction
  constexpr int XI = XROWS / RPX;      // activation load instructions per step
  constexpr int UNITS = BW / 32;       // 32-wide MFMA K units per band
  constexpr int RSW = BW + 16;         // LDS bytes per staged weight row
  constexpr int RSX = BX + 16;         // ... per staged activation row
  constexpr int WSTRIP = 16 * CB * RSW;
  constexpr int XSTRIP = XROWS * RSX;
  constexpr int WAVE_LDS = WSTRIP + XSTRIP;
  static_assert(XROWS % RPX == 0, "whole load instructions");
  static_assert(WAVE_LDS >= 2 * CB * 256 * (int)sizeof(float), "reduction scratch fits");
  __shared__ __attribute__((aligned(16))) unsigned char smem[NW * WAVE_LDS];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int nw = blockDim.x >> 6;
  const int j = lane & 15, g = lane >> 4;          // operand order
  const int hw = lane / LPW, cw = lane % LPW;      // weight load order: row RPW*i + hw, piece cw
  const int hx = lane / LPX, cx = lane % LPX;      // activation load order: row RPX*i + hx, piece cx
  const int n0 = blockIdx.x * (16 * CB);
  const int nbands = (K + BW - 1) / BW;            // K % 128 == 0: the last band may be partial
  // scale of the output this thread writes at the end, fetched ahead of the weight stream
  static_assert(16 * 16 * CB <= 64 * NW, "one output per thread");
  const uint32_t scale_raw =
      scale_fetch(scale, n0 + (int)threadIdx.x % (16 * CB), threadIdx.x < 16 * 16 * CB);
  unsigned char* wstrip = smem + wave * WAVE_LDS;
  unsigned char* xstrip = wstrip + WSTRIP;
  const u32x4 zero = {0u, 0u, 0u, 0u};

  const int8_t* Wp = Wq + (size_t)(n0 + hw) * K + cw * 16;
  const half_t* Xp = X + (size_t)hx * K + cx * 8;
  bool xrow[XI];
#pragma unroll
  for (int i = 0; i < XI; ++i) xrow[i] = (RPX * i + hx) < M;
  const int stw_off = hw * RSW + cw * 16;
  const int stx_off = hx * RSX + cx * 16;
  const int ldw_off = j * RSW + g * 8;
  const int ldx_off = (j % XROWS) * RSX + g * 16;  // MFMA rows beyond XROWS re-read staged rows; unused

  auto load_band = [&](int band, u32x4(&w)[WI], u32x4(&x)[XI]) {
    const bool okw = band < nbands && (band * BW + cw * 16) < K;
    const bool okx = band < nbands && (band * BW + cx * 8) < K;
#pragma unroll
    for (int i = 0; i < WI; ++i)
      w[i] = okw ? load16<true>(Wp + (size_t)(RPW * i) * K + (size_t)band * BW) : zero;
#pragma unroll
    for (int i = 0; i < XI; ++i)
      x[i] = (okx && xrow[i]) ? load16<false>(Xp + (size_t)(RPX * i) * K + (size_t)band * BW) : zero;
  };
  float4_t acc[CB], xacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int b = 0; b < CB; ++b) acc[b] = float4_t{0.f, 0.f, 0.f, 0.f};
  const half8_t ones8 = {static_cast<half_t>(1.f), static_cast<half_t>(1.f), static_cast<half_t>(1.f),
                         static_cast<half_t>(1.f), static_cast<half_t>(1.f), static_cast<half_t>(1.f),
                         static_cast<half_t>(1.f), static_cast<half_t>(1.f)};
  auto multiply = [&](const u32x4(&w)[WI], const u32x4(&x)[XI]) {
#pragma unroll
    for (int i = 0; i < WI; ++i) *reinterpret_cast<u32x4*>(wstrip + stw_off + RPW * i * RSW) = w[i];
#pragma unroll
    for (int i = 0; i < XI; ++i) *reinterpret_cast<u32x4*>(xstrip + stx_off + RPX * i * RSX) = x[i];
    wave_lds_sync();
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const u32x4 xv = *reinterpret_cast<const u32x4*>(xstrip + ldx_off + u * 64);
#pragma unroll
      for (int b = 0; b < CB; ++b) {
        const u32x2 wv = *reinterpret_cast<const u32x2*>(wstrip + b * 16 * RSW + ldw_off + u * 32);
        // bytes as fp16 subnormals: (w + 128) 2^-24, two integer operations fewer per register than
        // building normal numbers and subtracting their bias; the 128 leaves with the zero point
        const uint32_t t0 = wv.x ^ 0x80808080u, t1 = wv.y ^ 0x80808080u;
        const u32x4 wb = {__builtin_amdgcn_perm(0u, t0, 0x04010400u), __builtin_amdgcn_perm(0u, t0, 0x04030402u),
                          __builtin_amdgcn_perm(0u, t1, 0x04010400u), __builtin_amdgcn_perm(0u, t1, 0x04030402u)};
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_half8(xv), as_half8(wb), acc[b], 0, 0, 0);
      }
      xacc = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_half8(xv), ones8, xacc, 0, 0, 0);
    }
    wave_lds_sync();
  };

  // DEPTH bands of a wave in flight or in use: the loads of band t + DEPTH - 1 go out before band t is
  // multiplied
  u32x4 wbuf[DEPTH][WI], xbuf[DEPTH][XI];
  const int nsteps = (nbands + nw - 1) / nw;
  int step = stagger_start(nsteps, 0);
  auto next_band = [&]() {
    const int band = step * nw + wave;
    step = step + 1 == nsteps ? 0 : step + 1;
    return band;
  };
#pragma unroll
  for (int d = 0; d < DEPTH - 1; ++d)
    if (d < nsteps) load_band(next_band(), wbuf[d], xbuf[d]);
  for (int it = 0; it < nsteps; it += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if (it + d >= nsteps) break;
      if (it + d + DEPTH - 1 < nsteps)
        load_band(next_band(), wbuf[(d + DEPTH - 1) % DEPTH], xbuf[(d + DEPTH - 1) % DEPTH]);
      multiply(wbuf[d], xbuf[d]);
    }
  }

  // acc[b][r] = D[m = 4g + r][column 16b + j] (xacc: sum of x of row m in every column); the waves
  // meet in LDS: red[wave][0] = products [16][16*CB], red[wave][1] = activation sums [16][16]
  constexpr int TN = 16 * CB;
  __syncthreads();
  float(*red)[2][16 * TN] = reinterpret_cast<float(*)[2][16 * TN]>(smem);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int b = 0; b < CB; ++b) red[wave][0][(4 * g + r) * TN + 16 * b + j] = acc[b][r];
    red[wave][1][(4 * g + r) * 16 + j] = xacc[r];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 16 * TN; e += blockDim.x) {
    const int m = e / TN, n = n0 + e % TN;
    if (m < M) {
      const float sum = lds_sum<NW>(&red[0][0][e], 2 * 16 * TN, nw);
      const float xs = lds_sum<NW>(&red[0][1][m * 16 + (e & 15)], 2 * 16 * TN, nw);
      float v = sum * 16777216.f - (zero_point + 128.f) * xs;
      if (not_finite(xs))
        v = elementwise_dot<8>(reinterpret_cast<const uint8_t*>(Wq) + (size_t)n * K, X + (size_t)m * K, K, zero_point);
      Y[(size_t)m * N + n] = static_cast<half_t>(v * (scalar_scale * scale_value(scale_raw)));
    }
  }
}

// ---------------------------------------------------------------------------------------
// w4a16 with both operands staged through wave-private LDS (4-bit sibling of w8a16_r_kernel).
// A band is 512 k: 256 bytes of each of the tile's 16 weight rows (4 rows x 256 B per load
// instruction) and 1 KB of each activation row (one row per instruction).  The activations are
// parked already paired the way the nibble conversion produces its halves -- (x0,x4),(x1,x5),
// (x2,x6),(x3,x7) per 8 k -- so the 4 bytes a lane reads per MFMA unit turn into the B operand with
// one shift, four v_and_or and four exact fp16 subtractions, and the dot products run on the
// matrix pipe.  XROWS = activation rows staged (4).
// ---------------------------------------------------------------------------------------
template <int XROWS>
__global__ __launch_bounds__(512) void w4a16_r_kernel(const uint8_t* __restrict__ Wq,
                                                      const half_t* __restrict__ X,
                                                      const half_t* __restrict__ scale,
                                                      float scalar_scale, float zero_point,
                                                      half_t* __restrict__ Y, int M, int N, int K) {
  constexpr int NW = 8;
  constexpr int RSW = 256 + 16;      // LDS bytes per staged weight row (512 k)
  constexpr int RSX = 1024 + 16;     // ... per staged activation row
  constexpr int WSTRIP = 16 * RSW;
  constexpr int XSTRIP = XROWS * RSX;
  constexpr int WAVE_LDS = WSTRIP + XSTRIP;
  static_assert(WAVE_LDS >= 2 * 256 * (int)sizeof(float), "reduction scratch fits");
  __shared__ __attribute__((aligned(16))) unsigned char smem[NW * WAVE_LDS];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int nw = blockDim.x >> 6;
  const int j = lane & 15, g = lane >> 4;        // operand order
  const int hw = lane >> 4, cw = lane & 15;      // weight load order: row 4i + hw, piece cw (32 k)
  const int n0 = blockIdx.x * 16;
  const int nbands = (K + 511) >> 9;             // K % 128 == 0: the last band may be partial
  const size_t rowb = (size_t)K >> 1;            // bytes per weight row
  const bool use_zp = zero_point != 0.f;
  // scale of the output this thread writes at the end, fetched ahead of the weight stream
  const uint32_t scale_raw = scale_fetch(scale, n0 + (int)(threadIdx.x & 15), threadIdx.x < 256);
  unsigned char* wstrip = smem + wave * WAVE_LDS;
  unsigned char* xstrip = wstrip + WSTRIP;
  const u32x4 zero = {0u, 0u, 0u, 0u};

  const uint8_t* Wp = Wq + (size_t)(n0 + hw) * rowb + cw * 16;
  const half_t* Xp = X + lane * 8;
  const int stw_off = hw * RSW + cw * 16;
  const int stx_off = lane * 16;
  const int ldw_off = j * RSW + g * 4;
  const int ldx_off = (j % XROWS) * RSX + g * 16;  // MFMA rows beyond XROWS re-read staged rows; unused

  auto load_band = [&](int band, u32x4(&w)[4], u32x4(&x)[XROWS]) {
    const bool okw = band < nbands && (band * 512 + cw * 32) < K;
    const bool okx = band < nbands && (band * 512 + lane * 8) < K;
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = okw ? load16<true>(Wp + (size_t)(4 * i) * rowb + (size_t)band * 256) : zero;
#pragma unroll
    for (int i = 0; i < XROWS; ++i)
      x[i] = (okx && i < M) ? load16<false>(Xp + (size_t)i * K + (size_t)band * 512) : zero;
  };
  float4_t acc = {0.f, 0.f, 0.f, 0.f}, xacc = {0.f, 0.f, 0.f, 0.f};
  const half8_t ones8 = {static_cast<half_t>(1.f), static_cast<half_t>(1.f), static_cast<half_t>(1.f),
                         static_cast<half_t>(1.f), static_cast<half_t>(1.f), static_cast<half_t>(1.f),
                         static_cast<half_t>(1.f), static_cast<half_t>(1.f)};
  const half2_t b1024 = {static_cast<half_t>(1024.f), static_cast<half_t>(1024.f)};
  const half2_t b64 = {static_cast<half_t>(64.f), static_cast<half_t>(64.f)};
  auto multiply = [&](const u32x4(&w)[4], const u32x4(&x)[XROWS]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(wstrip + stw_off + 4 * i * RSW) = w[i];
#pragma unroll
    for (int i = 0; i < XROWS; ++i) {
      const u32x4 xv = x[i];  // x0..x7 -> (x0,x4) (x1,x5) (x2,x6) (x3,x7)
      const u32x4 xp = {__builtin_amdgcn_perm(xv.z, xv.x, 0x05040100u), __builtin_amdgcn_perm(xv.z, xv.x, 0x07060302u),
                        __builtin_amdgcn_perm(xv.w, xv.y, 0x05040100u), __builtin_amdgcn_perm(xv.w, xv.y, 0x07060302u)};
      *reinterpret_cast<u32x4*>(xstrip + stx_off + i * RSX) = xp;
    }
    wave_lds_sync();
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const u32x4 xa = *reinterpret_cast<const u32x4*>(xstrip + ldx_off + u * 64);
      const uint32_t wd = *reinterpret_cast<const uint32_t*>(wstrip + ldw_off + u * 16), w8 = wd >> 8;
      const half2_t p0 = as_half2((wd & 0x000F000Fu) | 0x64006400u) - b1024;   // (n0, n4)
      const half2_t p1 = as_half2((wd & 0x00F000F0u) | 0x54005400u) - b64;     // (n1, n5)
      const half2_t p2 = as_half2((w8 & 0x000F000Fu) | 0x64006400u) - b1024;   // (n2, n6)
      const half2_t p3 = as_half2((w8 & 0x00F000F0u) | 0x54005400u) - b64;     // (n3, n7)
      const half8_t wb = {p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
      acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_half8(xa), wb, acc, 0, 0, 0);
      if (use_zp) xacc = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_half8(xa), ones8, xacc, 0, 0, 0);
    }
    wave_lds_sync();
  };

  u32x4 w0[4], w1[4], x0[XROWS], x1[XROWS];
  const int nsteps = (nbands + nw - 1) / nw;
  int step = stagger_start(nsteps, 0);
  auto next_band = [&]() {
    const int band = step * nw + wave;
    step = step + 1 == nsteps ? 0 : step + 1;
    return band;
  };
  load_band(next_band(), w0, x0);
  for (int it = 0; it < nsteps; it += 2) {
    if (it + 1 < nsteps) load_band(next_band(), w1, x1);
    multiply(w0, x0);
    if (it + 1 >= nsteps) break;
    if (it + 2 < nsteps) load_band(next_band(), w0, x0);
    multiply(w1, x1);
  }

  // acc[r] = D[m = 4g + r][column j] (xacc: sum of x of row m in every column); waves meet in LDS
  __syncthreads();
  float(*red)[2][256] = reinterpret_cast<float(*)[2][256]>(smem);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    red[wave][0][(4 * g + r) * 16 + j] = acc[r];
    red[wave][1][(4 * g + r) * 16 + j] = xacc[r];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 256; e += blockDim.x) {
    const int m = e >> 4, n = n0 + (e & 15);
    if (m < M) {
      const float sum = lds_sum<NW>(&red[0][0][e], 512, nw);
      const float xs = lds_sum<NW>(&red[0][1][e], 512, nw);
      float v = sum - zero_point * xs;
      if (not_finite(xs)) v = elementwise_dot<4>(Wq + (size_t)n * rowb, X + (size_t)m * K, K, zero_point);
      Y[(size_t)m * N + n] = static_cast<half_t>(v * (scalar_scale * scale_value(scale_raw)));
    }
  }
}

// ---------------------------------------------------------------------------------------
// w4a16, two to four activation rows: all activations in LDS as one panel (4 rows x KC k, 8 bytes a k), staged
// once a workgroup, which then walks over column tiles of 16; the weights of a tile go from memory through
// registers and two KB of wave-private LDS into MFMA operands.  Launched with K <= KC.
//  * All loads are row-contiguous: eight lanes read the 128 bytes of a line.  A CU takes 64 bytes a clock
//    that way; where neighbouring lanes sit on different rows, as the operand order of the MFMA would have it,
//    it takes 18 (measured: reads of L2-resident data on every CU, 129 GB/s a CU against 38).
//  * Every wave has its whole share of a tile in flight; the registers of a load are filled again, with the next
//    tile's, as soon as it has been parked.
//  * Lane (j, g) takes 16 bytes = 32 k of row j: four words of eight nibbles.  The even nibbles of
//    two words make one MFMA operand (nibbles 0,4,2,6 of each), the odd ones a second: masked in
//    place they are fp16 subnormals, n 2^-24 and n 2^-20, exactly, so five integer operations
//    decode eight weights and two accumulators keep the two powers of two apart.
//  * The panel lies in LDS in that order: 16-byte pieces [128 k][word pair][even, odd][g][row], so one
//    operand read of a wave covers 256 contiguous bytes (the lanes of rows 4..15 repeat rows 0..3).  The rows
//    of a group are permuted by its number: the threads that stage it have consecutive k of one row.
//  * The row sums for the zero point are taken while the panel is staged.
// Loads return in order, so their order counts: activations, then the scales (cold), then the weights (the scales
// last: 0.35 us more on every call).
// What bounds it: the way of the weights through LDS, one pair after the other in every wave (park, wait, read, decode,
// multiply), which the loads hide only in part.  M=4, weights from memory, us: N=4096 K=14336 (eight waves, seven pairs each)
// 9.6; an empty kernel of its LDS and waves 1.7, the kernel with every load answered by zeros at once 6.9, with the
// activations' loads alone 7.1, with the weights' alone 9.0.  N = K = 8192 8.8, 1.7, 6.3, 6.2, 8.5; N = K = 4096 4.1, 1.7,
// 3.6, 3.6, 3.9.  Against the same panel with the loads in operand order and one tile a workgroup: N=4096 K=14336 11.8 / 9.6,
// N = K = 8192 10.9 / 8.8, N=14336 K=4096 9.1 / 7.9, N=28672 K=2304 11.2 / 8.9, N=4096 K=4096 4.4 / 4.1.
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ float wave_sum(float v) {
  v = row16_allreduce(v);
  float s = 0.f;
#pragma unroll
  for (int r = 0; r < 4; ++r) s += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 16 * r));
  return s;
}
template <int KC, int NW>
__global__ __launch_bounds__(64 * NW) void w4a16_x_kernel(const uint8_t* __restrict__ Wq, const half_t* __restrict__ X,
                                                      const half_t* __restrict__ scale, float scalar_scale,
                                                      float zero_point, half_t* __restrict__ Y, int M, int N, int K) {
  constexpr int PAIRS = KC / 256 / NW;           // 16 rows x 128 bytes of weights: two loads a wave
  constexpr int SEGS = KC / 512 / (NW / 4);      // 1 KB of an activation row: one load a wave
  static_assert(KC % (256 * NW) == 0 && KC % (128 * NW) == 0, "whole pairs and segments");
  constexpr int STRIP = 2048;
  constexpr bool kOwnRed = KC * 8 + NW * (STRIP + 2 * 516) <= 160 * 1024 - 64;
  constexpr int RED = 129;                       // floats a wave hands over: two powers of two of 4 x 16 sums, one row sum
  __shared__ u32x4 panel[KC / 2];
  __shared__ __attribute__((aligned(16))) unsigned char strips[NW * STRIP];
  __shared__ float own_red[kOwnRed ? 2 * NW * RED : 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, g = lane >> 4;        // operand order
  const int lr = lane >> 3, lp = lane & 7;       // load order: row, 16-byte piece of its 128
  const size_t rowb = (size_t)K >> 1;
  constexpr int kNonTemporal = 2;
  constexpr int kBeyond = 0x7ffffff0;            // past the descriptors: the load returns zeros

  // activations first: loads return in order, and the panel must not wait for the weights
  const int per_row = M == 2 ? NW / 2 : (M == 3 ? NW / 3 : NW / 4);  // waves that stage a row
  const int xm = wave / per_row, xs0 = wave - xm * per_row;
  const __amdgpu_buffer_rsrc_t xrs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(X + (size_t)xm * K), 0, xm < M ? K * 2 : 0, 0x00020000);
  u32x4 x[SEGS];
#pragma unroll
  for (int i = 0; i < SEGS; ++i)
    x[i] = __builtin_bit_cast(
        u32x4, __builtin_amdgcn_raw_buffer_load_b128(xrs, (xs0 + per_row * i) * 1024 + lane * 16, 0, 0));
  __builtin_amdgcn_sched_barrier(0);

  u32x4 w[PAIRS][2];
  int w_off[PAIRS];
#pragma unroll
  for (int t = 0; t < PAIRS; ++t) {
    const int kb = (wave + NW * t) * 128 + lp * 16;
    w_off[t] = kb < (int)rowb ? lr * (int)rowb + kb : kBeyond;
  }
  const int tiles = N >> 4;
  auto load_pair = [&](int tile, int t) {
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(Wq + (size_t)tile * 16 * rowb), 0, tile < tiles ? (int)(16 * rowb) : 0, 0x00020000);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      w[t][h] = __builtin_bit_cast(
          u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                     wrs, w_off[t] == kBeyond ? kBeyond : w_off[t] + 8 * h * (int)rowb, 0, kNonTemporal));
  };
  int tile = blockIdx.x;
  // scale of the output this thread writes, ahead of the tile's weights
  uint32_t scale_raw = scale_fetch(scale, tile * 16 + ((tid >> 2) & 15), tid < 256);
#pragma unroll
  for (int t = 0; t < PAIRS; ++t) {
    load_pair(tile, t);
    __builtin_amdgcn_sched_barrier(0);           // in this order: they are waited for one after the other
  }
  __builtin_amdgcn_sched_barrier(0);

  const half2_t ones = {static_cast<half_t>(1.f), static_cast<half_t>(1.f)};
  float xsum = 0.f;
#pragma unroll
  for (int i = 0; i < SEGS; ++i) {
    const int seg = xs0 + per_row * i;
    if (xm < M && seg * 512 < KC) {
      const u32x4 a = x[i];
#pragma unroll
      for (int c = 0; c < 4; ++c) xsum = __builtin_amdgcn_fdot2(as_half2(a[c]), ones, xsum, false);
      constexpr uint32_t kLow = 0x05040100u, kHigh = 0x07060302u;
      const int q = seg * 32 + (lane >> 1);      // 16-k group
      const int piece = (q >> 3) * 64 + (q & 1) * 32 + ((q >> 1) & 3) * 4 + (xm ^ ((q >> 3) & 3));
      u32x2* at = reinterpret_cast<u32x2*>(panel + piece) + (lane & 1);
      at[0] = u32x2{__builtin_amdgcn_perm(a.z, a.x, kLow), __builtin_amdgcn_perm(a.w, a.y, kLow)};
      at[32] = u32x2{__builtin_amdgcn_perm(a.z, a.x, kHigh), __builtin_amdgcn_perm(a.w, a.y, kHigh)};
    }
  }
  __syncthreads();
  xsum = wave_sum(xsum);

  unsigned char* const strip = strips + wave * STRIP;
  for (int parity = 0; tile < tiles; tile += gridDim.x, parity ^= 1) {
    float4_t even = {0.f, 0.f, 0.f, 0.f}, odd = {0.f, 0.f, 0.f, 0.f};
    const int next = tile + (int)gridDim.x;
    const uint32_t scale_now = scale_raw;
    scale_raw = scale_fetch(scale, next * 16 + ((tid >> 2) & 15), tid < 256 && next < tiles);
#pragma unroll
    for (int t = 0; t < PAIRS; ++t) {
      const int pair = wave + NW * t;
      // the panel's operands do not wait for the weights
      u32x4 xe[2][2], xo[2][2];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const u32x4* at = panel + ((pair * 2 + u) * 2 + p) * 32 + g * 4 + ((j ^ (pair * 2 + u)) & 3);
          xe[u][p] = at[0];
          xo[u][p] = at[16];
        }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < 2; ++h) *reinterpret_cast<u32x4*>(strip + h * 1024 + lr * 128 + 16 * (lp ^ lr)) = w[t][h];
      wave_lds_sync();
      load_pair(next, t);
#pragma unroll
      for (int u = 0; u < 2; ++u) {              // (past the end of K: zero weights on a zero panel)
        const u32x4 wv = *reinterpret_cast<const u32x4*>(strip + j * 128 + 16 * ((4 * u + g) ^ (j & 7)));
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const uint32_t a = wv[2 * p], b = wv[2 * p + 1], a8 = a >> 8, b8 = b >> 8;
          const u32x4 we = {a & 0x000F000Fu, a8 & 0x000F000Fu, b & 0x000F000Fu, b8 & 0x000F000Fu};  // 0,4 2,6 of both
          const u32x4 wo = {a & 0x00F000F0u, a8 & 0x00F000F0u, b & 0x00F000F0u, b8 & 0x00F000F0u};  // 1,5 3,7
          even = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_half8(xe[u][p]), as_half8(we), even, 0, 0, 0);
          odd = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_half8(xo[u][p]), as_half8(wo), odd, 0, 0, 0);
        }
      }
      wave_lds_sync();
    }
    // lanes 0..15 hold rows 0..3 of column j in registers 0..3
    float* const red = kOwnRed ? own_red + parity * NW * RED : reinterpret_cast<float*>(strips);
    constexpr int kRedStep = kOwnRed ? RED : STRIP / 4;
    if (lane < 16) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        red[wave * kRedStep + r * 16 + j] = even[r];
        red[wave * kRedStep + 64 + r * 16 + j] = odd[r];
      }
    }
    if (lane == 0) red[wave * kRedStep + 128] = xsum;
    __syncthreads();
    // four threads an output: a quarter of the waves each
    if (tid < 256) {
      const int e = tid >> 2, m = e >> 4, n = tile * 16 + (e & 15), part = tid & 3;
      const float* const r = red + part * (NW / 4) * kRedStep + e;
      float v = lds_sum<NW / 4>(r, kRedStep, NW / 4) * 16777216.f + lds_sum<NW / 4>(r + 64, kRedStep, NW / 4) * 1048576.f;
      v += dpp_f32<0xB1>(v);
      v += dpp_f32<0x4E>(v);
      if (part == 0 && m < M) {
        const float xs = lds_sum<NW / 2>(red + m * per_row * kRedStep + 128, kRedStep, per_row);
        v -= zero_point * xs;
        if (not_finite(xs)) v = elementwise_dot<4>(Wq + (size_t)n * rowb, X + (size_t)m * K, K, zero_point);
        Y[(size_t)m * N + n] = static_cast<half_t>(v * (scalar_scale * scale_value(scale_now)));
      }
    }
    if (!kOwnRed) __syncthreads();
  }
}

// ---------------------------------------------------------------------------------------
// w8a16, two to sixteen activation rows whose panel fits LDS: as w4a16_x_kernel above.  A workgroup stages the panel
// once, XR rows (4, 8 or 16; M <= XR) of K fp16 in operand order, and walks over 16-column tiles with only weights left
// to load.  The row-load kernel reads the activations again for every tile, and a CU takes HBM and L2 lines in the order
// it asked for them, some 50 GB/s together: with 16 rows the activations are two thirds of its bytes.  Lane (j, g) takes
// 16 bytes = 16 k of row j, the operands of two MFMAs; the panel's 16-byte pieces lie as [64 k][lower, upper 8 k of a
// lane's 16][g][row], the rows of a piece permuted by its number against bank conflicts.  With few waves (NW < XR) a wave
// stages several rows.  Bound by HBM for outputs of several tiles a CU (N=128256 K=2048, sixteen rows 44.2 us, 5.9 TB/s;
// row-load kernel 86.7), by the panel's way through L2 and the first weights' latency for one.  us, before / this one:
//   M=16  4096 x 4096 7.4 / 6.4   8192 x 2048 7.1 / 5.6   14336 x 4096 17.1 / 12.8   28672 x 1024 14.8 / 7.5
//   M=8   5120 x 5120 10.4 / 8.5  11008 x 4096 14.2 / 10.1   8192 x 8192 15.1 / 14.3   14336 x 4096 13.0 / 12.2
//   M=4   4096 x 4096 6.1 / 5.4   8192 x 2048 5.8 / 4.9   28672 x 2048 13.0 / 10.9   M=2 4096 x 2048 4.3 / 3.6
// Launched with K <= KC.
// ---------------------------------------------------------------------------------------
template <int XR, int KC, int NW>
__global__ __launch_bounds__(64 * NW) void w8a16_x_kernel(const int8_t* __restrict__ Wq, const half_t* __restrict__ X,
                                                          const half_t* __restrict__ scale, float scalar_scale,
                                                          float zero_point, half_t* __restrict__ Y, int M, int N, int K) {
  constexpr int PAIRS = KC / 128 / NW;                // 16 rows x 128 bytes of weights: two loads a wave
  constexpr int SEGS = KC / 512 * XR / NW;            // 1 KB of an activation row: one load a wave
  static_assert(KC % (128 * NW) == 0 && KC % 512 == 0 && KC / 512 * XR % NW == 0, "whole pairs and segments");
  constexpr int ROWS = NW < XR ? XR / NW : 1;         // rows a wave stages; or NW / M waves stage a row
  constexpr int STRIP = 2048, RED = XR * 16 + ROWS;   // floats a wave hands over: sums, and its parts of sums of x
  constexpr bool kOwnRed = XR * KC * 2 + NW * (STRIP + 8 * RED) <= 160 * 1024 - 64;
  __shared__ u32x4 panel[XR * KC / 8];
  __shared__ __attribute__((aligned(16))) unsigned char strips[NW * STRIP];
  __shared__ float own_red[kOwnRed ? 2 * NW * RED : 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, g = lane >> 4;             // operand order
  const int lr = lane >> 3, lp = lane & 7;            // load order: row, 16-byte piece of its 128
  constexpr int kNonTemporal = 2;
  constexpr int kBeyond = 0x7ffffff0;                 // past the descriptors: the load returns zeros
  constexpr int kShift = XR == 16 ? 0 : (XR == 8 ? 1 : 2);
  auto place = [&](int piece, int row) { return piece * XR + (row ^ ((piece >> kShift) & (XR - 1))); };
  // activations first: loads return in order, and the panel must not wait for the weights
  int per_row = NW < XR ? 1 : NW / XR;                // waves that stage a row: NW / M
  if constexpr (XR == 4) per_row = M == 2 ? NW / 2 : (M == 3 ? NW / 3 : NW / 4);
  else if constexpr (XR == 8 && NW == 16) per_row = M == 5 ? 3 : 2;
  const int xm = NW < XR ? wave * ROWS : wave / per_row, xs0 = wave - wave / per_row * per_row;
  u32x4 x[SEGS];
#pragma unroll
  for (int i = 0; i < SEGS; ++i) {
    const int m = xm + i % ROWS;
    const __amdgpu_buffer_rsrc_t xrs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(X + (size_t)m * K), 0, m < M ? K * 2 : 0, 0x00020000);
    x[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                         xrs, (xs0 + per_row * (i / ROWS)) * 1024 + lane * 16, 0, 0));
  }
  __builtin_amdgcn_sched_barrier(0);
  const int tiles = N >> 4;
  int tile = blockIdx.x;
  // scale of the output this thread writes, ahead of the tile's weights
  uint32_t scale_raw = scale_fetch(scale, tile * 16 + j, tid < XR * 16);
  u32x4 w[PAIRS][2];
  int w_off[PAIRS];
#pragma unroll
  for (int t = 0; t < PAIRS; ++t) {
    const int kb = (wave + NW * t) * 128 + lp * 16;
    w_off[t] = kb < K ? lr * K + kb : kBeyond;
  }
  auto load_pair = [&](int of, int t) {
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(Wq + (size_t)of * 16 * K), 0, of < tiles ? 16 * K : 0, 0x00020000);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      w[t][h] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                              wrs, w_off[t] == kBeyond ? kBeyond : w_off[t] + 8 * h * K, 0, kNonTemporal));
  };
#pragma unroll
  for (int t = 0; t < PAIRS; ++t) {
    load_pair(tile, t);
    __builtin_amdgcn_sched_barrier(0);                // in this order: they are waited for one after the other
  }
  const half2_t ones = {static_cast<half_t>(1.f), static_cast<half_t>(1.f)};
  float xsum[ROWS] = {};
#pragma unroll
  for (int i = 0; i < SEGS; ++i) {
    const int m = xm + i % ROWS, k8 = (xs0 + per_row * (i / ROWS)) * 64 + lane;   // row, 8-k group
    asm volatile("" : "+v"(x[i]));                    // (or the load sinks below the weights', to its only use)
#pragma unroll
    for (int c = 0; c < 4; ++c) xsum[i % ROWS] = __builtin_amdgcn_fdot2(as_half2(x[i][c]), ones, xsum[i % ROWS], false);
    if (m < M && k8 < KC / 8) panel[place((k8 >> 3) * 8 + (k8 & 1) * 4 + ((k8 >> 1) & 3), m)] = x[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < ROWS; ++i) xsum[i] = wave_sum(xsum[i]);

  unsigned char* const strip = strips + wave * STRIP;
  for (int parity = 0; tile < tiles; tile += gridDim.x, parity ^= 1) {
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
    const int next = tile + (int)gridDim.x;
    const uint32_t scale_now = scale_raw;
    scale_raw = scale_fetch(scale, next * 16 + j, tid < XR * 16 && next < tiles);
    auto walk = [&](auto more) {
#pragma unroll
      for (int t = 0; t < PAIRS; ++t) {
        const int pair = wave + NW * t;
        u32x4 xv[2][2];                               // the panel's operands do not wait for the weights
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int h = 0; h < 2; ++h) xv[u][h] = panel[place(((pair * 2 + u) * 2 + h) * 4 + g, j & (XR - 1))];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int h = 0; h < 2; ++h) *reinterpret_cast<u32x4*>(strip + h * 1024 + lr * 128 + 16 * (lp ^ lr)) = w[t][h];
        wave_lds_sync();
        if constexpr (more) load_pair(next, t);
#pragma unroll
        for (int u = 0; u < 2; ++u) {                 // (past the end of K: zero activations)
          const u32x4 wv = *reinterpret_cast<const u32x4*>(strip + j * 128 + 16 * ((4 * u + g) ^ (j & 7)));
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            // bytes as fp16 subnormals, (w + 128) 2^-24; the 128 leaves with the zero point
            const uint32_t t0 = wv[2 * h] ^ 0x80808080u, t1 = wv[2 * h + 1] ^ 0x80808080u;
            const u32x4 wb = {__builtin_amdgcn_perm(0u, t0, 0x04010400u), __builtin_amdgcn_perm(0u, t0, 0x04030402u),
                              __builtin_amdgcn_perm(0u, t1, 0x04010400u), __builtin_amdgcn_perm(0u, t1, 0x04030402u)};
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_half8(xv[u][h]), as_half8(wb), acc, 0, 0, 0);
          }
        }
        wave_lds_sync();
      }
    };
    if (NW == 8 && next >= tiles) walk(std::false_type{});
    else walk(std::true_type{});
    // acc[r]: row 4g + r, column j
    float* const red = kOwnRed ? own_red + parity * NW * RED : reinterpret_cast<float*>(strips);
    constexpr int kRedStep = kOwnRed ? RED : STRIP / 4;
    if (4 * g < XR) {
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave * kRedStep + (4 * g + r) * 16 + j] = acc[r];
    }
    if (lane == 0) {
#pragma unroll
      for (int i = 0; i < ROWS; ++i) red[wave * kRedStep + XR * 16 + i] = xsum[i];
    }
    __syncthreads();
    if (tid < XR * 16 && (tid >> 4) < M) {
      const int m = tid >> 4, n = tile * 16 + j;
      const float sum = lds_sum<NW>(red + tid, kRedStep, NW);
      const float* const xr = red + (m / ROWS) * per_row * kRedStep + XR * 16 + m % ROWS;
      const float xs = lds_sum<(NW < XR ? 1 : XR == 4 ? NW / 2 : NW / XR + 1)>(xr, kRedStep, per_row);
      float v = sum * 16777216.f - (zero_point + 128.f) * xs;
      if (not_finite(xs))
        v = elementwise_dot<8>(reinterpret_cast<const uint8_t*>(Wq) + (size_t)n * K, X + (size_t)m * K, K, zero_point);
      Y[(size_t)m * N + n] = static_cast<half_t>(v * (scalar_scale * scale_value(scale_now)));
    }
    if (!kOwnRed) __syncthreads();
  }
}

// ---------------------------------------------------------------------------------------
// Host launchers.  The integer-dot kernel, beyond what i8i8_go says of two to four rows: rows per workgroup
// 8 when that still yields >= 512 workgroups, else 4; waves as many (<= 4) as the row has 1 KB pieces.
// ---------------------------------------------------------------------------------------
static int i8_waves(int K) {
  const int pieces = (K / 16 + 63) / 64;
  return pieces >= 4 ? 4 : (pieces >= 2 ? 2 : 1);
}

// One activation row.  A wave's chunk is 1 KB of each weight row (2048 k of int4 in four units a
// lane, 1024 k of int8 in two); a workgroup has as many waves as K has chunks, up to 8, rounded up
// to a power of two, and takes four weight rows -- two when the whole matrix is 8 MiB or less,
// where four rows leave too few workgroups.  Measured, us per call, previous kernels -> these
// (N x K): int4 8192 x 8192 10.6 -> 8.7, 4096 x 4096 5.7 -> 4.1, 28672 x 4096 16.2 -> 11.6,
// 4096 x 14336 10.1 -> 8.1, 16384 x 16384 27.9 -> 24.5; int8 8192 x 8192 13.3 -> 12.1,
// 4096 x 4096 5.7 -> 5.25, 28672 x 4096 20.8 -> 18.8, 4096 x 14336 12.6 -> 11.4, 16384 x 16384
// 41.9 -> 40.6.  int8 with four units a lane (2 KB of a row per wave): 8192 x 8192 13.0.
// Loads through buffer descriptors that end with the row (no predicate, so no branch around each of
// the 10 .. 20 small loads of a chunk), six alternating runs each: int4 8192 x 8192 8.57 -> 8.15, 4096
// x 4096 4.08 -> 3.98; int8 12.25 -> 12.17, 5.30 -> 5.21.
// Two activation rows of int4 (MR = 2) against the row-load MFMA kernel: 8192 x 8192 11.4 -> 10.6,
// 4096 x 4096 5.7 -> 5.0, 4096 x 14336 11.6 -> 10.7, 28672 x 4096 level; the second row costs 2 us at
// 8192 x 8192 because its x traffic (64 MiB from L2) is twice the weights'; eight weight rows a
// workgroup to halve it lose more in occupancy (11.9).  (Now only where the panel kernel does not pay.)
template <int BITS, int MR>
static void launch_wq_m1(const W8A16Args& a, hipStream_t s) {
  auto* Wq = static_cast<const uint8_t*>(a.Wq);
  auto* X = static_cast<const half_t*>(a.x);
  auto* sc = static_cast<const half_t*>(a.scale);
  auto* Y = static_cast<half_t*>(a.y);
  constexpr int UD = BITS == 4 ? 4 : 2;
  const int chunks = (a.K + 512 * UD - 1) / (512 * UD);
  const bool small = (size_t)a.N * a.K * BITS / 8 <= (8u << 20);
#define FG_WQ_M1(RN, NWV)                                                                         \
  hipLaunchKernelGGL((wq_m1_kernel<BITS, RN, NWV, UD, MR>), dim3(a.N / RN), dim3(64 * NWV), 0, s, Wq, \
                     X, sc, a.scalar_scale, a.zero_point, Y, a.N, a.K)
#define FG_WQ_M1_ROWS(NWV) \
  if (small) FG_WQ_M1(2, NWV); else FG_WQ_M1(4, NWV)
  if (chunks > 4) { FG_WQ_M1_ROWS(8); }
  else if (chunks > 2) { FG_WQ_M1_ROWS(4); }
  else if (chunks > 1) { FG_WQ_M1_ROWS(2); }
  else { FG_WQ_M1_ROWS(1); }
#undef FG_WQ_M1_ROWS
#undef FG_WQ_M1
}

// Workgroups of a panel kernel: one a CU walks over up to `each` tiles, more where there are more tiles and LDS holds
// them (`most`).  What a workgroup has in flight is one tile, 16 weight rows, and short rows leave a CU idle (int4 M=4
// N=28672 K=2304 one / two a CU 11.9 / 8.9 us, K=1024 two / four 6.0 / 5.6), while for two tiles of longer rows a second
// workgroup only stages the panel again (N=8192 K=3072 5.4 / 5.8, K=2048 3.9 / 4.2; K=1024 the other way, 3.4 / 3.3).
static int panel_grid(int tiles, int cus, int each, int most) {
  return std::min(tiles, cus * std::min(most, (tiles + each * cus - 1) / (each * cus)));
}
// Panel kernel (w8a16_x_kernel): where it measured ahead of the row-load and lanes-over-x kernels (us, the better of
// those / this one):
//  * nine rows and more, wherever the panel fits: N=512 K=128 3.1 / 2.6, N=4096 K=4096 7.4 / 6.4, N=28672 K=2048 23.5 /
//    11.8, N=14336 K=4096 17.1 / 12.8;
//  * five to eight: N = K = 512 3.1 / 2.5, N=5120 K=5120 10.4 / 8.5, N = K = 8192 14.9 / 14.1 -- except one tile of long
//    rows on nearly every CU, which waits for the panel with little to spread it over (N=4096 K=6400 8.6 / 8.9, K=8192
//    9.6 / 9.8; N=3584 K=7168 8.8 / 8.6);
//  * two to four, for which the others read few activations: K <= 2048 (N=28672 K=1536 11.5 / 8.6, N=512 K=1792 3.3 /
//    2.9), and from there outputs wide enough to pay for the panel.  Four: N=1024 K=3072 4.0 / 3.7, N=512 K=2560 3.5 /
//    3.6; N=1536 K=4608 5.7 / 5.2, N=1024 K=4096 4.4 / 4.5.  Three: N=1536 K=2560 4.0 / 3.7, N=512 3.3 / 3.6; N=2048
//    K=4096 4.9 / 4.7, N=1536 4.4 / 4.6; N=3072 K=8192 8.5 / 7.8, N=1536 6.6 / 7.0.  Two: N=2048 K=3072 3.9 / 3.8; N=4096
//    K=4096 5.9 / 5.4, N=2048 4.3 / 4.6, N=14336 12.5 / 12.1, N=5120 6.5 / 6.9 (the second round a quarter full);
//    N=11008 K=8192 18.0 / 16.4, N=3072 7.4 / 7.7;
//  * not K > 6144 where 16-column tiles come out even, N = 8192 K=8192 four rows 12.9 / 13.2, two 11.5 / 11.9 at K=7168.
static bool w8_panel(const W8A16Args& a) {
  const int tiles = a.N / 16, cus = compute_units(), rounds = (tiles + cus - 1) / cus;
  if (a.M >= 9) return a.K <= 4096;
  if (a.M >= 5) return a.K <= 6144 || (a.K <= 8192 && (8 * tiles <= 7 * cus || rounds > 1));
  if (a.K <= 2048) return true;
  if (a.K > 8192 || (a.K > 6144 && tiles == rounds * cus)) return false;
  if (a.M == 4) return 8 * tiles >= (a.K <= 3072 ? 2 : 3) * cus;
  if (a.M == 3) return 4 * tiles >= (a.K <= 3072 ? 1 : (a.K <= 6144 ? 2 : 3)) * cus;
  if (a.K <= 3072 && rounds <= 2) return 2 * tiles >= cus;
  if (rounds == 1) return a.K <= 6144 && 8 * tiles >= 5 * cus;
  return 4 * tiles > 3 * rounds * cus;
}
static void launch_w8_panel(const W8A16Args& a, hipStream_t s) {
  // KC: the smallest that holds K.  Few waves with several pairs each where that keeps loads enough in flight (us, eight
  // rows, one way / the other: N=8192 K=2560 eight waves of three pairs 6.7 / four of five 5.7; K=5120 sixteen waves 10.6
  // / eight of five 10.0; K=7168 12.4 sixteen / 11.5 eight of seven); more where one tile is all a workgroup does (N=1024
  // K=2048 four / eight 3.7 / 3.5), and at K = 4096 sixteen of two pairs (N=8192 eight of four 8.7 / 8.1).
  const int tiles = a.N / 16, cus = compute_units();
  const bool many = tiles > cus;
#define FG_W8_X(XR, KC, NW, MOST)                                                                                  \
  hipLaunchKernelGGL((w8a16_x_kernel<XR, KC, NW>), dim3(panel_grid(tiles, cus, KC <= 512 ? 1 : 2, MOST)), dim3(64 * NW), \
                     0, s, static_cast<const int8_t*>(a.Wq), static_cast<const half_t*>(a.x),                      \
                     static_cast<const half_t*>(a.scale), a.scalar_scale, a.zero_point, static_cast<half_t*>(a.y), \
                     a.M, a.N, a.K)
  if (a.M <= 4) {
    if (a.K <= 512) FG_W8_X(4, 512, 4, 4);
    else if (a.K <= 1024) FG_W8_X(4, 1024, 8, 4);
    else if (a.K <= 1536) FG_W8_X(4, 1536, 4, 4);
    else if (a.K <= 2048) FG_W8_X(4, 2048, 8, 2);
    else if (a.K <= 2560) FG_W8_X(4, 2560, 4, 3);
    else if (a.K <= 3072) FG_W8_X(4, 3072, 8, 2);
    else if (a.K <= 4096 && !many) FG_W8_X(4, 4096, 8, 1);
    else if (a.K <= 4096) FG_W8_X(4, 4096, 16, 1);
    else if (a.K <= 5120) FG_W8_X(4, 5120, 8, 1);
    else if (a.K <= 6144 && !many) FG_W8_X(4, 6144, 8, 1);
    else if (a.K <= 6144) FG_W8_X(4, 6144, 16, 1);
    else if (a.K <= 7168) FG_W8_X(4, 7168, 8, 1);
    else FG_W8_X(4, 8192, 16, 1);
  } else if (a.M <= 8) {
    if (a.K <= 512) FG_W8_X(8, 512, 4, 4);
    else if (a.K <= 1024) FG_W8_X(8, 1024, 8, 3);
    else if (a.K <= 1536) FG_W8_X(8, 1536, 4, 3);
    else if (a.K <= 2048 && !many) FG_W8_X(8, 2048, 8, 1);
    else if (a.K <= 2048) FG_W8_X(8, 2048, 4, 2);
    else if (a.K <= 2560) FG_W8_X(8, 2560, 4, 2);
    else if (a.K <= 3072) FG_W8_X(8, 3072, 8, 2);
    else if (a.K <= 4096 && !many) FG_W8_X(8, 4096, 8, 1);
    else if (a.K <= 4096) FG_W8_X(8, 4096, 16, 1);
    else if (a.K <= 5120) FG_W8_X(8, 5120, 8, 1);
    else if (a.K <= 6144) FG_W8_X(8, 6144, 8, 1);
    else if (a.K <= 7168) FG_W8_X(8, 7168, 8, 1);
    else FG_W8_X(8, 8192, 16, 1);
  } else {
    if (a.K <= 512) FG_W8_X(16, 512, 4, 4);
    else if (a.K <= 1024) FG_W8_X(16, 1024, 4, 2);
    else if (a.K <= 2048 && !many) FG_W8_X(16, 2048, 8, 1);
    else if (a.K <= 2048) FG_W8_X(16, 2048, 4, 1);
    else if (a.K <= 3072 && !many) FG_W8_X(16, 3072, 8, 1);
    else if (a.K <= 3072) FG_W8_X(16, 3072, 4, 1);
    else FG_W8_X(16, 4096, 16, 1);
  }
#undef FG_W8_X
}

// An earlier kernel with lanes along K (16 weight bytes a lane) against the row-load kernel on 256-byte
// bands, us per call: K = N = 8192 M=1 12.6 / 14.3, M=2 15.1 / 14.2, M=4 21.1 / 14.9, M=8 32.9 / 17.2.
// The row-load kernel exists with 8 waves only.
bool launch_w8a16(const W8A16Args& a, hipStream_t s) {
  auto* Wq = static_cast<const int8_t*>(a.Wq);
  auto* X = static_cast<const half_t*>(a.x);
  auto* sc = static_cast<const half_t*>(a.scale);
  auto* Y = static_cast<half_t*>(a.y);
  const int t32 = a.N / 32;
  // 32-column tiles on 128-byte bands read half the activation bytes per weight byte.  Measured
  // against 16-column tiles (us):
  //  * two workgroups (16 waves) on every CU, 448..512 tiles or a multiple of 512: K = N = 16384 M=8
  //    44.8 / 49.3 -- but not with rows 8 KB apart: K=8192 N=16384 M=8 27.6 / 25.2;
  //  * one workgroup on every CU (N = 8192): long rows or 12..16 activation rows only, K=16384 M=8
  //    25.4 / 27.3, K=28672 M=14 47.8 / 55.4, against K=28672 M=4 40.0 / 38.7;
  //  * 13..16 rows from 160 tiles on: N=5120 K=11008 M=16 19.5 / 23.0, N=14336 K=14336 44.5 / 55.1.
  const bool aligned = a.N % 32 == 0;
  const bool two_per_cu = aligned && ((t32 >= 448 && t32 <= 512) || (t32 >= 512 && t32 % 512 == 0)) &&
                          (a.K != 8192 || a.M > 8);
  const bool one_per_cu = aligned && t32 == 256 &&
                          (a.M >= 12 || (a.K >= 16384 && (a.M >= 5 || a.K < 24576)));
  const bool many_rows = aligned && a.M >= 13 && t32 >= 160 && t32 != 256;
  const bool wide = two_per_cu || one_per_cu || many_rows;
  // 16-column tiles take 128-byte bands (smaller strips, more steps in flight): M=8, 128- / 256-byte
  // bands: K=11008 N=5120 17.7 / 19.3 -- except long rows of narrow outputs, K=14336 N=4096 M=4 14.8 / 13.9.
  const bool bw256 = a.N <= 4096 && a.K >= 14336;
#define FG_W8A16_R(XR, BW, CB)                                                                    \
  hipLaunchKernelGGL((w8a16_r_kernel<XR, 8, BW, CB>), dim3(a.N / (16 * CB)), dim3(512), 0, s, Wq, \
                     X, sc, a.scalar_scale, a.zero_point, Y, a.M, a.N, a.K)
  // Two rows run the lanes-over-x kernel on two rows -- except where the 16-column tiles of the row-load
  // kernel fill the CUs evenly (us, two-row kernel / row-load kernel: K=14336 N=4096 13.2 / 14.7; N=2048 K=8192
  // 6.1 / 6.8; but N=8192 K=8192 14.6 / 13.5, K=11008 18.4 / 17.0; N=16384 K=8192 25.5 / 23.5).  Three and four
  // rows only against narrow outputs, which leave the row-load kernel on half the CUs or fewer (M=4: N=1024
  // K=4096 4.5 / 5.3, N=2048 K=8192 7.8 / 8.1).
  const bool even_tiles = a.N % 8192 == 0;
  if (a.M == 1) {
    launch_wq_m1<8, 1>(a, s);
  } else if (w8_panel(a)) {
    launch_w8_panel(a, s);
  } else if (a.M == 2 && !even_tiles) {
    launch_wq_m1<8, 2>(a, s);
  } else if (a.M == 3 && a.N <= 2048) {
    launch_wq_m1<8, 3>(a, s);
  } else if (a.M == 4 && a.N <= 2048) {
    launch_wq_m1<8, 4>(a, s);
  } else if (a.M <= 4) {  // (two rows take the 4-row strip too)
    if (wide) FG_W8A16_R(4, 128, 2);
    else if (bw256) FG_W8A16_R(4, 256, 1);
    else FG_W8A16_R(4, 128, 1);
  } else if (a.M <= 8) {
    if (wide) FG_W8A16_R(8, 128, 2);
    else if (bw256) FG_W8A16_R(8, 256, 1);
    else FG_W8A16_R(8, 128, 1);
  } else if (a.M <= 16) {
    // 16-row activation strip on 128-byte bands only (the 256-byte form would need 100 KB of LDS).
    // 32-column tiles with three bands of a wave in flight instead of two (us): N = K = 8192 M=16 17.3 /
    // 18.2, K=16384 25.9 / 27.5; N=16384 K=8192 31.3 / 32.7 -- with eight rows level or behind (N = K = 8192
    // 15.3 / 14.7 against 16-column tiles), and 16-column tiles lose with any deeper pipeline (M=16 19.9 with
    // three, 21.4 with four).  With three in flight the one-a-CU form at N = 8192 pays from 12 rows on (K=8192
    // M=13 17.0 / 17.5; M=9 level).
    if (wide)
      hipLaunchKernelGGL((w8a16_r_kernel<16, 8, 128, 2, 3>), dim3(a.N / 32), dim3(512), 0, s, Wq, X, sc,
                         a.scalar_scale, a.zero_point, Y, a.M, a.N, a.K);
    else FG_W8A16_R(16, 128, 1);
  } else {
    return false;
  }
#undef FG_W8A16_R
  return true;
}

// Panel kernel (w4a16_x_kernel): where it measured ahead of the lanes-over-x kernel and, for K <= 16384 and more
// than 2048 columns, everywhere ahead of the row-load kernel (us, the other / this one, M = 2, 3, 4 where three pairs
// stand).  It stages the whole panel whatever N is, so long rows need columns to spread that over; more activation
// rows cost the lanes-over-x kernel as many more reads of x:
//  * K <= 2048 always (N=512 K=512 2.6 / 2.5, 2.9 / 2.5, 3.3 / 2.5); K = 4096 N=1024 3.5 / 3.5, 4.0 / 3.6, 4.6 / 3.7,
//    N=512 3.0 / 3.4, 3.4 / 3.5, 3.7 / 3.6;
//  * K = 6144 N=1024 3.8 / 4.2, 4.5 / 4.4, 5.0 / 4.5, N=1536 4.3 / 4.3, 5.0 / 4.4, 5.4 / 4.5;
//  * K = 8192 N=1024 4.1 / 4.9, 4.7 / 5.0, 5.2 / 5.3, N=1536 4.6 / 5.0, 5.4 / 5.1, 6.3 / 5.4, N=2048 5.1 / 5.1, N=3072
//    5.9 / 5.6;
//  * K = 12288 N=1024 4.9 / 6.5, 5.8 / 6.8, 6.6 / 7.1, N=1536 6.2 / 6.7, 7.4 / 6.9, 10.7 / 7.2, N=3072 7.6 / 7.2;
//  * K = 16384 N=1536 6.6 / 7.9, 7.8 / 8.4, 10.9 / 8.7, N=2048 6.9 / 8.1, 8.2 / 8.5, N=3072 8.9 / 8.7, 10.9 / 9.1.
// Against the row-load kernel N=4096 K=14336 M=4 13.0, N = K = 8192 12.7, N=5120 K=11008 16.9 (this one 9.6, 8.8, 10.4).
static bool w4_panel(const W8A16Args& a) {
  if (a.K > 16384) return false;
  if (a.K <= 2048) return true;
  if (a.K <= 4096) return a.M == 4 || a.N >= 1024;
  if (a.K <= 6144) return a.N >= (a.M == 2 ? 1536 : 1024);
  if (a.K <= 8192) return a.M == 2 ? a.N > 2048 : a.N >= 1536;
  if (a.M == 2) return a.N >= 3072;
  return a.M == 4 ? a.N >= 1536 : (a.K <= 12288 ? a.N >= 2048 : a.N > 2048);
}
static void launch_w4_panel(const W8A16Args& a, hipStream_t s) {
  // KC: the smallest that holds K.  Few waves with several pairs each, the same number for every wave, where that keeps
  // loads enough in flight (us, one way / the other): up to K = 1024 (N=4096 eight 3.1 / four 2.7), K=3072 N=4096 M=2
  // eight of one or two 4.0 / four of three 3.5, K=14336 N=8192 sixteen 15.2 / eight of seven 13.3, K=9216 sixteen 11.2 /
  // eight of five 9.4.  K = 4224..5120: eight waves of three pairs, or four of five where rows are whole lines (K a multiple
  // of 256; the same loads touch fewer of them) and no CU has more than two tiles: 0.88..1.03 of the time of eight (N=4096
  // K=5120 0.89, K=4352 0.91).  Rows that end half way into a line: three and four rows 0.98..1.08, two 0.95..1.01 from K =
  // 4736 on; more tiles 1.01..1.13.  K = 1152..2048: up to three workgroups a CU (240 calls 0.99 of the time with two; M=2
  // N=32768 K=1152 7.5 / 6.7, with one tile a workgroup 6.6); four waves instead, 1.02.
  const int tiles = a.N / 16, cus = compute_units();
#define FG_W4_X(KC, NW, MOST)                                                                                  \
  hipLaunchKernelGGL((w4a16_x_kernel<KC, NW>), dim3(panel_grid(tiles, cus, KC <= 1024 ? 1 : 2, MOST)), dim3(64 * NW), 0, s, \
                     static_cast<const uint8_t*>(a.Wq), static_cast<const half_t*>(a.x),                       \
                     static_cast<const half_t*>(a.scale), a.scalar_scale, a.zero_point, static_cast<half_t*>(a.y), \
                     a.M, a.N, a.K)
  const bool many = tiles > cus;
  if (a.K <= 1024) FG_W4_X(1024, 4, 4);
  else if (a.K <= 2048) FG_W4_X(2048, 8, 3);
  else if (a.K <= 3072) FG_W4_X(3072, 4, 2);
  else if (a.K <= 4096) FG_W4_X(4096, 8, 2);
  else if (a.K <= 5120 && (a.K % 256 == 0 || (a.M == 2 && a.K > 4608)) && tiles <= 2 * cus) FG_W4_X(5120, 4, 2);
  else if (a.K <= 6144) FG_W4_X(6144, 8, 1);
  else if (a.K <= 8192) FG_W4_X(8192, 8, 1);
  else if (a.K <= 10240) FG_W4_X(10240, 8, 1);
  else if (a.K <= 12288 && !many) FG_W4_X(12288, 16, 1);
  else if (a.K <= 12288) FG_W4_X(12288, 8, 1);
  else if (a.K <= 14336) FG_W4_X(14336, 8, 1);
  else FG_W4_X(16384, 16, 1);
#undef FG_W4_X
}

bool launch_w4a16(const W8A16Args& a, hipStream_t s) {
  auto* Wq = static_cast<const uint8_t*>(a.Wq);
  auto* X = static_cast<const half_t*>(a.x);
  auto* sc = static_cast<const half_t*>(a.scale);
  auto* Y = static_cast<half_t*>(a.y);
  if (a.M < 1 || a.M > 4) return false;
  if (a.M == 1) {
    launch_wq_m1<4, 1>(a, s);
  } else if (w4_panel(a)) {
    launch_w4_panel(a, s);
  } else if (a.M == 2) {
    launch_wq_m1<4, 2>(a, s);
  } else if (a.N <= 2048) {
    // narrow outputs leave the 16-column tiles of the row-load kernel on half the CUs or fewer (M=4, us,
    // lanes-over-x / row-load: N=1024 K=8192 5.3 / 7.4; towards 2048 columns they meet)
    if (a.M == 3) launch_wq_m1<4, 3>(a, s);
    else launch_wq_m1<4, 4>(a, s);
  } else {
    hipLaunchKernelGGL((w4a16_r_kernel<4>), dim3(a.N / 16), dim3(512), 0, s, Wq, X, sc, a.scalar_scale,
                       a.zero_point, Y, a.M, a.N, a.K);
  }
  return true;
}

template <int MB>
static void i8i8_go(const void* Wq, const void* xq, int32_t* acc, int M, int N, int K,
                    hipStream_t s) {
  auto* W = static_cast<const int8_t*>(Wq);
  auto* X = static_cast<const int8_t*>(xq);
  // Two to four rows.  One form has four weight rows a workgroup, one 1 KB piece of each in flight a
  // wave, and three or four waves, whichever leaves fewer of the last step's waves without a piece; the
  // other, below, eight rows (four for narrow outputs), two pieces a wave, four waves.  One after the other in
  // a replayed graph, us, the second form / the first:
  //  * two and three rows: the first throughout (M=2 N = K = 8192 12.6 / 12.1, N=28672 K=8192 36.5 / 34.7, K=12288 52.0 /
  //    51.7, M=3 53.4 / 54.9);
  //  * four rows: the first (N=16384 K=11008 33.6 / 32.6) but for twelve pieces against wide outputs, where the
  //    second's waves all have as many (N = K = 12288 26.0 / 28.2, N=28672 K=11520 52.0 / 55.9; N=11008 K=12288
  //    25.0 / 25.2);
  //  * narrow outputs keep the second, their workgroups do not fill the chip (N=2048 K=14336 M=4 7.9 / 8.5), and so
  //    do the longest rows (N=4096 K=14336 M=4 12.8 / 13.0).
  if (MB == 2 || MB == 4) {
    const int pieces = (K / 16 + 63) / 64;
    const bool full_steps = M == 4 && pieces == 12 && N >= 1024 * pieces;
    if (N > 2048 && pieces <= 12 && !full_steps) {
      const int waves = pieces <= 4 ? pieces : ((pieces + 2) / 3 * 3 < (pieces + 3) / 4 * 4 ? 3 : 4);
      hipLaunchKernelGGL((i8i8_kernel<MB, 4, 1>), dim3(N / 4), dim3(64 * waves), 0, s, W, X, acc, M, N, K);
      return;
    }
  }
  const dim3 block(64 * i8_waves(K));
  if (MB == 1) {
    hipLaunchKernelGGL((i8i8_kernel<1, 4, 1>), dim3(N / 4), block, 0, s, W, X, acc, M, N, K);
    return;
  }
  if (N / 8 >= 512 && MB <= 4) {
    hipLaunchKernelGGL((i8i8_kernel<MB, 8, 2>), dim3(N / 8), block, 0, s, W, X, acc, M, N, K);
  } else {
    hipLaunchKernelGGL((i8i8_kernel<MB, 4, 2>), dim3(N / 4), block, 0, s, W, X, acc, M, N, K);
  }
}

// Panel kernel (i8i8_x_kernel): where it measured ahead, us, the v_dot4 kernel (or an earlier panel kernel, with loads
// in operand order and one tile a workgroup) / this one.  It stages the whole panel whatever N is, so long rows need
// columns to spread that over:
//  * five rows and more: N=1024 K=4096 M=8 4.6 / 3.8, K=6144 5.1 / 4.8, K=8192 5.5 / 6.0; N=1536 K=8192 7.4 / 6.2, K=12288
//    9.6 / 8.6; N=2048 K=14336 M=5 9.4 / 10.4, N=3072 M=8 14.4 / 11.7; N = K = 5120 11.4 / 7.3, N = K = 8192 15.9 / 12.4,
//    N=14336 K=4096 16.6 / 11.3;
//  * four: N=1024 K=4096 3.7 / 3.4, K=5120 4.0 / 4.4; N=1536 K=8192 5.7 / 5.6; N=2048 K=9216 6.9 / 7.3, N=3072 7.7 / 7.9; N =
//    K = 5120 7.5 / 7.2, N=4096 K=8192 8.6 / 7.5, N=14336 K=4096 12.4 / 11.2, N = K = 8192 13.5 / 12.3;
//  * three, less: N=2176 K=7296 6.2 / 5.6, N=2048 K=7680 5.7 / 5.9, N=9216 K=5120 10.0 / 10.3; K > 7168 not where the second
//    or third round is a quarter full or less (N=5120 K=8192 9.4 / 9.6, N=8320 K=7808 13.2 / 14.0, against N=5632 0.94 and
//    N=9728 0.98 of the v_dot4 kernel's time);
//  * three and four to K = 10240 where the rounds come out full: N=4096 three 9.8 / 9.0, four 10.2 / 9.1, N=8192 16.8 / 14.4;
//    N=5120 11.3 / 12.0;
//  * two, for which the v_dot4 kernel reads few activations: K <= 2048 (N=28672 10.9 / 10.3, N=2048 3.3 / 2.9), to K = 4096
//    with one tile a CU at most (N=4096 5.2 / 4.7), to 6144 where one or two tiles a CU come out even (N=8192 9.6 / 9.0,
//    N=7168 8.8 / 8.2; N=5120 7.3 / 7.7, N=9216 10.5 / 11.3).
static bool i8_panel(int M, int N, int K) {
  if (M < 2 || K > 16384) return false;
  if (M >= 5) return K <= 4096 || N >= (K <= 6144 ? 1024 : (K <= 12288 ? 1536 : 2176));
  if (K <= 2048) return true;
  const int tiles = N / 16, cus = compute_units(), rounds = (tiles + cus - 1) / cus;
  if (M >= 3) {
    if (K <= 4096) return N >= (M == 4 ? 512 : 1024);
    if (K <= 8192 && M == 4) return N >= 1536;
    if (K <= 8192) return K <= 7168 ? N >= 2048 : (rounds == 1 ? N > 2048 : rounds > 3 || 4 * tiles > (4 * rounds - 3) * cus);
    return K <= 10240 && 4 * tiles > 3 * rounds * cus;
  }
  return (K <= 4096 && rounds == 1 && N >= 2048) || (K <= 6144 && rounds <= 2 && 8 * tiles >= 7 * rounds * cus);
}

bool launch_i8i8_i32(const void* Wq, const void* xq, int32_t* acc, int M, int N, int K,
                     hipStream_t s) {
  if (M < 1 || M > 8) return false;
  if (i8_panel(M, N, K)) {
    auto* W = static_cast<const int8_t*>(Wq);
    auto* X = static_cast<const int8_t*>(xq);
    // Workgroups a CU, and waves with the same number of pairs each, as in launch_w4_panel (eight rows, us, KC the next
    // power of two or 6144, 12288 / as here: N=4096 K=2560 4.3 / 3.7, N=2048 K=3072 3.9 / 3.3, N = K = 5120 7.3 / 6.8,
    // N=4096 K=7168 7.7 / 7.1, K=14336 13.3 / 12.7).
    const int tiles = N / 16, cus = compute_units();
#define FG_I8_X(XR, KC, NW, MOST)                                                                    \
  hipLaunchKernelGGL((i8i8_x_kernel<XR, KC, NW>), dim3(panel_grid(tiles, cus, KC <= 1024 ? 1 : 2, MOST)), \
                     dim3(64 * NW), 0, s, W, X, acc, M, N, K)
    if (M <= 4) {
      if (K <= 512) FG_I8_X(4, 512, 4, 4);
      else if (K <= 1024) FG_I8_X(4, 1024, 4, 4);
      else if (K <= 1536) FG_I8_X(4, 1536, 4, 4);
      else if (K <= 2048) FG_I8_X(4, 2048, 8, 3);
      else if (K <= 2560) FG_I8_X(4, 2560, 4, 3);
      else if (K <= 3072) FG_I8_X(4, 3072, 8, 2);
      else if (K <= 4096) FG_I8_X(4, 4096, 8, 2);
      else if (K <= 5120) FG_I8_X(4, 5120, 8, 2);
      else if (K <= 6144) FG_I8_X(4, 6144, 8, 2);
      else if (K <= 7168) FG_I8_X(4, 7168, 8, 2);
      else if (K <= 8192) FG_I8_X(4, 8192, 8, 2);
      else FG_I8_X(4, 10240, 8, 1);             // (longer rows: see i8_panel)
    } else if (K <= 512) FG_I8_X(8, 512, 4, 4);
    else if (K <= 1024) FG_I8_X(8, 1024, 8, 3);
    else if (K <= 1536) FG_I8_X(8, 1536, 4, 4);
    else if (K <= 2048) FG_I8_X(8, 2048, 8, 2);
    else if (K <= 2560) FG_I8_X(8, 2560, 4, 3);
    else if (K <= 3072) FG_I8_X(8, 3072, 8, 2);
    else if (K <= 4096) FG_I8_X(8, 4096, 8, 2);
    else if (K <= 5120) FG_I8_X(8, 5120, 8, 1);
    else if (K <= 6144) FG_I8_X(8, 6144, 8, 1);
    else if (K <= 7168) FG_I8_X(8, 7168, 8, 1);
    else if (K <= 8192) FG_I8_X(8, 8192, 8, 1);
    else if (K <= 10240) FG_I8_X(8, 10240, 16, 1);
    else if (K <= 12288) FG_I8_X(8, 12288, 16, 1);
    else if (K <= 14336) FG_I8_X(8, 14336, 16, 1);
    else FG_I8_X(8, 16384, 16, 1);
#undef FG_I8_X
  } else if (M == 1) {
    i8i8_go<1>(Wq, xq, acc, M, N, K, s);
  } else if (M == 2) {
    i8i8_go<2>(Wq, xq, acc, M, N, K, s);
  } else if (M <= 4) {
    i8i8_go<4>(Wq, xq, acc, M, N, K, s);
  } else {
    i8i8_go<8>(Wq, xq, acc, M, N, K, s);
  }
  return true;
}

void launch_dequant_i32_f16(const int32_t* acc, const void* scale, float x_scale, void* y, int M,
                            int N, hipStream_t s) {
  const size_t total = (size_t)M * N;
  const int blocks = (int)((total + 255) / 256 < 1024 ? (total + 255) / 256 : 1024);
  hipLaunchKernelGGL(dequant_i32_f16_kernel, dim3(blocks), dim3(256), 0, s, acc,
                     static_cast<const half_t*>(scale), x_scale, static_cast<half_t*>(y), M, N);
}

}  // namespace fg
