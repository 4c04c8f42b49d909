// fp16 kernel for more than 16 activation rows, both weight layouts.
//
// The kernels for 1..16 rows give every workgroup one block of rows; run on M rows they read the
// weights ceil(M / 16) (or 32) times and put both operands of every MFMA through wave-private LDS.
// Here a workgroup owns BM rows x BN columns of C with BM covering all rows where it can (up to
// 128), so the weights leave memory once, and its waves share both operands through LDS.
//
//  * Per step the workgroup stages BK k of its BN weight columns and of its BM activation rows:
//    16-byte loads into registers, P steps ahead (weights non-temporal unless row blocks exchange
//    steps, activations from L2), from there into one of two LDS buffers -- one barrier a step.  Rows
//    beyond M load as zeros and are never stored.
//  * k-contiguous rows lie in LDS as 16-byte pieces permuted by their row, so the operand-order reads
//    (ds_read_b128, row j, piece g) hit distinct banks without padding.  [K,N] rows lie as they come, 16 columns = 32 bytes a
//    group, groups permuted by k so that the four k rows a transposing read (ds_read_b64_tr_b16)
//    gathers sit on distinct banks; that read hands each lane four consecutive k of its column, so
//    no register transposition is needed.
//  * mfma_f32_16x16x32_f16 with the weights as first operand: a lane then holds four consecutive
//    columns of one row of C (8-byte stores, 16-byte partials).
//  * One-dimensional grid.  Workgroups go to the XCDs round-robin by id; the row blocks of one
//    (column tile, K range) get ids that differ by the XCD count, so they read the same weights
//    through the same L2 at about the same time (in exchanged steps, see PAIRED).
// What bounds it (128 x 128 tile, 2 x 4 waves of 64 x 32, 64 k a step, M = 256 N = 13824 K = 5120, counters
// over the steps of one workgroup a CU, row blocks in step): a step takes 1390 cycles.  The matrix cores are busy for 512
// of them, the LDS for 650 (every wave reads 64 + 32 rows, 96 KB in all, and 32 KB are written; no bank
// conflicts), the loads take about 650 (32 KB at the 50 bytes a clock a CU takes from L2).  None of the
// three is full: two waves a SIMD meet at a barrier every step, a wave spends a quarter of its time
// ([N,K]: a sixth) waiting to issue to the LDS, and reads and products overlap only in part.
// 64 x 64 wave tiles would read 64 KB.  K-splitting the waves (WK) halves the operand reads of the
// narrow tiles, where every wave would otherwise read all rows.
// Measured (us, the kernels for few rows repeated / this one): [K,N] M=256 N=13824 K=5120 333 / 54 (670
// TFLOP/s; a large product through the vendor library reaches 1145 on the card), M=128 N = K = 8192
// 104 / 41; [N,K] M=48 N=4096 K=11008 40 / 21 (4.4 TB/s), M=96 N = K = 8192 91 / 34.
// A split over K completes as for the other kernels: two passes, the counter protocol, or one
// fixed-point atomic per element; partials are added in ascending order of the K range.
#include "fg_device.h"
#include "fg_internal.h"

namespace fg {

namespace {

typedef half_t half4_v __attribute__((ext_vector_type(4)));
typedef short short4_v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4_v lds_short4;
typedef __attribute__((address_space(3))) unsigned char lds_byte;

// Group (32 bytes) permutation of k row `k` in the [K,N] LDS layout, GROUPS groups a row.  A wave's
// transposing read takes rows 8g + 0..3 (or 4..7) of one group for g = 0..3; 32 lanes at a time hit
// rows 0..3 and 8..11, which must land on eight different 32-byte slots of the 256 bytes the banks span.
template <int GROUPS>
__device__ __forceinline__ int kn_swizzle(int k) {
  if constexpr (GROUPS % 8 == 0) return (k & 3) | (((k >> 3) & 1) << 2);
  else if constexpr (GROUPS % 4 == 0) return ((k >> 1) & 1) | (((k >> 3) & 1) << 1);
  else if constexpr (GROUPS % 2 == 0) return (k >> 3) & 1;
  else return 0;
}

struct TileArgs {
  const half_t* A;
  const half_t* W;
  half_t* C;
  float* ws;
  int* counters;
  const void* bias;
  int M, N, K, flags, ldw;
  int ntiles, mblocks, splitk, xccs;
};

// PAIRED: several row blocks, which read the same weights side by side on one XCD.  In step they wait for the same
// lines: each asks HBM for half of what its own CU could take.  So the odd ones walk K with the pairs of steps in each
// four exchanged (2 3 0 1): either block brings half of the weights from HBM and finds the other half, two steps old,
// in the L2.  For that the weights may not be non-temporal, and all tiles start at the same step: they read the same
// activations at the same time.
// A row's result must not depend on the block it lies in, so either order gives the same bits: steps 0 and 1 of each four
// go into one sum, 2 and 3 into another, and the two meet once, after the last whole four (a + b is b + a); the steps
// behind it go in order.  One sum in the order of the walk / two, us: [K,N] M=256 N=13824 K=5120 53.9 / 54.1, [N,K]
// 54.9 / 53.1; level over 355 sizes of 33..512 rows (the worst M=419 N=2176 K=7040 39.8 / 41.8).
// us, all in step / this, call after call: M=256 N=13824 K=5120 [K,N] 57.8 / 54.1, [N,K] 60.2 / 53.1; N = K = 8192 [K,N]
// 64.5 / 57.9; M=200 N=4864 K=8320 [N,K] 49.2 / 38.4.  Loads alone 53 / 45.6; exchanging single steps or fours, a start
// by XCD or by tile, or weights kept non-temporal (60.2) gave less.
// FAR: [K,N] rows so far apart that the offsets over the rows of a step leave 32 bits (16 Mi elements and
// more); the same steps and sums with 64-bit addresses for the weights.
template <bool KN, bool FAR, bool PAIRED, int BM, int BN, int BK, int WM, int WN, int WK, int P>
__global__ __launch_bounds__(64 * WM * WN * WK, PAIRED && !FAR && BM == 64 && BN / WN == 32 ? 4 : 2)  // (4: two a CU)
void tile_kernel(TileArgs t) {
  constexpr int NT = 64 * WM * WN * WK;
  constexpr int TM = BM / WM, TN = BN / WN;  // wave tile
  constexpr int MB = TM / 16, NB = TN / 16;
  constexpr int UNITS = BK / 32 / WK;        // 32-k units of a step per wave
  static_assert(TM % 16 == 0 && TN % 16 == 0 && BK % (32 * WK) == 0 && (WK & (WK - 1)) == 0, "whole MFMA blocks");
  constexpr int RS = BK * 2;                 // LDS bytes per k-contiguous row
  constexpr int ABYTES = BM * RS;
  constexpr int WBYTES = KN ? BK * BN * 2 : BN * RS;
  constexpr int STAGE = ABYTES + WBYTES;
  constexpr int CPR = BK / 8;                // 16-byte pieces of a k-contiguous row
  constexpr int SW = CPR < 16 ? CPR - 1 : 15;  // pieces of row r are permuted by r & SW
  constexpr int WPR = KN ? BN / 8 : CPR;     // ... of a weight row
  constexpr int ACH = BM * CPR, WCH = BN * CPR;
  constexpr int AI = ACH / NT, WI = WCH / NT;
  static_assert(ACH % NT == 0 && WCH % NT == 0, "every thread stages as many pieces");
  constexpr int GROUPS = BN / 16;
  constexpr int RP = BN + 4;                 // floats per row of the tile when its sums are in LDS
  constexpr int SLOT = BM * RP;              // ... per K group of waves
  constexpr int SLOTS = WK > 1 ? WK / 2 : 1;
  constexpr int LDS = 2 * STAGE > SLOTS * SLOT * 4 ? 2 * STAGE : SLOTS * SLOT * 4;
  __shared__ __attribute__((aligned(16))) unsigned char smem[LDS];
  __shared__ int s_arrival;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, g = lane >> 4;
  const int wm = wave % WM, wn = wave / WM % WN, wk = wave / (WM * WN);
  // id -> (row block, column tile, K range)
  const int xcd = (int)blockIdx.x % t.xccs, local = (int)blockIdx.x / t.xccs;
  const int mblk = local % t.mblocks;
  const int unit = (local / t.mblocks) * t.xccs + xcd;
  const int S = t.splitk;
  if (unit >= t.ntiles * S) return;
  const int z = unit % S, tile = unit / S;
  const int m0 = mblk * BM, n0 = tile * BN;
  const int K = t.K, N = t.N, M = t.M;

  const int steps = K / BK;  // the launcher only takes forms whose BK divides K
  const int s0 = (int)((long long)steps * z / S), count = (int)((long long)steps * (z + 1) / S) - s0;

  // Where this thread's pieces come from (bytes from the tile's first row and the step's first k)
  // and go to.  All loads are buffer loads (FAR's weights apart): activation rows beyond M lie behind the descriptor's
  // end and read as zeros, and a step behind the last one has an empty descriptor.  No load sits
  // behind a branch, so the number in flight is the same on every path and the waits are exact; with
  // the loads in branches the compiler waits for all of them before every park (M = 256, N = 13824,
  // K = 5120: 64 us).
  unsigned a_off[AI], w_off[WI];
  int a_lds[AI], w_lds[WI];
#pragma unroll
  for (int i = 0; i < AI; ++i) {
    const int c = i * NT + tid, row = c / CPR, piece = c % CPR;
    a_off[i] = (unsigned)row * (unsigned)K * 2u + piece * 16;
    a_lds[i] = row * RS + 16 * (piece ^ (row & SW));
  }
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const int c = i * NT + tid, row = c / WPR, piece = c % WPR;
    w_off[i] = (unsigned)row * (unsigned)(KN ? t.ldw : K) * 2u + piece * 16;
    w_lds[i] = ABYTES + (KN ? row * (BN * 2) + 32 * ((piece >> 1) ^ kn_swizzle<GROUPS>(row)) + 16 * (piece & 1)
                            : row * RS + 16 * (piece ^ (row & SW)));
  }
  const int rows = M - m0 < BM ? M - m0 : BM;
  const half_t* const At = t.A + (size_t)m0 * K;
  const half_t* const Wt = t.W + (KN ? (size_t)n0 : (size_t)n0 * K);
  const unsigned a_bytes = (unsigned)rows * (unsigned)K * 2u;
  const unsigned w_bytes = KN ? ((unsigned)(BK - 1) * (unsigned)t.ldw + BN) * 2u : (unsigned)BN * (unsigned)K * 2u;

  u32x4 ra[P][AI], rw[P][WI];
  // step numbers wrap around from a start that differs from tile to tile: rows are a power of two
  // apart for the usual K, and workgroups in lockstep would sit on the same memory channels (PAIRED: see above)
  const int start = PAIRED || count == 0 ? 0 : tile % count;
  const int swapped = PAIRED && (mblk & 1) ? count & ~3 : 0;
  int issued = 0;
  auto load = [&](u32x4(&a)[AI], u32x4(&w)[WI]) {
    constexpr int kNonTemporal = PAIRED ? 0 : 2;  // the nt bit of a buffer load's cache policy
    const bool live = issued < count;
    int step = start + (issued < swapped ? issued ^ 2 : issued);
    if (!PAIRED && step >= count) step -= count;
    ++issued;
    const int k0 = (s0 + (FAR && !live ? 0 : step)) * BK;
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<half_t*>(Wt + (KN ? (size_t)k0 * t.ldw : (size_t)k0)), 0,
        (int)(live ? w_bytes - (KN ? 0u : (unsigned)k0 * 2u) : 0u), 0x00020000);
    const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<half_t*>(At + k0), 0, (int)(live ? a_bytes - (unsigned)k0 * 2u : 0u), 0x00020000);
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      if constexpr (FAR) {  // (a step behind the last one reads the first again; it is never multiplied)
        const int c = i * NT + tid;
        w[i] = load16<!PAIRED>(Wt + (size_t)(k0 + c / WPR) * t.ldw + c % WPR * 8);
      } else {
        w[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, (int)w_off[i], 0, kNonTemporal));
      }
    }
#pragma unroll
    for (int i = 0; i < AI; ++i)
      a[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ar, (int)a_off[i], 0, 0));
  };
  auto park = [&](int buf, const u32x4(&a)[AI], const u32x4(&w)[WI]) {
    unsigned char* b = smem + buf * STAGE;
#pragma unroll
    for (int i = 0; i < WI; ++i)
      *reinterpret_cast<u32x4*>(b + w_lds[i]) = w[i];
#pragma unroll
    for (int i = 0; i < AI; ++i)
      *reinterpret_cast<u32x4*>(b + a_lds[i]) = a[i];
  };

  constexpr int HALVES = PAIRED ? 2 : 1;     // (see PAIRED)
  float4_t sums[HALVES][NB][MB];
#pragma unroll
  for (int h = 0; h < HALVES; ++h)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int m = 0; m < MB; ++m) sums[h][b][m] = float4_t{0.f, 0.f, 0.f, 0.f};
  float4_t(&acc)[NB][MB] = sums[0];

  const int a_rd = (wm * TM + j) * RS;
  const int w_rd = ABYTES + (wn * TN + j) * RS;  // [N,K]
  // [K,N]: lane (j, g) addresses row 8g + j/4 of a 32-k unit, four columns 4 (j % 4) of a 16-column group;
  // rows 4 further have the same permutation, and so have rows 32 further
  const int t_row = 8 * g + (j >> 2);
  const int t_sw = kn_swizzle<GROUPS>(t_row);
  // Operands of one 32-k unit, two register sets: while one is multiplied the next is on its way from
  // LDS, across the steps' barriers too (otherwise all waves read, then all multiply).
  u32x4 av[2][MB], wv[2][NB];
  auto fetch = [&](int set, int buf, int uu) {
    const unsigned char* b = smem + buf * STAGE;
    const int u = uu * WK + wk;
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if constexpr (KN) {
        lds_byte* p = (lds_byte*)(smem + buf * STAGE + ABYTES + (u * 32 + t_row) * (BN * 2) +
                                  32 * ((wn * NB + i) ^ t_sw) + 8 * (j & 3));
        const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)p));
        const u32x2 hi =
            __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(p + 4 * (BN * 2))));
        wv[set][i] = u32x4{lo.x, lo.y, hi.x, hi.y};
      } else {
        wv[set][i] = *reinterpret_cast<const u32x4*>(b + w_rd + i * 16 * RS + 16 * ((4 * u + g) ^ (j & SW)));
      }
    }
#pragma unroll
    for (int m = 0; m < MB; ++m) av[set][m] = *reinterpret_cast<const u32x4*>(b + a_rd + m * 16 * RS + 16 * ((4 * u + g) ^ (j & SW)));
  };
  auto multiply = [&](int set, int half = 0) {
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int m = 0; m < MB; ++m)
        sums[half][i][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_half8(wv[set][i]), as_half8(av[set][m]),
                                                                  sums[half][i][m], 0, 0, 0);
  };
  auto clear_operands = [&](int set) {
#pragma unroll
    for (int i = 0; i < NB; ++i) wv[set][i] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int m = 0; m < MB; ++m) av[set][m] = u32x4{0u, 0u, 0u, 0u};
  };
  clear_operands(1);

#pragma unroll
  for (int p = 0; p < P; ++p) {
    load(ra[p], rw[p]);
    __builtin_amdgcn_sched_barrier(0);  // oldest first: the loop's waits count on this order
  }
  park(0, ra[0], rw[0]);
  load(ra[0], rw[0]);
  __builtin_amdgcn_sched_barrier(0);
  // register sets, LDS buffers and (PAIRED) the sum a step adds to have constant numbers inside a round
  constexpr int U = PAIRED ? 4 : (P % 2 ? 2 * P : P);
  static_assert(U % P == 0 && U % 2 == 0, "whole turns of the register sets and of the LDS buffers");
  // Order within a step: a unit's operand reads go out first, then the products of the unit read before
  // it, with the LDS writes and the global loads dealt out between them -- issued in one piece they
  // hold every wave at the load unit while the matrix cores idle.
  constexpr int PIECE_OPS = AI + WI, MFMAS = MB * NB, GAP = UNITS * MFMAS / (2 * PIECE_OPS);
  auto one_step = [&](int u, bool fours) {
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int uu = 0; uu < UNITS; ++uu) {
      fetch((u * UNITS + uu) & 1, u & 1, uu);
      multiply((u * UNITS + uu + 1) & 1, fours ? ((uu == 0 ? u + 3 : u) >> 1) & 1 : 0);
    }
    park((u + 1) & 1, ra[(u + 1) % P], rw[(u + 1) % P]);
    load(ra[(u + 1) % P], rw[(u + 1) % P]);
    constexpr int kMfma = 0x8, kVmemRead = 0x20, kDsRead = 0x100, kDsWrite = 0x200;
    constexpr int READS = MB + (KN ? 2 : 1) * NB;
#pragma unroll
    for (int uu = 0; uu < UNITS; ++uu) {
      __builtin_amdgcn_sched_group_barrier(kDsRead, READS, 0);
#pragma unroll
      for (int i = PIECE_OPS * uu / UNITS; i < PIECE_OPS * (uu + 1) / UNITS; ++i) {
        if constexpr (GAP > 0) __builtin_amdgcn_sched_group_barrier(kMfma, GAP, 0);
        __builtin_amdgcn_sched_group_barrier(kDsWrite, 1, 0);
        if constexpr (GAP > 0) __builtin_amdgcn_sched_group_barrier(kMfma, GAP, 0);
        __builtin_amdgcn_sched_group_barrier(kVmemRead, 1, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  int it = 0;
  for (; it + U <= count; it += U) {  // whole rounds only: a way out inside would blur the counts again
#pragma unroll
    for (int u = 0; u < U; ++u) one_step(u, PAIRED);
  }
  if constexpr (PAIRED) {
    multiply(1, 1);  // (the last unit of the fours)
    clear_operands(1);
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int m = 0; m < MB; ++m) acc[i][m] += sums[1][i][m];
  }
#pragma unroll
  for (int u = 0; u < U - 1; ++u) {
    if (it + u >= count) break;
    one_step(u, false);
  }
  if (!PAIRED || (count & 3)) {  // (the last unit; PAIRED, whole fours: they are through)
    if ((count * UNITS) & 1) multiply(0);
    else multiply(1);
  }

  // acc[i][m][r]: column wn TN + 16 i + 4 g + r of row wm TM + 16 m + j of the tile.  The K groups of
  // waves meet in LDS, the upper half of them handing over to the lower half until one is left; the
  // sums then lie in LDS row by row and every thread finishes whole pieces of four columns.
  float* red = reinterpret_cast<float*>(smem);
  const int r_off = (wm * TM + j) * RP + wn * TN + 4 * g;
  auto put = [&](float* slot) {
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int m = 0; m < MB; ++m) *reinterpret_cast<float4_t*>(slot + r_off + 16 * m * RP + 16 * i) = acc[i][m];
  };
#pragma unroll
  for (int h = WK / 2; h > 0; h >>= 1) {
    __syncthreads();
    if (wk >= h && wk < 2 * h) put(red + (wk - h) * SLOT);
    __syncthreads();
    if (wk < h) {
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int m = 0; m < MB; ++m)
          acc[i][m] += *reinterpret_cast<const float4_t*>(red + wk * SLOT + r_off + 16 * m * RP + 16 * i);
    }
  }
  __syncthreads();
  if (wk == 0) put(red);
  __syncthreads();

  constexpr int PIECES = BM * BN / 4;        // of four columns
  constexpr int NQ = (PIECES + NT - 1) / NT;
  const size_t MN = (size_t)M * N;
  auto write_out = [&](int row, int n, float4_t v) {
    half4_v* c = reinterpret_cast<half4_v*>(t.C + (size_t)row * N + n);
    if (t.flags & (kFlagAccumulate | kFlagTailMask)) {
      if (t.flags & kFlagAccumulate) {
        const half4_v old = *c;
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] += static_cast<float>(old[k]);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = apply_tail(v[k], n + k, t.bias, t.flags);
    }
    half4_v out;
#pragma unroll
    for (int k = 0; k < 4; ++k) out[k] = static_cast<half_t>(v[k]);
    *c = out;
  };
  uint64_t* facc = reinterpret_cast<uint64_t*>(reinterpret_cast<unsigned char*>(t.counters) + kWsCounterBytes);
  uint32_t* fcls = reinterpret_cast<uint32_t*>(facc + kWsAccElems);
  for (int q = 0; q < NQ; ++q) {
    const int e = q * NT + tid, row = m0 + e / (BN / 4), n = n0 + e % (BN / 4) * 4;
    const bool ok = e < PIECES && row < M;
    const float4_t v = ok ? *reinterpret_cast<const float4_t*>(red + (row - m0) * RP + (n - n0)) : float4_t{0.f, 0.f, 0.f, 0.f};
    if (S == 1) {
      if (ok) write_out(row, n, v);
    } else if (t.flags & kFlagFixSplit) {
      const size_t at = ok ? (size_t)row * N + n : 0;
      const size_t idx[4] = {at, at + 1, at + 2, at + 3};
      const float p[4] = {v[0], v[1], v[2], v[3]};
      const bool valid[4] = {ok, ok, ok, ok};
      fix_arrive<4>(facc, fcls, t.ws, z, MN, idx, p, valid, S, t.C, N, t.bias, t.flags);
    } else if (ok) {
      store_partial4(t.ws, (size_t)z * MN + (size_t)row * N + n, v, t.counters != nullptr);
    }
  }
  // without counters a second kernel sums the partials
  if (S == 1 || (t.flags & kFlagFixSplit) || t.counters == nullptr) return;
  if (splitk_arrive(t.counters + mblk * t.ntiles + tile, S, &s_arrival) == 0) return;
  for (int q = 0; q < NQ; ++q) {
    const int e = q * NT + tid, row = m0 + e / (BN / 4), n = n0 + e % (BN / 4) * 4;
    if (e >= PIECES || row >= M) continue;
    const int off[1] = {(row * N + n) * 4};  // the in-launch completion keeps all partials below 2 GiB
    float4_t tot[1];
    sum_partials_z<1, true>(t.ws, S, M * N * 4, off, tot);
    write_out(row, n, tot[0]);
  }
}

template <bool KN, bool FAR, int BM, int BN, int BK, int WM, int WN, int WK, int P>
void tile_go(const TileArgs& t, hipStream_t s) {
  const int units = t.ntiles * t.splitk;
  const dim3 grid((unsigned)((units + t.xccs - 1) / t.xccs * t.xccs) * (unsigned)t.mblocks), block(64 * WM * WN * WK);
  // Several row blocks exchange their steps (see PAIRED) but where that measured behind; 1900 calls of 33..4096 rows, their
  // time exchanged / in step on average 0.93, us of the worst in step / exchanged:
  //  * [K,N], 128 x 128 tiles of two to four blocks with K <= 2048, too few steps to pay: 1.02 (M=160 N=14336 K=1024 13.8 /
  //    14.9); five blocks and more gain there too (M=2048 N=4096 K=2048 46.4 / 43.8).  [N,K], two blocks, K < 2048: level,
  //    1.05..1.1 at worst (M=256 N=28672 K=512 19.7 / 21.7).
  //  * [N,K] rows a power of two apart, from 4 KB on: all tiles start in step, on the same channels.  With two blocks of the
  //    smaller tiles (three of 64 x 128) that costs as much as the exchange gives or more: up to 64 columns and rows 1.11
  //    unsplit (M=64 N=8192 K=2048 10.2 / 12.2) and 1.02 split from K=8192 on (K=16384 N=1024 in eight 12.9 / 14.1; K=4096
  //    0.97); 96 and 128 rows over all of K 0.81 at K=4096 but 1.02..1.09 at K = 2048 and 8192 (M=160 N=8192 14.0 / 15.3,
  //    44.2 / 46.7), split 0.98; 64 x 128 1.03 (M=149 N=10240 K=8192 50.2 / 53.9).  With more blocks the exchange wins there
  //    as well (K=2048 0.94, 4096 0.94, 8192 0.83; split 0.99, 0.95, 0.90; worst M=350 N=10240 K=2048 22.4 / 22.8), and with
  //    128 x 128 tiles of two (0.94).
  // The worst that is exchanged all the same: [K,N] M=400 N=4096 K=3072 19.7 / 21.0, [N,K] M=160 N=4096 K=16384 in two splits
  // 44.6 / 49.4.
  const bool largest = BM * BN >= 128 * 128, smallest = BM * BN <= 64 * 64;
  const bool power_apart = !KN && t.K % 2048 == 0 && (t.K & (t.K - 1)) == 0;
  const bool in_step = largest ? (KN ? t.K <= 2048 && t.mblocks <= 4 : t.K < 2048 && t.mblocks == 2)
                               : power_apart && t.mblocks <= (BM == 64 && BN == 128 ? 3 : 2) &&
                                     (t.splitk == 1 || (smallest && t.K >= 8192));
  if (t.mblocks == 1 || in_step) {
    hipLaunchKernelGGL((tile_kernel<KN, FAR, false, BM, BN, BK, WM, WN, WK, P>), grid, block, 0, s, t);
    return;
  }
  // 64 x 128 with two sums: 32 x 64 a wave take 168 registers, one workgroup a CU; 32 x 32 a wave on all of K leave room
  // for two, but read a third more from LDS.  [K,N] one a CU at most: 1.02..1.04 of one sum's time against 0.98..1.01, more:
  // 1.02 against 1.11..1.17; [N,K] 0.97..1.0 against 0.96..1.17.  (Eight XCDs of 32 CUs whatever the library counts: a plan
  // adds in the same order everywhere.)
  if constexpr (BM == 64 && BN == 128) {
    if (!KN || (units + 7) / 8 * t.mblocks > 32) {
      hipLaunchKernelGGL((tile_kernel<KN, FAR, true, BM, BN, BK, 2, 4, 1, P>), grid, block, 0, s, t);
      return;
    }
  }
  if constexpr (KN || BM != 64 || BN != 128)
    hipLaunchKernelGGL((tile_kernel<KN, FAR, true, BM, BN, BK, WM, WN, WK, P>), grid, block, 0, s, t);
}

}  // namespace

bool launch_tile(int form, bool kn, const fg_plan_t& p, const GemmArgs& a, hipStream_t s) {
  TileForm f;
  if (!tile_form_info(form, &f) || a.N % f.cols || a.K % f.bk) return false;
  TileArgs t{static_cast<const half_t*>(a.A), static_cast<const half_t*>(a.W), static_cast<half_t*>(a.C),
             a.ws, a.counters, a.bias, a.M, a.N, a.K, a.accumulate, a.ldw,
             a.N / f.cols, (a.M + f.rows - 1) / f.rows, p.splitk, a.xccs > 0 ? a.xccs : 1};
  if (((long long)t.ntiles * t.splitk + t.xccs) * t.mblocks > 0x7fffffffll) return false;
  const bool far = kn && 2ull * f.bk * a.ldw >= (1ull << 32);
#define FG_TILE(ID, BM, BN, BK, WM, WN, WK, P)                       \
  case ID:                                                           \
    if (far) tile_go<true, true, BM, BN, BK, WM, WN, WK, P>(t, s);   \
    else if (kn) tile_go<true, false, BM, BN, BK, WM, WN, WK, P>(t, s); \
    else tile_go<false, false, BM, BN, BK, WM, WN, WK, P>(t, s);     \
    return true
  switch (form) {
    FG_TILE(0, 32, 64, 128, 1, 2, 4, 2);
    FG_TILE(1, 32, 128, 128, 1, 4, 2, 2);
    FG_TILE(2, 64, 64, 128, 2, 2, 2, 2);
    FG_TILE(3, 96, 64, 128, 2, 2, 2, 2);
    FG_TILE(4, 128, 64, 128, 2, 2, 2, 2);
    FG_TILE(5, 128, 128, 64, 2, 4, 1, 2);
    FG_TILE(6, 64, 128, 64, 2, 2, 2, 2);
    default: return false;
  }
#undef FG_TILE
}

}  // namespace fg
