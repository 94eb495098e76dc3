// o_proj after the attention over Q4_L weights: y[v] += W x[v] for a batch of
// vectors (the reference's q4l_gemv_accumulate_multirow, lns_decode.metal:
// 1174-1225, once per vector).  W is rows x cols in device blocks of 144 bytes
// (8 f16 effective scales, then 256 weight nibbles: bit 3 sign, bits 0-2
// magnitude m; the weight is sign * scale * 2^(m - 5), m = 0 exact zero).
//
// On the matrix cores.  Within one 32-weight sub-block a row's scale is
// constant, so the sub-block's products take the weights as the exact f16
// powers of two +-2^(m - 5) and the row's scale is applied afterwards in f32:
// no f16 rounding of small weights.  x enters as two f16 parts, hi = f16(x)
// and lo = f16(x - hi), both rounded toward zero (x = hi + lo to 2^-20):
//   D[vec][row] = sum_k A[vec][k] * B[k][row],  A = x parts, B = weight codes
// with v_mfma_f32_16x16x32_f16 over 16 vectors and 16 rows.  Lane (g, n) =
// (lane / 16, lane % 16) holds A row n (vector n of the tile) and B column n
// (weight row n), k = 8g..8g+7, and receives D[vectors 4g..4g+3][row n], so
// the scale it applies is its own row's.  The lane's dword g of a sub-block
// holds its columns 8g..8g+7; a sub-block is two products with the same B,
// the hi parts then the lo parts, chained through the accumulator (so the
// products sum (hi + lo) * w), each dword of k holding two columns:
//   B  = [ w(0, 2),    w(4, 6),    w(1, 3),    w(5, 7)  ]
//   A1 = [hi(x0, x2), hi(x4, x6), hi(x1, x3), hi(x5, x7)],  A2 the lo parts.
// Per sub-block, row tile and vector tile: two products, then four f32
// multiply-adds for the scale.
//
// Work split.  A workgroup of 4 waves owns 16 RT weight rows (RT row tiles:
// 4, or 2 for up to 16 vectors) and a range of whole blocks; wave q takes
// blocks q, q + 4, ... of the range.  Per block a wave brings the RT tiles'
// weights into its LDS by LDS DMA (the next block's while it multiplies this
// one), then for each sub-block forms the x operands once and multiplies them
// with all RT row tiles.  When there are too few row groups to fill the GPU, the blocks of a
// row are split over S workgroups: each stores its partial sums, and the last
// of the S to finish (an arrival count per row group) adds the S partials in
// split order to y.  All sums run in a fixed order (sub-blocks, waves, then
// splits), so every call gives the same bits whichever workgroup finishes
// last.
#include <algorithm>

#include "lnskv_device.h"

namespace lnskv {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kQ4lBlockBytes = LNSKV_Q4L_DEVICE_BYTES;
constexpr int kQ4lTileVecs = 16;   // vectors per product (A rows)
constexpr int kQ4lMaxTiles = 4;    // vector tiles of q4l_gemv_acc_kernel (64 vectors)
constexpr int kQ4lWaves = 4;       // waves per workgroup (split of a range's blocks)
constexpr int kQ4lTargetWgs = 256; // workgroups wanted per launch: one per CU
// Buffer resource word 3 for raw dword access (DATA_FORMAT = 32-bit).
constexpr int kQ4lBufferFormat = 0x00020000;
typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef __attribute__((address_space(3))) uint32_t lds_u32;

// High byte of the f16 +2^(m - 5) for m = 0..7 (m = 0: zero): (m + 10) << 2,
// bytes m = 0..3 and m = 4..7, for v_perm_b32.
constexpr uint32_t kMagLo = 0x34302C00u;
constexpr uint32_t kMagHi = 0x44403C38u;

// Eight weight nibbles (one dword: weights 2i and 2i+1 in byte i) -> the f16
// codes as dwords (w0, w2), (w4, w6), (w1, w3), (w5, w7).
__device__ __forceinline__ u32x4 weight_codes(uint32_t w) {
  const uint32_t he = __builtin_amdgcn_perm(kMagHi, kMagLo, w & 0x07070707u) | ((w << 4) & 0x80808080u);
  const uint32_t ho = __builtin_amdgcn_perm(kMagHi, kMagLo, (w >> 4) & 0x07070707u) | (w & 0x80808080u);
  // f16 k (low half) and k+1 (high half) of each dword: high bytes only
  u32x4 d;
  d.x = __builtin_amdgcn_perm(he, ho, 0x050C040Cu);  // he bytes 0, 1
  d.y = __builtin_amdgcn_perm(he, ho, 0x070C060Cu);  // he bytes 2, 3
  d.z = __builtin_amdgcn_perm(he, ho, 0x010C000Cu);  // ho bytes 0, 1
  d.w = __builtin_amdgcn_perm(he, ho, 0x030C020Cu);  // ho bytes 2, 3
  return d;
}

// The hi and lo f16 parts of two x values, each as one dword (a in the low
// half): hi = f16(x) and lo = f16(x - hi), rounded toward zero.  x - hi is
// exact in f32 (hi is x with its low mantissa bits cleared), formed as one
// mixed-precision fma of the f16 hi with m1 = -1 (a value the compiler cannot
// see, so that it keeps the fma instead of a conversion and a subtraction).
__device__ __forceinline__ void x_pair_parts(float a, float b, float m1, uint32_t& hi, uint32_t& lo) {
  const auto h = __builtin_amdgcn_cvt_pkrtz(a, b);
  const auto l = __builtin_amdgcn_cvt_pkrtz(__builtin_fmaf((float)h[0], m1, a), __builtin_fmaf((float)h[1], m1, b));
  hi = __builtin_bit_cast(uint32_t, h);
  lo = __builtin_bit_cast(uint32_t, l);
}

// Waits until at most N vector-memory loads of this wave are outstanding
// (gfx9 s_waitcnt: vmcnt bits [3:0] and [15:14]; expcnt and lgkmcnt left open).
template <int N>
__device__ __forceinline__ void q4l_wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// 16-row tiles per workgroup (and per wave) for T vector tiles: each x
// operand a wave splits serves this many tiles; with one vector tile, two
// (measured faster: more row groups and a shorter merge).
constexpr int q4l_row_tiles(int T) { return T == 1 ? 2 : 4; }
// Outputs (vector, row) one workgroup produces for T vector tiles.
constexpr int q4l_wg_outputs(int T) { return T * kQ4lTileVecs * 16 * q4l_row_tiles(T); }

struct Q4lArgs {
  const uint8_t* W;
  const float* x;
  float* y;
  float* part;    // [S][groups][q4l_wg_outputs(T)] partial sums (S > 1)
  uint32_t* cnt;  // [groups] arrival counts, zero between calls (S > 1)
  uint32_t* err;  // host word set to 1 on a count above S - 1 (a header that was not zero)
  int64_t x_stride, y_stride;
  int rows, bpr, n_vec;
  int groups;     // row groups of 16 q4l_row_tiles(T) rows
  int split;      // S: workgroups per row group
  int bpw;        // blocks per workgroup (the last may hold fewer)
  int tiles;      // q4l_gemm_acc_kernel: 64-vector tiles (groups = row groups x tiles)
};

// Workgroup (row group rg, split sp) = blockIdx.x (rg fastest).
template <int T>
__global__ __launch_bounds__(kQ4lWaves * kWave) void q4l_gemv_acc_kernel(Q4lArgs a) {
  constexpr int RT = q4l_row_tiles(T);
  constexpr int RW = 16 * RT;                                // rows per workgroup
  constexpr int E = q4l_wg_outputs(T);                       // outputs per workgroup
  constexpr int kPer = E / (kQ4lWaves * kWave);              // outputs per thread
  constexpr int kChunks = RW * 9;                            // 16-byte chunks of a weight tile
  constexpr int kDma = (kChunks + kWave - 1) / kWave;        // LDS DMA instructions per tile
  constexpr int kTileStride = kDma * kWave * 16;             // LDS bytes per tile slot (padding included)
  constexpr int kRedBytes = kQ4lWaves * E * 4;
  constexpr int kTileBytes = kQ4lWaves * 2 * kTileStride;   // two slots per wave
  constexpr int kLds = kTileBytes > kRedBytes ? kTileBytes : kRedBytes;
  static_assert(E % (kQ4lWaves * kWave) == 0, "outputs per thread");
  __shared__ __attribute__((aligned(16))) uint8_t lds[kLds];
  __shared__ int merge;

  const int tid = (int)threadIdx.x;
  // q: the wave index, made visibly uniform so that offsets derived from it
  // stay in scalar registers
  const int lane = tid & (kWave - 1), q = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int g = lane >> 4, n = lane & 15;
  const int rg = (int)blockIdx.x % a.groups, sp = (int)blockIdx.x / a.groups;
  const int row0 = rg * RW;
  const int b_end = min(a.bpr, (sp + 1) * a.bpw);

  // the y entries this thread adds to (if it is the one to add them) are
  // loaded now so that the read-modify-write adds no memory round trip at the
  // end
  float yv[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int idx = tid + u * kQ4lWaves * kWave;
    const int t = idx / (kQ4lTileVecs * RW), v = (idx / RW) % kQ4lTileVecs, r = idx % RW;
    const int vec = t * kQ4lTileVecs + v;
    yv[u] = vec < a.n_vec && row0 + r < a.rows ? a.y[(int64_t)vec * a.y_stride + row0 + r] : 0.0f;
  }

  float4v acc[T][RT];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[t][r] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

  const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)a.W, (short)0, (int)((int64_t)a.rows * a.bpr * kQ4lBlockBytes), kQ4lBufferFormat);
  lds_u8* const wslot = (lds_u8*)&lds[q * 2 * kTileStride];
  // this lane's x row for each tile (vectors past n_vec read vector 0; their
  // outputs are never stored), at its 8 columns of a sub-block
  const float* xrow[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int vec = t * kQ4lTileVecs + n;
    xrow[t] = a.x + (int64_t)(vec < a.n_vec ? vec : 0) * a.x_stride + 8 * g;
  }

  float m1;
  asm volatile("v_mov_b32 %0, -1.0" : "=v"(m1));
  // The RT tiles of block b (RW rows x 144 bytes, chunk 9 r + c) into LDS by
  // LDS DMA; lanes past the tile load its first chunk into the padding.  Rows
  // past the matrix read row 0 of the group (their outputs are never stored).
  auto weight_dma = [&](int b, lds_u8* dst) {
#pragma unroll
    for (int k = 0; k < kDma; ++k) {
      const int idx = kWave * k + lane;
      const int r = idx < kChunks ? idx / 9 : 0, c = idx < kChunks ? idx % 9 : 0;
      const int rr = row0 + r < a.rows ? row0 + r : row0;
      const int off = (int)(((int64_t)rr * a.bpr + b) * kQ4lBlockBytes + 16 * c);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wrsrc, (__attribute__((address_space(3))) void*)(dst + 1024 * k), 16,
                                               off, 0, 0, 0);
    }
  };
  // Two tile slots per wave: the next block's tiles are on their way while
  // this block is multiplied (its slot's LDS reads are all consumed by then).
  int b = sp * a.bpw + q;
  if (b < b_end) weight_dma(b, wslot);
  for (int i = 0; b < b_end; b += kQ4lWaves, ++i) {  // wave-uniform
    lds_u8* const wl = wslot + (i & 1) * kTileStride;
    const bool more = b + kQ4lWaves < b_end;
    __builtin_amdgcn_sched_barrier(0);
    if (more) weight_dma(b + kQ4lWaves, wslot + ((i + 1) & 1) * kTileStride);
    // x of sub-block j + 1 is loaded while sub-block j is multiplied
    float4v xb[2][T][2];
    auto load_x = [&](int j, float4v (&dst)[T][2]) {
#pragma unroll
      for (int t = 0; t < T; ++t) {
        dst[t][0] = *reinterpret_cast<const float4v*>(xrow[t] + 256 * b + 32 * j);
        dst[t][1] = *reinterpret_cast<const float4v*>(xrow[t] + 256 * b + 32 * j + 4);
      }
    };
    __builtin_amdgcn_sched_barrier(0);
    load_x(0, xb[0]);
    // The compiler does not order LDS reads after an LDS DMA: this block's
    // DMAs were issued before the next block's and sub-block 0's x loads, and
    // loads complete in order, so once no more than those are outstanding the
    // tiles are in LDS.
    __builtin_amdgcn_sched_barrier(0);
    if (more)
      q4l_wait_vmcnt<kDma + T * 2>();
    else
      q4l_wait_vmcnt<T * 2>();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j + 1 < 8) load_x(j + 1, xb[(j + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      // x columns 8g + 0..7 of vector n (p: 0..3, v: 4..7), hi parts in
      // A1, lo parts in A2, in the k order of weight_codes
      half8 a1[T], a2[T];
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const float4v p = xb[j & 1][t][0], v = xb[j & 1][t][1];
        uint32_t h0, h1, h2, h3, l0, l1, l2, l3;
        x_pair_parts(p[0], p[2], m1, h0, l0);
        x_pair_parts(v[0], v[2], m1, h1, l1);
        x_pair_parts(p[1], p[3], m1, h2, l2);
        x_pair_parts(v[1], v[3], m1, h3, l3);
        a1[t] = __builtin_bit_cast(half8, u32x4{h0, h1, h2, h3});
        a2[t] = __builtin_bit_cast(half8, u32x4{l0, l1, l2, l3});
      }
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        const lds_u8* trow = wl + kQ4lBlockBytes * (16 * r + n);
        const uint32_t wj = *(const lds_u32*)(trow + 16 + 16 * j + 4 * g);
        const uint32_t sw = *(const lds_u32*)(trow + 4 * (j >> 1));
        const half8 codes = __builtin_bit_cast(half8, weight_codes(wj));
        const float scale = (float)__builtin_bit_cast(_Float16, (uint16_t)((j & 1) ? (sw >> 16) : (sw & 0xFFFFu)));
#pragma unroll
        for (int t = 0; t < T; ++t) {
          float4v d = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1[t], codes, float4v{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_f16(a2[t], codes, d, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[t][r][e] = fmaf(scale, d[e], acc[t][r][e]);
        }
      }
    }
  }

  // lane (g, n): vectors 4g..4g+3 of each tile, row n of each row tile.  The
  // weight tiles are dead once every wave is past its products.
  __syncthreads();
  float* red = reinterpret_cast<float*>(lds);  // [wave][t][vector][row]
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int e = 0; e < 4; ++e) red[((q * T + t) * kQ4lTileVecs + 4 * g + e) * RW + 16 * r + n] = acc[t][r][e];
  __syncthreads();
  float sum[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int idx = tid + u * kQ4lWaves * kWave;
    float s = red[idx];
#pragma unroll
    for (int w = 1; w < kQ4lWaves; ++w) s += red[w * E + idx];
    sum[u] = s;
  }
  if (a.split > 1) {
    // Store this workgroup's partials as device-scope stores (written through
    // to where every XCD reads), wait until they have completed, then count
    // the workgroup in; the last of the row group's S adds them up.
    float* mine = a.part + ((int64_t)sp * a.groups + rg) * E;
#pragma unroll
    for (int u = 0; u < kPer; ++u)
      __hip_atomic_store(mine + tid + u * kQ4lWaves * kWave, sum[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      const uint32_t old = __hip_atomic_fetch_add(a.cnt + rg, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const bool last = old == (uint32_t)(a.split - 1);
      if (old > (uint32_t)(a.split - 1) && a.err)  // not a zeroed header: flagged for lnskv_sync
        __hip_atomic_store(a.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      if (last) __hip_atomic_store(a.cnt + rg, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      merge = last;
    }
    __syncthreads();
    if (!merge) return;  // workgroup-uniform
    for (int s0 = 0; s0 < a.split; ++s0) {  // split order
      const float* ps = a.part + ((int64_t)s0 * a.groups + rg) * E;
      float pv[kPer];
#pragma unroll
      for (int u = 0; u < kPer; ++u)
        pv[u] = __hip_atomic_load(ps + tid + u * kQ4lWaves * kWave, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int u = 0; u < kPer; ++u) sum[u] = s0 == 0 ? pv[u] : sum[u] + pv[u];
    }
  }
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int idx = tid + u * kQ4lWaves * kWave;
    const int t = idx / (kQ4lTileVecs * RW), v = (idx / RW) % kQ4lTileVecs, r = idx % RW;
    const int vec = t * kQ4lTileVecs + v;
    if (vec >= a.n_vec || row0 + r >= a.rows) continue;
    a.y[(int64_t)vec * a.y_stride + row0 + r] = yv[u] + sum[u];
  }
}

// More than 64 vectors (a prompt chunk's o_proj): a workgroup of 8 waves owns
// 64 vectors x 128 rows; wave w multiplies rows 32 (w % 4) .. with all 64
// vectors over half w / 4 (128 columns) of every block of its range.  The
// kernel above re-reads the weights and splits x again for every 64 vectors and
// every 64 rows; here x is split once per 128 rows, into LDS, and a decoded
// weight operand serves 64 vectors.
//   D[vec][row] = sum_k A[vec][k] B[k][row]   (v_mfma_f32_32x32x16_f16)
// Lane (hl, n) = (lane / 32, lane % 32) holds A of vector n and B of weight
// row n, k = 8 hl .. + 7, and receives D[vectors 8 (i / 4) + 4 hl + i % 4]
// [row n].  Of a 32-weight sub-block the lane decodes dwords 2 hl and 2 hl + 1:
// k step t multiplies the columns 16 hl + 8 t + 0..7, lo and hi parts, four
// products per sub-block and 32 vectors.
// A half block's sums stay in the products' accumulators: its weights enter as
// scale * 2^(m - 5) * 2^k, exact in f16, with one k per row and half block that
// takes the largest of the four scales to [2^13, 2^14).  The scales of a block
// are f16(g * 2^(sl - 7)), within 2^15 of each other, so the smallest weight is
// still a normal number.  (Scales further apart than 2^23, which no disk block
// has, would lose low bits of weights below 2^-24 of the largest.)  The halves
// then add up in f32, times 2^-k: 16 multiply-adds for 32 vectors and 128
// columns instead of 64.
// x and weights go through LDS a block at a time, both loaded in whole 128-byte
// lines two blocks ahead.  x in LDS, per half block: [k step s = 2 j + t][hi,
// lo][hl][vector ^ sw] 16-byte chunks of 8 columns, sw = 2 ((2 s + hl) % 8): 16
// lanes read 256 contiguous bytes, and the XOR spreads the stores of one
// vector's chunks over the banks.
// Bound by issue: a block takes a SIMD's two waves 2048 matrix cycles, ~2450
// issuing the other vector work (a third of it decoding weights) and, of the
// LDS, ~3000 (each wave reads the half's 32 KiB of x); what hides one behind
// another is the order below (without the slices, every LDS read waited for
// right before its product: 10% more time).  4096 x 4096: 46.7 to 51.5 us from
// card to card at 512 vectors, 21.1 at 128 (135.3 and 34.2 as launches of 64
// vectors); 8192 x 8192 at 512 vectors 174 (333).  Waves of 64 rows x a quarter
// block halve the LDS reads but leave no registers for operands read ahead: 15%
// more time.
constexpr int kGemmVecs = 64;              // vectors per workgroup
constexpr int kGemmRows = 128;             // weight rows per workgroup
constexpr int kGemmWaves = 8;
constexpr int kGemmOut = kGemmVecs * kGemmRows;
constexpr size_t kGemmPartBytes = kGemmOut * sizeof(float);  // partial sums of one workgroup
constexpr int kGemmHalf = 128;             // columns staged at once
constexpr float kGemmMaxScale = 16376.0f;  // the largest f16 below 2^14
constexpr int kGemmBuf = kGemmVecs * kGemmHalf * 4;  // LDS bytes of one half (hi and lo)

typedef float float16v __attribute__((ext_vector_type(16)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// weight_codes in the order (w0, w2), (w1, w3), (w4, w6), (w5, w7): the first
// two dwords belong to columns 0..3, the others to 4..7.
__device__ __forceinline__ u32x4 weight_codes_split(uint32_t w) {
  const u32x4 d = weight_codes(w);
  return u32x4{d.x, d.z, d.y, d.w};
}

// The hi and lo f16 parts of two x values: hi rounded toward zero (so that a
// finite x past 65504 keeps a finite hi and the rest in lo, to 131008), lo to
// nearest even (x = hi + lo to 2^-22): x - hi is exact, formed and rounded by
// one mixed-precision fma of the f16 hi with m1 = -1 (hidden from the compiler
// as above).
__device__ __forceinline__ void x_pair_split(float a, float b, float m1, uint32_t& hi, uint32_t& lo) {
  typedef _Float16 half2v __attribute__((ext_vector_type(2)));
  const auto h = __builtin_amdgcn_cvt_pkrtz(a, b);
  const half2v l = {(_Float16)__builtin_fmaf((float)h[0], m1, a), (_Float16)__builtin_fmaf((float)h[1], m1, b)};
  hi = __builtin_bit_cast(uint32_t, h);
  lo = __builtin_bit_cast(uint32_t, l);
}

// Workgroup barrier after this wave's LDS accesses; unlike __syncthreads() it
// leaves the loads of the next half in flight.
__device__ __forceinline__ void gemm_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__global__ __launch_bounds__(kGemmWaves * kWave) void q4l_gemm_acc_kernel(Q4lArgs a) {
  constexpr int kChunks = kGemmRows * 9;                                 // 16-byte chunks of a block's weights
  constexpr int kThreads = kGemmWaves * kWave;
  constexpr int kLoads = (kChunks + kThreads - 1) / kThreads;
  __shared__ __attribute__((aligned(16))) uint8_t xs_[4 * kGemmBuf];     // [2 blocks][half]
  __shared__ __attribute__((aligned(16))) uint8_t ws[kGemmRows * kQ4lBlockBytes];
  __shared__ int merge;
  const int tid = (int)threadIdx.x;
  const int lane = tid & (kWave - 1), w = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int kh = w >> 2;  // the half of every block this wave multiplies (and its threads stage)
  const int hl = lane >> 5, n = lane & 31;
  // vector tiles fastest: with blocks dealt to the XCDs in turn, workgroups
  // that share x (4 bytes a column and vector; the weights are 0.56) share an L2
  const int vt = (int)blockIdx.x % a.tiles, rest = (int)blockIdx.x / a.tiles;
  const int rgs = a.groups / a.tiles;
  const int rg = rest % rgs, sp = rest / rgs;
  const int vec0 = vt * kGemmVecs, row0 = rg * kGemmRows;
  const int b0 = sp * a.bpw, nb = min(a.bpr - b0, a.bpw);  // blocks of this split

  // x staging: columns 4c .. 4c + 3 of half kh, vectors sv + 8u; vectors past
  // n_vec read the last one (never stored).  Loads past the last block re-read
  // it, unused: a branch around them would make the compiler wait for the
  // loads of the block before as if none were in flight.
  const int c = tid & 31, sv = (tid & 255) >> 5;
  float m1;
  asm volatile("v_mov_b32 %0, -1.0" : "=v"(m1));
  float4v xr[8];
  auto load_x1 = [&](int i, int u) {
    xr[u] = *reinterpret_cast<const float4v*>(a.x + (int64_t)min(vec0 + sv + 8 * u, a.n_vec - 1) * a.x_stride +
                                              256 * (b0 + min(i, nb - 1)) + kGemmHalf * kh + 4 * c);
  };
  // chunk c / 2: sub-block c / 8, its dword (c / 2) % 4 = 2 hl + t, so k step s
  const int ss = 2 * (c >> 3) + ((c >> 1) & 1), sh = (c >> 2) & 1;
  const uint32_t xdst = (uint32_t)(kh * kGemmBuf + ss * 4096 + sh * 1024 + 8 * (c & 1));
  const uint32_t xsw = 2u * (uint32_t)((2 * ss + sh) & 7);
  auto stage_x1 = [&](int buf, int u) {
    uint32_t h0, h1, l0, l1;
    x_pair_split(xr[u][0], xr[u][2], m1, h0, l0);
    x_pair_split(xr[u][1], xr[u][3], m1, h1, l1);
    uint8_t* dst = xs_ + buf * (2 * kGemmBuf) + xdst + 16u * ((uint32_t)(sv + 8 * u) ^ xsw);
    *reinterpret_cast<u32x2*>(dst) = u32x2{h0, h1};
    *reinterpret_cast<u32x2*>(dst + 2048) = u32x2{l0, l1};
  };
  // weight staging: chunks tid + 512 u of the tile's rows (rows past the
  // matrix read its last one)
  u32x4 wr[kLoads];
  auto load_w = [&](int i) {
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int idx = min(tid + kThreads * u, kChunks - 1);
      wr[u] = *reinterpret_cast<const u32x4*>(
          a.W + ((int64_t)min(row0 + idx / 9, a.rows - 1) * a.bpr + b0 + min(i, nb - 1)) * kQ4lBlockBytes + 16 * (idx % 9));
    }
  };
  auto stage_w = [&]() {
#pragma unroll
    for (int u = 0; u < kLoads; ++u)
      if (tid + kThreads * u < kChunks) *reinterpret_cast<u32x4*>(ws + 16 * (tid + kThreads * u)) = wr[u];
  };

  float16v acc[2];
#pragma unroll
  for (int q = 0; q < 32; ++q) acc[q >> 4][q & 15] = 0.0f;
  const uint8_t* wl = ws + (32 * (w & 3) + n) * kQ4lBlockBytes;
#pragma unroll
  for (int u = 0; u < 8; ++u) load_x1(0, u);
  load_w(0);
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    stage_x1(0, u);
    load_x1(1, u);
  }
  stage_w();
  load_w(1);
  gemm_barrier();
  for (int i = 0; i < nb; ++i) {
    const uint8_t* xb = xs_ + (i & 1) * (2 * kGemmBuf) + kh * kGemmBuf + 1024 * hl;
    // x operands of sub-block j: [k step][lo, hi][32 vectors]
    half8 xa[2][2][2][2];
    auto read_x = [&](int j, half8 (&o)[2][2][2]) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const uint8_t* x0 = xb + (2 * j + t) * 4096 + 16u * ((uint32_t)n ^ (2u * (uint32_t)((4 * j + 2 * t + hl) & 7)));
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          o[t][0][v] = *reinterpret_cast<const half8*>(x0 + 512 * v + 2048);
          o[t][1][v] = *reinterpret_cast<const half8*>(x0 + 512 * v);
        }
      }
    };
    // this lane's weights of the block, then the next block may be stored
    u32x2 wt[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) wt[j] = *reinterpret_cast<const u32x2*>(wl + 16 + 64 * kh + 16 * j + 8 * hl);
    const u32x2 scr = *reinterpret_cast<const u32x2*>(wl + 8 * kh);
    read_x(0, xa[0]);
    gemm_barrier();
    // the exponent of the largest |scale| (field e, 2^(e - 15); a subnormal one
    // counts as e = 1) to 13
    const uint32_t mag0 = scr[0] & 0x7FFF7FFFu, mag1 = scr[1] & 0x7FFF7FFFu;
    const uint32_t top = max(max(mag0 & 0xFFFFu, mag0 >> 16), max(mag1 & 0xFFFFu, mag1 >> 16));
    // Infinite scales (an effective scale past f16) enter as the largest finite
    // one, the finite ones beside them as zero, and the half's sum is multiplied
    // by infinity: as products they would meet x parts and codes of zero.  NaN
    // scales likewise.
    const bool nonfinite = top >= 0x7C00u;
    const int k = nonfinite ? -64 : 28 - max((int)(top >> 10), 1);
    auto weights = [&](int j, int t) {
      const uint32_t sb = scr[j >> 1];
      const float s0 = (float)__builtin_bit_cast(_Float16, (uint16_t)((j & 1) ? sb >> 16 : sb & 0xFFFFu));
      const _Float16 s1 = (_Float16)__builtin_amdgcn_fmed3f(ldexpf(s0, k), -kGemmMaxScale, kGemmMaxScale);
      return __builtin_bit_cast(half8, weight_codes_split(wt[j][t])) * half8{s1, s1, s1, s1, s1, s1, s1, s1};
    };
    float16v d[2];
#pragma unroll
    for (int q = 0; q < 32; ++q) d[q >> 4][q & 15] = 0.0f;
    half8 wa[2][2];  // the weight operands of sub-blocks j and j + 1, [k step]
    wa[0][0] = weights(0, 0);
    wa[0][1] = weights(0, 1);
    // Sub-block j's products, the lo parts first (their roundings are 2^-11 of
    // the hi parts'); between each two, a slice of the other work: sub-block j +
    // 1's operands, the next block's x to LDS and the loads of the one after.
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      auto products = [&](int p) {
#pragma unroll
        for (int v = 0; v < 2; ++v)
          d[v] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xa[j & 1][p & 1][p >> 1][v], wa[j & 1][p & 1], d[v], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      };
      __builtin_amdgcn_sched_barrier(0);
      if (j < 3) read_x(j + 1, xa[(j + 1) & 1]);
      products(0);
      stage_x1((i + 1) & 1, 2 * j);  // that buffer was last read before the barrier at this block's start
      load_x1(i + 2, 2 * j);
      products(1);
      if (j < 3) wa[(j + 1) & 1][0] = weights(j + 1, 0);
      products(2);
      stage_x1((i + 1) & 1, 2 * j + 1);
      load_x1(i + 2, 2 * j + 1);
      products(3);
      if (j < 3) wa[(j + 1) & 1][1] = weights(j + 1, 1);
    }
    stage_w();
    load_w(i + 2);
    const float back = nonfinite ? (float)__builtin_bit_cast(_Float16, (uint16_t)top) : ldexpf(1.0f, -k);
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[v][q] = fmaf(back, d[v][q], acc[v][q]);
    gemm_barrier();
  }

  // The two halves of the waves swap: kh = 0 keeps vectors 0..31 of the tile,
  // kh = 1 vectors 32..63.
  float* swap = reinterpret_cast<float*>(xs_) + (w & 3) * (16 * kWave) + lane;
  float16v sum;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    swap[kh * (64 * kWave) + i * kWave] = kh ? acc[0][i] : acc[1][i];
    sum[i] = kh ? acc[1][i] : acc[0][i];
  }
  gemm_barrier();
#pragma unroll
  for (int i = 0; i < 16; ++i) sum[i] += swap[(1 - kh) * (64 * kWave) + i * kWave];

  if (a.split > 1) {
    // as above: the last of the group's splits adds all of them in split order
    float* part = a.part + (int64_t)(rg * a.tiles + vt) * kGemmOut + tid;
    const int64_t step = (int64_t)a.groups * kGemmOut;
#pragma unroll
    for (int i = 0; i < 16; ++i)
      __hip_atomic_store(part + sp * step + i * kGemmWaves * kWave, sum[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      uint32_t* cnt = a.cnt + rg * a.tiles + vt;
      const uint32_t old = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const bool all = old == (uint32_t)(a.split - 1);
      if (old > (uint32_t)(a.split - 1) && a.err)
        __hip_atomic_store(a.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      if (all) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      merge = all;
    }
    __syncthreads();
    if (!merge) return;  // workgroup-uniform
    for (int s0 = 0; s0 < a.split; ++s0) {
      float pv[16];
#pragma unroll
      for (int i = 0; i < 16; ++i)
        pv[i] = __hip_atomic_load(part + s0 * step + i * kGemmWaves * kWave, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int i = 0; i < 16; ++i) sum[i] = s0 == 0 ? pv[i] : sum[i] + pv[i];
    }
  }
  const int row = row0 + 32 * (w & 3) + n;
  if (row >= a.rows) return;
  const int v0 = vec0 + 32 * kh + 4 * hl;  // this lane's vectors: v0 + 8 (i / 4) + i % 4
  float yv[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int vec = v0 + 8 * (i >> 2) + (i & 3);
    yv[i] = vec < a.n_vec ? a.y[(int64_t)vec * a.y_stride + row] : 0.0f;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int vec = v0 + 8 * (i >> 2) + (i & 3);
    if (vec < a.n_vec) a.y[(int64_t)vec * a.y_stride + row] = yv[i] + sum[i];
  }
}

// The launch plan for rw rows per workgroup: row groups, split and blocks per
// workgroup.
void q4l_plan(int rows, int bpr, int rw, int* groups, int* split, int* bpw) {
  const int G = (rows + rw - 1) / rw;
  int S = 1;
  if (G < kQ4lTargetWgs) S = std::max(1, std::min((kQ4lTargetWgs + G - 1) / G, bpr / kQ4lWaves));
  const int per = (bpr + S - 1) / S;
  *groups = G;
  *split = (bpr + per - 1) / per;
  *bpw = per;
}

template <int T>
void launch_q4l(Q4lArgs a, hipStream_t st) {
  q4l_plan(a.rows, a.bpr, 16 * q4l_row_tiles(T), &a.groups, &a.split, &a.bpw);
  q4l_gemv_acc_kernel<T><<<(unsigned)(a.groups * a.split), kQ4lWaves * kWave, 0, st>>>(a);
}

// The many-vector kernel's plan: blocks are split over S workgroups while there
// is a CU without one (its LDS holds one workgroup), each with at least 4 blocks
// (four take 13.5 us at 1024 x 1024, four and a merge 18.2 at 1024 x 4096), as
// far as a workspace of ws_bytes holds the partial sums.  Us with this split |
// within the partial sums of 64-vector launches (half the workgroups or fewer) |
// as such launches: 65 vectors, 4096 x 4096 20.7 | 25.2 | 24.3, 8192 x 8192
// 47.9 | 71.6 | 56.4, 16 x 4096 17.2 | 36.6 | 20.3; 129 vectors, 4096 x 14336
// 70.2 | 118 | 96.9.
void q4l_gemm_plan(Q4lArgs* a, size_t ws_bytes) {
  a->tiles = (a->n_vec + kGemmVecs - 1) / kGemmVecs;
  a->groups = (a->rows + kGemmRows - 1) / kGemmRows * a->tiles;
  const size_t fit = ws_bytes > kWsHeaderBytes ? (ws_bytes - kWsHeaderBytes) / kGemmPartBytes : 0;
  const int by_shape = std::min(kQ4lTargetWgs / a->groups, a->bpr / 4);
  const int S = std::max(1, (int)std::min((size_t)by_shape, fit / (size_t)a->groups));
  a->bpw = (a->bpr + S - 1) / S;
  a->split = (a->bpr + a->bpw - 1) / a->bpw;
}

// Workspace: the arrival counts (LNSKV_WORKSPACE_HEADER_BYTES, zero between
// calls) and the partial sums of a split launch.  A split needs fewer than
// kQ4lTargetWgs row groups, so S * groups < 2 kQ4lTargetWgs whatever the rows
// (q4l_wg_outputs grows with T, so the launch with the most tiles is largest);
// with fewer than 2 kQ4lWaves blocks a row there is no split and no workspace.
size_t q4l_ws_bytes(int cols, int n_vec) {
  const int bpr = cols / 256;
  if (bpr < 2 * kQ4lWaves) return 0;
  const int T = std::min((n_vec + kQ4lTileVecs - 1) / kQ4lTileVecs, kQ4lMaxTiles);
  return kWsHeaderBytes + (size_t)2 * kQ4lTargetWgs * (size_t)q4l_wg_outputs(T) * sizeof(float);
}

// What launches of the gemv kernel, 64 vectors at a time, use: 0 when none of
// them splits (then they need no workspace at all), else at most
// q4l_ws_bytes(cols, n_vec).
size_t q4l_gemv_ws_bytes(int rows, int cols, int n_vec) {
  const int bpr = cols / 256;
  const int n_tiles = (n_vec + kQ4lTileVecs - 1) / kQ4lTileVecs;
  size_t most = 0;
  for (int t0 = 0; t0 < n_tiles; t0 += kQ4lMaxTiles) {
    const int T = std::min(n_tiles - t0, kQ4lMaxTiles);
    int groups = 0, split = 0, bpw = 0;
    q4l_plan(rows, bpr, 16 * q4l_row_tiles(T), &groups, &split, &bpw);
    if (split > 1) most = std::max(most, (size_t)split * groups * (size_t)q4l_wg_outputs(T) * sizeof(float));
  }
  return most > 0 ? kWsHeaderBytes + most : 0;
}

}  // namespace
}  // namespace lnskv

using namespace lnskv;

extern "C" int lnskv_q4l_workspace_size(int32_t cols, int32_t n_vec, size_t* bytes) {
  clear_error();
  if (!bytes) return fail(LNSKV_ERR_INVALID, "bytes must be non-null");
  if (cols <= 0 || n_vec <= 0) return fail(LNSKV_ERR_INVALID, "cols %d and n_vec %d must be positive", cols, n_vec);
  if (cols % 256 != 0) return fail(LNSKV_ERR_UNSUPPORTED, "cols %d must be a multiple of 256", cols);
  *bytes = q4l_ws_bytes(cols, n_vec);
  return LNSKV_OK;
}

extern "C" int lnskv_q4l_gemv_accumulate(const void* blocks_dev, const float* x_dev, float* y_dev, int32_t rows,
                                         int32_t cols, int32_t n_vec, int32_t x_stride, int32_t y_stride,
                                         void* ws, size_t ws_bytes, lnskv_stream_t stream) {
  clear_error();
  if (!blocks_dev || !x_dev || !y_dev) return fail(LNSKV_ERR_INVALID, "blocks, x and y must be non-null");
  if (rows <= 0 || cols <= 0 || n_vec <= 0)
    return fail(LNSKV_ERR_INVALID, "rows %d, cols %d and n_vec %d must be positive", rows, cols, n_vec);
  if (cols % 256 != 0) return fail(LNSKV_ERR_UNSUPPORTED, "cols %d must be a multiple of 256", cols);
  if (x_stride < cols || y_stride < rows)
    return fail(LNSKV_ERR_INVALID, "x_stride %d must be >= cols %d and y_stride %d >= rows %d", x_stride, cols,
                y_stride, rows);
  if ((int64_t)rows * (cols / 256) * LNSKV_Q4L_DEVICE_BYTES > INT32_MAX)
    return fail(LNSKV_ERR_UNSUPPORTED, "a Q4L matrix over 2 GiB of blocks (%d x %d)", rows, cols);
  if (x_stride % 4 != 0 || (reinterpret_cast<uintptr_t>(x_dev) & 15) != 0 ||
      (reinterpret_cast<uintptr_t>(blocks_dev) & 15) != 0)
    return fail(LNSKV_ERR_INVALID, "x and the blocks must be 16-byte aligned and x_stride a multiple of 4");
  const hipStream_t st = (hipStream_t)stream;
  Q4lArgs a{};
  a.W = static_cast<const uint8_t*>(blocks_dev);
  a.x = x_dev;
  a.y = y_dev;
  a.x_stride = x_stride;
  a.y_stride = y_stride;
  a.rows = rows;
  a.bpr = cols / 256;
  a.n_vec = n_vec;
  const bool many = n_vec > kQ4lMaxTiles * kQ4lTileVecs;
  // need: what the launch uses.  The many-vector kernel also takes a workspace
  // below the size query's answer, or a library buffer that cannot grow under
  // capture, that holds what gemv launches would use, and then splits less.
  size_t need = q4l_gemv_ws_bytes(rows, cols, n_vec), least = need;
  if (many) {
    q4l_gemm_plan(&a, SIZE_MAX);
    need = a.split > 1 ? kWsHeaderBytes + (size_t)a.split * (size_t)a.groups * kGemmPartBytes : 0;
    least = std::min(least, need);
  }
  if (need > 0) {
    size_t have = ws_bytes;
    if (ws == nullptr) {
      if (int rc = library_buffer(2, need, least, &ws, &have, st)) return rc;
    } else if (ws_bytes < least) {
      return fail(LNSKV_ERR_WORKSPACE, "workspace of %zu bytes, %zu needed", ws_bytes, need);
    } else if ((reinterpret_cast<uintptr_t>(ws) & 15) != 0) {
      return fail(LNSKV_ERR_WORKSPACE, "workspace must be 16-byte aligned");
    }
    if (have < need) q4l_gemm_plan(&a, least);
    a.cnt = static_cast<uint32_t*>(ws);
    a.part = reinterpret_cast<float*>(static_cast<uint8_t*>(ws) + kWsHeaderBytes);
    a.err = ws_error_word(stream, true);
  }
  // past 64 vectors the gemv kernel would run once per 64.  Over 418 shapes of
  // 16 to 50000 rows, 256 to 14336 columns and 65 to 640 vectors the other kernel
  // took less time at every one: nearest (0.99) for a second round of a few
  // workgroups (16385 x 14336 at 65 vectors, 251.8 us against 254.2), 20.7
  // against 24.3 at 4096 x 4096 and 65, 48.1 against 139.5 at 512
  if (many) {
    q4l_gemm_acc_kernel<<<(unsigned)(a.groups * a.split), kGemmWaves * kWave, 0, st>>>(a);
    return hip_check("q4l gemm kernel launch");
  }
  switch ((n_vec + kQ4lTileVecs - 1) / kQ4lTileVecs) {
    case 1: launch_q4l<1>(a, st); break;
    case 2: launch_q4l<2>(a, st); break;
    case 3: launch_q4l<3>(a, st); break;
    default: launch_q4l<4>(a, st); break;
  }
  return hip_check("q4l gemv kernel launch");
}
