// Blockwise symmetric FP8 (OCP e4m3) quantiser for gfx950.
//
// Replaces fp8_blockwise_symmetric_quantization<QUANT_M, 128, SCALE_TRANSPOSE>
// (reference: examples/005.fp8.mm.cu:439-563): per block amax -> s = amax / 448.f ->
// q = e4m3(s ? x / s : 0), the code of the IEEE-correct fp32 quotient (quotient_codes below
// finds it without dividing), round-to-nearest-even and
// saturation to +-448; a block of zeros gives s = 0 and q = 0.  Scale layouts:
//   QUANT_M == 1:   transposed s[(n/128)*M + m]      plain s[m*ceil(N/128) + n/128]
//   QUANT_M == 128: transposed s[(n/128)*M + m/128]  plain s[(m/128)*ceil(N/128) + n/128]
// (row stride M in both transposed forms, as written at :494 and :532).
// HBM-bound: x is read once (4 B/element) and q written once (1 B/element); the 128x128 form
// keeps its block in registers between the amax pass and the conversion.
// Rows may be ragged (any M); N must be a multiple of 4 (float4 accesses, as in the reference).
#include "device_common.hip.h"
#include "kernels.h"
#include "quotient.hip.h"

namespace llmmm {

// e4m3 codes of v[0..3] / s, s = amax / 448, equal bit for bit to converting the correctly rounded fp32 quotients by the correctly rounded scale -- almost
// always without computing those.  An IEEE fp32 division per element made the quantisers ALU-bound (the same element rate from bf16 and from fp32 inputs).
// Instead: v * (rcp(s) (1 - 2^-21)) and v * (rcp(s) (1 + 2^-21)): rcp(s) is within 2^-23 (relative) of 1 / s, its product with the
// factor and the product with v add 2^-24 each, so both are within 2^-22 of the quotient times its factor and bracket the quotient
// and its fp32 rounding; if they convert to the same code, then -- the conversion being monotone -- so does the
// correctly rounded quotient (`plain`).
// No clamp there: |v rcp(s)| < 448 (1 + 2^-20), and everything below 464 converts to 448.
// Otherwise the lane computes the quotients (rounded_codes): where one lies within 2^-20 of a rounding boundary of the 3-bit mantissa (about 3 in 10^5
// elements), where an element is NaN -- the hardware's code 0xFF in both brackets, the only one with all of its low seven bits set; the code becomes
// 0x7F --, and where amax lies outside 2^-60 .. 2^100 (a block that holds an infinity or nothing but NaN, one so small or large that something on the
// way leaves the normal range), here by division.  A block of zeros has the codes 0.
struct BlockScale {
  float s;       // amax / 448
  float dn, up;  // rcp(s) (1 -+ 2^-21)
  bool  plain;   // they hold
  bool  zero;    // a block of zeros: codes 0
};
__device__ __forceinline__ BlockScale block_scale(float amax)
{
  const float s = scale_of_amax(amax), r = __builtin_amdgcn_rcpf(s);
  return {s, r * (1.0f - 0x1p-21f), r * (1.0f + 0x1p-21f), amax >= 0x1p-60f && amax <= 0x1p100f, amax == 0.f};
}
__device__ __forceinline__ uint32_t bracketed_codes(f32x4 v, const BlockScale& k, bool& plain)
{
  int lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[0] * k.dn, v[1] * k.dn, 0, false);
  lo     = __builtin_amdgcn_cvt_pk_fp8_f32(v[2] * k.dn, v[3] * k.dn, lo, true);
  int hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[0] * k.up, v[1] * k.up, 0, false);
  hi     = __builtin_amdgcn_cvt_pk_fp8_f32(v[2] * k.up, v[3] * k.up, hi, true);
  const uint32_t nan = (((uint32_t)lo & 0x7F7F7F7Fu) + 0x01010101u) & 0x80808080u;
  plain = (((((uint32_t)lo ^ (uint32_t)hi) | nan) == 0u) & k.plain) | k.zero;
  return k.zero ? 0u : (uint32_t)lo;
}
__device__ __forceinline__ uint32_t divided_codes(f32x4 v, float amax, float& s)
{
  s = amax / 448.0f;
  if (s == 0.f) return 0u;
  return pack_e4m3x4_sat(v[0] / s, v[1] / s, v[2] / s, v[3] / s);
}
__device__ __forceinline__ uint32_t rounded_codes(f32x4 v, float amax, float& s)
{
  if (__builtin_expect(!(amax >= 0x1p-60f && amax <= 0x1p100f), 0)) return divided_codes(v, amax, s);
  s             = scale_of_amax(amax);
  const float y = refined_reciprocal(s, __builtin_amdgcn_rcpf(s));
  return pack_e4m3x4_in_range(rounded_quotient(v[0], s, y), rounded_quotient(v[1], s, y), rounded_quotient(v[2], s, y), rounded_quotient(v[3], s, y));
}
__device__ __forceinline__ uint32_t quotient_codes(f32x4 v, float amax, const BlockScale& k, float& s)
{
  bool     plain;
  uint32_t c = bracketed_codes(v, k, plain);
  s          = k.s;
  if (__builtin_expect(!plain, 0)) c = divided_codes(v, amax, s);
  return c;
}

// The NI chunks of a thread of the row kernels (t, t + 256, ..; those past the row's end dropped): codes, and the scales from the first lane of each block.
// On many rows these kernels are bound by the vector instructions they issue, on few by the one pass a workgroup makes through code that is not in the
// instruction cache yet.  So the chunks run side by side without a branch, and the chunks in doubt go one after the other through one piece of code, instead
// of each through a copy of its own behind a branch of its own.  us per launch, RMSNorm and quantiser on bf16 rows that are not in the caches, with a division
// for the scale and for each chunk in doubt / with the scale by scale_of_amax, behind branches of every chunk / now: 1 x 2560 2.17 / 2.14 / 2.04,
// 1 x 8192 3.76 / 3.67 / 3.11, 16 x 4096 2.83 / 2.75 / 2.54, 2048 x 2560 8.1 / 7.9 / 7.9, 4096 x 8192 30.5 / 29.3 / 28.5; rows of zeros, for which the first
// did nothing at all, 2048 x 2560 5.5 / 6.5 / 6.2.
template <int NI>
__device__ __forceinline__ void quantise_row(const f32x4 (&v)[NI], const float (&amax)[NI], unsigned t, unsigned chunks, uint8_t* __restrict__ q,
                                             float* __restrict__ scale, int M, int m)
{
  uint32_t code[NI];
  float    s[NI];
  unsigned doubt = 0;  // bit i: chunk i
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const BlockScale k = block_scale(amax[i]);
    bool             plain;
    code[i] = bracketed_codes(v[i], k, plain);
    s[i]    = k.s;
    doubt |= (plain | (t + 256u * i >= chunks)) ? 0u : 1u << i;
  }
  while (doubt != 0u) {
    const int i = __builtin_ctz(doubt);
    doubt &= doubt - 1u;
    f32x4 vi = v[0];
    float ai = amax[0], si;
#pragma unroll
    for (int j = 1; j < NI; ++j) vi = i == j ? v[j] : vi, ai = i == j ? amax[j] : ai;
    const uint32_t ci = rounded_codes(vi, ai, si);
#pragma unroll
    for (int j = 0; j < NI; ++j) code[j] = i == j ? ci : code[j], s[j] = i == j ? si : s[j];
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const unsigned c = t + 256u * i;
    if (c < chunks) {
      *(uint32_t*)(q + 4 * c) = code[i];
      if ((t & 31) == 0) scale[(c >> 5) * (unsigned)M + m] = s[i];
    }
  }
}

// The reference starts its block maximum from (float)INT_MIN (examples/005.fp8.mm.cu:456) and its comparison never
// takes a NaN, so a block that holds nothing but NaN keeps that seed: scale INT_MIN / 448, codes 0x7F.  fmaxf drops
// NaN operands the same way.
constexpr float QUANT_AMAX_SEED = -2147483648.f;

__device__ __forceinline__ float amax4(float m, f32x4 v)
{
  return fmaxf(fmaxf(m, fmaxf(__builtin_fabsf(v[0]), __builtin_fabsf(v[1]))), fmaxf(__builtin_fabsf(v[2]), __builtin_fabsf(v[3])));
}

// 1 x 128 blocks.  Half a wavefront (32 lanes x float4) owns one block; a workgroup of 256
// threads covers 8 consecutive rows of one 128-column group per step and strides over rows.
template <bool TRANSPOSE>
__global__ void __launch_bounds__(256) quant_1x128_kernel(const float* __restrict__ x, uint8_t* __restrict__ q,
                                                          float* __restrict__ scale, int M, int N, int rows_per_wg)
{
  const int tid   = threadIdx.x;
  const int sub   = tid >> 5;        // which of the 8 rows of a step
  const int l32   = tid & 31;
  const int nb    = blockIdx.x;      // 128-column group
  const int n     = nb * 128 + l32 * 4;
  const int nbn   = (N + 127) >> 7;
  const int mbeg  = blockIdx.y * rows_per_wg;
  const int mend  = min(M, mbeg + rows_per_wg);
  const bool live = n < N;
  // four rows per thread and pass: their loads go out together, before the first row's cross-lane amax and divisions
  constexpr int U = 4;
  for (int m0 = mbeg + sub; m0 < mend; m0 += 8 * U) {
    f32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int m = m0 + 8 * u;
      v[u]        = f32x4{0.f, 0.f, 0.f, 0.f};
      if (live && m < mend) v[u] = __builtin_nontemporal_load((const f32x4*)(x + (size_t)m * N + n));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int m = m0 + 8 * u;
      if (m >= mend) break;  // uniform over the half-wavefront that shares the row
      float a = QUANT_AMAX_SEED;
      if (live) a = amax4(a, v[u]);
      a = half_wave_max(a);
      float          s;
      const uint32_t c = quotient_codes(v[u], a, block_scale(a), s);
      if (live) *(uint32_t*)(q + (size_t)m * N + n) = c;
      if (l32 == 0) {
        if (TRANSPOSE)
          scale[(size_t)nb * M + m] = s;
        else
          scale[(size_t)m * nbn + nb] = s;
      }
    }
  }
}

// 128 x 128 blocks: one workgroup of 256 threads per block, 16 float4 per thread in registers.  Bound by HBM on whole weights
// (19456 x 2560: 43.3 us = 5.8 TB/s, 49.4 with dependent loads; 8192 x 4096: 29.9, 33.8; 2560 x 9728: 22.2, 29.0), by one block's
// load latency on small ones (1024 x 1024: 5.2 us, 11.3).
template <bool TRANSPOSE>
__global__ void __launch_bounds__(256) quant_128x128_kernel(const float* __restrict__ x, uint8_t* __restrict__ q,
                                                            float* __restrict__ scale, int M, int N)
{
  __shared__ float wmax[4];
  const int tid  = threadIdx.x;
  const int l32  = tid & 31;
  const int sub  = tid >> 5;
  const int nb   = blockIdx.x;
  const int mb   = blockIdx.y;
  const int n    = nb * 128 + l32 * 4;
  const int nbn  = (N + 127) >> 7;
  const bool live = n < N;
  // Sixteen loads without a condition, all in flight before the first maximum: a lane past the last row or column takes the
  // last one of this block again, which the maximum does not notice and the stores below drop.  (Behind a condition each load
  // and its maximum share a branch, and every load waits for the one before it.)
  const int nc = min(n, N - 4);
  f32x4     v[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = __builtin_nontemporal_load((const f32x4*)(x + (size_t)min(mb * 128 + r * 8 + sub, M - 1) * N + nc));
  float a = QUANT_AMAX_SEED;
#pragma unroll
  for (int r = 0; r < 16; ++r) a = amax4(a, v[r]);
  a = half_wave_max(a);
  a = wave_xor_max<32>(a);
  if ((tid & 63) == 0) wmax[tid >> 6] = a;
  __syncthreads();
  a             = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
  // The scale is the workgroup's: what hangs on it is decided here, once, and not for every chunk.  A scale of zero: codes of zero (whatever NaN the block
  // holds: the maximum drops them).  Where the brackets do not hold otherwise they become NaN, and every chunk divides.
  // (With flags looked at per chunk 256 x 512 took 4.08 us, now 3.65; 1024 x 1024 4.33 / 3.86; 4096 x 4096 16.9 / 16.6; zeros 2048 x 2560 6.0 / 4.7.)
  BlockScale k = block_scale(a);
  if (__builtin_expect(!k.plain, 0)) {
    k.s  = a / 448.0f;
    k.dn = k.up = __builtin_nanf("");
  }
  k.plain = true, k.zero = false;
  if (tid == 0) {
    if (TRANSPOSE)
      scale[(size_t)nb * M + mb] = k.s;
    else
      scale[(size_t)mb * nbn + nb] = k.s;
  }
  if (__builtin_expect(k.s == 0.f, 0)) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = mb * 128 + r * 8 + sub;
      if (live && m < M) *(uint32_t*)(q + (size_t)m * N + n) = 0u;
    }
    return;
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int m = mb * 128 + r * 8 + sub;
    bool      plain;
    uint32_t  c = bracketed_codes(v[r], k, plain);
    if (__builtin_expect(!plain, 0)) c = pack_e4m3x4_sat(v[r][0] / k.s, v[r][1] / k.s, v[r][2] / k.s, v[r][3] / k.s);
    if (live && m < M) *(uint32_t*)(q + (size_t)m * N + n) = c;
  }
}

// RMSNorm fused in front of the 1 x 128 activation quantiser (the "RMSNorm + fp8 dynamic quant" fusion the reference
// plans, README.md:16; no reference kernel):
//   y[m,k] = (x[m,k] * r) * w[k],  r = 1 / sqrt(sum_k x[m,k]^2 / K + eps),  then q, s = quant_1x128(y), scales transposed.
// The sum of squares has one fixed order, which the CPU oracle restates, so that results are bit-exact and do not
// depend on which of the two kernels below runs: the row is cut into chunks of four elements; chunk c belongs to
// virtual lane c % 256, which accumulates its chunks in ascending order with one fused multiply-add per element;
// the 256 partial sums are combined per group of 64 by an xor butterfly (32, 16, .. 1) and the four group sums as
// (G0 + G1) + (G2 + G3).  A second pass normalises and quantises: a 128-column group is 32 consecutive chunks =
// half a wavefront in either kernel, so its amax needs five cross-lane steps.  HBM traffic: x once, q once.
//   * rmsnorm_quant_row_kernel:   one 256-thread workgroup per row (a thread is a virtual lane), the row held in
//     registers: K <= 10240.  Measured at K = 2560 against a wavefront per row: 3.2 instead of 8.2 us at M = 16 (a
//     single wavefront works through the row's 40 divisions per lane on its own), 6.9 instead of 9.4 us at M = 2048.
//   * rmsnorm_quant_1x128_kernel: one wavefront per row (a lane plays four virtual lanes), the row read twice:
//     longer rows.
// One chunk (4 elements) per lane of row m: normalise, take the amax of the 128-column group (the 32 chunks of this
// half of the wavefront), quantise, store codes and the group's scale.
__device__ __forceinline__ void rmsnorm_quant_chunk(f32x4 v, float r, const float* __restrict__ w, uint8_t* __restrict__ q,
                                                    float* __restrict__ scale, int m, int M, int K, int c, int chunks, int lane)
{
  const bool live = c < chunks;
  f32x4      y    = {0.f, 0.f, 0.f, 0.f};
  if (live) {
    const f32x4 wv = *(const f32x4*)(w + 4 * c);
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = (v[e] * r) * wv[e];
  }
  float a = amax4(0.f, y);
  a = half_wave_max(a);
  float          s;
  const uint32_t cd = quotient_codes(y, a, block_scale(a), s);
  if (live) {
    *(uint32_t*)(q + (size_t)m * K + 4 * c) = cd;
    if ((lane & 31) == 0) scale[(size_t)(c >> 5) * M + m] = s;
  }
}

// One wavefront per row, any K: the row is read twice (the second time from the L2).  A lane plays the four
// virtual lanes lane, lane + 64, lane + 128, lane + 192.
template <typename IN_T>
__global__ void __launch_bounds__(256) rmsnorm_quant_1x128_kernel(const IN_T* __restrict__ x, const float* __restrict__ w, float eps,
                                                                  uint8_t* __restrict__ q, float* __restrict__ scale, int M, int K)
{
  const int lane = threadIdx.x & 63;
  const int m    = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (m >= M) return;  // whole wavefronts leave: no barrier below
  const IN_T* xr      = x + (size_t)m * K;
  const int   chunks  = K >> 2;
  float       part[4] = {0.f, 0.f, 0.f, 0.f};
  for (int c0 = 0; c0 < chunks; c0 += 256) {
#pragma unroll
    for (int gidx = 0; gidx < 4; ++gidx) {
      const int c = c0 + 64 * gidx + lane;
      if (c < chunks) {
        const f32x4 v = load_row4<IN_T>(xr + 4 * c);
#pragma unroll
        for (int e = 0; e < 4; ++e) part[gidx] = __builtin_fmaf(v[e], v[e], part[gidx]);
      }
    }
  }
#pragma unroll
  for (int gidx = 0; gidx < 4; ++gidx) part[gidx] = wave_sum(part[gidx]);
  const float acc = (part[0] + part[1]) + (part[2] + part[3]);
  const float ms  = acc / (float)K;
  const float r   = 1.0f / __builtin_sqrtf(ms + eps);
  // second pass: lanes beyond the row's end still take part in the cross-lane maxima (with zeros)
  for (int c0 = 0; c0 < chunks; c0 += 64) {
    const int c = c0 + lane;
    f32x4     v = {0.f, 0.f, 0.f, 0.f};
    if (c < chunks) v = load_row4<IN_T>(xr + 4 * c);
    rmsnorm_quant_chunk(v, r, w, q, scale, m, M, K, c, chunks, lane);
  }
}

// One workgroup of 256 threads per row: thread t is virtual lane t and owns chunks t, t + 256, ...  NI = chunks per
// thread held in registers (K <= 1024 * NI).
template <typename IN_T, int NI>
__global__ void __launch_bounds__(256) rmsnorm_quant_row_kernel(const IN_T* __restrict__ x, const float* __restrict__ w, float eps,
                                                                uint8_t* __restrict__ q, float* __restrict__ scale, int M, int K)
{
  __shared__ float group_sum[4];
  const unsigned t   = threadIdx.x;
  const int   m      = blockIdx.x;
  const IN_T* xr     = x + (size_t)m * K;
  uint8_t*    qr     = q + (size_t)m * K;  // (a row's base is uniform: a lane adds 32 bits to it)
  const unsigned chunks = (unsigned)K >> 2;
  f32x4       held[NI], wv[NI];
  float       acc = 0.f;
  // every load without a condition (threads past the end of the row load its last chunk and drop it): behind one, the bf16
  // values are converted inside the branch, and each chunk's load waits for the one before it
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const unsigned c = min(t + 256u * i, chunks - 1u);
    held[i]     = load_row4<IN_T>(xr + 4 * c);
    wv[i]       = *(const f32x4*)(w + 4 * c);
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    if (t + 256u * i >= chunks) held[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_fmaf(held[i][e], held[i][e], acc);
  }
  acc = wave_sum(acc);
  if ((t & 63) == 0) group_sum[t >> 6] = acc;
  __syncthreads();
  const float total = (group_sum[0] + group_sum[1]) + (group_sum[2] + group_sum[3]);
  const float ms    = total / (float)K;
  const float r     = 1.0f / __builtin_sqrtf(ms + eps);
  float       amax[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) held[i][e] = (held[i][e] * r) * wv[i][e];  // zeros beyond the row's end
    amax[i] = amax4(0.f, held[i]);
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) amax[i] = half_wave_max(amax[i]);
  quantise_row<NI>(held, amax, t, chunks, qr, scale, M, m);
}

// The decoder-block epilogue behind a projection back to the hidden size (O, down), in one kernel behind the GEMM's
// fp32 planes:  h = (plane 0 + plane 1 + ... in split order) + residual,  hidden = T(h) (the new residual stream),
// y = RMSNorm(float(hidden)) * weight,  q, s = quant_1x128(y) -- the A operand of the next projection.  It takes the
// place of the split-K reduce kernel and of the separate RMSNorm + quantiser launch; the norm sees the rounded hidden
// state, exactly what a separate kernel reading `hidden` would see, and follows the same fixed summation order
// (rmsnorm_quant_row_kernel), so its codes and scales are those of the unfused sequence, bit for bit.
// One 256-thread workgroup per row; N <= 1024 * NI columns.
template <typename T, int NI>
__global__ void __launch_bounds__(256) planes_add_rmsnorm_quant_kernel(const float* __restrict__ planes, int S, const T* residual, T* hidden,
                                                                       const float* __restrict__ w, float eps, uint8_t* __restrict__ q,
                                                                       float* __restrict__ scale, int M, int N)
{
  __shared__ float group_sum[4];
  const unsigned t    = threadIdx.x;
  const int    m      = blockIdx.x;
  const unsigned chunks = (unsigned)N >> 2;
  const size_t plane  = (size_t)M * N;
  const T*     res    = residual + (size_t)m * N;  // (bases are uniform: a lane adds 32 bits to them)
  T*           hid    = hidden + (size_t)m * N;
  uint8_t*     qr     = q + (size_t)m * N;
  f32x4        held[NI], wv[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    held[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    wv[i]   = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // Everything that does not depend on the planes is requested first; then the planes, W of them in flight per chunk,
  // summed in split order (0 + p0 + p1 + ...: the order of the split-K reduce kernel).  Threads past the end of the
  // row load its last chunk and drop it.
  f32x4 rv[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const unsigned c = min(t + 256u * i, chunks - 1u);
    rv[i]       = load_row4<T>(res + 4 * c);
    wv[i]       = *(const f32x4*)(w + 4 * c);
  }
  // W planes in flight: 64 to 128 registers of loads beside the row's own; only the planes that exist are asked for.  That costs waves:
  // 177 VGPRs and two per SIMD for three chunks, 256 and one for eight and ten, where a form that held eight planes of three chunks or
  // two of ten, existing or not, took 126 and four, 170 and two.  With the GEMM in front of it that form was slower or even on
  // 1 .. 2048 rows of 2048 .. 10240 columns behind 1 .. 8 planes (us, then / now: 640 x 2560 x 4096 25.6 / 25.1, 768 x 3072 x 8192
  // 44.6 / 43.7, 16 x 8192 x 8192 24.5 / 22.0, 16 x 10240 x 2048 15.5 / 14.3).
  constexpr int W = NI <= 4 ? 8 : 32 / NI;
  for (int s0 = 0; s0 < S; s0 += W) {
    f32x4 p[W][NI];
#pragma unroll
    for (int u = 0; u < W; ++u)
      if (s0 + u < S) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const unsigned c = min(t + 256u * i, chunks - 1u);
          p[u][i]     = __builtin_nontemporal_load((const f32x4*)(planes + (size_t)(s0 + u) * plane + (size_t)m * N + 4 * c));
        }
      }
#pragma unroll
    for (int u = 0; u < W; ++u)
      if (s0 + u < S) {
#pragma unroll
        for (int i = 0; i < NI; ++i) held[i] += p[u][i];
      }
  }
  float acc = 0.f;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const unsigned c = t + 256u * i;
    if (c < chunks) {
      const f32x4 h = held[i] + rv[i];
      store_row4<T>(hid + 4 * c, h);
      // the norm reads the hidden state as stored (rounded to T)
      if constexpr (sizeof(T) == 4)
        held[i] = h;
      else {
#pragma unroll
        for (int e = 0; e < 4; ++e) held[i][e] = (float)(T)h[e];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_fmaf(held[i][e], held[i][e], acc);
    }
    else
      held[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  acc = wave_sum(acc);
  if ((t & 63) == 0) group_sum[t >> 6] = acc;
  __syncthreads();
  const float total = (group_sum[0] + group_sum[1]) + (group_sum[2] + group_sum[3]);
  const float ms    = total / (float)N;
  const float r     = 1.0f / __builtin_sqrtf(ms + eps);
  float       amax[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) held[i][e] = (held[i][e] * r) * wv[i][e];
    amax[i] = amax4(0.f, held[i]);
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) amax[i] = half_wave_max(amax[i]);
  quantise_row<NI>(held, amax, t, chunks, qr, scale, M, m);
}

// Chunks a thread of the two row kernels holds: the smallest of these that covers the row.  With 3 and 10 only, a row of 4096
// columns behind eight planes loaded ten chunks of every plane where it has four, two planes at a time: 16 rows
// 13.2 us, now 5.9 (and 5.3 -> 3.7 for rmsnorm_quant_row_kernel on 16 rows of 4096, 3.0 -> 2.5 on one of 2560, with the loads and the
// reductions below).
#define LLMMM_ROW_CHUNKS(COLUMNS, GO) \
  switch (((COLUMNS) + 1023) / 1024) { \
    case 1:                           \
    case 2: GO(2); break;             \
    case 3: GO(3); break;             \
    case 4: GO(4); break;             \
    case 5: GO(5); break;             \
    case 6:                           \
    case 7:                           \
    case 8: GO(8); break;             \
    default: GO(10); break;           \
  }

template <typename T>
static void launch_planes_add_rmsnorm_quant(const float* planes, int S, const void* residual, void* hidden, const float* w, float eps, void* q, float* scale,
                                            int M, int N, hipStream_t stream)
{
#define LLMMM_GO(NI)                                                                                                                             \
  hipLaunchKernelGGL((planes_add_rmsnorm_quant_kernel<T, NI>), dim3(M), dim3(256), 0, stream, planes, S, (const T*)residual, (T*)hidden, w, eps, \
                     (uint8_t*)q, scale, M, N)
  LLMMM_ROW_CHUNKS(N, LLMMM_GO)
#undef LLMMM_GO
}

hipError_t planes_add_rmsnorm_quant_launch(int hidden_dtype, const float* planes, int S, const void* residual, void* hidden, const float* w,
                                           float eps, void* q, float* scale, int M, int N, hipStream_t stream)
{
  if (N > 1024 * 10) return hipErrorInvalidValue;
  switch (hidden_dtype) {
    case LLMMM_DTYPE_F16: launch_planes_add_rmsnorm_quant<_Float16>(planes, S, residual, hidden, w, eps, q, scale, M, N, stream); break;
    case LLMMM_DTYPE_BF16: launch_planes_add_rmsnorm_quant<__bf16>(planes, S, residual, hidden, w, eps, q, scale, M, N, stream); break;
    case LLMMM_DTYPE_F32: launch_planes_add_rmsnorm_quant<float>(planes, S, residual, hidden, w, eps, q, scale, M, N, stream); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <typename T>
static void launch_rmsnorm_quant(const void* x, const float* w, float eps, void* q, float* scale, int M, int K, hipStream_t stream)
{
#define LLMMM_GO(NI) hipLaunchKernelGGL((rmsnorm_quant_row_kernel<T, NI>), dim3(M), dim3(256), 0, stream, (const T*)x, w, eps, (uint8_t*)q, scale, M, K)
  if (K <= 1024 * 10)
    LLMMM_ROW_CHUNKS(K, LLMMM_GO)
  else
    hipLaunchKernelGGL((rmsnorm_quant_1x128_kernel<T>), dim3((M + 3) / 4), dim3(256), 0, stream, (const T*)x, w, eps, (uint8_t*)q, scale, M, K);
#undef LLMMM_GO
}

hipError_t rmsnorm_quant_launch(int in_dtype, const void* x, const float* w, float eps, void* q, float* scale, int M, int K,
                                hipStream_t stream)
{
  switch (in_dtype) {
    case LLMMM_DTYPE_F16: launch_rmsnorm_quant<_Float16>(x, w, eps, q, scale, M, K, stream); break;
    case LLMMM_DTYPE_BF16: launch_rmsnorm_quant<__bf16>(x, w, eps, q, scale, M, K, stream); break;
    case LLMMM_DTYPE_F32: launch_rmsnorm_quant<float>(x, w, eps, q, scale, M, K, stream); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

__global__ void fill_u32_kernel(uint32_t* p, uint32_t value, size_t n)
{
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = value;
}

hipError_t fill_u32_launch(uint32_t* p, uint32_t value, size_t n, hipStream_t stream)
{
  hipLaunchKernelGGL(fill_u32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, p, value, n);
  return hipGetLastError();
}

hipError_t quant_fp8_launch(int quant_m, int transpose, const float* x, void* q, float* scale, int M, int N, hipStream_t stream)
{
  const int nbn = (N + 127) / 128;
  if (quant_m == 1) {
    // enough workgroups to fill the chip, at least 8 rows each
    int rows_per_wg = 64;
    while (rows_per_wg > 8 && (long)nbn * ((M + rows_per_wg - 1) / rows_per_wg) < 2048) rows_per_wg >>= 1;
    dim3 grid(nbn, (M + rows_per_wg - 1) / rows_per_wg);
    if (transpose)
      hipLaunchKernelGGL(quant_1x128_kernel<true>, grid, dim3(256), 0, stream, x, (uint8_t*)q, scale, M, N, rows_per_wg);
    else
      hipLaunchKernelGGL(quant_1x128_kernel<false>, grid, dim3(256), 0, stream, x, (uint8_t*)q, scale, M, N, rows_per_wg);
  }
  else {
    dim3 grid(nbn, (M + 127) / 128);
    if (transpose)
      hipLaunchKernelGGL(quant_128x128_kernel<true>, grid, dim3(256), 0, stream, x, (uint8_t*)q, scale, M, N);
    else
      hipLaunchKernelGGL(quant_128x128_kernel<false>, grid, dim3(256), 0, stream, x, (uint8_t*)q, scale, M, N);
  }
  return hipGetLastError();
}

}  // namespace llmmm
