// Device-side building blocks shared by the gfx950 GEMM kernels: vector types, the LDS tile
// layout with its bank-conflict-free swizzle, the direct global->LDS tile loader and small
// wavefront helpers.  gfx950 (CDNA4) only: 64-wide wavefronts, 160 KB LDS, 64 LDS banks.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace llmmm {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));

#define LLMMM_LDS __attribute__((address_space(3)))
#define LLMMM_GLOBAL __attribute__((address_space(1)))

// ---------------------------------------------------------------------------------------------
// K-major operand tiles in LDS (FP8): a tile row holds 128 bytes of the K extent as eight 16-byte chunks;
// row r / chunk c lives at  r * 128 + ((c ^ swz(r)) << 4).
// ds_read_b128 serves a wavefront in four passes of 16 lanes -- {0-3,12-15,20-23,24-27},
// {4-11,16-19,28-31} and the same two sets + 32 (measured on gfx950) -- and a pass is
// conflict-free when its 16 lanes touch 16 different 16-byte slots of the 256-byte bank row.
// SWZ_ROWS16 is matched to the lane -> (row, chunk) pattern of the 16x16x128 fp8 MFMA operands: lanes 16g..16g+15 read
// 16 consecutive rows at chunk 2g (+1).  The chunk is XOR-ed with row bits 1..3 and, for rows 4..11 of every 16, with
// 2, which cancels the chunk difference between the two halves of a pass.
// ---------------------------------------------------------------------------------------------
enum { SWZ_ROWS16 = 1 };

template <int SWZ>
struct KMajor {
  static_assert(SWZ == SWZ_ROWS16, "one placement only");
  static constexpr int ROW    = 128;  // bytes per tile row
  static constexpr int CHUNKS = ROW / 16;
  static constexpr int ROWS_PER_KB = 1024 / ROW;              // tile rows covered by one 1 KB load
};

template <int SWZ>
__device__ __forceinline__ int kmajor_swz(int r)
{
  return ((r >> 1) & 7) ^ ((((r >> 2) ^ (r >> 3)) & 1) << 1);
}
template <int SWZ>
__device__ __forceinline__ int kmajor_offset(int r, int c)
{
  return r * KMajor<SWZ>::ROW + ((c ^ kmajor_swz<SWZ>(r)) << 4);
}

// One wave copies 1024 bytes of a tile with a single LDS-direct load: lane l owns the 16 bytes
// at lds_group + 16*l, and fetches the logical (row, chunk) that the swizzle places there.
struct KMajorLane {
  int row;    // logical tile row this lane fetches
  int chunk;  // logical 16-byte chunk within the row
};
template <int SWZ>
__device__ __forceinline__ KMajorLane kmajor_lane(int group, int lane)
{
  KMajorLane p;
  p.row   = group * KMajor<SWZ>::ROWS_PER_KB + lane / KMajor<SWZ>::CHUNKS;
  p.chunk = (lane % KMajor<SWZ>::CHUNKS) ^ kmajor_swz<SWZ>(p.row);
  return p;
}

// 16 bytes per lane, global -> LDS without passing through registers (lane l's data lands at lds_addr + 16*l), written
// as inline assembly so that it stays invisible to the compiler's wait-count bookkeeping.
// While an LDS-direct load that the compiler knows about is in flight, every wait it inserts on
// its own becomes "all loads done", which defeats a deep software pipeline; kernels that keep
// many slices in flight issue all their vector-memory loads through these helpers and place the
// s_waitcnt themselves.  lds_addr is the wave-uniform LDS byte address (goes to M0).
__device__ __forceinline__ void asm_load_lds_16B(const void* gptr, unsigned lds_addr)
{
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(gptr), "s"(lds_addr) : "memory");
}
__device__ __forceinline__ void asm_load_16B(i32x4& dst, const void* gptr)
{
  asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(dst) : "v"(gptr) : "memory");
}
__device__ __forceinline__ void asm_load_8B(i32x2& dst, const void* gptr)
{
  asm volatile("global_load_dwordx2 %0, %1, off" : "=v"(dst) : "v"(gptr) : "memory");
}
__device__ __forceinline__ void asm_load_f32(float& dst, const void* gptr)
{
  asm volatile("global_load_dword %0, %1, off" : "=v"(dst) : "v"(gptr) : "memory");
}

// s_waitcnt vmcnt(N) lgkmcnt(0): at most N of this wave's vector-memory loads still in flight,
// every LDS access done.  simm16 = vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[5:4] << 14.
template <int N>
__device__ __forceinline__ void wait_vmcnt()
{
  static_assert(N >= 0 && N < 64, "vmcnt out of range");
  __builtin_amdgcn_s_waitcnt((N & 15) | 0x70 | ((N >> 4) << 14));
}

// Clock readings for the phase-accounting builds of the tile kernels: the constant 100 MHz counter and the shader's cycle
// counter (scalar reads; the values are stored with ordinary vector stores at the end of the kernel).
struct PhaseClock {
  unsigned long long real, cycles;
};
__device__ __forceinline__ PhaseClock phase_clock()
{
  PhaseClock c;
  c.real   = __builtin_amdgcn_s_memrealtime();
  c.cycles = __builtin_amdgcn_s_memtime();
  return c;
}

// Logical tile id -> (tm, tn).  Hardware hands consecutive workgroup ids to the 8 XCDs in turn,
// so ids congruent mod 8 share an L2: give each XCD a contiguous run of the grouped order
// (groups of up to four tile rows swept along n, all of one height but the last: 5 rows as 3 + 2, 13 as 4 + 4 + 4 + 1), whose members reuse the same few A and B panels.
// (Any number of tiles: XCD x owns tiles/8 of them and one more if x < tiles%8.  Dealing the ids of a tile count that 8 does not
// divide out in turn made every XCD read nearly all of both operands: FP8 384 x 3584 x 18944 in 84 tiles x 3 splits 45.4 us, 37.9 so;
// FP16 1152 x 3456 x 2048 in 243 tiles of 128 x 128 22.4 us, 19.7 so.)
// in_turn: tile ids in the hardware's order instead, in groups of four rows (see splits_in_turn in fp8_gemm.hip).
__device__ __forceinline__ void tile_coords(int wg, int tiles_m, int tiles_n, int& tm, int& tn, bool in_turn = false)
{
  const int tiles   = tiles_m * tiles_n;
  const int x       = wg & 7, rem = tiles & 7;
  const int L       = in_turn ? wg : x * (tiles >> 3) + (x < rem ? x : rem) + (wg >> 3);
  const int groups  = (tiles_m + 3) >> 2;
  const int group_m = in_turn ? 4 : (tiles_m + groups - 1) / groups;
  const int per     = group_m * tiles_n;
  const int group   = L / per;
  const int first   = group * group_m;
  const int gm      = (tiles_m - first) < group_m ? (tiles_m - first) : group_m;
  const int in      = L - group * per;
  tm                = first + in % gm;
  tn                = in / gm;
}

// mask = 16: v_permlane16_swap exchanges the odd 16-lane rows of its first register with the even rows of its second; from (v, v)
// it gives a = the even row of each pair in both rows, b = the odd row in both.  mask = 32: v_permlane32_swap, likewise for the
// halves of the wavefront.
// (The empty asm keeps them two values: the compiler otherwise takes both results for v and drops the operation on them.)
struct WavePair {
  float a, b;
};
template <int MASK>
__device__ __forceinline__ WavePair wave_swap_pair(float v)
{
  static_assert(MASK == 16 || MASK == 32, "row or half swap");
  const unsigned u = __builtin_bit_cast(unsigned, v);
  unsigned       x, y;
  if constexpr (MASK == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    x = r[0], y = r[1];
  }
  else {
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    x = r[0], y = r[1];
  }
  asm("" : "+v"(x), "+v"(y));
  return {__builtin_bit_cast(float, x), __builtin_bit_cast(float, y)};
}
// The value lane (l ^ mask) holds, for mask = 1, 2, 4, 8, 16 or 32.  Register moves but for 16: the reductions of the row kernels are
// chains of these, eleven long, and with ds_swizzle for 4, 8 and 16 (about 60 cycles a step instead of 8) seven of the eleven waited
// on the LDS crossbar (sums and maxima over 16 take the row swap above, which yields both operands):
//   1, 2     DPP quad permutes,
//   4        lane l + 4 for the lanes with bit 2 clear, l - 4 for the others: two DPP row shifts with complementary bank masks,
//   8        a DPP rotation of the 16-lane row by 8,
//   16       ds_swizzle, through the LDS crossbar after all: the row swap and its selection hold two more registers per value, and
//            in the kernel that fetches four values at once (the rotary embedding behind split-K planes) they cost the fifth wave
//            per SIMD: 107 instead of 93 VGPRs, 10240 columns at M = 128 29.0 -> 29.9 us,
//   32       the half swap above.
template <int MASK>
__device__ __forceinline__ float wave_xor_get(float v)
{
  const int iv = __builtin_bit_cast(int, v);
  if constexpr (MASK == 1)
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(iv, 0xB1, 0xf, 0xf, true));  // quad_perm [1,0,3,2]
  else if constexpr (MASK == 2)
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(iv, 0x4E, 0xf, 0xf, true));  // quad_perm [2,3,0,1]
  else if constexpr (MASK == 4) {
    const int up = __builtin_amdgcn_update_dpp(iv, iv, 0x104, 0xf, 0x5, false);                     // row_shl:4 into banks 0 and 2
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(up, iv, 0x114, 0xf, 0xa, false));  // row_shr:4 into banks 1 and 3
  }
  else if constexpr (MASK == 8)
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(iv, 0x128, 0xf, 0xf, true));  // row_ror:8
  else if constexpr (MASK == 16)
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(iv, (16 << 10) | 0x1f));
  else {
    const WavePair p = wave_swap_pair<MASK>(v);
    return (__lane_id() & MASK) ? p.a : p.b;
  }
}

// v op (the value of lane l ^ MASK), op = maximum / sum.  For 16 and 32 the swap already yields both operands, and both
// operations are commutative, so nothing has to be selected.
template <int MASK>
__device__ __forceinline__ float wave_xor_max(float v)
{
  if constexpr (MASK >= 16) {
    const WavePair p = wave_swap_pair<MASK>(v);
    return fmaxf(p.a, p.b);
  }
  else
    return fmaxf(v, wave_xor_get<MASK>(v));
}
template <int MASK>
__device__ __forceinline__ float wave_xor_sum(float v)
{
  if constexpr (MASK >= 16) {
    const WavePair p = wave_swap_pair<MASK>(v);
    return p.a + p.b;
  }
  else
    return v + wave_xor_get<MASK>(v);
}
// Maximum over the 32 lanes of each half of the wavefront, of block maxima: values that are never NaN and not negative, or the
// quantisers' one negative seed.  Such floats are ordered like their bits read as signed integers, and an integer maximum takes
// its DPP operand in the same instruction, where fmaxf costs three (the move, a quieting of the moved value, the maximum).  What
// bounds the row kernels on many rows is how many vector instructions a wave issues (2048 rows of 2560 bf16: about 500, eight
// waves on each SIMD); this form takes 12 fewer per maximum, less than the runs of a whole decoder layer differ by.  After
// the steps 1 and 2 all lanes of a quad agree, so a mirrored half row serves for step 4.
__device__ __forceinline__ float half_wave_max(float v)
{
  int a = __builtin_bit_cast(int, v);
  a     = max(a, __builtin_amdgcn_mov_dpp(a, 0xB1, 0xf, 0xf, true));   // quad_perm [1,0,3,2]
  a     = max(a, __builtin_amdgcn_mov_dpp(a, 0x4E, 0xf, 0xf, true));   // quad_perm [2,3,0,1]
  a     = max(a, __builtin_amdgcn_mov_dpp(a, 0x141, 0xf, 0xf, true));  // row_half_mirror
  a     = max(a, __builtin_amdgcn_mov_dpp(a, 0x128, 0xf, 0xf, true));  // row_ror:8
  const WavePair p = wave_swap_pair<16>(__builtin_bit_cast(float, a));
  return __builtin_bit_cast(float, max(__builtin_bit_cast(int, p.a), __builtin_bit_cast(int, p.b)));
}
// Sums over the halves and over all 64 lanes, the distant lanes first (the order the CPU oracle adds in).
__device__ __forceinline__ float half_wave_sum(float v) { return wave_xor_sum<1>(wave_xor_sum<2>(wave_xor_sum<4>(wave_xor_sum<8>(wave_xor_sum<16>(v))))); }
__device__ __forceinline__ float wave_sum(float v) { return half_wave_sum(wave_xor_sum<32>(v)); }

// ---------------------------------------------------------------------------------------------
// fp32 -> OCP e4m3, four codes per dword, as the reference's __nv_fp8_e4m3(float) gives them (round to nearest even,
// saturate to +-448, every NaN -> 0x7F; examples/005.fp8.mm.cu:482-485, examples/005.fp8.mm.opt.cu:445-454).
// v_cvt_pk_fp8_f32 rounds to nearest even and converts everything below 464 to 448, but writes 0xFF for a NaN of
// either sign and sign | 0x7F for larger magnitudes and infinities (measured).
// ---------------------------------------------------------------------------------------------
// Bytes whose low seven bits are all ones (the two NaN codes) lose their sign bit; other bytes are unchanged.
__device__ __forceinline__ uint32_t e4m3x4_nan_codes_to_7f(uint32_t c)
{
  const uint32_t m = ((c & 0x7F7F7F7Fu) + 0x01010101u) & 0x80808080u;
  return c & ~m;
}
// For values that are NaN or lie within +-448 (1 + 2^-20): quotients by a block's own scale, products with
// 448 / amax.  No clamp is needed then, and the only 0x7F / 0xFF bytes the hardware writes stand for NaN.
__device__ __forceinline__ uint32_t pack_e4m3x4_in_range(float a, float b, float c, float d)
{
  int v = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
  v     = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, v, true);
  return e4m3x4_nan_codes_to_7f((uint32_t)v);
}
// For any value: clamped to +-448 first (v_med3_f32 turns a NaN into a bound, so NaN is put back by hand).
__device__ __forceinline__ uint32_t pack_e4m3x4_sat(float a, float b, float c, float d)
{
  const uint32_t nan = (a != a ? 0x000000FFu : 0u) | (b != b ? 0x0000FF00u : 0u) | (c != c ? 0x00FF0000u : 0u) | (d != d ? 0xFF000000u : 0u);
  a     = __builtin_amdgcn_fmed3f(a, -448.f, 448.f);
  b     = __builtin_amdgcn_fmed3f(b, -448.f, 448.f);
  c     = __builtin_amdgcn_fmed3f(c, -448.f, 448.f);
  d     = __builtin_amdgcn_fmed3f(d, -448.f, 448.f);
  int v = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
  v     = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, v, true);
  return ((uint32_t)v & ~nan) | (0x7F7F7F7Fu & nan);
}

// 448 / amax of the fused re-quantisation (examples/005.fp8.mm.opt.cu:439-446), or 0 where that quotient is not finite: a
// group of zeros (the reference multiplies by 448 / 0 and writes NaN codes) and a group so small -- amax below 2^-119 --
// that the reciprocal overflows (the reference then writes +-448 for every non-zero element and NaN for the zeros).
// Such a group gets codes 0 (a NaN element stays NaN, 0x7F) next to its scale amax / 448; with a finite reciprocal every
// product lies within +-448 (1 + 2^-20), which is what pack_e4m3x4_in_range asks for.
__device__ __forceinline__ float requant_inv(float amax)
{
  const float inv = 448.f / amax;
  return inv < __builtin_inff() ? inv : 0.f;
}

// Four consecutive row elements of type float / bf16 / fp16 <-> fp32 (one 16- or 8-byte access).
template <typename IN_T>
__device__ __forceinline__ f32x4 load_row4(const IN_T* p);
template <>
__device__ __forceinline__ f32x4 load_row4<float>(const float* p)
{
  return *(const f32x4*)p;
}
template <>
__device__ __forceinline__ f32x4 load_row4<__bf16>(const __bf16* p)
{
  typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
  const bf16x4   v = *(const bf16x4*)p;
  return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}
template <>
__device__ __forceinline__ f32x4 load_row4<_Float16>(const _Float16* p)
{
  const f16x4 v = *(const f16x4*)p;
  return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}

template <typename T>
__device__ __forceinline__ void store_row4(T* p, f32x4 v);
template <>
__device__ __forceinline__ void store_row4<float>(float* p, f32x4 v)
{
  *(f32x4*)p = v;
}
template <>
__device__ __forceinline__ void store_row4<__bf16>(__bf16* p, f32x4 v)
{
  typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
  *(bf16x4*)p = bf16x4{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
}
template <>
__device__ __forceinline__ void store_row4<_Float16>(_Float16* p, f32x4 v)
{
  *(f16x4*)p = f16x4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
}

// ---------------------------------------------------------------------------------------------
// The hand-over of row maxima between the two workgroups that hold the halves of one 1x128 quantisation group (the SwiGLU outputs:
// 64 gate and the matching 64 up columns per workgroup).  `area` is [buffer 2][group][16-row block][half 2][16 rows] words of device
// memory, zero when the library is loaded, one per stream.  A slot holds (bits of the maximum) + 1 -- never 0, maxima of absolute
// values being neither negative nor NaN -- or 0 for "not written in this launch".  Two buffers take turns: a launch works in the one
// that holds zeros and clears its own slots of the other.  Which is which, a workgroup reads off its own row-0 slot of buffer 0 at kernel
// entry: written by nobody else, and both halves of a block take part in every launch that touches it, so they agree.  The state
// is kept per block of 16 rows, so launches with other row counts may follow each other.
// Device-scope relaxed atomics and no fence: the slots are all that is shared.  Waiting is safe because of where the halves sit
// (pair_place).  The wait is bounded all the same (20 ms of the 100 MHz clock); a wave that gives up counts itself in *timeouts
// and goes on with what it has.
// ---------------------------------------------------------------------------------------------
constexpr int PAIR_BLOCKS = 8;  // 16-row blocks of an area: M <= 128

// The group and half of a workgroup of `total` (an even number).  Ids go to the eight XCDs in turn and each XCD dispatches its share in order.
// Up to 31 workgroups per XCD the halves are neighbours by id: the smallest incomplete pair makes progress, and a second launch that waits
// like this one cannot take an XCD whole, even where two XCDs begin the two in different order.  A larger launch can (32 CUs, one workgroup
// on each), so its halves are eight ids apart, neighbours on one XCD, which then holds at most one incomplete pair of it.
// (Of the last ids, fewer than 16, the halves lie closer: a workgroup or two of each XCD.)  Not for all launches, because it moves what the XCDs
// read at a time: 28672 x 4096 pre-shuffled 22.5 us at M = 16 as neighbours by id, 25.4 on one XCD; other shapes differ by -3 .. +2 %.
__device__ __forceinline__ void pair_place(int id, int total, int& group, int& half)
{
  if (total <= 8 * 31) {
    group = id >> 1, half = id & 1;
    return;
  }
  const int first = id & ~15, r = id - first;
  const int apart = total - first >= 16 ? 8 : (total - first) >> 1;
  half  = r >= apart ? 1 : 0;
  group = (first >> 1) + r - half * apart;
}

struct PairSlots {
  unsigned* area;
  int       groups, group, half;
  __device__ __forceinline__ unsigned* slot(int buffer, int block, int h) const
  {
    return area + ((((size_t)buffer * groups + group) * PAIR_BLOCKS + block) * 2 + h) * 16;
  }
  // lane i < 16 of a 16-lane row: row i's maximum over this half
  __device__ __forceinline__ void publish(int cur, int block, int i, float a) const
  {
    __hip_atomic_store(slot(cur ^ 1, block, half) + i, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(slot(cur, block, half) + i, __builtin_bit_cast(unsigned, a) + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  // row i's maximum over the other half
  __device__ __forceinline__ float other(int cur, int block, int i, unsigned* timeouts) const
  {
    const unsigned*          src = slot(cur, block, half ^ 1) + i;
    const unsigned long long t0  = __builtin_amdgcn_s_memrealtime();
    unsigned                 w;
    for (;;) {
      w = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (__builtin_amdgcn_ballot_w64(w == 0u) == 0ull) break;
      if (__builtin_amdgcn_s_memrealtime() - t0 > 2000000ull) {
        if (__lane_id() == 0) atomicAdd(timeouts, 1u);
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    return __builtin_bit_cast(float, w - 1u);
  }
};

// silu(g) * u with the hardware's exp2 and reciprocal (each within about one ulp of fp32): far below the
// resolution of the e4m3 codes the result is quantised to.  g -> -inf gives -0, g -> +inf gives g * u.
__device__ __forceinline__ float silu_mul(float g, float u)
{
  const float e = __builtin_amdgcn_exp2f(g * -1.44269504088896340736f);  // exp(-g)
  return g * __builtin_amdgcn_rcpf(1.f + e) * u;
}

}  // namespace llmmm
