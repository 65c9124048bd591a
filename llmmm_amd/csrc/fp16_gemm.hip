// FP16 / BF16 GEMM for gfx950:  C[M,N] = A[M,K] * B,  fp32 accumulation, output rounded to T.
//
// Replaces the kernel behind LLMMM::fp16_mm<T> (reference: src/mm/fp16/mm.cu:6-42 launching
// src/mm/fp16/mm.cuh:657-684).  Layouts follow the reference: A[m*K+k] (mm.cuh:102),
// B[k*N+n] (mm.cuh:103), C[m*N+n] (mm.cuh:236).  A second B layout, Bt[n*K+k], is an extension.
//
// Design (nothing here is translated from the reference's mma.sync/ldmatrix code):
//  * one workgroup computes a BM x BN tile, one wavefront a WM x WN sub-tile built from v_mfma_f32_16x16x32_{f16,bf16}: on
//    this power-limited part that shape sustains about 16 % more FLOP/s than 32x32x16 on random operands.  The MFMA is issued
//    with B as the row operand and A as the column operand, so that each lane ends up with 4 consecutive n of one row m;
//  * the 256 x 256 tile is four waves of 128 x 128, one per SIMD: 256 accumulators in AGPRs, two sets of operand fragments in
//    VGPRs.  What a CU moves decides this kernel -- it takes in at most about 32 bytes per clock from its L2 and the board is at
//    its power limit -- and a 128 x 128 wave reads 16 fragments from LDS for 64 MFMAs where two 64 x 128 waves read 24.  A lone
//    wave must never wait, so the schedule is written out: every LDS read is issued a whole k step (64 MFMAs) before its data is
//    used, one LDS read or one half of a global load behind every second MFMA (an MFMA occupies the matrix pipe for four issue
//    slots), the MFMAs as inline assembly with the accumulator tied in place (left to the register allocator, the loop moves
//    160 accumulator registers per k step through VGPRs);
//  * K advances 64 elements per stage (two k steps): tile rows of 128 bytes, whole cache lines.  With 64-byte rows the same
//    kernel took 106 us at 4096^3 with Bt (98 us with whole lines): two half lines cost what two lines do;
//  * A and B tiles have LDS rings of their own (DA and DB stages), filled by LDS-direct loads.  One workgroup barrier per stage,
//    between its two k steps: by then every wave has its last fragments of the stage in registers, so the barrier frees the
//    stage's buffers, and it publishes the next stage.  The B tile of stage s + DB goes out behind the barrier, the A tile of
//    stage s + DA in the k step after it;
//  * A (and Bt) tiles are K-major and read with one ds_read_b128 per 16-row fragment (chunk XOR-ed with row bits 1..3:
//    conflict-free); a row-major B tile is kept as [k][n] and read with the transposing ds_read_b64_tr_b16, its 32-byte column
//    chunks XOR-ed with k bits;
//  * the epilogue lays each wave's result out row-major in LDS and stores whole rows;
//  * workgroup ids are remapped so that the tiles resident on one XCD share A/B panels in its L2.
// Measured (f16, us, row-major B / Bt; before: eight 64 x 128 waves, 64-byte rows, a ring of four 32-wide stages): 4096^3
// 109.7 / 108.9 -> 100.2 / 95.8 (1.37 / 1.43 PFLOP/s), 8192^3 829 / 846 -> 763 / 733, 3072^3 62.8 / 63.5 -> 58.0 / 54.1.
// At 4096^3 (row-major B) the matrix pipe is busy for 79 % of the K loop's cycles (clock readings in the kernel: 2592 per stage, 2048 of
// them MFMAs) and for 64 % of all shader cycles of a launch (counters); the clock is at the power limit, 1.8 - 2.0 GHz.
#include <utility>

#include "device_common.hip.h"
#include "kernels.h"

namespace llmmm {

template <typename T>
struct Vec16;
template <>
struct Vec16<_Float16> {
  typedef f16x8 vec;
};
template <>
struct Vec16<__bf16> {
  typedef bf16x8 vec;
};

// c += x * y, the accumulator tied to its AGPRs.  The compiler does not know this for an MFMA: whoever reads c afterwards
// places the wait states itself (see the end of the K loop).
template <typename T>
__device__ __forceinline__ void mfma_16x16x32(f32x4& c, typename Vec16<T>::vec x, typename Vec16<T>::vec y)
{
  if constexpr (__is_same(T, _Float16))
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(x), "v"(y));
  else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(x), "v"(y));
}

// WM x WN = a wave's sub-tile; DA, DB = stages in the LDS rings of the A and the B tile.
template <int BM, int BN, int WM, int WN, int DA_, int DB_>
struct Fp16Tile {
  static constexpr int MF = WM / 16, NF = WN / 16;  // 16-row / 16-column fragments per wave
  static constexpr int WAVES_M = BM / WM, WAVES_N = BN / WN, NW = WAVES_M * WAVES_N, NT = NW * 64;
  static constexpr int DA = DA_, DB = DB_;
  static constexpr int BK      = 64;        // elements of K per stage
  static constexpr int A_BYTES = BM * 128;  // K-major, 128 bytes per row
  static constexpr int B_BYTES = BN * 128;  // either layout: 64 x BN x 2 bytes
  static constexpr int B_ROW   = BN * 2;    // row pitch of the [k][n] layout
  static constexpr int B_RING  = DA * A_BYTES;  // LDS offset of the B ring
  static constexpr int LDS     = DA * A_BYTES + DB * B_BYTES;
  static constexpr int A_LOADS = (BM / 8) / NW, B_LOADS = (BN / 8) / NW, LOADS = A_LOADS + B_LOADS;  // 1 KB loads per wave and stage
  static constexpr int ROWS_PER_LOAD   = 8 * NW;        // K-major tiles: tile rows between two loads of a wave
  static constexpr int B_KROWS_PER_GRP = 1024 / B_ROW;  // [k][n] tile: k rows per 1 KB load
  static constexpr int READS = MF + NF, MFMAS = MF * NF;  // per k step
  static constexpr int AHEAD = DA - 1 > DB ? DA - 1 : DB;  // how far in front of the stage being computed loads go out
  // loads of a wave that may still be in flight when stage s + 1 has to be in LDS (those issued behind its own, see the K loop)
  static constexpr int IN_FLIGHT = DA > DB ? A_LOADS + (DB - 2) * LOADS : (DA - 2) * LOADS;
  static constexpr int PROLOGUE  = (DA - 2) * A_LOADS + (DB - 1) * B_LOADS;  // the same behind the prologue, for stage 0
  static_assert(DA >= 2 && DB >= 2 && PROLOGUE < 64 && IN_FLIGHT < 64, "vmcnt is a 6-bit counter");
  static_assert(NW % 2 == 0 && (BN & (BN - 1)) == 0, "the swizzles repeat every 16 rows; a [k][n] row divides 1 KB");
  static_assert(BM * BN * 2 <= LDS && LDS <= 160 * 1024, "the epilogue stages the tile in the rings");
};

// K-major tile: lanes 16g .. 16g+15 read 16 consecutive rows at chunk g (+ 4 in the second k step).  Two rows fill a 256-byte
// bank row; XOR-ing row bits 1..3 into the chunk keeps the 16 lanes of every ds_read_b128 pass on 16 different slots.
__device__ __forceinline__ int k128_swz(int r) { return (r >> 1) & 7; }
__device__ __forceinline__ int k128_offset(int r, int c) { return r * 128 + ((c ^ k128_swz(r)) << 4); }
// [k][n] tile: a transposing 64-bit read takes 4 x 4 row / chunk patches of rows 0..3 and 8..11 (+ 16 ..) in one pass.  The
// 32-byte column chunk of row k is XOR-ed with k bits that tell those eight rows apart; the 128-byte rows of a 64-column tile
// lie two to a bank row and need four values only.
template <int BN>
__device__ __forceinline__ int kn_swz(int k)
{
  return BN >= 128 ? (k & 3) | (((k >> 3) & 1) << 2) : ((k >> 1) & 1) | (((k >> 3) & 1) << 1);
}

// What a wave carries through the K loop.  Loads are LDS-direct and inline assembly (wave-uniform base in SGPRs, one constant
// byte offset per load in a VGPR), waits are placed by hand: the compiler, which would turn every wait it inserts into "all
// loads done" while it knows of an LDS-direct load in flight, never sees one.
template <typename T, int BM, int BN, int WM, int WN, int DA, int DB, bool B_NK>
struct Fp16Wave {
  typedef Fp16Tile<BM, BN, WM, WN, DA, DB> TC;
  typedef typename Vec16<T>::vec           vec;
  static constexpr int MF = TC::MF, NF = TC::NF;
  const T*        Ag;  // the tile's first row of A / of Bt, or its first column of B
  const T*        Bg;
  size_t          b_step;  // elements of B from one stage to the next
  int             K, wave, lane;
  unsigned        a_off[TC::A_LOADS], b_off[TC::B_LOADS];  // byte offsets of the lane's 16 bytes per load
  int             a_k, b_k[TC::B_LOADS];                   // k offset inside a stage of what the lane loads
  int             a_rd, b_rd[B_NK ? 1 : NF];               // LDS offsets of the lane's operand reads, first k step
  char LLMMM_LDS* lds;
  unsigned        lds_addr;
  f32x4           acc[NF][MF];

  // Load I of the A (B) tile of a stage into the ring slot at LDS offset `slot`.  A stage that K cuts short zero-fills the
  // missing part, so that the MFMAs need no masking.
  template <int I>
  __device__ __forceinline__ void load_a(int stage, unsigned slot) const
  {
    const unsigned dst = slot + (wave + I * TC::NW) * 1024;
    if (a_k < K - stage * TC::BK)
      sload(Ag + (size_t)stage * TC::BK, a_off[I], lds_addr + dst);
    else
      *(i32x4 LLMMM_LDS*)(lds + dst + lane * 16) = i32x4{0, 0, 0, 0};
  }
  template <int J>
  __device__ __forceinline__ void load_b(int stage, unsigned slot) const
  {
    const unsigned dst = slot + (wave + J * TC::NW) * 1024;
    if (b_k[J] < K - stage * TC::BK)
      sload(Bg + (size_t)stage * b_step, b_off[J], lds_addr + dst);
    else
      *(i32x4 LLMMM_LDS*)(lds + dst + lane * 16) = i32x4{0, 0, 0, 0};
  }
  static __device__ __forceinline__ void sload(const T* sbase, unsigned voff, unsigned lds_addr)
  {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_addr) : "memory");
  }
  template <int... I>
  __device__ __forceinline__ void load_a_tile(int stage, unsigned slot, std::integer_sequence<int, I...>) const
  {
    if (K - stage * TC::BK >= TC::BK)
      (sload(Ag + (size_t)stage * TC::BK, a_off[I], lds_addr + slot + (wave + I * TC::NW) * 1024), ...);
    else
      (load_a<I>(stage, slot), ...);
  }
  template <int... J>
  __device__ __forceinline__ void load_b_tile(int stage, unsigned slot, std::integer_sequence<int, J...>) const
  {
    if (K - stage * TC::BK >= TC::BK)
      (sload(Bg + (size_t)stage * b_step, b_off[J], lds_addr + slot + (wave + J * TC::NW) * 1024), ...);
    else
      (load_b<J>(stage, slot), ...);
  }

  // Fragment R (the A fragments first) of k step H of the stage whose tiles lie at LDS offsets sa, sb.
  template <int R, int H>
  __device__ __forceinline__ void read(unsigned sa, unsigned sb, vec (&a)[MF], vec (&b)[NF]) const
  {
    if constexpr (R < MF)
      a[R] = *(const vec LLMMM_LDS*)(lds + ((sa + a_rd) ^ (H * 64)) + R * 2048);
    else {
      constexpr int nf = R - MF;
      if constexpr (B_NK)
        b[nf] = *(const vec LLMMM_LDS*)(lds + ((sb + b_rd[0]) ^ (H * 64)) + nf * 2048);
      else {
        union {
          i16x4 h[2];
          vec   v;
        } u;
        u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((i16x4 LLMMM_LDS*)(lds + sb + b_rd[nf] + H * 32 * TC::B_ROW));
        u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((i16x4 LLMMM_LDS*)(lds + sb + b_rd[nf] + (H * 32 + 4) * TC::B_ROW));
        b[nf]  = u.v;
      }
    }
  }
  template <int H, int... R>
  __device__ __forceinline__ void read_all(unsigned sa, unsigned sb, vec (&a)[MF], vec (&b)[NF], std::integer_sequence<int, R...>) const
  {
    (read<R, H>(sa, sb, a, b), ...);
  }

  // Where in a k step things happen: read R behind MFMA read_pos(R) -- the last ones early enough to be back at the step's end --
  // and half P of the loads (even: M0 with the LDS address, odd: the load itself, so that an MFMA lies between the two) behind
  // MFMA load_pos(P).
  static constexpr int READ_SPAN = TC::MFMAS * 10 / 16;
  static constexpr int read_pos(int r) { return r * READ_SPAN / TC::READS; }
  static constexpr int load_pos(int p, int loads) { return (2 * p + 1) * TC::MFMAS / (4 * loads); }

  template <int H, int Q, int R>
  __device__ __forceinline__ void read_at(unsigned sa, unsigned sb, vec (&a)[MF], vec (&b)[NF]) const
  {
    if constexpr (read_pos(R) == Q) {
      __builtin_amdgcn_sched_barrier(0);
      read<R, H>(sa, sb, a, b);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  template <bool STEADY, bool IS_B, int Q, int P>
  __device__ __forceinline__ void load_at(const T* base, unsigned dst, int stage, unsigned slot, bool more) const
  {
    constexpr int NL = IS_B ? TC::B_LOADS : TC::A_LOADS, L = P / 2;
    static_assert(load_pos(2 * L, NL) < load_pos(2 * L + 1, NL), "M0 is written one MFMA ahead of the load");
    if constexpr (load_pos(P, NL) == Q) {
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (STEADY) {
        if constexpr (P % 2 == 0)
          asm volatile("s_add_u32 m0, %0, %1" ::"s"(dst), "n"(L * TC::NW * 1024) : "memory", "scc");
        else if constexpr (IS_B)
          asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(b_off[L]), "s"(base) : "memory");
        else
          asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(a_off[L]), "s"(base) : "memory");
      }
      else if constexpr (P % 2 == 1) {
        if (more) {
          if constexpr (IS_B)
            load_b<L>(stage, slot);
          else
            load_a<L>(stage, slot);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  template <bool STEADY, int H, bool IS_B, int Q, int... R, int... P>
  __device__ __forceinline__ void mfma_and_company(const vec (&aC)[MF], const vec (&bC)[NF], vec (&aN)[MF], vec (&bN)[NF], unsigned sa, unsigned sb, const T* base,
                                                   unsigned dst, int stage, unsigned slot, bool more, std::integer_sequence<int, R...>, std::integer_sequence<int, P...>)
  {
    constexpr int nf = Q % NF, mf = Q / NF;
    mfma_16x16x32<T>(acc[nf][mf], bC[nf], aC[mf]);
    (read_at<H, Q, R>(sa, sb, aN, bN), ...);
    (load_at<STEADY, IS_B, Q, P>(base, dst, stage, slot, more), ...);
  }
  // One k step: the MFMAs of fragments (aC, bC); meanwhile (aN, bN) receive k step H of the stage at (sa, sb) and the B (IS_B) or
  // A tile of stage `stage` is requested into `slot` (STEADY: it exists and is full; otherwise if `more`).
  template <bool STEADY, int H, bool IS_B, int... Q>
  __device__ __forceinline__ void k_step(const vec (&aC)[MF], const vec (&bC)[NF], vec (&aN)[MF], vec (&bN)[NF], unsigned sa, unsigned sb, int stage, unsigned slot,
                                         bool more, std::integer_sequence<int, Q...>)
  {
    const T*       base = IS_B ? Bg + (size_t)stage * b_step : Ag + (size_t)stage * TC::BK;
    const unsigned dst  = lds_addr + slot + wave * 1024;
    (mfma_and_company<STEADY, H, IS_B, Q>(aC, bC, aN, bN, sa, sb, base, dst, stage, slot, more, std::make_integer_sequence<int, TC::READS>(),
                                          std::make_integer_sequence<int, 2 * (IS_B ? TC::B_LOADS : TC::A_LOADS)>()),
     ...);
    __builtin_amdgcn_sched_barrier(0);
  }
};

// The kernel's body for tile `tile_index` of the tiles_m x tiles_n tiles of the column range that starts at n_base (0 and
// the whole matrix for the plain kernel); lds: the workgroup's rings.
// STAMP: the phase-accounting build -- clock readings at five points of every wave, stored to `stamps` at the end.
// SPLIT: the workgroup takes share `sp` of `S` of the K stages (pitch = the matrices' K, K = its own range) and stores its partial
// sums to plane sp of `planes` (fp16_splitk_reduce_kernel) instead of C.
template <typename T, int BM, int BN, int WM, int WN, int DA, int DB, bool B_NK, bool STAMP = false, bool SPLIT = false>
__device__ __forceinline__ void fp16_gemm_body(const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C, int M, int N, int pitch, int tiles_m,
                                               int tiles_n, char LLMMM_LDS* lds, int tile_index, int n_base, unsigned long long* stamps = nullptr,
                                               float* __restrict__ planes = nullptr, int sp = 0, int S = 1)
{
  typedef Fp16Tile<BM, BN, WM, WN, DA, DB> TC;
  typedef typename Vec16<T>::vec           vec;
  constexpr int                            MF = TC::MF, NF = TC::NF;
  PhaseClock                               ph[STAMP ? PHASE_POINTS : 1];
  unsigned long long                       wait_cycles = 0, load_wait_cycles = 0;  // STAMP: shader cycles in the K loop's waits; of which for the loads
  if constexpr (STAMP) ph[0] = phase_clock();

  const int tid  = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm   = wave % TC::WAVES_M;
  const int wn   = wave / TC::WAVES_M;
  int       tm, tn;
  tile_coords(tile_index, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = n_base + tn * BN;

  const int stages = (pitch + TC::BK - 1) / TC::BK, first = SPLIT ? sp * stages / S : 0;  // whole stages: a share ends on a multiple of BK or with K
  const int K      = SPLIT ? min(pitch, (sp + 1) * stages / S * TC::BK) - first * TC::BK : pitch;

  Fp16Wave<T, BM, BN, WM, WN, DA, DB, B_NK> w;
  w.K = K, w.wave = wave, w.lane = lane, w.lds = lds, w.lds_addr = (unsigned)(size_t)lds;
  w.Ag     = A + (size_t)m0 * pitch;
  w.Bg     = B_NK ? B + (size_t)n0 * pitch : B + n0;
  w.b_step = B_NK ? (size_t)TC::BK : (size_t)TC::BK * N;
  if constexpr (SPLIT) w.Ag += (size_t)first * TC::BK, w.Bg += (size_t)first * w.b_step;
  // ---- loader: lane -> what the 16 bytes at (1 KB load base + 16*lane) must hold.  (The byte offsets fit 32 bits: BM rows of
  // A or BN of Bt are part of matrices below 2^31 elements, and so are the k rows below K.)
  {
    const int r = wave * 8 + (lane >> 3);           // tile row of the first load; the others lie ROWS_PER_LOAD apart
    const int c = (lane & 7) ^ k128_swz(r);         // logical chunk placed at physical chunk lane%8
    w.a_k       = c * 8;
#pragma unroll
    for (int i = 0; i < TC::A_LOADS; ++i) w.a_off[i] = ((unsigned)(r + i * TC::ROWS_PER_LOAD) * (unsigned)pitch + c * 8) * 2u;
#pragma unroll
    for (int i = 0; i < TC::B_LOADS; ++i) {
      if constexpr (B_NK) {
        w.b_off[i] = ((unsigned)(r + i * TC::ROWS_PER_LOAD) * (unsigned)pitch + c * 8) * 2u;
        w.b_k[i]   = c * 8;
      }
      else {
        const int k     = (wave + i * TC::NW) * TC::B_KROWS_PER_GRP + (lane * 16) / TC::B_ROW;
        const int pbyte = (lane * 16) % TC::B_ROW;
        const int ch    = (pbyte >> 5) ^ kn_swz<BN>(k);  // logical 32-byte chunk stored at physical chunk pbyte/32
        w.b_off[i]      = ((unsigned)k * (unsigned)N + ((ch << 5) + (pbyte & 31)) / 2) * 2u;
        w.b_k[i]        = k;
      }
    }
  }
  // ---- operand reads.  lane = (g = lane/16, i = lane%16): row i of a 16-row fragment, k = 8g .. 8g+7
  const int g  = lane >> 4;
  const int li = lane & 15;
  w.a_rd       = k128_offset(wm * WM + li, g);
  if constexpr (B_NK)
    w.b_rd[0] = k128_offset(wn * WN + li, g);
  else {
    // transposing read: inside the 16-lane block, lane j supplies the 8 bytes (4 columns) j%4 of k row 8g + j/4
    const int k = 8 * g + (li >> 2);
#pragma unroll
    for (int nf = 0; nf < NF; ++nf) w.b_rd[nf] = k * TC::B_ROW + (((wn * NF + nf) ^ kn_swz<BN>(k)) << 5) + (li & 3) * 8;
  }
#pragma unroll
  for (int nf = 0; nf < NF; ++nf)
#pragma unroll
    for (int mf = 0; mf < MF; ++mf) w.acc[nf][mf] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int KS = (K + TC::BK - 1) / TC::BK, full_stages = K / TC::BK;
  const int KT = (K + 31) / 32;  // k steps

  vec aX[MF], aY[MF], bX[NF], bY[NF];  // fragments of a stage's first / second k step
  constexpr auto LA = std::make_integer_sequence<int, TC::A_LOADS>();
  constexpr auto LB = std::make_integer_sequence<int, TC::B_LOADS>();
  constexpr auto SQ = std::make_integer_sequence<int, TC::MFMAS>();
  // prologue: A_0 B_0 A_1 B_1 .. in flight, all of the rings but the last A stage, which the K loop requests first
#pragma unroll
  for (int u = 0; u < (DA > DB ? DA : DB); ++u) {
    if (u < DA - 1 && u < KS) w.load_a_tile(u, u * TC::A_BYTES, LA);
    if (u < DB && u < KS) w.load_b_tile(u, TC::B_RING + u * TC::B_BYTES, LB);
  }
  if (full_stages >= (DA - 1 > DB ? DA - 1 : DB))
    wait_vmcnt<TC::PROLOGUE>();
  else
    wait_vmcnt<0>();  // fewer or cut stages: the counts do not hold
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if constexpr (STAMP) ph[1] = phase_clock();
  w.template read_all<0>(0u, TC::B_RING, aX, bX, std::make_integer_sequence<int, TC::READS>());

  unsigned ra = 0, rb = TC::B_RING;             // LDS offsets of stage s in the two rings
  unsigned ra_prev = (DA - 1) * TC::A_BYTES;    // of stage s - 1 in the A ring: where A of stage s + DA - 1 goes
  int      s = 0;
#define LLMMM_STAGE(STEADY)                                                                                                             \
  {                                                                                                                                     \
    w.template k_step<STEADY, 1, false>(aX, bX, aY, bY, ra, rb, s + DA - 1, ra_prev, s + DA - 1 < KS, SQ);                              \
    const unsigned ra_next = ra + TC::A_BYTES == TC::B_RING ? 0u : ra + TC::A_BYTES;                                                    \
    const unsigned rb_next = rb + TC::B_BYTES == TC::LDS ? (unsigned)TC::B_RING : rb + TC::B_BYTES;                                     \
    unsigned long long tw_ = 0;                                                                                                         \
    if constexpr (STAMP) tw_ = __builtin_amdgcn_s_memtime();                                                                            \
    if constexpr (STEADY)                                                                                                               \
      wait_vmcnt<TC::IN_FLIGHT>(); /* stage s + 1 has landed; this wave's reads of stage s are back (lgkmcnt 0) */                      \
    else                                                                                                                                \
      wait_vmcnt<0>();                                                                                                                  \
    if constexpr (STAMP) load_wait_cycles += __builtin_amdgcn_s_memtime() - tw_;                                                        \
    __builtin_amdgcn_s_barrier();                                                                                                       \
    asm volatile("" ::: "memory"); /* no LDS read in front of the barrier */                                                            \
    if constexpr (STAMP) wait_cycles += __builtin_amdgcn_s_memtime() - tw_;                                                             \
    __builtin_amdgcn_sched_barrier(0);                                                                                                  \
    w.template k_step<STEADY, 0, true>(aY, bY, aX, bX, ra_next, rb_next, s + DB, rb, s + DB < KS, SQ);                                  \
    ra_prev = ra, ra = ra_next, rb = rb_next;                                                                                           \
  }
#pragma clang loop unroll(disable)
  for (; s + TC::AHEAD < full_stages; ++s) LLMMM_STAGE(true)
#pragma clang loop unroll(disable)
  for (; 2 * s + 1 < KT; ++s) LLMMM_STAGE(false)  // the fragments read behind the last stage are stale and not used
  if (2 * s < KT) w.template k_step<false, 1, false>(aX, bX, aY, bY, ra, rb, 0, 0u, false, SQ);  // K ends with a stage's first k step
#undef LLMMM_STAGE
  // the last MFMAs' results: wait states, then a use of every accumulator that nothing can be moved in front of
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int nf = 0; nf < NF; ++nf)
#pragma unroll
    for (int mf = 0; mf < MF; ++mf) asm volatile("" : "+a"(w.acc[nf][mf]));
  if constexpr (SPLIT) {
    // a plane is a row of 1 KB blocks, one per 16 x 16 fragment, in the accumulators' own lane order: every store is one linear
    // kilobyte, whatever the tile, and the reduce kernel finds 8 rows x 16 bytes of a fragment in one cache line
    float* plane = planes + (size_t)sp * M * N;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (nothing is left in flight; the compiler counts its own stores from here)
#pragma unroll
    for (int mf = 0; mf < MF; ++mf)
#pragma unroll
      for (int nf = 0; nf < NF; ++nf)
        *(f32x4*)(plane + ((size_t)((m0 + wm * WM) / 16 + mf) * (N / 16) + (n0 + wn * WN) / 16 + nf) * 256 + lane * 4) = w.acc[nf][mf];
    return;
  }
  if constexpr (STAMP) ph[2] = phase_clock();
  __builtin_amdgcn_s_barrier();  // every wave is through with the operands: the rings are free
  asm volatile("" ::: "memory");

  // ---- epilogue: lane (g, li) holds rows m = .. + mf*16 + li, columns nf*16 + 4g + r.
  // Stored straight from this layout, one instruction would write 8 bytes to each of 16 rows, and the memory pipeline pays
  // per row segment.  Instead every wave lays its result out row-major (16-byte chunks XOR-ed with the row so that the
  // ds_read_b128 below is conflict-free) in a private piece of the rings and stores whole rows, 16 bytes per lane.
  {
    typedef T             tx4 __attribute__((ext_vector_type(4)));
    char LLMMM_LDS* const stg = lds + wave * (WM * WN * 2);
    constexpr int         CPR = WN / 8;  // 16-byte chunks per row
#pragma unroll
    for (int mf = 0; mf < MF; ++mf) {
      const int r = mf * 16 + li;
#pragma unroll
      for (int nf = 0; nf < NF; ++nf) {
        const f32x4 v = w.acc[nf][mf];
        tx4         o;
        o[0] = (T)v[0];
        o[1] = (T)v[1];
        o[2] = (T)v[2];
        o[3] = (T)v[3];
        *(tx4 LLMMM_LDS*)(stg + r * (WN * 2) + (((nf * 2 + (g >> 1)) ^ (r & (CPR - 1))) << 4) + 8 * (g & 1)) = o;
      }
    }
    T* cbase = C + (size_t)(m0 + wm * WM) * N + n0 + wn * WN;
#pragma unroll
    for (int j = 0; j < WM * CPR / 64; ++j) {
      const int   r = (64 / CPR) * j + lane / CPR, ch = lane % CPR;
      const i32x4 v = *(const i32x4 LLMMM_LDS*)(stg + r * (WN * 2) + ((ch ^ (r & (CPR - 1))) << 4));
      *(i32x4*)(cbase + (size_t)r * N + ch * 8) = v;
    }
  }
  if constexpr (STAMP) {
    ph[3] = phase_clock();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stores are acknowledged
    ph[4] = phase_clock();
    static_assert(!STAMP || TC::NW == 4, "two records per wave");
    if (lane == 0)
      for (int half = 0; half < 2; ++half) {  // eight records per workgroup, one wave per SIMD: every wave fills two
        unsigned long long* o = stamps + ((size_t)tile_index * 8 + wave + half * 4) * PHASE_RECORD;
#pragma unroll
        for (int p = 0; p < PHASE_POINTS; ++p) o[2 * p] = ph[p].real, o[2 * p + 1] = ph[p].cycles;
        o[PHASE_STAMPS] = wait_cycles, o[PHASE_STAMPS + 1] = load_wait_cycles;
      }
  }
}

template <typename T>
__global__ void __launch_bounds__(256)
fp16_gemm_phases_kernel(const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C, int M, int N, int K, int tiles_m, int tiles_n,
                        unsigned long long* stamps)
{
  __shared__ __attribute__((aligned(1024))) char lds[Fp16Tile<256, 256, 128, 128, 3, 2>::LDS];
  fp16_gemm_body<T, 256, 256, 128, 128, 3, 2, false, true>(A, B, C, M, N, K, tiles_m, tiles_n, (char LLMMM_LDS*)lds, blockIdx.x, 0, stamps);
}

template <typename T, int BM, int BN, int WM, int WN, int DA, int DB, bool B_NK>
__global__ void __launch_bounds__((BM / WM) * (BN / WN) * 64)
fp16_gemm_kernel(const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C, int M, int N, int K, int tiles_m, int tiles_n)
{
  __shared__ __attribute__((aligned(1024))) char lds[Fp16Tile<BM, BN, WM, WN, DA, DB>::LDS];
  fp16_gemm_body<T, BM, BN, WM, WN, DA, DB, B_NK>(A, B, C, M, N, K, tiles_m, tiles_n, (char LLMMM_LDS*)lds, blockIdx.x, 0);
}

// split-K: S workgroups per tile, each over its share of the K stages, and a second kernel that adds their planes (where it pays:
// heuristic_split_fp16 in capi.cpp).  What bounds it besides the product is the planes' way through memory, so both kernels deal the
// tiles to the XCDs alike -- XCD x (workgroup ids = x mod 8) owns a contiguous run of tiles with all S shares of each -- and the reduce
// kernel finds the planes in its own L2.
// Workgroup wg of 8 * ceil(tiles / 8) * per: item 0 .. tiles * per - 1 of XCD-contiguous tiles with `per` items each; false: none.
__device__ __forceinline__ bool split_item(int wg, int tiles, int per, int& tile_id, int& item)
{
  const int x = wg & 7, j = wg >> 3, mine = (tiles >> 3) + (x < (tiles & 7) ? 1 : 0);
  if (j >= mine * per) return false;
  const int t = j % mine;
  item        = j / mine;
  tile_id     = t * 8 + x;  // tile_coords takes the ids = x mod 8 for XCD x's run
  return true;
}

template <typename T, int BM, int BN, int WM, int WN, int DA, int DB, bool B_NK>
__global__ void __launch_bounds__((BM / WM) * (BN / WN) * 64)
fp16_split_gemm_kernel(const T* __restrict__ A, const T* __restrict__ B, float* __restrict__ planes, int M, int N, int K, int tiles_m, int tiles_n, int S)
{
  __shared__ __attribute__((aligned(1024))) char lds[Fp16Tile<BM, BN, WM, WN, DA, DB>::LDS];
  int tile_id, sp;
  if (!split_item(blockIdx.x, tiles_m * tiles_n, S, tile_id, sp)) return;
  fp16_gemm_body<T, BM, BN, WM, WN, DA, DB, B_NK, false, true>(A, B, nullptr, M, N, K, tiles_m, tiles_n, (char LLMMM_LDS*)lds, tile_id, 0, nullptr, planes, sp, S);
}

// Adds the S planes in order and rounds to T.  A wave takes 8 rows x 64 columns: lane l row l / 8, columns 8 (l % 8) .. +7, i.e. two
// 16-byte pieces of a fragment whose eight rows lie in one cache line, and its stores are eight whole 128-byte lines.
// All loads of a lane go out together (a launch of this size is one latency long): S is a constant.
template <typename T, int S, int BM, int BN>
__global__ void __launch_bounds__(256)
fp16_splitk_reduce_kernel(const float* __restrict__ planes, T* __restrict__ C, int M, int N, int tiles_m, int tiles_n)
{
  constexpr int UNITS = BM * BN / 2048;  // workgroups per tile
  int           tile_id, unit, tm, tn;
  if (!split_item(blockIdx.x, tiles_m * tiles_n, UNITS, tile_id, unit)) return;
  tile_coords(tile_id, tiles_m, tiles_n, tm, tn);
  const int    lane = threadIdx.x & 63, w = unit * 4 + (threadIdx.x >> 6);
  const int    row = tm * BM + w / (BN / 64) * 8 + (lane >> 3), col = tn * BN + w % (BN / 64) * 64 + (lane & 7) * 8;
  const float* p = planes + ((size_t)(row >> 4) * (N >> 4) + (col >> 4)) * 256 + ((col & 8) * 4 + (row & 15)) * 4;
  f32x4        v[S][2];
#pragma unroll
  for (int s = 0; s < S; ++s) v[s][0] = *(const f32x4*)(p + (size_t)s * M * N), v[s][1] = *(const f32x4*)(p + (size_t)s * M * N + 64);
  typedef T tx8 __attribute__((ext_vector_type(8)));
  tx8       o;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    f32x4 t = v[0][h];
#pragma unroll
    for (int s = 1; s < S; ++s) t += v[s][h];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[4 * h + e] = (T)t[e];
  }
  *(tx8*)(C + (size_t)row * N + col) = o;
}

// 256 x 256 tiles whose number is not a multiple of the 256 CUs end with a round that keeps part of the chip busy for a
// whole tile's time (2048 x 19456: 608 tiles, the third round 96 of them).  One launch of both shapes: the columns that fill
// whole rounds go to 256 x 256 tiles (workgroups 0 .. tiles_m_big * cols_big - 1, dispatched first), the remaining columns
// to twice as many 128 x 256 tiles of four 64 x 128 waves -- the same K loop, half the rows per wave, the same results.
template <typename T, bool B_NK>
__global__ void __launch_bounds__(256)
fp16_gemm_hybrid_kernel(const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C, int M, int N, int K, int tiles_m_big, int cols_big,
                        int cols_small)
{
  static_assert(Fp16Tile<128, 256, 64, 128, 3, 3>::LDS <= Fp16Tile<256, 256, 128, 128, 3, 2>::LDS, "the small tiles fit the large tiles' rings");
  __shared__ __attribute__((aligned(1024))) char lds[Fp16Tile<256, 256, 128, 128, 3, 2>::LDS];
  const int n_big = tiles_m_big * cols_big;
  if ((int)blockIdx.x < n_big)
    fp16_gemm_body<T, 256, 256, 128, 128, 3, 2, B_NK>(A, B, C, M, N, K, tiles_m_big, cols_big, (char LLMMM_LDS*)lds, blockIdx.x, 0);
  else
    fp16_gemm_body<T, 128, 256, 64, 128, 3, 3, B_NK>(A, B, C, M, N, K, 2 * tiles_m_big, cols_small, (char LLMMM_LDS*)lds, (int)blockIdx.x - n_big,
                                                     cols_big * 256);
}

// --------------------------------------------------------------------------------------------- host
template <typename T, int BM, int BN, int WM, int WN, int DA, int DB, bool B_NK>
static hipError_t launch_fp16(const void* A, const void* B, void* C, int M, int N, int K, hipStream_t stream)
{
  const int tiles_m = M / BM, tiles_n = N / BN;
  if constexpr (BM == 256 && BN == 256) {
    // more than one round of the chip with a partly filled last one: whole rounds in 256 x 256 tiles, the remaining
    // columns in 128 x 256 tiles, if those fit one round (fp16_gemm_hybrid_kernel)
    const int  cus   = num_cus();
    const long tiles = (long)tiles_m * tiles_n, full = tiles / cus * cus;
    if (tiles > cus && tiles_m > 1 && full % tiles_m == 0) {
      const int cols_big = (int)(full / tiles_m), cols_small = tiles_n - cols_big;
      if (cols_small > 0 && (long)cols_small * tiles_m * 2 <= cus) {
        hipLaunchKernelGGL((fp16_gemm_hybrid_kernel<T, B_NK>), dim3(tiles_m * cols_big + 2 * tiles_m * cols_small), dim3(256), 0, stream, (const T*)A,
                           (const T*)B, (T*)C, M, N, K, tiles_m, cols_big, cols_small);
        return hipGetLastError();
      }
    }
  }
  hipLaunchKernelGGL((fp16_gemm_kernel<T, BM, BN, WM, WN, DA, DB, B_NK>), dim3(tiles_m * tiles_n), dim3(Fp16Tile<BM, BN, WM, WN, DA, DB>::NT), 0, stream,
                     (const T*)A, (const T*)B, (T*)C, M, N, K, tiles_m, tiles_n);
  return hipGetLastError();
}

template <typename T, int BM, int BN, int WM, int WN, int DA, int DB>
static hipError_t launch_fp16_split(bool b_nk, const void* A, const void* B, void* C, int M, int N, int K, int S, float* planes, hipStream_t stream)
{
  const int  tiles_m = M / BM, tiles_n = N / BN, runs = (tiles_m * tiles_n + 7) / 8 * 8;
  const dim3 grid(runs * S), block(Fp16Tile<BM, BN, WM, WN, DA, DB>::NT), reduce_grid(runs * (BM * BN / 2048));
  if (b_nk)
    hipLaunchKernelGGL((fp16_split_gemm_kernel<T, BM, BN, WM, WN, DA, DB, true>), grid, block, 0, stream, (const T*)A, (const T*)B, planes, M, N, K, tiles_m, tiles_n, S);
  else
    hipLaunchKernelGGL((fp16_split_gemm_kernel<T, BM, BN, WM, WN, DA, DB, false>), grid, block, 0, stream, (const T*)A, (const T*)B, planes, M, N, K, tiles_m, tiles_n, S);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  switch (S) {
#define LLMMM_GO(n) \
  case n: hipLaunchKernelGGL((fp16_splitk_reduce_kernel<T, n, BM, BN>), reduce_grid, dim3(256), 0, stream, planes, (T*)C, M, N, tiles_m, tiles_n); break
    LLMMM_GO(2);
    LLMMM_GO(3);
    LLMMM_GO(4);
    LLMMM_GO(5);
    LLMMM_GO(6);
    LLMMM_GO(7);
    LLMMM_GO(8);
#undef LLMMM_GO
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <typename T>
static hipError_t fp16_split(bool b_nk, int tile, const void* A, const void* B, void* C, int M, int N, int K, int S, float* planes, hipStream_t stream)
{
  switch (tile) {
    case LLMMM_TILE_128x128: return launch_fp16_split<T, 128, 128, 64, 64, 5, 5>(b_nk, A, B, C, M, N, K, S, planes, stream);
    case LLMMM_TILE_64x128: return launch_fp16_split<T, 64, 128, 32, 64, 3, 3>(b_nk, A, B, C, M, N, K, S, planes, stream);
    case LLMMM_TILE_64x64: return launch_fp16_split<T, 64, 64, 32, 32, 4, 4>(b_nk, A, B, C, M, N, K, S, planes, stream);
    default: return hipErrorInvalidValue;
  }
}

// K in S shares through fp32 planes (S * M * N floats), 2 <= S <= FP16_MAX_SPLIT, S <= the number of 64-wide K stages.
hipError_t fp16_gemm_split_launch(int dtype, int b_layout, int tile, const void* A, const void* B, void* C, int M, int N, int K, int S, float* planes,
                                  hipStream_t stream)
{
  if (S < 2 || S > FP16_MAX_SPLIT || S > (K + 63) / 64 || !planes || M % 128 || N % 128) return hipErrorInvalidValue;
  return dtype == 0 ? fp16_split<_Float16>(b_layout != 0, tile, A, B, C, M, N, K, S, planes, stream)
                    : fp16_split<__bf16>(b_layout != 0, tile, A, B, C, M, N, K, S, planes, stream);
}

// The rings of the 128 x 128 tile.  Up to one tile per CU and from K = 1024 on they take the whole LDS (1920 x 1536 x 5312, 180 tiles:
// 38 us deep, 44 us shallow; at K = 1024 the two are even).  Beyond one tile two workgroups share a CU (3968 x 2944 x 576, 713 tiles:
// 20.6 us shallow, 24.7 us deep), and a shorter K is over before the deep rings have paid for their start (1664 x 1408, us, shallow /
// deep: K = 512 7.8 / 8.5, 640 8.7 / 9.3, 800 10.3 / 10.7).
bool fp16_deep(int M, int N, int K) { return (long)(M / 128) * (N / 128) <= num_cus() && K >= 1024; }

template <typename T, bool B_NK>
static hipError_t dispatch_fp16(int tile, const void* A, const void* B, void* C, int M, int N, int K, hipStream_t stream)
{
  switch (tile) {
    case LLMMM_TILE_256x256: return launch_fp16<T, 256, 256, 128, 128, 3, 2, B_NK>(A, B, C, M, N, K, stream);
    // half tiles of eight 64 x 64 waves, two per SIMD: ahead of four 128 x 64 waves by 1-3 % (2048 x 2560 x 9728: 119 / 123 us)
    case LLMMM_TILE_128x256: return launch_fp16<T, 128, 256, 64, 64, 3, 3, B_NK>(A, B, C, M, N, K, stream);
    case LLMMM_TILE_256x128: return launch_fp16<T, 256, 128, 64, 64, 3, 3, B_NK>(A, B, C, M, N, K, stream);
    case LLMMM_TILE_128x128:
      return fp16_deep(M, N, K) ? launch_fp16<T, 128, 128, 64, 64, 5, 5, B_NK>(A, B, C, M, N, K, stream)
                                                      : launch_fp16<T, 128, 128, 64, 64, 3, 2, B_NK>(A, B, C, M, N, K, stream);
    case LLMMM_TILE_64x128: return launch_fp16<T, 64, 128, 32, 64, 3, 3, B_NK>(A, B, C, M, N, K, stream);
    case LLMMM_TILE_64x64: return launch_fp16<T, 64, 64, 32, 32, 4, 4, B_NK>(A, B, C, M, N, K, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t fp16_gemm_phases_launch(int dtype, const void* A, const void* B, void* C, int M, int N, int K, unsigned long long* stamps, hipStream_t stream)
{
  if (M % 256 || N % 256 || K % 32 || !stamps) return hipErrorInvalidValue;
  const int tiles_m = M / 256, tiles_n = N / 256;
  if (dtype == 0)
    hipLaunchKernelGGL((fp16_gemm_phases_kernel<_Float16>), dim3(tiles_m * tiles_n), dim3(256), 0, stream, (const _Float16*)A, (const _Float16*)B, (_Float16*)C, M,
                       N, K, tiles_m, tiles_n, stamps);
  else
    hipLaunchKernelGGL((fp16_gemm_phases_kernel<__bf16>), dim3(tiles_m * tiles_n), dim3(256), 0, stream, (const __bf16*)A, (const __bf16*)B, (__bf16*)C, M, N, K,
                       tiles_m, tiles_n, stamps);
  return hipGetLastError();
}

hipError_t fp16_gemm_launch(int dtype, int b_layout, int tile, const void* A, const void* B, void* C, int M, int N, int K,
                            hipStream_t stream)
{
  if (dtype == 0)
    return b_layout ? dispatch_fp16<_Float16, true>(tile, A, B, C, M, N, K, stream)
                    : dispatch_fp16<_Float16, false>(tile, A, B, C, M, N, K, stream);
  return b_layout ? dispatch_fp16<__bf16, true>(tile, A, B, C, M, N, K, stream)
                  : dispatch_fp16<__bf16, false>(tile, A, B, C, M, N, K, stream);
}

}  // namespace llmmm
