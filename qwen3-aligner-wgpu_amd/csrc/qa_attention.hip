// qa_attention.hip -- causal GQA prefill attention for gfx950 (hd = 128).
//
// Replaces the reference's prefill attention chain (src/decoder.rs:1346-1600:
// repeat_kv, a scores GEMM per key slab, softmax, the P.V GEMM and the slab
// merge; WGSL src/shaders.rs:2079-2505) with one flash-style kernel; the
// arithmetic it must match is the CPU twin, src/cpu_decoder.rs:324-411: f32
// scores q.k / sqrt(hd), softmax in f32, out = round(sum_t p_t v_t).
//
// Block = one kv head x a tile of RG x 32 query rows x its REP q heads; waves:
// NS key splits x REP heads x RG row groups of 32.  Split s takes the key
// blocks kb = s, s + NS, ... (64 keys each) below the tile's causal bound, so
// the long rows' key range is processed by NS wave groups at once; the partial
// results merge through LDS at the end in a fixed order.  Two shapes of eight
// waves (REP = 2):
//  * RG = 2, NS = 2: each K / V tile feeds 64 rows.  Once the grid is a few
//    blocks per CU, the stream and the phases per FLOP decide (4334 rows: 127
//    us against 138 with the other shape).
//  * RG = 1, NS = 4: twice the blocks and half the steps in a row, for grids
//    that leave CUs idle, where the length of the longest block's chain of
//    steps decides (a phase is ~1 us however few blocks run).  Its four
//    groups hold one K and one V tile each (NB = 1: 128 KB), refilled during
//    the VALU phase, longer than the L2 takes to answer; with two of each of
//    half the keys a step's fixed costs double (1024 rows: 20.1 us).
//    Measured, f16, repeated launches, RG = 2 -> RG = 1: 61 rows 7.7 -> 6.7 us,
//    323 rows 12.9 -> 10.4, 1024 rows 24.5 -> 16.9, 2048 rows (256 blocks of 64)
//    41.9 -> 36.3, 2200 rows (280) 46.0 -> 48.3; 771 rows from position 1536 with
//    16-bit probabilities 38.6 -> 24.4.  Hence the line at one block of 64 rows
//    per CU.
//    Behind a long past the blocks are all about equally long, and 257 to 512
//    of 32 rows take two full rounds: 8 kv heads, 1200 rows from position
//    1000 43.0 -> 40.3 us, 1500 51.1 -> 50.6, 2000 58.8 -> 60.9, 4000 91 ->
//    100, 8000 154 -> 182; 2048 rows from 2000 88 -> 84, 4000 133 -> 133, 8000
//    223 -> 229.  Hence the 64-row shape there from 1.5 times the rows on.
//
// Per key block, per wave (32 query rows):
//  * S = K . Q^T on v_mfma_f32_32x32x16 (A = 32 keys x 16 d from LDS, B = the
//    wave's Q fragments, kept in registers for the whole kernel): the lane
//    holds one query row and 16 of each 32-key tile's scores.
//  * online softmax in the log2 domain (v_exp_f32): the row max over the
//    lane's values plus its partner lane (lane ^ 32, same row); the running max
//    moves only when a block's max exceeds it by more than 2^8, and then the
//    running output and sum are rescaled by exp2(m_old - m_new); each lane
//    keeps its half of the row sum until the end.
//  * O^T += V^T . P^T: P goes from the score registers straight into the
//    MFMA's B operand.  The reference's GPU path rounds its probabilities to
//    the 16-bit format before its P.V GEMM (PS = 1 here), which costs up to
//    2^-11 (f16) / 2^-8 (bf16) relative per weight; by default (PS = 2) the
//    rounding residue goes through a second MFMA as a second 16-bit term, so
//    the product carries ~2^-22 / 2^-16 and the result tracks the f32 CPU
//    path.  f16 probabilities are formed scaled by 2^7 so that they stay in
//    the normal range (the scale cancels in the final division).  A lane half holds
//    keys {16j+4h..+3, 16j+8+4h..+3} of slice j, so the transposed V cache
//    stores each aligned group of 16 keys in the order 0-3, 8-11, 4-7, 12-15
//    (bits 2 and 3 of the key swapped): one 16-byte read per V fragment.
//  * K and V tiles stream L2 -> LDS with buffer_load ... lds, NB buffers of
//    each per split group; chunks are XOR-swizzled per row so the 32-row fragment
//    reads hit distinct banks.
#include <type_traits>

#include "qa_internal.h"

namespace qa {

#ifdef QA_PHASE_STAMPS
// Measurement build only (make stamps): every wave of an attention_kernel
// launch adds up s_memtime (shader clock) cycles by phase -- the prologue up
// to the phase loop, the MFMA phases (P.V + S issued), the VALU phases
// (softmax, DMA issue), the phases with no work of its own, the block
// barrier after each phase, the merge and output, and the DMA and LDS waits
// before each barrier -- and counts its MFMA and VALU phases.  Words per
// wave: those seven sums, the two counts.
constexpr int kAttnStampBlocks = 2048, kAttnStampWaves = 8, kAttnStampWords = 9;
__device__ unsigned long long attn_stamp_log[kAttnStampBlocks * kAttnStampWaves * kAttnStampWords];
#endif
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

#define QA_LDS __attribute__((address_space(3)))

constexpr uint32_t OOB = 0x80000000u;  // byte offset past every buffer's num_records
constexpr int HD = 128;  // head dim
constexpr int KB = 64;   // keys per step
constexpr float kLog2e = 1.44269504088896341f;
// The running row max is raised only when a block's max exceeds it by more
// than this (log2 units): probabilities then stay <= 2^kLazy and the output
// rescale runs once per such jump instead of once per block.
constexpr float kLazy = 8.f;

// Max / sum of a value over lane pairs (l, l ^ 32), on v_permlane32_swap: the
// two results hold the wave's lower and upper 32-lane halves exchanged in one
// of them, so a symmetric combination of both is the pair's result on every
// lane, identical on the two lanes of a pair.
__device__ __forceinline__ float pair_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pair_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int DT>
struct AFmt;
template <>
struct AFmt<QA_F16> {
  __device__ static __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  // two values, RNE, element a in the low half (v_cvt_pk_f16_f32)
  __device__ static __forceinline__ uint32_t pack2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, f16x2));
  }
  __device__ static __forceinline__ f32x2 unpack2(uint32_t h) {
    return __builtin_convertvector(__builtin_bit_cast(f16x2, h), f32x2);
  }
  // (a, b) minus their 16-bit roundings h (packed: a's in the low half), as
  // two 16-bit values.  Each difference is exact in f32 (a and h agree in
  // their leading bits), so v_fma_mix_f32 (-h) * 1 + a, which reads h
  // straight from its half of the packed word, gives the same bits as
  // widening h and subtracting, in one instruction instead of two.  a and b
  // are v_exp_f32 results, and the compiler puts no wait state ahead of an
  // asm statement; h = pack2(a, b) is a compiler instruction that reads both
  // and precedes these by its data dependency, so the transcendental's
  // one-instruction wait state has passed when they read a and b.
  __device__ static __forceinline__ uint32_t residue2(uint32_t h, float a, float b) {
    float d0, d1;
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(d0) : "v"(h), "v"(a));
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(d1) : "v"(h), "v"(b));
    return pack2(d0, d1);
  }
  // Probabilities are formed as p * 2^7; with the running max allowed to lag
  // the true one by up to 2^8 (kLazy) they stay <= 2^15, and the f16 range
  // keeps them normal down to p = 2^-21, so rounding them loses only relative
  // precision (below that, at most 2^-32 absolute).
  static constexpr float kPBias = 7.f;
};
template <>
struct AFmt<QA_BF16> {
  __device__ static __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  // two values, RNE (v_cvt_pk_bf16_f32): for finite values the reference's
  // (u + 0x7fff + ((u >> 16) & 1)) >> 16, src/shaders.rs:169-179
  __device__ static __forceinline__ uint32_t pack2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
  }
  __device__ static __forceinline__ f32x2 unpack2(uint32_t h) {
    return (f32x2){__uint_as_float(h << 16), __uint_as_float(h & 0xffff0000u)};
  }
  __device__ static __forceinline__ uint32_t residue2(uint32_t h, float a, float b) {
    const f32x2 hv = unpack2(h);
    return pack2(a - hv[0], b - hv[1]);
  }
  static constexpr float kPBias = 0.f;
};

// A value the caller knows to be equal in every lane, as a scalar register.
__device__ __forceinline__ int wave_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}
__device__ __forceinline__ void wait_lds() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xF | (0x3 << 14) | (0x7 << 4) | (0x0 << 8));
}
__device__ __forceinline__ void exec_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// LDS tile layouts.  K tile: 64 key rows x 256 B (16 chunks of 8 d); chunk c of
// row r at c ^ (r & 15).  V tile: 128 d rows x 128 B (8 chunks of 8 stored key
// positions); chunk c of row d at c ^ ((d >> 1) & 7).
__device__ __forceinline__ int kswz(int r) { return r & 15; }
__device__ __forceinline__ int vswz(int d) { return (d >> 1) & 7; }

// RG row groups of 32 query rows per block, NS key splits, NB buffers of each
// split's K and V tiles.
template <int DT, int REP, int PS, int RG, int NS, int NB>
__global__ void __launch_bounds__(NS * REP * RG * 64) attention_kernel(const AttnParams p) {
  constexpr int QT = 32 * RG;          // query rows per block
  constexpr int KT = KB / 32;          // 32-key score tiles per step
  constexpr int GW = REP * RG;         // waves per split group
  constexpr int VCH = KB / 8;          // 16-byte chunks per V tile row
  constexpr int VR = 64 / VCH;         // V tile rows per DMA instruction
  constexpr int KTILE = KB * HD * 2;
  constexpr int VTILE = HD * KB * 2;
  constexpr int KI = KB * HD * 2 / 1024 / GW;  // K DMA instructions per wave per block
  constexpr int VI = HD * KB * 2 / 1024 / GW;  // V DMA instructions per wave per block
  constexpr int LPS = KI + VI;
  static_assert(KI * GW * 4 == KB && VI * GW * VR == HD, "DMA row coverage");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[NS * NB * (KTILE + VTILE)];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int split = wave / GW, wg = wave % GW;
  const int hh = wg / RG, rg = wg % RG;
  // Phase offset (see the phases below): a SIMD runs waves w and w + 4, so the
  // upper half of the split groups runs one phase behind the lower half.
  const int off = split / (NS / 2);
  const int fr = lane & 31, fh = lane >> 5;
#ifdef QA_PHASE_STAMPS
  // s_memtime cycles by phase: prologue, MFMA, VALU, no work, barrier,
  // merge, DMA + LDS waits
  unsigned long long cyc[7] = {0, 0, 0, 0, 0, 0, 0}, nmma = 0, nvalu = 0;
  __builtin_amdgcn_sched_barrier(0);
  unsigned long long c_mark = __builtin_amdgcn_s_memtime();
  __builtin_amdgcn_sched_barrier(0);
#endif

  // Block b -> kv head b % nkvh, row tile T - 1 - b / nkvh: the longest key
  // ranges of every head are dispatched first, and with blocks dealt
  // round-robin over the 8 XCDs all blocks of a head land on one XCD (for
  // nkvh a multiple of 8), whose L2 then holds that head's K and V.
  const int T = (int)((p.rows + QT - 1) / QT);
  const int t = T - 1 - (int)(blockIdx.x / p.nkvh);
  const int kvh = (int)(blockIdx.x % p.nkvh);
  const int head = kvh * REP + hh;
  const int64_t row0 = (int64_t)t * QT;
  const int64_t kend = p.q0 + min(row0 + QT, p.rows);  // keys 0..kend-1 are visible
  const int nkb = (int)((kend + KB - 1) / KB);

  // ---- LDS: per split group, K slots 0/1 then V slots 0/1 ----
  unsigned char* gsm = smem + split * NB * (KTILE + VTILE);
  auto kslot = [&](int it) { return gsm + (it & (NB - 1)) * KTILE; };
  auto vslot = [&](int it) { return gsm + NB * KTILE + (it & (NB - 1)) * VTILE; };
  // this group's steps: key blocks split, split + NS, ... below nkb
  const int nst = (nkb - split + NS - 1) / NS;

  // ---- DMA (the group's GW waves share each tile) ----
  const uint16_t* kbase = p.k_cache + (int64_t)kvh * p.cap * HD;
  const uint16_t* vbase = p.v_cache + (int64_t)kvh * HD * p.cap;
  const __amdgpu_buffer_rsrc_t rsk = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(kbase), (short)0, (int)(p.cap * HD * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsv = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(vbase), (short)0, (int)(p.cap * HD * 2), 0x00020000);
  // K instruction j fills key rows 4 (GW j + wg) + lane / 16 and V instruction
  // j d rows VR (GW j + wg) + lane / VCH.  Over j the chunk swizzle of a lane's
  // V rows stays the same, and that of its K rows (row & 15) does for GW = 4
  // and alternates in bit 3 for GW = 2: an instruction's offset is the lane's
  // offset at j = 0 (that bit toggled) plus a wave-uniform amount, one add.
  // K rows at or past cap lie past the buffer's num_records and read as zeros;
  // a V column at or past cap (the last block, cap % KB != 0) would not, as it
  // lies inside the next d row, so those lanes get OOB.
  // (The lane offsets are recomputed at each refill, a few instructions, from
  // a copy of the lane index the compiler cannot hoist: kept live across the
  // loop they would push the kernel past its register budget.)
  auto lane_opaque = [&]() {
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  };
  static_assert(GW * 4 % 16 == 0 || GW * 4 % 16 == 8, "K chunk swizzle over j");
  static_assert(GW * VR % 16 == 0, "V chunk swizzle over j");
  auto issue_k = [&](int it) {
    unsigned char* sk = smem + wave_uniform((int)(kslot(it) - smem) + wg * 1024);
    const int l = lane_opaque(), rk = wg * 4 + (l >> 4);
    const uint32_t koff0 = (uint32_t)((rk * HD + (((l & 15) ^ kswz(rk)) << 3)) * 2);
    const uint32_t kb0 = (uint32_t)(split + NS * it) * (KB * HD * 2);
#pragma unroll
    for (int j = 0; j < KI; ++j) {
      const uint32_t flip = GW * 4 * j % 16 * 16;  // bit 3 of the chunk
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsk, (QA_LDS void*)(sk + j * GW * 1024), 16,
                                               (koff0 ^ flip) + kb0 + 4 * GW * j * HD * 2, 0, 0, 0);
    }
  };
  auto issue_v = [&](int it) {
    unsigned char* sv = smem + wave_uniform((int)(vslot(it) - smem) + wg * 1024);
    const int l = lane_opaque(), dv = wg * VR + l / VCH;
    const uint32_t cap2 = (uint32_t)p.cap * 2;
    const uint32_t col = (uint32_t)(((l % VCH) ^ vswz(dv)) << 3) + (uint32_t)(split + NS * it) * KB;
    const uint32_t voff0 = (uint32_t)dv * cap2 + col * 2;
    const bool vin = col < (uint32_t)p.cap;
#pragma unroll
    for (int j = 0; j < VI; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsv, (QA_LDS void*)(sv + j * GW * 1024), 16,
                                               vin ? voff0 + (uint32_t)(VR * GW * j) * cap2 : OOB, 0, 0, 0);
  };
  // Loads issued by refill(j), in the VALU phase of step j: K(j + NB) into K
  // slot j % NB (S(j) has read it) and V(j + NB - 1) (P.V of step j - 1 has
  // read its slot).  The MFMA phase of step i needs K(i) and V(i - 1), issued
  // by refill(i - NB): with NB = 2 refill(i - 1)'s loads may still be in
  // flight, with NB = 1 nothing.
  auto refill_count = [&](int j) {
    return NB == 1 ? 0 : (j + 2 < nst ? KI : 0) + (j + 1 < nst ? VI : 0);
  };
  auto wait_refill = [&](int c) {
    static_assert(KI == VI, "refill counts are 0, VI or KI + VI");
    if (c == LPS)
      wait_vmcnt<LPS>();
    else if (c == VI)
      wait_vmcnt<VI>();
    else
      wait_vmcnt<0>();
  };

  // ---- this wave's 32 query rows, as MFMA B fragments (8 slices of 16 d) ----
  const int64_t qrow = row0 + rg * 32 + fr;
  // Lanes past the last row repeat it, position and all, and store nothing.  A
  // position of their own would let them see cache entries that this call
  // never wrote, and a large score there moves the running max of the
  // wave's valid rows too (the ballot in softmax).
  const int64_t lrow = min(qrow, p.rows - 1);
  u32x4 qf[8];
  {
    const uint16_t* q = p.q + ((int64_t)head * p.rows + lrow) * HD + fh * 8;
#pragma unroll
    for (int s = 0; s < 8; ++s) qf[s] = *reinterpret_cast<const u32x4*>(q + s * 16);
  }
  const int pos = (int)(p.q0 + lrow);                   // this lane's query position
  const int wpos0 = (int)(p.q0 + row0 + rg * 32);       // the wave's first position
  const float sc = p.scale * kLog2e;

  f32x16 o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = f32x16{0};
  float m_run = -INFINITY, l_run = 0.f;
  f32x16 s[KT] = {};
  u32x4 pf[2 * KT], pl[2 * KT];

  // MFMA phase of step it: P.V of step it - 1 (V slot (it - 1) & 1) and
  // S = K.Q^T of step it (K slot it & 1).  Per 16-deep slice st: the P.V
  // MFMAs of the value terms, the two S MFMAs, then the residue terms, so the
  // two MFMAs on one O accumulator are never adjacent; the fragments of
  // slice st + 1 are read from LDS while slice st multiplies (the schedule
  // groups below keep the compiler from sinking the reads next to their use).
  auto mma = [&](auto pv_tag, auto s_tag, int it) {
    constexpr bool PV = decltype(pv_tag)::value, SQ = decltype(s_tag)::value;
    // A fragment row's chunk 2 i + fh sits at ((2 i + fh) ^ swizzle) << 4, so
    // over i the address is the one of i = 0 with bits 5.. toggled.  The lane's
    // part is formed here from an opaque copy of the lane index: hoisted out of
    // the loop, the addresses would spill.
    const int l = lane_opaque(), r = l & 31, h = l >> 5;
    const int ka = (int)(kslot(it) - smem) + r * 256 + ((h ^ kswz(r)) << 4);
    const int va = (int)(vslot(it - 1) - smem) + r * (KB * 2) + ((h ^ vswz(r)) << 4);
    if constexpr (SQ) {
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) s[kt] = f32x16{0};
    }
    auto rd_v = [&](int st, u32x4* vf) {
#pragma unroll
      for (int u = 0; u < KT; ++u) {
        const int q = KT * st + u, dt = q & 3, j = q >> 2;
        vf[u] = *reinterpret_cast<const u32x4*>(smem + (va ^ (j << 5)) + dt * 32 * KB * 2);
      }
    };
    auto rd_k = [&](int st, u32x4* kf) {
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
        kf[kt] = *reinterpret_cast<const u32x4*>(smem + (ka ^ (st << 5)) + kt * 32 * 256);
    };
    u32x4 vf[2][KT], kf[2][KT];
    if constexpr (PV) rd_v(0, vf[0]);
    if constexpr (SQ) rd_k(0, kf[0]);
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      const int cur = st & 1, nxt = cur ^ 1;
      if (st + 1 < 8) {
        if constexpr (PV) rd_v(st + 1, vf[nxt]);
        if constexpr (SQ) rd_k(st + 1, kf[nxt]);
      }
      if constexpr (PV) {
#pragma unroll
        for (int u = 0; u < KT; ++u) {
          const int q = KT * st + u, dt = q & 3, j = q >> 2;
          o[dt] = AFmt<DT>::mfma(vf[cur][u], pf[j], o[dt]);
        }
      }
      if constexpr (SQ) {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) s[kt] = AFmt<DT>::mfma(kf[cur][kt], qf[st], s[kt]);
      }
      if constexpr (PV && PS == 2) {
#pragma unroll
        for (int u = 0; u < KT; ++u) {
          const int q = KT * st + u, dt = q & 3, j = q >> 2;
          o[dt] = AFmt<DT>::mfma(vf[cur][u], pl[j], o[dt]);
        }
      }
    }
    if constexpr (PV && SQ) {
      // the fragment reads of a slice, then the MFMAs of the one before
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * KT, 0);
#pragma unroll
      for (int st = 0; st < 7; ++st) {
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * KT, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, KT * (PS + 1), 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, KT * (PS + 1), 0);
    }
  };

  // VALU phase of step it: causal mask, online softmax, P to 16-bit terms,
  // rescale of O.
  auto softmax = [&](int it) {
    const int kb = split + NS * it;
    if (kb * KB + KB - 1 > wpos0) {  // only blocks that cross this wave's diagonal
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (kb * KB + kt * 32 + 8 * g + 4 * fh + e > pos) s[kt][4 * g + e] = -INFINITY;
    }
    // row max of the raw scores (four independent chains); the scale (> 0)
    // is applied to the max and, fused, in the exponent: exp2(s sc - m)
    float mx[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx[i & 3] = fmaxf(mx[i & 3], s[kt][i]);
    const float bm = pair_max(fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3]))) * sc;
    if (__builtin_amdgcn_ballot_w64(bm > m_run + kLazy)) {  // some row's max jumped
      const float m_new = fmaxf(m_run, bm);
      const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.f : m_new));
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) o[dt] *= alpha;
      m_run = m_new;
    }
    const float m_b = (m_run == -INFINITY ? 0.f : m_run) - AFmt<DT>::kPBias;
    float rs[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float pv[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          pv[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][4 * g + e], sc, -m_b));
          rs[e] += pv[e];
        }
        // slice j = 2 kt + g / 2 holds groups g = 2(j%2), 2(j%2)+1 of tile kt
        const int j = 2 * kt + (g >> 1), half = g & 1;
        pf[j][2 * half] = AFmt<DT>::pack2(pv[0], pv[1]);
        pf[j][2 * half + 1] = AFmt<DT>::pack2(pv[2], pv[3]);
        if constexpr (PS == 2) {  // the rounding residue as a second 16-bit term
          pl[j][2 * half] = AFmt<DT>::residue2(pf[j][2 * half], pv[0], pv[1]);
          pl[j][2 * half + 1] = AFmt<DT>::residue2(pf[j][2 * half + 1], pv[2], pv[3]);
        }
      }
    // this lane's half of the row sum; the halves are added once at the end
    l_run += (rs[0] + rs[1]) + (rs[2] + rs[3]);
  };

  // ---- phases: the two halves of the split groups run half a step apart ----
  // ("ping-pong").  A group's step it is an MFMA phase (P.V(it - 1) + S(it))
  // followed by a VALU phase (softmax(it)); the upper half of the groups runs
  // one phase behind the lower, so on every SIMD (one wave of each half) one
  // wave's MFMAs overlap the other's softmax.  Every phase ends in a block barrier, which also orders each
  // group's LDS reads before the refills that overwrite them.
  const int n0 = (nkb + NS - 1) / NS, n1 = (nkb + NS / 2 - 1) / NS;
  const int phases = max(2 * n0 + 1, 2 * n1 + 2);
  using T_ = std::true_type;
  using F_ = std::false_type;
  if (nst > 0) issue_k(0);  // refill(-2)
  if (NB == 2 && nst > 1) issue_k(1);  // refill(-1): K(1), V(0)
  if (NB == 2 && nst > 0) issue_v(0);
  if (off == 0) wait_refill(refill_count(-1));
  exec_barrier();
#ifdef QA_PHASE_STAMPS
  auto stamp = [&](int bucket) {  // charge the cycles since the last mark to a bucket
    __builtin_amdgcn_sched_barrier(0);
    const unsigned long long now = __builtin_amdgcn_s_memtime();
    __builtin_amdgcn_sched_barrier(0);
    cyc[bucket] += now - c_mark;
    c_mark = now;
  };
  stamp(0);
#endif
  for (int ph = 0; ph < phases; ++ph) {
    const int my = ph - off;
#ifdef QA_PHASE_STAMPS
    int bucket = 3;
#endif
    if (my >= 0 && my <= 2 * nst) {
      const int it = my >> 1;
      if ((my & 1) == 0) {
        if (it >= 1 && it < nst)
          mma(T_{}, T_{}, it);
        else if (it == 0 && nst > 0)
          mma(F_{}, T_{}, it);
        else if (it == nst && it >= 1)
          mma(T_{}, F_{}, it);
#ifdef QA_PHASE_STAMPS
        bucket = 1;
        ++nmma;
#endif
      } else {
        if (it + NB < nst) issue_k(it + NB);
        if (it + NB - 1 < nst) issue_v(it + NB - 1);
        softmax(it);
#ifdef QA_PHASE_STAMPS
        bucket = 2;
        ++nvalu;
#endif
      }
    }
#ifdef QA_PHASE_STAMPS
    stamp(bucket);
#endif
    const int nx = ph + 1 - off;  // this wave's next phase
    if (nx >= 0 && (nx & 1) == 0 && (nx >> 1) <= nst) wait_refill(refill_count((nx >> 1) - 1));
    wait_lds();
#ifdef QA_PHASE_STAMPS
    stamp(6);
#endif
    exec_barrier();
#ifdef QA_PHASE_STAMPS
    stamp(4);
#endif
  }

  // ---- merge the key splits (in order) and write the output ----
  l_run = pair_sum(l_run);  // both lane halves of the row
  __syncthreads();
  float* xch = reinterpret_cast<float*>(smem);  // [NS - 1][GW waves][66 values][64 lanes]
  constexpr int XS = GW * 66 * 64;               // one split's floats
  static_assert((NS - 1) * XS * 4 <= (int)sizeof(smem), "merge buffer");
  uint16_t* out = p.out + qrow * p.ldo + (int64_t)head * HD;
  auto store = [&](int dt, int g, const float* v) {
    const u32x2 pk = {AFmt<DT>::pack2(v[0], v[1]), AFmt<DT>::pack2(v[2], v[3])};
    *reinterpret_cast<u32x2*>(out + dt * 32 + 8 * g + 4 * fh) = pk;
  };
  if (nkb == 1) {  // one key block: split 0 holds every key
    if (split == 0 && qrow < p.rows) {
      const float inv = 1.0f / l_run;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = o[dt][4 * g + e] * inv;
          store(dt, g, v);
        }
    }
  } else {
    if (split > 0) {
      float* dst = xch + (split - 1) * XS + wg * 66 * 64 + lane;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) dst[(dt * 16 + v) * 64] = o[dt][v];
      dst[64 * 64] = m_run;
      dst[65 * 64] = l_run;
    }
    __syncthreads();
    if (split == 0 && qrow < p.rows) {
      const float* src = xch + wg * 66 * 64 + lane;
      float mm = m_run;
#pragma unroll
      for (int i = 0; i < NS - 1; ++i) mm = fmaxf(mm, src[i * XS + 64 * 64]);
      const float mu = mm == -INFINITY ? 0.f : mm;
      const float a0 = __builtin_amdgcn_exp2f(m_run - mu);
      float a[NS - 1], sum = l_run * a0;
#pragma unroll
      for (int i = 0; i < NS - 1; ++i) {
        a[i] = __builtin_amdgcn_exp2f(src[i * XS + 64 * 64] - mu);
        sum += src[i * XS + 65 * 64] * a[i];
      }
      const float inv = 1.0f / sum;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = o[dt][4 * g + e] * a0;
#pragma unroll
            for (int i = 0; i < NS - 1; ++i) v[e] += src[i * XS + (dt * 16 + 4 * g + e) * 64] * a[i];
            v[e] *= inv;
          }
          store(dt, g, v);
        }
    }
  }
#ifdef QA_PHASE_STAMPS
  stamp(5);
  if (lane == 0 && blockIdx.x < (unsigned)kAttnStampBlocks && wave < kAttnStampWaves) {
    unsigned long long* d =
        attn_stamp_log + ((size_t)blockIdx.x * kAttnStampWaves + wave) * kAttnStampWords;
    for (int i = 0; i < 7; ++i) d[i] = cyc[i];
    d[7] = nmma;
    d[8] = nvalu;
  }
#endif
}

}  // namespace

namespace {

template <int DT, int REP, int PS, int RG, int NS, int NB>
hipError_t launch_shape(const AttnParams& p, hipStream_t s) {
  const dim3 grid((unsigned)((p.rows + 32 * RG - 1) / (32 * RG) * p.nkvh));
  hipLaunchKernelGGL((attention_kernel<DT, REP, PS, RG, NS, NB>), grid, dim3(NS * REP * RG * 64), 0, s, p);
  return hipGetLastError();
}

template <int DT, int PS>
hipError_t launch_ps(const AttnParams& p, hipStream_t s) {
  const int rep = p.nqh / p.nkvh;
  if (rep == 1) return launch_shape<DT, 1, PS, 2, 2, 2>(p, s);
  if (rep != 2) return hipErrorInvalidValue;  // rejected by qa_attention_prefill's validation
  if (attention_32_row_blocks(p)) return launch_shape<DT, 2, PS, 1, 4, 1>(p, s);
  return launch_shape<DT, 2, PS, 2, 2, 2>(p, s);
}

}  // namespace

hipError_t launch_attention(int dtype, const AttnParams& p, bool p16, hipStream_t s) {
  if (dtype == QA_BF16) return p16 ? launch_ps<QA_BF16, 1>(p, s) : launch_ps<QA_BF16, 2>(p, s);
  return p16 ? launch_ps<QA_F16, 1>(p, s) : launch_ps<QA_F16, 2>(p, s);
}

}  // namespace qa

#ifdef QA_PHASE_STAMPS
// The measurement build's attention records: kAttnStampBlocks x
// kAttnStampWaves x kAttnStampWords words (see attn_stamp_log), copied to
// `out`; *blocks, *waves and *words get the sizes.
extern "C" int qa_attn_stamps_read(unsigned long long* out, int* blocks, int* waves, int* words) {
  if (blocks) *blocks = qa::kAttnStampBlocks;
  if (waves) *waves = qa::kAttnStampWaves;
  if (words) *words = qa::kAttnStampWords;
  if (!out) return QA_OK;
  const hipError_t e =
      hipMemcpyFromSymbol(out, HIP_SYMBOL(qa::attn_stamp_log), sizeof(qa::attn_stamp_log));
  return e == hipSuccess ? QA_OK : QA_EDEVICE;
}
// Zeroes every record (synchronous; call outside stream capture).
extern "C" int qa_attn_stamps_clear(void) {
  static unsigned long long zeros[sizeof(qa::attn_stamp_log) / 8];
  const hipError_t e =
      hipMemcpyToSymbol(HIP_SYMBOL(qa::attn_stamp_log), zeros, sizeof(qa::attn_stamp_log));
  return e == hipSuccess ? QA_OK : QA_EDEVICE;
}
#endif
