// qa_head.hip -- the aligner's ends around the two towers, on the GPU:
//  * the input rows: the token embedding gather with the audio tower's rows
//    scattered into the audio positions (align_raw_rows, src/align_inference.rs:
//    688-714, done on the host by the reference);
//  * the timestamp head: the final RMSNorm on the <timestamp> rows in its
//    folded form (the weight inside the variance), the f32 score head and the
//    argmax (src/align_inference.rs:738-805, host f32 in the reference).
#include "qa_internal.h"

namespace qa {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr uint32_t kOob = 0x80000000u;  // byte offset past every operand's num_records

// One 16-byte-per-lane DMA of a buffer into LDS: lane l's 16 bytes at byte
// offset `off` land at lds + 16 l.
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rs, unsigned char* lds, uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)lds, 16, off,
                                           0, 0, 0);
}

template <int DT>
__device__ __forceinline__ float widen(uint16_t h) {
  if constexpr (DT == QA_F16) return (float)__builtin_bit_cast(_Float16, h);
  else return __uint_as_float((uint32_t)h << 16);
}

// out[r] = table[src[r]] for src >= 0, audio[-src[r] - 1] for src < 0; an
// index out of range gives a zero row.  One wave per row, 16-byte copies.
__global__ void __launch_bounds__(256) embed_scatter_kernel(const EmbedParams p) {
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= p.rows) return;
  const int s = p.src[r];
  const uint16_t* from = nullptr;
  if (s >= 0 && s < p.vocab) from = p.table + (int64_t)s * p.hidden;
  if (s < 0 && -(int64_t)s - 1 < p.n_audio) from = p.audio + (-(int64_t)s - 1) * p.hidden;
  uint16_t* to = p.out + r * p.hidden;
  for (int i = lane * 8; i < p.hidden; i += 512)
    *reinterpret_cast<u32x4*>(to + i) =
        from ? *reinterpret_cast<const u32x4*>(from + i) : u32x4{0, 0, 0, 0};
}

// normed[r][j] = x_j w_j / sqrt(sum_j (x_j w_j)^2 / n + eps) for x the row
// h[pos[r]] (src/align_inference.rs:760-775); one wave per row.  Latency-bound
// (160 KB at 78 rows): with VEC (n a multiple of 8, rows and weights 16-byte
// aligned) a lane loads 8 elements at a time, so a 1024-wide row is two loads in
// flight instead of sixteen 2-byte ones, one after another (12.5 -> 3.8 us).
template <int DT, bool VEC>
__global__ void __launch_bounds__(256) head_norm_kernel(const HeadParams p) {
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= p.rows) return;
  const int pos = p.pos[r];
  const bool ok = pos >= 0 && pos < p.h_rows;
  const uint16_t* x = p.h + (ok ? (int64_t)pos : 0) * p.ldh;
  float* y = p.normed + r * p.n;
  auto row_inv = [&](float s) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    return 1.0f / sqrtf(s / (float)p.n + p.eps);
  };
  if constexpr (VEC) {
    auto products = [&](int j, float* v) {  // x_j w_j .. x_{j+7} w_{j+7}
      const u32x4 h = ok ? *reinterpret_cast<const u32x4*>(x + j) : u32x4{0, 0, 0, 0};
      const f32x4 w0 = *reinterpret_cast<const f32x4*>(p.w + j);
      const f32x4 w1 = *reinterpret_cast<const f32x4*>(p.w + j + 4);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        v[e] = widen<DT>((uint16_t)(h[e >> 1] >> (16 * (e & 1)))) * (e < 4 ? w0[e & 3] : w1[e & 3]);
    };
    float s = 0.f;
    for (int j = lane * 8; j < p.n; j += 512) {
      float v[8];
      products(j, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) s += v[e] * v[e];
    }
    const float inv = row_inv(s);
    for (int j = lane * 8; j < p.n; j += 512) {
      float v[8];
      products(j, v);
#pragma unroll
      for (int e = 0; e < 2; ++e)
        *reinterpret_cast<f32x4*>(y + j + 4 * e) =
            ok ? f32x4{v[4 * e] * inv, v[4 * e + 1] * inv, v[4 * e + 2] * inv, v[4 * e + 3] * inv}
               : f32x4{0, 0, 0, 0};
    }
  } else {
    float s = 0.f;
    for (int j = lane; j < p.n; j += 64) {
      const float v = ok ? widen<DT>(x[j]) * p.w[j] : 0.f;
      s += v * v;
    }
    const float inv = row_inv(s);
    for (int j = lane; j < p.n; j += 64) y[j] = ok ? widen<DT>(x[j]) * p.w[j] * inv : 0.f;
  }
}

// logits[r][l] = sum_j normed[r][j] score[l][j] in f32 on the f32 matrix cores
// (v_mfma_f32_32x32x2_f32: f32 products and sums).  A block takes 32 rows x
// 32 LT labels: its eight waves are LT label tiles x 8 / LT parts of every
// 64-deep k slab, the parts' sums added through LDS in order at the end.  The
// MFMA's A operand is 32 labels, its B operand 32 rows, so a lane holds one
// row and runs of 4 labels.
//
// Slabs stream L2 -> LDS by DMA (a 1 KB instruction is 4 whole 256-byte row
// slabs) into a ring of three, 16-byte chunk c of row r at c ^ (r & 15): a
// fragment read is one chunk of each of 32 rows, two k halves, without bank
// conflicts.  The product does not care which k a slot holds as long as both
// operands agree, so a lane's 16 bytes (4 consecutive k) feed four MFMAs.
// Bound by the f32 matrix cores (157 TFLOP/s; 78 rows x 5000 labels are 96 x
// 5056 in tiles, 6.3 us) and the fill: 17 us at 78 rows, 36 at 240, against
// 44 and 78 on the VALU with 16-byte loads of 64 rows at a time.  Eight waves,
// because a wave that issues DMA does not issue MFMAs (four: 18.6 us at 78);
// three slabs, so that two blocks share a CU (six, one block: 52 against 43 us
// for the whole head at 240 rows).
//
// Needs n % 4 == 0, 16-byte aligned operands and each operand below 2 GiB;
// rows, labels and chunks past the edge read zeros through the range check.
template <int LT>
__global__ void __launch_bounds__(512) head_logits_kernel(const HeadParams p) {
  constexpr int NW = 8, KS = 64, KP = NW / LT;  // k per slab, k parts of a slab
  constexpr int S = 3;                       // ring slabs: 72 or 48 KB, so two blocks fit a CU
  constexpr int RB = 32, LB = 32 * LT;        // rows, labels per block
  constexpr int STAGE = (RB + LB) * KS * 4, INS = (RB + LB) / 4 / NW;  // bytes, DMAs per wave
  constexpr int CPW = KS / 8 / KP;  // chunk pairs of 8 k per wave per slab
  static_assert((S - 1) * INS < 16, "vmcnt's low four bits");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[S * STAGE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lt = wave % LT, kp = wave / LT;
  const int fr = lane & 31, fh = lane >> 5;
  // Block b runs on XCD b % 8: the row blocks of one label block follow each
  // other 8 apart, so its score rows enter one XCD's L2 only.
  const int rb = (int)((p.rows + RB - 1) / RB), group = (int)blockIdx.x / (8 * rb);
  const int64_t r0 = (int64_t)((int)blockIdx.x / 8 % rb) * RB;
  const int64_t l0 = (int64_t)(group * 8 + (int)blockIdx.x % 8) * LB;
  if (l0 >= p.labels) return;  // the last group may hold fewer than 8 label blocks
  const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc(
      p.normed, (short)0, (int)(p.rows * p.n * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(p.score), (short)0, (int)(p.labels * p.n * 4), 0x00020000);
  // DMA instruction i = 8 j + wave fills tile rows 4 i .. 4 i + 3 (rows of
  // `normed` first, then labels); this lane fetches one chunk of one of them.
  uint32_t off[INS];
  int kc[INS];
#pragma unroll
  for (int j = 0; j < INS; ++j) {
    const int t = (NW * j + wave) * 4 + (lane >> 4);  // tile row
    kc[j] = ((lane & 15) ^ (t & 15)) * 4;
    const int64_t row = t < RB ? r0 + t : l0 + t - RB;
    off[j] = row < (t < RB ? p.rows : p.labels) ? (uint32_t)((row * p.n + kc[j]) * 4) : kOob;
  }
  const int nk = (p.n + KS - 1) / KS;
  auto issue = [&](int it) {
#pragma unroll
    for (int j = 0; j < INS; ++j) {
      const int i = NW * j + wave;  // RB / 4 = 8 instructions of rows: j = 0
      const uint32_t o = it * KS + kc[j] < p.n && off[j] != kOob ? off[j] + (uint32_t)it * KS * 4 : kOob;
      dma16(NW * j < RB / 4 ? rsa : rsb, smem + (it % S) * STAGE + i * 1024, o);
    }
  };
  f32x4 fa[2][CPW], fb[2][CPW];
  auto read = [&](int it, int slot) {
    const unsigned char* sa = smem + (it % S) * STAGE;
    const unsigned char* sb = sa + (RB + lt * 32) * KS * 4;
#pragma unroll
    for (int q = 0; q < CPW; ++q) {
      const int at = fr * (KS * 4) + (((2 * (kp * CPW + q) + fh) ^ (fr & 15)) << 4);
      fb[slot][q] = *reinterpret_cast<const f32x4*>(sa + at);
      fa[slot][q] = *reinterpret_cast<const f32x4*>(sb + at);
    }
  };
  // Slab `it` is in (`newer` slabs after it may be in flight) and this wave's
  // reads have returned (lgkmcnt 0); after the barrier both hold for every
  // wave.  No memory fence: it would drain the DMA in flight.
  auto arrive = [&](int newer) {
    __builtin_amdgcn_sched_barrier(0);
    if (newer >= 2)
      __builtin_amdgcn_s_waitcnt(2 * INS | (0x7 << 4));
    else if (newer == 1)
      __builtin_amdgcn_s_waitcnt(INS | (0x7 << 4));
    else
      __builtin_amdgcn_s_waitcnt(0x7 << 4);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // The fragments of slab it + 1 are read while slab it multiplies, and slab
  // it's slot refills behind the barrier that follows its last read.
  f32x16 acc = f32x16{0};
  auto step = [&](int it, int slot) {
    if (it + 1 < nk) {
      arrive(min(S - 2, nk - 2 - it));
      if (it + S < nk) issue(it + S);
      read(it + 1, slot ^ 1);
    }
#pragma unroll
    for (int q = 0; q < CPW; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[slot][q][e], fb[slot][q][e], acc, 0, 0, 0);
  };
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (s < nk) issue(s);
  arrive(min(S - 1, nk - 1));
  read(0, 0);
  for (int it = 0; it < nk; it += 2) {
    step(it, 0);
    if (it + 1 < nk) step(it + 1, 1);
  }
  // the k parts' sums, in order
  float* part = reinterpret_cast<float*>(smem);  // [KP - 1][LT][16][64]
  __syncthreads();
  if (kp > 0) {
#pragma unroll
    for (int v = 0; v < 16; ++v) part[(((kp - 1) * LT + lt) * 16 + v) * 64 + lane] = acc[v];
  }
  __syncthreads();
  if (kp > 0) return;
#pragma unroll
  for (int k = 1; k < KP; ++k)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] += part[(((k - 1) * LT + lt) * 16 + v) * 64 + lane];
  const int64_t r = r0 + fr;
  if (r >= p.rows) return;
  float* out = p.logits + r * p.labels;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int64_t l = l0 + lt * 32 + 8 * g + 4 * fh;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (l + e < p.labels) out[l + e] = acc[4 * g + e];
  }
}

// The same for rows that are not whole aligned 16-byte chunks, or an operand of
// 2 GiB or more, on the VALU (each sum one chain of FMAs, j in order): a block
// takes 64 rows x 64 labels, k in slabs of 64 through LDS stored k-major; a
// thread owns 4 rows x 4 labels.
__global__ void __launch_bounds__(256) head_logits_ragged_kernel(const HeadParams p) {
  constexpr int KS = 64, PR = 4, RB = 16 * PR, LB = 64;
  __shared__ __attribute__((aligned(16))) float as[KS][RB];
  __shared__ __attribute__((aligned(16))) float bs[KS][LB];
  const int t = threadIdx.x;
  const int64_t r0 = (int64_t)blockIdx.y * RB, l0 = (int64_t)blockIdx.x * LB;
  const int tr = t >> 4, tl = t & 15;  // rows tr + 16 u (u < PR), labels 4 tl .. 4 tl + 3
  const int lr = t & 63, lk = (t >> 6) * 16;  // loader: row and label lr, k lk .. lk + 15
  const bool arow = r0 + lr < p.rows, brow = l0 + lr < p.labels;
  const float* ap = p.normed + (arow ? (r0 + lr) * p.n : 0);
  const float* bp = p.score + (brow ? (l0 + lr) * p.n : 0);
  float acc[PR][4] = {};
  for (int k0 = 0; k0 < p.n; k0 += KS) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int k = k0 + lk + e;
      as[lk + e][lr] = (arow && k < p.n) ? ap[k] : 0.f;
      bs[lk + e][lr] = (brow && k < p.n) ? bp[k] : 0.f;
    }
    __syncthreads();
#pragma unroll 4
    for (int kk = 0; kk < KS; ++kk) {
      const f32x4 b4 = *reinterpret_cast<const f32x4*>(&bs[kk][4 * tl]);
#pragma unroll
      for (int u = 0; u < PR; ++u) {
        const float a = as[kk][tr + 16 * u];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[u][i] += a * b4[i];
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < PR; ++u) {
    const int64_t r = r0 + tr + 16 * u;
    if (r >= p.rows) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t l = l0 + 4 * tl + i;
      if (l < p.labels) p.logits[r * p.labels + l] = acc[u][i];
    }
  }
}

// cls[r] = the first index of the largest logit of row r (the reference's
// `v > best_v` scan); one block per row, so that 78 rows keep 78 CUs loading
// (one wave per row: 9.0 us, one block: 3.9).
__global__ void __launch_bounds__(256) head_argmax_kernel(const HeadParams p) {
  __shared__ float wv[4];
  __shared__ int wi[4];
  const int t = threadIdx.x;
  const int64_t r = blockIdx.x;
  const float* row = p.logits + r * p.labels;
  const int none = (int)p.labels;
  float bv = -INFINITY;
  int bi = none;
  // 8 loads in flight per lane, then its labels in increasing order
  for (int64_t l0 = t; l0 < p.labels; l0 += 2048) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = l0 + 256 * u < p.labels ? row[l0 + 256 * u] : -INFINITY;
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (v[u] > bv) {
        bv = v[u];
        bi = (int)(l0 + 256 * u);
      }
  }
  auto take = [&](float ov, int oi) {
    if (ov > bv || (ov == bv && oi < bi)) {
      bv = ov;
      bi = oi;
    }
  };
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) take(__shfl_xor(bv, o, 64), __shfl_xor(bi, o, 64));
  if ((t & 63) == 0) {
    wv[t >> 6] = bv;
    wi[t >> 6] = bi;
  }
  __syncthreads();
  if (t > 0) return;
#pragma unroll
  for (int w = 1; w < 4; ++w) take(wv[w], wi[w]);
  p.cls[r] = bi < none ? bi : 0;
}

template <int DT>
void launch_head_norm(const HeadParams& p, hipStream_t s) {
  auto al = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  const dim3 rows4((unsigned)((p.rows + 3) / 4));
  if (p.n % 8 == 0 && p.ldh % 8 == 0 && al(p.h) && al(p.w) && al(p.normed))
    hipLaunchKernelGGL((head_norm_kernel<DT, true>), rows4, dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL((head_norm_kernel<DT, false>), rows4, dim3(256), 0, s, p);
}

}  // namespace

hipError_t launch_embed_scatter(const EmbedParams& p, hipStream_t s) {
  hipLaunchKernelGGL(embed_scatter_kernel, dim3((unsigned)((p.rows + 3) / 4)), dim3(256), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_timestamp_head(int dtype, const HeadParams& p, hipStream_t s) {
  if (dtype == QA_BF16)
    launch_head_norm<QA_BF16>(p, s);
  else
    launch_head_norm<QA_F16>(p, s);
  constexpr int64_t kSpan = (int64_t)1 << 31;
  const dim3 t(256), t8(512);
  if (p.n % 4 == 0 && (reinterpret_cast<uintptr_t>(p.score) & 15) == 0 &&
      (reinterpret_cast<uintptr_t>(p.normed) & 15) == 0 && p.rows * p.n * 4 < kSpan &&
      p.labels * p.n * 4 < kSpan) {
    const int64_t rb = (p.rows + 31) / 32;
    auto blocks = [&](int64_t lb) { return dim3((unsigned)(((p.labels + lb - 1) / lb + 7) / 8 * 8 * rb)); };
    // 64 labels per block read the rows half as often; 32 as long as the blocks
    // then make one round (up to 128 blocks of 64: up to 32 slots of 5000
    // labels).  The whole head with 32 / 64 labels a block, us: 5000 labels, 32
    // rows (79 blocks of 64) 17.5 / 21.7, 33 (158) 25.0 / 21.8, 78 (237) 25.5 /
    // 22.4, 240 (632) 49.0 / 43.5; 2500 labels, 96 rows (120) 16.9 / 21.2, 97
    // (160) 24.1 / 22.1; 10000 labels, 32 rows (157) 26.8 / 24.2.
    if ((p.labels + 63) / 64 * rb > 128)
      hipLaunchKernelGGL(head_logits_kernel<2>, blocks(64), t8, 0, s, p);
    else
      hipLaunchKernelGGL(head_logits_kernel<1>, blocks(32), t8, 0, s, p);
  } else {
    hipLaunchKernelGGL(head_logits_ragged_kernel,
                       dim3((unsigned)((p.labels + 63) / 64), (unsigned)((p.rows + 63) / 64)), t, 0, s, p);
  }
  hipLaunchKernelGGL(head_argmax_kernel, dim3((unsigned)p.rows), t, 0, s, p);
  return hipGetLastError();
}

}  // namespace qa
