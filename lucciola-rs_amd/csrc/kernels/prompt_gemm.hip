// The products of a prompt's rows for gfx950: y = x W^T for M rows x of K bf16
// elements and W row-major [N][K] (the reference's linear weights; its
// Qwen2Model::matmul_bf16, src/models.rs:252-295, at M > 1), on
// v_mfma_f32_32x32x16_bf16 with f32 accumulation, in three forms:
//   store: y = round(x W^T)                                  (q/k/v)
//   part:  f32 partials of K ranges [split][M][N], summed into the residual
//          rows by luc_reduce_norm                           (o, down)
//   silu:  W holds [gate rows (N) | up rows (N)], y = round(silu(g) * u) with g
//          and u rounded to bf16 first, as the unfused product and
//          luc_silu_mul give it                              (gate/up)
// and luc_reduce_norm: h = round(h + the partials in split order), one rounding
// (matmul_bf16's beta = 1), and the RMSNorm of the new row for the product that
// follows.
//
// A workgroup of 4 waves takes a tile of BM rows of x (64 or 128) and BN of W (64 or
// 128; 128 for the gate/up pairs: 64 gates with their 64 ups), wave (wn, wm) the W
// rows BN/2 wn .. and the x rows BM/2 wm ...  Both operands are K-contiguous, so a K
// step of 64 is 128 bytes of every row, loaded straight into LDS
// (global_load_lds_dwordx4, one wave-wide load = 8 rows) into a ring of as many stages
// (2 to 4) as leave room for two workgroups per CU; 16-byte chunk c of tile row r sits
// at slot c ^ ((r >> 1) & 7), so a 16-lane pass of the operand reads covers every LDS
// bank.  W is the MFMA's A operand and x its B operand: a lane then holds 4
// consecutive columns of one row of y.
//
// What bounds it (hidden 896, intermediate 4864): a workgroup runs 14 steps (q/k/v, gate/up),
// 4 to 7 (o, in K ranges) or 4 to 38 (down), each a barrier, LDS reads and
// loads from L2 (8 to 10 TB/s in all); larger tiles halve the reads and loads per
// MFMA and win once the rows fill the chip with them (us, hidden 896, intermediate
// 4864): gate/up 28.7 on 64-row tiles and 24.1 on 128 at 700 rows, 15.7 and 16.1 at
// 200; down 49.0 and 33.8 at 2000 rows, 19.2 and 21.6 at 700.  Four stages at one workgroup per
// CU are slower (gate/up 30.7).
//
// Qwen2.5-0.5B, 700 rows, per layer (us): q/k/v 8.8, o 7.3, gate/up with silu 24.1, down
// 19.2, the two reductions with their norms 4.7 each; hipBLASLt with separate norm and
// silu kernels took 11.5, 11.5, 23.3 + 6.3, 28.5 and 3.9 each, with ten launches a layer queued from Python.
//
// They are for prompts of few rows (5 to 1500), so the tiles are small to fill 256
// CUs, and o and down, with N = hidden, are split over K as well.  The tiles of a W row
// block go to one XCD (workgroup id mod 8), so W is read from HBM once and x
// (which fits every XCD's L2) by all.  Rows and columns past the end re-read the
// last one and are not stored.
#include "luc_common.h"

namespace luc {

typedef __attribute__((address_space(3))) void lds_void_g;
typedef __attribute__((address_space(3))) char lds_char_g;

struct GemmArgs {
  const uint16_t* x;  // [m][k]
  const uint16_t* w;  // [n][k], or [2 n][k] for silu
  void* y;            // bf16 [m][n], or f32 [splits][m][n] for part
  int32_t m, n, k;    // k a multiple of 64, n of 4
  int32_t splits;     // K ranges (part), else 1
  int32_t m_tiles, n_tiles;
};

enum GemmEpi { kGemmStore = 0, kGemmPart = 1, kGemmSilu = 2 };
constexpr int kGemmK = 64;

// The operand reads of two 16-k steps, not valid before the wait below.
__device__ inline void gemm_read2(uint32_t a0, uint32_t a1, u32x4_t* x) {
  asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3"
               : "=&v"(x[0]), "=&v"(x[1])
               : "v"(a0), "v"(a1)
               : "memory");
}
// waits for reads issued above while N later ones may be outstanding
template <int N>
__device__ inline void gemm_wait2(u32x4_t* x) {
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(x[0]), "+v"(x[1]) : "n"(N) : "memory");
}

template <int N>
struct GemmIC {  // a compile-time index passed to a generic lambda
  static constexpr int value = N;
};

template <int EPI, int FN, int FM, int NS>
__device__ void gemm_impl(const GemmArgs& A) {
  constexpr int BN = 64 * FN, BM = 64 * FM;    // FN (FM) 32-row fragments of W (x) per wave
  constexpr int CN = EPI == kGemmSilu ? 64 : BN;  // columns of y per workgroup
  static_assert(EPI != kGemmSilu || FN == 2, "a wave's gates and their ups");
  constexpr int STAGE = (BM + BN) * 2 * kGemmK;  // bytes
  constexpr int LOADS = STAGE / 1024 / 4;        // wave-wide loads per wave and stage
  __shared__ __attribute__((aligned(16))) char s_ab[NS][STAGE];  // W rows, then x rows
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = w & 1, wm = w >> 1;
  // W row blocks n = 8 i + id % 8, the row tiles and splits of one in turn
  const int q = blockIdx.x >> 3;
  const int per = A.m_tiles * A.splits;
  const int nt = (q / per) * 8 + (blockIdx.x & 7);
  if (nt >= A.n_tiles) return;
  const int rem = q % per;
  const int mt = rem % A.m_tiles, split = rem / A.m_tiles;
  const int n0 = nt * CN, m0 = mt * BM;
  const int steps_all = A.k / kGemmK;
  const int s0 = (int)((int64_t)steps_all * split / A.splits);
  const int steps = (int)((int64_t)steps_all * (split + 1) / A.splits) - s0;

  // load i of the wave: tile rows 8 j .. 8 j + 7, j = 4 i + w; lane l takes slot
  // l % 8 of row l / 8
  const char* src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int r = 8 * (4 * i + w) + (lane >> 3);  // tile row: W rows 0 .. BN - 1, then x rows
    const int c = (lane & 7) ^ ((r >> 1) & 7);
    const uint16_t* row;
    if (4 * i < BN / 8) {  // (LOADS splits between W and x at a multiple of four)
      // silu: wave wn's gates (32) then their ups
      const int nr = EPI == kGemmSilu ? min(n0 + (r >> 6) * 32 + (r & 31), A.n - 1) + ((r >> 5) & 1) * A.n
                                      : min(n0 + r, A.n - 1);
      row = A.w + (int64_t)nr * A.k;
    } else {
      row = A.x + (int64_t)min(m0 + r - BN, A.m - 1) * A.k;
    }
    src[i] = (const char*)(row + (int64_t)s0 * kGemmK + 8 * c);
  }
  auto issue = [&](int step) __attribute__((always_inline)) {
    char* const dst = s_ab[step % NS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_global_load_lds(src[i] + (int64_t)step * (2 * kGemmK),
                                       (lds_void_g*)(dst + (4 * i + w) * 1024), 16, 0, 0);
  };
  // operand addresses within a stage: row lane % 32 of the fragment, chunk 2 kk + g
  const int g = lane >> 5, lr = lane & 31;
  uint32_t rel[4];  // slot of 16-k step kk (fragments start at multiples of 32 rows: same key)
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) rel[kk] = lr * 128 + (((2 * kk + g) ^ ((lr >> 1) & 7)) << 4);
  const uint32_t wrow = wn * (BN / 2) * 128, xrow = (BN + wm * (BM / 2)) * 128;

  f32x16 acc[FM][FN];
#pragma unroll
  for (int h = 0; h < FM; ++h)
#pragma unroll
    for (int f = 0; f < FN; ++f)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[h][f][e] = 0.0f;

#pragma unroll
  for (int j = 0; j < NS - 1; ++j)
    if (j < steps) issue(j);
  for (int t = 0; t < steps; ++t) {
    // step t has landed; up to NS - 2 newer ones may be in flight
    const int newer = min(steps - 1 - t, NS - 2);
    if (newer >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LOADS) : "memory");
    else if (newer == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // every wave's loads of step t, and every wave done with step t - 1, whose
    // stage step t + NS - 1 takes
    __builtin_amdgcn_s_barrier();
    if (t + NS - 1 < steps) issue(t + NS - 1);
    const uint32_t base = (uint32_t)(uintptr_t)(const lds_char_g*)s_ab[t % NS];
    u32x4_t a[FN][4], b[FM][4];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
      for (int h = 0; h < FM; ++h)
        gemm_read2(base + xrow + h * 4096 + rel[2 * p], base + xrow + h * 4096 + rel[2 * p + 1], b[h] + 2 * p);
#pragma unroll
      for (int f = 0; f < FN; ++f)
        gemm_read2(base + wrow + f * 4096 + rel[2 * p], base + wrow + f * 4096 + rel[2 * p + 1], a[f] + 2 * p);
    }
    auto half = [&](auto pc) __attribute__((always_inline)) {  // 16-k steps 2 p and 2 p + 1
      constexpr int p = decltype(pc)::value;
      constexpr int later = p == 0 ? 2 * (FN + FM) : 0;  // reads that may be outstanding
#pragma unroll
      for (int h = 0; h < FM; ++h) gemm_wait2<later>(b[h] + 2 * p);
#pragma unroll
      for (int f = 0; f < FN; ++f) gemm_wait2<later>(a[f] + 2 * p);
#pragma unroll
      for (int kk = 2 * p; kk < 2 * p + 2; ++kk)
#pragma unroll
        for (int h = 0; h < FM; ++h)
#pragma unroll
          for (int f = 0; f < FN; ++f)
            acc[h][f] = mfma32<kBF16>(__builtin_bit_cast(uint4, a[f][kk]), __builtin_bit_cast(uint4, b[h][kk]),
                                      acc[h][f]);
    };
    half(GemmIC<0>{});
    half(GemmIC<1>{});
  }

  // lane: row m of fragment hh, columns nf + 8 i + 4 g .. + 3 of fragment f (silu:
  // gate in f = 0, its up in f = 1)
#pragma unroll
  for (int hh = 0; hh < FM; ++hh) {
    const int m = m0 + wm * (BM / 2) + hh * 32 + lr;
    if (m >= A.m) break;
#pragma unroll
    for (int f = 0; f < (EPI == kGemmSilu ? 1 : FN); ++f)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = n0 + wn * (CN / 2) + f * 32 + 8 * i + 4 * g;
        if (n >= A.n) continue;  // (n a multiple of 4)
        const f32x16& v = acc[hh][f];
        if constexpr (EPI == kGemmPart) {
          float* const y = (float*)A.y + ((int64_t)split * A.m + m) * A.n + n;
          *(float4*)y = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
        } else {
          uint32_t o[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if constexpr (EPI == kGemmSilu) {
#pragma clang fp contract(off)
              const float gt = St<kBF16>::load(St<kBF16>::store(v[4 * i + j]));
              const float up = St<kBF16>::load(St<kBF16>::store(acc[hh][FN - 1][4 * i + j]));
              const float s = gt / (1.0f + expf(-gt));
              o[j] = St<kBF16>::store(s * up);
            } else {
              o[j] = St<kBF16>::store(v[4 * i + j]);
            }
          }
          *(uint2*)((uint16_t*)A.y + (int64_t)m * A.n + n) = make_uint2(o[0] | o[1] << 16, o[2] | o[3] << 16);
        }
      }
  }
}

// h[row] = round(h[row] + sum over splits of part[s][row]), and out[row] =
// RMSNorm(h[row]) * weight (rmsnorm.cu's formula; the sum order is
// luc_rmsnorm_bf16's) unless weight is null.  One workgroup per row of n <= 8192
// elements, a multiple of 8.
constexpr int kReduceThreads = 256, kReduceChunks = 4;
__device__ void reduce_norm_impl(uint16_t* h, const float* part, int splits, uint16_t* out,
                                 const uint16_t* weight, float eps, int rows, int n) {
#pragma clang fp contract(off)
  __shared__ float red[kReduceThreads];
  const int t = threadIdx.x;
  const int64_t row = blockIdx.x;
  uint4* const hr = (uint4*)(h + row * n);
  const int chunks = n / 8;
  uint4 v[kReduceChunks];
  float s = 0.0f;
#pragma unroll
  for (int k = 0; k < kReduceChunks; ++k) {
    const int c = t + k * kReduceThreads;
    if (c >= chunks) continue;
    const uint4 old = hr[c];
    float a[8] = {};
    for (int sp = 0; sp < splits; ++sp) {
      const float4* const p = (const float4*)(part + ((int64_t)sp * rows + row) * n) + 2 * c;
      const float4 p0 = p[0], p1 = p[1];
      a[0] += p0.x; a[1] += p0.y; a[2] += p0.z; a[3] += p0.w;
      a[4] += p1.x; a[5] += p1.y; a[6] += p1.z; a[7] += p1.w;
    }
    uint16_t o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      o[e] = St<kBF16>::store(a[e] + St<kBF16>::load(chunk_elem(old, e)));
      const float f = St<kBF16>::load(o[e]);
      s = fmaf(f, f, s);
    }
    v[k] = chunk_pack(o);
    hr[c] = v[k];
  }
  if (!weight) return;
  red[t] = s;
  __syncthreads();
  if (t < 64) {
    float a = (red[t] + red[t + 128]) + (red[t + 64] + red[t + 192]);
#pragma unroll
    for (int k = 32; k > 0; k >>= 1) a = a + __shfl_down(a, k);
    if (t == 0) red[0] = a;
  }
  __syncthreads();
  const float inv = 1.0f / sqrtf(red[0] / (float)n + eps);
  const uint4* const wr = (const uint4*)weight;
  uint4* const y = (uint4*)(out + row * n);
#pragma unroll
  for (int k = 0; k < kReduceChunks; ++k) {
    const int c = t + k * kReduceThreads;
    if (c >= chunks) continue;
    const uint4 wc = wr[c];
    uint16_t o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float f = St<kBF16>::load(chunk_elem(v[k], e)) * inv;
      o[e] = St<kBF16>::store(f * St<kBF16>::load(chunk_elem(wc, e)));
    }
    y[c] = chunk_pack(o);
  }
}

}  // namespace luc

#define LUC_GEMM(NAME, EPI, FN, FM, NS)                                          \
  extern "C" __global__ __launch_bounds__(256, 2) void NAME(luc::GemmArgs a) {   \
    luc::gemm_impl<luc::EPI, FN, FM, NS>(a);                                     \
  }
LUC_GEMM(luc_gemm_store_bf16, kGemmStore, 1, 1, 4)
LUC_GEMM(luc_gemm_part_bf16, kGemmPart, 1, 1, 4)
LUC_GEMM(luc_gemm_part_bf16_m128, kGemmPart, 2, 2, 2)
LUC_GEMM(luc_gemm_silu_bf16, kGemmSilu, 2, 1, 3)
LUC_GEMM(luc_gemm_silu_bf16_m128, kGemmSilu, 2, 2, 2)

extern "C" __global__ __launch_bounds__(256) void luc_reduce_norm_bf16(uint16_t* h, const float* part,
                                                                       int splits, uint16_t* out,
                                                                       const uint16_t* weight, float eps,
                                                                       int rows, int n) {
  luc::reduce_norm_impl(h, part, splits, out, weight, eps, rows, n);
}
