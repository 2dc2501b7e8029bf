// fp32 tall-convention polynomial chain (the dtype-preserving path of
//   _horner_iterate   defmuon/optim/deflation_batched.py:196-204
// for fp32 input: G = X^T X;  B = b G + (c G) G;  X <- a X + X B, all in fp32).
//
// The bf16 chain (ns_chain.hip) is the training path; this one serves callers that
// hand the iteration fp32 matrices (the reference's own convergence study runs it in
// fp32), one launch per GEMM phase over the batch.  gemm_split (below) runs it on the bf16
// matrix cores with split operands; gemm_f32, on the fp32 matrix cores, takes the matrices
// whose planes gemm_split cannot address, and large batches of small ones, whose planes would
// be mostly padding.  In gemm_f32 each phase has the reference's
// rounding points (c G and b G rounded on their own, each sum of two rounded terms rounded
// once; gemm_split scales the sum G G by c instead of G):
//   C[i][j] = fl(fl(beta * R[i][j]) + fl(sum_k fl(s * P(i, k)) Q(j, k)))
// (the R term only where beta != 0, the scale s of P applied as its K slices are
// staged) with P and Q read through element strides, so T^T T, (c G) G and X B need
// no transposed copies.  The products run on the fp32 matrix cores
// (v_mfma_f32_32x32x2_f32, fp32 products and accumulation): 128 x 128 output tiles,
// 4 waves of 64 x 64 (2 x 2 blocks of 32 x 32), 16-deep K slices double-buffered in
// LDS as [k][row] (one barrier per slice), the next slice loaded into registers while
// the current one is multiplied.  Without packed fp32 (which this build leaves off)
// the vector units peak at half the matrix cores' 157.3 TFLOP/s.
#include "common.h"

#include <stdlib.h>

#include <algorithm>

namespace dmh {

constexpr int F_TILE = 128;
constexpr int F_BK = 16;
constexpr int F_LD = F_TILE + 4;   // LDS row stride (floats): 16-byte aligned rows

struct F32Gemm {
  const float* P; long long p_bs; int p_si, p_sk;   // P(i, k) = P[b*p_bs + i*p_si + k*p_sk]
  float p_scale;                                     // staged as fl(p_scale * P(i, k))
  const float* Q; long long q_bs; int q_sj, q_sk;   // Q(j, k)
  const float* R; long long r_bs; int r_ld;         // R[i][j] (beta != 0 only)
  float* C; long long c_bs; int c_ld;               // C[i][j]
  int I, J, K;
  float beta;
};

// One operand's K slice: 8 values per thread, held in registers between the global
// loads and the LDS stores.  KMAJ: the operand's rows are contiguous (element (r, k)
// at r + k * sk): thread t takes rows 4 (t % 32) .. +3 of slice rows k = t / 32 and
// t / 32 + 8.  Otherwise (k contiguous, (r, k) at r * sr + k): rows t / 4 and
// t / 4 + 64, k = 4 (t % 4) .. +3.  VEC: 16-byte loads (every bound and stride a
// multiple of 4 and the base 16-byte aligned, so a float4 is wholly in or out).
template <bool KMAJ, bool VEC>
struct F32Slice {
  float4 v[2];
  __device__ __forceinline__ void load(const float* base, int sr, int sk, int r0, int rows,
                                       int k0, int K, float scale) {
    const int t = threadIdx.x;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int r = KMAJ ? r0 + 4 * (t & 31) : r0 + (t >> 2) + 64 * u;
      const int k = KMAJ ? k0 + (t >> 5) + 8 * u : k0 + 4 * (t & 3);
      float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
      if (VEC) {
        if (r < rows && k < K) x = *(const float4*)(base + (long long)r * sr + (long long)k * sk);
      } else {
        float e[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int rq = KMAJ ? r + q : r, kq = KMAJ ? k : k + q;
          e[q] = (rq < rows && kq < K) ? base[(long long)rq * sr + (long long)kq * sk] : 0.f;
        }
        x = make_float4(e[0], e[1], e[2], e[3]);
      }
      if (scale != 1.f)
        x = make_float4(__fmul_rn(scale, x.x), __fmul_rn(scale, x.y), __fmul_rn(scale, x.z),
                        __fmul_rn(scale, x.w));
      v[u] = x;
    }
  }
  // S[k][r]: slice row k holds the operand's values for contraction index k0 + k
  __device__ __forceinline__ void store(float (*S)[F_LD]) const {
    const int t = threadIdx.x;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (KMAJ) {
        *(float4*)&S[(t >> 5) + 8 * u][4 * (t & 31)] = v[u];
      } else {
        const int r = (t >> 2) + 64 * u, k = 4 * (t & 3);
        S[k][r] = v[u].x;
        S[k + 1][r] = v[u].y;
        S[k + 2][r] = v[u].z;
        S[k + 3][r] = v[u].w;
      }
    }
  }
};

__device__ __forceinline__ f32x16 mfma_f32_32x32x2(float a, float b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// P K-major (PK: its rows contiguous) or k-contiguous; Q always K-major.  At most 128
// VGPRs, so that four workgroups share a CU (4% faster than the compiler's 140).
// grid (ceil(J / 128), ceil(I / 128), batch)
template <bool PK, bool VEC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
void gemm_f32(F32Gemm g) {
  __shared__ __attribute__((aligned(16))) float Ps[2][F_BK][F_LD];
  __shared__ __attribute__((aligned(16))) float Qs[2][F_BK][F_LD];
  const int b = blockIdx.z;
  const int i0 = blockIdx.y * F_TILE, j0 = blockIdx.x * F_TILE;
  const float* P = g.P + (long long)b * g.p_bs;
  const float* Q = g.Q + (long long)b * g.q_bs;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wi = 64 * (wave >> 1), wj = 64 * (wave & 1);   // the wave's 64 x 64 block
  const int r32 = lane & 31, kh = lane >> 5;
  F32Slice<PK, VEC> sp;
  F32Slice<true, VEC> sq;
  const int p_sr = PK ? 1 : g.p_si, p_sk = PK ? g.p_sk : 1;
  f32x16 acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[x][y][e] = 0.f;
  const int nk = (g.K + F_BK - 1) / F_BK;
  sp.load(P, p_sr, p_sk, i0, g.I, 0, g.K, g.p_scale);
  sq.load(Q, 1, g.q_sk, j0, g.J, 0, g.K, 1.f);
  sp.store(Ps[0]);
  sq.store(Qs[0]);
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < nk) {   // next slice into registers under this slice's products
      sp.load(P, p_sr, p_sk, i0, g.I, (kt + 1) * F_BK, g.K, g.p_scale);
      sq.load(Q, 1, g.q_sk, j0, g.J, (kt + 1) * F_BK, g.K, 1.f);
    }
#pragma unroll
    for (int kk = 0; kk < F_BK; kk += 2) {
      // lanes 0-31 hold contraction index kk, lanes 32-63 kk + 1
      const float a0 = Ps[cur][kk + kh][wi + r32], a1 = Ps[cur][kk + kh][wi + 32 + r32];
      const float b0 = Qs[cur][kk + kh][wj + r32], b1 = Qs[cur][kk + kh][wj + 32 + r32];
      acc[0][0] = mfma_f32_32x32x2(a0, b0, acc[0][0]);
      acc[0][1] = mfma_f32_32x32x2(a0, b1, acc[0][1]);
      acc[1][0] = mfma_f32_32x32x2(a1, b0, acc[1][0]);
      acc[1][1] = mfma_f32_32x32x2(a1, b1, acc[1][1]);
    }
    if (kt + 1 < nk) {
      // the other buffer was last read in slice kt - 1, before the previous barrier
      sp.store(Ps[cur ^ 1]);
      sq.store(Qs[cur ^ 1]);
    }
    __syncthreads();
  }
  // acc[x][y][e] holds C[wi + 32 x + 8 (e / 4) + 4 kh + e % 4][wj + 32 y + r32]
  float* C = g.C + (long long)b * g.c_bs;
  const float* R = g.beta != 0.f ? g.R + (long long)b * g.r_bs : nullptr;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const int j = j0 + wj + 32 * y + r32;
      if (j >= g.J) continue;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int i = i0 + wi + 32 * x + 8 * (e >> 2) + 4 * kh + (e & 3);
        if (i >= g.I) continue;
        float v = acc[x][y][e];
        if (R) v = __fadd_rn(__fmul_rn(g.beta, R[(long long)i * g.r_ld + j]), v);
        C[(long long)i * g.c_ld + j] = v;
      }
    }
}

__global__ __launch_bounds__(256) void copy_f32(const float* __restrict__ src, float* __restrict__ dst,
                                                long long count) {
  for (long long e = blockIdx.x * 256LL + threadIdx.x; e < count; e += 256LL * gridDim.x)
    dst[e] = src[e];
}

static bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

static int launch_f32(const F32Gemm& g, int batch, hipStream_t stream, const char* what) {
  const bool pk = g.p_si == 1;
  if (g.q_sj != 1 || (!pk && g.p_sk != 1)) {
    set_error("%s: operand layout not supported (P strides %d,%d, Q strides %d,%d)", what,
              g.p_si, g.p_sk, g.q_sj, g.q_sk);
    return DMH_EINVAL;
  }
  // 16-byte staging loads when every float4 lies wholly inside or outside the operand
  const bool vec = al16(g.P) && al16(g.Q) && g.p_bs % 4 == 0 && g.q_bs % 4 == 0 &&
                   g.q_sk % 4 == 0 && g.J % 4 == 0 &&
                   (pk ? (g.p_sk % 4 == 0 && g.I % 4 == 0) : (g.p_si % 4 == 0 && g.K % 4 == 0));
  const dim3 grid(ceil_div(g.J, F_TILE), ceil_div(g.I, F_TILE), batch);
  if (pk && vec) hipLaunchKernelGGL((gemm_f32<true, true>), grid, dim3(256), 0, stream, g);
  else if (pk) hipLaunchKernelGGL((gemm_f32<true, false>), grid, dim3(256), 0, stream, g);
  else if (vec) hipLaunchKernelGGL((gemm_f32<false, true>), grid, dim3(256), 0, stream, g);
  else hipLaunchKernelGGL((gemm_f32<false, false>), grid, dim3(256), 0, stream, g);
  DMH_CHECK_LAUNCH(what);
  return DMH_OK;
}

// ---------------------------------------------------------------------------
// The same chain on the bf16 matrix cores, the operands split into three bf16 terms.
//
// An fp32 value is exactly the sum of three bf16 values x = x_0 + x_1 + x_2 (each the
// rounding of what the ones before leave), and the six products x_s y_t with s + t <= 2
// carry all of x y but 2^-26 of it, summed in fp32 accumulators, smallest first.  Six bf16
// MFMAs take 3/8 of the time of the fp32 MFMAs they replace, and the sum of the leading
// products rounds once per 16 of them.  Relative error against 64 bits after five steps,
// fp32 matrix cores / here: 8 x (1536, 768) 3.4e-6 / 1.4e-6, (4096, 1024) 3.7e-6 / 1.4e-6,
// (333, 100) 1.4e-6 / 6.1e-7, Polar Express 4.0e-6 / 1.5e-6 on the first.  Only the upper
// tiles of the symmetric G and B are computed.  us for five steps, fp32 cores / here: 8 x
// (1536, 768) 2735 / 905, 24 x (3072, 768) 9025 / 4088, 20 x (1280, 1280) 10752 / 4768,
// (1000, 333) 1030 / 333, (40, 32) 103 / 91.
//
// X, G and B live as their three planes, bf16, zero-padded to multiples of 128, in blocks of
// 64 rows x 32 columns (split_off): a K stage of 32 is one contiguous run per plane of a
// row operand, and 2 KB runs of a K-major one (G = X^T X contracts over X's rows).  The
// epilogues read their fp32 term back from the planes, which hold it exactly.
//
// 128 x 128 tiles, 8 waves (two per SIMD) of 64 x 32, K stages of 32 (48 KB: two operands,
// three planes) in a 3-slot ring filled by direct-to-LDS loads; a wave reads 9 KB of
// fragments for 12 MFMAs of 32 cycles, so the MFMAs bound the loop (1.05-1.2 PFLOP/s of
// executed bf16 products at 24 x (3072, 768): the rate the bf16 chain's power allows too).
// ---------------------------------------------------------------------------
constexpr int S_TILE = 128;
constexpr int S_TK = 32;
constexpr int S_ROWB = S_TK * 2;                 // bytes of a block row
constexpr int S_PLANE = S_TILE * S_ROWB;         // 8 KB: one operand's plane of a stage
constexpr int S_OP = 3 * S_PLANE;
constexpr int S_STAGE = 2 * S_OP;                // 48 KB
constexpr int S_NST = 3;
constexpr int S_THREADS = 512;
constexpr int S_PITCH = S_TILE + 4;              // epilogue rows (floats)
constexpr int S_LPS = 6;                         // loads per wave and stage
static_assert(S_TILE * S_PITCH * 4 <= S_NST * S_STAGE, "the epilogue reuses the ring");

typedef __attribute__((address_space(3))) void* s_lds_ptr;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* s_lds_s16x4;

// element (i, j) of a plane with R rows (a multiple of 64)
__host__ __device__ __forceinline__ long long split_off(int i, int j, int R) {
  return ((long long)(j >> 5) * (R >> 6) + (i >> 6)) * 2048 + (i & 63) * 32 + (j & 31);
}

// x = t[0] + t[1] + t[2] for 2^-102 <= |x| < 3.3962e38 (below, the last terms run out of
// exponents).  Larger and infinite x give NaN: the square of one is infinite in G, so no result
// is finite on the fp32 matrix cores either.
__device__ __forceinline__ void split3(const float (&x)[8], bf16x8 (&t)[3]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float r = x[e];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const bf16 h = f2bf(r);
      t[p][e] = h;
      r -= bf2f(h);
    }
  }
}

enum { SEPI_STORE = 0, SEPI_POLY = 1, SEPI_AXPY = 2 };

struct SplitGemm {
  const bf16* P; int p_rows, p_cols;     // planes of the row operand i (p_rows x p_cols padded)
  const bf16* Q; int q_rows, q_cols;     // planes of the row operand j
  int K;                                 // multiple of 32: past it both operands are zero
  int tiles_m, tiles_n, sym;
  float alpha, beta;                     // POLY: fl(alpha R) + fl(beta C); AXPY: fl(alpha R) + C
  const bf16* R; int r_rows, r_cols;     // the added term's planes (indexed like C)
  bf16* out; int o_rows, o_cols;         // planes of C (and of its mirror image), or
  float* outf; int n, m;                 // ... fp32, row-major n x m
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t s_rsrc(const bf16* p, long long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ void s_load(__amdgpu_buffer_rsrc_t r, char* lds, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (s_lds_ptr)lds, 16, voff, soff, 0, 0);
}
// transposing LDS read of 8 consecutive k of one column: rows of 64 bytes, two reads 4 rows
// apart (lane layout beside lds_tr_frag in ns_chain.hip, and why the pointer is restrict)
__device__ __forceinline__ bf16x8 s_tr_frag(const char* __restrict__ p) {
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s_lds_s16x4)(p));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s_lds_s16x4)(p + 4 * S_ROWB));
  const bf16x4 l4 = __builtin_bit_cast(bf16x4, lo), h4 = __builtin_bit_cast(bf16x4, hi);
  return __builtin_shufflevector(l4, h4, 0, 1, 2, 3, 4, 5, 6, 7);
}
__device__ __forceinline__ f32x16 s_mfma(const bf16x8& a, const bf16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// the 8 values at plane offset off, back in fp32 (both sums are exact)
__device__ __forceinline__ void s_join(const bf16* base, long long plane, long long off,
                                       float (&x)[8]) {
  const bf16x8 t0 = *(const bf16x8*)(base + off), t1 = *(const bf16x8*)(base + plane + off),
               t2 = *(const bf16x8*)(base + 2 * plane + off);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (bf2f(t0[e]) + bf2f(t1[e])) + bf2f(t2[e]);
}

// C[i][j] = sum_k P(i, k) Q(j, k).  TNL = 0: P and Q hold rows i and j; TNL = 1: both are
// K-major (row k holds the values of every i).  grid: batch * tiles
template <int EPI, int TNL>
__global__ __launch_bounds__(S_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_split(SplitGemm g) {
  __shared__ __attribute__((aligned(1024))) char smem[S_NST * S_STAGE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lid = xcd_remap(blockIdx.x, gridDim.x);
  int b, ti, tj;
  if (g.sym) {   // upper triangle by rows
    const int T = g.tiles_m, per = T * (T + 1) / 2;
    b = lid / per;
    int rem = lid - b * per;
    ti = 0;
    while (rem >= T - ti) { rem -= T - ti; ++ti; }
    tj = ti + rem;
  } else {
    const int per = g.tiles_m * g.tiles_n;
    b = lid / per;
    const int t = lid - b * per;
    ti = t / g.tiles_n;
    tj = t - ti * g.tiles_n;
  }
  const int i0 = ti * S_TILE, j0 = tj * S_TILE;
  const long long planeP = (long long)g.p_rows * g.p_cols, planeQ = (long long)g.q_rows * g.q_cols;
  const long long baseP = (long long)b * 3 * planeP + (TNL ? split_off(0, i0, g.p_rows) : split_off(i0, 0, g.p_rows));
  const long long baseQ = (long long)b * 3 * planeQ + (TNL ? split_off(0, j0, g.q_rows) : split_off(j0, 0, g.q_rows));
  // a plane's bytes from the tile's first element: 4 whole block columns (K-major), or the
  // tile's rows in every block column
  const int nk = g.K / S_TK;
  const int stepP = TNL ? S_TK * S_ROWB : g.p_rows * S_ROWB, stepQ = TNL ? S_TK * S_ROWB : g.q_rows * S_ROWB;
  const long long bytesP = TNL ? (long long)4 * g.p_rows * S_ROWB : (long long)(nk - 1) * stepP + S_PLANE;
  const long long bytesQ = TNL ? (long long)4 * g.q_rows * S_ROWB : (long long)(nk - 1) * stepQ + S_PLANE;
  __amdgpu_buffer_rsrc_t rP[3], rQ[3];
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    rP[p] = s_rsrc(g.P + baseP + p * planeP, bytesP);
    rQ[p] = s_rsrc(g.Q + baseQ + p * planeQ, bytesQ);
  }
  // Wave w's load fills 1 KB of a plane: 16 rows of 64 bytes.  rows: rows 16 w .., 16-byte
  // chunk c of row r in slot c ^ ((r >> 2) & 3), so that 16 rows' chunks cover the 256 bytes
  // of the banks once; K-major: k 16 (w & 1) .. of block column w / 2, where a transposing
  // read takes whole rows.
  int voffP, voffQ;
  {
    const int r = 16 * wave + lane / 4;
    if (TNL) {
      const int cb = wave >> 1, k = 16 * (wave & 1) + lane / 4, o = k * S_ROWB + (lane % 4) * 16;
      voffP = cb * g.p_rows * S_ROWB + o;
      voffQ = cb * g.q_rows * S_ROWB + o;
    } else {
      voffP = voffQ = r * S_ROWB + ((lane % 4) ^ ((r >> 2) & 3)) * 16;
    }
  }
  char* const lds_wave = smem + wave * 1024;
  int issued = 0, slot_next = 0;
  auto issue_next = [&]() {
    char* d = lds_wave + slot_next * S_STAGE;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      s_load(rP[p], d + p * S_PLANE, voffP, issued * stepP);
      s_load(rQ[p], d + S_OP + p * S_PLANE, voffQ, issued * stepQ);
    }
    ++issued;
    slot_next = slot_next + 1 == S_NST ? 0 : slot_next + 1;
  };
  const int wm = wave >> 2, wn = wave & 3, r32 = lane & 31, hi = lane >> 5;
  auto frag_off = [&](int c0, int st) {   // rows / columns c0 .. c0 + 31, k 16 st .. + 15
    if (TNL) {
      const int gq = lane >> 4, e = (lane >> 2) & 3, q = lane & 3;
      const int k = 16 * st + 8 * (gq >> 1) + e;
      return (c0 >> 5) * (S_TK * S_ROWB) + k * S_ROWB + (16 * (gq & 1) + 4 * q) * 2;
    }
    const int row = c0 + r32;
    return row * S_ROWB + ((2 * st + hi) ^ ((row >> 2) & 3)) * 16;
  };
  int offP[2][2], offQ[2];
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    offP[0][st] = frag_off(64 * wm, st);
    offP[1][st] = frag_off(64 * wm + 32, st);
    offQ[st] = S_OP + frag_off(32 * wn, st);
  }
  bf16x8 fp[2][2][2][3], fq[2][2][3];   // [buffer][substep][block][plane]
  auto rd = [&](const char* p) { return TNL ? s_tr_frag(p) : *(const bf16x8*)p; };
  auto read = [&](int slot, int x) {
    const char* base = smem + slot * S_STAGE;
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        fp[x][st][0][p] = rd(base + offP[0][st] + p * S_PLANE);
        fp[x][st][1][p] = rd(base + offP[1][st] + p * S_PLANE);
        fq[x][st][p] = rd(base + offQ[st] + p * S_PLANE);
      }
  };
  // the products of the leading terms have accumulators of their own: one rounding at the
  // sum's magnitude per 16 products instead of six (the tall G's sums of squares lost up to
  // 1.4 times the fp32 units' error otherwise)
  f32x16 acc[2], low[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = low[i][e] = 0.f;
  auto mma = [&](int x) {
    // the six term pairs, smallest first, the two blocks in turn
    constexpr int TP[5] = {1, 0, 2, 0, 1}, TQ[5] = {1, 2, 0, 1, 0};
#pragma unroll
    for (int st = 0; st < 2; ++st) {
#pragma unroll
      for (int t = 0; t < 5; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          low[i] = s_mfma(fq[x][st][TQ[t]], fp[x][st][i][TP[t]], low[i]);
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[i] = s_mfma(fq[x][st][0], fp[x][st][i][0], acc[i]);
    }
  };
  auto wait_vm = [](int stages) {   // until at most this many stages are in flight
    if (stages >= 2) __builtin_amdgcn_s_waitcnt(0x0F70 | (2 * S_LPS));
    else if (stages == 1) __builtin_amdgcn_s_waitcnt(0x0F70 | S_LPS);
    else __builtin_amdgcn_s_waitcnt(0x0F70);
  };
  static_assert(2 * S_LPS < 16, "the waits above use the low vmcnt bits");
  auto barrier = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  for (int s = 0; s < S_NST && s < nk; ++s) issue_next();
  wait_vm(issued - 1);
  barrier();
  read(0, 0);
  int slot = 0;
  // as in gemm_ring (ns_chain.hip): once stage s + 1 has landed it is read under stage s's
  // MFMAs, and stage s's slot takes stage s + 3; branch-free pairs while stages are loaded
  auto full_step = [&](int x) {
    slot = slot + 1 == S_NST ? 0 : slot + 1;
    wait_vm(S_NST - 2);
    barrier();
    read(slot, x ^ 1);
    issue_next();
    mma(x);
  };
  auto last_step = [&](int s, int x) {
    if (s + 1 < nk) {
      slot = slot + 1 == S_NST ? 0 : slot + 1;
      wait_vm(issued - (s + 2));
      barrier();
      read(slot, x ^ 1);
      if (issued < nk) issue_next();
    }
    mma(x);
  };
  int s = 0;
  for (; s + 1 + S_NST < nk; s += 2) {
    full_step(0);
    full_step(1);
  }
  for (; s + 1 < nk; s += 2) {
    last_step(s, 0);
    last_step(s + 1, 1);
  }
  if (s < nk) last_step(s, 0);

  // epilogue: acc[i][4 q + e] holds C[64 wm + 32 i + r32][32 wn + 8 q + 4 hi + e]
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] += low[i][e];
  __syncthreads();   // the ring is read out
  float* const S = (float*)smem;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *(float4*)&S[(64 * wm + 32 * i + r32) * S_PITCH + 32 * wn + 8 * q + 4 * hi] =
          make_float4(acc[i][4 * q], acc[i][4 * q + 1], acc[i][4 * q + 2], acc[i][4 * q + 3]);
  __syncthreads();
  const bool mirror = g.sym && ti != tj;
  const long long planeO = (long long)g.o_rows * g.o_cols, planeR = (long long)g.r_rows * g.r_cols;
  const bool vec = (g.m & 3) == 0 && (((uintptr_t)g.outf) & 15) == 0;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    // a wave takes 16 rows of one block column: 1 KB of each plane
    const int u = tid + S_THREADS * v;
    const int r = ((u >> 2) & 15) + 16 * (u >> 8), c = 8 * ((u & 3) + 4 * ((u >> 6) & 3));
    float* sp = S + r * S_PITCH + c;
    const float4 lo = *(const float4*)sp, h4 = *(const float4*)(sp + 4);
    float x[8] = {lo.x, lo.y, lo.z, lo.w, h4.x, h4.y, h4.z, h4.w};
    const int gi = i0 + r, gj = j0 + c;
    if (EPI != SEPI_STORE) {
      float y[8];
      s_join(g.R + (long long)b * 3 * planeR, planeR, split_off(gi, gj, g.r_rows), y);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        x[e] = __fadd_rn(__fmul_rn(g.alpha, y[e]), EPI == SEPI_POLY ? __fmul_rn(g.beta, x[e]) : x[e]);
    }
    if (g.outf) {
      if (gi >= g.n) continue;
      float* o = g.outf + (long long)b * g.n * g.m + (long long)gi * g.m + gj;
      if (vec && gj + 7 < g.m) {
        *(float4*)o = make_float4(x[0], x[1], x[2], x[3]);
        *(float4*)(o + 4) = make_float4(x[4], x[5], x[6], x[7]);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (gj + e < g.m) o[e] = x[e];
      }
      continue;
    }
    bf16x8 t[3];
    split3(x, t);
    bf16* o = g.out + (long long)b * 3 * planeO + split_off(gi, gj, g.o_rows);
#pragma unroll
    for (int p = 0; p < 3; ++p) *(bf16x8*)(o + p * planeO) = t[p];
    if (EPI == SEPI_POLY && mirror) {
      *(float4*)sp = make_float4(x[0], x[1], x[2], x[3]);
      *(float4*)(sp + 4) = make_float4(x[4], x[5], x[6], x[7]);
    }
  }
  if (!mirror) return;
  if (EPI == SEPI_POLY) __syncthreads();   // the polynomial's values replaced the sums
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int u = tid + S_THREADS * v;
    const int j = ((u >> 2) & 15) + 16 * (u >> 8), c = 8 * ((u & 3) + 4 * ((u >> 6) & 3));
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = S[(c + e) * S_PITCH + j];
    bf16x8 t[3];
    split3(x, t);
    bf16* o = g.out + (long long)b * 3 * planeO + split_off(j0 + j, i0 + c, g.o_rows);
#pragma unroll
    for (int p = 0; p < 3; ++p) *(bf16x8*)(o + p * planeO) = t[p];
  }
}

// planes of X (n x m, row-major) padded to np x mp; one thread per 8 columns.
// grid (ceil(np mp / 8 / 256), batch)
__global__ __launch_bounds__(256) void split_entry(const float* __restrict__ X, int n, int m, int np,
                                                   int mp, bf16* __restrict__ out) {
  const int b = blockIdx.y;
  const long long u = blockIdx.x * 256LL + threadIdx.x;
  const long long plane = (long long)np * mp;
  if (u * 8 >= plane) return;
  // in the order of the planes: a block column's rows of four chunks each
  const int ch = (int)(u & 3);
  const long long rowu = u >> 2;
  const int i = (int)(rowu % np), j = 32 * (int)(rowu / np) + 8 * ch;
  float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (i < n) {
    const float* src = X + (long long)b * n * m + (long long)i * m + j;
    if (j + 7 < m && (m & 3) == 0 && (((uintptr_t)X) & 15) == 0) {
      const float4 lo = *(const float4*)src, hi = *(const float4*)(src + 4);
      x[0] = lo.x; x[1] = lo.y; x[2] = lo.z; x[3] = lo.w;
      x[4] = hi.x; x[5] = hi.y; x[6] = hi.z; x[7] = hi.w;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (j + e < m) x[e] = src[e];
    }
  }
  bf16x8 t[3];
  split3(x, t);
  bf16* o = out + (long long)b * 3 * plane + split_off(i, j, np);
#pragma unroll
  for (int p = 0; p < 3; ++p) *(bf16x8*)(o + p * plane) = t[p];
}

template <int EPI, int TNL>
static int launch_split(const SplitGemm& g, int batch, hipStream_t stream, const char* what) {
  const long long per = g.sym ? (long long)g.tiles_m * (g.tiles_m + 1) / 2
                              : (long long)g.tiles_m * g.tiles_n;
  if (per * batch > 0x7fffffffLL) {
    set_error("%s: bad grid (%lld tiles)", what, per * batch);
    return DMH_EINVAL;
  }
  hipLaunchKernelGGL((gemm_split<EPI, TNL>), dim3((int)(per * batch)), dim3(S_THREADS), 0, stream, g);
  DMH_CHECK_LAUNCH(what);
  return DMH_OK;
}

// Whether the traffic of planes padded to 128 costs a batch of small matrices more than the
// split products give: gemm_f32 pads in LDS only.  It is bound by the K walk of a lone tile in
// a small batch and by its traffic from some hundreds of matrices on, so the line is a batch
// size.  us for five steps, fp32 cores / split, above the lines: 128 x (32, 32) 112 / 134, 192 x
// (128, 32) 157 / 173, 256 x (1024, 32) 674 / 694, 384 x (64, 64) 290 / 296, 768 x (200, 64) 715
// / 801, 1024 x (100, 100) 794 / 881, 2048 x (40, 32) 433 / 1289, (64, 64) 860 / 1385, (100, 100)
// 1515 / 1682, and (16, 16) in any batch, 1: 76 / 99, 2048: 234 / 1214; below: 64 x (64, 32) 130 /
// 117, 128 x (1024, 32) 596 / 399, 256 x (64, 64) 222 / 200, 512 x (128, 64) 381 / 366, 768 x (100,
// 100) 661 / 641, and larger matrices in any batch, 2048 x (256, 100) 2453 / 2404, (130, 130)
// 7180 / 5973.
static bool padding_bound(int batch, int n, int m) {
  const long long nm = (long long)n * m;
  if (m <= 32) return nm <= 256 || batch >= (n <= 64 ? 96 : n <= 256 ? 192 : 256);
  if (m <= 64) return batch >= (n <= 64 ? 320 : 576);
  return n <= S_TILE && m <= S_TILE && 5 * nm <= 4 * S_TILE * S_TILE && batch >= 1024;
}

// The split chain addresses a plane with 32-bit offsets; larger matrices run on the fp32 matrix
// cores, as do those it would pad too much.  DMH_HORNER_SPLIT (for comparisons): 0 none, 1 all
// that it can address.
static bool use_split(int batch, int n, int m) {
  const char* env = getenv("DMH_HORNER_SPLIT");
  if (env && env[0] == '0') return false;
  const long long np = ceil_div(n, S_TILE) * (long long)S_TILE, mp = ceil_div(m, S_TILE) * (long long)S_TILE;
  if (np * mp * 2 >= (1LL << 31) || mp * mp * 2 >= (1LL << 31)) return false;
  return (env && env[0] == '1') || !padding_bound(batch, n, m);
}

static size_t gemm_f32_ws(int batch, int n, int m) {
  return (size_t)batch * (2 * (size_t)m * m + (size_t)n * m) * sizeof(float);
}

// planes of X (twice), G and B
static size_t split_ws(int batch, int n, int m) {
  const size_t np = (size_t)ceil_div(n, S_TILE) * S_TILE, mp = (size_t)ceil_div(m, S_TILE) * S_TILE;
  return (size_t)batch * 3 * (2 * np * mp + 2 * mp * mp) * sizeof(bf16);
}

// Matrices taken at a time: the planes are at least 2.25 times what gemm_f32 needs for the same
// batch, so a batch goes in equal parts whose planes stay within that or within 1 GiB, whichever
// is more (or one matrix); 1 GiB is ten matrices of (5120, 1280), several rounds of tiles.
static int split_part(int batch, int n, int m) {
  const size_t limit = std::max(gemm_f32_ws(batch, n, m), (size_t)1 << 30);
  const size_t fit = std::min<size_t>(std::max<size_t>(limit / split_ws(1, n, m), 1), 65535);
  const int parts = (int)((batch + fit - 1) / fit);
  return parts > 1 ? ceil_div(batch, parts) : batch;
}

static int horner_split(hipStream_t stream, const float* x, int batch, int n, int m, float* out,
                        const double* coeffs, int steps, void* ws) {
  const int np = ceil_div(n, S_TILE) * S_TILE, mp = ceil_div(m, S_TILE) * S_TILE;
  const size_t xs = (size_t)batch * 3 * np * mp, gs = (size_t)batch * 3 * mp * mp;
  bf16* cur = (bf16*)ws;
  bf16* nxt = cur + xs;
  bf16* G = nxt + xs;
  bf16* B = G + gs;
  hipLaunchKernelGGL(split_entry, dim3((unsigned)ceil_div((long long)np * mp / 8, 256), batch),
                     dim3(256), 0, stream, x, n, m, np, mp, cur);
  DMH_CHECK_LAUNCH("dmh_horner_f32 split");
  // contraction lengths without the stages that are all padding
  const int kn = ceil_div(n, S_TK) * S_TK, km = ceil_div(m, S_TK) * S_TK;
  for (int it = 0; it < steps; ++it) {
    int rc;
    SplitGemm g{};
    g.tiles_m = g.tiles_n = mp / S_TILE;
    g.sym = 1;
    g.P = g.Q = cur; g.p_rows = g.q_rows = np; g.p_cols = g.q_cols = mp;
    g.K = kn;
    g.out = G; g.o_rows = g.o_cols = mp;
    if ((rc = launch_split<SEPI_STORE, 1>(g, batch, stream, "dmh_horner_f32 G"))) return rc;
    g.P = g.Q = g.R = G; g.p_rows = g.q_rows = g.r_rows = g.p_cols = g.q_cols = g.r_cols = mp;
    g.K = km;
    g.alpha = (float)coeffs[3 * it + 1];
    g.beta = (float)coeffs[3 * it + 2];
    g.out = B;
    if ((rc = launch_split<SEPI_POLY, 0>(g, batch, stream, "dmh_horner_f32 B"))) return rc;
    g.sym = 0;
    g.tiles_m = np / S_TILE;
    g.P = g.R = cur; g.p_rows = g.r_rows = np; g.p_cols = g.r_cols = mp;
    g.Q = B;
    g.alpha = (float)coeffs[3 * it];
    g.out = nxt; g.o_rows = np; g.o_cols = mp;
    if (it + 1 == steps) g.outf = out;
    g.n = n; g.m = m;
    if ((rc = launch_split<SEPI_AXPY, 0>(g, batch, stream, "dmh_horner_f32 X"))) return rc;
    bf16* t = cur; cur = nxt; nxt = t;
  }
  return DMH_OK;
}

static size_t horner_f32_ws(int batch, int n, int m) {
  return use_split(batch, n, m) ? split_ws(split_part(batch, n, m), n, m) : gemm_f32_ws(batch, n, m);
}

}  // namespace dmh

using namespace dmh;

extern "C" {

int dmh_horner_f32_workspace_size(int batch, int n, int m, size_t* bytes) {
  if (batch < 0 || n <= 0 || m <= 0 || !bytes) {
    set_error("dmh_horner_f32_workspace_size: bad arguments");
    return DMH_EINVAL;
  }
  *bytes = horner_f32_ws(batch, n, m);
  return DMH_OK;
}

int dmh_horner_f32(hipStream_t stream, const float* x, int batch, int n, int m, float* out,
                   const double* coeffs, int steps, void* ws, size_t ws_bytes) {
  if (batch == 0) return DMH_OK;
  if (!x || !out || batch < 0 || n <= 0 || m <= 0 || steps < 0 || (steps > 0 && !coeffs)) {
    set_error("dmh_horner_f32: bad arguments (batch=%d n=%d m=%d steps=%d)", batch, n, m, steps);
    return DMH_EINVAL;
  }
  const size_t need = horner_f32_ws(batch, n, m);
  if (!ws || ws_bytes < need) {
    set_error("dmh_horner_f32: workspace %zu < %zu bytes", ws_bytes, need);
    return DMH_EWORKSPACE;
  }
  const long long tsz = (long long)n * m, gsz = (long long)m * m;
  if (steps == 0) {
    const long long count = tsz * batch;
    const int blocks = (int)std::min<long long>((count + 255) / 256, 8192);
    hipLaunchKernelGGL(copy_f32, dim3(blocks), dim3(256), 0, stream, x, out, count);
    DMH_CHECK_LAUNCH("dmh_horner_f32 copy");
    return DMH_OK;
  }
  if (use_split(batch, n, m)) {
    const int part = split_part(batch, n, m);
    for (int b = 0; b < batch; b += part) {
      const int rc = horner_split(stream, x + b * tsz, std::min(part, batch - b), n, m, out + b * tsz,
                                  coeffs, steps, ws);
      if (rc) return rc;
    }
    return DMH_OK;
  }
  float* G = (float*)ws;
  float* Bm = G + gsz * batch;
  float* tmp = Bm + gsz * batch;
  const float* src = x;
  for (int it = 0; it < steps; ++it) {
    const float a = (float)coeffs[3 * it], b = (float)coeffs[3 * it + 1],
                c = (float)coeffs[3 * it + 2];
    float* dst = ((steps - 1 - it) % 2 == 0) ? out : tmp;   // the last step lands in out
    int rc;
    // G = X^T X: P(i, k) = Q(i, k) = X[k][i]
    F32Gemm g1{src, tsz, 1, m, 1.f, src, tsz, 1, m, nullptr, 0, 0, G, gsz, m, m, m, n, 0.f};
    if ((rc = launch_f32(g1, batch, stream, "dmh_horner_f32 G"))) return rc;
    // B = b G + (c G) G: P(i, k) = c G[i][k], Q(j, k) = G[k][j]
    F32Gemm g2{G, gsz, m, 1, c, G, gsz, 1, m, G, gsz, m, Bm, gsz, m, m, m, m, b};
    if ((rc = launch_f32(g2, batch, stream, "dmh_horner_f32 B"))) return rc;
    // X' = a X + X B: P(i, k) = X[i][k], Q(j, k) = B[k][j]
    F32Gemm g3{src, tsz, m, 1, 1.f, Bm, gsz, 1, m, src, tsz, m, dst, tsz, m, n, m, m, a};
    if ((rc = launch_f32(g3, batch, stream, "dmh_horner_f32 X"))) return rc;
    src = dst;
  }
  return DMH_OK;
}

}  // extern "C"
