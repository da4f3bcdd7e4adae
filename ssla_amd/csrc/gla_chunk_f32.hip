// Chunked GLA in fp32: forward and backward for fp32 q, k, v, g (the
// reference runs its chunk pipeline for fp32 inputs too: ops/gla/chunk.py
// 906-960 forward, 963-1053 backward, with TF32 operands in most of its
// dots; here every product is fp32).
//
// Chunks of 64 rows restart at every sequence start; G is the chunk-local
// inclusive cumsum of g (log2-scaled), gamma = G at the chunk's last row,
// s = scale:
//   A_ij = s sum_k q_ik k_jk 2^(G_ik - G_jk)  (j <= i)
//   o    = s (q 2^G) S_c + A v
//   S_c+1 = 2^gamma S_c + (k 2^(gamma - G))^T v
// Every decay factor is kept at or below 1, so the exponent clamp at -126
// (v_exp_f32 range) only ever replaces a value that is itself below 2^-126:
// * diagonal 16-row blocks (j, i in one block, j <= i): 2^(G_i - G_j)
//   directly, one exponential of a non-positive argument per term;
// * blocks J < I: 2^(G_i - G_j) = 2^(G_i - E_J) 2^(E_J - G_j) with E_J = G at
//   the last row of block J (both factors <= 1): k~_j = k_j 2^(E_J - G_j)
//   per row, and the q side per (row, J) -- A and dq; or
//   2^(G_i - S_I) 2^(S_I - G_j) with S_I = G at the first row of block I:
//   q~_i = q_i 2^(G_i - S_I) per row, and the k side per (row, I) -- dk;
// * o, the state and dh use 2^G and 2^(gamma - G) (<= 1) directly.
// All products are fp32: on the matrix cores' fp32 instruction in the
// chunk-parallel kernels, on the VALU in the serial walk.
//
// ssla_gla_chunk_f32_fwd_ws and ssla_gla_chunk_f32_bwd give every chunk its own
// workgroup (below, with their workspace); ssla_gla_chunk_f32_fwd, for callers
// that have no workspace, walks the chunks with one workgroup per (sequence,
// head, 16-column V tile) and its state tile in LDS.  Backward of a chunk
// (K, V <= 64), h its entering state and dh its leaving gradient:
// dv = A^T dO + k_d dh,
// dq, dk from dO h^T, v dh^T and dA = (dO v^T) masked, dg = reverse cumsum
// of dG = q dq - k dk plus the chunk-total decay's term, dh <- 2^gamma dh +
// s (q 2^G)^T dO.  dG is formed without the terms that cancel exactly (the
// j = i term of A, and the state term of dk against the same term of the
// chunk-total decay's gradient): with strongly decaying gates dg is small
// next to q dq and k dk, and those terms would leave only their rounding.
#include "seq_slots.h"

namespace ssla {
namespace {

constexpr int kC = 64;        // chunk rows
constexpr int kP = 65;        // LDS row pitch (floats): conflict-free column walks
constexpr int kVT = 16;       // value columns per forward workgroup
constexpr int kThreads = 256;

__device__ __forceinline__ float ex2c(float x) { return fast_exp2(fminf(fmaxf(x, -126.f), 126.f)); }

__device__ __forceinline__ void seq_bounds(const int64_t *cu, int n, int64_t T, int64_t &bos, int64_t &eos) {
  bos = min(max(cu[n], (int64_t)0), T);
  eos = min(max(cu[n + 1], bos), T);
}

// Per-key references of a chunk (64 threads, one key each, after the
// cumsum): E[J] = G at row 16 J + 15, PE[J] = 2^(gamma - E[J]), DL = 2^gamma.
struct ChunkRefs {
  float E[4][64], PE[4][64], DL[64];
};

// Chunk-local cumsum of the gates (log2-scaled, in place) and the
// references; rows past the chunk hold g = 0, so G stays at gamma there.
__device__ __forceinline__ void chunk_cumsum(float (*sG)[kP], ChunkRefs &R) {
  const int kk = threadIdx.x;
  if (kk >= 64) return;
  float acc = 0.f;
  for (int r = 0; r < kC; ++r) {
    acc += sG[r][kk];
    sG[r][kk] = acc;
  }
#pragma unroll
  for (int I = 0; I < 4; ++I) {
    R.E[I][kk] = sG[16 * I + 15][kk];
    R.PE[I][kk] = ex2c(acc - sG[16 * I + 15][kk]);
  }
  R.DL[kk] = ex2c(acc);
}

// k~_j = k_j 2^(E_J - G_j) (into sKt).
__device__ __forceinline__ void chunk_tilde(const float (*sK)[kP], const float (*sG)[kP], const ChunkRefs &R,
                                            float (*sKt)[kP]) {
  for (int e = threadIdx.x; e < kC * 64; e += kThreads) {
    const int r = e >> 6, kk = e & 63, B = r >> 4;
    sKt[r][kk] = sK[r][kk] * ex2c(R.E[B][kk] - sG[r][kk]);
  }
}

// The 16 entries A_i,16J..16J+15 of thread (i, J), scale applied (zero
// above the diagonal): blocks J < I as (q_i 2^(G_i - E_J)) . k~_j, the
// diagonal block term by term.
__device__ __forceinline__ void a_row16(const float (*sQ)[kP], const float (*sK)[kP], const float (*sKt)[kP],
                                        const float (*sG)[kP], const ChunkRefs &R, int K, int i, int J, float scale,
                                        float (&a)[16]) {
  const int I = i >> 4;
#pragma unroll
  for (int jj = 0; jj < 16; ++jj) a[jj] = 0.f;
  if (J > I) return;
  if (J < I) {
    for (int kk = 0; kk < K; ++kk) {
      const float qv = sQ[i][kk] * ex2c(sG[i][kk] - R.E[J][kk]);
#pragma unroll
      for (int jj = 0; jj < 16; ++jj) a[jj] = fmaf(qv, sKt[16 * J + jj][kk], a[jj]);
    }
  } else {
    const int il = i - 16 * I;   // j = 16 I + jj <= i
    for (int kk = 0; kk < K; ++kk) {
      const float qv = sQ[i][kk], gi = sG[i][kk];
#pragma unroll
      for (int jj = 0; jj < 16; ++jj)
        if (jj <= il) a[jj] = fmaf(qv * sK[16 * I + jj][kk], ex2c(gi - sG[16 * I + jj][kk]), a[jj]);
    }
  }
#pragma unroll
  for (int jj = 0; jj < 16; ++jj) a[jj] *= scale;
}

// ---------------------------------------------------------------- forward --
__global__ __launch_bounds__(kThreads) void f32_fwd_kernel(
    const float *__restrict__ q, const float *__restrict__ k, const float *__restrict__ v,
    const float *__restrict__ g, const int64_t *__restrict__ cu, int n_seq, int64_t T, int H, int K, int V,
    float scale, const float *__restrict__ h0, float *__restrict__ o, float *__restrict__ ht) {
  __shared__ float sQ[kC][kP], sK[kC][kP], sKt[kC][kP], sG[kC][kP], sA[kC][kP];
  __shared__ float sV[kC][kVT], sS[64][kVT];
  __shared__ ChunkRefs R;
  const int tid = threadIdx.x;
  const int nvt = (V + kVT - 1) / kVT;
  const int64_t wg = blockIdx.x;
  const int vt = static_cast<int>(wg % nvt);
  const int h = static_cast<int>((wg / nvt) % H);
  const int n = static_cast<int>(wg / (static_cast<int64_t>(nvt) * H));
  const int v0 = vt * kVT;
  int64_t bos, eos;
  seq_bounds(cu, n, T, bos, eos);
  const int64_t sb = (static_cast<int64_t>(n) * H + h) * K * V;   // this (sequence, head)'s state
  for (int e = tid; e < 64 * kVT; e += kThreads) {
    const int kk = e / kVT, c = e % kVT;
    sS[kk][c] = (h0 && kk < K && v0 + c < V) ? h0[sb + static_cast<int64_t>(kk) * V + v0 + c] : 0.f;
  }
  const int ri = tid >> 2, q4 = tid & 3;   // row (or key) of this thread, and its quarter
  for (int64_t t0 = bos; t0 < eos; t0 += kC) {
    const int nc = static_cast<int>(min(static_cast<int64_t>(kC), eos - t0));
    __syncthreads();   // the previous chunk is done with the tiles
    for (int e = tid; e < kC * 64; e += kThreads) {
      const int r = e >> 6, kk = e & 63;
      const bool ok = r < nc && kk < K;
      const int64_t idx = ((t0 + r) * H + h) * K + kk;
      sQ[r][kk] = ok ? q[idx] : 0.f;
      sK[r][kk] = ok ? k[idx] : 0.f;
      sG[r][kk] = ok ? g[idx] * kLog2e : 0.f;
    }
    for (int e = tid; e < kC * kVT; e += kThreads) {
      const int r = e / kVT, c = e % kVT;
      sV[r][c] = (r < nc && v0 + c < V) ? v[((t0 + r) * H + h) * V + v0 + c] : 0.f;
    }
    __syncthreads();
    chunk_cumsum(sG, R);
    __syncthreads();
    chunk_tilde(sK, sG, R, sKt);
    __syncthreads();
    {   // A, thread (row ri, block q4)
      float a[16];
      a_row16(sQ, sK, sKt, sG, R, K, ri, q4, scale, a);
#pragma unroll
      for (int jj = 0; jj < 16; ++jj) sA[ri][16 * q4 + jj] = a[jj];
    }
    __syncthreads();
    {   // o: thread (row ri, columns 4 q4 .. 4 q4 + 3)
      const int c0 = 4 * q4;
      float acc[4] = {0.f, 0.f, 0.f, 0.f};
      for (int kk = 0; kk < K; ++kk) {
        const float qg = sQ[ri][kk] * ex2c(sG[ri][kk]);   // q 2^G
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] = fmaf(qg, sS[kk][c0 + c], acc[c]);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[c] *= scale;
      for (int j = 0; j <= ri; ++j) {
        const float aij = sA[ri][j];
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] = fmaf(aij, sV[j][c0 + c], acc[c]);
      }
      if (ri < nc) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (v0 + c0 + c < V) o[((t0 + ri) * H + h) * V + v0 + c0 + c] = acc[c];
      }
    }
    __syncthreads();
    {   // S <- 2^gamma S + (k~ 2^(gamma - E_J))^T v: thread (key ri, columns 4 q4 ..)
      const int c0 = 4 * q4;
      float acc[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[c] = sS[ri][c0 + c] * R.DL[ri];
      for (int j = 0; j < kC; ++j) {
        const float kd = sKt[j][ri] * R.PE[j >> 4][ri];
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] = fmaf(kd, sV[j][c0 + c], acc[c]);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) sS[ri][c0 + c] = acc[c];
    }
  }
  __syncthreads();
  if (ht) {
    for (int e = tid; e < 64 * kVT; e += kThreads) {
      const int kk = e / kVT, c = e % kVT;
      if (kk < K && v0 + c < V) ht[sb + static_cast<int64_t>(kk) * V + v0 + c] = sS[kk][c];
    }
  }
}

// ------------------------------------------------ chunk-parallel kernels --
// Forward and backward with every chunk its own workgroup and all products
// on v_mfma_f32_16x16x4_f32 (fp32 products, fp32 sums):
//   f32_states_kernel   each chunk's own contribution to the state,
//                       L = (k 2^(gamma - G))^T v, and (backward) to the state
//                       gradient, R = s (q 2^G)^T dO, with its decay 2^gamma
//   f32_prefix_kernel   S <- 2^gamma S + L over the chunks of a sequence (and
//                       dh <- 2^gamma dh + R from its end), element by element,
//                       leaving the entering value in each chunk's slot
//   f32_out_kernel / f32_grad_kernel   o, or dq, dk, dv, dg, of a chunk from
//                       its entering state (and leaving gradient)
// The walks they replace ran one workgroup per (sequence, head), 48 of them
// on 256 CUs at 12 ragged sequences of 8,209 rows in all, H = 4, K = V = 64:
// 14.4 ms for forward and backward against 0.159 ms here.  (Under the profiler,
// which drains the device between kernels, grad 73, states 35 and prefix 38 in
// two launches each, out 32 us: 179 in all.)  What bounds them now is latency: each workgroup's load, cumsum, stage and product
// phases follow one another with one or two workgroups per CU, and the prefix
// is a serial chain over the longest sequence's chunks.
//
// A 64 x 64 fp32 tile in LDS holds row r's 16-byte segment s at s ^ (r & 15).
// MFMA operands are read from it two ways, over the same order of the
// contraction index (step 4t + e of lane group gq: index 16t + 4gq + e):
//   row operand   lane r of the group holds row r's 4 columns 16t + 4gq ..
//                 (one 16-byte read for 4 steps)
//   col operand   lane r holds column c0 + r of row 16t + 4gq + e (4-byte
//                 reads; the four groups fall on different banks)
// A 16 x 16 result sits in the lanes as D[4gq + x][r]: as the second operand
// of a product that contracts over its row index it needs no exchange, so
// the blocks of A and dA feed the next product from registers.
//
// Decays inside a chunk: the gates are summed within each 16-row block, and
// the decay between rows of two blocks is put together from their own sums
// and the totals of the blocks between.  q~_i = q_i 2^(G_i - S_I) and
// k~_j = k_j 2^(E_J - G_j) are staged once; a block pair takes the per-key factor 2^(S_I - E_J) on one
// operand, or 2^(G_i - E_J) / 2^(S_I - G_j) on its result, all <= 1 for J < I.
// For J = I the factor undoes at most the block's own decay, and the block runs
// on the matrix cores like the others while |G - S_I| stays within 40 and q and
// k are zero or within 2^-46 .. 2^47: then q~, k~ and either of them times the
// factor are normal numbers (exponents of at most 80 and 40).  Any other chunk
// (`slow`, uniform over the workgroup) adds its diagonal blocks term by term,
// from raw q and k with exponentials of non-positive arguments only -- and so
// does one with an infinity or NaN in its rows (of v and dO as well): the
// matrix cores multiply a masked zero with every row of the block, which would
// carry it to rows before its own (after, in dk and dv).

constexpr float kDiagRange = 40.f;
constexpr uint32_t kInputMin = (127u - 46) << 23;   // the bits of 2^-46
constexpr float kInputMax = 0x1p47f;

__device__ __forceinline__ int tix(int r, int c) { return r * 64 + ((((c >> 2) ^ (r & 15)) << 2) | (c & 3)); }
__device__ __forceinline__ f32x4 row4(const float *t, int r, int c) {
  return *reinterpret_cast<const f32x4 *>(t + tix(r, c));
}
__device__ __forceinline__ void put4(float *t, int r, int c, const f32x4 &x) {
  *reinterpret_cast<f32x4 *>(t + tix(r, c)) = x;
}
__device__ __forceinline__ f32x4 mfma4(float a, float b, const f32x4 &c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 ref4(const float *p) { return *reinterpret_cast<const f32x4 *>(p); }

// 4 columns from c of a row of C floats (zero where !ok or past C); VEC: C is
// a multiple of 4 and the rows are 16-byte aligned.
template <bool VEC>
__device__ __forceinline__ f32x4 load4(const float *row, bool ok, int c, int C) {
  f32x4 x = {0.f, 0.f, 0.f, 0.f};
  if (!ok) return x;
  if (VEC) {
    if (c < C) x = *reinterpret_cast<const f32x4 *>(row + c);
  } else {
#pragma unroll
    for (int m = 0; m < 4; ++m)
      if (c + m < C) x[m] = row[c + m];
  }
  return x;
}
template <bool VEC>
__device__ __forceinline__ void store4(float *row, int c, int C, const f32x4 &x) {
  if (VEC) {
    if (c < C) *reinterpret_cast<f32x4 *>(row + c) = x;
  } else {
#pragma unroll
    for (int m = 0; m < 4; ++m)
      if (c + m < C) row[c + m] = x[m];
  }
}

// A chunk's workspace slot is its slot in units of 64 rows (seq_slots.h).
struct ChunkAt {
  int nc;           // rows
  int64_t t0;       // first row
  bool first, last; // of its sequence
};

// The chunk of a slot (false: none).
__device__ __forceinline__ bool chunk_of_slot(const int64_t *cu, int n_seq, int64_t T, int64_t slot, ChunkAt &at) {
  int n;
  int64_t bos, eos, first;
  if (!seq_of_slot(cu, n_seq, T, kC, slot, n, bos, eos, first)) return false;
  at.t0 = bos + (slot - first) * kC;
  if (at.t0 >= eos) return false;
  at.nc = static_cast<int>(min(static_cast<int64_t>(kC), eos - at.t0));
  at.first = slot == first;
  at.last = at.t0 + kC >= eos;
  return true;
}

// Cumsum of the gates (log2-scaled, in place) local to each 16-row block:
// thread (quad, group) holds rows RPT group .. of keys 4 quad ..; a wavefront
// holds 4 RPT rows.  Block-local sums keep the differences between rows exact
// to the block's own decay (a chunk-wide sum loses two bits and more of them),
// and every partial sum is formed in row order, so a row and the rows without
// decay after it hold the same value.  wtot: each wavefront's total (a block's
// when RPT is 4).  One barrier.
template <int RPT>
__device__ __forceinline__ void cumsum_rows(f32x4 (&g)[RPT], float (*wtot)[64]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, gq = lane >> 4, quad = lane & 15;
#pragma unroll
  for (int m = 0; m < RPT; ++m) {
    g[m] *= kLog2e;
    if (m) g[m] += g[m - 1];
  }
  f32x4 t[3];   // totals of groups 0 .. 2
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const float own = g[RPT - 1][x];
#pragma unroll
    for (int i = 0; i < 3; ++i) t[i][x] = __shfl(own, 16 * i + quad);
  }
  if (gq == 3) *reinterpret_cast<f32x4 *>(&wtot[w][4 * quad]) = ((t[0] + t[1]) + t[2]) + g[RPT - 1];
  __syncthreads();
  f32x4 off = {0.f, 0.f, 0.f, 0.f};
  if (RPT == 2 && (w & 1)) off = ref4(&wtot[w - 1][4 * quad]);   // the block's first eight rows
#pragma unroll
  for (int i = 0; i < 3; ++i)
    if (i < gq) off += t[i];
#pragma unroll
  for (int m = 0; m < RPT; ++m) g[m] += off;
}

// Decay of the whole blocks strictly between a and b at 4 keys: sE[B] = block
// B's total (G at its last row).
__device__ __forceinline__ f32x4 between(const float (*sE)[64], int a, int b, int col) {
  f32x4 x = {0.f, 0.f, 0.f, 0.f};
  for (int B = a + 1; B < b; ++B) x += ref4(&sE[B][col]);
  return x;
}

struct F32Args {
  const float *q, *k, *v, *g, *dO, *h0, *dht;
  const int64_t *cu;
  float *o, *ht, *dq, *dk, *dv, *dg, *dh0;
  float *sh, *sd;       // per (slot, head, value group): entering state / leaving gradient, [64][64]
  float *eh, *ed;       // per (slot, head): 2^gamma of the keys, as each of them uses it
  int64_t T, n_slots;
  int n_seq, H, K, V, nvg;
  float scale;
};

// L or R of one chunk (blockIdx.y: 0 = L, 1 = R); one workgroup per (slot,
// head, value group), wavefront w the keys 16w ..
template <bool VEC>
__global__ __launch_bounds__(256) void f32_states_kernel(F32Args a, int need_last, int need_first) {
  __shared__ __attribute__((aligned(16))) float sX[64 * 64], sY[64 * 64], wtot[4][64];
  const bool rev = blockIdx.y;
  const int vg = static_cast<int>(blockIdx.x % a.nvg);
  const int h = static_cast<int>(blockIdx.x / a.nvg % a.H);
  const int64_t slot = blockIdx.x / a.nvg / a.H;
  ChunkAt at;
  if (!chunk_of_slot(a.cu, a.n_seq, a.T, slot, at)) return;
  if (rev ? (at.first && !need_first) : (at.last && !need_last)) return;   // nothing follows it
  const int tid = threadIdx.x, quad = tid & 15, r0 = (tid >> 4) * 4, K = a.K, V = a.V, v0 = 64 * vg;
  const float *X = rev ? a.q : a.k, *Y = rev ? a.dO : a.v;
  f32x4 x[4], y[4], g[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const bool ok = r0 + m < at.nc;
    const int64_t row = (at.t0 + r0 + m) * a.H + h;
    g[m] = load4<VEC>(a.g + row * K, ok, 4 * quad, K);
    x[m] = load4<VEC>(X + row * K, ok, 4 * quad, K);
    y[m] = load4<VEC>(Y + row * V, ok, v0 + 4 * quad, V);
  }
  cumsum_rows<4>(g, wtot);
  const int lane = tid & 63, w = tid >> 6, r = lane & 15, gq = lane >> 4;
  const f32x4 tot = ref4(&wtot[w][4 * quad]);
  const f32x4 far = rev ? between(wtot, -1, w, 4 * quad) : between(wtot, w, 4, 4 * quad);   // the other blocks' share
#pragma unroll
  for (int m = 0; m < 4; ++m) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      x[m][e] *= rev ? a.scale * ex2c(g[m][e] + far[e]) : ex2c((tot[e] - g[m][e]) + far[e]);
    put4(sX, r0 + m, 4 * quad, x[m]);
    put4(sY, r0 + m, 4 * quad, y[m]);
  }
  const int64_t sl = slot * a.H + h;
  if (vg == 0 && tid < 64)
    (rev ? a.ed : a.eh)[sl * 64 + tid] = ex2c(((wtot[0][tid] + wtot[1][tid]) + wtot[2][tid]) + wtot[3][tid]);
  __syncthreads();
  f32x4 acc[4] = {};
#pragma unroll 4
  for (int s = 0; s < 16; ++s) {
    const int row = 16 * (s >> 2) + 4 * gq + (s & 3);
    const float xv = sX[tix(row, 16 * w + r)];
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = mfma4(sY[tix(row, 16 * c + r)], xv, acc[c]);
  }
  float *out = (rev ? a.sd : a.sh) + (sl * a.nvg + vg) * 4096 + (16 * w + r) * 64 + 4 * gq;
#pragma unroll
  for (int c = 0; c < 4; ++c) *reinterpret_cast<f32x4 *>(out + 16 * c) = acc[c];
}

// Entering states (blockIdx.y 0) or leaving state gradients (1) from the
// chunks' own contributions, in place; 4 values per thread, kPre chunks per
// round trip.  Four workgroups per (sequence, head, value group).
constexpr int kPre = 8;
__global__ __launch_bounds__(256) void f32_prefix_kernel(F32Args a) {
  const bool rev = blockIdx.y;
  const int part = static_cast<int>(blockIdx.x & 3);
  const int vg = static_cast<int>((blockIdx.x >> 2) % a.nvg);
  const int h = static_cast<int>((blockIdx.x >> 2) / a.nvg % a.H);
  const int n = static_cast<int>((blockIdx.x >> 2) / a.nvg / a.H);
  int64_t bos, eos;
  seq_bounds(a.cu, n, a.T, bos, eos);
  const int64_t nch = (eos - bos + kC - 1) / kC;
  const int e = part * 1024 + 4 * static_cast<int>(threadIdx.x), key = e >> 6, c = 64 * vg + (e & 63);
  const int64_t sb = ((static_cast<int64_t>(n) * a.H + h) * a.K + key) * a.V + c;
  const float *init = rev ? a.dht : a.h0;
  float *fin = rev ? a.dh0 : a.ht;
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  if (init && key < a.K) {
#pragma unroll
    for (int m = 0; m < 4; ++m)
      if (c + m < a.V) S[m] = init[sb + m];
  }
  const int64_t s0 = bos / kC + n;
  float *st = rev ? a.sd : a.sh;
  const float *dec = rev ? a.ed : a.eh;
  for (int64_t i0 = 0; i0 < nch; i0 += kPre) {
    f32x4 L[kPre];
    float d[kPre];
    float *p[kPre];
#pragma unroll
    for (int u = 0; u < kPre; ++u) {
      const int64_t i = min(i0 + u, nch - 1);
      const int64_t sl = min(s0 + (rev ? nch - 1 - i : i), a.n_slots - 1) * a.H + h;
      p[u] = st + (sl * a.nvg + vg) * 4096 + e;
      L[u] = *reinterpret_cast<const f32x4 *>(p[u]);
      d[u] = dec[sl * 64 + key];
    }
#pragma unroll
    for (int u = 0; u < kPre; ++u) {
      if (i0 + u < nch) {
        *reinterpret_cast<f32x4 *>(p[u]) = S;
        S = d[u] * S + L[u];
      }
    }
  }
  if (fin && key < a.K) {
#pragma unroll
    for (int m = 0; m < 4; ++m)
      if (c + m < a.V) fin[sb + m] = S[m];
  }
}

// Largest magnitude of the values (NaN if one is), and the smallest but zero
// as twice its bits less one (a zero gives the largest number).
struct Magnitudes {
  float most = 0.f;
  uint32_t least = 0xffffffffu;
  template <int RPT, bool LEAST>
  __device__ __forceinline__ void add(const f32x4 (&x)[RPT]) {
#pragma unroll
    for (int m = 0; m < RPT; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float f = x[m][e];   // (a bit cast of the element itself reads element 0)
        most = __builtin_elementwise_maximum(most, fabsf(f));
        if (LEAST) least = min(least, (__builtin_bit_cast(uint32_t, f) << 1) - 1);
      }
  }
};

// q~ / k~ of the thread's rows into their tiles; sets *slow where one of them
// (`most`: or another operand's largest magnitude) leaves the range of the
// matrix-core diagonal.
template <int RPT>
__device__ __forceinline__ void stage_tilde(const f32x4 (&q)[RPT], const f32x4 (&k)[RPT], const f32x4 (&g)[RPT],
                                            const float (*sS)[64], const float (*sE)[64], int r0, int quad, float *tq,
                                            float *tk, float most, int *slow) {
  const int B = r0 >> 4;
  const f32x4 S = ref4(&sS[B][4 * quad]), E = ref4(&sE[B][4 * quad]);
  Magnitudes qk;
  qk.add<RPT, true>(q);
  qk.add<RPT, true>(k);
  // (a NaN fails either comparison)
  bool out = !(most < __builtin_inff()) | !(qk.most <= kInputMax) | (qk.least < 2 * kInputMin - 1);
#pragma unroll
  for (int m = 0; m < RPT; ++m) {
    f32x4 a, b;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float d = g[m][e] - S[e];
      out |= !(fabsf(d) <= kDiagRange);
      a[e] = q[m][e] * ex2c(d);
      b[e] = k[m][e] * ex2c(E[e] - g[m][e]);
    }
    put4(tq, r0 + m, 4 * quad, a);
    put4(tk, r0 + m, 4 * quad, b);
  }
  if (out) *slow = 1;
}

// The block references S (first row) and E (last row) of the thread's rows.
template <int RPT>
__device__ __forceinline__ void stage_refs(const f32x4 (&g)[RPT], int r0, int quad, float (*sS)[64], float (*sE)[64]) {
  if ((r0 & 15) == 0) *reinterpret_cast<f32x4 *>(&sS[r0 >> 4][4 * quad]) = g[0];
  if ((r0 & 15) == 16 - RPT) *reinterpret_cast<f32x4 *>(&sE[r0 >> 4][4 * quad]) = g[RPT - 1];
}

// 2^x of 4 keys.
__device__ __forceinline__ f32x4 exp4(const f32x4 &x) {
  f32x4 y;
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = ex2c(x[e]);
  return y;
}

// One block pair's term-by-term sums sum_k q_ik k_jk 2^(G_i - G_j) as
// D[4gq + x][r] with row index `row` of q (i) and column index of k (j) when
// QROWS, or j and i when not; terms j > i are zero.
template <bool QROWS>
__device__ __forceinline__ f32x4 diag_terms(const float *tq, const float *tk, const float *tg, int B, int gq, int r,
                                            int K) {
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int x = 0; x < 4; ++x) {
    const int i = 16 * B + (QROWS ? 4 * gq + x : r), j = 16 * B + (QROWS ? r : 4 * gq + x);
    float acc = 0.f;
    if (j <= i) {
#pragma unroll 1
      for (int kk = 0; kk < K; kk += 4) {
        const f32x4 qv = row4(tq, i, kk), kv = row4(tk, j, kk), gi = row4(tg, i, kk), gj = row4(tg, j, kk);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = fmaf(qv[e] * kv[e], ex2c(gi[e] - gj[e]), acc);
      }
    }
    if (x == 0) s[0] = acc;
    if (x == 1) s[1] = acc;
    if (x == 2) s[2] = acc;
    if (x == 3) s[3] = acc;
  }
  return s;
}

// o of one chunk: one workgroup per (slot, head, value group), wavefront I
// the rows 16I ..; 66 KB of LDS, two workgroups per CU.
template <bool VEC>
__global__ __launch_bounds__(256, 2) void f32_out_kernel(F32Args a) {
  __shared__ __attribute__((aligned(16))) float tQ[4096], tK[4096], tV[4096], tS[4096];
  __shared__ __attribute__((aligned(16))) float wtot[4][64], sS[4][64], sE[4][64];
  __shared__ int slow;
  const int vg = static_cast<int>(blockIdx.x % a.nvg);
  const int h = static_cast<int>(blockIdx.x / a.nvg % a.H);
  const int64_t slot = blockIdx.x / a.nvg / a.H;
  ChunkAt at;
  if (!chunk_of_slot(a.cu, a.n_seq, a.T, slot, at)) return;
  const int tid = threadIdx.x, quad = tid & 15, r0 = (tid >> 4) * 4, K = a.K, V = a.V, v0 = 64 * vg;
  const float *st = a.sh + ((slot * a.H + h) * a.nvg + vg) * 4096;
  f32x4 q[4], k[4], g[4], v[4], s[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const bool ok = r0 + m < at.nc;
    const int64_t row = (at.t0 + r0 + m) * a.H + h;
    g[m] = load4<VEC>(a.g + row * K, ok, 4 * quad, K);
    q[m] = load4<VEC>(a.q + row * K, ok, 4 * quad, K);
    k[m] = load4<VEC>(a.k + row * K, ok, 4 * quad, K);
    v[m] = load4<VEC>(a.v + row * V, ok, v0 + 4 * quad, V);
    s[m] = ref4(st + (r0 + m) * 64 + 4 * quad);
  }
  if (tid == 0) slow = 0;
  Magnitudes of;
  of.add<4, false>(v);
  cumsum_rows<4>(g, wtot);
  stage_refs<4>(g, r0, quad, sS, sE);
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    put4(tV, r0 + m, 4 * quad, v[m]);
    put4(tS, r0 + m, 4 * quad, s[m]);
  }
  __syncthreads();
  stage_tilde<4>(q, k, g, sS, sE, r0, quad, tQ, tK, of.most, &slow);
  __syncthreads();
  const int lane = tid & 63, I = tid >> 6, r = lane & 15, gq = lane >> 4;
  const bool diag = !slow;
  f32x4 acc[4] = {};
  f32x4 qr[4];   // q~ of row 16 I + r, keys 16 t + 4 gq ..
#pragma unroll
  for (int t = 0; t < 4; ++t) qr[t] = row4(tQ, 16 * I + r, 16 * t + 4 * gq);
  // q 2^G against the entering state
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const f32x4 S = ref4(&sS[I][16 * t + 4 * gq]) + between(sE, -1, I, 16 * t + 4 * gq);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float qg = qr[t][e] * ex2c(S[e]);
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[c] = mfma4(tS[tix(16 * t + 4 * gq + e, 16 * c + r)], qg, acc[c]);
    }
  }
  for (int J = 0; J <= I; ++J) {
    if (J == I && !diag) break;
    f32x4 p = {0.f, 0.f, 0.f, 0.f};   // A[i = r][j = 4 gq + x]
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int kc = 16 * t + 4 * gq;
      const f32x4 S = ref4(&sS[I][kc]);
      const f32x4 f = qr[t] * exp4(J == I ? S - ref4(&sE[I][kc]) : S + between(sE, J, I, kc));   // 2^(S_I - E_J)
      const f32x4 kr = row4(tK, 16 * J + r, 16 * t + 4 * gq);
#pragma unroll
      for (int e = 0; e < 4; ++e) p = mfma4(kr[e], f[e], p);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const float pv = (J < I || 4 * gq + x <= r) ? p[x] : 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[c] = mfma4(tV[tix(16 * J + 4 * gq + x, 16 * c + r)], pv, acc[c]);
    }
  }
  if (!diag) {   // the diagonal blocks term by term, from raw q, k and G (in the state's tile)
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const bool ok = r0 + m < at.nc;
      const int64_t row = (at.t0 + r0 + m) * a.H + h;
      q[m] = load4<VEC>(a.q + row * K, ok, 4 * quad, K);
      k[m] = load4<VEC>(a.k + row * K, ok, 4 * quad, K);
      g[m] = load4<VEC>(a.g + row * K, ok, 4 * quad, K);
    }
    cumsum_rows<4>(g, wtot);   // its barrier also ends the products above
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      put4(tQ, r0 + m, 4 * quad, q[m]);
      put4(tK, r0 + m, 4 * quad, k[m]);
      put4(tS, r0 + m, 4 * quad, g[m]);
    }
    __syncthreads();
    const f32x4 p = diag_terms<false>(tQ, tK, tS, I, gq, r, K);   // A[i = r][j = 4 gq + x]
#pragma unroll 1
    for (int jg = 0; jg < 4; ++jg)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float aij = __shfl(p[x], 16 * jg + r);
        if (4 * jg + x > r) continue;   // later rows are left out, not multiplied by zero
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] += aij * row4(tV, 16 * I + 4 * jg + x, 16 * c + 4 * gq);
      }
  }
  if (16 * I + r < at.nc) {
    float *o = a.o + ((at.t0 + 16 * I + r) * a.H + h) * V;
#pragma unroll
    for (int c = 0; c < 4; ++c) store4<VEC>(o, v0 + 16 * c + 4 * gq, V, acc[c] * a.scale);
  }
}

// Reverse inclusive scan over the 16 lanes of each DPP row.
template <int N>
__device__ __forceinline__ float row_shl(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
      0, __builtin_bit_cast(int, x), 0x100 + N, 0xf, 0xf, true));
}
__device__ __forceinline__ float row_suffix_scan(float x) {
  x += row_shl<1>(x);
  x += row_shl<2>(x);
  x += row_shl<4>(x);
  x += row_shl<8>(x);
  return x;
}

// dq, dk, dv, dg of one chunk: one workgroup of 8 wavefronts per (slot,
// head); wavefront (I, P) the rows 16 I .. and the key / value tiles 2P,
// 2P + 1.  Seven tiles: 128 KB of LDS, one workgroup per CU.  Results are
// formed transposed (D[key][row]) so that a lane holds 4 consecutive keys of
// one row, and the scans of dg over rows run across 16 lanes.
constexpr int kGradThreads = 512;
struct GradLds {
  float tQ[4096], tK[4096], tV[4096], tO[4096], tH[4096], tD[4096], tG[4096];
  float sDA[4][2][16][17];          // dA of the diagonal blocks (term by term), one copy per wavefront
  float wtot[8][64], sS[4][64], sE[4][64], sDgH[64], totT[4][64], totG[4][64];
  int slow;
};
template <bool VEC>
__global__ __launch_bounds__(kGradThreads) void f32_grad_kernel(F32Args a) {
  __shared__ __attribute__((aligned(16))) GradLds L;
  const int h = static_cast<int>(blockIdx.x % a.H);
  const int64_t slot = blockIdx.x / a.H;
  ChunkAt at;
  if (!chunk_of_slot(a.cu, a.n_seq, a.T, slot, at)) return;
  const int tid = threadIdx.x, quad = tid & 15, r0 = (tid >> 4) * 2, K = a.K, V = a.V;
  const float *sh = a.sh + (slot * a.H + h) * 4096, *sd = a.sd + (slot * a.H + h) * 4096;
  {
    f32x4 q[2], k[2], g[2], v[2], d[2], hs[2], dh[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const bool ok = r0 + m < at.nc;
      const int64_t row = (at.t0 + r0 + m) * a.H + h;
      g[m] = load4<VEC>(a.g + row * K, ok, 4 * quad, K);
      q[m] = load4<VEC>(a.q + row * K, ok, 4 * quad, K);
      k[m] = load4<VEC>(a.k + row * K, ok, 4 * quad, K);
      v[m] = load4<VEC>(a.v + row * V, ok, 4 * quad, V);
      d[m] = load4<VEC>(a.dO + row * V, ok, 4 * quad, V);
      hs[m] = ref4(sh + (r0 + m) * 64 + 4 * quad);
      dh[m] = ref4(sd + (r0 + m) * 64 + 4 * quad);
    }
    if (tid == 0) L.slow = 0;
    Magnitudes of;
    of.add<2, false>(v);
    of.add<2, false>(d);
    cumsum_rows<2>(g, L.wtot);
    stage_refs<2>(g, r0, quad, L.sS, L.sE);
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      put4(L.tV, r0 + m, 4 * quad, v[m]);
      put4(L.tO, r0 + m, 4 * quad, d[m]);
      put4(L.tH, r0 + m, 4 * quad, hs[m]);
      put4(L.tD, r0 + m, 4 * quad, dh[m]);
      put4(L.tG, r0 + m, 4 * quad, g[m]);
      // sum over the values of dh h, per key (row of the state)
      float s = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) s = fmaf(hs[m][e], dh[m][e], s);
      s = row_inclusive_scan(s);
      if (quad == 15) L.sDgH[r0 + m] = s;
    }
    __syncthreads();
    stage_tilde<2>(q, k, g, L.sS, L.sE, r0, quad, L.tQ, L.tK, of.most, &L.slow);
  }
  const int lane = tid & 63, w = tid >> 6, I = w >> 1, P = w & 1, r = lane & 15, gq = lane >> 4;
  const int i0 = 16 * I + r;                       // this lane's row
  const bool in = i0 < at.nc;
  const int64_t grow = (at.t0 + i0) * a.H + h;
  f32x4 qv[2], kv[2];                              // raw q, k of the row at this lane's keys
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    qv[c] = load4<VEC>(a.q + grow * K, in, 32 * P + 16 * c + 4 * gq, K);
    kv[c] = load4<VEC>(a.k + grow * K, in, 32 * P + 16 * c + 4 * gq, K);
  }
  __syncthreads();
  const bool diag = !L.slow;
  f32x4 Gr[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) Gr[c] = row4(L.tG, i0, 32 * P + 16 * c + 4 * gq);
  f32x4 dor[4], vr[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    dor[t] = row4(L.tO, i0, 16 * t + 4 * gq);
    vr[t] = row4(L.tV, i0, 16 * t + 4 * gq);
  }
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 pq[2] = {zero, zero}, pk[2] = {zero, zero}, ov[2] = {zero, zero};   // dO h^T, v dh^T, k_d dh
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const f32x4 kd = row4(L.tK, i0, 16 * t + 4 * gq) * exp4(between(L.sE, I, 4, 16 * t + 4 * gq));
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int c0 = 32 * P + 16 * c;
      const f32x4 hr = row4(L.tH, c0 + r, 16 * t + 4 * gq), dr = row4(L.tD, c0 + r, 16 * t + 4 * gq);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        pq[c] = mfma4(hr[e], dor[t][e], pq[c]);
        pk[c] = mfma4(dr[e], vr[t][e], pk[c]);
        ov[c] = mfma4(L.tD[tix(16 * t + 4 * gq + e, c0 + r)], kd[e], ov[c]);
      }
    }
  }
  float dii = 0.f;                                    // dA_ii of this lane's row
  auto own_diag = [&](const f32x4 &da) {              // D[r][r] sits in lane 16 (r / 4) + r, element r % 4
    const float x = (r & 2) ? ((r & 1) ? da[3] : da[2]) : ((r & 1) ? da[1] : da[0]);
    return __shfl(x, 16 * (r >> 2) + r);
  };
  f32x4 rq[2] = {zero, zero}, rk[2] = {zero, zero};   // intra-chunk parts of dq, dk (no diagonal, no scale)
  // The pair (i, j) enters dq_i and dk_j with the same three factors,
  // 2^(G_i - S_I) 2^(S_I - E_J) 2^(E_J - G_j): what each adds to dG then cancels
  // but for the products' rounding (dg 1.2e-6 -> 0.7e-6 off fp64 at strong
  // gates against other splits of the exponent in dq and in dk).
  f32x4 fi[2], fj[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int kc = 32 * P + 16 * c + 4 * gq;
    fi[c] = exp4(Gr[c] - ref4(&L.sS[I][kc]));
    fj[c] = exp4(ref4(&L.sE[I][kc]) - Gr[c]);
  }
  for (int J = 0; J <= I; ++J) {                      // dq: earlier rows j
    if (J == I && !diag) break;
    f32x4 da = zero;                                  // dA[i = r][j = 4 gq + x]
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const f32x4 vj = row4(L.tV, 16 * J + r, 16 * t + 4 * gq);
#pragma unroll
      for (int e = 0; e < 4; ++e) da = mfma4(vj[e], dor[t][e], da);
    }
    if (J == I) {
      dii = own_diag(da);
#pragma unroll
      for (int x = 0; x < 4; ++x)
        if (4 * gq + x >= r) da[x] = 0.f;
    }
    f32x4 part[2] = {zero, zero};
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        part[c] = mfma4(L.tK[tix(16 * J + 4 * gq + x, 32 * P + 16 * c + r)], da[x], part[c]);
#pragma unroll
    for (int c = 0; c < 2; ++c) {   // 2^(G_i - S_I) 2^(S_I - E_J)
      const int kc = 32 * P + 16 * c + 4 * gq;
      const f32x4 S = ref4(&L.sS[I][kc]);
      rq[c] += (fi[c] * exp4(J == I ? S - ref4(&L.sE[I][kc]) : S + between(L.sE, J, I, kc))) * part[c];
    }
  }
  for (int B = I; B < 4; ++B) {                       // dk, dv: later rows i of block B
    if (B == I && !diag) continue;
    f32x4 da = zero, A = zero;                        // dA, A [i = 4 gq + x][j = r]
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const f32x4 oi = row4(L.tO, 16 * B + r, 16 * t + 4 * gq), qi = row4(L.tQ, 16 * B + r, 16 * t + 4 * gq);
      const int kc = 16 * t + 4 * gq;
      const f32x4 S = ref4(&L.sS[B][kc]);
      const f32x4 kf =
          row4(L.tK, i0, kc) * exp4(B == I ? S - ref4(&L.sE[I][kc]) : S + between(L.sE, I, B, kc));   // 2^(S_B - E_I)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        da = mfma4(oi[e], vr[t][e], da);
        A = mfma4(qi[e], kf[e], A);
      }
    }
    f32x4 part[2] = {zero, zero};
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const float d = (B > I || 4 * gq + x > r) ? da[x] : 0.f;
      const float s = (B > I || 4 * gq + x >= r) ? A[x] * a.scale : 0.f;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int at_ = tix(16 * B + 4 * gq + x, 32 * P + 16 * c + r);
        part[c] = mfma4(L.tQ[at_], d, part[c]);
        ov[c] = mfma4(L.tO[at_], s, ov[c]);
      }
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {   // 2^(E_I - G_j) 2^(S_B - E_I)
      const int kc = 32 * P + 16 * c + 4 * gq;
      const f32x4 S = ref4(&L.sS[B][kc]);
      rk[c] += (fj[c] * exp4(B == I ? S - ref4(&L.sE[I][kc]) : S + between(L.sE, I, B, kc))) * part[c];
    }
  }
  if (!diag) {
    __syncthreads();   // q~ and k~ are read: raw q, k take their place
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const bool ok = r0 + m < at.nc;
      const int64_t row = (at.t0 + r0 + m) * a.H + h;
      put4(L.tQ, r0 + m, 4 * quad, load4<VEC>(a.q + row * K, ok, 4 * quad, K));
      put4(L.tK, r0 + m, 4 * quad, load4<VEC>(a.k + row * K, ok, 4 * quad, K));
    }
    f32x4 da = zero;   // dA[i = 4 gq + x][j = r]
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) da = mfma4(dor[t][e], vr[t][e], da);
    dii = own_diag(da);
#pragma unroll
    for (int x = 0; x < 4; ++x) L.sDA[I][P][4 * gq + x][r] = da[x];
    __syncthreads();
    const f32x4 A = diag_terms<true>(L.tQ, L.tK, L.tG, I, gq, r, K);   // A[i = 4 gq + x][j = r]
#pragma unroll 1
    for (int ig = 0; ig < 4; ++ig)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float aij = __shfl(A[x], 16 * ig + r) * a.scale;
        if (4 * ig + x < r) continue;   // earlier rows are left out, not multiplied by zero
#pragma unroll
        for (int c = 0; c < 2; ++c) ov[c] += aij * row4(L.tO, 16 * I + 4 * ig + x, 32 * P + 16 * c + 4 * gq);
      }
#pragma unroll 1
    for (int j = 0; j < 16; ++j) {
      const int row = 16 * I + j;
      const float dij = j < r ? L.sDA[I][P][r][j] : 0.f, dji = j > r ? L.sDA[I][P][j][r] : 0.f;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int kc = 32 * P + 16 * c + 4 * gq;
        const f32x4 qj = row4(L.tQ, row, kc), kj = row4(L.tK, row, kc), gj = row4(L.tG, row, kc);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (j < r) rq[c][e] = fmaf(dij * kj[e], ex2c(Gr[c][e] - gj[e]), rq[c][e]);
          if (j > r) rk[c][e] = fmaf(dji * qj[e], ex2c(gj[e] - Gr[c][e]), rk[c][e]);
        }
      }
    }
  }
  // dv of the row: values 32 P + 16 c + 4 gq ..
  if (in) {
#pragma unroll
    for (int c = 0; c < 2; ++c) store4<VEC>(a.dv + grow * V, 32 * P + 16 * c + 4 * gq, V, ov[c]);
  }
  // dq, dk; dG and the state term of dk with their scans over the rows
  f32x4 pre[2], suf[2], eg[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int kc = 32 * P + 16 * c + 4 * gq;
    // 2^G and 2^(gamma - G) of the row, from the start and to the end of the chunk
    const f32x4 eG = exp4(Gr[c] + between(L.sE, -1, I, kc));
    const f32x4 eE = exp4((ref4(&L.sE[I][kc]) - Gr[c]) + between(L.sE, I, 4, kc));
    f32x4 dqv, dkv;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float part = fmaf(eG[e], pq[c][e], rq[c][e]);
      dqv[e] = a.scale * fmaf(dii, kv[c][e], part);
      dkv[e] = fmaf(eE[e], pk[c][e], a.scale * fmaf(dii, qv[c][e], rk[c][e]));
      const float dG = qv[c][e] * (a.scale * part) - kv[c][e] * (a.scale * rk[c][e]);
      const float tdk = kv[c][e] * eE[e] * pk[c][e];
      const float ps = row_inclusive_scan(tdk);
      pre[c][e] = row_shr<1>(ps);
      suf[c][e] = row_suffix_scan(dG);
      eg[c][e] = ps;
    }
    if (r == 15) *reinterpret_cast<f32x4 *>(&L.totT[I][kc]) = eg[c];
    if (r == 0) *reinterpret_cast<f32x4 *>(&L.totG[I][kc]) = suf[c];
    if (in) {
      store4<VEC>(a.dq + grow * K, kc, K, dqv);
      store4<VEC>(a.dk + grow * K, kc, K, dkv);
    }
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int kc = 32 * P + 16 * c + 4 * gq;
    f32x4 x = ref4(&L.sDgH[kc]) * exp4(between(L.sE, -1, 4, kc)) + (pre[c] + suf[c]);
    for (int B = 0; B < 4; ++B) {
      if (B < I) x += ref4(&L.totT[B][kc]);
      if (B > I) x += ref4(&L.totG[B][kc]);
    }
    if (in) store4<VEC>(a.dg + grow * K, kc, K, x);
  }
}

inline int64_t f32_slots(int n_seq, int64_t T) { return T / kC + n_seq + 1; }
constexpr size_t kF32Align = 16;

}  // namespace
}  // namespace ssla

extern "C" int ssla_gla_chunk_f32_fwd(const float *q, const float *k, const float *v, const float *g,
                                      const int64_t *cu_seqlens, int n_seq, int64_t T, int H, int K, int V,
                                      float scale, const float *h0, float *o, float *ht, void *stream) {
  using namespace ssla;
  clear_error();
  SSLA_CHECK_ARG(n_seq >= 0 && T >= 0 && H > 0 && K > 0 && V > 0,
                 "gla_chunk_f32_fwd: bad sizes n_seq=%d T=%lld H=%d K=%d V=%d", n_seq, (long long)T, H, K, V);
  if (K > 64 || V > 256) {
    set_error("gla_chunk_f32_fwd: K=%d V=%d (K <= 64 and V <= 256 per call)", K, V);
    return SSLA_ERR_UNSUPPORTED;
  }
  if (n_seq == 0) return SSLA_OK;
  SSLA_CHECK_ARG(cu_seqlens && (T == 0 || (q && k && v && g && o)), "gla_chunk_f32_fwd: null pointer");
  const int nvt = (V + kVT - 1) / kVT;
  const int64_t blocks = static_cast<int64_t>(n_seq) * H * nvt;
  SSLA_CHECK_ARG(blocks < 0x7fffffff, "gla_chunk_f32_fwd: too many (sequence, head, tile) items");
  hipLaunchKernelGGL(f32_fwd_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0,
                     static_cast<hipStream_t>(stream), q, k, v, g, cu_seqlens, n_seq, T, H, K, V, scale, h0, o, ht);
  return launch_status("gla_chunk_f32_fwd");
}

extern "C" size_t ssla_gla_chunk_f32_fwd_workspace_size(int n_seq, int64_t T, int H, int K, int V) {
  if (n_seq < 0 || T < 0 || H <= 0 || K <= 0 || V <= 0) return 0;
  const size_t items = static_cast<size_t>(ssla::f32_slots(n_seq, T)) * H;
  return items * (64 + static_cast<size_t>((V + 63) / 64) * 4096) * sizeof(float) + ssla::kF32Align;
}

extern "C" int ssla_gla_chunk_f32_fwd_ws(const float *q, const float *k, const float *v, const float *g,
                                         const int64_t *cu_seqlens, int n_seq, int64_t T, int H, int K, int V,
                                         float scale, const float *h0, float *o, float *ht, void *workspace,
                                         size_t workspace_bytes, void *stream) {
  using namespace ssla;
  clear_error();
  SSLA_CHECK_ARG(n_seq >= 0 && T >= 0 && H > 0 && K > 0 && V > 0,
                 "gla_chunk_f32_fwd: bad sizes n_seq=%d T=%lld H=%d K=%d V=%d", n_seq, (long long)T, H, K, V);
  if (K > 64 || V > 256) {
    set_error("gla_chunk_f32_fwd: K=%d V=%d (K <= 64 and V <= 256 per call)", K, V);
    return SSLA_ERR_UNSUPPORTED;
  }
  if (n_seq == 0) return SSLA_OK;
  SSLA_CHECK_ARG(cu_seqlens && (T == 0 || (q && k && v && g && o)), "gla_chunk_f32_fwd: null pointer");
  const size_t need = ssla_gla_chunk_f32_fwd_workspace_size(n_seq, T, H, K, V);
  if (workspace == nullptr || workspace_bytes < need) {
    set_error("gla_chunk_f32_fwd: workspace of %zu bytes needed, %zu given", need, workspace_bytes);
    return SSLA_ERR_WORKSPACE;
  }
  F32Args a = {};
  a.q = q, a.k = k, a.v = v, a.g = g, a.h0 = h0, a.cu = cu_seqlens, a.o = o, a.ht = ht;
  a.T = T, a.n_slots = f32_slots(n_seq, T), a.n_seq = n_seq, a.H = H, a.K = K, a.V = V, a.nvg = (V + 63) / 64;
  a.scale = scale;
  a.sh = reinterpret_cast<float *>((reinterpret_cast<uintptr_t>(workspace) + kF32Align - 1) / kF32Align * kF32Align);
  a.eh = a.sh + static_cast<size_t>(a.n_slots) * H * a.nvg * 4096;
  const int64_t chunks = a.n_slots * H * a.nvg, seqs = static_cast<int64_t>(n_seq) * H * a.nvg * 4;
  SSLA_CHECK_ARG(chunks < 0x7fffffff && seqs < 0x7fffffff, "gla_chunk_f32_fwd: too many (chunk, head, tile) items");
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const bool vec = K % 4 == 0 && V % 4 == 0 && aligned(q, 16) && aligned(k, 16) && aligned(v, 16) && aligned(g, 16) &&
                   aligned(o, 16);
  const dim3 gc(static_cast<unsigned>(chunks));
  if (T > 0) {
    if (vec)
      hipLaunchKernelGGL(f32_states_kernel<true>, gc, dim3(256), 0, s, a, ht != nullptr, 0);
    else
      hipLaunchKernelGGL(f32_states_kernel<false>, gc, dim3(256), 0, s, a, ht != nullptr, 0);
  }
  hipLaunchKernelGGL(f32_prefix_kernel, dim3(static_cast<unsigned>(seqs)), dim3(256), 0, s, a);
  if (T > 0) {
    if (vec)
      hipLaunchKernelGGL(f32_out_kernel<true>, gc, dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL(f32_out_kernel<false>, gc, dim3(256), 0, s, a);
  }
  return launch_status("gla_chunk_f32_fwd");
}

extern "C" size_t ssla_gla_chunk_f32_bwd_workspace_size(int n_seq, int64_t T, int H) {
  if (n_seq < 0 || T < 0 || H <= 0) return 0;
  return static_cast<size_t>(ssla::f32_slots(n_seq, T)) * H * 2 * (64 + 4096) * sizeof(float) + ssla::kF32Align;
}

extern "C" int ssla_gla_chunk_f32_bwd(const float *q, const float *k, const float *v, const float *g,
                                      const int64_t *cu_seqlens, int n_seq, int64_t T, int H, int K, int V,
                                      float scale, const float *h0, const float *do_, const float *dht, float *dq,
                                      float *dk, float *dv, float *dg, float *dh0, void *workspace,
                                      size_t workspace_bytes, void *stream) {
  using namespace ssla;
  clear_error();
  SSLA_CHECK_ARG(n_seq >= 0 && T >= 0 && H > 0 && K > 0 && V > 0,
                 "gla_chunk_f32_bwd: bad sizes n_seq=%d T=%lld H=%d K=%d V=%d", n_seq, (long long)T, H, K, V);
  if (K > 64 || V > 64) {
    set_error("gla_chunk_f32_bwd: K=%d V=%d (K, V <= 64 per call)", K, V);
    return SSLA_ERR_UNSUPPORTED;
  }
  if (n_seq == 0) return SSLA_OK;
  SSLA_CHECK_ARG(cu_seqlens && (T == 0 || (q && k && v && g && do_ && dq && dk && dv && dg)),
                 "gla_chunk_f32_bwd: null pointer");
  SSLA_CHECK_ARG(h0 == nullptr || dh0 != nullptr, "gla_chunk_f32_bwd: dh0 needed with an initial state");
  const size_t need = ssla_gla_chunk_f32_bwd_workspace_size(n_seq, T, H);
  if (workspace == nullptr || workspace_bytes < need) {
    set_error("gla_chunk_f32_bwd: workspace of %zu bytes needed, %zu given", need, workspace_bytes);
    return SSLA_ERR_WORKSPACE;
  }
  F32Args a = {};
  a.q = q, a.k = k, a.v = v, a.g = g, a.dO = do_, a.h0 = h0, a.dht = dht, a.cu = cu_seqlens;
  a.dq = dq, a.dk = dk, a.dv = dv, a.dg = dg, a.dh0 = dh0;
  a.T = T, a.n_slots = f32_slots(n_seq, T), a.n_seq = n_seq, a.H = H, a.K = K, a.V = V, a.nvg = 1, a.scale = scale;
  const size_t items = static_cast<size_t>(a.n_slots) * H;
  a.sh = reinterpret_cast<float *>((reinterpret_cast<uintptr_t>(workspace) + kF32Align - 1) / kF32Align * kF32Align);
  a.sd = a.sh + items * 4096;
  a.eh = a.sd + items * 4096;
  a.ed = a.eh + items * 64;
  const int64_t chunks = a.n_slots * H, seqs = static_cast<int64_t>(n_seq) * H * 4;
  SSLA_CHECK_ARG(chunks < 0x7fffffff && seqs < 0x7fffffff, "gla_chunk_f32_bwd: too many (chunk, head) items");
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const bool vec = K % 4 == 0 && V % 4 == 0 && aligned(q, 16) && aligned(k, 16) && aligned(v, 16) && aligned(g, 16) &&
                   aligned(do_, 16) && aligned(dq, 16) && aligned(dk, 16) && aligned(dv, 16) && aligned(dg, 16);
  const dim3 gs(static_cast<unsigned>(chunks), 2), gc(static_cast<unsigned>(chunks));
  if (T > 0) {
    if (vec)
      hipLaunchKernelGGL(f32_states_kernel<true>, gs, dim3(256), 0, s, a, 0, dh0 != nullptr);
    else
      hipLaunchKernelGGL(f32_states_kernel<false>, gs, dim3(256), 0, s, a, 0, dh0 != nullptr);
  }
  hipLaunchKernelGGL(f32_prefix_kernel, dim3(static_cast<unsigned>(seqs), 2), dim3(256), 0, s, a);
  if (T > 0) {
    if (vec)
      hipLaunchKernelGGL(f32_grad_kernel<true>, gc, dim3(kGradThreads), 0, s, a);
    else
      hipLaunchKernelGGL(f32_grad_kernel<false>, gc, dim3(kGradThreads), 0, s, a);
  }
  return launch_status("gla_chunk_f32_bwd");
}
