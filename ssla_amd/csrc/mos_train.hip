// Training form of the MosAttention layer (reference layers/mos_attention.py:
// 103-140 with _apply_scatter_proj / _apply_gather_proj, :148-167, and
// utils/async_utils.py:243-264): forward with what the backward needs kept,
// and the backward.  The layer's matrices come folded per kernel position a,
//   Wa[a] = [Wq; Wv; Wg] Ws[a]   [3H, Cin]        Wb[a] = Wgp[a] Wo   [H, H],
// so that every copy of event e at position a needs
//   (q, v, g) = Wa[a] x_e,  s = sigmoid(g),  h = s h_prev + v along its patch,
//   y = q h,                out_e = sum_a Wb[a] y_{e,a}  (+ Win x_e).
//
// All row tensors lie in (event, position) order, [E, A, .]: the projections
// and their gradients are then dense fp32 products over the events, with the
// sum over an event's copies inside the product's reduction -- no gathered
// event rows, no sort by position, no row sums afterwards -- and only the two
// scans walk the patches, through the patch rows' (event, position).  The
// composed forward and backward ran some 475 launches, with library products
// of 52k-long reductions into 48 x 48 results at 135-425 us each and 440 us
// per row sum: 11.6 ms for a training step of a 24 -> 48 layer on 52,000
// events (9 positions), 1.16 ms here.  The kernels are bound by their row
// traffic (468,000 rows of 48 channels): scans 113 and 153 us at 4 TB/s,
// projection 70, the wide weight gradient 95, d events 65 us.
//
// Copies that lie in no patch (frame borders) hold zeros in y and in the
// gradient rows, so the products may include them.
#include "common.h"

namespace ssla {
namespace {

__device__ __forceinline__ f32x4 mma(float a, float b, const f32x4 &c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <bool VEC>
__device__ __forceinline__ f32x4 ld4(const float *row, bool ok, int c, int C) {
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

// ------------------------------------------------------------- products --
// C[E, N] = A[E, K] B[N, K]^T, fp32 on v_mfma_f32_16x16x4_f32.  A workgroup
// takes 64 RT events and 16 NT columns, a wavefront 16 RT events and all the
// columns; A goes from global memory straight into the operand layout (lane
// 16 gq + r: event r, 4 consecutive k at 16 t + 4 gq), B is staged through LDS
// in pieces of 32 k with the next piece's loads in flight.  The product is
// formed transposed, so a lane holds 4 consecutive columns of one event.
// epi 1: columns n with n % period >= from become sigmoid(n) ; epi 2: C += .
constexpr int kPitch = 36;   // LDS row pitch of B: 16 rows' 16-byte reads fall on different banks
struct TallArgs {
  const float *A, *B;
  float *C;
  int64_t E;
  int lda, N, K, epi, period, from;
};
template <int RT, int NT, bool VEC>
__global__ __launch_bounds__(256) void mos_tall_gemm(TallArgs a) {
  __shared__ __attribute__((aligned(16))) float sB[2][16 * NT][kPitch];
  constexpr int BL = (NT * 128 + 255) / 256;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r = lane & 15, gq = lane >> 4;
  const int64_t e0 = static_cast<int64_t>(blockIdx.x) * (64 * RT) + 16 * RT * w;
  f32x4 acc[RT][NT] = {}, an[RT][2], bn[BL];
  // step (n0, kc): the pieces of one column block, then the next block
  int n0 = blockIdx.y * 16 * NT, kc = 0;
  const int dn = gridDim.y * 16 * NT;
  auto load = [&](int n1, int k1) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int64_t e = e0 + 16 * i + r;
        an[i][t] = ld4<VEC>(a.A + e * a.lda, e < a.E, k1 + 16 * t + 4 * gq, a.K);
      }
#pragma unroll
    for (int i = 0; i < BL; ++i) {
      const int id = tid + 256 * i, n = n1 + (id >> 3);
      bn[i] = ld4<VEC>(a.B + static_cast<int64_t>(n) * a.K, id < NT * 128 && n < a.N, k1 + 4 * (id & 7), a.K);
    }
  };
  if (n0 < a.N) load(n0, 0);
  for (int buf = 0; n0 < a.N; buf ^= 1) {
    f32x4 av[RT][2];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int t = 0; t < 2; ++t) av[i][t] = an[i][t];
#pragma unroll
    for (int i = 0; i < BL; ++i) {
      const int id = tid + 256 * i;
      if (id < NT * 128) *reinterpret_cast<f32x4 *>(&sB[buf][id >> 3][4 * (id & 7)]) = bn[i];
    }
    // this buffer was last read two steps ago, before the previous barrier
    __syncthreads();
    const bool last = kc + 32 >= a.K;
    const int n1 = last ? n0 + dn : n0, k1 = last ? 0 : kc + 32;
    if (n1 < a.N) load(n1, k1);
    // each piece sums from zero and is added whole: a reduction of 1,296
    // terms rounds like one of 41 + 8 (d events 5.0e-7 -> 2.0e-7 off fp64)
#pragma unroll
    for (int c = 0; c < NT; ++c) {
      f32x4 p[RT] = {};
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const f32x4 b = *reinterpret_cast<const f32x4 *>(&sB[buf][16 * c + r][16 * t + 4 * gq]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < RT; ++i) p[i] = mma(b[e], av[i][t][e], p[i]);
      }
#pragma unroll
      for (int i = 0; i < RT; ++i) acc[i][c] += p[i];
    }
    if (last) {
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const int64_t e = e0 + 16 * i + r;
        float *row = a.C + e * a.N;
#pragma unroll
        for (int c = 0; c < NT; ++c) {
          const int n = n0 + 16 * c + 4 * gq;
          f32x4 x = acc[i][c];
          acc[i][c] = (f32x4){0.f, 0.f, 0.f, 0.f};
          if (e >= a.E) continue;
          if (a.epi == 1) {
#pragma unroll
            for (int m = 0; m < 4; ++m)
              if ((n + m) % a.period >= a.from) x[m] = 1.f / (1.f + expf(-x[m]));
          }
          if (VEC) {
            if (n < a.N) {
              f32x4 *p = reinterpret_cast<f32x4 *>(row + n);
              if (a.epi == 2) x += *p;
              *p = x;
            }
          } else {
#pragma unroll
            for (int m = 0; m < 4; ++m)
              if (n + m < a.N) row[n + m] = a.epi == 2 ? row[n + m] + x[m] : x[m];
          }
        }
      }
    }
    n0 = n1;
    kc = k1;
  }
}

// part[s][M, N] = sum over the s-th slice of events of A[e, m] B[e, n] (the
// weight gradients: reductions of 1e4..1e6 events into small matrices, bound
// by reading B).  A wavefront takes all M rows, 64 columns and one slice;
// both operands come from global memory in the operand layout (4 events per
// step, one per lane group; lane r holds A's column 16 i + r and B's columns
// 4 r .. 4 r + 3, one per product), kStep steps in flight.
constexpr int kStep = 4;
template <int MT, bool VEC>
__global__ __launch_bounds__(256) void mos_wgrad(const float *__restrict__ A, const float *__restrict__ B, int64_t E,
                                                 int M, int N, int64_t slice, int n_slices, float *__restrict__ part) {
  const int lane = threadIdx.x & 63, r = lane & 15, gq = lane >> 4;
  const int s = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (s >= n_slices) return;
  const int n = blockIdx.x * 64 + 4 * r;
  const int64_t lo = s * slice, hi = min(lo + slice, E);
  f32x4 acc[MT][4] = {};
  for (int64_t e0 = lo; e0 < hi; e0 += 4 * kStep) {
    float av[kStep][MT];
    f32x4 bv[kStep];
#pragma unroll
    for (int u = 0; u < kStep; ++u) {
      const int64_t e = e0 + 4 * u + gq;
      const bool ok = e < hi;
      bv[u] = ld4<VEC>(B + e * N, ok, n, N);
#pragma unroll
      for (int i = 0; i < MT; ++i) av[u][i] = (ok && 16 * i + r < M) ? A[e * M + 16 * i + r] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < kStep; ++u)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = mma(av[u][i], bv[u][j], acc[i][j]);
  }
  float *out = part + static_cast<int64_t>(s) * M * N;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int m = 16 * i + 4 * gq + x;
      if (m >= M) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (n + j < N) out[static_cast<int64_t>(m) * N + n + j] = acc[i][j][x];
    }
}

// out[i] = sum over the slices of part[s][i], in slice order within each of
// 4 quarters (deterministic).
__global__ __launch_bounds__(256) void mos_wgrad_sum(const float *__restrict__ part, int n_slices, int64_t n,
                                                     float *__restrict__ out) {
  __shared__ float q[4][64];
  const int t = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 64 + t;
  const int per = (n_slices + 3) / 4, lo = w * per, hi = min(lo + per, n_slices);
  float acc = 0.f;
  if (i < n) {
    for (int s0 = lo; s0 < hi; s0 += 8) {
      float x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = s0 + u < hi ? part[(s0 + u) * n + i] : 0.f;
#pragma unroll
      for (int u = 0; u < 8; ++u) acc += x[u];
    }
  }
  q[w][t] = acc;
  __syncthreads();
  if (w == 0 && i < n) out[i] = ((q[0][t] + q[1][t]) + q[2][t]) + q[3][t];
}

// ---------------------------------------------------------------- scans --
// A wavefront holds `slots` patches side by side, `ch` lanes (at least
// kAhead, one channel each while c < H) per patch, channel block blockIdx.y,
// and walks them kAhead rows at a time.  A batch's row places are one
// coalesced load by the patch's lanes, handed round by lane reads; its values
// are in flight while the batch before is worked on, without branches (rows
// past the end read the last row again).
constexpr int kAhead = 8;
struct ScanArgs {
  const int64_t *src, *pos, *cu;   // patch rows: event and position; patch offsets [P + 1]
  int64_t P, R;
  int A, H, ch, slots;
};

// Workgroups are dealt to the 8 XCDs in turn: each XCD takes one contiguous
// eighth of the patches, so that the copies of one event (neighbouring
// patches, sharing cache lines) meet in one L2.
struct ScanAt {
  int64_t lo, hi;   // the patch's rows
  int c, j, l0;     // channel, lane within the patch's lanes, their first lane
};
__device__ __forceinline__ bool scan_place(const ScanArgs &a, ScanAt &p) {
  const int lane = threadIdx.x & 63, slot = lane / a.ch;
  const int64_t per = gridDim.x / 8, blk = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  const int64_t patch = (blk * 4 + (threadIdx.x >> 6)) * a.slots + slot;
  p.j = lane - slot * a.ch;
  p.l0 = slot * a.ch;
  p.c = blockIdx.y * a.ch + p.j;
  if (slot >= a.slots || patch >= a.P) return false;
  p.lo = min(max(a.cu[patch], (int64_t)0), a.R);
  p.hi = min(max(a.cu[patch + 1], p.lo), a.R);
  return p.lo < p.hi;
}
// Place (event * A + position) of row i0 + dir * j, clamped into the patch.
__device__ __forceinline__ int scan_row(const ScanArgs &a, const ScanAt &p, int64_t i) {
  i = min(max(i, p.lo), p.hi - 1);
  return static_cast<int>(a.src[i]) * a.A + static_cast<int>(a.pos[i]);
}

// In qvh [E, A, 3H]: h takes v's place; y [E, A, H] = q h; valid[e, a] = 1.
__global__ __launch_bounds__(256) void mos_scan_fwd(ScanArgs a, float *__restrict__ qvh, float *__restrict__ y,
                                                    unsigned char *__restrict__ valid) {
  ScanAt p;
  if (!scan_place(a, p)) return;
  const int H = a.H, c = min(p.c, H - 1);   // lanes past H read with it and write nothing
  const bool mine = p.c < H;
  int at[kAhead];
  float q[kAhead], v[kAhead], s[kAhead];
  auto values = [&](int rows) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      at[u] = __shfl(rows, p.l0 + u);
      const float *row = qvh + static_cast<int64_t>(at[u]) * 3 * H + c;
      q[u] = row[0];
      v[u] = row[H];
      s[u] = row[2 * H];
    }
  };
  values(scan_row(a, p, p.lo + p.j));
  int next = scan_row(a, p, p.lo + kAhead + p.j);
  float h = 0.f;
  for (int64_t i0 = p.lo; i0 < p.hi; i0 += kAhead) {
    float cq[kAhead], cv[kAhead], cs[kAhead];
    int ca[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) cq[u] = q[u], cv[u] = v[u], cs[u] = s[u], ca[u] = at[u];
    if (i0 + kAhead < p.hi) {
      values(next);
      next = scan_row(a, p, i0 + 2 * kAhead + p.j);
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      h = fmaf(cs[u], h, cv[u]);
      if (mine && i0 + u < p.hi) {
        qvh[static_cast<int64_t>(ca[u]) * 3 * H + H + c] = h;
        y[static_cast<int64_t>(ca[u]) * H + c] = cq[u] * h;
        if (c == 0) valid[ca[u]] = 1;
      }
    }
  }
}

// Reverse: dh = q dy + s_next dh_next; d [E, A, 3H] = (dy h, dh, dh h_prev s (1 - s)).
__global__ __launch_bounds__(256) void mos_scan_bwd(ScanArgs a, const float *__restrict__ qvh,
                                                    const float *__restrict__ dy, float *__restrict__ d) {
  ScanAt p;
  if (!scan_place(a, p)) return;
  const int H = a.H, c = min(p.c, H - 1);
  const bool mine = p.c < H;
  int at[kAhead];
  float q[kAhead], h[kAhead], s[kAhead], g[kAhead];
  auto values = [&](int rows) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      at[u] = __shfl(rows, p.l0 + u);
      const float *row = qvh + static_cast<int64_t>(at[u]) * 3 * H + c;
      q[u] = row[0];
      h[u] = row[H];
      s[u] = row[2 * H];
      g[u] = dy[static_cast<int64_t>(at[u]) * H + c];
    }
  };
  values(scan_row(a, p, p.hi - 1 - p.j));
  int next = scan_row(a, p, p.hi - 1 - kAhead - p.j);
  float carry = 0.f;   // s_next dh_next
  for (int64_t i0 = p.hi - 1; i0 >= p.lo; i0 -= kAhead) {
    float cq[kAhead], chh[kAhead + 1], cs[kAhead], cg[kAhead];
    int ca[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) cq[u] = q[u], chh[u] = h[u], cs[u] = s[u], cg[u] = g[u], ca[u] = at[u];
    if (i0 - kAhead >= p.lo) {
      values(next);
      next = scan_row(a, p, i0 - 2 * kAhead - p.j);
    }
    chh[kAhead] = h[0];   // h before the batch's last row: the next batch's first
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int64_t i = i0 - u;
      const float prev = i > p.lo ? chh[u + 1] : 0.f;
      const float dh = fmaf(cq[u], cg[u], carry);
      if (mine && i >= p.lo) {
        float *row = d + static_cast<int64_t>(ca[u]) * 3 * H + c;
        row[0] = cg[u] * chh[u];
        row[H] = dh;
        row[2 * H] = dh * prev * cs[u] * (1.f - cs[u]);
      }
      carry = cs[u] * dh;
    }
  }
}

// Zero the rows of the copies that lie in no patch.
__global__ __launch_bounds__(256) void mos_zero_rows(const unsigned char *__restrict__ valid, int64_t n, int W,
                                                     float *__restrict__ x) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n || valid[i]) return;
  for (int c = 0; c < W; ++c) x[i * W + c] = 0.f;
}

template <int RT, int NT>
void launch_tall(const TallArgs &a, bool vec, hipStream_t st) {
  // about 2048 workgroups, each with an equal share of the column blocks
  const int64_t gx = (a.E + 64 * RT - 1) / (64 * RT), blocks = (a.N + 16 * NT - 1) / (16 * NT);
  const int64_t per = std::max<int64_t>(1, gx * blocks / 2048);
  const dim3 grid(static_cast<unsigned>(gx), static_cast<unsigned>((blocks + per - 1) / per));
  if (vec)
    hipLaunchKernelGGL((mos_tall_gemm<RT, NT, true>), grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((mos_tall_gemm<RT, NT, false>), grid, dim3(256), 0, st, a);
}

void tall_gemm(const float *A, int lda, const float *B, float *C, int64_t E, int N, int K, int epi, int period,
               int from, hipStream_t st) {
  TallArgs a = {A, B, C, E, lda, N, K, epi, period, from};
  const bool vec = N % 4 == 0 && K % 4 == 0 && lda % 4 == 0 && aligned(A, 16) && aligned(B, 16) && aligned(C, 16);
  // up to 64 columns per workgroup, the widths the layers use without a ragged tile; 128 events per
  // workgroup where that still gives two per CU
  const int nt = N <= 16 ? 1 : N <= 32 ? 2 : N <= 48 ? 3 : (N % 48 == 0 && N % 64 != 0) ? 3 : 4;
  const bool two = (E + 127) / 128 * ((N + 16 * nt - 1) / (16 * nt)) >= 512;
  switch (nt) {
    case 1: two ? launch_tall<2, 1>(a, vec, st) : launch_tall<1, 1>(a, vec, st); break;
    case 2: two ? launch_tall<2, 2>(a, vec, st) : launch_tall<1, 2>(a, vec, st); break;
    case 3: two ? launch_tall<2, 3>(a, vec, st) : launch_tall<1, 3>(a, vec, st); break;
    default: two ? launch_tall<2, 4>(a, vec, st) : launch_tall<1, 4>(a, vec, st); break;
  }
}

// Slices of a weight gradient: about 2048 wavefronts, at least 64 events each.
inline int wgrad_slices(int64_t E, int N) {
  const int64_t groups = (N + 63) / 64;
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>((2048 + groups - 1) / groups, (E + 63) / 64)));
}

template <bool VEC>
void wgrad_launch(const float *A, const float *B, int64_t E, int M, int N, int64_t slice, int ns, float *part,
                  hipStream_t st) {
  const dim3 grid((N + 63) / 64, (ns + 3) / 4);
#define SSLA_WG(MT_)                                                                                             \
  case MT_:                                                                                                      \
    hipLaunchKernelGGL((mos_wgrad<MT_, VEC>), grid, dim3(256), 0, st, A, B, E, M, N, slice, ns, part);            \
    break
  switch ((M + 15) / 16) {
    SSLA_WG(1);
    SSLA_WG(2);
    SSLA_WG(3);
    SSLA_WG(4);
    SSLA_WG(5);
    SSLA_WG(6);
    SSLA_WG(7);
    SSLA_WG(8);
  }
#undef SSLA_WG
}

// out[M, N] = A[E, M]^T B[E, N] (M <= 128).
void wgrad(const float *A, const float *B, int64_t E, int M, int N, float *part, float *out, hipStream_t st) {
  const int ns = wgrad_slices(E, N);
  const int64_t slice = ((E + ns - 1) / ns + 3) / 4 * 4;
  if (N % 4 == 0 && aligned(B, 16))
    wgrad_launch<true>(A, B, E, M, N, slice, ns, part, st);
  else
    wgrad_launch<false>(A, B, E, M, N, slice, ns, part, st);
  const int64_t n = static_cast<int64_t>(M) * N;
  hipLaunchKernelGGL(mos_wgrad_sum, dim3(static_cast<unsigned>((n + 63) / 64)), dim3(256), 0, st, part, ns, n, out);
}

ScanArgs scan_args(const int64_t *src, const int64_t *pos, const int64_t *cu, int64_t P, int64_t R, int A, int H) {
  ScanArgs a = {src, pos, cu, P, R, A, H, 0, 0};
  const int blocks = (H + 63) / 64;
  a.ch = std::max((H + blocks - 1) / blocks, kAhead);
  a.slots = 64 / a.ch;
  return a;
}
dim3 scan_grid(const ScanArgs &a) {
  const int64_t per = 4 * a.slots;
  return dim3(static_cast<unsigned>((a.P + per - 1) / per + 7) / 8 * 8, (a.H + a.ch - 1) / a.ch);
}

size_t up16(size_t x) { return (x + 15) / 16 * 16; }

// ------------------------------------------------------------ layer norm --
// LayerNorm over the H <= 128 channels of a row and its backward, 16 lanes per
// row: lane j holds channels j, j + 16, ..., the row sums are lane rotations.
// A row is read once (the centred second moment is taken in registers), so
// both passes are bound by their rows: 52,000 x 48 forward 6 us and backward
// 8 + 7 us, where the library's took 53 us (a workgroup of one wavefront per row)
// and 81 us (the weight gradients alone 50).  A workgroup's rows are summed
// per lane for the weight gradients, then over its 16 row groups, then over
// the workgroups (norm_grad_sum): no atomics, the same bits every run.
constexpr int kNormBlocks = 1024;
template <int N>
__device__ __forceinline__ float ror16(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 + N, 0xf, 0xf, false));
}
__device__ __forceinline__ float sum16(float x) {
  x += ror16<8>(x);
  x += ror16<4>(x);
  x += ror16<2>(x);
  return x + ror16<1>(x);
}

template <int CPL>
__device__ __forceinline__ void row_ld(const float *p, int j, int H, float (&x)[CPL]) {
#pragma unroll
  for (int i = 0; i < CPL; ++i) x[i] = j + 16 * i < H ? p[j + 16 * i] : 0.f;
}

template <int CPL>
__global__ __launch_bounds__(256) void row_norm_fwd(const float *__restrict__ x, int64_t n, int H,
                                                    const float *__restrict__ w, const float *__restrict__ b, float eps,
                                                    float *__restrict__ y, float2 *__restrict__ stats) {
  const int j = threadIdx.x & 15;
  float wj[CPL], bj[CPL];
  row_ld(w, j, H, wj);
  row_ld(b, j, H, bj);
  for (int64_t r = static_cast<int64_t>(blockIdx.x) * 16 + (threadIdx.x >> 4); r < n;
       r += static_cast<int64_t>(gridDim.x) * 16) {
    float v[CPL], s = 0.f, m2 = 0.f;
    row_ld(x + r * H, j, H, v);
#pragma unroll
    for (int i = 0; i < CPL; ++i) s += v[i];
    const float mean = sum16(s) / H;
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
      v[i] -= mean;
      if (j + 16 * i < H) m2 = fmaf(v[i], v[i], m2);
    }
    const float rstd = 1.f / sqrtf(sum16(m2) / H + eps);
#pragma unroll
    for (int i = 0; i < CPL; ++i)
      if (j + 16 * i < H) y[r * H + j + 16 * i] = fmaf(v[i] * rstd, wj[i], bj[i]);
    if (j == 0) stats[r] = make_float2(mean, rstd);
  }
}

// part (nullable): [gridDim.x, 2, H], this workgroup's sums of dy xhat and dy.
template <int CPL>
__global__ __launch_bounds__(256) void row_norm_bwd(const float *__restrict__ dy, const float *__restrict__ x,
                                                    const float2 *__restrict__ stats, int64_t n, int H,
                                                    const float *__restrict__ w, float *__restrict__ dx,
                                                    float *__restrict__ part) {
  __shared__ float s_g[16][2][16 * CPL + 1];
  const int j = threadIdx.x & 15, gr = threadIdx.x >> 4;
  float wj[CPL], dw[CPL], db[CPL];
  row_ld(w, j, H, wj);
#pragma unroll
  for (int i = 0; i < CPL; ++i) dw[i] = db[i] = 0.f;
  for (int64_t r = static_cast<int64_t>(blockIdx.x) * 16 + gr; r < n; r += static_cast<int64_t>(gridDim.x) * 16) {
    float g[CPL], h[CPL], s1 = 0.f, s2 = 0.f;
    row_ld(dy + r * H, j, H, g);
    row_ld(x + r * H, j, H, h);
    const float2 st = stats[r];
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
      h[i] = (h[i] - st.x) * st.y;
      dw[i] = fmaf(g[i], h[i], dw[i]);
      db[i] += g[i];
      g[i] *= wj[i];
      if (j + 16 * i < H) {
        s1 += g[i];
        s2 = fmaf(g[i], h[i], s2);
      }
    }
    const float m1 = sum16(s1) / H, m2 = sum16(s2) / H;
    if (dx) {
#pragma unroll
      for (int i = 0; i < CPL; ++i)
        if (j + 16 * i < H) dx[r * H + j + 16 * i] = st.y * (g[i] - m1 - h[i] * m2);
    }
  }
  if (part == nullptr) return;
#pragma unroll
  for (int i = 0; i < CPL; ++i) {
    s_g[gr][0][j + 16 * i] = dw[i];
    s_g[gr][1][j + 16 * i] = db[i];
  }
  __syncthreads();
  for (int c = threadIdx.x; c < 2 * H; c += 256) {
    const int m = c / H, ch = c - m * H;
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) s += s_g[k][m][ch];
    part[static_cast<int64_t>(blockIdx.x) * 2 * H + c] = s;
  }
}

// out[c] = sum over the workgroups of part[., c], 64 threads per 4 channels.
__global__ __launch_bounds__(256) void norm_grad_sum(const float *__restrict__ part, int blocks, int H,
                                                     float *__restrict__ dw, float *__restrict__ db) {
  __shared__ float s_p[4][65];
  const int c = blockIdx.x * 4 + (threadIdx.x & 3), p = threadIdx.x >> 2;
  float s = 0.f;
  if (c < 2 * H)
    for (int k = p; k < blocks; k += 64) s += part[static_cast<int64_t>(k) * 2 * H + c];
  s_p[threadIdx.x & 3][p] = s;
  for (int d = 32; d > 0; d >>= 1) {
    __syncthreads();
    if (p < d) s_p[threadIdx.x & 3][p] += s_p[threadIdx.x & 3][p + d];
  }
  if (p == 0 && c < 2 * H) {
    float *out = c < H ? dw : db;
    if (out) out[c < H ? c : c - H] = s_p[threadIdx.x & 3][0];
  }
}

int norm_blocks(int64_t n) { return static_cast<int>(std::min<int64_t>((n + 15) / 16, kNormBlocks)); }

template <typename F>
void for_lane_channels(int H, F f) {   // f(channels per lane): 1, 2, 3, 4, 6 or 8
  const int c = (H + 15) / 16;
  if (c <= 1) f(std::integral_constant<int, 1>{});
  else if (c <= 2) f(std::integral_constant<int, 2>{});
  else if (c <= 3) f(std::integral_constant<int, 3>{});
  else if (c <= 4) f(std::integral_constant<int, 4>{});
  else if (c <= 6) f(std::integral_constant<int, 6>{});
  else f(std::integral_constant<int, 8>{});
}

int train_check(const char *what, int64_t E, int Cin, int64_t R, int64_t P, int A, int H) {
  SSLA_CHECK_ARG(E > 0 && Cin > 0 && R >= 0 && P >= 0 && A > 0 && H > 0, "%s: bad sizes E=%lld Cin=%d R=%lld P=%lld "
                 "A=%d H=%d", what, (long long)E, Cin, (long long)R, (long long)P, A, H);
  if (Cin > 128 || H > 128 || A > 49) {
    set_error("%s: needs input and hidden up to 128 and at most 49 positions (Cin=%d H=%d A=%d)", what, Cin, H, A);
    return SSLA_ERR_UNSUPPORTED;
  }
  if (E * A >= 0x7fffffff) {   // row places are 32-bit
    set_error("%s: %lld events at %d positions (below 2^31 copies per call)", what, (long long)E, A);
    return SSLA_ERR_UNSUPPORTED;
  }
  SSLA_CHECK_ARG(P < 0x7fffffff, "%s: too many patches", what);
  return SSLA_OK;
}

}  // namespace
}  // namespace ssla

extern "C" int ssla_mos_train_fwd(const float *events, int64_t E, int Cin, const int64_t *src, const int64_t *pos,
                                  int64_t R, const int64_t *cu, int64_t P, int A, const float *Wa, const float *WbT,
                                  const float *Win, int H, float *qvh, float *y, unsigned char *valid, float *out,
                                  void *stream) {
  using namespace ssla;
  clear_error();
  const int ok = train_check("mos_train_fwd", E, Cin, R, P, A, H);
  if (ok != SSLA_OK) return ok;
  SSLA_CHECK_ARG(events && src && pos && cu && Wa && WbT && qvh && y && valid && out, "mos_train_fwd: null pointer");
  const hipStream_t st = static_cast<hipStream_t>(stream);
  tall_gemm(events, Cin, Wa, qvh, E, A * 3 * H, Cin, 1, 3 * H, 2 * H, st);
  const ScanArgs sa = scan_args(src, pos, cu, P, R, A, H);
  if (P > 0) hipLaunchKernelGGL(mos_scan_fwd, scan_grid(sa), dim3(256), 0, st, sa, qvh, y, valid);
  if (R < E * A)
    hipLaunchKernelGGL(mos_zero_rows, dim3(static_cast<unsigned>((E * A + 255) / 256)), dim3(256), 0, st, valid, E * A,
                       H, y);
  tall_gemm(y, A * H, WbT, out, E, H, A * H, 0, 1, 0, st);
  if (Win) tall_gemm(events, Cin, Win, out, E, H, Cin, 2, 1, 0, st);
  return launch_status("mos_train_fwd");
}

extern "C" size_t ssla_mos_train_bwd_workspace_size(int64_t E, int Cin, int A, int H) {
  using namespace ssla;
  if (E <= 0 || Cin <= 0 || A <= 0 || H <= 0) return 0;
  const size_t rows = static_cast<size_t>(E) * A * H * sizeof(float);
  size_t part = 0;
  part = std::max(part, static_cast<size_t>(wgrad_slices(E, 3 * A * H)) * Cin * 3 * A * H);
  part = std::max(part, static_cast<size_t>(wgrad_slices(E, A * H)) * H * A * H);
  part = std::max(part, static_cast<size_t>(wgrad_slices(E, H)) * Cin * H);
  return up16(rows) + up16(3 * rows) + part * sizeof(float) + 16;
}

extern "C" int ssla_mos_train_bwd(const float *dout, const float *events, int64_t E, int Cin, const int64_t *src,
                                  const int64_t *pos, int64_t R, const int64_t *cu, int64_t P, int A,
                                  const float *WaT, const float *Wbp, const float *WinT, int H, const float *qvh,
                                  const float *y, const unsigned char *valid, float *devents, float *dWaT,
                                  float *dWbT, float *dWinT, void *workspace, size_t workspace_bytes, void *stream) {
  using namespace ssla;
  clear_error();
  const int ok = train_check("mos_train_bwd", E, Cin, R, P, A, H);
  if (ok != SSLA_OK) return ok;
  SSLA_CHECK_ARG(dout && events && src && pos && cu && WaT && Wbp && qvh && y && valid, "mos_train_bwd: null pointer");
  const size_t need = ssla_mos_train_bwd_workspace_size(E, Cin, A, H);
  if (workspace == nullptr || workspace_bytes < need) {
    set_error("mos_train_bwd: workspace of %zu bytes needed, %zu given", need, workspace_bytes);
    return SSLA_ERR_WORKSPACE;
  }
  const hipStream_t st = static_cast<hipStream_t>(stream);
  const size_t rows = static_cast<size_t>(E) * A * H * sizeof(float);
  char *ws = reinterpret_cast<char *>(up16(reinterpret_cast<uintptr_t>(workspace)));
  float *dy = reinterpret_cast<float *>(ws), *d = reinterpret_cast<float *>(ws + up16(rows));
  float *part = reinterpret_cast<float *>(ws + up16(rows) + up16(3 * rows));
  if (dWbT) wgrad(dout, y, E, H, A * H, part, dWbT, st);
  if (dWinT) wgrad(events, dout, E, Cin, H, part, dWinT, st);
  if (devents || dWaT) {
    tall_gemm(dout, H, Wbp, dy, E, A * H, H, 0, 1, 0, st);
    const ScanArgs sa = scan_args(src, pos, cu, P, R, A, H);
    if (P > 0) hipLaunchKernelGGL(mos_scan_bwd, scan_grid(sa), dim3(256), 0, st, sa, qvh, dy, d);
    if (R < E * A)
      hipLaunchKernelGGL(mos_zero_rows, dim3(static_cast<unsigned>((E * A + 255) / 256)), dim3(256), 0, st, valid,
                         E * A, 3 * H, d);
    if (dWaT) wgrad(events, d, E, Cin, 3 * A * H, part, dWaT, st);
    if (devents) {
      tall_gemm(d, 3 * A * H, WaT, devents, E, Cin, 3 * A * H, 0, 1, 0, st);
      if (WinT) tall_gemm(dout, H, WinT, devents, E, Cin, H, 2, 1, 0, st);
    }
  }
  return launch_status("mos_train_bwd");
}

extern "C" int ssla_row_norm_fwd(const float *x, int64_t n, int H, const float *w, const float *b, float eps, float *y,
                                 float *stats, void *stream) {
  using namespace ssla;
  clear_error();
  SSLA_CHECK_ARG(n > 0 && H > 0 && x && w && b && y && stats, "row_norm_fwd: bad arguments");
  SSLA_CHECK_ARG((reinterpret_cast<uintptr_t>(stats) & 7) == 0, "row_norm_fwd: stats must be 8-byte aligned");
  if (H > 128) {
    set_error("row_norm_fwd: H=%d exceeds 128", H);
    return SSLA_ERR_UNSUPPORTED;
  }
  for_lane_channels(H, [&](auto c) {
    hipLaunchKernelGGL(row_norm_fwd<decltype(c)::value>, dim3(norm_blocks(n)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), x, n, H, w, b, eps, y, reinterpret_cast<float2 *>(stats));
  });
  return launch_status("row_norm_fwd");
}

extern "C" size_t ssla_row_norm_bwd_workspace_size(int64_t n, int H) {
  return n > 0 && H > 0 ? sizeof(float) * 2 * H * ssla::norm_blocks(n) : 0;
}

extern "C" int ssla_row_norm_bwd(const float *dy, const float *x, const float *stats, int64_t n, int H, const float *w,
                                 float *dx, float *dw, float *db, void *workspace, size_t workspace_bytes,
                                 void *stream) {
  using namespace ssla;
  clear_error();
  SSLA_CHECK_ARG(n > 0 && H > 0 && dy && x && stats && w, "row_norm_bwd: bad arguments");
  SSLA_CHECK_ARG((reinterpret_cast<uintptr_t>(stats) & 7) == 0, "row_norm_bwd: stats must be 8-byte aligned");
  if (H > 128) {
    set_error("row_norm_bwd: H=%d exceeds 128", H);
    return SSLA_ERR_UNSUPPORTED;
  }
  const size_t need = ssla_row_norm_bwd_workspace_size(n, H);
  if ((dw || db) && (workspace == nullptr || workspace_bytes < need)) {
    set_error("row_norm_bwd: workspace of %zu bytes needed, %zu given", need, workspace_bytes);
    return SSLA_ERR_WORKSPACE;
  }
  const hipStream_t st = static_cast<hipStream_t>(stream);
  float *part = dw || db ? static_cast<float *>(workspace) : nullptr;
  const int blocks = norm_blocks(n);
  for_lane_channels(H, [&](auto c) {
    hipLaunchKernelGGL(row_norm_bwd<decltype(c)::value>, dim3(blocks), dim3(256), 0, st, dy, x,
                       reinterpret_cast<const float2 *>(stats), n, H, w, dx, part);
  });
  if (part) hipLaunchKernelGGL(norm_grad_sum, dim3((2 * H + 3) / 4), dim3(256), 0, st, part, blocks, H, dw, db);
  return launch_status("row_norm_bwd");
}
