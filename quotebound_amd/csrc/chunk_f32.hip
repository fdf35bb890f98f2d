// The recurrence on float32 inputs at Dk = 128, chunkwise, on float32 matrix instructions: what the recurrent design's
// entry points run on long sequences (rec.hip chooses). The recurrent kernels spend every step of every state row on
// the vector pipes (64-71% busy); here a chunk of 64 steps is a few products of 64 x 128 and 128 x 128 matrices on
// v_mfma_f32_16x16x4_f32, every operand and sum float32, so the results keep the recurrent form's accuracy (measured
// against 64-bit values: 1e-7 to 2e-7 in both). The residuals are the recurrent design's: the chunk-start states and
// e = v - u per token and state row, so either backward reads either forward's.
//
// With G the chunk's cumulative log-decays, E_ij = exp(G_i - G_j), M = strict_lower(E * K K^T), P = lower_incl(E *
// Q K^T) and D = diag(exp(G_63 - G)), a chunk's forward is
//   R = V - diag(exp G) K S0^T,  e = (I + M diag(beta))^-1 R,  Delta = diag(beta) e
//   Y = diag(exp G) Q S0^T + P Delta,  S1 = exp(G_63) S0 + Delta^T D K
// (so e comes without a division by beta), and its backward, with T = (I + diag(beta) M)^-1,
//   dDelta = P^T dY + D K dS1^T,  w = T^T dDelta,  dV = diag(beta) w,  dbeta = rowsum(w * e)
//   dS0 = exp(G_63) dS1 + dY^T diag(exp G) Q - dV^T diag(exp G) K
//   dP = dY Delta^T,  dM = -dV Delta^T,  N = lower_incl(dP * E),  X = strict_lower(dM * E)
//   dQ = diag(exp G) dY S0 + N K,  dK = -diag(exp G) dV S0 + D Delta dS1 + N^T Q + (X + X^T) K
// and dG from every exponential (the equations of the reference's step-by-step sweep, src/delta_grad.cpp:14-18).
//
// Four kernels: prep (E, the inverse, P: no state in it), the two state passes (one block per sequence, value head
// and 16 state rows, over the chunks in order) and the per-chunk gradients.
//
// A product contracts over 16 indices at a time: a lane of group g = lane / 16 supplies indices 4g .. 4g + 3 of the
// 16, one per instruction (element e of all lanes: indices 4g + e), so rows are read 16 bytes at a time and both
// operands follow the same order.
//
// Bound by the matrix pipes' float32 rate (256 operations a cycle and CU) and the latency of the chain of products in
// the state passes: about half of that rate each. At B = 1, T = 4096, 16 key and 32 value heads of 128: prep 38 us,
// forward 218, prep again 39, backward state pass 214, gradients 299, where the step-by-step kernels took 819 us
// forward and 1,877 + 202 backward.
//
// Every sum is taken 16 terms at a time from zero (four instructions) and the partial sums added up: a chain of 128
// terms in one accumulator rounds 128 times at the size of the whole sum (dq 6e-7 from the 64-bit values where the
// recurrent form is 1.2e-7 off).
//
// A value that is not finite spreads in a product to positions that the step-by-step form would not touch (zeros of a
// triangular matrix times it). The kernels look for such values in what they form and raise a flag; the recurrent
// kernels follow each pass and do its work again if the flag is up, and return at once if not.
#include "chunk_common.h"
#include "gdn_kernels.h"

namespace qbgdn {
namespace {

constexpr int Dk = 128;
constexpr int kR = 16;       // state rows per block of the state passes
constexpr int kLW = 20;      // pitch of the [64 positions][16 rows] matrices
constexpr int kLX = 132;     // pitch of the [16][128] hand-over of the backward state pass
constexpr double kLogFloor = -150.0;

// Per (chunk slot, value head), written by prep: the inverse, P and (for the backward) E as their ten 16 x 16 blocks on
// or below the diagonal (tri_off), and the per-position vectors.
struct TileF {
  float t[kTri];
  float p[kTri];
  float e[kTri];
  float gam[kC];   // exp(G_i)
  float dec[kC];   // exp(G_63 - G_i)
  float beta[kC];
};
static_assert(sizeof(TileF) % 16 == 0, "TileF records stay 16-byte aligned");

struct F32Args {
  const float *q, *k, *v, *g, *beta, *s0;
  float *y, *s_out, *ckpt, *e_res;
  const float *dy, *ds_out;
  float *dq, *dk, *dv, *dg, *dbeta, *ds0;
  TileF* tiles;
  float* dsend;  // [NC][Hv][Dv][Dk]: the cotangent of each chunk's end state
  float* w;      // [tokens][Hv][Dv]: the cotangent of Delta, through the inverse
  int* flag;     // raised when a value formed is not finite; cleared by prep
  int64_t NC;
  int Hk, Hv, Dv, N, nblk, g_is_log;
  SeqTable tab;
};

__device__ __forceinline__ f32x4 mmaf(f32x4 c, float a, float b) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The four instructions over 16 indices, from zero.
__device__ __forceinline__ f32x4 dot16(const f32x4& a, const f32x4& b) {
  return mmaf(mmaf(mmaf(mmaf(zero4(), a[0], b[0]), a[1], b[1]), a[2], b[2]), a[3], b[3]);
}

// N of them side by side: an instruction waits for the one before it in its sum about as long again as it runs, so a
// wave alternates between sums. Returns their sum.
template <int N>
__device__ __forceinline__ f32x4 dot16n(const f32x4 (&a)[N], const f32x4 (&b)[N]) {
  f32x4 x[N];
#pragma unroll
  for (int n = 0; n < N; ++n) x[n] = zero4();
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int n = 0; n < N; ++n) x[n] = mmaf(x[n], a[n][e], b[n][e]);
  if constexpr (N == 4) return (x[0] + x[1]) + (x[2] + x[3]);
  f32x4 r = x[0];
#pragma unroll
  for (int n = 1; n < N; ++n) r += x[n];
  return r;
}
// Element (r, c) of a float32 LDS matrix of row length ld (64 or 128): the 16-byte units of a row are permuted by its
// index, so that 16 rows read 16 bytes wide at one column, and the rows 4g + e (g = 0..3) read at 16 consecutive
// columns, each cover the 64 banks once.
__device__ __forceinline__ int fsw(int r, int c, int ld) { return r * ld + (c ^ (4 * (r & 15))); }
// The same for rows of 32.
__device__ __forceinline__ int psw(int r, int c) { return r * 32 + (c ^ (4 * ((r >> 1) & 7))); }

__device__ __forceinline__ f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ void st4(float* p, const f32x4& x) { *reinterpret_cast<f32x4*>(p) = x; }
__device__ __forceinline__ f32x4 as_f4(const uint4& u) { return __builtin_bit_cast(f32x4, u); }

// NaN once a value that is not finite has been added.
__device__ __forceinline__ void watch(float& m, const f32x4& x) {
#pragma unroll
  for (int j = 0; j < 4; ++j) m = fmaf(x[j], 0.f, m);
}
__device__ __forceinline__ void raise(int* flag, float m) {
  if (!(m == 0.f)) atomicOr(flag, 1);
}

// ---- prep -----------------------------------------------------------------------------------------------------------

// A and the inverse in LDS, float32, as the padded blocks of chunk_prep.hip (rows of 20, blocks 324 apart).
constexpr int kLdPad = 20, kBlkPad = 16 * kLdPad + 4, kTriPad = 10 * kBlkPad;
__device__ __forceinline__ int tri_pad(int i, int j) {
  return ((i >> 4) * ((i >> 4) + 1) / 2 + (j >> 4)) * kBlkPad + (i & 15) * kLdPad + (j & 15);
}

// One block per (chunk slot, key head), its value heads in turn, or per (chunk slot, value head) where those blocks
// fit on the device at once (hpb = 1). kBwd: the inverse of I + diag(beta) M, else of I + M diag(beta).
template <bool kBwd>
__global__ __launch_bounds__(256, 4) void f32_prep_kernel(F32Args a, int hpb) {
  constexpr int kH = Dk / 2;  // K and Q are staged 64 columns at a time, so that four blocks share a CU
  __shared__ __align__(16) float smem[2 * kC * kH];  // K and Q columns, then A and the inverse in the same bytes
  __shared__ double Gd[kC];
  __shared__ float Bs[kC], Sg[kC];
  static_assert(2 * kTriPad <= 2 * kC * kH, "A and the inverse fit in the k/q staging bytes");
  float *Kb = smem, *Qb = smem + kC * kH, *Am = smem, *Tm = smem + kTriPad;
  if (blockIdx.x == 0 && threadIdx.x == 0) *a.flag = 0;

  const int units = a.Hv / hpb, total = int(a.NC) * units, grp = a.Hv / a.Hk;
  const int wid = xcd_remap(blockIdx.x, total);
  const int64_t slot = wid / units;
  const int hv0 = (wid % units) * hpb, hk = hv0 / grp;
  const SlotPos sp = slot_pos(a.tab, slot);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 4, li = lane & 15;
  const uint32_t L = uint32_t(sp.L);
  const int sk = a.Hk * Dk;
  // The ten lower-triangular blocks (I, J) of K K^T and Q K^T, formed transposed: lane -> row i = 16 I + li, columns
  // 16 J + 4g + jj. In registers for every value head.
  f32x4 kk[3], qk[3];
#pragma unroll
  for (int u = 0; u < 3; ++u) kk[u] = zero4(), qk[u] = zero4();
  {
    const auto kr = buffer_rsrc(a.k + sp.tok * sk + hk * Dk, L * uint32_t(sk) * 4u);
    const auto qr = buffer_rsrc(a.q + sp.tok * sk + hk * Dk, L * uint32_t(sk) * 4u);
    uint4 kv[4], qv[4];
    const auto load = [&](int c0) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int e = tid + 256 * j;
        const uint32_t off = uint32_t((e >> 4) * sk + c0 + (e & 15) * 4) * 4u;
        kv[j] = buf_ld16(kr, off), qv[j] = buf_ld16(qr, off);
      }
    };
    load(0);
#pragma unroll
    for (int c0 = 0; c0 < Dk; c0 += kH) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int e = tid + 256 * j, at = fsw(e >> 4, (e & 15) * 4, kH);
        st4(Kb + at, as_f4(kv[j])), st4(Qb + at, as_f4(qv[j]));
      }
      __syncthreads();
      if (c0 == 0) load(kH);
#pragma unroll
      for (int u = 0; u < 3; ++u) {
        const int b = w + 4 * u, I = (b >= 1) + (b >= 3) + (b >= 6), J = b - I * (I + 1) / 2;
        if (b < 10) {
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            const int c = 16 * s + 4 * g;
            const f32x4 aj = ld4(Kb + fsw(16 * J + li, c, kH)), ki = ld4(Kb + fsw(16 * I + li, c, kH));
            const f32x4 qi = ld4(Qb + fsw(16 * I + li, c, kH));
            kk[u] += dot16(aj, ki), qk[u] += dot16(aj, qi);
          }
        }
      }
      if (c0 == 0) __syncthreads();
    }
  }
  for (int vh = 0; vh < hpb; ++vh) {
    const int hv = hv0 + vh;
    TileF* tile = a.tiles + (slot * a.Hv + hv);
    __syncthreads();  // every wave is done with the K and Q rows, or with the previous head's A and inverse
    if (tid < kC) {
      const int64_t at = (sp.tok + tid) * a.Hv + hv;
      const bool in = uint32_t(tid) < L;
      const float gx = in ? a.g[at] : 0.f, bx = in ? a.beta[at] : 0.f;
      // The log-decay, floored where its exponential is 0 in float32 (so that a factor of 0 does not make G_i - G_j a
      // NaN); a decay factor's sign is kept apart.
      double G = 0.0;
      bool neg = false;
      if (in) {
        G = a.g_is_log ? double(gx) : log(fabs(double(gx)));
        if (G < kLogFloor) G = kLogFloor;
        neg = !a.g_is_log && gx < 0.f;
      }
      const uint64_t nm = __ballot(neg);
      Gd[tid] = wave_prefix_sum(G), Bs[tid] = bx;
      Sg[tid] = __popcll(nm & ((uint64_t(2) << tid) - 1)) & 1 ? -1.f : 1.f;
    }
    __syncthreads();
    if (w == 3) {  // the tile's vectors: a wave with two blocks where two others have three
      const double G = Gd[lane], Glast = Gd[kC - 1];
      tile->gam[lane] = Sg[lane] * expf(float(G));
      tile->dec[lane] = Sg[lane] * Sg[kC - 1] * expf(float(Glast - G));
      tile->beta[lane] = Bs[lane];
    }
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      const int b = w + 4 * u, I = (b >= 1) + (b >= 3) + (b >= 6), J = b - I * (I + 1) / 2;
      if (b < 10) {
        const int i = 16 * I + li, j0 = 16 * J + 4 * g;
        f32x4 av, pv, xv;
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const int j = j0 + jj;
          const float e = j <= i ? Sg[i] * Sg[j] * expf(float(Gd[i] - Gd[j])) : 0.f;
          av[jj] = j < i ? (kBwd ? Bs[i] : Bs[j]) * e * kk[u][jj] : 0.f;
          pv[jj] = j <= i ? e * qk[u][jj] : 0.f;
          xv[jj] = e;
        }
        st4(Am + tri_pad(i, j0), av);
        st4(tile->p + tri_off(i, j0), pv);
        if constexpr (kBwd) st4(tile->e + tri_off(i, j0), xv);
      }
    }
    __syncthreads();
    // The diagonal blocks by substitution, thread -> column; then the blocks at distance d below them,
    // T_IJ = -T_II sum_{J <= K < I} A_IK T_KJ, one wave per block.
    if (tid < kC) {
      const int jl = tid & 15, b0 = tid & ~15;
      float x[16], col[16];
#pragma unroll
      for (int il = 0; il < 16; ++il) col[il] = Am[tri_pad(b0 + il, b0 + jl)];
      lower_inverse16(col, x, jl);
#pragma unroll
      for (int il = 0; il < 16; ++il) Tm[tri_pad(b0 + il, b0 + jl)] = x[il];
    }
    __syncthreads();
    for (int d = 1; d < 4; ++d) {
      if (w < 4 - d) {
        const int I = d + w, J = w;
        f32x4 W = zero4();
        for (int K = J; K < I; ++K) {
          f32x4 tk;
#pragma unroll
          for (int e = 0; e < 4; ++e) tk[e] = Tm[tri_pad(16 * K + 4 * g + e, 16 * J + li)];
          W += dot16(ld4(Am + tri_pad(16 * I + li, 16 * K + 4 * g)), tk);
        }
        const f32x4 R = dot16(ld4(Tm + tri_pad(16 * I + li, 16 * I + 4 * g)), W);
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) Tm[tri_pad(16 * I + 4 * g + jj, 16 * J + li)] = -R[jj];
      }
      __syncthreads();
    }
    {
      const int i = tid >> 2, j0 = (tid & 3) * 16;
      if (j0 <= i) {
#pragma unroll
        for (int j = 0; j < 16; j += 4) st4(tile->t + tri_off(i, j0 + j), ld4(Tm + tri_pad(i, j0 + j)));
      }
    }
  }
}

// Rows r .. r + 3 of a [64][16] matrix (pitch kLW) at column c.
__device__ __forceinline__ f32x4 rows4(const float* m, int r, int c) {
  return f32x4{m[r * kLW + c], m[(r + 1) * kLW + c], m[(r + 2) * kLW + c], m[(r + 3) * kLW + c]};
}
// Rows r .. r + 3 of a [64][128] matrix (fsw) at column c.
__device__ __forceinline__ f32x4 cols4(const float* m, int r, int c) {
  return f32x4{m[fsw(r, c, Dk)], m[fsw(r + 1, c, Dk)], m[fsw(r + 2, c, Dk)], m[fsw(r + 3, c, Dk)]};
}

// A lane's offsets into [..][128] matrices (fsw), formed once: an offset formed at each read costs the chain two or
// three vector instructions, and a wave issues one in about five cycles. The asm keeps them from being formed again.
struct RowOff {  // row i (i & 15 = li) at columns 16 s + 4g, s = 0 .. 3 (64 columns on: + 64)
  int o[4];
  __device__ RowOff(int i, int g, int li) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      o[s] = i * Dk + ((16 * s + 4 * g) ^ (4 * li));
      asm volatile("" : "+v"(o[s]));
    }
  }
};
struct ColOff {  // rows 4g + e at columns c + 16 t, c a multiple of 32 plus li (16 rows on: + 16 Dk)
  int o[4][2];
  __device__ ColOff(int c, int g) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        o[e][t] = (4 * g + e) * Dk + ((c + 16 * t) ^ (16 * g + 4 * e));
        asm volatile("" : "+v"(o[e][t]));
      }
  }
};
// The sum over columns 64 h .. 64 h + 63 of a row of A times a row of B.
__device__ __forceinline__ f32x4 dot_rows(const float* A, const RowOff& i, const float* B, const RowOff& j, int h) {
  f32x4 x[4], y[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) x[s] = ld4(A + i.o[s] + 64 * h), y[s] = ld4(B + j.o[s] + 64 * h);
  return dot16n(x, y);
}
// up[t] += the sum over the positions 32 h .. of column c + 16 t of K times a row's entries d of those positions.
__device__ __forceinline__ void dot_cols(f32x4 (&up)[2], const float* K, const ColOff& c, const f32x4& d0,
                                         const f32x4& d1, int h) {
  f32x4 x[2][2];
#pragma unroll
  for (int t = 0; t < 2; ++t) x[0][t] = zero4(), x[1][t] = zero4();
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      x[0][t] = mmaf(x[0][t], K[c.o[e][t] + 32 * h * Dk], d0[e]);
      x[1][t] = mmaf(x[1][t], K[c.o[e][t] + (32 * h + 16) * Dk], d1[e]);
    }
#pragma unroll
  for (int t = 0; t < 2; ++t) up[t] += x[0][t] + x[1][t];
}
// Over the positions j of the first N tiles: the sum of m[j][li] A[ip][j], A packed lower triangular, N - 1 = ip's tile.
template <int N>
__device__ __forceinline__ f32x4 tri_rows_n(const float* m, const float* A, int ip, int g, int li) {
  f32x4 x[N], y[N];
#pragma unroll
  for (int J = 0; J < N; ++J) x[J] = rows4(m, 16 * J + 4 * g, li), y[J] = ld4(A + tri_off(ip, 16 * J + 4 * g));
  return dot16n(x, y);
}
__device__ __forceinline__ f32x4 tri_rows(const float* m, const float* A, int wp, int ip, int g, int li) {
  switch (wp) {
    case 0: return tri_rows_n<1>(m, A, ip, g, li);
    case 1: return tri_rows_n<2>(m, A, ip, g, li);
    case 2: return tri_rows_n<3>(m, A, ip, g, li);
    default: return tri_rows_n<4>(m, A, ip, g, li);
  }
}
// Over the positions i of the last N tiles: the sum of m[i][li] A[i][ip], ip's tile the first of them (index 4e + g at
// step e: the four rows a step reads then lie on distinct banks).
template <int N>
__device__ __forceinline__ f32x4 tri_cols_n(const float* m, const float* A, int ip, int g, int li) {
  f32x4 x[N], y[N];
#pragma unroll
  for (int I = 0; I < N; ++I) {
    const int i = 16 * (4 - N + I) + g;
    x[I] = f32x4{m[i * kLW + li], m[(i + 4) * kLW + li], m[(i + 8) * kLW + li], m[(i + 12) * kLW + li]};
    // Rows 4 apart of block (I, J): 64 elements.
    const float* b = A + (((4 - N + I) * (5 - N + I) / 2 + 4 - N) << 8) + (g << 4) + (ip & 15);
    y[I] = f32x4{b[0], b[64], b[128], b[192]};
  }
  return dot16n(x, y);
}
__device__ __forceinline__ f32x4 tri_cols(const float* m, const float* A, int wp, int ip, int g, int li) {
  switch (wp) {
    case 0: return tri_cols_n<4>(m, A, ip, g, li);
    case 1: return tri_cols_n<3>(m, A, ip, g, li);
    case 2: return tri_cols_n<2>(m, A, ip, g, li);
    default: return tri_cols_n<1>(m, A, ip, g, li);
  }
}

// ---- the forward state pass -----------------------------------------------------------------------------------------

// Waves 0-3 carry the state (wave w: positions 16w .., then state columns 32w ..), waves 4-7 form y, waves 8-11 load
// the next chunk's inputs into registers a chunk ahead and stage them in LDS where their last readers are done. Three
// barriers per chunk: S in LDS | K S^T, R | e, Delta | the update of S; y's S Q^T runs beside the first two and its P
// Delta beside the third (S Q^T whole beside the second: 247 -> 239 us at 4,096 steps, 63.8 -> 64.6 at 777). A block issues 464 matrix instructions per chunk, 3,712 cycles on its four pipes.
__global__ __launch_bounds__(768) void f32_fwd_kernel(F32Args a) {
  __shared__ __align__(16) float Sm[2][kR * Dk], Kb[2][kC * Dk], Qb[kC * Dk], Tb[kTri], Pb[kTri];
  __shared__ __align__(16) float Wr[kC * kLW], Wd[kC * kLW], We[kC * kLW], Vs[kC * kR], Gs[2][256];
  const int total = a.nblk * a.Hv * a.N;
  const StateItem item = state_item(a.tab, blockIdx.x, a.nblk, a.Hv, a.Hk, total);
  const int hv = item.hv, n = item.n, hk = hv / (a.Hv / a.Hk), row0 = kR * item.blk;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, li = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wp = (w & 4) ? 3 - (w & 3) : w & 3, ip = 16 * wp + li, u = tid & 255;
  const Seq sq = seq_of(a.tab, n);
  const int nch = (sq.len + kC - 1) / kC;
  const int sk = a.Hk * Dk, sv = a.Hv * a.Dv;

  if (w >= 8) {
    uint4 k[8], q[8], t[3], p[3], v;
    float gd;
    const auto rows = [&](uint4 (&x)[8], const float* src, int c) {
      const int64_t tok = sq.tok0 + int64_t(c) * kC;
      const auto r = buffer_rsrc(src + tok * sk + hk * Dk, uint32_t(min(kC, sq.len - c * kC)) * uint32_t(sk) * 4u);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int e = u + 256 * j;
        x[j] = buf_ld16(r, uint32_t((e >> 5) * sk + (e & 31) * 4) * 4u);
      }
    };
    const auto tile = [&](int c) { return a.tiles + ((sq.slot0 + c) * a.Hv + hv); };
    const auto tri = [&](uint4 (&x)[3], const float* src) {
      const auto r = buffer_rsrc(src, kTri * 4);
#pragma unroll
      for (int j = 0; j < 3; ++j) x[j] = buf_ld16(r, uint32_t(u + 256 * j) * 16u);
    };
    const auto small = [&](int c) {  // v rows u / 4, and exp G, D, beta (the rest unused)
      const int64_t tok = sq.tok0 + int64_t(c) * kC;
      const auto r = buffer_rsrc(a.v + tok * sv + hv * a.Dv + row0,
                                 uint32_t(min(kC, sq.len - c * kC)) * uint32_t(sv) * 4u);
      v = buf_ld16(r, uint32_t((u >> 2) * sv + 4 * (u & 3)) * 4u);
      gd = buf_ld4(buffer_rsrc(tile(c)->gam, 3 * kC * 4), uint32_t(u) * 4u);
    };
    const auto put_rows = [&](float* dst, const uint4 (&x)[8]) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int e = u + 256 * j;
        st4(dst + fsw(e >> 5, (e & 31) * 4, Dk), as_f4(x[j]));
      }
    };
    const auto put_tri = [&](float* dst, const uint4 (&x)[3]) {
      static_assert(kTri / 4 == 640, "two units per thread and one for the first two waves");
#pragma unroll
      for (int j = 0; j < 2; ++j) st4(dst + 4 * (u + 256 * j), as_f4(x[j]));
      if (w < 10) st4(dst + 4 * (u + 512), as_f4(x[2]));  // the last 128 units: whole waves, so no masked store
    };
    const auto put_small = [&](int b) { st4(Vs + 4 * u, as_f4(v)), Gs[b][u] = gd; };
    if (nch == 0) return;
    rows(k, a.k, 0), rows(q, a.q, 0), tri(t, tile(0)->t), small(0);
    put_rows(Kb[0], k), put_rows(Qb, q), put_tri(Tb, t), put_small(0);
    const int c1 = min(1, nch - 1);
    tri(p, tile(0)->p), rows(k, a.k, c1), small(c1), rows(q, a.q, c1), tri(t, tile(c1)->t);
    for (int c = 0; c < nch; ++c) {
      const int cn = min(c + 1, nch - 1), c2 = min(c + 2, nch - 1), b1 = (c & 1) ^ 1;
      __syncthreads();
      put_tri(Pb, p);  // P of chunk c: y of chunk c - 1 is formed
      tri(p, tile(cn)->p);
      __syncthreads();
      put_rows(Kb[b1], k), put_small(b1);  // of chunk c + 1: the last readers of these bytes were chunk c - 1's
      rows(k, a.k, c2), small(c2);
      __syncthreads();
      put_rows(Qb, q), put_tri(Tb, t);  // S Q^T and e of chunk c are formed
      rows(q, a.q, c2), tri(t, tile(c2)->t);
    }
    return;
  }
  float bad = 0.f;
  const RowOff so(li, g, li), ko(ip, g, li);
  if (w >= 4) {
    for (int c = 0; c < nch; ++c) {
      const int b = c & 1;
      __syncthreads();
      f32x4 x = dot_rows(Sm[b], so, Qb, ko, 0);
      __syncthreads();
      x += dot_rows(Sm[b], so, Qb, ko, 1);
      __syncthreads();
      const f32x4 y = Gs[b][ip] * x + tri_rows(Wd, Pb, wp, ip, g, li);
      const int64_t tok = sq.tok0 + int64_t(c) * kC;
      const auto yr = buffer_rsrc(a.y + tok * sv + hv * a.Dv + row0,
                                  uint32_t(min(kC, sq.len - c * kC)) * uint32_t(sv) * 4u);
      BufIO<float>::st4(yr, uint32_t(ip * sv + 4 * g), y);
      watch(bad, y);
    }
    raise(a.flag, bad);
    return;
  }
  // S tile t holds S[li][32 wp + 16 t + 4g + jj].
  const int64_t srow = (int64_t(n) * a.Hv + hv) * a.Dv + row0 + li;
  f32x4 S[2] = {zero4(), zero4()};
  const ColOff uo(32 * wp + li, g);
  if (a.s0) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) S[t][jj] = a.s0[srow * Dk + 32 * wp + 16 * t + 4 * g + jj];
  }
  const uint32_t ck_bytes = a.ckpt ? uint32_t(kR) * Dk * 4 : 0u;
  for (int c = 0; c < nch; ++c) {
    const int64_t slot = sq.slot0 + c, tok = sq.tok0 + int64_t(c) * kC;
    const uint32_t L = uint32_t(min(kC, sq.len - c * kC));
    const int b = c & 1;
    {
      const auto ck = buffer_rsrc(a.ckpt ? a.ckpt + ((slot * a.Hv + hv) * a.Dv + row0) * Dk : a.k, ck_bytes);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int col = 32 * wp + 16 * t + 4 * g;
        st4(Sm[b] + fsw(li, col, Dk), S[t]);
        BufIO<float>::st4(ck, uint32_t(li * Dk + col), S[t]);
      }
    }
    __syncthreads();
    {
      const f32x4 x = dot_rows(Sm[b], so, Kb[b], ko, 0) + dot_rows(Sm[b], so, Kb[b], ko, 1);
      st4(Wr + ip * kLW + 4 * g, ld4(Vs + ip * kR + 4 * g) - Gs[b][ip] * x);
    }
    __syncthreads();
    {
      const f32x4 ev = tri_rows(Wr, Tb, wp, ip, g, li);
      const f32x4 dl = Gs[b][2 * kC + ip] * ev;
      st4(Wd + ip * kLW + 4 * g, dl);
      st4(We + ip * kLW + 4 * g, Gs[b][kC + ip] * dl);
      const auto er = buffer_rsrc(a.e_res ? a.e_res + tok * sv + hv * a.Dv + row0 : a.k,
                                  a.e_res ? L * uint32_t(sv) * 4u : 0u);
      BufIO<float>::st4(er, uint32_t(ip * sv + 4 * g), ev);
      watch(bad, ev);
    }
    __syncthreads();
    const float glast = Gs[b][kC - 1];
    f32x4 up[2] = {zero4(), zero4()};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      dot_cols(up, Kb[b], uo, rows4(We, 32 * h + 4 * g, li), rows4(We, 32 * h + 16 + 4 * g, li), h);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) S[t] = glast * S[t] + up[t];
  }
  watch(bad, S[0]), watch(bad, S[1]);
  raise(a.flag, bad);
  if (a.s_out) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) a.s_out[srow * Dk + 32 * wp + 16 * t + 4 * g + jj] = S[t][jj];
  }
}

// ---- the backward state pass ----------------------------------------------------------------------------------------

// The same shape over the chunks in reverse: waves 0-3 carry dS (K dS^T, dDelta | w = T^T dDelta, dv | the update),
// waves 4-7 form what has no dS in it, Z = dY^T P of the next chunk and X = Q^T diag(exp G) dY of this one, waves
// 8-11 load and stage.
__global__ __launch_bounds__(768) void f32_bwd_state_kernel(F32Args a) {
  __shared__ __align__(16) float dSm[kR * Dk], Kb[2][kC * Dk], Qb[kC * Dk], Tb[kTri], Pb[kTri], Ys[2][kC * kLW];
  __shared__ __align__(16) float Zs[kC * kLW], Wd[kC * kLW], We[kC * kLW], Xs[kR * kLX], Gs[2][256];
  const int total = a.nblk * a.Hv * a.N;
  const StateItem item = state_item(a.tab, blockIdx.x, a.nblk, a.Hv, a.Hk, total);
  const int hv = item.hv, n = item.n, hk = hv / (a.Hv / a.Hk), row0 = kR * item.blk;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, li = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wp = (w & 4) ? 3 - (w & 3) : w & 3, ip = 16 * wp + li, u = tid & 255;
  const Seq sq = seq_of(a.tab, n);
  const int nch = (sq.len + kC - 1) / kC;
  const int sk = a.Hk * Dk, sv = a.Hv * a.Dv;

  if (w >= 8) {
    uint4 k[8], q[8], t[3], p[3], yv;
    float gd;
    const auto rows = [&](uint4 (&x)[8], const float* src, int c) {
      const int64_t tok = sq.tok0 + int64_t(c) * kC;
      const auto r = buffer_rsrc(src + tok * sk + hk * Dk, uint32_t(min(kC, sq.len - c * kC)) * uint32_t(sk) * 4u);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int e = u + 256 * j;
        x[j] = buf_ld16(r, uint32_t((e >> 5) * sk + (e & 31) * 4) * 4u);
      }
    };
    const auto tile = [&](int c) { return a.tiles + ((sq.slot0 + c) * a.Hv + hv); };
    const auto tri = [&](uint4 (&x)[3], const float* src) {
      const auto r = buffer_rsrc(src, kTri * 4);
#pragma unroll
      for (int j = 0; j < 3; ++j) x[j] = buf_ld16(r, uint32_t(u + 256 * j) * 16u);
    };
    const auto small = [&](int c) {  // dY rows u / 4, and exp G, D, beta (the rest unused)
      const int64_t tok = sq.tok0 + int64_t(c) * kC;
      const auto r = buffer_rsrc(a.dy + tok * sv + hv * a.Dv + row0,
                                 uint32_t(min(kC, sq.len - c * kC)) * uint32_t(sv) * 4u);
      yv = buf_ld16(r, uint32_t((u >> 2) * sv + 4 * (u & 3)) * 4u);
      gd = buf_ld4(buffer_rsrc(tile(c)->gam, 3 * kC * 4), uint32_t(u) * 4u);
    };
    const auto put_rows = [&](float* dst, const uint4 (&x)[8]) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int e = u + 256 * j;
        st4(dst + fsw(e >> 5, (e & 31) * 4, Dk), as_f4(x[j]));
      }
    };
    const auto put_tri = [&](float* dst, const uint4 (&x)[3]) {
      static_assert(kTri / 4 == 640, "two units per thread and one for the first two waves");
#pragma unroll
      for (int j = 0; j < 2; ++j) st4(dst + 4 * (u + 256 * j), as_f4(x[j]));
      if (w < 10) st4(dst + 4 * (u + 512), as_f4(x[2]));  // the last 128 units: whole waves, so no masked store
    };
    const auto put_small = [&](int b) { st4(Ys[b] + (u >> 2) * kLW + 4 * (u & 3), as_f4(yv)), Gs[b][u] = gd; };
    if (nch == 0) return;
    const int c0 = nch - 1, c1 = max(nch - 2, 0);
    rows(k, a.k, c0), rows(q, a.q, c0), tri(t, tile(c0)->t), tri(p, tile(c0)->p), small(c0);
    put_rows(Kb[c0 & 1], k), put_rows(Qb, q), put_tri(Tb, t), put_tri(Pb, p), put_small(c0 & 1);
    __syncthreads();  // the first Z is formed
    small(c1), tri(p, tile(c1)->p), rows(k, a.k, c1), rows(q, a.q, c1), tri(t, tile(c1)->t);
    for (int c = nch - 1; c >= 0; --c) {
      const int c2 = max(c - 2, 0), b1 = (c & 1) ^ 1;
      __syncthreads();
      put_tri(Pb, p);  // of chunk c - 1: Z of chunk c is formed
      tri(p, tile(c2)->p);
      __syncthreads();
      put_rows(Kb[b1], k), put_small(b1);  // of chunk c - 1: the last readers of these bytes were chunk c + 1's
      rows(k, a.k, c2), small(c2);
      __syncthreads();
      put_rows(Qb, q), put_tri(Tb, t);  // X and w of chunk c are formed
      rows(q, a.q, c2), tri(t, tile(c2)->t);
    }
    return;
  }
  if (w >= 4) {
    // Z at rows r = 4g + jj, position ip: sum over i of dY[i][r] P[i][ip], from LDS buffer b.
    const auto form_z = [&](int b) { st4(Zs + ip * kLW + 4 * g, tri_cols(Ys[b], Pb, wp, ip, g, li)); };
    const ColOff uo(32 * wp + li, g);
    if (nch == 0) return;
    __syncthreads();
    form_z((nch - 1) & 1);
    for (int c = nch - 1; c >= 0; --c) {
      const int b = c & 1;
      // X at state columns 32 wp + 16 t + 4g + jj, row li.
      f32x4 x[2] = {zero4(), zero4()};
      const auto half = [&](int h) {
        const int i = 32 * h + 4 * g;
        dot_cols(x, Qb, uo, ld4(Gs[b] + i) * rows4(Ys[b], i, li), ld4(Gs[b] + i + 16) * rows4(Ys[b], i + 16, li), h);
      };
      __syncthreads();
      half(0);
      __syncthreads();
      half(1);
#pragma unroll
      for (int t = 0; t < 2; ++t) st4(Xs + li * kLX + 32 * wp + 16 * t + 4 * g, x[t]);
      __syncthreads();
      if (c > 0) form_z(b ^ 1);
    }
    return;
  }
  const int64_t srow = (int64_t(n) * a.Hv + hv) * a.Dv + row0 + li;
  float bad = 0.f;
  f32x4 dS[2] = {zero4(), zero4()};
  const RowOff so(li, g, li), ko(ip, g, li);
  const ColOff uo(32 * wp + li, g);
  if (a.ds_out) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) dS[t][jj] = a.ds_out[srow * Dk + 32 * wp + 16 * t + 4 * g + jj];
  }
  if (nch > 0) __syncthreads();
  for (int c = nch - 1; c >= 0; --c) {
    const int64_t slot = sq.slot0 + c, tok = sq.tok0 + int64_t(c) * kC;
    const uint32_t bytes = uint32_t(min(kC, sq.len - c * kC)) * uint32_t(sv) * 4u;
    const int b = c & 1;
    {
      const auto out = buffer_rsrc(a.dsend + ((slot * a.Hv + hv) * a.Dv + row0) * Dk, kR * Dk * 4);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int col = 32 * wp + 16 * t + 4 * g;
        st4(dSm + fsw(li, col, Dk), dS[t]);
        BufIO<float>::st4(out, uint32_t(li * Dk + col), dS[t]);
      }
    }
    __syncthreads();
    {
      const f32x4 x = dot_rows(dSm, so, Kb[b], ko, 0) + dot_rows(dSm, so, Kb[b], ko, 1);
      st4(Wd + ip * kLW + 4 * g, Gs[b][kC + ip] * x + ld4(Zs + ip * kLW + 4 * g));
    }
    __syncthreads();
    {
      const f32x4 wv = tri_cols(Wd, Tb, wp, ip, g, li);
      const f32x4 dv = Gs[b][2 * kC + ip] * wv;
      st4(We + ip * kLW + 4 * g, -Gs[b][ip] * dv);
      const auto wr = buffer_rsrc(a.w + tok * sv + hv * a.Dv + row0, bytes);
      const auto vr = buffer_rsrc(a.dv + tok * sv + hv * a.Dv + row0, bytes);
      BufIO<float>::st4(wr, uint32_t(ip * sv + 4 * g), wv);
      BufIO<float>::st4(vr, uint32_t(ip * sv + 4 * g), dv);
      watch(bad, wv);
    }
    __syncthreads();
    const float glast = Gs[b][kC - 1];
    f32x4 up[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) up[t] = ld4(Xs + li * kLX + 32 * wp + 16 * t + 4 * g);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      dot_cols(up, Kb[b], uo, rows4(We, 32 * h + 4 * g, li), rows4(We, 32 * h + 16 + 4 * g, li), h);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) dS[t] = glast * dS[t] + up[t];
  }
  watch(bad, dS[0]), watch(bad, dS[1]);
  raise(a.flag, bad);
  if (a.ds0) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) a.ds0[srow * Dk + 32 * wp + 16 * t + 4 * g + jj] = dS[t][jj];
  }
}

// sum16 in 64 bits.
__device__ __forceinline__ double sum16d(double x) {
  const auto add = [&x](auto ctrl) {
    constexpr int c = decltype(ctrl)::value;
    const int64_t b = __builtin_bit_cast(int64_t, x);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0, int(b), c, 0xf, 0xf, false);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0, int(b >> 32), c, 0xf, 0xf, false);
    x += __builtin_bit_cast(double, int64_t(uint64_t(hi) << 32 | lo));
  };
  using std::integral_constant;
  add(integral_constant<int, 0xb1>{}), add(integral_constant<int, 0x4e>{});
  add(integral_constant<int, 0x141>{}), add(integral_constant<int, 0x140>{});
  return x;
}

// ---- the gradients of a chunk ---------------------------------------------------------------------------------------

// The key tile (16 positions) that accumulator mi of the wave at position tile pw, half hw holds in dP and dM: tiles
// m <= pw only, dealt so that both halves have some.
__device__ __forceinline__ int key_tile(int pw, int hw, int mi) { return pw < 2 ? hw + 2 * mi : 2 * hw + mi; }

// One work item per (chunk slot, key head), its value heads in turn with dq and dk summed in registers, so in a fixed
// order; as many blocks as CUs, each looping over items. Per value head the state rows come in blocks of 32: S0, dS,
// dY, e and w through registers into one of two LDS buffers while the products run on the other. Wave (pw, hw) holds
// positions 16 pw .. and, of the 128 columns, 64 hw .. .
constexpr int kBlk = 32;
// x[t] += the sum over the rows r + e of a[e] times column c + 16 t of m (fsw), four sums side by side.
__device__ __forceinline__ void add4(f32x4 (&x)[4], const f32x4& a, const float* m, int r, int c) {
  f32x4 u[4], y[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) u[t] = zero4(), y[t] = cols4(m, r, c + 16 * t);
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int t = 0; t < 4; ++t) u[t] = mmaf(u[t], a[e], y[t][e]);
#pragma unroll
  for (int t = 0; t < 4; ++t) x[t] += u[t];
}
constexpr int oS = 0, oDS = oS + kBlk * Dk, oY = oDS + kBlk * Dk, oE = oY + kC * kBlk, oW = oE + kC * kBlk;
constexpr int kBuf = oW + kC * kBlk;
constexpr int eQ = 0, eN = eQ + kC * Dk, eX = eN + kC * kC;  // after the row blocks, in the same bytes: Q rows, N, X
static_assert(eX + kC * kC <= 2 * kBuf, "the 64 x 64 part fits in the row blocks' bytes");

__global__ __launch_bounds__(512) void f32_bwd_grads_kernel(F32Args a) {
  __shared__ __align__(16) float sm[2 * kBuf], Kr[kC * Dk];
  __shared__ __align__(16) float gam[kC], dec[kC], bet[kC];
  __shared__ double rowx[2][kC], colx[4][kC];
  __shared__ float vpos[2][kC], hpos[2][kC], bpos[kC], red[8];
  const int grp = a.Hv / a.Hk, total = int(a.NC) * a.Hk;
  const int tid = threadIdx.x;
  // The two waves of a SIMD hold position tiles p and 3 - p: the triangular products, which grow with p, even out.
  const int hw = __builtin_amdgcn_readfirstlane(tid >> 8);
  const int pw = __builtin_amdgcn_readfirstlane(((tid >> 6) ^ (3 * (tid >> 8))) & 3);
  const int sk = a.Hk * Dk, sv = a.Hv * a.Dv, nb = a.Dv / kBlk;
  // The lane's places, re-formed where they are used from an opaque copy of the thread index, so that their address
  // expressions are not held (spilled) across the loops.
  struct Lane {
    int lt, g, li, ip, i0, col;
  };
  const auto lane_of = [&] {
    int lt = tid;
    asm volatile("" : "+v"(lt));
    const int g = (lt >> 4) & 3, li = lt & 15;
    return Lane{lt, g, li, 16 * pw + li, 16 * pw + 4 * g, 64 * hw + li};
  };
  struct Item {
    int64_t slot, tok;
    int hk, L;
  };
  const auto item_at = [&](int id) {
    const int wid = xcd_remap(id, total);
    const int64_t slot = wid / a.Hk;
    const SlotPos sp = slot_pos(a.tab, slot);
    return Item{slot, sp.tok, wid % a.Hk, sp.L};
  };
  f32x4 xs[2], ys[2], dyv, ev, wv;  // a row block in flight
  const auto load_block = [&](const Item& it, int hv, int r0) {
    const int64_t st = ((it.slot * a.Hv + hv) * a.Dv + r0) * Dk + 4 * tid, at = (it.tok * a.Hv + hv) * a.Dv + r0;
    xs[0] = ld4(a.ckpt + st), xs[1] = ld4(a.ckpt + st + 2048);
    ys[0] = ld4(a.dsend + st), ys[1] = ld4(a.dsend + st + 2048);
    const uint32_t bytes = uint32_t(it.L) * uint32_t(sv) * 4u, off = uint32_t((tid >> 3) * sv + 4 * (tid & 7)) * 4u;
    dyv = as_f4(buf_ld16(buffer_rsrc(a.dy + at, bytes), off));
    ev = as_f4(buf_ld16(buffer_rsrc(a.e_res + at, bytes), off));
    wv = as_f4(buf_ld16(buffer_rsrc(a.w + at, bytes), off));
  };
  float bad = 0.f;
  {
    const Item first = item_at(blockIdx.x);
    load_block(first, first.hk * grp, 0);
  }
  for (int id = blockIdx.x; id < total; id += gridDim.x) {
    const Item cur = item_at(id);
    const int hk = cur.hk;
    const uint32_t kbytes = uint32_t(cur.L) * uint32_t(sk) * 4u;
    const int64_t kat = cur.tok * sk + hk * Dk;
    __syncthreads();  // the previous item's readers of the K rows are done
    {
      const auto kr = buffer_rsrc(a.k + kat, kbytes);
      uint4 kv[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int e = tid + 512 * j;
        kv[j] = buf_ld16(kr, uint32_t((e >> 5) * sk + (e & 31) * 4) * 4u);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int e = tid + 512 * j;
        st4(Kr + fsw(e >> 5, (e & 31) * 4, Dk), as_f4(kv[j]));
      }
    }
    f32x4 dQ[4], dK[4], kk[2];  // dQ, dK: rows i0 + jj, columns col + 16 t; kk = K K^T: columns of the key tiles
#pragma unroll
    for (int t = 0; t < 4; ++t) dQ[t] = zero4(), dK[t] = zero4();
    for (int h = 0; h < grp; ++h) {
      const int hv = hk * grp + h;
      // The head whose first block the last row block reads ahead: the group's next, the next item's first, or this
      // one again (unused).
      Item nx = cur;
      int nhv = hv;
      if (h + 1 < grp) {
        nhv = hv + 1;
      } else if (id + int(gridDim.x) < total) {
        nx = item_at(id + gridDim.x);
        nhv = nx.hk * grp;
      }
      const auto load_next = [&](int b) {
        if (b < nb)
          load_block(cur, hv, b * kBlk);
        else
          load_block(nx, nhv, 0);
      };
      float sds = 0.f, bsum = 0.f;
      const auto put_block = [&](float* buf) {
        const int r = tid >> 5, c = (tid & 31) * 4, at = psw(tid >> 3, 4 * (tid & 7));
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          st4(buf + oS + fsw(r + 16 * j, c, Dk), xs[j]), st4(buf + oDS + fsw(r + 16 * j, c, Dk), ys[j]);
#pragma unroll
          for (int e = 0; e < 4; ++e) sds = fmaf(xs[j][e], ys[j][e], sds);
        }
        st4(buf + oY + at, dyv), st4(buf + oE + at, ev), st4(buf + oW + at, wv);
#pragma unroll
        for (int e = 0; e < 4; ++e) bsum = fmaf(ev[e], wv[e], bsum);
      };
      const TileF* tile = a.tiles + (cur.slot * a.Hv + hv);
      __syncthreads();  // the previous head's end phase is done
      if (tid < kC) gam[tid] = tile->gam[tid], dec[tid] = tile->dec[tid], bet[tid] = tile->beta[tid];
      put_block(sm);
      load_next(1);
      if (h == 0) {
        const auto [lt, g, li, ip, i0, col] = lane_of();
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) {
          const int m = key_tile(pw, hw, mi);
          kk[mi] = zero4();
          if (m <= pw) {
            const RowOff i(ip, g, li), j(16 * m + li, g, li);
            kk[mi] = dot_rows(Kr, i, Kr, j, 0) + dot_rows(Kr, i, Kr, j, 1);
          }
        }
      }
      f32x4 dQi[4], dKa[4], dKb[4], dP[2], dM[2];  // dY S0, w S0, e dS; dY e^T, w e^T
#pragma unroll
      for (int t = 0; t < 4; ++t) dQi[t] = zero4(), dKa[t] = zero4(), dKb[t] = zero4();
#pragma unroll
      for (int mi = 0; mi < 2; ++mi) dP[mi] = zero4(), dM[mi] = zero4();
      for (int b = 0; b < nb; ++b) {
        __syncthreads();  // this block is in LDS; the products of the one before are done
        const auto [lt, g, li, ip, i0, col] = lane_of();
        const float* buf = sm + (b & 1) * kBuf;
        if (b + 1 < nb) {
          put_block(sm + ((b + 1) & 1) * kBuf);
          load_next(b + 2);
        }
#pragma unroll 1
        for (int s = 0; s < 2; ++s) {
          const int at = psw(ip, 16 * s + 4 * g);
          const f32x4 ya = ld4(buf + oY + at), wa = ld4(buf + oW + at), ea = ld4(buf + oE + at);
#pragma unroll
          for (int mi = 0; mi < 2; ++mi) {
            const int m = key_tile(pw, hw, mi);
            if (m <= pw) {
              const f32x4 em = ld4(buf + oE + psw(16 * m + li, 16 * s + 4 * g));
              f32x4 u = zero4(), v = zero4();
#pragma unroll
              for (int e = 0; e < 4; ++e) u = mmaf(u, ya[e], em[e]), v = mmaf(v, wa[e], em[e]);
              dP[mi] += u, dM[mi] += v;
            }
          }
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const f32x4 s0 = cols4(buf + oS, 16 * s + 4 * g, col + 16 * t), ds = cols4(buf + oDS, 16 * s + 4 * g, col + 16 * t);
            f32x4 u0 = zero4(), u1 = zero4(), u2 = zero4();
#pragma unroll
            for (int e = 0; e < 4; ++e) u0 = mmaf(u0, ya[e], s0[e]), u1 = mmaf(u1, wa[e], s0[e]), u2 = mmaf(u2, ea[e], ds[e]);
            dQi[t] += u0, dKa[t] += u1, dKb[t] += u2;
          }
        }
      }
      {
        const auto [lt, g, li, ip, i0, col] = lane_of();
        // Q rows, and P's and E's entries at the lane's places of dP and dM (0 above the diagonal): asked for here, where
        // the products' registers are free again (asked for a block earlier they spill).
        uint4 qv[4];
        f32x4 pv[2], xv[2];
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) {
          const int m = key_tile(pw, hw, mi);
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) {
            const int at = tri_off(i0 + jj, 16 * m + li);
            pv[mi][jj] = m <= pw ? tile->p[at] : 0.f, xv[mi][jj] = m <= pw ? tile->e[at] : 0.f;
          }
        }
        const auto qr = buffer_rsrc(a.q + kat, kbytes);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int e = lt + 512 * j;
          qv[j] = buf_ld16(qr, uint32_t((e >> 5) * sk + (e & 31) * 4) * 4u);
        }
        __syncthreads();
        // E1: N and X, then Q, into the row blocks' bytes; the terms of dG that N and X give (row sums, column sums).
        // Row and column sums add the same values with opposite signs, and dg adds them up again along the positions:
        // in 64 bits, so that what cancels cancels.
        double rx[4] = {0.0, 0.0, 0.0, 0.0};
        const f32x4 bp = ld4(bet + i0);
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) {
          const int mt = key_tile(pw, hw, mi), m = 16 * mt + li;
          const float bm = bet[m];
          const f32x4 dp = bm * dP[mi] * xv[mi];  // E is 0 above the diagonal
          f32x4 dm = -bm * bp * dM[mi] * xv[mi];
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) dm[jj] = m < i0 + jj ? dm[jj] : 0.f;
          const f32x4 d = bm * dP[mi] * pv[mi] + dm * kk[mi];
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) rx[jj] += d[jj];
          if (mt <= pw) {
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) sm[eN + fsw(i0 + jj, m, kC)] = dp[jj], sm[eX + fsw(i0 + jj, m, kC)] = dm[jj];
          }
          double cx = (double(d[0]) + d[1]) + (double(d[2]) + d[3]);
          cx += __shfl_xor(cx, 16), cx += __shfl_xor(cx, 32);
          colx[pw][m] = cx;  // the same bits in the four lane groups
        }
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) rowx[hw][i0 + jj] = sum16d(rx[jj]);
        bsum += dpp_mov<0xb1>(bsum), bsum += dpp_mov<0x4e>(bsum), bsum += dpp_mov<0x141>(bsum);
        bpos[tid >> 3] = bsum;  // the eight lanes of a position
        red[tid >> 6] = swap32_sum(swap16_sum(sum16(sds)));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int e = lt + 512 * j;
          st4(sm + eQ + fsw(e >> 5, (e & 31) * 4, Dk), as_f4(qv[j]));
        }
      }
      __syncthreads();
      {
      const auto [lt, g, li, ip, i0, col] = lane_of();
      // E2: the head's dQ and dK and the rest of dG's terms.
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const int i = i0 + jj;
        const float gi = gam[i], gb = gi * bet[i], db = dec[i] * bet[i];
        float qd = 0.f, ka = 0.f, kb = 0.f;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float kx = Kr[fsw(i, col + 16 * t, Dk)];
          qd = fmaf(sm[eQ + fsw(i, col + 16 * t, Dk)], dQi[t][jj], qd);
          ka = fmaf(kx, dKa[t][jj], ka), kb = fmaf(kx, dKb[t][jj], kb);
          dQ[t][jj] = fmaf(gi, dQi[t][jj], dQ[t][jj]);
          dK[t][jj] += db * dKb[t][jj] - gb * dKa[t][jj];
        }
        const float hs = db * kb;
        vpos[hw][i] = sum16(gi * qd - gb * ka);
        hpos[hw][i] = sum16(hs);
      }
      for (int m = 0; m <= pw; ++m) {
        const int at = fsw(ip, 16 * m + 4 * g, kC);
        const f32x4 na = ld4(sm + eN + at), xa = ld4(sm + eX + at);
        add4(dQ, na, Kr, 16 * m + 4 * g, col), add4(dK, xa, Kr, 16 * m + 4 * g, col);
      }
      for (int I = pw; I < 4; ++I) {
        const int i = 16 * I + 4 * g;
        f32x4 nt, xt;
#pragma unroll
        for (int e = 0; e < 4; ++e) nt[e] = sm[eN + fsw(i + e, ip, kC)], xt[e] = sm[eX + fsw(i + e, ip, kC)];
        add4(dK, nt, sm + eQ, i, col), add4(dK, xt, Kr, i, col);
      }
      __syncthreads();
      }
      // E3 (one wave): dG per position, dg = its reverse cumulative sum (lane l takes position 63 - l), and dbeta.
      if (tid < kC) {
        const int t = kC - 1 - tid;
        float sds_all = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) sds_all += red[j];
        // exp(G_63 - G_j) at a position j counts at the chunk's end and against j: sum and scan in 64 bits, as above.
        const double hs = double(hpos[0][t]) + hpos[1][t];
        double vd = double(vpos[0][t]) + vpos[1][t] - hs + rowx[0][t] + rowx[1][t] -
                    ((colx[0][t] + colx[1][t]) + (colx[2][t] + colx[3][t]));
        double hsum = hs;
#pragma unroll
        for (int off = 1; off < kC; off <<= 1) hsum += __shfl_xor(hsum, off);
        if (t == kC - 1) vd += hsum + gam[kC - 1] * sds_all;
#pragma unroll
        for (int off = 1; off < kC; off <<= 1) {
          const double u = __shfl_up(vd, off);
          if (tid >= off) vd += u;
        }
        const float v = float(vd);
        if (t < cur.L) {
          const int64_t at = (cur.tok + t) * a.Hv + hv;
          a.dg[at] = v, a.dbeta[at] = bpos[t];
          bad = fmaf(v, 0.f, fmaf(bpos[t], 0.f, bad));
        }
      }
    }
    const auto [lt, g, li, ip, i0, col] = lane_of();
    const auto dqr = buffer_rsrc(a.dq + kat, kbytes), dkr = buffer_rsrc(a.dk + kat, kbytes);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      watch(bad, dQ[t]), watch(bad, dK[t]);
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const uint32_t at = uint32_t((i0 + jj) * sk + col + 16 * t);
        BufIO<float>::st(dqr, at, dQ[t][jj]), BufIO<float>::st(dkr, at, dK[t][jj]);
      }
    }
  }
  raise(a.flag, bad);
}

// ---- host -----------------------------------------------------------------------------------------------------------

size_t tiles_bytes(const Problem& p) { return size_t(p.NC) * p.Hv * sizeof(TileF); }
size_t dsend_bytes(const Problem& p) { return size_t(p.NC) * p.Hv * p.Dv * Dk * 4; }
size_t w_bytes(const Problem& p) { return size_t(p.BT) * p.Hv * p.Dv * 4; }

F32Args base_args(const Problem& p, void* ws, size_t flag_at) {
  F32Args a{};
  a.NC = p.NC, a.Hk = p.Hk, a.Hv = p.Hv, a.Dv = p.Dv, a.N = p.N, a.nblk = p.Dv / kR, a.g_is_log = p.g_is_log;
  a.tab = p.tab;
  a.tiles = static_cast<TileF*>(ws);
  a.flag = reinterpret_cast<int*>(static_cast<unsigned char*>(ws) + flag_at);
  return a;
}

hipError_t device_cus(int* cus) {
  int dev = 0;
  const hipError_t e = hipGetDevice(&dev);
  return e != hipSuccess ? e : hipDeviceGetAttribute(cus, hipDeviceAttributeMultiprocessorCount, dev);
}

template <bool kBwd>
void launch_prep(const F32Args& a, int cus, hipStream_t s) {
  // Four blocks (33 KB of LDS, 128 registers) fit a CU: a block per value head while those all fit at once, else per
  // key head.
  const int hpb = a.NC * a.Hv <= int64_t(4) * cus ? 1 : a.Hv / a.Hk;
  hipLaunchKernelGGL(f32_prep_kernel<kBwd>, dim3(int(a.NC) * (a.Hv / hpb)), dim3(256), 0, s, a, hpb);
}

}  // namespace

bool chunk_f32_takes(const Problem& p, int steps, size_t ws_bytes) {
  if (p.in_bf16 || p.Dk != Dk || p.Dv % kBlk) return false;
  // A chunk's rows of k and of v are addressed by 32-bit byte offsets.
  if (int64_t(p.Hk) * Dk * kC * 4 >= (int64_t(1) << 31) || int64_t(p.Hv) * p.Dv * kC * 4 >= (int64_t(1) << 31)) return false;
  int longest = p.T;
  if (p.tab.n > 0) {
    longest = 0;
    for (int i = 0; i < p.tab.n; ++i)
      if (p.tab.tok0[i + 1] - p.tab.tok0[i] > longest) longest = p.tab.tok0[i + 1] - p.tab.tok0[i];
  }
  return longest >= steps && p.NC * p.Hv < (int64_t(1) << 30) &&
         tiles_bytes(p) + dsend_bytes(p) + w_bytes(p) <= ws_bytes;
}

hipError_t chunk_f32_fwd(const Problem& p, const FwdPtrs& f, void* ws, size_t flag_at, const int** redo, hipStream_t s) {
  F32Args a = base_args(p, ws, flag_at);
  a.q = static_cast<const float*>(f.q), a.k = static_cast<const float*>(f.k), a.v = static_cast<const float*>(f.v);
  a.g = f.g, a.beta = static_cast<const float*>(f.beta), a.s0 = f.s0;
  a.y = static_cast<float*>(f.y), a.s_out = f.s_out, a.ckpt = f.ckpt;
  a.e_res = f.ckpt ? f.ckpt + int64_t(p.NC) * p.Hv * p.Dv * p.Dk : nullptr;
  int cus = 0;
  hipError_t e = device_cus(&cus);
  if (e != hipSuccess) return e;
  launch_prep<false>(a, cus, s);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(f32_fwd_kernel, dim3(a.nblk * a.Hv * a.N), dim3(768), 0, s, a);
  *redo = a.flag;
  return hipGetLastError();
}

hipError_t chunk_f32_bwd(const Problem& p, const BwdPtrs& b, void* ws, size_t flag_at, const int** redo, hipStream_t s) {
  F32Args a = base_args(p, ws, flag_at);
  unsigned char* at = static_cast<unsigned char*>(ws) + tiles_bytes(p);
  a.dsend = reinterpret_cast<float*>(at), a.w = reinterpret_cast<float*>(at + dsend_bytes(p));
  a.q = static_cast<const float*>(b.q), a.k = static_cast<const float*>(b.k), a.v = static_cast<const float*>(b.v);
  a.g = b.g, a.beta = static_cast<const float*>(b.beta);
  a.ckpt = const_cast<float*>(b.ckpt), a.e_res = a.ckpt + int64_t(p.NC) * p.Hv * p.Dv * p.Dk;
  a.dy = static_cast<const float*>(b.dy), a.ds_out = b.ds_out;
  a.dq = static_cast<float*>(b.dq), a.dk = static_cast<float*>(b.dk), a.dv = static_cast<float*>(b.dv);
  a.dg = b.dg, a.dbeta = static_cast<float*>(b.dbeta), a.ds0 = b.ds0;
  int cus = 0;
  hipError_t e = device_cus(&cus);
  if (e != hipSuccess) return e;
  launch_prep<true>(a, cus, s);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(f32_bwd_state_kernel, dim3(a.nblk * a.Hv * a.N), dim3(768), 0, s, a);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  const int total = int(a.NC) * a.Hk, grid = total <= cus ? total : (cus >= 8 ? cus & ~7 : cus);
  hipLaunchKernelGGL(f32_bwd_grads_kernel, dim3(grid), dim3(512), 0, s, a);
  *redo = a.flag;
  return hipGetLastError();
}

}  // namespace qbgdn
