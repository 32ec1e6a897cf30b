// symeig.hip -- symmetric eigensolver of the rSVD pipeline on the GPU, the
// device replacement of LAPACKE_dsyev on BB^T (MKL/mvf.c:1206-1209, vnum = 2,
// called from rra.c:191) and of compute_evals_and_evecs_of_symm_matrix.
//
// Two-sided cyclic block Jacobi.  The n columns are cut into blocks of B = 16;
// a round pairs the blocks with the circle method (every block meets every
// other once per sweep).  A round has two roles, which one launch
// (symj_step_kernel) runs side by side -- the apply of round r next to the
// solve of round r + 1:
//   solve : one workgroup per block pair forms the pair's S x S (S = 2B)
//           diagonal tile H of G and runs an inner sweep of two-sided Jacobi
//           on it (B disjoint rotations per step; all pairs in the first round
//           of a sweep, only the cross-block pairs afterwards), accumulating
//           the S x S orthogonal J with H <- J^T H J;
//   apply : every S x S tile of G in pair order becomes J_a^T T J_b (the
//           upper tiles are computed and mirrored, so G stays exactly
//           symmetric) and every S-row strip of V's pair columns becomes
//           V J -- hundreds of independent workgroups.
// Unlike one-sided Jacobi no Gram matrix is formed: the tile is read from G
// itself, and the O(n^2) work of a round is spread over the whole GPU.
// A sweep in which no pair met had |g_pq| > 1e-10 sqrt(|g_pp g_qq|) ends the
// loop: Jacobi converges quadratically, so that sweep's rotations leave the
// off-diagonals near the rounding floor.
// Off-diagonals below 4 eps ||G||_F are not rotated (they are below the
// absolute accuracy of any backward-stable eigensolver, LAPACK's included).
#include <cmath>
#include <cstring>

#include "jacobi_rot.h"
#include "rsvd_internal.h"

namespace rsvd {

namespace {


__device__ __forceinline__ int player(int pos, int r, int N) {
  int x = pos - 1 + r;  // 0 <= r < N - 1
  x = x >= N - 1 ? x - (N - 1) : x;
  return pos == 0 ? 0 : 1 + x;
}

// The columns of block pair w in round r: slot s (0..2B-1) is column
// first[s / B] + s % B, or -1 when the slot is padding (dummy block or past n).
template <int B>
struct PairCols {
  int64_t first[2];
  int64_t n;
  __device__ __forceinline__ PairCols(int w, int r, int N, int nblocks, int64_t n_) : n(n_) {
    const int ba = player(w, r, N), bb = player(N - 1 - w, r, N);
    first[0] = ba < nblocks ? (int64_t)ba * B : -1;
    first[1] = bb < nblocks ? (int64_t)bb * B : -1;
  }
  __device__ __forceinline__ int64_t col(int s) const {
    const int64_t f = first[s >= B];
    const int64_t c = f + (s & (B - 1));
    return (f >= 0 && c < n) ? c : -1;
  }
};

template <int B>
__device__ __forceinline__ int64_t pair_col(int w, int s, int r, int N, int nblocks, int64_t n) {
  return PairCols<B>(w, r, N, nblocks, n).col(s);
}

// The inner sweep.  Round 0 of a sweep meets every pair of its 2B columns: first
// the pairs inside each of the two blocks (B - 1 steps, jac_within), then the
// B x B cross pairs (B steps, jac_cross); the other rounds only the cross pairs.
// Every pair of columns meets once per sweep, and the inner steps per sweep are
// about n instead of 2n.

// A 64-bit value moved inside each 16-lane row of the wave (a data-parallel
// move, no trip through the LDS crossbar): CTRL 0x150 (row_newbcast:0) gives
// every lane lane 0's, 0x12f (row_ror:15) the next lane's, 0x121 (row_ror:1) the
// previous lane's, both cyclically.
template <int CTRL>
__device__ __forceinline__ double row_move(double v) {
  union {
    double d;
    int i[2];
  } u = {v};
  u.i[0] = __builtin_amdgcn_mov_dpp(u.i[0], CTRL, 0xf, 0xf, true);
  u.i[1] = __builtin_amdgcn_mov_dpp(u.i[1], CTRL, 0xf, 0xf, true);
  return u.d;
}
__device__ __forceinline__ double row_first(double v) { return row_move<0x150>(v); }
__device__ __forceinline__ double row_next(double v) { return row_move<0x12f>(v); }
__device__ __forceinline__ double row_prev(double v) { return row_move<0x121>(v); }

// The pairs inside the two blocks of the S x S tile (S = 2B) in LDS, H in Ha
// (double-buffered with Hb), J accumulated in Jl (row-major, padded HP): step m
// rotates column i against i xor m in both blocks.  Thread (bi, x) (bi = t / B,
// x = t % B) computes the rotation of pair bj = (bi + x) mod B -- the 16 lanes of
// a row of a wave compute the 16 rotations, its lane 0 that of pair bi, which
// the row takes from there -- applies R_bi^T . R_bj to the 2 x 2 block of H at
// (pair bi rows, pair bj columns) -- the blocks partition H -- and R_bi to rows
// 2 x, 2 x + 1 of J's columns of pair bi.  One barrier per step.  Returns the
// buffer holding the final H; *any_sig |= a rotation of the lane's counted.
template <int B>
__device__ double* jac_within(double* Ha, double* Hb, double* Jl, float flo, RotStop stop,
                              bool* any_sig) {
  constexpr int S = 2 * B, HP = S + 1;
  const int tid = threadIdx.x;
  const int bi = tid / B, x = tid % B, bj = (bi + x) % B;
  double* Hc = Ha;
  double* Hn = Hb;
  // pair k of step m: the (k mod B/2)-th i without m's top bit, in block k / (B/2)
  auto pair = [](int k, int m, int top, int* p, int* q) {
    const int h = k & (B / 2 - 1), lo = h & (top - 1);
    const int i = 2 * (h - lo) + lo, base = (k / (B / 2)) * B;
    *p = base + i;
    *q = base + (i ^ m);
  };
  for (int m = 1; m < B; ++m) {
    const int top = 1 << (31 - __builtin_clz(m));
    int pi, qi, pj, qj;
    pair(bi, m, top, &pi, &qi);
    pair(bj, m, top, &pj, &qj);
    const int x0 = 2 * x;
    // every LDS read of the step first, so that one latency covers them
    const double aj = Hc[pj * HP + pj], bbj = Hc[qj * HP + qj], gj = Hc[pj * HP + qj];
    const double h00 = Hc[pi * HP + pj], h01 = Hc[pi * HP + qj];
    const double h10 = Hc[qi * HP + pj], h11 = Hc[qi * HP + qj];
    const double j00 = Jl[x0 * HP + pi], j01 = Jl[x0 * HP + qi];
    const double j10 = Jl[(x0 + 1) * HP + pi], j11 = Jl[(x0 + 1) * HP + qi];
    double cj, sj;
    bool sgj;
    rotation(aj, bbj, gj, flo, stop, &cj, &sj, &sgj);
    *any_sig |= sgj;
    const double ci = row_first(cj), si = row_first(sj);
    // X = H_blk R_j, then R_i^T X
    const double x00 = cj * h00 - sj * h01, x01 = sj * h00 + cj * h01;
    const double x10 = cj * h10 - sj * h11, x11 = sj * h10 + cj * h11;
    const double y01 = ci * x01 - si * x11;
    double y10 = si * x00 + ci * x10;
    if (x == 0) y10 = y01;  // a diagonal block stays exactly symmetric
    Hn[pi * HP + pj] = ci * x00 - si * x10;
    Hn[pi * HP + qj] = y01;
    Hn[qi * HP + pj] = y10;
    Hn[qi * HP + qj] = si * x01 + ci * x11;
    Jl[x0 * HP + pi] = ci * j00 - si * j01;
    Jl[x0 * HP + qi] = si * j00 + ci * j01;
    Jl[(x0 + 1) * HP + pi] = ci * j10 - si * j11;
    Jl[(x0 + 1) * HP + qi] = si * j10 + ci * j11;
    __syncthreads();
    double* tmp = Hc;
    Hc = Hn;
    Hn = tmp;
  }
  return Hc;
}

// The cross pairs: step t rotates column p_k = k of block a against column
// q_k = (k + t) mod B of block b.  Thread (bi, x) keeps the 2 x 2 block of H at
// (pair bi rows, pair bj columns), bj = (bi + x) mod B, and rows 2 bi, 2 bi + 1 of
// J's columns of pair bj in registers.  From a step to the next p stays and q
// moves by one pair, so H(p, p) and J(p) stay, H(p, q) and J(q) come from the next
// lane of the row (a data-parallel move), and only H(q, p) and H(q, q) cross rows:
// they go through LDS (E), with the entries of the next rotations (R and E's
// diagonal).  One barrier per step (E and R double-buffered).  After B steps every
// entry is back where it started.  E: 2 B B pairs, R: 2 B pairs (LDS).
// What bounds a step is LDS traffic and latency: with H and J in LDS (19
// accesses a thread and step instead of 5) a step took 1195 cycles, here 800.
typedef double d2_t __attribute__((ext_vector_type(2)));

template <int B>
__device__ void jac_cross(const double* H, const double* Jl, d2_t* E, d2_t* R, float flo,
                          RotStop stop, bool* any_sig, double* __restrict__ Jw,
                          double* __restrict__ Hw) {
  static_assert(B == 16, "a row of 16 lanes holds the B rotations of a step");
  constexpr int S = 2 * B, HP = S + 1;
  const int tid = threadIdx.x;
  const int bi = tid / B, x = tid % B, bj = (bi + x) % B, r0 = 2 * bi;
  double h00 = H[bi * HP + bj], h01 = H[bi * HP + B + bj];
  double h10 = H[(B + bi) * HP + bj], h11 = H[(B + bi) * HP + B + bj];
  double a = H[bj * HP + bj], b = H[(B + bj) * HP + B + bj], g = H[bj * HP + B + bj];
  double jp0 = Jl[r0 * HP + bj], jq0 = Jl[r0 * HP + B + bj];
  double jp1 = Jl[(r0 + 1) * HP + bj], jq1 = Jl[(r0 + 1) * HP + B + bj];
  const int up = (tid + B) % (B * B);              // the same lane of pair bi + 1's row
  const int dj = ((bj + 1) % B) * B;               // lane 0 of pair bj + 1's row
  bool sig = false;
#pragma unroll 2
  for (int t = 0; t < B; ++t) {
    d2_t* Et = E + (t & 1) * B * B;
    d2_t* Rt = R + (t & 1) * B;
    double c, s;
    bool sg;
    rotation(a, b, g, flo, stop, &c, &s, &sg);
    sig |= sg;
    const double ci = row_first(c), si = row_first(s);
    // X = H_blk R_j, then R_i^T X
    const double x00 = c * h00 - s * h01, x01 = s * h00 + c * h01;
    const double x10 = c * h10 - s * h11, x11 = s * h10 + c * h11;
    const double y01 = ci * x01 - si * x11, y11 = si * x01 + ci * x11;
    double y10 = si * x00 + ci * x10;
    if (x == 0) y10 = y01;  // a diagonal block stays exactly symmetric
    h00 = ci * x00 - si * x10;
    h01 = row_next(y01);
    Et[tid] = d2_t{row_prev(y10), y11};
    if (x == 0) Rt[bi] = d2_t{h00, h01};
    const double n0 = s * jp0 + c * jq0, n1 = s * jp1 + c * jq1;
    jp0 = c * jp0 - s * jq0;
    jp1 = c * jp1 - s * jq1;
    jq0 = row_next(n0);
    jq1 = row_next(n1);
    __syncthreads();
    const d2_t e = Et[up], r = Rt[bj];
    b = Et[dj][1];
    h10 = e[0];
    h11 = e[1];
    a = r[0];
    g = r[1];
  }
  *any_sig |= sig;
  Jw[r0 * S + bj] = jp0;
  Jw[r0 * S + B + bj] = jq0;
  Jw[(r0 + 1) * S + bj] = jp1;
  Jw[(r0 + 1) * S + B + bj] = jq1;
  Hw[bi * S + bj] = h00;
  Hw[bi * S + B + bj] = h01;
  Hw[(B + bi) * S + bj] = h10;
  Hw[(B + bi) * S + B + bj] = h11;
}

// The whole inner sweep of pair w; J and the final tile out (row-major S x S
// each).  Ha holds the tile, Jl the identity; Hb is scratch.  The flag is set
// when a rotation counted for the stop.
template <int B>
__device__ void jac_solve(double* Ha, double* Hb, double* Jl, d2_t* R, bool cross, float flo,
                          RotStop stop, int w, double* __restrict__ Jout,
                          double* __restrict__ Hout, unsigned long long* __restrict__ flag) {
  constexpr int S = 2 * B, HP = S + 1;
  static_assert(2 * B * B * sizeof(d2_t) <= S * HP * sizeof(double), "E fits a tile's region");
  bool sig = false;
  double* Hc = cross ? Ha : jac_within<B>(Ha, Hb, Jl, flo, stop, &sig);
  d2_t* E = reinterpret_cast<d2_t*>(Hc == Ha ? Hb : Ha);
  jac_cross<B>(Hc, Jl, E, R, flo, stop, &sig, Jout + (size_t)w * S * S, Hout + (size_t)w * S * S);
  if (__any(sig) && (threadIdx.x & 63) == 0) atomicOr(flag, 1ULL);
}

// First round of the iteration: the pair tiles are read from G.
template <int B>
__global__ void __launch_bounds__(256)
symj_solve_kernel(int64_t n, const double* __restrict__ G, int64_t ldg, int nblocks, int N,
                  int round, const double* __restrict__ scal, RotStop stop,
                  double* __restrict__ Jout, double* __restrict__ Hout,
                  unsigned long long* __restrict__ flag) {
  constexpr int S = 2 * B, HP = S + 1;
  __shared__ __align__(16) double Ha[S * HP], Hb[S * HP], Jl[S * HP];
  __shared__ d2_t R[2 * B];
  __shared__ int64_t cols[S];
  const int w = blockIdx.x;
  const int tid = threadIdx.x;
  if (tid < S) cols[tid] = pair_col<B>(w, tid, round, N, nblocks, n);
  __syncthreads();
  for (int e = tid; e < S * S; e += 256) {
    const int i = e % S, j = e / S;
    const int64_t ci = cols[i], cj = cols[j];
    Ha[i * HP + j] = (ci >= 0 && cj >= 0) ? G[ci + cj * ldg] : 0.0;
    Jl[i * HP + j] = (i == j) ? 1.0 : 0.0;
  }
  const float flo = (float)scal[0];
  __syncthreads();
  jac_solve<B>(Ha, Hb, Jl, R, round > 0, flo, stop, w, Jout, Hout, flag);
}

typedef double d4_t __attribute__((ext_vector_type(4)));

// The 16 x 16 block (bm, bn) of the product op(P) Q with inner dimension 32,
// P and Q in LDS (row-major, leading dimensions lp and lq; op(P) = P^T reads
// P[k][m]), on the FP64 matrix cores: eight v_mfma_f64_16x16x4f64 steps along
// k.  srcA carries Q[k][n] and srcB op(P)[m][k] (lane l: n or m = l % 16,
// k = 4 s + l / 16), so lane l's accumulator register r holds
// C[16 bm + l % 16][16 bn + 4 r + l / 16].
template <bool TA>
__device__ __forceinline__ d4_t blk_mfma(const double* __restrict__ P, int lp,
                                         const double* __restrict__ Q, int lq, int bm, int bn) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  d4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const int k = 4 * s + lk;
    const double q = Q[k * lq + 16 * bn + li];
    const double p = TA ? P[k * lp + 16 * bm + li] : P[(16 * bm + li) * lp + k];
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(q, p, acc, 0, 0, 0);
  }
  return acc;
}

// Stores block (bm, bn) (the layout of blk_mfma) into C (leading dimension ldc).
__device__ __forceinline__ void blk_store(const d4_t& acc, double* __restrict__ C, int ldc,
                                          int bm, int bn) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) C[(16 * bm + li) * ldc + 16 * bn + 4 * r + lk] = acc[r];
}

// The wave's 16 x 16 quadrant (wave / 2, wave % 2) of the 32 x 32 product
// op(P) Q, P and Q padded to HP = 33.  Two LDS reads per 16 multiply-adds a
// lane, where a register-blocked scalar product reads one per two.
template <bool TA>
__device__ __forceinline__ d4_t tile_mfma(const double* __restrict__ P,
                                          const double* __restrict__ Q) {
  const int wave = threadIdx.x >> 6;
  return blk_mfma<TA>(P, 33, Q, 33, wave >> 1, wave & 1);
}

__device__ __forceinline__ void tile_store(const d4_t& acc, double* __restrict__ C) {
  const int wave = threadIdx.x >> 6;
  blk_store(acc, C, 33, wave >> 1, wave & 1);
}

// Apply round r's rotations (the apply role of symj_step_kernel): blocks
// [0, ntg) take the upper pair tiles (w1 <= w2) of Gin and write J_w1^T T J_w2
// to both triangles of Gout; the rest take 2S-row strips of V (in place):
// V(rows, cols(w)) <- V(rows, cols(w)) J_w.  Every element of Gout and V is
// written by exactly one workgroup.  Every global read of a workgroup is
// issued before its first wait (one memory latency), ahead of the skip test;
// padding slots read an in-bounds element and drop it.
template <int B>
__device__ void jac_apply(int bid, int64_t n, const double* __restrict__ Gin,
                          double* __restrict__ Gout, int64_t ldg, double* __restrict__ V,
                          int64_t ldv, int nblocks, int N, int round,
                          const double* __restrict__ Jall, int ntg, double* T, double* Ja,
                          double* Jb, double* X, bool skip) {
  static_assert(B == 16, "the tile products are 32 x 32, one 16 x 16 quadrant a wave");
  constexpr int S = 2 * B, HP = S + 1;
  const int pairs = N / 2;
  const int tid = threadIdx.x;
  if (bid < ntg) {
    int w1 = 0;
    while (bid >= pairs - w1) {
      bid -= pairs - w1;
      ++w1;
    }
    const int w2 = w1 + bid;
    const PairCols<B> pa(w1, round, N, nblocks, n), pb(w2, round, N, nblocks, n);
    const double* J1 = Jall + (size_t)w1 * S * S;
    const double* J2 = Jall + (size_t)w2 * S * S;
    // thread: row r of the tile, columns c0 + 8 it; column r of the J, rows
    // c0 + 8 it
    const int r = tid % S, c0 = tid / S;
    const int64_t gr = pa.col(r);
    double tv[4], av[4], bv[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int c = c0 + 8 * it;
      const int64_t gc = pb.col(c);
      const double g = Gin[(gr < 0 ? 0 : gr) + (gc < 0 ? 0 : gc) * ldg];
      tv[it] = (gr >= 0 && gc >= 0) ? g : 0.0;
      av[it] = J1[c * S + r];
      bv[it] = J2[c * S + r];
    }
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int c = c0 + 8 * it;
      T[r * HP + c] = tv[it];
      Ja[c * HP + r] = av[it];
      Jb[c * HP + r] = bv[it];
    }
    if (skip) return;
    __syncthreads();
    tile_store(tile_mfma<false>(T, Jb), X);  // X = T J_w2
    __syncthreads();
    // Y = J_w1^T X into T (T is not read again: its last reads were before
    // the barrier above)
    tile_store(tile_mfma<true>(Ja, X), T);
    __syncthreads();
    if (w1 == w2) {
      // diagonal pair tile: the upper triangle, mirrored
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const int c = c0 + 8 * it;
        const int64_t gc = pb.col(c);
        if (gr >= 0 && gc >= 0) Gout[gr + gc * ldg] = (r <= c) ? T[r * HP + c] : T[c * HP + r];
      }
    } else {
      const int64_t gr2 = pb.col(r);
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const int c = c0 + 8 * it;
        const int64_t gc = pb.col(c), gc2 = pa.col(c);
        if (gr >= 0 && gc >= 0) Gout[gr + gc * ldg] = T[r * HP + c];
        // mirror: row cols(w2)[r], column cols(w1)[c]
        if (gr2 >= 0 && gc2 >= 0) Gout[gr2 + gc2 * ldg] = T[c * HP + r];
      }
    }
    return;
  }
  if (V == nullptr) return;
  // V strip: rows [r0, r0 + 2S) of the pair's columns, in two S-row halves
  // (T and X).  Thread: row r of the strip, columns cq + 4 it; J_w element
  // (tid / S + 8 it, tid % S).
  bid -= ntg;
  const int w = bid % pairs;
  const int64_t r0 = (int64_t)(bid / pairs) * (2 * S);
  const PairCols<B> pc(w, round, N, nblocks, n);
  const double* Jw = Jall + (size_t)w * S * S;
  const int r = tid % (2 * S), cq = tid / (2 * S);
  const bool row_ok = r0 + r < n;
  double vv[8], jv[4];
#pragma unroll
  for (int it = 0; it < 8; ++it) {
    const int64_t gc = pc.col(cq + 4 * it);
    const double v = V[(row_ok ? r0 + r : 0) + (gc < 0 ? 0 : gc) * ldv];
    vv[it] = (gc >= 0 && row_ok) ? v : 0.0;
  }
  const int jr = tid % S, jc0 = tid / S;
#pragma unroll
  for (int it = 0; it < 4; ++it) jv[it] = Jw[(jc0 + 8 * it) * S + jr];
  double* Vh = r < S ? T + r * HP : X + (r - S) * HP;  // this thread's row of the strip
#pragma unroll
  for (int it = 0; it < 8; ++it) Vh[cq + 4 * it] = vv[it];
#pragma unroll
  for (int it = 0; it < 4; ++it) Jb[(jc0 + 8 * it) * HP + jr] = jv[it];
  if (skip) return;
  __syncthreads();
  const d4_t o1 = tile_mfma<false>(T, Jb), o2 = tile_mfma<false>(X, Jb);
  __syncthreads();
  tile_store(o1, T);
  tile_store(o2, X);
  __syncthreads();
  if (!row_ok) return;
#pragma unroll
  for (int it = 0; it < 8; ++it) {
    const int64_t gc = pc.col(cq + 4 * it);
    if (gc >= 0) V[(r0 + r) + gc * ldv] = Vh[cq + 4 * it];
  }
}

// One launch per round: the apply of round r (blocks nsolve..) and, in the
// same launch, the inner sweeps of round r1 = the next round (blocks
// 0..nsolve-1), so a round costs max(apply, solve) instead of their sum.  A
// solve workgroup builds its pair's tile of G_{r+1} = J_r^T G_r J_r itself:
// its two blocks a and b sat in pairs wa and wb of round r, so the diagonal
// blocks are sub-blocks of those pairs' final tiles (Hin, kept by round r's
// solves) and the off-diagonal block is Ja^T G_r(cols(wa), cols(wb)) Jb with
// Ja, Jb the columns of J_wa, J_wb that belong to a and b.  G is read from
// Gin and written to Gout (double-buffered), J and the tiles alternate too.
template <int B>
__global__ void __launch_bounds__(256)
symj_step_kernel(int64_t n, const double* __restrict__ Gin, double* __restrict__ Gout,
                 int64_t ldg, double* __restrict__ V, int64_t ldv, int nblocks, int N, int round,
                 int round1, int nsolve, const double* __restrict__ scal, RotStop stop,
                 const double* __restrict__ Jin, const double* __restrict__ Hin,
                 double* __restrict__ Jout, double* __restrict__ Hout, int ntg,
                 unsigned long long* __restrict__ flag,
                 const unsigned long long* __restrict__ prev) {
  constexpr int S = 2 * B, HP = S + 1, BP = B + 1;
  // Device-side stop: every launch of a sweep reads the previous sweep's
  // rotation flags (complete: that sweep's launches have finished) and does
  // nothing when they say it converged, so the host can queue a sweep before
  // it has read the last one's flags.  Read here and tested after the other
  // global reads are issued (before any global write), so one memory latency
  // covers them all.
  const bool skip = prev && *prev == 0;
  // Apply role: four S x HP regions T, Ja, Jb, X.  Solve role: Ha, Jl and
  // Tab (later Hb) S x HP each, then JBq, X3 and JAq S x BP each; no region
  // changes tenant before the inner sweep.  Both footprints let four
  // workgroups share a CU.
  constexpr int kSm = (4 * S * HP > 3 * S * HP + 3 * S * BP) ? 4 * S * HP : 3 * S * HP + 3 * S * BP;
  __shared__ __align__(16) double sm[kSm];
  __shared__ d2_t R[2 * B];
  const int tid = threadIdx.x;
  if ((int)blockIdx.x >= nsolve) {
    jac_apply<B>((int)blockIdx.x - nsolve, n, Gin, Gout, ldg, V, ldv, nblocks, N, round, Jin, ntg,
                 sm, sm + S * HP, sm + 2 * S * HP, sm + 3 * S * HP, skip);
    return;
  }
  double* Ha = sm;
  double* Jl = sm + S * HP;
  double* Tab = sm + 2 * S * HP;
  double* Hb = Tab;  // from the first inner step on
  double* JBq = sm + 3 * S * HP;  // JBq[i * BP + c] = J_wb(i, hb B + c)
  double* X3 = JBq + S * BP;      // Tab JBq
  double* JAq = X3 + S * BP;      // JAq[i * BP + c] = J_wa(i, ha B + c)
  const int w = blockIdx.x;
  // the blocks of pair w in round1 and where they sat in round r
  const int xa = player(w, round1, N), xb = player(N - 1 - w, round1, N);
  auto locate = [&](int x, int* wp, int* h) {
    const int y = x - 1 - round;
    const int pos = (x == 0) ? 0 : 1 + (y < 0 ? y + N - 1 : y);
    if (pos < N / 2) {
      *wp = pos;
      *h = 0;
    } else {
      *wp = N - 1 - pos;
      *h = 1;
    }
  };
  int wa, ha, wb, hb;
  locate(xa, &wa, &ha);
  locate(xb, &wb, &hb);
  const PairCols<B> pa(wa, round, N, nblocks, n), pb(wb, round, N, nblocks, n);
  const double* JA = Jin + (size_t)wa * S * S;
  const double* JB = Jin + (size_t)wb * S * S;
  const double* HA = Hin + (size_t)wa * S * S;
  const double* HB = Hin + (size_t)wb * S * S;
  // every global read first: thread row i of Tab (columns j0 + 8 it), rows
  // dd + B it of JAq and JBq (column dc), and entry (dd, dc) of the two diagonal
  // blocks
  const int i = tid % S, j0 = tid / S;
  const int dc = tid % B, dd = tid / B;
  const int64_t gi = pa.col(i);
  double tv[4], av[2], bv[2];
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    // padding slots read column 0 / row 0 (in bounds) and drop the value
    const int64_t gj = pb.col(j0 + 8 * it);
    const double g = Gin[(gi < 0 ? 0 : gi) + (gj < 0 ? 0 : gj) * ldg];
    tv[it] = (gi >= 0 && gj >= 0) ? g : 0.0;
  }
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    av[it] = JA[(dd + B * it) * S + ha * B + dc];
    bv[it] = JB[(dd + B * it) * S + hb * B + dc];
  }
  const double hav = HA[(ha * B + dd) * S + ha * B + dc];
  const double hbv = HB[(hb * B + dd) * S + hb * B + dc];
  // the rotation floor goes through LDS: its load then completes with the
  // others instead of being deferred to its first use in the inner sweep
  __shared__ float flo_s;
  if (tid == 0) flo_s = (float)scal[0];
  // J starts as the identity (its region has no other tenant)
#pragma unroll
  for (int it = 0; it < 4; ++it) Jl[i * HP + j0 + 8 * it] = (i == j0 + 8 * it) ? 1.0 : 0.0;
#pragma unroll
  for (int it = 0; it < 4; ++it) Tab[i * HP + j0 + 8 * it] = tv[it];
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    JAq[(dd + B * it) * BP + dc] = av[it];
    JBq[(dd + B * it) * BP + dc] = bv[it];
  }
  // diagonal blocks of the new tile from round r's final tiles
  Ha[dd * HP + dc] = hav;
  Ha[(B + dd) * HP + B + dc] = hbv;
  // the skip test after the LDS stores, so that no global read waits for it
  if (skip) return;
  __syncthreads();
  // off-diagonal block H_ab = J_a^T G_r(cols(wa), cols(wb)) J_b on the FP64
  // matrix cores: X3 = Tab JBq (S x B, waves 0 and 1), then H_ab = JAq^T X3
  // (B x B, wave 0), mirrored into H_ba
  const int wave = tid >> 6;
  if (wave < 2) blk_store(blk_mfma<false>(Tab, HP, JBq, BP, wave, 0), X3, BP, wave, 0);
  __syncthreads();
  if (wave == 0) {
    const d4_t h = blk_mfma<true>(JAq, BP, X3, BP, 0, 0);
    const int lane = tid & 63, c = lane & 15, d0 = lane >> 4;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      Ha[c * HP + B + 4 * r + d0] = h[r];
      Ha[(B + 4 * r + d0) * HP + c] = h[r];
    }
  }
  __syncthreads();
  jac_solve<B>(Ha, Hb, Jl, R, round1 > 0, flo_s, stop, w, Jout, Hout, flag);
}

// Gs = sc G with sc the power of two of unit_scale (so that no rotation has to
// scale its entries), V = I, the sweeps' flags cleared, scal = {rotation floor,
// 1 / sc}.  fro2: ||G||_F^2; where that over- or underflowed every workgroup
// finds the largest entry for itself.
__global__ void __launch_bounds__(256)
symj_prep_kernel(int64_t n, const double* __restrict__ G, int64_t ldg, double* __restrict__ Gs,
                 double* __restrict__ V, int64_t ldv, const double* __restrict__ fro2,
                 double* __restrict__ scal, unsigned long long* __restrict__ flags, int nflags) {
  __shared__ double red[256];
  const int64_t total = n * n;
  double sc = norm_scale(*fro2), fro = sqrt(*fro2) * sc;
  if (sc == 0.0) {
    double mx = 0.0;
    for (int64_t idx = threadIdx.x; idx < total; idx += 256)
      mx = fmax(mx, fabs(G[idx % n + (idx / n) * ldg]));
    red[threadIdx.x] = mx;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
      if ((int)threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
      __syncthreads();
    }
    sc = unit_scale(red[0]);
    fro = 1.0;
  }
  for (int64_t idx = blockIdx.x * (int64_t)256 + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * 256) {
    const int64_t i = idx % n, j = idx / n;
    Gs[i + j * ldg] = sc * G[i + j * ldg];
    if (V) V[i + j * ldv] = (i == j) ? 1.0 : 0.0;
  }
  if (blockIdx.x == 0) {
    for (int e = threadIdx.x; e < nflags; e += 256) flags[e] = 0;
    if (threadIdx.x == 0) {
      scal[0] = 4.0 * 2.220446049250313e-16 * fro;
      scal[1] = 1.0 / sc;
    }
  }
}

__global__ void symj_diag_kernel(int64_t n, const double* __restrict__ G, int64_t ldg,
                                 const double* __restrict__ scal, double* __restrict__ d) {
  const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (j < n) d[j] = G[j + j * ldg] * scal[1];
}

// The whole iteration for n <= kSmallN in one workgroup: G (upper triangle) and
// V live in LDS, a step is one rotation of every pair of the round-robin order.
// The block solver is launch- and latency-bound at these sizes (a round of one
// block pair takes as long as one of seventeen): a whole call at n = 26 took
// 0.39 ms with it and 0.19 ms here, at n = 40 0.66 and 0.32 ms.  A step's LDS
// traffic, all of H and V, grows as n^2 and there are n steps: at n = 64 this
// kernel takes 0.72 ms, more than the block solver's three rounds a sweep.
// Per step: wave 0 computes the rotations while the other waves apply the
// previous step's to V; after a barrier every thread applies the step's to its
// 2 x 2 block of H (pairs bi <= bj; entry (i, j) is kept at row min, column max).
constexpr int kSmallN = 48, kSmallThreads = 1024, kSmallLd = kSmallN + 1;

__device__ __forceinline__ double& upper(double* H, int i, int j) {
  return i < j ? H[i * kSmallLd + j] : H[j * kSmallLd + i];
}

__global__ void __launch_bounds__(kSmallThreads)
symj_small_kernel(int n, const double* __restrict__ G, int64_t ldg, double* __restrict__ V, int64_t ldv,
                  double* __restrict__ evals, int max_sweeps, RotStop stop,
                  int* __restrict__ sweeps) {
  __shared__ double H[kSmallN * kSmallLd], J[kSmallN * kSmallLd];
  __shared__ double rc[2][kSmallN / 2], rs[2][kSmallN / 2];
  __shared__ int pp[2][kSmallN / 2], qq[2][kSmallN / 2];
  __shared__ double red[kSmallThreads / 64];
  __shared__ int sig_s;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int np = n + (n & 1), half = np / 2;
  double ss = 0.0;
  for (int e = tid; e < np * kSmallN; e += kSmallThreads) {
    const int i = e % kSmallN, j = e / kSmallN;
    const double v = (i < n && j < n) ? G[i + j * ldg] : 0.0;
    if (i >= np) continue;
    if (i <= j) H[i * kSmallLd + j] = v;
    J[i * kSmallLd + j] = (i == j) ? 1.0 : 0.0;
    if (i <= j) ss += (i < j ? 2.0 : 1.0) * v * v;
  }
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  double fro2 = 0.0;
  for (int w = 0; w < kSmallThreads / 64; ++w) fro2 += red[w];
  double sc = norm_scale(fro2), fro = sqrt(fro2) * sc;
  if (sc == 0.0) {  // the squares over- or underflowed: scale by the largest entry
    double mx = 0.0;
    for (int e = lane; e < np * np; e += 64) mx = fmax(mx, fabs(upper(H, e % np, e / np)));
    for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
    sc = unit_scale(mx);
    fro = 1.0;
    __syncthreads();  // every wave has read the unscaled entries
  }
  const float flo = (float)(4.0 * 2.220446049250313e-16 * fro);
  for (int e = tid; e < np * kSmallN; e += kSmallThreads) {
    const int i = e % kSmallN, j = e / kSmallN;
    if (i <= j) H[i * kSmallLd + j] *= sc;
  }
  __syncthreads();
  // this thread's block (bi, bj) of the upper triangle of pairs, row by row
  const int nblk = half * (half + 1) / 2;
  int bi = 0, bj = tid;
  if (tid < nblk) {
    while (bj >= half - bi) {
      bj -= half - bi;
      ++bi;
    }
    bj += bi;
  }
  auto rotate_v = [&](int buf, int first, int stride) {
    if (lane >= np) return;
    for (int k = first; k < half; k += stride) {
      const double c = rc[buf][k], s = rs[buf][k];
      const int p = pp[buf][k], q = qq[buf][k];
      const double x = J[lane * kSmallLd + p], y = J[lane * kSmallLd + q];
      J[lane * kSmallLd + p] = c * x - s * y;
      J[lane * kSmallLd + q] = s * x + c * y;
    }
  };
  int buf = 0, sweep = 0;
  bool pending = false;  // the previous step's rotations are not in V yet
  while (sweep < max_sweeps && np > 1) {
    bool sig = false;
    for (int t = 0; t < np - 1; ++t) {
      if (wave == 0) {
        if (lane < half) {
          auto pos = [&](int x) {
            int y = x - 1 + t;
            y = y >= np - 1 ? y - (np - 1) : y;
            return x == 0 ? 0 : 1 + y;
          };
          const int p = pos(lane), q = pos(np - 1 - lane);
          double c, s;
          bool sg;
          rotation(H[p * kSmallLd + p], H[q * kSmallLd + q], upper(H, p, q), flo, stop, &c, &s,
                   &sg);
          rc[buf][lane] = c;
          rs[buf][lane] = s;
          pp[buf][lane] = p;
          qq[buf][lane] = q;
          sig |= sg;
        }
      } else if (V && pending) {
        rotate_v(buf ^ 1, wave - 1, kSmallThreads / 64 - 1);
      }
      __syncthreads();
      if (tid < nblk) {
        const int pi = pp[buf][bi], qi = qq[buf][bi], pj = pp[buf][bj], qj = qq[buf][bj];
        const double ci = rc[buf][bi], si = rs[buf][bi], cj = rc[buf][bj], sj = rs[buf][bj];
        double &e00 = upper(H, pi, pj), &e01 = upper(H, pi, qj), &e10 = upper(H, qi, pj),
               &e11 = upper(H, qi, qj);
        const double h00 = e00, h01 = e01, h10 = e10, h11 = e11;
        const double x00 = cj * h00 - sj * h01, x01 = sj * h00 + cj * h01;
        const double x10 = cj * h10 - sj * h11, x11 = sj * h10 + cj * h11;
        e00 = ci * x00 - si * x10;
        e01 = ci * x01 - si * x11;  // a diagonal block: the same entry as e10
        if (bi != bj) e10 = si * x00 + ci * x10;
        e11 = si * x01 + ci * x11;
      }
      __syncthreads();
      buf ^= 1;
      pending = true;
    }
    if (tid == 0) sig_s = 0;
    __syncthreads();
    if (sig) sig_s = 1;
    __syncthreads();
    ++sweep;
    if (sig_s == 0) break;
    __syncthreads();
  }
  if (V && pending) rotate_v(buf ^ 1, wave, kSmallThreads / 64);
  __syncthreads();
  for (int e = tid; e < n * kSmallN; e += kSmallThreads) {
    const int i = e % kSmallN, j = e / kSmallN;
    if (i >= n) continue;
    if (V) V[i + j * ldv] = J[i * kSmallLd + j];
    if (evals && i == j) evals[i] = H[i * kSmallLd + i] / sc;
  }
  if (tid == 0 && sweeps) *sweeps = sweep;
}

// Eigenvalues only, for n <= kTriN: Householder tridiagonalisation in LDS and
// multisection with Sturm counts, one workgroup.  Where the vectors are not
// wanted this takes 0.145 ms at n = 64 against 0.45 ms for the block Jacobi
// iteration, both to the rounding of ||G||; what bounds it is the chain of
// n - 2 reflections and 24 n Sturm steps.
constexpr int kTriN = 64, kTriLd = kTriN + 1, kTriThreads = 256;

// Sum over the wave, in every lane, by data-parallel moves.
__device__ __forceinline__ double wave_sum(double v) {
  v += row_move<0xb1>(v);   // quad_perm [1, 0, 3, 2]
  v += row_move<0x4e>(v);   // quad_perm [2, 3, 0, 1]
  v += row_move<0x141>(v);  // row_half_mirror: the other quad of eight lanes
  v += row_move<0x140>(v);  // row_mirror: the other half of the row
  v += __shfl_xor(v, 16, 64);
  v += __shfl_xor(v, 32, 64);
  return v;
}

__global__ void __launch_bounds__(kTriThreads)
symtri_values_kernel(int n, const double* __restrict__ G, int64_t ldg, double* __restrict__ evals) {
  constexpr int P = kTriThreads / kTriN;  // threads a row / an eigenvalue
  constexpr int CW = kTriN / P;           // columns of a thread's part of a row
  __shared__ double A[kTriN * kTriLd];
  __shared__ double vs[kTriN], ws[kTriN], part[P][kTriN], dd[kTriN], ee[kTriN],
      e2[kTriN];
  __shared__ int cnt[kTriN * P];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double mx = 0.0;
  for (int e = tid; e < kTriN * kTriN; e += kTriThreads) {
    const int i = e % kTriN, j = e / kTriN;
    const double v = (i < n && j < n) ? (i <= j ? G[i + j * ldg] : G[j + i * ldg]) : 0.0;
    A[i * kTriLd + j] = v;
    mx = (fabs(v) > mx || isnan(v)) ? fabs(v) : mx;
  }
  // scaled by a power of two: the squares below stay in range
  for (int off = 32; off > 0; off >>= 1) {
    const double o = __shfl_xor(mx, off, 64);
    mx = (o > mx || isnan(o)) ? o : mx;
  }
  if (lane == 0) ws[wave] = mx;
  __syncthreads();
  for (int w = 0; w < kTriThreads / 64; ++w) mx = (ws[w] > mx || isnan(ws[w])) ? ws[w] : mx;
  const double sc = unit_scale(mx);
  for (int e = tid; e < kTriN * kTriN; e += kTriThreads)
    A[(e % kTriN) * kTriLd + e / kTriN] *= sc;
  __syncthreads();
  // reflection k maps A(k + 1 .., k) to a multiple of the first unit vector; a
  // wave has nothing to do once its columns are behind k
  const int c0 = wave * CW;
  for (int k = 0; k + 2 < n; ++k) {
    const double x = lane > k ? A[k * kTriLd + lane] : 0.0;
    const double alpha = A[k * kTriLd + k + 1];
    const double tail2 = wave_sum(lane > k + 1 ? x * x : 0.0);
    if (tail2 == 0.0) {  // nothing to annihilate (the same in every thread)
      if (tid == 0) ee[k] = alpha;
      continue;
    }
    const double beta = -copysign(sqrt(alpha * alpha + tail2), alpha);
    const double tau = (beta - alpha) * rcp_nr(beta);
    const double v = lane == k + 1 ? 1.0 : x * rcp_nr(alpha - beta);  // zero up to k
    if (tid == 0) ee[k] = beta;
    if (wave == 0) vs[lane] = v;
    __syncthreads();
    // p = A v, a part of the columns a wave
    double p = 0.0;
    if (c0 + CW > k + 1) {
#pragma unroll
      for (int c = 0; c < CW; ++c) p = fma(A[lane * kTriLd + c0 + c], vs[c0 + c], p);
    }
    part[wave][lane] = p;
    __syncthreads();
    p = 0.0;
    for (int w = 0; w < P; ++w) p += part[w][lane];
    if (lane <= k) p = 0.0;
    const double w = tau * (p - 0.5 * tau * wave_sum(p * v) * v);
    if (wave == 0) ws[lane] = w;
    __syncthreads();
    // A <- A - v w^T - w v^T on the rows and columns past k
    if (c0 + CW > k + 1) {
#pragma unroll
      for (int c = 0; c < CW; ++c) {
        double& a = A[lane * kTriLd + c0 + c];
        a = fma(-w, vs[c0 + c], fma(-v, ws[c0 + c], a));
      }
    }
    __syncthreads();
  }
  if (tid < n) dd[tid] = A[tid * kTriLd + tid];
  if (tid == 0) {
    if (n > 1) ee[n - 2] = A[(n - 2) * kTriLd + n - 1];
    ee[n - 1] = 0.0;
  }
  __syncthreads();
  // Gershgorin bounds, the same in every thread
  double lo = 1e300, hi = -1e300;
  for (int i = 0; i < n; ++i) {
    const double r = fabs(ee[i]) + (i > 0 ? fabs(ee[i - 1]) : 0.0);
    lo = (dd[i] - r < lo || isnan(dd[i] - r)) ? dd[i] - r : lo;
    hi = (dd[i] + r > hi || isnan(dd[i] + r)) ? dd[i] + r : hi;
  }
  const double span = hi - lo, tiny = 1e-290;
  lo -= 1e-15 * span;
  hi += 1e-15 * span;
  if (tid < n) e2[tid] = tid > 0 ? ee[tid - 1] * ee[tid - 1] : 0.0;
  __syncthreads();
  // eigenvalue j (ascending): P interior points of its interval a round; 24
  // rounds divide it by 5^24 = 6e16
  const int j = tid / P, q = tid % P;
  for (int round = 0; round < 24; ++round) {
    const double step = (hi - lo) * (1.0 / (P + 1));
    const double x = lo + step * (q + 1);
    int below = 0;
    double s = 1.0;
#pragma unroll 4
    for (int i = 0; i < n; ++i) {
      // one Newton step: the quotient's error (about 2^-48 of it) shifts the eigenvalues as
      // the same change of e2 would, by 4e-15 of the norm
      double r = __builtin_amdgcn_rcp(s);
      r = fma(r, fma(-s, r, 1.0), r);
      s = fma(-e2[i], r, dd[i] - x);
      s = fabs(s) < tiny ? -tiny : s;
      below += s < 0.0;
    }
    cnt[tid] = below;
    __syncthreads();
    int t = 0;  // points with at most j eigenvalues below
    for (int u = 0; u < P; ++u) t += cnt[j * P + u] <= j;
    __syncthreads();
    hi = t < P ? lo + step * (t + 1) : hi;
    lo = t > 0 ? lo + step * t : lo;
  }
  // descending; NaN input gives NaN
  if (q == 0 && j < n) evals[n - 1 - j] = 0.5 * (lo + hi) / sc;
}

}  // namespace

int symeig_values_f64(Context* c, int64_t n, const double* G, int64_t ldg, double* evals) {
  if (n <= 0) return 0;
  if (n > kTriN) return set_error("symeig_values: n=%lld above %d", (long long)n, kTriN);
  if (ldg < n) return set_error("symeig_values: leading dimension < n");
  KTimer kt(c, "symeig");
  hipLaunchKernelGGL(symtri_values_kernel, dim3(1), dim3(kTriThreads), 0, c->stream, (int)n, G, ldg,
                     evals);
  RSVD_LAUNCH_CHECK();
  return 0;
}

namespace {

template <int B>
int run_sweeps(Context* c, int64_t n, double* G, int64_t ldg, double* V, int64_t ldv,
               double* evals, int max_sweeps, int loose, int* sweep_out) {
  constexpr int S = 2 * B;
  const int nblocks = (int)((n + B - 1) / B);
  const int N = nblocks + (nblocks & 1);
  const int pairs = N / 2;
  const int ntg = pairs * (pairs + 1) / 2;
  const int ntv = V ? pairs * (int)((n + 2 * S - 1) / (2 * S)) : 0;
  const RotStop stop = rot_stop(loose);
  DBuf<double> G2, Jb, Hb, fro2, scal;
  DBuf<unsigned long long> flags;
  const size_t js = (size_t)pairs * S * S;
  RSVD_TRY(G2.alloc((size_t)(ldg * n)));
  RSVD_TRY(Jb.alloc(2 * js));
  RSVD_TRY(Hb.alloc(2 * js));
  RSVD_TRY(fro2.alloc(1));
  RSVD_TRY(scal.alloc(2));
  RSVD_TRY(flags.alloc((size_t)max_sweeps + 2));
  RSVD_TRY(sumsq_f64(c, n, n, G, ldg, fro2.p));
  {
    int blocks = (int)((n * n + 255) / 256);
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL(symj_prep_kernel, dim3(blocks), dim3(256), 0, c->stream, n,
                       (const double*)G, ldg, G2.p, V, ldv, (const double*)fro2.p, scal.p, flags.p,
                       max_sweeps + 2);
    RSVD_LAUNCH_CHECK();
  }
  double* cur = G2.p;
  double* nxt = G;
  int jc = 0;
  int sweep = 0;
  KTimer kt(c, "symeig");
  if (n > 1) {
    // round 0 of sweep 0 from G itself; afterwards every launch applies
    // round r and solves the next round
    hipLaunchKernelGGL(symj_solve_kernel<B>, dim3(pairs), dim3(256), 0, c->stream, n,
                       (const double*)cur, ldg, nblocks, N, 0, (const double*)scal.p, stop, Jb.p,
                       Hb.p, flags.p);
    RSVD_LAUNCH_CHECK();
    // The first launches of sweep s are queued before the host looks at
    // sweep s - 1's flags (copied to pinned memory behind sweep s - 1 and
    // waited for while those launches run); when s - 1 converged they return
    // at once (the device-side stop above), the rest of the sweep is never
    // queued, and the state is the one sweep s started from.
    constexpr int kAhead = 4;  // launches of sweep s queued before the wait
    volatile unsigned long long* slot = static_cast<unsigned long long*>(c->pinned);
    hipEvent_t ev[2] = {nullptr, nullptr};
    RSVD_HIP(hipEventCreateWithFlags(&ev[0], hipEventDisableTiming));
    RSVD_HIP(hipEventCreateWithFlags(&ev[1], hipEventDisableTiming));
    int rc = 0;
    bool done = false;
    for (; sweep < max_sweeps && rc == 0 && !done; ++sweep) {
      double* cur0 = cur;
      const int jc0 = jc;
      const unsigned long long* prev = sweep > 0 ? flags.p + sweep - 1 : nullptr;
      for (int r = 0; r < N - 1; ++r) {
        const bool wrap = r + 1 == N - 1;
        const int r1 = wrap ? 0 : r + 1;
        unsigned long long* fl = flags.p + (wrap ? sweep + 1 : sweep);
        hipLaunchKernelGGL(symj_step_kernel<B>, dim3(pairs + ntg + ntv), dim3(256), 0, c->stream,
                           n, (const double*)cur, nxt, ldg, V, ldv, nblocks, N, r, r1, pairs,
                           (const double*)scal.p, stop, (const double*)(Jb.p + jc * js),
                           (const double*)(Hb.p + jc * js), Jb.p + (1 - jc) * js,
                           Hb.p + (1 - jc) * js, ntg, fl, prev);
        if (hipGetLastError() != hipSuccess) {
          rc = set_error("symeig: step launch failed");
          break;
        }
        double* tmp = cur;
        cur = nxt;
        nxt = tmp;
        jc = 1 - jc;
        // after the first kAhead launches (or the whole sweep, if shorter):
        // sweep - 1's verdict
        if (sweep > 0 && (r + 1 == kAhead || (r + 1 == N - 1 && N - 1 < kAhead))) {
          if (hipEventSynchronize(ev[(sweep - 1) & 1]) != hipSuccess) {
            rc = set_error("symeig: flag wait failed");
            break;
          }
          // no rotation of sweep - 1 counted for the stop: this sweep's
          // launches did nothing
          if (slot[(sweep - 1) & 1] == 0) {
            cur = cur0;
            jc = jc0;
            done = true;
            break;
          }
        }
      }
      if (rc || done) break;
      if (hipMemcpyAsync((void*)(slot + (sweep & 1)), flags.p + sweep, sizeof(unsigned long long),
                         hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
          hipEventRecord(ev[sweep & 1], c->stream) != hipSuccess) {
        rc = set_error("symeig: flag copy failed");
        break;
      }
    }
    (void)hipEventDestroy(ev[0]);
    (void)hipEventDestroy(ev[1]);
    if (rc) return rc;
  }
  if (evals) {
    hipLaunchKernelGGL(symj_diag_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       c->stream, n, (const double*)cur, ldg, (const double*)scal.p, evals);
    RSVD_LAUNCH_CHECK();
  }
  *sweep_out = sweep;
  return 0;
}

}  // namespace

int symeig_jacobi_f64(Context* c, int64_t n, double* G, int64_t ldg, double* V, int64_t ldv,
                      double* evals, int max_sweeps, int* sweeps_out, int loose) {
  if (sweeps_out) *sweeps_out = 0;
  if (n <= 0) return 0;
  if (ldg < n || (V && ldv < n)) return set_error("symeig: leading dimension < n");
  if (n <= kSmallN) {
    DBuf<int> sw;
    if (sweeps_out) RSVD_TRY(sw.alloc(1));
    {
      KTimer kt(c, "symeig");
      hipLaunchKernelGGL(symj_small_kernel, dim3(1), dim3(kSmallThreads), 0, c->stream, (int)n, 
                         (const double*)G, ldg, V, ldv, evals, max_sweeps, rot_stop(loose), sw.p);
      RSVD_LAUNCH_CHECK();
    }
    if (sweeps_out) RSVD_TRY(read_small(c, sweeps_out, sw.p, sizeof(int)));
    return 0;
  }
  int sweep = 0;
  // B = 16: each thread owns one 2x2 block and computes one rotation per
  // step; a larger B trades launches for a slower, LDS-bound inner sweep
  RSVD_TRY(run_sweeps<16>(c, n, G, ldg, V, ldv, evals, max_sweeps, loose, &sweep));
  if (sweeps_out) *sweeps_out = sweep;
  return 0;
}

}  // namespace rsvd
