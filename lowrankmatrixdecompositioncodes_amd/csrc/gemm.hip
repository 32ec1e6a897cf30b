// gemm.hip -- FP64 / FP32 GEMM on CDNA4 matrix cores for the A-streaming passes
// of the rSVD / blocked QB pipeline (Y = A*Omega, Z = A^T*Y, B = Q^T*A, the
// deflation A -= Qp*Bp, U = Q*Uhat, ...), replacing the cblas_dgemm calls of
// MKL/mvf.c:538-561.
//
// A 16x16x4 FP64 MFMA holds its SIMD for 64 cycles and needs 1 KB of operands,
// so no two waves need to share them: every wave runs on its own, without a
// barrier in the k loop, with the next k block's loads in flight behind the
// current block's products.  A k block is one 128-byte line of a k-contiguous
// row (16 FP64 or 32 FP32 elements).  The k index inside a block is permuted so
// that a lane's loads are 16 bytes wide: MFMA step s multiplies the elements
// kmap(g, s) of the lane groups g = lane / 16 (any order of k serves, as long as
// both operands use it).
//  * An operand stored row-contiguous is loaded into registers in MFMA lane
//    order, 16 lanes covering 32 rows of one k; its rows are dealt to the 16-row
//    blocks in pairs (row 2 (lane % 16) + (b & 1) of a 32-row group belongs to
//    block b), the same for both operands and the stores of C.
//  * An operand stored k-contiguous is loaded eight full lines a time and
//    transposed to lane order through a region of LDS of the wave's own
//    (loaded in lane order it would take 16 half lines a load: 50 TF against
//    60 TF for A^T B at 6000 x 288 x 16384).
// Measured (FP64, the kernel's own time; the former kernel staged 128 x 64 tiles
// through one LDS buffer with two barriers a slice): 16384 x 288 x 6000 N N 29 ->
// 60 TF, A^T B as above 40 -> 60 TF, 2000 x 110 x 1000 112 -> 17 us, a 110 x 110
// Gram of 2000 rows 38 -> 8 us.  The large ones are bound by the MFMAs (71 TF at
// the clock a large product reaches) and, where A outgrows the caches, by reading
// it again (gemm_plan); the small ones by latency.  FP32 products that read too
// much this way take a staged kernel (gemm_staged).
// Operand lane layout of the 16x16x4 MFMAs (per 64-lane wave):
//   srcA: lane l holds X[i = l%16][k = l/16]
//   srcB: lane l holds Y[k = l/16][j = l%16]
//   dst : lane l, register r holds D[i][j = l%16] with
//         i = 4*(l/16) + r   for v_mfma_f32_16x16x4f32
//         i = 4*r + l/16     for v_mfma_f64_16x16x4f64
// srcA is fed from op(B) and srcB from op(A), so accumulator lanes run along M
// and the epilogue writes contiguous segments of column-major C.
//
// The same kernel with the FP32 operands rounded (or split) to bf16 in registers
// serves the smaller products of gemm_lp.hip.
#include <algorithm>
#include <climits>
#include <cmath>
#include <type_traits>

#include <rocblas/rocblas.h>

#include "rsvd_internal.h"

namespace rsvd {

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

template <typename T>
struct Mfma;
template <>
struct Mfma<double> {
  typedef d4_t acc_t;
  // two elements, and the k-contiguous elements of one load (16 bytes), at
  // their natural alignment (the hardware's wide global accesses need four
  // bytes)
  typedef double v2_t __attribute__((ext_vector_type(2), aligned(8)));
  typedef v2_t vk_t;
  typedef double vl_t __attribute__((ext_vector_type(2)));  // the same in LDS
  static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // accumulator row held by lane group g (= lane/16), register r
  static __device__ __forceinline__ int row(int g, int r) { return 4 * r + g; }
};
template <>
struct Mfma<float> {
  typedef f4_t acc_t;
  typedef float v2_t __attribute__((ext_vector_type(2), aligned(4)));
  typedef float vk_t __attribute__((ext_vector_type(4), aligned(4)));
  typedef float vl_t __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int g, int r) { return 4 * g + r; }
};

constexpr int kThreads = 256;
// Depth of a k block, MFMA steps of a block, elements of a 16-byte load.
template <typename T>
struct KBlock {
  static constexpr int kDepth = 128 / sizeof(T);
  static constexpr int kSteps = kDepth / 4;
  static constexpr int kVec = 16 / sizeof(T);
  // element of the k block that lane group g multiplies in MFMA step s
  static __device__ __forceinline__ int kmap(int g, int s) {
    return kVec * (g + 4 * (s / kVec)) + s % kVec;
  }
};

// row of a wave's 16-row block b held by index x (0..15)
__device__ __forceinline__ int block_row(int b, int x) { return 32 * (b >> 1) + 2 * x + (b & 1); }

// One operand of a wave: TT 16-row blocks of op(X) from row r0, `lim` rows in
// all (rows past the end read the last row; their products are not stored).
// KC: element (row, k) at X[k + row ld] (k-contiguous), else X[row + k ld].
// A block is loaded into raw registers (load) and read from them in lane order
// (frags).
template <typename T, bool KC, int TT>
struct Operand;

template <typename T, int TT>
struct Operand<T, false, TT> {
  typedef typename Mfma<T>::v2_t v2_t;
  static constexpr int SS = KBlock<T>::kSteps;
  static constexpr int kLds = 0;
  struct Raw {
    T f[TT][SS];
  };
  const T* X;
  int64_t ld, r0, last;
  bool full;  // every row of the wave's blocks is valid
  __device__ __forceinline__ Operand(const T* X_, int64_t ld_, int64_t r, int64_t lim, char*)
      : X(X_), ld(ld_), r0(r), last(lim - 1), full(r + 16 * TT <= lim) {}
  // FULL: every row valid; TAIL: zero where k >= kend
  template <bool FULL, bool TAIL>
  __device__ __forceinline__ void load(int64_t k0, int64_t kend, Raw& w) const {
    const int li = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int s = 0; s < SS; ++s) {
      const int64_t k = k0 + KBlock<T>::kmap(lk, s);
      const bool ok = !TAIL || k < kend;
      const T* p = X + (ok ? k : kend - 1) * ld;
#pragma unroll
      for (int b = 0; b < TT; b += 2) {
        const int64_t r = r0 + block_row(b, li);
        if constexpr (FULL) {
          const v2_t v = *reinterpret_cast<const v2_t*>(p + r);
          w.f[b][s] = ok ? v[0] : T(0);
          w.f[b + 1][s] = ok ? v[1] : T(0);
        } else {
          const T v0 = p[r < last ? r : last], v1 = p[r + 1 < last ? r + 1 : last];
          w.f[b][s] = ok ? v0 : T(0);
          w.f[b + 1][s] = ok ? v1 : T(0);
        }
      }
    }
  }
  __device__ __forceinline__ void frags(const Raw& w, T (&f)[TT][SS]) const {
#pragma unroll
    for (int b = 0; b < TT; ++b)
#pragma unroll
      for (int s = 0; s < SS; ++s) f[b][s] = w.f[b][s];
  }
};

// Load j takes rows 8 j + lane / 8, 16-byte chunk lane % 8 of each row's line.
// In LDS row r keeps its chunk c at position c ^ ((r / 2) % 8): the sixteen
// rows 2 x (or 2 x + 1) that a frag read takes at equal c spread over the banks.
template <typename T, int TT>
struct Operand<T, true, TT> {
  static constexpr int SS = KBlock<T>::kSteps, VK = KBlock<T>::kVec;
  static constexpr int kLds = TT * 16 * 128;  // bytes of the wave's region
  typedef typename Mfma<T>::vk_t vk_t;
  struct Raw {
    vk_t v[2 * TT];
  };
  const T* X;
  int64_t ld, r0, last;
  bool full;
  char* lds;
  __device__ __forceinline__ Operand(const T* X_, int64_t ld_, int64_t r, int64_t lim, char* lds_)
      : X(X_), ld(ld_), r0(r), last(lim - 1), full(r + 16 * TT <= lim), lds(lds_) {}
  template <bool FULL, bool TAIL>
  __device__ __forceinline__ void load(int64_t k0, int64_t kend, Raw& w) const {
    const int lane = threadIdx.x & 63;
    const int64_t k = k0 + VK * (lane & 7);
#pragma unroll
    for (int j = 0; j < 2 * TT; ++j) {
      const int64_t r = r0 + 8 * j + (lane >> 3);
      const T* p = X + (FULL || r < last ? r : last) * ld + k;
      if constexpr (!TAIL) {
        w.v[j] = *reinterpret_cast<const vk_t*>(p);
      } else {
#pragma unroll
        for (int e = 0; e < VK; ++e) w.v[j][e] = (k + e < kend) ? p[e] : T(0);
      }
    }
  }
  __device__ __forceinline__ void frags(const Raw& w, T (&f)[TT][SS]) const {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    // one wave's LDS operations complete in order; the fences keep the
    // compiler from moving the reads over the writes or the next block's
    // writes over these reads
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int j = 0; j < 2 * TT; ++j) {
      const int r = 8 * j + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
      *reinterpret_cast<typename Mfma<T>::vl_t*>(lds + r * 128 + 16 * c) = w.v[j];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int b = 0; b < TT; ++b) {
      const int r = block_row(b, li);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int c = (lk + 4 * q) ^ ((r >> 1) & 7);
        const auto v = *reinterpret_cast<const typename Mfma<T>::vl_t*>(lds + r * 128 + 16 * c);
#pragma unroll
        for (int e = 0; e < VK; ++e) f[b][VK * q + e] = v[e];
      }
    }
  }
};

// Arguments of a launch: C = alpha op(A) op(B) + beta C, M x N, inner K in
// slices of kchunk (a multiple of the k block), slice z into C + z zstride.
template <typename T>
struct GemmArgs {
  int64_t M, N, K, kchunk;
  T alpha;
  const T* A;
  int64_t lda;
  const T* B;
  int64_t ldb;
  T beta;
  T* C;
  int64_t ldc, zstride;
  double* sumsq;  // optional: per-workgroup sums of squares of the stored C
  int sym;        // Gram: form the entries on and above the diagonal only
  int mirror;     // sym: store each also below the diagonal
  int gx, gy;     // tiles
};

// Row tiles of column tile tn with an entry on or above the diagonal.
__host__ __device__ __forceinline__ int64_t sym_tiles(int64_t tn, int64_t gx, int64_t bm,
                                                      int64_t bn) {
  const int64_t up = ((tn + 1) * bn + bm - 1) / bm;
  return up < gx ? up : gx;
}

// A workgroup (four waves) owns a (16 TM WM) x (16 TN WN) tile of C; KS = 4 /
// (WM WN) waves share a wave tile and deal its k blocks among them, their
// partial tiles added in wave order through LDS at the end.
// SPLIT (FP32 operands): 0 multiplies on the FP32 matrix cores; 1 rounds the
// operands to bf16, 3 splits them into bf16 hi + lo and takes hi hi + hi lo + lo
// hi (gemm_lp.hip), both in registers on the way to v_mfma_f32_16x16x32_bf16 --
// one MFMA (three) for the 32-deep block, the same accumulator layout.
template <typename T, bool TA, bool TB, int TM, int TN, int WM, int WN, int SPLIT = 0>
__global__ void __launch_bounds__(kThreads, 2)
gemm_kernel(const GemmArgs<T> g) {
  constexpr int KS = 4 / (WM * WN);
  constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
  typedef typename Mfma<T>::acc_t acc_t;
  typedef typename Mfma<T>::v2_t v2_t;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int ks = wave / (WM * WN), wt = wave % (WM * WN);
  // Tile order.  Workgroups are handed to the 8 XCDs round-robin by
  // dispatch order (b % 8), each XCD with its own L2: XCD x takes a
  // contiguous run of tiles, walked with the dimension that has fewer tiles
  // fastest, so the workgroups that run together on one XCD share the large
  // operand's panel (the n / l column tiles of one row block of A run side by
  // side and A leaves HBM once instead of once per column tile).
  int64_t tm, tn;
  {
    const int64_t gx = g.gx, gy = g.gy, nt = gridDim.x;
    const int64_t b = blockIdx.x;
    const int64_t xcd = b & 7, j = b >> 3, q = nt >> 3, r = nt & 7;
    const int64_t t = xcd * q + (xcd < r ? xcd : r) + j;
    if (g.sym) {
      // a Gram: the tiles of column tn that reach the diagonal, column by column
      tm = t;
      for (tn = 0; tm >= sym_tiles(tn, gx, BM, BN); ++tn) tm -= sym_tiles(tn, gx, BM, BN);
    } else if (gy <= gx) {
      tn = t % gy;
      tm = t / gy;
    } else {
      tm = t % gx;
      tn = t / gx;
    }
  }
  const int64_t m0 = tm * BM + (wt % WM) * 16 * TM;
  const int64_t n0 = tn * BN + (wt / WM) * 16 * TN;
  const int64_t kbeg = (int64_t)blockIdx.y * g.kchunk;
  const int64_t kend = (kbeg + g.kchunk < g.K) ? kbeg + g.kchunk : g.K;
  T* __restrict__ C = g.C + (int64_t)blockIdx.y * g.zstride;

  acc_t acc[TN][TM];
#pragma unroll
  for (int a = 0; a < TN; ++a)
#pragma unroll
    for (int b = 0; b < TM; ++b) acc[a][b] = acc_t{0, 0, 0, 0};

  // the waves' transposition regions, then their partial tiles
  typedef Operand<T, TA, TM> OpA;
  typedef Operand<T, !TB, TN> OpB;
  constexpr int kStage = 4 * (OpA::kLds + OpB::kLds);
  constexpr int kPart = KS > 1 ? KS * TN * TM * 4 * 64 * (int)sizeof(T) : 0;
  constexpr int kSm = kStage > kPart ? kStage : kPart;
  __shared__ __align__(16) char sm[kSm > 0 ? kSm : 16];

  const bool live = m0 < g.M && n0 < g.N;
  if (live) {
    constexpr int KD = KBlock<T>::kDepth, SS = KBlock<T>::kSteps;
    char* ws = sm + wave * (OpA::kLds + OpB::kLds);
    const OpA oa(g.A, g.lda, m0, g.M, ws);
    const OpB ob(g.B, g.ldb, n0, g.N, ws + OpA::kLds);
    typename OpA::Raw a0, a1;
    typename OpB::Raw b0, b1;
    T fa[TM][SS], fb[TN][SS];
    auto mma = [&]() {
      if constexpr (SPLIT != 0) {
        bf16x8_t ah[TM], al[TM], bh[TN], bl[TN];
        auto cut = [](const T(&x)[KBlock<T>::kSteps], bf16x8_t& h, bf16x8_t& l) {
#pragma unroll
          for (int s = 0; s < KBlock<T>::kSteps; ++s) {
            const __bf16 v = (__bf16)x[s];
            h[s] = v;
            if (SPLIT == 3) l[s] = (__bf16)(x[s] - (float)v);
          }
        };
#pragma unroll
        for (int a = 0; a < TN; ++a) cut(fb[a], bh[a], bl[a]);
#pragma unroll
        for (int b = 0; b < TM; ++b) cut(fa[b], ah[b], al[b]);
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
          for (int b = 0; b < TM; ++b) {
            f4_t d = acc[a][b];
            if (SPLIT == 3) {
              d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[a], al[b], d, 0, 0, 0);
              d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bl[a], ah[b], d, 0, 0, 0);
            }
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[a], ah[b], d, 0, 0, 0);
          }
        return;
      }
#pragma unroll
      for (int s = 0; s < SS; ++s)
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
          for (int b = 0; b < TM; ++b) acc[a][b] = Mfma<T>::mma(fb[a][s], fa[b][s], acc[a][b]);
    };
    const int64_t full = (kend - kbeg) / KD;
    // two register buffers, unrolled by two so that they swap by name
    auto loop = [&](auto ft) {
      constexpr bool F = decltype(ft)::value;
      auto load = [&](int64_t kb, typename OpA::Raw& ra, typename OpB::Raw& rb) {
        oa.template load<F, false>(kbeg + kb * KD, kend, ra);
        ob.template load<F, false>(kbeg + kb * KD, kend, rb);
      };
      int64_t kb = ks;
      if (kb < full) load(kb, a0, b0);
      for (; kb + KS < full; kb += 2 * KS) {
        oa.frags(a0, fa);
        ob.frags(b0, fb);
        load(kb + KS, a1, b1);
        mma();
        oa.frags(a1, fa);
        ob.frags(b1, fb);
        if (kb + 2 * KS < full) load(kb + 2 * KS, a0, b0);
        mma();
      }
      if (kb < full) {
        oa.frags(a0, fa);
        ob.frags(b0, fb);
        mma();
      }
    };
    if (oa.full && ob.full) loop(std::true_type{});
    else loop(std::false_type{});
    if (kbeg + full * KD < kend && full % KS == ks) {
      oa.template load<false, true>(kbeg + full * KD, kend, a0);
      ob.template load<false, true>(kbeg + full * KD, kend, b0);
      oa.frags(a0, fa);
      ob.frags(b0, fb);
      mma();
    }
  }

  double ss = 0.0;
  // rows 2 li and 2 li + 1 of block pair bp, the four columns of block a
  auto store = [&](int a, int bp, const acc_t& x0, const acc_t& x1) {
    const int64_t gm = m0 + 32 * bp + 2 * li;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t gn = n0 + block_row(a, Mfma<T>::row(lk, r));
      if (gm >= g.M || gn >= g.N) continue;
      if (g.sym) {  // beta = 0
        const T v[2] = {g.alpha * x0[r], g.alpha * x1[r]};
#pragma unroll
        for (int e = 0; e < 2; ++e)
          if (gm + e <= gn) {
            C[gm + e + gn * g.ldc] = v[e];
            if (g.mirror) C[gn + (gm + e) * g.ldc] = v[e];
          }
        continue;
      }
      T* cp = C + gm + gn * g.ldc;
      if (gm + 1 < g.M) {
        v2_t v = {g.alpha * x0[r], g.alpha * x1[r]};
        if (g.beta != T(0)) {
          const v2_t c = *reinterpret_cast<const v2_t*>(cp);
          v[0] += g.beta * c[0];
          v[1] += g.beta * c[1];
        }
        *reinterpret_cast<v2_t*>(cp) = v;
        ss += (double)v[0] * (double)v[0] + (double)v[1] * (double)v[1];
      } else {
        T v = g.alpha * x0[r];
        if (g.beta != T(0)) v += g.beta * (*cp);
        *cp = v;
        ss += (double)v * (double)v;
      }
    }
  };
  if constexpr (KS == 1) {
    if (live) {
#pragma unroll
      for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int bp = 0; bp < TM / 2; ++bp) store(a, bp, acc[a][2 * bp], acc[a][2 * bp + 1]);
    }
  } else {
    static_assert(WM * WN == 1 && KS == 4, "the four waves share one tile");
    T(*part)[TN * TM * 4][64] = reinterpret_cast<T(*)[TN * TM * 4][64]>(sm);
    __syncthreads();
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
      for (int b = 0; b < TM; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[wave][(a * TM + b) * 4 + r][lane] = acc[a][b][r];
    __syncthreads();
    // block pairs dealt to the waves, partial tiles added in wave order
    for (int t = wave; t < TN * TM / 2; t += 4) {
      const int a = t / (TM / 2), bp = t % (TM / 2);
      acc_t x[2];
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = (a * TM + 2 * bp + e) * 4 + r;
          x[e][r] = ((part[0][i][lane] + part[1][i][lane]) + part[2][i][lane]) + part[3][i][lane];
        }
      store(a, bp, x[0], x[1]);
    }
  }
  if (g.sumsq) {
    __shared__ double red[kThreads / 64];
    for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    if (tid == 0) {
      double t = 0;
      for (int w = 0; w < kThreads / 64; ++w) t += red[w];
      g.sumsq[tm + (int64_t)g.gx * tn] = t;
    }
  }
}

// FP32 with the operands staged: 128 x BN tiles of C, 16 elements of k at a time in LDS,
// for the products that gemm_staged chooses.  An FP32 MFMA takes half the cycles of an
// FP64 one for the same element count, and a wave of gemm_kernel that reads two
// row-contiguous operands off the cache lines' boundaries fetches five lines where three
// hold its data; here a workgroup fetches each once.
template <bool TA, bool TB, int BN>
__global__ void __launch_bounds__(kThreads, 2)
gemm_staged_kernel(const GemmArgs<float> g) {
  constexpr int BM = 128, BK = 16, PAD = 4;
  constexpr int TM = 4, TN = BN / 32;  // 16 x 16 blocks of a wave (two waves along each side)
  constexpr int EA = BM * BK / kThreads, EB = BN * BK / kThreads;
  __shared__ float As[BK][BM + PAD], Bs[BK][BN + PAD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  // the tile order of gemm_kernel
  const int64_t gx = g.gx, gy = g.gy, nt = gridDim.x;
  const int64_t xcd = blockIdx.x & 7, q = nt >> 3, r = nt & 7;
  const int64_t t = xcd * q + (xcd < r ? xcd : r) + (blockIdx.x >> 3);
  const int64_t m0 = (gy <= gx ? t / gy : t % gx) * BM, n0 = (gy <= gx ? t % gy : t / gx) * BN;
  const int64_t kbeg = (int64_t)blockIdx.y * g.kchunk;
  const int64_t kend = (kbeg + g.kchunk < g.K) ? kbeg + g.kchunk : g.K;
  float* C = g.C + (int64_t)blockIdx.y * g.zstride;
  // this thread's elements of a stage: row ma and k ka of A (and of B), the e-th one
  // sa elements further along the other dimension
  const int ma = TA ? tid / BK : tid % BM, ka = TA ? tid % BK : tid / BM;
  const int nb = TB ? tid % BN : tid / BK, kb = TB ? tid / BN : tid % BK;
  constexpr int RA = TA ? kThreads / BK : 0, KA = TA ? 0 : kThreads / BM;
  constexpr int RB = TB ? 0 : kThreads / BK, KB = TB ? kThreads / BN : 0;
  const float* pa = g.A + (TA ? kbeg + ka + (m0 + ma) * g.lda : m0 + ma + (kbeg + ka) * g.lda);
  const float* pb = g.B + (TB ? n0 + nb + (kbeg + kb) * g.ldb : kbeg + kb + (n0 + nb) * g.ldb);
  const int64_t sa = (TA ? RA : KA) * g.lda, sb = (TB ? KB : RB) * g.ldb;
  const int64_t na = TA ? BK : BK * g.lda, nbs = TB ? BK * g.ldb : BK;  // to the next stage
  const int mleft = (int)(g.M - m0 < BM ? g.M - m0 : BM);
  const int nleft = (int)(g.N - n0 < BN ? g.N - n0 : BN);
  float ra[EA], rb[EB];
  auto load = [&](int64_t k0) {
    const int kleft = (int)(kend - k0 < BK ? kend - k0 : BK);
#pragma unroll
    for (int e = 0; e < EA; ++e)
      ra[e] = (ma + RA * e < mleft && ka + KA * e < kleft) ? pa[e * sa] : 0.0f;
#pragma unroll
    for (int e = 0; e < EB; ++e)
      rb[e] = (nb + RB * e < nleft && kb + KB * e < kleft) ? pb[e * sb] : 0.0f;
    pa += na;
    pb += nbs;
  };
  f4_t acc[TN][TM];
#pragma unroll
  for (int a = 0; a < TN; ++a)
#pragma unroll
    for (int b = 0; b < TM; ++b) acc[a][b] = f4_t{0, 0, 0, 0};
  const int wm0 = (wave & 1) * 64, wn0 = (wave >> 1) * (BN / 2);
  load(kbeg);
  for (int64_t k0 = kbeg; k0 < kend; k0 += BK) {
    __syncthreads();
#pragma unroll
    for (int e = 0; e < EA; ++e) As[ka + KA * e][ma + RA * e] = ra[e];
#pragma unroll
    for (int e = 0; e < EB; ++e) Bs[kb + KB * e][nb + RB * e] = rb[e];
    __syncthreads();
    if (k0 + BK < kend) load(k0 + BK);
#pragma unroll
    for (int s = 0; s < BK / 4; ++s) {
      float av[TM], bv[TN];
#pragma unroll
      for (int a = 0; a < TN; ++a) bv[a] = Bs[4 * s + lk][wn0 + 16 * a + li];
#pragma unroll
      for (int b = 0; b < TM; ++b) av[b] = As[4 * s + lk][wm0 + 16 * b + li];
#pragma unroll
      for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[a][b] = Mfma<float>::mma(bv[a], av[b], acc[a][b]);
    }
  }
#pragma unroll
  for (int a = 0; a < TN; ++a)
#pragma unroll
    for (int b = 0; b < TM; ++b) {
      const int64_t gm = m0 + wm0 + 16 * b + li;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t gn = n0 + wn0 + 16 * a + Mfma<float>::row(lk, e);
        if (gm >= g.M || gn >= g.N) continue;
        float* cp = C + gm + gn * g.ldc;
        const float v = g.alpha * acc[a][b][e];
        *cp = g.beta != 0.0f ? v + g.beta * *cp : v;
      }
    }
}

// C = sum_z W[z] (+ beta*C), W[z] is M x N with leading dimension M, added in
// double.  sym: the
// entries on and above the diagonal, each stored on both sides of it.
template <typename T>
__global__ void splitk_reduce_kernel(int64_t M, int64_t N, int splits, const T* __restrict__ W,
                                     T beta, T* __restrict__ C, int64_t ldc, int sym) {
  int64_t total = M * N;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    int64_t i = idx % M, j = idx / M;
    if (sym && i > j) continue;
    double s = 0.0;
    // loads issued ahead of the (in-order) adds
#pragma unroll 8
    for (int z = 0; z < splits; ++z) s += (double)W[(int64_t)z * total + idx];
    T* cp = C + i + j * ldc;
    T v = (T)s;
    if (beta != T(0)) v += beta * (*cp);
    *cp = v;
    if (sym) C[j + i * ldc] = v;
  }
}

// Fixed-order sum of n doubles into *out (single workgroup).
__global__ void sum_partials_kernel(int64_t n, const double* __restrict__ part,
                                    double* __restrict__ out) {
  __shared__ double red[256];
  double s = 0;
  for (int64_t i = threadIdx.x; i < n; i += 256) s += part[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
}

// How a product is cut: the workgroup tile and the number of k slices.
enum GemmTile { kTile128x64 = 0, kTile64x32 = 1, kTile32x32 = 2 };
struct GemmPlan {
  int tile;
  int splits;
  int64_t gx, gy, tiles, kchunk;
};

// The model's constants of a precision, in microseconds: a k block of a 16 x 16 block
// of C on one wave; the time of each tile over that, with op(A) row-contiguous and
// k-contiguous; the workgroups a CU that a lone one takes the time of (its waves wait
// for their operands with nothing else to run); a workgroup's start and end; what
// slices add, once and an element; what a long k loop adds.
struct CutCost {
  double block, slow[2][3], alone[3], group[3], launch, elem, drift;
};

// The cheapest cut by a model of the kernel's time: rounds of one workgroup a CU (one
// wave on every SIMD), each as long as a wave's k blocks -- its MFMAs, 64 cycles each
// in FP64 and 32 in FP32; the split modes (16 each) wait for their operands far
// longer.  In FP64 workgroups that share operands drift apart in a long k loop and
// fetch them again: past 96 blocks a wave the time grows, by `drift` at 192.
// Fitted to a grid of cuts of 1750 FP64 and 870 FP32 and split products and Grams (16
// to 90000 rows, even and odd sizes, every transposition): its choice is 2.2% (FP64)
// and 2.5% (FP32) slower than the fastest of them in the geometric mean.  With rounds
// and MFMAs alone it chose one workgroup a CU with a long loop too often, above all
// for odd sizes, whose rows straddle cache lines: A^T B at 4013 x 50 x 18712 373 us,
// now 235, at 2271 x 110 x 14730 279 and 205 us, at 100 x 4073 x 43721 1478 and 998 us.
// Slices cost their second launch: 4 us in a chain of small FP64 products (three slices
// for 26 x 26 x 400 and 200 x 26 x 400 saved 2 us of their kernels' 7).
// The slices hold at most kMaxSliceElems elements: what they save on a larger output,
// part of a last round of workgroups, is not worth the memory.  In an allocation-free
// call they are also no more than the largest free range of the scratch array holds: a
// call never needs more than its panels for the sake of a slice.
constexpr int64_t kMaxSliceElems = int64_t(1) << 28;
template <typename T>
static GemmPlan gemm_plan(Context* c, bool ka, int64_t M, int64_t N, int64_t K, bool sym,
                          bool one_slice, int split = 0) {
  static const struct {
    int bm, bn, ks, blocks;  // blocks of C a wave owns
  } kTiles[3] = {{128, 64, 1, 8}, {64, 32, 4, 8}, {32, 32, 4, 4}};
  static const CutCost
      kF64 = {256.0 / 2400, {{1.1, 1.1, 1.13}, {1.26, 1.26, 1.1}}, {1.3, 2.0, 1.1},
              {0.5, 0.8, 0.8}, 4.0, 1.5e-6, 0.4},
      kF32 = {256.0 / 2400, {{1.1, 1.1, 1.0}, {1.1, 1.1, 1.0}}, {1.6, 1.4, 1.0},
              {0.3, 0.3, 0.3}, 2.0, 5e-7, 0.0},
      kSplit = {0.1, {{1.2, 1.05, 1.0}, {0.88, 0.9, 1.0}}, {1.4, 1.3, 1.2},
                {0.1, 0.1, 0.1}, 2.0, 1e-6, 0.0};
  const CutCost& m = sizeof(T) == 8 ? kF64 : (split == 0 ? kF32 : kSplit);
  constexpr int64_t depth = KBlock<T>::kDepth;
  // Large A^T B: 32 x 32 tiles fetch half as much again as 64 x 32 ones, and their reads
  // reach what the memory gives (16384 x 544 x 65536 in FP64: 7.5 TB/s).  With constants
  // of their own, FP64 from 40 GFLOP on: 36 products take 0.89 of the time in the geometric
  // mean (0.68 to 1.2; 16384 x 544 x 65536 22.1 ms, now 19.4, 4987 x 576 x 18539 2.64 and
  // 1.80).  Not with one narrow ragged column of tiles (12001 x 101 x 40003 2.48 and 2.88 ms)
  // nor fewer rows than columns.  FP32 from 20 GFLOP on: 40 products 0.5 to 1.02 of the time
  // (256 x 10180 x 85045 8.96 and 4.92 ms, 65867 x 760 x 10522 15.8 and 10.9).
  static const double kLargeSlow[3] = {1.0, 1.04, 1.08};
  const double flops = 2.0 * (double)M * (double)N * (double)K;
  const bool large = ka && !sym && split == 0 &&
                    (sizeof(T) == 8 ? flops > 4e10 && M >= N && (N % 32 == 0 || N >= 288)
                                    : flops > 2e10);
  const double* slow = large ? kLargeSlow : m.slow[ka];
  const int64_t cus = c->num_cus > 0 ? c->num_cus : 256;
  const int64_t kblocks = (K + depth - 1) / depth;
  int64_t room = kMaxSliceElems / (M * N);
  if (c->scratch_mode) room = std::min(room, (int64_t)(scratch_room(c) / sizeof(T)) / (M * N));
  // FP32: a wave's running sum takes at most `longest` products as far as 64 slices
  // allow (its rounding grows with the length).  512 where the output is small: at
  // 65536 rows the Gram behind the last CholeskyQR step needs it.  For larger ones what
  // 128 x 64 tiles sliced for two workgroups a CU take, 256 products a slice or more;
  // of two such tiles a CU or more the sums are not cut.
  int64_t longest = 0;
  if (sizeof(T) == 4 && !one_slice) {
    longest = 512;
    if (M * N > (int64_t(1) << 20)) {
      const int64_t gx = (M + 127) / 128, gy = (N + 63) / 64;
      int64_t tiles = gx * gy;
      if (sym) {
        tiles = 0;
        for (int64_t y = 0; y < gy; ++y) tiles += sym_tiles(y, gx, 128, 64);
      }
      const int64_t most = tiles < 2 * cus ? std::min<int64_t>(64, K / 256) : 1;
      const int64_t slices = most > 1 ? pick_k_slices(tiles, 2 * cus, most) : 1;
      longest = std::max<int64_t>(longest, (K + slices - 1) / slices);
    }
  }
  GemmPlan best{};
  double best_cost = 1e300;
  for (int t = 0; t < 3; ++t) {
    const auto& d = kTiles[t];
    const int64_t gx = (M + d.bm - 1) / d.bm, gy = (N + d.bn - 1) / d.bn;
    int64_t tiles = gx * gy;
    if (sym) {
      tiles = 0;
      for (int64_t y = 0; y < gy; ++y) tiles += sym_tiles(y, gx, d.bm, d.bn);
    }
    int64_t smax = one_slice ? 1 : kblocks / (2 * d.ks);
    smax = smax > room ? room : smax;
    smax = smax < 1 ? 1 : (smax > 64 ? 64 : smax);
    int64_t smin = 1;
    if (longest > 0) {
      smin = (K + longest * d.ks - 1) / (longest * d.ks);
      smin = smin < smax ? smin : smax;
    }
    for (int64_t s = smin; s <= smax; ++s) {
      const int64_t kb = (kblocks + s - 1) / s;
      if ((kblocks + kb - 1) / kb != s && s > smin) continue;  // as with a smaller s
      const double rounds = (double)((tiles * s + cus - 1) / cus);
      const double blocks = (double)((kb + d.ks - 1) / d.ks);
      double wave = blocks * d.blocks * m.block * slow[t];
      if (blocks > 96) wave *= 1.0 + m.drift * std::min(1.0, std::log2(blocks / 96.0));
      double cost = std::max(rounds, m.alone[t]) * wave + rounds * m.group[t];
      if (s > 1) cost += m.launch + m.elem * (double)s * (double)M * (double)N;
      if (cost < best_cost) {
        best_cost = cost;
        best = GemmPlan{t, (int)((kblocks + kb - 1) / kb), gx, gy, tiles, kb * depth};
      }
    }
  }
  return best;
}

template <typename T, bool TA, bool TB, int SPLIT>
static void gemm_launch_tile(Context* c, int tile, dim3 grid, const GemmArgs<T>& g) {
  if (tile == kTile128x64)
    hipLaunchKernelGGL((gemm_kernel<T, TA, TB, 4, 2, 2, 2, SPLIT>), grid, dim3(kThreads), 0,
                       c->stream, g);
  else if (tile == kTile64x32)
    hipLaunchKernelGGL((gemm_kernel<T, TA, TB, 4, 2, 1, 1, SPLIT>), grid, dim3(kThreads), 0,
                       c->stream, g);
  else
    hipLaunchKernelGGL((gemm_kernel<T, TA, TB, 2, 2, 1, 1, SPLIT>), grid, dim3(kThreads), 0,
                       c->stream, g);
}

template <typename T>
static int launch_splitk_reduce(Context* c, int64_t M, int64_t N, int splits, const T* work, T beta,
                                T* C, int64_t ldc, bool sym) {
  const int64_t blocks = std::min<int64_t>((M * N + 255) / 256, 4096);
  hipLaunchKernelGGL(splitk_reduce_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, c->stream, M, N,
                     splits, work, beta, C, ldc, sym ? 1 : 0);
  RSVD_LAUNCH_CHECK();
  return 0;
}

template <typename T, int SPLIT = 0>
static int launch_gemm(Context* c, const GemmPlan& pl, char ta, char tb, int64_t M, int64_t N,
                       int64_t K, T alpha, const T* A, int64_t lda, const T* B, int64_t ldb, T beta,
                       T* C, int64_t ldc, double* sumsq_partials, bool sym, const char* tag) {
  DBuf<T> work;
  GemmArgs<T> g{M, N, K, pl.kchunk, alpha, A, lda, B, ldb, beta, C, ldc, 0, sumsq_partials,
                sym ? 1 : 0, sym ? 1 : 0, (int)pl.gx, (int)pl.gy};
  if (pl.splits > 1) {
    RSVD_TRY(work.alloc((size_t)(M * N * pl.splits)));
    g.C = work.p;
    g.ldc = M;
    g.zstride = M * N;
    g.beta = T(0);
    g.mirror = 0;
  }
  {
    KTimer kt(c, tag);
    const dim3 grid((unsigned)pl.tiles, (unsigned)pl.splits);
    const bool tA = (ta == 'T' || ta == 't'), tB = (tb == 'T' || tb == 't');
    if (!tA && !tB) gemm_launch_tile<T, false, false, SPLIT>(c, pl.tile, grid, g);
    else if (tA && !tB) gemm_launch_tile<T, true, false, SPLIT>(c, pl.tile, grid, g);
    else if (!tA && tB) gemm_launch_tile<T, false, true, SPLIT>(c, pl.tile, grid, g);
    else gemm_launch_tile<T, true, true, SPLIT>(c, pl.tile, grid, g);
    RSVD_LAUNCH_CHECK();
  }
  return pl.splits > 1 ? launch_splitk_reduce<T>(c, M, N, pl.splits, work.p, beta, C, ldc, sym) : 0;
}

// The FP32 products of gemm_staged_kernel.  Over 500 products of 0.1 to 200 GFLOP
// gemm_kernel takes 0.65 to 0.9 of its time below 1 GFLOP and for outputs of few rows, and
// 0.8 to 0.95 above, but 1.1 to 1.5 times as long where both operands are row-contiguous
// off the 128-byte lines (N T, odd sizes), or one is in a long k loop, or k is so short
// that the tail of its 32-deep blocks weighs (46256 x 1611 x 89 290 us, here 230).
static bool gemm_staged(bool tA, bool tB, int64_t M, int64_t N, int64_t K, int64_t lda,
                        int64_t ldb) {
  const int off = (!tA && lda % 32 != 0) + (tB && ldb % 32 != 0);
  const double flops = 2.0 * (double)M * (double)N * (double)K;
  if (M < (off == 2 ? 96 : 192) || flops < (K < 100 ? 5e8 : 1e9)) return false;
  return off == 2 || (off == 1 && K > 10000) || K < 300;
}

static int launch_gemm_staged(Context* c, const char* tag, bool tA, bool tB, int64_t M, int64_t N,
                              int64_t K, float alpha, const float* A, int64_t lda, const float* B,
                              int64_t ldb, float beta, float* C, int64_t ldc) {
  const int bn = N <= 32 ? 32 : 64;
  const int64_t gx = (M + 127) / 128, gy = (N + bn - 1) / bn, tiles = gx * gy;
  // slices for two workgroups a CU, 256 products or more each
  const int64_t target = 2LL * (c->num_cus > 0 ? c->num_cus : 256);
  int64_t splits = 1;
  if (tiles < target && K >= 4 * 256)
    splits = pick_k_slices(tiles, target, std::min<int64_t>(K / 256, bn == 32 ? 128 : 64));
  const int64_t kchunk = ((K + splits - 1) / splits + 15) / 16 * 16;
  splits = (K + kchunk - 1) / kchunk;
  DBuf<float> work;
  GemmArgs<float> g{M, N, K, kchunk, alpha, A, lda, B, ldb, beta, C, ldc, 0, nullptr, 0, 0,
                    (int)gx, (int)gy};
  if (splits > 1) {
    RSVD_TRY(work.alloc((size_t)(M * N * splits)));
    g.C = work.p;
    g.ldc = M;
    g.zstride = M * N;
    g.beta = 0.0f;
  }
  {
    KTimer kt(c, tag);
    const dim3 grid((unsigned)tiles, (unsigned)splits);
#define RSVD_STAGED(TA_, TB_)                                                                   \
  do {                                                                                          \
    if (bn == 32)                                                                               \
      hipLaunchKernelGGL((gemm_staged_kernel<TA_, TB_, 32>), grid, dim3(kThreads), 0, c->stream, \
                         g);                                                                    \
    else                                                                                        \
      hipLaunchKernelGGL((gemm_staged_kernel<TA_, TB_, 64>), grid, dim3(kThreads), 0, c->stream, \
                         g);                                                                    \
  } while (0)
    if (!tA && !tB) RSVD_STAGED(false, false);
    else if (tA && !tB) RSVD_STAGED(true, false);
    else if (!tA && tB) RSVD_STAGED(false, true);
    else RSVD_STAGED(true, true);
#undef RSVD_STAGED
    RSVD_LAUNCH_CHECK();
  }
  return splits > 1 ? launch_splitk_reduce<float>(c, M, N, (int)splits, work.p, beta, C, ldc, false)
                    : 0;
}

static int check_dims(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc,
                      char ta, char tb) {
  if (M < 0 || N < 0 || K < 0) return set_error("gemm: negative dimension");
  const bool tA = (ta == 'T' || ta == 't'), tB = (tb == 'T' || tb == 't');
  if (lda < (tA ? (K > 0 ? K : 1) : (M > 0 ? M : 1)))
    return set_error("gemm: lda=%lld too small", (long long)lda);
  if (ldb < (tB ? (N > 0 ? N : 1) : (K > 0 ? K : 1)))
    return set_error("gemm: ldb=%lld too small", (long long)ldb);
  if (ldc < (M > 0 ? M : 1)) return set_error("gemm: ldc=%lld too small", (long long)ldc);
  return 0;
}

template <typename T>
__global__ void scale_kernel(int64_t M, int64_t N, T beta, T* C, int64_t ldc) {
  int64_t total = M * N;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    int64_t i = idx % M, j = idx / M;
    C[i + j * ldc] = beta == T(0) ? T(0) : beta * C[i + j * ldc];
  }
}

// With rsvd_set_fp64_vendor_gemm(1), the A-streaming FP64 products of the
// plain path (Y = A X, Z = A^T Y, B^T = A^T Q: K in the thousands, 10+ GFLOP)
// run on rocBLAS's dgemm instead of gemm_kernel: a vendor reference the
// plain method can be timed against (off by default).  Never inside an
// allocation-free call (rocBLAS takes its own workspace), nor for dimensions
// beyond rocBLAS's 32-bit integers.
static int vendor_f64(Context* c, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                      int64_t ldc, bool* use) {
  *use = false;
  if (!c->fp64_vendor || c->scratch_mode) return 0;
  if (2.0 * (double)M * (double)N * (double)K < 1e10 || M * N < (int64_t(1) << 22) || K < 4096)
    return 0;
  for (int64_t v : {M, N, K, lda, ldb, ldc})
    if (v > INT_MAX) return 0;
  if (!c->blas) {
    rocblas_handle h = nullptr;
    if (rocblas_create_handle(&h) != rocblas_status_success)
      return set_error("rocblas_create_handle failed");
    if (rocblas_set_stream(h, c->stream) != rocblas_status_success) {
      rocblas_destroy_handle(h);
      return set_error("rocblas_set_stream failed");
    }
    c->blas = h;
  }
  *use = true;
  return 0;
}

template <typename T>
static int gemm_any(Context* c, char ta, char tb, int64_t M, int64_t N, int64_t K, T alpha,
                    const T* A, int64_t lda, const T* B, int64_t ldb, T beta, T* C, int64_t ldc,
                    const char* tag) {
  RSVD_TRY(check_dims(M, N, K, lda, ldb, ldc, ta, tb));
  if (M == 0 || N == 0) return 0;
  if constexpr (sizeof(T) == 8) {
    bool vendor = false;
    if (K > 0) RSVD_TRY(vendor_f64(c, M, N, K, lda, ldb, ldc, &vendor));
    if (vendor) {
      KTimer kt(c, tag);
      const bool tA = (ta == 'T' || ta == 't'), tB = (tb == 'T' || tb == 't');
      const double a = alpha, b = beta;
      const rocblas_status st = rocblas_dgemm(
          (rocblas_handle)c->blas, tA ? rocblas_operation_transpose : rocblas_operation_none,
          tB ? rocblas_operation_transpose : rocblas_operation_none, (rocblas_int)M,
          (rocblas_int)N, (rocblas_int)K, &a, A, (rocblas_int)lda, B, (rocblas_int)ldb, &b, C,
          (rocblas_int)ldc);
      if (st != rocblas_status_success)
        return set_error("rocblas_dgemm failed: %s", rocblas_status_to_string(st));
      return 0;
    }
  }
  if (K == 0) {
    int blocks = (int)((M * N + 255) / 256);
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(scale_kernel<T>, dim3(blocks), dim3(256), 0, c->stream, M, N, beta, C,
                       ldc);
    RSVD_LAUNCH_CHECK();
    return 0;
  }
  // no limit of the grid's (its x counts every tile, under 2^24 of them for any matrix that
  // fits the memory); more columns have always been refused
  if (N > 32 && (N + 63) / 64 > 65535)
    return set_error("gemm: N=%lld too large for the grid", (long long)N);
  // A^T A or B B^T with beta = 0: the entries on and above the diagonal are
  // formed and stored on both sides of it
  const bool tA = (ta == 'T' || ta == 't'), tB = (tb == 'T' || tb == 't');
  const bool sym = A == B && lda == ldb && tA != tB && M == N && beta == T(0);
  if constexpr (sizeof(T) == 4) {
    if (!sym && gemm_staged(tA, tB, M, N, K, lda, ldb))
      return launch_gemm_staged(c, tag, tA, tB, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
  }
  return launch_gemm<T>(c, gemm_plan<T>(c, tA, M, N, K, sym, false), ta, tb, M, N, K, alpha, A, lda, B,
                        ldb, beta, C, ldc, nullptr, sym, tag);
}

int gemm_split(Context* c, const char* tag, char ta, char tb, int64_t M, int64_t N, int64_t K,
               float alpha, const float* A, int64_t lda, const float* B, int64_t ldb, float beta,
               float* C, int64_t ldc, int split) {
  const bool tA = (ta == 'T' || ta == 't'), tB = (tb == 'T' || tb == 't');
  const bool sym = A == B && lda == ldb && tA != tB && M == N && beta == 0.0f;
  const GemmPlan pl = gemm_plan<float>(c, tA, M, N, K, sym, false, split);
  return split == 1 ? launch_gemm<float, 1>(c, pl, ta, tb, M, N, K, alpha, A, lda, B, ldb, beta, C,
                                            ldc, nullptr, sym, tag)
                    : launch_gemm<float, 3>(c, pl, ta, tb, M, N, K, alpha, A, lda, B, ldb, beta, C,
                                            ldc, nullptr, sym, tag);
}

int gemm_f64(Context* c, char ta, char tb, int64_t M, int64_t N, int64_t K, double alpha,
             const double* A, int64_t lda, const double* B, int64_t ldb, double beta, double* C,
             int64_t ldc) {
  return gemm_any<double>(c, ta, tb, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc,
                          "gemm_f64");
}

int gemm_f64_tag(Context* c, const char* tag, char ta, char tb, int64_t M, int64_t N, int64_t K,
                 double alpha, const double* A, int64_t lda, const double* B, int64_t ldb,
                 double beta, double* C, int64_t ldc) {
  return gemm_any<double>(c, ta, tb, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, tag);
}

int gemm_f32(Context* c, char ta, char tb, int64_t M, int64_t N, int64_t K, float alpha,
             const float* A, int64_t lda, const float* B, int64_t ldb, float beta, float* C,
             int64_t ldc) {
  return gemm_any<float>(c, ta, tb, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, "gemm_f32");
}

int gemm_f64_deflate(Context* c, int64_t M, int64_t N, int64_t K, const double* Q, int64_t ldq,
                     const double* B, int64_t ldb, double* C, int64_t ldc, double* sumsq) {
  RSVD_TRY(check_dims(M, N, K, ldq, ldb, ldc, 'N', 'N'));
  if (M == 0 || N == 0) {
    RSVD_HIP(hipMemsetAsync(sumsq, 0, sizeof(double), c->stream));
    return 0;
  }
  const int64_t k = K > 0 ? K : 1;
  const GemmPlan pl = gemm_plan<double>(c, false, M, N, k, false, true);
  const int64_t nparts = pl.gx * pl.gy;
  DBuf<double> part;
  RSVD_TRY(part.alloc((size_t)nparts));
  RSVD_TRY(launch_gemm<double>(c, pl, 'N', 'N', M, N, k, -1.0, Q, ldq, B, ldb, 1.0, C, ldc, part.p,
                               false, "gemm_f64_deflate"));
  hipLaunchKernelGGL(sum_partials_kernel, dim3(1), dim3(256), 0, c->stream, nparts,
                     (const double*)part.p, sumsq);
  RSVD_LAUNCH_CHECK();
  return 0;
}

}  // namespace rsvd
