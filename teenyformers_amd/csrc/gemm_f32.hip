// fp32 linear layer y[M, N] = x[M, K] . w[N, K]^T at the reference's
// precision (teeny-core's Linear behind sym_linear, src/layers/mod.rs:54-58,
// runs in fp32; src/loader.rs:41,66-80 decodes every weight to f32).
//
// teeny_linear_f32 hands its products to hipBLASLt; these kernels are the
// library's own path for up to 4 rows of short products (the rule and its
// figures: capi.cpp) and where hipBLASLt does not take the device, shape or
// stream (a product under graph capture).
//
// Up to 64 rows (a decode step, one row per sequence): teeny_gemm_f32_sk_*,
// below.  More rows: teeny_gemm_f32_nt, each output one fp32 fused
// multiply-add chain over k in increasing order, so the result does not
// depend on the tiling.
//
// Tiling of teeny_gemm_f32_nt: a workgroup of 256 threads owns a 128 x 128 tile of y; 16-deep K
// slices of x and w are staged in LDS transposed (k-major), two buffers, so
// the next slice's global loads are in flight while the current one is
// multiplied; each thread accumulates an 8 x 8 block (rows ty*4 + {0..3} and
// 64 + ty*4 + {0..3}, columns likewise from tx) with 16-byte LDS reads.
// Rows past M or N and k past K load zeros and are never stored.
#include "f32_mfma.h"

namespace {

constexpr int TM = 128, TN = 128, TK = 16, PAD = 4;

struct Smem {
  float a[2][TK][TM + PAD];  // x slice, k-major
  float b[2][TK][TN + PAD];  // w slice, k-major
};

DEVI f32x4 load4(const float* __restrict__ base, long row, int nrows, int k, int K) {
  if (row < nrows && k < K) return *reinterpret_cast<const f32x4*>(base + row * K + k);
  return f32x4{0.0f, 0.0f, 0.0f, 0.0f};
}

}  // namespace

extern "C" __global__ __launch_bounds__(256) void teeny_gemm_f32_nt(
    const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ y, int M,
    int N, int K) {
  __shared__ Smem sm;
  const int tid = threadIdx.x;
  const int tx = tid & 15, ty = tid >> 4;
  const long m0 = (long)blockIdx.y * TM, n0 = (long)blockIdx.x * TN;

  // staging: each thread brings two 4-float k-runs of x and two of w per
  // slice: tile row r = tid / 4 (+64), k = 4 (tid % 4)
  const int lr = tid >> 2, lk = 4 * (tid & 3);
  auto fetch = [&](int k0, f32x4* ra, f32x4* rb) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      ra[h] = load4(x, m0 + lr + 64 * h, M, k0 + lk, K);
      rb[h] = load4(w, n0 + lr + 64 * h, N, k0 + lk, K);
    }
  };
  auto stash = [&](int buf, const f32x4* ra, const f32x4* rb) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        sm.a[buf][lk + j][lr + 64 * h] = ra[h][j];
        sm.b[buf][lk + j][lr + 64 * h] = rb[h][j];
      }
  };

  float acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = 0.0f;

  const int n_slices = (K + TK - 1) / TK;
  f32x4 ra[2], rb[2];
  fetch(0, ra, rb);
  stash(0, ra, rb);
  __syncthreads();
  for (int s = 0; s < n_slices; ++s) {
    const int buf = s & 1;
    if (s + 1 < n_slices) fetch((s + 1) * TK, ra, rb);
#pragma unroll
    for (int k = 0; k < TK; ++k) {
      const f32x4 a0 = *reinterpret_cast<const f32x4*>(&sm.a[buf][k][4 * ty]);
      const f32x4 a1 = *reinterpret_cast<const f32x4*>(&sm.a[buf][k][64 + 4 * ty]);
      const f32x4 b0 = *reinterpret_cast<const f32x4*>(&sm.b[buf][k][4 * tx]);
      const f32x4 b1 = *reinterpret_cast<const f32x4*>(&sm.b[buf][k][64 + 4 * tx]);
      const float av[8] = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
      const float bv[8] = {b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]};
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = __builtin_fmaf(av[i], bv[j], acc[i][j]);
    }
    if (s + 1 < n_slices) stash(buf ^ 1, ra, rb);
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const long m = m0 + (i < 4 ? 4 * ty + i : 64 + 4 * ty + i - 4);
    if (m >= M) continue;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const long n = n0 + 64 * h + 4 * tx;
      float* yr = y + m * N + n;
      if (n + 3 < N && (N & 3) == 0) {
        *reinterpret_cast<f32x4*>(yr) =
            f32x4{acc[i][4 * h], acc[i][4 * h + 1], acc[i][4 * h + 2], acc[i][4 * h + 3]};
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (n + j < N) yr[j] = acc[i][4 * h + j];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Few rows: y[M, N] = x[M, K] . w[N, K]^T, M <= 16 MT, bound by reading w once.
//
// A workgroup of 8 wavefronts owns 16 RT rows of w; the wavefronts take its
// 64-wide k chunks in turn (8 c + wavefront), so that each CU streams whole
// rows and the loop has no barrier, and their sums are added in wavefront
// order through LDS.  w rows are the A operand of v_mfma_f32_16x16x4_f32 and x
// rows the B operand: a 16-byte load of a lane (row l % 16, k = 4 (l / 16)) of
// each feeds four products (the k order inside 16 only has to agree).  The k
// order does not depend on RT and MT, so neither do the bits of an output on M.
// Rows past M or N repeat the last one and are not stored; the k past K of the
// last chunk load zeros.
//
// Measured from HBM (weights rotated past the last-level cache), 16 wavefronts
// per CU at M = 1: N32000 K2048 46 us (5.7 TB/s), N28672 K4096 83 us (5.7),
// N4096 K14336 41 us (5.7), N2048 K8192 21 us, N3072 K2048 8 us; the 128 x 128
// tiles took 0.5 ms each (2 ms at K8192).  Two or more chunks per register
// set, or two row tiles, leave one workgroup per CU and lost 2-20 % there; at
// M = 16 the x loads cost as much as w's, and two row tiles (half the x loads)
// gain up to 12 % once the grid still fills the CUs twice, and up to 25 % at
// M = 64.
// ---------------------------------------------------------------------------
namespace {

constexpr int SKW = 8;   // wavefronts per workgroup
constexpr int SKC = 64;  // k per chunk

template <int RT, int MT>
__device__ __forceinline__ void gemm_f32_sk(const float* __restrict__ x,
                                            const float* __restrict__ w, float* __restrict__ y,
                                            int M, int N, int K) {
  __shared__ __attribute__((aligned(16))) float red[SKW][RT * MT][64][4];
  const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long row0 = (long)blockIdx.x * (16 * RT);
  const float* wr[RT];
  const float* xr[MT];
#pragma unroll
  for (int r = 0; r < RT; ++r) wr[r] = w + min(row0 + 16 * r + j, (long)N - 1) * K + 4 * g;
#pragma unroll
  for (int m = 0; m < MT; ++m) xr[m] = x + (long)min(16 * m + j, M - 1) * K + 4 * g;
  f32x4 acc[RT][MT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[r][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 a[2][4][RT], b[2][4][MT];  // two register sets of a chunk
  auto load = [&](int set, int c) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = c * SKC + 16 * u;
#pragma unroll
      for (int r = 0; r < RT; ++r) a[set][u][r] = *reinterpret_cast<const f32x4*>(wr[r] + k);
#pragma unroll
      for (int m = 0; m < MT; ++m) b[set][u][m] = *reinterpret_cast<const f32x4*>(xr[m] + k);
    }
    // every load is issued before the products that follow wait for one
    __builtin_amdgcn_sched_barrier(0);
  };
  auto products = [&](int set) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int m = 0; m < MT; ++m)
            acc[r][m] = mfma4(a[set][u][r][e], b[set][u][m][e], acc[r][m]);
    __builtin_amdgcn_sched_barrier(0);
  };
  // this wavefront's whole chunks, the next one's loads in flight
  // (straight-line bodies: a branch around the loads would make the products
  // wait for all of them)
  const int n = max(0, (K / SKC - wave + SKW - 1) / SKW);
  int c = wave;
  if (n > 0) {
    int i = 0;
    load(0, c);
    for (; i + 2 < n; i += 2, c += 2 * SKW) {
      load(1, c + SKW);
      products(0);
      load(0, c + 2 * SKW);
      products(1);
    }
    if (i + 1 < n) {
      load(1, c + SKW);
      products(0);
      products(1);
      c += 2 * SKW;
    } else {
      products(0);
      c += SKW;
    }
  }
  // the last chunk of K, if it is not whole; K is a multiple of 4, so a load
  // is within K or past it
  if (c * SKC < K) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = c * SKC + 16 * u;
      const bool in = k + 4 * g < K;
#pragma unroll
      for (int r = 0; r < RT; ++r)
        a[0][u][r] = in ? *reinterpret_cast<const f32x4*>(wr[r] + k) : f32x4{0, 0, 0, 0};
#pragma unroll
      for (int m = 0; m < MT; ++m)
        b[0][u][m] = in ? *reinterpret_cast<const f32x4*>(xr[m] + k) : f32x4{0, 0, 0, 0};
    }
    products(0);
  }
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int m = 0; m < MT; ++m) *reinterpret_cast<f32x4*>(red[wave][r * MT + m][lane]) = acc[r][m];
  __syncthreads();
  // output (row 16 r + 4 g + i of w, row 16 m + j of x) is value i of lane
  // (j, g) of block (r, m): one lane of the workgroup per four w rows
  for (int t = threadIdx.x; t < RT * MT * 64; t += 64 * SKW) {
    const int blk = t >> 6, l = t & 63;
    f32x4 s = *reinterpret_cast<const f32x4*>(red[0][blk][l]);
#pragma unroll
    for (int v = 1; v < SKW; ++v) s += *reinterpret_cast<const f32x4*>(red[v][blk][l]);
    const int m = 16 * (blk % MT) + (l & 15);
    const long n = row0 + 16 * (blk / MT) + 4 * (l >> 4);
    if (m >= M) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n + i < N) y[(long)m * N + n + i] = s[i];
  }
}

}  // namespace

#define TEENY_GEMM_F32_SK(RT, MT)                                                          \
  extern "C" __global__ __launch_bounds__(64 * SKW) void teeny_gemm_f32_sk_r##RT##_m##MT( \
      const float* x, const float* w, float* y, int M, int N, int K) {                     \
    gemm_f32_sk<RT, MT>(x, w, y, M, N, K);                                                 \
  }
TEENY_GEMM_F32_SK(1, 1)
TEENY_GEMM_F32_SK(2, 1)
TEENY_GEMM_F32_SK(1, 2)
TEENY_GEMM_F32_SK(2, 2)
TEENY_GEMM_F32_SK(1, 4)
TEENY_GEMM_F32_SK(2, 4)
