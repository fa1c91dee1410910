// fp32 flash-attention 2, forward and backward: the reference's precision,
// on the fp32 matrix instruction v_mfma_f32_16x16x4_f32.
//
// Reference: flash_attn2_causal_fwd (src/kernels/flash_attn2.rs:61-126), the
// bidirectional forward it mirrors (:57-58), flash_attn2_causal_bwd (:135-203)
// and flash_attn2_backward (:209-279).  The reference runs one 128-thread CTA
// per query row and walks every key, masked ones included, and adds dK/dV
// with fp32 atomics.  Here:
//   forward  a wavefront per 16 query rows, 64 rows per workgroup, the online
//            softmax per 32-key tile, causal blocks skipped;
//   backward split like FA2's two-kernel form: a q-parallel kernel for dQ,
//            which also stores Delta = rowsum(O * dO), and a k-parallel
//            kernel for dK/dV (no atomics, deterministic).
// Layout [B, H, S, D] contiguous (= the reference's [BH, S, D]); GQA maps q
// head h to kv head h / (Hq / Hkv).
//
// Bound: the fp32 matrix rate (145 TFLOP/s measured on a 4096^3 product),
// and at short sequences one wavefront's chain through its tiles.  Every
// product is fp32 with fp32 accumulation, as before, so the results are as
// exact as those of the lane-per-row form that this replaced.
// B2 H16 S1024 D64 causal, this against that form: forward 66 us (1141), dQ 83
// (1035 + 7 for Delta), dK/dV 102 (1752); B4 Hq32 Hkv8 S2048 D128, 1280, 1680
// and 2320 us, 108 TFLOP/s in the forward.  Reading the operands two chunks
// ahead took dK/dV from 110 to 102 us and left the others; a second group of 4
// wavefronts per workgroup on every second tile gained up to 1.1 at D = 32 and
// lost up to 1.15 at large grids (its barrier puts every wavefront's softmax
// in the same place), and was left out.
//
// The 16x16x4 layout (lane l, j = l % 16, g = l / 16): A[i][k] has i = j and
// k = g, B[k][j] has k = g, and C[i][j] register r is row i = 4 g + r.  So
//   * a 16-byte read of four consecutive d of a row feeds four products (the
//     summation index may be permuted as long as A and B agree): product t of
//     chunk c sums d = 16 c + 4 g + t;
//   * scores are formed transposed, S^T = K Q^T (dK/dV: S = Q K^T), so a lane
//     owns one query (key) column and register r of a 16-row subtile is row
//     4 g + r, which is the B operand of product r of the next contraction
//     over those rows without any exchange between lanes;
//   * that contraction's A operand, X^T[d][row 4 g + t], is read 16 bytes (4
//     consecutive d) at a time as well: the four values feed the four output
//     tiles whose row i stands for d = 4 i + tile, so a lane ends up with 16
//     consecutive d of its column.
// Tiles of 32 rows stream into LDS by buffer_load ... lds one tile ahead (two
// buffers); the 16-byte chunks of a row are XOR-permuted so that 16 rows read
// at one chunk, and 16 chunks of one row, fall into distinct banks.
#include "f32_mfma.h"

namespace {

constexpr int kWaves = 4;            // wavefronts per workgroup
constexpr int kRows = 16 * kWaves;   // query (or key) rows per workgroup
constexpr int kTile = 32;            // rows per LDS tile

// 16-byte chunk index of chunk c of tile row r: rows of D / 4 chunks, the
// chunk XORed with the row's line (256 bytes) so that 16 consecutive rows'
// chunk c lie in distinct banks.
template <int D>
DEVI int chunk_at(int r, int c) {
  constexpr int CPR = D / 4;
  constexpr int RPL = CPR >= 16 ? 1 : 16 / CPR;      // rows per 256-byte line
  constexpr int M = (CPR >= 16 ? 16 : CPR) - 1;
  return r * CPR + (c ^ ((r / RPL) & M));
}

template <int D>
struct Tile : Geo<D> {
  static constexpr int CPR = D / 4;           // 16-byte chunks per row
  static constexpr int TILE = kTile * D * 4;  // bytes of a tile
  static constexpr int NLD = TILE / 1024;     // 1 KiB loads per tile
};

// Rows row0 .. row0 + 31 of a [n, D] head at `base` into LDS; rows at or past
// n load as zeros (outside the descriptor's range).  The descriptor is built
// per tile, so a head may be larger than its 32-bit offsets reach.  A tensor
// that is not 16-byte aligned is copied through registers.
template <int D>
DEVI void load_tile(const float* base, int row0, int n, char* lds, int wave, int lane) {
  const int rows = min(kTile, n - row0);
  if ((reinterpret_cast<uintptr_t>(base) & 15) != 0) {
    for (int x = wave * 64 + lane; x < kTile * D; x += 64 * kWaves) {
      const int r = x / D, d = x % D;
      reinterpret_cast<float*>(lds)[chunk_at<D>(r, d / 4) * 4 + (d & 3)] =
          r < rows ? base[(long)row0 * D + x] : 0.0f;
    }
    return;
  }
  const auto rs = make_rsrc(base + (long)row0 * D, rows * D * 4);
#pragma unroll
  for (int i0 = 0; i0 < Tile<D>::NLD; i0 += kWaves) {
    const int i = i0 + wave;
    if (i < Tile<D>::NLD) {
      const int L = i * 64 + lane, r = L / Tile<D>::CPR, c = L % Tile<D>::CPR;
      dma16(rs, lds + i * 1024, (uint32_t)chunk_at<D>(r, c) * 16, 0);
    }
  }
}

// A row-wise A operand of one tile row: chunk c's four d
template <int D>
DEVI f32x4 row_chunk(const char* tile, int r, int c, int g) {
  if constexpr (D == 8) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(tile + chunk_at<D>(r, g & 1) * 16);
    return g < 2 ? x : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  } else {
    return *reinterpret_cast<const f32x4*>(tile + chunk_at<D>(r, 4 * c + g) * 16);
  }
}
// out[u] = (rows 16 u + i of the tile) . (the lane's column), u = 0, 1: two
// independent chains
template <int D>
DEVI void score(const char* tile, const f32x4* col, int j, int g, f32x4* out) {
#pragma unroll
  for (int u = 0; u < 2; ++u) out[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // operands are read two chunks ahead of their products
  constexpr int NC = Geo<D>::NC, RA = 2;
  f32x4 a[RA + 1][2];
  auto read = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u) a[c % (RA + 1)][u] = row_chunk<D>(tile, 16 * u + j, c, g);
  };
#pragma unroll
  for (int c = 0; c < RA && c < NC; ++c) read(c);
  sched_group(kDsRead, 2 * (RA < NC ? RA : NC));
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (c + RA < NC) read(c + RA);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) out[u] = mfma4(a[c % (RA + 1)][u][t], col[c][t], out[u]);
    if (c + RA < NC) sched_group(kDsRead, 2);
    sched_group(kMfma, 8);
  }
  __builtin_amdgcn_sched_barrier(0);
}

// acc += (tile)^T . p, p[u][t] at tile row 16 u + 4 g + t
template <int D>
DEVI void accumulate(const char* tile, const f32x4* p, int j, int g,
                     f32x4 (*acc)[Geo<D>::VW]) {
  // operands are read RA rows ahead of their products
  constexpr int VW = Geo<D>::VW, NH = Geo<D>::NH, RA = D == 128 ? 1 : 2;
  float a[RA + 1][NH][VW];
  auto read = [&](int s) __attribute__((always_inline)) {
    const int r = 16 * (s >> 2) + 4 * g + (s & 3);
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      float* x = a[s % (RA + 1)][h];
      if constexpr (VW == 4) {
        const f32x4 y = *reinterpret_cast<const f32x4*>(tile + chunk_at<D>(r, 16 * h + j) * 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = y[e];
      } else if constexpr (VW == 2) {
        const f32x2 y = *reinterpret_cast<const f32x2*>(tile + chunk_at<D>(r, j / 2) * 16 +
                                                        8 * (j & 1));
        x[0] = y[0];
        x[1] = y[1];
      } else {
        const int d = D == 8 ? (j & 7) : j;
        x[0] = *reinterpret_cast<const float*>(tile + chunk_at<D>(r, d / 4) * 16 + 4 * (d & 3));
        if (D == 8 && j >= 8) x[0] = 0.0f;
      }
    }
  };
#pragma unroll
  for (int s = 0; s < RA; ++s) read(s);
  sched_group(kDsRead, RA * NH);
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    if (s + RA < 8) read(s + RA);
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
      for (int e = 0; e < VW; ++e)
        acc[h][e] = mfma4(a[s % (RA + 1)][h][e], p[s >> 2][s & 3], acc[h][e]);
    if (s + RA < 8) sched_group(kDsRead, NH);
    sched_group(kMfma, NH * VW);
  }
  __builtin_amdgcn_sched_barrier(0);
}

// Whether every element of the tile is finite (0 * x is 0, or NaN)
template <int D>
DEVI bool tile_finite(const char* tile, int lane) {
  constexpr int N = D / 8;  // 16-byte reads per lane, up to 8 in flight
  f32x4 t = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i0 = 0; i0 < N; i0 += 8) {
    f32x4 x[8];
#pragma unroll
    for (int i = 0; i < 8 && i0 + i < N; ++i)
      x[i] = *reinterpret_cast<const f32x4*>(tile + ((i0 + i) * 64 + lane) * 16);
#pragma unroll
    for (int i = 0; i < 8 && i0 + i < N; ++i) t += 0.0f * x[i];
    __builtin_amdgcn_sched_barrier(0);
  }
  const float s = (t[0] + t[1]) + (t[2] + t[3]);
  return __builtin_amdgcn_ballot_w64(s != s) == 0;
}

// A causal tile on the diagonal that is not finite is left out of the products
// (0 * Inf of a masked row is NaN in a sum over rows); its rows are then added
// one by one, from global memory and after the walk, to the columns that see
// them: row_dot is a row's product with the lane's column, add_row adds w * row.
// The walk itself keeps its registers; the test of one tile per walk took the
// backward of B2 H16 S1024 D64 from 170 to 173 us and that of B4 Hq32 Hkv8 S2048
// D128 from 3.98 to 4.03 ms, the forwards are within a run's spread.
template <int D>
DEVI float row_dot(const float* row, const f32x4* col, int g) {
  f32x4 x[Geo<D>::NC];
  row_regs<D>(row, g, x);
  float s = 0.0f;
#pragma unroll
  for (int c = 0; c < Geo<D>::NC; ++c)
#pragma unroll
    for (int t = 0; t < 4; ++t) s += x[c][t] * col[c][t];
  return sum_g(s);
}
template <int D>
DEVI void add_row(const float* row, float w, int g, f32x4 (*acc)[Geo<D>::VW]) {
  constexpr int VW = Geo<D>::VW;
  if (D == 8 && g >= 2) return;
#pragma unroll
  for (int h = 0; h < Geo<D>::NH; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int e = 0; e < VW; ++e)
        acc[h][e][r] += w * row[16 * VW * h + VW * (4 * g + r) + e];
}

// Work item of a workgroup: (rank, head), rank 0 a head's longest walk, all
// heads' rank 0 first.  With a multiple of 8 heads one XCD (ids deal round
// robin) sees whole heads.  Where everything is resident at once, the time is
// that of the CU with the most work: every second round of 32 workgroups per
// XCD is taken backwards, so that a CU that got a long walk in one round gets
// a short one in the next (B2 H16 S1024 D64 causal,
// against row blocks in order: forward 99 -> 66 us, dQ 127 -> 84, dK/dV 161 -> 110).
DEVI void work_item(int heads, int& rank, int& head) {
  constexpr int kRound = 32 * TEENY_NUM_XCD;
  int s = blockIdx.x;
  const int round = s / kRound, p = s - round * kRound;
  if ((round & 1) && (round + 1) * kRound <= (int)gridDim.x)
    s = round * kRound + (31 - p / TEENY_NUM_XCD) * TEENY_NUM_XCD + p % TEENY_NUM_XCD;
  rank = s / heads;
  head = s - rank * heads;
}

// one barrier per tile: this wavefront's loads of the tile have landed, then
// everyone's have, and everyone is done with the buffer that is loaded next
DEVI void tile_ready() {
  __builtin_amdgcn_s_waitcnt(kVmWaitLgkm0<0>());
  barrier_only();
}

template <int D, bool CAUSAL>
__device__ __forceinline__ void fwd_f32(const float* __restrict__ q, const float* __restrict__ k,
                                        const float* __restrict__ v, float* __restrict__ o,
                                        float* __restrict__ lse, int nq, int nk, float scale,
                                        int hq, int hkv, int heads) {
  struct __attribute__((aligned(16))) Smem {
    char k[2][Tile<D>::TILE];
    char v[2][Tile<D>::TILE];
  };
  __shared__ Smem sm;
  const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int rank, bh;
  work_item(heads, rank, bh);
  const int b = bh / hq, h = bh - b * hq;
  const long kvh = (long)b * hkv + h / (hq / hkv);
  const int row0 = (CAUSAL ? (nq - 1) / kRows - rank : rank) * kRows;
  const int w0 = row0 + 16 * wave;  // this wavefront's first row
  const int qpos = w0 + j;
  const float* kb = k + kvh * (long)nk * D;
  const float* vb = v + kvh * (long)nk * D;
  const int kend = CAUSAL ? min(nk, row0 + kRows) : nk;
  const int n_tiles = (kend + kTile - 1) / kTile;
  auto load = [&](int i, int buf) __attribute__((always_inline)) {
    if (i < n_tiles) {
      load_tile<D>(kb, i * kTile, nk, sm.k[buf], wave, lane);
      load_tile<D>(vb, i * kTile, nk, sm.v[buf], wave, lane);
    }
  };
  load(0, 0);
  f32x4 qf[Geo<D>::NC];
  row_regs<D>(q + ((long)bh * nq + min(qpos, nq - 1)) * D, g, qf);
  f32x4 acc[Geo<D>::NH][Geo<D>::VW];
  zero_acc<D>(acc);
  float m = -INFINITY, l = 0.0f;
  int redo = -1;  // the first row of a tile that was left out
  for (int i = 0; i < n_tiles; ++i) {
    const int buf = i & 1, t0 = i * kTile;
    tile_ready();
    load(i + 1, buf ^ 1);
    if (CAUSAL && t0 > w0 + 15) continue;  // past every row of this wavefront
    f32x4 s[2];
    score<D>(sm.k[buf], qf, j, g, s);
    const bool edge = t0 + kTile > nk || (CAUSAL && t0 + kTile - 1 > w0);
    float mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float x = s[u][r] * scale;
        if (edge) {
          const int kr = t0 + 16 * u + 4 * g + r;
          if (kr >= nk || (CAUSAL && kr > qpos)) x = -INFINITY;
        }
        s[u][r] = x;
        mx = fmaxf(mx, x);
      }
    // key 0 is in the first tile of every row, so m is its score or more
    const float m_new = fmaxf(m, max_g(mx));
    const float alpha = expf(m - m_new);
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[u][r] = expf(s[u][r] - m_new);
        l += s[u][r];
      }
#pragma unroll
    for (int hh = 0; hh < Geo<D>::NH; ++hh)
#pragma unroll
      for (int e = 0; e < Geo<D>::VW; ++e) acc[hh][e] *= alpha;
    if (CAUSAL && edge && !tile_finite<D>(sm.v[buf], lane)) {
      redo = t0;  // a wavefront's last tile
      continue;
    }
    accumulate<D>(sm.v[buf], s, j, g, acc);
  }
  if (CAUSAL && redo >= 0)
#pragma unroll 1
    for (int r = redo; r < min(nk, min(redo + kTile, w0 + 16)); ++r) {
      const float p = expf(row_dot<D>(kb + (long)r * D, qf, g) * scale - m);
      if (r <= qpos) add_row<D>(vb + (long)r * D, p, g, acc);
    }
  l = sum_g(l);
  if (qpos >= nq) return;
  store_col<D>(o + ((long)bh * nq + qpos) * D, acc, g, [&](float x) { return x / l; });
  if (g == 0) lse[(long)bh * nq + qpos] = m + logf(l);
}

// dQ: a wavefront per 16 query rows, walking keys 0..q (causal) or all keys;
// it also stores Delta[bh, q] = sum_d O * dO (flash_attn2.rs:171 / :247) for
// the dK/dV kernel that follows.
template <int D, bool CAUSAL>
__device__ __forceinline__ void bwd_dq_f32(const float* __restrict__ q,
                                           const float* __restrict__ k,
                                           const float* __restrict__ v,
                                           const float* __restrict__ o,
                                           const float* __restrict__ dout,
                                           const float* __restrict__ lse,
                                           float* __restrict__ delta, float* __restrict__ dq,
                                           int nq, int nk, float scale, int hq, int hkv,
                                           int heads) {
  struct __attribute__((aligned(16))) Smem {
    char k[2][Tile<D>::TILE];
    char v[2][Tile<D>::TILE];
  };
  __shared__ Smem sm;
  const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int rank, bh;
  work_item(heads, rank, bh);
  const int b = bh / hq, h = bh - b * hq;
  const long kvh = (long)b * hkv + h / (hq / hkv);
  const int row0 = (CAUSAL ? (nq - 1) / kRows - rank : rank) * kRows;
  const int w0 = row0 + 16 * wave;
  const int qpos = w0 + j;
  const long row = (long)bh * nq + min(qpos, nq - 1);
  const float* kb = k + kvh * (long)nk * D;
  const float* vb = v + kvh * (long)nk * D;
  const int kend = CAUSAL ? min(nk, row0 + kRows) : nk;
  const int n_tiles = (kend + kTile - 1) / kTile;
  auto load = [&](int i, int buf) __attribute__((always_inline)) {
    if (i < n_tiles) {
      load_tile<D>(kb, i * kTile, nk, sm.k[buf], wave, lane);
      load_tile<D>(vb, i * kTile, nk, sm.v[buf], wave, lane);
    }
  };
  load(0, 0);
  f32x4 qf[Geo<D>::NC], dof[Geo<D>::NC];
  row_regs<D>(q + row * D, g, qf);
  row_regs<D>(dout + row * D, g, dof);
  float dl = 0.0f;
  {
    f32x4 of[Geo<D>::NC];
    row_regs<D>(o + row * D, g, of);
#pragma unroll
    for (int c = 0; c < Geo<D>::NC; ++c)
#pragma unroll
      for (int t = 0; t < 4; ++t) dl += of[c][t] * dof[c][t];
    dl = sum_g(dl);
  }
  if (g == 0 && qpos < nq) delta[row] = dl;
  const float L = lse[row];
  f32x4 acc[Geo<D>::NH][Geo<D>::VW];
  zero_acc<D>(acc);
  int redo = -1;  // as in the forward
  for (int i = 0; i < n_tiles; ++i) {
    const int buf = i & 1, t0 = i * kTile;
    tile_ready();
    load(i + 1, buf ^ 1);
    if (CAUSAL && t0 > w0 + 15) continue;
    const bool edge = t0 + kTile > nk || (CAUSAL && t0 + kTile - 1 > w0);
    if (CAUSAL && edge && !tile_finite<D>(sm.k[buf], lane)) {
      redo = t0;
      continue;
    }
    f32x4 s[2], dp[2];
    score<D>(sm.k[buf], qf, j, g, s);
    score<D>(sm.v[buf], dof, j, g, dp);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float ds = expf(s[u][r] * scale - L) * (dp[u][r] - dl);
        if (edge) {
          const int kr = t0 + 16 * u + 4 * g + r;
          if (kr >= nk || (CAUSAL && kr > qpos)) ds = 0.0f;
        }
        s[u][r] = ds;
      }
    accumulate<D>(sm.k[buf], s, j, g, acc);
  }
  if (CAUSAL && redo >= 0)
#pragma unroll 1
    for (int r = redo; r < min(nk, min(redo + kTile, w0 + 16)); ++r) {
      const float p = expf(row_dot<D>(kb + (long)r * D, qf, g) * scale - L);
      const float ds = p * (row_dot<D>(vb + (long)r * D, dof, g) - dl);
      if (r <= qpos) add_row<D>(kb + (long)r * D, ds, g, acc);
    }
  if (qpos >= nq) return;
  store_col<D>(dq + row * D, acc, g, [&](float x) { return x * scale; });
}

// dK, dV: a wavefront per 16 key rows of a kv head, walking the 32-row q tiles
// of every q head in its GQA group (q >= key when causal).  `shares`
// workgroups share the walk's (head, tile) items out; with more than one
// the sums go to part as fp32 [dK | dV][share][B, Hkv, nk, D] (dK
// unscaled), which the merge kernel adds in order.
template <int D, bool CAUSAL>
__device__ __forceinline__ void bwd_dkdv_f32(const float* __restrict__ q,
                                             const float* __restrict__ k,
                                             const float* __restrict__ v,
                                             const float* __restrict__ dout,
                                             const float* __restrict__ lse,
                                             const float* __restrict__ delta,
                                             float* __restrict__ dk, float* __restrict__ dv,
                                             float* __restrict__ part, int nq, int nk,
                                             float scale, int hq, int hkv, int heads,
                                             int shares) {
  struct __attribute__((aligned(16))) Smem {
    char q[2][Tile<D>::TILE];
    char dout[2][Tile<D>::TILE];
    float ld[2][2][kTile];  // LSE, Delta of the tile's rows
  };
  __shared__ Smem sm;
  const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int rank, kvh;
  work_item(heads * shares, rank, kvh);
  const int share = kvh / heads;
  kvh -= share * heads;  // b * hkv + hk
  const int b = kvh / hkv, hk = kvh - b * hkv;
  const int group = hq / hkv;
  const int row0 = rank * kRows;
  const int w0 = row0 + 16 * wave;
  const int kpos = w0 + j;
  const long krow = (long)kvh * nk + min(kpos, nk - 1);
  // the walk: q tiles first .. n_q - 1 of each head of the group
  const int n_q = (nq + kTile - 1) / kTile;
  const int first = CAUSAL ? min(row0 / kTile, n_q) : 0;
  const int per_head = n_q - first;
  const int items = group * per_head;  // below 2^31 (the host's shape check)
  const int i0 = (int)((long)items * share / shares);
  const int i1 = (int)((long)items * (share + 1) / shares);
  float rv = 0.0f;  // threads 0..63: the next tile's LSE or Delta of one row
  auto tile_row = [&](int i) { return (first + i % per_head) * kTile; };
  auto load = [&](int i, int buf) __attribute__((always_inline)) {
    if (i >= i1) return;
    const long bh = (long)b * hq + (long)hk * group + i / per_head;
    const int t0 = tile_row(i);
    load_tile<D>(q + bh * nq * D, t0, nq, sm.q[buf], wave, lane);
    load_tile<D>(dout + bh * nq * D, t0, nq, sm.dout[buf], wave, lane);
    if (tid < 2 * kTile) {
      // rows past the end: P = exp(0 - inf) = 0, masked below too (0 * inf)
      const int r = t0 + (tid & (kTile - 1));
      const float* src = tid < kTile ? lse : delta;
      rv = r < nq ? src[bh * nq + r] : tid < kTile ? INFINITY : 0.0f;
    }
  };
  load(i0, 0);
  f32x4 kf[Geo<D>::NC], vf[Geo<D>::NC];
  row_regs<D>(k + krow * D, g, kf);
  row_regs<D>(v + krow * D, g, vf);
  f32x4 dka[Geo<D>::NH][Geo<D>::VW], dva[Geo<D>::NH][Geo<D>::VW];
  zero_acc<D>(dka);
  zero_acc<D>(dva);
  int buf = 0, redo = i1;  // the first item whose diagonal tile was left out
  for (int i = i0; i < i1; ++i, buf ^= 1) {
    const int t0 = tile_row(i);
    if (tid < 2 * kTile) sm.ld[buf][tid / kTile][tid & (kTile - 1)] = rv;
    tile_ready();
    load(i + 1, buf ^ 1);
    if (CAUSAL && t0 + kTile - 1 < w0) continue;  // before every key of this wavefront
    if (CAUSAL && t0 < w0 + 15 &&
        (i >= redo || !(tile_finite<D>(sm.dout[buf], lane) && tile_finite<D>(sm.q[buf], lane)))) {
      redo = min(redo, i);
      continue;
    }
    f32x4 s[2], dp[2];
    score<D>(sm.q[buf], kf, j, g, s);
    score<D>(sm.dout[buf], vf, j, g, dp);
    const bool edge = t0 + kTile > nq || (CAUSAL && t0 < w0 + 15);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const f32x4 L = *reinterpret_cast<const f32x4*>(&sm.ld[buf][0][16 * u + 4 * g]);
      const f32x4 dl = *reinterpret_cast<const f32x4*>(&sm.ld[buf][1][16 * u + 4 * g]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = expf(s[u][r] * scale - L[r]), ds = p * (dp[u][r] - dl[r]);
        const int qr = t0 + 16 * u + 4 * g + r;
        const bool off = edge && (qr >= nq || (CAUSAL && kpos > qr));
        s[u][r] = off ? 0.0f : p;
        dp[u][r] = off ? 0.0f : ds;
      }
    }
    accumulate<D>(sm.dout[buf], s, j, g, dva);
    accumulate<D>(sm.q[buf], dp, j, g, dka);
  }
  if (CAUSAL)
#pragma unroll 1
    for (int i = redo; i < i1; ++i) {
      const int t0 = tile_row(i);
      if (t0 >= w0 + 15) continue;
      const long bh = (long)b * hq + (long)hk * group + i / per_head;
#pragma unroll 1
      for (int r = max(t0, w0); r < min(nq, t0 + kTile); ++r) {
        const float* qr = q + (bh * nq + r) * D;
        const float* dor = dout + (bh * nq + r) * D;
        const float p = expf(row_dot<D>(qr, kf, g) * scale - lse[bh * nq + r]);
        const float ds = p * (row_dot<D>(dor, vf, g) - delta[bh * nq + r]);
        if (r >= kpos) {
          add_row<D>(dor, p, g, dva);
          add_row<D>(qr, ds, g, dka);
        }
      }
    }
  if (kpos >= nk) return;
  if (shares > 1) {
    const long n = (long)heads * nk * D;
    float* pk = part + share * n + krow * D;
    store_col<D>(pk, dka, g, [&](float x) { return x; });
    store_col<D>(pk + shares * n, dva, g, [&](float x) { return x; });
    return;
  }
  store_col<D>(dk + krow * D, dka, g, [&](float x) { return x * scale; });
  store_col<D>(dv + krow * D, dva, g, [&](float x) { return x; });
}

}  // namespace

#define TEENY_FA2_F32_INST_C(D, SFX, CAUSAL)                                                      \
  extern "C" __global__ __launch_bounds__(256) void teeny_fa2_fwd_f32_d##D##SFX(                 \
      const float* q, const float* k, const float* v, float* o, float* l, int nq, int nk,         \
      float scale, int hq, int hkv, int heads) {                                                  \
    fwd_f32<D, CAUSAL>(q, k, v, o, l, nq, nk, scale, hq, hkv, heads);                             \
  }                                                                                               \
  extern "C" __global__ __launch_bounds__(256) void teeny_fa2_bwd_dq_f32_d##D##SFX(              \
      const float* q, const float* k, const float* v, const float* o, const float* dout,          \
      const float* lse, float* delta, float* dq, int nq, int nk, float scale, int hq, int hkv,    \
      int heads) {                                                                                \
    bwd_dq_f32<D, CAUSAL>(q, k, v, o, dout, lse, delta, dq, nq, nk, scale, hq, hkv, heads);       \
  }                                                                                               \
  extern "C" __global__ __launch_bounds__(256) void teeny_fa2_bwd_dkdv_f32_d##D##SFX(            \
      const float* q, const float* k, const float* v, const float* dout, const float* lse,        \
      const float* delta, float* dk, float* dv, float* part, int nq, int nk, float scale, int hq, \
      int hkv, int heads, int shares) {                                                           \
    bwd_dkdv_f32<D, CAUSAL>(q, k, v, dout, lse, delta, dk, dv, part, nq, nk, scale, hq, hkv,      \
                            heads, shares);                                                       \
  }
#define TEENY_FA2_F32_INST(D)         \
  TEENY_FA2_F32_INST_C(D, _c, true)   \
  TEENY_FA2_F32_INST_C(D, _n, false)

TEENY_FA2_F32_INST(8)
TEENY_FA2_F32_INST(16)
TEENY_FA2_F32_INST(32)
TEENY_FA2_F32_INST(64)
TEENY_FA2_F32_INST(128)
