// MFMA GEMMs for many activation rows:  out[m, n] = epi( sum_k X[m, k] * W[n, k] )
// gemm_rows_kernel (below): 65 to 256 rows (tree verification).  gemm_tile_kernel, here: the LM head
// over 65 to 128 rows, and products whose 32-bit offsets neither it nor the four-wave kernel reach
// (rows or weights of 4 GiB and more); the dispatch to gemm_quad.hip and the split reduction sit here too,
// with the epilogues of the decode GEMM (store / residual / SwiGLU / per-tile argmax for the LM
// head) -- the large-M counterpart of the reference's tensor-core GEMMs (gemv.py:61-116 with
// BLOCK_M >= 16, fast.py:161-213) and of its cuBLAS prefill (engine.py:550-592).
//
// CDNA4 mapping (v_mfma_f32_16x16x32_bf16, wave64, 160 KiB LDS per CU):
//  * a workgroup of 4 waves owns a 128 (weight rows) x 128 (activation rows) output tile; wave
//    (wn, wm) owns the 64 x 64 quarter (4 x 4 MFMA tiles, 64 fp32 accumulators per lane);
//  * K advances in stages of 64: both 128-row x 128-byte tiles are staged in LDS, each row as 8
//    16-byte units stored at unit ^ (row & 7), so the fragment reads (16 rows x one 16-byte unit)
//    and the staging writes (8 rows x 8 units per 8 lanes) hit distinct banks;
//  * two LDS buffers (64 KiB, two workgroups per CU) and a two-deep register ring: the global
//    loads of stage s + 2 are issued before stage s is contracted, stage s + 1 is written to the
//    other buffer after it, so one barrier per stage and two stages of loads in flight;
//  * A = weight rows, B = activation rows: the accumulator lane (c, q) holds output columns
//    n..n+3 (4 q + r) of row m (c), so every epilogue store is one 8-byte write;
//  * workgroup ids are remapped so the tiles that one XCD runs are consecutive in (M block
//    fastest, then N block): the M blocks that share a weight tile run on one XCD and meet in its
//    L2 instead of each XCD fetching the tile from HBM;
//  * when the tile grid is too small to fill the chip (few rows, narrow N), K is split over
//    workgroups; the fp32 partial tiles go to a caller-provided workspace and a second kernel
//    sums them in split order and applies the epilogue (deterministic).
// Requirements (checked by gemm_tile_ok): K % 64 == 0, N % 128 == 0 (SwiGLU: N % 64 == 0),
// 16-byte aligned X / W rows, 8-byte aligned output / residual rows.
#include "qd_launch.h"

namespace {

constexpr int TM = 128, TN = 128, TK = 64;
#ifndef QD_TILE_RING
#define QD_TILE_RING 2
#endif
// K stages of loads in flight per thread (even).  Measured on MI355X: 4 stages (250 VGPRs)
// took 8.18 ms per config-5 verify forward against 8.01 ms with 2 and left the 4 x 8192
// prefill unchanged -- the 256-row projections are not bound by load latency.
constexpr int TILE_RING = QD_TILE_RING;
static_assert(TILE_RING % 2 == 0, "the ring slots and the two LDS buffers advance together");
#ifndef QD_TILE_GROUP_M
#define QD_TILE_GROUP_M 8
#endif
constexpr int TILE_GROUP_M = QD_TILE_GROUP_M;
#ifndef QD_TILE_ROWS
#define QD_TILE_ROWS 1     // all-rows kernel at 65..256 rows
#endif
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

__device__ __forceinline__ bf16x8_t as_bf8(uint4 v) { return __builtin_bit_cast(bf16x8_t, v); }

struct TileLds {
  uint4 w[2][TN * 8];
  uint4 x[2][TM * 8];
};

// one stage of one thread's staging units: 4 weight and 4 activation 16-byte units (named
// registers: arrays here end up in scratch or LDS)
struct Stage {
  uint4 w0, w1, w2, w3, x0, x1, x2, x3;
};
struct Src {
  const uint4 *W, *X;
  int64_t w0, w1, w2, w3, x0, x1, x2, x3;   // uint4 offsets of the thread's 4 + 4 rows
};
__device__ __forceinline__ void load_stage(Stage& st, const Src& s, int64_t kk) {
  st.w0 = ld_stream(s.W + s.w0 + kk);
  st.w1 = ld_stream(s.W + s.w1 + kk);
  st.w2 = ld_stream(s.W + s.w2 + kk);
  st.w3 = ld_stream(s.W + s.w3 + kk);
  st.x0 = s.X[s.x0 + kk];
  st.x1 = s.X[s.x1 + kk];
  st.x2 = s.X[s.x2 + kk];
  st.x3 = s.X[s.x3 + kk];
}
__device__ __forceinline__ void store_stage(const Stage& st, uint4* lw, uint4* lx) {
  lw[0] = st.w0;
  lw[256] = st.w1;
  lw[512] = st.w2;
  lw[768] = st.w3;
  lx[0] = st.x0;
  lx[256] = st.x1;
  lx[512] = st.x2;
  lx[768] = st.x3;
}

template <int EPI, bool SPLIT>
__global__ __launch_bounds__(256, 2) void gemm_tile_kernel(
    const bf16_t* __restrict__ X, int64_t x_stride, int M, const bf16_t* __restrict__ W, int N,
    int K, int mblocks, int nblocks, int ks_per, bf16_t* out, int64_t out_stride, const bf16_t* res,
    int64_t res_stride, float* pval, int32_t* pidx, float* logits, float* part) {
  __shared__ TileLds sm;
  __shared__ float amax_v[2][2][64];
  __shared__ int32_t amax_i[2][2][64];
  // XCD-aware remap: hardware workgroup h runs on XCD h % 8; give each XCD a contiguous run of
  // logical tiles
  const int total = gridDim.x, h = blockIdx.x;
  const int xq = total >> 3, xr = total & 7, xcd = h & 7, slot = h >> 3;
  const int L = xcd < xr ? xcd * (xq + 1) + slot : xr * (xq + 1) + (xcd - xr) * xq + slot;
  // within a K split, tiles go in groups of TILE_GROUP_M M blocks: M fastest inside a group,
  // then N, so the workgroups one XCD runs at a time cover a few M blocks x many N blocks and
  // both the weight tiles and the activation tiles they read are shared in that XCD's L2
  const int tiles = mblocks * nblocks;
  const int split = L / tiles;
  const int Lt = L - split * tiles;
  const int group = Lt / (TILE_GROUP_M * nblocks);
  const int first = group * TILE_GROUP_M;
  const int gm = min(TILE_GROUP_M, mblocks - first);
  const int rr = Lt - first * nblocks;
  const int mb = first + rr % gm;
  const int nb = rr / gm;

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int c = lane & 15, q = lane >> 4;
  const int wn = wave & 1, wm = wave >> 1;
  const int64_t m0 = (int64_t)mb * TM;
  const int ksteps = K / TK;
  const int kbeg = split * ks_per;
  const int kend = min(ksteps, kbeg + ks_per);

  // staging: thread tid moves units u = tid + 256 i (i < 4) of both tiles: row r0 + 32 i
  // (r0 = tid / 8), unit tid % 8.  Weight row of LDS row r0 + 32 i: nb*128 + r0 + 32 i, or for
  // SwiGLU (gate | up halves of W, 64 output columns per block) nb*64 + r0 + 32 (i / 2) plus N
  // for odd i (the up rows).
  const int r0 = tid >> 3, unit0 = tid & 7;
  const int Nrows = EPI == EPI_SWIGLU ? 2 * N : N;
  auto wrow_of = [&](int i) -> int64_t {
    const int64_t wr = EPI == EPI_SWIGLU
                           ? (int64_t)nb * 64 + r0 + 32 * (i >> 1) + ((i & 1) ? N : 0)
                           : (int64_t)nb * TN + r0 + 32 * i;
    return (wr < Nrows ? wr : Nrows - 1) * (K / 8) + unit0;          // in uint4 units
  };
  auto xrow_of = [&](int i) -> int64_t {
    const int64_t xm = m0 + r0 + 32 * i;
    return (xm < M ? xm : M - 1) * (x_stride / 8) + unit0;
  };
  const Src src{reinterpret_cast<const uint4*>(W), reinterpret_cast<const uint4*>(X),
                wrow_of(0), wrow_of(1), wrow_of(2), wrow_of(3),
                xrow_of(0), xrow_of(1), xrow_of(2), xrow_of(3)};
  uint4* lw0 = &sm.w[0][r0 * 8 + (unit0 ^ (r0 & 7))];              // + 256 i: rows + 32 i
  uint4* lx0 = &sm.x[0][r0 * 8 + (unit0 ^ (r0 & 7))];
  Stage st[TILE_RING];
// (the scheduling barrier keeps the loads at the head of the stage: left free, the scheduler
// moves them behind the contraction and shortens the prefetch distance)
#define QD_LOAD(SLOT, KS)                                          \
  {                                                                \
    load_stage(st[SLOT], src, ((KS) < kend ? (KS) : kend - 1) * 8);\
    __builtin_amdgcn_sched_barrier(0);                             \
  }
#define QD_STORE(SLOT, BUF) store_stage(st[SLOT], lw0 + (BUF) * (TN * 8), lx0 + (BUF) * (TM * 8))
  f32x4_t acc[4][4];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) acc[nt][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int fa = (64 * wn + c) * 8, fb = (64 * wm + c) * 8;           // fragment rows (+ 128 t)
#define QD_COMPUTE(BUF)                                                                        \
  _Pragma("unroll") for (int s_ = 0; s_ < 2; ++s_) {                                           \
    const int u_ = (4 * s_ + q) ^ (c & 7);                                                     \
    uint4 a_[4], b_[4];                                                                        \
    _Pragma("unroll") for (int t = 0; t < 4; ++t) a_[t] = sm.w[BUF][fa + 128 * t + u_];        \
    _Pragma("unroll") for (int t = 0; t < 4; ++t) b_[t] = sm.x[BUF][fb + 128 * t + u_];        \
    _Pragma("unroll") for (int nt = 0; nt < 4; ++nt)                                           \
    _Pragma("unroll") for (int mt = 0; mt < 4; ++mt)                                           \
      acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf8(a_[nt]), as_bf8(b_[mt]),    \
                                                            acc[nt][mt], 0, 0, 0);             \
  }

  // Stage s sits in LDS buffer s & 1 while the loads of stages s + 1 .. s + TILE_RING are in
  // flight in the register ring (slot s % TILE_RING is refilled with stage s + TILE_RING once
  // stage s is in LDS).  Each stage: refill, contract, write stage s + 1 into the other buffer,
  // one barrier.  The loop body is TILE_RING stages with no exit between them (an exit there lets
  // the compiler sink loads to their use, behind the contraction they are meant to overlap);
  // the last partial round is guarded stage by stage.  Loads past the last stage are clamped.
#pragma unroll
  for (int r = 0; r < TILE_RING; ++r) QD_LOAD(r, kbeg + r);
  QD_STORE(0, 0);
  lds_barrier();
  int ks = kbeg;
  for (; ks + TILE_RING <= kend; ks += TILE_RING) {
#pragma unroll
    for (int r = 0; r < TILE_RING; ++r) {
      QD_LOAD(r, ks + r + TILE_RING);
      QD_COMPUTE(r & 1);
      QD_STORE((r + 1) % TILE_RING, (r + 1) & 1);
      lds_barrier();
    }
  }
#pragma unroll
  for (int r = 0; r < TILE_RING; ++r) {
    if (ks + r < kend) {
      QD_COMPUTE(r & 1);
      if (ks + r + 1 < kend) {
        QD_STORE((r + 1) % TILE_RING, (r + 1) & 1);
        lds_barrier();
      }
    }
  }
#undef QD_LOAD
#undef QD_STORE
#undef QD_COMPUTE

  // ---------------------------------------------------------------- epilogue
  // lane (c, q) of acc[nt][mt] holds rows 4 q + r (r < 4) of the weight tile = output columns
  // n .. n + 3, for activation row m = m0 + 64 wm + 16 mt + c
  if constexpr (SPLIT) {
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int64_t m = m0 + 64 * wm + 16 * mt + c;
      if (m >= M) continue;
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        const int64_t n = (int64_t)nb * TN + 64 * wn + 16 * nt + 4 * q;
        *reinterpret_cast<f32x4_t*>(part + ((int64_t)split * M + m) * N + n) = acc[nt][mt];
      }
    }
  } else if constexpr (EPI == EPI_ARGMAX) {
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int64_t m = m0 + 64 * wm + 16 * mt + c;
      const bool ok = m < M;
      float bv = -INFINITY;
      int32_t bi = 0x7FFFFFFF;
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        const int64_t n = (int64_t)nb * TN + 64 * wn + 16 * nt + 4 * q;
        if (ok && logits) *reinterpret_cast<f32x4_t*>(logits + m * (int64_t)N + n) = acc[nt][mt];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = rbf(acc[nt][mt][r]);
          if (v > bv) { bv = v; bi = (int32_t)(n + r); }   // ascending n within the lane
        }
      }
      // across the four q lanes of row c (interleaved column ranges): lowest index on ties
#pragma unroll
      for (int sh = 0; sh < 2; ++sh) {
        const float ov = sh ? lane_xor32(bv) : lane_xor16(bv);
        const int32_t oi = sh ? __builtin_bit_cast(int32_t, lane_xor32(__builtin_bit_cast(float, bi)))
                              : __builtin_bit_cast(int32_t, lane_xor16(__builtin_bit_cast(float, bi)));
        if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
      }
      if (q == 0) {
        amax_v[wm][wn][16 * mt + c] = bv;
        amax_i[wm][wn][16 * mt + c] = bi;
      }
    }
    lds_barrier();
    if (tid < 128) {
      const int wm2 = tid >> 6, r = tid & 63;
      const int64_t m = m0 + 64 * wm2 + r;
      if (m < M) {
        float bv = amax_v[wm2][0][r];
        int32_t bi = amax_i[wm2][0][r];
        const float ov = amax_v[wm2][1][r];
        const int32_t oi = amax_i[wm2][1][r];
        if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
        pval[m * (int64_t)nblocks + nb] = bv;
        pidx[m * (int64_t)nblocks + nb] = bi;
      }
    }
  } else {
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int64_t m = m0 + 64 * wm + 16 * mt + c;
      if (m >= M) continue;
      if constexpr (EPI == EPI_SWIGLU) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          const int64_t n = (int64_t)nb * 64 + 32 * wn + 16 * nt + 4 * q;
          float y[4];
#pragma unroll
          for (int r = 0; r < 4; ++r)
            y[r] = silu_rbf(rbf(acc[nt][mt][r])) * rbf(acc[nt + 2][mt][r]);
          *reinterpret_cast<uint2*>(out + m * out_stride + n) =
              make_uint2(pack2(y[0], y[1]), pack2(y[2], y[3]));
        }
      } else {
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
          const int64_t n = (int64_t)nb * TN + 64 * wn + 16 * nt + 4 * q;
          float y[4];
          if constexpr (EPI == EPI_RES) {
            const uint2 rv = *reinterpret_cast<const uint2*>(res + m * res_stride + n);
            y[0] = bflo(rv.x) + rbf(acc[nt][mt][0]);
            y[1] = bfhi(rv.x) + rbf(acc[nt][mt][1]);
            y[2] = bflo(rv.y) + rbf(acc[nt][mt][2]);
            y[3] = bfhi(rv.y) + rbf(acc[nt][mt][3]);
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) y[r] = acc[nt][mt][r];
          }
          *reinterpret_cast<uint2*>(out + m * out_stride + n) =
              make_uint2(pack2(y[0], y[1]), pack2(y[2], y[3]));
        }
      }
    }
  }
}

// Sum of the split partials in split order + epilogue (store / residual); one thread per four
// consecutive output columns.
template <int EPI>
__global__ __launch_bounds__(256) void gemm_split_reduce_kernel(const float* __restrict__ part,
                                                                int splits, int64_t M, int64_t N,
                                                                bf16_t* out, int64_t out_stride,
                                                                const bf16_t* res,
                                                                int64_t res_stride) {
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t n4 = N / 4;
  if (g >= M * n4) return;
  const int64_t m = g / n4, n = 4 * (g % n4);
  // partials summed in split order, loaded eight at a time before any of them is added
  constexpr int RB = 8;
  f32x4_t a = *reinterpret_cast<const f32x4_t*>(part + m * N + n);
  for (int z0 = 1; z0 < splits; z0 += RB) {
    f32x4_t v[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
      v[i] = z0 + i < splits ? *reinterpret_cast<const f32x4_t*>(part + ((int64_t)(z0 + i) * M + m) * N + n)
                             : f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < RB; ++i)
      if (z0 + i < splits) a += v[i];
  }
  float y[4];
  if constexpr (EPI == EPI_RES) {
    const uint2 rv = *reinterpret_cast<const uint2*>(res + m * res_stride + n);
    y[0] = bflo(rv.x) + rbf(a[0]);
    y[1] = bfhi(rv.x) + rbf(a[1]);
    y[2] = bflo(rv.y) + rbf(a[2]);
    y[3] = bfhi(rv.y) + rbf(a[3]);
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = a[r];
  }
  *reinterpret_cast<uint2*>(out + m * out_stride + n) = make_uint2(pack2(y[0], y[1]), pack2(y[2], y[3]));
}

// ------------------------------------------------------------------ all rows per workgroup (65..256)
// At a few hundred activation rows (a tree-verification forward: B x T = 256) a workgroup owns a
// block of weight rows for 128 MT of the activation rows (all of them, or one of two halves):
// 8 waves, wave w the 16 MT activation rows 16 MT w .. (NT x MT MFMA tiles; SwiGLU: NT gate
// tiles and the NT up tiles of the same outputs); K in stages of 64 that go from global memory
// straight into LDS (128-byte rows, unit u at u ^ (row & 7); the weight rows shared by the
// waves), RW_NBUF stage buffers, RW_NBUF - 1 stages in flight, one barrier per stage.  Every
// workgroup re-reads its activation rows' K range from L2, so the plan (rows_plan below) trades
// those re-reads against more K splits (fp32 partials for the consumer) or activation halves
// (each weight block read by two workgroups on one XCD, so the second read hits its L2).
// Measured on a config-5 verify (256 rows) against the 128 x 128 tiles: gate/up 58.6 -> 47.3 us,
// qkv 22.7 -> 20.3 us with the tiled kernel's split counts; stages of 32 in 7-8 buffers (twice
// the bytes in flight, twice the barriers) were slower (8.16 against 7.19 ms per verify).
constexpr int RW_MAXM = 256;                // activation rows per workgroup at most (8 waves x 32)
// Stage buffers: three (two stages in flight).  Four or five, which the LDS holds for every
// instantiation here, measured slower on a config-5 verify (6.56 / 6.60 against 6.51 ms): the
// loop's DMA, LDS reads and MFMAs each take about as long as the whole loop (timing copies),
// so deeper prefetch only adds LDS traffic.
#ifndef QD_RW_NBUF_MAX
#define QD_RW_NBUF_MAX 3
#endif
constexpr int RW_LDS_BYTES = 160 * 1024;
// stage buffers for `rows` staged rows (128 bytes each): as many as fit the CU's LDS, 3..max
__host__ __device__ constexpr int rw_nbuf(int rows) {
  return RW_LDS_BYTES / (rows * 128) > QD_RW_NBUF_MAX ? QD_RW_NBUF_MAX : RW_LDS_BYTES / (rows * 128);
}

template <int EPI, bool SPLIT, int NT, int MT>
__global__ __launch_bounds__(512, 1) void gemm_rows_kernel(
    const bf16_t* __restrict__ X, int64_t x_stride, int M, const bf16_t* __restrict__ W, int N,
    int K, int rows_per_wg, int S, int ks_per, int mh, bf16_t* out, int64_t out_stride,
    const bf16_t* res, int64_t res_stride, float* part) {
  constexpr bool SW = EPI == EPI_SWIGLU;
  constexpr int WT = SW ? 2 * NT : NT;       // weight tiles (gate tiles, then up tiles)
  constexpr int WR = 16 * WT;                // staged weight rows
  constexpr int RM = 128 * MT;               // staged activation rows
  constexpr int ROWS = WR + RM;              // staged rows per stage (weights, then activations)
  constexpr int NBLK = ROWS / 8;             // 1 KiB load blocks per stage (8 rows x 128 bytes)
  constexpr int PER = (NBLK + 7) / 8;        // loads per wave per stage (at most)
  constexpr int RW_NBUF = rw_nbuf(ROWS);
  static_assert(RW_NBUF >= 3 && RW_NBUF * ROWS * 128 <= RW_LDS_BYTES, "stage buffers");
  __shared__ uint4 sm[RW_NBUF][ROWS * 8];
  // workgroup -> (weight block, K split, activation half): the halves of one weight block are
  // workgroups g and g + 8 (dispatch puts workgroup g on XCD g % 8), so they share an L2
  const int nb = (N + rows_per_wg - 1) / rows_per_wg;
  int blkid = blockIdx.x, mb = 0;
  if (mh > 1) {
    const int slot = blockIdx.x >> 3;
    mb = slot % mh;
    blkid = (slot / mh) * 8 + (blockIdx.x & 7);
    if (blkid >= nb * S) return;             // the grid's padding to whole groups of 8
  }
  const int rb = blkid / S, split = blkid - rb * S;
  const int m0 = mb * RM;
  const int n0 = rb * rows_per_wg;
  const int nrows = min(rows_per_wg, N - n0);
  const int ksteps = K / TK;
  const int kbeg = split * ks_per, kend = min(ksteps, kbeg + ks_per);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // uniform: load bases in SGPRs
  const int c = lane & 15, q = lane >> 4;
  // LDS row r < WR: weight row n0 + r (SwiGLU: gate rows, then up rows + N); r >= WR: activation
  // row m0 + r - WR; rows past the block / past M reload a valid row (never stored)
  auto grow_off = [&](int r) -> uint32_t {
    if (r < WR) {
      int wr = SW ? (r % (16 * NT)) : r;
      wr = min(wr, nrows - 1);
      const int64_t row = (int64_t)n0 + wr + ((SW && r >= 16 * NT) ? N : 0);
      return (uint32_t)(row * K * 2);
    }
    const int xm = min(m0 + r - WR, M - 1);
    return (uint32_t)((int64_t)xm * x_stride * 2);
  };
  // wave w loads blocks w, w + 8, ... < NBLK (PER of them, or PER - 1 where NBLK is not a
  // multiple of 8: repeating blocks to even the waves out cost 10-12 % more load requests, the
  // stream this loop is bound by); lane l of a block: row l / 8, position l % 8, K unit
  // (l % 8) ^ (row % 8)
  static_assert(PER >= 2, "PER - 1 loads for the short waves");
  const bool full = wave + 8 * (PER - 1) < NBLK;   // uniform per wave
  uint32_t voff[PER];
  int blk[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    blk[j] = (wave + 8 * j) % NBLK;
    const int r = blk[j] * 8 + (lane >> 3);
    voff[j] = grow_off(r) + (uint32_t)(((lane & 7) ^ ((lane >> 3) & 7)) * 16);
  }
  const uint32_t lbase = __builtin_amdgcn_readfirstlane(lds_u32(&sm[0][0]));
  // loads j0 .. j1 - 1 of this wave's PER (or PER - 1) for stage ks into buffer buf
  auto issue = [&](int ks, int buf, int j0 = 0, int j1 = 1 << 30) {
    const char* wb = reinterpret_cast<const char*>(W) + (size_t)ks * (TK * 2);
    const char* xb = reinterpret_cast<const char*>(X) + (size_t)ks * (TK * 2);
    const uint32_t l = lbase + (uint32_t)buf * (ROWS * 128);
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (j >= j0 && j < j1 && (j < PER - 1 || full))
        dma16(blk[j] * 8 < WR ? wb : xb, voff[j], l + (uint32_t)blk[j] * 1024);
  };
  f32x4_t acc[WT][MT];
#pragma unroll
  for (int t = 0; t < WT; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const bool active = m0 + 16 * MT * wave < M;   // uniform per wave
  // contract the stage in buffer buf as two halves of K = 32, each preceded by half of the loads
  // of stage ks_next (< 0: none) into buf_next: issued between the MFMAs rather than all ahead of
  // them, the verify took 6.39 instead of 6.51 ms
  auto compute = [&](int buf, int ks_next, int buf_next) {
    const uint4* b0 = sm[buf];
#pragma unroll
    for (int s_ = 0; s_ < 2; ++s_) {
      if (ks_next >= 0) issue(ks_next, buf_next, s_ ? PER / 2 : 0, s_ ? PER : PER / 2);
      __builtin_amdgcn_sched_barrier(0);
      const int u_ = (4 * s_ + q) ^ (c & 7);
      uint4 a_[WT], b_[MT];
#pragma unroll
      for (int t = 0; t < WT; ++t) a_[t] = b0[(16 * t + c) * 8 + u_];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) b_[mt] = b0[(WR + 16 * MT * wave + 16 * mt + c) * 8 + u_];
#pragma unroll
      for (int t = 0; t < WT; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf8(a_[t]), as_bf8(b_[mt]),
                                                               acc[t][mt], 0, 0, 0);
    }
  };
  // stage kbeg + i in buffer i % RW_NBUF; at the top of step i this wave's loads of stage i have
  // landed once at most min(RW_NBUF - 2, stages after it) stages of its loads (PER or PER - 1 a
  // stage) are outstanding; after the barrier every wave's have, and every wave is done with
  // stage i - 1, whose buffer then takes stage i + RW_NBUF - 1
  constexpr int P = RW_NBUF - 1;
  const int nst = kend - kbeg;
#pragma unroll
  for (int i = 0; i < P; ++i)
    if (i < nst) issue(kbeg + i, i);
  int buf = 0;
  for (int i = 0; i < nst; ++i) {
    if (full) wait_stages<PER, P - 1>(nst - 1 - i);
    else wait_stages<PER - 1, P - 1>(nst - 1 - i);
    lds_barrier();
    const int kn = i + P < nst ? kbeg + i + P : -1, bn = buf + P < RW_NBUF ? buf + P : buf + P - RW_NBUF;
    if (active) compute(buf, kn, bn);
    else if (kn >= 0) issue(kn, bn);
    buf = buf + 1 < RW_NBUF ? buf + 1 : 0;
  }

  // epilogue: lane (c, q) of acc[t][mt] holds weight rows 4 q + r of tile t = output columns
  // n .. n + 3 of activation row m = m0 + 16 MT wave + 16 mt + c
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int64_t m = m0 + 16 * MT * wave + 16 * mt + c;
    if (m >= M) continue;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int u = 16 * t + 4 * q;          // output column offset in the block
      if (u >= nrows) continue;
      const int64_t n = (int64_t)n0 + u;
      if constexpr (SPLIT) {
        *reinterpret_cast<f32x4_t*>(part + ((int64_t)split * M + m) * N + n) = acc[t][mt];
      } else {
        float y[4];
        if constexpr (SW) {
#pragma unroll
          for (int r = 0; r < 4; ++r) y[r] = silu_rbf(rbf(acc[t][mt][r])) * rbf(acc[NT + t][mt][r]);
        } else if constexpr (EPI == EPI_RES) {
          const uint2 rv = *reinterpret_cast<const uint2*>(res + m * res_stride + n);
          y[0] = bflo(rv.x) + rbf(acc[t][mt][0]);
          y[1] = bfhi(rv.x) + rbf(acc[t][mt][1]);
          y[2] = bflo(rv.y) + rbf(acc[t][mt][2]);
          y[3] = bfhi(rv.y) + rbf(acc[t][mt][3]);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) y[r] = acc[t][mt][r];
        }
        *reinterpret_cast<uint2*>(out + m * out_stride + n) = make_uint2(pack2(y[0], y[1]), pack2(y[2], y[3]));
      }
    }
  }
}

int64_t tile_nblocks(int64_t N, int epi) { return epi == EPI_SWIGLU ? N / 64 : N / TN; }

}  // namespace

bool gemm_tile_ok(int64_t M, int64_t N, int64_t K, int epi, const void* x, int64_t x_stride,
                  const void* w, const void* out, int64_t out_stride, const void* res,
                  int64_t res_stride) {
  if (M <= 0 || K % TK != 0 || K < 2 * TK) return false;
  if (epi == EPI_SWIGLU ? N % 64 != 0 : N % TN != 0) return false;
  if (x_stride % 8 || reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(w) % 16)
    return false;
  if (epi != EPI_ARGMAX && (out_stride % 4 || reinterpret_cast<uintptr_t>(out) % 8)) return false;
  if (epi == EPI_RES && (res_stride % 4 || reinterpret_cast<uintptr_t>(res) % 8)) return false;
  return M * (int64_t)(N / 16) < (1ll << 40) && (M + TM - 1) / TM * tile_nblocks(N, epi) < (1ll << 30);
}


// K splits: only the store / residual epilogues split, when the tile grid leaves CUs idle; as
// many as keep the grid within one workgroup per CU (a grid a little past that puts two on some
// CUs, which then set the kernel's time: measured at 256 rows, 288 / 280-workgroup grids 9.09 ms
// per verify forward, the same GEMMs split to 192 / 240 workgroups 8.15 ms, to 480 8.72 ms), and
// at least 4 stages per split
int gemm_tile_splits(int64_t M, int64_t N, int64_t K, int epi) {
  if (epi != EPI_NONE && epi != EPI_RES) return 1;
  const int64_t tiles = (M + TM - 1) / TM * tile_nblocks(N, epi);
  if (tiles >= 160) return 1;
  int64_t sp = plan_cus() / tiles;
  const int64_t maxsp = (K / TK) / 4;
  if (sp > maxsp) sp = maxsp;
  return sp < 1 ? 1 : (int)sp;
}

// The all-rows kernel's plan for M <= 256 rows.  One round of workgroups; each workgroup moves
// (through its CU's L1 -> L2 request stream, which bounds this kernel) its weight rows' and its
// activation rows' K range, and with K splits writes fp32 partials that the consumer reads
// back.  The plan minimises that per-workgroup traffic over the K split count S (store /
// residual epilogues, when the caller takes partials), the activation halves (1 or 2) and the
// block height (a multiple of 4 rows, at most RW_NT_MAX MFMA tiles, the skinny GEMM's rule for
// the resulting workgroup count):
//   2 (K / S) (activation rows + weight rows) + [S > 1] 4 (activation rows x block rows
//   + S M N / CUs).
// On a config-5 verify (256 rows, 256 CUs) that picks two activation halves for every
// projection: qkv 96-row blocks in 2 K splits, o and down 124-row blocks in 6, gate/up 76 + 76
// rows (SwiGLU, no split); the four launches went from 105.9 to 98.7 us per layer (one half per
// workgroup for gate/up only: 6.86 against 6.63 ms per verify).
struct RowsPlan {
  int rows = 0, nt = 0, mt = 0, mh = 0, splits = 0, ks_per = 0;
};
constexpr int RW_NT_MAX = 8, RW_NT_MAX_SW = 5;

static int rows_nt_round(int nt, bool sw) {   // the instantiated block heights (MFMA tiles)
  if (sw) return nt < 2 ? 2 : nt;                              // 2..5
  if (nt <= 4) return nt;                                      // 1..4
  return nt <= 6 ? 6 : 8;
}

static bool rows_plan(int64_t M, int64_t N, int64_t K, int epi, bool can_split, RowsPlan& best) {
  best = RowsPlan();
  if (!QD_TILE_ROWS || M > RW_MAXM || epi == EPI_ARGMAX) return false;
  const bool sw = epi == EPI_SWIGLU;
  if ((sw ? 2 * N : N) * K * 2 >= (1ll << 32)) return false;
  const int64_t cus = plan_cus(), ksteps = K / TK;
  // the K split count stays the tiled kernel's (more splits measured slower at 256 rows: qkv in
  // 5 splits 20.2 -> 19.4 us, down in 12 splits 25.5 -> 24.0 us, but their consumers, which
  // read every split's partials, 8.8 -> 12.0 and 5.3 -> 7.7 us)
  const int64_t smax = can_split && !sw ? gemm_tile_splits(M, N, K, epi) : 1;
  double best_cost = 0;
  for (int mt = 1; mt <= 2; ++mt) {
    const int64_t rm = 128 * mt, mh = (M + rm - 1) / rm;
    if (mh > 2 || (mt == 2 && M <= 128)) continue;
    for (int64_t S0 = smax; S0 <= smax; ++S0) {
      const int64_t ks_per = (ksteps + S0 - 1) / S0, S = (ksteps + ks_per - 1) / ks_per;
      const int64_t per = cus / (S * mh);                      // weight blocks in one round
      if (per < 1) break;
      const int64_t rows = ((N + per - 1) / per + 3) / 4 * 4;
      const int nt = rows_nt_round((int)((rows + 15) / 16), sw);
      const int ntmax = sw ? RW_NT_MAX_SW : S > 1 ? RW_NT_MAX : 4;   // instantiated heights
      if (nt > ntmax || 16 * nt < rows) continue;
      const int64_t wgs = (N + rows - 1) / rows * S * mh;
      if (wgs > cus) continue;
      const double act = (double)(M < rm ? M : rm), wrows = (double)rows * (sw ? 2 : 1);
      double cost = 2.0 * ks_per * TK * (act + wrows);
      if (S > 1) cost += 4.0 * act * rows + 4.0 * S * M * N / cus;
      if (best.splits == 0 || cost < best_cost) {
        best_cost = cost;
        best.rows = (int)rows; best.nt = nt; best.mt = mt; best.mh = (int)mh;
        best.splits = (int)S; best.ks_per = (int)ks_per;
      }
    }
  }
  return best.splits > 0;
}

// The block height (MFMA tiles) of the instantiation launch_rows picks for a plan: SwiGLU 2..5,
// split-K 1..4, 6, 8, unsplit store / residual 1..4 (rows_plan's rounding and limits keep
// 16 x this >= the plan's rows).
static int rows_inst_nt(int nt, int epi, bool split) {
  if (epi == EPI_SWIGLU) return nt <= 2 ? 2 : nt >= 5 ? 5 : nt;
  if (split) return nt <= 1 ? 1 : nt <= 4 ? nt : nt <= 6 ? 6 : 8;
  return nt <= 1 ? 1 : nt >= 4 ? 4 : nt;
}

// What the launchers run on the all-rows kernel for (M, N, K, epi) with `part_floats` floats of
// split-partial room (0: none).  Returns -1 when the kernel does not take the shape (the tiled
// kernels do), 0 when it does but the caller only takes split partials (gemm_tile_partials) and
// no split fits, 1 with the plan to launch: split when the plan splits and the partials fit,
// else the unsplit plan.
static int rows_launch_plan(int64_t M, int64_t N, int64_t K, int epi, bool partials_only,
                            int64_t part_floats, RowsPlan& P) {
  if (M < GEMM_TILE_MIN_M || !rows_plan(M, N, K, epi, true, P)) return -1;
  const bool room = part_floats >= (int64_t)P.splits * M * N;
  if (partials_only) return P.splits > 1 && room ? 1 : 0;
  if (P.splits > 1 && !room) rows_plan(M, N, K, epi, false, P);   // no room for partials: S = 1
  return P.splits > 0 ? 1 : -1;
}

// the all-rows kernel's activation row offsets are 32-bit bytes
static bool rows_stride_ok(int64_t M, int64_t xs, int64_t K) { return ((M - 1) * xs + K) * 2 < (1ll << 32); }

template <int EPI, bool SPLIT>
static void launch_rows(const RowsPlan& P, const bf16_t* x, int64_t xs, int M, const bf16_t* w,
                        int N, int K, bf16_t* out, int64_t os, const bf16_t* res, int64_t rs,
                        float* part, hipStream_t s) {
  const int nblk = (N + P.rows - 1) / P.rows * P.splits;
  const int ng = P.mh > 1 ? (nblk + 7) / 8 * 8 * P.mh : nblk;
  const dim3 g((unsigned)ng), b(512);
#define QD_RW(NT, MT)                                                                           \
  gemm_rows_kernel<EPI, SPLIT, NT, MT><<<g, b, 0, s>>>(x, xs, M, w, N, K, P.rows, P.splits,       \
                                                       P.ks_per, P.mh, out, os, res, rs, part)
#define QD_RW_MT(NT) \
  do { if (P.mt == 1) QD_RW(NT, 1); else QD_RW(NT, 2); } while (0)
  const int nt = rows_inst_nt(P.nt, EPI, SPLIT);
  if constexpr (EPI == EPI_SWIGLU) {
    switch (nt) {
      case 2: QD_RW_MT(2); break;
      case 3: QD_RW_MT(3); break;
      case 4: QD_RW_MT(4); break;
      default: QD_RW_MT(5); break;
    }
  } else if constexpr (SPLIT) {
    switch (nt) {
      case 1: QD_RW_MT(1); break;
      case 2: QD_RW_MT(2); break;
      case 3: QD_RW_MT(3); break;
      case 4: QD_RW_MT(4); break;
      case 6: QD_RW_MT(6); break;
      default: QD_RW_MT(8); break;
    }
  } else {
    switch (nt) {
      case 1: QD_RW_MT(1); break;
      case 2: QD_RW_MT(2); break;
      case 3: QD_RW_MT(3); break;
      default: QD_RW_MT(4); break;
    }
  }
#undef QD_RW_MT
#undef QD_RW
}

int gemm_rows_query(int64_t M, int64_t N, int64_t K, int epi, bool partials_only,
                    int64_t part_floats, int64_t* out) {
  RowsPlan P;
  const int rp = rows_launch_plan(M, N, K, epi, partials_only, part_floats, P);
  if (rp != 1) return rp;
  const bool split = P.splits > 1;
  const int nt = rows_inst_nt(P.nt, split ? EPI_NONE : epi, split);
  const int64_t nblk = (N + P.rows - 1) / P.rows * P.splits;
  const int wt = (!split && epi == EPI_SWIGLU) ? 2 * nt : nt;
  out[0] = P.rows;
  out[1] = nt;
  out[2] = P.mt;
  out[3] = P.mh;
  out[4] = P.splits;
  out[5] = P.ks_per;
  out[6] = P.mh > 1 ? (nblk + 7) / 8 * 8 * P.mh : nblk;             // grid (launch_rows)
  out[7] = (int64_t)rw_nbuf(16 * wt + 128 * P.mt) * (16 * wt + 128 * P.mt) * 128;   // static LDS bytes
  return 1;
}

int64_t gemm_tile_ws_floats(int64_t M, int64_t N, int64_t K, int epi) {
  if (M < GEMM_TILE_MIN_M) return M >= GEMM_SMALL_MIN_M && K % TK == 0 ? quad_small_ws_floats(M, N, K) : 0;
  RowsPlan P;
  const int sp = rows_plan(M, N, K, epi, true, P) ? P.splits : gemm_tile_splits(M, N, K, epi);
  return sp > 1 ? (int64_t)sp * M * N : 0;
}

// Falls with the row count as well as growing with it: from 33 to 64 rows the plan takes fewer splits
// as rows are added, and past that the split count drops where a 128-row block is added (one count
// per number of blocks, so a block's largest need is at its last row count).
int64_t gemm_tile_ws_floats_upto(int64_t B, int64_t T, int64_t N, int64_t K, int epi) {
  int64_t most = 0;
  auto take = [&](int64_t t) {
    const int64_t f = gemm_tile_ws_floats(B * t, N, K, epi);
    if (f > most) most = f;
  };
  for (int64_t t = (GEMM_SMALL_MIN_M + B - 1) / B; t <= T && B * t < GEMM_TILE_MIN_M; ++t) take(t);
  for (int64_t rows = TM;; rows += TM) {
    const int64_t t = rows / B < T ? rows / B : T;
    if (B * t >= GEMM_TILE_MIN_M) take(t);
    if (t == T || gemm_tile_splits(rows, N, K, epi) <= 1) return most;
  }
}

// as gemm_tile_partials, for a decode step's rows: where the all-rows kernel's split count does
// not fit part_floats, the four-wave kernel takes fewer
int gemm_step_partials(const bf16_t* x, int64_t xs, int64_t M, const bf16_t* w, int64_t N,
                       int64_t K, float* part, int64_t part_floats, hipStream_t s) {
  if (M > 128 || gemm_tile_ws_floats(M, N, K, EPI_NONE) <= part_floats)
    return gemm_tile_partials(x, xs, M, w, N, K, part, part_floats, s);
  if (M < GEMM_SMALL_MIN_M || !gemm_tile_ok(M, N, K, EPI_NONE, x, xs, w, part, N, nullptr, 0)) return 0;
  return quad_small_partials(x, xs, M, w, N, K, part, part_floats, s);
}

int gemm_tile_partials(const bf16_t* x, int64_t xs, int64_t M, const bf16_t* w, int64_t N,
                       int64_t K, float* part, int64_t part_floats, hipStream_t s) {
  if (M < GEMM_SMALL_MIN_M || !part ||
      !gemm_tile_ok(M, N, K, EPI_NONE, x, xs, w, part, N, nullptr, 0))
    return 0;
  if (M < GEMM_TILE_MIN_M) return quad_small_partials(x, xs, M, w, N, K, part, part_floats, s);
  RowsPlan P;
  const int rp = rows_stride_ok(M, xs, K) ? rows_launch_plan(M, N, K, EPI_NONE, true, part_floats, P) : -1;
  if (rp == 0) return 0;
  if (rp == 1) {
    launch_rows<EPI_NONE, true>(P, x, xs, (int)M, w, (int)N, (int)K, nullptr, 0, nullptr, 0,
                                part, s);
    return P.splits;
  }
  int splits = gemm_tile_splits(M, N, K, EPI_NONE);
  if (splits <= 1 || part_floats < (int64_t)splits * M * N) return 0;
  const int ksteps = (int)(K / TK);
  const int ks_per = (ksteps + splits - 1) / splits;
  splits = (ksteps + ks_per - 1) / ks_per;              // no empty split
  if (launch_gemm_quad(x, xs, M, w, N, K, nullptr, 0, nullptr, 0, EPI_NONE, splits, ks_per, part, s))
    return splits;
  const int64_t mblocks = (M + TM - 1) / TM, nblocks = tile_nblocks(N, EPI_NONE);
  gemm_tile_kernel<EPI_NONE, true><<<dim3((unsigned)(mblocks * nblocks * splits)), dim3(256), 0, s>>>(
      x, xs, (int)M, w, (int)N, (int)K, (int)mblocks, (int)nblocks, ks_per, nullptr, 0, nullptr, 0,
      nullptr, nullptr, nullptr, part);
  return splits;
}

// K splits of a launch that reduces them itself, and stages per split
static int tile_launch_splits(int64_t M, int64_t N, int64_t K, int epi, int64_t part_floats, int& ks_per) {
  // from 1024 rows on, whole 256-column blocks are not split (the largest tiles fill the chip)
  int splits = M >= 1024 && N % 256 == 0 ? 1 : gemm_tile_splits(M, N, K, epi);
  if (splits > 1 && part_floats < (int64_t)splits * M * N) splits = 1;
  const int ksteps = (int)(K / TK);
  ks_per = (ksteps + splits - 1) / splits;
  return (ksteps + ks_per - 1) / ks_per;                // no empty split
}

int gemm_quad_query(int64_t M, int64_t N, int64_t K, int epi, int64_t part_floats, int64_t* out) {
  const void* a = reinterpret_cast<const void*>(256);
  RowsPlan P;
  if (M < GEMM_SMALL_MIN_M || !gemm_tile_ok(M, N, K, epi, a, K, a, a, N, a, N)) return 0;
  if (M < GEMM_TILE_MIN_M) {
    if (!quad_small_pays(M, N, K, epi, part_floats)) return 0;
    quad_small_query(M, N, K, epi, part_floats, out);
    return 1;
  }
  if (rows_launch_plan(M, N, K, epi, false, part_floats, P) == 1) return 0;
  int ks_per;
  const int splits = tile_launch_splits(M, N, K, epi, part_floats, ks_per);
  quad_query(M, N, K, epi, splits, ks_per, out);
  return 1;
}

// Returns the number of argmax partials per row written (EPI_ARGMAX), else 0.
int64_t launch_gemm_tile(const bf16_t* x, int64_t xs, int64_t M, const bf16_t* w, int64_t N,
                         int64_t K, bf16_t* out, int64_t os, const bf16_t* res, int64_t rs, int epi,
                         float* pval, int32_t* pidx, float* logits, float* part,
                         int64_t part_floats, hipStream_t s) {
  if (epi == EPI_ARGMAX) {
    const int64_t parts = launch_lm_quad(x, xs, M, w, N, K, pval, pidx, logits, s);
    if (parts > 0) return parts;
  }
  auto reduce = [&](int S) {
    const dim3 rg((unsigned)((M * (N / 4) + 255) / 256)), rb(256);
    if (epi == EPI_RES)
      gemm_split_reduce_kernel<EPI_RES><<<rg, rb, 0, s>>>(part, S, M, N, out, os, res, rs);
    else
      gemm_split_reduce_kernel<EPI_NONE><<<rg, rb, 0, s>>>(part, S, M, N, out, os, res, rs);
  };
  if (epi != EPI_ARGMAX && M < GEMM_TILE_MIN_M) {
    const int S = launch_quad_small(x, xs, M, w, N, K, out, os, res, rs, epi, part, part ? part_floats : 0, s);
    if (S > 0) reduce(S);
    if (S >= 0) return 0;
  }
  RowsPlan P;
  if (epi != EPI_ARGMAX && rows_stride_ok(M, xs, K) &&
      rows_launch_plan(M, N, K, epi, false, part ? part_floats : 0, P) == 1) {
    if (P.splits > 1) {
      launch_rows<EPI_NONE, true>(P, x, xs, (int)M, w, (int)N, (int)K, nullptr, 0, nullptr, 0,
                                  part, s);
      reduce(P.splits);
      return 0;
    }
    if (epi == EPI_RES)
      launch_rows<EPI_RES, false>(P, x, xs, (int)M, w, (int)N, (int)K, out, os, res, rs, part, s);
    else if (epi == EPI_SWIGLU)
      launch_rows<EPI_SWIGLU, false>(P, x, xs, (int)M, w, (int)N, (int)K, out, os, res, rs, part, s);
    else
      launch_rows<EPI_NONE, false>(P, x, xs, (int)M, w, (int)N, (int)K, out, os, res, rs, part, s);
    return 0;
  }
  const int64_t mblocks = (M + TM - 1) / TM, nblocks = tile_nblocks(N, epi);
  int ks_per;
  const int splits = tile_launch_splits(M, N, K, epi, part ? part_floats : 0, ks_per);
  // the four-wave kernel; the 128 x 128 tiles below where its 32-bit offsets do not reach, and
  // for the LM head's 65..128 rows
  const bool quad = epi != EPI_ARGMAX &&
                    launch_gemm_quad(x, xs, M, w, N, K, out, os, res, rs, epi, splits, ks_per, part, s);
  const dim3 grid((unsigned)(mblocks * nblocks * splits)), block(256);
  const int Mi = (int)M, Ni = (int)N, Ki = (int)K, mbi = (int)mblocks, nbi = (int)nblocks;
#define QD_TILE(E, SP)                                                                           \
  do {                                                                                           \
    if (!quad)                                                                                   \
      gemm_tile_kernel<E, SP><<<grid, block, 0, s>>>(x, xs, Mi, w, Ni, Ki, mbi, nbi, ks_per, out, \
                                                     os, res, rs, pval, pidx, logits, part);     \
  } while (0)
  if (splits > 1) {
    if (epi == EPI_RES) QD_TILE(EPI_RES, true);
    else QD_TILE(EPI_NONE, true);
    reduce(splits);
    return 0;
  }
  switch (epi) {
    case EPI_RES: QD_TILE(EPI_RES, false); break;
    case EPI_SWIGLU: QD_TILE(EPI_SWIGLU, false); break;
    case EPI_ARGMAX: QD_TILE(EPI_ARGMAX, false); return nblocks;
    default: QD_TILE(EPI_NONE, false); break;
  }
#undef QD_TILE
  return 0;
}
