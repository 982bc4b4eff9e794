// Four-wave MFMA GEMM:  out[m, n] = epi( sum_k X[m, k] * W[n, k] )  for 257 and more activation rows
// (prefill chunks) and for 33 to 64 (mid-sized batches, small trees), the split partials of decode steps
// of 65 to 128 rows, and the LM head over 33 to 64 and 129 and more  (the reference's cuBLAS prefill,
// engine.py:550-592, and its tensor-core GEMMs, gemv.py:61-116).
//
// A workgroup of 4 waves, one per SIMD, owns 32 MT activation rows x 32 NT weight rows (SwiGLU: 16 NT gate
// and the 16 NT up rows of the same outputs); wave (wm, wn) the quarter of 16 MT x 16 NT, MT x NT
// MFMA tiles of accumulators in the AGPRs.  The tile shapes are chosen per launch (quad_plan
// below): what decides at a few hundred to a few thousand rows is how evenly the tiles fill
// whole rounds of the CUs.
//  * K advances in stages of 64 (whole 128-byte lines of every row) that go from global memory
//    straight into LDS (global_load_lds_dwordx4: no staging registers), NBUF stage buffers deep;
//    one barrier per stage.
//  * A stage is contracted as two halves of K = 32.  While one half's MFMAs issue, the next
//    half's fragments are read into a second register set and (in a stage's second half) the
//    loads of the stage NBUF ahead go into the buffer that the barrier has just freed, one load
//    and one fragment read between every MT NT / (MT + NT) MFMAs (issuing the loads in bunches of
//    2, 4 or 16 instead: 2 / 3 / 6 % slower at 16384 rows).
//  * One wave per SIMD with a square-ish quarter reads (MT + NT) fragments for MT NT MFMAs: LDS
//    traffic per flop is 2/3 (8 x 8 tiles) to 1/2 of the 8-wave kernels this one replaced, which
//    at 128 x 128 tiles were bound by it.  256 AGPRs hold the accumulators, so the MFMAs are
//    written as asm with AGPR operands: left to the compiler, part of them lands in VGPRs and is
//    copied around the loop (100 moves per 128 MFMAs).
//  * With two stage buffers (the largest tiles) a load has half a stage to a stage to land,
//    enough from L2 but not from HBM: two waves touch the lines of stage s + 4 with one 4-byte
//    load each (into spare LDS), a share of the lines per workgroup such that the workgroups that
//    one XCD runs at a time (4 row blocks x 8 weight blocks) cover theirs once.  gate/up at 16384
//    rows 1356 -> 1243 us, 512 rows (128 x 160 pairs) 69 -> 58 us; with three and more buffers it
//    gains nothing.
//  * Weight rows enter the MFMA tiles pairwise interleaved (rd): the lane then holds eight
//    consecutive output columns of a tile pair, one 16-byte store per row instead of two 8-byte
//    stores in different lines.
// The accumulation of an output runs through its K range in order, 32 at a time: the bits are the
// same for every tile shape.
// Measured (MI355X, weights from HBM), against the 8-wave 128 x 128 and 256 x 256 kernels: see
// quad_plan.
#include "qd_launch.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

__device__ __forceinline__ bf16x8_t as_bf8(uint4 v) { return __builtin_bit_cast(bf16x8_t, v); }

constexpr int TK = 64;                         // K per stage: 128 bytes of every row

#ifndef QD_QUAD_GROUP_M
#define QD_QUAD_GROUP_M 4   // M blocks per group of the tile order
#endif

// WAIT: the 8 wait states that a VALU read of the result needs, in the same asm.  The compiler does
// not see the latency of an MFMA in asm and may copy an accumulator right behind one (it does where
// the main loop's accumulators become the tail's), so the last MFMA of a stage carries them, and of
// each half in the tail; the others are followed by an MFMA and the rest of that wait.
template <bool WAIT>
__device__ __forceinline__ void mfma_acc(f32x4_t& acc, uint4 a, uint4 b) {
  if constexpr (WAIT)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\ts_nop 7"
                 : "+a"(acc) : "v"(as_bf8(a)), "v"(as_bf8(b)));
  else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(as_bf8(a)), "v"(as_bf8(b)));
}

// one dword per lane into LDS (256 bytes at lds): brings the lanes' lines into this XCD's L2
__device__ __forceinline__ void touch_line(const void* base, uint32_t voff, uint32_t lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(base), "{m0}"(lds) : "memory");
}

__host__ __device__ constexpr int quad_lds_u4(int mt, int nt, int nbuf) {
  return nbuf * 32 * (mt + nt) * 8 + (nbuf == 2 ? 16 : 0);   // stages, and the touched dwords
}

// output columns of a workgroup's tile
__host__ __device__ constexpr int quad_outs(int nt, bool sw) { return sw ? 16 * nt : 32 * nt; }

template <int EPI, bool SPLIT, int MT, int NT, int NBUF>
__global__ __launch_bounds__(256, 1) void gemm_quad_kernel(
    const bf16_t* __restrict__ X, int64_t x_stride, int M, const bf16_t* __restrict__ W, int N,
    int K, int mblocks, int nblocks, int outs, int ks_per, bf16_t* out, int64_t out_stride,
    const bf16_t* res, int64_t res_stride, int wide, float* part, float* pval, int32_t* pidx,
    float* logits) {
  constexpr bool SW = EPI == EPI_SWIGLU && !SPLIT;
  constexpr int BM = 32 * MT, BN = 32 * NT, ROWS = BM + BN;   // LDS rows: weights, activations
  constexpr int PER = MT + NT;                 // 1 KiB load blocks per wave and stage
  constexpr int GT = SW ? NT / 2 : NT;         // tiles of one run of weight rows (gate, up)
  constexpr int PAIRED = 32 * (GT / 2);        // its interleaved rows; an odd last tile follows
  constexpr int TOUCH = NBUF == 2 ? 2 : 0;     // stages the line touches run ahead of the loads
  static_assert(!SW || NT % 2 == 0, "gate tiles, then up tiles");
  static_assert(MT * NT <= 64, "accumulators in the AGPRs");
  // [stage buffer][row * 8 + position]: a row's 128 bytes hold its eight 16-byte K units, unit u
  // at position u ^ key(row), the keys such that the 8 lanes of a fragment read (one unit of 8
  // rows) cover all banks
  __shared__ uint4 sm[quad_lds_u4(MT, NT, NBUF)];
  const int total = gridDim.x, h = blockIdx.x;
  const int xq = total >> 3, xr = total & 7, xcd = h & 7, slot = h >> 3;
  const int L = xcd < xr ? xcd * (xq + 1) + slot : xr * (xq + 1) + (xcd - xr) * xq + slot;
  const int tiles = mblocks * nblocks;
  const int split = L / tiles, Lt = L - split * tiles;
  const int group = Lt / (QD_QUAD_GROUP_M * nblocks);
  const int first = group * QD_QUAD_GROUP_M;
  const int gm = min(QD_QUAD_GROUP_M, mblocks - first);
  const int rr = Lt - first * nblocks;
  const int mb = first + rr % gm, nb = rr / gm;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, q = lane >> 4;
  const int wn = wave & 1, wm = wave >> 1;
  const int64_t m0 = (int64_t)mb * BM;
  const int n0 = nb * outs;                    // output columns per workgroup: at most quad_outs()
  const int nrows = min(outs, N - n0);
  const int mrows = (int)(M - m0 < BM ? M - m0 : BM);
  const int kbeg = split * ks_per;
  const int stages = min(K / TK, kbeg + ks_per) - kbeg;
  // weight row (relative to n0) of LDS row r < BN; rows past the operand reload its last row
  auto wrow = [&](int r) -> int64_t {
    if constexpr (SW) {
      const int o = 16 * GT * (r / (32 * GT)) + r % (16 * GT);
      return min(o, nrows - 1) + (int64_t)(((r / (16 * GT)) & 1) ? N : 0);
    } else {
      return min(r, nrows - 1);
    }
  };
  auto wkey = [&](int r) {
    return r % (16 * GT) < PAIRED ? (r & 3) | (((r >> 3) & 1) << 2) : r & 7;
  };
  // loads: block j (< NT weights, then activations) of wave w is LDS rows 8 (w + 4 j) .. + 7;
  // lane l of a block writes position l % 8 of row l / 8
  uint32_t off[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int r = 8 * (wave + 4 * j) + (lane >> 3);
    if (j < NT) {
      off[j] = (uint32_t)(wrow(r) * K * 2 + ((lane & 7) ^ wkey(r)) * 16);
    } else {
      off[j] = (uint32_t)((int64_t)min(r - BN, mrows - 1) * x_stride * 2 + ((lane & 7) ^ (r & 7)) * 16);
    }
  }
  const uint32_t lds = __builtin_amdgcn_readfirstlane(lds_u32(&sm[0]));
  const uint32_t lbase = lds + wave * 1024;
  const char* wbase = reinterpret_cast<const char*>(W + (int64_t)n0 * K + (int64_t)kbeg * TK);
  const char* xbase = reinterpret_cast<const char*>(X + m0 * x_stride + (int64_t)kbeg * TK);
  auto load = [&](int st, int b, int j) {
    dma16((j < NT ? wbase : xbase) + (size_t)st * (TK * 2), off[j],
          lbase + (uint32_t)b * (ROWS * 128) + 4096u * j);
  };
  // line touches: wave 0 this workgroup's quarter of the weight rows, wave 1 its eighth of the
  // activation rows
  constexpr int TW = BN / 4 < 64 ? BN / 4 : 64, TX = BM / 8;
  const bool toucher = TOUCH > 0 && wave < 2;
  uint32_t toff = 0;
  if (TOUCH > 0)
    toff = wave == 0 ? (uint32_t)(wrow(((rr % gm) & 3) * TW + min(lane, TW - 1)) * K * 2)
                     : (uint32_t)((int64_t)min((nb & 7) * TX + min(lane, TX - 1), mrows - 1) * x_stride * 2);
  auto touch = [&](int st) {
    st = st < stages ? st : stages - 1;
    touch_line((wave == 0 ? wbase : xbase) + (size_t)st * (TK * 2), toff, lds + NBUF * ROWS * 128);
  };
  f32x4_t acc[NT][MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // After a loop and at the end: the accumulators stay where they are until the last MFMA (with its
  // wait) is behind, and what the compiler has moved at a loop's end is two wait states old before
  // an MFMA reads it.
  auto settle = [&]() {
    asm volatile("s_nop 1");
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) asm volatile("" : "+a"(acc[nt][mt]));
  };
  // fragments of one K half: NT weight tiles, MT activation tiles, one 16-byte unit per lane each
  struct Frag {
    uint4 v[PER];
  };
  const int kw = c & 7;                        // key of the lane's rows, the same in every tile
  const int u0 = q ^ kw, u1 = (4 + q) ^ kw;
  const int pp = (16 * NT * wn + 8 * (c >> 2) + (c & 3)) * 8;   // paired weight tiles
  const int ps = (16 * NT * wn + c) * 8;                        // an odd last weight tile
  const int px = (BN + 16 * MT * wm + c) * 8;                   // activation tiles
  auto rd = [&](Frag& f, int b, int hf, int t) {
    const int u = (hf ? u1 : u0) + b * (ROWS * 8);
    if (t < NT) {
      const int g = t / GT, i = t % GT;        // run (gate, up) and tile in it
      if (32 * (i / 2) < PAIRED) f.v[t] = sm[pp + (16 * GT * g + 32 * (i / 2) + 4 * (i & 1)) * 8 + u];
      else f.v[t] = sm[ps + (16 * GT * g + 16 * i) * 8 + u];
    } else {
      f.v[t] = sm[px + 128 * (t - NT) + u];
    }
  };
  // contract the half in cur; RD: read half (rb, hf) into nxt; LD: load stage st into buffer lb;
  // WT: the last MFMA carries its wait
#define QD_HALF(WT, LD, RD, cur, nxt, rb, hf, st, lb)                                          \
  _Pragma("unroll") for (int g_ = 0; g_ < PER; ++g_) {                                         \
    if (LD) load(st, lb, g_);                                                                  \
    if (RD) rd(nxt, rb, hf, g_);                                                               \
    __builtin_amdgcn_sched_barrier(0);                                                         \
    _Pragma("unroll") for (int e_ = g_ * MT * NT / PER; e_ < (g_ + 1) * MT * NT / PER; ++e_) { \
      if (e_ + 1 < MT * NT) mfma_acc<false>(acc[e_ % NT][e_ / NT], cur.v[e_ % NT], cur.v[NT + e_ / NT]); \
      else mfma_acc<WT>(acc[e_ % NT][e_ / NT], cur.v[e_ % NT], cur.v[NT + e_ / NT]);           \
    }                                                                                          \
    __builtin_amdgcn_sched_barrier(0);                                                         \
  }
#pragma unroll
  for (int i = 0; i < NBUF; ++i)
    if (i < stages) {
#pragma unroll
      for (int j = 0; j < PER; ++j) load(i, i, j);
      if (toucher) touch(NBUF + i);
    }
  wait_stages<PER, NBUF - 1>(stages - 1);      // stage 0 landed
  lds_barrier();
  Frag f0, f1;
#pragma unroll
  for (int t = 0; t < PER; ++t) rd(f0, 0, 0, t);
  // Stage s sits in buffer s % NBUF.  After its first half every fragment of it is in registers;
  // once this wave's loads of stage s + 1 have landed (the loads of the NBUF - 2 stages after it,
  // and the touches issued since, may be outstanding) the waves meet: stage s + 1 is then
  // visible and stage s's buffer free.
  int b = 0, s = 0;
  for (; s + NBUF < stages; ++s) {
    QD_HALF(false, false, true, f0, f1, b, 1, 0, 0);
    if (toucher) wait_vm<PER * (NBUF - 2) + NBUF - 1>();
    else wait_vm<PER * (NBUF - 2)>();
    lds_barrier();
    const int bn = b + 1 < NBUF ? b + 1 : 0;
    QD_HALF(true, true, true, f1, f0, bn, 0, s + NBUF, b);
    if (toucher) touch(s + NBUF + TOUCH);
    b = bn;
  }
  settle();
  for (; s + 1 < stages; ++s) {                // the last stages: nothing left to load
    QD_HALF(true, false, true, f0, f1, b, 1, 0, 0);
    wait_stages<PER, NBUF - 2>(stages - 2 - s);
    lds_barrier();
    const int bn = b + 1 < NBUF ? b + 1 : 0;
    QD_HALF(true, false, true, f1, f0, bn, 0, 0, 0);
    settle();
    b = bn;
  }
  QD_HALF(true, false, true, f0, f1, b, 1, 0, 0);
  QD_HALF(true, false, false, f1, f0, b, 0, 0, 0);
#undef QD_HALF
  wait_vm<0>();                                // no load outlives the workgroup
  settle();

  // epilogue: lane (c, q) of acc[nt][mt] holds four consecutive output columns, of a tile pair
  // eight: columns 32 p + 8 q .. + 7 of the run (an odd last tile: 16 nt + 4 q .. + 3), for
  // activation row 16 MT wm + 16 mt + c of the block
  if constexpr (EPI == EPI_ARGMAX) {
    // LM head: per activation row the maximum bf16 logit of the block's vocabulary rows and its
    // lowest index (the lane's columns ascend with nt and r; lanes and waves hold interleaved
    // column ranges, so ties compare indices) -> pval / pidx[m][nb] for argmax_reduce_kernel
    static_assert(NT % 2 == 0, "paired tiles");
    float* av = reinterpret_cast<float*>(&sm[0]);                // [2][BM], then indices
    int32_t* ai = reinterpret_cast<int32_t*>(av + 2 * BM);
    lds_barrier();                             // every wave is done with the staged rows
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int row = 16 * MT * wm + 16 * mt + c;
      float bv = -INFINITY;
      int32_t bi = 0x7FFFFFFF;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int64_t n = (int64_t)n0 + 16 * NT * wn + 32 * (nt / 2) + 8 * q + 4 * (nt & 1);
        if (row < mrows && logits && n < N)
          *reinterpret_cast<f32x4_t*>(logits + (m0 + row) * (int64_t)N + n) = acc[nt][mt];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = rbf(acc[nt][mt][r]);
          if (n + r < N && v > bv) { bv = v; bi = (int32_t)(n + r); }
        }
      }
#pragma unroll
      for (int sh = 0; sh < 2; ++sh) {
        const float ov = sh ? lane_xor32(bv) : lane_xor16(bv);
        const int32_t oi = sh ? __builtin_bit_cast(int32_t, lane_xor32(__builtin_bit_cast(float, bi)))
                              : __builtin_bit_cast(int32_t, lane_xor16(__builtin_bit_cast(float, bi)));
        if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
      }
      if (q == 0) {
        av[wn * BM + row] = bv;
        ai[wn * BM + row] = bi;
      }
    }
    lds_barrier();
    if (tid < mrows) {
      float bv = av[tid];
      int32_t bi = ai[tid];
      const float ov = av[BM + tid];
      const int32_t oi = ai[BM + tid];
      if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
      pval[(m0 + tid) * (int64_t)nblocks + nb] = bv;
      pidx[(m0 + tid) * (int64_t)nblocks + nb] = bi;
    }
    return;
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int row = 16 * MT * wm + 16 * mt + c;
    if (row >= mrows) continue;
    const int64_t m = m0 + row;
#pragma unroll
    for (int i = 0; i < GT; ++i) {
      const bool paired = 32 * (i / 2) < PAIRED;
      if (paired && (i & 1)) continue;         // with its even tile
      const int u = 16 * GT * wn + (paired ? 16 * i + 8 * q : 16 * i + 4 * q);
      if (u >= nrows) continue;                // N and outs are multiples of 8 columns
      const int64_t n = (int64_t)n0 + u;
      {
        const f32x4_t lo = acc[i][mt], hi = acc[paired ? i + 1 : i][mt];
        if constexpr (SPLIT) {
          float* o = part + ((int64_t)split * M + m) * N + n;
          *reinterpret_cast<f32x4_t*>(o) = lo;
          if (paired) *reinterpret_cast<f32x4_t*>(o + 4) = hi;
        } else {
          uint4 y;
          if constexpr (SW) {
            const f32x4_t ulo = acc[GT + i][mt], uhi = acc[GT + (paired ? i + 1 : i)][mt];
            float v[8];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              v[r] = silu_rbf(rbf(lo[r])) * rbf(ulo[r]);
              v[4 + r] = paired ? silu_rbf(rbf(hi[r])) * rbf(uhi[r]) : 0.f;
            }
            y = make_uint4(pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7]));
          } else if constexpr (EPI == EPI_RES) {
            const bf16_t* rp = res + m * res_stride + n;
            uint4 rv;
            if (paired && (wide & 2)) {
              rv = *reinterpret_cast<const uint4*>(rp);
            } else {
              const uint2 a = *reinterpret_cast<const uint2*>(rp);
              const uint2 z = paired ? *reinterpret_cast<const uint2*>(rp + 4) : make_uint2(0, 0);
              rv = make_uint4(a.x, a.y, z.x, z.y);
            }
            y = make_uint4(pack2(bflo(rv.x) + rbf(lo[0]), bfhi(rv.x) + rbf(lo[1])),
                           pack2(bflo(rv.y) + rbf(lo[2]), bfhi(rv.y) + rbf(lo[3])),
                           pack2(bflo(rv.z) + rbf(hi[0]), bfhi(rv.z) + rbf(hi[1])),
                           pack2(bflo(rv.w) + rbf(hi[2]), bfhi(rv.w) + rbf(hi[3])));
          } else {
            y = make_uint4(pack2(lo[0], lo[1]), pack2(lo[2], lo[3]), pack2(hi[0], hi[1]), pack2(hi[2], hi[3]));
          }
          bf16_t* o = out + m * out_stride + n;
          if (paired && (wide & 1)) {
            *reinterpret_cast<uint4*>(o) = y;
          } else {
            *reinterpret_cast<uint2*>(o) = make_uint2(y.x, y.y);
            if (paired) *reinterpret_cast<uint2*>(o + 4) = make_uint2(y.z, y.w);
          }
        }
      }
    }
  }
}

// Tile shapes {MT, NT, stage buffers} and the time of one round of workgroups over the CUs,
// a + b x stages (SwiGLU: + QUAD_SWIGLU MT NT) in us: least squares over 14 row counts from 300 to
// 16384 x the four Qwen3-4B projections x every shape on MI355X, weights from HBM (single launches
// scatter by about 8 %).  The plan takes the shape whose rounds cost least: over 78 launches of other
// sizes the fastest shape in 61, 0.4 % off it on average, 5.8 % at most.  Times (us) with the
// kernels before (8 waves, 128 x 128 tiles to 1023 rows, 256 x 256 from 1024) -> now, o and down
// at 512 rows with their split reduce:
//   rows    qkv (6144 x 2560)  o (2560 x 4096)  gate/up (19456 x 2560)  down (2560 x 9728)
//   512        30.4 ->  24.8     27.9 ->  24.1      87.4 ->   58.2        43.8 ->  40.2
//   1024       64.9 ->  35.7     93.9 ->  32.2     135.1 ->  115.4       206.8 ->  70.7
//   3000      123.0 ->  88.9     96.6 ->  56.6     266.8 ->  261.4       206.2 -> 119.2
//   16384     418.3 -> 393.4    313.2 -> 293.7    1342.0 -> 1265.2       716.4 -> 657.9
// (the whole-round rates at 16384 rows are 1.17 to 1.31 PFLOP/s, the matrix cores 58 to 70 % busy at
// 32768.)  What is left is the line stream, a fifth of it past the L2, and a round's start and end,
// when the first lines come from HBM and the outputs are written with no MFMAs beside them (the
// fitted a: 4 to 13 us).
struct QuadShape {
  int mt, nt, nbuf;
  float a, b;
};
constexpr QuadShape QUAD[] = {
    {4, 3, 5, 3.6f, 0.409f},  {4, 4, 5, 5.8f, 0.479f},   {4, 5, 4, 5.5f, 0.569f},
    {4, 6, 4, 7.1f, 0.625f},  {4, 8, 3, 7.3f, 0.800f},   {4, 10, 2, 10.2f, 0.973f},
    {6, 5, 3, 6.6f, 0.700f},  {6, 6, 3, 9.2f, 0.790f},   {6, 8, 2, 10.2f, 0.993f},
    {8, 4, 3, 7.7f, 0.755f},  {8, 5, 3, 7.6f, 0.926f},   {8, 6, 2, 9.5f, 1.026f},
    {8, 8, 2, 13.2f, 1.232f},
};
constexpr double QUAD_SWIGLU = 0.06;
constexpr int QUADS = sizeof(QUAD) / sizeof(QUAD[0]);

constexpr bool quad_fits() {
  for (int i = 0; i < QUADS; ++i)
    if (quad_lds_u4(QUAD[i].mt, QUAD[i].nt, QUAD[i].nbuf) * 16 > 160 * 1024) return false;
  return true;
}
static_assert(quad_fits(), "the CU's LDS");


// Split launches take one of the first two: their splits times 128 x 128 tiles are at most the CUs
// (gemm_tile_splits), one round of {4, 4}.
constexpr int QUAD_SPLIT = 2;

// us of a launch in shape q
double quad_cost(const QuadShape& q, int64_t M, int64_t N, bool sw, int64_t splits, int64_t stages) {
  const int64_t bm = 32 * q.mt, bn = quad_outs(q.nt, sw);
  const int64_t wgs = (M + bm - 1) / bm * ((N + bn - 1) / bn) * splits;
  return (double)((wgs + plan_cus() - 1) / plan_cus()) *
         (q.a + (sw ? QUAD_SWIGLU * q.mt * q.nt : 0.0) + (double)q.b * stages);
}

int quad_plan(int64_t M, int64_t N, bool sw, int64_t splits, int64_t stages) {
  int best = -1;
  double best_t = 0;
  for (int i = 0; i < (splits > 1 ? QUAD_SPLIT : QUADS); ++i) {
    if (sw && QUAD[i].nt % 2) continue;
    const double t = quad_cost(QUAD[i], M, N, sw, splits, stages);
    if (best < 0 || t < best_t) {
      best = i;
      best_t = t;
    }
  }
  return best;
}

template <int I, int EPI, bool SPLIT>
void quad_go(const bf16_t* x, int64_t xs, int64_t M, const bf16_t* w, int64_t N, int64_t K, bf16_t* out,
             int64_t os, const bf16_t* res, int64_t rs, int splits, int ks_per, int wide,
             float* part, hipStream_t s) {
  constexpr QuadShape q = QUAD[I];
  constexpr int BM = 32 * q.mt, BN = quad_outs(q.nt, EPI == EPI_SWIGLU);
  const int64_t mbl = (M + BM - 1) / BM, nbl = (N + BN - 1) / BN;
  gemm_quad_kernel<EPI, SPLIT, q.mt, q.nt, q.nbuf><<<dim3((unsigned)(mbl * nbl * splits)), dim3(256), 0, s>>>(
      x, xs, (int)M, w, (int)N, (int)K, (int)mbl, (int)nbl, BN, ks_per, out, os, res, rs, wide, part,
      nullptr, nullptr, nullptr);
}

template <int EPI, bool SPLIT, int I = 0>
void quad_pick(int i, const bf16_t* x, int64_t xs, int64_t M, const bf16_t* w, int64_t N, int64_t K,
               bf16_t* out, int64_t os, const bf16_t* res, int64_t rs, int splits, int ks_per,
               int wide, float* part, hipStream_t s) {
  if constexpr (I < (SPLIT ? QUAD_SPLIT : QUADS)) {
    if constexpr (EPI != EPI_SWIGLU || QUAD[I].nt % 2 == 0) {
      if (i == I)
        return quad_go<I, EPI, SPLIT>(x, xs, M, w, N, K, out, os, res, rs, splits, ks_per, wide, part, s);
    }
    quad_pick<EPI, SPLIT, I + 1>(i, x, xs, M, w, N, K, out, os, res, rs, splits, ks_per, wide, part, s);
  }
}

// row offsets inside a block, and to the up rows, are 32-bit bytes
bool quad_offsets_ok(int64_t xs, int64_t N, int64_t K, int epi) {
  return 256 * xs * 2 < (1ll << 32) && ((epi == EPI_SWIGLU ? N : 0) + 320) * K * 2 < (1ll << 32) &&
         N < (1ll << 30) && K < (1ll << 30);
}

bool al16(const void* p, int64_t stride) { return reinterpret_cast<uintptr_t>(p) % 16 == 0 && stride % 8 == 0; }

}  // namespace

// The operands satisfy gemm_tile_ok.  splits > 1 (store / residual products only): fp32 partials
// part[splits][M][N] of K ranges of ks_per stages, nothing else written.  Returns false, with
// nothing launched, where the 32-bit offsets do not reach.
bool launch_gemm_quad(const bf16_t* x, int64_t xs, int64_t M, const bf16_t* w, int64_t N, int64_t K,
                      bf16_t* out, int64_t os, const bf16_t* res, int64_t rs, int epi, int splits,
                      int ks_per, float* part, hipStream_t s) {
  if (M >= (1ll << 31) || !quad_offsets_ok(xs, N, K, epi)) return false;
  const int i = quad_plan(M, N, epi == EPI_SWIGLU, splits, ks_per);
  const int wide = (al16(out, os) ? 1 : 0) | (res && al16(res, rs) ? 2 : 0);
#define QD_QUAD(E, SP) quad_pick<E, SP>(i, x, xs, M, w, N, K, out, os, res, rs, splits, ks_per, wide, part, s)
  if (splits > 1) QD_QUAD(EPI_NONE, true);
  else if (epi == EPI_RES) QD_QUAD(EPI_RES, false);
  else if (epi == EPI_SWIGLU) QD_QUAD(EPI_SWIGLU, false);
  else QD_QUAD(EPI_NONE, false);
#undef QD_QUAD
  return true;
}

// ------------------------------------------------------------------ 33..64 rows
// A batched decode step or a small tree: every weight byte is used 64 times at most and read once,
// so the weight stream is the cost and the workgroups (one row block of 64) must take equal shares
// of it in one round.  (Also the split partials of a decode step of 65..128 rows, two row blocks:
// its room for partials holds fewer splits than the all-rows kernel's plan there takes.)  Shapes
// {2, NT}; outs <= quad_outs(NT) columns per workgroup and S K splits
// (fp32 partials, for the store / residual products), the pair that costs least:
//   2.5 us + (0.08 + 0.0027 weight rows + 0.0018 staged weight rows) us per stage
//   + 8 S M N bytes of partials written and read back at 4 TB/s,
// fitted on MI355X to shapes {2, 2} .. {2, 6} and 1 to 8 splits at 33, 48 and 64 rows.  At 48 rows
// (weights from HBM, partials not reduced): qkv 20.8 -> 9.2 us, o 18.4 -> 6.3, gate/up 48.7 ->
// 28.3, down 36.3 -> 11.8 against the 16-row weight tiles of gemm_lds_kernel, which read every
// weight twice above 32 rows (reading the weights alone: 4.8, 3.2, 15.3, 7.7 us).
struct SmallPlan {
  int nt = 0, outs = 0, splits = 1, ks_per = 0;
};
constexpr int SMALL_SPLITS = 8;

static SmallPlan quad_small_plan(int64_t M, int64_t N, int64_t K, bool sw, int64_t max_splits) {
  SmallPlan best;
  double best_t = 0;
  const int64_t stages = K / TK, mbl = (M + 63) / 64;
  if (max_splits > SMALL_SPLITS) max_splits = SMALL_SPLITS;
  if (sw || max_splits < 1) max_splits = 1;
  for (int64_t S0 = 1; S0 <= max_splits && (S0 == 1 || stages / S0 >= 4); ++S0) {
    const int64_t ks_per = (stages + S0 - 1) / S0, S = (stages + ks_per - 1) / ks_per;
    for (int nt = 2; nt <= 6; ++nt) {
      if (nt == 5 || (sw && nt % 2)) continue;
      const int64_t most = quad_outs(nt, sw);
      const int64_t blocks = plan_cus() / (S * mbl) > 0 ? plan_cus() / (S * mbl) : 1;   // one round
      int64_t outs = ((N + blocks - 1) / blocks + 7) / 8 * 8;
      if (outs > most) outs = most;
      const int64_t wgs = (N + outs - 1) / outs * S * mbl;
      const double rows = (double)outs * (sw ? 2 : 1);
      const double t = (double)((wgs + plan_cus() - 1) / plan_cus()) *
                           (2.5 + (0.08 + 0.0027 * rows + 0.0018 * 32 * nt) * (double)ks_per) +
                       (S > 1 ? 8.0 * S * M * N / 4e6 : 0.0);
      if (best.nt == 0 || t < best_t) {
        best_t = t;
        best.nt = nt;
        best.outs = (int)outs;
        best.splits = (int)S;
        best.ks_per = (int)ks_per;
      }
    }
  }
  return best;
}

constexpr int quad_small_nbuf(int nt) { return nt == 2 || nt == 6 ? 4 : 3; }

template <int EPI, bool SPLIT>
static void quad_small_go(const SmallPlan& P, const bf16_t* x, int64_t xs, int64_t M, const bf16_t* w,
                          int64_t N, int64_t K, bf16_t* out, int64_t os, const bf16_t* res,
                          int64_t rs, int wide, float* part, hipStream_t s) {
  const int64_t mbl = (M + 63) / 64, nbl = (N + P.outs - 1) / P.outs;
#define QD_SMALL(NT)                                                                            \
  gemm_quad_kernel<EPI, SPLIT, 2, NT, quad_small_nbuf(NT)><<<dim3((unsigned)(mbl * nbl * P.splits)), dim3(256), \
                                                             0, s>>>(                           \
      x, xs, (int)M, w, (int)N, (int)K, (int)mbl, (int)nbl, P.outs, P.ks_per, out, os, res, rs, wide, part, \
      nullptr, nullptr, nullptr)
  if (P.nt == 2) QD_SMALL(2);
  else if (P.nt == 4) QD_SMALL(4);
  else if (P.nt == 6) QD_SMALL(6);
  else if constexpr (EPI != EPI_SWIGLU) QD_SMALL(3);
#undef QD_SMALL
}

// Whether a whole product of 33..64 rows is faster here than on gemm_lds_kernel (K a multiple of 512),
// whose workgroups of 16 columns split K over their waves: up to 2048 columns they are one round of the
// CUs, and its time hardly grows with K, while a workgroup here walks its K range stage by stage.  Past
// 2048 columns always.  Up to there the K splits win from K = 2048 on (to 2560: up to 1024 columns); SwiGLU, or
// a product without room for partials, has none.  33 rows, weights from HBM (us, there -> here):
//   N x K                 store, split       store, no room     SwiGLU (2N weight rows)
//   512 x 512             3.4 -> 5.7         3.4 -> 4.2          4.5 ->  4.8
//   2048 x 1024           5.1 -> 6.5         5.1 -> 6.2          7.5 ->  7.0
//   1024 x 2560           7.4 -> 6.9         7.4 -> 10.9        10.0 -> 12.0
//   2048 x 2560           8.1 -> 8.0 (64 rows 8.6 -> 8.9)  8.1 -> 11.2   11.7 -> 12.4
//   1024 x 8192          15.1 -> 9.7        15.1 -> 27.2        21.8 -> 29.6
//   3072 x 1024           8.2 -> 7.1         8.2 ->  6.3        11.6 ->  7.3
bool quad_small_pays(int64_t M, int64_t N, int64_t K, int epi, int64_t part_floats) {
  if (K % 512 || N > 2048) return true;
  if (epi == EPI_SWIGLU) return K < 1536 && N > K;
  return part_floats >= 2 * M * N && K > 1536 && (K > 2560 || N <= 1024);
}

// The operands satisfy gemm_tile_ok, 33 <= M <= 64 (quad_small_partials: 128).  quad_small_partials: fp32 partials
// part[S][M][N], S returned (0, nothing launched: no split fits part_floats or pays).
// launch_quad_small: the whole product; with splits its partials go to part, their count is
// returned and the caller reduces them, else 0 is returned and out is written; -1, with nothing
// launched, where the 32-bit offsets do not reach.
int quad_small_partials(const bf16_t* x, int64_t xs, int64_t M, const bf16_t* w, int64_t N, int64_t K,
                        float* part, int64_t part_floats, hipStream_t s) {
  if (!quad_offsets_ok(xs, N, K, EPI_NONE)) return 0;
  const SmallPlan P = quad_small_plan(M, N, K, false, part ? part_floats / (M * N) : 1);
  if (P.splits <= 1) return 0;
  quad_small_go<EPI_NONE, true>(P, x, xs, M, w, N, K, nullptr, 0, nullptr, 0, 0, part, s);
  return P.splits;
}

int launch_quad_small(const bf16_t* x, int64_t xs, int64_t M, const bf16_t* w, int64_t N, int64_t K,
                      bf16_t* out, int64_t os, const bf16_t* res, int64_t rs, int epi, float* part,
                      int64_t part_floats, hipStream_t s) {
  if (!quad_offsets_ok(xs, N, K, epi)) return -1;
  const SmallPlan P = quad_small_plan(M, N, K, epi == EPI_SWIGLU, part ? part_floats / (M * N) : 1);
  const int wide = (al16(out, os) ? 1 : 0) | (res && al16(res, rs) ? 2 : 0);
  if (P.splits > 1) {
    quad_small_go<EPI_NONE, true>(P, x, xs, M, w, N, K, nullptr, 0, nullptr, 0, 0, part, s);
    return P.splits;
  }
  if (epi == EPI_RES) quad_small_go<EPI_RES, false>(P, x, xs, M, w, N, K, out, os, res, rs, wide, part, s);
  else if (epi == EPI_SWIGLU) quad_small_go<EPI_SWIGLU, false>(P, x, xs, M, w, N, K, out, os, res, rs, wide, part, s);
  else quad_small_go<EPI_NONE, false>(P, x, xs, M, w, N, K, out, os, res, rs, wide, part, s);
  return 0;
}

// What the launchers above run, for qd_gemm_quad_plan: out = MT, NT, stage buffers, K splits, stages per
// split, output columns per workgroup.
void quad_query(int64_t M, int64_t N, int64_t K, int epi, int splits, int ks_per, int64_t* out) {
  const bool sw = epi == EPI_SWIGLU;
  const QuadShape& q = QUAD[quad_plan(M, N, sw, splits, ks_per)];
  const int64_t v[6] = {q.mt, q.nt, q.nbuf, splits, ks_per, quad_outs(q.nt, sw)};
  for (int i = 0; i < 6; ++i) out[i] = v[i];
}

void quad_small_query(int64_t M, int64_t N, int64_t K, int epi, int64_t part_floats, int64_t* out) {
  const SmallPlan P = quad_small_plan(M, N, K, epi == EPI_SWIGLU, part_floats / (M * N));
  const int64_t v[6] = {2, P.nt, quad_small_nbuf(P.nt), P.splits, P.ks_per, P.outs};
  for (int i = 0; i < 6; ++i) out[i] = v[i];
}

// split partials the two above can use at most
int64_t quad_small_ws_floats(int64_t M, int64_t N, int64_t K) {
  const SmallPlan P = quad_small_plan(M, N, K, false, SMALL_SPLITS);
  return P.splits > 1 ? (int64_t)P.splits * M * N : 0;
}

// LM head over 33..64 and 129 and more rows: argmax partials pval / pidx [M][return value] (one per
// block of vocabulary rows; the last block may pass the vocabulary: its missing rows reload a valid
// one and are never ranked); 0, with nothing launched, for other shapes.  129 and more rows: of three
// tile shapes the one that the cost above favours; with {8, 8} alone, 256 rows, the whole head over 129
// rows took 252 us at 151936 (8-wave kernel 246; {6, 8}: 239) and 62.9 at 16000 (60.0; {4, 4}: 31.7).
// 33..64 rows: 320 vocabulary rows per workgroup, two nearly full rounds (475 workgroups at 151936), three
// stages of 40 KiB of weights in LDS: 40 rows 275 -> 138 us (5.6 TB/s) against gemm_stream_kernel, which
// re-stages the activations with every chunk; 64 rows 285 -> 139 us ({2, 4} tiles 139 / 146, {2, 8} 157 /
// 159).  Under LM_SMALL_BLOCKS workgroups the stream kernel's 256 are faster (33 rows at 8192: 33.8 against
// 35.9).  65..128 rows stay on gemm_tile_kernel: 167 us at 100 rows against 174 with {4, 8} tiles here.
constexpr int64_t LM_SMALL_BLOCKS = 48;

template <int MT, int NT, int NBUF>
static int64_t lm_quad_go(const bf16_t* x, int64_t xs, int64_t M, const bf16_t* w, int64_t N, int64_t K,
                          float* pval, int32_t* pidx, float* logits, hipStream_t s) {
  const int64_t mbl = (M + 32 * MT - 1) / (32 * MT), nbl = (N + 32 * NT - 1) / (32 * NT);
  gemm_quad_kernel<EPI_ARGMAX, false, MT, NT, NBUF><<<dim3((unsigned)(mbl * nbl)), dim3(256), 0, s>>>(
      x, xs, (int)M, w, (int)N, (int)K, (int)mbl, (int)nbl, 32 * NT, (int)(K / TK), nullptr, 0, nullptr, 0, 0,
      nullptr, pval, pidx, logits);
  return nbl;
}

int64_t launch_lm_quad(const bf16_t* x, int64_t xs, int64_t M, const bf16_t* w, int64_t N, int64_t K,
                       float* pval, int32_t* pidx, float* logits, hipStream_t s) {
  const bool small = M >= 33 && M <= 64;
  if ((!small && M < 129) || M >= (1ll << 31) || N % 4 || N < 256 || K % TK ||
      !quad_offsets_ok(xs, N, K, EPI_ARGMAX))
    return 0;
  if (xs % 8 || reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(w) % 16) return 0;
  if (small) {
    if ((N + 319) / 320 < LM_SMALL_BLOCKS) return 0;
    return lm_quad_go<2, 10, 3>(x, xs, M, w, N, K, pval, pidx, logits, s);
  }
  constexpr QuadShape S0 = QUAD[1], S1 = QUAD[8], S2 = QUAD[12];
  static_assert(S0.nt % 2 == 0 && S1.mt == 6 && S1.nt == 8 && S2.mt == 8, "{4, 4}, {6, 8}, {8, 8}");
  const double t0 = quad_cost(S0, M, N, false, 1, K / TK), t1 = quad_cost(S1, M, N, false, 1, K / TK),
               t2 = quad_cost(S2, M, N, false, 1, K / TK);
  if (t0 < t1 && t0 < t2) return lm_quad_go<S0.mt, S0.nt, S0.nbuf>(x, xs, M, w, N, K, pval, pidx, logits, s);
  if (t1 < t2) return lm_quad_go<S1.mt, S1.nt, S1.nbuf>(x, xs, M, w, N, K, pval, pidx, logits, s);
  return lm_quad_go<S2.mt, S2.nt, S2.nbuf>(x, xs, M, w, N, K, pval, pidx, logits, s);
}
