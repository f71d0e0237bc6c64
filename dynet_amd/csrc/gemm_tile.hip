// Products of a few hundred tiles and more that the 256 x 256-tile kernel does not take (ragged, or not enough of them):
// C = epilogue(A * B [+ A1 * B1]) in the three layouts, single or strided-batched, at any alignment
// (dynet/matrix-multiply.h:16-37,97-117,162-180).  A 256-thread block (4 wavefronts, 2 x 2) owns a 128 x 128 tile; fp32 in
// and out, on the bf16 matrix cores with every operand as three bf16 values (split3.h).
//
// The 256-wide kernel at half the size, for its reason: a value is fetched and split once per block and reaches the
// wavefronts that share it through LDS.  (Without LDS sharing, 64 x 64 tiles and the depth over the wavefronts, the
// address units and the L2s are the limit: 10 000 x 700 x 650 in 90 us.)  A step is 16 deep: three planes (h, m, l) of
// [k half][128 slots][8 bf16] per operand, 24 KiB a stage, two stages; two blocks share a CU (their registers are the limit)
// and cover each other's barriers.  A slot is a row of the operand: row r itself for one stored along k, slot 32*j + i for row 4*i + j of
// one stored along its rows (the four rows of a lane's 128-bit load go to four places that neighbouring lanes continue);
// slots of the second k half are permuted by xor 4, which keeps the two halves of a row on different banks.
// Wavefronts 0, 1 stage A, wavefronts 2, 3 stage B: four 128-bit loads a lane (dword-aligned is enough), split into
// 4 rows x 4 k, three 64-bit LDS writes a row.  24 MFMAs a wavefront and step, plane by plane (l*h, m*h, m*m, h*m, h*l, h*h):
// the small planes' registers are free early, and the next step's fragments are read into them under this step's products.
// 10 000 x 700 x 650 76 us (128-wide tiles on the fp32 instruction 136), 2051 x 2050 x 650 as l*r^T 66 (120).
#include "gemm.h"
#include "split3.h"

namespace dyhip {

namespace {

typedef float tilex16 __attribute__((ext_vector_type(16)));
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float float2u __attribute__((ext_vector_type(2), aligned(4)));

constexpr unsigned kTileT = 128, kTilePlane = 4096, kTileOperand = 3 * kTilePlane, kTileStage = 2 * kTileOperand;

struct TileArgs {
  GemmSeg seg[kGemmMaxSeg];
  int nseg;
  unsigned M, N;
  float* C;
  float* partial;  // [splits][M*N] when set: no epilogue
  GemmEpiParams epi;
  size_t stride_a, stride_b, stride_c;  // between the items of a batch (blockIdx.z)
  TileOrder order;
  unsigned steps, steps_per_split;  // 16-deep steps of all segments laid end to end; of a block
};

template <bool AK, bool BKM>
__global__ __launch_bounds__(256, 2) void gemm_tile_kernel(TileArgs g) {
  __shared__ __attribute__((aligned(16))) char lds[2 * kTileStage];
  const unsigned lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned wm = w & 1, wn = w >> 1, l32 = lane & 31, lhi = lane >> 5;
  unsigned m0, n0;
  const TileOrder order = g.order;
  order.locate(blockIdx.x, m0, n0);
  m0 *= kTileT;
  n0 *= kTileT;
  const unsigned s0 = blockIdx.y * g.steps_per_split, s1 = min(g.steps, s0 + g.steps_per_split);

  // ---- loader: this wavefront's operand ----
  const bool stage_b = w >= 2;
  const bool kmajor = AK == BKM ? AK : stage_b ? BKM : AK;
  const unsigned w2 = w & 1, mn0 = stage_b ? n0 : m0, rows = (stage_b ? g.N : g.M) - mn0;
  // First of a lane's rows, and its k inside a step.  Groups of four rows that reach past the matrix edge are moved to its
  // last four, and written to those rows' slots (by several lanes then, with the same values); rows before the tile, where
  // fewer than four are left, to slots past the edge.
  const unsigned row0 = kmajor ? 16 * w2 + lane / 4 : rows >= 4 ? min(4 * (lane % 32), rows - 4) : mn0 > 0 ? rows - 4 : 0u;
  const unsigned quarter = kmajor ? lane % 4 : 2 * w2 + lane / 32, half = quarter / 2;
  const bool few = !kmajor && rows < 4 && mn0 == 0;
  unsigned load_at = s0, load_end = 0, load_k = 0, Kseg = 0;  // next step; end of its segment; its k; the segment's depth
  size_t ld = 0, off[4];
  const float* op = nullptr;  // the segment's operand at the tile's first row
#define DYHIP_TILE_SEG                                                                                   \
  if (load_at >= load_end) {                                                                             \
    unsigned first_ = 0;                                                                                 \
    bool second_ = false;                                                                                \
    load_end = (unsigned(g.seg[0].K) + 15) / 16;                                                         \
    if (g.nseg > 1 && load_at >= load_end) {                                                             \
      first_ = load_end;                                                                                 \
      second_ = true;                                                                                    \
      load_end += (unsigned(g.seg[1].K) + 15) / 16;                                                      \
    }                                                                                                    \
    Kseg = unsigned(second_ ? g.seg[1].K : g.seg[0].K);                                                  \
    ld = stage_b ? (second_ ? g.seg[1].ldb : g.seg[0].ldb) : (second_ ? g.seg[1].lda : g.seg[0].lda);    \
    op = (stage_b ? (second_ ? g.seg[1].B : g.seg[0].B) + size_t(blockIdx.z) * g.stride_b                \
                  : (second_ ? g.seg[1].A : g.seg[0].A) + size_t(blockIdx.z) * g.stride_a) +             \
         (kmajor ? size_t(mn0) * ld : size_t(mn0));                                                      \
    load_k = (load_at - first_) * 16;                                                                    \
    _Pragma("unroll") for (int j_ = 0; j_ < 4; ++j_) off[j_] =                                           \
        kmajor ? size_t(min(row0 + 32 * j_, rows - 1)) * ld + 4 * quarter : size_t(ptrdiff_t(int(row0))) + size_t(4 * quarter + j_) * ld; \
  }
  float4u raw[4];
  // loads past the block's last step repeat it
#define DYHIP_TILE_LOAD                                                                                  \
  {                                                                                                      \
    if (few || (load_at + 1 == load_end && Kseg % 16 != 0)) {                                            \
      const unsigned kb_ = load_k + 4 * quarter;                                                         \
      _Pragma("unroll") for (int j_ = 0; j_ < 4; ++j_) _Pragma("unroll") for (int c_ = 0; c_ < 4; ++c_) { \
        const unsigned r_ = min(kmajor ? row0 + 32 * j_ : row0 + c_, rows - 1);                          \
        const unsigned k_ = kb_ + (kmajor ? c_ : j_), kc_ = min(k_, Kseg - 1);                           \
        const float x_ = op[kmajor ? size_t(r_) * ld + kc_ : size_t(kc_) * ld + r_];                     \
        raw[j_][c_] = k_ < Kseg ? x_ : 0.f;                                                              \
      }                                                                                                  \
    } else {                                                                                             \
      const float* p_ = op + size_t(load_k) * (kmajor ? 1 : ld);                                         \
      _Pragma("unroll") for (int j_ = 0; j_ < 4; ++j_) raw[j_] = *reinterpret_cast<const float4u*>(p_ + off[j_]); \
    }                                                                                                    \
    if (load_at + 1 < s1) {                                                                              \
      ++load_at;                                                                                         \
      load_k += 16;                                                                                      \
      DYHIP_TILE_SEG                                                                                     \
    }                                                                                                    \
  }
  unsigned oa[2], ob[2], ow[4];  // fragments: a register per stage (see gemm_wide.hip); writes: one per row
  const unsigned frag = lhi * 2048 + (l32 ^ (4 * lhi)) * 16;
  oa[0] = frag + wm * 1024;
  ob[0] = kTileOperand + frag + wn * 1024;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const unsigned row = (row0 + (kmajor ? 32 * j : j)) % kTileT, slot = kmajor ? row : 32 * (row % 4) + row / 4;
    ow[j] = (stage_b ? kTileOperand : 0u) + half * 2048 + (slot ^ (4 * half)) * 16 + (quarter % 2) * 8;
  }
  oa[1] = oa[0] + kTileStage;
  ob[1] = ob[0] + kTileStage;
  asm volatile("" : "+v"(oa[1]), "+v"(ob[1]));
#define DYHIP_TILE_SPLIT(j, stage)                                                                       \
  {                                                                                                      \
    uint2 h_, m_, l_;                                                                                    \
    split3_pair_beside_products(kmajor ? raw[j][0] : raw[0][j], kmajor ? raw[j][1] : raw[1][j], h_.x, m_.x, l_.x);       \
    split3_pair_beside_products(kmajor ? raw[j][2] : raw[2][j], kmajor ? raw[j][3] : raw[3][j], h_.y, m_.y, l_.y);       \
    char* d_ = lds + ow[j] + (stage) * kTileStage;                                                            \
    *reinterpret_cast<uint2*>(d_) = h_;                                                                  \
    *reinterpret_cast<uint2*>(d_ + kTilePlane) = m_;                                                     \
    *reinterpret_cast<uint2*>(d_ + 2 * kTilePlane) = l_;                                                 \
  }
  bf16x8 ah[2], am[2], al[2], bh[2][2], bm[2], bl[2];
#define DYHIP_TILE_READ(f, o, plane) \
  _Pragma("unroll") for (int t_ = 0; t_ < 2; ++t_) f[t_] = *reinterpret_cast<const bf16x8*>(lds + (o) + (plane) * kTilePlane + t_ * 512);
#define DYHIP_TILE_MMA(fa, fb, sum)                               \
  _Pragma("unroll") for (int u_ = 0; u_ < 2; ++u_)                \
      _Pragma("unroll") for (int t_ = 0; t_ < 2; ++t_) sum[u_][t_] = \
          __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[u_], fa[t_], sum[u_][t_], 0, 0, 0);
#define DYHIP_TILE_FENCE __builtin_amdgcn_sched_barrier(0);
#define DYHIP_TILE_MIX(id, n, valu, rd, wr)                                \
  _Pragma("unroll") for (int x_ = 0; x_ < (n); ++x_) {                     \
    __builtin_amdgcn_sched_group_barrier(0x008, 1, id);                    \
    if (rd) __builtin_amdgcn_sched_group_barrier(0x100, rd, id);           \
    if (valu) __builtin_amdgcn_sched_group_barrier(0x002, valu, id);       \
    if (wr) __builtin_amdgcn_sched_group_barrier(0x200, wr, id);           \
  }
  tilex16 acc[2][2], low[2][2];  // sums of the products of the h parts, and of the five small ones (split3.h)
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[u][t][r] = low[u][t][r] = 0.f;

  if (s0 < s1) {
    if (!kmajor && rows < kTileT) {
      // Slots past the edge are never written.  Their outputs are dropped, but must not look like sums that are not finite:
      // zeros in this wavefront's half of them.
#pragma unroll
      for (unsigned x = 0; x < 12; ++x)
        *reinterpret_cast<uint4*>(lds + (stage_b ? kTileOperand : 0u) + half * 2048 + x / 6 * kTileStage + x % 6 / 2 * kTilePlane +
                                  x % 2 * 1024 + lane * 16) = make_uint4(0, 0, 0, 0);
    }
    DYHIP_TILE_SEG
    DYHIP_TILE_LOAD
#pragma unroll
    for (int j = 0; j < 4; ++j) DYHIP_TILE_SPLIT(j, 0)
    DYHIP_TILE_LOAD
#pragma unroll
    for (int j = 0; j < 4; ++j) DYHIP_TILE_SPLIT(j, 1)
    DYHIP_TILE_LOAD
    __syncthreads();
    DYHIP_TILE_READ(al, oa[0], 2)
    DYHIP_TILE_READ(bh[0], ob[0], 0)
    DYHIP_TILE_READ(am, oa[0], 1)
    DYHIP_TILE_READ(bm, ob[0], 1)
    for (unsigned s = s0; s < s1; s += 2) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        if (e == 1 && s + 1 >= s1) break;
        DYHIP_TILE_READ(ah, oa[e], 0)
        DYHIP_TILE_READ(bl, ob[e], 2)
        DYHIP_TILE_MMA(al, bh[e], low)
        DYHIP_TILE_MIX(0, 1, 0, 4, 0)
        DYHIP_TILE_MIX(0, 3, 0, 0, 0)
        DYHIP_TILE_FENCE
        // every wave's part of the next step is in LDS, and every wave holds its last fragments of this one, whose stage
        // is refilled below two steps ahead
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        DYHIP_TILE_FENCE
            DYHIP_TILE_MMA(am, bh[e], low)
        DYHIP_TILE_READ(al, oa[e ^ 1], 2)
        DYHIP_TILE_READ(bh[e ^ 1], ob[e ^ 1], 0)
        DYHIP_TILE_SPLIT(0, e)
        DYHIP_TILE_SPLIT(1, e)
        DYHIP_TILE_MIX(1, 2, 12, 2, 0)
        DYHIP_TILE_MIX(1, 2, 12, 0, 3)
        DYHIP_TILE_FENCE
        DYHIP_TILE_MMA(am, bm, low)
        DYHIP_TILE_SPLIT(2, e)
        DYHIP_TILE_SPLIT(3, e)
        DYHIP_TILE_MIX(2, 2, 12, 0, 0)
        DYHIP_TILE_MIX(2, 2, 12, 0, 3)
        DYHIP_TILE_FENCE
        DYHIP_TILE_READ(am, oa[e ^ 1], 1)
        DYHIP_TILE_MMA(ah, bm, low)
        DYHIP_TILE_FENCE
        DYHIP_TILE_LOAD
        DYHIP_TILE_READ(bm, ob[e ^ 1], 1)
        DYHIP_TILE_MMA(ah, bl, low)
        DYHIP_TILE_FENCE
        DYHIP_TILE_MMA(ah, bh[e], acc)
        DYHIP_TILE_FENCE
      }
    }
  }
#undef DYHIP_TILE_SEG
#undef DYHIP_TILE_LOAD
#undef DYHIP_TILE_SPLIT
#undef DYHIP_TILE_READ
#undef DYHIP_TILE_MMA
#undef DYHIP_TILE_FENCE
#undef DYHIP_TILE_MIX

  // the wavefront's sums, whole and to scale
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[u][t][r] = (acc[u][t][r] + low[u][t][r]) * kSplitOut;
      if (__builtin_expect(any_not_finite(acc[u][t]), 0)) {
        const unsigned m = min(m0 + (AK ? 64 * wm + 32 * t + l32 : 4 * l32 + 2 * wm + t), g.M - 1);
        const unsigned n = min(n0 + (BKM ? 64 * wn + 32 * u + l32 : 4 * l32 + 2 * wn + u), g.N - 1);
        sums16 s = {};
        unsigned first = 0;
        for (int sg = 0; sg < g.nseg; ++sg) {
          const GemmSeg& q = g.seg[sg];
          const unsigned count = (unsigned(q.K) + 15) / 16, b0 = max(s0, first) - first, b1 = max(min(s1, first + count), first) - first;
          add_products_fp32<AK, BKM>(s, q.A + size_t(blockIdx.z) * g.stride_a + (AK ? m * q.lda : m), q.lda,
                                     q.B + size_t(blockIdx.z) * g.stride_b + (BKM ? n * q.ldb : n), q.ldb, 16 * b0,
                                     min(16 * b1, unsigned(q.K)));
          first += count;
        }
        acc[u][t] = s;
      }
    }

  // acc[u][t][r] of a lane: two rows and, for each r, two columns
  float* out = g.partial != nullptr ? g.partial + size_t(blockIdx.y) * g.M * g.N : g.C + size_t(blockIdx.z) * g.stride_c;
  const bool direct = g.partial == nullptr;
  float bias[2] = {0.f, 0.f};
  unsigned m[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    m[t] = m0 + (AK ? 64 * wm + 32 * t + l32 : 4 * l32 + 2 * wm + t);
    if (direct && g.epi.kind != kEpiAxpby && m[t] < g.M) {
      bias[t] = g.epi.bias[m[t]];
      if (g.epi.kind == kEpiLstmGates && m[t] >= g.epi.H && m[t] < 2 * g.epi.H) bias[t] += 1.0f;  // forget-gate bias
    }
  }
  const float beta = direct && g.epi.kind == kEpiAxpby ? g.epi.beta : 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const unsigned i = 8 * (r / 4) + 4 * lhi + r % 4, n = n0 + (BKM ? 64 * wn + 32 * u + i : 4 * i + 2 * wn + u);
      if (n >= g.N) continue;
      float v[2] = {acc[u][0][r], acc[u][1][r]};
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if (m[t] >= g.M) continue;
        if (direct) {
          v[t] += bias[t];
          if (g.epi.kind == kEpiLstmGates)
            v[t] = m[t] < 3 * g.epi.H ? logistic(g.epi.logistic_mode, v[t]) : tanh_accurate(v[t]);
        }
      }
      float* p = out + size_t(n) * g.M;
      if (!AK && m[1] < g.M) {
        if (beta != 0.f) {
          const float2u o = *reinterpret_cast<const float2u*>(p + m[0]);
          v[0] += beta * o[0];
          v[1] += beta * o[1];
        }
        *reinterpret_cast<float2u*>(p + m[0]) = float2u{v[0], v[1]};
      } else {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          if (m[t] >= g.M) continue;
          if (beta != 0.f) v[t] += beta * p[m[t]];
          p[m[t]] = v[t];
        }
      }
    }
}

}  // namespace

int gemm_tile_launch(dyhip_device* dev, bool a_kmajor, bool b_kmajor, size_t M, size_t N, int nseg, const GemmSeg* segs,
                     float* C, float* partial, const GemmEpiParams& epi, const GemmBatch* batch, unsigned splits_wanted,
                     unsigned* splits) {
  TileArgs g;
  g.nseg = nseg;
  g.M = unsigned(M);
  g.N = unsigned(N);
  g.C = C;
  g.partial = partial;
  g.epi = epi;
  g.steps = 0;
  for (int s = 0; s < kGemmMaxSeg; ++s) {
    g.seg[s] = s < nseg ? segs[s] : GemmSeg{nullptr, 0, nullptr, 0, 0};
    g.steps += unsigned((g.seg[s].K + 15) / 16);
  }
  const unsigned items = batch != nullptr && batch->count > 1 ? batch->count : 1;
  g.stride_a = items > 1 ? batch->stride_a : 0;
  g.stride_b = items > 1 ? batch->stride_b : 0;
  g.stride_c = items > 1 ? batch->stride_c : 0;
  g.order = TileOrder::of(cdiv<unsigned>(g.M, kTileT), cdiv<unsigned>(g.N, kTileT), 1, 1);
  g.steps_per_split = g.steps <= splits_wanted ? 1 : cdiv<unsigned>(g.steps, splits_wanted);
  *splits = g.steps == 0 ? 1 : cdiv<unsigned>(g.steps, g.steps_per_split);
  const dim3 grid(g.order.tiles_m * g.order.tiles_n, *splits, items), block(256);
  if (a_kmajor && b_kmajor) hipLaunchKernelGGL((gemm_tile_kernel<true, true>), grid, block, 0, dev->stream, g);
  else if (a_kmajor) hipLaunchKernelGGL((gemm_tile_kernel<true, false>), grid, block, 0, dev->stream, g);
  else if (b_kmajor) hipLaunchKernelGGL((gemm_tile_kernel<false, true>), grid, block, 0, dev->stream, g);
  else hipLaunchKernelGGL((gemm_tile_kernel<false, false>), grid, block, 0, dev->stream, g);
  DYHIP_CHECK_LAUNCH();
  return DYHIP_OK;
}

}  // namespace dyhip
