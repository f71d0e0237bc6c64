// Products of ordinary size, C = epilogue(A * B [+ A1 * B1]) in any of the three layouts (l*r, l^T*r, l*r^T), single or
// strided-batched (dynet/matrix-multiply.h:16-37,97-117,162-180; cuBLAS sgemm and sgemmStridedBatched there), at any
// alignment: everything between the streaming kernels for a few rows or columns and the 256 x 256-tile kernel.
//
// A block owns a tile of 32*TM x 32*TN outputs; its wavefronts split the depth, each multiplies the whole tile over its
// part, and they meet in LDS once, at the end: no barrier in the loop.  fp32 in and out, on the bf16 matrix cores with every
// operand as three bf16 values (split3.h); depths below 32, which only a batch of more than 65 535 items, slices for another
// kernel and gates of a handful of inputs bring here, on the fp32 instruction in one form.
//
// Step of 16 k: 128-bit loads (dword-aligned is enough) in the order of memory, written to a piece of LDS that is the
// wavefront's own, read from there as fragments (lane 32*lhi + l32 holds k = 8*lhi .. 8*lhi + 7 of row l32), split in
// registers.  Four steps of loads are in flight and a step crosses LDS under the products of the one before it; with 2 x 2
// tiles, whose accumulators and fragments fill the registers, one, and it is read when its fragments are formed (1024^3
// 20.8 -> 22.2 us, against 26.4 with the sums of a step by themselves, which spilled).  Rows past the matrix are read at a
// clamped row and their outputs dropped; a depth that is not a multiple of 16 ends in a step of clamped, zeroed loads.
//
// What bounds it: the latency of a step's way through memory, LDS and the split, with one to three wavefronts a SIMD to
// cover it.  us in a graph, fp32 instruction in 128-wide tiles -> here: 1024 x 512 x 784 l*r 22.3 -> 13.5, 1024 x 784 x 512
// l*r^T 24.2 -> 14.9, 1024^3 33.6 -> 22.4.
#include <algorithm>
#include <type_traits>

#include "gemm.h"
#include "split3.h"

namespace dyhip {

namespace {

typedef float directx16 __attribute__((ext_vector_type(16)));
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));

struct DirectArgs {
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

// One operand's part of a 16-deep step, T tiles of 32 rows, on its way from memory through a wavefront's own piece of LDS
// into fragments.  Stored along k: a load instruction is 16 rows x 64 bytes, LDS holds [row][4 chunks of 16 bytes], chunk c
// of row r at position c ^ (r/4 % 4) (fragment reads of 16 neighbouring rows then cover all banks); tile t is rows
// 32*t + l32.  Stored along its rows: an instruction is 8/T k x 128*T bytes, LDS holds [k][32*T rows]; tile t is rows
// T*l32 + t.
// Offsets are in bytes from the tile's first row: 32 bits (Off) where a leading dimension is small enough for them.
template <bool KMAJOR, int T, typename Off>
struct DirectOperand {
  static constexpr int L = 2 * T;  // 128-bit loads a lane and step
  const float* base;  // the tile's first row, k = 0 (uniform)
  size_t ld;
  Off off[KMAJOR ? L : 1];
  unsigned K, rows;              // depth; rows inside the matrix from the tile's first
  // Groups of four rows past the matrix edge are moved to its last four rows; one that straddles the edge is shifted back
  // into place on its way to LDS.  back: rows before the tile that its only group then starts at.  few: the matrix has fewer
  // than four rows, every load is checked (uniform).
  unsigned shift, back;
  bool straddles, few;

  __device__ __forceinline__ void init(const float* p, size_t ld_, unsigned K_, unsigned mn0, unsigned MN, unsigned lane) {
    ld = ld_;
    K = K_;
    rows = MN - mn0;
    straddles = !KMAJOR && rows < 32 * T && rows % 4 != 0;
    few = !KMAJOR && rows < 4 && mn0 == 0;
    back = !KMAJOR && rows < 4 && mn0 > 0 ? 4 - rows : 0;
    base = p + (KMAJOR ? size_t(mn0) * ld : size_t(mn0 - back));
    shift = 0;
    if (KMAJOR) {
#pragma unroll
      for (int i = 0; i < L; ++i) off[i] = 4 * (Off(min(16u * i + lane / 4, rows - 1)) * Off(ld) + 4 * (((lane % 4) ^ (lane / 16)) % 4));
    } else {
      const unsigned r0 = 4 * (lane % (8 * T)), moved = min(r0, rows >= 4 ? rows - 4 : 0u);
      off[0] = 4 * (Off(lane / (8 * T)) * Off(ld) + moved);
      shift = min(r0 - moved + back, 3u);  // (3: a group wholly past the edge, whatever it holds)
    }
  }
  __device__ __forceinline__ void load(float4u (&v)[L], unsigned step) const {
    const float* p = base + size_t(step) * (KMAJOR ? 16 : 16 * ld);
#pragma unroll
    for (int i = 0; i < L; ++i) {
      v[i] = *reinterpret_cast<const float4u*>(reinterpret_cast<const char*>(p) + off[KMAJOR ? i : 0]);
      if (!KMAJOR) p += (8 / T) * ld;
    }
  }
  // the same for fewer than four rows, or for the last step of a depth that is not a multiple of 16: elements past an edge
  // are read at the last row or k, those past the depth are zeroed
  __device__ __forceinline__ void load_checked(float4u (&v)[L], unsigned step, unsigned lane) const {
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const unsigned r0 = KMAJOR ? 16 * i + lane / 4 : 4 * (lane % (8 * T));
      const unsigned k0 = step * 16 + (KMAJOR ? 4 * (((lane % 4) ^ (lane / 16)) % 4) : (8 / T) * i + lane / (8 * T));
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const unsigned r = min(KMAJOR ? r0 : r0 + c, rows - 1), k = KMAJOR ? k0 + c : k0;
        const float x = base[KMAJOR ? size_t(r) * ld + min(k, K - 1) : size_t(min(k, K - 1)) * ld + back + r];
        v[i][c] = k < K ? x : 0.f;
      }
    }
  }
  template <bool CHECKED>
  __device__ __forceinline__ void store(float* lds, const float4u (&v)[L], unsigned lane) const {
#pragma unroll
    for (int i = 0; i < L; ++i) {
      float4 x = make_float4(v[i][0], v[i][1], v[i][2], v[i][3]);
      if (!KMAJOR && !CHECKED && straddles) {
        x.x = shift & 1 ? x.y : x.x;
        x.y = shift & 1 ? x.z : x.y;
        x.z = shift & 1 ? x.w : x.z;
        x.x = shift & 2 ? x.z : x.x;
        x.y = shift & 2 ? x.w : x.y;
      }
      *reinterpret_cast<float4*>(lds + 256 * i + 4 * lane) = x;
    }
  }
  // k = 8*lhi .. 8*lhi + 7 of row (or column) l32 of every tile
  __device__ __forceinline__ void read(float (&x)[T][8], const float* lds, unsigned l32, unsigned lhi) const {
    if (KMAJOR) {
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const float* row = lds + (32 * t + l32) * 16;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const float4 y = *reinterpret_cast<const float4*>(row + 4 * ((2 * lhi + c) ^ (l32 / 4 % 4)));
          x[t][4 * c] = y.x; x[t][4 * c + 1] = y.y; x[t][4 * c + 2] = y.z; x[t][4 * c + 3] = y.w;
        }
      }
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float* q = lds + (8 * lhi + k) * (32 * T) + T * l32;
        if (T == 2) {
          const float2 y = *reinterpret_cast<const float2*>(q);
          x[0][k] = y.x;
          x[T - 1][k] = y.y;
        } else {
          x[0][k] = *q;
        }
      }
    }
  }
};

template <int T>
__device__ __forceinline__ void split_frags(const float (&v)[T][8], bf16x8 (&h)[T], bf16x8 (&m)[T], bf16x8 (&l)[T]) {
#pragma unroll
  for (int t = 0; t < T; ++t) {
    uint4 ph, pm, pl;
    split3_pair(v[t][0], v[t][1], ph.x, pm.x, pl.x);
    split3_pair(v[t][2], v[t][3], ph.y, pm.y, pl.y);
    split3_pair(v[t][4], v[t][5], ph.z, pm.z, pl.z);
    split3_pair(v[t][6], v[t][7], ph.w, pm.w, pl.w);
    h[t] = __builtin_bit_cast(bf16x8, ph);
    m[t] = __builtin_bit_cast(bf16x8, pm);
    l[t] = __builtin_bit_cast(bf16x8, pl);
  }
}

template <int TM, int TN>
__device__ __forceinline__ void direct_mma(const bf16x8 (&a)[TM], const bf16x8 (&b)[TN], directx16 (&acc)[TN][TM]) {
#pragma unroll
  for (int u = 0; u < TN; ++u)
#pragma unroll
    for (int t = 0; t < TM; ++t) acc[u][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[u], a[t], acc[u][t], 0, 0, 0);
}

// The fragments of one step, ready for the matrix cores: three bf16 parts, or the fp32 values themselves.
template <bool SPLIT, int T>
struct DirectFrags {
  bf16x8 h[T], m[T], l[T];
  __device__ __forceinline__ void from(const float (&v)[T][8]) { split_frags<T>(v, h, m, l); }
};
template <int T>
struct DirectFrags<false, T> {
  float x[T][8];
  __device__ __forceinline__ void from(const float (&v)[T][8]) {
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int k = 0; k < 8; ++k) x[t][k] = v[t][k];
  }
};

// A step's products.  The bf16 ones of the h parts have an accumulator of their own, the five small ones share another
// (split3.h); the fp32 ones have one.
template <int TM, int TN>
__device__ __forceinline__ void direct_step(const DirectFrags<true, TM>& a, const DirectFrags<true, TN>& b,
                                            directx16 (&acc)[TN][TM], directx16 (&low)[TN][TM]) {
  direct_mma<TM, TN>(a.l, b.h, low);
  direct_mma<TM, TN>(a.h, b.l, low);
  direct_mma<TM, TN>(a.m, b.m, low);
  direct_mma<TM, TN>(a.m, b.h, low);
  direct_mma<TM, TN>(a.h, b.m, low);
  direct_mma<TM, TN>(a.h, b.h, acc);
}
template <int TM, int TN>
__device__ __forceinline__ void direct_step(const DirectFrags<false, TM>& a, const DirectFrags<false, TN>& b,
                                            directx16 (&acc)[TN][TM], directx16 (&)[TN][TM]) {
#pragma unroll
  for (int k = 0; k < 8; ++k)
#pragma unroll
    for (int u = 0; u < TN; ++u)
#pragma unroll
      for (int t = 0; t < TM; ++t) acc[u][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(b.x[u][k], a.x[t][k], acc[u][t], 0, 0, 0);
}

// 2 x 2 tiles: accumulators and fragments fill the registers
template <int TM, int TN>
constexpr bool kDirectFull = TM * TN == 4;

template <bool AK, bool BKM, int TM, int TN, int WAVES, bool SPLIT>
__global__ __launch_bounds__(64 * WAVES, 2) void gemm_direct_kernel(DirectArgs g) {
  using Off = std::conditional_t<kDirectFull<TM, TN>, unsigned, size_t>;
  constexpr int R = 16 * TM * TN;                  // accumulator registers a lane
  constexpr int STAGE = 512 * (TM + TN);           // floats of a wavefront's step
  constexpr int LDS = WAVES * (R * 64 > STAGE ? R * 64 : STAGE);
  __shared__ __attribute__((aligned(16))) float lds[LDS];
  const unsigned lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned l32 = lane & 31, lhi = lane >> 5;
  unsigned m0, n0;
  const TileOrder order = g.order;
  order.locate(blockIdx.x, m0, n0);
  m0 *= 32 * TM;
  n0 *= 32 * TN;
  const unsigned s0 = blockIdx.y * g.steps_per_split, s1 = min(g.steps, s0 + g.steps_per_split);
  const unsigned w0 = s0 + (s1 - s0) * w / WAVES, w1 = s0 + (s1 - s0) * (w + 1) / WAVES;
  float* const la = lds + w * STAGE;
  float* const lb = la + 512 * TM;
  directx16 acc[TN][TM], low[TN][TM];
#pragma unroll
  for (int u = 0; u < TN; ++u)
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[u][t][r] = low[u][t][r] = 0.f;

  unsigned first = 0;  // first step of the segment
  for (int sg = 0; sg < g.nseg; ++sg) {
    const GemmSeg& q = g.seg[sg];
    const unsigned K = unsigned(q.K), count = (K + 15) / 16;
    const unsigned a0 = max(w0, first) - first, a1 = min(w1, first + count);
    const bool mine = a1 > first + a0;
    const unsigned e = mine ? a1 - first : a0;  // this wave's steps of the segment: [a0, e)
    first += count;
    if (!mine) continue;
    DirectOperand<AK, TM, Off> oa;
    DirectOperand<BKM, TN, Off> ob;
    oa.init(q.A + size_t(blockIdx.z) * g.stride_a, q.lda, K, m0, g.M, lane);
    ob.init(q.B + size_t(blockIdx.z) * g.stride_b, q.ldb, K, n0, g.N, lane);
    // Steps of loads in flight, and whether a step is read from LDS when its fragments are formed or one step ahead:
    // 2 x 2 tiles have no registers to spare beside their accumulators.
    constexpr bool LATE = kDirectFull<TM, TN>;
    constexpr int RAW = LATE ? 1 : 4;
    float4u ra[RAW][2 * TM], rb[RAW][2 * TN];
    float xa[TM][8], xb[TN][8];
    DirectFrags<SPLIT, TM> fa;
    DirectFrags<SPLIT, TN> fb;
    // Through LDS: write, then read; nobody else touches a wavefront's piece, and its LDS accesses stay in order.
#define DYHIP_DIRECT_STORE(buf, checked)                 \
  oa.template store<checked>(la, ra[buf], lane);         \
  ob.template store<checked>(lb, rb[buf], lane);         \
  __builtin_amdgcn_wave_barrier();
#define DYHIP_DIRECT_READ                                \
  oa.read(xa, la, l32, lhi);                             \
  ob.read(xb, lb, l32, lhi);                             \
  __builtin_amdgcn_wave_barrier();
    const unsigned full = oa.few || ob.few ? a0 : max(a0, min(e, K / 16));
    if (full > a0) {
      // A step crosses LDS under the MFMAs of the one before it.  Loads past the range repeat its last step
      // (unconditional: the compiler counts what is in flight only in straight-line code).
#define DYHIP_DIRECT_LOAD(buf, s)         \
  oa.load(ra[buf], min((s), full - 1));   \
  ob.load(rb[buf], min((s), full - 1));
#pragma unroll
      for (int r = 0; r < RAW; ++r) { DYHIP_DIRECT_LOAD(r, a0 + r) }
      DYHIP_DIRECT_STORE(0, false)
      if (!LATE) { DYHIP_DIRECT_READ }
      DYHIP_DIRECT_LOAD(0, a0 + RAW)
      for (unsigned s = a0; s < full; s += RAW) {
#pragma unroll
        for (int r = 0; r < RAW; ++r) {
          if (r > 0 && s + r >= full) break;
          constexpr int NB = RAW - 1;
          if (LATE) { DYHIP_DIRECT_READ }
          fa.from(xa);
          fb.from(xb);
          __builtin_amdgcn_sched_barrier(0);
          DYHIP_DIRECT_STORE((r + 1) & NB, false)
          if (!LATE) { DYHIP_DIRECT_READ }
          DYHIP_DIRECT_LOAD((r + 1) & NB, s + r + 1 + RAW)
          direct_step<TM, TN>(fa, fb, acc, low);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
#undef DYHIP_DIRECT_LOAD
    }
    for (unsigned s = full; s < e; ++s) {
      oa.load_checked(ra[0], s, lane);
      ob.load_checked(rb[0], s, lane);
      DYHIP_DIRECT_STORE(0, true)
      DYHIP_DIRECT_READ
      fa.from(xa);
      fb.from(xb);
      direct_step<TM, TN>(fa, fb, acc, low);
    }
#undef DYHIP_DIRECT_STORE
#undef DYHIP_DIRECT_READ
  }

  if (SPLIT) {  // this wavefront's sums, whole and to scale
#pragma unroll
    for (int u = 0; u < TN; ++u)
#pragma unroll
      for (int t = 0; t < TM; ++t) {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[u][t][r] = (acc[u][t][r] + low[u][t][r]) * kSplitOut;
        if (__builtin_expect(any_not_finite(acc[u][t]), 0)) {
          const unsigned m = min(m0 + (AK ? 32 * t + l32 : TM * l32 + t), g.M - 1);
          const unsigned n = min(n0 + (BKM ? 32 * u + l32 : TN * l32 + u), g.N - 1);
          sums16 s = {};
          unsigned fs = 0;
          for (int sg = 0; sg < g.nseg; ++sg) {
            const GemmSeg& q = g.seg[sg];
            const unsigned count = (unsigned(q.K) + 15) / 16, b0 = max(w0, fs) - fs, b1 = max(min(w1, fs + count), fs) - fs;
            add_products_fp32<AK, BKM>(s, q.A + size_t(blockIdx.z) * g.stride_a + (AK ? m * q.lda : m), q.lda,
                                       q.B + size_t(blockIdx.z) * g.stride_b + (BKM ? n * q.ldb : n), q.ldb, 16 * b0,
                                       min(16 * b1, unsigned(q.K)));
            fs += count;
          }
          acc[u][t] = s;
        }
      }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < TN; ++u)
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) lds[((w * TN + u) * TM + t) * 1024 + r * 64 + lane] = acc[u][t][r];
  __syncthreads();
  // wavefront w finishes 16 * TN / WAVES groups of TM outputs a lane
  float* out = g.partial != nullptr ? g.partial + size_t(blockIdx.y) * g.M * g.N : g.C + size_t(blockIdx.z) * g.stride_c;
#pragma unroll
  for (int x = 0; x < 16 * TN / WAVES; ++x) {
    const unsigned f = w * (16 * TN / WAVES) + x, r = f % 16, u = f / 16;
    const unsigned i = 8 * (r / 4) + 4 * lhi + r % 4, n = n0 + (BKM ? 32 * u + i : TN * i + u);
    if (n >= g.N) continue;
#pragma unroll
    for (int t = 0; t < TM; ++t) {
      const unsigned m = m0 + (AK ? 32 * t + l32 : TM * l32 + t);
      if (m >= g.M) continue;
      float v = lds[(u * TM + t) * 1024 + r * 64 + lane];
#pragma unroll
      for (int ww = 1; ww < WAVES; ++ww) v += lds[((ww * TN + u) * TM + t) * 1024 + r * 64 + lane];
      float* p = out + m + size_t(n) * g.M;
      if (g.partial == nullptr) {
        if (g.epi.kind == kEpiAxpby) {
          if (g.epi.beta != 0.f) v += g.epi.beta * *p;
        } else {
          float pre = g.epi.bias[m];
          if (g.epi.kind == kEpiLstmGates) {
            if (m >= g.epi.H && m < 2 * g.epi.H) pre += 1.0f;  // forget-gate bias
            pre += v;
            v = m < 3 * g.epi.H ? logistic(g.epi.logistic_mode, pre) : tanh_accurate(pre);
          } else {
            v += pre;
          }
        }
      }
      *p = v;
    }
  }
}

}  // namespace

int gemm_direct_launch(dyhip_device* dev, bool a_kmajor, bool b_kmajor, size_t M, size_t N, int nseg, const GemmSeg* segs,
                       float* C, float* partial, const GemmEpiParams& epi, const GemmBatch* batch, int tm, int tn,
                       int waves, unsigned splits_wanted, unsigned* splits) {
  DYHIP_REQUIRE((tm == 1 || tm == 2) && (tn == 1 || tn == tm) && (waves == 4 || (waves == 8 && tn == 1)), "no such tile");
  DirectArgs g;
  g.nseg = nseg;
  g.M = unsigned(M);
  g.N = unsigned(N);
  g.C = C;
  g.partial = partial;
  g.epi = epi;
  g.steps = 0;
  size_t depth = 0, ld = 0;
  for (int s = 0; s < kGemmMaxSeg; ++s) {
    g.seg[s] = s < nseg ? segs[s] : GemmSeg{nullptr, 0, nullptr, 0, 0};
    g.steps += unsigned((g.seg[s].K + 15) / 16);
    depth += g.seg[s].K;
    ld = std::max({ld, g.seg[s].lda, g.seg[s].ldb});
  }
  const unsigned items = batch != nullptr && batch->count > 1 ? batch->count : 1;
  g.stride_a = items > 1 ? batch->stride_a : 0;
  g.stride_b = items > 1 ? batch->stride_b : 0;
  g.stride_c = items > 1 ? batch->stride_c : 0;
  if (tn == 2 && ld >= (size_t(1) << 24)) tn = 1;  // 2 x 2 tiles: 32-bit offsets over 64 rows
  g.order = TileOrder::of(cdiv<unsigned>(g.M, 32 * tm), cdiv<unsigned>(g.N, 32 * tn), tm, tn);
  g.steps_per_split = std::max(1u, cdiv<unsigned>(std::max(1u, g.steps), splits_wanted));
  *splits = std::max(1u, cdiv<unsigned>(g.steps, g.steps_per_split));
  const dim3 grid(g.order.tiles_m * g.order.tiles_n, *splits, items);
#define DYHIP_DIRECT(TM, TN, W, SP)                                                                                           \
  do {                                                                                                                      \
    if (a_kmajor && b_kmajor) hipLaunchKernelGGL((gemm_direct_kernel<true, true, TM, TN, W, SP>), grid, dim3(64 * W), 0, dev->stream, g);       \
    else if (a_kmajor) hipLaunchKernelGGL((gemm_direct_kernel<true, false, TM, TN, W, SP>), grid, dim3(64 * W), 0, dev->stream, g);             \
    else if (b_kmajor) hipLaunchKernelGGL((gemm_direct_kernel<false, true, TM, TN, W, SP>), grid, dim3(64 * W), 0, dev->stream, g);             \
    else hipLaunchKernelGGL((gemm_direct_kernel<false, false, TM, TN, W, SP>), grid, dim3(64 * W), 0, dev->stream, g);                          \
  } while (0)
  if (depth < 32) DYHIP_DIRECT(1, 1, 4, false);
  else if (tm == 2 && tn == 2) DYHIP_DIRECT(2, 2, 4, true);
  else if (tm == 2 && waves == 8) DYHIP_DIRECT(2, 1, 8, true);
  else if (tm == 2) DYHIP_DIRECT(2, 1, 4, true);
  else if (waves == 8) DYHIP_DIRECT(1, 1, 8, true);
  else DYHIP_DIRECT(1, 1, 4, true);
#undef DYHIP_DIRECT
  DYHIP_CHECK_LAUNCH();
  return DYHIP_OK;
}

}  // namespace dyhip
