// GEMM for large outputs: a 512-thread block (8 wavefronts, 2 x 4) owns a 256 x 256 tile of C, one block per CU.  fp32 in
// and out; the products run on the bf16 matrix cores, each fp32 value as the sum of three bf16 values, with the precision
// of the fp32 matrix instruction (split3.h).  Same three forms as gemm.hip, which keeps the small, skinny, ragged,
// segmented and batched problems (dynet/matrix-multiply.h:16-37,97-117,162-180 are the callers this replaces
// cublasSgemm for).
//
// What bounds it.  Six bf16 products for one fp32 product: at the 2.2-2.4 PFLOP/s that register-resident 32x32x16 MFMAs
// reach here the ceiling is about 370 TFLOP/s of fp32 work.  The MFMAs keep the matrix cores 61 % busy (counters, 10000 x
// 4480 x 1024) at a shader clock that falls to 1.9 GHz; a third stage in LDS, which takes the two wavefronts of a SIMD out
// of step, changed nothing.  Measured, random operands, against v_mfma_f32_32x32x2_f32 in the same tiling (94 % busy,
// 157 TFLOP/s at most):
//   10000 x 4480 x 1024 l*r     708 -> 473 us (130 -> 194 TFLOP/s)   1024 x 4480 x 10000 l^T*r   712 -> 478 us
//   10000 x 1024 x 4480 l*r^T   688 -> 448 us (133 -> 205)            4096 x 1024 x 4480 l*r^T    285 -> 192 us
//
// Step of 16 k.  Operands are fetched as fp32 into registers (four 128-bit loads a thread), split there and written to
// LDS as three bf16 planes: splitting in the block re-does the work for every tile that shares an operand, but 104 vector
// instructions a wave and step hide under 48 MFMAs, where a pass of its own over the operands would move 10 bytes per
// element (450 MB for a 10000 x 4480 operand).  LDS holds two stages of 48 KiB; fragments are read as 128 bits a lane.
//
// Sums.  A matrix instruction rounds what it adds to, so six of them into one accumulator round a long sum six times in 16
// k, where the fp32 instruction rounds it once a product that is not zero: with half of the products zero (a rectifier's
// outputs) the sums were 13 % further from fp64 than the fp32 instruction's, with nine tenths zero 76 % (K = 512).  So the
// six products of a 32 x 32 tile form a sum of their own, from zero, which vector instructions add to the accumulator:
// one rounding of the long sum in 16 k.  Three times closer than the fp32 instruction on dense operands, as close with 3 %
// of the products left (1.0-1.2 times), 1.15-1.3 times as far with 1 %.  (An accumulator each for the large and the small
// products, as in the other kernels, does not fit beside 128 sums a lane.)  It costs 6 %: 128 vector instructions a step.
//
// Schedule of a step (48 MFMAs per wave): tile by tile, two column tiles for each of four row tiles.  A tile's sum is added
// up under the MFMAs of the next one.  The second tile of a pair uses the small planes of the row tile first, so that the
// next row tile's planes are read into the same registers as they fall free.  One barrier before the last row tile: there
// every wave holds the last fragments of this step's stage, which is refilled two steps ahead under what is left, and the
// loads for the step after that leave last.  Vector and LDS instructions are dealt between the MFMAs one by one (left
// alone the compiler puts them in front).
//
// Work distribution.  The tile count rarely divides the CU count, and a round of one tile per CU that is not full
// leaves CUs idle for the whole round.  So the units of work are k-tiles: all k-tiles of all tiles, tile by tile, form
// one sequence that is cut into one equal segment per CU, and a block walks its segment, loads running two k-tiles
// ahead of the MFMAs straight across tile boundaries (the next tile's operands arrive under the stores of the one
// just finished).  A tile that lies wholly inside a segment is written out by that block.  A tile cut by segment
// boundaries is completed in one of two ways:
//   * segments at least a tile long (more tiles than CUs): a tile is cut at most once.  The block that holds its later
//     k-tiles (the start of its segment) leaves a partial tile in the workspace and raises a flag; the block that
//     holds its first k-tiles (the end of its segment, hundreds of microseconds later) adds that partial tile to its
//     own, applies the epilogue and stores.  No second kernel, no float atomics, a fixed order of additions.
//     Segments are dealt in descending block order, so a block only ever waits for a block dispatched before it,
//     which itself waits for nobody before it raises its flag; the wait is bounded anyway, and a wait that gave up is
//     counted and reported by dyhip_device_sync.
//   * shorter segments (fewer tiles than CUs, or little more): a tile spans several segments, one CU adding all their
//     partial tiles would take longer than its share of the product (256 KiB per partial tile at one CU's ~30 GB/s
//     from beyond its L2), so every part goes to the workspace and a second kernel, 16 blocks per tile, adds them in
//     segment order and applies the epilogue.
// When the tiles are a whole number of rounds plus a few tile columns, the caller gives this kernel the leading
// columns (whole rounds, nothing cut) and the rest to the 128 x 128-tile kernel.
#include "gemm.h"
#include "split3.h"

namespace dyhip {

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float fvec2 __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(1))) void* global_ptr_t;
typedef __attribute__((address_space(3))) void* lds_ptr_t;

constexpr int kWideThreads = 512;
constexpr int kWT = 256;                  // tile extent along m and along n
constexpr int kWK = 32;                   // k-tile
constexpr int kStageFloats = 16384;       // 64 KiB, a stage of the shallow kernel
constexpr size_t kSlotFloats = size_t(kWT) * kWT;

struct WideArgs {
  const float* A;
  const float* B;
  float* C;
  const float* bias;    // C = bias[m] + sum when set (beta unused)
  float* slots;         // partial tiles, [32][512 threads][4] in the order the threads hold them: slot = segment when
                        // tiles are finished in the kernel, else 2 x segment + (0: the segment's first item, 1: its last)
  unsigned* flags;      // one per segment, zero between launches; the last of the kGemmFlagWords counts waits that gave up
  unsigned lda, ldb;
  unsigned M, N;
  unsigned nt;          // k-tiles of a tile
  unsigned tiles_m;
  unsigned units;       // tiles x nt, dealt to the blocks in equal segments
  unsigned spin_limit;  // polls (about a microsecond apart) before a wait for another block gives up
  int raise_flags;      // 1; 0 only in tests of the give-up path (the partial tile is stored, its flag stays down)
  int finish_in_kernel; // a cut tile is finished by the block that holds its first k-tiles; else by the second kernel
  float beta;
};

// One K step is 16 deep; a k-tile is two steps.  A step's stage: for each operand three planes (h, m, l), each
// [k half][256 slots][8 bf16]: the 16 bytes that one lane of a 32x32x16 fragment reads.  A slot is a row of the operand:
// row r itself for an operand stored along k; slot 64*j + i for row 4*i + j of one stored along mn, so that the four
// rows a lane fetches with one 128-bit load go to four places that neighbouring lanes continue.  Slots of the second k
// half are permuted by xor 4, which puts the two halves of a row's 64 bytes on different banks.
// Waves 0-3 stage A, waves 4-7 stage B: four 128-bit loads a lane (16 values), split into 4 rows x 4 k, three 64-bit
// LDS writes a row.
// LDS: [operand][stage][plane], so that the second stage is in reach of an LDS instruction's offset.
constexpr unsigned kPlaneBytes = 8192, kStageBytes = 3 * kPlaneBytes, kOperandBytes = 2 * kStageBytes;
constexpr size_t kWideLdsBytes = 2 * kOperandBytes;  // 96 KiB

// byte offsets (from the tile's first row and the step's first k) of this lane's four loads; rows and groups of
// four past the matrix edge are clamped to the last one inside (their values only reach outputs the epilogue masks)
__device__ __forceinline__ void load_offsets(bool kmajor, unsigned (&off)[4], unsigned ld, unsigned mn0, unsigned MN) {
  const unsigned lane = threadIdx.x & 63, w4 = (threadIdx.x >> 6) & 3;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    off[j] = 4 * (kmajor ? min(64u * j + 16 * w4 + lane / 4, MN - mn0 - 1) * ld + 4 * (lane % 4)
                         : min(lane * 4, MN - mn0 - 4) + (4 * w4 + j) * ld);
}

// LDS byte offset of this lane's first row inside an operand's stage (its row j is 1024*j bytes further)
__device__ __forceinline__ unsigned write_offset(bool kmajor) {
  const unsigned lane = threadIdx.x & 63, w4 = (threadIdx.x >> 6) & 3;
  const unsigned quarter = kmajor ? lane % 4 : w4, slot = kmajor ? 16 * w4 + lane / 4 : lane, half = quarter / 2;
  return half * 4096 + (slot ^ (4 * half)) * 16 + (quarter % 2) * 8;
}

__device__ __forceinline__ float component(const float4& q, int c) { return c == 0 ? q.x : c == 1 ? q.y : c == 2 ? q.z : q.w; }

// row j of the 4 rows x 4 k in v, split and written
__device__ __forceinline__ void split_row(bool kmajor, const float4 (&v)[4], int j, char* dst) {
  float x[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) x[k] = kmajor ? component(v[j], k) : component(v[k], j);
  uint2 h, m, l;
  split3_pair_beside_products(x[0], x[1], h.x, m.x, l.x);
  split3_pair_beside_products(x[2], x[3], h.y, m.y, l.y);
  *reinterpret_cast<uint2*>(dst + 1024 * j) = h;
  *reinterpret_cast<uint2*>(dst + 1024 * j + kPlaneBytes) = m;
  *reinterpret_cast<uint2*>(dst + 1024 * j + 2 * kPlaneBytes) = l;
}

__device__ __forceinline__ bf16x8 read_frag(const char* p) { return *reinterpret_cast<const bf16x8*>(p); }

// Where output (u, r) of a lane lies along n, inside its tile (r: accumulator element, u: column tile of the wave)
template <bool BKM>
__device__ __forceinline__ unsigned out_column(unsigned wn, unsigned u, unsigned i) {
  return BKM ? wn * 64 + 32 * u + i : 4 * (32 * (wn >> 1) + i) + 2 * (wn & 1) + u;
}

// Values that blocks on different L2s hand to each other inside one launch go past those caches (each L2 serves one
// eighth of the chip and does not see the others' lines): relaxed system-scope atomic accesses, which the compiler
// offers up to 64 bits, two per 128-bit group.  They are ordinary accesses to the compiler: it counts them, waits for
// them before their values are used and pads the stores' data registers itself.
typedef float wide_v4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ unsigned long long pack_through(float lo, float hi) {
  return (unsigned long long)__float_as_uint(lo) | ((unsigned long long)__float_as_uint(hi) << 32);
}
__device__ __forceinline__ void store_through(float* p, float x, float y, float z, float w) {
  unsigned long long* q = reinterpret_cast<unsigned long long*>(p);
  __hip_atomic_store(q, pack_through(x, y), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(q + 1, pack_through(z, w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ wide_v4 load_through(const float* p) {
  const unsigned long long* q = reinterpret_cast<const unsigned long long*>(p);
  const unsigned long long lo = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  const unsigned long long hi = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  const wide_v4 v = {__uint_as_float(unsigned(lo)), __uint_as_float(unsigned(lo >> 32)), __uint_as_float(unsigned(hi)),
                     __uint_as_float(unsigned(hi >> 32))};
  return v;
}

// first unit of segment s when `units` k-tiles are dealt to `segments` blocks: floor(s * units / segments) in 32-bit
// arithmetic (segments <= 65536)
__host__ __device__ __forceinline__ unsigned segment_start(unsigned s, unsigned units, unsigned segments) {
  const unsigned q = units / segments, rm = units - q * segments;
  return s * q + s * rm / segments;
}

template <bool AK>
__device__ __forceinline__ unsigned out_row(unsigned wm, unsigned t, unsigned l32) {
  return wm * 128 + (AK ? 32 * t + l32 : 4 * l32 + t);
}

// A wavefront's 128 x 64 sums over k-tiles kt0 .. kt1 - 1 of a tile once more, by the fp32 instruction, 32 x 32 at a time:
// to the slot of a partial tile (this thread's first element of it, past the L2), or, with the parts of segments s0 ..
// s1 - 1 (slot: of the first segment), through the epilogue to C.
template <bool AK, bool BKM>
__device__ __forceinline__ void redo_sums(const WideArgs& g, unsigned tile, unsigned kt0, unsigned kt1, bool part, float* slot,
                                          unsigned s0, unsigned s1) {
  const unsigned wm = (threadIdx.x >> 6) & 1, wn = threadIdx.x >> 7, l32 = threadIdx.x & 31, lhi = (threadIdx.x >> 5) & 1;
  const unsigned m0 = (tile % g.tiles_m) * kWT, n0 = (tile / g.tiles_m) * kWT;
#pragma unroll 1
  for (unsigned x = 0; x < 8; ++x) {
    const unsigned u = x / 4, t = x % 4, m = m0 + out_row<AK>(wm, t, l32);
    const unsigned mc = min(m, g.M - 1), nc = min(n0 + out_column<BKM>(wn, u, l32), g.N - 1);
    sums16 s = {};
    add_products_fp32<AK, BKM>(s, g.A + (AK ? size_t(mc) * g.lda : mc), g.lda, g.B + (BKM ? size_t(nc) * g.ldb : nc), g.ldb,
                               kt0 * kWK, kt1 * kWK);
    typedef __attribute__((address_space(1))) float* global_float;
    global_float at = (global_float)(slot + size_t(16 * u) * (4 * kWideThreads) + t);
#pragma unroll
    for (unsigned r = 0; r < 16; ++r, at += 4 * kWideThreads) {
      asm volatile("" : "+v"(at));  // addresses one by one
      float v = s[r];
      if (part) {
        __hip_atomic_store(at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        continue;
      }
      for (unsigned s2 = s0; s2 < s1; ++s2)
        v += __hip_atomic_load(at + size_t(s2) * kSlotFloats, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      const unsigned n = n0 + out_column<BKM>(wn, u, 8 * (r / 4) + 4 * lhi + r % 4);
      if (m >= g.M || n >= g.N) continue;
      float* p = g.C + m + size_t(n) * g.M;
      if (g.bias != nullptr) v += g.bias[m];
      else if (g.beta != 0.f) v += g.beta * *p;
      *p = v;
    }
  }
}

// AK: A(m,k) = A[k + m*lda], else A[m + k*lda].  BKM: B(k,n) = B[k + n*ldb], else B[n + k*ldb].
template <bool AK, bool BKM>
__global__ __launch_bounds__(kWideThreads, 1) void gemm_wide_kernel(WideArgs g) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = w & 1, wn = w >> 1;
  const int l32 = lane & 31, lhi = lane >> 5;
  const unsigned frag = lhi * 4096 + (l32 ^ (4 * lhi)) * 16;
  // This lane's fragments of A and B, and its first row (below).  Opaque: taken apart into what they share and constants,
  // they would put the second stage out of reach again.
  unsigned oa = frag + wm * (AK ? 128 : 32) * 16;
  unsigned ob = kOperandBytes + frag + (BKM ? wn * 64 : (wn & 1) * 128 + (wn >> 1) * 32) * 16;
  constexpr unsigned ta = AK ? 512 : 1024, tb = BKM ? 512 : 1024;  // bytes between a wave's row (column) tiles
  const unsigned nt = g.nt;

  // this block's segment of the unit sequence (tile-major, k-tiles ascending inside a tile).  Segments are handed out
  // in descending order of block index: the blocks that a block may have to wait for (below) have lower indices and
  // were therefore dispatched before it.
  const unsigned segments = gridDim.x, seg = segments - 1 - blockIdx.x;
  const unsigned u0 = segment_start(seg, g.units, segments), u1 = segment_start(seg + 1, g.units, segments);
  if (u0 == u1) return;

  // Loads run three steps ahead of the product, straight across tile boundaries, and repeat the segment's last step at
  // its end.  load_at: the next step to load; load_p: its first element; load_end: the end of its tile.
  const bool stage_b = w >= 4;
  const unsigned ld = stage_b ? g.ldb : g.lda;
  const float* const operand = stage_b ? g.B : g.A;
  const bool kmajor = AK == BKM ? AK : stage_b ? BKM : AK;
  const size_t step = kmajor ? 16 : size_t(16) * ld;
  unsigned ow = (stage_b ? kOperandBytes : 0u) + write_offset(kmajor);
  asm volatile("" : "+v"(oa), "+v"(ob), "+v"(ow));
  const unsigned last = 2 * u1 - 1;
  unsigned load_at = 2 * u0, load_end, off[4];
  const float* load_p;
#define DYHIP_WIDE_TILE(k0)                                                                      \
  {                                                                                              \
    const unsigned t_ = load_at / (2 * nt);                                                      \
    const unsigned mn0_ = (stage_b ? t_ / g.tiles_m : t_ % g.tiles_m) * kWT;                     \
    load_offsets(kmajor, off, ld, mn0_, stage_b ? g.N : g.M);                                    \
    load_p = operand + (kmajor ? size_t(mn0_) * ld : size_t(mn0_)) + (k0) * step;                \
    load_end = (t_ + 1) * 2 * nt;                                                                \
  }
  DYHIP_WIDE_TILE(load_at % (2 * nt))
  float4 raw[4];
#define DYHIP_WIDE_LOAD                                                                          \
  {                                                                                              \
    _Pragma("unroll") for (int j_ = 0; j_ < 4; ++j_) raw[j_] =                                   \
        *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(load_p) + off[j_]);                                      \
    const unsigned more_ = load_at < last ? 1u : 0u;                                             \
    load_at += more_;                                                                            \
    load_p += more_ * step;                                                                      \
  }
#define DYHIP_WIDE_LOAD_NEXT_TILE if (load_at == load_end) DYHIP_WIDE_TILE(0u)
#define DYHIP_WIDE_SPLIT(j, stage) split_row(kmajor, raw, (j), lds + ow + (stage) * kStageBytes);
  // Fragments (h, m, l) of one of the wave's row tiles and of both of its column tiles.  A step's products go tile by tile,
  // x = 2 t + u; a plane of the row tile is fetched for the next one where its last product has been issued.
  bf16x8 fa[3], fb[2][3];
#define DYHIP_WIDE_READ_A(p, t, stage) fa[p] = read_frag(lds + oa + (stage) * kStageBytes + (p) * kPlaneBytes + (t) * ta);
#define DYHIP_WIDE_READ_B(u, stage) \
  _Pragma("unroll") for (int p_ = 0; p_ < 3; ++p_) fb[u][p_] = read_frag(lds + ob + (stage) * kStageBytes + p_ * kPlaneBytes + (u) * tb);
#define DYHIP_WIDE_MMA(x, pa, pb) \
  sum[(x) % 2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[(x) % 2][pb], fa[pa], sum[(x) % 2], 0, 0, 0);
#define DYHIP_WIDE_CHAIN(x)                              \
  _Pragma("unroll") for (int r_ = 0; r_ < 16; ++r_) sum[(x) % 2][r_] = 0.f; \
  DYHIP_WIDE_MMA(x, 2, 0) DYHIP_WIDE_MMA(x, 1, 1) DYHIP_WIDE_MMA(x, 1, 0) DYHIP_WIDE_MMA(x, 0, 2) DYHIP_WIDE_MMA(x, 0, 1) \
  DYHIP_WIDE_MMA(x, 0, 0)
// the second tile of a pair, and the next row tile t of a stage behind it
#define DYHIP_WIDE_CHAIN_NEXT(x, t, stage)                              \
  _Pragma("unroll") for (int r_ = 0; r_ < 16; ++r_) sum[(x) % 2][r_] = 0.f; \
  DYHIP_WIDE_MMA(x, 2, 0) DYHIP_WIDE_READ_A(2, t, stage) DYHIP_WIDE_MMA(x, 1, 1) DYHIP_WIDE_MMA(x, 1, 0) \
  DYHIP_WIDE_READ_A(1, t, stage) DYHIP_WIDE_MMA(x, 0, 2) DYHIP_WIDE_MMA(x, 0, 1) DYHIP_WIDE_MMA(x, 0, 0) \
  DYHIP_WIDE_READ_A(0, t, stage)
#define DYHIP_WIDE_ADD(x) _Pragma("unroll") for (int r_ = 0; r_ < 16; ++r_) acc[(x) % 2][(x) / 2][r_] += sum[(x) % 2][r_];
// (keeps the additions where they are: the compiler would move them out of the loop, and spill the sums)
#define DYHIP_WIDE_PIN(x) _Pragma("unroll") for (int r_ = 0; r_ < 16; r_ += 8) {                                            \
    float* a_ = acc[(x) % 2][(x) / 2] + r_;                                                                               \
    asm volatile("" : "+v"(a_[0]), "+v"(a_[1]), "+v"(a_[2]), "+v"(a_[3]), "+v"(a_[4]), "+v"(a_[5]), "+v"(a_[6]), "+v"(a_[7])); \
  }
// n times: one MFMA, then so many LDS reads, vector instructions, LDS writes and global loads
#define DYHIP_WIDE_MIX(id, n, valu, rd, wr, ld_)                               \
  _Pragma("unroll") for (int x_ = 0; x_ < (n); ++x_) {                     \
    __builtin_amdgcn_sched_group_barrier(0x008, 1, id);                     \
    if (rd) __builtin_amdgcn_sched_group_barrier(0x100, rd, id);            \
    if (valu) __builtin_amdgcn_sched_group_barrier(0x002, valu, id);        \
    if (wr) __builtin_amdgcn_sched_group_barrier(0x200, wr, id);            \
    if (ld_) __builtin_amdgcn_sched_group_barrier(0x020, ld_, id);          \
  }
#define DYHIP_WIDE_FENCE __builtin_amdgcn_sched_barrier(0);

  for (unsigned pos = u0; pos < u1;) {
    const unsigned tile = pos / nt, ub = tile * nt, kt0 = pos - ub, kt1 = min(nt, u1 - ub);
    if (pos == u0) {
      DYHIP_WIDE_LOAD
#pragma unroll
      for (int j = 0; j < 4; ++j) DYHIP_WIDE_SPLIT(j, 0)
      DYHIP_WIDE_LOAD
#pragma unroll
      for (int j = 0; j < 4; ++j) DYHIP_WIDE_SPLIT(j, 1)
      DYHIP_WIDE_LOAD_NEXT_TILE
      DYHIP_WIDE_LOAD
      DYHIP_WIDE_LOAD_NEXT_TILE
      __syncthreads();
      DYHIP_WIDE_READ_A(2, 0, 0)
      DYHIP_WIDE_READ_A(1, 0, 0)
      DYHIP_WIDE_READ_A(0, 0, 0)
      DYHIP_WIDE_READ_B(0, 0)
    }
    pos += kt1 - kt0;
    float acc[2][4][16];
    floatx16 sum[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[u][t][r] = sum[u][r] = 0.f;
    }
    for (unsigned i = kt0; i < kt1; ++i) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        DYHIP_WIDE_READ_B(1, e)
        DYHIP_WIDE_CHAIN(0)
        DYHIP_WIDE_ADD(7)  // of the step before
        DYHIP_WIDE_MIX(0, 2, 0, 2, 0, 0)
        DYHIP_WIDE_MIX(0, 4, 4, 0, 0, 0)
        DYHIP_WIDE_PIN(7)
        DYHIP_WIDE_FENCE
        DYHIP_WIDE_CHAIN_NEXT(1, 1, e)
        DYHIP_WIDE_ADD(0)
        DYHIP_WIDE_MIX(1, 1, 0, 0, 0, 0)
        DYHIP_WIDE_MIX(1, 1, 0, 1, 0, 0)
        DYHIP_WIDE_MIX(1, 1, 5, 0, 0, 0)
        DYHIP_WIDE_MIX(1, 1, 5, 1, 0, 0)
        DYHIP_WIDE_MIX(1, 2, 3, 0, 0, 0)
        DYHIP_WIDE_PIN(0)
        DYHIP_WIDE_FENCE
        DYHIP_WIDE_CHAIN(2)
        DYHIP_WIDE_ADD(1)
        DYHIP_WIDE_MIX(2, 2, 0, 0, 0, 0)
        DYHIP_WIDE_MIX(2, 4, 4, 0, 0, 0)
        DYHIP_WIDE_PIN(1)
        DYHIP_WIDE_FENCE
        DYHIP_WIDE_CHAIN_NEXT(3, 2, e)
        DYHIP_WIDE_ADD(2)
        DYHIP_WIDE_MIX(3, 1, 0, 0, 0, 0)
        DYHIP_WIDE_MIX(3, 1, 0, 1, 0, 0)
        DYHIP_WIDE_MIX(3, 1, 5, 0, 0, 0)
        DYHIP_WIDE_MIX(3, 1, 5, 1, 0, 0)
        DYHIP_WIDE_MIX(3, 2, 3, 0, 0, 0)
        DYHIP_WIDE_PIN(2)
        DYHIP_WIDE_FENCE
        DYHIP_WIDE_CHAIN(4)
        DYHIP_WIDE_ADD(3)
        DYHIP_WIDE_MIX(4, 2, 0, 0, 0, 0)
        DYHIP_WIDE_MIX(4, 4, 4, 0, 0, 0)
        DYHIP_WIDE_PIN(3)
        DYHIP_WIDE_FENCE
        DYHIP_WIDE_CHAIN_NEXT(5, 3, e)
        DYHIP_WIDE_ADD(4)
        DYHIP_WIDE_MIX(5, 1, 0, 0, 0, 0)
        DYHIP_WIDE_MIX(5, 1, 0, 1, 0, 0)
        DYHIP_WIDE_MIX(5, 1, 5, 0, 0, 0)
        DYHIP_WIDE_MIX(5, 1, 5, 1, 0, 0)
        DYHIP_WIDE_MIX(5, 2, 3, 0, 0, 0)
        DYHIP_WIDE_PIN(4)
        DYHIP_WIDE_FENCE
        // every wave's part of the next step is in LDS, and every wave holds its last fragments of this one, whose stage
        // is refilled below two steps ahead
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        DYHIP_WIDE_FENCE
        DYHIP_WIDE_CHAIN(6)
        DYHIP_WIDE_ADD(5)
        DYHIP_WIDE_SPLIT(0, e)
        DYHIP_WIDE_SPLIT(1, e)
        DYHIP_WIDE_MIX(6, 2, 6, 0, 0, 0)
        DYHIP_WIDE_MIX(6, 4, 10, 0, 2, 0)
        DYHIP_WIDE_PIN(5)
        DYHIP_WIDE_FENCE
        DYHIP_WIDE_READ_B(0, e ^ 1)
        DYHIP_WIDE_CHAIN_NEXT(7, 0, e ^ 1)
        DYHIP_WIDE_ADD(6)
        DYHIP_WIDE_SPLIT(2, e)
        DYHIP_WIDE_SPLIT(3, e)
        DYHIP_WIDE_LOAD
        DYHIP_WIDE_MIX(7, 1, 6, 3, 0, 0)
        DYHIP_WIDE_MIX(7, 1, 6, 1, 0, 0)
        DYHIP_WIDE_MIX(7, 1, 10, 0, 2, 0)
        DYHIP_WIDE_MIX(7, 1, 10, 1, 2, 0)
        DYHIP_WIDE_MIX(7, 2, 10, 0, 1, 2)
        DYHIP_WIDE_PIN(6)
        DYHIP_WIDE_FENCE
        DYHIP_WIDE_LOAD_NEXT_TILE
      }
    }
    DYHIP_WIDE_ADD(7)
    // Sums to scale, and whether one is not finite: then this wavefront forms its part of them again where it would store
    // them (redo_sums).
    bool again;
    {
      float z = 0.f;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            acc[u][t][r] *= kSplitOut;
            z = fmaf(acc[u][t][r], 0.f, z);
          }
      again = __any(!(z == 0.f));
    }

    // the thread index as the compiler cannot see through: the addresses below are formed here, after the loop,
    // instead of being computed ahead of it and parked in scratch memory
    unsigned tid_e = threadIdx.x;
    asm volatile("" : "+v"(tid_e));
    // acc[u][t][r] of lane l: m = AK ? 32 t + l%32 : 4 (l%32) + t (+ 128 wm),
    // n = BKM ? 32 u + i : 2 i + u (+ 64 wn) with i = 8 (r/4) + 4 (l/32) + r%4.
    // A partial tile is stored as [u][r][thread][t]: one 128-bit access per thread and (u, r), whoever reads it.
    // Not the whole tile, and not this block's to finish: it goes to a slot, past the L2 for a block on another one.
    const bool part = kt0 > 0 || (kt1 < nt && !g.finish_in_kernel);
    float* slot = g.slots + 4 * tid_e;
    if (part) slot += size_t(g.finish_in_kernel ? seg : 2 * seg + (tile == u0 / nt ? 0 : 1)) * kSlotFloats;
    // This block holds the tile's first k-tiles (or all of them) and finishes the tile.  The segments that start inside
    // the tile computed their partial tiles first thing, long ago by now; the wait is bounded all the same, and a wait
    // that gives up is counted for the host to report.  Partial tiles are added in segment order.
    unsigned s_end = seg + 1;
    if (!part && kt1 < nt) {
      while (s_end < segments && segment_start(s_end, g.units, segments) < ub + nt) ++s_end;
      if (tid_e == 0) {
        for (unsigned s2 = seg + 1; s2 < s_end; ++s2) {
          unsigned spins = 0;
          while (__hip_atomic_load(g.flags + s2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u) {
            if (spins++ >= g.spin_limit) {
              atomicAdd(g.flags + kGemmFlagWords - 1, 1u);
              break;
            }
            __builtin_amdgcn_s_sleep(32);
          }
          __hip_atomic_store(g.flags + s2, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
        }
      }
      __syncthreads();
    }
    if (__builtin_expect(again, 0)) {
      redo_sums<AK, BKM>(g, tile, kt0, kt1, part, slot, seg + 1, s_end);
    } else if (part) {
      if (g.finish_in_kernel) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            store_through(slot + size_t(u * 16 + r) * (4 * kWideThreads), acc[u][0][r], acc[u][1][r], acc[u][2][r],
                          acc[u][3][r]);
      } else {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            *reinterpret_cast<float4*>(slot + size_t(u * 16 + r) * (4 * kWideThreads)) =
                make_float4(acc[u][0][r], acc[u][1][r], acc[u][2][r], acc[u][3][r]);
      }
    }
    if (part) {
      if (g.finish_in_kernel) {  // the segment's flag goes up once memory has acknowledged every store
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (tid_e == 0 && g.raise_flags) __hip_atomic_store(g.flags + seg, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      continue;
    }
    if (again) continue;
    const unsigned lane_e = tid_e & 63, wm_e = (tid_e >> 6) & 1, wn_e = tid_e >> 7, l32_e = lane_e & 31, lhi_e = lane_e >> 5;
    const unsigned m0 = (tile % g.tiles_m) * kWT, n0 = (tile / g.tiles_m) * kWT;
    float* out = g.C + m0 + size_t(n0) * g.M;
    const unsigned mlim = g.M - m0, nlim = g.N - n0;
    const float beta = g.bias == nullptr ? g.beta : 0.f;
    const bool add_bias = g.bias != nullptr;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r0 = 0; r0 < 16; r0 += 8) {
        float4 v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = make_float4(acc[u][0][r0 + q], acc[u][1][r0 + q], acc[u][2][r0 + q], acc[u][3][r0 + q]);
        for (unsigned s2 = seg + 1; s2 < s_end; ++s2) {  // eight loads in flight
          const float* slot = g.slots + size_t(s2) * kSlotFloats + 4 * tid_e + size_t(u * 16 + r0) * (4 * kWideThreads);
          wide_v4 o[8];
#pragma unroll
          for (int q = 0; q < 8; ++q) o[q] = load_through(slot + size_t(q) * (4 * kWideThreads));
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            v[q].x += o[q][0]; v[q].y += o[q][1]; v[q].z += o[q][2]; v[q].w += o[q][3];
          }
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const int r = r0 + q;
          const unsigned n = out_column<BKM>(wn_e, u, 8 * (r / 4) + 4 * lhi_e + (r % 4));
          if (n >= nlim) continue;
          if (!AK) {
            const unsigned m = out_row<AK>(wm_e, 0, l32_e);
            if (m >= mlim) continue;
            float* p = out + m + size_t(n) * g.M;
            float4 x = v[q];
            if (add_bias) {
              const float4 o = *reinterpret_cast<const float4*>(g.bias + m0 + m);
              x.x += o.x; x.y += o.y; x.z += o.z; x.w += o.w;
            } else if (beta != 0.f) {
              const float4 o = *reinterpret_cast<const float4*>(p);
              x.x += beta * o.x; x.y += beta * o.y; x.z += beta * o.z; x.w += beta * o.w;
            }
            *reinterpret_cast<float4*>(p) = x;
          } else {
            const float xs[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              const unsigned m = out_row<AK>(wm_e, t, l32_e);
              if (m >= mlim) continue;
              float* p = out + m + size_t(n) * g.M;
              float x = xs[t];
              if (add_bias) x += g.bias[m0 + m];
              else if (beta != 0.f) x += beta * *p;
              *p = x;
            }
          }
        }
      }
  }
#undef DYHIP_WIDE_TILE
#undef DYHIP_WIDE_LOAD
#undef DYHIP_WIDE_LOAD_NEXT_TILE
#undef DYHIP_WIDE_SPLIT
#undef DYHIP_WIDE_READ_A
#undef DYHIP_WIDE_READ_B
#undef DYHIP_WIDE_MMA
#undef DYHIP_WIDE_CHAIN
#undef DYHIP_WIDE_CHAIN_NEXT
#undef DYHIP_WIDE_PIN
#undef DYHIP_WIDE_ADD
#undef DYHIP_WIDE_MIX
#undef DYHIP_WIDE_FENCE
}

// Second kernel for products whose tiles span several segments each (fewer tiles than CUs, or little more): C tile =
// epilogue(sum of the tile's partial tiles in segment order).  Block (x, y) takes tile x and two of its 32 (u, r)
// groups, its threads standing for the threads of the main kernel (a partial tile is stored in their order).
template <bool AK, bool BKM>
__global__ __launch_bounds__(kWideThreads) void gemm_wide_fixup_kernel(WideArgs g, unsigned segments) {
  const unsigned nt = g.nt, tile = blockIdx.x, ub = tile * nt;
  // segments that hold k-tiles of this tile: s_lo holds its first, s_hi its last
  unsigned s_lo = min(ub / (g.units / segments), segments - 1);
  while (s_lo + 1 < segments && segment_start(s_lo + 1, g.units, segments) <= ub) ++s_lo;
  while (segment_start(s_lo, g.units, segments) > ub) --s_lo;
  unsigned s_hi = s_lo;
  while (s_hi + 1 < segments && segment_start(s_hi + 1, g.units, segments) < ub + nt) ++s_hi;
  if (s_lo == s_hi) return;  // one block had the whole tile and wrote it itself
  const unsigned tid = threadIdx.x, lane = tid & 63, wm = (tid >> 6) & 1, wn = tid >> 7, l32 = lane & 31, lhi = lane >> 5;
  const unsigned m0 = (tile % g.tiles_m) * kWT, n0 = (tile / g.tiles_m) * kWT;
  float* out = g.C + m0 + size_t(n0) * g.M;
  const unsigned mlim = g.M - m0, nlim = g.N - n0;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const unsigned ur = blockIdx.y * 2 + j, u = ur / 16, r = ur % 16;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    for (unsigned s2 = s_lo; s2 <= s_hi; ++s2) {
      // the tile is the first item of every segment but the one that holds its first k-tiles (unless that segment
      // starts with it)
      const unsigned first_tile = segment_start(s2, g.units, segments) / nt;
      const float4 o = *reinterpret_cast<const float4*>(g.slots + size_t(2 * s2 + (first_tile == tile ? 0 : 1)) * kSlotFloats +
                                                        size_t(ur) * (4 * kWideThreads) + 4 * tid);
      v.x += o.x; v.y += o.y; v.z += o.z; v.w += o.w;
    }
    const unsigned n = out_column<BKM>(wn, u, 8 * (r / 4) + 4 * lhi + (r % 4));
    if (n >= nlim) continue;
    if (!AK) {
      const unsigned m = out_row<AK>(wm, 0, l32);
      if (m >= mlim) continue;
      float* p = out + m + size_t(n) * g.M;
      if (g.bias != nullptr) {
        const float4 o = *reinterpret_cast<const float4*>(g.bias + m0 + m);
        v.x += o.x; v.y += o.y; v.z += o.z; v.w += o.w;
      } else if (g.beta != 0.f) {
        const float4 o = *reinterpret_cast<const float4*>(p);
        v.x += g.beta * o.x; v.y += g.beta * o.y; v.z += g.beta * o.z; v.w += g.beta * o.w;
      }
      *reinterpret_cast<float4*>(p) = v;
    } else {
      const float xs[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const unsigned m = out_row<AK>(wm, t, l32);
        if (m >= mlim) continue;
        float* p = out + m + size_t(n) * g.M;
        float x = xs[t];
        if (g.bias != nullptr) x += g.bias[m0 + m];
        else if (g.beta != 0.f) x += g.beta * *p;
        *p = x;
      }
    }
  }
}

// ---- shallow products: C[M x N] = beta*C + A[M x K] * B[N x K]^T with K <= 128 (the weight gradient of one timestep:
// K is the batch) -----------------------------------------------------------------------------------------------
// With four k-tiles a pipelined loop never fills: set-up, the exposed latency of each k-tile and the read-modify-write
// of C add up to more than the MFMAs.  Here a 512-thread block owns a 128 x 128 tile and fetches BOTH operand tiles
// whole (2 x 64 KiB, straight into LDS) plus its part of the old C in one burst at the start, so the block pays one
// memory latency, then 128 MFMAs per wave, then stores.  Wave w (2 x 4 over the tile) owns 64 m x 32 n.
// LDS: [half h of the depth][wave w][A 4 KiB][B 4 KiB]; the 1 KiB chunk u of wave w in half h holds rows
// k = 64h + 8w + 2u + {0, 1} of the operand tile (128 floats each), so that each half is one M0 window per wave.
struct ShallowArgs {
  const float* A;
  const float* B;
  float* C;
  unsigned lda, ldb;
  unsigned M, N, K;
  unsigned tiles_m;
  float beta;
};

constexpr size_t kShallowLdsBytes = sizeof(float) * 2 * kStageFloats;

__global__ __launch_bounds__(kWideThreads, 1) void gemm_shallow_nt_kernel(ShallowArgs g) {
  extern __shared__ __attribute__((aligned(16))) float lds_f[];
  const unsigned lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const unsigned wm = w & 1, wn = w >> 1, l32 = lane & 31, lhi = lane >> 5;
  const unsigned tm = blockIdx.x % g.tiles_m, tn = blockIdx.x / g.tiles_m;
  const unsigned m0 = tm * 128, n0 = tn * 128;

  // old C of this lane's outputs: m = m0 + 64 wm + 2 l32 + {0, 1}, n = n0 + 32 wn + i, i = 8 (r/4) + 4 lhi + r%4
  const unsigned m = m0 + wm * 64 + 2 * l32;
  fvec2 cold[16];
  if (g.beta != 0.f) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const unsigned n = n0 + wn * 32 + 8 * (r / 4) + 4 * lhi + (r % 4);
      cold[r] = fvec2{0.f, 0.f};
      if (m < g.M && n < g.N) cold[r] = *reinterpret_cast<const fvec2*>(g.C + m + size_t(n) * g.M);
    }
  }
  // operand tiles: rows past the depth are not fetched (nor read), groups of four past the edge are clamped
  unsigned am = m0 + 4 * l32, bn = n0 + 4 * l32;
  am = am < g.M ? am : g.M - 4;
  bn = bn < g.N ? bn : g.N - 4;
#define DYHIP_SHALLOW_LOADS(h)                                                                                     \
  {                                                                                                                \
    float* window = lds_f + (h) * kStageFloats + w * 2048 + 1024;                                                    \
    const unsigned k0 = 64 * (h) + 8 * w + lhi;                                                                    \
    const float* pa = g.A + am + size_t(k0) * g.lda;                                                               \
    const float* pb = g.B + bn + size_t(k0) * g.ldb;                                                               \
    if (64 * (h) + 8 * w + 0 < g.K) {                                                                              \
      __builtin_amdgcn_global_load_lds((global_ptr_t)(pa + 1024), (lds_ptr_t)window, 16, -4096, 0);                \
      __builtin_amdgcn_global_load_lds((global_ptr_t)(pb), (lds_ptr_t)window, 16, 0, 0);                           \
    }                                                                                                              \
    if (64 * (h) + 8 * w + 2 < g.K) {                                                                              \
      __builtin_amdgcn_global_load_lds((global_ptr_t)(pa + 2 * size_t(g.lda) + 768), (lds_ptr_t)window, 16, -3072, 0); \
      __builtin_amdgcn_global_load_lds((global_ptr_t)(pb + 2 * size_t(g.ldb) - 256), (lds_ptr_t)window, 16, 1024, 0);  \
    }                                                                                                              \
    if (64 * (h) + 8 * w + 4 < g.K) {                                                                              \
      __builtin_amdgcn_global_load_lds((global_ptr_t)(pa + 4 * size_t(g.lda) + 512), (lds_ptr_t)window, 16, -2048, 0); \
      __builtin_amdgcn_global_load_lds((global_ptr_t)(pb + 4 * size_t(g.ldb) - 512), (lds_ptr_t)window, 16, 2048, 0);  \
    }                                                                                                              \
    if (64 * (h) + 8 * w + 6 < g.K) {                                                                              \
      __builtin_amdgcn_global_load_lds((global_ptr_t)(pa + 6 * size_t(g.lda) + 256), (lds_ptr_t)window, 16, -1024, 0); \
      __builtin_amdgcn_global_load_lds((global_ptr_t)(pb + 6 * size_t(g.ldb) - 768), (lds_ptr_t)window, 16, 3072, 0);  \
    }                                                                                                              \
  }
  DYHIP_SHALLOW_LOADS(0)
  DYHIP_SHALLOW_LOADS(1)
#undef DYHIP_SHALLOW_LOADS

  floatx16 acc[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
  // group kg (8 k) of half h: step s of lane half lhi is row k = 8 kg + 4 lhi + s, i.e. chunk 2 lhi + s/2 of wave kg%8
  const float* la = lds_f + lhi * 512 + wm * 64 + 2 * l32;
  const float* lb = lds_f + 1024 + lhi * 512 + wn * 32 + l32;
  const unsigned groups = g.K / 8;
  fvec2 a[2][4];
  float b[2][4];
#define DYHIP_SHALLOW_READ(buf, kg)                                                        \
  _Pragma("unroll") for (int s = 0; s < 4; ++s) {                                          \
    const unsigned o = ((kg) / 8) * kStageFloats + ((kg) % 8) * 2048 + (s / 2) * 256 + (s % 2) * 128; \
    a[buf][s] = *reinterpret_cast<const fvec2*>(la + o);                                   \
    b[buf][s] = lb[o];                                                                     \
  }
#define DYHIP_SHALLOW_MMA(buf)                                                                          \
  __builtin_amdgcn_sched_barrier(0);                                                                    \
  _Pragma("unroll") for (int s = 0; s < 4; ++s) {                                                       \
    acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[buf][s], a[buf][s][0], acc[0], 0, 0, 0);            \
    acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[buf][s], a[buf][s][1], acc[1], 0, 0, 0);            \
  }                                                                                                     \
  __builtin_amdgcn_sched_barrier(0);
  // the first half of the depth can start while the second is still on its way (only when the whole second half
  // was asked for, so that every wave has the same number of loads in flight)
  const bool two_phase = g.K == 128;
  if (two_phase) __builtin_amdgcn_s_waitcnt(0x0F78);  // vmcnt(8): the eight loads of the second half may be in flight
  else __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();
  const unsigned first = two_phase ? 8 : groups;
  DYHIP_SHALLOW_READ(0, 0u)
  for (unsigned kg = 0; kg < first; kg += 2) {
    const unsigned k1 = kg + 1 < first ? kg + 1 : kg, k2 = kg + 2 < first ? kg + 2 : kg;
    DYHIP_SHALLOW_READ(1, k1)
    DYHIP_SHALLOW_MMA(0)
    DYHIP_SHALLOW_READ(0, k2)
    if (kg + 1 < first) { DYHIP_SHALLOW_MMA(1) }
  }
  if (two_phase) {
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    DYHIP_SHALLOW_READ(0, 8u)
    for (unsigned kg = 8; kg < 16; kg += 2) {
      const unsigned k2 = kg + 2 < 16 ? kg + 2 : kg;
      DYHIP_SHALLOW_READ(1, kg + 1)
      DYHIP_SHALLOW_MMA(0)
      DYHIP_SHALLOW_READ(0, k2)
      DYHIP_SHALLOW_MMA(1)
    }
  }
#undef DYHIP_SHALLOW_READ
#undef DYHIP_SHALLOW_MMA
  if (m >= g.M) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const unsigned n = n0 + wn * 32 + 8 * (r / 4) + 4 * lhi + (r % 4);
    if (n >= g.N) continue;
    fvec2 v = fvec2{acc[0][r], acc[1][r]};
    if (g.beta != 0.f) v += g.beta * cold[r];
    *reinterpret_cast<fvec2*>(g.C + m + size_t(n) * g.M) = v;
  }
}

template <bool AK, bool BKM>
int launch_wide(dyhip_device* dev, const WideArgs& g, unsigned blocks, unsigned bit) {
  const void* fn = reinterpret_cast<const void*>(&gemm_wide_kernel<AK, BKM>);
  if ((dev->wide_gemm_ready & (1u << bit)) == 0) {  // 96 KiB of LDS need the opt-in, once per device
    DYHIP_CHECK_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, int(kWideLdsBytes)));
    dev->wide_gemm_ready |= 1u << bit;
  }
  hipLaunchKernelGGL((gemm_wide_kernel<AK, BKM>), dim3(blocks), dim3(kWideThreads), kWideLdsBytes, dev->stream, g);
  return DYHIP_OK;
}

}  // namespace

// How the k-tiles are dealt to the blocks.  ok = false: leave the problem to the smaller tiles.
struct WidePlan {
  bool ok;
  bool finish_in_kernel;  // segments at least a tile long: a tile is cut at most once, and finished inside the kernel
  unsigned tiles_m, tiles, nt, units, segments;
};

static WidePlan plan_wide(const dyhip_device* dev, size_t M, size_t N, size_t K32) {
  const unsigned cus = dev->num_cus > 0 ? unsigned(dev->num_cus) : 256;
  WidePlan p{};
  p.tiles_m = unsigned(cdiv<size_t>(M, kWT));
  p.nt = unsigned(K32 / kWK);
  const size_t tiles = size_t(p.tiles_m) * cdiv<size_t>(N, kWT), units = tiles * p.nt;
  p.tiles = unsigned(tiles);
  p.units = unsigned(units);
  p.segments = cus;
  const size_t per = units / cus;
  p.finish_in_kernel = per >= p.nt;
  // Measured against 128 x 128 tiles: a block's set-up, its share of partial tiles and of the second kernel cost
  // about three k-tiles, so a problem of fewer tiles than CUs (nothing but cut tiles) needs long segments.
  p.ok = units < (size_t(1) << 31) && (p.finish_in_kernel ? p.nt >= 8 : per >= 16);
  return p;
}

bool gemm_wide_eligible(const dyhip_device* dev, bool a_kmajor, bool b_kmajor, size_t M, size_t N, size_t K,
                        const float* A, size_t lda, const float* B, size_t ldb, const float* C) {
  const size_t K32 = K / kWK * kWK;
  if (K32 < 256 || M < 192 || N < 192 || dev->max_lds_per_block < kWideLdsBytes) return false;
  if (!aligned16(A) || !aligned16(B) || !aligned16(C) || lda % 4 != 0 || ldb % 4 != 0) return false;
  if ((!a_kmajor && M % 4 != 0) || (!b_kmajor && N % 4 != 0)) return false;
  // 32-bit element offsets inside the kernel
  const size_t span_a = a_kmajor ? M * lda : K * lda, span_b = b_kmajor ? N * ldb : K * ldb;
  if (span_a >= (size_t(1) << 31) || span_b >= (size_t(1) << 31) || M * N >= (size_t(1) << 31)) return false;
  const size_t tiles = cdiv<size_t>(M, kWT) * cdiv<size_t>(N, kWT);
  const size_t cus = dev->num_cus > 0 ? size_t(dev->num_cus) : 256;
  // and 32-bit byte offsets from a tile's first element
  if (lda >= (size_t(1) << 21) || ldb >= (size_t(1) << 21)) return false;
  // edge tiles compute whole 256 x 256 tiles: ragged shapes stay with the smaller tiles
  if (double(M) * double(N) < 0.8 * double(tiles) * double(kSlotFloats)) return false;
  if (dev->gemm_ws == nullptr || dev->gemm_flags == nullptr || dev->gemm_ws_bytes < (2 * cus) * kSlotFloats * sizeof(float) ||
      cus + 1 > size_t(kGemmFlagWords))
    return false;
  return plan_wide(dev, M, N, K32).ok;
}

size_t gemm_wide_whole_rounds_columns(const dyhip_device* dev, bool a_kmajor, bool b_kmajor, size_t M, size_t N, size_t K,
                                      const float* A, size_t lda, const float* B, size_t ldb, const float* C) {
  const size_t cus = dev->num_cus > 0 ? size_t(dev->num_cus) : 256;
  const size_t tiles_m = cdiv<size_t>(M, kWT), tiles = tiles_m * cdiv<size_t>(N, kWT);
  const size_t direct = tiles / cus * cus;
  // From a depth of 768 on one sequence of k-tiles over all tiles is as fast or faster (l*r, apart against one sequence:
  // 4096 x 4480 K = 512 121 against 135 us, 768 176 and 176, 1024 222 against 219; 8192 x 2304 K = 512 130 against 137,
  // 768 182 against 179, 1024 234 against 221, 2048 441 against 407).
  if (K >= 768 || direct == 0 || direct == tiles || direct % tiles_m != 0 || tiles - direct > cus / 4) return 0;
  const size_t cols = direct / tiles_m * kWT;
  return cols < N && gemm_wide_eligible(dev, a_kmajor, b_kmajor, M, cols, K, A, lda, B, ldb, C) ? cols : 0;
}

int gemm_wide_run(dyhip_device* dev, bool a_kmajor, bool b_kmajor, size_t M, size_t N, size_t K32, const float* A,
                  size_t lda, const float* B, size_t ldb, float* C, float beta, const float* bias) {
  const WidePlan p = plan_wide(dev, M, N, K32);
  WideArgs g;
  g.A = A;
  g.B = B;
  g.C = C;
  g.bias = bias;
  g.slots = static_cast<float*>(dev->gemm_ws);
  g.flags = dev->gemm_flags;
  g.lda = unsigned(lda);
  g.ldb = unsigned(ldb);
  g.M = unsigned(M);
  g.N = unsigned(N);
  g.nt = p.nt;
  g.tiles_m = p.tiles_m;
  g.units = p.units;
  g.finish_in_kernel = p.finish_in_kernel ? 1 : 0;
  g.spin_limit = dev->gemm_spin_limit;  // seconds by default; a partial tile is normally there hundreds of microseconds before it is asked for
  g.raise_flags = dev->gemm_raise_flags;
  g.beta = beta;
  int st;
  if (a_kmajor && b_kmajor) st = launch_wide<true, true>(dev, g, p.segments, 0);
  else if (a_kmajor) st = launch_wide<true, false>(dev, g, p.segments, 1);
  else if (b_kmajor) st = launch_wide<false, true>(dev, g, p.segments, 2);
  else st = launch_wide<false, false>(dev, g, p.segments, 3);
  DYHIP_CHECK_STATUS(st);
  DYHIP_CHECK_LAUNCH();
  if (p.finish_in_kernel) {
    mark_gemm_flags_used(dev);
  } else {
    const dim3 grid(p.tiles, 16);
    if (a_kmajor && b_kmajor) hipLaunchKernelGGL((gemm_wide_fixup_kernel<true, true>), grid, dim3(kWideThreads), 0, dev->stream, g, p.segments);
    else if (a_kmajor) hipLaunchKernelGGL((gemm_wide_fixup_kernel<true, false>), grid, dim3(kWideThreads), 0, dev->stream, g, p.segments);
    else if (b_kmajor) hipLaunchKernelGGL((gemm_wide_fixup_kernel<false, true>), grid, dim3(kWideThreads), 0, dev->stream, g, p.segments);
    else hipLaunchKernelGGL((gemm_wide_fixup_kernel<false, false>), grid, dim3(kWideThreads), 0, dev->stream, g, p.segments);
    DYHIP_CHECK_LAUNCH();
  }
  return DYHIP_OK;
}

bool gemm_shallow_nt_eligible(const dyhip_device* dev, size_t M, size_t N, size_t K, const float* A, size_t lda,
                              const float* B, size_t ldb, const float* C) {
  if (K < 24 || K > 128 || K % 8 != 0 || M % 4 != 0 || N % 4 != 0 || M < 128 || N < 128) return false;
  if (dev->max_lds_per_block < kShallowLdsBytes) return false;
  if (!aligned16(A) || !aligned16(B) || lda % 4 != 0 || ldb % 4 != 0 || (reinterpret_cast<uintptr_t>(C) & 7u) != 0)
    return false;
  if (K * lda >= (size_t(1) << 31) || K * ldb >= (size_t(1) << 31) || M * N >= (size_t(1) << 31)) return false;
  const size_t cus = dev->num_cus > 0 ? size_t(dev->num_cus) : 256;
  return cdiv<size_t>(M, 128) * cdiv<size_t>(N, 128) * 2 >= cus;  // fewer tiles: smaller ones fill the GPU
}

int gemm_shallow_nt_run(dyhip_device* dev, size_t M, size_t N, size_t K, const float* A, size_t lda, const float* B,
                        size_t ldb, float* C, float beta) {
  ShallowArgs g;
  g.A = A;
  g.B = B;
  g.C = C;
  g.lda = unsigned(lda);
  g.ldb = unsigned(ldb);
  g.M = unsigned(M);
  g.N = unsigned(N);
  g.K = unsigned(K);
  g.tiles_m = unsigned(cdiv<size_t>(M, 128));
  g.beta = beta;
  if ((dev->wide_gemm_ready & (1u << 4)) == 0) {
    DYHIP_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_shallow_nt_kernel),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, int(kShallowLdsBytes)));
    dev->wide_gemm_ready |= 1u << 4;
  }
  const unsigned blocks = g.tiles_m * unsigned(cdiv<size_t>(N, 128));
  hipLaunchKernelGGL(gemm_shallow_nt_kernel, dim3(blocks), dim3(kWideThreads), kShallowLdsBytes, dev->stream, g);
  DYHIP_CHECK_LAUNCH();
  return DYHIP_OK;
}

// For tests of the hand-off between blocks without a GPU: the first unit of every segment (segments + 1 values, the
// last one = units) when the k-tiles of an M x N x K product are dealt to `segments` blocks, and how cut tiles are
// finished.  The same function as the kernels use.
void gemm_wide_describe(size_t M, size_t N, size_t K, unsigned segments, unsigned* starts, unsigned* k_tiles_per_tile,
                        int* finish_in_kernel) {
  const unsigned nt = unsigned(K / kWK);
  const size_t units = cdiv<size_t>(M, kWT) * cdiv<size_t>(N, kWT) * nt;
  for (unsigned s2 = 0; s2 <= segments; ++s2) starts[s2] = segment_start(s2, unsigned(units), segments);
  *k_tiles_per_tile = nt;
  *finish_in_kernel = units / segments >= nt ? 1 : 0;
}

}  // namespace dyhip
