// All timesteps of an LSTM layer in one launch, forward and backward (the chain of lstm_step_fwd_kernel /
// lstm_step_bwd_kernel launches of lstm.hip; dynet/lstm.cc:1044-1080, dynet/nodes-lstm.cc:101-703).
//
// A timestep as a launch of its own is bound by what every launch pays: dispatch and drain, the weights from the L2s
// once more (256 KB a CU), the state after them.  Here a block keeps its slice of the recurrent weights on chip for the
// whole sequence, as three bf16 parts (split3.h): two in registers, the third in LDS.  A timestep then reads the state
// alone, multiplies on the bf16 matrix cores, runs the cell update of its (unit, column) pairs and hands its part of the
// new state to the blocks that work on the same columns.
//
// us a timestep in a graph, a launch each -> 35 in one launch, forward / backward: H = 1024, B = 128 13.7 / 15.1 -> 8.5 /
// 10.9; H = 512, B = 64 5.9 / 8.6 -> 3.95 / 4.3; H = 650, B = 20 (two launches each) 11.2 / 9.0 -> 4.7 / 5.3.  What bounds
// it at H = 1024, B = 128, forward, by stamps inside the kernel (when a timestep took 9.1): 1.5 us until the last block's flag
// is seen, 5.4 for the state's way from the L2 (192 KB a CU) and the products (2.9 of matrix cores), 1.4 for the sums in LDS,
// 0.4 cell update, 0.4 until the state is in memory; backward the product is 8 us, 768 KB of state a CU, 96 GB/s.  Small
// layers: the hand-over.
#include <initializer_list>

#include "common.h"
#include "split3.h"

namespace dyhip {

hipError_t zero_fill(void* p, size_t nbytes, hipStream_t stream);

namespace {

constexpr unsigned kSeqWaves = 8, kSeqThreads = 64 * kSeqWaves;
typedef float sums4 __attribute__((ext_vector_type(4)));
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr unsigned kSeqRedBytes = kSeqWaves * 32 * 32 * sizeof(float);
// Polls, about a microsecond apart, before a waiting block looks for a tile that no block has taken.  What holds CUs has mostly
// ended by then, and a block with two tiles reads its weights again for every timestep: a model of H = 1024, B = 128, T = 35
// beside a queue of large products 4.1 ms with 8 polls, 3.4 with 64, 2.77 with 256 and with 1024 (3.19 with a launch a timestep);
// beside another such model 3.0 to 3.5, 2.7, 2.7 and 2.7 ms for both (3.11).
constexpr unsigned kSeqPatience = 256;

// Which block works on which tile, and how far the tiles are; zero at the start of a launch.
struct SeqSync {
  unsigned RT, CT;   // row tiles (units) x column tiles
  unsigned* claims;  // [CT][RT]: 1 + the block that works on the tile
  unsigned* flags;   // [CT][RT]: timesteps that the tile's part of the state is complete for
  unsigned* gave_up;
  unsigned spin_limit;
};

struct SeqFwdArgs {
  unsigned H, B, T;
  unsigned ksteps;     // groups of 16 units: ceil(H / 16)
  SeqSync sync;        // row tiles of 8 * TILES units, column tiles of 32
  const float* Wh;     // 4H x H, column-major
  const float* bias;
  const float* mask;   // H x B or null: the recurrent product reads h (.) mask
  const float* xproj;  // T x B x 4H; may be gates
  float *gates, *c, *h;
  unsigned* state;     // [T][CT][ksteps][3][64][4]: h of every timestep as the next one's operand, in parts (SeqState)
  int mode;
};

struct SeqBwdArgs {
  unsigned H, B, T;
  unsigned ksteps;     // groups of 32 of the 4 * 16 * RT gate rows (each gate's rows padded to a multiple of 16)
  SeqSync sync;        // row tiles of 16 units, column tiles of 16 * COLS
  const float* Wh;     // 4H x H, column-major
  const float* mask;   // H x B or null
  const float *gates, *c, *dh;
  float* dpre;
  unsigned* state;     // [T][column tiles of 16][ksteps][3][64][4]: dpre of every timestep as the next one's operand
  float* carry;        // [CT][RT][512]: dc between two timesteps of a tile whose block has several
};

// Position of block b when the blocks of an XCD (b modulo 8) take consecutive tiles: the tiles of a column tile, which
// read the same state, then share one or two L2s.
__device__ __forceinline__ unsigned seq_first_tile(unsigned b, unsigned n) {
  const unsigned x = b % 8;
  return x * (n / 8) + min(x, n % 8) + b / 8;
}

// Position of (row, column) in a 32 x 32 tile of sums in LDS.  Banks: a matrix-core result writes rows r and r + 4 of 32
// columns at once, the cell update reads 16 rows of 4 columns (8 rows of 8): without conflicts (two to a bank).
__device__ __forceinline__ unsigned seq_red_at(unsigned row, unsigned col) {
  return (row >> 1) * 64 + ((row ^ (row >> 2)) & 1) * 32 + (col ^ (4 * ((row >> 1) & 7)));
}

// The state as the products read it: every value as its three bf16 parts, formed once by the thread that has it (64 blocks
// read it, and splitting there took longer than the products; 6 bytes a value instead of 4).  A step of the depth holds
// [part][lane of the fragment][8 values].
struct SeqState {
  uint4 h, m, l;
  __device__ __forceinline__ void load(const unsigned* step, unsigned lane) {
    const uint4* p = reinterpret_cast<const uint4*>(step) + lane;
    h = p[0];
    m = p[64];
    l = p[128];
  }
  // value i of the eight; see seq_split for what the parts hold where the first one is no number
  __device__ __forceinline__ static float value(const unsigned* step, unsigned lane, unsigned i) {
    const unsigned short* p = reinterpret_cast<const unsigned short*>(step) + lane * 8 + i;
    const float h = __uint_as_float(unsigned(p[0]) << 16), m = __uint_as_float(unsigned(p[512]) << 16),
                l = __uint_as_float(unsigned(p[1024]) << 16);
    return h * 0.f == 0.f ? (h + (m + l)) * (1.f / kSplitIn) : __uint_as_float(unsigned(p[512]) << 16 | p[1024]);
  }
  // Where the pair of values that depth k is one of lies in a step of `width` depths and 64 / (width / 8) columns: the
  // first part's word; the others are 256 words on.
  template <unsigned WIDTH>
  __device__ __forceinline__ static unsigned word(unsigned k, unsigned col) {
    return k / WIDTH * 768 + (k % WIDTH / 8 * (512 / WIDTH) + col) * 4 + k % 8 / 2;
  }
  __device__ __forceinline__ static void put(unsigned* to, unsigned v) {
    __hip_atomic_store(to, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
};
// The parts of 2^16 times this thread's value and its neighbour's (threads 2i and 2i + 1 have neighbouring units), packed.
// Each value by itself: split3_pair would spread an infinity to the other value of its pair.  A value of about 2^111 or more,
// an infinity and a NaN leave a first part that is no number, and the products with it are formed again by the fp32
// instruction: with KEEP the other two parts hold such a value as it is.  That is rare, and a wavefront that has one
// (seq_keeps) puts its parts a second time.
template <bool KEEP>
__device__ __forceinline__ void seq_split(float v, unsigned (&part)[3]) {
  const unsigned bits = __float_as_uint(v);
  bool keep = false;
  v *= kSplitIn;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    unsigned mine = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{v, 0.f}, bf16x2));
    v -= __uint_as_float(mine << 16);
    if (KEEP && i == 0) keep = (mine & 0x7f80u) == 0x7f80u;
    if (KEEP && i > 0 && keep) mine = i == 1 ? bits >> 16 : bits & 0xffffu;
    const unsigned other = __builtin_amdgcn_update_dpp(0, mine, 0xB1, 0xF, 0xF, false);
    part[i] = threadIdx.x & 1 ? mine << 16 | other : other << 16 | mine;
  }
}
__device__ __forceinline__ bool seq_keeps(float v) { return !(fabsf(v) < 0x1p110f); }

// Waits, with all threads of the block, until every row tile of a column tile has finished `want` timesteps.
__device__ __forceinline__ void seq_wait(const SeqSync& y, unsigned ct, unsigned want, bool& dead) {
  if (threadIdx.x < 64) {
    const unsigned* flags = y.flags + size_t(ct) * y.RT;
    for (unsigned polls = 0; !dead; ++polls) {
      bool ok = true;
      for (unsigned at = threadIdx.x; at < y.RT; at += 64)
        ok = ok && __hip_atomic_load(flags + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) >= want;
      if (__all(ok)) break;
      if (polls >= y.spin_limit) {
        dead = true;
        if (threadIdx.x == 0) atomicAdd(y.gave_up, 1u);
      }
      __builtin_amdgcn_s_sleep(1);
    }
  }
  __syncthreads();
}

// After this block's part of the state has been written through: raises its flag.  What a timestep writes for later launches
// (gates, c and h, or dpre) comes behind it: stored while the flags were on their way it held them up, all blocks' at once, by
// 0.65 us at H = 1024, B = 128 backward (11.9 -> 11.2 us a timestep) and 0.4 at H = 650, B = 20 forward (5.1 -> 4.7).  Up to eight
// row tiles there is too little of it, and the wait is the longer one (H = 128, B = 32 backward 3.2 -> 3.35; 16 tiles, H = 256,
// 3.6 either way).
__device__ __forceinline__ void seq_raise(const SeqSync& y, unsigned ct, unsigned rt, unsigned steps) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(y.flags + size_t(ct) * y.RT + rt, steps, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  if (y.RT > 8) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
}

// Which block works on which tile.  Every tile has a block of its own in the grid; a block that runs takes its tile
// (claims) before it does anything else.  Nothing says that all blocks run at the same time: another queue or process can
// hold CUs for as long as it likes, another launch of this kernel even until this one has ended.  So a block that has
// waited a while for the first timestep takes tiles that no block has taken, and does them beside its own; a block that
// starts later and finds its tile taken ends at once.  After the first timestep all tiles of the block's columns belong
// to blocks that run, and a block waits for nothing but blocks that run and the timestep before: the launch ends
// whatever else the GPU is doing.  (A wait has a bound all the same; one that gives up is counted and reported as the
// matrix products' are.)
//
// What the blocks hand each other.  The threads of a block write its part of the state with stores that go through to
// memory, wait until they are there, and one raises a flag in memory; whoever needs it polls the flag there and then
// reads the state with ordinary loads.  These cannot hit a stale line: every timestep has a place of its own, whole
// 128-byte lines of which are written by one block and read by none before the flags of that place are up, so no cache
// has them from earlier in this launch, and none keeps them from before it (caches hold nothing across launches that
// another XCD may write).  With release and acquire fences instead, which write back and drop whole L2s, a hand-over
// takes 34 us where it takes 1.7 (256 blocks, 64 to a column tile).
template <class K>
__device__ __forceinline__ void seq_run(K& k, const SeqSync& y, unsigned T, unsigned* word) {
  const unsigned me = blockIdx.x + 1, tile = seq_first_tile(blockIdx.x, y.RT * y.CT);
  const unsigned ct = tile / y.RT, own = tile % y.RT;
  unsigned* claims = y.claims + size_t(ct) * y.RT;
  const auto claim = [&](unsigned rt) {
    unsigned nobody = 0;
    return __hip_atomic_compare_exchange_strong(claims + rt, &nobody, me, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_SYSTEM);
  };
  if (threadIdx.x == 0) word[0] = claim(own) ? 1u : 0u;
  __syncthreads();
  if (word[0] == 0) return;  // uniform
  k.columns(ct);
  float carry = k.first_step(own);
  k.load_weights(own);
  unsigned tiles = 1;
  for (unsigned polls = 0;;) {
    __syncthreads();
    if (threadIdx.x < 64) {
      const unsigned* flags = y.flags + size_t(ct) * y.RT;
      unsigned next = 0;  // 1: the first timestep is complete; 2 + rt: taken over
      for (unsigned i = 0; i < kSeqPatience && next == 0; ++i) {
        bool ok = true;
        for (unsigned at = threadIdx.x; at < y.RT; at += 64)
          ok = ok && __hip_atomic_load(flags + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) >= 1;
        if (__all(ok)) next = 1;
        else __builtin_amdgcn_s_sleep(8);
      }
      polls += kSeqPatience;
      if (threadIdx.x == 0) {
        for (unsigned rt = 0; rt < y.RT && next == 0; ++rt)
          if (__hip_atomic_load(claims + rt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) == 0 && claim(rt)) next = 2 + rt;
        if (next == 0 && polls > y.spin_limit) {
          next = 1;
          atomicAdd(y.gave_up, 1u);
        }
        word[0] = next;
      }
    }
    __syncthreads();
    const unsigned next = word[0];
    if (next == 1) break;
    if (next >= 2) {
      k.keep(next - 2, k.first_step(next - 2));
      ++tiles;
    }
  }
  __syncthreads();
  if (tiles == 1) {
    k.own_steps(own, carry);
    return;
  }
  k.keep(own, carry);
  for (unsigned s = 1; s < T; ++s)
    for (unsigned rt = 0; rt < y.RT; ++rt)
      if (__hip_atomic_load(claims + rt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) == me) k.other_step(rt, s);  // uniform
}

template <int TILES, int KS>
struct SeqFwd {
  static constexpr unsigned UB = 8 * TILES;  // units of a tile; its 32 * TILES weight rows are q * UB + unit
  static constexpr int RAW = 2;   // steps of the state in flight; more spill
  const SeqFwdArgs& a;
  bf16x8* low;       // this wavefront's low parts, [TILES][KS][64]
  float* red;
  unsigned wave, lane, l32, lhi, ct, eu, col, ecol, lcol;
  bf16x8 wh[TILES][KS], wm[TILES][KS];
  bool dead = false;

  __device__ __forceinline__ SeqFwd(const SeqFwdArgs& a, char* lds) : a(a) {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    lane = threadIdx.x % 64;
    l32 = lane % 32;
    lhi = lane / 32;
    low = reinterpret_cast<bf16x8*>(lds) + wave * (TILES * KS * 64) + lane;
    red = reinterpret_cast<float*>(lds + kSeqWaves * TILES * KS * 64 * sizeof(bf16x8));
    eu = threadIdx.x % UB;
    col = threadIdx.x / UB;
  }
  __device__ __forceinline__ void columns(unsigned ct_) {
    ct = ct_;
    ecol = ct * 32 + col;
    lcol = min(ecol, a.B - 1);
  }
  __device__ __forceinline__ bool updates() const { return TILES == 2 || threadIdx.x < 256; }

  // this lane's eight weights of row tile j, step g of 16 k
  __device__ __forceinline__ void weights8(unsigned rt, int j, unsigned g, float (&x)[8]) const {
    const unsigned row = j * 32 + l32, unit = rt * UB + row % UB, k = 16 * g + 8 * lhi;
    const unsigned at = row / UB * a.H + min(unit, a.H - 1);
#pragma unroll
    for (unsigned i = 0; i < 8; ++i) x[i] = a.Wh[min(k + i, a.H - 1) * (4 * a.H) + at];  // 4 * H * H fits 32 bits
#pragma unroll
    for (unsigned i = 0; i < 8; ++i) x[i] = unit < a.H && k + i < a.H ? x[i] : 0.f;
  }
  __device__ __forceinline__ void load_weights(unsigned rt) {
    constexpr int N = TILES * KS, C = N < 8 ? N : 8;  // 8 x 8 loads in flight: the registers that the parts will take
#pragma unroll
    for (int n0 = 0; n0 < N; n0 += C) {
      float x[C][8];
#pragma unroll
      for (int n = n0; n < n0 + C && n < N; ++n) weights8(rt, n % TILES, wave * KS + n / TILES, x[n - n0]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = n0; n < n0 + C && n < N; ++n) {
        const float(&y)[8] = x[n - n0];
        Split3 s;
        s.from(make_float4(y[0], y[1], y[2], y[3]), make_float4(y[4], y[5], y[6], y[7]));
        wh[n % TILES][n / TILES] = s.h;
        wm[n % TILES][n / TILES] = s.m;
        low[(n % TILES * KS + n / TILES) * 64] = s.l;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // The sum of a 32 x 32 tile over this wavefront's part of the depth again, by the fp32 instruction.
  __device__ __forceinline__ sums16 redo(const unsigned* sp, unsigned rt, int j) const {
    sums16 s = {0};
    const unsigned g0 = wave * KS, g1 = min(g0 + KS, a.ksteps);
#pragma unroll 1
    for (unsigned g = g0; g < g1; ++g) {
      float x[8];
      weights8(rt, j, g, x);
#pragma unroll
      for (unsigned i = 0; i < 8; ++i)
        s = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i], SeqState::value(sp + g * 768, lane, i), s, 0, 0, 0);
    }
    return s;
  }

  __device__ __forceinline__ void publish(unsigned rt, unsigned t, float hv) {
    unsigned* to = a.state + (size_t(t) * a.sync.CT + ct) * a.ksteps * 768 + SeqState::word<16>(rt * UB + eu, col);
    const bool odd = threadIdx.x & 1;
    const auto put = [&](const unsigned (&part)[3]) {
      SeqState::put(to + (odd ? 256 : 0), odd ? part[1] : part[0]);
      if (!odd) SeqState::put(to + 512, part[2]);
    };
    unsigned part[3];
    seq_split<false>(hv, part);
    put(part);
    if (__builtin_expect(__any(seq_keeps(hv)), 0)) {
      seq_split<true>(hv, part);
      put(part);
    }
  }

  // Cell update of this thread's (unit, column); h goes to the blocks that wait for it before anything else is written.
  __device__ __forceinline__ float finish(unsigned rt, unsigned t, const float (&pre)[4], float cp, float mh) {
    const unsigned ej = rt * UB + eu;
    const bool in = updates() && ej < a.H && ecol < a.B;
    float gi = 0.f, gf = 0.f, go = 0.f, gg = 0.f, cv = 0.f, hv = 0.f;
    if (updates()) {
      gi = logistic(a.mode, pre[0]);
      gf = logistic(a.mode, pre[1]);
      go = logistic(a.mode, pre[2]);
      gg = tanh_accurate(pre[3]);
      cv = t > 0 ? gi * gg + gf * cp : gi * gg;
      hv = go * tanh_accurate(cv);
      publish(rt, t, in ? hv * mh : 0.f);
    }
    seq_raise(a.sync, ct, rt, t + 1);
    if (in) {
      float* g = a.gates + (size_t(t) * a.B + ecol) * 4 * a.H + ej;
      const size_t s = (size_t(t) * a.B + ecol) * a.H + ej;
      g[0] = gi;
      g[a.H] = gf;
      g[2 * size_t(a.H)] = go;
      g[3 * size_t(a.H)] = gg;
      a.c[s] = cv;
      a.h[s] = hv;
    }
    return cv;
  }

  // Wx * x and the bias of this thread's (unit, column)
  __device__ __forceinline__ void inputs(unsigned rt, unsigned t, float (&x)[4]) {
    const float* xp = a.xproj + (size_t(t) * a.B + lcol) * 4 * a.H + min(rt * UB + eu, a.H - 1);
#pragma unroll
    for (int q = 0; q < 4; ++q) x[q] = xp[size_t(q) * a.H];
  }
  __device__ __forceinline__ void biases(unsigned rt, float (&b)[4]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) b[q] = a.bias[q * a.H + min(rt * UB + eu, a.H - 1)];
  }
  __device__ __forceinline__ float mask_of(unsigned rt) {
    return a.mask != nullptr ? a.mask[size_t(lcol) * a.H + min(rt * UB + eu, a.H - 1)] : 1.f;
  }

  __device__ __forceinline__ float first_step(unsigned rt) {
    float x[4] = {0.f, 0.f, 0.f, 0.f}, b[4] = {0.f, 0.f, 0.f, 0.f}, pre[4], mh = 1.f;
    if (updates()) {
      inputs(rt, 0, x);
      biases(rt, b);
      mh = mask_of(rt);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) pre[q] = (q == 1 ? b[q] + 1.0f : b[q]) + x[q];
    return finish(rt, 0, pre, 0.f, mh);
  }

  // six products of parts: the large one into sum, the others into small
  __device__ __forceinline__ static void products(sums16& sum, sums16& small, const bf16x8& h, const bf16x8& m, const bf16x8& l,
                                                  const SeqState& v) {
    const bf16x8 vh = __builtin_bit_cast(bf16x8, v.h), vm = __builtin_bit_cast(bf16x8, v.m), vl = __builtin_bit_cast(bf16x8, v.l);
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h, vl, small, 0, 0, 0);
    sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h, vh, sum, 0, 0, 0);
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(m, vm, small, 0, 0, 0);
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h, vm, small, 0, 0, 0);
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(m, vh, small, 0, 0, 0);
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l, vh, small, 0, 0, 0);
  }

  // Weights from registers and LDS (OWN), or from memory step by step: the same products in the same order.  What the
  // cell update reads is fetched under the last products, when the registers of the state are free.
  template <bool OWN>
  __device__ __forceinline__ float step(unsigned rt, unsigned t, float cp, float mh) {
    float b[4] = {0.f, 0.f, 0.f, 0.f}, x[4] = {0.f, 0.f, 0.f, 0.f}, pre[4];
    const unsigned g0 = wave * KS, last = a.ksteps - 1;
    seq_wait(a.sync, ct, t, dead);
    const unsigned* sp = a.state + (size_t(t - 1) * a.sync.CT + ct) * a.ksteps * 768;
    sums16 sum[TILES], small[TILES];
#pragma unroll
    for (int j = 0; j < TILES; ++j) { sum[j] = sums16{0}; small[j] = sums16{0}; }
    if (OWN) {
      SeqState v[RAW];
#pragma unroll
      for (int i = 0; i < RAW; ++i) v[i].load(sp + min(g0 + i, last) * 768, lane);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
        for (int j = 0; j < TILES; ++j) products(sum[j], small[j], wh[j][ks], wm[j][ks], low[(j * KS + ks) * 64], v[ks % RAW]);
        if (ks + RAW < KS) v[ks % RAW].load(sp + min(g0 + ks + RAW, last) * 768, lane);
        if (ks == KS - RAW && updates()) {
          inputs(rt, t, x);
          biases(rt, b);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll 1
      for (int ks = 0; ks < KS; ++ks) {
        SeqState v;
        v.load(sp + min(g0 + ks, last) * 768, lane);
#pragma unroll
        for (int j = 0; j < TILES; ++j) {
          float y[8];
          weights8(rt, j, g0 + ks, y);
          Split3 w;
          w.from(make_float4(y[0], y[1], y[2], y[3]), make_float4(y[4], y[5], y[6], y[7]));
          products(sum[j], small[j], w.h, w.m, w.l, v);
        }
      }
      if (updates()) {
        inputs(rt, t, x);
        biases(rt, b);
      }
    }
    // the eight parts of the depth meet in LDS, a row tile at a time
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      sum[j] = (sum[j] + small[j]) * kSplitOut;
      if (__builtin_expect(any_not_finite(sum[j]), 0)) sum[j] = redo(sp, rt, j);
#pragma unroll
      for (int r = 0; r < 16; ++r) red[wave * 1024 + seq_red_at(8 * (r / 4) + 4 * lhi + r % 4, l32)] = sum[j][r];
      __syncthreads();
      if (updates()) {
#pragma unroll
        for (int q = 0; q < 4 / TILES; ++q) {
          const unsigned at = seq_red_at(q * UB + eu, col);
          float sum_q = red[at];
#pragma unroll
          for (unsigned w = 1; w < kSeqWaves; ++w) sum_q += red[w * 1024 + at];
          pre[j * (4 / TILES) + q] = sum_q;
        }
      }
      if (j + 1 < TILES) __syncthreads();  // (seq_raise waits for the last one's readers)
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) pre[q] += (q == 1 ? b[q] + 1.0f : b[q]) + x[q];
    return finish(rt, t, pre, cp, mh);
  }

  __device__ __forceinline__ void own_steps(unsigned rt, float c) {
    const float mh = updates() ? mask_of(rt) : 1.f;
    for (unsigned t = 1; t < a.T; ++t) c = step<true>(rt, t, c, mh);
  }
  __device__ __forceinline__ void keep(unsigned, float) {}  // c is written anyway
  __device__ __forceinline__ void other_step(unsigned rt, unsigned t) {
    float cp = 0.f, mh = 1.f;
    if (updates()) {
      cp = a.c[(size_t(t - 1) * a.B + lcol) * a.H + min(rt * UB + eu, a.H - 1)];  // this thread wrote it
      mh = mask_of(rt);
    }
    step<false>(rt, t, cp, mh);
  }
};

template <int TILES, int KS>
__global__ __launch_bounds__(kSeqThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void lstm_sequence_fwd_kernel(SeqFwdArgs a) {
  extern __shared__ char lds[];
  SeqFwd<TILES, KS> k(a, lds);
  seq_run(k, a.sync, a.T, reinterpret_cast<unsigned*>(k.red));
}

// The backward timesteps, last one first: step s is timestep T - 1 - s.  A block owns 16 units x 16 * COLS columns and the
// whole depth of Wh^T * dpre, 4H, an eighth a wavefront; v_mfma_f32_16x16x32_bf16, lane 16 * lq + l16 holding depth
// 32 * g + 8 * lq + 0..7 of row (column) l16.
template <int COLS, int KS>
struct SeqBwd {
  static constexpr int RAW = COLS * KS > 24 ? 2 : 4;  // steps of the state in flight; more spill
  const SeqBwdArgs& a;
  bf16x8* low;  // this wavefront's low parts, [KS][64]
  float* red;
  unsigned wave, lane, l16, lq, ct, eu, col, ecol, lcol, Hp;
  bf16x8 wh[KS], wm[KS];
  bool dead = false;

  // what the cell update of a timestep reads: gates, c of the timestep before, dh
  struct Cell {
    float g[4], cp, dh;
  };

  __device__ __forceinline__ SeqBwd(const SeqBwdArgs& a, char* lds) : a(a) {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    lane = threadIdx.x % 64;
    l16 = lane % 16;
    lq = lane / 16;
    low = reinterpret_cast<bf16x8*>(lds) + wave * (KS * 64) + lane;
    red = reinterpret_cast<float*>(lds + kSeqWaves * KS * 64 * sizeof(bf16x8));
    eu = threadIdx.x % 16;
    col = threadIdx.x / 16;
    Hp = 16 * a.sync.RT;
  }
  __device__ __forceinline__ void columns(unsigned ct_) {
    ct = ct_;
    ecol = ct * (16 * COLS) + col;
    lcol = min(ecol, a.B - 1);
  }
  __device__ __forceinline__ bool updates() const { return COLS == 2 || threadIdx.x < 256; }

  // this lane's eight weights of step g of 32 k: one run of Wh, within the rows of a gate
  __device__ __forceinline__ void weights8(unsigned rt, unsigned g, float (&x)[8]) const {
    const unsigned k = 32 * g + 8 * lq, q = k / Hp, row = k - q * Hp, unit = rt * 16 + l16;
    const bool in = unit < a.H && q < 4;
    const float* p = a.Wh + (min(unit, a.H - 1) * (4 * a.H) + min(q, 3u) * a.H);
    if (a.H >= 8 && __all(row + 8 <= a.H || row >= a.H)) {
      const float* r = p + min(row, a.H - 8);
      const float4u lo = *reinterpret_cast<const float4u*>(r), hi = *reinterpret_cast<const float4u*>(r + 4);
#pragma unroll
      for (unsigned i = 0; i < 4; ++i) {
        x[i] = lo[i];
        x[4 + i] = hi[i];
      }
    } else {
#pragma unroll
      for (unsigned i = 0; i < 8; ++i) x[i] = p[min(row + i, a.H - 1)];
    }
#pragma unroll
    for (unsigned i = 0; i < 8; ++i) x[i] = in && row + i < a.H ? x[i] : 0.f;
  }
  __device__ __forceinline__ void load_weights(unsigned rt) {
    constexpr int C = KS < 8 ? KS : 8;
#pragma unroll
    for (int n0 = 0; n0 < KS; n0 += C) {
      float x[C][8];
#pragma unroll
      for (int n = n0; n < n0 + C && n < KS; ++n) weights8(rt, wave * KS + n, x[n - n0]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = n0; n < n0 + C && n < KS; ++n) {
        const float(&y)[8] = x[n - n0];
        Split3 s;
        s.from(make_float4(y[0], y[1], y[2], y[3]), make_float4(y[4], y[5], y[6], y[7]));
        wh[n] = s.h;
        wm[n] = s.m;
        low[n * 64] = s.l;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  __device__ __forceinline__ const unsigned* state_of(unsigned s, int c) const {
    return a.state + ((size_t(s) * a.sync.CT + ct) * COLS + c) * a.ksteps * 768;
  }

  // The sum of a column tile over this wavefront's part of the depth again, by the fp32 instruction.
  __device__ __forceinline__ sums4 redo(const unsigned* sp, unsigned rt) const {
    sums4 sum = {0.f, 0.f, 0.f, 0.f};
    const unsigned g0 = wave * KS, g1 = min(g0 + KS, a.ksteps);
#pragma unroll 1
    for (unsigned g = g0; g < g1; ++g) {
      float x[8];
      weights8(rt, g, x);
#pragma unroll
      for (unsigned i = 0; i < 8; ++i)
        sum = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], SeqState::value(sp + g * 768, lane, i), sum, 0, 0, 0);
    }
    return sum;
  }

  __device__ __forceinline__ Cell cell(unsigned rt, unsigned t) const {
    const unsigned lj = min(rt * 16 + eu, a.H - 1);
    const size_t at = size_t(t) * a.B + lcol, before = size_t(t > 0 ? t - 1 : 0) * a.B + lcol;
    Cell o;
#pragma unroll
    for (int q = 0; q < 4; ++q) o.g[q] = a.gates[at * 4 * a.H + q * a.H + lj];
    o.cp = a.c[before * a.H + lj];
    o.dh = a.dh[at * a.H + lj];
    return o;
  }
  __device__ __forceinline__ float c_of(unsigned rt, unsigned t) const {
    return a.c[(size_t(t) * a.B + lcol) * a.H + min(rt * 16 + eu, a.H - 1)];
  }
  __device__ __forceinline__ float mask_of(unsigned rt) const {
    return a.mask != nullptr ? a.mask[size_t(lcol) * a.H + min(rt * 16 + eu, a.H - 1)] : 1.f;
  }

  // Cell backward of this thread's (unit, column); dpre goes to the blocks that wait for it first.  Returns dc of t - 1.
  __device__ __forceinline__ float finish(unsigned rt, unsigned t, const Cell& o, float cv, float dc, float rec) {
    const unsigned ej = rt * 16 + eu, s = a.T - 1 - t;
    const bool in = updates() && ej < a.H && ecol < a.B;
    float out[4] = {0.f, 0.f, 0.f, 0.f}, dc_next = 0.f;
    if (updates()) {
      const float gi = o.g[0], gf = o.g[1], go = o.g[2], gg = o.g[3];
      const float dh = o.dh + rec, th = tanh_accurate(cv);
      const float dcv = dc + dh * go * (1.f - th * th);
      const float d_o = dh * th;
      const float d_i = dcv * gg, d_f = t > 0 ? dcv * o.cp : 0.f, d_g = dcv * gi;
      dc_next = dcv * gf;
      out[0] = d_i * gi * (1.f - gi);
      out[1] = d_f * gf * (1.f - gf);
      out[2] = d_o * go * (1.f - go);
      out[3] = d_g * (1.f - gg * gg);
      if (t > 0) {  // the rest of the state's rows and columns is zero
        unsigned* to = a.state + ((size_t(s) * a.sync.CT + ct) * COLS + col / 16) * a.ksteps * 768;
        unsigned part[4][3];
        const bool odd = threadIdx.x & 1;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          seq_split<false>(in ? out[q] : 0.f, part[q]);
          SeqState::put(to + SeqState::word<32>(q * Hp + ej, col % 16) + (odd ? 256 : 0), odd ? part[q][1] : part[q][0]);
        }
#pragma unroll
        for (int q = 0; q < 4; q += 2)
          SeqState::put(to + SeqState::word<32>((q + odd) * Hp + ej, col % 16) + 512, odd ? part[q + 1][2] : part[q][2]);
        const float largest = fmaxf(fmaxf(fabsf(out[0]), fabsf(out[1])), fmaxf(fabsf(out[2]), fabsf(out[3])));
        if (__builtin_expect(__any(in && seq_keeps(largest)), 0)) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            unsigned kept[3];
            seq_split<true>(in ? out[q] : 0.f, kept);
            unsigned* at = to + SeqState::word<32>(q * Hp + ej, col % 16);
            SeqState::put(at + (odd ? 256 : 0), odd ? kept[1] : kept[0]);
            if (!odd) SeqState::put(at + 512, kept[2]);
          }
        }
      }
    }
    seq_raise(a.sync, ct, rt, s + 1);
    if (in) {
      float* d = a.dpre + (size_t(t) * a.B + ecol) * 4 * a.H + ej;
#pragma unroll
      for (int q = 0; q < 4; ++q) d[size_t(q) * a.H] = out[q];
    }
    return dc_next;
  }

  __device__ __forceinline__ float first_step(unsigned rt) {
    Cell o = {};
    float cv = 0.f;
    if (updates()) {
      o = cell(rt, a.T - 1);
      cv = c_of(rt, a.T - 1);
    }
    return finish(rt, a.T - 1, o, cv, 0.f, 0.f);
  }

  __device__ __forceinline__ static sums4 mma(const bf16x8& x, const uint4& y, const sums4& s) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, __builtin_bit_cast(bf16x8, y), s, 0, 0, 0);
  }
  // six products of parts for every column tile: the large ones into sum, the others into small
  __device__ __forceinline__ static void products(sums4 (&sum)[COLS], sums4 (&small)[COLS], const bf16x8& h, const bf16x8& m,
                                                  const bf16x8& l, const SeqState (&v)[COLS]) {
#define SEQ_EACH(stmt) _Pragma("unroll") for (int c = 0; c < COLS; ++c) stmt;
    SEQ_EACH(small[c] = mma(h, v[c].l, small[c]))
    SEQ_EACH(sum[c] = mma(h, v[c].h, sum[c]))
    SEQ_EACH(small[c] = mma(m, v[c].m, small[c]))
    SEQ_EACH(small[c] = mma(h, v[c].m, small[c]))
    SEQ_EACH(small[c] = mma(m, v[c].h, small[c]))
    SEQ_EACH(small[c] = mma(l, v[c].h, small[c]))
#undef SEQ_EACH
  }

  // Step s >= 1 of a tile; cv: c of its timestep, on return of the one before.
  template <bool OWN>
  __device__ __forceinline__ float step(unsigned rt, unsigned s, float& cv, float dc, float mh) {
    const unsigned t = a.T - 1 - s, g0 = wave * KS;
    Cell o = {};
    seq_wait(a.sync, ct, s, dead);
    const unsigned* sp[COLS];
    sums4 sum[COLS], small[COLS];
#pragma unroll
    for (int c = 0; c < COLS; ++c) {
      sp[c] = state_of(s - 1, c);
      sum[c] = sums4{0.f, 0.f, 0.f, 0.f};
      small[c] = sums4{0.f, 0.f, 0.f, 0.f};
    }
    const unsigned last = a.ksteps - 1;
    if (OWN) {
      SeqState v[RAW][COLS];
#pragma unroll
      for (int i = 0; i < RAW; ++i)
#pragma unroll
        for (int c = 0; c < COLS; ++c) v[i][c].load(sp[c] + min(g0 + i, last) * 768, lane);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        products(sum, small, wh[ks], wm[ks], low[ks * 64], v[ks % RAW]);
#pragma unroll
        for (int c = 0; c < COLS; ++c)
          if (ks + RAW < KS) v[ks % RAW][c].load(sp[c] + min(g0 + ks + RAW, last) * 768, lane);
        if (ks == KS - RAW && updates()) o = cell(rt, t);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll 1
      for (int ks = 0; ks < KS; ++ks) {
        float x[8];
        weights8(rt, g0 + ks, x);
        Split3 w;
        w.from(make_float4(x[0], x[1], x[2], x[3]), make_float4(x[4], x[5], x[6], x[7]));
        SeqState v[COLS];
#pragma unroll
        for (int c = 0; c < COLS; ++c) v[c].load(sp[c] + min(g0 + ks, last) * 768, lane);
        products(sum, small, w.h, w.m, w.l, v);
      }
      if (updates()) o = cell(rt, t);
    }
#pragma unroll
    for (int c = 0; c < COLS; ++c) {
      sum[c] = (sum[c] + small[c]) * kSplitOut;
      float z = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) z = fmaf(sum[c][r], 0.f, z);
      if (__builtin_expect(__any(!(z == 0.f)), 0)) sum[c] = redo(sp[c], rt);
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave * 512 + seq_red_at(4 * lq + r, c * 16 + l16)] = sum[c][r];
    }
    __syncthreads();
    float rec = 0.f;
    if (updates()) {
      const unsigned at = seq_red_at(eu, col);
#pragma unroll
      for (unsigned w = 0; w < kSeqWaves; ++w) rec += red[w * 512 + at];
    }
    const float c_now = cv;
    cv = o.cp;
    return finish(rt, t, o, c_now, dc, a.mask != nullptr ? rec * mh : rec);
  }

  __device__ __forceinline__ void own_steps(unsigned rt, float dc) {
    float cv = 0.f, mh = 1.f;
    if (a.T > 1 && updates()) {
      cv = c_of(rt, a.T - 2);
      mh = mask_of(rt);
    }
    for (unsigned s = 1; s < a.T; ++s) dc = step<true>(rt, s, cv, dc, mh);
  }
  __device__ __forceinline__ void keep(unsigned rt, float dc) {
    a.carry[(size_t(ct) * a.sync.RT + rt) * kSeqThreads + threadIdx.x] = dc;
  }
  __device__ __forceinline__ void other_step(unsigned rt, unsigned s) {
    float cv = 0.f, mh = 1.f;
    if (updates()) {
      cv = c_of(rt, a.T - 1 - s);
      mh = mask_of(rt);
    }
    const float dc = a.carry[(size_t(ct) * a.sync.RT + rt) * kSeqThreads + threadIdx.x];  // this thread wrote it
    keep(rt, step<false>(rt, s, cv, dc, mh));
  }
};

template <int COLS, int KS>
__global__ __launch_bounds__(kSeqThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void lstm_sequence_bwd_kernel(SeqBwdArgs a) {
  extern __shared__ char lds[];
  SeqBwd<COLS, KS> k(a, lds);
  seq_run(k, a.sync, a.T, reinterpret_cast<unsigned*>(k.red));
}

constexpr size_t kSeqAlign = 256;

// What a sequence needs of its workspace: the sync words (zeroed by each launch), the carries and every timestep's state.
struct SeqPlan {
  bool ok;
  int tiles, ks;  // of the kernel instance
  unsigned RT, CT, ksteps;
  size_t sync_words, carry_floats, state_words;
  size_t head() const { return (sync_words * 4 + kSeqAlign - 1) / kSeqAlign * kSeqAlign; }
  size_t bytes() const { return head() + (carry_floats + state_words) * sizeof(float); }
};

// Small tiles (8 units x 32 columns forward, 16 x 16 backward) while that gives no more blocks than CUs: half the products
// a block (us a timestep, small tiles / large: H = 512, B = 128 forward 4.4 / 5.2, backward 5.0 / 6.6; H = 650, B = 20 5.2 /
// 6.6 and 5.7 / 9.4); twice that beyond.  More blocks than CUs could not all keep their weights, and a hidden size beyond
// 1024 does not fit a CU: not ok.
SeqPlan plan_sequence(const dyhip_device* dev, bool backward, unsigned H, unsigned B, unsigned T) {
  SeqPlan p{};
  const unsigned cus = unsigned(dev->num_cus > 0 ? dev->num_cus : 256), tiles16 = (H + 15) / 16;
  if (H > 1024 || B > 32 * cus || dev->gemm_flags == nullptr) return p;
  size_t lds;
  if (backward) {
    p.RT = tiles16;
    p.tiles = p.RT * ((B + 15) / 16) <= cus ? 1 : 2;
    p.CT = (B + 16 * p.tiles - 1) / (16 * p.tiles);
    p.ksteps = 2 * p.RT;
    p.ks = int((p.RT + 15) / 16 * 4);
    p.carry_floats = size_t(p.CT) * p.RT * kSeqThreads;
    p.state_words = size_t(T) * p.CT * p.tiles * p.ksteps * 768;
    lds = kSeqWaves * size_t(p.ks * 64 * 16 + 512 * 4);
  } else {
    p.CT = (B + 31) / 32;
    p.tiles = 2 * tiles16 * p.CT <= cus ? 1 : 2;
    p.RT = p.tiles == 1 ? 2 * tiles16 : tiles16;
    p.ksteps = tiles16;
    p.ks = int((tiles16 + 15) / 16 * 2);
    p.state_words = size_t(T) * p.CT * p.ksteps * 768;
    lds = kSeqWaves * size_t(p.tiles * p.ks * 64 * 16) + kSeqRedBytes;
  }
  p.sync_words = size_t(p.CT) * p.RT * 2;
  p.ok = p.RT * p.CT <= cus && dev->max_lds_per_block >= lds;
  return p;
}

template <class Args>
int launch_sequence(dyhip_device* dev, void (*kernel)(Args), unsigned instance, size_t lds, const SeqPlan& p, const Args& a) {
  if ((dev->sequence_ready & (1u << instance)) == 0) {  // more than 64 KiB of LDS need the opt-in, once per device
    DYHIP_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
    dev->sequence_ready |= 1u << instance;
  }
  DYHIP_CHECK_HIP(zero_fill(a.sync.claims, p.sync_words * sizeof(unsigned), dev->stream));
  const unsigned tiles = p.RT * p.CT, most = dev->sequence_blocks;
  hipLaunchKernelGGL(kernel, dim3(most > 0 && most < tiles ? most : tiles), dim3(kSeqThreads), lds, dev->stream, a);
  DYHIP_CHECK_LAUNCH();
  mark_gemm_flags_used(dev);
  return DYHIP_OK;
}

template <int TILES, int KS>
int launch_fwd(dyhip_device* dev, const SeqPlan& p, const SeqFwdArgs& a) {
  return launch_sequence(dev, &lstm_sequence_fwd_kernel<TILES, KS>, (TILES - 1) * 4 + KS / 2 - 1,
                         kSeqWaves * size_t(TILES * KS * 64 * 16) + kSeqRedBytes, p, a);
}
template <int COLS, int KS>
int launch_bwd(dyhip_device* dev, const SeqPlan& p, const SeqBwdArgs& a) {
  return launch_sequence(dev, &lstm_sequence_bwd_kernel<COLS, KS>, 8 + (COLS - 1) * 4 + KS / 4 - 1,
                         kSeqWaves * size_t(KS * 64 * 16 + 512 * 4), p, a);
}

SeqSync sync_of(const dyhip_device* dev, const SeqPlan& p, void* ws) {
  unsigned* words = static_cast<unsigned*>(ws);
  return SeqSync{p.RT, p.CT, words, words + p.CT * p.RT, dev->gemm_flags + kGemmFlagWords - 1, dev->gemm_spin_limit};
}

int check_sequence(const SeqPlan& p, unsigned H, unsigned B, unsigned T, const void* ws, size_t ws_bytes) {
  DYHIP_REQUIRE(H >= 1 && B >= 1 && T >= 1, "LSTM sequence: bad hidden (%u), batch (%u) or sequence (%u) size", H, B, T);
  DYHIP_REQUIRE(p.ok, "LSTM sequence: unsupported hidden (%u) or batch (%u) size", H, B);
  DYHIP_REQUIRE(ws && ws_bytes >= p.bytes() && reinterpret_cast<uintptr_t>(ws) % kSeqAlign == 0,
                "LSTM sequence: workspace of %zu bytes on a 256-byte boundary needed", p.bytes());
  return DYHIP_OK;
}

}  // namespace
}  // namespace dyhip

using namespace dyhip;

extern "C" {

int dyhip_device_set_sequence_blocks(dyhip_device* dev, unsigned blocks) {
  DYHIP_CHECK_DEV(dev);
  dev->sequence_blocks = blocks;
  return DYHIP_OK;
}

int dyhip_lstm_sequence_workspace(dyhip_device* dev, unsigned H, unsigned B, unsigned T, size_t* bytes) {
  DYHIP_CHECK_DEV(dev);
  DYHIP_REQUIRE(bytes, "null output pointer");
  DYHIP_REQUIRE(H >= 1 && B >= 1 && T >= 1, "LSTM sequence: bad hidden (%u), batch (%u) or sequence (%u) size", H, B, T);
  const SeqPlan f = plan_sequence(dev, false, H, B, T), b = plan_sequence(dev, true, H, B, T);
  *bytes = !f.ok || !b.ok ? 0 : f.bytes() > b.bytes() ? f.bytes() : b.bytes();
  return DYHIP_OK;
}

int dyhip_lstm_sequence_forward(dyhip_device* dev, unsigned H, unsigned B, unsigned T, const float* Wh, const float* mask_h,
                                const float* xproj, const float* b, int logistic_mode, float* gates, float* c, float* h,
                                void* ws, size_t ws_bytes) {
  DYHIP_CHECK_DEV(dev);
  DYHIP_REQUIRE(Wh && xproj && b && gates && c && h, "LSTM sequence: null tensor pointer");
  DYHIP_REQUIRE(logistic_mode == DYHIP_LOGISTIC_PACKET || logistic_mode == DYHIP_LOGISTIC_SCALAR,
                "unknown logistic mode %d", logistic_mode);
  const SeqPlan p = plan_sequence(dev, false, H, B, T);
  DYHIP_CHECK_STATUS(check_sequence(p, H, B, T, ws, ws_bytes));
  const SeqFwdArgs a{H, B, T, p.ksteps, sync_of(dev, p, ws), Wh, b, mask_h, xproj, gates, c, h,
                     reinterpret_cast<unsigned*>(static_cast<char*>(ws) + p.head()), logistic_mode};
#define DYHIP_SEQ(f, n, m)                                  \
  switch (p.ks) {                                           \
    case 1 * m: return f<n, 1 * m>(dev, p, a);              \
    case 2 * m: return f<n, 2 * m>(dev, p, a);              \
    case 3 * m: return f<n, 3 * m>(dev, p, a);              \
    default: return f<n, 4 * m>(dev, p, a);                 \
  }
  if (p.tiles == 1) DYHIP_SEQ(launch_fwd, 1, 2)
  DYHIP_SEQ(launch_fwd, 2, 2)
}

int dyhip_lstm_sequence_backward(dyhip_device* dev, unsigned H, unsigned B, unsigned T, const float* Wh, const float* mask_h,
                                 const float* gates, const float* c, const float* dh, float* dpre, void* ws, size_t ws_bytes) {
  DYHIP_CHECK_DEV(dev);
  DYHIP_REQUIRE(Wh && gates && c && dh && dpre, "LSTM sequence: null tensor pointer");
  const SeqPlan p = plan_sequence(dev, true, H, B, T);
  DYHIP_CHECK_STATUS(check_sequence(p, H, B, T, ws, ws_bytes));
  float* carry = reinterpret_cast<float*>(static_cast<char*>(ws) + p.head());
  const SeqBwdArgs a{H, B, T, p.ksteps, sync_of(dev, p, ws), Wh, mask_h, gates, c, dh, dpre,
                     reinterpret_cast<unsigned*>(carry + p.carry_floats), carry};
  if (p.tiles == 1) DYHIP_SEQ(launch_bwd, 1, 4)
  DYHIP_SEQ(launch_bwd, 2, 4)
#undef DYHIP_SEQ
}

}  // extern "C"
