// Attention on the matrix cores for wide heads (D = 256: fp32 MFMA; 512: three-term bf16 products): the SD-VAE mid-block call
// (app/models/vae.js:86: one head, D = C = 512, 1024 tokens), which the reference sends down its
// unfused GEMM -> softmax -> GEMM path (app/gpu/ops.js:119-147).
//
// Work decomposition (wide_mfma_kernel, D = 256; D = 512 runs wide_split_kernel, described there)
//   One workgroup = NW = 4 wave64s = 32 queries x one chunk of keys. Wave w owns the head-dim
//   slice [w*D/NW, (w+1)*D/NW) of Q, K, V and O:
//   per 32-key block it computes the partial score tile S_w^T = K_w Q_w^T over its slice
//   (v_mfma_f32_32x32x2f32, the same transposed layout as the flash kernel), the NW partial tiles
//   are summed through LDS in two stages in a fixed order (so every wave derives bit-identical
//   probabilities), and each wave accumulates O_w^T += V_w^T P^T for its slice. K and V slices are
//   private to their wave: each wave streams its own slice into LDS with global_load_lds_dwordx4,
//   and only the score exchange needs workgroup barriers.
//   One head of 1024 queries gives just 32 query groups, so the keys are also split across
//   workgroups (nks chunks). Each workgroup writes its partial (O, m, l) to a workspace and a
//   second, fully parallel kernel merges the chunks of every query group with the online-softmax
//   rescale (the kernel boundary orders the two; no atomics or cross-XCD fences).
//
// LDS per workgroup: K and V slices [32 keys][D/NW] per wave (XOR-swizzled as in the flash kernel)
// plus the score exchange: 80 KiB for D = 256 (two workgroups per CU).

#include <algorithm>
#include <cstring>
#include <type_traits>
#include <utility>

#include "common.h"
#include "kernels.h"
#include "split.h"

namespace sa {

namespace {

constexpr float kRescaleSlack = 8.f;

// Asks the scheduler for N times one MFMA and V VALU instructions, in turn.
template <int N, int V>
__device__ __forceinline__ void mix() {
  static_for<N>([](auto) {
    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x2, V, 0);
  });
}

// Arguments of the attention kernels, packed into 112 bytes (launches start about 0.8 us sooner
// with at most 112 bytes of explicit arguments, as measured for the flash kernels): pointers carry
// the callers' element offsets, strides are 32-bit (calls with larger strides take the generic
// kernel), and `o` is the output with one key chunk, the workspace of partial records otherwise.
struct WideArgs {
  const float* q;
  const float* k;
  const float* v;
  float* o;
  const void* mask;   // key lengths (int32) | key mask (uint8)
  const float* bias;  // dense bias
  int32_t sq, sk, sv;  // batch strides
  union {
    int32_t so;     // one key chunk: output batch stride
    int32_t first;  // key chunks: the launch's first query group (its records start at the workspace)
  };
  int32_t ldq, ldk, ldv, ldo;  // row strides
  int32_t Lq, Lk;
  int32_t sbias, smask;  // dense-bias and key-mask batch strides
  int32_t tiles;         // workgroups of the launch (the grid size, for the XCD remap)
  int32_t chunk;         // keys per chunk
  float scale_log2;
  int16_t H, nks;        // heads, key chunks per query group
};
static_assert(sizeof(WideArgs) == 112, "wide kernel arguments must stay within 112 bytes");

// Arguments of the merge kernel: query groups [first, first + groups), whose records (nks each)
// start at ws.
struct MergeArgs {
  float* o;  // output + its element offset
  const float* ws;
  int32_t H, Lq, so, ldo, q_groups, nks, nwg, first, groups;
};

// Dense bias and key mask of one 32-key block in the 32x32 score layout, where lane (col, half)
// holds query col's keys k0 + 8(r/4) + 4 half + r%4 in score register r: four runs of 4 keys per
// lane. Loaded before the block's score products (load), folded into the base-2 scores after them
// (apply). Runs are 16-byte (bias) or 4-byte (mask) loads where the rows allow it and the run lies
// inside the keys, element loads clamped to the last key otherwise; keys at or past Lk read the
// last key's entry and are masked by the caller's key bound.
template <int BIAS, int MASK>
struct BlockTerms {
  static constexpr bool kBias = BIAS == BIAS_DENSE;
  static constexpr bool kMask = MASK == MASK_KEY_MASK;
  f32x4 bv[kBias ? 4 : 1];
  uint32_t km[kMask ? 4 : 1];

  struct Rows {
    const float* brow;     // dense bias row of the lane's query (rows past Lq re-read the last row)
    const uint8_t* kmask;  // key-mask row of the sequence
    bool bias_vec, mask_vec;
    int Lk;
  };
  __device__ static Rows rows(const WideArgs& p, int b, int h, int qi) {
    Rows r;
    r.Lk = p.Lk;
    r.brow = nullptr;
    r.kmask = nullptr;
    r.bias_vec = r.mask_vec = false;
    if constexpr (kBias) {
      r.brow = p.bias + (int64_t)b * p.sbias + ((int64_t)h * p.Lq + min(qi, p.Lq - 1)) * p.Lk;
      // 16-byte runs: the table 16-byte aligned and every row start a multiple of 4 floats (keys of a
      // run start at multiples of 4)
      r.bias_vec = (reinterpret_cast<uintptr_t>(p.bias) & 15) == 0 && (p.Lk & 3) == 0 && (p.sbias & 3) == 0;
    }
    if constexpr (kMask) {
      r.kmask = static_cast<const uint8_t*>(p.mask) + (int64_t)b * p.smask;
      r.mask_vec = (reinterpret_cast<uintptr_t>(r.kmask) & 3) == 0;
    }
    return r;
  }
  __device__ void load(const Rows& r, int k0, int half) {
#pragma unroll
    for (int k4 = 0; k4 < 4; ++k4) {
      const int kk = k0 + 8 * k4 + 4 * half;  // keys kk .. kk + 3
      if constexpr (kBias) {
        if (r.bias_vec && kk + 4 <= r.Lk) {
          bv[k4] = *reinterpret_cast<const f32x4*>(r.brow + kk);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) bv[k4][e] = r.brow[min(kk + e, r.Lk - 1)];
        }
      }
      if constexpr (kMask) {
        if (r.mask_vec && kk + 4 <= r.Lk) {
          km[k4] = *reinterpret_cast<const uint32_t*>(r.kmask + kk);
        } else {
          uint32_t w = 0;
#pragma unroll
          for (int e = 0; e < 4; ++e) w |= (uint32_t)r.kmask[min(kk + e, r.Lk - 1)] << (8 * e);
          km[k4] = w;
        }
      }
    }
  }
  // u: base-2 scores; bias in natural units, so it enters times log2(e)
  __device__ void apply(float* u) const {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      if constexpr (kBias) u[r] = fmaf(bv[r >> 2][r & 3], kLog2e, u[r]);
      if constexpr (kMask) u[r] = ((km[r >> 2] >> (8 * (r & 3))) & 0xffu) != 0 ? u[r] : -INFINITY;
    }
  }
};

template <int BIAS, int MASK>
__global__ __launch_bounds__(256, 1) void wide_mfma_kernel(WideArgs p) {
  constexpr int D = 256, NW = 4;
  constexpr int DS = D / NW;      // head dims per wave
  constexpr int QREG = DS / 2;    // Q values per lane
  constexpr int NDB = DS / 32;    // 32-dim output tiles per wave
  constexpr int CPR = DS / 4;     // 16-byte chunks per slice row
  constexpr int SLICE = 32 * DS;  // floats per K or V slice tile
  constexpr int NI = 32 * CPR / 64;  // LDS-DMA instructions per slice per wave
  constexpr int REC = 32 * D + 64;   // workspace floats per partial: O [32][D], m [32], l [32]
  static_assert(NI * 64 == 32 * CPR, "slice must split into whole wave loads");

  // K and V slices in separate arrays: the compiler then only waits for the DMA into the array a
  // read touches, so V of the next block can stay in flight while K is read
  __shared__ __attribute__((aligned(16))) float lds_k[NW * SLICE];  // [wave][SLICE]
  __shared__ __attribute__((aligned(16))) float lds_v[NW * SLICE];
  __shared__ __attribute__((aligned(16))) f32x4 lds_s[NW * 4 * 64];      // [wave][r/4][lane]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31;
  const int half = lane >> 5;

  const int q_groups = (p.Lq + 31) >> 5, nks = p.nks, chunk = p.chunk;
  int tile = xcd_remap(blockIdx.x, p.tiles);
  const int kc = tile % nks;
  tile /= nks;                       // the launch's query group
  const int slot_base = tile * nks;  // its chunks' records
  if (nks > 1) tile += p.first;
  const int g = tile % q_groups;
  tile /= q_groups;
  const int h = tile % p.H;
  const int b = tile / p.H;
  const int q0 = g * 32;
  const int qi = q0 + col;
  const bool q_valid = qi < p.Lq;

  int kv_len = p.Lk;
  if constexpr (MASK == MASK_KEY_LEN) kv_len = min(max(static_cast<const int32_t*>(p.mask)[b], 0), p.Lk);
  const int kbeg = kc * chunk;
  const int kend = min(kbeg + chunk, kv_len);
  const int nblk = kend > kbeg ? (kend - kbeg + 31) >> 5 : 0;
  using Terms = BlockTerms<BIAS, MASK>;
  constexpr bool kTerms = Terms::kBias || Terms::kMask;
  const typename Terms::Rows trows = Terms::rows(p, b, h, qi);

  float* const kt = lds_k + wave * SLICE;
  float* const vt = lds_v + wave * SLICE;
  const float* kbase = p.k + (int64_t)b * p.sk + h * D + wave * DS;
  const float* vbase = p.v + (int64_t)b * p.sv + h * D + wave * DS;

  // own K / V slice of block j; rows past the chunk's last key re-read that key
  auto issue_k = [&](int j) {
    const int key0 = kbeg + 32 * j;
#pragma unroll
    for (int n = 0; n < NI; ++n) {
      const int pc_all = n * 64 + lane;
      const int row = pc_all / CPR;
      const int pc = pc_all % CPR;
      const int key = min(key0 + row, kend - 1);
      load_to_lds16(kbase + (int64_t)key * p.ldk + 4 * (pc ^ (row & 15)), kt + n * 256);
    }
  };
  auto issue_v = [&](int j) {
    const int key0 = kbeg + 32 * j;
#pragma unroll
    for (int n = 0; n < NI; ++n) {
      const int pc_all = n * 64 + lane;
      const int row = pc_all / CPR;
      const int pc = pc_all % CPR;
      const int key = min(key0 + row, kend - 1);
      load_to_lds16(vbase + (int64_t)key * p.ldv + 4 * (pc ^ (((row >> 2) & 1) << 3)), vt + n * 256);
    }
  };

  if (nblk > 0) {
    issue_k(0);
    issue_v(0);
  }

  // Q slice in registers, pre-scaled: lane holds scale*log2(e)*Q[qi][wave*DS + half*DS/2 + s]
  float qr[QREG];
  {
    const float* src = p.q + (int64_t)b * p.sq + (int64_t)qi * p.ldq + h * D + wave * DS + half * (DS / 2);
#pragma unroll
    for (int i = 0; i < QREG / 4; ++i) {
      f32x4 x = {0.f, 0.f, 0.f, 0.f};
      if (q_valid) x = *reinterpret_cast<const f32x4*>(src + 4 * i);
      qr[4 * i + 0] = x[0] * p.scale_log2;
      qr[4 * i + 1] = x[1] * p.scale_log2;
      qr[4 * i + 2] = x[2] * p.scale_log2;
      qr[4 * i + 3] = x[3] * p.scale_log2;
    }
  }

  f32x16 oacc[NDB];
#pragma unroll
  for (int t = 0; t < NDB; ++t) oacc[t] = zero16();
  float m = kMaxSeed;
  float l = 0.f;
  wait_vmcnt<0>();  // Q and the first block's slices

  for (int j = 0; j < nblk; ++j) {
    const int k0 = kbeg + 32 * j;
    // own K slice of block j has landed (the last NI loads in flight are V of block j, or the Q
    // loads on the first block); wave-private, so no barrier
    wait_vmcnt<NI>();
    // the block's bias / mask terms, used after the score exchange (register loads: the compiler
    // waits for them where they are used)
    Terms terms;
    if constexpr (kTerms) terms.load(trows, k0, half);
    // ---- partial scores over this wave's head-dim slice
    f32x16 s = zero16();
    const float* krow = kt + col * DS;
    const int ksw = col & 15;
#pragma unroll
    for (int i = 0; i < QREG / 4; ++i) {
      const int c = (half * (CPR / 2) + i) ^ ksw;
      const f32x4 kv = *reinterpret_cast<const f32x4*>(krow + 4 * c);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[0], qr[4 * i + 0], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[1], qr[4 * i + 1], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[2], qr[4 * i + 2], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[3], qr[4 * i + 3], s, 0, 0, 0);
    }
    // ---- sum the four partial tiles (fixed order: identical probabilities in every wave)
    __syncthreads();  // everyone has read the previous exchange
#pragma unroll
    for (int k4 = 0; k4 < 4; ++k4) {
      f32x4 x;
      x[0] = s[4 * k4 + 0];
      x[1] = s[4 * k4 + 1];
      x[2] = s[4 * k4 + 2];
      x[3] = s[4 * k4 + 3];
      lds_s[(wave * 4 + k4) * 64 + lane] = x;
    }
    __syncthreads();
    // Two-stage sum: wave w adds up its 1/NW of the tile over all NW partials (in wave order) and
    // writes the sum back into partial 0 at the same places, which no other wave reads; after the
    // barrier every wave reads the summed tile from partial 0.
    {
      float* ldsf = reinterpret_cast<float*>(lds_s);
      const int e0 = wave * (1024 / NW) + lane * 4;  // four floats of the tile per lane
      f32x4 a = *reinterpret_cast<const f32x4*>(ldsf + e0);
#pragma unroll
      for (int ww = 1; ww < NW; ++ww) a += *reinterpret_cast<const f32x4*>(ldsf + ww * 1024 + e0);
      *reinterpret_cast<f32x4*>(ldsf + e0) = a;
    }
    __syncthreads();
    float u[16];
#pragma unroll
    for (int k4 = 0; k4 < 4; ++k4) {
      const f32x4 a = lds_s[k4 * 64 + lane];
      u[4 * k4 + 0] = a[0];
      u[4 * k4 + 1] = a[1];
      u[4 * k4 + 2] = a[2];
      u[4 * k4 + 3] = a[3];
    }
    if (j + 1 < nblk) issue_k(j + 1);  // own K slice consumed: the next one streams in meanwhile
    if constexpr (kTerms) terms.apply(u);
    if (k0 + 32 > kend) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = k0 + 8 * (r >> 2) + 4 * half + (r & 3);
        u[r] = key < kend ? u[r] : -INFINITY;
      }
    }
    // ---- online softmax with a lazily moved reference
    float mb = u[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mb = max_nan(mb, u[r]);
    mb = max_with_partner(mb);
    if (j == 0) {
      // the wave's first block: its maximum becomes the reference (O and l are still zero, so there is
      // nothing to rescale; -FLT_MAX stays for rows with every key masked)
      m = max_nan(m, mb);
    } else if (__builtin_amdgcn_ballot_w64(mb > m + kRescaleSlack) != 0) {
      const float m_new = max_nan(m, mb);
      const float alpha = fast_exp2(m - m_new);
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int t = 0; t < NDB; ++t) oacc[t] *= alpha;
    }
    float ps = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      u[r] = fast_exp2(u[r] - m);
      ps += u[r];
    }
    l += ps;
    // ---- O_w^T += V_w^T P^T (V of block j: only the next K may still be in flight)
    if (j + 1 < nblk) {
      wait_vmcnt<NI>();
    } else {
      wait_vmcnt<0>();
    }
    const float* vrow = vt + (4 * half) * DS + col;
#pragma unroll
    for (int t = 0; t < NDB; ++t) {
      const float* vcol = vrow + 32 * (t ^ half);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float vv = vcol[(8 * (r >> 2) + (r & 3)) * DS];
        oacc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv, u[r], oacc[t], 0, 0, 0);
      }
    }
    if (j + 1 < nblk) issue_v(j + 1);  // after this wave's last read of its V slice
  }

  const float lt = sum_with_partner(l);
  if (nks == 1) {
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    if (q_valid) {
      float* dst = p.o + (int64_t)b * p.so + (int64_t)qi * p.ldo + h * D + wave * DS + 4 * half;
#pragma unroll
      for (int t = 0; t < NDB; ++t)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          f32x4 x;
          x[0] = oacc[t][4 * g4 + 0] * inv;
          x[1] = oacc[t][4 * g4 + 1] * inv;
          x[2] = oacc[t][4 * g4 + 2] * inv;
          x[3] = oacc[t][4 * g4 + 3] * inv;
          *reinterpret_cast<f32x4*>(dst + 32 * t + 8 * g4) = x;
        }
    }
    return;
  }

  // ---- publish this chunk's partial: O (unnormalised, relative to m), m, l; the merge kernel
  // combines the chunks of each query group
  float* rec = p.o + (int64_t)(slot_base + kc) * REC;
  float* orow = rec + col * D + wave * DS + 4 * half;
#pragma unroll
  for (int t = 0; t < NDB; ++t)
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      f32x4 x;
      x[0] = oacc[t][4 * g4 + 0];
      x[1] = oacc[t][4 * g4 + 1];
      x[2] = oacc[t][4 * g4 + 2];
      x[3] = oacc[t][4 * g4 + 3];
      *reinterpret_cast<f32x4*>(orow + 32 * t + 8 * g4) = x;
    }
  if (wave == 0 && half == 0) {
    rec[32 * D + col] = m;
    rec[32 * D + 32 + col] = lt;
  }
}

// D = 512, on the bf16 matrix cores with three-term operands (split.h; six term products per product,
// smallest first): one workgroup = 8 waves = 32 queries x one chunk of keys, in rounds of four 32-key blocks.
// In a round wave w computes a quarter of the head dims (128 (w % 4)) of the score tiles of two blocks
// (2 (w / 4) and the next); the four quarter sums meet in LDS, and each wave finishes 16 keys of one block:
// maxima and row sums of all waves give one reference m per query for the round. Each wave
// publishes its probabilities, split once, and accumulates O^T for 64 head dims over all four blocks. Head
// dim 2i + t of those sits on row i of output tile t, so an 8-byte load of a V row feeds both tiles.
// K and V rows come straight from memory into registers, pipelined ahead of their products, and are split
// there: with 32 queries per workgroup every element is used once, 7 VALU instructions per MFMA, put
// between the products that cover them. That is what bounds it: a wave alone issues one of them per
// 6 cycles, two waves per SIMD one per 4.4, so 8 waves and not 4 (the VAE block of 4096 tokens: 331 against 345 us,
// fp32 products 401; its attention alone 256 us, fp32 299). Q is split once, into LDS; two blocks per wave halve its reads, which at one block
// would take LDS (64 bytes per clock and CU) as long as the MFMAs.
// Writes the same partial records as wide_mfma_kernel (merged by wide_merge_kernel).
template <int BIAS, int MASK>
__global__ __launch_bounds__(512, 2) void wide_split_kernel(WideArgs p) {
  constexpr int D = 512;
  constexpr int DS = D / 8;          // output head dims per wave
  constexpr int NS = D / 64;         // product steps of a quarter of the head dims
  constexpr int REC = 32 * D + 64;   // workspace floats per partial: O [32][D], m [32], l [32]
  constexpr int KR = BIAS == BIAS_NONE ? 3 : 2;  // product steps whose K loads are in flight (three do not fit beside a bias)

  __shared__ u32x4 lds_q[D / 16 * 3 * 64];  // [product step][term][half][query ^ chunk], then the output
  __shared__ u32x4 lds_p[8 * 3 * 2 * 64];   // probability terms [16 keys][term][lane] (8 * 3 * 64); before that
                                            // the quarter sums [wave][neighbour][2][lane]
  __shared__ float lds_m[8 * 32];           // [16 keys][query]
  __shared__ float lds_l[8 * 32];
  __shared__ int lds_bad;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31;
  const int half = lane >> 5;

  const int q_groups = (p.Lq + 31) >> 5, nks = p.nks, chunk = p.chunk;
  int tile = xcd_remap(blockIdx.x, p.tiles);
  const int kc = tile % nks;
  tile /= nks;                       // the launch's query group
  const int slot_base = tile * nks;  // its chunks' records
  if (nks > 1) tile += p.first;
  const int g = tile % q_groups;
  tile /= q_groups;
  const int h = tile % p.H;
  const int b = tile / p.H;
  const int q0 = g * 32;

  int kv_len = p.Lk;
  if constexpr (MASK == MASK_KEY_LEN) kv_len = min(max(static_cast<const int32_t*>(p.mask)[b], 0), p.Lk);
  const int kbeg = kc * chunk;
  const int kend = min(kbeg + chunk, kv_len);
  const int rounds = kend > kbeg ? (kend - kbeg + 127) >> 7 : 0;
  using Terms = BlockTerms<BIAS, MASK>;
  constexpr bool kTerms = Terms::kBias || Terms::kMask;
  const typename Terms::Rows trows = Terms::rows(p, b, h, q0 + col);

  const float* qbase = p.q + (int64_t)b * p.sq + h * D;
  const float* kbase = p.k + (int64_t)b * p.sk + h * D;
  const float* vbase = p.v + (int64_t)b * p.sv + h * D + wave * DS;

  // ---- K of product step i (dims 128 (w % 4) + 16 i + 8 half + 0..7) of blocks 2 (w / 4) + 0 and 1: rows
  // past the chunk's last key re-read it
  f32x4 kring[KR][2][2];
  const float* kr[2];
  auto aim_k = [&](int rb0) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
      kr[e] = kbase + (int64_t)min(rb0 + 64 * (wave >> 2) + 32 * e + col, kend - 1) * p.ldk + 128 * (wave & 3) + 8 * half;
  };
  auto load_k = [&](int i) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int x = 0; x < 2; ++x) kring[i % KR][e][x] = *reinterpret_cast<const f32x4*>(kr[e] + 16 * i + 4 * x);
  };
  // V rows of one block for this wave's head dims: register r holds V[key][2*col, 2*col + 1] of key
  // 8(r/4) + 4*half + r%4 of the block (the keys of score register r). The buffer ends after the chunk's
  // last valid key, so rows past it read as zeros and no load needs a branch.
  unsigned vrow_off[16];  // byte offset of register r's row and columns from the block's first row
#pragma unroll
  for (int r = 0; r < 16; ++r) vrow_off[r] = 4u * (unsigned)((4 * half + 8 * (r >> 2) + (r & 3)) * (int)p.ldv + 2 * col);
  auto load_v = [&](int kb0, f32x2* dst) {
    // (in a scalar register: a clamp on the vector unit would make every load a waterfall loop)
    const int rows = __builtin_amdgcn_readfirstlane(max(0, min(32, kend - kb0)));
    const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(vbase + (int64_t)kb0 * p.ldv), 0, rows * (int)p.ldv * 4, 0x00020000);
#pragma unroll
    for (int r = 0; r < 16; ++r)
      dst[r] = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(vr, vrow_off[r], 0, 0));
  };

  if (rounds > 0) {
    aim_k(kbeg);
#pragma unroll
    for (int i = 0; i < KR; ++i) load_k(i);
  }
  // ---- Q terms into LDS, pre-scaled, and times kUp, so the scores come out in units of kDown (rows past Lq
  // re-read the last row). K needs no scaling: an element below 2^-110 is short of bits by at most 2^-134,
  // which a scaled query below 2^104 turns into at most 2^-30 of a score; a larger one overflows here.
  if (tid == 0) lds_bad = 0;
  const float sc = p.scale_log2 * kUp;
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const int row = (n * 512 + tid) >> 6, c = lane;
    const float* src = qbase + (int64_t)min(q0 + row, p.Lq - 1) * p.ldq + 8 * c;
    const Split8 t = split8<true>(*reinterpret_cast<const f32x4*>(src), *reinterpret_cast<const f32x4*>(src + 4), sc);
    u32x4* d = lds_q + (c >> 1) * 192 + (c & 1) * 32 + (row ^ (c & 31));
    d[0] = t.h;
    d[64] = t.m;
    d[128] = t.l;
  }
  __syncthreads();

  f32x16 oacc[2] = {zero16(), zero16()};
  float m = kMaxSeed;
  float l = 0.f;
  const int blk = 2 * (wave >> 2) + ((wave >> 1) & 1), sub = wave & 1;  // the 16 keys this wave finishes

  for (int rd = 0; rd < rounds; ++rd) {
    const int rb0 = kbeg + 128 * rd;  // first key of the round
    const int kb0 = rb0 + 32 * blk;   // the block this wave finishes 16 keys of
    Terms terms;                      // its bias / mask terms, used after the score products
    if constexpr (kTerms) terms.load(trows, kb0, half);
    f32x2 vbuf[2][16];  // V of the round's blocks, double-buffered
    f32x16 s[2] = {zero16(), zero16()};
    if (rb0 + 64 * (wave >> 2) < kend) {
      auto read_q = [&](int i, u32x4 (&x)[3]) {
        const int ii = NS * (wave & 3) + i;
        const u32x4* f = lds_q + ii * 192 + half * 32 + (col ^ ((2 * ii + half) & 31));
#pragma unroll
        for (int t = 0; t < 3; ++t) x[t] = f[64 * t];
      };
      u32x4 qx[2][3];
      Split8 kx[2][2];
      read_q(0, qx[0]);
#pragma unroll
      for (int e = 0; e < 2; ++e) kx[0][e] = split8(kring[0][e][0], kring[0][e][1]);
      static_for<NS>([&](auto I) {
        constexpr int i = decltype(I)::value, cur = i & 1;
        if constexpr (i + KR < NS) load_k(i + KR);
        if constexpr (i == NS - 3) load_v(rb0, vbuf[0]);  // the round's first V block streams in under the last products
        if constexpr (i + 1 < NS) {
          read_q(i + 1, qx[cur ^ 1]);
#pragma unroll
          for (int e = 0; e < 2; ++e)
            kx[cur ^ 1][e] = split8(kring[(i + 1) % KR][e][0], kring[(i + 1) % KR][e][1]);
        }
        auto products = [&](auto kt, int qt) {
#pragma unroll
          for (int e = 0; e < 2; ++e) s[e] = mfma32(kt(kx[cur][e]), qx[cur][qt], s[e]);
        };
        products([](const Split8& x) { return x.l; }, 0);
        products([](const Split8& x) { return x.h; }, 2);
        products([](const Split8& x) { return x.m; }, 1);
        products([](const Split8& x) { return x.m; }, 0);
        products([](const Split8& x) { return x.h; }, 1);
        products([](const Split8& x) { return x.h; }, 0);
        if constexpr (i + 1 < NS) mix<12, 8>();
        // keeps each load where it is issued (left free, the scheduler sinks loads to their use)
        __builtin_amdgcn_sched_barrier(0);
      });
    } else {
      load_v(rb0, vbuf[0]);
    }
    // ---- quarter sums of the other three waves' 16 keys (wave ^ x finishes block (.. ^ x) / 2, half (.. ^ x) % 2)
#pragma unroll
    for (int x = 1; x < 4; ++x) {
      const int to = (wave & 3) ^ x;
      u32x4* out = lds_p + (wave * 3 + x - 1) * 128 + lane;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        f32x4 v;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float lo = (to & 1) ? s[0][8 + 4 * e + c] : s[0][4 * e + c];
          const float hi = (to & 1) ? s[1][8 + 4 * e + c] : s[1][4 * e + c];
          v[c] = (to & 2) ? hi : lo;
        }
        out[64 * e] = __builtin_bit_cast(u32x4, v);
      }
    }
    float u[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const float lo = sub ? s[0][8 + r] : s[0][r], hi = sub ? s[1][8 + r] : s[1][r];
      u[r] = (wave & 2) ? hi : lo;
    }
    __syncthreads();
#pragma unroll
    for (int x = 1; x < 4; ++x) {
      const u32x4* in = lds_p + ((wave ^ x) * 3 + x - 1) * 128 + lane;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const f32x4 v = __builtin_bit_cast(f32x4, in[64 * e]);
#pragma unroll
        for (int c = 0; c < 4; ++c) u[4 * e + c] += v[c];
      }
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) u[r] *= kDown;
    if constexpr (kTerms) {  // of the block's 16 registers per lane, this wave's 8
      float w[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) w[r] = u[r & 7];
      terms.apply(w);
      // (opaque: a choice between two loads of w would become one at a run-time index, and w memory)
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        float lo = w[r], hi = w[8 + r];
        asm("" : "+v"(lo), "+v"(hi));
        u[r] = sub ? hi : lo;
      }
    }
    if (kb0 + 32 > kend) {
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int key = kb0 + 16 * sub + 8 * (r >> 2) + 4 * half + (r & 3);
        u[r] = key < kend ? u[r] : -INFINITY;
      }
    }
    if (rd + 1 < rounds) {  // the next round's first K rows stream in under the rest of this one
      aim_k(rb0 + 128);
#pragma unroll
      for (int i = 0; i < KR; ++i) load_k(i);
    }
    // ---- one reference per query for the round: the maximum over the four blocks
    float mb = u[0];
#pragma unroll
    for (int r = 1; r < 8; ++r) mb = max_nan(mb, u[r]);
    mb = max_with_partner(mb);
    if (half == 0) lds_m[wave * 32 + col] = mb;
    __syncthreads();  // also: every quarter sum has been read
    float m_new = m;
#pragma unroll
    for (int w = 0; w < 8; ++w) m_new = max_nan(m_new, lds_m[32 * w + col]);
    if (rd > 0) {
      const float alpha = fast_exp2(m - m_new);
      l *= alpha;
      oacc[0] *= alpha;
      oacc[1] *= alpha;
    }
    m = m_new;
    float ps = 0.f;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      u[r] = fast_exp2(u[r] - m);
      ps += u[r];
    }
    ps = sum_with_partner(ps);
    if (half == 0) lds_l[wave * 32 + col] = ps;
    {
      const Split8 t = split8(f32x4{u[0], u[1], u[2], u[3]}, f32x4{u[4], u[5], u[6], u[7]}, kUp);
      u32x4* d = lds_p + (blk * 2 + sub) * 192 + lane;
      d[0] = t.h;
      d[64] = t.m;
      d[128] = t.l;
    }
    __syncthreads();
    {
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < 8; ++w) sum += lds_l[32 * w + col];
      l += sum;
    }
    // ---- O^T += V^T P^T over the round's blocks, this wave's 64 head dims, 16 keys (8 registers per lane) at a
    // time; the next block's V is requested before this block's products
    static_for<4>([&](auto J) {
      constexpr int j = decltype(J)::value;
      if constexpr (j + 1 < 4) load_v(rb0 + 32 * (j + 1), vbuf[(j + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      if (rb0 + 32 * j < kend) {  // wave-uniform: blocks past the chunk's keys hold no probabilities
        Split8 vx[2][2];
        u32x4 px[2][3];
        auto prep = [&](auto I) {
          constexpr int i = decltype(I)::value;
          const f32x2* vb = vbuf[j & 1] + 8 * i;
#pragma unroll
          for (int t = 0; t < 2; ++t)
            vx[i][t] = split8(f32x4{vb[0][t], vb[1][t], vb[2][t], vb[3][t]}, f32x4{vb[4][t], vb[5][t], vb[6][t], vb[7][t]});
#pragma unroll
          for (int t = 0; t < 3; ++t) px[i][t] = lds_p[(j * 2 + i) * 192 + 64 * t + lane];
        };
        prep(std::integral_constant<int, 0>{});
        static_for<2>([&](auto I) {
          constexpr int i = decltype(I)::value;
          if constexpr (i == 0) prep(std::integral_constant<int, 1>{});
          auto products = [&](auto vt, int pt) {
#pragma unroll
            for (int t = 0; t < 2; ++t) oacc[t] = mfma32(vt(vx[i][t]), px[i][pt], oacc[t]);
          };
          products([](const Split8& v) { return v.l; }, 0);
          products([](const Split8& v) { return v.h; }, 2);
          products([](const Split8& v) { return v.m; }, 1);
          products([](const Split8& v) { return v.m; }, 0);
          products([](const Split8& v) { return v.h; }, 1);
          products([](const Split8& v) { return v.h; }, 0);
          if constexpr (i == 0) mix<12, 8>();
          __builtin_amdgcn_sched_barrier(0);
        });
      }
    });
    if (rd + 1 < rounds) __syncthreads();  // every wave is done with the round's exchange
  }

  // Values without three terms, as in flash_split_kernel: anything not finite in a wave's state, or an output that
  // is not zero and below 2^26 times what V elements below 2^-110 may have cost it. If any wave finds one,
  // all take the chunk again with fp32 products straight from memory.
  {
    float most = fabsf(l), least = INFINITY;
    const float floor = l * (0x1p-108f * kUp);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        most = max_nan(most, fabsf(oacc[t][r]));
        least = min_nan(least, fabsf(oacc[t][r]));
      }
    bool redo = !(most < INFINITY);
    if (least < floor) {  // zeros too, which are exact: look again
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) redo |= oacc[t][r] != 0.f && fabsf(oacc[t][r]) < floor;
    }
    if (__builtin_amdgcn_ballot_w64(redo) != 0 && lane == 0) lds_bad = 1;
    __syncthreads();  // also: every wave is done with the Q terms
    if (lds_bad != 0) {
#pragma unroll
      for (int t = 0; t < 2; ++t) oacc[t] = zero16();
      m = kMaxSeed;
      l = 0.f;
      const float* qrow = qbase + (int64_t)min(q0 + col, p.Lq - 1) * p.ldq;
#pragma unroll 1
      for (int kb = kbeg; kb < kend; kb += 32) {
        const float* krow = kbase + (int64_t)min(kb + col, kend - 1) * p.ldk;
        f32x16 s = zero16();
#pragma unroll 1
        for (int d = 0; d < D; d += 2) s = __builtin_amdgcn_mfma_f32_32x32x2f32(krow[d + half], qrow[d + half], s, 0, 0, 0);
        Terms terms;
        if constexpr (kTerms) terms.load(trows, kb, half);
        float u[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) u[r] = s[r] * p.scale_log2;
        if constexpr (kTerms) terms.apply(u);
        float mb = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          u[r] = kb + 8 * (r >> 2) + 4 * half + (r & 3) < kend ? u[r] : -INFINITY;
          mb = max_nan(mb, u[r]);
        }
        const float m_new = max_nan(m, max_with_partner(mb));
        const float alpha = fast_exp2(m - m_new);
        l *= alpha;
#pragma unroll
        for (int t = 0; t < 2; ++t) oacc[t] *= alpha;
        m = m_new;
        float ps = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          u[r] = fast_exp2(u[r] - m);
          ps += u[r];
        }
        l += sum_with_partner(ps);
        f32x2 vb[16];
        load_v(kb, vb);
#pragma unroll
        for (int r = 0; r < 16; ++r)
#pragma unroll
          for (int t = 0; t < 2; ++t) oacc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(vb[r][t], u[r], oacc[t], 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t) oacc[t] *= kDown;  // P was scaled
    }
  }

  // ---- output: O^T tile t, register r holds head dim 64*wave + 2i + t of query col, with
  // i = 8(r/4) + 4*half + r%4, so the two tiles' registers r and r + 1 (r even) are four consecutive head
  // dims. The wave stages its 32 x 64 slice in LDS (the Q terms are dead), 16-byte chunk c of query q
  // at c ^ (q & 15), and stores it back as 256-byte row pieces, four rows per instruction.
  const float inv = nks == 1 ? (l > 0.f ? 1.f / l : 0.f) : 1.f;
  float* stage = reinterpret_cast<float*>(lds_q) + wave * 32 * DS;
#pragma unroll
  for (int r = 0; r < 16; r += 2) {
    const int c = 4 * (r >> 2) + 2 * half + ((r & 3) >> 1);
    const f32x4 x = {oacc[0][r] * inv, oacc[1][r] * inv, oacc[0][r + 1] * inv, oacc[1][r + 1] * inv};
    *reinterpret_cast<f32x4*>(stage + col * DS + 4 * (c ^ (col & 15))) = x;
  }
  float* dst;
  int64_t ld;
  if (nks == 1) {
    dst = p.o + (int64_t)b * p.so + (int64_t)q0 * p.ldo + h * D + wave * DS;
    ld = p.ldo;
  } else {
    float* rec = p.o + (int64_t)(slot_base + kc) * REC;
    dst = rec + wave * DS;
    ld = D;
    if (wave == 0 && half == 0) {
      rec[32 * D + col] = m;
      rec[32 * D + 32 + col] = l;
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int row = 4 * j + (lane >> 4), c = lane & 15;
    const f32x4 x = *reinterpret_cast<const f32x4*>(stage + row * DS + 4 * (c ^ (row & 15)));
    if (nks > 1 || q0 + row < p.Lq) *reinterpret_cast<f32x4*>(dst + (int64_t)row * ld + 4 * c) = x;
  }
}

// Combines the nks partial records of every query group: one thread per (query, 4 dims),
// O = sum_c O_c exp2(m_c - m) / sum_c l_c exp2(m_c - m) with m = max_c m_c (0 if every l_c is 0).
template <int D>
__global__ __launch_bounds__(256) void wide_merge_kernel(MergeArgs p) {
  const int q_groups = p.q_groups, nks = p.nks;
  constexpr int REC = 32 * D + 64;
  constexpr int C4 = D / 4;
  // the same XCD remap as the attention kernel, whose workgroups wrote a query group's records from
  // one XCD: consecutive merge workgroups (one query group's queries) run there and find the records
  // in that XCD's L2
  const int64_t idx = (int64_t)xcd_remap(blockIdx.x, p.nwg) * 256 + threadIdx.x;
  const int64_t total = (int64_t)p.groups * 32 * C4;
  if (idx >= total) return;
  const int d4 = (int)(idx % C4);
  int64_t r = idx / C4;
  const int qq = (int)(r % 32);
  r /= 32;  // the launch's query group
  const float* recs = p.ws + r * nks * REC;
  r += p.first;  // (b*H + h)*q_groups + g
  const int g = (int)(r % q_groups);
  const int bh = (int)(r / q_groups);
  const int h = bh % p.H;
  const int b = bh / p.H;
  const int qi = g * 32 + qq;
  if (qi >= p.Lq) return;
  // One pass over the chunks in groups of 8 whose loads are all issued before any is used
  // (indexes clamped to the last chunk, surplus entries of a group skipped), with a running
  // maximum: the sums so far are rescaled when a group raises it. A query costs ceil(nks/8) load
  // round trips (one for the VAE call's 8 chunks); with a single group the rescale only touches
  // the zero-initialized sums, so the result equals the two-pass (maximum first) merge bit for bit.
  float mt = kMaxSeed;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  float lsum = 0.f;
  for (int c0 = 0; c0 < nks; c0 += 8) {
    float mv[8], lv[8];
    f32x4 xv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float* rc = recs + (int64_t)min(c0 + u, nks - 1) * REC;
      mv[u] = rc[32 * D + qq];
      lv[u] = rc[32 * D + 32 + qq];
      xv[u] = *reinterpret_cast<const f32x4*>(rc + qq * D + 4 * d4);
    }
    float mg = mt;
#pragma unroll
    for (int u = 0; u < 8; ++u) mg = fmaxf(mg, mv[u]);  // a repeated last chunk changes nothing
    const float sc = fast_exp2(mt - mg);
    lsum *= sc;
    acc[0] *= sc;
    acc[1] *= sc;
    acc[2] *= sc;
    acc[3] *= sc;
    mt = mg;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (c0 + u >= nks) break;
      const float a = fast_exp2(mv[u] - mt);
      lsum = fmaf(lv[u], a, lsum);
      acc[0] = fmaf(xv[u][0], a, acc[0]);
      acc[1] = fmaf(xv[u][1], a, acc[1]);
      acc[2] = fmaf(xv[u][2], a, acc[2]);
      acc[3] = fmaf(xv[u][3], a, acc[3]);
    }
  }
  const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
  f32x4 y;
  y[0] = acc[0] * inv;
  y[1] = acc[1] * inv;
  y[2] = acc[2] * inv;
  y[3] = acc[3] * inv;
  *reinterpret_cast<f32x4*>(p.o + (int64_t)b * p.so + (int64_t)qi * p.ldo + h * D + 4 * d4) = y;
}

template <int D, int BIAS, int MASK>
void launch_main(const WideArgs& a, dim3 grid, hipStream_t stream) {
  if constexpr (D == 512)
    hipLaunchKernelGGL((wide_split_kernel<BIAS, MASK>), grid, dim3(512), 0, stream, a);
  else
    hipLaunchKernelGGL((wide_mfma_kernel<BIAS, MASK>), grid, dim3(256), 0, stream, a);
}

template <int D, int BIAS>
hipError_t launch_mask(const WideArgs& a, int mask_mode, dim3 grid, hipStream_t stream) {
  switch (mask_mode) {
    case MASK_NONE: launch_main<D, BIAS, MASK_NONE>(a, grid, stream); break;
    case MASK_KEY_LEN: launch_main<D, BIAS, MASK_KEY_LEN>(a, grid, stream); break;
    case MASK_KEY_MASK: launch_main<D, BIAS, MASK_KEY_MASK>(a, grid, stream); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

bool fits32(int64_t x) { return x >= 0 && x <= 0x7fffffff; }

template <int D>
hipError_t launch_d(const AttnParams& p, const WidePlan& plan, float* ws, hipStream_t stream) {
  const int64_t groups = (int64_t)p.B * p.H * plan.q_groups;
  const int64_t whole = plan.nks > 1 ? plan.whole : groups;  // leading groups, unsplit
  const int64_t split = groups - whole;                      // the rest, in nks chunks each
  if (whole > 0x7fffffff || split * plan.nks > 0x7fffffff) return hipErrorInvalidConfiguration;
  WideArgs a;
  memset(&a, 0, sizeof a);
  a.q = p.q + p.q_off;
  a.k = p.k + p.k_off;
  a.v = p.v + p.v_off;
  a.mask = p.mask_mode == MASK_KEY_LEN ? static_cast<const void*>(p.key_len) : static_cast<const void*>(p.key_mask);
  a.bias = p.bias;
  a.sq = (int32_t)p.sq;
  a.sk = (int32_t)p.sk;
  a.sv = (int32_t)p.sv;
  a.ldq = (int32_t)p.ldq;
  a.ldk = (int32_t)p.ldk;
  a.ldv = (int32_t)p.ldv;
  a.ldo = (int32_t)p.ldo;
  a.Lq = p.Lq;
  a.Lk = p.Lk;
  a.sbias = (int32_t)p.sbias;
  a.smask = (int32_t)p.smask;
  a.scale_log2 = p.scale_log2;
  a.H = (int16_t)p.H;
  auto attend = [&](int64_t n) -> hipError_t {
    a.tiles = (int32_t)n;
    const dim3 grid((unsigned)n);
    if (p.bias_mode == BIAS_NONE) return launch_mask<D, BIAS_NONE>(a, p.mask_mode, grid, stream);
    if (p.bias_mode == BIAS_DENSE) return launch_mask<D, BIAS_DENSE>(a, p.mask_mode, grid, stream);
    return hipErrorInvalidValue;
  };
  if (whole > 0) {
    a.o = p.o + p.o_off;
    a.so = (int32_t)p.so;
    a.nks = 1;
    a.chunk = plan.whole_chunk;
    const hipError_t e = attend(whole);
    if (e != hipSuccess || split == 0) return e;
  }
  a.o = ws;
  a.first = (int32_t)whole;
  a.nks = (int16_t)plan.nks;
  a.chunk = plan.chunk;
  const hipError_t e = attend(split * plan.nks);
  if (e != hipSuccess) return e;
  const int64_t threads = split * 32 * (D / 4);
  const int64_t blocks = (threads + 255) / 256;
  if (blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
  MergeArgs m;
  m.o = p.o + p.o_off;
  m.ws = ws;
  m.H = p.H;
  m.Lq = p.Lq;
  m.so = (int32_t)p.so;
  m.ldo = (int32_t)p.ldo;
  m.q_groups = plan.q_groups;
  m.nks = plan.nks;
  m.nwg = (int32_t)blocks;
  m.first = (int32_t)whole;
  m.groups = (int32_t)split;
  hipLaunchKernelGGL((wide_merge_kernel<D>), dim3((unsigned)blocks), dim3(256), 0, stream, m);
  return hipGetLastError();
}

}  // namespace

bool wide_mfma_supported(const AttnParams& p) {
  // 32-bit strides and at most 32767 heads (the packed arguments); other calls take the generic kernel
  const bool fit = fits32(p.sq) && fits32(p.sk) && fits32(p.sv) && fits32(p.so) && fits32(p.ldq) && fits32(p.ldk) &&
                   fits32(p.ldv) && fits32(p.ldo) && fits32(p.sbias) && fits32(p.smask) && p.H <= 32767;
  return fit && (p.D == 256 || p.D == 512) && (p.bias_mode == BIAS_NONE || p.bias_mode == BIAS_DENSE) &&
         (p.mask_mode == MASK_NONE || p.mask_mode == MASK_KEY_LEN || p.mask_mode == MASK_KEY_MASK);
}

int wide_mfma_variants(FlashVariant* out, int cap) {
  int n = 0;
  for (int D = 256; D <= 512; D *= 2)
    for (int bias = BIAS_NONE; bias <= BIAS_DENSE; ++bias)
      for (int mask = MASK_NONE; mask <= MASK_KEY_MASK; ++mask) {
        if (n < cap) out[n] = {D, 1, bias, mask};
        ++n;
      }
  return n;
}

// Key chunks per query group: of the plans whose merge records fit kWideMaxRecordBytes, the one
// with the shortest modelled makespan (ties: the first found, fewer chunks). A workgroup costs the
// key blocks of its chunk plus about two blocks of start-up and stores; workgroups run in rounds of
// one per CU (D = 512: 8 waves, 146 KiB of LDS) or two (D = 256: 80 KiB of LDS); a split
// adds the merge, about half a block plus one block per 22 MB of records. One block is 32 queries x
// 32 keys over all head dims. (At D = 512 the constants are those of an fp32 kernel of 4.7 us per block; wide_split_kernel
// takes 3.9 us per block, 0.5 to 1.6 blocks more per workgroup, and its merge of 16.8 MB 5.2 us, 1.3 blocks, as
// modelled.) The plans: every group in the same
// number of chunks (up to kWideMaxChunks), or, when the groups fill whole rounds and a few more,
// the whole rounds unsplit and only the groups past them in chunks, in a second launch. For one
// head of 1024 tokens this is 8 chunks of 4 blocks (256 workgroups, one round); for 2304 tokens 3
// chunks of 24 blocks (216 workgroups) rather than 4 of 20 blocks, whose 288 workgroups would take
// two rounds; for 9216 tokens (288 groups) 256 groups unsplit, then 32 groups in 8 chunks.
WidePlan wide_mfma_plan(const AttnParams& p, int num_cus) {
  WidePlan plan;
  plan.q_groups = (p.Lq + 31) / 32;
  const int64_t base = (int64_t)p.B * p.H * plan.q_groups;
  const int64_t slots = (int64_t)num_cus * (p.D == 512 ? 1 : 2);
  const int nblk = (p.Lk + 31) / 32;
  // D = 512 takes keys in rounds of four blocks (wide_split_kernel): chunks of whole rounds
  const int unit = p.D == 512 ? 4 : 1;
  const int64_t rec_bytes = (int64_t)(32 * p.D + 64) * (int64_t)sizeof(float);
  auto rounds = [&](int64_t wgs) { return (double)((wgs + slots - 1) / slots); };
  auto merge = [&](int64_t wgs) { return 0.5 + (double)(wgs * rec_bytes) / 22e6; };
  auto fits = [&](int64_t wgs) { return wgs * rec_bytes <= kWideMaxRecordBytes; };
  const int full = (nblk + unit - 1) / unit * unit;  // blocks of an unsplit group
  double best = rounds(base) * (full + 2);
  plan.nks = 1;
  plan.chunk = plan.whole_chunk = 32 * full;
  plan.whole = 0;
  // split groups: `split` of them (the last ones) in n chunks of bpc blocks, after `whole` unsplit
  auto consider = [&](int64_t whole, int64_t split) {
    for (int want = 2; want <= kWideMaxChunks; ++want) {
      const int bpc = (nblk + want * unit - 1) / (want * unit) * unit;
      const int n = (nblk + bpc - 1) / bpc;  // chunks that hold at least one key
      if (n == 1 || !fits(split * n)) continue;
      const double cost = (whole > 0 ? rounds(whole) * (full + 2) : 0.0) + rounds(split * n) * (bpc + 2) +
                          merge(split * n);
      if (cost < best) {
        best = cost;
        plan.nks = n;
        plan.chunk = 32 * bpc;
        plan.whole = whole;
      }
    }
  };
  consider(0, base);
  if (base > slots && base % slots != 0 && base <= 0x7fffffff) consider(base / slots * slots, base % slots);
  plan.ws_floats = plan.nks > 1 ? (base - plan.whole) * plan.nks * (int64_t)(32 * p.D + 64) : 0;
  return plan;
}

const char* wide_mfma_name(int D) { return D == 512 ? "wide_mfma_d512" : "wide_mfma_d256"; }

hipError_t launch_wide_mfma(const AttnParams& p, const WidePlan& plan, float* ws, hipStream_t stream) {
  if (p.D == 512) return launch_d<512>(p, plan, ws, stream);
  if (p.D == 256) return launch_d<256>(p, plan, ws, stream);
  return hipErrorInvalidValue;
}

}  // namespace sa
