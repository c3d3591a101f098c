// Flash attention on the bf16 matrix cores of gfx950, head dim 64 or 128, for launches that fill the chip
// (app/gpu/kernels.js:164-316 and, with bias and masks fused, the unfused chain of
// app/gpu/ops.js:119-147): every float32 operand as three bfloat16 terms (split.h), every product as
// six term products summed in float32, smallest first. Packed arguments and launch classes: flash_mfma.hip.
//
// Work decomposition
//   A workgroup is QG * KS waves: QG groups of 32 queries of one (sequence, head), each seen by KS waves
//   that take every KS-th block of 32 keys and merge their softmax states through LDS at the end. A step
//   covers KS blocks. All waves load the step's K and V rows into registers one step ahead, split
//   them once for the workgroup, and leave the terms in LDS in operand order.
//   Scores S^T = K Q^T and output O^T += V^T P^T with v_mfma_f32_32x32x16_bf16: a lane holds query l%32 and
//   keys 8(r/4) + 4(l/32) + r%4 in register r, as with the fp32 32x32x2 products (the retry below uses them on the
//   same softmax). The row maximum is an in-lane chain and one exchange between the half-waves, the row sum a
//   per-lane partial until the end. The 8 keys that a half-wave multiplies per product step of 16
//   are the 8 of its own registers (order of the sum over keys: any), so P needs no exchange: V is laid out
//   to match. Q is pre-scaled and split once.
//   LDS: K terms [product step][term][half][key ^ chunk], so that the 8 threads of a row write 8 different
//   bank groups; V terms [product step][32 dims][term][half][dim], transposed by loading a
//   row of 64 dims per instruction, 8 keys per thread. Q and P are split as 2^24 times themselves.

#include <string.h>

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "split.h"

namespace sa {

namespace {

// O and l are rescaled only when a block's maximum exceeds the reference by more than this (log2 units: p
// stays <= 256); numerator and denominator share the reference.
constexpr float kRescaleSlack = 8.f;

struct FlashOrder {
  uint8_t order[kMaxOrder];
};
struct NoOrder {};

template <int D, int QG, int KS, int STAGES, int WPE, int BIAS, int MASK, typename Order>
__global__ __launch_bounds__(64 * QG * KS, WPE) void flash_split_kernel(FlashArgs p, Order ord) {
  constexpr int NW = QG * KS;
  constexpr int QT = 32 * QG;            // queries per workgroup
  constexpr int KT = 32 * KS;            // keys per step
  constexpr int FK = D / 16;             // product steps of the scores
  constexpr int NDB = D / 32;            // 32-dim output tiles
  constexpr int CPR = D / 8;             // chunks of 8 dims per K row
  constexpr int NC = D / (16 * QG);      // K chunks and V units per thread and step
  constexpr int KBLK = FK * 3 * 64;      // 16-byte chunks of one block's K terms (V: the same)
  constexpr int BLK = 2 * KBLK;
  constexpr int STAGE = KS * BLK;
  constexpr int MSTRIDE = 16 * NDB + 2;  // merge record per lane: O tiles, m, l
  constexpr bool kLen = MASK == MASK_KEY_LEN || MASK == MASK_KEY_LEN_ORDERED;
  static_assert(NC * 16 * QG == D, "a step's rows must split over the threads");
  constexpr int OUT = KS == 1 ? NW * 32 * D / 4 : 0;  // the output rows reuse the tiles
  constexpr int LDS = STAGES * STAGE > OUT ? STAGES * STAGE : OUT;
  static_assert((KS - 1) * QG * 64 * MSTRIDE <= 4 * LDS, "merge records must fit in the tiles");

  constexpr int RB = QT + KT - 1;        // relative distances per step
  static_assert(BIAS != BIAS_RELPOS || RB <= 64 * NW, "one relative distance per thread");
  static_assert(KT <= 64 * NW, "one key mask per thread");

  __shared__ u32x4 lds[LDS];
  __shared__ float lds_rb[BIAS == BIAS_RELPOS ? STAGES * RB : 1];
  __shared__ float lds_km[MASK == MASK_KEY_MASK ? STAGES * KT : 1];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qg = wave % QG;
  const int ks = wave / QG;
  const int col = lane & 31;
  const int half = lane >> 5;

  const int q_tiles = (p.Lq + QT - 1) / QT;
  int tile = xcd_remap(blockIdx.x, p.tiles);
  const int qtile = tile % q_tiles;
  tile /= q_tiles;
  const int h = tile % p.H;
  int b = tile / p.H;
  if constexpr (MASK == MASK_KEY_LEN_ORDERED) b = ord.order[b];  // the host schedule
  const int q0 = qtile * QT;
  const int qi = q0 + qg * 32 + col;
  const bool q_valid = qi < p.Lq;

  int kv_len = p.Lk;
  if constexpr (kLen) kv_len = min(max(static_cast<const int32_t*>(p.mask)[b], 0), p.Lk);
  const int nblk = (kv_len + 31) >> 5;
  const int nstep = (nblk + KS - 1) / KS;
  const uint8_t* kmask = MASK == MASK_KEY_MASK ? static_cast<const uint8_t*>(p.mask) + (int64_t)b * p.aux : nullptr;
  const float* kbase = p.k + (int64_t)b * p.sk + h * D;
  const float* vbase = p.v + (int64_t)b * p.sv + h * D;
  const float* qrow = p.q + (int64_t)b * p.sq + (int64_t)min(qi, p.Lq - 1) * p.ldq + h * D;
  const float* brow = nullptr;
  if constexpr (BIAS == BIAS_DENSE) brow = p.bias + (int64_t)b * p.sbias + ((int64_t)h * p.Lq + min(qi, p.Lq - 1)) * p.Lk;

  // ---- a step's K and V as loaded: rows past the last valid key re-read it (masked out of the softmax).
  // With them the step's bias and mask: the dense-bias values of the lane's 16 keys; the table value of
  // one relative distance per thread (its bucket is loaded a step earlier) and one key's mask, which go
  // to LDS with the terms.
  f32x4 kx[NC][2];
  float vx[NC][8];
  float bx[BIAS == BIAS_DENSE ? 16 : 1];
  float rbx = 0.f, kmx = 0.f;
  int bucket = -1;
  float bcur[BIAS == BIAS_DENSE ? 16 : 1];
  auto load_bucket = [&](int step) {
    // entry e covers LUT index key0 - (q0 + QT - 1) + (Lq - 1) + e
    const int li = step * KT - (q0 + QT - 1) + (p.Lq - 1) + tid;
    bucket = tid < RB && li >= 0 && li <= p.Lq + p.Lk - 2 ? max(p.lut[li], 0) : -1;
  };
  auto load = [&](int step) {
    const int key0 = step * KT;
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      const int id = n * 64 * NW + tid;
      const float* src = kbase + (int64_t)min(key0 + id / CPR, kv_len - 1) * p.ldk + 8 * (id % CPR);
      kx[n][0] = *reinterpret_cast<const f32x4*>(src);
      kx[n][1] = *reinterpret_cast<const f32x4*>(src + 4);
    }
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      const int u = n * NW + wave;  // unit: block u / (D/16), product step, half, 64 dims
      const int s = (u / (D / 64)) >> 1 & 1, hh = (u / (D / 64)) & 1;
      const int k0 = key0 + 32 * (u / (D / 16)) + 16 * s + 4 * hh;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = min(k0 + (j & 3) + 8 * (j >> 2), kv_len - 1);
        vx[n][j] = vbase[(int64_t)key * p.ldv + 64 * (u % (D / 64)) + lane];
      }
    }
    if constexpr (BIAS == BIAS_DENSE) {
      const int k0 = key0 + 32 * ks + 4 * half;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (key0 + 32 * ks + 32 <= p.Lk) {  // runs of 4 keys at any 4-byte alignment
          const f32x4_a4 v = *reinterpret_cast<const f32x4_a4*>(brow + k0 + 8 * g);
#pragma unroll
          for (int e = 0; e < 4; ++e) bx[4 * g + e] = v[e];
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) bx[4 * g + e] = brow[min(k0 + 8 * g + e, p.Lk - 1)];
        }
      }
    }
    if constexpr (BIAS == BIAS_RELPOS) {
      rbx = bucket >= 0 ? p.bias[min(bucket, p.num_buckets - 1) * p.H + h] : 0.f;
      load_bucket(step + 1);
    }
    if constexpr (MASK == MASK_KEY_MASK) {
      const int key = key0 + tid;
      kmx = tid < KT && key < p.Lk && kmask[min(key, p.Lk - 1)] != 0 ? 0.f : -INFINITY;
    }
  };
  auto store = [&](int stage) {
    u32x4* base = lds + stage * STAGE;
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      const int id = n * 64 * NW + tid;
      const int key = id / CPR, c = id % CPR;
      const Split8 t = split8(kx[n][0], kx[n][1]);
      u32x4* d = base + (key >> 5) * BLK + (c >> 1) * 192 + (c & 1) * 32 + ((key & 31) ^ (c & 7));
      d[0] = t.h;
      d[64] = t.m;
      d[128] = t.l;
    }
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      const int u = n * NW + wave;
      const int s = (u / (D / 64)) >> 1 & 1, hh = (u / (D / 64)) & 1;
      const int t32 = 2 * (u % (D / 64)) + half;
      const Split8 t = split8(f32x4{vx[n][0], vx[n][1], vx[n][2], vx[n][3]}, f32x4{vx[n][4], vx[n][5], vx[n][6], vx[n][7]});
      u32x4* d = base + (u / (D / 16)) * BLK + KBLK + (s * NDB + t32) * 192 + hh * 32 + col;
      d[0] = t.h;
      d[64] = t.m;
      d[128] = t.l;
    }
    if constexpr (BIAS == BIAS_DENSE) {
#pragma unroll
      for (int r = 0; r < 16; ++r) bcur[r] = bx[r];
    }
    if constexpr (BIAS == BIAS_RELPOS) {
      if (tid < RB) lds_rb[stage * RB + tid] = rbx * kLog2e;
    }
    if constexpr (MASK == MASK_KEY_MASK) {
      if (tid < KT) lds_km[stage * KT + tid] = kmx;
    }
  };

  if constexpr (BIAS == BIAS_RELPOS) load_bucket(0);
  if (nstep > 0) load(0);

  // ---- Q terms, pre-scaled: product step s holds dims 16s + 8*half + 0..7 of query qi. Times kUp, so the
  // scores come out in units of kDown. (K needs no scaling: an element below 2^-110 is short of bits by at
  // most 2^-134, which a scaled query below 2^104 turns into at most 2^-30 of a score; a larger
  // one overflows here.)
  Split8 q[FK];
  {
    const float sc = q_valid ? p.scale_log2 * kUp : 0.f;
#pragma unroll
    for (int s = 0; s < FK; ++s) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(qrow + 16 * s + 8 * half);
      const f32x4 c = *reinterpret_cast<const f32x4*>(qrow + 16 * s + 8 * half + 4);
      q[s] = split8<true>(a, c, sc);
    }
  }

  f32x16 oacc[NDB];
#pragma unroll
  for (int t = 0; t < NDB; ++t) oacc[t] = zero16();
  float m = kMaxSeed;
  float l = 0.f;

  // Scores of the 32 keys from k0 -> probabilities; moves (m, l, O) on. split: scores of the three-term
  // products, which are in units of kDown unless a bias has brought them to base 2.
  auto softmax = [&](float (&u)[16], int k0, bool first, auto split) {
    constexpr float kUnit = decltype(split)::value && BIAS == BIAS_NONE ? kDown : 1.f;
    if (MASK != MASK_KEY_MASK && k0 + 32 > kv_len) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = k0 + 8 * (r >> 2) + 4 * half + (r & 3);
        u[r] = key < kv_len ? u[r] : -INFINITY;
      }
    }
    float mb = u[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mb = max_nan(mb, u[r]);
    mb = max_with_partner(mb) * kUnit;
    if (first) {
      m = max_nan(m, mb);
    } else if (__builtin_amdgcn_ballot_w64(mb > m + kRescaleSlack) != 0) {
      const float m_new = max_nan(m, mb);
      const float alpha = fast_exp2(m - m_new);
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int t = 0; t < NDB; ++t) oacc[t] *= alpha;
    }
    u[0] = fast_exp2(fmaf(u[0], kUnit, -m));
    float ps = u[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) {
      u[r] = fast_exp2(fmaf(u[r], kUnit, -m));
      ps += u[r];
    }
    l += ps;
  };

  // scores of block blk from stage `stage` (in units of kDown, base 2 with a bias), bias and key mask added
  auto scores = [&](int stage, float (&u)[16]) {
    const u32x4* kb = lds + stage * STAGE + ks * BLK;
    f32x16 s = zero16();
#pragma unroll
    for (int i = 0; i < FK; ++i) {
      const u32x4* f = kb + i * 192 + half * 32 + (col ^ ((2 * i + half) & 7));
      const u32x4 kh = f[0], km = f[64], kl = f[128];
      s = mfma32(kl, q[i].h, s);
      s = mfma32(kh, q[i].l, s);
      s = mfma32(km, q[i].m, s);
      s = mfma32(km, q[i].h, s);
      s = mfma32(kh, q[i].m, s);
      s = mfma32(kh, q[i].h, s);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      u[r] = BIAS == BIAS_NONE ? s[r] : s[r] * kDown;
      const int e = 8 * (r >> 2) + 4 * half + (r & 3);  // the register's key in the block
      if constexpr (BIAS == BIAS_DENSE) u[r] = fmaf(bcur[r], kLog2e, u[r]);
      if constexpr (BIAS == BIAS_RELPOS) u[r] += lds_rb[stage * RB + 32 * ks + e - qi + q0 + QT - 1];
      if constexpr (MASK == MASK_KEY_MASK) u[r] += lds_km[stage * KT + 32 * ks + e];
    }
  };
  auto output = [&](int stage, const float (&pr)[16]) {
    const u32x4* vb = lds + stage * STAGE + ks * BLK + KBLK;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const Split8 pt = split8(f32x4{pr[8 * i], pr[8 * i + 1], pr[8 * i + 2], pr[8 * i + 3]},
                               f32x4{pr[8 * i + 4], pr[8 * i + 5], pr[8 * i + 6], pr[8 * i + 7]}, kUp);
#pragma unroll
      for (int t0 = 0; t0 < NDB; t0 += 2) {
        u32x4 v[2][3];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int e = 0; e < 3; ++e) v[t][e] = vb[(i * NDB + t0 + t) * 192 + e * 64 + lane];
        auto products = [&](int e, const u32x4& x) {
#pragma unroll
          for (int t = 0; t < 2; ++t) oacc[t0 + t] = mfma32(v[t][e], x, oacc[t0 + t]);
        };
        products(2, pt.h);
        products(0, pt.l);
        products(1, pt.m);
        products(1, pt.h);
        products(0, pt.m);
        products(0, pt.h);
      }
    }
  };

  if (nstep > 0) {
    store(0);
    if (nstep > 1) load(1);
  }
  __syncthreads();
  for (int step = 0; step < nstep; ++step) {
    const int stage = STAGES == 2 ? step & 1 : 0;
    const int blk = step * KS + ks;
    if (blk < nblk) {
      float u[16];
      scores(stage, u);
      softmax(u, blk * 32, step == 0, std::true_type{});
      output(stage, u);
    }
    if constexpr (STAGES == 1) __syncthreads();  // every wave is done with the stage
    if (step + 1 < nstep) {
      store(STAGES == 2 ? stage ^ 1 : 0);
      if (step + 2 < nstep) load(step + 2);
    }
    __syncthreads();
  }

  // Two kinds of values have no three terms, and a wave whose sums they may have reached takes its key blocks
  // again with fp32 products straight from memory, so such inputs give what float32 products give:
  // infinity, NaN, keys and values past the bfloat16 range and scaled queries from 2^104 up, which turn into NaN,
  // and sums past the scaled range, which turn into infinities: anything not finite in its state;
  // elements of V below 2^-110, whose terms are short by up to 2^-134, which costs an output at most 2^-134 l: one
  // that is not zero and below 2^26 times that.
  {
    float most = fabsf(l), least = INFINITY;
    const float floor = sum_with_partner(l) * (0x1p-108f * kUp);
#pragma unroll
    for (int t = 0; t < NDB; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        most = max_nan(most, fabsf(oacc[t][r]));
        least = min_nan(least, fabsf(oacc[t][r]));
      }
    bool redo = !(most < INFINITY);
    if (least < floor) {  // zeros too, which are exact: look again
#pragma unroll
      for (int t = 0; t < NDB; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) redo |= oacc[t][r] != 0.f && fabsf(oacc[t][r]) < floor;
    }
    if (__builtin_amdgcn_ballot_w64(redo) != 0) {
#pragma unroll
      for (int t = 0; t < NDB; ++t) oacc[t] = zero16();
      m = kMaxSeed;
      l = 0.f;
      const float sc = q_valid ? p.scale_log2 : 0.f;
#pragma unroll 1
      for (int blk = ks; blk < nblk; blk += KS) {
        const float* krow = kbase + (int64_t)min(blk * 32 + col, kv_len - 1) * p.ldk;
        f32x16 s = zero16();
#pragma unroll 1
        for (int d = 0; d < D; d += 2) s = __builtin_amdgcn_mfma_f32_32x32x2f32(krow[d + half], qrow[d + half] * sc, s, 0, 0, 0);
        float pr[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = blk * 32 + 8 * (r >> 2) + 4 * half + (r & 3), kc = min(key, p.Lk - 1);
          pr[r] = s[r];
          if constexpr (BIAS == BIAS_DENSE) pr[r] = fmaf(brow[kc], kLog2e, pr[r]);
          if constexpr (BIAS == BIAS_RELPOS) {
            const int bk = min(max(p.lut[kc - min(qi, p.Lq - 1) + p.Lq - 1], 0), p.num_buckets - 1);
            pr[r] = fmaf(p.bias[bk * p.H + h], kLog2e, pr[r]);
          }
          if constexpr (MASK == MASK_KEY_MASK) pr[r] += key < p.Lk && kmask[kc] != 0 ? 0.f : -INFINITY;
        }
        softmax(pr, blk * 32, blk == ks, std::false_type{});
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float* vrow = vbase + (int64_t)min(blk * 32 + 8 * (r >> 2) + 4 * half + (r & 3), kv_len - 1) * p.ldv + col;
#pragma unroll
          for (int t = 0; t < NDB; ++t) oacc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(vrow[32 * t], pr[r], oacc[t], 0, 0, 0);
        }
      }
    } else {
#pragma unroll
      for (int t = 0; t < NDB; ++t) oacc[t] *= kDown;  // P was scaled
    }
  }

  // ---- merge the key splits: waves ks > 0 publish (O, m, l), wave ks == 0 combines
  float* const ldsf = reinterpret_cast<float*>(lds);
  if constexpr (KS > 1) {
    if (ks > 0) {
      float* rec = ldsf + ((ks - 1) * QG + qg) * 64 * MSTRIDE + lane;
#pragma unroll
      for (int t = 0; t < NDB; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) rec[(16 * t + r) * 64] = oacc[t][r];
      rec[(16 * NDB) * 64] = m;
      rec[(16 * NDB + 1) * 64] = l;
    }
    __syncthreads();
    if (ks > 0) return;
    float mt = m;
#pragma unroll
    for (int sp = 1; sp < KS; ++sp) mt = fmaxf(mt, ldsf[((sp - 1) * QG + qg) * 64 * MSTRIDE + lane + (16 * NDB) * 64]);
    const float a0 = fast_exp2(m - mt);
    l *= a0;
#pragma unroll
    for (int t = 0; t < NDB; ++t) oacc[t] *= a0;
#pragma unroll
    for (int sp = 1; sp < KS; ++sp) {
      const float* o2 = ldsf + ((sp - 1) * QG + qg) * 64 * MSTRIDE + lane;
      const float a = fast_exp2(o2[(16 * NDB) * 64] - mt);
      l = fmaf(o2[(16 * NDB + 1) * 64], a, l);
#pragma unroll
      for (int t = 0; t < NDB; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[t][r] = fmaf(o2[(16 * t + r) * 64], a, oacc[t][r]);
    }
  }

  // ---- normalise and store: lane holds O[qi][32t + 8g + 4*half + 0..3] in registers 4g..4g+3
  const float lt = sum_with_partner(l);
  const float inv = lt > 0.f ? __builtin_amdgcn_rcpf(lt) : 0.f;  // v_rcp_f32 (1 ulp)
  if constexpr (KS == 1) {
    // through LDS, as whole rows (16-byte chunks swizzled by row); each wave its own 32 x D tile
    constexpr int CPO = D / 4;       // 16-byte chunks per row
    constexpr int RPI = 64 / CPO;    // rows per store instruction
    float* ot = ldsf + wave * 32 * D;
#pragma unroll
    for (int t = 0; t < NDB; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 x = {oacc[t][4 * g] * inv, oacc[t][4 * g + 1] * inv, oacc[t][4 * g + 2] * inv, oacc[t][4 * g + 3] * inv};
        *reinterpret_cast<f32x4*>(ot + col * D + 4 * ((8 * t + 2 * g + half) ^ (col & 15))) = x;
      }
    const int rsub = lane / CPO, cidx = lane % CPO;
    float* obase = p.o + (int64_t)b * p.so + h * D;
#pragma unroll
    for (int j = 0; j < 32 / RPI; ++j) {
      const int row = RPI * j + rsub;
      const f32x4 x = *reinterpret_cast<const f32x4*>(ot + row * D + 4 * (cidx ^ (row & 15)));
      const int orow = q0 + qg * 32 + row;
      // non-temporal: O is not read again here, and K/V tiles of the neighbouring workgroups stay in the L2
      if (orow < p.Lq) __builtin_nontemporal_store(x, reinterpret_cast<f32x4*>(obase + (int64_t)orow * p.ldo + 4 * cidx));
    }
  } else if (q_valid) {
    float* dst = p.o + (int64_t)b * p.so + (int64_t)qi * p.ldo + h * D + 4 * half;
#pragma unroll
    for (int t = 0; t < NDB; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 x = {oacc[t][4 * g] * inv, oacc[t][4 * g + 1] * inv, oacc[t][4 * g + 2] * inv, oacc[t][4 * g + 3] * inv};
        *reinterpret_cast<f32x4*>(dst + 32 * t + 8 * g) = x;
      }
  }
}

template <int D, int QG, int KS, int STAGES, int WPE, int BIAS, int MASK>
hipError_t launch_one(const AttnParams& p, hipStream_t stream) {
  const int64_t n = (int64_t)p.B * p.H * ((p.Lq + 32 * QG - 1) / (32 * QG));
  if (n > 0x7fffffff) return hipErrorInvalidConfiguration;
  const FlashArgs a = flash_args(p, n);
  const dim3 grid((unsigned)n), block(64 * QG * KS);
  if constexpr (MASK == MASK_KEY_LEN_ORDERED) {
    FlashOrder ord;
    memcpy(ord.order, p.order, sizeof ord.order);
    hipLaunchKernelGGL((flash_split_kernel<D, QG, KS, STAGES, WPE, BIAS, MASK, FlashOrder>), grid, block, 0, stream, a, ord);
  } else {
    hipLaunchKernelGGL((flash_split_kernel<D, QG, KS, STAGES, WPE, BIAS, MASK, NoOrder>), grid, block, 0, stream, a, NoOrder{});
  }
  return hipGetLastError();
}

template <int D, int QG, int KS, int STAGES, int WPE, int BIAS>
hipError_t launch_mask(const AttnParams& p, hipStream_t stream) {
  switch (p.mask_mode) {
    case MASK_NONE: return launch_one<D, QG, KS, STAGES, WPE, BIAS, MASK_NONE>(p, stream);
    case MASK_KEY_LEN:
      if (p.order_n > 0) return launch_one<D, QG, KS, STAGES, WPE, BIAS, MASK_KEY_LEN_ORDERED>(p, stream);
      return launch_one<D, QG, KS, STAGES, WPE, BIAS, MASK_KEY_LEN>(p, stream);
    case MASK_KEY_MASK: return launch_one<D, QG, KS, STAGES, WPE, BIAS, MASK_KEY_MASK>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

template <int D, int QG, int KS, int STAGES, int WPE>
hipError_t launch_bias(const AttnParams& p, hipStream_t stream) {
  switch (p.bias_mode) {
    case BIAS_NONE: return launch_mask<D, QG, KS, STAGES, WPE, BIAS_NONE>(p, stream);
    case BIAS_DENSE: return launch_mask<D, QG, KS, STAGES, WPE, BIAS_DENSE>(p, stream);
    case BIAS_RELPOS: return launch_mask<D, QG, KS, STAGES, WPE, BIAS_RELPOS>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

// Groups of 32 queries x key splits per workgroup, [stages], by the workgroups a launch makes. Means of
// 1416 (head dim 128) and 888 (64) calls of 1 to 58 sequences x 4 to 12 heads, 4 to 700 queries, 8 to 1000 keys, with and without
// dense bias and key lengths, as a ratio to the fp32 MFMA kernel that these replaced:
//   head dim 64                                       2x2 [2]  2x2 [1]  2x4 [1]  4x2 [2]  4x1 [2]
//     up to 256 workgroups of 64 queries, 2-4 blocks    0.91     0.92     1.04     1.18     1.11
//       5-10 blocks                                     0.85     0.89     0.90     1.04     1.16
//       more                                            0.80     0.85     0.71     0.93     1.14
//     at most 64 queries, more workgroups, 2+ blocks    1.08     0.83     1.05     1.23     1.03
//     up to 256 of 128 queries, 2 / 3-4 blocks          1.2      0.9      1.3      0.95/0.78  0.83/0.76
//       5-10 blocks                                     1.03     0.81     1.09     0.71     0.75
//     more                                              1.1-1.5  0.7-1.0  0.9-1.9  0.7-1.3  0.62-0.74
//     one block of keys                                 1.0-2.3  0.9-1.5  1.2-3.0  1.1-1.7  0.71-0.91
//   head dim 128                                      2x2 [1]  4x1 [2]  4x1 [1], no bias
//     one block of keys                                 1.0-1.8  0.87-1.0  0.9-1.2
//     up to 128 units of 128 queries                    0.71-0.99  1.04-1.2  1.4-2.2
//     257-512 units, 3+ blocks                          0.90     0.94     0.92 (600 units of 1000 keys 168 us against 201)
//     more                                              0.7-1.1  0.56-0.83  0.78-0.84
// Head dim 64 therefore counts the workgroups of a shape; head dim 128, where one workgroup fills a CU, takes the
// least of three estimates fitted to the same calls (us per round of workgroups). 4x1 [1] puts two workgroups
// on a CU at 256 registers a wave and spills 47 to 65 of them, more with a bias (1.4 times the fp32 kernel):
// it is not compiled with one.
FlashShape flash_shape(const AttnParams& p, int num_cus) {
  const int64_t units = (int64_t)p.B * p.H * ((p.Lq + 127) / 128), half_units = (int64_t)p.B * p.H * ((p.Lq + 63) / 64);
  const int nblk = (p.Lk + 31) / 32;
  if (nblk == 1) return {4, 1, 2};
  if (p.D == 64) {
    if (half_units <= num_cus) return nblk <= 8 ? FlashShape{2, 2, 2} : FlashShape{2, 4, 1};
    if (p.Lq <= 64) return {2, 2, 1};
    if (units <= num_cus && nblk > 8) return {4, 2, 2};
    return {4, 1, 2};
  }
  const int64_t per_cu = (units + num_cus - 1) / num_cus, half_per_cu = (half_units + num_cus - 1) / num_cus;
  const bool bias = p.bias_mode != BIAS_NONE;
  const int steps = (nblk + 1) / 2;  // of two blocks
  const double split = (double)half_per_cu * (bias ? 6.2 + 4.45 * steps : 5.4 + 4.1 * steps);
  const double whole = (double)per_cu * (bias ? 5.9 + 3.5 * nblk : 5.5 + 2.98 * nblk);
  const double pairs = 1.03 * ((double)(per_cu / 2) * (10 + 5.8 * nblk) + (double)(per_cu % 2) * (6 + 3.9 * nblk));
  if (!bias && pairs < std::min(split, whole)) return {4, 1, 1};
  return split < whole ? FlashShape{2, 2, 1} : FlashShape{4, 1, 2};
}

hipError_t launch_flash_split(const AttnParams& p, int num_cus, hipStream_t stream) {
  const FlashShape s = flash_shape(p, num_cus);
  if (p.D == 64) {
    if (s.groups == 2 && s.splits == 4) return launch_bias<64, 2, 4, 1, 2>(p, stream);
    if (s.groups == 2) return s.stages == 2 ? launch_bias<64, 2, 2, 2, 2>(p, stream) : launch_bias<64, 2, 2, 1, 2>(p, stream);
    return s.splits == 2 ? launch_bias<64, 4, 2, 2, 2>(p, stream) : launch_bias<64, 4, 1, 2, 2>(p, stream);
  }
  if (p.D == 128) {
    if (s.groups == 2) return launch_bias<128, 2, 2, 1, 1>(p, stream);
    return s.stages == 2 ? launch_bias<128, 4, 1, 2, 1>(p, stream) : launch_mask<128, 4, 1, 1, 2, BIAS_NONE>(p, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace sa
