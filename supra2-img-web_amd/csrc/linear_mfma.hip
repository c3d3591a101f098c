// Linear layer y = epilogue(alpha * x W^T) on the matrix cores of gfx950: the projections either side of
// the attention operator (app/gpu/ops.js:35-43 `linear`, app/gpu/gemm.js:116-223 `matmulShader`
// with A mode "rows" and B format "f32"): the DiT qkv / proj / q / kv / cproj / fc1 / fc2 layers.
//
//   x [M, K] rows at x + x_off + m*ldx;  W [N, K] (PyTorch layout) rows at w + n*ldw
//   r = alpha * sum_k x[m][k] W[n][k] (+ bias[n]), then act (GELU erf / GELU tanh / SiLU), then
//   y[m][n] = r, y[m][n] += r, or y[m][n] += gate[gate_off + n] * r (gemm.js:127-137).
//
// Three kernels: linear_split_kernel (large and medium grids, bf16 matrix cores, described there),
// linear_mfma_kernel (fp32 MFMA, grids between those and the small ones) and linear_ksplit_kernel (small
// grids, fp32 MFMA); split_tile and linear_class choose. Any other alignment: linear_generic_kernel.
//
// Work decomposition of linear_mfma_kernel
//   A workgroup is 4 wave64s in a 2 x 2 grid computing a 64 x 64 tile; each wave owns 32 x 32 outputs, one
//   accumulator of v_mfma_f32_32x32x2f32. The x rows are the MFMA A operand and the W rows the B operand, so
//   lane l of an accumulator holds column n = l%32 and rows 8*(r/4) + 4*(l/32) + r%4 of register r:
//   every store instruction writes 128 contiguous bytes of two rows.
//   K advances in tiles of 32. Within a group of 8 consecutive k, half-wave h supplies
//   k = 8g + 4h + s at MFMA step s (s = 0..3): one b128 LDS read per operand row and group feeds
//   four MFMAs, and every (x, W) pair of k meets exactly once.
//
// Tiles move HBM/L2 -> LDS with buffer_load_dwordx4 ... lds (no VGPR staging; scalar descriptor and
// k offset, loop-invariant lane offsets), two stages, one barrier per k-tile. The k-loop advances two
// tiles at a time so every stage index is a compile-time constant: the steady-state loop issues
// no VALU instruction, which on gfx950 would serialize with the MFMAs of the SIMD. LDS rows are
// 32 floats (8 chunks of 16 bytes); chunk c of row r sits at c ^ ((r / 2) % 8) (two rows per 256
// bytes), which makes the b128 operand reads of 16 consecutive rows
// conflict-free (measured SQ_LDS_BANK_CONFLICT = 0). The operands of the next
// group of 8 k are read from LDS while the MFMAs of the current group run, and the barrier of the
// next k-tile sits before the last group's MFMAs.
//
// The epilogue shares the SIMD datapath with the fp32 MFMAs, so it is kept short: activation and
// store mode are template parameters (no per-element branches), stores are raw buffer stores with
// scalar descriptors and row offsets, whole tiles skip the bounds checks.
// Rows past M (x) or N (W) re-read the last row (finite data, never stored); the k-tile holding K
// clamps its column to K - 8 and only its valid groups of 8 are multiplied (K % 8 == 0).
//
// Tile order (TileOrder): consecutive tiles run on one XCD (xcd_remap), and the tiles are cut into
// row super-blocks of about one XCD's share of the x row blocks. Inside a super-block the N tiles go
// in groups of W panels small enough to stay in the XCD's 4 MB L2 (the host sizes the groups), and
// inside a group the row blocks go in turn, each with the group's panels. A row block's x rows are
// then read once per group, while they are hot, and a panel once per super-block, instead of all
// of W cycling through the L2 once per row block.

#include <algorithm>
#include <type_traits>

#include <cstring>

#include "common.h"
#include "kernels.h"
#include "split.h"


namespace sa {

namespace {

// Activations of app/gpu/gemm.js:21-36. The epilogue runs on the same SIMD datapath as the fp32
// MFMAs, so the two logistic forms use one hardware exp2 and one reciprocal:
//   GELU (tanh) 0.5 x (1 + tanh(u)) = x / (1 + e^(-2u)),  u = sqrt(2/pi) (x + 0.044715 x^3);
//   SiLU        x / (1 + e^(-x)).
// Both saturate correctly: e^(...) -> inf gives x * 0, e^(...) -> 0 gives x. GELU (erf) calls erff.
__device__ __forceinline__ float logistic_times(float x, float z) {  // x / (1 + e^z)
  return x * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(z * kLog2e));
}

template <int ACT>
__device__ __forceinline__ float apply_act(float v) {
  if constexpr (ACT == LIN_ACT_GELU) return 0.5f * v * (1.f + erff(v * 0.70710678118654752f));
  if constexpr (ACT == LIN_ACT_GELU_TANH) {
    const float u = v * fmaf(0.035677408136300125f, v * v, 0.79788456080286536f);  // sqrt(2/pi) * (1, 0.044715)
    return logistic_times(v, -2.f * u);
  }
  if constexpr (ACT == LIN_ACT_SILU) return logistic_times(v, -v);
  return v;
}

// Row block and N tile of logical tile t: super-blocks of sb_rows row blocks (the last may be
// shorter), inside one the N tiles in groups of group_n (the last may be narrower), inside a group
// the row blocks, each with the group's N tiles. Bijective on [0, tiles_m * tiles_n).
struct TileOrder {
  int tiles_m, tiles_n, group_n, sb_rows;
};

// Arguments of the MFMA kernels: 80 bytes, 96 with the tile order (launches with at most 112 bytes
// of explicit arguments start sooner). Pointers carry the callers' element offsets, resid is the
// residual rows (y itself when the caller gave none), and the row strides fit 32 bits under
// linear_mfma_supported.
struct LinArgs {
  const float* x;
  const float* w;
  const float* bias;
  const float* gate;
  float* y;
  const float* resid;
  int32_t ldx, ldw, ldy;
  int32_t M, N, K;
  float alpha;
};
static_assert(sizeof(LinArgs) + sizeof(TileOrder) <= 112, "linear kernel arguments must stay within 112 bytes");

__device__ __forceinline__ void tile_coords(int t, const TileOrder& o, int& mi, int& ni) {
  const int sb_tiles = o.sb_rows * o.tiles_n;
  const int sb = t / sb_tiles;
  const int rem = t - sb * sb_tiles;
  const int rows = min(o.sb_rows, o.tiles_m - sb * o.sb_rows);
  const int g = rem / (rows * o.group_n);
  const int off = rem - g * rows * o.group_n;
  const int w = min(o.group_n, o.tiles_n - g * o.group_n);
  mi = sb * o.sb_rows + off / w;
  ni = g * o.group_n + off % w;
}

// Waves per SIMD that the register budget of linear_split_kernel is set for (its VGPRs: 64 x 64 106,
// 64 x 96 116, 128 x 96 168, 256 x 144 198, 256 x 192 228; no scratch).
template <int NW, int MT, int NT>
constexpr int split_waves_per_simd() {
  return MT * NT <= 6 ? 4 : MT * NT <= 12 ? 3 : 2;
}

// Rows [m0, m0 + rows) x columns [n0, n0 + cols) in fp32 products straight from memory, by one wave (lane =
// 16 lc + lr), 16 x 16 outputs at a time and stored from here: merged with the caller's accumulators and
// epilogue instead, it cost the main loop up to 6% (fc2 of 16384 rows 209 -> 196 us without).
template <int ACT, int EPI>
__device__ __forceinline__ void redo_tile(const LinArgs& p, int m0, int n0, int rows, int cols, int lr, int lc) {
#pragma unroll 1
  for (int mt = m0; mt < min(m0 + rows, p.M); mt += 16) {
#pragma unroll 1
    for (int nt = n0; nt < min(n0 + cols, p.N); nt += 16) {
      const float* x = p.x + (int64_t)min(mt + lr, p.M - 1) * p.ldx + lc;
      const float* w = p.w + (int64_t)min(nt + lr, p.N - 1) * p.ldw + lc;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int k = 0; k < p.K; k += 4) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[k], x[k], acc, 0, 0, 0);
      const int m = mt + lr;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = nt + 4 * lc + e;
        if (m >= p.M || n >= p.N) continue;
        float v = apply_act<ACT>(fmaf(acc[e], p.alpha, p.bias ? p.bias[n] : 0.f));
        const int64_t at = (int64_t)m * p.ldy + n;
        if constexpr (EPI != LIN_EPI_STORE) v = fmaf(EPI == LIN_EPI_RESID_GATE ? p.gate[n] : 1.f, v, p.resid[at]);
        p.y[at] = v;
      }
    }
  }
}

// Large and medium grids: the product on the bf16 matrix cores, each float32 operand as three bfloat16
// terms (split.h) and each product as the six term products of 2^-24 and more of its size, smallest
// first, summed in the float32 accumulators: x w ~ xl wh + xh wl + xm wm + xm wh + xh wm + xh wh.
// Error against 64 bits (2-norm, N(0, 1) rows, K = 576 / 2304): 3.6e-7 / 7.4e-7, the fp32 MFMA chain
// 4.3e-7 / 8.6e-7: one rounding per 32 k and term product instead of one per 2 k, and the terms
// dropped are below the rounding of the sum.
//
// A workgroup is NW waves stacked along the rows; a wave owns 16*MT rows x 16*NT columns as MT x NT
// accumulators of v_mfma_f32_16x16x32_bf16. W is the A operand and x the B operand, so a lane holds 4
// consecutive columns of one row and stores 16 bytes. Each wave loads its own x rows straight into the
// operand layout (nobody shares them) and splits them in registers; the 16-column fragments of W are
// dealt to the waves, which split them and leave the terms in LDS in operand order (every access is one
// contiguous 1 KB row: no bank conflicts), two stages, one barrier per 32 k. So each element of W is
// split once per row block, and an LDS read of one term feeds MT or more MFMAs.
//
// What bounds it: the matrix cores at the clock they hold under this load (random operands: 2.06 of
// the nominal 2.5 PFLOP/s measured with nothing but these MFMAs, i.e. 344 TFLOP/s of products) and the
// issue slots the split takes beside them (11 VALU instructions per two elements; without the split,
// results discarded, 263 TFLOP/s at K = 2304, with it 235, with the row norms of the retry 225). 16x16x32 measured faster than 32x32x16 on
// whole grids (qkv layer of 16384 rows 160 against 191-211 us), and 8 waves over 256 rows faster than
// twice 4 waves over 128 (half the W splits).
template <int NW, int MT, int NT, int ACT, int EPI>
__global__ __launch_bounds__(64 * NW, (split_waves_per_simd<NW, MT, NT>())) void linear_split_kernel(LinArgs p, TileOrder order) {
  constexpr int BM = 16 * MT * NW, BN = 16 * NT, BK = 32;
  constexpr int GW = NT % 3 == 0 ? 3 : 2;   // column fragments per group: MT * GW independent chains
  constexpr int G = NT / GW;
  constexpr int NF = (NT + NW - 1) / NW;    // W fragments per wave (the last waves may have one less)
  constexpr int STAGE = NT * 3 * 64;        // 16-byte chunks per stage: [fragment][term][lane]
  // Sums per output: two on the smallest tile, which takes calls of the two-split fp32 kernel and must not be
  // less exact: the products of first terms, and all others, whose sum is too small to round them (2-norm at
  // K = 576 / 2304: 1.4e-7 / 2.9e-7, in one sum 3.6e-7 / 7.4e-7, that kernel 3.05e-7 / 6.1e-7)
  constexpr int CH = MT * NT <= 4 ? 2 : 1;
  static_assert(G * GW == NT, "column fragments must split into groups");

  __shared__ u32x4 lds[2 * STAGE];
  __shared__ unsigned lds_norm;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15;  // operand row (x row or W row) of the lane
  const int lc = lane >> 4;  // its 8 consecutive k of every 32

  int mi, ni;
  tile_coords(xcd_remap(blockIdx.x, order.tiles_m * order.tiles_n), order, mi, ni);
  const int mw = mi * BM + wave * 16 * MT;  // the wave's first row; waves past M re-read the last row
  const int n0 = ni * BN;
  const int mb = min(mw, p.M - 1);
  const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(p.x + (int64_t)mb * p.ldx);
  const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(p.w + (int64_t)n0 * p.ldw);
  unsigned xoff[MT], woff[NF];
#pragma unroll
  for (int i = 0; i < MT; ++i) xoff[i] = 4u * (unsigned)(min(16 * i + lr, p.M - 1 - mb) * p.ldx + 8 * lc);
#pragma unroll
  for (int f = 0; f < NF; ++f) woff[f] = 4u * (unsigned)(min(16 * (f * NW + wave) + lr, p.N - 1 - n0) * p.ldw + 8 * lc);
  const int nkt = (p.K + BK - 1) / BK;
  const int nfull = p.K / BK;  // whole k-tiles; with K % 32 != 0 the last tile (nfull) holds K

  f32x4 xa[MT][2], wb[NF][2];  // the next k-tile as loaded
  auto load = [&](int kt) {
    const unsigned s = 4u * (unsigned)(kt * BK);
    unsigned back = 0;  // chunks of 8 k past K re-read the last one (zeroed by cut)
    if (kt >= nfull) back = 4u * (unsigned)max(kt * BK + 8 * lc + 8 - p.K, 0);
    auto ld = [&](__amdgpu_buffer_rsrc_t r, unsigned v) {
      return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, v, s, 0));
    };
#pragma unroll
    for (int f = 0; f < NF; ++f)
      if (f * NW + wave < NT) {
        wb[f][0] = ld(wr, woff[f] - back);
        wb[f][1] = ld(wr, woff[f] - back + 16);
      }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      xa[i][0] = ld(xr, xoff[i] - back);
      xa[i][1] = ld(xr, xoff[i] - back + 16);
    }
  };
  auto cut = [&](int kt) {
    if (kt >= nfull && kt * BK + 8 * lc >= p.K) {
#pragma unroll
      for (int f = 0; f < NF; ++f) wb[f][0] = wb[f][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < MT; ++i) xa[i][0] = xa[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  f32x4 norm = {0.f, 0.f, 0.f, 0.f};  // on its diagonal, sums of squares over the rows of x and W that the wave splits
  auto put = [&](int f, int stage) {
    if (f * NW + wave < NT) {
      const Split8 s = split8(wb[f][0], wb[f][1]);
      u32x4* d = lds + stage * STAGE + (f * NW + wave) * 192 + lane;
      d[0] = s.h;
      d[64] = s.m;
      d[128] = s.l;
      norm = mfma16(s.h, s.h, norm);
    }
  };
  Split8 a[2][MT];
  f32x4 acc[CH][MT][NT];
#pragma unroll
  for (int c = 0; c < CH; ++c)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[c][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // k-tile kt from stage C; the splits of the next tile go between the groups' MFMAs
  auto step = [&](int kt, auto stage) {
    constexpr int C = decltype(stage)::value;
    const bool more = kt + 1 < nkt;
    if (more) cut(kt + 1);
#pragma unroll
    for (int i = 0; i < MT; ++i) norm = mfma16(a[C][i].h, a[C][i].h, norm);
    static_for<G>([&](auto gg) {
      constexpr int g = decltype(gg)::value;
      u32x4 b[GW][3];
#pragma unroll
      for (int j = 0; j < GW; ++j)
#pragma unroll
        for (int t = 0; t < 3; ++t) b[j][t] = lds[C * STAGE + (g * GW + j) * 192 + t * 64 + lane];
      auto products = [&](int t, auto term, int ch = 0) {
#pragma unroll
        for (int j = 0; j < GW; ++j)
#pragma unroll
          for (int i = 0; i < MT; ++i) acc[ch][i][g * GW + j] = mfma16(b[j][t], term(a[C][i]), acc[ch][i][g * GW + j]);
      };
      products(2, [](const Split8& s) { return s.h; });
      products(0, [](const Split8& s) { return s.l; });
      products(1, [](const Split8& s) { return s.m; });
      products(1, [](const Split8& s) { return s.h; });
      products(0, [](const Split8& s) { return s.m; });
      products(0, [](const Split8& s) { return s.h; }, CH - 1);
      if (more) {
#pragma unroll
        for (int f = 0; f < NF; ++f)
          if (f % G == g) put(f, C ^ 1);
#pragma unroll
        for (int i = 0; i < MT; ++i)
          if ((i + NF) % G == g) a[C ^ 1][i] = split8(xa[i][0], xa[i][1]);
      }
    });
    if (kt + 2 < nkt) load(kt + 2);
    __syncthreads();
  };
  if (tid == 0) lds_norm = 0;
  load(0);
  cut(0);
#pragma unroll
  for (int f = 0; f < NF; ++f) put(f, 0);
#pragma unroll
  for (int i = 0; i < MT; ++i) a[0][i] = split8(xa[i][0], xa[i][1]);
  if (nkt > 1) load(1);
  __syncthreads();
  int kt = 0;
  for (; kt + 2 <= nkt; kt += 2) {
    step(kt, std::integral_constant<int, 0>{});
    step(kt + 1, std::integral_constant<int, 1>{});
  }
  if (kt < nkt) step(kt, std::integral_constant<int, 0>{});
  if constexpr (CH == 2) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[0][i][j] += acc[1][i][j];
  }

  // Two kinds of operands have no three terms, and a wave whose sums they may have reached takes its whole tile
  // again with fp32 MFMAs straight from memory, so such inputs give what float32 products give:
  // infinity, NaN and magnitudes that round past the bfloat16 range, whose differences turn into NaN: anything
  // not finite in the sums;
  // magnitudes below 2^-110, whose terms are short by up to 2^-134. That costs a sum at most 2^-134 (|x|_1 + |w|_1)
  // <= 2^-133 sqrt(K) n, with n^2 the largest sum of squares over a row of x or W: a sum below 2^26 times that
  // (zeros, which are mostly those of zero rows, only where it may be more than 2^-106 off). The squares come from the matrix cores, which have the time: one product of each
  // fragment's first terms with themselves per 32 k. (Scaling every operand by 2^24 instead, at 2 VALU
  // instructions per pair, took 10 to 20% longer: 16384 x 576 x 576 62.7 us against 56.6.)
  if (lr >> 2 == lc) atomicMax(&lds_norm, __float_as_uint(norm[lr & 3]));
  float most = 0.f, least = INFINITY;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        most = max_nan(most, fabsf(acc[0][i][j][e]));
        least = min_nan(least, fabsf(acc[0][i][j][e]));
      }
  __syncthreads();
  const float floor = 0x1p-107f * sqrtf(static_cast<float>(p.K)) * sqrtf(__uint_as_float(lds_norm));
  bool redo = !(most < INFINITY);
  if (!(least >= floor)) {  // look again: zeros are exact, or off by no more than 2^-106
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) redo |= !(fabsf(acc[0][i][j][e]) >= floor) && (acc[0][i][j][e] != 0.f || floor > 0x1p-80f);
  }
  if (__builtin_amdgcn_ballot_w64(redo) != 0) {
    redo_tile<ACT, EPI>(p, mw, n0, 16 * MT, BN, lr, lc);
    return;
  }

  // ---- epilogue: lane holds columns n0 + 16j + 4*lc .. +3 of row mw + 16i + lr. Rows, bias and gate are
  // read and written 16 bytes at a time at any alignment, element by element at the edge of N. Plain stores are
  // non-temporal where four lanes write a whole 64-byte piece: y is not read back here, and keeping it out
  // of the L2 leaves the W panels and x rows there. Rows at other alignments need the L2 to put their lines
  // together (5714 x 1107 x 56 in rows of 1108: 22.6 us non-temporal, 15.6 without); the residual
  // epilogues, which have just read their rows, keep the default policy too.
  const bool whole = (reinterpret_cast<uintptr_t>(p.y) & 63) == 0 && (p.ldy & 15) == 0;
  auto load4 = [&](const float* src, int left) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (left >= 4) return f32x4(*reinterpret_cast<const f32x4_a4*>(src));
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < left) v[e] = src[e];
    return v;
  };
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = mw + 16 * i + lr;
    if (m >= p.M) continue;
    const int nl = n0 + 4 * lc;
    const int64_t row = (int64_t)m * p.ldy;
    f32x4 old[EPI != LIN_EPI_STORE ? NT : 1];
    if constexpr (EPI != LIN_EPI_STORE) {  // the old values of the row together, then combined
#pragma unroll
      for (int j = 0; j < NT; ++j)
        if (nl + 16 * j < p.N) old[j] = load4(p.resid + row + nl + 16 * j, p.N - nl - 16 * j);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int n = nl + 16 * j;
      const int left = p.N - n;
      if (left <= 0) continue;
      f32x4 v = {0.f, 0.f, 0.f, 0.f}, g = {1.f, 1.f, 1.f, 1.f};
      if (p.bias) v = load4(p.bias + n, left);
      if constexpr (EPI == LIN_EPI_RESID_GATE) g = load4(p.gate + n, left);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = apply_act<ACT>(fmaf(acc[0][i][j][e], p.alpha, v[e]));
        if constexpr (EPI != LIN_EPI_STORE) v[e] = fmaf(g[e], v[e], old[j][e]);
      }
      float* dst = p.y + row + n;
      if (EPI == LIN_EPI_STORE && whole && left >= 4) {
        __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(dst));
      } else if (left >= 4) {
        *reinterpret_cast<f32x4_a4*>(dst) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (e < left) dst[e] = v[e];
      }
    }
  }
}

// 64 x 64 tiles, one 32 x 32 accumulator per wave, 32 k per tile, two tiles in flight (LDS stages); the
// activation and the epilogue are compile-time, so the store loop has no per-element branches.
template <int ACT, int EPI>
__global__ __launch_bounds__(256, 2) void linear_mfma_kernel(LinArgs p, TileOrder order) {
  constexpr int BM = 64, BN = 64, BK = 32;
  constexpr int CPR = BK / 4;            // 16-byte chunks per tile row
  constexpr int RP = 64 / BK;            // tile rows per 256 bytes (one pass over the 64 banks)
  constexpr int NG = BK / 8;             // groups of 8 k per tile
  constexpr int A_TILE = BM * BK;        // floats per stage
  constexpr int B_TILE = BN * BK;
  constexpr int STAGE = A_TILE + B_TILE;
  constexpr int NI = BM * CPR / 256;     // DMA instructions per wave, operand and stage (64 chunks each)
  static_assert(NI * 256 == BM * CPR && BM == BN, "tiles must split into whole wave copies");
  static_assert(NG % 2 == 0, "an even number of groups per tile");

  __shared__ __attribute__((aligned(16))) float lds[2 * STAGE];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1;
  const int wn = wave & 1;
  const int col = lane & 31;
  const int half = lane >> 5;

  int mi, ni;
  tile_coords(xcd_remap(blockIdx.x, order.tiles_m * order.tiles_n), order, mi, ni);
  const int m0 = mi * BM;
  const int n0 = ni * BN;
  const float* xbase = p.x + (int64_t)m0 * p.ldx;
  const float* wbase = p.w + (int64_t)n0 * p.ldw;
  const int mlast = min(BM, p.M - m0) - 1;  // last valid tile row
  const int nlast = min(BN, p.N - n0) - 1;

  // Per-lane byte offsets (from the tile's first row at k = 0) of this lane's 16-byte chunk in
  // each DMA instruction: instruction n of wave w fills physical chunks (n*4 + w)*64 + lane; the
  // chunk c of row r sits at physical chunk c ^ ((r / RP) % CPR).
  unsigned aoff[NI], boff[NI];
  int kcol[NI];  // logical column (floats) of the chunk, for the clamped k-tile
#pragma unroll
  for (int n = 0; n < NI; ++n) {
    const int pc_all = (n * 4 + wave) * 64 + lane;
    const int row = pc_all / CPR;
    const int c = (pc_all % CPR) ^ ((row / RP) % CPR);
    kcol[n] = 4 * c;
    aoff[n] = 4u * (unsigned)(min(row, mlast) * (int)p.ldx + 4 * c);
    boff[n] = 4u * (unsigned)(min(row, nlast) * (int)p.ldw + 4 * c);
  }

  // Copies through buffer descriptors: the tile's first row is the descriptor base (scalar), the
  // k-tile's column offset the scalar soffset, and the lane's row/chunk offset a loop-invariant
  // 32-bit voffset, so the copies need no per-lane address arithmetic (VALU work serializes with
  // the MFMAs on a SIMD).
  const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(xbase);
  const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(wbase);
  const int nkt = (p.K + BK - 1) / BK;
  const int nfull = p.K / BK;  // whole k-tiles; with K % BK != 0 the last tile (nfull) holds K
  // Copies of k-tile kt into LDS stage S. The stage is a compile-time constant (the main loop
  // advances two tiles at a time), so every LDS address below is a constant offset.
  auto issue = [&](int kt, auto stage) {
    constexpr int S = decltype(stage)::value;
    float* at = lds + S * STAGE;
    float* bt = at + A_TILE;
    // the tile holding K (always tile nfull, so its offsets are loop-invariant): columns at or
    // past K re-read the last group (never multiplied)
    const bool last = kt >= nfull;
    const int k0 = last ? nfull * BK : kt * BK;
    const unsigned soff = 4u * (unsigned)k0;
    const int kmax = p.K - 8 - k0;
    unsigned back[NI];  // whole groups back
#pragma unroll
    for (int n = 0; n < NI; ++n) back[n] = last && kcol[n] > kmax + 4 ? 4u * (unsigned)((kcol[n] & ~7) - kmax) : 0u;
#pragma unroll
    for (int n = 0; n < NI; ++n) buffer_to_lds16(xr, aoff[n] - back[n], at + (n * 4 + wave) * 256, soff);
#pragma unroll
    for (int n = 0; n < NI; ++n) buffer_to_lds16(wr, boff[n] - back[n], bt + (n * 4 + wave) * 256, soff);
  };

  f32x16 acc = zero16();

  // LDS read offsets (floats) of this lane's operand chunk in group g: row `col` of the
  // wave's block, logical chunk 2g + half
  const int swz = (col / RP) % CPR;
  int goff[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) goff[g] = col * BK + 4 * ((2 * g + half) ^ swz);
  const int arow0 = wm * 32 * BK;  // wave's first A row, in floats
  const int brow0 = wn * 32 * BK;

  // Operands of one group in registers, double-buffered: group g + 1 (or group 0 of the next
  // tile) is read from LDS while the MFMAs of group g run.
  f32x4 ra[2], rb[2];
  auto read_group = [&](auto stage, int g, int slot) {
    constexpr int S = decltype(stage)::value;
    ra[slot] = *reinterpret_cast<const f32x4*>(lds + S * STAGE + arow0 + goff[g]);
    rb[slot] = *reinterpret_cast<const f32x4*>(lds + S * STAGE + A_TILE + brow0 + goff[g]);
  };
  // tile kt (in stage S) has landed for this thread; the barrier makes it whole and guarantees every wave has
  // read the stage the next copies overwrite: tile kt + 1 goes to stage S ^ 1, the one tile kt - 1 used
  auto sync_tile = [&](int kt, auto stage) {
    constexpr int S = decltype(stage)::value;
    wait_vmcnt<0>();
    __syncthreads();
    if (kt + 1 < nkt) issue(kt + 1, std::integral_constant<int, S ^ 1>{});
  };
  // the MFMAs of tile kt (stage S); the operands of group g + 1, or of the next tile's group 0,
  // are read while those of group g are multiplied
  auto step = [&](int kt, auto stage) {
    constexpr int S = decltype(stage)::value;
    using Next = std::integral_constant<int, S ^ 1>;
    const int ng = kt < nfull ? NG : (p.K - nfull * BK) >> 3;  // valid groups of 8 k in this tile
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int cur = g & 1;  // NG is even, so group 0 of every tile sits in slot 0
      if (g + 1 < NG) {
        read_group(stage, g + 1, cur ^ 1);
      } else if (kt + 1 < nkt) {
        sync_tile(kt + 1, Next{});
        read_group(Next{}, 0, cur ^ 1);
      }
      if (g < ng) {
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ra[cur][s], rb[cur][s], acc, 0, 0, 0);
      }
    }
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;

  issue(0, S0{});  // tile 0 (a tile always exists: K >= 8)
  sync_tile(0, S0{});
  read_group(S0{}, 0, 0);
  int kt = 0;
  for (; kt + 2 <= nkt; kt += 2) {
    step(kt, S0{});
    step(kt + 1, S1{});
  }
  if (kt < nkt) step(kt, S0{});

  // ---- epilogue: lane holds column n = nw + col, rows mw + 8(r/4) + 4*half + r%4.
  // Buffer loads/stores over the wave's output block: a scalar descriptor, a 32-bit per-lane
  // offset and a scalar per-row offset (no 64-bit address arithmetic per element); whole tiles
  // skip the bounds checks.
  const int mw = m0 + wm * 32;
  const int nw = n0 + wn * 32;
  const bool full = m0 + BM <= p.M && n0 + BN <= p.N;
  const __amdgpu_buffer_rsrc_t yr =
      __builtin_amdgcn_make_buffer_rsrc(p.y + (int64_t)mw * p.ldy + nw, 0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t rr_ = buffer_rsrc(p.resid + (int64_t)mw * p.ldy + nw);  // residual rows
  const int ldy4 = 4 * (int)p.ldy;
  // Plain stores are non-temporal (cache policy NT): y is not read back here, and keeping it out of
  // the L2 leaves the W panels and x rows there. The residual epilogues keep the default policy.
  constexpr int kStoreCpol = EPI == LIN_EPI_STORE ? 2 : 0;
  auto store = [&](auto check) {
    constexpr bool kCheck = decltype(check)::value;
    const bool n_ok = !kCheck || nw + col < p.N;
    const float bias_n = (p.bias && n_ok) ? p.bias[nw + col] : 0.f;
    float gate_n = 1.f;
    if constexpr (EPI == LIN_EPI_RESID_GATE) gate_n = n_ok ? p.gate[nw + col] : 0.f;
    const int voff = 4 * half * ldy4 + 4 * col;
    // residual epilogues: the 16 old values of the block are loaded together, then combined
    float old[16];
    if constexpr (EPI != LIN_EPI_STORE) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int rr = 8 * (r >> 2) + (r & 3);
        old[r] = 0.f;
        if (!kCheck || (n_ok && mw + 4 * half + rr < p.M))
          old[r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rr_, voff, rr * ldy4, 0));
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int rr = 8 * (r >> 2) + (r & 3);
      if (!kCheck || (n_ok && mw + 4 * half + rr < p.M)) {
        float v = apply_act<ACT>(fmaf(acc[r], p.alpha, bias_n));
        if constexpr (EPI != LIN_EPI_STORE) v = fmaf(gate_n, v, old[r]);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), yr, voff, rr * ldy4, kStoreCpol);
      }
    }
  };
  if (full) {
    store(std::false_type{});
  } else {
    store(std::true_type{});
  }
}

// Small products (under two 64 x 64 tiles per CU: the VAE projections, batch-2 DiT calls): one
// workgroup per (32*TM) x (32*TN) output tile with KS waves on each of its 32 x 32 blocks, each of
// them on different k (32 x 32 tiles with four splits, 32 x 64 tiles with two). K advances in 64-deep tiles of 8 groups of 8; the KS waves of a block
// multiply 8/KS groups each, so a wave's MFMA chain is K/KS long and short grids spread over KS
// times the waves. The partial sums meet in LDS, and the KS waves of a block add them up (in wave
// order) for 16/KS of its accumulator registers each and run the epilogue for those rows. Copies,
// swizzle and the clamped last k-tile as in linear_mfma_kernel.
template <int TM, int TN, int KS, int ACT, int EPI>
__global__ __launch_bounds__(64 * TM * TN * KS) void linear_ksplit_kernel(LinArgs p, TileOrder order) {
  constexpr int BM = 32 * TM, BN = 32 * TN, BK = 64, NS = 2;
  constexpr int NWAVE = TM * TN * KS;
  constexpr int NT = 64 * NWAVE;     // threads
  constexpr int CPR = BK / 4;        // 16-byte chunks per tile row
  constexpr int NG = BK / 8;         // groups of 8 k per tile
  constexpr int GPW = NG / KS;       // groups per wave
  constexpr int RPW = 16 / KS;       // accumulator registers each wave finishes
  constexpr int A_TILE = BM * BK;
  constexpr int STAGE = (BM + BN) * BK;
  constexpr int NIA = BM * CPR / NT;  // DMA instructions per thread and stage
  constexpr int NIB = BN * CPR / NT;
  static_assert(NIA * NT == BM * CPR && NIB * NT == BN * CPR, "tiles must split into whole copies");
  static_assert(GPW * KS == NG && RPW * KS == 16 && RPW % 4 == 0, "k split must divide the groups and rows");
  static_assert(NWAVE * 16 * 64 <= NS * STAGE, "partial sums must fit in the tiles");

  __shared__ __attribute__((aligned(16))) float lds[NS * STAGE];  // the partial sums reuse it

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int blk = wave % (TM * TN);  // the wave's 32 x 32 block: rows 32*(blk / TN), columns 32*(blk % TN)
  const int ks = wave / (TM * TN);   // its share of k
  const int col = lane & 31;
  const int half = lane >> 5;

  int mi, ni;
  tile_coords(xcd_remap(blockIdx.x, order.tiles_m * order.tiles_n), order, mi, ni);
  const int m0 = mi * BM;
  const int n0 = ni * BN;
  const int mlast = min(BM, p.M - m0) - 1;
  const int nlast = min(BN, p.N - n0) - 1;

  // chunk of DMA instruction n: physical chunk n*NT + tid, row pc / CPR, logical chunk c at
  // physical c ^ (row % CPR)
  unsigned aoff[NIA], boff[NIB];
  int acol[NIA], bcol[NIB];
#pragma unroll
  for (int n = 0; n < NIA; ++n) {
    const int pc_all = n * NT + tid;
    const int row = pc_all / CPR;
    const int c = (pc_all % CPR) ^ (row % CPR);
    acol[n] = 4 * c;
    aoff[n] = 4u * (unsigned)(min(row, mlast) * (int)p.ldx + 4 * c);
  }
#pragma unroll
  for (int n = 0; n < NIB; ++n) {
    const int pc_all = n * NT + tid;
    const int row = pc_all / CPR;
    const int c = (pc_all % CPR) ^ (row % CPR);
    bcol[n] = 4 * c;
    boff[n] = 4u * (unsigned)(min(row, nlast) * (int)p.ldw + 4 * c);
  }
  const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(p.x + (int64_t)m0 * p.ldx);
  const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(p.w + (int64_t)n0 * p.ldw);
  const int nkt = (p.K + BK - 1) / BK;
  const int nfull = p.K / BK;
  auto issue = [&](int kt, auto stage) {
    constexpr int S = decltype(stage)::value;
    float* at = lds + S * STAGE;
    float* bt = at + A_TILE;
    // whole tiles copy at the k-tile's column; the tile holding K (always tile nfull) re-reads the
    // last group for columns at or past K (never multiplied)
    const bool last = kt >= nfull;
    const int k0 = kt * BK;
    const unsigned soff = 4u * (unsigned)k0;
    const int kmax = p.K - 8 - k0;
#pragma unroll
    for (int n = 0; n < NIA; ++n) {
      const unsigned shift = last && acol[n] > kmax + 4 ? 4u * (unsigned)((acol[n] & ~7) - kmax) : 0u;
      buffer_to_lds16(xr, aoff[n] - shift, at + (n * NWAVE + wave) * 256, soff);
    }
#pragma unroll
    for (int n = 0; n < NIB; ++n) {
      const unsigned shift = last && bcol[n] > kmax + 4 ? 4u * (unsigned)((bcol[n] & ~7) - kmax) : 0u;
      buffer_to_lds16(wr, boff[n] - shift, bt + (n * NWAVE + wave) * 256, soff);
    }
  };

  f32x16 acc = zero16();
  const int swz = col % CPR;
  const int arow = 32 * (blk / TN) + col;  // the lane's A row and B row in the tile
  const int brow = 32 * (blk % TN) + col;
  auto step = [&](int kt, auto stage) {
    constexpr int S = decltype(stage)::value;
    wait_vmcnt<0>();
    __syncthreads();  // tile kt is whole, and every wave is done with the stage the next copy fills
    if (kt + 1 < nkt) issue(kt + 1, std::integral_constant<int, S ^ 1>{});
    const int ng = kt < nfull ? NG : (p.K - nfull * BK) >> 3;  // valid groups of 8 k in this tile
    const float* at = lds + S * STAGE + arow * BK;
    const float* bt = lds + S * STAGE + A_TILE + brow * BK;
#pragma unroll
    for (int u = 0; u < GPW; ++u) {
      const int g = GPW * ks + u;
      if (g < ng) {
        const int c = 4 * ((2 * g + half) ^ swz);
        const f32x4 ra = *reinterpret_cast<const f32x4*>(at + c);
        const f32x4 rb = *reinterpret_cast<const f32x4*>(bt + c);
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ra[s], rb[s], acc, 0, 0, 0);
      }
    }
  };
  issue(0, std::integral_constant<int, 0>{});
  int kt = 0;
  for (; kt + 2 <= nkt; kt += 2) {
    step(kt, std::integral_constant<int, 0>{});
    step(kt + 1, std::integral_constant<int, 1>{});
  }
  if (kt < nkt) step(kt, std::integral_constant<int, 0>{});

  // ---- partial sums through LDS: wave w's register r of lane l at red[(w*16 + r)*64 + l]
  __syncthreads();  // every wave is done with the tiles
  float* red = lds;
#pragma unroll
  for (int r = 0; r < 16; ++r) red[(wave * 16 + r) * 64 + lane] = acc[r];
  __syncthreads();
  // ---- epilogue: the wave finishes registers RPW*ks .. of its block: register r holds row
  // 8(r/4) + 4*half + r%4 of column col
  const int n = n0 + 32 * (blk % TN) + col;
  if (n >= p.N) return;
  const float bias_n = p.bias ? p.bias[n] : 0.f;
  float gate_n = 1.f;
  if constexpr (EPI == LIN_EPI_RESID_GATE) gate_n = p.gate[n];
  const float* rsrc = p.resid;
#pragma unroll
  for (int k = 0; k < RPW; ++k) {
    const int r = RPW * ks + k;
    const int m = m0 + 32 * (blk / TN) + 8 * (r >> 2) + 4 * half + (r & 3);
    if (m < p.M) {
      float sum = red[(blk * 16 + r) * 64 + lane];
#pragma unroll
      for (int w = 1; w < KS; ++w) sum += red[((w * TM * TN + blk) * 16 + r) * 64 + lane];
      float v = apply_act<ACT>(fmaf(sum, p.alpha, bias_n));
      const int64_t e = (int64_t)m * p.ldy + n;
      if constexpr (EPI != LIN_EPI_STORE) v = fmaf(gate_n, v, rsrc[e]);
      if constexpr (EPI == LIN_EPI_STORE) {
        __builtin_nontemporal_store(v, p.y + e);  // not read back here, as in linear_mfma_kernel
      } else {
        p.y[e] = v;
      }
    }
  }
}

// Any shape and alignment: one thread per output, 16 x 16 outputs per workgroup, K in steps of
// 16 through LDS. Used when rows are not 16-byte aligned or K % 8 != 0.
__global__ __launch_bounds__(256) void linear_generic_kernel(LinearParams p) {
  __shared__ float xs[16][17];
  __shared__ float ws[16][17];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int m = blockIdx.y * 16 + ty;
  const int n = blockIdx.x * 16 + tx;
  const int mload = blockIdx.y * 16 + ty;  // row loaded by this thread (x tile)
  const int nload = blockIdx.x * 16 + ty;  // row loaded by this thread (W tile)
  float acc = 0.f;
  for (int k0 = 0; k0 < p.K; k0 += 16) {
    const int k = k0 + tx;
    xs[ty][tx] = (mload < p.M && k < p.K) ? p.x[p.x_off + (int64_t)mload * p.ldx + k] : 0.f;
    ws[ty][tx] = (nload < p.N && k < p.K) ? p.w[(int64_t)nload * p.ldw + k] : 0.f;
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) acc = fmaf(xs[ty][kk], ws[tx][kk], acc);
    __syncthreads();
  }
  if (m < p.M && n < p.N) {
    float v = fmaf(acc, p.alpha, p.bias ? p.bias[n] : 0.f);
    switch (p.act) {
      case LIN_ACT_GELU: v = apply_act<LIN_ACT_GELU>(v); break;
      case LIN_ACT_GELU_TANH: v = apply_act<LIN_ACT_GELU_TANH>(v); break;
      case LIN_ACT_SILU: v = apply_act<LIN_ACT_SILU>(v); break;
      default: break;
    }
    const int64_t e = p.y_off + (int64_t)m * p.ldy + n;
    if (p.epi == LIN_EPI_STORE) p.y[e] = v;
    else p.y[e] = fmaf(p.epi == LIN_EPI_RESID_GATE ? p.gate[p.gate_off + n] : 1.f, v, (p.resid ? p.resid : p.y)[e]);
  }
}

// Groups of W panels of at most 2 MB (half an XCD's L2: the other half holds the x rows in flight),
// as few and as even as possible, over super-blocks of one XCD's share of the row blocks. Grouping
// reads each x row block once per group; it is used when those extra reads come to at most twice
// W, which the plain order fetches several times per XCD once W outgrows the L2. Measured FETCH_SIZE
// at 16384 rows: qkv (W 4 MB, x 4.7 MB per XCD, 2 groups) 150 -> 54 MiB with the NT stores, fc1
// (W 5.3 MB, 3 groups) 144 -> 83 MiB; fc2 (W 5.3 MB but x 19 MB per XCD) went up 156 -> 199-256 MiB
// when grouped and keeps the plain order. Timings were unchanged (the layers are MFMA-bound).
TileOrder tile_order(const LinearParams& p, int bm, int bn) {
  constexpr int64_t kGroupBytes = 2 << 20;
  TileOrder o;
  o.tiles_m = (int)((p.M + bm - 1) / bm);
  o.tiles_n = (int)((p.N + bn - 1) / bn);
  o.sb_rows = (o.tiles_m + 7) / 8;
  o.group_n = o.tiles_n;
  const int64_t panel = (int64_t)bn * p.K * 4;
  const int64_t w_bytes = o.tiles_n * panel;
  const int64_t groups = std::min<int64_t>((w_bytes + kGroupBytes - 1) / kGroupBytes, o.tiles_n);
  if (groups > 1) {
    const int group_n = (int)((o.tiles_n + groups - 1) / groups);
    const int64_t x_share = (int64_t)o.sb_rows * bm * p.K * 4;
    const int64_t n_groups = (o.tiles_n + group_n - 1) / group_n;
    if (group_n >= 2 && (n_groups - 1) * x_share <= 2 * w_bytes) o.group_n = group_n;
  }
  return o;
}

LinArgs lin_args(const LinearParams& p) {
  LinArgs a;
  memset(&a, 0, sizeof a);
  a.x = p.x + p.x_off;
  a.w = p.w;
  a.bias = p.bias;
  a.gate = p.gate ? p.gate + p.gate_off : nullptr;
  a.y = p.y + p.y_off;
  a.resid = (p.resid ? p.resid : p.y) + p.y_off;
  a.ldx = (int32_t)p.ldx;
  a.ldw = (int32_t)p.ldw;
  a.ldy = (int32_t)p.ldy;
  a.M = p.M;
  a.N = p.N;
  a.K = p.K;
  a.alpha = p.alpha;
  return a;
}

template <int ACT, int EPI>
hipError_t launch_tiles(const LinearParams& p, hipStream_t stream) {
  const int64_t tm = (p.M + 63) / 64;
  const int64_t tn = (p.N + 63) / 64;
  if (tm * tn > 0x7fffffff) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((linear_mfma_kernel<ACT, EPI>), dim3((unsigned)(tm * tn)), dim3(256), 0, stream, lin_args(p),
                     tile_order(p, 64, 64));
  return hipGetLastError();
}

template <int ACT>
hipError_t launch_epi(const LinearParams& p, hipStream_t stream) {
  switch (p.epi) {
    case LIN_EPI_STORE: return launch_tiles<ACT, LIN_EPI_STORE>(p, stream);
    case LIN_EPI_RESID: return launch_tiles<ACT, LIN_EPI_RESID>(p, stream);
    case LIN_EPI_RESID_GATE: return launch_tiles<ACT, LIN_EPI_RESID_GATE>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

template <int NW, int MT, int NT, int ACT, int EPI>
hipError_t launch_split_tiles(const LinearParams& p, hipStream_t stream) {
  const int64_t tm = (p.M + 16 * MT * NW - 1) / (16 * MT * NW);
  const int64_t tn = (p.N + 16 * NT - 1) / (16 * NT);
  if (tm * tn > 0x7fffffff) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((linear_split_kernel<NW, MT, NT, ACT, EPI>), dim3((unsigned)(tm * tn)), dim3(64 * NW), 0, stream,
                     lin_args(p), tile_order(p, 16 * MT * NW, 16 * NT));
  return hipGetLastError();
}

template <int NW, int MT, int NT, int ACT>
hipError_t launch_split_epi(const LinearParams& p, hipStream_t stream) {
  switch (p.epi) {
    case LIN_EPI_STORE: return launch_split_tiles<NW, MT, NT, ACT, LIN_EPI_STORE>(p, stream);
    case LIN_EPI_RESID: return launch_split_tiles<NW, MT, NT, ACT, LIN_EPI_RESID>(p, stream);
    case LIN_EPI_RESID_GATE: return launch_split_tiles<NW, MT, NT, ACT, LIN_EPI_RESID_GATE>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

template <int NW, int MT, int NT>
hipError_t launch_split(const LinearParams& p, hipStream_t stream) {
  switch (p.act) {
    case LIN_ACT_NONE: return launch_split_epi<NW, MT, NT, LIN_ACT_NONE>(p, stream);
    case LIN_ACT_GELU: return launch_split_epi<NW, MT, NT, LIN_ACT_GELU>(p, stream);
    case LIN_ACT_GELU_TANH: return launch_split_epi<NW, MT, NT, LIN_ACT_GELU_TANH>(p, stream);
    case LIN_ACT_SILU: return launch_split_epi<NW, MT, NT, LIN_ACT_SILU>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

template <int TM, int TN, int KS, int ACT, int EPI>
hipError_t launch_ksplit_tiles(const LinearParams& p, hipStream_t stream) {
  TileOrder o;
  o.tiles_m = (p.M + 32 * TM - 1) / (32 * TM);
  o.tiles_n = (p.N + 32 * TN - 1) / (32 * TN);
  o.group_n = o.tiles_n;  // the operands of these small products stay in the L2
  o.sb_rows = (o.tiles_m + 7) / 8;
  const int64_t n = (int64_t)o.tiles_m * o.tiles_n;
  if (n > 0x7fffffff) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((linear_ksplit_kernel<TM, TN, KS, ACT, EPI>), dim3((unsigned)n), dim3(64 * TM * TN * KS), 0, stream,
                     lin_args(p), o);
  return hipGetLastError();
}

template <int TM, int TN, int KS, int ACT>
hipError_t launch_ksplit_epi(const LinearParams& p, hipStream_t stream) {
  switch (p.epi) {
    case LIN_EPI_STORE: return launch_ksplit_tiles<TM, TN, KS, ACT, LIN_EPI_STORE>(p, stream);
    case LIN_EPI_RESID: return launch_ksplit_tiles<TM, TN, KS, ACT, LIN_EPI_RESID>(p, stream);
    case LIN_EPI_RESID_GATE: return launch_ksplit_tiles<TM, TN, KS, ACT, LIN_EPI_RESID_GATE>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

template <int TM, int TN, int KS>
hipError_t launch_ksplit(const LinearParams& p, hipStream_t stream) {
  switch (p.act) {
    case LIN_ACT_NONE: return launch_ksplit_epi<TM, TN, KS, LIN_ACT_NONE>(p, stream);
    case LIN_ACT_GELU: return launch_ksplit_epi<TM, TN, KS, LIN_ACT_GELU>(p, stream);
    case LIN_ACT_GELU_TANH: return launch_ksplit_epi<TM, TN, KS, LIN_ACT_GELU_TANH>(p, stream);
    case LIN_ACT_SILU: return launch_ksplit_epi<TM, TN, KS, LIN_ACT_SILU>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_act(const LinearParams& p, hipStream_t stream) {
  switch (p.act) {
    case LIN_ACT_NONE: return launch_epi<LIN_ACT_NONE>(p, stream);
    case LIN_ACT_GELU: return launch_epi<LIN_ACT_GELU>(p, stream);
    case LIN_ACT_GELU_TANH: return launch_epi<LIN_ACT_GELU_TANH>(p, stream);
    case LIN_ACT_SILU: return launch_epi<LIN_ACT_SILU>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

bool linear_mfma_supported(const LinearParams& p) {
  auto a16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  // copies address a tile's rows as 32-bit byte offsets from its first row (up to 128 x rows and
  // 192 W rows, plus the k offset <= the row stride); stores address up to 128 output rows likewise
  // (the same bounds keep the row strides within the 32 bits of the kernels' arguments)
  return p.K % 8 == 0 && a16(p.x) && a16(p.w) && p.x_off % 4 == 0 && p.ldx % 4 == 0 && p.ldw % 4 == 0 &&
         (int64_t)(64 * 2 + 1) * p.ldx * 4 < 0x7fffffffLL && (int64_t)(64 * 3 + 1) * p.ldw * 4 < 0x7fffffffLL &&
         (int64_t)64 * 2 * p.ldy * 4 < 0x7fffffffLL;
}

namespace {

// Size class of a call: the tile of the fp32 kernels that its grid fills, and the kernel's name in the
// API. Classes 128 x 192 and 64 x 192 (at least one 128 x 192 tile per CU, or three 64 x 192 ones) run
// linear_split_kernel, class 64 x 64 that or linear_mfma_kernel, the 32 x 64 class that or
// linear_ksplit_kernel (split_tile below).
// Grids of fewer 64 x 64 tiles than 1.25 per CU take linear_ksplit_kernel, whose quarter-K waves
// spread them over the SIMDs (us, 64 x 64 -> k-split: VAE output projection 1024 x 512 x 512 11.75 ->
// 8.1, context k|v 77 x 1152 x 576 13.2 -> 6.3, batch-2 proj/q/cproj 512 x 576 x 576 12.6-13.0 ->
// 8.4-8.7, fc1 512 x 2304 x 576 21.4 -> 19.2, fc2 512 x 576 x 2304 43.4 -> 23.0). Grids of 1.25 to 2
// such tiles per CU are the class of 32 x 64 tiles with k split in two, whose count is twice that and so shares
// out more evenly over the CUs (VAE q|k|v 1024 x 1536 x 512, 384 tiles: 64 x 64 18.7-19.2, 32 x 64 /
// two splits 17.4, 64 x 32 17.5, 64 x 32 / four splits 17.9, 64 x 64 / two splits 20.7, 32 x 32 / four
// splits 18.9-19.4). The split kernel's smallest tiles (64 x 48, 32 x 48) measured slower on the small grids:
// 13-20 against 6-15 us at K = 576, with one, two or four k-tiles of loads in flight alike: a wave alone
// on its SIMD issues one VALU instruction per 6 cycles, and the splits are most of its work.
enum LinearClass { kClass128x192, kClass64x192, kClass64x64, kClass32x64, kClass32x32 };
LinearClass linear_class(const LinearParams& p, int num_cus) {
  const int64_t tiles_wide = ((p.M + 127) / 128) * ((p.N + 191) / 192);
  const int64_t tiles_tall = ((p.M + 63) / 64) * ((p.N + 191) / 192);
  const int64_t tiles_64 = ((p.M + 63) / 64) * ((p.N + 63) / 64);
  if (p.N >= 2048 && tiles_wide >= num_cus) return kClass128x192;
  if ((p.N % 192 == 0 || p.N >= 1024) && tiles_tall >= 3 * (int64_t)num_cus) return kClass64x192;
  if (4 * tiles_64 < 5 * (int64_t)num_cus) return kClass32x32;
  if (tiles_64 < 2 * (int64_t)num_cus) return kClass32x64;
  return kClass64x64;
}

// The tile that linear_split_kernel runs a call of the larger classes with, or one of the fp32 kernels:
// kMfma64 (linear_mfma_kernel, 64 x 64) in its class, kKsplit32x64 in its own. Each candidate's time is
// estimated from how many of its tiles every CU gets, a + b u us for 1, 2, ... of them at once (u = K / 576), fitted
// over 12 (N, K) of 512..2304 x 64..2304 and 15 row counts of 512 to 16128, plus what the residual epilogues
// add per million outputs (0.2 us to the fp32 64 x 64 kernel, 0.65 to four-wave tiles, 1.05 to eight-wave ones).
// Measured over those 278 calls: the choices take 17.54 ms, the best tile each time 17.49, the fp32 kernels alone
// 23.2 (none of the choices more than 4% longer). The fp32 64 x 64 kernel, the less exact, is taken from 7%
// faster on: short K (6144 x 1024 x 128: 17 against 20 us), and 4096 x 512 x 2048 (72 / 79). The class of the
// two-split fp32 kernel takes only the 64 x 64 split tile beside it, whose two sums per output are more
// exact than its two halves of k.
enum SplitTile { kMfma64, kKsplit32x64, kSplit64x64, kSplit64x96, kSplit128x96, kSplit256x144, kSplit256x192 };
SplitTile split_tile(const LinearParams& p, int num_cus, LinearClass cls) {
  struct Line {
    double a, b;
  };
  static constexpr Line k64x64[] = {{3.4, 14.4}, {5.5, 18.5}, {6.8, 23.7}, {7.2, 31.3}};
  static constexpr Line k64x96[] = {{5.0, 17.7}, {6.7, 22.5}, {7.8, 30.3}, {7.9, 42.3}};
  static constexpr Line k128x96[] = {{7.4, 23.8}, {9.6, 32.4}, {10.4, 48.5}};
  static constexpr Line k256x144[] = {{12.3, 39.5}};
  static constexpr Line k256x192[] = {{14.1, 59.0}};
  const double u = p.K / 576.0;
  const double resid = p.epi == LIN_EPI_STORE ? 0 : 1e-6 * p.M * (double)p.N;  // million outputs read back
  auto per_cu = [&](int bm, int bn) {
    const int64_t tiles = (int64_t)((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn);
    return (tiles + num_cus - 1) / num_cus;
  };
  // n tiles per CU: whole residencies, then the rest at once; where several tiles share a CU the next one's start
  // covers half of the last one's
  auto cost = [&](int bm, int bn, const auto& lines, double per_output) {
    constexpr int64_t cap = sizeof(lines) / sizeof(Line);
    const int64_t n = per_cu(bm, bn);
    auto t = [&](int64_t k) { return k == 0 ? 0.0 : lines[k - 1].a + lines[k - 1].b * u; };
    const double covered = cap == 1 ? 0.0 : 0.5 * (double)((n - 1) / cap) * lines[cap - 1].a;
    return n / cap * t(cap) + t(n % cap) - covered + per_output * resid;
  };
  double best = cost(64, 64, k64x64, 0.65);
  SplitTile t = kSplit64x64;
  auto take = [&](double c, SplitTile tile) {
    if (c < best) {
      best = c;
      t = tile;
    }
  };
  if (cls == kClass32x64) {  // three or four 32 x 64 tiles per CU
    take((per_cu(32, 64) <= 3 ? 4.4 + 14.6 * u : 5.2 + 20.6 * u) + 0.85 * resid, kKsplit32x64);
    return t;
  }
  take(cost(64, 96, k64x96, 0.65), kSplit64x96);
  take(cost(128, 96, k128x96, 0.65), kSplit128x96);
  take(cost(256, 144, k256x144, 1.05), kSplit256x144);
  take(cost(256, 192, k256x192, 1.05), kSplit256x192);
  if (cls == kClass64x64) take(1.07 * (3.4 + per_cu(64, 64) * (0.4 + 8.45 * u) + 0.2 * resid), kMfma64);
  return t;
}

}  // namespace

const char* linear_kernel_name(const LinearParams& p, int num_cus) {
  if (!linear_mfma_supported(p)) return "linear_generic";
  switch (linear_class(p, num_cus)) {
    case kClass128x192: return "linear_mfma_128x192";
    case kClass64x192: return "linear_mfma_64x192";
    case kClass32x64: return "linear_mfma_32x64_ksplit";
    case kClass32x32: return "linear_mfma_32x32_ksplit";
    default: return "linear_mfma_64x64";
  }
}

void linear_tile(const LinearParams& p, int num_cus, int* rows, int* cols, int* terms) {
  struct Tile {
    int rows, cols, terms;
  };
  static constexpr Tile kTiles[] = {{64, 64, 1}, {32, 64, 1}, {64, 64, 3}, {64, 96, 3}, {128, 96, 3}, {256, 144, 3}, {256, 192, 3}};
  Tile t = {16, 16, 1};  // linear_generic_kernel
  if (linear_mfma_supported(p)) {
    const LinearClass cls = linear_class(p, num_cus);
    t = cls == kClass32x32 ? Tile{32, 32, 1} : kTiles[split_tile(p, num_cus, cls)];
  }
  *rows = t.rows;
  *cols = t.cols;
  *terms = t.terms;
}

hipError_t launch_linear(const LinearParams& p, int num_cus, hipStream_t stream) {
  if (!linear_mfma_supported(p)) {
    const dim3 grid((unsigned)((p.N + 15) / 16), (unsigned)((p.M + 15) / 16));
    if ((p.N + 15) / 16 > 0x7fffffff || (p.M + 15) / 16 > 65535) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL(linear_generic_kernel, grid, dim3(256), 0, stream, p);
    return hipGetLastError();
  }
  const LinearClass cls = linear_class(p, num_cus);
  if (cls == kClass32x32) return launch_ksplit<1, 1, 4>(p, stream);
  switch (split_tile(p, num_cus, cls)) {
    case kKsplit32x64: return launch_ksplit<1, 2, 2>(p, stream);
    case kSplit64x64: return launch_split<4, 1, 4>(p, stream);
    case kSplit64x96: return launch_split<4, 1, 6>(p, stream);
    case kSplit128x96: return launch_split<4, 2, 6>(p, stream);
    case kSplit256x144: return launch_split<8, 2, 9>(p, stream);
    case kSplit256x192: return launch_split<8, 2, 12>(p, stream);
    default: return launch_act(p, stream);
  }
}

}  // namespace sa
