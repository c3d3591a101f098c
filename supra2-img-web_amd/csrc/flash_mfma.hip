// Host side of the flash attention launches (head dim 64 or 128, csrc/flash_split.hip): the packed kernel
// arguments, and the launch classes that a plan reports and the key-length schedule works on. A class
// counts a call in units of 128 queries (64 with a 2-way key split, calls of under 2048 groups of 32), which is
// not how it is launched: flash_shape groups queries and splits keys, and one grid runs them all.

#include <string.h>

#include "common.h"
#include "kernels.h"

namespace sa {

FlashArgs flash_args(const AttnParams& p, int64_t tiles) {
  FlashArgs a;
  memset(&a, 0, sizeof a);
  a.q = p.q + p.q_off;
  a.k = p.k + p.k_off;
  a.v = p.v + p.v_off;
  a.o = p.o + p.o_off;
  a.sq = (int32_t)p.sq;
  a.sk = (int32_t)p.sk;
  a.sv = (int32_t)p.sv;
  a.so = (int32_t)p.so;
  a.ldq = (int32_t)p.ldq;
  a.ldk = (int32_t)p.ldk;
  a.ldv = (int32_t)p.ldv;
  a.ldo = (int32_t)p.ldo;
  a.Lq = p.Lq;
  a.Lk = p.Lk;
  a.tiles = (int32_t)tiles;
  a.H = (int16_t)p.H;
  a.scale_log2 = p.scale_log2;
  if (p.mask_mode == MASK_KEY_LEN) a.mask = p.key_len;
  if (p.mask_mode == MASK_KEY_MASK) {
    a.mask = p.key_mask;
    a.aux = (int32_t)p.smask;
  }
  a.bias = p.bias;
  if (p.bias_mode == BIAS_RELPOS) {
    a.lut = p.lut;
    a.num_buckets = (int16_t)p.num_buckets;
  } else {
    a.sbias = p.sbias;
  }
  return a;
}

bool flash_mfma_args_fit(const AttnParams& p) {
  const int64_t lim = 0x7fffffff;
  return p.ldq <= lim && p.ldk <= lim && p.ldv <= lim && p.ldo <= lim && p.sq <= lim && p.sk <= lim &&
         p.sv <= lim && p.so <= lim && p.H <= 0x7fff && (p.mask_mode != MASK_KEY_MASK || p.smask <= lim) &&
         (p.bias_mode != BIAS_RELPOS || p.num_buckets <= 0x7fff);
}

const char* flash_mfma_name(int D, int nsplit) {
  if (D == 64) return nsplit == 2 ? "flash_mfma_d64_split2" : "flash_mfma_d64";
  if (D == 128) return nsplit == 2 ? "flash_mfma_d128_split2" : "flash_mfma_d128";
  return nullptr;
}

// The key splits that classes have; every (bias, mask) pair exists for each of them.
constexpr int kSplits64[] = {1, 2};
constexpr int kSplits128[] = {1, 2};

static int class_split(int nsplit) { return nsplit >= 2 ? 2 : 1; }

FlashVariant flash_mfma_variant(const AttnParams& p, int nsplit) {
  int mask = p.mask_mode;
  if (mask == MASK_KEY_LEN && p.order_n > 0) mask = MASK_KEY_LEN_ORDERED;
  return {p.D, class_split(nsplit), p.bias_mode, mask};
}

// Units of a class past the last whole round of four per CU, and what plans call them: few enough for 32-query
// groups or 64-query units at one per CU. No launch of theirs follows: flash_split_kernel runs every
// unit in one grid (three workgroups per CU without a mask, two in the other variants, by registers), where the
// leftover of a round costs what it holds: batch 57 / 60 / 64 of the DiT self-attention take 57 / 59 / 62 us.
int64_t flash_mfma_tail_units(const AttnParams& p, int nsplit, int num_cus) {
  const bool eligible = p.D == 64 && class_split(nsplit) == 1 && p.bias_mode == BIAS_NONE &&
                        p.mask_mode == MASK_NONE && p.Lk > 32;
  if (!eligible) return 0;
  const int64_t tiles = (int64_t)p.B * p.H * ((p.Lq + 127) / 128);
  const int64_t slots = 4 * (int64_t)num_cus;
  if (tiles <= slots) return 0;
  const int64_t rest = tiles % slots;
  return 2 * rest <= num_cus ? rest : 0;
}

int flash_mfma_tail_kernel(const AttnParams& p, int nsplit, int num_cus) {
  const int64_t tail = flash_mfma_tail_units(p, nsplit, num_cus);
  if (tail == 0) return TAIL_NONE;
  if (4 * tail <= num_cus) return TAIL_SMALL;
  // one round plus the leftover: folded into the round's first workgroups
  const int64_t tiles = (int64_t)p.B * p.H * ((p.Lq + 127) / 128);
  return tiles < 8 * (int64_t)num_cus ? TAIL_FOLD : TAIL_SPLIT2;
}

int64_t flash_mfma_tail_groups(const AttnParams& p, int nsplit, int num_cus, int64_t* first) {
  const int64_t tail = flash_mfma_tail_units(p, nsplit, num_cus);
  *first = 0;
  if (tail == 0) return 0;
  // unit t = (b*H + h)*q_tiles + qtile holds the 32-query groups from (b*H + h)*q_groups + 4*qtile
  // on (the 64-query units from (b*H + h)*q_units + 2*qtile), and the units after it the ones after
  const int64_t q_tiles = (p.Lq + 127) / 128;
  const int64_t per = flash_mfma_tail_kernel(p, nsplit, num_cus) == TAIL_SMALL ? 4 : 2;  // sub-units per unit
  const int64_t q_sub = (p.Lq + 128 / per - 1) / (128 / per);
  const int64_t t = (int64_t)p.B * p.H * q_tiles - tail;
  *first = (t / q_tiles) * q_sub + per * (t % q_tiles);
  return (int64_t)p.B * p.H * q_sub - *first;
}

int flash_mfma_unit_queries(int nsplit) { return 32 * (4 / class_split(nsplit)); }

// Four and one are what the schedule's model does best with, not what fits a CU (two of the scheduled
// variant's workgroups at head dim 64): batch 64, prompts of 1 to 128 tokens 27.7 / 27.1 / 27.7 us over three draws
// with four, 29.2 / 27.6 / 28.9 with two, 29.4 / 27.7 / 28.9 with one, 31.8 / 30.6 / 29.6 in launch order; batch 24 in 64-query
// units and one per CU 13.5 / 15.0 / 12.5, in 128-query units and two 14.4 / 15.3 / 13.7.
int flash_mfma_per_cu(const AttnParams& p, int nsplit) {
  const FlashVariant v = flash_mfma_variant(p, nsplit);
  const bool four = v.D == 64 && v.nsplit == 1 && v.bias == BIAS_NONE && v.mask != MASK_KEY_MASK;
  return four ? 4 : 1;
}

int64_t flash_mfma_workgroups(const AttnParams& p, int nsplit, int num_cus) {
  const int qt = 32 * (4 / class_split(nsplit));
  return (int64_t)p.B * p.H * ((p.Lq + qt - 1) / qt) - flash_mfma_tail_units(p, nsplit, num_cus);
}

int flash_mfma_variants(FlashVariant* out, int cap) {
  int n = 0;
  auto add = [&](int D, int s) {
    for (int bias = BIAS_NONE; bias <= BIAS_RELPOS; ++bias)
      for (int mask = MASK_NONE; mask <= MASK_KEY_LEN_ORDERED; ++mask) {
        if (n < cap) out[n] = {D, s, bias, mask};
        ++n;
      }
  };
  for (int s : kSplits64) add(64, s);
  for (int s : kSplits128) add(128, s);
  return n;
}

}  // namespace sa
