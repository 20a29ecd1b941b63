// How the network passes share the neighbour list among waves (device code, and
// host code for the check that every pair is taken once).
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define HMD_NN_ITEMS_FN __device__ inline
#else
#define HMD_NN_ITEMS_FN inline
#endif

// An item is an entry, or one of its 2^split groups of i-sub-clusters, and wave
// v of n takes the items v, v + n, ...  An entry of a dense liquid holds 0 to
// 4,096 pairs (about 1,000 on average), so a short list is split until there are
// HMD_NN_ITEMS items (or eight groups an entry): eight of the 2,048 waves the
// chip holds of the forward pass.  Whole entries in contiguous shares left a CU
// with 1.2 of 8 waves running on average at 9,999 atoms.
#define HMD_NN_ITEMS 16384u
struct HmdNnItems {
  uint32_t n, split;
  HMD_NN_ITEMS_FN HmdNnItems(uint32_t entries, uint32_t want) : split(0) {
    while (split < 3u && (entries << split) < want) ++split;
    n = entries << split;
  }
  HMD_NN_ITEMS_FN uint32_t entry(uint32_t w) const { return w >> split; }
  // Item w's sub-clusters.  Which group of its entry an item takes turns from
  // round to round of the waves: the first and last i-sub-clusters of an entry
  // hold different numbers of pairs, and with a number of waves that is a
  // multiple of eight a wave would take the same group every time.  The turn is
  // that of the entry's first item, so the groups of an entry are all taken
  // once whatever the number of waves.
  HMD_NN_ITEMS_FN uint32_t mask(uint32_t w, uint32_t n_waves) const {
    const uint32_t per = 1u << split, group = 8u >> split;
    const uint32_t turn = (w & ~(per - 1u)) / n_waves;
    return ((1u << group) - 1u) << (group * ((w + turn) & (per - 1u)));
  }
};
