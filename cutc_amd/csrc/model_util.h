// model_util.h — small helpers shared by the host-side solver drivers.
#pragma once

#include <algorithm>

#include "ctc_internal.h"
#include "kernels_common.h"

namespace ctc {

inline CissArgs ciss_args(const DevCiss &d) {
  CissArgs a{};
  for (int s = 0; s < 3; ++s) a.oidx[s] = d.oidx[s];
  a.vals = d.vals;
  a.tile_slot = d.tile_slot;
  a.tile_mask = d.tile_mask;
  a.directory = d.directory;
  a.rowptr = d.rowptr;
  a.nnz = d.nnz;
  a.ntiles = d.ntiles;
  a.dlength = d.dlength;
  return a;
}

// factor pointers relative to a CISS mode: f[0] = own mode, f[1+s] = mode+1+s
inline FactorArgs rel_factors(float *const *F, uint32_t N, uint32_t mode) {
  FactorArgs f{};
  for (uint32_t s = 0; s < N; ++s) f.f[s] = F[(mode + s) % N];
  return f;
}

// tiles per span from the options' tile_len (nonzeros per wave work unit)
inline uint32_t span_tiles_of(const ctc_options *o) {
  uint32_t tl = o && o->tile_len ? o->tile_len : 1024;  // 0: the measured default
  tl = std::max<uint32_t>(64, (tl + 63) / 64 * 64);
  return tl / 64;
}

// tiles per span of the ALS span kernels over nnz nonzeros.  An asked-for
// tile_len stands; the default shrinks the span until the walk has about
// kSpanWaves waves, because a span is one wave's serial chain.
// k_als_gram at R = 16 with spans of 1024 nonzeros and by this rule: 20K
// nonzeros 78 -> 8 us, 1M nonzeros 74 -> 28 us; from 8.4M nonzeros on the span is 1024.
// A span adds a piece to the scratch: at most 16383, 138 MB at R = 32 (1M nonzeros
// 132 MB beside their rows' own pieces, 8 MB with spans of 1024).
constexpr uint64_t kSpanWaves = 8192;
inline uint32_t als_span_tiles(const ctc_options *o, uint64_t nnz) {
  const uint32_t most = span_tiles_of(o);
  if (o && o->tile_len) return most;
  const uint64_t ntiles = (nnz + kTile - 1) / kTile;
  return (uint32_t)std::min<uint64_t>(most, std::max<uint64_t>(1, ntiles / kSpanWaves));
}

inline unsigned block_of(const ctc_options *o) {
  unsigned b = o && o->block ? o->block : 256;
  if (b < 64) b = 64;
  if (b > 256) b = 256;
  return b / 64 * 64;
}

}  // namespace ctc
