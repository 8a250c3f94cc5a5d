// kernels.hip — gfx950 kernels of libctc: CISS tile walks for SGD, ALS
// (MFMA Gram + MTTKRP, FP64 Cholesky solve), MTTKRP, the loss adjoint and the
// RMSE reductions.
//
// Execution model shared by the walks ("walkers"):
//   * The nonzeros of a mode's CISS are cut into spans of whole 64-nonzero
//     tiles.  A walker owns one span and visits its nonzeros in order.
//   * A walker is W = min(R, 64) lanes; lane w holds columns w, w+W, ... of
//     every factor row it touches, so each row access is one contiguous
//     W*4-byte load or atomic (coalesced), and a dot product is a W-lane DPP /
//     swizzle reduction.  64/W walkers share a wave.
//   * A wave loads W nonzeros at a time (indices, value, row-start bit from the
//     tile mask) with one coalesced load per stream, then hands nonzero q to
//     its walker lanes with ds_bpermute; the row starts come from one ballot.
//   * Row (directory-slot) changes are found from the tile mask; the slot of a
//     walker's first nonzero is the tile header's first slot.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "kernels_common.h"
#include "kernels_launch.h"

namespace ctc {

// ==========================================================================
// SGD epoch (reference rule SG/sgd.cu:75-99: every row of a nonzero is
// updated from its pre-update values; step = lr * scale).
//
// A walker keeps the rows of its current nonzero in registers.  How a row it
// shares with concurrent walkers is read and written is chosen per mode
// (PA for the CISS mode, PB for the next mode, PC for the others):
//   P_RACY     read at the start of a run of equal indices, apply own updates
//              in registers, store the row after every nonzero (concurrent
//              writers overwrite each other).
//   P_ATOMIC   read every nonzero, add every update with a device-scope float
//              atomic (the reference's atomicAdd, SG/sgd.cu:96-98).
//   P_RUN      read at the start of a run, apply own updates in registers, add
//              the run's accumulated delta with atomics when the run ends.
//   P_HOT      per row: P_RACY if the row's bit is set in the mode's hot-row
//              bitmap (rows with more updates per sweep than a threshold,
//              whose atomics would serialise on one L2 channel), else P_ATOMIC.
//   P_HOTRUN   per row: P_RACY for a hot row, else P_RUN with runs cut
//              after kRunCap nonzeros (the row is then added and re-read, so
//              a walker's copy is never more than kRunCap own updates away
//              from the shared row: uncut runs of thousands of nonzeros on a
//              row many walkers share add up deltas taken from one stale copy
//              and diverge).  In mode-0 order the nonzeros of one mode-0 row
//              come sorted by the next mode, so runs of one next-mode row are
//              common and each run costs one atomic row update instead of one
//              per nonzero.
// The float atomics are the kernel's limit (the L2 completes about one
// 4-byte atomic per channel per clock), so fewer atomic rows is what pays.
// Walker w processes span (w * stride) mod nspans (stride 1 = natural order).
// ==========================================================================
enum { P_RACY = 0, P_ATOMIC = 1, P_RUN = 2, P_HOT = 3, P_HOTRUN = 4 };
constexpr int kRunCap = 8;

template <int R, int N, int PA, int PB, int PC>
__global__ void __launch_bounds__(256) k_sgd(CissArgs c, FactorArgs fa, HotRows hot, uint32_t span,
                                             uint64_t nspans, uint64_t stride, float step, float lam) {
  constexpr int W = R < 64 ? R : 64;
  constexpr int CPL = R / W;
  constexpr int WPW = 64 / W;
  constexpr uint32_t NONE = 0xFFFFFFFFu;
  const int lane = lane_id();
  const int sub = lane / W;
  const int wl = lane % W;
  const uint64_t wave = (uint64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const uint64_t walker = wave * WPW + sub;
  if (wave * WPW >= nspans) return;  // whole wave idle (uniform)
  const bool live = walker < nspans;
  const uint64_t sp = live ? (walker * stride) % nspans : 0;
  const uint64_t s0 = sp * span;
  const uint64_t s1 = !live ? 0 : (s0 + span < c.nnz ? s0 + span : c.nnz);

  // row slots: 0 = CISS mode (A), 1.. = modes mode+1, ... (B, C, D)
  float *Fm[N];
#pragma unroll
  for (int s = 0; s < N; ++s) Fm[s] = fa.f[s];
  float v[N][CPL], del[N][CPL];
  uint32_t cur[N];
#pragma unroll
  for (int s = 0; s < N; ++s) {
    cur[s] = NONE;
#pragma unroll
    for (int q = 0; q < CPL; ++q) v[s][q] = 0.f, del[s][q] = 0.f;
  }
  uint32_t slot = 0;

  auto pol = [](int s) { return s == 0 ? PA : (s == 1 ? PB : PC); };
  auto bitmapped = [&](int s) { return pol(s) == P_HOT || pol(s) == P_HOTRUN; };
  auto flush_run = [&](int s) {
#pragma unroll
    for (int q2 = 0; q2 < CPL; ++q2) atomic_add_f32(Fm[s] + (size_t)cur[s] * R + wl + q2 * W, del[s][q2]);
  };
  // the cached row of slot s is a P_RUN row whose delta is not yet added, and
  // the nonzeros its run has taken so far
  bool pend[N];
  int runlen[N];
#pragma unroll
  for (int s = 0; s < N; ++s) pend[s] = false, runlen[s] = 0;

  for (uint32_t ch = 0; ch < span; ch += W) {
    const uint64_t el = s0 + ch + wl;
    const bool vl = el < s1;
    uint32_t il[N - 1];
    float xl = 0.f;
    bool hl = false;
    if (vl) {
#pragma unroll
      for (int s = 0; s < N - 1; ++s) il[s] = c.oidx[s][el];
      xl = c.vals[el];
      hl = (c.tile_mask[el >> 6] >> (el & 63)) & 1ull;
    } else {
#pragma unroll
      for (int s = 0; s < N - 1; ++s) il[s] = 0;
    }
    const uint64_t hm = __ballot(vl && hl);
    // hot-row bits of this lane's nonzero, one bit per slot, looked up once
    // per chunk rather than on every nonzero's dependency chain
    int hotl = 0;
#pragma unroll
    for (int s = 1; s < N; ++s)
      if (bitmapped(s) && vl) hotl |= (int)((hot.bits[s][il[s - 1] >> 5] >> (il[s - 1] & 31)) & 1u) << s;
    for (int q = 0; q < W; ++q) {
      const int src = sub * W + q;
      uint32_t idx[N];
#pragma unroll
      for (int s = 0; s < N - 1; ++s) idx[1 + s] = (uint32_t)__shfl((int)il[s], src, 64);
      const float x = __shfl(xl, src, 64);
      const int hotq = __shfl(hotl, src, 64);
      const uint64_t e = s0 + ch + q;
      if (e < s1) {
        const bool head = (hm >> src) & 1ull;
        if (cur[0] == NONE || head) {
          slot = cur[0] == NONE ? c.tile_slot[s0 >> 6] : slot + 1;
          idx[0] = c.directory[slot];
        } else {
          idx[0] = cur[0];
        }
        int pr[N];  // per-row policy of this nonzero
#pragma unroll
        for (int s = 0; s < N; ++s) {
          int P = pol(s);
          if (P == P_HOT) P = ((hotq >> s) & 1) ? P_RACY : P_ATOMIC;
          if (P == P_HOTRUN) P = ((hotq >> s) & 1) ? P_RACY : P_RUN;
          pr[s] = P;
        }
#pragma unroll
        for (int s = 0; s < N; ++s) {
          const int P = pr[s];
          const bool capped = pol(s) == P_HOTRUN && pend[s] && runlen[s] >= kRunCap;
          if (P == P_ATOMIC || idx[s] != cur[s] || capped) {
            if (pend[s]) flush_run(s);  // the cached row's run ends here
            pend[s] = P == P_RUN;
            runlen[s] = 0;
            // an atomic row is re-read at every nonzero: forget it as the cached row
            cur[s] = P == P_ATOMIC ? NONE : idx[s];
#pragma unroll
            for (int q2 = 0; q2 < CPL; ++q2) {
              v[s][q2] = Fm[s][(size_t)idx[s] * R + wl + q2 * W];
              del[s][q2] = 0.f;
            }
          }
        }
        // prediction and error
        float part = 0.f;
#pragma unroll
        for (int q2 = 0; q2 < CPL; ++q2) {
          float pv = v[0][q2];
#pragma unroll
          for (int s = 1; s < N; ++s) pv *= v[s][q2];
          part += pv;
        }
        const float err = x - group_sum<W>(part);
#pragma unroll
        for (int q2 = 0; q2 < CPL; ++q2) {
          // products of all rows but one, from pre-update values
          float oth[N];
#pragma unroll
          for (int s = 0; s < N; ++s) {
            float o = 1.f;
#pragma unroll
            for (int s2 = 0; s2 < N; ++s2)
              if (s2 != s) o *= v[s2][q2];
            oth[s] = o;
          }
          const int col = wl + q2 * W;
#pragma unroll
          for (int s = 0; s < N; ++s) {
            const int P = pr[s];
            const float d = step * (err * oth[s] - lam * v[s][q2]);
            float *dst = Fm[s] + (size_t)idx[s] * R + col;
            if (P == P_ATOMIC) {
              atomic_add_f32(dst, d);
            } else {
              v[s][q2] += d;
              del[s][q2] += d;
              if (P == P_RACY) *dst = v[s][q2];
            }
          }
        }
#pragma unroll
        for (int s = 0; s < N; ++s) runlen[s] += 1;
      }
    }
  }
#pragma unroll
  for (int s = 0; s < N; ++s)
    if (pend[s]) flush_run(s);
}

// ==========================================================================
// Bulk-synchronous SGD (the default schedule).  One launch of k_sgd_sync is
// one sub-step: walker w runs nonzeros [w*span + s*sub, +sub) of its span
// from the factors as they stood when the sub-step began; k_sgd_settle and
// k_sgd_fold then add every row's handed-in deltas to the factors.
//   * Along a run of consecutive nonzeros with the same index in a mode the
//     walker keeps its copy of that row in registers (read where the run
//     starts) and applies the reference step to it (SG/sgd.cu:86-99).
//   * Modes 1..: when a run ends its delta is written to the run's staging
//     slot (a static table numbers every chunk's runs in walk order), and
//     k_sgd_settle adds, per row, the sum of its slots (a cold row: the
//     reference's atomicAdd, SG/sgd.cu:96-98) or their mean (a hot row:
//     replica averaging, NC/sgd.cu:229-262 with the sum of :523-525), summed
//     in a fixed order.  No atomics: the sweep is bitwise reproducible.
//   * Mode 0: a row of at most long_min - 1 nonzeros cannot meet a second
//     walker within one sub-step (two walkers' nonzeros of one sub-step are at
//     least span - sub + 1 positions apart), so its walker stores its copy in
//     place.  A longer row's run deltas are added as 64-bit fixed-point
//     integers (2^-32 units) into its delta sum D (integer addition is
//     associative, so the sum does not depend on the order the walkers finish
//     in), a hot row's into kSyncReplicas replicas with a count of runs, and
//     k_sgd_settle adds the sum (cold) or the mean (hot) and clears them.
// ==========================================================================
constexpr double kFixScale = 4294967296.0;        // 2^32
constexpr double kFixInv = 1.0 / 4294967296.0;    // 2^-32

// Lane shape of the merge and of the row walks below: a walker is W = R / 4
// lanes of a wave; lane l holds the row elements 4l .. 4l + 3, so a row moves
// with one 16-byte access per lane and a wave carries 256 / R walkers (eight at
// R = 32).
template <int R>
struct SyncShape {
  static constexpr int CPL = 4;
  static constexpr int W = R / CPL;
  static constexpr int WPW = 64 / W;
};

template <int CPL>
__device__ inline void load_row4(const float *p, float (&v)[CPL]) {
#pragma unroll
  for (int j = 0; j < CPL; j += 4) {
    const float4 t = *reinterpret_cast<const float4 *>(p + j);
    v[j] = t.x, v[j + 1] = t.y, v[j + 2] = t.z, v[j + 3] = t.w;
  }
}

template <int CPL>
__device__ inline void store_row4(float *p, const float (&v)[CPL]) {
#pragma unroll
  for (int j = 0; j < CPL; j += 4) *reinterpret_cast<float4 *>(p + j) = make_float4(v[j], v[j + 1], v[j + 2], v[j + 3]);
}

// Staged deltas are written once and read once by the next launch: streamed
// past the caches.
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Four BF16 entries per lane (8 bytes): the mixed path's staged deltas.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Lane shape of the SGD walk: a lane holds CPL elements of a row.  A walker's
// time is its chain of instructions per nonzero, which is shorter with two
// elements, while four take fewer instructions in all: see launch_sgd_sync.
template <int R, int CPL>
struct WalkShape {
  static constexpr int W = R / CPL;
  static constexpr int WPW = 64 / W;
};

template <int CPL>
using Cols = float __attribute__((ext_vector_type(CPL)));

// a staged delta, FP32 or BF16 (round to nearest even)
template <int CPL, bool MIX>
__device__ inline void stage_cols(float *stage, size_t at, Cols<CPL> v) {
  if constexpr (MIX) {
    uint32_t __attribute__((ext_vector_type(CPL / 2))) t;
#pragma unroll
    for (int j = 0; j < CPL / 2; ++j) t[j] = (uint32_t)f2bf(v[2 * j]) | ((uint32_t)f2bf(v[2 * j + 1]) << 16);
    __builtin_nontemporal_store(t, reinterpret_cast<decltype(t) *>(reinterpret_cast<uint16_t *>(stage) + at));
  } else {
    __builtin_nontemporal_store(v, reinterpret_cast<Cols<CPL> *>(stage + at));
  }
}

// MIX (the mixed-precision path): the run deltas of modes 1.. are staged in
// BF16 (round to nearest even), halving the staging traffic; the factors, the
// walker's arithmetic and the sums of the deltas stay FP32 / FP64.
//
// A walker's nonzeros are one dependent chain (each step starts from the
// rows the last one left), so what a step waits for and the instructions it
// takes set the time.  Rows of a sub-step do not change while it runs (an
// in-place mode-0 row has one reader, its own walker), so nothing has to wait
// but the arithmetic:
//   * the indices, values, mode-0 rows, run ends and staging positions of
//     SyncMeta::CH nonzeros are read at once and kept in LDS;
//   * the rows of nonzero t + 4 are requested when nonzero t has been
//     consumed, whether a run starts there or not (a row that goes on is a
//     cache hit, and unconditional loads leave the compiler exact wait counts).
// Time of a sub-step's walk at R = 32: 12.5M nonzeros 39 -> 21 us, 50M nonzeros
// 64 -> 53 us (the staged deltas, 200 MB, are written at 3.8 TB/s); R = 64 mixed,
// 5M nonzeros 41 -> 21 us; R = 16, 20K nonzeros 24 -> 14 us.
enum : uint32_t { kOwnRow = 1u, kRunEnd = 2u };  // kRunEnd << k: the run in mode k ends with this nonzero

template <int R, int N, bool MIX, int CPL>
struct SyncMeta {
  static constexpr int W = WalkShape<R, CPL>::W;
  static constexpr int CH = 4 * W < 32 ? 4 * W : 32;      // nonzeros of a walker per round: at most 4 per lane
  static constexpr int WORDS = N + 2 + (MIX ? N - 1 : 0);  // other modes' rows, value, mode-0 row, flags, positions
  // one nonzero more than are kept (read ahead, not used); odd: the walkers'
  // broadcasts fall on different banks
  static constexpr int STRIDE = ((CH + 1) * WORDS) | 1;
  static constexpr size_t kWaveBytes = (size_t)WalkShape<R, CPL>::WPW * STRIDE * sizeof(uint32_t);
};

template <int R, int N, bool MIX, int CPL>
__global__ void __launch_bounds__(256) k_sgd_sync(CissArgs c, FactorArgs fa, SyncArgs sy, uint32_t span,
                                                  uint32_t sub, uint32_t s, uint64_t nspans, uint32_t long_min,
                                                  float step, float lam) {
  constexpr int W = WalkShape<R, CPL>::W;
  constexpr int WPW = WalkShape<R, CPL>::WPW;
  using Meta = SyncMeta<R, N, MIX, CPL>;
  constexpr int CH = Meta::CH, NW = Meta::WORDS, J = CH / W;
  constexpr int B = 4;  // nonzeros whose rows are in flight
  extern __shared__ uint32_t meta_s[];
  const int lane = lane_id();
  const int wl = lane % W;
  const uint64_t wave = (uint64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const uint64_t walker = wave * WPW + lane / W;
  if (wave * WPW >= nspans) return;  // whole wave idle (uniform)
  uint32_t *meta = meta_s + (threadIdx.x / W) * Meta::STRIDE;
  uint64_t e0 = 0;
  uint32_t len = 0;  // this walker's nonzeros in the sub-step
  if (walker < nspans) {
    const uint64_t send = (walker + 1) * span < c.nnz ? (walker + 1) * span : c.nnz;
    e0 = walker * span + (uint64_t)s * sub;
    if (e0 < send) len = (uint32_t)(send - e0 < sub ? send - e0 : sub);
  }
  using V = Cols<CPL>;
  V v[N], del[N];
  bool fresh[N];  // the next nonzero starts a run in mode k
  uint32_t rslot[N];  // modes 1..: the next staging slot
#pragma unroll
  for (int k = 0; k < N; ++k) {
    fresh[k] = true;
    rslot[k] = k >= 1 ? sy.sbase[k][(size_t)s * nspans + (walker < nspans ? walker : nspans - 1)] : 0u;
    v[k] = del[k] = 0.f;
  }

  // the rows in flight of nonzero t (in slot t % B), and what is known of it;
  // what LDS holds of a nonzero is read one nonzero before its rows are requested
  V g[B][N];
  float xb[B], xm = 0.f;
  uint32_t row0[B], fl[B], rm[N], fm = 0;
  auto peek = [&](int t) {
    const uint32_t *w = meta + t * NW;
#pragma unroll
    for (int k = 0; k < N; ++k) rm[k] = w[k == 0 ? N : k - 1];
    xm = __uint_as_float(w[N - 1]);
    fm = w[N + 1];
  };
  auto request = [&](int b) {
    xb[b] = xm, row0[b] = rm[0], fl[b] = fm;
#pragma unroll
    for (int k = 0; k < N; ++k)
      g[b][k] = *reinterpret_cast<const V *>(fa.f[k] + (size_t)rm[k] * R + wl * CPL);
  };
  // a mode-0 run ends: its row is stored in place where no other walker meets
  // it; the deltas of a longer row are added as fixed-point integers
  auto end_row0 = [&](uint32_t row, bool own) {
    if (own) {
      *reinterpret_cast<V *>(fa.f[0] + (size_t)row * R + wl * CPL) = v[0];
      return;
    }
    const uint32_t h = sy.hidx[0][row];
    unsigned long long *d;
    if (h == 0xFFFFFFFFu) {
      d = (unsigned long long *)sy.D[0] + (size_t)row * R;
    } else {
      // a hot row's mean needs its count of runs; a cold row adds its delta
      // sum, so the merge needs no count (an untouched row's sum is 0)
      const size_t r = (size_t)h * kSyncReplicas + walker % kSyncReplicas;
      d = (unsigned long long *)sy.Dh[0] + r * R;
      if (wl == 0) atomicAdd(sy.ch[0] + r, 1u);
    }
#pragma unroll
    for (int j = 0; j < CPL; ++j)
      atomicAdd(d + wl * CPL + j, (unsigned long long)__double2ll_rn((double)del[0][j] * kFixScale));
  };
  auto consume = [&](int t, int b) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      v[k] = fresh[k] ? g[b][k] : v[k];
      del[k] = fresh[k] ? V(0.f) : del[k];
    }
    float part = 0.f;
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      float pv = v[0][j];
#pragma unroll
      for (int k = 1; k < N - 1; ++k) pv *= v[k][j];
      part = fmaf(pv, v[N - 1][j], part);
    }
    const float err = xb[b] - group_sum<W>(part);
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      float d[N];  // the step over its rate
#pragma unroll
      for (int k = 0; k < N; ++k) {
        float o = 1.f;
#pragma unroll
        for (int k2 = 0; k2 < N; ++k2)
          if (k2 != k) o *= v[k2][j];
        d[k] = fmaf(err, o, -(lam * v[k][j]));
      }
#pragma unroll
      for (int k = 0; k < N; ++k) {
        v[k][j] = fmaf(step, d[k], v[k][j]);
        del[k][j] = fmaf(step, d[k], del[k][j]);
      }
    }
#pragma unroll
    for (int k = 0; k < N; ++k) fresh[k] = (fl[b] & (kRunEnd << k)) != 0;
#pragma unroll
    for (int k = 1; k < N; ++k)
      if (fresh[k]) {  // the run's delta goes to its staging slot / position
        const uint32_t at = MIX ? meta[t * NW + N + 1 + k] : rslot[k]++;
        stage_cols<CPL, MIX>(sy.stage[k], (size_t)at * R + wl * CPL, del[k]);
      }
    if (fresh[0]) end_row0(row0[b], (fl[b] & kOwnRow) != 0);
  };

  for (uint32_t ch = 0; ch < sub; ch += CH) {
    wave_sync();  // the last round's reads are done
    const uint32_t n = ch < len ? (len - ch < (uint32_t)CH ? len - ch : (uint32_t)CH) : 0u;
    if (__ballot(n > 0) == 0) break;
    // unconditional, so that all the loads of a step are in flight together
    // (past the walker's end: its last nonzero again, or nonzero 0)
    const uint64_t last = len ? e0 + len - 1 : 0;
    uint32_t ix[J][N - 1], nx[J][N - 1], slot[J], row[J], r0[J], r1[J];
    uint64_t mask[J];
    float x[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const uint64_t at = e0 + ch + j * W + wl, e = at < last ? at : last, f = e < last ? e + 1 : e;
      slot[j] = c.tile_slot[e >> 6], mask[j] = c.tile_mask[e >> 6];
#pragma unroll
      for (int k = 0; k < N - 1; ++k) ix[j][k] = c.oidx[k][e], nx[j][k] = c.oidx[k][f];
      x[j] = c.vals[e];
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const uint64_t at = e0 + ch + j * W + wl, e = at < last ? at : last;
      slot[j] = tile_lane_slot(slot[j], mask[j], (int)(e & 63));
      row[j] = c.directory[slot[j]];
      r0[j] = c.rowptr[slot[j]], r1[j] = c.rowptr[slot[j] + 1];
    }
    uint32_t fl_t[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const uint64_t at = e0 + ch + j * W + wl;
      fl_t[j] = r1[j] - r0[j] < long_min ? kOwnRow : 0u;
      if (at >= last || (uint64_t)r1[j] == at + 1) fl_t[j] |= kRunEnd;
#pragma unroll
      for (int k = 1; k < N; ++k)
        if (at >= last || nx[j][k - 1] != ix[j][k - 1]) fl_t[j] |= kRunEnd << k;
    }
    uint32_t pos[J][N];
    if constexpr (MIX) {
      // staging positions of the runs that end here: the slots counted on from
      // the walker's next one, in walk order
#pragma unroll
      for (int k = 1; k < N; ++k)
#pragma unroll
        for (int j = 0; j < J; ++j) {
          const bool ends = (uint32_t)(j * W + wl) < n && (fl_t[j] & (kRunEnd << k));
          const uint64_t mine = (__ballot(ends) >> (lane - wl)) & (W == 64 ? ~0ull : (1ull << W) - 1);
          pos[j][k] = ends ? sy.dest[k][rslot[k] + __popcll(mine & ((1ull << wl) - 1))] : 0u;
          rslot[k] += __popcll(mine);
        }
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
      uint32_t *w = meta + (j * W + wl) * NW;
#pragma unroll
      for (int k = 0; k < N - 1; ++k) w[k] = ix[j][k];
      w[N - 1] = __float_as_uint(x[j]);
      w[N] = row[j];
      w[N + 1] = fl_t[j];
      if constexpr (MIX)
#pragma unroll
        for (int k = 1; k < N; ++k) w[N + 1 + k] = pos[j][k];
    }
    wave_sync();
#pragma unroll
    for (int b = 0; b < B; ++b) {
      peek(b);
      request(b);
    }
    peek(B);
#pragma unroll 1
    for (int q = 0; q < CH - B; q += B)
#pragma unroll
      for (int b = 0; b < B; ++b) {
        if ((uint32_t)(q + b) < n) consume(q + b, b);
        request(b);
        peek(q + B + b + 1);  // of the last: one past the round's nonzeros, not used
      }
#pragma unroll
    for (int b = 0; b < B; ++b)
      if ((uint32_t)(CH - B + b) < n) consume(CH - B + b, b);
  }
}

// Mode 0's long rows (k_sgd_sync's fixed-point sums) as block `blk` of a
// 256-thread launch: a cold row adds its delta sum D, a hot row the mean of
// its replicas' sums Dh over their count of runs ch; both are cleared.
template <int R>
__device__ inline void sgd_merge_block(const MergeArgs &a, uint64_t blk) {
  constexpr int W = R < 64 ? R : 64;
  constexpr int CPL = R / W;
  constexpr int WPW = 64 / W;
  const int lane = lane_id();
  const int wl = lane % W;
  const uint64_t wave = blk * 4 + (threadIdx.x >> 6);
  const uint64_t i = wave * WPW + lane / W;
  if (i >= a.off[a.nseg]) return;
  int g = 0;
  while (g + 1 < a.nseg && i >= a.off[g + 1]) ++g;
  const int m = a.mode[g];
  const uint64_t k = i - a.off[g];
  if (a.is_hot[g]) {
    // hot row k of mode m: sum its replicas, add the mean of its runs' deltas;
    // the loads of eight replicas at a time, the clearing after them
    static_assert(kSyncReplicas % 8 == 0, "replicas are read in eights");
    uint32_t cnt = 0;
    const uint4 *ch = reinterpret_cast<const uint4 *>(a.ch[m] + k * kSyncReplicas);
#pragma unroll
    for (int r = 0; r < kSyncReplicas / 4; ++r) {
      const uint4 t = ch[r];
      cnt += (t.x + t.y) + (t.z + t.w);
    }
    if (cnt == 0) return;
    const uint32_t row = a.hrow[m][k];
    float *gr = a.F[m] + (size_t)row * R;
    long long *d = a.Dh[m] + k * kSyncReplicas * R;
    const double sc = 1.0 / (double)cnt;
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      const int col = wl + j * W;
      long long sum = 0;
#pragma unroll
      for (int r = 0; r < kSyncReplicas; r += 8) {
        long long x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = d[(size_t)(r + u) * R + col];
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += x[u];
      }
#pragma unroll
      for (int r = 0; r < kSyncReplicas; ++r) d[(size_t)r * R + col] = 0;
      gr[col] = (float)((double)gr[col] + (double)sum * kFixInv * sc);
    }
    if (wl < kSyncReplicas) a.ch[m][k * kSyncReplicas + wl] = 0u;
    if (W < kSyncReplicas)
      for (int r = wl + W; r < kSyncReplicas; r += W) a.ch[m][k * kSyncReplicas + r] = 0u;
    return;
  }
  // cold row: add its delta sum where it is nonzero
  const uint32_t row = a.rows[g] ? a.rows[g][k] : (uint32_t)k;
  float *gr = a.F[m] + (size_t)row * R;
  long long *d = a.D[m] + (size_t)row * R;
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
    const int col = wl + j * W;
    const long long dv = d[col];
    if (dv != 0) {
      gr[col] = (float)((double)gr[col] + (double)dv * kFixInv);
      d[col] = 0;
    }
  }
}

// acc += the staged deltas at positions p, p + stride, ... before e, in that
// order, in FP64.  FP32 deltas sit at their slot, BF16 ones at the position
// itself (positions are numbered over the epoch, s0 is the sub-step's first).
// What a long list waits for is its round trips, so eight deltas are in flight,
// and their slots are read while the eight before them are.
template <int R, bool MIX>
__device__ inline void sum_staged(const float *stage, const uint32_t *slots, uint32_t s0, uint32_t p, uint32_t e,
                                  uint32_t stride, int col, double (&acc)[SyncShape<R>::CPL]) {
  constexpr int CPL = SyncShape<R>::CPL, U = 8;
  static_assert(CPL == 4, "a lane's share of a delta is one 16-byte (BF16: 8-byte) load");
  uint32_t at[U];
  auto slot = [&](uint32_t q) -> uint32_t { return q >= e ? 0u : MIX ? q - s0 : slots[q]; };
#pragma unroll
  for (int u = 0; u < U; ++u) at[u] = slot(p + u * stride);
  for (; p < e; p += U * stride) {
    u32x2 xb[U];  // BF16 deltas as they are stored
    f32x4 xf[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (p + u * stride < e) {
        const size_t i = (size_t)at[u] * R + col;
        if constexpr (MIX)
          xb[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x2 *>(reinterpret_cast<const uint16_t *>(stage) + i));
        else
          xf[u] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(stage + i));
      }
#pragma unroll
    for (int u = 0; u < U; ++u) at[u] = slot(p + (U + u) * stride);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (p + u * stride < e) {
        if constexpr (MIX) {
          acc[0] += (double)bf_lo(xb[u].x), acc[1] += (double)bf_hi(xb[u].x);
          acc[2] += (double)bf_lo(xb[u].y), acc[3] += (double)bf_hi(xb[u].y);
        } else {
#pragma unroll
          for (int j = 0; j < CPL; ++j) acc[j] += (double)xf[u][j];
        }
      }
  }
}

// A row of at most kSettleLight runs, settled by one walker (W lanes) of
// light block lblk: its runs' deltas summed in position order in FP64, the
// sum (cold row) or the mean (hot row) added to the row.
template <int R, bool MIX>
__device__ inline void sgd_settle_light(const SettleArgs &a, uint64_t lblk) {
  constexpr int CPL = SyncShape<R>::CPL;
  constexpr int W = SyncShape<R>::W;
  constexpr int NW = 256 / W;
  const uint64_t li = lblk * NW + threadIdx.x / W;
  const int wl = threadIdx.x % W;
  int k = 1;
  while (k < 3 && li >= a.lb[k + 1]) ++k;
  if (li >= a.lb[k + 1]) return;
  const uint32_t gp = a.light[k][li - a.lb[k]];
  const uint32_t b = a.piece_start[k][gp], e = a.piece_start[k][gp + 1];
  const uint32_t row = a.piece_row[k][gp];
  float *fr = a.F[k] + (size_t)row * R + wl * CPL;
  float fv[CPL];
  load_row4<CPL>(fr, fv);
  const uint32_t hw = a.hot[k][row >> 5];
  double acc[CPL];
#pragma unroll
  for (int j = 0; j < CPL; ++j) acc[j] = 0.0;
  sum_staged<R, MIX>(a.stage[k], a.slots[k], (uint32_t)a.slot0[k], b, e, 1, wl * CPL, acc);
  const double sc = ((hw >> (row & 31)) & 1u) ? 1.0 / (double)(e - b) : 1.0;
  float out[CPL];
#pragma unroll
  for (int j = 0; j < CPL; ++j) out[j] = (float)((double)fv[j] + acc[j] * sc);
  store_row4<CPL>(fr, out);
}

// One launch per sub-step settles every piece of the staged modes and mode 0's
// long rows.  Blocks 0 .. pb[4] - 1: one heavy piece each, whose walkers take
// the piece's positions in turn (FP64 partial sums) and add their partials in
// walker order; a piece that holds a whole row applies it, the others leave
// their sums for k_sgd_fold.  The next nb_light blocks: NW light rows each
// (sgd_settle_light).  The rest: mode 0 (sgd_merge_block).  Every order is
// fixed, so the result is reproducible.  Both lists are sorted by their runs,
// longest first: the walkers of a wave have like counts, and the long pieces
// do not start last.  Bound by the round trips of the longest lists, then by the
// staged deltas (12.5M nonzeros at R = 32: 50 MB): 15.8 us a sub-step (21.4 us
// unsorted, with four deltas in flight; 16.9 us with four and eight waves per
// SIMD), 50M nonzeros 30.9 us (34.4 us), 200 MB at 6.5 TB/s.  With mode 0 here,
// k_sgd_fold (5 us) runs only where a row has several pieces.
template <int R, bool MIX>
__global__ void __launch_bounds__(256, MIX ? 8 : 6) k_sgd_settle(SettleArgs a) {
  constexpr int CPL = SyncShape<R>::CPL;  // a slot's row moves as 16-byte pieces
  constexpr int W = SyncShape<R>::W;
  constexpr int NW = 256 / W;  // walkers per workgroup
  constexpr int G = 256 / R;   // first-level groups of the reduction
  __shared__ double part[NW][R];
  __shared__ double red[G][R];
  const uint64_t pblk = blockIdx.x;
  if (pblk >= a.pb[4]) {  // uniform per block: these paths have no barrier
    if (pblk < a.pb[4] + a.nb_light)
      sgd_settle_light<R, MIX>(a, pblk - a.pb[4]);
    else
      sgd_merge_block<R>(a.mg, pblk - a.pb[4] - a.nb_light);
    return;
  }
  int k = 1;
  while (k < 3 && pblk >= a.pb[k + 1]) ++k;
  const uint64_t gp = a.heavy[k][pblk - a.pb[k]];
  const int wid = threadIdx.x / W;
  const int wl = threadIdx.x % W;
  const uint32_t b = a.piece_start[k][gp], e = a.piece_start[k][gp + 1];
  // a whole row's factor entry and hot bit, read while the slots are summed
  const uint32_t row = a.piece_row[k][gp];
  float fv = 0.f;
  uint32_t hw = 0;
  if (row != 0xFFFFFFFFu && threadIdx.x < R) {
    fv = a.F[k][(size_t)row * R + threadIdx.x];
    hw = a.hot[k][row >> 5];
  }
  double acc[CPL];
#pragma unroll
  for (int j = 0; j < CPL; ++j) acc[j] = 0.0;
  sum_staged<R, MIX>(a.stage[k], a.slots[k], (uint32_t)a.slot0[k], b + wid, e, NW, wl * CPL, acc);
#pragma unroll
  for (int j = 0; j < CPL; ++j) part[wid][wl * CPL + j] = acc[j];
  __syncthreads();
  // walker partials in a fixed order: group g sums walkers g, g + G, ... of
  // those that took a slot, then the groups in order
  const uint32_t used = e - b < (uint32_t)NW ? e - b : (uint32_t)NW;
  {
    const int col = threadIdx.x % R, g = threadIdx.x / R;
    double t = 0.0;
    for (uint32_t w = g; w < used; w += G) t += part[w][col];
    red[g][col] = t;
  }
  __syncthreads();
  if (threadIdx.x < R) {
    double t = 0.0;
#pragma unroll
    for (int g = 0; g < G; ++g) t += red[g][threadIdx.x];
    if (row == 0xFFFFFFFFu) {
      a.part[k][(gp - a.piece0[k]) * R + threadIdx.x] = t;
    } else {
      const double sc = ((hw >> (row & 31)) & 1u) ? 1.0 / (double)(e - b) : 1.0;
      a.F[k][(size_t)row * R + threadIdx.x] = (float)((double)fv + t * sc);
    }
  }
}

// One walker per staged row of more than one piece adds its pieces' partial
// sums in order, then the total (a cold row) or the total over its count of
// runs (a hot row) to the row.
template <int R>
__global__ void __launch_bounds__(256) k_sgd_fold(SettleArgs a) {
  constexpr int W = R < 64 ? R : 64;
  constexpr int CPL = R / W;
  constexpr int WPW = 64 / W;
  const int wl = lane_id() % W;
  const uint64_t i = ((uint64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * WPW + lane_id() / W;
  int k = 1;
  while (k < 3 && i >= a.fb[k + 1]) ++k;
  if (i >= a.fb[k + 1]) return;
  const FoldSeg sg = a.fold[k][i - a.fb[k]];
  const double *pt = a.part[k];
  double t[CPL];
#pragma unroll
  for (int j = 0; j < CPL; ++j) t[j] = 0.0;
#pragma unroll 4
  for (uint32_t q = 0; q < sg.npiece; ++q)
#pragma unroll
    for (int j = 0; j < CPL; ++j) t[j] += pt[(size_t)(sg.piece + q) * R + wl + j * W];
  const uint32_t *hot = a.hot[k];
  const double sc = ((hot[sg.row >> 5] >> (sg.row & 31)) & 1u) ? 1.0 / (double)sg.runs : 1.0;
  float *gr = a.F[k] + (size_t)sg.row * R;
#pragma unroll
  for (int j = 0; j < CPL; ++j) gr[wl + j * W] = (float)((double)gr[wl + j * W] + t[j] * sc);
}

// ==========================================================================
// MTTKRP / adjoint walk: per row, acc = sum over its nonzeros of w * h with
// h = hadamard of the other modes' rows and
//   w = x                       (kWalkMttkrp: SG/als.cu:295-312 intent), or
//   w = x - <F_mode(row), h>    (kWalkAdjoint, kWalkJacobi: the residual).
// A row that starts and ends inside a walker's span is stored.  The rows open
// at the ends of the spans (a walker's first, where it continues, and its
// last) are first joined in LDS along the workgroup's walkers, whose spans are
// consecutive, and each joined row is added with one atomic per entry into the
// initialised output.  A hot row so costs one atomic row per workgroup: one
// per walker queued on the row's memory channel for longer than the walk took.
// For the adjoint, out holds lambda c F (c = the row's nonzeros or 1) and
// receives -acc, and loss_part the per-block sum of squared residuals.
// kWalkJacobi is the reference's CCD sums (SG/ccd.cu:157-195): out receives
// acc = sum e h and den the sum of h * h, per column, all from the factors as
// they were at launch.  kWalkLoss only sums the squared residuals into
// loss_part (the training loss of tc_loss_sq, SG/completion.c:166-189).
// Bound by the gathers of the other modes' rows: the rows of four nonzeros are
// gathered together, the next chunk's indices one chunk ahead (44 registers at
// N = 3).  MTTKRP of 8M nonzeros at R = 32 132 us per mode (117 us with spans of
// 256, see walk_span: 2.1 times the indices, values and rows a CU can take from
// its cache at 64 B per clock); with an atomic row per walker and row 258 us.  The
// adjoint of 20M nonzeros of a 4-way tensor 495 us per mode (1087 us).  Two or
// eight nonzeros at a time: 128 / 145 us and 525 / 504 us.
// ==========================================================================
enum : int { kWalkMttkrp = 0, kWalkAdjoint = 1, kWalkJacobi = 2, kWalkLoss = 3 };

template <int R, int N, int KIND>
__global__ void __launch_bounds__(256) k_mttkrp(CissArgs c, FactorArgs fa, uint32_t span, float *out,
                                                double *loss_part, float *den, float lam, int per_occ) {
  constexpr bool ADJ = KIND != kWalkMttkrp;  // w is the residual
  constexpr bool SQ = KIND == kWalkJacobi;
  // a walker is R / 4 lanes, each holding 4 consecutive entries of a row, so
  // a gathered row is one 16-byte load per lane and a wave carries 256 / R
  // walkers (the shape of the SGD walk)
  constexpr int W = SyncShape<R>::W;
  constexpr int CPL = SyncShape<R>::CPL;
  constexpr int WPW = SyncShape<R>::WPW;
  constexpr uint32_t NONE = 0xFFFFFFFFu;
  constexpr int NWK = 256 / W;  // walkers of a workgroup, and the open rows they leave: first, last
  constexpr bool SUMS = KIND != kWalkLoss;
  __shared__ double red[4];
  __shared__ float open_s[SUMS ? 2 * NWK : 1][R], open_q[SQ ? 2 * NWK : 1][R];
  __shared__ uint32_t open_id[2 * NWK];
  const int lane = lane_id();
  const int sub = lane / W;
  const int wl = lane % W;
  const int wk = threadIdx.x / W;
  const uint64_t wave = (uint64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const uint64_t walker = wave * WPW + sub;
  const uint64_t s0 = walker * span;
  const uint64_t s1 = s0 + span < c.nnz ? s0 + span : c.nnz;
  const bool wave_idle = wave * WPW * (uint64_t)span >= c.nnz;

  float acc[CPL], own[CPL], sq[CPL];
  double lsum = 0.0;
  uint32_t arow = NONE, cnt = 0;
  bool cont = false;  // the open row began before this span
  if (SUMS && wl == 0) open_id[2 * wk] = open_id[2 * wk + 1] = NONE;
#pragma unroll
  for (int q = 0; q < CPL; ++q) acc[q] = 0.f, own[q] = 0.f, sq[q] = 0.f;
  constexpr bool LOSS = KIND == kWalkAdjoint || KIND == kWalkLoss;  // the squared residuals are summed
  constexpr int B = W < 4 ? W : 4;  // nonzeros whose rows are gathered together
  auto leave_open = [&](int e) {
    if (wl == 0) open_id[e] = arow;
    store_row4<CPL>(&open_s[SUMS ? e : 0][wl * CPL], acc);
    if (SQ) store_row4<CPL>(&open_q[SQ ? e : 0][wl * CPL], sq);
  };
  auto end_row = [&]() {  // a row that ends inside the span
    if (!SUMS) return;
    if (cont) {
      leave_open(2 * wk);
      cont = false;
      return;
    }
    float v[CPL];
    const float reg = lam * (per_occ ? (float)cnt : 1.f);
#pragma unroll
    for (int q2 = 0; q2 < CPL; ++q2) v[q2] = KIND == kWalkAdjoint ? reg * own[q2] - acc[q2] : acc[q2];
    store_row4<CPL>(out + (size_t)arow * R + wl * CPL, v);
    if (SQ) store_row4<CPL>(den + (size_t)arow * R + wl * CPL, sq);
  };

  if (!wave_idle) {
    // the next chunk's indices, value and tile word of this lane's nonzero
    uint32_t in[N - 1], tsn = 0;
    float xn = 0.f;
    uint64_t mn = 0;
    auto fetch = [&](uint32_t ch) {
      const uint64_t el = s0 + ch + wl;
#pragma unroll
      for (int s = 0; s < N - 1; ++s) in[s] = 0;
      if (ch < span && el < s1) {
#pragma unroll
        for (int s = 0; s < N - 1; ++s) in[s] = c.oidx[s][el];
        xn = c.vals[el];
        mn = c.tile_mask[el >> 6];
        tsn = c.tile_slot[el >> 6];
      }
    };
    fetch(0);
    for (uint32_t ch = 0; ch < span; ch += W) {
      const uint64_t el = s0 + ch + wl;
      uint32_t il[N - 1], rl = 0;
#pragma unroll
      for (int s = 0; s < N - 1; ++s) il[s] = in[s];
      const float xl = xn;
      bool hl = false;
      if (el < s1) {
        hl = (mn >> (el & 63)) & 1ull;
        rl = c.directory[tile_lane_slot(tsn, mn, (int)(el & 63))];
      }
      const uint64_t hm = __ballot(hl);
      fetch(ch + W);
#pragma unroll 1
      for (int q0 = 0; q0 < W; q0 += B) {
        float g[B][N - 1][CPL], og[ADJ ? B : 1][CPL];
        uint32_t rb[B];
        bool nw[B];
#pragma unroll
        for (int b = 0; b < B; ++b) {
          const int src = sub * W + q0 + b;
          rb[b] = (uint32_t)__shfl((int)rl, src, 64);
          nw[b] = ((hm >> src) & 1ull) || (ch + q0 + b == 0);  // starts a row or the walker's span
#pragma unroll
          for (int s = 0; s < N - 1; ++s)  // past the end: row 0, not used
            load_row4<CPL>(fa.f[1 + s] + (size_t)(uint32_t)__shfl((int)il[s], src, 64) * R + wl * CPL, g[b][s]);
          if constexpr (ADJ)
            if (nw[b]) load_row4<CPL>(fa.f[0] + (size_t)rb[b] * R + wl * CPL, og[b]);
        }
#pragma unroll
        for (int b = 0; b < B; ++b) {
          const float x = __shfl(xl, sub * W + q0 + b, 64);
          if (s0 + ch + q0 + b < s1) {
            if (nw[b]) {
              if (arow != NONE)
                end_row();
              else
                cont = !((hm >> (sub * W + q0 + b)) & 1ull);
              arow = rb[b];
              cnt = 0;
#pragma unroll
              for (int q2 = 0; q2 < CPL; ++q2) {
                acc[q2] = 0.f, sq[q2] = 0.f;
                if (ADJ) own[q2] = og[b][q2];
              }
            }
            float h[CPL];
#pragma unroll
            for (int q2 = 0; q2 < CPL; ++q2) h[q2] = g[b][0][q2];
#pragma unroll
            for (int s = 1; s < N - 1; ++s)
#pragma unroll
              for (int q2 = 0; q2 < CPL; ++q2) h[q2] *= g[b][s][q2];
            float w = x;
            if (ADJ) {
              float part = 0.f;
#pragma unroll
              for (int q2 = 0; q2 < CPL; ++q2) part += own[q2] * h[q2];
              w = x - group_sum<W>(part);
              if (LOSS && wl == 0) lsum += (double)w * (double)w;
            }
            ++cnt;
#pragma unroll
            for (int q2 = 0; q2 < CPL; ++q2) {
              acc[q2] += w * h[q2];
              if (SQ) sq[q2] += h[q2] * h[q2];
            }
          }
        }
      }
    }
    if (SUMS && arow != NONE) leave_open(2 * wk + 1);
  }
  if (SUMS) {
    __syncthreads();
    // join the open rows of consecutive walkers: a row's first entry takes it
    auto add = [&](int e, bool more) {
      float s[CPL], s2[CPL];
      const uint32_t id = open_id[e];
      load_row4<CPL>(&open_s[e][wl * CPL], s);
      if (SQ) load_row4<CPL>(&open_q[SQ ? e : 0][wl * CPL], s2);
      for (int v = wk + 1; more && v < (int)(blockDim.x / W); ++v) {
        const uint32_t f = open_id[2 * v];
        const int from = f == id ? 2 * v : f == NONE && open_id[2 * v + 1] == id ? 2 * v + 1 : -1;
        if (from < 0) break;
        float t[CPL];
        load_row4<CPL>(&open_s[from][wl * CPL], t);
#pragma unroll
        for (int q2 = 0; q2 < CPL; ++q2) s[q2] += t[q2];
        if (SQ) {
          load_row4<CPL>(&open_q[SQ ? from : 0][wl * CPL], t);
#pragma unroll
          for (int q2 = 0; q2 < CPL; ++q2) s2[q2] += t[q2];
        }
        if (from == 2 * v) break;  // it ended inside that span
      }
#pragma unroll
      for (int q2 = 0; q2 < CPL; ++q2) {
        atomic_add_f32(out + (size_t)id * R + wl * CPL + q2, KIND == kWalkAdjoint ? -s[q2] : s[q2]);
        if (SQ) atomic_add_f32(den + (size_t)id * R + wl * CPL + q2, s2[q2]);
      }
    };
    const uint32_t first = open_id[2 * wk], last = open_id[2 * wk + 1];
    if (first != NONE && wk == 0) add(0, false);
    if (last != NONE && (wk == 0 || first != NONE || open_id[2 * wk - 1] != last)) add(2 * wk + 1, true);
  }
  if (LOSS) {
    double t = wave_sum_d(lsum);
    if (lane == 0) red[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
      double s = 0.0;
      for (int w2 = 0; w2 < (int)(blockDim.x >> 6); ++w2) s += red[w2];
      loss_part[blockIdx.x] = s;
    }
  }
}

// ==========================================================================
// ALS, phase 1: Gram + MTTKRP walk on the FP64 matrix cores.
//
// One wave per span.  Per row segment the wave accumulates
//   G += h h^T  with v_mfma_f64_16x16x4_f64 (h = hadamard of the other
//               modes' rows, formed exactly in FP64 from the FP32 factors)
//   m += x h    in FP64 on the VALUs
// and writes (G, m) as an FP64 "piece" when the row ends or the span ends.
// Piece ids are slot + span_off[span], so the pieces of a slot are contiguous
// and written exactly once: no atomics, fixed summation order
// (deterministic).  Lane l holds column (l % 16) + 16 q of nonzero l / 16 of
// the current 4-nonzero step, which is exactly the A (16 x 4) and B (4 x 16)
// operand layout of the 16x16x4 shape, so both operands are the same h
// registers; block (bi, bj) of G (bi >= bj) takes A = h[bi], B = h[bj].
// FP64 accumulation keeps the normal equations within 1e-5 of an FP64
// reference even when (G + lambda I) is poorly conditioned.
//
// tile_thin (null: none) marks the nonzeros of rows that are solved in their
// dual form: the walk passes over them and writes no piece for their rows.
// ==========================================================================
typedef double doublex4 __attribute__((ext_vector_type(4)));

template <int R, int N>
__device__ __forceinline__ void als_gram_walk(const CissArgs &c, const FactorArgs &fa, uint32_t span_tiles,
                                              uint64_t nspans, const uint32_t *span_off, const uint64_t *tile_thin,
                                              double *pieces) {
  constexpr int CG = (R + 15) / 16;      // 16-column groups
  constexpr int NB = CG * (CG + 1) / 2;  // lower-triangle 16x16 blocks
  constexpr int NPS = 4;                 // nonzeros per MFMA step
  constexpr size_t PSZ = (size_t)R * R + R;
  const int lane = lane_id();
  const uint64_t w = (uint64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (w >= nspans) return;
  const uint64_t t0 = w * span_tiles;
  const uint64_t t1 = t0 + span_tiles < c.ntiles ? t0 + span_tiles : c.ntiles;
  const uint32_t poff = span_off[w];
  uint32_t slot = c.tile_slot[t0];
  bool skip = false;  // the open row is marked in tile_thin
  const int col = lane & 15;
  const int nsub = lane >> 4;

  doublex4 acc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[b] = doublex4{0.0, 0.0, 0.0, 0.0};
  double macc[CG];
#pragma unroll
  for (int q = 0; q < CG; ++q) macc[q] = 0.0;

  auto flush = [&](uint32_t pid) {
    double *P = pieces + (size_t)pid * PSZ;
    int b = 0;
#pragma unroll
    for (int bi = 0; bi < CG; ++bi) {
#pragma unroll
      for (int bj = 0; bj <= bi; ++bj, ++b) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          // f64 16x16x4 output: accumulator v of lane l is row 4 v + l / 16
          const int row = 16 * bi + 4 * v + nsub, cc = 16 * bj + col;
          if (row < R && cc < R) P[row * R + cc] = acc[b][v];
          acc[b][v] = 0.0;
        }
      }
    }
#pragma unroll
    for (int q = 0; q < CG; ++q) {
      double mt = macc[q];
      mt += __shfl_xor(mt, 16, 64);
      mt += __shfl_xor(mt, 32, 64);
      if (lane < 16 && 16 * q + lane < R) P[R * R + 16 * q + lane] = mt;
      macc[q] = 0.0;
    }
  };

  for (uint64_t t = t0; t < t1; ++t) {
    const uint64_t base = t * kTile;
    const uint32_t cnt = (uint32_t)((c.nnz - base) < (uint64_t)kTile ? (c.nnz - base) : kTile);
    uint32_t jl = 0, kl = 0, ll = 0;
    float xl = 0.f;
    if ((uint32_t)lane < cnt) {
      jl = c.oidx[0][base + lane];
      kl = c.oidx[1][base + lane];
      if (N == 4) ll = c.oidx[2][base + lane];
      xl = c.vals[base + lane];
    }
    uint64_t mask = c.tile_mask[t];
    if (cnt < 64) mask &= (1ull << cnt) - 1ull;
    const uint64_t thin = tile_thin ? tile_thin[t] : 0ull;
    uint32_t pos = 0;
    while (pos < cnt) {
      if ((mask >> pos) & 1ull) {
        if (!(t == t0 && pos == 0)) {
          if (!skip) flush(slot + poff);
          ++slot;
        }
      }
      skip = (thin >> pos) & 1ull;
      if (skip) {  // on to the next nonzero that is not marked, past the rows that start on the way
        const uint64_t stop = ~thin >> pos;
        uint32_t to = stop ? pos + (uint32_t)__ffsll((unsigned long long)stop) - 1u : cnt;
        if (to > cnt) to = cnt;
        const uint64_t upto = to >= 64 ? ~0ull : (1ull << to) - 1ull;
        slot += (uint32_t)__popcll(mask & upto & ~((2ull << pos) - 1ull));
        pos = to;
        continue;
      }
      const uint64_t rest = (pos >= 63) ? 0ull : ((mask >> (pos + 1)) << (pos + 1));
      uint32_t nxt = rest ? (uint32_t)__ffsll((unsigned long long)rest) - 1u : cnt;
      if (nxt > cnt) nxt = cnt;
      // the factor values of step e are gathered one step ahead (inside the
      // row segment), so a wave has the next step's loads in flight under
      // the current step's MFMAs
      float f1[CG], f2[CG], f3[CG];
      auto fetch = [&](uint32_t e, float (&g1)[CG], float (&g2)[CG], float (&g3)[CG]) {
        const uint32_t my = e + (uint32_t)nsub;
        const int src = (int)(my < 64 ? my : 63);
        const uint32_t j = (uint32_t)__shfl((int)jl, src, 64);
        const uint32_t k = (uint32_t)__shfl((int)kl, src, 64);
        const uint32_t l = N == 4 ? (uint32_t)__shfl((int)ll, src, 64) : 0u;
#pragma unroll
        for (int q = 0; q < CG; ++q) {
          const int cq = col + 16 * q;
          g1[q] = g2[q] = g3[q] = 0.f;
          if (my < nxt && cq < R) {
            g1[q] = fa.f[1][(size_t)j * R + cq];
            g2[q] = fa.f[2][(size_t)k * R + cq];
            if (N == 4) g3[q] = fa.f[3][(size_t)l * R + cq];
          }
        }
      };
      fetch(pos, f1, f2, f3);
      for (uint32_t e = pos; e < nxt; e += NPS) {
        const uint32_t my = e + (uint32_t)nsub;
        const bool valid = my < nxt;
        const int src = (int)(my < 64 ? my : 63);
        const double x = (double)__shfl(xl, src, 64);
        float n1[CG], n2[CG], n3[CG];
        if (e + NPS < nxt) fetch(e + NPS, n1, n2, n3);
        double h[CG];
#pragma unroll
        for (int q = 0; q < CG; ++q) {
          double v = 0.0;
          if (valid && col + 16 * q < R) {
            v = (double)f1[q] * (double)f2[q];
            if (N == 4) v *= (double)f3[q];
          }
          h[q] = v;
          macc[q] += x * v;
        }
        int b = 0;
#pragma unroll
        for (int bi = 0; bi < CG; ++bi)
#pragma unroll
          for (int bj = 0; bj <= bi; ++bj, ++b)
            acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(h[bi], h[bj], acc[b], 0, 0, 0);
#pragma unroll
        for (int q = 0; q < CG; ++q) f1[q] = n1[q], f2[q] = n2[q], f3[q] = n3[q];
      }
      pos = nxt;
    }
  }
  if (!skip) flush(slot + poff);
}

// Occupancy: at R <= 32 the walk (with its one-step gather lookahead) is held
// to 6 waves per SIMD, about 80 registers; at R = 64, and at R = 32 with four
// modes (which would spill at 80), it keeps the compiler's default.  Measured on
// the 100M-nonzero tensor at R = 32: 4.56 ms per mode without lookahead at the
// default occupancy, 4.27 ms without lookahead at 7 waves, 4.00 ms with lookahead
// at 6.
template <int R, int N>
__global__ void __launch_bounds__(256, 6) k_als_gram(CissArgs c, FactorArgs fa, uint32_t span_tiles,
                                                     uint64_t nspans, const uint32_t *span_off,
                                                     const uint64_t *tile_thin, double *pieces) {
  als_gram_walk<R, N>(c, fa, span_tiles, nspans, span_off, tile_thin, pieces);
}
template <int R, int N>
__global__ void __launch_bounds__(256) k_als_gram_wide(CissArgs c, FactorArgs fa, uint32_t span_tiles,
                                                       uint64_t nspans, const uint32_t *span_off,
                                                       const uint64_t *tile_thin, double *pieces) {
  als_gram_walk<R, N>(c, fa, span_tiles, nspans, span_off, tile_thin, pieces);
}

// ==========================================================================
// ALS, phase 2: per directory slot, sum its pieces in FP64, add lambda to the
// diagonal (p_update_matrice, SG/als.cu:484-487), factor the R x R system by
// Cholesky (right-looking, Golub & Van Loan 4.2) in FP64 in LDS, solve, and
// optionally refine once: x += (G+lambda I)^-1 (m - (G+lambda I) x).
// One 64-thread workgroup per slot.  Replaces cusolverDnDpotrfBatched +
// DpotrsBatched (SG/als.cu:715-716).
// ==========================================================================
__device__ inline int tri_row(int t) {
  int a = (int)((sqrtf(8.f * (float)t + 1.f) - 1.f) * 0.5f);
  if ((a + 1) * (a + 2) / 2 <= t) ++a;
  if (a * (a + 1) / 2 > t) --a;
  return a;
}

// Heavy slots (more pieces than the solve's serial sum should take) are first
// reduced in fixed groups of consecutive pieces.  A thread owns one element of
// a group's sum (blockIdx.y: 256 elements of the piece), eight pieces' loads in
// flight, added in piece order: the rank-32 class of a batch (1.8M nonzeros) 41 us per
// mode, 1M nonzeros at R = 16 7 us; on the span kernels 20M nonzeros at R = 32 take 32 us
// (218 us with one 64-thread workgroup per group and a load at a time).
template <int R>
__global__ void __launch_bounds__(256) k_piece_reduce(const double *pieces, const uint32_t *grp_piece,
                                                      const uint32_t *grp_n, double *gsum) {
  constexpr uint32_t PSZ = R * R + R;
  const uint32_t e = blockIdx.y * 256 + threadIdx.x;
  if (e >= PSZ) return;
  const uint64_t g = blockIdx.x;
  const double *P = pieces + (size_t)grp_piece[g] * PSZ + e;
  const uint32_t n = grp_n[g];
  double acc = 0.0;
  uint32_t q = 0;
  for (; q + 8 <= n; q += 8) {
    double x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = P[(size_t)(q + u) * PSZ];
#pragma unroll
    for (int u = 0; u < 8; ++u) acc += x[u];
  }
  for (; q < n; ++q) acc += P[(size_t)q * PSZ];
  gsum[g * PSZ + e] = acc;
}

template <int R, bool REFINE>
__global__ void __launch_bounds__(64) k_als_solve(const double *pieces, const uint32_t *slot_pb,
                                                  const double *gsum, const uint32_t *slot_gb,
                                                  const uint32_t *directory, uint64_t dlength,
                                                  double lam, float *A, uint32_t *flag) {
  constexpr int LD = R + 1;
  constexpr size_t PSZ = (size_t)R * R + R;
  constexpr int PER = (R * R + 63) / 64;
  __shared__ double Gs[R * LD];
  __shared__ double G0[REFINE ? R * LD : 1];
  __shared__ double ys[R], rs[R];
  const int lane = threadIdx.x;
  const uint64_t s = blockIdx.x;
  if (s >= dlength) return;
  uint32_t p0 = slot_pb[s], p1 = slot_pb[s + 1];
  const double *src = pieces;
  if (slot_gb && slot_gb[s + 1] > slot_gb[s]) {  // heavy slot: read its group sums
    p0 = slot_gb[s];
    p1 = slot_gb[s + 1];
    src = gsum;
  }

  double g[PER];
#pragma unroll
  for (int t = 0; t < PER; ++t) g[t] = 0.0;
  double mv = 0.0;
  for (uint32_t p = p0; p < p1; ++p) {
    const double *P = src + (size_t)p * PSZ;
#pragma unroll
    for (int t = 0; t < PER; ++t) {
      const int idx = lane + 64 * t;
      if (idx < R * R) {
        const int i = idx / R, j = idx % R;
        const int hi = i > j ? i : j, lo = i > j ? j : i;
        g[t] += P[hi * R + lo];
      }
    }
    if (lane < R) mv += P[R * R + lane];
  }
#pragma unroll
  for (int t = 0; t < PER; ++t) {
    const int idx = lane + 64 * t;
    if (idx < R * R) {
      const int i = idx / R, j = idx % R;
      const double v = g[t] + (i == j ? lam : 0.0);
      Gs[i * LD + j] = v;
      if (REFINE) G0[i * LD + j] = v;
    }
  }
  if (lane < R) {
    ys[lane] = mv;
    rs[lane] = mv;
  }
  __syncthreads();

  bool bad = false;
  for (int k = 0; k < R; ++k) {
    double d = Gs[k * LD + k];
    if (!(d > 0.0)) {
      bad = true;
      d = 1.0;
    }
    const double lkk = sqrt(d), inv = 1.0 / lkk;
    __syncthreads();
    if (lane == 0) Gs[k * LD + k] = lkk;
    for (int i = k + 1 + lane; i < R; i += 64) Gs[i * LD + k] *= inv;
    __syncthreads();
    const int n = R - k - 1;
    const int T = n * (n + 1) / 2;
    for (int t = lane; t < T; t += 64) {
      const int a = tri_row(t), b = t - a * (a + 1) / 2;
      const int i = k + 1 + a, j = k + 1 + b;
      Gs[i * LD + j] -= Gs[i * LD + k] * Gs[j * LD + k];
    }
    __syncthreads();
  }

  auto solve = [&](double *y) __attribute__((always_inline)) {
    for (int k = 0; k < R; ++k) {  // L y = b
      const double yk = y[k] / Gs[k * LD + k];
      __syncthreads();
      if (lane == 0) y[k] = yk;
      for (int i = k + 1 + lane; i < R; i += 64) y[i] -= Gs[i * LD + k] * yk;
      __syncthreads();
    }
    for (int k = R - 1; k >= 0; --k) {  // L^T x = y
      const double xk = y[k] / Gs[k * LD + k];
      __syncthreads();
      if (lane == 0) y[k] = xk;
      for (int i = lane; i < k; i += 64) y[i] -= Gs[k * LD + i] * xk;
      __syncthreads();
    }
  };
  solve(ys);
  if (REFINE) {
    if (lane < R) {
      double r = rs[lane];
      for (int j = 0; j < R; ++j) {
        const int hi = lane > j ? lane : j, lo = lane > j ? j : lane;
        r -= G0[hi * LD + lo] * ys[j];
      }
      rs[lane] = r;
    }
    __syncthreads();
    solve(rs);
    if (lane < R) ys[lane] += rs[lane];
    __syncthreads();
  }
  const uint32_t row = directory[s];
  if (lane < R) A[(size_t)row * R + lane] = bad ? 0.f : (float)ys[lane];
  if (bad && lane == 0) atomicOr(flag, 1u);
}

// Same solve without refinement for R <= 32, one half-wave (32 lanes) per
// slot, eight slots per 256-thread workgroup, no workgroup barriers.  Lane c
// keeps column c of G in registers (rows i >= c; the upper part of the
// register column holds don't-care values).  Root-free right-looking LDL^T:
// at step k lane k publishes its column and right-hand-side entry to a
// per-slot LDS buffer; d_k = buf[k] + lambda (lambda only ever sits on the
// diagonal, so it is added when the pivot is read); every lane c > k
// subtracts buf[i] * buf[c] / d_k from its column and l_ck z_k from its
// right-hand-side entry, so the forward solve L z = m rides along.  Masking is
// done by zero coefficients, not branches.  Then x = L^-T (D^-1 z), with
// l_kc = g[k] / d_c read from lane c's own registers.  Instruction count per
// system is about R^2 FMAs plus R reciprocals; the kernel is issue-bound, so
// that count is its time.
template <int R>
__global__ void __launch_bounds__(256) k_als_solve_h(const double *pieces, const uint32_t *slot_pb,
                                                     const double *gsum, const uint32_t *slot_gb,
                                                     const uint32_t *directory, const uint32_t *list, uint64_t count,
                                                     double lam, float *A, uint32_t *flag) {
  static_assert(R <= 32, "one half-wave per slot");
  constexpr size_t PSZ = (size_t)R * R + R;
  constexpr int CB = R + 2;  // column k, then z_k / x_k; even, so every half's buffer is 16-byte aligned
  __shared__ __align__(16) double cbuf[8][CB];
  const int lane = lane_id();
  const int c = lane & 31;
  const int cc = c < R ? c : R - 1;  // clamped column for lanes past the rank
  const int hw = (int)(threadIdx.x >> 5);
  const uint64_t i0 = (uint64_t)blockIdx.x * 8 + (uint64_t)hw;
  const bool live = i0 < count;
  const uint64_t s = live && list ? list[i0] : i0;
  double *buf = cbuf[hw];

  double g[R];
#pragma unroll
  for (int i = 0; i < R; ++i) g[i] = 0.0;
  double b = 0.0;
  if (live && c < R) {
    uint32_t p0 = slot_pb[s], p1 = slot_pb[s + 1];
    const double *src = pieces;
    if (slot_gb && slot_gb[s + 1] > slot_gb[s]) {  // heavy slot: its group sums
      p0 = slot_gb[s];
      p1 = slot_gb[s + 1];
      src = gsum;
    }
#pragma unroll 1
    for (uint32_t p = p0; p < p1; ++p) {
      const double *P = src + (size_t)p * PSZ;
      // rows i < c are above the diagonal: don't-care (inside the piece, never used)
#pragma unroll
      for (int i = 0; i < R; ++i) g[i] += P[i * R + c];
      b += P[R * R + c];
    }
  }

  bool bad = false;
  double rd = 1.0;  // lane c: 1 / d_c
#pragma unroll
  for (int k = 0; k < R; ++k) {
    if (c == k) {
#pragma unroll
      for (int i = k; i < R; ++i) buf[i] = g[i];
      buf[R] = b;
    }
    wave_sync();
    double d = buf[k] + lam;
    if (!(d > 0.0)) {
      bad = true;
      d = 1.0;
    }
    const double rk = rcp_f64(d);
    const double zk = buf[R];
    const double lck = c > k ? buf[cc] * rk : 0.0;  // l_ck for the lanes still to factor, else 0
#pragma unroll
    for (int i = k + 1; i < R; ++i) g[i] = __builtin_fma(-buf[i], lck, g[i]);
    b = __builtin_fma(-lck, zk, b);
    if (c == k) rd = rk;
    wave_sync();
  }
  // w = D^-1 z, then L^T x = w
  b *= rd;
#pragma unroll
  for (int k = R - 1; k >= 0; --k) {
    if (c == k) buf[R] = b;
    wave_sync();
    const double xk = buf[R];
    const double lkc = c < k ? g[k] * rd : 0.0;  // l_kc (unit lower factor) for lanes before k
    b = __builtin_fma(-lkc, xk, b);
    wave_sync();
  }
  if (live && c < R) A[(size_t)directory[s] * R + c] = bad ? 0.f : (float)b;
  if (live && bad && c == 0) atomicOr(flag, 1u);
}

// ==========================================================================
// Evaluation: sum of squared errors over a COO (validation / test) or per
// problem of a batch, FP64 accumulation, one partial per block (fixed grid,
// fixed order -> deterministic).  The training loss is a walk of the mode-0
// CISS (k_mttkrp, kWalkLoss).
// ==========================================================================
template <int N>
__device__ inline float predict_row(const float *const *F, const uint32_t *ix, int R) {
  const float *r0 = F[0] + (size_t)ix[0] * R;
  const float *r1 = F[1] + (size_t)ix[1] * R;
  const float *r2 = N > 2 ? F[2] + (size_t)ix[2] * R : nullptr;
  const float *r3 = N > 3 ? F[3] + (size_t)ix[3] * R : nullptr;
  float acc = 0.f;
  for (int f = 0; f < R; f += 4) {
    float4 a = *(const float4 *)(r0 + f);
    float4 b = *(const float4 *)(r1 + f);
    float4 v = make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w);
    if (N > 2) {
      float4 cc = *(const float4 *)(r2 + f);
      v = make_float4(v.x * cc.x, v.y * cc.y, v.z * cc.z, v.w * cc.w);
    }
    if (N > 3) {
      float4 d = *(const float4 *)(r3 + f);
      v = make_float4(v.x * d.x, v.y * d.y, v.z * d.z, v.w * d.w);
    }
    acc += (v.x + v.y) + (v.z + v.w);
  }
  return acc;
}

__device__ inline void block_store_sum(double v, double *out) {
  __shared__ double red[8];
  v = wave_sum_d(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += red[w];
    *out = s;
  }
}

template <int N>
__global__ void __launch_bounds__(256) k_eval_coo(CooArgs c, FactorArgs fa, int R, double *part) {
  double acc = 0.0;
  const float *F[4] = {fa.f[0], fa.f[1], fa.f[2], fa.f[3]};
  for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < c.nnz;
       p += (uint64_t)gridDim.x * blockDim.x) {
    uint32_t ix[4];
#pragma unroll
    for (int m = 0; m < N; ++m) ix[m] = c.ind[m][p];
    const double e = (double)c.vals[p] - (double)predict_row<N>(F, ix, R);
    acc += e * e;
  }
  block_store_sum(acc, part + blockIdx.x);
}

// Squared error per segment [seg[b], seg[b+1]) of the nonzeros (a segment = one
// problem of a batch): gridDim.y blocks per segment, each leaving one partial,
// part[b * gridDim.y + y].  CISS=true reads mode-0 CISS order, false a COO.
// Bound by the row gathers.  Walkers of R / 4 lanes move a row as one 16-byte
// load per lane, the walkers of a segment's blocks take its nonzeros in turn,
// and the FP32 prediction is summed over the walker's lanes.  A long segment is
// shared by several blocks (eval_seg_blocks): with one block per segment and a
// lane per nonzero, the RMSE of 24 problems of 0.3M nonzeros (six per rank) took
// 24 ms; with 64 blocks per segment its longest kernel, of the six at rank 64, takes
// 0.53 ms.
template <int R, int N, bool CISS>
__global__ void __launch_bounds__(256) k_eval_seg(CissArgs c, CooArgs co, FactorArgs fa, const uint64_t *seg,
                                                  double *part) {
  constexpr int W = SyncShape<R>::W, CPL = SyncShape<R>::CPL, NW = 256 / W;
  const int wl = threadIdx.x % W;
  double acc = 0.0;
  const uint64_t p1 = seg[blockIdx.x + 1];
  const uint64_t G = (uint64_t)gridDim.y * NW;
  for (uint64_t p = seg[blockIdx.x] + (uint64_t)blockIdx.y * NW + threadIdx.x / W; p < p1; p += G) {
    uint32_t ix[N];
    float x;
    if (CISS) {
      const uint64_t t = p >> 6;
      ix[0] = c.directory[tile_lane_slot(c.tile_slot[t], c.tile_mask[t], (int)(p & 63))];
#pragma unroll
      for (int s = 0; s < N - 1; ++s) ix[1 + s] = c.oidx[s][p];
      x = c.vals[p];
    } else {
#pragma unroll
      for (int m = 0; m < N; ++m) ix[m] = co.ind[m][p];
      x = co.vals[p];
    }
    float h[CPL];
    load_row4<CPL>(fa.f[0] + (size_t)ix[0] * R + wl * CPL, h);
#pragma unroll
    for (int m = 1; m < N; ++m) {
      float g[CPL];
      load_row4<CPL>(fa.f[m] + (size_t)ix[m] * R + wl * CPL, g);
#pragma unroll
      for (int j = 0; j < CPL; ++j) h[j] *= g[j];
    }
    const double e = (double)x - (double)group_sum<W>((h[0] + h[1]) + (h[2] + h[3]));
    if (wl == 0) acc += e * e;
  }
  block_store_sum(acc, part + (size_t)blockIdx.x * gridDim.y + blockIdx.y);
}

// blockIdx.y: one of several arrays, n[y] entries
__global__ void __launch_bounds__(256) k_sumsq(FactorArgs x, RowCounts len, double *part) {
  double acc = 0.0;
  const float *f = x.f[blockIdx.y];
  const uint64_t n = len.n[blockIdx.y];
  for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n;
       p += (uint64_t)gridDim.x * blockDim.x) {
    const double v = f[p];
    acc += v * v;
  }
  block_store_sum(acc, part + (size_t)blockIdx.y * gridDim.x + blockIdx.x);
}

// out[0] = sum of first[0 .. nfirst), out[1 + k] = sum of part[k * nb .. k * nb + nb),
// each in a fixed order
__global__ void __launch_bounds__(256) k_reduce_stats(const double *first, uint32_t nfirst, const double *part,
                                                      uint32_t nb, double *out) {
  const double *p = blockIdx.x ? part + (size_t)(blockIdx.x - 1) * nb : first;
  const uint32_t n = blockIdx.x ? nb : nfirst;
  double acc = 0.0;
  for (uint32_t i = threadIdx.x; i < n; i += 256) acc += p[i];
  block_store_sum(acc, out + blockIdx.x);
}

// out[k] = sum of part[k * nb .. k * nb + nb) in a fixed order
__global__ void __launch_bounds__(256) k_reduce_parts(const double *part, uint32_t nb, double *out) {
  const double *p = part + (size_t)blockIdx.x * nb;
  double acc = 0.0;
  for (uint32_t i = threadIdx.x; i < nb; i += 256) acc += p[i];
  block_store_sum(acc, out + blockIdx.x);
}

// ==========================================================================
// elementwise helpers
// ==========================================================================
__global__ void __launch_bounds__(256) k_fill(float *x, uint64_t n, float v) {
  for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n;
       p += (uint64_t)gridDim.x * blockDim.x)
    x[p] = v;
}

// plain streaming copy of n 16-byte words: the bandwidth yardstick and the
// known-size kernel that calibrates HBM traffic counters.  (Four loads in
// flight per lane before the stores measured the same rate, 4.59 TB/s.)
__global__ void __launch_bounds__(256) k_copy(const uint4 *__restrict__ src, uint4 *__restrict__ dst, uint64_t n) {
  for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n;
       p += (uint64_t)gridDim.x * blockDim.x)
    dst[p] = src[p];
}

// The gradient's regulariser, before the adjoint walk adds to it: grad =
// lambda * c_i * F for the rows of a CISS directory (c_i = row nnz) or, when
// per_occ == 0, for every row (c_i = 1); part: its share of the loss.  A
// stream of 16-byte loads and stores: 45 us at 1M rows of R = 32 (20 us of zero
// fill and 156 us of 4-byte updates after the walk, before).
__global__ void __launch_bounds__(256) k_reg_rows(const uint32_t *directory, const uint32_t *rowptr,
                                                  uint64_t nrows, int R, float lam, int per_occ,
                                                  const float *F, float *G, double *part) {
  double acc = 0.0;
  const uint32_t Q = (uint32_t)R / 4;  // 16-byte parts of a row: a power of two
  const uint64_t total = nrows * (uint64_t)Q;
  for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < total;
       p += (uint64_t)gridDim.x * blockDim.x) {
    uint64_t at = p;
    float cnt = 1.f;
    if (per_occ) {
      const uint64_t s = p / Q;
      at = (uint64_t)directory[s] * Q + p % Q;
      cnt = (float)(rowptr[s + 1] - rowptr[s]);
    }
    float a[4], g[4];
    load_row4<4>(F + at * 4, a);
    double q = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      g[j] = lam * cnt * a[j];
      q += (double)a[j] * (double)a[j];
    }
    store_row4<4>(G + at * 4, g);
    acc += 0.5 * (double)lam * (double)cnt * q;
  }
  block_store_sum(acc, part + blockIdx.x);
}

// ==========================================================================
// launchers
// ==========================================================================
#define CTC_R_SWITCH(R, ...)                                        \
  switch (R) {                                                      \
    case 8: { constexpr int RR = 8; __VA_ARGS__; } break;           \
    case 16: { constexpr int RR = 16; __VA_ARGS__; } break;         \
    case 32: { constexpr int RR = 32; __VA_ARGS__; } break;         \
    case 64: { constexpr int RR = 64; __VA_ARGS__; } break;         \
    case 128: { constexpr int RR = 128; __VA_ARGS__; } break;       \
    default: return hipErrorInvalidValue;                           \
  }

static inline unsigned grid_for(uint64_t waves, unsigned block) {
  const uint64_t wpb = block / 64;
  return (unsigned)((waves + wpb - 1) / wpb);
}

// policy code = PA * 64 + PB * 8 + PC
template <int N>
static hipError_t launch_sgd_n(hipStream_t st, const CissArgs &c, const FactorArgs &f, const HotRows &hot, int R,
                               uint32_t span,
                               uint64_t nspans, uint64_t stride, int code, float step, float lam, unsigned grid,
                               unsigned block) {
#define CTC_SGD_P(PA, PB, PC) \
  case PA * 64 + PB * 8 + PC:  \
    CTC_R_SWITCH(R, hipLaunchKernelGGL((k_sgd<RR, N, PA, PB, PC>), dim3(grid), dim3(block), 0, st, c, f, hot, span, nspans, stride, step, lam)); \
    break;
  switch (code) {
    CTC_SGD_P(P_RACY, P_HOT, P_HOT)
    CTC_SGD_P(P_RACY, P_HOTRUN, P_HOTRUN)
    CTC_SGD_P(P_RACY, P_ATOMIC, P_ATOMIC)
    CTC_SGD_P(P_RACY, P_RACY, P_RACY)
    CTC_SGD_P(P_RACY, P_RACY, P_ATOMIC)
    default:
      return hipErrorInvalidValue;
  }
#undef CTC_SGD_P
  return hipGetLastError();
}

hipError_t launch_sgd(hipStream_t st, const CissArgs &c, const FactorArgs &f, const HotRows &hot, int nmodes, int R,
                      uint32_t span, uint64_t stride, int code, float step, float lam, unsigned block) {
  if (c.nnz == 0) return hipSuccess;
  const uint64_t nspans = (c.nnz + span - 1) / span;
  const int W = R < 64 ? R : 64;
  const uint64_t waves = (nspans + (64 / W) - 1) / (64 / W);
  const unsigned grid = grid_for(waves, block);
  if (nmodes == 3) return launch_sgd_n<3>(st, c, f, hot, R, span, nspans, stride, code, step, lam, grid, block);
  if (nmodes == 4) return launch_sgd_n<4>(st, c, f, hot, R, span, nspans, stride, code, step, lam, grid, block);
  return hipErrorInvalidValue;
}

template <int R, int N, bool MIX, int CPL>
static void launch_sync_as(hipStream_t st, const CissArgs &c, const FactorArgs &f, const SyncArgs &sy, uint32_t span,
                           uint32_t sub, uint32_t s, uint64_t nspans, uint32_t long_min, float step, float lam,
                           unsigned block) {
  constexpr uint64_t wpw = WalkShape<R, CPL>::WPW;
  const size_t lds = (block / 64) * SyncMeta<R, N, MIX, CPL>::kWaveBytes;
  hipLaunchKernelGGL((k_sgd_sync<R, N, MIX, CPL>), dim3(grid_for((nspans + wpw - 1) / wpw, block)), dim3(block), lds, st,
                     c, f, sy, span, sub, s, nspans, long_min, step, lam);
}

hipError_t launch_sgd_sync(hipStream_t st, const CissArgs &c, const FactorArgs &f, const SyncArgs &sy, int nmodes,
                           int R, uint32_t span, uint32_t sub, uint32_t s, uint32_t long_min, float step, float lam,
                           unsigned block, bool mixed) {
  if (c.nnz == 0) return hipSuccess;
  if (nmodes != 3 && nmodes != 4) return hipErrorInvalidValue;
  const uint64_t nspans = (c.nnz + span - 1) / span;
  // Two elements per lane while four would leave a SIMD with less than two
  // waves (R = 32: 12.5M nonzeros 3113 us an epoch against 3230, 50M nonzeros 6104
  // against 5957; R = 16, 20K nonzeros 1424 against 1628).  From R = 64 on the sum
  // over a walker of more than 16 lanes would cost more.  Mixed: always four,
  // the order of that sum decides how the staged deltas round.
  constexpr uint64_t kTwoPerSimd = 2048;
  const bool two = R <= 32 && nspans / (256 / (uint64_t)R) < kTwoPerSimd;
#define CTC_SYNC(NN)                                                                                             \
  CTC_R_SWITCH(R, constexpr int kFew = RR <= 32 ? 2 : 4;                                                         \
               (mixed ? launch_sync_as<RR, NN, true, 4> : two ? launch_sync_as<RR, NN, false, kFew>              \
                                                              : launch_sync_as<RR, NN, false, 4>)(               \
                   st, c, f, sy, span, sub, s, nspans, long_min, step, lam, block))
  if (nmodes == 3) {
    CTC_SYNC(3);
  } else {
    CTC_SYNC(4);
  }
#undef CTC_SYNC
  return hipGetLastError();
}

hipError_t launch_sgd_settle(hipStream_t st, SettleArgs a, int R, bool mixed) {
  const int W = R < 64 ? R : 64;
  const uint64_t items = a.mg.off[a.mg.nseg];
  const uint64_t nw = 1024 / (uint64_t)R;  // light rows per block: 256 / (R / 4) walkers
  a.nb_light = (a.lb[4] + nw - 1) / nw;
  const uint64_t sb = a.pb[4] + a.nb_light + grid_for((items + (64 / W) - 1) / (64 / W), 256);
  if (sb > 0x7FFFFFFFull) return hipErrorInvalidValue;
  if (sb > 0) {
    if (mixed) {
      CTC_R_SWITCH(R, hipLaunchKernelGGL((k_sgd_settle<RR, true>), dim3((unsigned)sb), dim3(256), 0, st, a));
    } else {
      CTC_R_SWITCH(R, hipLaunchKernelGGL((k_sgd_settle<RR, false>), dim3((unsigned)sb), dim3(256), 0, st, a));
    }
  }
  const uint64_t fg = grid_for((a.fb[4] + (64 / W) - 1) / (64 / W), 256);
  if (fg > 0) CTC_R_SWITCH(R, hipLaunchKernelGGL((k_sgd_fold<RR>), dim3((unsigned)fg), dim3(256), 0, st, a));
  return hipGetLastError();
}

hipError_t launch_mttkrp(hipStream_t st, const CissArgs &c, const FactorArgs &f, int nmodes, int R,
                         uint32_t span, bool adjoint, float *out, double *loss_part,
                         unsigned *grid_out, unsigned block, float lam, int per_occ) {
  const unsigned grid = (unsigned)mttkrp_grid(c.nnz, R, span, block);
  *grid_out = grid;
  if (c.nnz == 0) return hipSuccess;
  float *none = nullptr;
  if (nmodes == 3) {
    if (adjoint) {
      CTC_R_SWITCH(R, hipLaunchKernelGGL((k_mttkrp<RR, 3, kWalkAdjoint>), dim3(grid), dim3(block), 0, st, c, f, span, out, loss_part, none, lam, per_occ));
    } else {
      CTC_R_SWITCH(R, hipLaunchKernelGGL((k_mttkrp<RR, 3, kWalkMttkrp>), dim3(grid), dim3(block), 0, st, c, f, span, out, loss_part, none, lam, per_occ));
    }
  } else if (nmodes == 4) {
    if (adjoint) {
      CTC_R_SWITCH(R, hipLaunchKernelGGL((k_mttkrp<RR, 4, kWalkAdjoint>), dim3(grid), dim3(block), 0, st, c, f, span, out, loss_part, none, lam, per_occ));
    } else {
      CTC_R_SWITCH(R, hipLaunchKernelGGL((k_mttkrp<RR, 4, kWalkMttkrp>), dim3(grid), dim3(block), 0, st, c, f, span, out, loss_part, none, lam, per_occ));
    }
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_ccd_jacobi(hipStream_t st, const CissArgs &c, const FactorArgs &f, int nmodes, int R,
                             uint32_t span, float *num, float *den, unsigned block) {
  if (c.nnz == 0) return hipSuccess;
  const unsigned grid = (unsigned)mttkrp_grid(c.nnz, R, span, block);
  double *none = nullptr;
  if (nmodes == 3) {
    CTC_R_SWITCH(R, hipLaunchKernelGGL((k_mttkrp<RR, 3, kWalkJacobi>), dim3(grid), dim3(block), 0, st, c, f, span, num, none, den, 0.f, 0));
  } else if (nmodes == 4) {
    CTC_R_SWITCH(R, hipLaunchKernelGGL((k_mttkrp<RR, 4, kWalkJacobi>), dim3(grid), dim3(block), 0, st, c, f, span, num, none, den, 0.f, 0));
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_loss_walk(hipStream_t st, const CissArgs &c, const FactorArgs &f, int nmodes, int R,
                            uint32_t span, double *part, unsigned block) {
  if (c.nnz == 0) return hipSuccess;
  const unsigned grid = (unsigned)mttkrp_grid(c.nnz, R, span, block);
  float *none = nullptr;
  if (nmodes == 3) {
    CTC_R_SWITCH(R, hipLaunchKernelGGL((k_mttkrp<RR, 3, kWalkLoss>), dim3(grid), dim3(block), 0, st, c, f, span, none, part, none, 0.f, 0));
  } else if (nmodes == 4) {
    CTC_R_SWITCH(R, hipLaunchKernelGGL((k_mttkrp<RR, 4, kWalkLoss>), dim3(grid), dim3(block), 0, st, c, f, span, none, part, none, 0.f, 0));
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

uint64_t mttkrp_walkers_per_block(int R, unsigned block) { return (uint64_t)(block / 64) * (64 / (R / 4)); }

// Spans of 256 where they fill the chip, down to 32 for smaller tensors: about 4096
// waves (the loss of 1M nonzeros at R = 16: 14 us, 89 us with 256).  A span between
// two powers of two costs: MTTKRP of 8M nonzeros at R = 32 132 us with the 224 it
// gets, 117 / 124 / 123 / 133 us with 256 / 128 / 64 / 32, the adjoint of 4M
// nonzeros 92 us with 96, 79 us with 64.  Rounding down to the power of two would take
// that back but leaves more partial sums of a hot row to the FP32 atomics: at one
// size the error of the sums against 64 bits grew from 9e-8 to 1.2e-7 of their norm.
uint32_t walk_span(uint64_t nnz, int R) {
  const uint64_t per = nnz / (4096 * (uint64_t)(256 / R)) / 32 * 32;
  return (uint32_t)(per < 32 ? 32 : per > 256 ? 256 : per);
}

uint64_t mttkrp_grid(uint64_t nnz, int R, uint32_t span, unsigned block) {
  const uint64_t walkers = (nnz + span - 1) / span;
  const uint64_t wpw = 64 / (R / 4);  // walkers per wave (SyncShape<R>)
  const uint64_t waves = (walkers + wpw - 1) / wpw;
  return grid_for(waves, block);
}

hipError_t launch_als_gram(hipStream_t st, const CissArgs &c, const FactorArgs &f, int nmodes, int R,
                           uint32_t span_tiles, uint64_t nspans, const uint32_t *span_off, const uint64_t *tile_thin,
                           double *pieces, unsigned block) {
  if (c.nnz == 0) return hipSuccess;
  const unsigned grid = grid_for(nspans, block);
#define CTC_GRAM(RR)                                                                                     \
  do {                                                                                                    \
    if (nmodes == 3)                                                                                      \
      hipLaunchKernelGGL((k_als_gram<RR, 3>), dim3(grid), dim3(block), 0, st, c, f, span_tiles, nspans, \
                         span_off, tile_thin, pieces);                                                    \
    else                                                                                                  \
      hipLaunchKernelGGL((k_als_gram<RR, 4>), dim3(grid), dim3(block), 0, st, c, f, span_tiles, nspans, \
                         span_off, tile_thin, pieces);                                                    \
  } while (0)
  switch (R) {
    case 8: CTC_GRAM(8); break;
    case 16: CTC_GRAM(16); break;
    case 32:
      if (nmodes == 3)
        CTC_GRAM(32);
      else  // four modes need more than the 80 registers of 6 waves per SIMD (it would spill)
        hipLaunchKernelGGL((k_als_gram_wide<32, 4>), dim3(grid), dim3(block), 0, st, c, f, span_tiles, nspans,
                           span_off, tile_thin, pieces);
      break;
    case 64:
      if (nmodes == 3)
        hipLaunchKernelGGL((k_als_gram_wide<64, 3>), dim3(grid), dim3(block), 0, st, c, f, span_tiles, nspans,
                           span_off, tile_thin, pieces);
      else
        hipLaunchKernelGGL((k_als_gram_wide<64, 4>), dim3(grid), dim3(block), 0, st, c, f, span_tiles, nspans,
                           span_off, tile_thin, pieces);
      break;
    default: return hipErrorInvalidValue;
  }
#undef CTC_GRAM
  return hipGetLastError();
}

hipError_t launch_piece_reduce(hipStream_t st, const double *pieces, const uint32_t *grp_piece,
                               const uint32_t *grp_n, uint64_t ngroups, int R, double *gsum) {
  if (ngroups == 0) return hipSuccess;
#define CTC_REDUCE(RR)                                                                                               \
  case RR:                                                                                                           \
    hipLaunchKernelGGL((k_piece_reduce<RR>), dim3((unsigned)ngroups, (RR * RR + RR + 255) / 256), dim3(256), 0, st, \
                       pieces, grp_piece, grp_n, gsum);                                                              \
    break
  switch (R) {
    CTC_REDUCE(8);
    CTC_REDUCE(16);
    CTC_REDUCE(32);
    CTC_REDUCE(64);
    default: return hipErrorInvalidValue;
  }
#undef CTC_REDUCE
  return hipGetLastError();
}

hipError_t launch_als_solve(hipStream_t st, const double *pieces, const uint32_t *slot_pb, const double *gsum,
                            const uint32_t *slot_gb, const uint32_t *directory, const uint32_t *list, uint64_t count,
                            int R, double lam, bool refine, float *A, uint32_t *flag) {
  if (count == 0) return hipSuccess;
  if (list && (refine || R > 32)) return hipErrorInvalidValue;
  const uint64_t dlength = count;
  const unsigned grid = (unsigned)dlength;
  if (!refine && R <= 32) {
    const unsigned g8 = (unsigned)((dlength + 7) / 8);
    switch (R) {
      case 8: hipLaunchKernelGGL((k_als_solve_h<8>), dim3(g8), dim3(256), 0, st, pieces, slot_pb, gsum, slot_gb, directory, list, count, lam, A, flag); break;
      case 16: hipLaunchKernelGGL((k_als_solve_h<16>), dim3(g8), dim3(256), 0, st, pieces, slot_pb, gsum, slot_gb, directory, list, count, lam, A, flag); break;
      case 32: hipLaunchKernelGGL((k_als_solve_h<32>), dim3(g8), dim3(256), 0, st, pieces, slot_pb, gsum, slot_gb, directory, list, count, lam, A, flag); break;
      default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
  }
#define CTC_SOLVE(RR)                                                                                      \
  do {                                                                                                      \
    if (refine)                                                                                             \
      hipLaunchKernelGGL((k_als_solve<RR, true>), dim3(grid), dim3(64), 0, st, pieces, slot_pb, gsum,      \
                         slot_gb, directory, dlength, lam, A, flag);                                        \
    else                                                                                                    \
      hipLaunchKernelGGL((k_als_solve<RR, false>), dim3(grid), dim3(64), 0, st, pieces, slot_pb, gsum,     \
                         slot_gb, directory, dlength, lam, A, flag);                                        \
  } while (0)
  switch (R) {  // without refinement only rank 64 comes here
    case 8: hipLaunchKernelGGL((k_als_solve<8, true>), dim3(grid), dim3(64), 0, st, pieces, slot_pb, gsum, slot_gb, directory, dlength, lam, A, flag); break;
    case 16: hipLaunchKernelGGL((k_als_solve<16, true>), dim3(grid), dim3(64), 0, st, pieces, slot_pb, gsum, slot_gb, directory, dlength, lam, A, flag); break;
    case 32: hipLaunchKernelGGL((k_als_solve<32, true>), dim3(grid), dim3(64), 0, st, pieces, slot_pb, gsum, slot_gb, directory, dlength, lam, A, flag); break;
    case 64: CTC_SOLVE(64); break;
    default: return hipErrorInvalidValue;
  }
#undef CTC_SOLVE
  return hipGetLastError();
}

hipError_t launch_eval_coo(hipStream_t st, const CooArgs &c, const FactorArgs &f, int nmodes, int R,
                           unsigned nblocks, double *part) {
  if (nmodes == 3)
    hipLaunchKernelGGL((k_eval_coo<3>), dim3(nblocks), dim3(256), 0, st, c, f, R, part);
  else if (nmodes == 4)
    hipLaunchKernelGGL((k_eval_coo<4>), dim3(nblocks), dim3(256), 0, st, c, f, R, part);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

// Blocks that share a segment: eight nonzeros for each walker of the longest
// segment's blocks, and no more than 8192 blocks for all segments, 32 a CU, since a
// block costs more than a short segment's nonzeros.  RMSE of a batch of 2000 problems
// of 300 nonzeros 127 us, 400 of 4000 137 us, 4 of 5000 115 us; with 64 blocks for
// every segment 243 / 154 / 124 us, with one 145 / 281 / 272 us; 4, 16 and 32 nonzeros
// a walker differ by up to 2, 7 and 25 percent.
unsigned eval_seg_blocks(int R, uint32_t nseg, uint64_t longest) {
  const uint64_t share = 8 * 1024 / (uint64_t)R;  // a block has 256 / (R / 4) walkers
  const uint64_t most = std::min<uint64_t>(kSegBlocks, std::max<uint64_t>(1, 8192 / nseg));
  return (unsigned)std::min(most, std::max<uint64_t>(1, (longest + share - 1) / share));
}

hipError_t launch_eval_seg(hipStream_t st, const CissArgs *c, const CooArgs *co, const FactorArgs &f,
                           int nmodes, int R, const uint64_t *seg, uint32_t nseg, unsigned blocks, double *part) {
  if (nseg == 0) return hipSuccess;
  const CissArgs ca = c ? *c : CissArgs{};
  const CooArgs cb = co ? *co : CooArgs{};
#define CTC_SEG(NN)                                                                                                  \
  do {                                                                                                               \
    if (c) {                                                                                                         \
      CTC_R_SWITCH(R, hipLaunchKernelGGL((k_eval_seg<RR, NN, true>), dim3(nseg, blocks), dim3(256), 0, st, ca, cb, \
                                         f, seg, part));                                                             \
    } else {                                                                                                         \
      CTC_R_SWITCH(R, hipLaunchKernelGGL((k_eval_seg<RR, NN, false>), dim3(nseg, blocks), dim3(256), 0, st, ca, cb, \
                                         f, seg, part));                                                             \
    }                                                                                                                \
  } while (0)
  if (nmodes == 3)
    CTC_SEG(3);
  else if (nmodes == 4)
    CTC_SEG(4);
  else
    return hipErrorInvalidValue;
#undef CTC_SEG
  return hipGetLastError();
}

hipError_t launch_sumsq(hipStream_t st, const FactorArgs &x, const RowCounts &len, int count, unsigned nblocks,
                        double *part) {
  hipLaunchKernelGGL(k_sumsq, dim3(nblocks, (unsigned)count), dim3(256), 0, st, x, len, part);
  return hipGetLastError();
}

hipError_t launch_reduce_stats(hipStream_t st, const double *first, uint32_t nfirst, const double *part, uint32_t nb,
                               uint32_t groups, double *out) {
  hipLaunchKernelGGL(k_reduce_stats, dim3(1 + groups), dim3(256), 0, st, first, nfirst, part, nb, out);
  return hipGetLastError();
}

hipError_t launch_reduce_parts(hipStream_t st, const double *part, uint32_t nb, uint32_t groups,
                               double *out) {
  hipLaunchKernelGGL(k_reduce_parts, dim3(groups), dim3(256), 0, st, part, nb, out);
  return hipGetLastError();
}

hipError_t launch_fill(hipStream_t st, float *x, uint64_t n, float v) {
  if (n == 0) return hipSuccess;
  uint64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_fill, dim3((unsigned)blocks), dim3(256), 0, st, x, n, v);
  return hipGetLastError();
}

hipError_t launch_copy(hipStream_t st, const void *src, void *dst, uint64_t bytes) {
  const uint64_t n = bytes / 16;
  if (n == 0) return hipSuccess;
  uint64_t blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(k_copy, dim3((unsigned)blocks), dim3(256), 0, st, (const uint4 *)src, (uint4 *)dst, n);
  return hipGetLastError();
}

hipError_t launch_reg_rows(hipStream_t st, const uint32_t *directory, const uint32_t *rowptr,
                           uint64_t nrows, int R, float lam, int per_occ, const float *F, float *G,
                           unsigned nblocks, double *part) {
  hipLaunchKernelGGL(k_reg_rows, dim3(nblocks), dim3(256), 0, st, directory, rowptr, nrows, R, lam,
                     per_occ, F, G, part);
  return hipGetLastError();
}

}  // namespace ctc
