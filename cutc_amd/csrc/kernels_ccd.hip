// kernels_ccd.hip — CCD++ column kernels for gfx950 (canonical CCD++ as the
// reference states it in comments, SG/ccd.cu:532-554 and NC/ccd.cu:28-180:
// for each column f, add the rank-one component back to the residual, update
// column f of every mode as a 1-D ridge solve a_if = sum(r h) / (lambda +
// sum h^2), then subtract the new component).
//
// Layout.  Every mode's CISS carries its own copy of the residual in its own
// nonzero order, so each column pass streams it coalesced.  The factors are
// mirrored column-major (R x dims) during an epoch.  A copy stores "x minus
// every component except column `pending`"; the pass of column f over mode m
// first completes the previous column (subtracting its new component), then
// adds column f back with its pre-update values (saved before the column's
// first mode update), and sums num/den.  The three values a pass needs of a
// row (pending column's new value, column f saved, column f current) sit in
// one 16-byte record per row, built at the start of each column: a nonzero
// costs one gather per mode instead of three.  Divergent gathers are what
// the pass is limited by (the texture addresser is the busy unit), so the
// number of gather instructions, not their width, sets its time.
//
// Reductions.  One wave walks a span of tiles, one lane per nonzero.  Row
// sums inside a tile use a segmented inclusive scan that takes each lane's
// distance to its row's start from the tile mask; the row still open at the end
// of a tile is carried in a wave-uniform value into the next tile.  Completed
// rows are written as (num, den) pieces with the same piece numbering as the ALS
// Gram pieces, so the per-row sums have a fixed order (deterministic, no atomics).
//
// The three passes of a column over 20M nonzeros (480K x 18K x 2K): 137 / 173 /
// 196 us (169 / 182 / 219 us with the whole scan on the LDS pipe and no tile in
// flight); the 16 bytes per nonzero that a pass streams take 68 us.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels_ccd.h"
#include "kernels_common.h"

namespace ctc {

// x of lane - D (what lanes below D get is not used): whole-wave DPP shifts by
// one for 1 and 2, a swap of the wave's halves for 32, else a shuffle
template <int D>
__device__ inline float lane_before(float x) {
  int v = __float_as_int(x);
  if constexpr (D <= 2) {
#pragma unroll
    for (int i = 0; i < D; ++i) v = __builtin_amdgcn_update_dpp(0, v, 0x138, 0xF, 0xF, false);
  } else if constexpr (D == 32) {
    v = (int)__builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false)[0];
  } else {
    return __shfl_up(x, D, 64);
  }
  return __int_as_float(v);
}

template <int D>
__device__ inline void scan_step(float &a, float &b, int dist) {
  const float ua = lane_before<D>(a), ub = lane_before<D>(b);
  a += dist >= D ? ua : 0.f;
  b += dist >= D ? ub : 0.f;
}

// Inclusive segmented scan over the wave; dist = lanes from the start of the
// lane's segment to it, so no flag is carried along (18 shuffles on the LDS pipe
// per tile before, 6 now; with 12 an epoch of 20M nonzeros took 18.05 ms, now 17.45).
// The order of the sums is kept: a row of few nonzeros can turn a rounding of its
// sums into a thousand times that in its value.
__device__ inline void seg_scan(float &a, float &b, int dist) {
  scan_step<1>(a, b, dist);
  scan_step<2>(a, b, dist);
  scan_step<4>(a, b, dist);
  scan_step<8>(a, b, dist);
  scan_step<16>(a, b, dist);
  scan_step<32>(a, b, dist);
}

__device__ inline float lane_value(float x, uint32_t lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), (int)lane));
}

// The pass of wave w (uniform) over its span.  LS >= 0: the records of other
// mode LS (a mode of at most kCcdLdsRows rows) are read from the workgroup's
// copy xs in LDS instead of gathered from memory.  The indices and the
// residual of tile t + 2 and the records of tile t + 1 are in flight while
// tile t is summed.
template <int N, int LS>
__device__ __forceinline__ void ccd_col_wave(const CcdColArgs &a, uint64_t w, const float4 *xs) {
  const int lane = lane_id();
  const CissArgs &c = a.c;
  const uint64_t t0 = w * a.span_tiles;
  const uint64_t t1 = t0 + a.span_tiles < c.ntiles ? t0 + a.span_tiles : c.ntiles;
  const uint32_t poff = a.span_off[w];
  const bool fix = a.sub_col >= 0 || a.add_back;  // this pass rewrites the residual
  double carry_n = 0.0, carry_d = 0.0;
  uint32_t carry_slot = 0;
  bool have_carry = false;
  double2 *pieces = reinterpret_cast<double2 *>(a.pieces);

  uint32_t ix[N - 1], row = 0;  // of the tile after the next
  float en;
  auto indices = [&](uint64_t t) {
    t = t < t1 ? t : t1 - 1;  // past the span: its last tile again, not used
    const uint64_t at = t * kTile + lane, p = at < c.nnz ? at : c.nnz - 1;
#pragma unroll
    for (int s = 0; s < N - 1; ++s) ix[s] = c.oidx[s][p];
    en = a.resid[p];
    // lanes past the end take a valid row's slot too
    if (fix) row = c.directory[tile_lane_slot(c.tile_slot[t], c.tile_mask[t], (int)(p & 63))];
  };
  float4 qn[N];
  float e1;
  uint32_t ln = 0;  // the record in LDS is read when its tile is summed
  auto records = [&]() {
#pragma unroll
    for (int s = 0; s < N - 1; ++s)
      if (s == LS)
        ln = ix[s];
      else
        qn[1 + s] = a.x[1 + s][ix[s]];
    if (fix) qn[0] = a.x[0][row];  // the own mode's row: pending and saved values
    e1 = en;
  };
  indices(t0);
  records();
  indices(t0 + 1);
  for (uint64_t t = t0; t < t1; ++t) {
    float4 q[N];
#pragma unroll
    for (int s = 0; s < N; ++s) q[s] = s == 1 + LS && LS >= 0 ? xs[ln] : qn[s];
    float e = e1;
    records();
    indices(t + 2);
    const uint64_t base = t * kTile;
    const uint32_t cnt = (uint32_t)((c.nnz - base) < (uint64_t)kTile ? (c.nnz - base) : kTile);
    uint64_t mask = c.tile_mask[t];
    if (cnt < 64) mask &= (1ull << cnt) - 1ull;
    const uint32_t first_slot = c.tile_slot[t];
    const bool valid = (uint32_t)lane < cnt;
    if (fix) {
      if (a.sub_col >= 0) {
        float v = q[0].x;
#pragma unroll
        for (int s = 1; s < N; ++s) v *= q[s].x;
        e -= v;
      }
      if (a.add_back) {
        float v = q[0].y;
#pragma unroll
        for (int s = 1; s < N; ++s) v *= q[s].y;
        e += v;
      }
      if (valid) a.resid[base + lane] = e;
    }
    float h = q[1].z;
#pragma unroll
    for (int s = 2; s < N; ++s) h *= q[s].z;
    float num = valid ? e * h : 0.f, den = valid ? h * h : 0.f;
    const uint64_t upto = (mask | 1ull) & (lane == 63 ? ~0ull : (2ull << lane) - 1ull);
    seg_scan(num, den, lane - (63 - __clzll((long long)upto)));

    // first segment: lanes [0, fh); fh = first row start after lane 0
    const uint64_t later = mask & ~1ull;
    const uint32_t fh = later ? (uint32_t)__ffsll((unsigned long long)later) - 1u : cnt;
    const bool join = (t > t0) && !(mask & 1ull);  // lane 0 continues the carried row
    if (have_carry && !join) {
      if (lane == 0) pieces[carry_slot + poff] = make_double2(carry_n, carry_d);
      have_carry = false;
      carry_n = carry_d = 0.0;
    }
    const double fn = (double)lane_value(num, fh - 1) + (join ? carry_n : 0.0);
    const double fd = (double)lane_value(den, fh - 1) + (join ? carry_d : 0.0);
    if (fh < cnt) {
      if (lane == 0) pieces[first_slot + poff] = make_double2(fn, fd);
      // complete middle segments end at lanes i in [fh, cnt-1) whose next lane
      // starts a row; the last segment (ending at cnt-1) becomes the carry
      const bool tail = (uint32_t)lane >= fh && (uint32_t)lane + 1 < cnt && ((mask >> (lane + 1)) & 1ull);
      if (tail) pieces[tile_lane_slot(first_slot, mask, lane) + poff] = make_double2((double)num, (double)den);
      carry_n = (double)lane_value(num, cnt - 1);
      carry_d = (double)lane_value(den, cnt - 1);
      carry_slot = tile_lane_slot(first_slot, mask, (int)cnt - 1);
    } else {
      carry_n = fn;
      carry_d = fd;
      carry_slot = first_slot;
    }
    have_carry = true;
  }
  if (have_carry && lane == 0) pieces[carry_slot + poff] = make_double2(carry_n, carry_d);
}

// the wave's span, as the uniform value it is: the tile words are scalar loads
__device__ inline uint64_t wave_index() {
  return (uint64_t)blockIdx.x * (blockDim.x >> 6) + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

template <int N>
__global__ void __launch_bounds__(256) k_ccd_col(CcdColArgs a) {
  const uint64_t w = wave_index();
  if (w >= a.nspans) return;
  ccd_col_wave<N, -1>(a, w, nullptr);
}

// 1024-thread workgroups (16 spans) sharing one LDS copy of the records of a
// small other mode: its gathers no longer go through the texture addresser.
template <int N, int LS>
__global__ void __launch_bounds__(1024, 8) k_ccd_col_lds(CcdColArgs a) {
  __shared__ float4 xs[kCcdLdsRows];
  const float4 *src = a.x[1 + LS];
  for (uint32_t i = threadIdx.x; i < a.lds_rows; i += blockDim.x) xs[i] = src[i];
  __syncthreads();
  const uint64_t w = wave_index();
  if (w >= a.nspans) return;
  ccd_col_wave<N, LS>(a, w, xs);
}

// a_f(row) = num / (lambda + den) per directory slot (SG/ccd.cu:345 form),
// written to the factor mirror and to the row's record (the current value
// later modes' passes gather).  Each slot's pieces are summed in a fixed order
// (deterministic).
__device__ inline void ccd_finish_slot(uint64_t slot, double n, double d, const uint32_t *directory, double lam,
                                       float *col, float4 *x) {
  const uint32_t row = directory[slot];
  const float v = (float)(n / (lam + d));
  col[row] = v;
  x[row].z = v;
}

// one wave per slot: lane l sums pieces l, l + 64, ... into four partial sums
// (piece l + 64 i into partial i mod 4, so four loads are in flight), adds
// them in order, and a fixed shuffle tree adds the lanes (parallel over the
// thousands of pieces of a long row)
__device__ inline void ccd_finish_wave(uint64_t slot, const double *pieces, const uint32_t *slot_pb,
                                       const uint32_t *directory, double lam, float *col, float4 *x) {
  const int lane = lane_id();
  const double2 *pc = reinterpret_cast<const double2 *>(pieces);
  const uint32_t p1 = slot_pb[slot + 1];
  double n4[4] = {0.0, 0.0, 0.0, 0.0}, d4[4] = {0.0, 0.0, 0.0, 0.0};
  uint32_t p = slot_pb[slot] + lane;
  for (; p + 3 * 64 < p1; p += 4 * 64) {
    double2 q[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) q[u] = pc[p + u * 64];
#pragma unroll
    for (int u = 0; u < 4; ++u) n4[u] += q[u].x, d4[u] += q[u].y;
  }
  for (int u = 0; p < p1; p += 64, ++u) n4[u] += pc[p].x, d4[u] += pc[p].y;
  double n = (n4[0] + n4[1]) + (n4[2] + n4[3]), d = (d4[0] + d4[1]) + (d4[2] + d4[3]);
  for (int o = 32; o > 0; o >>= 1) {
    n += __shfl_xor(n, o, 64);
    d += __shfl_xor(d, o, 64);
  }
  if (lane == 0) ccd_finish_slot(slot, n, d, directory, lam, col, x);
}

// Blocks 0 .. hb - 1 take the slots of more than kHeavyPieces pieces (listed by
// the host), a wave each as above; the blocks after them 256 consecutive slots
// each, a lane per slot, whose few pieces are added in piece order.  The slots,
// their rows and their records are consecutive, so the kernel is a stream; with
// the slots dealt to the blocks in a stride, which kept the long rows (the
// hottest are numbered first) apart, 480K slots took 25 us; the three modes of
// that tensor now take 5.5 us on average.
__global__ void __launch_bounds__(256) k_ccd_finish(const double *pieces, const uint32_t *slot_pb,
                                                    const uint32_t *heavy, uint64_t nheavy, uint32_t hb,
                                                    const uint32_t *directory, uint64_t dlength, double lam,
                                                    float *col, float4 *x) {
  if (blockIdx.x < hb) {
    const uint64_t h = (uint64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (h < nheavy) ccd_finish_wave(heavy[h], pieces, slot_pb, directory, lam, col, x);
    return;
  }
  const uint64_t s = (uint64_t)(blockIdx.x - hb) * 256 + threadIdx.x;
  if (s >= dlength) return;
  const uint32_t p0 = slot_pb[s], p1 = slot_pb[s + 1];
  if (p1 - p0 > kHeavyPieces) return;
  double n = 0.0, d = 0.0;
  for (uint32_t p = p0; p < p1; ++p) {
    const double2 q = reinterpret_cast<const double2 *>(pieces)[p];
    n += q.x;
    d += q.y;
  }
  ccd_finish_slot(s, n, d, directory, lam, col, x);
}

// per-row records of every mode at the start of a column's update; the column's
// mirror is cleared for the rows without nonzeros, the finish writes the others
__global__ void __launch_bounds__(256) k_ccd_pack(CcdPackArgs a) {
  const uint64_t n = a.off[4];
  for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (uint64_t)gridDim.x * blockDim.x) {
    int m = 0;
    while (m < 3 && p >= a.off[m + 1]) ++m;
    const uint64_t i = p - a.off[m], rows = a.off[m + 1] - a.off[m];
    float *cur = a.ft[m] + (size_t)a.col * rows + i;
    const float v = *cur;
    a.x[m][i] = make_float4(a.sub_col >= 0 ? a.ft[m][(size_t)a.sub_col * rows + i] : 0.f, v, v, 0.f);
    *cur = 0.f;
  }
}

// residual copy of a mode: r = x - <rows>, row-major factors in CISS-relative
// order, the products and their sum in FP64 (the residual is updated from
// here on for a whole solve).  Walkers of R / 4 lanes with 4 entries of a row
// per lane (one 16-byte load per row), walker g of G taking nonzeros g, g + G,
// ...  (One lane per nonzero with R scalar loads per row took 15.1 ms per mode
// on the 100M-nonzero tensor; this shape 3.9 ms; four nonzeros per walker at a
// time 5.4 ms.)
template <int R, int N>
__global__ void __launch_bounds__(256) k_ccd_resid(CissArgs c, FactorArgs fa, float *resid) {
  constexpr int CPL = 4, W = R / CPL, WPW = 64 / W;
  const int lane = lane_id();
  const int sub = lane / W, wl = lane % W;
  const uint64_t G = (uint64_t)gridDim.x * (blockDim.x >> 6) * WPW;
  const uint64_t g = ((uint64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * WPW + sub;
  for (uint64_t p = g; p < c.nnz; p += G) {  // uniform over the walker's lanes
    const uint64_t t = p >> 6;
    const uint32_t slot = tile_lane_slot(c.tile_slot[t], c.tile_mask[t], (int)(p & 63));
    const float4 a = *reinterpret_cast<const float4 *>(fa.f[0] + (size_t)c.directory[slot] * R + wl * CPL);
    double v[CPL] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int s = 0; s < N - 1; ++s) {
      const float4 o = *reinterpret_cast<const float4 *>(fa.f[1 + s] + (size_t)c.oidx[s][p] * R + wl * CPL);
      v[0] *= o.x, v[1] *= o.y, v[2] *= o.z, v[3] *= o.w;
    }
    double pr = (v[0] + v[1]) + (v[2] + v[3]);
#pragma unroll
    for (int o = 1; o < W; o <<= 1) pr += __shfl_xor(pr, o, 64);  // within the walker's lanes
    if (wl == 0) resid[p] = (float)((double)c.vals[p] - pr);
  }
}

// The reference's CCD update of a mode (SG/ccd.cu:318-348): every column of
// each directory row from the sums of the Jacobi walk, in place; rows outside
// the directory keep their values.
__global__ void __launch_bounds__(256) k_ccd_jacobi_rows(const uint32_t *directory, uint64_t dlength, int R,
                                                         const float *num, const float *den, double lam, float *F) {
  const uint64_t n = dlength * (uint64_t)R;
  for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n;
       p += (uint64_t)gridDim.x * blockDim.x) {
    const size_t e = (size_t)directory[p / R] * R + p % R;
    F[e] = (float)((double)num[e] / (lam + (double)den[e]));
  }
}

// out (R x rows, column-major) <-> in (rows x R, row-major)
__global__ void __launch_bounds__(256) k_transpose(const float *in, float *out, uint64_t rows, int R,
                                                   int to_colmajor) {
  const uint64_t n = rows * (uint64_t)R;
  for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n;
       p += (uint64_t)gridDim.x * blockDim.x) {
    if (to_colmajor) {
      const uint64_t f = p / rows, i = p % rows;  // write-coalesced
      out[p] = in[i * R + f];
    } else {
      const uint64_t i = p / R, f = p % R;
      out[p] = in[f * rows + i];
    }
  }
}

hipError_t launch_ccd_col(hipStream_t st, const CcdColArgs &a, int nmodes, unsigned block) {
  if (a.c.nnz == 0) return hipSuccess;
  if (a.lds_s >= 0 && a.lds_rows <= kCcdLdsRows) {
    const unsigned g = (unsigned)((a.nspans + 15) / 16);
    if (nmodes == 3 && a.lds_s == 0)
      hipLaunchKernelGGL((k_ccd_col_lds<3, 0>), dim3(g), dim3(1024), 0, st, a);
    else if (nmodes == 3 && a.lds_s == 1)
      hipLaunchKernelGGL((k_ccd_col_lds<3, 1>), dim3(g), dim3(1024), 0, st, a);
    else
      return hipErrorInvalidValue;
    return hipGetLastError();
  }
  const uint64_t wpb = block / 64;
  const unsigned grid = (unsigned)((a.nspans + wpb - 1) / wpb);
  if (nmodes == 3)
    hipLaunchKernelGGL((k_ccd_col<3>), dim3(grid), dim3(block), 0, st, a);
  else if (nmodes == 4)
    hipLaunchKernelGGL((k_ccd_col<4>), dim3(grid), dim3(block), 0, st, a);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_ccd_finish(hipStream_t st, const double *pieces, const uint32_t *slot_pb, const uint32_t *heavy,
                             uint64_t nheavy, const uint32_t *directory, uint64_t dlength, double lam, float *col,
                             float4 *x) {
  if (dlength == 0) return hipSuccess;
  const uint32_t hb = (uint32_t)((nheavy + 3) / 4);
  hipLaunchKernelGGL(k_ccd_finish, dim3(hb + (unsigned)((dlength + 255) / 256)), dim3(256), 0, st, pieces, slot_pb,
                     heavy, nheavy, hb, directory, dlength, lam, col, x);
  return hipGetLastError();
}

hipError_t launch_ccd_pack(hipStream_t st, const CcdPackArgs &a) {
  if (a.off[4] == 0) return hipSuccess;
  uint64_t blocks = (a.off[4] + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_ccd_pack, dim3((unsigned)blocks), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_ccd_resid(hipStream_t st, const CissArgs &c, const FactorArgs &f, int nmodes, int R,
                            float *resid) {
  if (c.nnz == 0) return hipSuccess;
  const unsigned blocks = 4096;  // 4 waves each: 16 per CU
  switch (R * 8 + nmodes) {
#define CTC_RESID(RR, NN) \
  case RR * 8 + NN: hipLaunchKernelGGL((k_ccd_resid<RR, NN>), dim3(blocks), dim3(256), 0, st, c, f, resid); break;
    CTC_RESID(8, 3) CTC_RESID(16, 3) CTC_RESID(32, 3) CTC_RESID(64, 3) CTC_RESID(128, 3)
    CTC_RESID(8, 4) CTC_RESID(16, 4) CTC_RESID(32, 4) CTC_RESID(64, 4) CTC_RESID(128, 4)
#undef CTC_RESID
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_ccd_jacobi_rows(hipStream_t st, const uint32_t *directory, uint64_t dlength, int R,
                                  const float *num, const float *den, double lam, float *F) {
  const uint64_t n = dlength * (uint64_t)R;
  if (n == 0) return hipSuccess;
  uint64_t blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(k_ccd_jacobi_rows, dim3((unsigned)blocks), dim3(256), 0, st, directory, dlength, R, num, den,
                     lam, F);
  return hipGetLastError();
}

hipError_t launch_transpose(hipStream_t st, const float *in, float *out, uint64_t rows, int R,
                            bool to_colmajor) {
  const uint64_t n = rows * (uint64_t)R;
  if (n == 0) return hipSuccess;
  uint64_t blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(k_transpose, dim3((unsigned)blocks), dim3(256), 0, st, in, out, rows, R,
                     to_colmajor ? 1 : 0);
  return hipGetLastError();
}

}  // namespace ctc
