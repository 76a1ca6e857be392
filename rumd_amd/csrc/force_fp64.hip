// All-FP64 LJ 12-6 force / energy / virial kernels (gfx950): the comparison
// path for the FP32 kernels of force.hip.
//
// Reference arithmetic: fij (include/rumd/PairPotential.h:1198-1244) with
// Pot_IPL_12_6::ComputeInteraction (include/rumd/PairPotential.h:161-168),
// evaluated in double.  Positions are r (+ rlo in mixed mode) widened to
// double; the minimum image is formed in double; the cut-off shifts u(rc) and
// s(rc) rc are recomputed in double from the table's rc, A12 and A6 (RUMD
// computes them in float on the host, src/PairPotential.cu:82-125); the
// per-particle sums are double and are rounded once into the float4 outputs.
//
// The list formats are those of the FP32 kernels: tile lists (sorted method)
// are served by a tile kernel staging the halo as double positions in LDS;
// N2 lists and the no-list case by several lanes per particle reading
// positions from global memory.  FP64 arithmetic issues at the rate of plain
// FP32 here, so a pair costs its operation count: one reciprocal square root
// by iteration instead of a divide and a square root, no branch before the pair
// term, and no image correction where a tile's halo is staged in the shifted frame.
#include "force_kernels.h"

namespace rumdx {
namespace {

// Per type pair, in LDS: {rc^2, A12, A6, s(rc) rc, energy shift, unused}, the
// shift being -u(rc) for SP and -(u(rc) + s(rc) rc^2) for SF.
constexpr uint32_t kTabD = 6;

template <int CUT>
__device__ __forceinline__ void load_table_f64(double* s_tab, const float* __restrict__ params, uint32_t nt) {
  for (uint32_t k = threadIdx.x; k < nt * nt; k += blockDim.x) {
    const float* q = params + static_cast<size_t>(k) * RUMDX_NUM_PARAM;
    const double rc = q[0], a12 = q[1], a6 = q[2];
    const double i2 = 1.0 / (rc * rc), i6 = i2 * i2 * i2;
    const double ucut = i6 * (a12 * i6 + a6);
    const double src = i6 * i2 * (12.0 * a12 * i6 + 6.0 * a6) * rc;  // s(rc) rc = -u'(rc)
    double* t = s_tab + kTabD * k;
    t[0] = rc * rc;
    t[1] = a12;
    t[2] = a6;
    t[3] = src;
    t[4] = CUT == RUMDX_CUTOFF_SF ? -(ucut + src * rc) : -ucut;
    t[5] = 0.0;
  }
}

struct AccD {
  double fx = 0.0, fy = 0.0, fz = 0.0, u = 0.0, vir = 0.0;
  double sxx = 0.0, syy = 0.0, szz = 0.0, syz = 0.0, sxz = 0.0, sxy = 0.0;
};

struct PosD {
  double x, y, z;
  uint32_t t, pad;
};

__device__ __forceinline__ PosD pos_d(const float4* __restrict__ r, const float4* __restrict__ rlo, uint32_t j) {
  const float4 h = r[j];
  PosD p{static_cast<double>(h.x), static_cast<double>(h.y), static_cast<double>(h.z), __float_as_uint(h.w), 0u};
  if (rlo != nullptr) {
    const float4 l = rlo[j];
    p.x += static_cast<double>(l.x);
    p.y += static_cast<double>(l.y);
    p.z += static_cast<double>(l.z);
  }
  return p;
}

// 1/sqrt(x) to double precision: v_rsq_f64 (relative error about 2^-24) and
// one third-order step of the Householder iteration.
__device__ __forceinline__ double rsqrt_f64(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

// One pair; WRAP: the displacement needs the minimum image.  The pair term is
// formed for every pair, so that a group's pairs overlap, and added only inside
// rc: a masked factor of zero would still carry an infinite or undefined
// coordinate into the sums (0 x NaN).  19.0 us at KA N = 32,768 either way (20.0
// with the displacements masked as well).  kTinyD2 is added in d2's first product:
// the iteration of rsqrt_f64 has no start at zero, and r^-12 is infinite there.
constexpr double kTinyD2 = 1e-300;

template <int CUT, bool STR, bool WRAP>
__device__ __forceinline__ void pair_f64(const PosD& pi, const PosD& pj, const double* trow, const Box& bx,
                                         AccD& a) {
  double dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
  if (WRAP) {
    dx -= bx.Ld[0] * rint(dx * bx.iLd[0]);
    dy -= bx.Ld[1] * rint(dy * bx.iLd[1]);
    dz -= bx.Ld[2] * rint(dz * bx.iLd[2]);
  }
  const double d2 = fma(dz, dz, fma(dy, dy, fma(dx, dx, kTinyD2)));
  const double* t = trow + kTabD * pj.t;
  const double rinv = rsqrt_f64(d2), inv2 = rinv * rinv, inv6 = inv2 * inv2 * inv2;
  const double x = t[1] * inv6;  // A12 / r^6
  double s = 6.0 * inv6 * inv2 * fma(2.0, x, t[2]);
  double u = inv6 * (x + t[2]);
  if (CUT == RUMDX_CUTOFF_SP) {
    u += t[4];
  } else if (CUT == RUMDX_CUTOFF_SF) {
    s = fma(-t[3], rinv, s);
    u += fma(t[3], d2 * rinv, t[4]);
  }
  if (d2 < t[0]) {
    a.fx += dx * s;
    a.fy += dy * s;
    a.fz += dz * s;
    a.u += u;
    a.vir += d2 * s;
    if (STR) {
      a.sxx -= dx * dx * s;
      a.syy -= dy * dy * s;
      a.szz -= dz * dz * s;
      a.syz -= dy * dz * s;
      a.sxz -= dx * dz * s;
      a.sxy -= dx * dy * s;
    }
  }
}

// Sums a particle's partial accumulators over the 2^lg lanes that share it (a
// fixed butterfly).  Called by every lane of the wave.
template <bool STR>
__device__ __forceinline__ void combine_f64(AccD& a, uint32_t lg) {
  for (uint32_t o = 1; o < (1u << lg); o <<= 1) {
    a.fx += __shfl_xor(a.fx, o, 64);
    a.fy += __shfl_xor(a.fy, o, 64);
    a.fz += __shfl_xor(a.fz, o, 64);
    a.u += __shfl_xor(a.u, o, 64);
    a.vir += __shfl_xor(a.vir, o, 64);
    if (STR) {
      a.sxx += __shfl_xor(a.sxx, o, 64);
      a.syy += __shfl_xor(a.syy, o, 64);
      a.szz += __shfl_xor(a.szz, o, 64);
      a.syz += __shfl_xor(a.syz, o, 64);
      a.sxz += __shfl_xor(a.sxz, o, 64);
      a.sxy += __shfl_xor(a.sxy, o, 64);
    }
  }
}

template <bool STR, bool INIT>
__device__ __forceinline__ void store_f64(uint32_t i, const AccD& a, float4* __restrict__ f, float4* __restrict__ w,
                                          float4* __restrict__ sts) {
  const double u = 0.5 * a.u;  // each pair energy was counted from both ends
  if (INIT) {
    f[i] = make_float4(static_cast<float>(a.fx), static_cast<float>(a.fy), static_cast<float>(a.fz),
                       static_cast<float>(u));
    w[i] = make_float4(0.f, STR ? static_cast<float>(a.sxz) : 0.f, STR ? static_cast<float>(a.sxy) : 0.f,
                       static_cast<float>(a.vir));
    if (STR)
      sts[i] = make_float4(static_cast<float>(a.sxx), static_cast<float>(a.syy), static_cast<float>(a.szz),
                           static_cast<float>(a.syz));
  } else {
    const float4 fo = f[i];
    f[i] = make_float4(static_cast<float>(fo.x + a.fx), static_cast<float>(fo.y + a.fy),
                       static_cast<float>(fo.z + a.fz), static_cast<float>(fo.w + u));
    float4 wo = w[i];
    wo.w = static_cast<float>(wo.w + a.vir);
    if (STR) {
      wo.y = static_cast<float>(wo.y + a.sxz);
      wo.z = static_cast<float>(wo.z + a.sxy);
      const float4 so = sts[i];
      sts[i] = make_float4(static_cast<float>(so.x + a.sxx), static_cast<float>(so.y + a.syy),
                           static_cast<float>(so.z + a.szz), static_cast<float>(so.w + a.syz));
    }
    w[i] = wo;
  }
}

// A coordinate in the tile's shifted frame (shift_coord in double: the moved
// coordinate is off by one rounding of a double at most).
__device__ __forceinline__ double shift_f64(double x, uint32_t fl, int axis, double len) {
  const uint32_t f = fl >> (2 * axis);
  if ((f & kTileShiftDown) && x >= 0.0) return x - len;
  if ((f & kTileShiftUp) && x < 0.0) return x + len;
  return x;
}

__device__ __forceinline__ PosD shifted_f64(PosD p, uint32_t fl, const Box& bx) {
  p.x = shift_f64(p.x, fl, 0, bx.Ld[0]);
  p.y = shift_f64(p.y, fl, 1, bx.Ld[1]);
  p.z = shift_f64(p.z, fl, 2, bx.Ld[2]);
  return p;
}

// The staged halo in LDS, one array per coordinate: 8-byte reads of scattered
// particles spread over all banks (a 32-byte record leaves half of them idle)
// and 25 bytes a particle admit three workgroups per CU.
struct HaloD {
  double* x;
  double* y;
  double* z;
  uint8_t* t;

  __device__ __forceinline__ HaloD(void* lds, uint32_t cap) {
    x = static_cast<double*>(lds);
    y = x + cap;
    z = y + cap;
    t = reinterpret_cast<uint8_t*>(z + cap);
  }
  __device__ __forceinline__ PosD get(uint32_t h) const { return PosD{x[h], y[h], z[h], t[h], 0u}; }
  __device__ __forceinline__ void put(uint32_t h, const PosD& p) const {
    x[h] = p.x;
    y[h] = p.y;
    z[h] = p.z;
    t[h] = static_cast<uint8_t>(p.t);
  }
};
static_assert(RUMDX_MAX_TYPES <= 256, "types are staged as bytes");

// A particle's stored list against the staged halo, this lane's groups part,
// part + step, ... (the FP32 tile kernel's split of a list over lanes).
template <int CUT, bool STR, bool WRAP>
__device__ __forceinline__ void list_f64(const PosD& pi, uint32_t i, uint32_t nn, uint32_t part, uint32_t step,
                                         const uint16_t* __restrict__ nbl16, uint32_t nvp, const HaloD& s_pd,
                                         bool bytes, const double* trow, const Box& bx, AccD& a) {
  const u32x4* grp = reinterpret_cast<const u32x4*>(nbl16);
  const uint32_t sh = bytes ? 4u : 0u;
  for (uint32_t g = part; g * 8u < nn; g += step) {
    const u32x4 q = __builtin_nontemporal_load(grp + static_cast<size_t>(g) * nvp + i);
    const uint32_t m = nn - g * 8u;
    if (m >= 8u) {
#pragma unroll
      for (int e = 0; e < 8; ++e) pair_f64<CUT, STR, WRAP>(pi, s_pd.get(group_entry(q, e) >> sh), trow, bx, a);
    } else {
#pragma unroll
      for (int e = 0; e < 7; ++e)
        if (static_cast<uint32_t>(e) < m)
          pair_f64<CUT, STR, WRAP>(pi, s_pd.get(group_entry(q, e) >> sh), trow, bx, a);
    }
  }
}

// Tile lists of the sorted method: `split` workgroups per tile, the halo as
// double positions in LDS by one gather over the slot list the build recorded,
// a particle's list spread over as many of its lanes as fit.  Bound by VALU
// issue (45 operations a pair, 57 where the image is needed) with the LDS reads
// close behind (64 bytes a pair).  At KA N = 32,768 56.5 -> 20.6 us in 216 tiles
// against one lane per particle walking 2-byte entries (19.3 in the 726 smaller
// tiles a sample of this size has); 24.4 us with 32-byte records in LDS.
//
// The workgroup's size goes by the mean number of particles in a tile.  Where
// the tiles are few (four workgroups per CU), 384 lanes for up to 128 particles,
// else 512.  384 against 512 lanes: 14.0 / 16.0 us at 18 particles a tile (KA n =
// 9,000), 19.3 / 22.4 at 45 (32,768), 28.2 / 28.3 at 87 (60,000), but 36.4 / 30.9 at
// 215 (110,000); 256 lanes 13.6 for 11.5 at 23 (12,000).  Where they are many, lanes
// without a particle only hold back other workgroups: the smallest power of two
// with two lanes for each.  Such a workgroup against 384 lanes, LJ: 98 / 392 us at
// 1,000,000 particles cut at 1.2 (46,656 tiles of 21), 23 / 57 at 200,000 cut at 1.5
// (4,913 of 41), 129 / 197 at 1,000,000 cut at 2.0 (12,167 of 82).
constexpr uint32_t kFewTilesF64 = 1024;

uint32_t block_f64(uint32_t n, uint32_t ntiles) {
  const auto holds = [&](uint32_t per_tile) { return n <= static_cast<uint64_t>(per_tile) * ntiles; };
  if (ntiles <= kFewTilesF64) return holds(128) ? 384u : 512u;
  return holds(32) ? 64u : holds(64) ? 128u : holds(128) ? 256u : 512u;
}

template <int CUT, bool STR, bool INIT, uint32_t BLOCK>
__global__ __launch_bounds__(BLOCK) void k_lj_tiles_f64(
    const float4* __restrict__ r, const float4* __restrict__ rlo, float4* __restrict__ f, float4* __restrict__ w,
    float4* __restrict__ sts, const uint16_t* __restrict__ nbl16, const uint32_t* __restrict__ num_nbrs,
    const uint16_t* __restrict__ lane_order, const float* __restrict__ params, uint32_t nt, Box bx,
    const uint4* __restrict__ tile_info, const uint32_t* __restrict__ halo_slots, uint32_t halo_cap, uint32_t cap,
    CellFallback fb, uint32_t nvp, uint32_t max_nbrs, uint32_t split) {
  extern __shared__ double s_dd[];
  double* s_tab = s_dd;
  const HaloD s_pd(s_dd + kTabD * nt * nt, cap);
  load_table_f64<CUT>(s_tab, params, nt);
  const uint32_t b = xcd_block(blockIdx.x, gridDim.x);
  const uint32_t t = b / split, share = b % split;
  const uint4 info = tile_info[t];
  // staged by the build (its halo list is written) and fits here in double
  const bool staged = (info.y >> 16) == halo_cap && info.x <= halo_cap && info.x <= cap;
  const bool fast = (info.y & kTileFast) != 0u;
  const uint32_t shifts = fast ? info.y : 0u;
  const bool bytes = info.x <= kByteEntryHalo;
  if (staged) {
    const uint32_t* hs = halo_slots + static_cast<size_t>(t) * halo_cap;
    // slots of four particles, then their positions: each set in flight together
    for (uint32_t q0 = threadIdx.x; q0 < info.x; q0 += 4u * BLOCK) {
      uint32_t slot[4];
      PosD p[4];
#pragma unroll
      for (uint32_t u = 0; u < 4u; ++u) {
        const uint32_t q = q0 + u * BLOCK;
        slot[u] = hs[q < info.x ? q : q0];
      }
#pragma unroll
      for (uint32_t u = 0; u < 4u; ++u) p[u] = pos_d(r, rlo, slot[u]);
#pragma unroll
      for (uint32_t u = 0; u < 4u; ++u)
        if (q0 + u * BLOCK < info.x) s_pd.put(q0 + u * BLOCK, shifted_f64(p[u], shifts, bx));
    }
  }
  __syncthreads();
  // this workgroup's particles: every split-th of the lane order, so that the
  // shares of a tile have lists of like lengths
  const uint32_t all = info.w - info.z;
  const uint32_t np = all > share ? (all - share + split - 1u) / split : 0u;
  uint32_t lg = 0;
  while (lg < 3u && (np << (lg + 1u)) <= BLOCK) ++lg;
  const uint32_t part = threadIdx.x & ((1u << lg) - 1u), step = 1u << lg;
  for (uint32_t c0 = 0; c0 < np; c0 += BLOCK >> lg) {
    const uint32_t k = c0 + (threadIdx.x >> lg);
    const bool live = k < np;
    AccD a;
    uint32_t i = 0;
    if (live) {
      i = info.z + lane_order[info.z + k * split + share];
      const PosD pi = pos_d(r, rlo, i);
      const double* trow = s_tab + kTabD * nt * pi.t;
      const uint32_t nn = num_nbrs[i];
      if (staged && nn < max_nbrs) {
        if (fast)
          list_f64<CUT, STR, false>(shifted_f64(pi, shifts, bx), i, nn, part, step, nbl16, nvp, s_pd, bytes, trow, bx, a);
        else
          list_f64<CUT, STR, true>(pi, i, nn, part, step, nbl16, nvp, s_pd, bytes, trow, bx, a);
      } else if (part == 0) {
        const uint32_t lin = fb.slot_cell[i];
        const int cx = static_cast<int>(lin % fb.nc0);
        const int cy = static_cast<int>((lin / fb.nc0) % fb.nc1);
        const int cz = static_cast<int>(lin / (static_cast<uint32_t>(fb.nc0) * fb.nc1));
        for (int dz = -2; dz <= 2; ++dz)
          for (int dy = -2; dy <= 2; ++dy)
            for (int dx = -2; dx <= 2; ++dx) {
              const int ox = (cx + dx + fb.nc0) % fb.nc0, oy = (cy + dy + fb.nc1) % fb.nc1,
                        oz = (cz + dz + fb.nc2) % fb.nc2;
              const uint32_t rank = fb.cell_rank[ox + oy * fb.nc0 + oz * fb.nc0 * fb.nc1];
              for (uint32_t j = fb.cell_start[rank]; j < fb.cell_start[rank + 1]; ++j)
                if (j != i) pair_f64<CUT, STR, true>(pi, pos_d(r, rlo, j), trow, bx, a);
            }
      }
    }
    combine_f64<STR>(a, lg);
    if (live && part == 0) store_f64<STR, INIT>(i, a, f, w, sts);
  }
}

// N2 lists (u32 slots, column-major) or, with nbl == nullptr, all pairs: 2^lg
// lanes share a particle.
template <int CUT, bool STR, bool INIT>
__global__ __launch_bounds__(kBlock) void k_lj_slots_f64(const float4* __restrict__ r, const float4* __restrict__ rlo,
                                                         float4* __restrict__ f, float4* __restrict__ w,
                                                         float4* __restrict__ sts, const uint32_t* __restrict__ nbl,
                                                         const uint32_t* __restrict__ num_nbrs,
                                                         const float* __restrict__ params, uint32_t nt, Box bx,
                                                         uint32_t n, uint32_t nvp, uint32_t max_nbrs, uint32_t lg) {
  extern __shared__ double s_dd[];
  load_table_f64<CUT>(s_dd, params, nt);
  __syncthreads();
  const uint32_t gid = xcd_block(blockIdx.x, gridDim.x) * (kBlock >> lg) + (threadIdx.x >> lg);
  const uint32_t part = threadIdx.x & ((1u << lg) - 1u), step = 1u << lg;
  const bool live = gid < n;
  const uint32_t i = live ? gid : n - 1u;
  AccD a;
  if (live) {
    const PosD pi = pos_d(r, rlo, i);
    const double* trow = s_dd + kTabD * nt * pi.t;
    const uint32_t nn = nbl != nullptr ? num_nbrs[i] : 0u;
    if (nbl != nullptr && nn < max_nbrs) {
      for (uint32_t k = part; k < nn; k += step)
        pair_f64<CUT, STR, true>(pi, pos_d(r, rlo, nbl[static_cast<size_t>(k) * nvp + i]), trow, bx, a);
    } else {
      for (uint32_t j = part; j < n; j += step)
        if (j != i) pair_f64<CUT, STR, true>(pi, pos_d(r, rlo, j), trow, bx, a);
    }
  }
  combine_f64<STR>(a, lg);
  if (live && part == 0) store_f64<STR, INIT>(i, a, f, w, sts);
}

// LDS of the tile kernel: the table and the halo positions.
constexpr size_t kHaloDBytes = 3 * sizeof(double) + 1;
size_t tiles_f64_lds(uint32_t cap, uint32_t nt) { return sizeof(double) * kTabD * nt * nt + kHaloDBytes * cap; }

// The halo capacity of the tile kernel: the list's, bounded by the device's
// LDS per workgroup (halos beyond it read positions from global memory).
uint32_t tiles_f64_cap(uint32_t cap, uint32_t nt) {
  int dev = 0, lds = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || lds <= 0)
    lds = 64 * 1024;
  const size_t fixed = sizeof(double) * kTabD * nt * nt + 256;
  const size_t most = static_cast<size_t>(lds) > fixed ? (static_cast<size_t>(lds) - fixed) / kHaloDBytes : 0;
  return cap < most ? cap : static_cast<uint32_t>(most);
}

template <int CUT, bool STR, bool INIT>
int launch_f64(const rumdx_particles* p, const rumdx_nblist* nb, const float* params, uint32_t nt, const Box& bx,
               hipStream_t st) {
  const float4* r = reinterpret_cast<const float4*>(p->r_dev);
  const float4* rlo = reinterpret_cast<const float4*>(p->rlo_dev);
  float4* f = reinterpret_cast<float4*>(p->f_dev);
  float4* w = reinterpret_cast<float4*>(p->w_dev);
  float4* sts = reinterpret_cast<float4*>(p->sts_dev);
  if (nb != nullptr && nb->nbl16_dev != nullptr) {
    const uint32_t cap = tiles_f64_cap(nb->halo_cap, nt);
    const CellFallback fb{nb->cell_rank_dev, nb->cell_start_dev, nb->slot_cell_dev, nb->nc[0], nb->nc[1], nb->nc[2], {}};
    // A small sample has fewer tiles than the chip holds workgroups: several
    // workgroups then share a tile, each staging its halo.  One / two / four:
    // 27 / 18 / 13 us at 64 tiles (n = 9,000), 23 / 16 / 16 at 125 (20,000),
    // 32 / 30 / 40 at 343 (60,000), 31 / 36 / 51 at 512 (110,000), in 4^3 tiles.
    const uint32_t split = nb->ntiles >= 384u ? 1u : nb->ntiles >= 96u ? 2u : 4u;
    const auto launch = [&](auto kernel, uint32_t block) {
      hipLaunchKernelGGL(kernel, dim3(nb->ntiles * split), dim3(block), tiles_f64_lds(cap, nt), st, r, rlo, f, w, sts,
                         nb->nbl16_dev, nb->num_nbrs_dev, nb->lane_order_dev, params, nt, bx,
                         reinterpret_cast<const uint4*>(nb->tile_info_dev), nb->tile_halo_dev, nb->halo_cap, cap, fb,
                         p->nvp, nb->max_nbrs, split);
    };
    switch (block_f64(p->n, nb->ntiles)) {
      case 64: launch(k_lj_tiles_f64<CUT, STR, INIT, 64>, 64); break;
      case 128: launch(k_lj_tiles_f64<CUT, STR, INIT, 128>, 128); break;
      case 256: launch(k_lj_tiles_f64<CUT, STR, INIT, 256>, 256); break;
      case 384: launch(k_lj_tiles_f64<CUT, STR, INIT, 384>, 384); break;
      default: launch(k_lj_tiles_f64<CUT, STR, INIT, 512>, 512); break;
    }
  } else {
    // a wave per particle over all pairs; 16 lanes over a list (some 90
    // entries), so that a sample of a thousand particles fills the CUs
    const uint32_t lg = nb != nullptr ? 4u : 6u;
    hipLaunchKernelGGL((k_lj_slots_f64<CUT, STR, INIT>), dim3(blocks_for(p->n, kBlock >> lg)), dim3(kBlock),
                       sizeof(double) * kTabD * nt * nt, st, r, rlo, f, w, sts, nb != nullptr ? nb->nbl_dev : nullptr,
                       nb != nullptr ? nb->num_nbrs_dev : nullptr, params, nt, bx, p->n, p->nvp,
                       nb != nullptr ? nb->max_nbrs : 0u, lg);
  }
  return check_launch("rumdx_pair_lj_fp64");
}

template <int CUT>
int dispatch_f64(const rumdx_particles* p, const rumdx_nblist* nb, const float* params, uint32_t nt, const Box& bx,
                 bool init, bool str, hipStream_t st) {
  if (str) return init ? launch_f64<CUT, true, true>(p, nb, params, nt, bx, st)
                       : launch_f64<CUT, true, false>(p, nb, params, nt, bx, st);
  return init ? launch_f64<CUT, false, true>(p, nb, params, nt, bx, st)
              : launch_f64<CUT, false, false>(p, nb, params, nt, bx, st);
}

}  // namespace
}  // namespace rumdx

extern "C" int rumdx_pair_lj_fp64(const rumdx_particles* p, const rumdx_nblist* nb, const float* params_dev,
                                  uint32_t ntypes, const float box[8], int cutoff_method, int initialize,
                                  int calc_stresses, void* stream) {
  using namespace rumdx;
  if (p == nullptr || box == nullptr || params_dev == nullptr)
    return fail(RUMDX_E_INVALID, "rumdx_pair_lj_fp64: null argument");
  if (p->r_dev == nullptr || p->f_dev == nullptr || p->w_dev == nullptr)
    return fail(RUMDX_E_INVALID, "rumdx_pair_lj_fp64: particle arrays not allocated");
  if (calc_stresses && p->sts_dev == nullptr)
    return fail(RUMDX_E_INVALID, "rumdx_pair_lj_fp64: stresses requested but sts is null");
  if (nb != nullptr && nb->excl_start_dev != nullptr)
    return fail(RUMDX_E_INVALID, "rumdx_pair_lj_fp64: the FP64 comparison path takes lists without exclusions");
  if (ntypes == 0 || ntypes > RUMDX_MAX_TYPES) return fail(RUMDX_E_INVALID, "rumdx_pair_lj_fp64: ntypes out of range");
  if (p->n == 0) return RUMDX_OK;
  if (nb != nullptr && ((nb->nbl_dev == nullptr && nb->nbl16_dev == nullptr) || nb->num_nbrs_dev == nullptr ||
                        nb->max_nbrs == 0))
    return fail(RUMDX_E_INVALID, "rumdx_pair_lj_fp64: neighbour list not allocated");
  if (nb != nullptr && nb->nbl16_dev != nullptr &&
      (nb->ntiles == 0 || nb->tile_first_rank_dev == nullptr || nb->tile_origin_dev == nullptr ||
       nb->slot_cell_dev == nullptr || nb->cell_rank_dev == nullptr || nb->cell_start_dev == nullptr ||
       nb->lane_order_dev == nullptr || nb->tile_info_dev == nullptr || nb->tile_halo_dev == nullptr))
    return fail(RUMDX_E_INVALID, "rumdx_pair_lj_fp64: tile arrays not allocated");
  const Box bx = make_box(box);
  const hipStream_t st = as_stream(stream);
  const bool init = initialize != 0, str = calc_stresses != 0;
  switch (cutoff_method) {
    case RUMDX_CUTOFF_NS: return dispatch_f64<RUMDX_CUTOFF_NS>(p, nb, params_dev, ntypes, bx, init, str, st);
    case RUMDX_CUTOFF_SP: return dispatch_f64<RUMDX_CUTOFF_SP>(p, nb, params_dev, ntypes, bx, init, str, st);
    case RUMDX_CUTOFF_SF: return dispatch_f64<RUMDX_CUTOFF_SF>(p, nb, params_dev, ntypes, bx, init, str, st);
    default: return fail(RUMDX_E_INVALID, "rumdx_pair_lj_fp64: invalid cutoff method");
  }
}
