// fv_sweep.h -- the fused finite-volume stage kernel.
//
// One workgroup updates one block of the level; a lane owns one (x, y)
// column of the block (BX x BX lanes: 256 for 16^2 blocks, rounded up to
// whole waves for 8^2 and 10^2).  The block's stencil data never round-trips through HBM ghost
// cells: halo cells are read straight from the face neighbours' interiors
// through the level's neighbour table (or from a physical-boundary rule),
// converted to primitive variables once and staged in LDS.  In 3-D the
// workgroup marches along z with a per-lane register window of 2*NG
// primitive planes; x/y faces of the current plane come from LDS, the z face
// from the window, and each z-face flux is computed once and carried.  On a
// level with too few blocks to fill the GPU a block's planes are split over
// several workgroups (blockIdx.y), each with its own window and first face.
//
// Per cell and stage the kernel does what finite_volume
// (src/mod_finite_volume.t:116-339) or hancock (:19-113) plus addsource2
// (src/mod_source.t:130-160) do for one block, fused with the RK
// combination of src/mod_advance.t:251-267:
//   wnew = init + sum_d [ (-qdt/dx_d) fC_d(i+1/2) - (-qdt/dx_d) fC_d(i-1/2) ]
//          + sources(wCT)
// with init = psb, psb = base, or a*base + b*psa.
#pragma once

#include <type_traits>

#include "fv_device.h"

namespace fvc {
constexpr int BX = 16;  // block_nx(1) = block_nx(2) of the fastest kernels
constexpr int NTHREADS = 256;

struct SweepArgs {
  const double* src;   // psa (stage input, wCT)
  const double* base;  // RK base slot (comb_mode 1, 2)
  double* dst;         // psb
  const int* nbr;      // [nb][3^ndim]
  int nblocks;
  int bx;              // block_nx(1) = block_nx(2)
  int bnz;             // block_nx(3) (1 in 2-D)
  int per_xcd;         // ceil(nblocks/8)
  int zc;              // planes of a workgroup (3-D; bnz: the block is not split)
  int src_al16;        // src is aligned to 16 bytes
  int comb_mode;       // 0: init = dst, 1: init = base, 2: init = a*base + b*src,
                       // 3: init = src (base is the stage input itself)
  double comb_a, comb_b;
  double dq[3];        // -qdt/dx_d
  double qdt;
  double ch;           // cmax_global (GLM)
  double glm_decay;    // exp(-qdt*ch*alpha/min dx)
  int bc[6];           // physical boundary type per side
  int* crash;
  // block-structured AMR (all nullptr / unused on a uniform level)
  const int* blevel;        // level-1 of each block: cell size dx/2^blevel
  double glm_decay_lev[8];  // psi decay factor per level
  double* freg;             // scaled block-boundary face fluxes (refluxing)
  const int* fregoff;       // [nb][2*ndim] register offset of a face, -1: none
  int nface;                // transverse cells of a face (register stride)
  int linde;                // Linde's source follows the stage (linde_kernel)
  // CFL partials of the output (uniform level, mixed form): per block, which is
  // one workgroup, the max over cells of sum_d cmax_d/dx_d and of cmax, as
  // getdt_courant needs them; nullptr: not wanted
  double* dt_part;
};

constexpr int MAXLEV = 8;

}  // namespace fvc

namespace FV_NS {
using fvc::BX;
using fvc::NTHREADS;
using fvc::SweepArgs;

// lanes of the stage kernel for BX x BX blocks (whole waves)
template <int BXc>
constexpr int kLanes = (BXc * BXc + 63) / 64 * 64;

// Block id of a workgroup: consecutive blocks of the Morton-ordered level go
// to the same XCD (workgroups are dealt round-robin over the 8 XCDs), so that
// halo reads of neighbouring blocks hit the XCD's own L2.
__device__ __forceinline__ int wg_block(int per_xcd) {
  const int g = blockIdx.x;
  return (g & 7) * per_xcd + (g >> 3);
}

// Resolve the source of cell (x,y,z) (block-local, may lie outside the
// block by up to NG) for block b: returns the source block and rewrites the
// coordinates into it; *sign = -1 for an antisymmetric boundary.
// (BXc = 0: the block size a.bx of the arguments; else the compile-time one)
template <int NDIM, int BXc = 0>
__device__ __forceinline__ int locate(const SweepArgs& a, int b, int& x, int& y, int& z, double& sign) {
  int c[3] = {x, y, z};
  const int bx = BXc ? BXc : a.bx;
  const int n[3] = {bx, bx, a.bnz};
  int dir[3] = {0, 0, 0};
  sign = 1.0;
#pragma unroll
  for (int d = 0; d < NDIM; ++d) dir[d] = c[d] < 0 ? -1 : (c[d] >= n[d] ? 1 : 0);
  int nn = 1, idx = 0;
#pragma unroll
  for (int d = 0; d < NDIM; ++d) { idx += (dir[d] + 1) * nn; nn *= 3; }
  int nb = a.nbr[b * nn + idx];
  if (nb >= 0) {
#pragma unroll
    for (int d = 0; d < NDIM; ++d) c[d] -= dir[d] * n[d];
    x = c[0]; y = c[1]; z = c[2];
    return nb;
  }
  // physical boundary: apply cont / symm / asymm in every direction whose
  // face neighbour is a boundary, then take the remaining offset from the
  // neighbour in the other directions
  // (bc_phys src/mod_boundary_conditions.t:12-120)
  int rem[3] = {0, 0, 0};
#pragma unroll
  for (int d = 0; d < NDIM; ++d) {
    if (dir[d] == 0) continue;
    int fidx = 0, m = 1;
#pragma unroll
    for (int e = 0; e < NDIM; ++e) { fidx += ((e == d ? dir[d] : 0) + 1) * m; m *= 3; }
    if (a.nbr[b * nn + fidx] >= 0) { rem[d] = dir[d]; continue; }
    const int t = a.bc[2 * d + (dir[d] > 0 ? 1 : 0)];
    if (t == 2) {  // cont
      c[d] = dir[d] < 0 ? 0 : n[d] - 1;
    } else {       // symm / asymm
      c[d] = dir[d] < 0 ? -1 - c[d] : 2 * n[d] - 1 - c[d];
      if (t == 4) sign = -sign;
    }
  }
  int ridx = 0, m = 1;
#pragma unroll
  for (int d = 0; d < NDIM; ++d) { ridx += (rem[d] + 1) * m; m *= 3; }
  int src = b;
  if (ridx != (nn - 1) / 2) {
    src = a.nbr[b * nn + ridx];
#pragma unroll
    for (int d = 0; d < NDIM; ++d) c[d] -= rem[d] * n[d];
  }
  x = c[0]; y = c[1]; z = c[2];
  return src;
}

template <class P>
__device__ __forceinline__ void load_cons(const double* __restrict__ w, int b, int x, int y, int z, int bx,
                                          int bnz, double* c) {
  const size_t cells = (size_t)bx * bx * bnz;
  const size_t off = (size_t)b * P::NW * cells + ((size_t)z * bx + y) * bx + x;
#pragma unroll
  for (int iw = 0; iw < P::NW; ++iw) c[iw] = w[off + iw * cells];
}

// conserved state of an arbitrary (possibly halo) cell, with the sign of an
// antisymmetric boundary applied
template <class P, int NDIM, int BXc = 0>
__device__ __forceinline__ void load_cons_at(const SweepArgs& a, int b, int x, int y, int z, double* c) {
  double sign;
  const int sb = locate<NDIM, BXc>(a, b, x, y, z, sign);
  load_cons<P>(a.src, sb, x, y, z, BXc ? BXc : a.bx, a.bnz, c);
  if (sign < 0.0) {
#pragma unroll
    for (int iw = 0; iw < P::NW; ++iw) c[iw] = -c[iw];
  }
}

// primitive state (FP64 conversion, rounded to R) of conserved state c
template <class P, class R>
__device__ __forceinline__ void prim_of(const double* c, R* out, const FVParams& fp) {
  double w[P::NW];
  to_prim<P>(c, w, fp);
#pragma unroll
  for (int iw = 0; iw < P::NW; ++iw) out[iw] = R(w[iw]);
}

// primitive state of an arbitrary (possibly halo) cell
template <class P, class R, int NDIM, int BXc = 0>
__device__ __forceinline__ void load_prim(const SweepArgs& a, const FVParams& fp, int b, int x, int y,
                                          int z, R* w) {
  double c[P::NW];
  load_cons_at<P, NDIM, BXc>(a, b, x, y, z, c);
  prim_of<P, R>(c, w, fp);
}

// The RK base and the output are touched once per launch: they stream
// through L2 (non-temporal) so that they do not displace the stage input,
// whose planes are re-read as halos by neighbouring workgroups.
constexpr int kNonTemporal = 2;  // nt bit of the cache policy
// bytes at p (the same for the whole wave) as a raw buffer
__device__ __forceinline__ __amdgpu_buffer_rsrc_t block_buffer(const double* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(p), 0, bytes, 0x00020000);
}
typedef unsigned uint2v __attribute__((ext_vector_type(2)));
template <int POLICY>
__device__ __forceinline__ double buffer_ld(__amdgpu_buffer_rsrc_t r, unsigned lane, unsigned off) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, lane, off, POLICY));
}
template <int POLICY>
__device__ __forceinline__ void buffer_st(double v, __amdgpu_buffer_rsrc_t r, unsigned lane, unsigned off) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2v, v), r, lane, off, POLICY);
}

// Cell t of the four NG-deep halo strips of a plane (x and y block-local,
// outside the block on one side), t < 4*NG*BX; then the 4 NG x NG corners.
template <int NG, int BX>
__device__ __forceinline__ void strip_cell(int t, int& x, int& y) {
  constexpr int NSTRIP = 4 * NG * BX;
  if (t < NSTRIP) {
    const int s = t / (NG * BX), r = t % (NG * BX);
    const int along = r % BX, depth = r / BX;
    if (s == 0) { x = -NG + depth; y = along; }
    else if (s == 1) { x = BX + depth; y = along; }
    else if (s == 2) { x = along; y = -NG + depth; }
    else { x = along; y = BX + depth; }
  } else {
    const int u = t - NSTRIP;
    const int q = u / (NG * NG), r = u % (NG * NG);
    const int ox = r % NG, oy = r / NG;
    x = (q & 1) ? BX + ox : -NG + ox;
    y = (q & 2) ? BX + oy : -NG + oy;
  }
}

// The halo strips of a plane as 16-byte pairs of neighbouring cells in x, 64
// per variable of a 16^2 cross-section: pair p < 64 of the strips x-, x+ (16
// rows), y-, y+ (2 rows of 8 pairs).  Offset of the pair's first cell in the
// state, plane 0, variable 0; a physical boundary takes the cells of the
// block that bc_phys mirrors or extends (which of the two, and the sign, is
// the reader's: halo_elem).
template <int NW>
__device__ __forceinline__ size_t halo_pair(const SweepArgs& a, int b, int p) {
  const int s = p >> 4, q = p & 15;
  const int hi = s & 1, dim = s >> 1;
  const int nbk = a.nbr[b * 27 + 13 + (hi ? 1 : -1) * (dim ? 3 : 1)];
  const int depth = q >> 3;
  int x, y;
  if (dim == 0) {
    y = q;
    x = (nbk >= 0) == (hi != 0) ? 0 : 14;
  } else {
    x = 2 * (q & 7);
    if (nbk >= 0) y = hi ? depth : 14 + depth;
    else if (a.bc[2 + hi] == 2) y = hi ? 15 : 0;
    else y = hi ? 15 - depth : 1 - depth;
  }
  const size_t cells = (size_t)256 * a.bnz;
  return (size_t)(nbk >= 0 ? nbk : b) * NW * cells + y * 16 + x;
}
// Position (2 pair + element) of halo cell t < 128 (strip_cell's order) among
// the pairs, and the sign of an antisymmetric boundary
__device__ __forceinline__ int halo_elem(const SweepArgs& a, int b, int t, bool& neg) {
  const int s = t >> 5, along = t & 15, depth = (t >> 4) & 1;
  const int hi = s & 1, dim = s >> 1;
  const bool phys = a.nbr[b * 27 + 13 + (hi ? 1 : -1) * (dim ? 3 : 1)] < 0;
  const int bc = a.bc[2 * dim + hi];
  neg = phys && bc == 4;
  if (dim == 1) return 2 * (s * 16 + depth * 8 + (along >> 1)) + (along & 1);
  const int e = !phys ? depth : (bc == 2 ? hi : 1 - depth);
  return 2 * (s * 16 + along) + e;
}

// Occupancy: FP64 kernels run 2 waves per SIMD (LDS and registers), FP32
// kernels are held to 3 (at most 168 VGPRs).
template <class R>
constexpr int kMinWaves = std::is_same<R, float>::value ? 3 : 2;

// Scheme constants of a block's level: every length scales by 2^-lev
// (dx(level) = dx(level-1)/2, src/mod_initialize.t:101), so the products
// below are exact and match a level-wise evaluation bit for bit.
__device__ __forceinline__ void level_params(const SweepArgs& a, int b, FVParams& fp, double* dq,
                                             double& glm_decay) {
  dq[0] = a.dq[0]; dq[1] = a.dq[1]; dq[2] = a.dq[2];
  glm_decay = a.glm_decay;
  if (!a.blevel) return;
  const int lev = a.blevel[b];
  if (lev == 0) return;
  const double sc = double(1 << lev), sc2 = sc * sc;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    fp.dx[d] = fp.dx[d] / sc;
    fp.dxinv[d] = fp.dxinv[d] * sc;
    fp.rdelinv[d] = fp.rdelinv[d] * sc2;
    fp.cada3k[d] = fp.cada3k[d] * sc2;
    fp.cada3t[d] = fp.cada3t[d] / sc2;
    dq[d] = dq[d] * sc;
  }
  fp.invds2 = fp.invds2 * sc2;
  fp.mindx = fp.mindx / sc;
  glm_decay = a.glm_decay_lev[lev];
}

// Cell-centred field: nothing beside the flux update
struct NoCt {};

// AMR: level-dependent scheme constants and the refluxing registers; the
// uniform-level kernels are compiled without them (their registers would
// spill in the 3-D MHD kernels).
// CTA: a 3-D stage of constrained transport (its face field, face data and
// edge fields; fv_ct3.hip): the faces take their normal field from it and give
// it what the edge fields need, and the update leaves out the field.
template <class P, class R, int RIEM, int LIM, int NG, bool AMR, int BXc, class CTA = NoCt>
__global__ void __launch_bounds__(kLanes<BXc>, kMinWaves<R>)
sweep_kernel(SweepArgs a, FVParams fp0, CTA ct) {
  constexpr int BX = BXc;                 // block_nx(1) = block_nx(2)
  constexpr int NTHREADS = kLanes<BXc>;   // lanes of the workgroup
  constexpr bool FULL = BX * BX == NTHREADS;
  constexpr int NDIM = P::NDIM;
  constexpr int NW = P::NW;
  constexpr int PX = BX + 2 * NG;
  constexpr bool HANCOCK = RIEM == RIEM_HANCOCK;
  constexpr bool CT = !std::is_same<CTA, NoCt>::value;
  constexpr int NF = CT ? P::MAG : NW;    // variables updated from their fluxes
  // Any extra runtime branch in the z loop of the specialised kernels (a
  // compile-time TVD limiter on a uniform level of 16^2 cross-sections)
  // costs the FP64 form about 12% (measured): they carry no small-value
  // checks (runs with fix_small_values take the runtime-limiter kernel),
  // and only the FP32-reconstruction form, where the fused CFL partials cost
  // 2% and save the separate pass over ps, computes them.
  constexpr bool SPECIAL = LIM != 0 && LIM != LIM_WENO5 && !AMR && BXc == 16;
  constexpr bool SMALLCHK = !SPECIAL && !CT;
  constexpr bool CFL = !AMR && !CT && BXc == 16 && std::is_same<R, float>::value;
  constexpr int NSTRIP = 4 * NG * BX;
  constexpr int NHALO = NSTRIP;
  // 3-D, FP32 reconstruction: the halo strips of the NG planes ahead are
  // loaded together with the window's lookahead plane and kept in an LDS ring
  // (the face neighbours read the same planes at the same time, so the loads
  // hit L2).  The FP64 kernel keeps to 2 workgroups per CU within 160 KB of
  // LDS by loading the halo of the current plane instead.
  constexpr bool HRING = NDIM == 3 && std::is_same<R, float>::value;

  __shared__ R sp[NW][PX][PX];          // primitive plane with halo
  __shared__ R fxs[HANCOCK ? 1 : NF][BX][BX + 1];  // x faces: fxs[iw][y][f]
  __shared__ R fys[HANCOCK ? 1 : NF][BX + 1][BX];  // y faces: fys[iw][f][x]
  __shared__ R hring[HRING ? NG : 1][HRING ? NW : 1][HRING ? NSTRIP : 1];
  // the conserved halo pairs of the next plane, loaded straight into LDS
  constexpr bool HPAIR = NDIM == 3 && !HRING && NG == 2 && BX == 16;
  __shared__ __align__(16) double hraw[HPAIR ? NW : 1][HPAIR ? 128 : 1];

  const int b = wg_block(a.per_xcd);
  if (b >= a.nblocks) return;
  __shared__ int nbs[CT ? 27 : 1];        // the block's neighbours (CT)
  if constexpr (CT) {
    if (threadIdx.x < 27) nbs[threadIdx.x] = a.nbr[b * 27 + threadIdx.x];
    __syncthreads();
  }
  FVParams fp = fp0;
  double dq[3], glm_decay;
  // refluxing registers of the block's faces (x-, x+, y-, y+, z-, z+)
  int freg[2 * NDIM];
  if constexpr (AMR) {
    level_params(a, b, fp, dq, glm_decay);
#pragma unroll
    for (int f = 0; f < 2 * NDIM; ++f) freg[f] = a.fregoff ? a.fregoff[b * 2 * NDIM + f] : -1;
  } else {
    dq[0] = a.dq[0]; dq[1] = a.dq[1]; dq[2] = a.dq[2];
    glm_decay = a.glm_decay;
  }
  const int tid = threadIdx.x;
  // lane -> column; the lanes past BX*BX (8^2 and 10^2 blocks) repeat
  // column 0's arithmetic and store nothing of it
  const bool own = FULL || tid < BX * BX;
  const int cid = own ? tid : 0;
  const int tx = cid % BX;
  const int ty = cid / BX;
  const R ch = R(a.ch);
  int crash = 0;
  double dt_maxtot = -1.0e99, dt_cmax = 0.0;  // CFL partials of this lane's column
  const size_t cells = (size_t)BX * BX * a.bnz;
  const size_t boff = (size_t)b * NW * cells;
  // Accesses to a block's planes in this lane's column: the block as a buffer
  // in scalar registers, a scalar offset for plane and variable and this 32-bit
  // lane offset, so that they take no vector address arithmetic.
  const unsigned loff = 8u * (unsigned)(ty * BX + tx);
  const unsigned vbytes = 8u * (unsigned)cells, bbytes = NW * vbytes;
  auto block_ld = [&](const double* p, int k, double* c) {  // plane k of the block at p
    const __amdgpu_buffer_rsrc_t r = block_buffer(p, bbytes);
#pragma unroll
    for (int iw = 0; iw < NW; ++iw) c[iw] = buffer_ld<0>(r, loff, k * (BX * BX * 8) + iw * vbytes);
  };
  auto block_ld_stream = [&](const double* p, int k, double* c) {
    const __amdgpu_buffer_rsrc_t r = block_buffer(p, bbytes);
#pragma unroll
    for (int iw = 0; iw < NF; ++iw) c[iw] = buffer_ld<kNonTemporal>(r, loff, k * (BX * BX * 8) + iw * vbytes);
  };
  auto block_st_stream = [&](double* p, int k, const double* c) {
    const __amdgpu_buffer_rsrc_t r = block_buffer(p, bbytes);
#pragma unroll
    for (int iw = 0; iw < NF; ++iw) buffer_st<kNonTemporal>(c[iw], r, loff, k * (BX * BX * 8) + iw * vbytes);
  };

  // lane's pair and halo cell
  const double* hsrc = nullptr;
  int hel = 0;
  bool hneg = false;
  if constexpr (HPAIR) {
    hsrc = a.src + halo_pair<NW>(a, b, tid & 63);
    hel = halo_elem(a, b, tid & 127, hneg);
  }
  // pairs of plane z into hraw: one 16-byte load per lane and variable; they
  // are there after land_pairs and the barrier behind it.  A caller's array
  // that is not aligned to 16 bytes is read in 8-byte loads.
  auto load_pairs = [&](int z) {
    if constexpr (HPAIR) {
#pragma unroll
      for (int i = 0; i < (NW + 3) / 4; ++i) {
        const int iw = i * 4 + __builtin_amdgcn_readfirstlane(tid >> 6);
        if (iw < NW) {
          const double* p = hsrc + (size_t)z * BX * BX + iw * cells;
          if (a.src_al16) {
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)p,
                                             (__attribute__((address_space(3))) void*)hraw[iw], 16, 0, 0);
          } else {
            hraw[iw][2 * (tid & 63)] = p[0];
            hraw[iw][2 * (tid & 63) + 1] = p[1];
          }
        }
      }
    }
  };
  auto land_pairs = [&]() {
    if constexpr (HPAIR) __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  };
  const int nz = NDIM == 3 ? a.bnz : 1;
  const int z0 = NDIM == 3 ? (int)blockIdx.y * a.zc : 0;  // this workgroup's planes z0 .. z1-1
  const int z1 = NDIM == 3 ? (z0 + a.zc < nz ? z0 + a.zc : nz) : 1;

  // z window (3-D): Wp[m] = primitive plane k-NG+1+m (m < NG, the current
  // plane last), Wc[m] = conserved plane k+1+m as stored (FP64).  The current
  // plane's conserved state is the RK input of comb modes 2 and 3, so the
  // block's own planes are read from HBM once.
  constexpr int NWP = NDIM == 3 ? NG : 1;
  R Wp[NWP][NW];
  double Wc[NWP][NW];
  R fz_carry[NW];
  // primitive planes k-NG+1 .. k+NG of this lane's column
  auto zstencil = [&](R (*Z)[NW]) {
#pragma unroll
    for (int m = 0; m < NG; ++m)
#pragma unroll
      for (int iw = 0; iw < NW; ++iw) Z[m][iw] = Wp[m][iw];
#pragma unroll
    for (int m = 0; m < NG; ++m) prim_of<P, R>(Wc[m], Z[NG + m], fp);
  };
  // the neighbours above and below are the same for all lanes
  int nbz[2] = {0, 0};
  if constexpr (NDIM == 3)
#pragma unroll
    for (int sd = 0; sd < 2; ++sd) nbz[sd] = __builtin_amdgcn_readfirstlane(a.nbr[b * 27 + 13 + (2 * sd - 1) * 9]);
  // conserved plane z of this lane's column, z within NG of the block
  // (locate for a cell outside the block in z alone)
  auto load_plane = [&](int z, double* c) {
    const double* pz = a.src + boff;
    int zz = z;
    bool neg = false;
    if (z < 0 || z >= nz) {
      const int sd = z < 0 ? 0 : 1;
      const int nbk = sd ? nbz[1] : nbz[0];
      if (nbk >= 0) {
        pz = a.src + (size_t)nbk * NW * cells;
        zz = sd ? z - nz : z + nz;
      } else {
        const int t = a.bc[4 + sd];
        zz = t == 2 ? (sd ? nz - 1 : 0) : (sd ? 2 * nz - 1 - z : -1 - z);
        neg = t == 4;
      }
    }
    block_ld(pz, zz, c);
    if (neg)
#pragma unroll
      for (int iw = 0; iw < NW; ++iw) c[iw] = -c[iw];
  };
  R zp[NW];  // primitive plane k+1, the next plane's own after it
  if constexpr (NDIM == 3) {
    load_pairs(z0);
    // prologue: planes z0-NG .. z0+NG-1, halo ring of planes z0 .. z0+NG-1,
    // carried face z0-1/2
#pragma unroll
    for (int m = 0; m < NG; ++m) {
      double c[NW];
      load_plane(z0 + m - NG, c);
      prim_of<P, R>(c, Wp[m], fp);
    }
#pragma unroll
    for (int m = 0; m < NG; ++m) load_plane(z0 + m, Wc[m]);
    prim_of<P, R>(Wc[0], zp, fp);
    if constexpr (HRING) {
      for (int p = z0; p < z0 + NG && p < z1; ++p)
        for (int t = tid; t < NSTRIP; t += NTHREADS) {
          int x, y;
          strip_cell<NG, BX>(t, x, y);
          R w[NW];
          load_prim<P, R, NDIM, BX>(a, fp, b, x, y, p, w);
#pragma unroll
          for (int iw = 0; iw < NW; ++iw) hring[p % NG][iw][t] = w[iw];
        }
    }
    if constexpr (!HANCOCK) {
      R Z[2 * NG][NW];
      zstencil(Z);
      [[maybe_unused]] CtIO io;
      if constexpr (CT) ct.template face_in<RIEM, 2>(a, io, nbs, tx, ty, z0 - 1);
      face_flux<P, R, RIEM, 2, LIM, NG, CT, true>(Z, fp, ch, fz_carry, crash, &io);
    }
    land_pairs();
    if constexpr (HRING || HPAIR) __syncthreads();
  }

  // Plane k in LDS (primitive, with x/y halo); w: this lane's cell.  In 3-D the
  // next plane is staged while this one's flux divergence is formed, which
  // reads the face arrays and registers only: two barriers per plane (with the
  // addresses above in scalar registers and the halo pairs, 256^3 MHD-GLM: FP64
  // 1785 -> 1590 us, mixed 1226 -> 1148 us for the barriers, 1037 -> 1015 us for
  // the addresses).
  auto stage_plane = [&](int k, const R* w) {
    if (own)
#pragma unroll
      for (int iw = 0; iw < NW; ++iw) sp[iw][ty + NG][tx + NG] = w[iw];
    if constexpr (HRING) {
      const int slot = k % NG;
      for (int t = tid; t < NSTRIP; t += NTHREADS) {
        int x, y;
        strip_cell<NG, BX>(t, x, y);
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) sp[iw][y + NG][x + NG] = hring[slot][iw][t];
      }
    } else if constexpr (HPAIR) {
      // halo strips of plane k from the pairs, by alternate wave pairs from
      // plane to plane
      if (((tid >> 7) ^ k) & 1) {
        int x, y;
        strip_cell<NG, BX>(tid & 127, x, y);
        double c[NW];
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) c[iw] = hneg ? -hraw[iw][hel] : hraw[iw][hel];
        R w[NW];
        prim_of<P, R>(c, w, fp);
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) sp[iw][y + NG][x + NG] = w[iw];
      }
    } else {
      // halo strips of plane k (FP64: loaded by alternate wave pairs from
      // plane to plane)
      const int th = std::is_same<R, double>::value && NTHREADS == 256 ? (tid + 128 * (k & 1)) % NTHREADS : tid;
      for (int t = th; t < NHALO; t += NTHREADS) {
        int x, y;
        strip_cell<NG, BX>(t, x, y);
        R w[NW];
        load_prim<P, R, NDIM, BX>(a, fp, b, x, y, k, w);
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) sp[iw][y + NG][x + NG] = w[iw];
      }
    }
  };
  if constexpr (NDIM == 3) stage_plane(z0, zp);

  for (int k = z0; k < z1; ++k) {
    double cons_k[NW];  // wCT of this lane's cell
    double acc[NW];
    // RK base (src/mod_advance.t:251-267), streamed; the combination with
    // the stage input is formed once the base has arrived
    // (the production kernels fuse the stage input's product in 2-D and the
    // base's in 3-D, whatever code surrounds the combination)
    auto rk_init = [&]() {
      if (a.comb_mode == 0) {
        block_ld_stream(a.dst + boff, k, acc);
      } else if (a.comb_mode == 1) {
        block_ld_stream(a.base + boff, k, acc);
      } else if (a.comb_mode == 2) {
        block_ld_stream(a.base + boff, k, acc);
#pragma unroll
        for (int iw = 0; iw < NF; ++iw)
          acc[iw] = kExact ? a.comb_a * acc[iw] + a.comb_b * cons_k[iw]
                           : NDIM == 2 ? fma(a.comb_b, cons_k[iw], a.comb_a * acc[iw])
                                       : fma(a.comb_a, acc[iw], a.comb_b * cons_k[iw]);
      } else {
#pragma unroll
        for (int iw = 0; iw < NF; ++iw) acc[iw] = cons_k[iw];
      }
    };
    if constexpr (NDIM == 3) {
      // advance the window and issue the lookahead plane k+NG
#pragma unroll
      for (int iw = 0; iw < NW; ++iw) cons_k[iw] = Wc[0][iw];
      // fix_small_values: phys_to_primitive checks every cell it converts
      // (src/hd/mod_hd_phys.t:713-715, src/mhd/mod_mhd_phys.t:1750-1753);
      // over the level, the blocks' own cells are every converted cell
      if (SMALLCHK && fp.fix_small && small_cons<P>(cons_k, fp)) crash = 1;
#pragma unroll
      for (int m = 0; m < NG - 1; ++m)
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) Wp[m][iw] = Wp[m + 1][iw];
#pragma unroll
      for (int iw = 0; iw < NW; ++iw) Wp[NG - 1][iw] = zp[iw];
#pragma unroll
      for (int m = 0; m < NG - 1; ++m)
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) Wc[m][iw] = Wc[m + 1][iw];
      load_plane(k + NG, Wc[NG - 1]);
      if constexpr (CT) ct.template cell_out<P, R>(fp, cons_k, Wp[NG - 1], b, tx, ty, k);
    } else {
      block_ld(a.src + boff, k, cons_k);
      if (SMALLCHK && fp.fix_small && small_cons<P>(cons_k, fp)) crash = 1;
      R w[NW];
      prim_of<P, R>(cons_k, w, fp);
      stage_plane(k, w);
    }
    __syncthreads();
    if constexpr (HRING) {
      // halo of plane k+NG into the ring slot just copied out
      if (k + NG < z1) {
        const int slot = k % NG;
        // by the upper waves: the lower ones take the partial face pass
        const int th = NTHREADS == 256 ? (tid + 128) % NTHREADS : tid;
        for (int t = th; t < NSTRIP; t += NTHREADS) {
          int x, y;
          strip_cell<NG, BX>(t, x, y);
          R w[NW];
          load_prim<P, R, NDIM, BX>(a, fp, b, x, y, k + NG, w);
#pragma unroll
          for (int iw = 0; iw < NW; ++iw) hring[slot][iw][t] = w[iw];
        }
      }
    }

    // z neighbours of this lane's cell for the sources and the Hancock
    // predictor: primitive planes k-1 and k+1
    R zm[NW];
    if constexpr (NDIM == 3) {
#pragma unroll
      for (int iw = 0; iw < NW; ++iw) zm[iw] = Wp[NG - 2][iw];
    }
    // extended GLM sources: the gradients of psi and B and the cell's own
    // field, read from the plane before the next one takes its place
    double glm_gp[2], glm_divb, glm_b[P::NDIR];
    auto glm_gradients = [&]() {
      if constexpr (P::GLM) {
        constexpr int S = P::PSI;
        const int cx = tx + NG, cy = ty + NG;
        glm_gp[0] = div_by((double(sp[S][cy][cx + 1]) - double(sp[S][cy][cx - 1])) * 0.5, fp.dx[0], fp.dxinv[0]);
        glm_gp[1] = div_by((double(sp[S][cy + 1][cx]) - double(sp[S][cy - 1][cx])) * 0.5, fp.dx[1], fp.dxinv[1]);
        glm_divb = 0.0;
        glm_divb = glm_divb + 0.5 * (double(sp[P::MAG][cy][cx + 1]) - double(sp[P::MAG][cy][cx - 1])) * fp.dxinv[0];
        glm_divb =
            glm_divb + 0.5 * (double(sp[P::MAG + 1][cy + 1][cx]) - double(sp[P::MAG + 1][cy - 1][cx])) * fp.dxinv[1];
#pragma unroll
        for (int d = 0; d < P::NDIR; ++d) glm_b[d] = double(sp[P::MAG + d][cy][cx]);
      }
    };

    if constexpr (!HANCOCK) {
      // ---- face fluxes of this plane --------------------------------------
      constexpr int NXF = BX * (BX + 1);             // x faces (272 for 16^2)
      constexpr int XSLOTS = (NXF + 63) / 64 * 64;   // padded to a wave multiple
      constexpr int NSLOT = XSLOTS + NXF;            // + the y faces
      // FP64: the waves that take the third, partial pass change from plane
      // to plane, so that the co-resident workgroups' heavy waves spread
      // over the SIMDs (measured 1.6% faster; the FP32 form is not helped)
      const int t0 = std::is_same<R, double>::value ? (tid + 64 * (k & 3)) % NTHREADS : tid;
      // Where one list of x and y faces takes fewer passes of the workgroup than
      // two padded ones (8^2 cross-sections: 3 instead of 4), the y faces are
      // computed as x faces of the stencil with the first two components
      // swapped: the same operations, sums of two terms in the other order.
      // (16^2: 9 wave passes instead of 10, measured no faster.)  HLLD's
      // transverse components are not symmetric in that order.
      constexpr bool SWAP = NDIM == 3 && std::is_same<R, double>::value && !CT && RIEM != RIEM_HLLD &&
                            (2 * NXF + NTHREADS - 1) / NTHREADS < (NSLOT + NTHREADS - 1) / NTHREADS;
      if constexpr (SWAP) {
        for (int t = tid; t < 2 * NXF; t += NTHREADS) {
          const int isy = t >= NXF, u = isy ? t - NXF : t;
          const int r = u / (BX + 1), f = u % (BX + 1);  // row or column, face between f-1 and f
          auto comp = [&](int iw) {
            const int v = P::MHD && iw >= P::MAG ? P::MAG : P::MOM;
            return iw == v ? v + isy : (iw == v + 1 ? v + 1 - isy : iw);
          };
          const R* p = &sp[0][0][0] + (isy ? f * PX + r + NG : (r + NG) * PX + f);
          const int step = isy ? PX : 1;
          R st[2 * NG][NW];
#pragma unroll
          for (int s = 0; s < 2 * NG; ++s)
#pragma unroll
            for (int iw = 0; iw < NW; ++iw) st[s][iw] = p[comp(iw) * (PX * PX) + s * step];
          FVParams fq = fp;
          fq.rdelinv[0] = isy ? fp.rdelinv[1] : fp.rdelinv[0];
          fq.cada3k[0] = isy ? fp.cada3k[1] : fp.cada3k[0];
          R fc[NW];
          face_flux<P, R, RIEM, 0, LIM, NG>(st, fq, ch, fc, crash);
          R* o = isy ? &fys[0][f][r] : &fxs[0][r][f];
#pragma unroll
          for (int iw = 0; iw < NW; ++iw) o[comp(iw) * (BX * (BX + 1))] = fc[iw];
        }
      } else for (int t = t0; t < NSLOT; t += NTHREADS) {
        if (t < NXF) {
          const int y = t / (BX + 1), f = t % (BX + 1);  // face between f-1 and f
          R st[2 * NG][NW];
#pragma unroll
          for (int s = 0; s < 2 * NG; ++s)
#pragma unroll
            for (int iw = 0; iw < NW; ++iw) st[s][iw] = sp[iw][y + NG][f + s];
          R fc[NW];
          [[maybe_unused]] CtIO io;
          if constexpr (CT) ct.template face_in<RIEM, 0>(a, io, nbs, f - 1, y, k);
          face_flux<P, R, RIEM, 0, LIM, NG, CT>(st, fp, ch, fc, crash, &io);
          if constexpr (CT)
            if (f > 0) ct.template face_out<P, R, 0>(io, fc, b, f - 1, y, k);
#pragma unroll
          for (int iw = 0; iw < NF; ++iw) fxs[iw][y][f] = fc[iw];
        } else if (t >= XSLOTS) {
          const int u = t - XSLOTS;
          const int f = u / BX, x = u % BX;  // face between f-1 and f
          R st[2 * NG][NW];
#pragma unroll
          for (int s = 0; s < 2 * NG; ++s)
#pragma unroll
            for (int iw = 0; iw < NW; ++iw) st[s][iw] = sp[iw][f + s][x + NG];
          R fc[NW];
          [[maybe_unused]] CtIO io;
          if constexpr (CT) ct.template face_in<RIEM, 1>(a, io, nbs, x, f - 1, k);
          face_flux<P, R, RIEM, 1, LIM, NG, CT>(st, fp, ch, fc, crash, &io);
          if constexpr (CT)
            if (f > 0) ct.template face_out<P, R, 1>(io, fc, b, x, f - 1, k);
#pragma unroll
          for (int iw = 0; iw < NF; ++iw) fys[iw][f][x] = fc[iw];
        }
      }
      if (HPAIR && k + 1 < z1) load_pairs(k + 1);
      rk_init();
      // z face k+1/2 last, so that the lookahead load has landed
      R fz_new[NW];
      if constexpr (NDIM == 3) {
        R Z[2 * NG][NW];
        zstencil(Z);
        [[maybe_unused]] CtIO io;
        if constexpr (CT) ct.template face_in<RIEM, 2>(a, io, nbs, tx, ty, k);
        face_flux<P, R, RIEM, 2, LIM, NG, CT>(Z, fp, ch, fz_new, crash, &io);
        if constexpr (CT) ct.template face_out<P, R, 2>(io, fz_new, b, tx, ty, k);
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) zp[iw] = Z[NG][iw];
      }
      glm_gradients();
      land_pairs();
      __syncthreads();
      if (NDIM == 3 && k + 1 < z1) stage_plane(k + 1, zp);
      // ---- store_flux (src/mod_fix_conserve.t:597-648): the scaled fluxes
      //      of the block-boundary faces, for refluxing --------------------
      if (AMR && a.freg && own) {
        const size_t nf = (size_t)a.nface;
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) {
          if (tx == 0 && freg[0] >= 0)
            a.freg[freg[0] + iw * nf + ty + BX * k] = dq[0] * double(fxs[iw][ty][0]);
          if (tx == BX - 1 && freg[1] >= 0)
            a.freg[freg[1] + iw * nf + ty + BX * k] = dq[0] * double(fxs[iw][ty][BX]);
          if (ty == 0 && freg[2] >= 0)
            a.freg[freg[2] + iw * nf + tx + BX * k] = dq[1] * double(fys[iw][0][tx]);
          if (ty == BX - 1 && freg[3] >= 0)
            a.freg[freg[3] + iw * nf + tx + BX * k] = dq[1] * double(fys[iw][BX][tx]);
          if constexpr (NDIM == 3) {
            if (k == 0 && freg[4] >= 0) a.freg[freg[4] + iw * nf + tx + BX * ty] = dq[2] * double(fz_carry[iw]);
            if (k == nz - 1 && freg[5] >= 0) a.freg[freg[5] + iw * nf + tx + BX * ty] = dq[2] * double(fz_new[iw]);
          }
        }
      }
      // ---- flux divergence, dimension by dimension (:269-284) ------------
#pragma unroll
      for (int iw = 0; iw < NF; ++iw) {
        acc[iw] = acc[iw] + dq[0] * double(fxs[iw][ty][tx + 1]) - dq[0] * double(fxs[iw][ty][tx]);
        acc[iw] = acc[iw] + dq[1] * double(fys[iw][ty + 1][tx]) - dq[1] * double(fys[iw][ty][tx]);
        if constexpr (NDIM == 3) {
          acc[iw] = acc[iw] + dq[2] * double(fz_new[iw]) - dq[2] * double(fz_carry[iw]);
          fz_carry[iw] = fz_new[iw];
        }
      }
    } else {
      // ---- Hancock predictor (src/mod_finite_volume.t:19-113) -------------
      if (HPAIR && k + 1 < z1) load_pairs(k + 1);
      rk_init();
      if constexpr (NDIM == 3) prim_of<P, R>(Wc[0], zp, fp);
      const R inv_g1 = R(fp.inv_gamma_1);
      auto hancock_dim = [&](auto IDc, const R* wm, const R* w0, const R* wp) {
        constexpr int ID = decltype(IDc)::value;
        R wL[NW], wR[NW];
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) {
          R ldw, rdw;
          dwlimiter<R, LIM>(fp.limiter, w0[iw] - wm[iw], wp[iw] - w0[iw], R(fp.rdelinv[ID]), ldw, rdw);
          wL[iw] = w0[iw] + R(0.5) * ldw;
          wR[iw] = w0[iw] - R(0.5) * rdw;
        }
        R wLC[NW], wRC[NW], fL[NW], fR[NW];
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) { wLC[iw] = wL[iw]; wRC[iw] = wR[iw]; }
        to_cons<P, R>(wLC, inv_g1);
        to_cons<P, R>(wRC, inv_g1);
        phys_flux<P, R, ID>(wRC, wR, ch, fR);
        phys_flux<P, R, ID>(wLC, wL, ch, fL);
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) acc[iw] = acc[iw] + dq[ID] * double(fL[iw] - fR[iw]);
      };
      R wm[NW], w0[NW], wp[NW];
#pragma unroll
      for (int iw = 0; iw < NW; ++iw) {
        wm[iw] = sp[iw][ty + NG][tx + NG - 1];
        w0[iw] = sp[iw][ty + NG][tx + NG];
        wp[iw] = sp[iw][ty + NG][tx + NG + 1];
      }
      hancock_dim(std::integral_constant<int, 0>(), wm, w0, wp);
#pragma unroll
      for (int iw = 0; iw < NW; ++iw) {
        wm[iw] = sp[iw][ty + NG - 1][tx + NG];
        wp[iw] = sp[iw][ty + NG + 1][tx + NG];
      }
      hancock_dim(std::integral_constant<int, 1>(), wm, w0, wp);
      if constexpr (NDIM == 3) hancock_dim(std::integral_constant<int, 2>(), zm, w0, zp);
      glm_gradients();
      land_pairs();
      if constexpr (NDIM == 3) {
        __syncthreads();
        if (k + 1 < z1) stage_plane(k + 1, zp);
      }
    }

    // ---- unphysical values after the flux update (finite_volume
    //      :325-333, hancock :109-111: small_values_method 'error' sets
    //      crash, after which the run stops).  The reconstructed face
    //      states of the TVD limiters lie between their cells' values, so
    //      the face checks of reconstruct_LR (:1213-1216) flag nothing more
    // (hancock checks only after its sources, GLM here or Linde's kernel)
    if constexpr (!(HANCOCK && P::GLM))
      if (!(HANCOCK && a.linde) && SMALLCHK && fp.fix_small && small_cons<P>(acc, fp)) crash = 1;
    // ---- sources: addsource2 -> mhd_add_source (src/mod_source.t:130-160,
    //      src/mhd/mod_mhd_phys.t:4565-4695) -----------------------------
    if constexpr (P::GLM) {
      // add_source_glm src/mhd/mod_mhd_phys.t:5472-5531
      constexpr int S = P::PSI;
      acc[S] = glm_decay * acc[S];
      if (fp.glm_extended) {
        double gp[3] = {glm_gp[0], glm_gp[1], 0.0}, divb = glm_divb;
        const double* bn = glm_b;
        if constexpr (NDIM == 3) {
          gp[2] = div_by((double(zp[S]) - double(zm[S])) * 0.5, fp.dx[2], fp.dxinv[2]);
          divb = divb + 0.5 * (double(zp[P::MAG + 2]) - double(zm[P::MAG + 2])) * fp.dxinv[2];
        }
#pragma unroll
        for (int d = 0; d < NDIM; ++d) acc[P::E] = acc[P::E] - a.qdt * bn[d] * gp[d];
#pragma unroll
        for (int d = 0; d < P::NDIR; ++d) acc[P::MOM + d] = acc[P::MOM + d] - a.qdt * bn[d] * divb;
      }
    }
    // Linde's source (add_source_linde) follows in linde_kernel: div B at
    // the neighbours needs the field beyond this kernel's planes and rim
    // the GLM source checks again (src/mhd/mod_mhd_phys.t:5529)
    if constexpr (P::GLM)
      if (SMALLCHK && fp.fix_small && small_cons<P>(acc, fp)) crash = 1;
    if (own)
      block_st_stream(a.dst + boff, k, acc);
    if constexpr (CFL)
      if (a.dt_part) cfl_cell<P>(acc, fp, dt_maxtot, dt_cmax);
  }
  if (crash) *a.crash = 1;
  if constexpr (CFL) {
    if (a.dt_part) {
      // block max: wave64 shuffles, then the 4 waves through LDS
      for (int off = 32; off > 0; off >>= 1) {
        dt_maxtot = fmax(dt_maxtot, __shfl_xor(dt_maxtot, off, 64));
        dt_cmax = fmax(dt_cmax, __shfl_xor(dt_cmax, off, 64));
      }
      __shared__ double dtr[2][NTHREADS / 64];
      if ((tid & 63) == 0) { dtr[0][tid >> 6] = dt_maxtot; dtr[1][tid >> 6] = dt_cmax; }
      __syncthreads();
      if (tid == 0) {
        double m = dtr[0][0], c = dtr[1][0];
        for (int i = 1; i < NTHREADS / 64; ++i) { m = fmax(m, dtr[0][i]); c = fmax(c, dtr[1][i]); }
        a.dt_part[2 * b] = m;
        a.dt_part[2 * b + 1] = c;
      }
    }
  }
}

}  // namespace FV_NS
