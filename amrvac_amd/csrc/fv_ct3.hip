// Constrained transport on a uniform periodic 3-D level (ideal MHD, ndir = 3,
// staggered face field, typedivbfix = 'ct').
//
// A stage is three launches; what one hands to the next lies in per-block
// arrays in HBM, indexed by the block's own cells.  A face or edge quantity
// belongs to the cell whose upper face or edge it is, is formed by that cell's
// block alone and read from there by the neighbours: the level is periodic, so
// every face is some cell's upper face.
//   sweep_kernel       (fv_sweep.h) marches through the planes as the stage
//                      without a face field does: all faces' fluxes
//                      (finite_volume src/mod_finite_volume.t:183-190 with
//                      mhd_modify_wLR :6338-6345), the update of density,
//                      momentum and energy, and for the edge fields the fluxes
//                      of the two transverse field components, the face data
//                      of mhd_get_ct_velocity_* (src/mhd/mod_mhd_phys.t:
//                      3261-3326) and, for uct_contact, b x v at cell centres
//                      (FP64);
//   ct3_edge_kernel    one thread per edge: the edge electric field times qdt
//                      and the edge length (mhd_update_faces_average /
//                      _contact / _hll :6951-7479), the edge along idir at the
//                      upper corner of each cell in the two other directions;
//   ct3_update_kernel  the faces from the circulation of the edge fields (a
//                      plane's lower ones in the same operations as their
//                      owner, which stores them) and the cell field from the
//                      faces (mhd_face_to_center :7586-7648).
// The new upper faces go to ws_new, which then replaces psb's face field.
//
// Bound by memory: the primitive state, all fluxes on every halo face and the
// update as launches of their own moved 1.9 times as much (128 x 128 x 256,
// uct_contact, FP64: a stage 1580 -> 660 us).
//
// Face field layout: ws[nb][3][16][16][16], component d of cell (i, j, k) is
// the field on the upper d face of that cell.
#include "fv_ct_common.h"

namespace FV_NS {
namespace {

using fvc::BX;
constexpr size_t C3 = (size_t)BX * BX * BX;  // cells of a block

// scratch per block, in doubles: transverse field fluxes [3][2][C3] (in the
// face precision, whose values they are), face data [3][4][C3], b x v [3][C3],
// edge fields [3][C3]
constexpr size_t kCt3Flux = 6 * C3, kCt3Data = 12 * C3, kCt3Ecc = 3 * C3, kCt3Edges = 3 * C3;
// face data of the edge fields (FP64): the face velocity of uct_contact, the
// signal speeds and velocity averages of uct_hll
constexpr int VN = 0, CBMIN = 0, CBMAX = 1, VB1 = 2, VB2 = 3;

__device__ __forceinline__ size_t cidx(int x, int y, int z) { return ((size_t)z * BX + y) * BX + x; }

// A cell within a block of the block's own cells, by its owner.  nbs: the
// block's 27 neighbours in LDS, which cost a lane less than a look into the
// level's table before each load (128 x 128 x 256: edge kernel 155 -> 129 us, update 204 -> 105); on the
// periodic level all exist.
struct Owner {
  int b;
  size_t c;
  __device__ __forceinline__ Owner(const int* nbs, int x, int y, int z) {
    const int sx = x < 0 ? -1 : (x >= BX ? 1 : 0), sy = y < 0 ? -1 : (y >= BX ? 1 : 0);
    const int sz = z < 0 ? -1 : (z >= BX ? 1 : 0);
    b = nbs[13 + 9 * sz + 3 * sy + sx];
    c = cidx(x - sx * BX, y - sy * BX, z - sz * BX);
  }
};
__device__ __forceinline__ void load_neighbours(const SweepArgs& a, int b, int* nbs) {
  if (threadIdx.x < 27) nbs[threadIdx.x] = a.nbr[(size_t)b * 27 + threadIdx.x];
}

__device__ __forceinline__ double ws_at3(const double* ws, const Owner& o, int d) {
  return ws[((size_t)o.b * 3 + d) * C3 + o.c];
}

// the face field a slot combination gives (the RK initial state of psb)
__device__ __forceinline__ double ws_comb3(const SweepArgs& a, const CtArgs& t, int mode, const Owner& o, int d) {
  if (mode == 0) return ws_at3(t.ws_dst, o, d);
  if (mode == 1) return ws_at3(t.ws_base, o, d);
  if (mode == 2) return a.comb_a * ws_at3(t.ws_base, o, d) + a.comb_b * ws_at3(t.ws_src, o, d);
  return ws_at3(t.ws_src, o, d);
}

// flux of B_comp through the d faces of a block, in the face precision
template <class R>
__device__ __forceinline__ R* flux_ptr(const CtArgs& t, int b, int d, int comp) {
  return reinterpret_cast<R*>(t.faces + (size_t)b * kCt3Flux) + (size_t)(2 * d + (comp == (d + 1) % 3 ? 0 : 1)) * C3;
}
__device__ __forceinline__ double* data_ptr(const CtArgs& t, int b, int d, int k) {
  return t.data + (size_t)b * kCt3Data + (size_t)(4 * d + k) * C3;
}

// the sweep's side: cell (x, y, z) owns the face
struct Ct3Sweep : CtArgs {
  template <int RIEM, int ID>
  __device__ __forceinline__ void face_in(const SweepArgs& a, CtIO& io, const int* nbs, int x, int y, int z) const {
    const Owner o(nbs, x, y, z);
    io.bn = ws_at3(ws_src, o, ID);
    if constexpr (RIEM == RIEM_HLLD)
      io.bx = bx_mode < 0 ? ws_at3(ws_block, o, ID) : ws_comb3(a, *this, bx_mode, o, ID);
  }
  template <class P, class R, int ID>
  __device__ __forceinline__ void face_out(const CtIO& io, const R* f, int b, int x, int y, int z) const {
    constexpr int iN = (ID + 1) % 3, iE = (ID + 2) % 3;
    const size_t c = cidx(x, y, z);
    flux_ptr<R>(*this, b, ID, iN)[c] = f[P::MAG + iN];
    flux_ptr<R>(*this, b, ID, iE)[c] = f[P::MAG + iE];
    if (ct == CT_CONTACT) data_ptr(*this, b, ID, VN)[c] = 0.5 * (io.vL[ID] + io.vR[ID]);
    if (ct == CT_HLL) {
      const double cbmax = io.cmax > 0.0 ? io.cmax : 0.0;
      const double cbmin = tvdlf ? cbmax : (-io.cmin > 0.0 ? -io.cmin : 0.0);
      data_ptr(*this, b, ID, CBMIN)[c] = cbmin;
      data_ptr(*this, b, ID, CBMAX)[c] = cbmax;
      data_ptr(*this, b, ID, VB1)[c] = (cbmax * io.vL[iN] + cbmin * io.vR[iN]) / (cbmax + cbmin);
      // the second average takes vbarRC(:,idim,1), as the reference does
      data_ptr(*this, b, ID, VB2)[c] = (cbmax * io.vL[iE] + cbmin * io.vR[iN]) / (cbmax + cbmin);
    }
  }
  // ECC = b x v (components x, y, z) of the FP64 primitive state
  template <class P, class R>
  __device__ __forceinline__ void cell_out(const FVParams& fp, const double* cons, const R* prim, int b, int x, int y,
                                           int z) const {
    if (ct != CT_CONTACT) return;
    double w[P::NW];
    if constexpr (std::is_same<R, double>::value) {
#pragma unroll
      for (int iw = 0; iw < P::NW; ++iw) w[iw] = prim[iw];
    } else {
      to_prim<P>(cons, w, fp);
    }
    double* e = ecc + (size_t)b * kCt3Ecc + cidx(x, y, z);
    const int b1 = P::MAG, b2 = P::MAG + 1, b3 = P::MAG + 2, m1 = P::MOM, m2 = P::MOM + 1, m3 = P::MOM + 2;
    e[0 * C3] = w[b2] * w[m3] - w[b3] * w[m2];
    e[1 * C3] = w[b3] * w[m1] - w[b1] * w[m3];
    e[2 * C3] = w[b1] * w[m2] - w[b2] * w[m1];
  }
};

// blockIdx.x: plane, blockIdx.y: edge direction idir, blockIdx.z: block; the
// edge at the upper (idim1, idim2) corner of each cell, with (idim1, idim2,
// idir) cyclic (lvc = 1)
template <class P, class R, int LIM>
__global__ void __launch_bounds__(fvc::NTHREADS) ct3_edge_kernel(SweepArgs a, CtArgs t, FVParams fp) {
  __shared__ int nbs[27];
  const int idir = blockIdx.y, b = blockIdx.z, q = threadIdx.x;
  load_neighbours(a, b, nbs);
  __syncthreads();
  const int c[3] = {q % BX, q / BX, (int)blockIdx.x};
  const int idim1 = (idir + 1) % 3, idim2 = (idir + 2) % 3;
  int e1[3] = {0, 0, 0}, e2[3] = {0, 0, 0};
  e1[idim1] = 1;
  e2[idim2] = 1;
  // the cell s1 up along idim1 and s2 up along idim2
  auto at = [&](int s1, int s2) {
    return Owner(nbs, c[0] + s1 * e1[0] + s2 * e2[0], c[1] + s1 * e1[1] + s2 * e2[1], c[2] + s1 * e1[2] + s2 * e2[2]);
  };
  // FM(cell, component, face direction): flux of B_component through the
  // upper face of the cell
  auto FM = [&](const Owner& o, int comp, int fd) { return double(flux_ptr<R>(t, o.b, fd, comp)[o.c]); };
  auto FQ = [&](const Owner& o, int k, int fd) { return data_ptr(t, o.b, fd, k)[o.c]; };
  double e;
  if (t.ct != CT_HLL) {
    const Owner o00 = at(0, 0), o10 = at(1, 0), o01 = at(0, 1);
    const double fy0 = FM(o00, idim1, idim2), fy1 = FM(o10, idim1, idim2);
    const double fx0 = FM(o00, idim2, idim1), fx1 = FM(o01, idim2, idim1);
    e = 0.25 * (fy0 + fy1 - fx0 - fx1);
    if (t.ct == CT_CONTACT) {
      auto E = [&](const Owner& o) { return t.ecc[(size_t)o.b * kCt3Ecc + (size_t)idir * C3 + o.c]; };
      const double E00 = E(o00), E10 = E(o10), E01 = E(o01), E11 = E(at(1, 1));
      const double v10 = FQ(o00, VN, idim1), v11 = FQ(o01, VN, idim1);
      const double v20 = FQ(o00, VN, idim2), v21 = FQ(o10, VN, idim2);
      // first pair: idim2-face fluxes of B_idim1 at c, c + e1
      {
        const double ELc = fy0 - E00, ELp = fy1 - E10;
        const double ERc = fy0 - E01, ERp = fy1 - E11;
        double ELC, ERC;
        if (v10 > 0.0) ELC = ELc;
        else if (v10 < 0.0) ELC = ELp;
        else ELC = 0.5 * (ELc + ELp);
        if (v11 > 0.0) ERC = ERc;
        else if (v11 < 0.0) ERC = ERp;
        else ERC = 0.5 * (ERc + ERp);
        e = e + 0.25 * (ELC + ERC);
      }
      // second pair: idim1-face fluxes of B_idim2 at c, c + e2
      {
        const double ELc = -fx0 - E00, ELp = -fx1 - E01;
        const double ERc = -fx0 - E10, ERp = -fx1 - E11;
        double ELC, ERC;
        if (v20 > 0.0) ELC = ELc;
        else if (v20 < 0.0) ELC = ELp;
        else ELC = 0.5 * (ELc + ELp);
        if (v21 > 0.0) ERC = ERc;
        else if (v21 < 0.0) ERC = ERp;
        else ERC = 0.5 * (ERc + ERp);
        e = e + 0.25 * (ELC + ERC);
      }
    }
    e = e * a.qdt * fp.dx[idir];
  } else {
    const double r1 = fp.rdelinv[idim1], r2 = fp.rdelinv[idim2];
    double vtL1, vtR1, vtL2, vtR2, bL1, bR1, bL2, bR2;
    const Owner o00 = at(0, 0), o0m = at(0, -1), o01 = at(0, 1), o02 = at(0, 2), om0 = at(-1, 0), o10 = at(1, 0),
              o20 = at(2, 0);
    // vbarC(idim1 faces, 1) along idim2 -> vtil(:, 2)
    ct_recon<LIM>(fp, r2, FQ(o0m, VB1, idim1), FQ(o00, VB1, idim1), FQ(o01, VB1, idim1), FQ(o02, VB1, idim1), vtL2,
                  vtR2);
    // vbarC(idim2 faces, 2) along idim1 -> vtil(:, 1)
    ct_recon<LIM>(fp, r1, FQ(om0, VB2, idim2), FQ(o00, VB2, idim2), FQ(o10, VB2, idim2), FQ(o20, VB2, idim2), vtL1,
                  vtR1);
    // face field of the stage input: B_idim1 along idim2, B_idim2 along idim1
    auto W = [&](const Owner& o, int comp) { return ws_at3(t.ws_src, o, comp); };
    ct_recon<LIM>(fp, r2, W(o0m, idim1), W(o00, idim1), W(o01, idim1), W(o02, idim1), bL1, bR1);
    ct_recon<LIM>(fp, r1, W(om0, idim2), W(o00, idim2), W(o10, idim2), W(o20, idim2), bL2, bR2);
    auto mx = [](double u, double v) { return u > v ? u : v; };
    const double cm1 = mx(FQ(o01, CBMIN, idim1), FQ(o00, CBMIN, idim1));
    const double cp1 = mx(FQ(o01, CBMAX, idim1), FQ(o00, CBMAX, idim1));
    const double cm2 = mx(FQ(o10, CBMIN, idim2), FQ(o00, CBMIN, idim2));
    const double cp2 = mx(FQ(o10, CBMAX, idim2), FQ(o00, CBMAX, idim2));
    e = -(cp1 * vtL1 * bL2 + cm1 * vtR1 * bR2 - cp1 * cm1 * (bR2 - bL2)) / (cp1 + cm1) +
        (cp2 * vtL2 * bL1 + cm2 * vtR2 * bR1 - cp2 * cm2 * (bR1 - bL1)) / (cp2 + cm2);
    e = a.qdt * fp.dx[idir] * e;
  }
  t.edges[(size_t)b * kCt3Edges + (size_t)idir * C3 + cidx(c[0], c[1], c[2])] = e;
}

// one workgroup per plane (blockIdx.x) of a block (blockIdx.y), one lane per
// cell: the plane's edge fields with the lower neighbours', then its faces with
// the lower ones, go through LDS
template <class P>
__global__ void __launch_bounds__(fvc::NTHREADS) ct3_update_kernel(SweepArgs a, CtArgs t, FVParams fp) {
  constexpr int B1 = BX + 1;
  static_assert(BX * BX == fvc::NTHREADS, "one lane per cell of a plane");
  __shared__ double ez[B1][B1];                     // E_z at (x, y), each from -1
  __shared__ double ey[2][BX][B1], ex[2][B1][BX];   // E_y at (x, y), E_x at (x, y) of planes k-1 and k
  __shared__ double fx[BX][B1], fy[B1][BX];         // new x faces from x = -1, new y faces from y = -1
  __shared__ int nbs[27];
  const int b = blockIdx.y, k = blockIdx.x, tid = threadIdx.x;
  load_neighbours(a, b, nbs);
  __syncthreads();
  auto EF = [&](int idir, int x, int y, int z) {
    const Owner o(nbs, x, y, z);
    return t.edges[(size_t)o.b * kCt3Edges + (size_t)idir * C3 + o.c];
  };
  for (int q = tid; q < B1 * B1; q += fvc::NTHREADS) ez[q / B1][q % B1] = EF(2, q % B1 - 1, q / B1 - 1, k);
  for (int q = tid; q < BX * B1; q += fvc::NTHREADS)
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      ey[m][q / B1][q % B1] = EF(1, q % B1 - 1, q / B1, k - 1 + m);
      ex[m][q / BX][q % BX] = EF(0, q % BX, q / BX - 1, k - 1 + m);
    }
  __syncthreads();
  const double sC[3] = {fp.dx[1] * fp.dx[2], fp.dx[0] * fp.dx[2], fp.dx[0] * fp.dx[1]};
  // the new field on the upper d face of a cell; circulation: the terms in the
  // order of idim2, idir ascending, with the sign lvc(d, idim2, idir)
  for (int q = tid; q < BX * B1; q += fvc::NTHREADS) {
    {
      const int f = q % B1, y = q / B1;
      double c = 0.0;
      c = c + (ez[y + 1][f] - ez[y][f]);
      c = c - (ey[1][y][f] - ey[0][y][f]);
      fx[y][f] = ws_comb3(a, t, a.comb_mode, Owner(nbs, f - 1, y, k), 0) - c / sC[0];
    }
    {
      const int x = q % BX, f = q / BX;
      double c = 0.0;
      c = c - (ez[f][x + 1] - ez[f][x]);
      c = c + (ex[1][f][x] - ex[0][f][x]);
      fy[f][x] = ws_comb3(a, t, a.comb_mode, Owner(nbs, x, f - 1, k), 1) - c / sC[1];
    }
  }
  const int i = tid % BX, j = tid / BX;
  double fz[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    double c = 0.0;
    c = c + (ey[m][j][i + 1] - ey[m][j][i]);
    c = c - (ex[m][j + 1][i] - ex[m][j][i]);
    fz[m] = ws_comb3(a, t, a.comb_mode, Owner(nbs, i, j, k - 1 + m), 2) - c / sC[2];
  }
  __syncthreads();
  const size_t cell = cidx(i, j, k);
  const double up[3] = {fx[j][i + 1], fy[j + 1][i], fz[1]}, lo[3] = {fx[j][i], fy[j][i], fz[0]};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    t.ws_new[((size_t)b * 3 + d) * C3 + cell] = up[d];
    a.dst[((size_t)b * P::NW + P::MAG + d) * C3 + cell] = 0.5 / sC[d] * (up[d] * sC[d] + lo[d] * sC[d]);
  }
}

template <class P, int RIEM, int LIM>
hipError_t launch_ct3_lim(int mixed, const SweepArgs& a, const Ct3Sweep& t, const FVParams& fp, hipStream_t s) {
  const dim3 ge(BX, 3, a.nblocks), gu(BX, a.nblocks);
  const dim3 gs = sweep_grid(a, 8 * a.per_xcd), th(fvc::NTHREADS);
  if (mixed) {
    if constexpr (kExact) return hipErrorInvalidValue;  // the bit-reproducible build is FP64 only
    else {
      hipLaunchKernelGGL((sweep_kernel<P, float, RIEM, LIM, 2, false, BX, Ct3Sweep>), gs, th, 0, s, a, fp, t);
      hipLaunchKernelGGL((ct3_edge_kernel<P, float, LIM>), ge, th, 0, s, a, t, fp);
    }
  } else {
    hipLaunchKernelGGL((sweep_kernel<P, double, RIEM, LIM, 2, false, BX, Ct3Sweep>), gs, th, 0, s, a, fp, t);
    hipLaunchKernelGGL((ct3_edge_kernel<P, double, LIM>), ge, th, 0, s, a, t, fp);
  }
  hipLaunchKernelGGL((ct3_update_kernel<P>), gu, th, 0, s, a, t, fp);
  return hipGetLastError();
}

template <class P, int RIEM>
hipError_t launch_ct3_riem(int mixed, int lim, const SweepArgs& a, const Ct3Sweep& t, const FVParams& fp,
                           hipStream_t s) {
  switch (lim) {
    case LIM_MINMOD: return launch_ct3_lim<P, RIEM, LIM_MINMOD>(mixed, a, t, fp, s);
    case LIM_VANLEER: return launch_ct3_lim<P, RIEM, LIM_VANLEER>(mixed, a, t, fp, s);
    case LIM_CADA3: return launch_ct3_lim<P, RIEM, LIM_CADA3>(mixed, a, t, fp, s);
    default: return launch_ct3_lim<P, RIEM, 0>(mixed, a, t, fp, s);
  }
}

using P3 = Phys<3, 3, true, DIVB_NONE>;

}  // namespace

// one constrained-transport stage in 3-D (ideal MHD, ndir = 3, 16^3 blocks,
// TVD limiters; mixed: FP32 reconstruction and Riemann solver, FP64 state,
// face field and edge fields).  scratch: ct3_scratch_doubles(nblocks)
// doubles.
hipError_t launch_ct3_stage(int mixed, int riem, int lim, int ct, const fvc::SweepArgs& a, const double* ws_src,
                            const double* ws_base, const double* ws_dst, const double* ws_block, int bx_mode,
                            double* scratch, double* ws_new, const fvc::FVParams& fp, hipStream_t s) {
  if (a.bx != BX || a.bnz != BX) return hipErrorInvalidValue;
  Ct3Sweep t{};
  t.ws_src = ws_src;
  t.ws_base = ws_base;
  t.ws_dst = ws_dst;
  t.ws_block = ws_block;
  t.bx_mode = bx_mode;
  const size_t nb = (size_t)a.nblocks;
  t.faces = scratch;
  t.data = scratch + nb * kCt3Flux;
  t.ecc = t.data + nb * kCt3Data;
  t.edges = t.ecc + nb * kCt3Ecc;
  t.ws_new = ws_new;
  t.ct = ct;
  t.tvdlf = riem == RIEM_TVDLF;
  switch (riem) {
    case RIEM_HLL: return launch_ct3_riem<P3, RIEM_HLL>(mixed, lim, a, t, fp, s);
    case RIEM_TVDLF: return launch_ct3_riem<P3, RIEM_TVDLF>(mixed, lim, a, t, fp, s);
    case RIEM_HLLC: return launch_ct3_riem<P3, RIEM_HLLC>(mixed, lim, a, t, fp, s);
    case RIEM_HLLD: return launch_ct3_riem<P3, RIEM_HLLD>(mixed, lim, a, t, fp, s);
    default: return hipErrorInvalidValue;
  }
}

size_t ct3_scratch_doubles(int nblocks) {
  return (size_t)nblocks * (kCt3Flux + kCt3Data + kCt3Ecc + kCt3Edges);
}

}  // namespace FV_NS
