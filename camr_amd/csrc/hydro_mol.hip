// hydro_mol.hip -- the method of lines' hydro source in four launches.
//
//   k_mol_prim   hydro_ctoprim of Sborder into compact primitives
//   k_mol_divu   nodal divergence
//   k_mol_xy     slopes, face states, Riemann solves and adjust_fluxes of the
//                x and y faces, their share of every cell's divergence
//   k_mol_z      the same of z, and the update
//
// The stage-by-stage kernels (k_mol_face and k_update, which per-box calls
// and levels with flux registers run) write 12 values per face and read them
// back: 344 of the 689 us of a 128^3 source in the update and the stores.
// Here no face value reaches memory: 595 us, 293 of them x and y, 182 z (at
// four waves per SIMD neither the rate of memory nor of the VALUs, a wave
// waits half its time).  All three directions in one launch, marching in z,
// need 256 VGPRs: 577 us at two waves per SIMD.
// The arithmetic per face and cell is theirs (mol_slopes, mol_face_state,
// face_flux, adjust_face_jump, hydro_update's order), hence the same bits.
#include "hydro_mol.h"
#include "hydro_fused.h"
#include "hydro_kernels.h"

namespace camr {

namespace {


// Box of block w from the prefix blk[0..n]; lb its block within the box.
__device__ __forceinline__ int mol_box(const int *blk, int n, int w, int &lb) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (blk[mid] <= w) lo = mid;
        else hi = mid - 1;
    }
    lb = w - blk[lo];
    return lo;
}

// The logical block of this one: XCD x (hardware block w runs on w % 8) owns a
// contiguous run of them, so that tiles beside each other share an L2.
__device__ __forceinline__ int xcd_block() {
    const unsigned n = gridDim.x, w = blockIdx.x, q = n / kXCD, r = n % kXCD, x = w % kXCD;
    return (int)(x * q + (x < r ? x : r) + w / kXCD);
}

__global__ void __launch_bounds__(kBlock)
k_mol_prim(const MolBox *tab, const int *blk, int n, HydroConst hc, int *status) {
    int lb;
    const MolBox &B = tab[mol_box(blk, n, (int)blockIdx.x, lb)];
    int i, j, k;
    if (!range_point(range_of(grow(B.bx, CAMR_NGROW)), (int64_t)lb * kBlock + threadIdx.x, i, j, k))
        return;
    const CView u = cview(B.Lu, B.u, NVAR);
    const unsigned vu = B.Lu.off(i, j, k);
    double v[NVAR], o[NQC], e;
#pragma unroll
    for (int c = 0; c < NVAR; ++c) v[c] = u.ld(vu, c);
    if (!prim_compact(v, o, e, hc, status)) return;
    const CView q = cview(B.L, B.q, NQC);
    const unsigned vq = B.L.off(i, j, k);
#pragma unroll
    for (int c = 0; c < NQC; ++c) q.st(vq, c, o[c]);
}

__global__ void __launch_bounds__(kBlock)
k_mol_divu(const MolBox *tab, const int *blk, int n, HydroConst hc) {
    int lb;
    const MolBox &B = tab[mol_box(blk, n, (int)blockIdx.x, lb)];
    int i, j, k;
    if (!range_point(range_of(nodes(nodes(nodes(B.bx, 0), 1), 2)),
                     (int64_t)lb * kBlock + threadIdx.x, i, j, k))
        return;
    const CView q = cview(B.L, B.q, NQC), d = cview(B.L, B.divu, 1);
    d.st(B.L.off(i, j, k), 0, divu_node(q, i, j, k, hc));
}

// The state that the cell at offset v hands to its low and high face of
// direction D, from its own and its two neighbours' primitives.
template <int D>
__device__ __forceinline__ void mol_cell_states(const CView &q, unsigned v, unsigned sd,
                                                const double *c, double cc, const HydroConst &hc,
                                                double *lo, double *hi) {
    double m[NS], p[NS], dq[NMS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        m[s] = q.ld(v - sd, s);
        p[s] = q.ld(v + sd, s);
    }
    mol_slopes(D, m, c, p, cc, hc.plm_iorder, hc.small_dens, dq);
    mol_face_state(D, 1.0, c, dq, cc, &p[SY], hc.small_dens, hc.small_pres, hi);
    mol_face_state(D, -1.0, c, dq, cc, &c[SY], hc.small_dens, hc.small_pres, lo);
}

// What adjust_fluxes reads at the low D-face of the cell at (offset v of q, vu
// of Sborder): the sum of the face's nodal divergences and the jump of U.
template <int D>
__device__ __forceinline__ double mol_jump(const CView &u, const CView &dv, unsigned v, unsigned vu,
                                           const Canon &L, const Canon &Lu, double *du) {
    const unsigned s1 = D == 0 ? L.sy() : 8u, s2 = D == 2 ? L.sy() : L.sz();
    const unsigned su = D == 0 ? 8u : (D == 1 ? Lu.sy() : Lu.sz());
#pragma unroll
    for (int n = 0; n < NVAR; ++n) du[n] = n == UTEMP ? 0.0 : u.ld(vu, n) - u.ld(vu - su, n);
    return dv.ld(v, 0) + dv.ld(v + s1, 0) + dv.ld(v + s2, 0) + dv.ld(v + s1 + s2, 0);
}

// Flux of that face from the states on both sides: f the NVAR fluxes without
// UTEMP's 0 (compact order FR..FY) times the area, g Godunov (u, p).
template <int D>
__device__ __forceinline__ void mol_face(double dsum, const double *du, int idx, double *ql,
                                         double *qr, const FaceAux &a, const HydroConst &hc,
                                         double area, double *f, double *g) {
    int mut;
    face_flux(D, idx, hc, ql, qr, a, f, g, &mut);
    double fu[NVAR];
    fu[URHO] = f[FR]; fu[UMX] = f[FMX]; fu[UMY] = f[FMY]; fu[UMZ] = f[FMZ];
    fu[UEDEN] = f[FE]; fu[UEINT] = f[FEI]; fu[UTEMP] = 0.0;
#pragma unroll
    for (int s = 0; s < NSPEC; ++s) fu[UFS + s] = f[FY + s];
    adjust_face_jump<D>(fu, dsum, du, idx, area, hc);
    f[FR] = fu[URHO]; f[FMX] = fu[UMX]; f[FMY] = fu[UMY]; f[FMZ] = fu[UMZ];
    f[FE] = fu[UEDEN]; f[FEI] = fu[UEINT];
#pragma unroll
    for (int s = 0; s < NSPEC; ++s) f[FY + s] = fu[UFS + s];
}

// One direction of a tile: LDS slot t of a thread is its cell's, slot t - s
// the cell below's in direction D.  A thread forms its cell's states once,
// hands the upper one to the thread above, solves the cell's low face with
// the one it is handed, and hands that flux to the thread below; then
// part[0..NF) += low flux - high flux and pp = the cell's pdivu term, whose
// sums go in hydro_update's order (FIRST: they start here).
//   state: the cell takes part;  face: its low face is solved;  out: both of
//   its faces are.  Every thread of the block calls.
constexpr int kMolSlots = NS + 2;
static_assert(NF == NS && NG == 2, "states and fluxes share the LDS slots");
template <int D, bool FIRST>
__device__ __forceinline__ void mol_dir(double *sh, int t, int s, bool state, bool face, bool out,
                                        const CView &q, const CView &u, const CView &dv,
                                        const Canon &L, const Canon &Lu, int i, int j, int k,
                                        const HydroConst &hc, double area, double *part,
                                        double &pp) {
    const unsigned v = L.off(i, j, k), vu = Lu.off(i, j, k);
    double lo[NS], f[NF], g[NG];
    FaceAux a;
    a.gam_l = a.gam_r = kGamma;
    if (state) {
        double c[NS], hi[NS];
#pragma unroll
        for (int n = 0; n < NS; ++n) c[n] = q.ld(v, n);
        a.c_r = q.ld(v, SC);
        a.csml_r = q.ld(v, SCS);
        mol_cell_states<D>(q, v, D == 0 ? 8u : (D == 1 ? L.sy() : L.sz()), c, a.c_r, hc, lo, hi);
#pragma unroll
        for (int n = 0; n < NS; ++n) sh[n * kBlock + t] = hi[n];
        sh[NS * kBlock + t] = a.c_r;
        sh[(NS + 1) * kBlock + t] = a.csml_r;
    }
    double du[NVAR], ds = 0.0;
    if (face) ds = mol_jump<D>(u, dv, v, vu, L, Lu, du);
    __syncthreads();
    if (face) {
        double ql[NS];
#pragma unroll
        for (int n = 0; n < NS; ++n) ql[n] = sh[n * kBlock + t - s];
        a.c_l = sh[NS * kBlock + t - s];
        a.csml_l = sh[(NS + 1) * kBlock + t - s];
        mol_face<D>(ds, du, D == 0 ? i : (D == 1 ? j : k), ql, lo, a, hc, area, f, g);
    }
    __syncthreads();
    if (face) {
#pragma unroll
        for (int n = 0; n < NF; ++n) sh[n * kBlock + t] = f[n];
        sh[NF * kBlock + t] = g[GUN];
        sh[(NF + 1) * kBlock + t] = g[GP];
    }
    __syncthreads();
    if (out) {
        const double *h = sh + t + s;
#pragma unroll
        for (int n = 0; n < NF; ++n)
            part[n] = FIRST ? f[n] - h[n * kBlock] : part[n] + f[n] - h[n * kBlock];
        const double x = (h[(NF + 1) * kBlock] + g[GP]) * (h[NF * kBlock] * area - g[GUN] * area);
        pp = FIRST ? x : pp + x;
    }
}

// Where compact component n of a cell's sums is kept in dS/dt between the two
// kernels below (the pdivu sum in UTEMP's place).
__device__ __forceinline__ constexpr int mol_comp(int n) {
    return n == FR ? URHO : n == FMX ? UMX : n == FMY ? UMY : n == FMZ ? UMZ : n == FE ? UEDEN
         : n == FEI ? UEINT : UFS + (n - FY);
}

// x and y: a block owns a tile of w x h cells of a plane, one thread each;
// the inner (w - 2) x (h - 2) cells' sums go to dS/dt.
__global__ void __launch_bounds__(kBlock, 3)
k_mol_xy(const MolBox *tab, const int *blk, int nbox, HydroConst hc) {
    __shared__ double sh[kMolSlots * kBlock];
    int lb;
    const MolBox &B = tab[mol_box(blk, nbox, xcd_block(), lb)];
    const Box bx = B.bx;
    const int w = B.w, h = B.h, t = (int)threadIdx.x;
    const int bz = lb / (B.ntx * B.nty), r = lb - bz * B.ntx * B.nty;
    const int by = r / B.ntx, bxi = r - by * B.ntx;
    const int ty = t / w, tx = t - ty * w;
    const int i = bx.lo[0] - 1 + bxi * (w - 2) + tx, j = bx.lo[1] - 1 + by * (h - 2) + ty;
    const int k = bx.lo[2] + bz;
    const bool live = ty < h && i <= bx.hi[0] + 1 && j <= bx.hi[1] + 1;
    const bool inx = live && i >= bx.lo[0] && i <= bx.hi[0];
    const bool iny = live && j >= bx.lo[1] && j <= bx.hi[1];
    const bool out = inx && iny && tx > 0 && tx < w - 1 && ty > 0 && ty < h - 1;
    const CView q = cview(B.L, B.q, NQC), u = cview(B.Lu, B.u, NVAR), dv = cview(B.L, B.divu, 1);
    double part[NF], pp;
    // (the rim's rows have no part in x, its columns none in y)
    const bool row = iny && ty > 0 && ty < h - 1, col = inx && tx > 0 && tx < w - 1;
    mol_dir<0, true>(sh, t, 1, row, row && tx > 0 && i >= bx.lo[0], out, q, u, dv, B.L, B.Lu, i, j,
                     k, hc, hc.dx[1] * hc.dx[2], part, pp);
    __syncthreads();
    mol_dir<1, false>(sh, t, w, col, col && ty > 0 && j >= bx.lo[1], out, q, u, dv, B.L, B.Lu, i, j,
                      k, hc, hc.dx[0] * hc.dx[2], part, pp);
    if (!out) return;
    double *o = B.dsdt.ptr(i, j, k);
#pragma unroll
    for (int n = 0; n < NF; ++n) o[mol_comp(n) * B.dsdt.ns] = part[n];
    o[UTEMP * B.dsdt.ns] = pp;
}

// z and the update: tiles of zw x zh cells of the x-z plane, the inner
// zh - 2 planes written.
__global__ void __launch_bounds__(kBlock, 3)
k_mol_z(const MolBox *tab, const int *blk, int nbox, HydroConst hc) {
    __shared__ double sh[kMolSlots * kBlock];
    int lb;
    const MolBox &B = tab[mol_box(blk, nbox, xcd_block(), lb)];
    const Box bx = B.bx;
    const int w = B.zw, h = B.zh, t = (int)threadIdx.x;
    // z tiles fastest, then x: blocks that share planes run together
    const int r = lb / B.ntz, bz = lb - r * B.ntz;
    const int jj = r / B.nzx, bxi = r - jj * B.nzx;
    const int tz = t / w, tx = t - tz * w;
    const int i = bx.lo[0] + bxi * w + tx, j = bx.lo[1] + jj, k = bx.lo[2] - 1 + bz * (h - 2) + tz;
    const bool live = tz < h && i <= bx.hi[0] && k <= bx.hi[2] + 1;
    const bool out = live && k >= bx.lo[2] && k <= bx.hi[2] && tz > 0 && tz < h - 1;
    const CView q = cview(B.L, B.q, NQC), u = cview(B.Lu, B.u, NVAR), dv = cview(B.L, B.divu, 1);
    double part[NF], pp = 0.0;
    double *o = B.dsdt.ptr(i, j, k);
    const int64_t ns = B.dsdt.ns;
    if (out) {
#pragma unroll
        for (int n = 0; n < NF; ++n) part[n] = o[mol_comp(n) * ns];
        pp = o[UTEMP * ns];
    }
    mol_dir<2, false>(sh, t, w, live, live && tz > 0 && k >= bx.lo[2], out, q, u, dv, B.L, B.Lu, i, j,
                      k, hc, hc.dx[0] * hc.dx[1], part, pp);
    if (!out) return;
    // hydro_pdivu and hydro_update, written as 0 + the divergence
    const double vol = hc.dx[0] * hc.dx[1] * hc.dx[2], volinv = 1.0 / vol;
    const double pdivu = 0.5 * pp / vol;
#pragma unroll
    for (int n = 0; n < NF; ++n) {
        double d = 0.0 + part[n] * volinv;
        if (n == FEI) d -= pdivu;
        o[mol_comp(n) * ns] = d;
    }
    o[UTEMP * ns] = 0.0;
}

} // namespace

bool MolEngine::fits(const Box &bx) { return canon_fits(bx); }

MolEngine::~MolEngine() { release(); }

void MolEngine::release() {
    if (tab_) (void)hipFree(tab_);
    if (blk_) (void)hipFree(blk_);
    if (buf_) (void)hipFree(buf_);
    tab_ = nullptr;
    blk_ = nullptr;
    buf_ = nullptr;
}

int MolEngine::setup(const std::vector<Box> &boxes, const std::vector<Arr> &sb,
                     const std::vector<Arr> &dsdt) {
    const int n = (int)boxes.size();
    host_.resize(n);
    size_t total = 0;
    for (const Box &b : boxes) total += ((size_t)(NQC + 1) * canon_box(b).npts() + 31) & ~size_t(31);
    // where the primitives of all boxes at once are much of what is free, or
    // are not to be had, the level stays with one box's scratch per stream
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) != hipSuccess || total * sizeof(double) > free_b / 4)
        return CAMR_OK;
    if (hipMalloc(&buf_, total * sizeof(double)) != hipSuccess ||
        hipMalloc(&blk_, (size_t)4 * (n + 1) * sizeof(int)) != hipSuccess ||
        hipMalloc(&tab_, std::max(n, 1) * sizeof(MolBox)) != hipSuccess) {
        release();
        (void)hipGetLastError();  // not a later launch's
        return CAMR_OK;
    }
    blk_host_.assign((size_t)4 * (n + 1), 0);
    double *p = buf_;
    for (int b = 0; b < n; ++b) {
        MolBox &m = host_[b];
        const Box bx = boxes[b], cb = canon_box(bx), G = grow(bx, CAMR_NGROW);
        m.bx = bx;
        m.L = canon_of(bx);
        m.q = p;
        m.divu = p + (size_t)NQC * cb.npts();
        p += ((size_t)(NQC + 1) * cb.npts() + 31) & ~size_t(31);
        m.Lu.lo0 = G.lo[0]; m.Lu.lo1 = G.lo[1]; m.Lu.lo2 = G.lo[2];
        m.Lu.js = G.len(0);
        m.Lu.ks = G.len(0) * G.len(1);
        m.Lu.cs = (unsigned)G.npts();
        m.u = sb[b].p;
        m.dsdt = dsdt[b];
        // the tile whose inner cells fill the box's plane with the fewest
        // threads (rows of at least 8 inner cells where the box has them)
        const int n0 = bx.len(0), n1 = bx.len(1);
        int64_t best = INT64_MAX;
        for (int w = 4; w <= 66; ++w) {
            if (w > 4 && (w - 2 > n0 || (w < 10 && n0 >= 8))) continue;
            const int h = std::min(kBlock / w, n1 + 2);
            if (h < 3) continue;
            const int64_t tiles =
                (int64_t)((n0 + w - 3) / (w - 2)) * ((n1 + h - 3) / (h - 2));
            if (tiles <= best) {  // equal: the longer rows
                best = tiles;
                m.w = w;
                m.h = h;
            }
        }
        m.ntx = (n0 + m.w - 3) / (m.w - 2);
        m.nty = (n1 + m.h - 3) / (m.h - 2);
        // z: rows of 32 cells where the box has them (128^3: 182 us, of 16
        // cells 190, of 64 213)
        m.zw = std::min(n0, 32);
        m.zh = std::min(kBlock / m.zw, bx.len(2) + 2);
        m.nzx = (n0 + m.zw - 1) / m.zw;
        m.ntz = (bx.len(2) + m.zh - 3) / (m.zh - 2);
        const int64_t nb[4] = {(G.npts() + kBlock - 1) / kBlock,
                               (nodes(nodes(nodes(bx, 0), 1), 2).npts() + kBlock - 1) / kBlock,
                               (int64_t)m.ntx * m.nty * bx.len(2),
                               (int64_t)m.nzx * m.ntz * n1};
        for (int r = 0; r < 4; ++r) {
            int *row = &blk_host_[(size_t)r * (n + 1)];
            if (row[b] + nb[r] > 0x7fffffff) {
                set_error("method of lines: grid exceeds 2^31 blocks");
                return CAMR_ERR_SHAPE;
            }
            row[b + 1] = row[b] + (int)nb[r];
        }
    }
    if (n > 0 &&
        (hipMemcpy(tab_, host_.data(), n * sizeof(MolBox), hipMemcpyHostToDevice) != hipSuccess ||
         hipMemcpy(blk_, blk_host_.data(), blk_host_.size() * sizeof(int), hipMemcpyHostToDevice) !=
             hipSuccess)) {
        set_error("method of lines: table upload failed");
        return CAMR_ERR_HIP;
    }
    return CAMR_OK;
}

int MolEngine::source(const HydroConst &hc, hipStream_t st, int *status, Prof *prof) const {
    const int n = (int)host_.size();
    if (n == 0) return CAMR_OK;
    auto grid = [&](int r) { return dim3((unsigned)blk_host_[(size_t)r * (n + 1) + n]); };
    auto row = [&](int r) { return (const int *)(blk_ + (size_t)r * (n + 1)); };
    {
        Region reg(prof, "prim", st);
        hipLaunchKernelGGL(k_mol_prim, grid(0), dim3(kBlock), 0, st, tab_, row(0), n, hc, status);
    }
    {
        Region reg(prof, "divu", st);
        hipLaunchKernelGGL(k_mol_divu, grid(1), dim3(kBlock), 0, st, tab_, row(1), n, hc);
    }
    Region reg(prof, "mol_source", st);
    hipLaunchKernelGGL(k_mol_xy, grid(2), dim3(kBlock), 0, st, tab_, row(2), n, hc);
    hipLaunchKernelGGL(k_mol_z, grid(3), dim3(kBlock), 0, st, tab_, row(3), n, hc);
    return hipGetLastError() == hipSuccess ? CAMR_OK : CAMR_ERR_HIP;
}

} // namespace camr
