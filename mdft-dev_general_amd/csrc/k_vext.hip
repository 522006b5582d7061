// k_vext.hip -- external potential vext(io, r) of a solute on the device.
//
// Lennard-Jones between solute atoms and solvent sites with Lorentz-Berthelot
// mixing and a spherical cut-off (src/module_lennardjones.f90:9-226, rvdw
// default 10 A), plus the Coulomb energy of the solvent site charges in the
// solute's field taken at the minimum image, and the clip at qfact/2 of
// src/module_vext.f90:638-640.  The reference computes the electrostatic part
// with a periodic Poisson solver (src/module_fastpoissonsolver.f90:121-288);
// the minimum-image sum here is the reference's direct_sum alternative in
// spirit; the Poisson path itself is in k_poisson.hip (the Coulomb term and the
// clip are then off here, and the clip follows the sum).
//
// A site that stands at few distinct places over the orientations (at the
// molecule's origin: one; on its axis: one per (theta, phi)) has its potential
// summed over the atoms once per place (site_potential), and the orientations
// read it; only the other sites are summed per orientation.
#include "mdft_internal.h"

namespace {

constexpr int kThreads = 256;
constexpr int kTile = 256;

struct VextArgs {
    int nx, ny, nz, no, nsite, natom;
    double dx, dy, dz, lx, ly, lz, ilx, ily, ilz, rc2, qfact, clip;
    int coulomb;  // 1: minimum-image Coulomb of the site charges in the solute's field
    const double *site_off;  // [no][nsite][3]
    const double *site_p;    // [nsite][3]: q, sigma, epsilon
    const double *atoms;     // [natom][6]: x, y, z, q, sigma, epsilon
};

// squared minimum-image distance.  (Dividing by the box length instead of multiplying by its
// inverse would differ at half a box only, where both images are as far.)
__device__ inline double min_image2(double x, double y, double z, const VextArgs &a) {
    x -= a.lx * rint(x * a.ilx);
    y -= a.ly * rint(y * a.ily);
    z -= a.lz * rint(z * a.ilz);
    return fmax(x * x + y * y + z * z, 1e-12);
}

constexpr int kBx = 8, kBy = 8, kBz = 4;  // points of a workgroup: a brick, so that its atoms are near

// S[r][col] = sum over the atoms of the potential of site col_site[col] at r + col_pos[col].  The
// atoms that can reach the brick (all of them with a Coulomb term) are gathered in LDS, 256 tested
// at a time, and every thread sums over those: bound by FP64 arithmetic, about 50 instructions per
// point and atom within reach.  64^3, 1000 atoms, mmax 3: 0.217 ms; 96^3, 20 atoms: 0.013 ms (one
// sum per orientation over all atoms and sites: 109 and 8.0 ms).
__global__ __launch_bounds__(kThreads) void site_potential(double *__restrict__ S, int ncols,
                                                          const double *__restrict__ col_pos,
                                                          const int *__restrict__ col_site, VextArgs a) {
    struct Atom {
        double x, y, z, sg2, e4, qq;
    };
    __shared__ Atom at[kTile];
    __shared__ int base[kThreads / 64];
    const int nbx = (a.nx + kBx - 1) / kBx, nby = (a.ny + kBy - 1) / kBy;
    const int bx = blockIdx.x % nbx * kBx, by = blockIdx.x / nbx % nby * kBy, bz = blockIdx.x / (nbx * nby) * kBz;
    const int tid = threadIdx.x, col = blockIdx.y, s = col_site[col];
    const int ix = bx + tid % kBx, iy = by + tid / kBx % kBy, iz = bz + tid / (kBx * kBy);
    const double ox = col_pos[3 * col], oy = col_pos[3 * col + 1], oz = col_pos[3 * col + 2];
    const double sx = ix * a.dx + ox, sy = iy * a.dy + oy, sz = iz * a.dz + oz;
    const double hx = 0.5 * (kBx - 1) * a.dx, hy = 0.5 * (kBy - 1) * a.dy, hz = 0.5 * (kBz - 1) * a.dz;
    const double cx = bx * a.dx + ox + hx, cy = by * a.dy + oy + hy, cz = bz * a.dz + oz + hz;
    const double qs = a.site_p[3 * s], sgs = a.site_p[3 * s + 1], eps_s = a.site_p[3 * s + 2];
    const int lane = tid & 63, wv = tid >> 6;
    double acc = 0.0;
    for (int t0 = 0; t0 < a.natom; t0 += kTile) {
        bool in = t0 + tid < a.natom;
        Atom m{};
        if (in) {
            const double *p = a.atoms + (size_t)(t0 + tid) * 6;
            m.x = p[0];
            m.y = p[1];
            m.z = p[2];
            const double e = eps_s * p[5], sg = 0.5 * (sgs + p[4]);
            m.sg2 = sg * sg;
            m.e4 = e > 0.0 ? 4.0 * sqrt(e) : 0.0;
            m.qq = a.coulomb ? qs * p[3] : 0.0;
            // the distance to the brick along each axis is at least the centre's less its half width
            const double ux = cx - m.x, uy = cy - m.y, uz = cz - m.z;
            const double fx = fmax(0.0, fabs(ux - a.lx * rint(ux * a.ilx)) - hx);
            const double fy = fmax(0.0, fabs(uy - a.ly * rint(uy * a.ily)) - hy);
            const double fz = fmax(0.0, fabs(uz - a.lz * rint(uz * a.ilz)) - hz);
            const bool far = fx * fx + fy * fy + fz * fz > a.rc2 * (1.0 + 1e-9) + 1e-9;
            if (far) m.e4 = 0.0;
            in = m.e4 != 0.0 || m.qq != 0.0;
        }
        const unsigned long long mask = __ballot(in);
        __syncthreads();  // the last tile's list has been read
        if (lane == 0) base[wv] = __popcll(mask);
        __syncthreads();
        int at0 = 0, nt = 0;
        for (int w = 0; w < kThreads / 64; w++) {
            if (w < wv) at0 += base[w];
            nt += base[w];
        }
        if (in) at[at0 + __popcll(mask & ((1ull << lane) - 1))] = m;
        __syncthreads();
        for (int k = 0; k < nt; k++) {
            const Atom b = at[k];
            const double r2 = min_image2(sx - b.x, sy - b.y, sz - b.z, a);
            if (b.e4 != 0.0 && r2 < a.rc2) {
                const double sr2 = b.sg2 / r2;
                const double sr6 = sr2 * sr2 * sr2;
                acc += b.e4 * (sr6 * sr6 - sr6);
            }
            if (b.qq != 0.0) acc += a.qfact * b.qq / sqrt(r2);
        }
    }
    if (ix < a.nx && iy < a.ny && iz < a.nz) S[(((size_t)iz * a.ny + iy) * a.nx + ix) * ncols + col] = acc;
}

// The sum over the places of the sites of orientation io at point r.
__device__ inline double place_sum(const VextPlaces &b, size_t r, int io) {
    double v = 0.0;
    for (int s = 0; s < b.nsite; s++) {
        v += b.S[r * b.ncols + b.col[io * b.nsite + s]];
    }
    return v;
}

constexpr int kChunk = 16 * kThreads;  // elements of a workgroup

// vext where every site stands at few places: one read of them, one write per orientation
__global__ __launch_bounds__(kThreads) void vext_from_places(double *__restrict__ vext, size_t total, unsigned no,
                                                            VextPlaces b, double clip) {
    const size_t g0 = (size_t)blockIdx.x * kChunk, r0 = g0 / no;
    const unsigned o0 = (unsigned)(g0 - r0 * no);
    for (unsigned i = threadIdx.x; i < kChunk && g0 + i < total; i += kThreads) {
        const unsigned q = (o0 + i) / no;
        vext[g0 + i] = fmin(place_sum(b, r0 + q, (int)(o0 + i - q * no)), clip);
    }
}

// One thread per (grid point, orientation) for the sites whose place depends on the orientation (sites[0 ..
// nlive)); solute atoms are staged through LDS in tiles shared by the workgroup.
__global__ __launch_bounds__(kThreads) void vext_kernel(double *__restrict__ vext, VextArgs a, VextPlaces b, int nlive,
                                                       const int *__restrict__ sites) {
    __shared__ double at[kTile][6];
    const size_t total = (size_t)a.nx * a.ny * a.nz * a.no;
    const size_t g = (size_t)blockIdx.x * kThreads + threadIdx.x;
    const bool live = g < total;
    const size_t r = live ? g / a.no : 0;
    const int io = live ? (int)(g % a.no) : 0;
    const int ix = (int)(r % a.nx), iy = (int)((r / a.nx) % a.ny), iz = (int)(r / ((size_t)a.nx * a.ny));
    const double px = ix * a.dx, py = iy * a.dy, pz = iz * a.dz;
    double acc = b.ncols > 0 && live ? place_sum(b, r, io) : 0.0;
    for (int t0 = 0; t0 < a.natom; t0 += kTile) {
        const int nt = min(kTile, a.natom - t0);
        __syncthreads();
        for (int i = threadIdx.x; i < nt * 6; i += kThreads) at[i / 6][i % 6] = a.atoms[(size_t)t0 * 6 + i];
        __syncthreads();
        if (!live) continue;
        for (int l = 0; l < nlive; l++) {
            const int s = sites[l];
            const double *off = a.site_off + ((size_t)io * a.nsite + s) * 3;
            const double sx = px + off[0], sy = py + off[1], sz = pz + off[2];
            const double qs = a.site_p[3 * s], sgs = a.site_p[3 * s + 1], eps_s = a.site_p[3 * s + 2];
            for (int k = 0; k < nt; k++) {
                const double r2 = min_image2(sx - at[k][0], sy - at[k][1], sz - at[k][2], a);
                const double e = eps_s * at[k][5];
                if (e > 0.0 && r2 < a.rc2) {
                    const double sg = 0.5 * (sgs + at[k][4]);
                    const double sr2 = sg * sg / r2;
                    const double sr6 = sr2 * sr2 * sr2;
                    acc += 4.0 * sqrt(e) * (sr6 * sr6 - sr6);
                }
                const double qq = qs * at[k][3];
                if (a.coulomb && qq != 0.0) acc += a.qfact * qq / sqrt(r2);
            }
        }
    }
    if (live) vext[g] = fmin(acc, a.clip);
}

VextArgs vext_args(mdft_ctx *c, int natom, const double *d_atoms, int nsite, const double *d_site_p,
                   const double *d_site_off, double rcut, double qfact, double clip, bool coulomb) {
    VextArgs a;
    a.coulomb = coulomb ? 1 : 0;
    a.nx = c->d.nx;
    a.ny = c->d.ny;
    a.nz = c->d.nz;
    a.no = c->no;
    a.nsite = nsite;
    a.natom = natom;
    a.dx = c->d.lx / c->d.nx;
    a.dy = c->d.ly / c->d.ny;
    a.dz = c->d.lz / c->d.nz;
    a.lx = c->d.lx;
    a.ly = c->d.ly;
    a.lz = c->d.lz;
    a.ilx = 1.0 / c->d.lx;
    a.ily = 1.0 / c->d.ly;
    a.ilz = 1.0 / c->d.lz;
    a.rc2 = rcut * rcut;
    a.qfact = qfact;
    a.clip = clip;
    a.site_off = d_site_off;
    a.site_p = d_site_p;
    a.atoms = d_atoms;
    return a;
}

}  // namespace

hipError_t launch_site_potential(mdft_ctx *c, int natom, const double *d_atoms, int nsite, const double *d_site_p,
                                 double rcut, double qfact, bool coulomb, int ncols, const double *d_col_pos,
                                 const int *d_col_site, double *S) {
    const VextArgs a = vext_args(c, natom, d_atoms, nsite, d_site_p, nullptr, rcut, qfact, 0.0, coulomb);
    const size_t nb = (size_t)((a.nx + kBx - 1) / kBx) * ((a.ny + kBy - 1) / kBy) * ((a.nz + kBz - 1) / kBz);
    hipLaunchKernelGGL(site_potential, dim3((unsigned)nb, (unsigned)ncols), dim3(kThreads), 0, c->stream, S, ncols,
                       d_col_pos, d_col_site, a);
    return hipGetLastError();
}

hipError_t launch_vext_from_places(mdft_ctx *c, const VextPlaces &b, double clip) {
    const size_t total = c->N * (size_t)c->no;
    hipLaunchKernelGGL(vext_from_places, dim3((unsigned)((total + kChunk - 1) / kChunk)), dim3(kThreads), 0, c->stream,
                       c->d_vext, total, (unsigned)c->no, b, clip);
    return hipGetLastError();
}

hipError_t launch_vext(mdft_ctx *c, int natom, const double *d_atoms, int nsite, const double *d_site_p,
                       const double *d_site_off, double rcut, double qfact, double clip, bool coulomb,
                       const VextPlaces &b, int nlive, const int *d_sites) {
    const VextArgs a = vext_args(c, natom, d_atoms, nsite, d_site_p, d_site_off, rcut, qfact, clip, coulomb);
    const size_t total = c->N * (size_t)c->no;
    const size_t nb = (total + kThreads - 1) / kThreads;
    hipLaunchKernelGGL(vext_kernel, dim3((unsigned)nb), dim3(kThreads), 0, c->stream, c->d_vext, a, b, nlive, d_sites);
    return hipGetLastError();
}
