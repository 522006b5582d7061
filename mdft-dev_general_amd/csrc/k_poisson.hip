// k_poisson.hip -- electrostatic part of vext by the reference's fast Poisson
// solver (src/module_fastpoissonsolver.f90:121-288, "new construction"), on
// the device.
//
//  1. the solute point charges are spread onto the 8 surrounding nodes with
//     trilinear (cloud-in-cell) weights, periodic, and divided by the volume
//     element (src/module_solute.f90:193-232 with floorNode / ceilingNode /
//     distToFloorNode of src/module_mathematica.f90:134-220);
//  2. rho(k) = sum_r rho(r) exp(-i k.r) (FFTW's forward r2c), and
//     V(k) = 4 pi rho(k) / k^2, 0 where k^2 <= DBL_EPSILON, with k from the
//     integer frequencies m = i - 1 for i <= n/2, else i - 1 - n (:201-219);
//  3. for each orientation io, vextq(io, r) = qfact / N * c2r[V(k) conj(sigma_io(k))]
//     (:239-249), sigma_io(k) = sum_sites q_s exp(-i k.R_io r_s) exp(-0.5^2 k^2 / 2),
//     the smeared charge density of a solvent molecule in orientation io, with k
//     from the grid's wave vectors (+pi/d on the Nyquist index;
//     src/module_solvent.f90:367-426);
//  4. vext = vext_LJ + vextq, then the clip at qfact/2 (src/module_vext.f90:600-669).
//
// The c2r of FFTW reads the half spectrum kx = 0 .. nx/2 and takes the real part
// of the kx = 0 (and, nx even, kx = nx/2) planes after the y and z transforms.
// Its result is the inverse transform of the Hermitian spectrum S that has the
// half spectrum on 0 < kx < nx/2, its conjugate at the opposite wave vectors, and
// the Hermitian part of those two planes.  Two orientations share one complex
// transform: S_1 + i S_2 gives one as the real and the other as the imaginary part.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <map>
#include <vector>

#include "mdft_internal.h"

namespace {

constexpr int kThreads = 256;
constexpr double kSmootherRadius = 0.5;  // src/module_solvent.f90:381

struct PoissonArgs {
    int nx, ny, nz, no, j0, batch;  // columns j0 .. j0 + batch - 1 of the transforms, orientations 2 j and 2 j + 1
    int ncol;                       // all columns, (no + 1) / 2
    double lx, ly, lz;
    double q0;                      // charge at the molecule's origin
    const double *q;                // [nq] charges of the sites elsewhere
    const double2 *ph;              // phases exp(i k o): [axis: ny, nz, nx][index][site][orientation of the column][ncol]
};

__device__ inline double wave(int i, int n, double len) {  // the grid's wave vectors: +pi/d on the Nyquist index
    return 2.0 * acos(-1.0) * (i <= n / 2 ? i : i - n) / len;
}

// X <- 4 pi X / k^2 exp(-0.5^2 k^2 / 2), with X [N] the inverse-normalised transform of the charge
// density (N undoes its 1/N): V(k) times the smearing of sigma_io(k).
__global__ __launch_bounds__(kThreads) void poisson_field(double2 *__restrict__ X, PoissonArgs a) {
    const size_t N = (size_t)a.nx * a.ny * a.nz;
    const double twopi = 2.0 * acos(-1.0);
    for (size_t r = (size_t)blockIdx.x * kThreads + threadIdx.x; r < N; r += (size_t)gridDim.x * kThreads) {
        const int ix = (int)(r % a.nx), iy = (int)((r / a.nx) % a.ny), iz = (int)(r / ((size_t)a.nx * a.ny));
        // integer frequencies of the Poisson kernel
        const int m1 = ix < a.nx / 2 ? ix : ix - a.nx;
        const int m2 = iy < a.ny / 2 ? iy : iy - a.ny;
        const int m3 = iz < a.nz / 2 ? iz : iz - a.nz;
        const double q1 = twopi * m1 / a.lx, q2 = twopi * m2 / a.ly, q3 = twopi * m3 / a.lz;
        const double k2 = q1 * q1 + q2 * q2 + q3 * q3;
        const double kx = wave(ix, a.nx, a.lx), ky = wave(iy, a.ny, a.ly), kz = wave(iz, a.nz, a.lz);
        const double smooth = exp(-kSmootherRadius * kSmootherRadius * (kx * kx + ky * ky + kz * kz) / 2.0);
        const double f = fabs(k2) > DBL_EPSILON ? (double)N * 2.0 * twopi / k2 * smooth : 0.0;
        X[r] = make_double2(X[r].x * f, X[r].y * f);
    }
}

// phases of one axis: ph[i][(site, orientation)][column] = exp(i k_i o), o the axis's component of the
// site's place in orientation 2 column + orientation
__global__ __launch_bounds__(kThreads) void poisson_phases(double2 *__restrict__ ph, int n, double len, int axis, int no,
                                                          int ncol, int nq, const int *__restrict__ qsite, int nsite,
                                                          const double *__restrict__ site_off) {
    const size_t total = (size_t)n * nq * 2 * ncol;
    for (size_t g = (size_t)blockIdx.x * kThreads + threadIdx.x; g < total; g += (size_t)gridDim.x * kThreads) {
        const int j = (int)(g % ncol), t = (int)(g / ncol % (2 * nq)), i = (int)(g / ((size_t)ncol * 2 * nq));
        const int io = 2 * j + (t & 1);
        const double o = io < no ? site_off[((size_t)io * nsite + qsite[t >> 1]) * 3 + axis] : 0.0;
        double s, c;
        sincos(wave(i, n, len) * o, &s, &c);
        ph[g] = make_double2(c, s);
    }
}

__device__ inline double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// Z [N][batch] = S_1 + i S_2 of each column (see above).  A workgroup takes one (ky, kz) line, its
// threads (column, kx); the phase of a wave vector is the product of its axes' phases, of which ky
// and kz are multiplied once per thread (NQ sites).  One evaluation serves k and -k.  Bound by its
// writes: 42 orientations at 96^3 in 0.07-0.10 ms, 3-4.4 TB/s (with a sine and a cosine per site and
// element, and half of the elements zero, 28 orientations took 0.29 ms).
template <int NQ>
__global__ __launch_bounds__(kThreads) void poisson_spectrum(const double2 *__restrict__ X, double2 *__restrict__ Z,
                                                            PoissonArgs a) {
    const int iy = blockIdx.x % a.ny, iz = blockIdx.x / a.ny;
    const int my = iy ? a.ny - iy : 0, mz = iz ? a.nz - iz : 0;
    const int rows = kThreads / a.batch > 0 ? kThreads / a.batch : 1;
    const int T = 2 * NQ * a.ncol;  // phases of one index
    const double2 *py = a.ph, *pz = py + (size_t)a.ny * T, *px = pz + (size_t)a.nz * T;
    for (int jj = threadIdx.x % (kThreads / rows); jj < a.batch; jj += kThreads / rows) {
        const int row = threadIdx.x / (kThreads / rows), col = a.j0 + jj;
        if (row >= rows || col >= a.ncol) continue;
        const bool two = 2 * col + 1 < a.no;
        constexpr int NR = NQ > 0 ? 2 * NQ : 1;
        double2 yz[NR];
#pragma unroll
        for (int t = 0; t < 2 * NQ; t++)
            yz[t] = cmul(py[(size_t)iy * T + t * a.ncol + col], pz[(size_t)iz * T + t * a.ncol + col]);
        // U_o = V conj(sigma_o) at kx index ix with the y, z phases p
        auto spectrum = [&](int ix, const double2 *p, double2 V, double2 &u1, double2 &u2) {
            double2 s[2] = {make_double2(a.q0, 0.0), make_double2(a.q0, 0.0)};
#pragma unroll
            for (int t = 0; t < 2 * NQ; t++) {
                const double2 e = cmul(p[t], px[(size_t)ix * T + t * a.ncol + col]);
                s[t & 1].x += a.q[t >> 1] * e.x;
                s[t & 1].y += a.q[t >> 1] * e.y;
            }
            u1 = cmul(V, s[0]);
            u2 = two ? cmul(V, s[1]) : make_double2(0.0, 0.0);
        };
        const size_t line = ((size_t)iz * a.ny + iy) * a.nx, mline = ((size_t)mz * a.ny + my) * a.nx;
        for (int ix = row; ix <= a.nx / 2; ix += rows) {
            double2 u1, u2;
            spectrum(ix, yz, X[line + ix], u1, u2);
            const bool own = ix == 0 || 2 * ix == a.nx;
            if (own) {  // the Hermitian part of the plane
                double2 myz[NR], v1, v2;
#pragma unroll
                for (int t = 0; t < 2 * NQ; t++)
                    myz[t] = cmul(py[(size_t)my * T + t * a.ncol + col], pz[(size_t)mz * T + t * a.ncol + col]);
                spectrum(ix, myz, X[mline + ix], v1, v2);
                u1 = make_double2(0.5 * (u1.x + v1.x), 0.5 * (u1.y - v1.y));
                u2 = make_double2(0.5 * (u2.x + v2.x), 0.5 * (u2.y - v2.y));
            }
            Z[(line + ix) * a.batch + jj] = make_double2(u1.x - u2.y, u1.y + u2.x);
            if (!own) Z[(mline + a.nx - ix) * a.batch + jj] = make_double2(u1.x + u2.y, u2.x - u1.y);
        }
    }
}

// One read of Z and one write of vext, whose runs of 2 batch values straddle lines: 42 orientations
// at 96^3 in 0.167 ms, 3.6 TB/s.
// vext[r][2 j], vext[r][2 j + 1] = min(base + scale (Re, Im) Z[r][j], clip), base the potential of the
// sites' places, or (places.ncols < 0) vext itself
constexpr int kPerThread = 8, kChunk = kPerThread * kThreads;
__global__ __launch_bounds__(kThreads) void poisson_store(const double2 *__restrict__ Z, double *__restrict__ vext,
                                                         size_t total, int no, int j0, unsigned batch, double scale,
                                                         VextPlaces places, double clip) {
    const size_t g0 = (size_t)blockIdx.x * kChunk, r0 = g0 / batch;
    const unsigned c0 = (unsigned)(g0 - r0 * batch);
    double2 z[kPerThread];  // all loads before the first store
    double b0[kPerThread];
    const bool one = places.ncols == 1 && places.nsite == 1;  // a single place: every orientation reads it
#pragma unroll
    for (int k = 0; k < kPerThread; k++) {
        const unsigned i = threadIdx.x + k * kThreads;
        const size_t g = g0 + i < total ? g0 + i : total - 1;
        z[k] = Z[g];
        b0[k] = one ? places.S[r0 + (c0 + (unsigned)(g - g0)) / batch] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < kPerThread; k++) {
        const unsigned i = threadIdx.x + k * kThreads;
        if (g0 + i >= total) break;
        const unsigned q = (c0 + i) / batch;
        const size_t r = r0 + q;
        const int io = 2 * (j0 + (int)(c0 + i - q * batch));
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (io + h >= no) break;
            double *v = vext + r * no + io + h;
            double b = b0[k];
            if (places.ncols < 0) {
                b = *v;
            } else if (!one) {
                for (int s = 0; s < places.nsite; s++)
                    b += places.S[r * places.ncols + places.col[(io + h) * places.nsite + s]];
            }
            b += scale * (h ? z[k].y : z[k].x);
            *v = b > clip ? clip : b;
        }
    }
}

__global__ __launch_bounds__(kThreads) void zero_field(double2 *__restrict__ X, size_t N) {
    for (size_t g = (size_t)blockIdx.x * kThreads + threadIdx.x; g < N; g += (size_t)gridDim.x * kThreads)
        X[g] = make_double2(0.0, 0.0);
}

__global__ void scatter_set(double2 *__restrict__ X, const long long *idx, const double *val, int nval) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nval) X[idx[i]] = make_double2(val[i], 0.0);
}

__global__ __launch_bounds__(kThreads) void clip_kernel(double *__restrict__ v, size_t total, double clip) {
    for (size_t g = (size_t)blockIdx.x * kThreads + threadIdx.x; g < total; g += (size_t)gridDim.x * kThreads)
        if (v[g] > clip) v[g] = clip;
}

unsigned blocks_for(size_t total) {
    size_t nb = (total + kThreads - 1) / kThreads;
    return (unsigned)(nb > 65536 ? 65536 : nb);
}

}  // namespace

hipError_t launch_vext_clip(mdft_ctx *c, double clip) {
    const size_t total = c->N * (size_t)c->no;
    hipLaunchKernelGGL(clip_kernel, dim3(blocks_for(total)), dim3(kThreads), 0, c->stream, c->d_vext, total, clip);
    return hipGetLastError();
}

// vext <- min(base + the Poisson electrostatic energy of the solvent sites (steps 1-3 above), clip),
// base from the sites' places or vext itself (places.ncols < 0).  h_atoms [natom][6] (x, y, z, q,
// sigma, epsilon), h_site_q [nsite] and h_site_off [no][nsite][3] on the host, d_site_off the
// offsets on the device.  *done false: the solute has no charge, nothing was written.
hipError_t launch_poisson_vext(mdft_ctx *c, int natom, const double *h_atoms, int nsite, const double *h_site_q,
                               const double *h_site_off, const double *d_site_off, double qfact,
                               const VextPlaces &places, double clip, bool *done) {
    *done = false;
    const int n[3] = {c->d.nx, c->d.ny, c->d.nz};
    const double len[3] = {c->d.lx, c->d.ly, c->d.lz};
    // 1. cloud-in-cell charges (the reference's do concurrent over sites, in site order)
    std::map<long long, double> rho;
    bool charged = false;
    for (int s = 0; s < natom; s++) {
        const double q = h_atoms[6 * s + 3];
        if (!(fabs(q) > DBL_EPSILON)) continue;
        charged = true;
        int m[3], p[3];
        double wp[3], wm[3];
        for (int a = 0; a < 3; a++) {
            const double x = h_atoms[6 * s + a], d = len[a] / n[a];
            m[a] = (int)floor(fmod(fmod(x, len[a]) + len[a], len[a]) / d);  // floorNode - 1 (0-based)
            if (m[a] >= n[a]) m[a] -= n[a];
            p[a] = (m[a] + 1) % n[a];                                     // ceilingNode - 1
            wp[a] = fabs(x / d - floor(x / d));                            // distToFloorNode
            wm[a] = 1.0 - wp[a];
        }
        for (int corner = 0; corner < 8; corner++) {
            const int cx = (corner & 1) ? p[0] : m[0], cy = (corner & 2) ? p[1] : m[1], cz = (corner & 4) ? p[2] : m[2];
            // q * w1 * w2 * w3, left to right as in the reference
            const double qw = q * ((corner & 1) ? wp[0] : wm[0]) * ((corner & 2) ? wp[1] : wm[1]) *
                              ((corner & 4) ? wp[2] : wm[2]);
            rho[((long long)cz * n[1] + cy) * n[0] + cx] += qw;
        }
    }
    if (!charged) return hipSuccess;  // no solute charge: no electrostatic potential (src/module_vext.f90:154-164)
    const double dvol = (len[0] / n[0]) * (len[1] / n[1]) * (len[2] / n[2]);
    std::vector<long long> idx;
    std::vector<double> val;
    bool nonzero = false;
    for (auto &kv : rho) {
        idx.push_back(kv.first);
        val.push_back(kv.second / dvol);
        nonzero = nonzero || fabs(kv.second / dvol) > DBL_EPSILON;
    }
    if (!nonzero) return hipSuccess;  // all |rho| <= DBL_EPSILON (:187-190)
    *done = true;
    const size_t N = c->N;
    // charged sites, those at the molecule's origin in every orientation apart: their phase is 1
    double q0 = 0.0;
    std::vector<int> qsite;
    std::vector<double> qs;
    for (int s = 0; s < nsite; s++) {
        if (fabs(h_site_q[s]) <= DBL_EPSILON) continue;
        bool origin = true;
        for (int io = 0; io < c->no; io++)
            for (int k = 0; k < 3; k++) origin = origin && h_site_off[((size_t)io * nsite + s) * 3 + k] == 0.0;
        if (origin) {
            q0 += h_site_q[s];
        } else {
            qsite.push_back(s);
            qs.push_back(h_site_q[s]);
        }
    }
    // sites are summed in groups of at most kMaxQ (the phases of one group in registers): each group is a
    // transform of its own, added to the one before it
    constexpr int kMaxQ = 4;
    const int ngroup = qsite.empty() ? 1 : ((int)qsite.size() + kMaxQ - 1) / kMaxQ;
    // two orientations per column, at most np columns at a time
    const int ncol = (c->no + 1) / 2, nchunk = (ncol + c->np - 1) / c->np, B = (ncol + nchunk - 1) / nchunk;
    const size_t nph = (size_t)(n[0] + n[1] + n[2]) * 2 * kMaxQ * ncol;
    double2 *X = nullptr, *Z = nullptr, *ph = nullptr;
    long long *d_idx = nullptr;
    double *d_val = nullptr, *d_q = nullptr;
    int *d_qsite = nullptr;
    hipError_t e = dev_malloc(&X, sizeof(double2) * N);
    if (e == hipSuccess) e = dev_malloc(&Z, sizeof(double2) * N * B);
    if (e == hipSuccess) e = dev_malloc(&ph, sizeof(double2) * nph);
    if (e == hipSuccess) e = dev_malloc(&d_idx, sizeof(long long) * idx.size());
    if (e == hipSuccess) e = dev_malloc(&d_val, sizeof(double) * val.size());
    if (e == hipSuccess) e = dev_malloc(&d_q, sizeof(double) * (qs.size() + 1));
    if (e == hipSuccess) e = dev_malloc(&d_qsite, sizeof(int) * (qs.size() + 1));
    if (e == hipSuccess) e = hipMemcpy(d_idx, idx.data(), sizeof(long long) * idx.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(d_val, val.data(), sizeof(double) * val.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess && !qs.empty()) e = hipMemcpy(d_q, qs.data(), sizeof(double) * qs.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess && !qs.empty())
        e = hipMemcpy(d_qsite, qsite.data(), sizeof(int) * qs.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(zero_field, dim3(blocks_for(N)), dim3(kThreads), 0, c->stream, X, N);
        hipLaunchKernelGGL(scatter_set, dim3(((unsigned)val.size() + 255) / 256), dim3(256), 0, c->stream, X, d_idx,
                           d_val, (int)val.size());
        e = hipGetLastError();
    }
    // 2. forward transform exp(-i k.r), normalised by 1/N (undone in poisson_field)
    if (e == hipSuccess) e = launch_fft3d_f64(c, X, -1, 1);
    PoissonArgs a{n[0], n[1], n[2], c->no, 0, B, ncol, len[0], len[1], len[2], 0.0, d_q, ph};
    if (e == hipSuccess) {
        hipLaunchKernelGGL(poisson_field, dim3(blocks_for(N)), dim3(kThreads), 0, c->stream, X, a);
        e = hipGetLastError();
    }
    // 3. per group of sites and chunk of columns: spectrum, unnormalised inverse exp(+i k.r), store
    for (int g = 0; e == hipSuccess && g < ngroup; g++) {
        const int nq = qsite.empty() ? 0 : std::min(kMaxQ, (int)qsite.size() - g * kMaxQ);
        a.q = d_q + g * kMaxQ;
        a.q0 = g == 0 ? q0 : 0.0;
        double2 *p = ph;
        const int axis[3] = {1, 2, 0};
        for (int k = 0; k < 3 && nq > 0; k++) {
            const int ax = axis[k];
            hipLaunchKernelGGL(poisson_phases, dim3(blocks_for((size_t)n[ax] * nq * 2 * ncol)), dim3(kThreads), 0,
                               c->stream, p, n[ax], len[ax], ax, c->no, ncol, nq, d_qsite + g * kMaxQ, nsite, d_site_off);
            p += (size_t)n[ax] * nq * 2 * ncol;
        }
        VextPlaces base = places;
        if (g > 0) base.ncols = -1;
        for (a.j0 = 0; e == hipSuccess && a.j0 < ncol; a.j0 += B) {
            const dim3 grid((unsigned)(n[1] * n[2]));
            switch (nq) {
#define POISSON_NQ(Q) \
    case Q: hipLaunchKernelGGL(poisson_spectrum<Q>, grid, dim3(kThreads), 0, c->stream, X, Z, a); break;
                POISSON_NQ(0) POISSON_NQ(1) POISSON_NQ(2) POISSON_NQ(3) POISSON_NQ(4)
#undef POISSON_NQ
            }
            e = hipGetLastError();
            if (e == hipSuccess) e = launch_fft3d_f64(c, Z, +1, B);
            if (e == hipSuccess) {
                const size_t total = N * B;
                hipLaunchKernelGGL(poisson_store, dim3((unsigned)((total + kChunk - 1) / kChunk)), dim3(kThreads), 0,
                                   c->stream, Z, c->d_vext, total, c->no, a.j0, (unsigned)B, qfact / (double)N, base,
                                   g + 1 == ngroup ? clip : HUGE_VAL);
                e = hipGetLastError();
            }
        }
    }
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    (void)dev_free(X, e == hipSuccess);
    (void)dev_free(Z, e == hipSuccess);
    (void)dev_free(ph, e == hipSuccess);
    (void)dev_free(d_qsite, e == hipSuccess);
    (void)dev_free(d_idx, e == hipSuccess);
    (void)dev_free(d_val, e == hipSuccess);
    (void)dev_free(d_q, e == hipSuccess);
    return e;
}
