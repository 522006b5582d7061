// k_angular.hip -- orientation <-> projection transforms and the fused
// gradient/free-energy pass, FP64.
//
// angl2proj restates src/module_orientation_projection_transform.f90:159-199
// (a 2D DFT over (psi, phi) for each theta node, then a Gauss-Legendre
// contraction in theta with Wigner d and sqrt(2m+1)), driven as in
// src/module_energy_cproj_mrso.f90:276-290 with o = rho0 (xi^2 - 1).
// The final pass fuses proj2angl (:202-243), the F_exc reduction and dF update
// of src/module_energy_cproj_mrso.f90:728-762 with the ideal+external term of
// src/module_energy_ideal_and_external.f90:48-72, so xi is read once, vext once
// and dF written once per evaluation.
//
// Layout: points r are processed in tiles of PT consecutive points per
// workgroup; xi/vext/df tiles [PT][no] and projection tiles [PT][np] are
// contiguous in HBM, so every global access is a coalesced stream.
#include <cfloat>

#include "mdft_internal.h"
#include "turns.h"

namespace {

constexpr int kThreads = 256;

__device__ inline double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

template <typename T> struct C2;
template <> struct C2<double> { using t = double2; };
template <> struct C2<float> { using t = float2; };
template <typename V> __device__ inline V mk(decltype(V::x) a, decltype(V::x) b) { V v; v.x = a; v.y = b; return v; }

// An FP32 value held in the low word of an FP64 register pair.  The tile prefetches keep the
// loaded word as it is and convert it where it is used: a conversion next to each load would
// make the wave wait for every load before issuing the next, one HBM latency per element.
__device__ inline double hold_f32(float v) { return __longlong_as_double((long long)__float_as_uint(v)); }
__device__ inline double held_f32(double h) { return (double)__uint_as_float((unsigned)__double_as_longlong(h)); }

template <int PT>
__global__ __launch_bounds__(kThreads) void angl2proj_f64(const double *__restrict__ xi, double2 *__restrict__ proj,
                                                         size_t N, AngTables t, double rho0) {
    extern __shared__ double smem[];
    const int no = t.no, np = t.np, nth = t.ntheta, nphi = t.nphi, npsi = t.npsi, H1 = t.H + 1,
              W = 2 * t.L + 1;
    double *o = smem;                                           // [PT][no]
    double2 *G = reinterpret_cast<double2 *>(o + PT * no);      // [PT][nth][nphi][H1]
    double2 *F = G + PT * nth * nphi * H1;                      // [PT][nth][W][H1]
    const size_t r0 = (size_t)blockIdx.x * PT;
    const int npts = (int)((N - r0) < (size_t)PT ? (N - r0) : (size_t)PT);
    const int tid = threadIdx.x;
    const double *src = xi + r0 * no;
    for (int i = tid; i < npts * no; i += kThreads) {
        double x = src[i];
        o[i] = rho0 * (x * x - 1.0);
    }
    __syncthreads();
    // DFT over psi: G = sum_ipsi o exp(+i mu2 psi)
    const int nG = npts * nth * nphi * H1;
    for (int i = tid; i < nG; i += kThreads) {
        const int mu2 = i % H1;
        const double *line = o + (i / H1) * npsi;
        double re = 0.0, im = 0.0;
        for (int ipsi = 0; ipsi < npsi; ipsi++) {
            const int k = (mu2 * ipsi) % npsi;
            const double v = line[ipsi];
            re += v * t.cps[k];
            im += v * t.sps[k];
        }
        G[i] = make_double2(re, im);
    }
    __syncthreads();
    // DFT over phi: F = sum_iphi G exp(+i mup phi) / (nphi npsi)
    const double norm = 1.0 / (double)(nphi * npsi);
    const int nF = npts * nth * W * H1;
    for (int i = tid; i < nF; i += kThreads) {
        const int mu2 = i % H1;
        int rest = i / H1;
        const int mup = rest % W - t.L;
        rest /= W;  // pt*nth + it
        const double2 *g = G + (size_t)rest * nphi * H1 + mu2;
        double re = 0.0, im = 0.0;
        for (int iphi = 0; iphi < nphi; iphi++) {
            int k = (mup * iphi) % nphi;
            k += (k < 0) ? nphi : 0;
            const double2 v = g[iphi * H1];
            re += v.x * t.cph[k] - v.y * t.sph[k];
            im += v.x * t.sph[k] + v.y * t.cph[k];
        }
        F[i] = make_double2(re * norm, im * norm);
    }
    __syncthreads();
    // Gauss-Legendre contraction in theta with Wigner d
    double2 *dst = proj + r0 * np;
    for (int i = tid; i < npts * np; i += kThreads) {
        const int pt = i / np, ip = i - pt * np;
        const int mup = t.pmup[ip], mu2 = t.pmu[ip] / t.mrso;
        const double2 *f = F + ((size_t)pt * nth * W + (mup + t.L)) * H1 + mu2;
        const double *a = t.a2p + ip * nth;
        double re = 0.0, im = 0.0;
        for (int it = 0; it < nth; it++) {
            const double2 v = f[(size_t)it * W * H1];
            re += v.x * a[it];
            im += v.y * a[it];
        }
        dst[i] = make_double2(re * t.fm[ip], im * t.fm[ip]);
    }
}

// products of the gradient with up to 3 vectors (FP32 or FP64, bit j of self: the gradient
// itself), accumulated in the final pass (mdft_energy_and_gradient_dots)
struct DotArgs {
    int k, self, f32;
    const void *p[3];
};

__device__ inline double dot_operand(const DotArgs &da, int j, size_t g, double gv) {
    if ((da.self >> j) & 1) return gv;
    return da.f32 ? (double)static_cast<const float *>(da.p[j])[g] : static_cast<const double *>(da.p[j])[g];
}

__device__ inline void block_reduce3(double &a, double &b, double &c, double *partials) {
    __shared__ double red[3][kThreads / 64];
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_down(a, off, 64);
        b += __shfl_down(b, off, 64);
        c += __shfl_down(c, off, 64);
    }
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) {
        red[0][wv] = a;
        red[1][wv] = b;
        red[2][wv] = c;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double s0 = 0, s1 = 0, s2 = 0;
        for (int k = 0; k < kThreads / 64; k++) {
            s0 += red[0][k];
            s1 += red[1][k];
            s2 += red[2][k];
        }
        partials[blockIdx.x * 3 + 0] = s0;
        partials[blockIdx.x * 3 + 1] = s1;
        partials[blockIdx.x * 3 + 2] = s2;
    }
}

struct FinalConsts {
    double rho0, kT, dv, prefactor;
};

// mode 0: df = ideal+ext gradient + excess gradient (energy_and_gradient)
// mode 1: df += excess gradient (excess_energy plug-in)
// mode 2: df = gamma(r, Omega) = -(prefactor / kT) proj2angl(proj), the OZ field in units of ln(rho/rho0)
// mode 3: proj holds gamma's projections, df = exp((-beta vext + proj2angl(proj)) / 2) (xi not read)
// mode 4: proj holds the projections of rho/rho0 - 1: df = 0 where the reference cold start
// excludes the solvent (beta vext >= -ln(DBL_EPSILON) - 0.05), else
// sqrt(max(1 + proj2angl(proj), MDFT_WS_DENSITY_FLOOR))
// mode 5 (specialised kernels only): df = proj2angl(proj)
template <int PT>
__global__ __launch_bounds__(kThreads) void final_f64(const double2 *__restrict__ proj, const double *__restrict__ xi,
                                                     const double *__restrict__ vext, double *__restrict__ df,
                                                     double *__restrict__ partials, size_t N, AngTables t,
                                                     FinalConsts k, int mode) {
    extern __shared__ double smem[];
    const int no = t.no, np = t.np, nth = t.ntheta, nphi = t.nphi, npsi = t.npsi, H1 = t.H + 1,
              W = 2 * t.L + 1, L = t.L;
    double2 *Gm = reinterpret_cast<double2 *>(smem);   // [PT][np]
    double2 *f = Gm + PT * np;                         // [PT][nth][W][H1]
    double2 *h = f + PT * nth * W * H1;                // [PT][nth][nphi][H1]
    const size_t r0 = (size_t)blockIdx.x * PT;
    const int npts = (int)((N - r0) < (size_t)PT ? (N - r0) : (size_t)PT);
    const int tid = threadIdx.x;
    const double2 *src = proj + r0 * np;
    for (int i = tid; i < npts * np; i += kThreads) Gm[i] = src[i];
    __syncthreads();
    // f(theta, mu2, mup) = sum_m p(m, mup, mu2) d(theta) fm(m)   (:215-224)
    const int nf = npts * nth * W * H1;
    for (int i = tid; i < nf; i += kThreads) {
        const int mu2 = i % H1;
        int rest = i / H1;
        const int mup = rest % W - L;
        rest /= W;
        const int it = rest % nth, pt = rest / nth;
        const int a = abs(mup), b = t.mrso * mu2;
        const int mlo = a > b ? a : b;
        double re = 0.0, im = 0.0;
        for (int m = mlo; m <= L; m++) {
            const int ip = t.pidx[(m * W + mup + L) * H1 + mu2];
            const double2 v = Gm[pt * np + ip];
            const double c = t.p2a[ip * nth + it];
            re += v.x * c;
            im += v.y * c;
        }
        f[i] = make_double2(re, im);
    }
    __syncthreads();
    // h(theta, phi, mu2) = sum_mup conj(f) exp(+i mup phi)
    const int nh = npts * nth * nphi * H1;
    for (int i = tid; i < nh; i += kThreads) {
        const int mu2 = i % H1;
        int rest = i / H1;
        const int iphi = rest % nphi;
        rest /= nphi;  // pt*nth + it
        const double2 *fr = f + (size_t)rest * W * H1 + mu2;
        double re = 0.0, im = 0.0;
        for (int mup = -L; mup <= L; mup++) {
            int kk = (mup * iphi) % nphi;
            kk += (kk < 0) ? nphi : 0;
            const double2 v = fr[(mup + L) * H1];
            // conj(v) * (c + i s)
            re += v.x * t.cph[kk] + v.y * t.sph[kk];
            im += v.x * t.sph[kk] - v.y * t.cph[kk];
        }
        h[i] = make_double2(re, im);
    }
    __syncthreads();
    double fid = 0.0, fext = 0.0, fexc = 0.0;
    const double rho0 = k.rho0, kT = k.kT, dv = k.dv;
    for (int i = tid; i < npts * no; i += kThreads) {
        const int pt = i / no, io = i - pt * no;
        const int ipsi = io % npsi, iphi = (io / npsi) % nphi, it = io / (npsi * nphi);
        const double2 *hr = h + ((size_t)(pt * nth + it) * nphi + iphi) * H1;
        // c2r: real part of the Hermitian-weighted sum over mu2 (weight 2 for mu2 > 0)
        double v = hr[0].x;
        for (int mu2 = 1; mu2 < H1; mu2++) {
            const int kk = (mu2 * ipsi) % npsi;
            v += 2.0 * (hr[mu2].x * t.cps[kk] - hr[mu2].y * t.sps[kk]);
        }
        const double wio = t.w[io];
        const double vexc = k.prefactor * wio * v;
        const size_t g = (r0 + pt) * (size_t)no + io;
        const double x = (mode >= 3) ? 0.0 : xi[g];
        const double rho = x * x * rho0;
        fexc += (x * x * rho0 - rho0) * vexc;
        if (mode == 0) {
            const double ve = vext[g];
            double gid = 0.0;
            if (rho > DBL_EPSILON) {
                const double lg = log(rho / rho0);
                fid += kT * dv * wio * (rho * lg - rho + rho0);
                fext += dv * wio * rho * ve;
                gid = wio * 2.0 * rho0 * x * (kT * lg + ve);
            } else {
                fid += kT * dv * wio * rho0;
            }
            if (df) df[g] = gid + 2.0 * rho0 * x * vexc;
        } else if (mode == 1) {
            if (df) df[g] += 2.0 * rho0 * x * vexc;
        } else if (mode == 2) {  // gamma(r, Omega) in units of ln(rho/rho0)
            if (df) df[g] = -(k.prefactor / kT) * v;
        } else if (mode == 3) {  // proj holds gamma's projections; df = exp((-beta vext + gamma) / 2)
            df[g] = exp(0.5 * fmin(fmax(-vext[g] / kT + v, -200.0), 7.0));
        } else {  // mode 4: proj holds the projections of rho/rho0 - 1;
                  // df = sqrt(max(1 + v, floor)), 0 where the cold start excludes the solvent
            df[g] = (vext[g] / kT >= -log(DBL_EPSILON) - 0.05) ? 0.0 : sqrt(fmax(1.0 + v, MDFT_WS_DENSITY_FLOOR));
        }
    }
    block_reduce3(fid, fext, fexc, partials);
}

// Ideal + external term alone (module_energy_ideal_and_external.f90:48-72); df accumulated.
__global__ __launch_bounds__(kThreads) void ideal_f64(const double *__restrict__ xi, const double *__restrict__ vext,
                                                     double *__restrict__ df, double *__restrict__ partials,
                                                     size_t total, int no, const double *__restrict__ w,
                                                     FinalConsts k) {
    double fid = 0.0, fext = 0.0, zero = 0.0;
    const double rho0 = k.rho0, kT = k.kT, dv = k.dv;
    for (size_t g = (size_t)blockIdx.x * kThreads + threadIdx.x; g < total; g += (size_t)gridDim.x * kThreads) {
        const int io = (int)(g % (size_t)no);
        const double x = xi[g], wio = w[io];
        const double rho = x * x * rho0;
        if (rho > DBL_EPSILON) {
            const double lg = log(rho / rho0);
            const double ve = vext[g];
            fid += kT * dv * wio * (rho * lg - rho + rho0);
            fext += dv * wio * rho * ve;
            if (df) df[g] += wio * 2.0 * rho0 * x * (kT * lg + ve);
        } else {
            fid += kT * dv * wio * rho0;
        }
    }
    block_reduce3(fid, fext, zero, partials);
}

// Sums of the per-workgroup (F_id, F_ext, F_exc) partials in a fixed order (so repeated
// evaluations are bitwise identical).  Workgroup (b, y) sums the b-th contiguous slice of array y
// (the gradient products are a second array of the same length) into out[y].
constexpr int kReduce = 1024;
struct ReduceArgs {
    const double *part[2];
    double *out[2];
};
__global__ __launch_bounds__(kReduce) void reduce3(ReduceArgs r, int nblocks) {
    const int per = (nblocks + gridDim.x - 1) / gridDim.x;
    const int lo = blockIdx.x * per, hi = min(nblocks, lo + per);
    const double *partials = r.part[blockIdx.y];
    double a = 0.0, b = 0.0, c = 0.0;
    for (int i = lo + threadIdx.x; i < hi; i += kReduce) {
        a += partials[3 * i + 0];
        b += partials[3 * i + 1];
        c += partials[3 * i + 2];
    }
    __shared__ double red[3][kReduce / 64];
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_down(a, off, 64);
        b += __shfl_down(b, off, 64);
        c += __shfl_down(c, off, 64);
    }
    const int wv = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        red[0][wv] = a;
        red[1][wv] = b;
        red[2][wv] = c;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        double s = 0.0;
        for (int w = 0; w < kReduce / 64; w++) s += red[threadIdx.x][w];
        r.out[blockIdx.y][3 * blockIdx.x + threadIdx.x] = s;
    }
}

// ---- specialisations for mrso = 2 with compile-time angular sizes: all
// index arithmetic uses constant divisors, loops have fixed trip counts, and
// the phase / Wigner / weight tables are staged in LDS once per workgroup.
template <int L>
struct Dims {
    static constexpr int NTH = L + 1, NPHI = 2 * L + 1, H = L / 2, H1 = H + 1, NPSI = 2 * H + 1, W = 2 * L + 1;
    static constexpr int NO = NTH * NPHI * NPSI;
    static constexpr int np_of(int m) { return m < 0 ? 0 : np_of(m - 1) + (2 * m + 1) * (m / 2 + 1); }
    static constexpr int NP = np_of(L);
};

// x / D for 0 <= x < NMAX as (x * M) >> S with a 24-bit multiply (one full-rate instruction;
// the 32-bit multiply-high of the compiler's constant division issues at a quarter rate).  M
// and S are chosen at compile time and checked against x / D for every x in the range.
template <unsigned D, unsigned NMAX>
struct DivC {
    static constexpr bool exact(unsigned long long m, unsigned s) {
        for (unsigned x = 0; x < NMAX; x++)
            if ((unsigned)((x * m) >> s) != x / D) return false;
        return true;
    }
    static constexpr unsigned pick() {
        for (unsigned s = 0; s < 32; s++) {
            const unsigned long long m = ((1ull << s) + D - 1) / D;
            if (m < (1ull << 24) && (NMAX - 1) * m < (1ull << 32) && exact(m, s)) return s;
        }
        return 32;
    }
    static constexpr unsigned S = pick();
    static_assert(S < 32 && NMAX <= (1u << 24), "no 24-bit reciprocal for this divisor and range");
    static constexpr unsigned M = (unsigned)(((1ull << S) + D - 1) / D);
    __device__ static unsigned q(unsigned x) { return __umul24(x, M) >> S; }
};

// a * b for a, b < 2^24 and a product below 2^32, kept a 24-bit multiply: the empty asm stops
// the compiler from folding the product into a subtraction or a 64-bit address, where it would
// become a quarter-rate 32-bit multiply again
__device__ inline unsigned mul24(unsigned a, unsigned b) {
    unsigned r = __umul24(a, b);
    asm("" : "+v"(r));
    return r;
}

// ---- the angular transforms by rows.  A row holds the values of one (point, theta) over
// (phi, psi), NPHI NPSI of them, and after the two DFTs its NF complex coefficients (mup, mu2):
// mu2 = 0: mup = 0 .. L (the others are their conjugates, the values being real), mu2 = 1 .. H:
// mup = -L .. L.  One thread transforms a row in registers, in place in LDS: both DFTs are of odd
// length n, so the terms j and n - j are added and subtracted first and the outputs k and -k share
// the sums, a third of the multiply-adds of the plain sums, and each value is read and written once
// (one thread per output reads n values and n twiddles for each).
template <int L> struct Rows : Dims<L> {
    using D = Dims<L>;
    static constexpr int ROW = D::NPHI * D::NPSI, NF = L + 1 + D::H * D::W;
    static constexpr int RS = (ROW > 2 * NF ? ROW : 2 * NF) | 1;  // odd: consecutive rows in different banks
    static constexpr int item(int mup, int mu2) { return mu2 == 0 ? mup : L + 1 + (mu2 - 1) * D::W + mup + L; }
};

// X(k) = sum_j x_j e^{+2 pi i j k / N}, k = -L .. L (at L + k), N = 2 L + 1
template <int N, typename T>
__device__ __forceinline__ void dft_odd(const T (&x)[N], const T (&y)[N], T (&ox)[N], T (&oy)[N]) {
    constexpr int L = N / 2;
    constexpr Turns<T, N> tw;
    T sx[L + 1], sy[L + 1], dx[L + 1], dy[L + 1];
    T x0 = x[0], y0 = y[0];
#pragma unroll
    for (int j = 1; j <= L; j++) {
        sx[j] = x[j] + x[N - j];
        sy[j] = y[j] + y[N - j];
        dx[j] = x[j] - x[N - j];
        dy[j] = y[j] - y[N - j];
        x0 += sx[j];
        y0 += sy[j];
    }
    ox[L] = x0;
    oy[L] = y0;
#pragma unroll
    for (int k = 1; k <= L; k++) {
        T ax = x[0], ay = y[0], bx = 0, by = 0;  // the cos sum, and the sin sum times i
#pragma unroll
        for (int j = 1; j <= L; j++) {
            const T c = tw.c[(j * k) % N], s = tw.s[(j * k) % N];
            ax = fma(sx[j], c, ax);
            ay = fma(sy[j], c, ay);
            bx = fma(-dy[j], s, bx);
            by = fma(dx[j], s, by);
        }
        ox[L + k] = ax + bx;
        oy[L + k] = ay + by;
        ox[L - k] = ax - bx;
        oy[L - k] = ay - by;
    }
}

template <int L, typename T> __device__ __forceinline__ void row_to_coefficients(T *row) {
    using R = Rows<L>;
    constexpr int NPHI = R::NPHI, NPSI = R::NPSI, H = R::H;
    constexpr Turns<T, NPHI> tw;
    constexpr Turns<T, NPSI> tp;
    T g0[NPHI], gx[H > 0 ? H : 1][NPHI], gy[H > 0 ? H : 1][NPHI];
#pragma unroll
    for (int j = 0; j < NPHI; j++) {
        const T v0 = row[j * NPSI];
        T s[H + 1], d[H + 1];
        g0[j] = v0;
#pragma unroll
        for (int p = 1; p <= H; p++) {
            const T a = row[j * NPSI + p], b = row[j * NPSI + NPSI - p];
            s[p] = a + b;
            d[p] = a - b;
            g0[j] += s[p];
        }
#pragma unroll
        for (int mu = 1; mu <= H; mu++) {
            T x = v0, y = 0;
#pragma unroll
            for (int p = 1; p <= H; p++) {
                x = fma(s[p], tp.c[(mu * p) % NPSI], x);
                y = fma(d[p], tp.s[(mu * p) % NPSI], y);
            }
            gx[mu - 1][j] = x;
            gy[mu - 1][j] = y;
        }
    }
    // mu2 = 0: real values, mup = 0 .. L
    {
        T x0 = g0[0], s[L + 1], d[L + 1];
#pragma unroll
        for (int j = 1; j <= L; j++) {
            s[j] = g0[j] + g0[NPHI - j];
            d[j] = g0[j] - g0[NPHI - j];
            x0 += s[j];
        }
        row[0] = x0;
        row[1] = x0;  // mup = 0 is real: its slot holds the value twice (see OutLane)
#pragma unroll
        for (int k = 1; k <= L; k++) {
            T a = g0[0], b = 0;
#pragma unroll
            for (int j = 1; j <= L; j++) {
                a = fma(s[j], tw.c[(j * k) % NPHI], a);
                b = fma(d[j], tw.s[(j * k) % NPHI], b);
            }
            row[2 * k] = a;
            row[2 * k + 1] = b;
        }
    }
#pragma unroll
    for (int mu = 0; mu < H; mu++) {
        T ox[NPHI], oy[NPHI];
        dft_odd<NPHI, T>(gx[mu], gy[mu], ox, oy);
#pragma unroll
        for (int k = 0; k < NPHI; k++) {
            row[2 * (L + 1 + mu * NPHI + k)] = ox[k];
            row[2 * (L + 1 + mu * NPHI + k) + 1] = oy[k];
        }
    }
}

// The phi synthesis of one (row, mu2), in place over its coefficients: mu2 = 0 (real values,
// coefficients doubled for mup > 0): h(phi_j) at row[j]; mu2 > 0: h(phi_j) = sum_mup conj(f) e^{i mup
// phi_j} at the item of mup = j - L.
template <int L, typename T> __device__ __forceinline__ void phi_synthesis0(T *row) {
    using R = Rows<L>;
    constexpr int N = R::NPHI;
    constexpr Turns<T, N> tw;
    T x[L + 1], y[L + 1], h0 = row[0];
    const T f0 = h0;
#pragma unroll
    for (int k = 1; k <= L; k++) {
        x[k] = row[2 * k];
        y[k] = row[2 * k + 1];
        h0 += x[k];
    }
    row[0] = h0;
#pragma unroll
    for (int j = 1; j <= L; j++) {
        T a = f0, b = 0;
#pragma unroll
        for (int k = 1; k <= L; k++) {
            a = fma(x[k], tw.c[(j * k) % N], a);
            b = fma(y[k], tw.s[(j * k) % N], b);
        }
        row[j] = a + b;
        row[N - j] = a - b;
    }
}
template <int L, typename T> __device__ __forceinline__ void phi_synthesis(T *f) {
    constexpr int N = 2 * L + 1;
    T x[N], y[N], ox[N], oy[N];
#pragma unroll
    for (int k = -L; k <= L; k++) {
        const int at = k < 0 ? N + k : k;
        x[at] = f[2 * (L + k)];
        y[at] = -f[2 * (L + k) + 1];
    }
    dft_odd<N, T>(x, y, ox, oy);
#pragma unroll
    for (int j = 0; j < N; j++) {
        const int at = j <= L ? L + j : j - L - 1;
        f[2 * j] = ox[at];
        f[2 * j + 1] = oy[at];
    }
}

// One projection of the theta contraction: out = (sum_it ax[it] F_it.x, sum_it ay[it] F_it.y) with
// F_it the coefficient at `item` of the rows of a point.  The signs of mup < 0 at mu2 = 0 (the
// conjugate of mup > 0 times (-1)^mup), the pairs of real projections and all norms are in the weights.
template <int L, typename T> struct OutLane {
    T ax[L + 1], ay[L + 1];
    int item;
};

// (m, mup, mu2) of packed entry e; of a pair of real projections m = 2 j and mup = 0
template <int L> __device__ inline void packed_entry(int e, int &m, int &mup, int &mu2) {
    using P = Packed<L>;
    m = mup = mu2 = 0;
    if (e >= P::pair0) {
        m = 2 * (e - P::pair0);
        return;
    }
    for (int it = 1; it < Rows<L>::NF; it++) {
        const int k = it <= L ? it : (it - L - 1) % P::W - L, u = it <= L ? 0 : (it - L - 1) / P::W + 1;
        const int o = P::off(k, u), lo = P::mlo(k, u);
        if (lo <= L && e >= o && e < o + L + 1 - lo) {
            m = lo + e - o;
            mup = k;
            mu2 = u;
            return;
        }
    }
}

// weights of the projections in the context's order, or (PACK) of the packed entries
template <int L, typename T, bool PACK>
__global__ void out_lanes_build(OutLane<L, T> *__restrict__ out, AngTables t) {
    using R = Rows<L>;
    constexpr int NOUT = PACK ? Packed<L>::np : R::NP;
    const double nrm = 1.0 / (double)(R::NPHI * R::NPSI);
    for (int i = threadIdx.x; i < NOUT; i += blockDim.x) {
        int m, mup, mu2, ip = i;
        if (PACK) {
            packed_entry<L>(i, m, mup, mu2);
            ip = t.pidx[(m * R::W + mup + L) * (R::H + 1) + mu2];
        } else {
            m = t.pm[ip];
            mup = t.pmup[ip];
            mu2 = t.pmu[ip] / 2;
        }
        const bool conj = mu2 == 0 && mup < 0, real = mu2 == 0 && mup == 0;
        const int ip2 = (PACK && real && m < L) ? t.pidx[((m + 1) * R::W + L) * (R::H + 1)] : -1;
        OutLane<L, T> o;
        for (int it = 0; it < R::NTH; it++) {
            // d^m(mup, 0) already has the sign (-1)^mup of d^m(-mup, 0)
            const double a = t.a2p[ip * R::NTH + it] * t.fm[ip] * nrm;
            const double a2 = ip2 < 0 ? 0.0 : t.a2p[ip2 * R::NTH + it] * t.fm[ip2] * nrm;
            o.ax[it] = (T)a;
            o.ay[it] = (T)(real ? a2 : (conj ? -a : a));
        }
        o.item = R::item(conj ? -mup : mup, mu2);
        out[i] = o;
    }
}

// feat = 0: o = rho0 (xi^2 - 1) (the excess term); feat = 1: o = clip(-beta xi / 2, -4, 4) / 4
// with xi the external potential -- the log of the square-root Boltzmann factor, bounded
// (features of the learned warm start); feat = 2: o = xi^2 - 1 = rho/rho0 - 1 (the
// warm start's density target; 0 in the bulk, -1 where the solvent is excluded); feat = 3:
// o = k0 aux / (xi w(io)) where xi^2 > MDFT_WS_DENSITY_FLOOR, else 0, with aux = dF at the
// density guess xi and k0 = dv / 2: dF/dr / w for r = rho/rho0, whose angl2proj is the
// adjoint of proj2angl up to a per-projection factor (the warm start's training gradient);
// feat = 4: o = xi (the plain transform). k0 is rho0 for feat 0.
// At 128^3, mmax 5, the stored 70 of 88 projections: FP64 reads 5.5 GB of xi and writes 2.35 GB in 1.61 ms, 4.9
// TB/s, HBM; FP32 with FP64 xi reads as much and writes 1.17 GB in 1.21 ms, 5.5 TB/s, HBM; with the FP32
// iterate of the fast minimiser it moves 3.9 GB in 1.16 ms, 3.4 TB/s, bound by vector issue (0.83 ms).  (One
// thread per psi sum, per phi sum and per projection, tables in LDS, all 88 projections: 2.22 ms FP32 and 3.72 ms
// FP64, the time of its reads of values and twiddles from LDS; by rows 1.22 and 1.79.)
// The theta contraction gives a thread one projection, its weights in registers, and a group of
// threads consecutive projections of a point, so the stores are whole records.
template <int L, int PT, int TH, typename T, bool PACK>
__global__ __launch_bounds__(TH) void angl2proj_t(const double *__restrict__ xi, typename C2<T>::t *__restrict__ proj,
                                                 size_t N, AngTables t, double k0, int feat, double beta,
                                                 const double *__restrict__ aux, const double *__restrict__ vsinv,
                                                 const float *__restrict__ xi32,
                                                 const OutLane<L, T> *__restrict__ lanes) {
    using R = Rows<L>;
    using V = typename C2<T>::t;
    constexpr int NO = R::NO, NTH = R::NTH, NOUT = PACK ? Packed<L>::np : R::NP, ROW = R::ROW, RS = R::RS;
    __shared__ T rows[NTH * PT * RS];  // row of (point, theta) at theta PT + point
    __shared__ double sth[NTH];        // 1 / s of each theta (the weights, hence s, depend on theta only)
    const int tid = threadIdx.x;
    const size_t r0 = (size_t)blockIdx.x * PT;
    const int npts = (int)((N - r0) < (size_t)PT ? (N - r0) : (size_t)PT);
    // all of a thread's loads are issued before the first is used
    constexpr int NIT = (PT * NO + TH - 1) / TH;
    const double *src = xi + r0 * NO;
    double xr[NIT];
#pragma unroll
    for (int q = 0; q < NIT; q++) {
        const int i = tid + q * TH;
        xr[q] = (i < npts * NO) ? (xi32 ? hold_f32(xi32[r0 * NO + i]) : src[i]) : 0.0;  // FP32 iterate: xi32
    }
    constexpr int G = TH / NOUT;  // groups of NOUT threads: each takes every G-th point of the theta contraction
    static_assert(G >= 1, "a projection per thread");
    const int grp = tid / NOUT, ip = tid - grp * NOUT;
    const OutLane<L, T> ln = lanes[ip];
    if (tid < NTH) sth[tid] = vsinv ? vsinv[tid * ROW] : 1.0;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NIT; q++) {
        const int i = tid + q * TH;
        if (i >= npts * NO) break;
        const unsigned pt = DivC<NO, PT * NO>::q(i);
        const unsigned io = i - mul24(pt, NO), it = DivC<ROW, NO>::q(io);
        T &o = rows[mul24(mul24(it, PT) + pt, RS) + (io - mul24(it, ROW))];
        const double xv = xi32 ? held_f32(xr[q]) : xr[q];
        const double x = vsinv ? xv * sth[it] : xv;  // scaled variables: xi = u / s
        if (feat == 0) o = (T)(k0 * (x * x - 1.0));
        else if (feat == 1) o = (T)(0.25 * fmin(fmax(-0.5 * beta * x, -4.0), 4.0));
        else if (feat == 2) o = (T)(x * x - 1.0);
        else if (feat == 4) o = (T)x;
        else o = (x * x > MDFT_WS_DENSITY_FLOOR * (1.0 + 1e-12)) ? (T)(k0 * aux[r0 * NO + i] / (x * t.w[io])) : (T)0;
    }
    __syncthreads();
    // points past the end leave their rows unread: nothing of them is stored
    for (int i = tid; i < NTH * PT; i += TH) row_to_coefficients<L, T>(rows + i * RS);
    __syncthreads();
    if (grp < G) {
        const T *f0 = rows + 2 * ln.item;
        V *dst = proj + r0 * NOUT + ip;
        for (int pt = grp; pt < npts; pt += G) {
            T re = 0, im = 0;
#pragma unroll
            for (int it = 0; it < NTH; it++) {
                const T *f = f0 + (it * PT + pt) * RS;
                re = fma(f[0], ln.ax[it], re);
                im = fma(f[1], ln.ay[it], im);
            }
            dst[(size_t)pt * NOUT] = mk<V>(re, im);
        }
    }
}

// ---- ln y, y > 0, by table (P. T. P. Tang, ACM Trans. Math. Softw. 16, 378 (1990)) ----------------
// y = 2^k z, z in [1/2, 1); d the multiple of 1/256 next to 1 / c, c the multiple of 1/256 next to z;
// r = z d - 1, |r| <= 0.005, all but exact in one fused operation; ln y = k ln 2 - ln d + ln(1 + r),
// the last by its series to r^7.  k ln 2 and -ln d are split at 2^-42, so that their upper parts add
// exactly (to 0 next to y = 1, where r is exact).  With the lower parts in the last sum: at most 0.57
// units in the last place (60 million values against extended precision).
constexpr int kLogC = 129;
constexpr double kLn2Hi = 0x1.62e42fefa38p-1, kLn2Lo = 0x1.ef35793c7673p-45;
struct LogTable {
    double2 c[kLogC];  // d, upper part of -ln d for c = 1/2 + j / 256
    double lo[kLogC];
};
__device__ __forceinline__ double log_table(double y, const LogTable &t) {
    const double z = __builtin_amdgcn_frexp_mant(y);
    const double k = (double)__builtin_amdgcn_frexp_exp(y);
    // the upper word of 1/2 ends in 21 zero bits: 7 bits of the fraction, rounded (infinity: 128; NaN: limited)
    const unsigned j0 = ((unsigned)__double2hiint(z) + 0x1000u) >> 13 & 0xffu, j = j0 < 128u ? j0 : 128u;
    const double2 c = t.c[j];
    const double r = fma(z, c.x, -1.0);
    double p = fma(r, 1.0 / 7, -1.0 / 6);
    p = fma(r, p, 1.0 / 5);
    p = fma(r, p, -1.0 / 4);
    p = fma(r, p, 1.0 / 3);
    p = fma(r, p, -1.0 / 2);
    const double h = fma(k, kLn2Hi, c.y), lo = fma(k, kLn2Lo, t.lo[j]);
    const double s = h + r, e = (h - s) + r;
    const double v = s + (e + fma(r * r, p, lo));
    return y < HUGE_VAL ? v : y;
}

// Points per tile of final_t and its least waves per SIMD: elements for whole rounds of 256 threads
// (330 x 6 = 7.7 rounds at mmax 5), as many as registers hold without spilling.  Measured, final
// pass at 128^3, mmax 5: fast variant 4, 5, 6, 7, 8 points 3.58, 3.42, 3.38, 3.55, 4.52 ms; FP32
// 4.54, 4.55, 3.85, 4.09, 3.97; FP64 6, 7, 8 points 4.32, 4.28, 4.69 ms; 100^3, mmax 4, FP64: 8, 9, 10
// points 1.37, 1.35, 1.34 ms; 96^3, mmax 3: 15, 18, 21 points 444, 439, 436 us.  5 waves per SIMD with
// smaller tiles: 5.97 ms, 1.84 ms, 456 us.
template <int L, typename T> struct FinalShape {
    static constexpr int PT32 = L == 5 ? 6 : L == 4 ? 9 : L == 3 ? 24 : L == 2 ? 32 : L == 1 ? 128 : 256;
    static constexpr int PT64 = L == 5 ? 7 : L == 4 ? 9 : L == 3 ? 18 : L == 2 ? 32 : L == 1 ? 128 : 256;
    static constexpr int PT = sizeof(T) == 4 ? PT32 : PT64;
    static constexpr int WAVES = 4;
};

// Bound by HBM: the fast variant moves 15.0 GB at 128^3, mmax 5, in 3.33 ms (4.5 TB/s; a plain copy
// reaches 4.8), FP64 19.0 GB in 4.28 ms (4.4).  (FP64 with the library's logarithm, 1.4 ms of vector issue, took
// 5.53 ms; 96^3, mmax 3 558 against 439 us, 75^3, mmax 2 152 against 115.)  The phi synthesis takes one
// thread per (row, mu2), in place; with one thread per (row, phi, mu2), each reading 11 coefficients
// and 11 twiddles from LDS for one output, the pass took 3.70 (fast) and 6.79 ms (FP64).
//
// Persistent: each workgroup stages the tables once and then takes tiles blockIdx.x,
// blockIdx.x + gridDim.x, ...  A tile needs no barrier beyond its three: every LDS array a
// tile writes was last read before a barrier that all threads have passed by then.  The
// free-energy sums and gradient products accumulate over a workgroup's tiles and are
// written once, one partial per workgroup.
// DOT32: mode 0 with an FP32 iterate, forming the gradient products over FP32 vectors (the
// evaluations of the fast minimiser), on at least PT points.  Every load of the tile is then
// issued on every path (the last partial round of a thread's elements with its index clamped
// into the tile), and dF is stored on every path: the wait before each use counts exactly the
// memory operations issued after it, so the product operands loaded ahead stay in flight.  The
// last tile of a grid that is not a whole number of tiles starts early, over points of the one
// before it (whose dF is written twice, with the same values); those add nothing to the sums.
template <int L, typename T, bool DOT32, bool PACK, bool EVAL = DOT32>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(FinalShape<L, T>::WAVES, 8))) void final_t(
    const typename C2<T>::t *__restrict__ proj, const double *__restrict__ xi, const double *__restrict__ vext,
    double *__restrict__ df, double *__restrict__ partials, size_t N, AngTables t, FinalConsts k, int mode,
    float *__restrict__ df32, const double *__restrict__ vsinv, DotArgs da, double *__restrict__ dpart,
    const float *__restrict__ xi32, const float *__restrict__ vext32) {
    using R = Rows<L>;
    using V = typename C2<T>::t;
    constexpr int PT = FinalShape<L, T>::PT;
    constexpr int NO = R::NO, NP = PACK ? Packed<L>::np : R::NP, NTH = R::NTH, NPSI = R::NPSI, H = R::H, W = R::W;
    constexpr int NW = PACK ? Packed<L>::pair0 + L + 1 : NP;  // rows of the theta weights
    constexpr int ROW = R::ROW, RS = R::RS, NF = R::NF;
    constexpr int NPS = NP | 1;  // odd: the records of consecutive points in different banks
    if constexpr (EVAL) mode = 0;
    if constexpr (EVAL && !DOT32) {
        xi32 = nullptr;
        df32 = nullptr;
    }
    __shared__ __align__(16) V Gm[PT * NPS];
    __shared__ T rows[NTH * PT * RS];  // row of (point, theta) at theta PT + point
    __shared__ V twpsi[NPSI * (H + 1)];  // (cos, sin)(2 pi mu2 ipsi / npsi) at [ipsi][mu2]
    // theta weights, twice the table's for mu2 > 0 (the weight of +-mu2 in the c2r) and, packed, for mup > 0
    // of mu2 = 0 (mup and -mup); by projection, or by packed entry with one row per m of the real ones
    __shared__ T p2a[NW * NTH];
    __shared__ double wth[NTH];          // the weights depend on theta only
    __shared__ double sth[NTH];          // 1 / s of each theta
    constexpr bool kLog = sizeof(T) == 8;
    __shared__ std::conditional_t<kLog, LogTable, char> lt;  // FP64
    // projection index or packed entry of (m, mup, mu2), projection index of (m, -mup, 0), as bytes: the loaded index is then known to be small
    // and its products stay 24-bit multiplies (entries with m below the item's lowest m are never read)
    static_assert(R::NP <= 255, "projection indices are stored as bytes");
    __shared__ unsigned char pidx[(L + 1) * NF], pneg[(L + 1) * (L + 1)];
    __shared__ unsigned char ford[NF];  // the theta synthesis' (mup, mu2) items, longest m loop first
    const int tid = threadIdx.x;
    auto mup_of = [](int it) { return it <= L ? it : (it - L - 1) % W - L; };
    auto mu_of = [](int it) { return it <= L ? 0 : (it - L - 1) / W + 1; };
    for (int i = tid; i < (L + 1) * NF; i += kThreads) {
        const int m = i / NF, it = i % NF, mup = mup_of(it), mu2 = mu_of(it), lo = Packed<L>::mlo(mup, mu2);
        const int ip = t.pidx[(m * W + mup + L) * (H + 1) + mu2];
        if (m < lo) continue;
        int row = ip;
        if constexpr (PACK) {
            row = it == 0 ? Packed<L>::pair0 + m : Packed<L>::off(mup, mu2) + m - lo;
            pidx[i] = (unsigned char)(it == 0 ? Packed<L>::pair0 + m / 2 : row);
        } else {
            pidx[i] = (unsigned char)ip;
        }
        const double f = (mu2 > 0 || (PACK && it != 0)) ? 2.0 : 1.0;
        for (int th = 0; th < NTH; th++) p2a[row * NTH + th] = (T)(f * t.p2a[ip * NTH + th]);
    }
    if constexpr (!PACK) {  // (mu2 = 0, mup < 0 has the weights of mup > 0 in its sum)
        for (int i = tid; i < (L + 1) * (L + 1); i += kThreads)
            pneg[i] = (unsigned char)t.pidx[((i / (L + 1)) * W - i % (L + 1) + L) * (H + 1)];
    }
    {
        // an item sums over m = max(|mup|, 2 mu2) .. L; ranked by that length (ties by index),
        // the lanes of a wave take loops of nearly one length
        auto len = [&](int it) {
            const int a = mup_of(it), b = 2 * mu_of(it);
            const int aa = a < 0 ? -a : a;
            return L + 1 - (aa > b ? aa : b);
        };
        for (int i = tid; i < NF; i += kThreads) {
            const int li = len(i);
            int r = 0;
            for (int j = 0; j < NF; j++) {
                const int lj = len(j);
                r += (lj > li || (lj == li && j < i)) ? 1 : 0;
            }
            ford[r] = (unsigned char)i;
        }
    }
    for (int i = tid; i < NPSI * (H + 1); i += kThreads) {
        const int kk = ((i % (H + 1)) * (i / (H + 1))) % NPSI;
        twpsi[i] = mk<V>((T)t.cps[kk], (T)t.sps[kk]);
    }
    for (int i = tid; i < NTH; i += kThreads) {
        wth[i] = t.w[i * ROW];
        sth[i] = vsinv ? vsinv[i * ROW] : 1.0;
    }
    if constexpr (kLog)
        for (int i = tid; i < (int)(sizeof(LogTable) / sizeof(double)); i += kThreads) reinterpret_cast<double *>(&lt)[i] = t.logt[i];
    double fid = 0.0, fext = 0.0, fexc = 0.0;
    double d0 = 0.0, d1 = 0.0, d2 = 0.0;  // products of dF with the DotArgs vectors
    double dss = 0.0;                     // DOT32: the product of dF with itself
    const double rho0 = k.rho0, kT = k.kT, dv = k.dv;
    const size_t ntiles = (N + PT - 1) / PT;
    for (size_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        // the thread index, opaque to the compiler in each tile: the tile's indices and LDS
        // addresses depend on the thread only, and hoisted out of the tile loop they would
        // all stay in registers (and spill)
        int tl = tid;
        asm volatile("" : "+v"(tl));
        const int skip = (DOT32 && (tile + 1) * PT > N) ? (int)((tile + 1) * PT - N) : 0;
        const size_t r0 = tile * PT - skip;
        const int npts = DOT32 ? PT : (int)((N - r0) < (size_t)PT ? (N - r0) : (size_t)PT);
        // DOT32: the tile's base pointers (uniform), indexed by 32-bit element offsets
        const float *xi32t = DOT32 ? xi32 + r0 * NO : nullptr, *vx32t = DOT32 ? vext32 + r0 * NO : nullptr;
        float *df32t = DOT32 ? df32 + r0 * NO : nullptr;
        const V *src = proj + r0 * NP;
        if constexpr (sizeof(T) == 4 && NP % 2 == 0) {  // FP32: 16-byte loads, two projections each
            for (int i = tl; i < npts * (NP / 2); i += kThreads) {
                const float4 v = reinterpret_cast<const float4 *>(src)[i];
                const unsigned pt = DivC<NP / 2, PT * (NP / 2)>::q(i);
                V *g = Gm + mul24(pt, NPS) + 2 * (i - mul24(pt, NP / 2));
                g[0] = mk<V>(v.x, v.y);
                g[1] = mk<V>(v.z, v.w);
            }
        } else {
            for (int i = tl; i < npts * NP; i += kThreads) {
                const unsigned pt = DivC<NP, PT * NP>::q(i);
                Gm[mul24(pt, NPS) + (i - mul24(pt, NP))] = src[i];
            }
        }
        // DOT32: the tile's FP32 iterate, FP32 vext and the FP32 operands of the first two
        // gradient products, loaded here so that their latency passes during the synthesis
        // phases; an operand that is not needed (the gradient itself, or beyond da.k) is read
        // from dF, which exists here
        constexpr int NIT = (PT * NO + kThreads - 1) / kThreads;
        float xr32[NIT], vr32[NIT];
        float dq[2][NIT];
        const float *dp0 = (da.k > 0 && !(da.self & 1)) ? static_cast<const float *>(da.p[0]) : df32;
        const float *dp1 = (da.k > 1 && !((da.self >> 1) & 1)) ? static_cast<const float *>(da.p[1]) : df32;
        const float *dp0t = DOT32 ? dp0 + r0 * NO : nullptr, *dp1t = DOT32 ? dp1 + r0 * NO : nullptr;
        if constexpr (DOT32) {
    #pragma unroll
            for (int q = 0; q < NIT; q++) {
                const int i = tl + q * kThreads;
                const int ii = i < npts * NO ? i : npts * NO - 1;
                xr32[q] = xi32t[ii];
                vr32[q] = vx32t[ii];
                dq[0][q] = dp0t[ii];
                dq[1][q] = dp1t[ii];
            }
        }
        // the general variant: the tile's xi and vext, all of a thread's loads issued together:
        // before the synthesis phases where the registers allow it (FP32, and FP64 for mmax <= 3: 96^3,
        // mmax 3: 0.577 -> 0.556 ms; FP64 at mmax 5 would spill), else before the loop that uses them
        constexpr bool kEarly = sizeof(T) == 4 || L <= 3;
        double xr[NIT], vr[NIT];
        auto load_general = [&]() {
    #pragma unroll
            for (int q = 0; q < NIT; q++) {
                const int i = tl + q * kThreads;
                xr[q] = 0.0;
                vr[q] = 0.0;
                if (i < npts * NO) {
                    const size_t g = r0 * NO + i;
                    if (mode < 3) xr[q] = xi32 ? hold_f32(xi32[g]) : xi[g];  // FP32 iterate: xi32
                    if (mode == 0 || mode == 3 || mode == 4) vr[q] = vext[g];
                }
            }
        };
        if constexpr (!DOT32 && kEarly) load_general();
        __syncthreads();
        // f(theta, mup, mu2) = sum_m p(m, mup, mu2) d(theta) fm(m): one thread per (point, mup, mu2),
        // all theta at once (each projection read once); items by rank of their loop length, the
        // tile's points innermost.  mu2 = 0: the psi step takes the real part of the sum over mup, so
        // the items mup > 0 hold p(m, mup, 0) + (-1)^mup conj(p(m, -mup, 0)), packed twice p(m, mup, 0),
        // and mup = 0 the real part
        for (int i = tl; i < PT * NF; i += kThreads) {
            const int rk = i / PT, pt = i - rk * PT;
            if (pt >= npts) continue;
            const int item = ford[rk];
            int mlo, neg = 0;  // lowest m; 1, 2: mu2 = 0 with mup > 0, = 0
            if (item <= L) {
                mlo = item;
                neg = item > 0 ? 1 : 2;
            } else {
                const int rest = item - (L + 1), mu1 = (int)DivC<W, (H > 0 ? H : 1) * W>::q(rest);
                const int mup = rest - mu1 * W - L, a = mup < 0 ? -mup : mup, b = 2 * mu1 + 2;
                mlo = a > b ? a : b;
            }
            [[maybe_unused]] const T sg = (item & 1) ? (T)-1 : (T)1;
            T re[NTH], im[NTH];
    #pragma unroll
            for (int it = 0; it < NTH; it++) re[it] = im[it] = (T)0;
            const V *gp = Gm + mul24(pt, NPS);
            for (int m = mlo; m <= L; m++) {
                const unsigned p = pidx[m * NF + item];
                V v = gp[p];
                const T *c = p2a + p * NTH;
                if constexpr (PACK) {
                    if (neg == 2) {
                        if (m & 1) v.x = v.y;
                        c = p2a + (Packed<L>::pair0 + m) * NTH;
                    }
                } else if (neg == 1) {
                    const V u = gp[pneg[m * (L + 1) + item]];
                    v.x = fma(sg, u.x, v.x);
                    v.y = fma(-sg, u.y, v.y);
                }
    #pragma unroll
                for (int it = 0; it < NTH; it++) {
                    re[it] += v.x * c[it];
                    im[it] += v.y * c[it];
                }
            }
            T *fo = rows + (mul24(pt, RS) + 2 * item);
    #pragma unroll
            for (int it = 0; it < NTH; it++) {
                fo[it * (PT * RS)] = re[it];
                fo[it * (PT * RS) + 1] = neg == 2 ? (T)0 : im[it];
            }
        }
        __syncthreads();
        // h(theta, phi, mu2), one thread per (row, mu2), in place; mu2-major, so that whole waves
        // take mu2 = 0 (points past the end: their rows are never read)
        for (int i = tl; i < NTH * PT * (H + 1); i += kThreads) {
            const int mu2 = (int)DivC<NTH * PT, NTH * PT * (H + 1)>::q(i), row = i - mu2 * (NTH * PT);
            T *f = rows + mul24(row, RS);
            if (mu2 == 0) phi_synthesis0<L, T>(f);
            else phi_synthesis<L, T>(f + 2 * (L + 1) + mul24(mu2 - 1, 2 * W));
        }
        __syncthreads();
        if constexpr (!DOT32 && !kEarly) load_general();
        // FP32 path: the free-energy terms of a thread's elements in this tile, summed in FP32
        // and added to the FP64 sums once per tile
        float fexc_t = 0.0f, fid_t = 0.0f, fext_t = 0.0f;
    #pragma unroll
        for (int q = 0; q < NIT; q++) {
            const int i = tl + q * kThreads;
            if (i >= npts * NO) break;
            double xq;
            float ve32 = 0.0f;
            if constexpr (DOT32) {
                float xv = xr32[q];
                ve32 = vr32[q];
                asm volatile("" : "+v"(xv), "+v"(ve32));  // the conversion stays here, not next to the load
                xq = (double)xv;
            } else {
                xq = xi32 ? held_f32(xr[q]) : xr[q];
            }
            // LDS offsets by 24-bit products: every operand here is small and non-negative
            const unsigned pt = DivC<NO, PT * NO>::q(i);
            const unsigned io = i - mul24(pt, NO), it = DivC<ROW, NO>::q(io);
            const unsigned col = io - mul24(it, ROW), iphi = DivC<NPSI, ROW>::q(col), ipsi = col - mul24(iphi, NPSI);
            const T *hr = rows + mul24(mul24(it, PT) + pt, RS);
            const V *tp = twpsi + mul24(ipsi, H + 1);
            T vt = hr[iphi];
            hr += 2 * (L + 1) + 2 * iphi;
    #pragma unroll
            for (int mu2 = 1; mu2 <= H; mu2++) {
                const T hx = hr[(mu2 - 1) * 2 * W], hy = hr[(mu2 - 1) * 2 * W + 1];
                vt = fma(-hy, tp[mu2].y, fma(hx, tp[mu2].x, vt));
            }
            const size_t g = r0 * NO + i;
            if constexpr (sizeof(T) == 4) {
                if (mode == 0) {
                    // FP32 path: the per-orientation terms in FP32 (the transforms feeding them
                    // are FP32 already), summed in FP32 over the thread's elements of the tile
                    // and in FP64 over the tiles; rho/rho0 - 1 is formed in FP64 first so that
                    // the excess term keeps its small deviations from the bulk
                    const double si = vsinv ? sth[it] : 1.0;  // scaled variables: xi = u / s, dF/du = dF/dxi / s
                    const double x = xq * si;
                    const double xx = x * x;
                    const float wf = (float)wth[it];
                    const float ws = DOT32 && (int)pt < skip ? 0.0f : wf;  // weight in the sums
                    const float vexcf = (float)k.prefactor * wf * vt;
                    const float drf = (float)(xx - 1.0);
                    const float rho0f = (float)rho0, x2 = (float)xx, xf = (float)x;
                    fexc_t += rho0f * drf * ((float)k.prefactor * ws * vt);
                    float gid = 0.0f;
                    if (xx * rho0 > DBL_EPSILON) {
                        // ln(rho / rho0) from the hardware base-2 logarithm: x2 > 6e-15 here (rho > DBL_EPSILON),
                        // a normal FP32 number, so logf's denormal scaling and its extra-precise
                        // product with ln 2 change nothing at this path's FP32 accuracy
                        const float lg = __builtin_amdgcn_logf(x2) * 0.693147181f;
                        const float ve = DOT32 ? ve32 : (float)vr[q];
                        const float kTf = (float)kT, dvf = (float)dv;
                        fid_t += kTf * dvf * ws * rho0f * (x2 * lg - drf);
                        fext_t += dvf * ws * rho0f * x2 * ve;
                        gid = wf * 2.0f * rho0f * xf * (kTf * lg + ve);
                    } else {
                        fid_t += (float)(kT * dv * rho0) * ws;
                    }
                    const float gv = (gid + 2.0f * rho0f * xf * vexcf) * (float)si;
                    if constexpr (DOT32) {
                        df32t[i] = gv;
                        const double gd = (int)pt < skip ? 0.0 : (double)gv;
                        // the empty asm keeps the conversions here: hoisted next to the loads above,
                        // they would make each load wait
                        float o0 = dq[0][q], o1 = dq[1][q];
                        asm volatile("" : "+v"(o0), "+v"(o1));
                        // every product is formed (an operand that is not needed was read from dF
                        // and is discarded at the end); the gradient's own product separately
                        dss = fma(gd, gd, dss);
                        d0 = fma(gd, (double)o0, d0);
                        d1 = fma(gd, (double)o1, d1);
                        if (da.k > 2 && !((da.self >> 2) & 1)) d2 += gd * (double)static_cast<const float *>(da.p[2])[g];
                        continue;
                    }
                    if (df32) df32[g] = gv;
                    else if (df) df[g] = (double)gv;
                    if (da.k > 0) {
                        d0 += (double)gv * dot_operand(da, 0, g, (double)gv);
                        if (da.k > 1) d1 += (double)gv * dot_operand(da, 1, g, (double)gv);
                        if (da.k > 2) d2 += (double)gv * dot_operand(da, 2, g, (double)gv);
                    }
                    continue;
                }
            }
            // from here on FP64: free-energy reductions, rho ln rho and the gradient
            const double v = (double)vt;
            const double wio = wth[it];
            const double vexc = k.prefactor * wio * v;
            const double si = (mode == 0 && vsinv) ? sth[it] : 1.0;  // scaled variables (mode 0)
            const double x = xq * si;
            const double rho = x * x * rho0;
            fexc += (x * x * rho0 - rho0) * vexc;
            if (mode == 0) {
                const double ve = vr[q];
                double gid = 0.0;
                if (rho > DBL_EPSILON) {
                    double lg = 0.0;  // ln(rho / rho0)
                    if constexpr (kLog) lg = log_table(x * x, lt);
                    fid += kT * dv * wio * (rho * lg - rho + rho0);
                    fext += dv * wio * rho * ve;
                    gid = wio * 2.0 * rho0 * x * (kT * lg + ve);
                } else {
                    fid += kT * dv * wio * rho0;
                }
                const double gv = (gid + 2.0 * rho0 * x * vexc) * si;
                if (df32) df32[g] = (float)gv;
                else if (df) df[g] = gv;
                // (the FP64 kernel forms no gradient products: its context runs the separate
                // multi-dot, which keeps this kernel's registers where they were)
            } else if (mode == 1) {
                if (df) df[g] += 2.0 * rho0 * x * vexc;
            } else if (mode == 2) {  // gamma(r, Omega) in units of ln(rho/rho0)
                if (df) df[g] = -(k.prefactor / kT) * v;
            } else if (mode == 3) {  // proj holds gamma's projections; df = exp((-beta vext + gamma) / 2)
                df[g] = exp(0.5 * fmin(fmax(-vr[q] / kT + v, -200.0), 7.0));
            } else if (mode == 4) {  // proj holds the projections of rho/rho0 - 1;
                                     // df = sqrt(max(1 + v, floor)), 0 where the cold start excludes the solvent
                df[g] = (vr[q] / kT >= -log(DBL_EPSILON) - 0.05) ? 0.0 : sqrt(fmax(1.0 + v, MDFT_WS_DENSITY_FLOOR));
            } else {  // mode 5: df = proj2angl(proj), the plain transform
                df[g] = v;
            }
        }
        fexc += (double)fexc_t;
        fid += (double)fid_t;
        fext += (double)fext_t;
    }
    block_reduce3(fid, fext, fexc, partials);
    if constexpr (sizeof(T) == 4) {
        if (da.k > 0) {
            if constexpr (DOT32) {
                if (da.self & 1) d0 = dss;
                if ((da.self >> 1) & 1) d1 = dss;
                if ((da.self >> 2) & 1) d2 = dss;
            }
            __syncthreads();
            block_reduce3(d0, d1, d2, dpart);
        }
    }
}

constexpr size_t kMinTile = 4;  // the specialised kernels take at least as many points per workgroup
constexpr int kPT = 4;  // points per workgroup tile (keeps the LDS tile under 64 KB at mmax = 5)

// Workgroups of a persistent kernel, never more than the tiles.  resident_grid: as many as
// the compute units hold at once (registers and LDS of that kernel); a larger grid leaves
// workgroups waiting for a slot until others have finished all their tiles.  The fast final
// pass runs faster so; the general final pass runs faster with 8 per compute unit (about twice the
// resident number), the later ones taking the slots of the first to finish.
template <typename K>
size_t resident_grid(const mdft_ctx *c, K kernel, size_t ntiles) {
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kThreads, 0) != hipSuccess || per_cu < 1) per_cu = 1;
    const size_t g = (size_t)per_cu * (size_t)(c->num_cus > 0 ? c->num_cus : 256);
    return ntiles < g ? ntiles : g;
}
size_t oversubscribed_grid(const mdft_ctx *c, size_t ntiles) {
    const size_t g = 8 * (size_t)(c->num_cus > 0 ? c->num_cus : 256);
    return ntiles < g ? ntiles : g;
}

size_t a2p_lds(const AngTables &t) {
    return sizeof(double) * kPT * t.no + sizeof(double2) * kPT * t.ntheta * t.nphi * (t.H + 1) +
           sizeof(double2) * kPT * t.ntheta * (2 * t.L + 1) * (t.H + 1);
}
size_t final_lds(const AngTables &t) {
    return sizeof(double2) * kPT * t.np + sizeof(double2) * kPT * t.ntheta * (2 * t.L + 1) * (t.H + 1) +
           sizeof(double2) * kPT * t.ntheta * t.nphi * (t.H + 1);
}

hipError_t ensure_partials(mdft_ctx *c, size_t nblocks) {
    if (c->partials_cap >= nblocks * 3) return hipSuccess;
    if (c->d_partials) (void)dev_free(c->d_partials);
    c->d_partials = nullptr;
    c->partials_cap = 0;
    hipError_t e = dev_malloc(&c->d_partials, sizeof(double) * nblocks * 3);
    if (e == hipSuccess) c->partials_cap = nblocks * 3;
    return e;
}

}  // namespace

// Points per workgroup and threads of angl2proj_t: about as many rows (L + 1 per point) as a
// workgroup's threads can take in one round, in LDS that leaves three or more workgroups on a
// compute unit.  Measured at 128^3, mmax 5, FP32 / FP64: 16 points, 256 threads 1.22 / 1.79 ms, 128
// threads 1.26 / 2.47; 32 points 1.26 / 3.69 (one FP64 workgroup per compute unit); 8 points, 128
// threads 1.27 / 1.78.  100^3, mmax 4, FP64: 192 threads 0.54, 256 0.64 ms.
template <int L> struct A2pShape {
    static constexpr int PT = L >= 4 ? 16 : L == 3 ? 32 : L == 2 ? 64 : L == 1 ? 128 : 256, TH = L == 4 ? 192 : 256;
};

template <typename T, bool PACK = false>
bool launch_a2p_t(mdft_ctx *c, const double *xi, typename C2<T>::t *proj, int feat = 0, const double *aux = nullptr,
                  size_t npts = 0) {
    if (!npts) npts = c->N;
    const double beta = 1.0 / c->d.kT;
    const double k0 = (feat == 3) ? 0.5 * c->dv : c->rho0;
    void *&img = c->d_a2p_img[(sizeof(T) == 8) + 2 * PACK];
    switch (c->L) {
#define A2P_CASE(LL) \
    case LL: { \
        using S = A2pShape<LL>; \
        if (!img) { \
            if (dev_malloc(&img, sizeof(OutLane<LL, T>) * Rows<LL>::NP) != hipSuccess) { img = nullptr; return false; } \
            hipLaunchKernelGGL((out_lanes_build<LL, T, PACK>), dim3(1), dim3(128), 0, c->stream, static_cast<OutLane<LL, T> *>(img), c->ang); \
        } \
        hipLaunchKernelGGL((angl2proj_t<LL, S::PT, S::TH, T, PACK>), dim3((unsigned)((npts + S::PT - 1) / S::PT)), dim3(S::TH), 0, c->stream, xi, proj, npts, c->ang, k0, feat, beta, aux, feat == 0 ? c->vsinv : nullptr, feat == 0 ? c->xi32 : nullptr, static_cast<const OutLane<LL, T> *>(img)); \
        return true; \
    }
        A2P_CASE(0) A2P_CASE(1) A2P_CASE(2) A2P_CASE(3) A2P_CASE(4) A2P_CASE(5)
#undef A2P_CASE
        default: return false;
    }
}

// the table of log_table, built in extended precision
int log_setup(mdft_ctx *c) {
    LogTable h;
    for (int j = 0; j < kLogC; j++) {
        const double d = nearbyint(256.0 / (0.5 + j / 256.0)) / 256.0;
        const long double l = -logl((long double)d);
        const double hi = (double)(nearbyintl(l * 0x1p42L) * 0x1p-42L);
        h.c[j] = make_double2(d, j == 0 ? -kLn2Hi : hi);
        h.lo[j] = j == 0 ? -kLn2Lo : (double)(l - (long double)hi);
    }
    void *p = nullptr;
    if (dev_malloc(&p, sizeof(h)) != hipSuccess) return MDFT_ENOMEM;
    c->d_logt = p;
    c->ang.logt = static_cast<const double *>(p);
    return hipMemcpy(p, &h, sizeof(h), hipMemcpyHostToDevice) == hipSuccess ? MDFT_OK : MDFT_EHIP;
}

template <typename T, bool PACK = false>
bool launch_final_t(mdft_ctx *c, const typename C2<T>::t *proj, const double *xi, double *df, int mode, FinalConsts k,
                    size_t npts = 0, size_t *grid_out = nullptr) {
    if (!npts) npts = c->N;
    DotArgs da{};
    if (mode == 0 && c->dot_k > 0) {
        da.k = c->dot_k;
        da.self = c->dot_self;
        da.f32 = c->df32 != nullptr;
        for (int j = 0; j < 3; j++) da.p[j] = c->dot_vec[j];
    }
    // the FP32 kernel forming products over FP32 vectors (dF then FP32 too) has its own variant
    [[maybe_unused]] const bool dot32 = sizeof(T) == 4 && mode == 0 && da.k > 0 && da.f32 && c->xi32 && c->vext32_ok;
    switch (c->L) {
#define FIN_CASE(LL) \
    case LL: { \
        constexpr int PT = FinalShape<LL, T>::PT; \
        const size_t ntiles = (npts + PT - 1) / PT; \
        if constexpr (PACK && sizeof(T) == 4) { \
            if (dot32 && npts >= PT) { \
                const size_t nb = resident_grid(c, final_t<LL, T, true, true>, ntiles); \
                if (grid_out) *grid_out = nb; \
                hipLaunchKernelGGL((final_t<LL, T, true, true>), dim3((unsigned)nb), dim3(kThreads), 0, c->stream, proj, xi, c->d_vext, df, c->d_partials, npts, c->ang, k, mode, c->df32, c->vsinv, da, c->d_dpart, c->xi32, c->d_vext32); \
                return true; \
            } \
        } \
        const size_t nb = oversubscribed_grid(c, ntiles); \
        if constexpr (PACK && sizeof(T) == 8) { \
            if (mode == 0 && !c->df32 && !c->xi32) { \
                if (grid_out) *grid_out = nb; \
                hipLaunchKernelGGL((final_t<LL, T, false, true, true>), dim3((unsigned)nb), dim3(kThreads), 0, c->stream, proj, xi, c->d_vext, df, c->d_partials, npts, c->ang, k, 0, nullptr, c->vsinv, da, c->d_dpart, nullptr, nullptr); \
                return true; \
            } \
        } \
        if (grid_out) *grid_out = nb; \
        hipLaunchKernelGGL((final_t<LL, T, false, PACK>), dim3((unsigned)nb), dim3(kThreads), 0, c->stream, proj, xi, c->d_vext, df, c->d_partials, npts, c->ang, k, mode, mode == 0 ? c->df32 : nullptr, mode == 0 ? c->vsinv : nullptr, da, c->d_dpart, mode == 0 ? c->xi32 : nullptr, nullptr); \
        return true; \
    }
        FIN_CASE(0) FIN_CASE(1) FIN_CASE(2) FIN_CASE(3) FIN_CASE(4) FIN_CASE(5)
#undef FIN_CASE
        default: return false;
    }
}


hipError_t launch_angl2proj_f64(mdft_ctx *c, const double *xi, double2 *proj) {
    if (c->packed) return launch_a2p_t<double, true>(c, xi, proj) ? hipGetLastError() : hipErrorNotSupported;
    if (c->d.mrso == 2 && launch_a2p_t<double>(c, xi, proj)) return hipGetLastError();
    const size_t nb = (c->N + kPT - 1) / kPT;
    if (a2p_lds(c->ang) > c->lds_limit) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL(angl2proj_f64<kPT>, dim3((unsigned)nb), dim3(kThreads), a2p_lds(c->ang), c->stream, xi, proj,
                       c->N, c->ang, c->rho0);
    return hipGetLastError();
}

hipError_t launch_final_f64(mdft_ctx *c, const double2 *proj, const double *xi, double *df, int mode,
                            int *nblocks_out) {
    const size_t nb = (c->N + kPT - 1) / kPT;
    if (final_lds(c->ang) > c->lds_limit) return hipErrorInvalidConfiguration;
    hipError_t e = ensure_partials(c, nb);
    if (e != hipSuccess) return e;
    FinalConsts k;
    k.rho0 = c->rho0;
    k.kT = c->d.kT;
    k.dv = c->dv;
    const double pi = acos(-1.0);
    const double fourpisq = 4.0 * pi * pi;
    k.prefactor = -c->d.kT * 2.0 * fourpisq / c->d.mrso / c->d.n0;  // cproj_mrso.f90:728
    if (c->d.mrso == 2) {
        const size_t nbt = (c->N + kMinTile - 1) / kMinTile;
        if ((e = ensure_partials(c, nbt)) != hipSuccess) return e;
        size_t grid = 0;
        if (c->packed ? launch_final_t<double, true>(c, proj, xi, df, mode, k, 0, &grid)
                      : launch_final_t<double>(c, proj, xi, df, mode, k, 0, &grid)) {
            *nblocks_out = (int)grid;
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL(final_f64<kPT>, dim3((unsigned)nb), dim3(kThreads), final_lds(c->ang), c->stream, proj, xi,
                       c->d_vext, df, c->d_partials, c->N, c->ang, k, mode);
    *nblocks_out = (int)nb;
    return hipGetLastError();
}

hipError_t launch_ideal_f64(mdft_ctx *c, const double *xi, double *df, int *nblocks_out) {
    const size_t total = c->N * (size_t)c->no;
    size_t nb = (total + kThreads - 1) / kThreads;
    if (nb > 65536) nb = 65536;
    hipError_t e = ensure_partials(c, nb);
    if (e != hipSuccess) return e;
    FinalConsts k;
    k.rho0 = c->rho0;
    k.kT = c->d.kT;
    k.dv = c->dv;
    k.prefactor = 0.0;
    hipLaunchKernelGGL(ideal_f64, dim3((unsigned)nb), dim3(kThreads), 0, c->stream, xi, c->d_vext, df, c->d_partials,
                       total, c->no, c->d_w, k);
    *nblocks_out = (int)nb;
    return hipGetLastError();
}

// out[0..2] <- the sums of d_partials and, where products is set, prod_out[0..2] <- those of d_dpart.  The
// outputs are pinned host memory, written by the kernel itself: a copy after it, and a reduction of
// its own for the products, made the end of an evaluation 20 us where this takes 8.
hipError_t launch_reduce3(mdft_ctx *c, int nblocks, double *out, double *prod_out) {
    constexpr int kSlices = 512;
    ReduceArgs r{{c->d_partials, c->d_dpart}, {out, prod_out}};
    const unsigned arrays = prod_out ? 2 : 1;
    if (nblocks > 8 * kReduce) {  // (the specialised final passes have at most 8 workgroups per compute unit)
        if (!c->d_slices) {
            hipError_t e = dev_malloc(&c->d_slices, sizeof(double) * 6 * kSlices);
            if (e != hipSuccess) return e;
        }
        ReduceArgs s{{c->d_partials, c->d_dpart}, {c->d_slices, c->d_slices + 3 * kSlices}};
        hipLaunchKernelGGL(reduce3, dim3(kSlices, arrays), dim3(kReduce), 0, c->stream, s, nblocks);
        r.part[0] = c->d_slices;
        r.part[1] = c->d_slices + 3 * kSlices;
        nblocks = kSlices;
    }
    hipLaunchKernelGGL(reduce3, dim3(1, arrays), dim3(kReduce), 0, c->stream, r, nblocks);
    return hipGetLastError();
}

FinalConsts final_consts(mdft_ctx *c) {
    FinalConsts k;
    k.rho0 = c->rho0;
    k.kT = c->d.kT;
    k.dv = c->dv;
    const double pi = acos(-1.0);
    k.prefactor = -c->d.kT * 2.0 * (4.0 * pi * pi) / c->d.mrso / c->d.n0;  // cproj_mrso.f90:728
    return k;
}

hipError_t launch_angl2proj_f32(mdft_ctx *c, const double *xi, float2 *proj) {
    if (c->packed) return launch_a2p_t<float, true>(c, xi, proj) ? hipGetLastError() : hipErrorNotSupported;
    if (c->d.mrso != 2 || !launch_a2p_t<float>(c, xi, proj)) return hipErrorNotSupported;
    return hipGetLastError();
}

hipError_t launch_final_f32(mdft_ctx *c, const float2 *proj, const double *xi, double *df, int mode, int *nblocks_out) {
    const size_t nbt = (c->N + kMinTile - 1) / kMinTile;
    hipError_t e = ensure_partials(c, nbt);
    if (e != hipSuccess) return e;
    size_t grid = 0;
    if (c->d.mrso != 2 || !(c->packed ? launch_final_t<float, true>(c, proj, xi, df, mode, final_consts(c), 0, &grid)
                                      : launch_final_t<float>(c, proj, xi, df, mode, final_consts(c), 0, &grid)))
        return hipErrorNotSupported;
    *nblocks_out = (int)grid;
    return hipGetLastError();
}

// angl2proj of a warm-start field into the context's projection buffer (mrso = 2 kernels):
// feat 1: the feature field of src = vext; feat 2: the density target rho/rho0 - 1 of src = xi;
// feat 3: the start gradient field of src = xi with aux = dF
hipError_t launch_angl2proj_feat(mdft_ctx *c, const double *src, int feat, const double *aux) {
    if (c->d.mrso != 2) return hipErrorNotSupported;
    if (!aux) aux = c->d_vext;
    bool ok = (c->d.precision == MDFT_PREC_FP64)
                  ? launch_a2p_t<double>(c, src, static_cast<double2 *>(c->d_proj), feat, aux)
                  : launch_a2p_t<float>(c, src, static_cast<float2 *>(c->d_proj), feat, aux);
    return ok ? hipGetLastError() : hipErrorNotSupported;
}

// The plain FP64 transforms of npts points (any count, not only the context's grid):
// proj [npts][np] = angl2proj(f [npts][no]) and f = proj2angl(proj); mrso = 2 kernels.
hipError_t launch_transform_f64(mdft_ctx *c, const double *f, double2 *proj, size_t npts, bool to_proj) {
    if (c->d.mrso != 2) return hipErrorNotSupported;
    if (to_proj) return launch_a2p_t<double>(c, f, proj, 4, nullptr, npts) ? hipGetLastError() : hipErrorNotSupported;
    hipError_t e = ensure_partials(c, (npts + kMinTile - 1) / kMinTile);
    if (e != hipSuccess) return e;
    return launch_final_t<double>(c, proj, nullptr, const_cast<double *>(f), 5, final_consts(c), npts)
               ? hipGetLastError()
               : hipErrorNotSupported;
}
