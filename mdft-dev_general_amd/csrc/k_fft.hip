// k_fft.hip -- batched 3D complex FFTs of all projections, FP64 and FP32.
//
// Replaces the FFTW plans of src/module_energy_cproj_mrso.f90:256-267 and the
// transforms at :306-329 (sign +1, unnormalised) and :690-719 (sign -1, then
// scaled by 1/(nx ny nz)).  The projection field is stored as the reference's
// deltarho_p(np,nx,ny,nz): projection index fastest.  A pass transforms one axis
// in place.  For each of them the field is [outer][n][C] with C contiguous columns:
// C = np along x, nx np along y and nx ny np along z.  A workgroup takes PB columns
// (128 bytes) of one outer index, runs a mixed-radix Stockham FFT and writes the
// lines back.  Along y and z the columns of a workgroup may belong to two grid points,
// so that every workgroup but the last has PB of them whatever np is.
#include "mdft_internal.h"
#include "turns.h"

namespace {

constexpr int kThreads = 256;

template <typename T> struct C2;
template <> struct C2<double> { using t = double2; };
template <> struct C2<float> { using t = float2; };

template <typename V> __device__ inline V mk(decltype(V::x) a, decltype(V::x) b) { V v; v.x = a; v.y = b; return v; }
template <typename V> __device__ inline V cmul(V a, V b) { return mk<V>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
template <typename V> __device__ inline V cadd(V a, V b) { return mk<V>(a.x + b.x, a.y + b.y); }
template <typename V> __device__ inline V csub(V a, V b) { return mk<V>(a.x - b.x, a.y - b.y); }
// multiply by s*i
template <typename V> __device__ inline V mul_si(V a, decltype(V::x) s) { return mk<V>(-s * a.y, s * a.x); }

template <int R, typename V>
struct Dft;  // composite radices below

template <typename V>
struct Dft<2, V> {
    static __device__ inline void run(V *v, decltype(V::x)) {
        V a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    }
};

template <typename V>
struct Dft<4, V> {
    static __device__ inline void run(V *v, decltype(V::x) s) {
        V a0 = cadd(v[0], v[2]), a1 = csub(v[0], v[2]);
        V b0 = cadd(v[1], v[3]), b1 = mul_si(csub(v[1], v[3]), s);
        v[0] = cadd(a0, b0);
        v[2] = csub(a0, b0);
        v[1] = cadd(a1, b1);
        v[3] = csub(a1, b1);
    }
};

template <typename V>
struct Dft<3, V> {
    static __device__ inline void run(V *v, decltype(V::x) s) {
        using T = decltype(V::x);
        const T c1 = (T)-0.5, s1 = (T)0.86602540378443864676;  // cos, sin of 2 pi / 3
        V t1 = cadd(v[1], v[2]), t2 = csub(v[1], v[2]);
        V y0 = cadd(v[0], t1);
        V m1 = mk<V>(v[0].x + c1 * t1.x, v[0].y + c1 * t1.y);
        V m2 = mul_si(t2, s * s1);
        v[0] = y0;
        v[1] = cadd(m1, m2);
        v[2] = csub(m1, m2);
    }
};

template <typename V>
struct Dft<5, V> {
    static __device__ inline void run(V *v, decltype(V::x) s) {
        using T = decltype(V::x);
        const T c1 = (T)0.30901699437494742410, c2 = (T)-0.80901699437494742410;
        const T s1 = (T)0.95105651629515357212, s2 = (T)0.58778525229247312917;
        V t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]);
        V t3 = csub(v[1], v[4]), t4 = csub(v[2], v[3]);
        V y0 = cadd(v[0], cadd(t1, t2));
        V a1 = mk<V>(v[0].x + c1 * t1.x + c2 * t2.x, v[0].y + c1 * t1.y + c2 * t2.y);
        V a2 = mk<V>(v[0].x + c2 * t1.x + c1 * t2.x, v[0].y + c2 * t1.y + c1 * t2.y);
        V b1 = mul_si(mk<V>(s1 * t3.x + s2 * t4.x, s1 * t3.y + s2 * t4.y), s);
        V b2 = mul_si(mk<V>(s2 * t3.x - s1 * t4.x, s2 * t3.y - s1 * t4.y), s);
        v[0] = y0;
        v[1] = cadd(a1, b1);
        v[4] = csub(a1, b1);
        v[2] = cadd(a2, b2);
        v[3] = csub(a2, b2);
    }
};

template <typename V>
struct Dft<8, V> {
    static __device__ inline void run(V *v, decltype(V::x) s) {
        using T = decltype(V::x);
        const T r2 = (T)0.70710678118654752440;
        V e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
        Dft<4, V>::run(e, s);
        Dft<4, V>::run(o, s);
        V w1 = mk<V>(r2, s * r2), w3 = mk<V>(-r2, s * r2);
        o[1] = cmul(o[1], w1);
        o[2] = mul_si(o[2], s);
        o[3] = cmul(o[3], w3);
        for (int k = 0; k < 4; k++) {
            v[k] = cadd(e[k], o[k]);
            v[k + 4] = csub(e[k], o[k]);
        }
    }
};

// e^{s 2 pi i k / N} v for compile-time k
template <int K, int N, typename V>
__device__ inline V turn(V v, decltype(V::x) s) {
    using T = decltype(V::x);
    if constexpr (K % N == 0) return v;
    else if constexpr ((4 * K) % N == 0) {
        constexpr int q = (4 * K / N) % 4;
        if constexpr (q == 1) return mul_si(v, s);
        else if constexpr (q == 2) return mk<V>(-v.x, -v.y);
        else return mul_si(v, -s);
    } else {
        constexpr T c = (T)cos_turn(K, N), w = (T)sin_turn(K, N);
        return cmul(v, mk<V>(c, s * w));
    }
}

// Composite radices: R = R1 R2 in registers, x[j2 + R2 j1] -> X[k1 + R1 k2]
constexpr int first_factor(int r) { return r % 4 == 0 && r != 12 ? 4 : (r % 3 == 0 ? 3 : (r % 5 == 0 ? 5 : 2)); }
template <int R, typename V>
struct Dft {
    static constexpr int R1 = first_factor(R), R2 = R / R1;
    template <int J2, int K1>
    static __device__ inline void twiddle(V *a, decltype(V::x) s) {
        a[K1] = turn<J2 * K1, R>(a[K1], s);
        if constexpr (K1 + 1 < R1) twiddle<J2, K1 + 1>(a, s);
    }
    template <int J2>
    static __device__ inline void first(V *v, V (*y)[R1], decltype(V::x) s) {
#pragma unroll
        for (int j1 = 0; j1 < R1; j1++) y[J2][j1] = v[J2 + R2 * j1];
        Dft<R1, V>::run(y[J2], s);
        twiddle<J2, 0>(y[J2], s);
        if constexpr (J2 + 1 < R2) first<J2 + 1>(v, y, s);
    }
    static __device__ inline void run(V *v, decltype(V::x) s) {
        V y[R2][R1];
        first<0>(v, y, s);
#pragma unroll
        for (int k1 = 0; k1 < R1; k1++) {
            V z[R2];
#pragma unroll
            for (int j2 = 0; j2 < R2; j2++) z[j2] = y[j2][k1];
            Dft<R2, V>::run(z, s);
#pragma unroll
            for (int k2 = 0; k2 < R2; k2++) v[k1 + R1 * k2] = z[k2];
        }
    }
};

// One Stockham stage of radix R over `rows` lines of length n held in LDS;
// twiddles read from the FP64 table and rounded to the working precision.
template <int R, typename V>
__device__ inline void stockham_stage(const V *src, V *dst, int n, int ld, int Ns, int rows,
                                      const double2 *__restrict__ tw, decltype(V::x) s) {
    using T = decltype(V::x);
    const int nb = n / R;
    const int tstep = n / (Ns * R);
    for (int task = threadIdx.x; task < rows * nb; task += kThreads) {
        const int row = task / nb, j = task - row * nb;
        const V *in = src + row * ld;
        V *out = dst + row * ld;
        const int k = j % Ns;
        V v[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            V x = in[j + r * nb];
            if (r > 0 && k > 0) {
                const double2 w = tw[(k * r * tstep) % n];
                x = cmul(x, mk<V>((T)w.x, (T)w.y * s));
            }
            v[r] = x;
        }
        Dft<R, V>::run(v, s);
        const int base = (j / Ns) * Ns * R + k;
#pragma unroll
        for (int r = 0; r < R; r++) out[base + r * Ns] = v[r];
    }
}

// The lines of one pass: [outer][n][C], C contiguous columns; a workgroup takes the pb columns
// from c0 = batch pb of one outer index.
struct Cols {
    size_t C;          // columns
    unsigned pb;       // columns per workgroup
    unsigned nbatch;   // workgroups per outer index
    unsigned nwg;      // all workgroups
    unsigned run;      // consecutive workgroups of one XCD
    unsigned lines;    // > 1: a workgroup takes whole lines of `lines` outer indices (C small), pb = lines C rows
    unsigned nouter;
};

// Workgroups go to the 8 XCDs round robin in dispatch order.  `run` consecutive ones are given to
// one XCD (one L2), so that the 128-byte lines that two workgroups share are read from HBM once,
// while all XCDs stay within 8 run workgroups of each other: ranges an eighth of the field apart
// meet in the same memory channels.  Measured per evaluation (128^3, mmax 5, FP64; 6 passes over all 88
// projections, each over the whole field): one range per XCD 7.00 ms, runs of 96 6.95, 24 6.55-7.0, 8 7.02, round
// robin 7.69 ms; FP32 (shared lines along x) 3.52, 3.45, 3.47, 3.52, 4.40 ms.
constexpr unsigned kRun = 24;
__device__ inline unsigned xcd_order(unsigned run) {
    const unsigned g = blockIdx.x / (8 * run), w = blockIdx.x - g * 8 * run;
    return (g * 8 + (w & 7)) * run + (w >> 3);
}

// Line lengths that are not known at compile time.
template <typename V>
__global__ __launch_bounds__(kThreads) void fft_axis(V *__restrict__ data, Cols g, FftAxisPlan plan, double sgn_d,
                                                    double scale_d) {
    using T = decltype(V::x);
    extern __shared__ __align__(16) unsigned char fft_smem[];
    V *sbuf = reinterpret_cast<V *>(fft_smem);
    const T sgn = (T)sgn_d, scale = (T)scale_d;
    const int n = plan.n, ld = n + 1, PB = (int)g.pb;
    const unsigned id = xcd_order(g.run);
    if (id >= g.nwg) return;
    V *A = sbuf, *B = sbuf + PB * ld;
    const unsigned o = id / g.nbatch;
    const size_t c0 = (size_t)(id % g.nbatch) * g.pb;
    V *base = data + (size_t)o * n * g.C + c0;
    const int pb = (int)(g.C - c0 < g.pb ? g.C - c0 : g.pb);
    for (int idx = threadIdx.x; idx < n * pb; idx += kThreads) {
        const int p = idx % pb, e = idx / pb;
        A[p * ld + e] = base[(size_t)e * g.C + p];
    }
    __syncthreads();
    V *src = A, *dst = B;
    int Ns = 1;
    for (int st = 0; st < plan.nst; st++) {
        const int R = plan.radix[st];
        switch (R) {
            case 8: stockham_stage<8, V>(src, dst, n, ld, Ns, pb, plan.tw, sgn); break;
            case 4: stockham_stage<4, V>(src, dst, n, ld, Ns, pb, plan.tw, sgn); break;
            case 2: stockham_stage<2, V>(src, dst, n, ld, Ns, pb, plan.tw, sgn); break;
            case 3: stockham_stage<3, V>(src, dst, n, ld, Ns, pb, plan.tw, sgn); break;
            default: stockham_stage<5, V>(src, dst, n, ld, Ns, pb, plan.tw, sgn); break;
        }
        Ns *= R;
        __syncthreads();
        V *t = src;
        src = dst;
        dst = t;
    }
    for (int idx = threadIdx.x; idx < n * pb; idx += kThreads) {
        const int p = idx % pb, e = idx / pb;
        V v = src[p * ld + e];
        v.x *= scale;
        v.y *= scale;
        base[(size_t)e * g.C + p] = v;
    }
}

// ---- line lengths known at compile time: constant trip counts and twiddle indices, one LDS
// buffer, the stages staged through registers.  A pass is bound by HBM: 4.8-5.3 TB/s of its one
// read and one write at 96-180 points, where a plain copy reaches 4.8.  The kernel above, with runtime
// radices, takes about twice as long, 3.6 times at most (six passes in an evaluation, FP32: 100^3, mmax 4 1.71
// against 0.73 ms, 180^3, mmax 5 24.7 against 6.9; FP64: 128^3, mmax 5 10.2 against 5.1, 48^3, mmax 1 56 against
// 30 us).  The lengths are all products of 2, 3 and 5 from 16 to 128, where boxes mostly are, and eight of the
// fourteen from there to 256.  135, 162, 216, 225, 243, 250 and all beyond 256 take the kernel above as the sizes
// below 16 do: no workload has them (216^3, mmax 3, FP32: 14.1 of an evaluation's 21.9 ms).
constexpr bool is_radix(int r) {
    return r == 2 || r == 3 || r == 4 || r == 5 || r == 6 || r == 8 || r == 9 || r == 10 || r == 12 || r == 15 || r == 16;
}
// The radix of the next stage for the remaining factor `rem`: two stages of nearly equal radix
// where both are at most rmax, else the largest radix.
constexpr int pick_radix(int rem, int rmax) {
    int best = 0;
    for (int r = 2; r <= rmax; r++)
        if (is_radix(r) && rem % r == 0 && is_radix(rem / r) && rem / r <= rmax && r >= rem / r && !best) best = r;
    if (best && rem > 5) return best;
    if (rem <= rmax && is_radix(rem)) return rem;
    for (int r = rmax; r >= 2; r--)
        if (is_radix(r) && rem % r == 0) return r;
    return 0;
}
// The largest radix: registers against passes over LDS.  FP64: a butterfly of 16 holds 64
// registers (128^3, all 88 projections: 16 and 8 took 7.85 ms where 8, 4 and 4 took 7.69).
template <typename V> constexpr int rmax() { return sizeof(V) == 16 ? 10 : 16; }

template <typename V> constexpr int columns() { return 128 / (int)sizeof(V); }

// Task t of a stage is (row = t % pb, butterfly j = t / pb), so a wave's consecutive lanes are
// consecutive columns: the first stage reads its inputs straight from HBM and the last writes
// its outputs straight back, in runs of 128 bytes.  LDS holds [element][row].
template <int N, int Ns, int REM, int T, bool FIRST, typename V>
__device__ inline void run_stages(V *A, const V *twl, decltype(V::x) s, V *__restrict__ base, size_t es, unsigned pb,
                                  unsigned magic, unsigned C, size_t ls, decltype(V::x) scale) {
    constexpr int R = FIRST ? pick_radix(N, rmax<V>()) : (REM <= rmax<V>() && is_radix(REM) ? REM : pick_radix(REM, rmax<V>()));
    constexpr int nb = N / R, tstep = N / (Ns * R), PB = columns<V>();
    constexpr bool LAST = (REM == R);
    constexpr int NT = (PB * nb + T - 1) / T;
    const unsigned ntask = pb * nb;
    V o[NT][R];
    unsigned off[NT];  // rows past the batch's lines: LDS offset and memory offset of a valid one
#pragma unroll
    for (int q = 0; q < NT; q++) {
        const unsigned task = threadIdx.x + q * T;
        if (q > 0 && task >= ntask) continue;
        const unsigned tk = task < ntask ? task : ntask - 1;
        const unsigned j = (tk * magic) >> 20, row = tk - j * pb, k = j % Ns;
        off[q] = (j / Ns * (Ns * R) + k) * pb + row;
        V v[R];
        if constexpr (FIRST) {
            // every load is issued unconditionally (a load under a branch made the wave wait for
            // it before issuing the next)
            const V *p = base + (ls ? (size_t)(row / C) * ls + row % C : (size_t)row) + (size_t)j * es;
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = p[(size_t)r * nb * es];
        } else {
#pragma unroll
            for (int r = 0; r < R; r++) {
                V x = A[(j + r * nb) * pb + row];
                if (r > 0) {
                    const V w = twl[k * r * tstep];
                    x = cmul(x, mk<V>(w.x, w.y * s));
                }
                v[r] = x;
            }
        }
        Dft<R, V>::run(v, s);
#pragma unroll
        for (int r = 0; r < R; r++) o[q][r] = v[r];
    }
    if constexpr (!FIRST) __syncthreads();  // every read of this stage precedes its in-place writes
#pragma unroll
    for (int q = 0; q < NT; q++) {
        const unsigned task = threadIdx.x + q * T;
        if (task >= ntask) continue;
        if constexpr (LAST) {
            const unsigned j = (task * magic) >> 20, row = task - j * pb, k = j % Ns;
            const unsigned e = j / Ns * (Ns * R) + k;
            V *p = base + (ls ? (size_t)(row / C) * ls + row % C : (size_t)row) + (size_t)e * es;
#pragma unroll
            for (int r = 0; r < R; r++) {
                V v = o[q][r];
                v.x *= scale;
                v.y *= scale;
                p[(size_t)r * Ns * es] = v;
            }
        } else {
#pragma unroll
            for (int r = 0; r < R; r++) A[off[q] + r * Ns * pb] = o[q][r];
        }
    }
    if constexpr (!LAST) {
        __syncthreads();
        run_stages<N, Ns * R, REM / R, T, false, V>(A, twl, s, base, es, pb, magic, C, ls, scale);
    }
}

// threads of a workgroup: the butterflies of its largest stage, at most 256 (one butterfly of the
// first stage each, which at 128 points of FP64 leaves half of them without a load: 128 threads
// took 7.14 against 7.00 ms per evaluation, over all 88 projections)
template <int N, int REM, typename V> constexpr int stage_tasks() {
    constexpr int R = REM <= rmax<V>() && is_radix(REM) && REM != N ? REM : pick_radix(REM, rmax<V>());
    constexpr int t = columns<V>() * (N / R);
    if constexpr (REM == R) return t;
    else {
        constexpr int u = stage_tasks<N, REM / R, V>();
        return t > u ? t : u;
    }
}
template <int N, typename V> constexpr int fft_threads() {
    constexpr int t = (stage_tasks<N, N, V>() + 63) / 64 * 64;
    return t > 256 ? 256 : t;
}

template <int N, typename V>
__global__ __launch_bounds__((fft_threads<N, V>())) void fft_cols(V *__restrict__ data, Cols g, unsigned magic,
                                                                 const double2 *__restrict__ tw, double sgn_d,
                                                                 double scale_d) {
    using T = decltype(V::x);
    constexpr int TH = fft_threads<N, V>();
    __shared__ V A[columns<V>() * N];
    __shared__ V twl[N];
    const unsigned id = xcd_order(g.run);
    if (id >= g.nwg) return;
    V *base;
    unsigned pb = g.pb;
    size_t ls = 0;
    if (g.lines > 1) {
        const unsigned o = id * g.lines, nl = g.nouter - o < g.lines ? g.nouter - o : g.lines;
        base = data + (size_t)o * N * g.C;
        pb = nl * (unsigned)g.C;
        ls = (size_t)N * g.C;
    } else {
        const unsigned o = id / g.nbatch;
        const size_t c0 = (size_t)(id - o * g.nbatch) * g.pb;
        base = data + (size_t)o * N * g.C + c0;
        if (g.C - c0 < pb) pb = (unsigned)(g.C - c0);
    }
    if (pb != g.pb) magic = (1u << 20) / pb + 1;
    for (int i = threadIdx.x; i < N; i += TH) twl[i] = mk<V>((T)tw[i].x, (T)tw[i].y);
    // (the barrier that ends the first stage covers the twiddles)
    run_stages<N, 1, N, TH, true, V>(A, twl, (T)sgn_d, base, g.C, pb, magic, (unsigned)g.C, ls, (T)scale_d);
}

template <typename V>
bool launch_cols(int n, const Cols &g, hipStream_t st, V *proj, const double2 *tw, double sign, double scale) {
    const dim3 grid((g.nwg + 8 * g.run - 1) / (8 * g.run) * 8 * g.run);
    const unsigned magic = (1u << 20) / g.pb + 1;  // exact quotients of task < 4096 by pb <= 16
    switch (n) {
#define FFT_C(NN) \
    case NN: hipLaunchKernelGGL((fft_cols<NN, V>), grid, dim3(fft_threads<NN, V>()), 0, st, proj, g, magic, tw, sign, scale); return true;
        FFT_C(16) FFT_C(18) FFT_C(20) FFT_C(24) FFT_C(25) FFT_C(27) FFT_C(30) FFT_C(32) FFT_C(36) FFT_C(40) FFT_C(45)
        FFT_C(48) FFT_C(50) FFT_C(54) FFT_C(60) FFT_C(64) FFT_C(72) FFT_C(75) FFT_C(80) FFT_C(81) FFT_C(90) FFT_C(96)
        FFT_C(100) FFT_C(108) FFT_C(120) FFT_C(125) FFT_C(128) FFT_C(144) FFT_C(150) FFT_C(160) FFT_C(180) FFT_C(192)
        FFT_C(200) FFT_C(240) FFT_C(256)
#undef FFT_C
        default: return false;
    }
}

// one axis of `outer` blocks [n][C] from `data` on, of a field of np numbers per grid point
template <typename V>
hipError_t launch_axis(mdft_ctx *c, V *data, int ax, size_t C, size_t outer, size_t np, double sign, double scale) {
    const int n = c->fft[ax].n;
    const unsigned PB = columns<V>();
    Cols g;
    g.C = C;
    g.nouter = (unsigned)outer;
    g.lines = 1;
    // equal batches: np = 70 in FP32 is 5 x 14, not 4 x 16 + 6
    g.nbatch = (unsigned)((C + PB - 1) / PB);
    g.pb = (unsigned)((C + g.nbatch - 1) / g.nbatch);
    if (2 * C <= PB) {  // few columns: whole lines of several outer indices
        g.lines = (unsigned)(PB / C);
        g.pb = (unsigned)(g.lines * C);
        g.nbatch = 1;
    }
    g.nwg = g.lines > 1 ? (g.nouter + g.lines - 1) / g.lines : g.nouter * g.nbatch;
    g.run = g.nwg < 8 * kRun ? (g.nwg + 7) / 8 : kRun;
    if (!launch_cols<V>(n, g, c->stream, data, c->fft[ax].tw, sign, scale)) {
        if (g.lines > 1) {
            g.lines = 1;
            g.pb = (unsigned)g.C;
            g.nwg = g.nouter;
        }
        // LDS holds the lines of the columns twice.  From 640 points on that is more than there is for PB of
        // them (160 KB); 4 are taken then where a point has fewer than PB numbers (mmax <= 1, in FP32 2), up to
        // 1279 points, in FP32 2559.
        const size_t line = sizeof(V) * 2 * (size_t)(n + 1);
        if (g.pb * line > c->lds_limit && g.pb > 4 && np < PB) {
            g.pb = 4;
            g.nbatch = (unsigned)((C + 3) / 4);
            g.nwg = g.nouter * g.nbatch;
        }
        const size_t lds = g.pb * line;
        if (lds > c->lds_limit) return hipErrorInvalidConfiguration;
        g.run = g.nwg < 8 * kRun ? (g.nwg + 7) / 8 : kRun;
        hipLaunchKernelGGL((fft_axis<V>), dim3((g.nwg + 8 * g.run - 1) / (8 * g.run) * 8 * g.run), dim3(kThreads), lds,
                           c->stream, data, g, c->fft[ax], sign, scale);
    }
    return hipGetLastError();
}

// The x and y passes of a field beyond the 256 MB memory-side cache run slab by slab (whole xy planes of
// at most that size), the second reading and writing what the first left in the cache: a pass there
// moves 7-8 TB/s, from HBM 5.0.  Six passes, whole field -> slabs of 128, 192, 256, 320 MB: 128^3, mmax 5
// FP64 5.63 -> 5.22, 5.10, 4.98, 5.49 ms; FP32 2.78 -> 2.65, 2.61, 2.55, 2.69; 100^3, mmax 4, FP64 (two
// slabs) 1.60 -> 1.42.  A field of 283 MB gains nothing (96^3, mmax 3, FP64: 0.612 ms either way), one of
// 335 MB 5 %.  The inverse takes z first, so that its last two axes are x and y as well.
template <typename V>
hipError_t launch_fft3d(mdft_ctx *c, V *proj, int sign, int batch) {
    const size_t nx = c->d.nx, ny = c->d.ny, nz = c->d.nz, np = batch > 0 ? batch : c->np;
    const double scale = (sign < 0) ? 1.0 / (double)(nx * ny * nz) : 1.0;
    constexpr size_t kCache = (size_t)256 << 20;
    const size_t plane = nx * ny * np, bytes = plane * nz * sizeof(V);
    size_t nslab = bytes <= kCache + kCache / 6 ? 1 : (bytes + kCache - 1) / kCache;
    if (nslab > nz) nslab = nz;
    const size_t planes = (nz + nslab - 1) / nslab;  // per slab
    hipError_t e = hipSuccess;
    if (sign < 0) e = launch_axis(c, proj, 2, plane, 1, np, sign, scale);
    for (size_t z = 0; e == hipSuccess && z < nz; z += planes) {
        const size_t m = nz - z < planes ? nz - z : planes;
        V *p = proj + z * plane;
        const int first = sign < 0 ? 1 : 0;
        for (int k = 0; e == hipSuccess && k < 2; k++) {
            const int ax = k == 0 ? first : 1 - first;
            e = ax == 0 ? launch_axis(c, p, 0, np, ny * m, np, sign, 1.0)
                        : launch_axis(c, p, 1, nx * np, m, np, sign, 1.0);
        }
    }
    if (e == hipSuccess && sign > 0) e = launch_axis(c, proj, 2, plane, 1, np, sign, scale);
    return e;
}

}  // namespace

// Radix plan: radix-8 stages while more than 8 remain, then 4, 2, 3, 5.
int fft_make_plan(int n, int *radix) {
    int k = 0;
    while (n % 8 == 0 && n > 8 && k < MDFT_FFT_MAX_STAGES) { radix[k++] = 8; n /= 8; }
    while (n % 4 == 0 && k < MDFT_FFT_MAX_STAGES) { radix[k++] = 4; n /= 4; }
    while (n % 2 == 0 && k < MDFT_FFT_MAX_STAGES) { radix[k++] = 2; n /= 2; }
    while (n % 3 == 0 && k < MDFT_FFT_MAX_STAGES) { radix[k++] = 3; n /= 3; }
    while (n % 5 == 0 && k < MDFT_FFT_MAX_STAGES) { radix[k++] = 5; n /= 5; }
    return (n == 1) ? k : -1;
}

hipError_t launch_fft3d_f64(mdft_ctx *c, double2 *proj, int sign, int batch) {
    return launch_fft3d<double2>(c, proj, sign, batch);
}

hipError_t launch_fft3d_f32(mdft_ctx *c, float2 *proj, int sign, int batch) {
    return launch_fft3d<float2>(c, proj, sign, batch);
}
