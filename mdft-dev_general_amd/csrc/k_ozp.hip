// k_ozp.hip -- the q-space step of the excess term for the lowest orders (mmax <= 2, molecular
// symmetry order 2, packed projections): one thread per (q, -q) pair.
//
// The same steps as k_ozm.hip (src/module_energy_cproj_mrso.f90:441-674): rotation to the frame of q,
// c interpolated linearly in |q|, the OZ sums, rotation back, the chops in FP64, the store rule.  At
// these orders a pair has at most 14 + 14 projections: they stay in a thread's registers throughout,
// all indices being compile-time constants, where the tiles of k_ozm.hip (8 pairs per workgroup of 256
// threads) leave most threads idle between barriers.  Pairs are sorted by interpolation interval, so
// that a wave's threads read the same two rows of c.  Bound by the gather of the pairs' records, at
// mmax 2 by the one (FP64) or two (FP32) waves per SIMD that the registers allow.  k_ozm.hip -> here, FP32 /
// FP64: 96^3, mmax 1 115 -> 24 / 162 -> 26 us; 75^3, mmax 2 117 -> 44 / 217 -> 81; 64^3, mmax 0 30 -> 9 / 40 -> 10.
#include <cfloat>
#include <type_traits>

#include "mdft_internal.h"

namespace {

// Threads of a workgroup.  FP64 at mmax 2 holds one wave per SIMD, which single waves fill as they end (64, 128, 256
// threads: 64^3 54, 60, 59 us, 128^3 330, 350, 353); FP32, 186, 179, 169 us at 128^3, shares the lines of c.
template <typename T> constexpr int threads() { return sizeof(T) == 8 ? 64 : 256; }

template <typename T> struct C2;
template <> struct C2<double> { using t = double2; };
template <> struct C2<float> { using t = float2; };

template <int L> struct Idx {
    static constexpr int nmu(int m) { return m / 2 + 1; }
    static constexpr int iabs(int x) { return x < 0 ? -x : x; }
    static constexpr int poff(int m) {
        int o = 0;
        for (int l = 0; l < m; l++) o += (2 * l + 1) * nmu(l);
        return o;
    }
    static constexpr int np = poff(L + 1);
    static constexpr int p(int m, int mup, int mu2) { return poff(m) + (mup + m) * nmu(m) + mu2; }
    static constexpr int kp = ((L + 2) / 2) * 2;  // Fourier coefficients stored per d entry
    static constexpr int roff(int m) { return m * (4 * m * m - 1) / 3; }
    // first coefficient of row (m, khi, mu2) in the relayouted c(k) table
    static constexpr int ia(int m, int khi, int mu2) {
        int i = 0;
        for (int a = 0; a <= L; a++)
            for (int k = -a; k <= a; k++)
                for (int u = 0; u < nmu(a); u++) {
                    if (a == m && k == khi && u == mu2) return i;
                    for (int n = iabs(k); n <= L; n++) i += 2 * (n / 2) + 1;
                }
        return i;
    }
    // its column of (n, nu2 = v) within block khi
    static constexpr int col(int khi, int n, int v) {
        int i = 0;
        for (int a = iabs(khi); a < n; a++) i += 2 * (a / 2) + 1;
        return i + v + n / 2;
    }
};

// a component below FLT_EPSILON becomes 0 and the other single precision (:491-492)
__device__ inline void chop_r(double &re, double &im) {
    if (fabs(re) < (double)FLT_EPSILON) {
        re = 0.0;
        im = (double)(float)im;
    }
    if (fabs(im) < (double)FLT_EPSILON) {
        im = 0.0;
        re = (double)(float)re;
    }
}
__device__ inline void chop_r(float &, float &) {}
// DBL_EPSILON chop of gamma (:618-623)
__device__ inline void chop_g(double &re, double &im) {
    if (fabs(re) < DBL_EPSILON && fabs(im) < DBL_EPSILON) re = im = 0.0;
    if (fabs(re) < DBL_EPSILON) {
        re = 0.0;
        im = (double)(float)im;
    }
    if (fabs(im) < DBL_EPSILON) {
        im = 0.0;
        re = (double)(float)re;
    }
}
__device__ inline void chop_g(float &, float &) {}

template <typename T> struct Frame {  // multiples of the angles of q
    T ct[3], st[3], cp[3], sp[3];
};

// f(A), f(A + 1), ..., f(B - 1) with compile-time arguments
template <int A, int B, typename F> __device__ __forceinline__ void each(F &&f) {
    if constexpr (A < B) {
        f(std::integral_constant<int, A>{});
        each<A + 1, B>(f);
    }
}

// R^m(mup, khi) = exp(-i mup phi) d^m(mup, khi)(theta), d from its Fourier series
template <int L, int M, int MUP, int KHI, typename T>
__device__ __forceinline__ typename C2<T>::t entry_r(const T *__restrict__ ftab, const Frame<T> &f) {
    using I = Idx<L>;
    constexpr int at = (I::roff(M) + (MUP + M) * (2 * M + 1) + KHI + M) * I::kp, a = MUP < 0 ? -MUP : MUP;
    T v = 0;
    each<0, M + 1>([&](auto k) { v += ftab[at + k] * (((MUP - KHI) & 1) ? f.st[k] : f.ct[k]); });
    typename C2<T>::t r;
    r.x = f.cp[a] * v;
    r.y = (MUP < 0 ? f.sp[a] : -f.sp[a]) * v;
    chop_r(r.x, r.y);
    return r;
}

// o += a b in four multiply-adds (as a sum of two products, one of each three becomes an addition)
template <typename T> __device__ __forceinline__ void mac(T &ox, T &oy, T ax, T ay, T bx, T by) {
    ox = fma(ax, bx, ox);
    oy = fma(ax, by, oy);
    ox = fma(-ay, by, ox);
    oy = fma(ay, bx, oy);
}

template <int L, typename T>
__global__ __launch_bounds__(threads<T>()) void ozp(typename C2<T>::t *__restrict__ proj, const TilePair *__restrict__ pairs,
                                               unsigned n, unsigned per, const double2 *__restrict__ ck, int npc,
                                               const T *__restrict__ ftab) {
    using C = typename C2<T>::t;
    using I = Idx<L>;
    using P = Packed<L>;
    constexpr int NP = I::np, NPK = P::np;
    // workgroups go to the 8 XCDs round robin: each takes a contiguous range of |q|
    const unsigned i = ((blockIdx.x & 7) * per + (blockIdx.x >> 3)) * threads<T>() + threadIdx.x;
    if (i >= n) return;
    const TilePair tp = pairs[i];
    if (tp.flag & 4) return;  // padding
    C *rq = proj + (size_t)tp.gq * NPK, *rm = proj + (size_t)tp.gmq * NPK;
    C iq[NPK], im[NPK], x[NP], y[NP];  // x, y: all projections of q and -q
    each<0, NPK>([&](auto e) {
        iq[e] = rq[e];
        im[e] = rm[e];
    });
    each<0, L + 1>([&](auto m) {
        each<-m, m + 1>([&](auto mup) {
            each<0, I::nmu(m)>([&](auto u) {
                C &a = x[I::p(m, mup, u)], &b = y[I::p(m, mup, u)];
                if constexpr (u > 0 || mup > 0) {
                    constexpr int e = P::off(mup, u) + m - P::mlo(mup, u);
                    a = iq[e];
                    b = im[e];
                } else if constexpr (mup < 0) {
                    constexpr int e = P::off(-mup, 0) + m + mup;
                    constexpr T s = (mup & 1) ? (T)-1 : (T)1;
                    a.x = s * im[e].x;
                    a.y = -s * im[e].y;
                    b.x = s * iq[e].x;
                    b.y = -s * iq[e].y;
                } else {
                    const C p = iq[P::pair0 + m / 2], q = im[P::pair0 + m / 2];
                    a.x = (T)0.5 * (m % 2 ? p.y + q.y : p.x + q.x);
                    a.y = (T)0.5 * (m % 2 ? q.x - p.x : p.y - q.y);
                    b.x = a.x;
                    b.y = -a.y;
                }
            });
        });
    });
    Frame<T> f;
    {
        double c = 1.0, s = 0.0, cp = 1.0, sp = 0.0;
        each<0, L + 1>([&](auto k) {
            f.ct[k] = (T)c;
            f.st[k] = (T)s;
            f.cp[k] = (T)cp;
            f.sp[k] = (T)sp;
            const double nc = c * tp.ct - s * tp.st, np = cp * tp.cp - sp * tp.sp;
            s = s * tp.ct + c * tp.st;
            c = nc;
            sp = sp * tp.cp + cp * tp.sp;
            cp = np;
        });
    }
    // to the frame of q: x(m, khi, u) <- sum_mup x(m, mup, u) R(mup, khi);
    // y(m, -khi, u) <- (-1)^m sum_mup y(m, mup, u) R(mup, khi)   (m = 0: R = 1)
    each<1, L + 1>([&](auto m) {
        constexpr int NU = I::nmu(m);
        constexpr T sg = (m & 1) ? (T)-1 : (T)1;
        C a[(2 * m + 1) * NU], b[(2 * m + 1) * NU];
        each<-m, m + 1>([&](auto khi) {
            each<0, NU>([&](auto u) {
                a[(khi + m) * NU + u].x = a[(khi + m) * NU + u].y = 0;
                b[(m - khi) * NU + u].x = b[(m - khi) * NU + u].y = 0;
            });
            each<-m, m + 1>([&](auto mup) {
                const C r = entry_r<L, m, mup, khi, T>(ftab, f);
                each<0, NU>([&](auto u) {
                    const C v = x[I::p(m, mup, u)], w = y[I::p(m, mup, u)];
                    C &oa = a[(khi + m) * NU + u], &ob = b[(m - khi) * NU + u];
                    mac(oa.x, oa.y, v.x, v.y, r.x, r.y);
                    mac(ob.x, ob.y, w.x, w.y, r.x, r.y);
                });
            });
        });
        each<0, (2 * m + 1) * NU>([&](auto k) {
            x[I::poff(m) + k] = a[k];
            y[I::poff(m) + k].x = sg * b[k].x;
            y[I::poff(m) + k].y = sg * b[k].y;
        });
    });
    // OZ: block khi reads and writes the entries (., khi, .) only
    const T al = (T)tp.al, be = (T)(1.0 - tp.al);
    const double2 *c0 = ck + (size_t)(tp.iq - 1) * npc, *c1 = c0 + npc;
    each<-L, L + 1>([&](auto khi) {
        constexpr int lo = khi < 0 ? -khi : khi;
        C g[NP], h[NP];
        each<lo, L + 1>([&](auto m) {
            each<0, I::nmu(m)>([&](auto u) {
                T gx = 0, gy = 0, hx = 0, hy = 0;
                each<lo, L + 1>([&](auto nn) {
                    each<-(nn / 2), nn / 2 + 1>([&](auto v) {
                        constexpr int ia = I::ia(m, khi, u) + I::col(khi, nn, v);
                        const double2 d0 = c0[ia], d1 = c1[ia];
                        const T cx = be * (T)d0.x + al * (T)d1.x, cy = be * (T)d0.y + al * (T)d1.y;
                        constexpr int e = I::p(nn, khi, v < 0 ? -v : v);
                        C p = v < 0 ? x[e] : y[e], q = v < 0 ? y[e] : x[e];
                        if constexpr (v >= 0) {
                            p.y = -p.y;
                            q.y = -q.y;
                        }
                        mac(gx, gy, p.x, p.y, cx, cy);
                        mac(hx, hy, q.x, q.y, cx, cy);
                    });
                });
                chop_g(gx, gy);
                chop_g(hx, hy);
                C &og = g[I::p(m, khi, u)], &oh = h[I::p(m, khi, u)];
                og.x = gx;
                og.y = gy;
                oh.x = hx;
                oh.y = hy;
            });
        });
        each<lo, L + 1>([&](auto m) {
            each<0, I::nmu(m)>([&](auto u) {
                x[I::p(m, khi, u)] = g[I::p(m, khi, u)];
                y[I::p(m, khi, u)] = h[I::p(m, khi, u)];
            });
        });
    });
    // back: x(m, mup, u) <- sum_khi x(m, khi, u) conj R(mup, khi);
    // y(m, mup, u) <- (-1)^m sum_khi y(m, -khi, u) conj R(mup, khi)
    each<1, L + 1>([&](auto m) {
        constexpr int NU = I::nmu(m);
        constexpr T sg = (m & 1) ? (T)-1 : (T)1;
        C a[(2 * m + 1) * NU], b[(2 * m + 1) * NU];
        each<-m, m + 1>([&](auto mup) {
            each<0, NU>([&](auto u) {
                a[(mup + m) * NU + u].x = a[(mup + m) * NU + u].y = 0;
                b[(mup + m) * NU + u].x = b[(mup + m) * NU + u].y = 0;
            });
            each<-m, m + 1>([&](auto khi) {
                const C r = entry_r<L, m, mup, khi, T>(ftab, f);
                each<0, NU>([&](auto u) {
                    const C v = x[I::p(m, khi, u)], w = y[I::p(m, -khi, u)];
                    C &oa = a[(mup + m) * NU + u], &ob = b[(mup + m) * NU + u];
                    mac(oa.x, oa.y, v.x, v.y, r.x, -r.y);
                    mac(ob.x, ob.y, w.x, w.y, r.x, -r.y);
                });
            });
        });
        each<0, (2 * m + 1) * NU>([&](auto k) {
            x[I::poff(m) + k] = a[k];
            y[I::poff(m) + k].x = sg * b[k].x;
            y[I::poff(m) + k].y = sg * b[k].y;
        });
    });
    // store rule (:648-656): q == -q keeps the second store, conjugated on a Nyquist plane
    const bool self = tp.flag & 1;
    if (self) {
        const T sg = (tp.flag & 2) ? (T)-1 : (T)1;
        each<0, NP>([&](auto k) {
            y[k].y *= sg;
            x[k] = y[k];
        });
    }
    // the packed projections of the real part (see pack_out of k_ozm.hip)
    each<0, L + 1>([&](auto m) {
        each<0, m + 1>([&](auto mup) {
            const C a = x[I::p(m, mup, 0)], b = y[I::p(m, mup, 0)], an = x[I::p(m, -mup, 0)], bn = y[I::p(m, -mup, 0)];
            constexpr T s = (mup & 1) ? (T)-1 : (T)1;
            C o, w;
            o.x = (T)0.5 * (a.x + s * bn.x);
            o.y = (T)0.5 * (a.y - s * bn.y);
            w.x = (T)0.5 * (b.x + s * an.x);
            w.y = (T)0.5 * (b.y - s * an.y);
            if constexpr (mup > 0) {
                iq[P::off(mup, 0) + m - mup] = o;
                im[P::off(mup, 0) + m - mup] = w;
            } else if constexpr (m % 2 == 0) {
                iq[P::pair0 + m / 2] = o;
                im[P::pair0 + m / 2] = w;
            } else {  // + i times the projection of odd m
                C &p = iq[P::pair0 + m / 2], &q = im[P::pair0 + m / 2];
                p.x -= o.y;
                p.y += o.x;
                q.x -= w.y;
                q.y += w.x;
            }
        });
    });
    each<1, L / 2 + 1>([&](auto u) {
        each<-L, L + 1>([&](auto mup) {
            each<P::mlo(mup, u), L + 1>([&](auto m) {
                iq[P::off(mup, u) + m - P::mlo(mup, u)] = x[I::p(m, mup, u)];
                im[P::off(mup, u) + m - P::mlo(mup, u)] = y[I::p(m, mup, u)];
            });
        });
    });
    each<0, NPK>([&](auto e) {
        if (!self) rq[e] = iq[e];
        rm[e] = im[e];
    });
}

template <int L, typename T> hipError_t launch_ozp_t(mdft_ctx *c, typename C2<T>::t *proj) {
    const unsigned n = 8u * (unsigned)c->pairs.ntiles;
    if (n == 0) return hipSuccess;
    constexpr unsigned TH = threads<T>();
    const unsigned nb = (n + TH - 1) / TH, per = (nb + 7) / 8;
    hipLaunchKernelGGL((ozp<L, T>), dim3(8 * per), dim3(TH), 0, c->stream, proj, c->pairs.tpair, n, per, c->d_ck,
                       c->npc, static_cast<const T *>(c->d_ozm_ftab));
    return hipGetLastError();
}

template <typename T> hipError_t launch_ozp_any(mdft_ctx *c, typename C2<T>::t *proj) {
    switch (c->L) {
        case 0: return launch_ozp_t<0, T>(c, proj);
        case 1: return launch_ozp_t<1, T>(c, proj);
        case 2: return launch_ozp_t<2, T>(c, proj);
        default: return hipErrorInvalidConfiguration;
    }
}

}  // namespace

hipError_t launch_ozp_f64(mdft_ctx *c, double2 *proj) { return launch_ozp_any<double>(c, proj); }
hipError_t launch_ozp_f32(mdft_ctx *c, float2 *proj) { return launch_ozp_any<float>(c, proj); }
