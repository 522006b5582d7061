// turns.h -- cos and sin of 2 pi k / n as compile-time constants.
#pragma once

// The angle is folded into [0, pi / 4] by its index (exact; [0, pi / 2] for odd n), where the
// Taylor series to x^23 is correct to the last bits.
constexpr double turn_taylor(double x, int first) {  // first 0: cos, 1: sin
    double t = first ? x : 1.0, s = 0.0;
    double terms[12] = {};
    for (int i = 0; i < 12; i++) {
        terms[i] = t;
        t *= -x * x / (double)((2 * i + 1 + first) * (2 * i + 2 + first));
    }
    for (int i = 11; i >= 0; i--) s += terms[i];
    return s;
}
constexpr double kTurnPi = 3.14159265358979323846;
constexpr double cos_turn(int k, int n);
constexpr double sin_turn(int k, int n) {
    k = ((k % n) + n) % n;
    if (2 * k > n) return -sin_turn(n - k, n);
    if (2 * k == n) return 0.0;
    if (4 * k > n) return n % 2 ? turn_taylor(kTurnPi * (n - 2 * k) / n, 1) : sin_turn(n / 2 - k, n);
    if (8 * k > n) return turn_taylor(kTurnPi * (n - 4 * k) / (2.0 * n), 0);
    return turn_taylor(2.0 * kTurnPi * k / n, 1);
}
constexpr double cos_turn(int k, int n) {
    k = ((k % n) + n) % n;
    if (2 * k > n) k = n - k;
    if (4 * k > n) return -(n % 2 ? turn_taylor(kTurnPi * (n - 2 * k) / n, 0) : cos_turn(n / 2 - k, n));
    if (8 * k > n) return turn_taylor(kTurnPi * (n - 4 * k) / (2.0 * n), 1);
    return turn_taylor(2.0 * kTurnPi * k / n, 0);
}
constexpr bool turn_is(double a, double b) { return a - b < 2e-16 && b - a < 2e-16; }
static_assert(turn_is(cos_turn(1, 8), 0.70710678118654752440) && turn_is(sin_turn(1, 8), 0.70710678118654752440), "");
static_assert(turn_is(sin_turn(2, 5), 0.58778525229247312917) && turn_is(cos_turn(2, 5), -0.80901699437494742410), "");
static_assert(turn_is(cos_turn(4, 9), -0.93969262078590838405) && turn_is(sin_turn(5, 9), -0.34202014332566873304), "");
static_assert(turn_is(cos_turn(5, 11), -0.95949297361449738989) && turn_is(sin_turn(3, 11), 0.98982144188093273238), "");

// cos(2 pi k / N) and sin(2 pi k / N), k = 0 .. N - 1
template <typename T, int N> struct Turns {
    T c[N] = {}, s[N] = {};
    constexpr Turns() {
        for (int k = 0; k < N; k++) {
            c[k] = (T)cos_turn(k, N);
            s[k] = (T)sin_turn(k, N);
        }
    }
};
