// CPU emulation of the t-line transform (fft_core.h: TCross, WaveX, t_order and
// the wavefront stages), thread by thread between its synchronisations, against a
// brute-force DFT in long double: the forward transform's frequency order,
// and the inverse of an array in that order.  Exit 1 on failure.
#include "../../mpc_amd/csrc/fft_core.h"
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

using namespace mpc;

/* a wavefront's Stockham stages over its region of WN elements */
template <class T, int NT, int WN, int E, int DIR, int Ns, int R, int... Rest> struct Wave {
    static void run(std::vector<cx<T>> &V, size_t t0, cx<T> *reg, const cx<T> *tw) {
        constexpr int L = WN / E;
        using X = WaveX<T, WN>;
        for (int lane = 0; lane < L; ++lane) {
            cx<T>(&v)[E] = *reinterpret_cast<cx<T>(*)[E]>(&V[(t0 + lane) * E]);
            fft_stage_t<T, WN, E, R, Ns, DIR, true, 0>(v, lane, reg, 1, TwFromTable<T, WN, R, Ns, DIR, NT / WN>{tw});
            if constexpr (sizeof...(Rest) != 0) X::template put<Ns>(v, lane, reg);
        }
        if constexpr (sizeof...(Rest) != 0) {
            for (int lane = 0; lane < L; ++lane) {
                cx<T>(&v)[E] = *reinterpret_cast<cx<T>(*)[E]>(&V[(t0 + lane) * E]);
                X::template get<Ns>(v, lane, reg);
            }
            Wave<T, NT, WN, E, DIR, Ns * R, Rest...>::run(V, t0, reg, tw);
        }
    }
};
template <class T, int NT, int DIR, class Rad> struct Line;
template <class T, int NT, int DIR, int... Rs> struct Line<T, NT, DIR, Radices<Rs...>> {
    static constexpr int E = 8, WN = t_wave_len(NT), R1 = NT / WN, TPL = NT / E, L = WN / E, RS = WaveX<T, WN>::ELEMS;
    static void run(std::vector<cx<T>> &V, const cx<T> *tw) {
        std::vector<cx<T>> lds(R1 * RS);
        auto at = [&](int tid) -> cx<T>(&)[E] { return *reinterpret_cast<cx<T>(*)[E]>(&V[(size_t)tid * E]); };
        auto waves = [&] {
            for (int w = 0; w < R1; ++w) Wave<T, NT, WN, E, DIR, 1, Rs...>::run(V, (size_t)w * L, lds.data() + w * RS, tw);
        };
        if constexpr (R1 == 1) {
            waves();
        } else if constexpr (DIR < 0) {
            for (int tid = 0; tid < TPL; ++tid) { TCross<T, NT, R1, E> x; x.load(tw, tid); x.fwd(at(tid), tid, lds.data()); }
            for (int tid = 0; tid < TPL; ++tid)
                for (int m = 0; m < E; ++m) at(tid)[m] = lds[tid / 64 * RS + tid % 64 + 64 * m];
            waves();
        } else {
            waves();
            for (int tid = 0; tid < TPL; ++tid)
                for (int m = 0; m < E; ++m) lds[tid / 64 * RS + tid % 64 + 64 * m] = at(tid)[m];
            for (int tid = 0; tid < TPL; ++tid) { TCross<T, NT, R1, E> x; x.load(tw, tid); x.inv(at(tid), tid, lds.data()); }
        }
    }
};

template <class T, int NT, int DIR> double check(unsigned seed) {
    constexpr int E = 8, TPL = NT / E;
    std::vector<cx<T>> tw(NT), V(NT);
    std::vector<long double> c(NT), s(NT), xr(NT), xi(NT);
    for (int k = 0; k < NT; ++k) {
        const long double a = 2.0L * 3.14159265358979323846264338327950288L * k / NT;
        c[k] = cosl(a);
        s[k] = sinl(a);
        tw[k] = mk((T)c[k], (T)-s[k]);
    }
    srand(seed);
    for (int i = 0; i < NT; ++i) { xr[i] = (T)(rand() / (double)RAND_MAX - 0.5); xi[i] = (T)(rand() / (double)RAND_MAX - 0.5); }
    /* element m of thread tid is position tid + TPL m: time tid + TPL m, or
     * frequency t_order of it */
    std::vector<int> seen(NT, 0);
    for (int p = 0; p < NT; ++p) {
        const int i = DIR < 0 ? p : t_order(NT, p);
        V[(size_t)(p % TPL) * E + p / TPL] = mk((T)xr[i], (T)xi[i]);
        seen[t_order(NT, p)]++;
    }
    for (int n : seen) if (n != 1) return 1.0;      /* t_order is a permutation */
    Line<T, NT, DIR, typename TPlan<t_wave_len(NT)>::R>::run(V, tw.data());
    double num = 0, den = 0;
    for (int p = 0; p < NT; ++p) {
        const long k = DIR < 0 ? t_order(NT, p) : p;
        long double sr = 0, si = 0;
        for (int j = 0; j < NT; ++j) {
            const int a = (int)((j * k) % NT);
            const long double cs = c[a], sn = DIR * s[a];
            sr += xr[j] * cs - xi[j] * sn;
            si += xr[j] * sn + xi[j] * cs;
        }
        const cx<T> g = V[(size_t)(p % TPL) * E + p / TPL];
        num += (double)((g.re - sr) * (g.re - sr) + (g.im - si) * (g.im - si));
        den += (double)(sr * sr + si * si);
    }
    return std::sqrt(num / den);
}
template <int NT> int run_n() {
    const double a = check<double, NT, -1>(NT), b = check<double, NT, +1>(NT + 1);
    const double d = check<float, NT, -1>(NT + 2), e = check<float, NT, +1>(NT + 3);
    printf("t line N=%5d f64 fwd %.3e inv %.3e  f32 fwd %.3e inv %.3e\n", NT, a, b, d, e);
    return a > 1e-14 || b > 1e-14 || d > 2e-6 || e > 2e-6;
}
int main() {
    const int bad = run_n<256>() | run_n<512>() | run_n<1024>() | run_n<2048>() | run_n<4096>();
    printf(bad ? "FAIL\n" : "OK\n");
    return bad;
}
