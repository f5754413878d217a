// CPU emulation of the t-line transform with each thread's twiddle powers cached
// (TCross and the TwChain of its wavefront's stages, as persistent workgroups
// keep them), against the form that reads the table (tline_emul.cpp, itself
// checked against a brute-force DFT): the same bits.  Exit 1 on failure.
#define main tline_emul_main
#include "tline_emul.cpp"
#undef main
#include <cstring>
#include <random>

/* a wavefront's stages; ch: the wavefront's threads' powers from this stage on */
template <class T, int NT, int WN, int E, int DIR, int Ns, int R, int... Rest> struct WaveC {
    using CH = TwChain<T, WN, E, Ns, R, Rest...>;
    static void run(std::vector<cx<T>> &V, size_t t0, cx<T> *reg, const std::vector<const CH *> &ch) {
        constexpr int L = WN / E;
        using X = WaveX<T, WN>;
        for (int lane = 0; lane < L; ++lane) {
            cx<T>(&v)[E] = *reinterpret_cast<cx<T>(*)[E]>(&V[(t0 + lane) * E]);
            fft_stage_t<T, WN, E, R, Ns, DIR, true, 0>(v, lane, reg, 1, TwFromPowers<T, R, E / R, DIR>{ch[lane]->p});
            if constexpr (sizeof...(Rest) != 0) X::template put<Ns>(v, lane, reg);
        }
        if constexpr (sizeof...(Rest) != 0) {
            std::vector<const TwChain<T, WN, E, Ns * R, Rest...> *> next;
            for (int lane = 0; lane < L; ++lane) {
                cx<T>(&v)[E] = *reinterpret_cast<cx<T>(*)[E]>(&V[(t0 + lane) * E]);
                X::template get<Ns>(v, lane, reg);
                next.push_back(&ch[lane]->next);
            }
            WaveC<T, NT, WN, E, DIR, Ns * R, Rest...>::run(V, t0, reg, next);
        }
    }
};
template <class T, int NT, int DIR, class Rad> struct LineC;
template <class T, int NT, int DIR, int... Rs> struct LineC<T, NT, DIR, Radices<Rs...>> {
    static constexpr int E = 8, WN = t_wave_len(NT), R1 = NT / WN, TPL = NT / E, L = WN / E, RS = WaveX<T, WN>::ELEMS;
    using CH = TwChain<T, WN, E, 1, Rs...>;
    static void run(std::vector<cx<T>> &V, const cx<T> *tw) {
        std::vector<cx<T>> lds(R1 * RS);
        std::vector<CH> w(TPL);
        std::vector<TCross<T, NT, R1 == 1 ? 2 : R1, E>> x(TPL);
        for (int tid = 0; tid < TPL; ++tid) {
            w[tid].load(tw, tid % L, R1);
            if (R1 > 1) x[tid].load(tw, tid);
        }
        auto at = [&](int tid) -> cx<T>(&)[E] { return *reinterpret_cast<cx<T>(*)[E]>(&V[(size_t)tid * E]); };
        auto waves = [&] {
            for (int v = 0; v < R1; ++v) {
                std::vector<const CH *> ch;
                for (int lane = 0; lane < L; ++lane) ch.push_back(&w[(size_t)v * L + lane]);
                WaveC<T, NT, WN, E, DIR, 1, Rs...>::run(V, (size_t)v * L, lds.data() + v * RS, ch);
            }
        };
        if constexpr (R1 == 1) {
            waves();
        } else if constexpr (DIR < 0) {
            for (int tid = 0; tid < TPL; ++tid) x[tid].fwd(at(tid), tid, lds.data());
            for (int tid = 0; tid < TPL; ++tid)
                for (int m = 0; m < E; ++m) at(tid)[m] = lds[tid / 64 * RS + tid % 64 + 64 * m];
            waves();
        } else {
            waves();
            for (int tid = 0; tid < TPL; ++tid)
                for (int m = 0; m < E; ++m) lds[tid / 64 * RS + tid % 64 + 64 * m] = at(tid)[m];
            for (int tid = 0; tid < TPL; ++tid) x[tid].inv(at(tid), tid, lds.data());
        }
    }
};

template <class T, int NT, int DIR> bool same() {
    using R = typename TPlan<t_wave_len(NT)>::R;
    std::vector<cx<T>> tw(NT), a(NT);
    std::mt19937 g(NT + DIR);
    std::uniform_real_distribution<double> u(-1, 1);
    for (int k = 0; k < NT; ++k) {
        const long double p = -2.0L * 3.14159265358979323846264338327950288L * k / NT;
        tw[k] = mk((T)cosl(p), (T)sinl(p));
        a[k] = mk((T)u(g), (T)u(g));
    }
    std::vector<cx<T>> b = a;
    Line<T, NT, DIR, R>::run(a, tw.data());
    LineC<T, NT, DIR, R>::run(b, tw.data());
    return std::memcmp(a.data(), b.data(), sizeof(cx<T>) * NT) == 0;
}
template <int NT> int run_c() {
    const bool ok[4] = {same<double, NT, -1>(), same<double, NT, +1>(), same<float, NT, -1>(), same<float, NT, +1>()};
    printf("cached N=%5d f64 fwd %d inv %d  f32 fwd %d inv %d\n", NT, ok[0], ok[1], ok[2], ok[3]);
    return !(ok[0] && ok[1] && ok[2] && ok[3]);
}
int main() {
    const int bad = run_c<256>() | run_c<512>() | run_c<1024>() | run_c<2048>() | run_c<4096>();
    printf(bad ? "FAIL\n" : "OK\n");
    return bad;
}
