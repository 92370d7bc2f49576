// ldlt!'s unblocked body (csrc/k_factor_dev.hpp) for one workgroup on the
// host: the lanes are fibers, the lanes of a wave meet at every shuffle, and
// between barriers the waves run one after another in an order drawn from a
// seed, each as far as it gets. Waves that meet at different barriers have
// taken different branches: the run stops there.
#include <algorithm>
#include <random>
#include <ucontext.h>
#include <vector>
#include "k_factor_dev.hpp"

namespace {

enum State { READY, EXCHANGE, BALLOT, BARRIER, DONE };
struct Lane {
    HostLane index{};
    ucontext_t context{};
    State state = READY;
    uint64_t value = 0, result = 0;
    int source = 0;
    int site = 0;
};
std::vector<Lane> lanes;
Lane *current = nullptr;
ucontext_t scheduler;
void (*body)() = nullptr;

void lane_main() {
    body();
    current->state = DONE;
    swapcontext(&current->context, &scheduler);
}
void wait_as(State s) {
    Lane *l = current;
    l->state = s;
    swapcontext(&l->context, &scheduler);
}

// one wave up to its next barrier or its end
bool run_wave(size_t first, size_t count) {
    for (;;) {
        for (size_t i = first + count; i-- > first;)         // the first lane, which moves diagonal elements, after the others have read them
            if (lanes[i].state == READY) {
                current = &lanes[i];
                swapcontext(&scheduler, &lanes[i].context);
            }
        const State s = lanes[first].state;
        for (size_t i = first; i < first + count; ++i)
            if (lanes[i].state != s || lanes[i].site != lanes[first].site) return false;   // the lanes of a wave apart
        if (s == BARRIER || s == DONE) return true;
        uint64_t ballot = 0;
        for (size_t i = 0; i < count; ++i) ballot |= (lanes[first + i].value & 1) << i;
        for (size_t i = first; i < first + count; ++i) lanes[i].result = s == BALLOT ? ballot : lanes[first + lanes[i].source].value;
        for (size_t i = first; i < first + count; ++i) lanes[i].state = READY;
    }
}

// barriers passed, or -1 where waves met at different ones
int64_t run_workgroup(int threads, uint64_t seed) {
    constexpr size_t kStack = 128 * 1024;
    std::vector<char> stacks(kStack * threads);
    lanes.assign(threads, Lane());
    for (int t = 0; t < threads; ++t) {
        Lane &l = lanes[t];
        l.index.thread.x = (unsigned)t;
        l.index.block_dim.x = (unsigned)threads;
        getcontext(&l.context);
        l.context.uc_stack.ss_sp = stacks.data() + kStack * t;
        l.context.uc_stack.ss_size = kStack;
        makecontext(&l.context, lane_main, 0);
    }
    std::mt19937_64 rng(seed);
    const int waves = threads / 64;
    std::vector<int> order(waves);
    for (int w = 0; w < waves; ++w) order[w] = w;
    for (int64_t barriers = 0;; ++barriers) {
        std::shuffle(order.begin(), order.end(), rng);
        for (int w : order)
            if (!run_wave(64 * (size_t)w, 64)) return -1;
        for (const Lane &l : lanes)
            if (l.state != lanes[0].state || l.site != lanes[0].site) return -1;
        if (lanes[0].state == DONE) return barriers;
        for (Lane &l : lanes) l.state = READY;
    }
}

template <int N> struct Call {
    static mfk::DV A, dsub;
    static int64_t n, *pivots, *info;
    static uint8_t *blocks;
    static mf::V<N> alpha;
    static std::vector<double> sv, coefs;
    static std::vector<int64_t> si;
    static void run() {
        mfk::ldlt_unblocked_body<N>(A, n, dsub, pivots, blocks, alpha, info, sv.data(), si.data(), coefs.empty() ? nullptr : coefs.data());
    }
};
template <int N> mfk::DV Call<N>::A;
template <int N> mfk::DV Call<N>::dsub;
template <int N> int64_t Call<N>::n;
template <int N> int64_t *Call<N>::pivots;
template <int N> int64_t *Call<N>::info;
template <int N> uint8_t *Call<N>::blocks;
template <int N> mf::V<N> Call<N>::alpha;
template <int N> std::vector<double> Call<N>::sv;
template <int N> std::vector<double> Call<N>::coefs;
template <int N> std::vector<int64_t> Call<N>::si;

template <int N>
int64_t ldlt(int64_t n, double *A, double *dsub, int64_t *pivots, uint8_t *blocks, int64_t *info, int threads, int with_coefs, uint64_t seed) {
    using C = Call<N>;
    C::A = mfk::DV{A, 1, n, n * n};
    C::dsub = mfk::DV{dsub, 1, n, n};
    C::n = n;
    C::pivots = pivots;
    C::blocks = blocks;
    C::info = info;
    C::alpha = mf::div(mf::add(mf::from<N>(1.0), mf::sqrt(mf::from<N>(17.0))), mf::from<N>(8.0));
    C::sv.assign((size_t)threads * N, 0.0);
    C::si.assign(threads, 0);
    C::coefs.assign(with_coefs ? 2 * n * N : 0, 0.0);
    body = C::run;
    return run_workgroup(threads, seed);
}

}  // namespace

HostLane &host_lane() { return current->index; }
int host_lane_id() { return (int)(current->index.thread.x & 63); }
void host_barrier(int line) {
    current->site = line;
    wait_as(BARRIER);
}
uint64_t host_exchange(uint64_t value, int source) {
    Lane *l = current;
    l->value = value;
    l->source = source & 63;
    wait_as(EXCHANGE);
    return l->result;
}
uint64_t host_ballot(bool p) {
    Lane *l = current;
    l->value = p;
    wait_as(BALLOT);
    return l->result;
}

extern "C" int64_t ldlt_waves(int limbs, int64_t n, double *A, double *dsub, int64_t *pivots, uint8_t *blocks, int64_t *info, int threads,
                              int with_coefs, uint64_t seed) {
    switch (limbs) {
        case 1: return ldlt<1>(n, A, dsub, pivots, blocks, info, threads, with_coefs, seed);
        case 2: return ldlt<2>(n, A, dsub, pivots, blocks, info, threads, with_coefs, seed);
        case 3: return ldlt<3>(n, A, dsub, pivots, blocks, info, threads, with_coefs, seed);
        default: return ldlt<4>(n, A, dsub, pivots, blocks, info, threads, with_coefs, seed);
    }
}
