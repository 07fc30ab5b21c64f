// The column loop of a small front (mf_pivots.h) by four wavefronts on the
// host: one coroutine each, switched before and after every access to what
// they share, in 24 orders of preference (a preferred wavefront runs until it
// waits at a barrier) and in random orders.  In every order all four must do
// the same updates, meet at the same number of barriers and leave with the
// same verdict, for a pivot that fails at each column and for none.
#include <ucontext.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "mf_pivots.h"

namespace {

constexpr int W = 4;
constexpr size_t STACK = 64 * 1024;

struct Wave {
    ucontext_t ctx;
    std::vector<char> stack;
    bool done = false, waiting = false, ok = false;
    int barriers = 0;
    std::vector<int> updated;
};

Wave wave[W];
ucontext_t host;
int now, shared_fail, nn, bad;
bool closed;

void yield() { swapcontext(&wave[now].ctx, &host); }

struct Fail {
    void set(int v) const {
        yield();
        shared_fail = v;
        yield();
    }
    int get() const {
        yield();
        const int v = shared_fail;
        yield();
        return v;
    }
};

void body() {
    const int g = now;
    Wave& w = wave[g];
    w.ok = mf::pivot_columns(
        nn, g, closed, [&](int k) { return k != bad; }, Fail(),
        [&] {
            ++w.barriers;
            w.waiting = true;
            yield();
        },
        [&](int k) { w.updated.push_back(k); });
    w.done = true;
    yield();
}

// false: the wavefronts disagree
template <typename Pick>
bool run(Pick pick) {
    shared_fail = 0;
    for (int g = 0; g < W; ++g) {
        Wave& w = wave[g];
        w.done = w.waiting = w.ok = false;
        w.barriers = 0;
        w.updated.clear();
        w.stack.resize(STACK);
        getcontext(&w.ctx);
        w.ctx.uc_stack.ss_sp = w.stack.data();
        w.ctx.uc_stack.ss_size = STACK;
        w.ctx.uc_link = &host;
        makecontext(&w.ctx, body, 0);
    }
    for (;;) {
        int ready[W], n = 0, waiting = 0, done = 0;
        for (int g = 0; g < W; ++g) {
            if (wave[g].done) ++done;
            else if (wave[g].waiting) ++waiting;
            else ready[n++] = g;
        }
        if (done == W) break;
        if (n == 0) {
            if (waiting != W) return false;  // some left, the others wait for them
            for (Wave& w : wave) w.waiting = false;
            continue;
        }
        now = pick(ready, n);
        swapcontext(&host, &wave[now].ctx);
    }
    for (const Wave& w : wave)
        if (w.barriers != wave[0].barriers || w.updated != wave[0].updated || w.ok != (bad >= nn)) return false;
    return (int)wave[0].updated.size() == std::min(bad, nn);
}

}  // namespace

int main() {
    long runs = 0;
    for (int c = 0; c < 2; ++c)
        for (nn = 1; nn <= 10; ++nn)
            for (bad = 0; bad <= nn; ++bad) {
                closed = c != 0;
                int order[W] = {0, 1, 2, 3};
                do {
                    ++runs;
                    if (!run([&](const int* ready, int n) {
                            for (int g : order)
                                if (std::find(ready, ready + n, g) != ready + n) return g;
                            return ready[0];
                        })) {
                        std::printf("order %d %d %d %d: columns %d, failing %d, closed %d\n", order[0], order[1], order[2],
                                    order[3], nn, bad, c);
                        return 1;
                    }
                } while (std::next_permutation(order, order + W));
                for (int seed = 0; seed < 20; ++seed) {
                    std::mt19937 rng(1000 * nn + 20 * bad + seed);
                    ++runs;
                    if (!run([&](const int* ready, int n) { return ready[rng() % n]; })) {
                        std::printf("seed %d: columns %d, failing %d, closed %d\n", seed, nn, bad, c);
                        return 1;
                    }
                }
            }
    std::printf("%ld runs\n", runs);
    return 0;
}
