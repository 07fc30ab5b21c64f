// The workspaces of a solve (mf_room.h) taken from memories of every size, one
// solve and a second, larger one after it: a solve that fits with the permuted
// columns, a staging copy and update vectors for all its columns is never
// refused, room is taken where it fits, and nothing is held beyond the memory.
#include <cstdio>
#include <cstdlib>

#include "mf_room.h"

namespace {

using std::int64_t;

struct Memory {
    int64_t size, used = 0;
    int64_t buf[4] = {0, 0, 0, 0};  // permuted columns, staging copy, update vectors, solutions
    // as ensure(): kept where it is large enough, else given back and taken anew
    bool take(int b, int64_t need) {
        if (buf[b] >= need && buf[b] > 0) return true;
        give(b);
        if (used + need > size) return false;
        buf[b] = need;
        used += need;
        return true;
    }
    void give(int b) {
        used -= buf[b];
        buf[b] = 0;
    }
};

int failures = 0;
void check(bool ok, const char* what, int64_t size, int64_t n, int64_t mv, int64_t nrhs) {
    if (ok) return;
    if (++failures <= 10)
        std::printf("%s: memory %lld, n %lld, update vectors %lld, columns %lld\n", what, (long long)size, (long long)n,
                    (long long)mv, (long long)nrhs);
}

bool solve(Memory& m, int64_t n, int64_t mv, int64_t nrhs, int64_t few, bool stage) {
    return mf::take_room(
        nrhs, few, [&] { return m.take(0, n * nrhs) && (!stage || m.take(1, n * nrhs)); },
        [&](int64_t c) { return m.take(2, mv * c) && m.take(3, 2 * n * c); },
        [&] { return m.take(2, mv * (nrhs < 5 ? nrhs : 5)); }, [&] { m.give(2), m.give(3); });
}

}  // namespace

int main() {
    const int64_t n = 10;
    for (int64_t mv : {1, 7, 25})
        for (int64_t few : {1, 5})
            for (bool stage : {false, true})
                for (int64_t first : {0, 1, 6, 40})
                    for (int64_t nrhs : {1, 4, 5, 6, 16, 17, 100})
                        for (int64_t size = 0; size < 2 * (4 * n + mv) * 112; size += 7) {
                            Memory m{size};
                            if (first) (void)solve(m, n, mv, first, few, stage);
                            const bool ok = solve(m, n, mv, nrhs, few, stage);
                            const int64_t columns = nrhs * n * (stage ? 2 : 1);
                            // buffers of the first solve that the second one keeps
                            const int64_t keep = first > nrhs ? (first - nrhs) * n * (stage ? 2 : 1) : 0;
                            if (columns + keep + mv * nrhs <= size) check(ok, "refused", size, n, mv, nrhs);
                            if (!ok) continue;
                            check(m.used <= size, "over the memory", size, n, mv, nrhs);
                            check(m.buf[0] >= n * nrhs && (!stage || m.buf[1] >= n * nrhs), "columns", size, n, mv, nrhs);
                            check(m.buf[2] >= mv * (nrhs < 5 ? nrhs : 5), "update vectors", size, n, mv, nrhs);
                            if (nrhs <= few) continue;
                            const int64_t all = mf::whole_blocks(nrhs), one = mf::ROOM_BLOCK;
                            if (columns + keep + (mv + 2 * n) * all <= size)
                                check(m.buf[2] >= mv * all && m.buf[3] >= 2 * n * all, "no room for all", size, n, mv, nrhs);
                            else if (columns + keep + (mv + 2 * n) * one <= size)
                                check(m.buf[2] >= mv * one && m.buf[3] >= 2 * n * one, "no room for a block", size, n, mv, nrhs);
                        }
    std::printf("%d failures\n", failures);
    return failures != 0;
}
