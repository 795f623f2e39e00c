// The host lists of the resident launches against their definition.
//   resident_lists_host NV R SEED THREADS ALLOCATIONS
// THREADS thread creations and ALLOCATIONS arrays of NV int32 succeed. Prints
// OK and the longest halo, REFUSED (the lists report failure) or WRONG.
#include <dlfcn.h>
#include <pthread.h>

#include <atomic>
#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <random>
#include <set>

#include "resident_lists.h"

static int threads_left = 1 << 20;
static std::atomic<int> arrays_left{1 << 20};
static size_t array_bytes = ~size_t(0);

extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
    using Fn = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    static const Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "pthread_create"));
    return threads_left-- > 0 ? real(t, a, f, arg) : EAGAIN;
}
void *operator new(size_t n) {
    if (n == array_bytes && arrays_left-- <= 0) throw std::bad_alloc();
    if (void *p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

int main(int, char **argv) {
    const int nv = std::atoi(argv[1]), R = std::atoi(argv[2]);
    std::mt19937 rng(static_cast<unsigned>(std::atoi(argv[3])));
    // a band and some far columns; rows of odd slices share the offsets +-1, +-2 (negative width)
    std::vector<std::set<int32_t>> cols(static_cast<size_t>(nv));
    const int ns = (nv + 63) / 64;
    for (int r = 0; r < nv; ++r) {
        cols[r].insert(r);
        const bool shared = (r / 64) & 1;
        const int far = shared ? 0 : static_cast<int>(rng() % 9);
        for (int o : {-2, -1, 1, 2})
            if (r + o >= 0 && r + o < nv && rng() % 8) cols[r].insert(r + o);
        for (int k = 0; k < far; ++k) cols[r].insert(static_cast<int32_t>(rng() % static_cast<unsigned>(nv)));
    }
    std::vector<int32_t> rp{0}, ci, width(static_cast<size_t>(ns));
    std::vector<std::vector<int32_t>> shared(static_cast<size_t>(ns));
    std::vector<int64_t> vptr{0};
    for (const auto &c : cols) {
        ci.insert(ci.end(), c.begin(), c.end());
        rp.push_back(static_cast<int32_t>(ci.size()));
    }
    for (int s = 0; s < ns; ++s) {
        int w = 0;
        for (int r = 64 * s; r < std::min(nv, 64 * s + 64); ++r) w = std::max<int>(w, rp[r + 1] - rp[r] - 1);
        if (s & 1) {
            shared[s] = {-2, -1, 1, 2};
            w = 4;
        }
        width[s] = (s & 1) ? -w : w;
        vptr.push_back(vptr.back() + 64 * w);
    }
    threads_left = std::atoi(argv[4]);
    arrays_left = std::atoi(argv[5]);
    array_bytes = sizeof(int32_t) * static_cast<size_t>(nv);
    fk::ResidentLists l;
    const bool ok = fk::resident_lists(nv, R, rp, ci, width, shared, vptr, l);
    array_bytes = ~size_t(0);
    if (!ok) {
        std::puts("REFUSED");
        return 0;
    }
    int longest = 0;
    const int nb = (nv + R - 1) / R;
    for (int b = 0; b < nb; ++b) {
        const int r0 = b * R, r1 = std::min(nv, r0 + R);
        std::set<int32_t> halo;
        for (int r = r0; r < r1; ++r)
            for (int32_t c : cols[r])
                if (c < r0 || c >= r1) halo.insert(c);
        const std::vector<int32_t> want(halo.begin(), halo.end());
        if (want != std::vector<int32_t>(l.halo.begin() + l.ptr[b], l.halo.begin() + l.ptr[b + 1])) return std::puts("WRONG halo"), 1;
        longest = std::max<int>(longest, static_cast<int>(want.size()));
        for (int r = r0; r < r1; ++r) {
            const int s = r / 64, lane = r % 64, W = std::abs(width[s]), ng = W / 4;
            std::vector<int32_t> row;  // column of every entry: its own row on padding
            if (width[s] < 0)
                for (int o : shared[s]) row.push_back(cols[r].count(r + o) ? r + o : r);
            else
                for (int32_t c : cols[r])
                    if (c != r) row.push_back(c);
            row.resize(static_cast<size_t>(W), r);
            for (int k = 0; k < W; ++k) {
                const int64_t e = vptr[s] + (k < 4 * ng ? 4 * (64 * (k / 4) + lane) + k % 4 : 256 * ng + 64 * (k - 4 * ng) + lane);
                const int i = l.idx[e], c = i < R ? r0 + i : want[i - R];
                if (c != row[k]) return std::puts("WRONG entry"), 1;
            }
        }
    }
    if (l.halo_max != longest) return std::puts("WRONG longest halo"), 1;
    std::printf("OK %d\n", longest);
    return 0;
}
