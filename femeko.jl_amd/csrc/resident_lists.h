// Host lists of the resident launches on the SELL copy.
#pragma once

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace fk {

struct ResidentLists {
    std::vector<uint16_t> idx;       // LDS index of every SELL entry, laid out like the values
    std::vector<int32_t> ptr, halo;  // block b: the rows halo[ptr[b] .. ptr[b + 1]) outside its own
    int32_t halo_max = 0;
};

// The LDS index of every SELL entry and the halo list of every block of R rows,
// from the host's copy of the pattern. A block's halo is the sorted set of the
// columns its rows have outside the block; on renumbered meshes it is 2.2 to
// 2.5 times the block's rows. False where an index exceeds 16 bits or memory
// runs out. Threads that cannot be had leave their part to the caller's.
inline bool resident_lists(int64_t nv, int R, const std::vector<int32_t> &rp, const std::vector<int32_t> &ci,
                           const std::vector<int32_t> &width, const std::vector<std::vector<int32_t>> &shared,
                           const std::vector<int64_t> &vptr, ResidentLists &out) {
    const int64_t ns = static_cast<int64_t>(width.size());
    const int nb = static_cast<int>((nv + R - 1) / R);
    std::vector<std::vector<int32_t>> halo(static_cast<size_t>(nb));
    std::vector<uint16_t> &idx = out.idx;
    idx.resize(static_cast<size_t>(vptr[ns]));
    const int nth = static_cast<int>(std::min<unsigned>(16u, std::max(1u, std::thread::hardware_concurrency())));
    bool fits = true;
    std::mutex mu;
    const auto give_up = [&] {
        const std::lock_guard<std::mutex> lock(mu);
        fits = false;
    };
    const auto blocks = [&](int b0, int b1) {
        std::vector<int32_t> place(static_cast<size_t>(nv), -1);  // halo position of a row of the block at hand
        for (int b = b0; b < b1; ++b) {
            const int64_t r0 = static_cast<int64_t>(b) * R, r1 = std::min(nv, r0 + R);
            std::vector<int32_t> &h = halo[b];
            for (int64_t k = rp[r0]; k < rp[r1]; ++k) {
                const int32_t c = ci[k];
                if ((c < r0 || c >= r1) && place[c] < 0) {
                    place[c] = 0;
                    h.push_back(c);
                }
            }
            std::sort(h.begin(), h.end());
            if (h.size() + R > 0xfffe) return give_up();
            for (size_t e = 0; e < h.size(); ++e) place[h[e]] = static_cast<int32_t>(e);
            auto at = [&](int64_t c) { return static_cast<uint16_t>(c >= r0 && c < r1 ? c - r0 : R + place[c]); };
            for (int64_t s = r0 / 64; s < std::min(ns, (r0 + R) / 64); ++s) {
                const int32_t W = width[s] < 0 ? -width[s] : width[s], ng = W >> 2;
                for (int lane = 0; lane < 64; ++lane) {
                    const int64_t r = s * 64 + lane;
                    const uint16_t own = static_cast<uint16_t>(r - r0);
                    const int32_t *lo = r < nv ? ci.data() + rp[r] : nullptr;
                    const int32_t *hi = r < nv ? ci.data() + rp[r + 1] : nullptr;
                    int32_t k = 0;
                    auto put = [&](uint16_t v) {
                        const int64_t o = k < 4 * ng ? 4 * (64 * static_cast<int64_t>(k >> 2) + lane) + (k & 3)
                                                     : 256 * static_cast<int64_t>(ng) + 64 * (k - 4 * ng) + lane;
                        idx[vptr[s] + o] = v;
                        ++k;
                    };
                    if (width[s] < 0) {
                        for (int32_t off : shared[s]) {
                            const int64_t c = r + off;
                            const int32_t *f = r < nv && c >= 0 && c < nv
                                                   ? std::lower_bound(lo, hi, static_cast<int32_t>(c))
                                                   : hi;
                            put(f != hi && *f == c ? at(c) : own);
                        }
                    } else {
                        for (const int32_t *c = lo; c != hi; ++c)
                            if (*c != r) put(at(*c));
                        while (k < W) put(own);
                    }
                }
            }
            for (int32_t c : h) place[c] = -1;
        }
    };
    const auto part = [&](int q) {
        try {
            blocks(nb * q / nth, nb * (q + 1) / nth);
        } catch (const std::bad_alloc &) {
            give_up();
        }
    };
    std::vector<std::thread> th;
    th.reserve(static_cast<size_t>(nth));
    int q = 1;
    try {
        for (; q < nth; ++q) th.emplace_back(part, q);
    } catch (const std::system_error &) {
    }
    part(0);
    for (; q < nth; ++q) part(q);
    for (auto &t : th) t.join();
    if (!fits) return false;
    out.ptr.assign(static_cast<size_t>(nb) + 1, 0);
    out.halo.clear();
    out.halo_max = 0;
    for (int b = 0; b < nb; ++b) {
        out.ptr[b + 1] = out.ptr[b] + static_cast<int32_t>(halo[b].size());
        out.halo_max = std::max(out.halo_max, static_cast<int32_t>(halo[b].size()));
        out.halo.insert(out.halo.end(), halo[b].begin(), halo[b].end());
    }
    return true;
}

}  // namespace fk
