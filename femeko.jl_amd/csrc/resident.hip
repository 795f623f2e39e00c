// Jacobi-PCG that stays on the chip: one cooperative launch runs a whole
// solve on the stencil copy of the matrix, with x, r, p and D^-1 (and, as far
// as they fit, the matrix values) in the registers of at most one block per
// CU.
//
// The three-kernel iteration of solve.hip moves 152 bytes per row in FP64
// (76 in FP32) and starts three kernels, each of which loads a state, sums
// the previous kernel's block partials and reduces its own: about 4.2 us per
// kernel however small the mesh. Here an iteration is one exchange between
// the resident blocks:
//   q = A p from LDS and the values, w = D^-1 q; w of the own rows out
//   all-reduce p.q, r.z, q.z, q.w and r.r (which also orders the stores of w)
//   alpha = r.z / p.q;  r'.z' = r.z - 2 alpha q.z + alpha^2 q.w;  beta = r'.z' / r.z
//   x += alpha p, z -= alpha w, p = z + beta p  for the own rows (registers)
//   and, from the neighbours' w, for every other row of the block's windows
// r.z is summed from z itself in every iteration; only beta takes the next
// r.z from the identity above, whose error is that of the sums (the terms are
// of the size of r.z). Copies of a row's z and p in several blocks go through
// the same operations on the same numbers and stay equal bit for bit.
// r = D z is not stored: the diagonal is kept beside D^-1.
//
// A block owns R = BLOCK * RPT consecutive rows. The rows its stencil reaches,
// [i0 + o, i0 + o + R) for every offset +-o, merge into a few windows, whose p
// lies in LDS; each window element outside the own rows belongs to one thread,
// which keeps its z in a register. 2 R + 4 m of them are exchanged per
// iteration for the 15-point patterns of an m^3 grid.
//
// Larger meshes go by bricks: with P the offset of the next plane, a block owns
// the rows z P + t of a few planes z and a run of t. Its halo, a plane above
// and below and a reach of a + 1 rows at both ends of every run, is far smaller
// than the windows (n = 160: 7.3k rows beside 16.8k own ones, where windows
// take 33k and do not fit), and a row's backward values are the forward ones
// the block has just read for the plane below, from L2. p lies in LDS alone, and
// only rows within reach of the brick's faces send their w.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <utility>
#include <vector>

#include "device.h"
#include "internal.h"
#include "resident.h"
#include "resident_lists.h"

namespace fk {

constexpr int kResK = 7;         // positive offsets of a resident stencil at most
constexpr int kResWindows = 3;   // separate windows at most
constexpr int kResLdsMax = 155 * 1024;

template <typename T>
struct ResidentArgs {
    const T *val;                 // K x ld value columns a(i, i + off[k])
    const T *dinv;
    const T *r0;                  // initial residual
    T *x;                         // solution out
    T *w;                         // exchange (AgentRows)
    u64 *slots;                   // cleared before the launch
    CgState *state;
    int32_t ld, n, K, nb, stride;
    int32_t off[kResK];
    int32_t lf[kResK], lb[kResK]; // LDS index of local row 0 shifted by +-off[k]
    int32_t lown;                 // LDS index of local row 0
    int32_t wbeg[kResWindows + 1];// LDS index of each window's first element; the number of elements
    int32_t wrow[kResWindows];    // row - i0 of an element - its LDS index, by window
    // SELL copy (any pattern): LDS index of every entry, laid out like the
    // values, and each block's list of rows outside its own (its halo)
    const int64_t *sptr;
    const int32_t *swidth;
    const uint16_t *sidx;
    const int32_t *halo_ptr, *halo;
    int32_t nslices, spare;       // LDS index of the spare element
    // bricks: rows z P + t, 0 <= t < P; a block owns len rows of several planes
    int32_t P, len, reach, S;     // reach of the stencil in t; S = len + 2 reach, a plane in LDS
    int32_t groups;               // blocks side by side in a plane
    double bb_ref, rtol;
    int64_t max_iter;
    // residual replacement (FP32 recursion, FP64 solution u)
    double *u;                    // FP64 solution, accumulates x / s
    const double *b;              // right-hand side, null: 0
    double *r64;                  // FP64 residual
    const double *val64, *diag64;
    T *p;                         // the direction of the own rows over a replacement
    RuState *ru;
    int32_t us;                   // distance of a row's values in u and r64 (right-hand sides side by side)
    double s, target2, thresh64, delta2;
    int32_t G;                    // iterations between two checks of the drop
    uint32_t first;               // tag of the first exchange; the waits of tag 0 give up
};

// A copy of v that the compiler takes for a new value: addresses computed from
// it inside the iteration loop are not hoisted out of it, where the 14 LDS
// and 8 value offsets of each row would occupy registers for the whole solve.
__device__ __forceinline__ int32_t fresh(int32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}

// LDS index of the e-th window element (the windows in LDS order, the own rows
// left out; elements past the last share one spare slot) and its row (spare: none)
template <typename Args>
__device__ __forceinline__ int32_t window_lds(Args &A, int32_t R, int32_t e) {
    return min(e < A.lown ? e : e + R, A.wbeg[kResWindows]);
}
template <typename Args>
__device__ __forceinline__ int32_t window_row(Args &A, int32_t i0, int32_t li) {
    // FP64 selects values: the compiler else selects the address and loads it,
    // a trip to memory before every element's w, one after another at four rows
    // per thread
    const auto at = [&](int k) {
        return sizeof(*A.val) == 8 ? __builtin_amdgcn_readfirstlane(A.wrow[k]) : A.wrow[k];
    };
    int32_t d = at(0);
#pragma unroll
    for (int k = 1; k < kResWindows; ++k) d = li >= A.wbeg[k] ? at(k) : d;
    return li < A.wbeg[kResWindows] ? i0 + li + d : -1;
}

// a row that no buffer holds: loads of it read zero, stores are dropped
constexpr int32_t kNoRow = 0x10000000;

// rows per thread whose x waits in LDS, past the windows: all of the FP64
// shapes with many rows, and half of the FP32 bricks that would spill
template <typename T>
constexpr int x_in_lds(int rpt, bool brick) {
    return sizeof(T) == 8 ? (rpt < 4 ? 0 : rpt > 16 ? 9 : rpt > 14 ? 12 : rpt) : brick && rpt > 22 ? rpt * 3 / 5 : 0;
}

// 1 / v to the last bit or so; v = 0: 0
__device__ __forceinline__ float reciprocal(float v) {
    const float y = __builtin_amdgcn_rcpf(v);
    return v != 0.f ? fmaf(y, fmaf(-v, y, 1.f), y) : 0.f;
}
__device__ __forceinline__ double reciprocal(double v) {
    double y = __builtin_amdgcn_rcp(v);
    y = fma(y, fma(-v, y, 1.0), y);
    return v != 0.0 ? fma(y, fma(-v, y, 1.0), y) : 0.0;
}

constexpr int64_t kClosing = int64_t(1) << 62;  // added to the iterations in the last round; past any limit
constexpr int kResRestarts = 32;  // direction restarts before the FP32 recursion gives up

// RPT rows per thread, the values of the first NK of them in registers (the
// others are streamed from L2 / MALL, a row ahead of their use); U window
// elements per thread at most.
//
// NE > 0: the SELL copy instead of the stencil, rows of at most NE entries.
// The own rows lie first in LDS, the rows of the block's halo list after them,
// and every entry keeps its value and the LDS index of its column.
//
// NE < 0: a brick of the stencil copy, runs of up to -NE x BLOCK rows in each of
// its planes, NK rows' values in flight. Slots past a run's end hold no row:
// their d, z and w are 0.
//
// REFINE (T = float): the reliable updates of solve.hip inside the launch. At
// the end of every G iterations in which ||r||^2 has fallen by delta2 since
// the last replacement, and when the recursion has reached its target, x / s
// is folded into the FP64 solution u, the FP64 residual b - A u of the free
// rows replaces the recursion's (times s), and p is kept; a recursion that has
// drifted below the true residual, or broken down, restarts from p = z. The
// solve ends on the FP64 residual.
template <typename T, int BLOCK, int RPT, int NK, int U, bool REFINE, int NE, typename Args>
__device__ __forceinline__ void resident_solve(Args &A, const int me, const int32_t i0) {
    extern __shared__ char lds_raw[];
    T *win = reinterpret_cast<T *>(lds_raw);
    __shared__ double sh[kReduceShared];
    [[maybe_unused]] __shared__ double before;  // thread 0: ||r||^2 before the step on the way out
    constexpr int K = kResK, R = BLOCK * RPT;
    constexpr bool GEN = NE > 0, BRICK = NE < 0;
    constexpr int TP = BRICK ? -NE : 1, BZ = RPT / TP;  // runs of BLOCK rows in a plane of a brick, planes
    static_assert(!BRICK || (NK > 0 && RPT % NK == 0 && RPT % TP == 0), "whole planes and turns of the ring");
    constexpr int E = GEN ? NE : 2 * K;  // entries per row: K forward, then K backward ones
    static_assert(!GEN || NK == RPT, "SELL values are not streamed");
    constexpr int XL = x_in_lds<T>(RPT, BRICK);
    T *xs = win + (GEN || BRICK ? A.spare : A.wbeg[kResWindows]) + 1;
    constexpr bool AHEAD = RPT > 1 && (sizeof(T) == 4 || (!GEN && RPT <= 3));
    const int32_t tid = threadIdx.x;
    const AgentRows<T> rows(A.w, A.stride);
    const ValueColumns<T> vals(A.val, A.K, A.ld);
    const int32_t n = A.n, lown = GEN ? 0 : A.lown;
    const int32_t bt = BRICK ? (i0 % A.P) : 0, blen = BRICK ? min(A.len, A.P - bt) : 0;
    const int32_t hbase = BRICK ? i0 - A.P - A.reach : 0;  // row of LDS element 0
    // row of thread t's j-th own element, n or more if there is none, and its LDS index
    const auto own_row = [&](int j, int32_t t) {
        if constexpr (BRICK) {
            const int32_t in = (j % TP) * BLOCK + t, first = i0 + (j / TP) * A.P;
            return in < min(blen, n - first) ? first + in : kNoRow;
        } else {
            return i0 + j * BLOCK + t;
        }
    };
    const auto own_lds = [&](int j, int32_t t) {
        return BRICK ? lown + (j / TP) * A.S + (j % TP) * BLOCK + t : lown + j * BLOCK + t;
    };
    const int32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int32_t h0 = GEN ? A.halo_ptr[i0 / R] : 0, nh = GEN ? A.halo_ptr[i0 / R + 1] - h0 : 0;
    uint32_t tag = A.first;
    if (tid == 0) sh[kReduceShared - 1] = 0.0;

    // z = D^-1 r of the own rows goes out
    double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
    for (int j = 0; j < RPT; ++j) {
        const int32_t row = own_row(j, tid);
        if (row >= n) continue;
        const T dj = A.dinv[row];
        T r = T(0);
        if (dj != T(0)) r = REFINE ? static_cast<T>(A.s * A.r64[static_cast<int64_t>(row) * A.us]) : A.r0[row];
        rows.store(tag, row, dj * r);
    }
    bool alive = all_reduce5<BLOCK>(s, A.slots, me, A.nb, tag, sh);

    double rr = 0.0, thresh = 0.0, bb = A.bb_ref;
    int64_t it = 0;
    int code = alive ? -1 : FK_ERR_HIP;  // -1: running
    [[maybe_unused]] double rr64 = 0.0, rr_last = 1.0;
    [[maybe_unused]] int32_t nrep = 0, restarts = 0, until_check = A.G;
    bool restart = true;  // p = z
    while (code < 0) {
        // ---- a run of iterations from z (exchanged) and p: state into registers
        const int32_t tl = fresh(tid);
        T d[RPT], g[BRICK ? 1 : RPT], x[XL < RPT ? RPT - XL : 1], z[RPT], p[BRICK ? 1 : RPT], w[RPT];
        T zw[U];
        [[maybe_unused]] T v[NK > 0 ? NK : 1][E];
        [[maybe_unused]] uint32_t pk[GEN ? RPT : 1][GEN ? NE / 2 : 1];  // LDS indices of two entries
        // rows of this thread's halo elements; bricks: LDS index and, from bit
        // 16, plane slot of each, the sign bit where there is no row
        [[maybe_unused]] int32_t hrow[GEN || BRICK ? U : 1];
        const auto xj = [&](int j, int32_t t) -> T & { return j < XL ? xs[j * BLOCK + t] : x[j < XL ? 0 : j - XL]; };
        // LDS index and row of the u-th window element (spare: none)
        const auto element = [&](int u, int32_t t, int32_t &row) {
            if constexpr (GEN) {
                row = hrow[u];
                return row >= 0 ? R + t + u * BLOCK : A.spare;
            } else if constexpr (BRICK) {
                const int32_t h = fresh(hrow[u]), li = h & 0xffff;
                row = h < 0 ? kNoRow : hbase + li + (h >> 16) * (A.P - A.S);
                return li;
            } else {
                const int32_t li = window_lds(A, R, t + u * BLOCK);
                row = window_row(A, i0, li);
                return li;
            }
        };
        // the value pairs of a row of the stencil
        const auto load_row = [&](int32_t row, T(&o)[E]) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                o[k] = o[K + k] = T(0);
                if (BRICK || k < A.K) {
                    o[k] = vals.load(k, row);
                    o[K + k] = vals.load(k, row - A.off[k]);
                }
            }
        };
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            const int32_t row = own_row(j, tl), at = min(row, n - 1);
            const T dj = A.dinv[at], pj = restart || BRICK ? T(0) : A.p[at];
            z[j] = rows.load(tag, row);  // 0 past the last row
            d[j] = row < n ? dj : T(0);
            if constexpr (!BRICK) p[j] = restart || row >= n ? z[j] : pj;
            xj(j, tl) = T(0);
            // a brick's p stays in LDS; its elements past a run belong to the halo
            if (restart && (!BRICK || (j % TP) * BLOCK + tl < blen))
                win[own_lds(j, tl)] = BRICK ? z[j] : p[BRICK ? 0 : j];
            if (BRICK && j % 8 == 7) __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (!BRICK) {
#pragma unroll
            for (int j = 0; j < RPT; ++j) g[j] = d[j] != T(0) ? T(1) / d[j] : T(0);
        }
        if constexpr (GEN) {
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                const int32_t sl = i0 / 64 + j * (BLOCK / 64) + wave, own = j * BLOCK + tl;
                const bool in = sl < A.nslices;
                const int64_t base = in ? A.sptr[sl] : 0;
                const int32_t W = in ? abs(A.swidth[sl]) : 0, ng = W >> 2, lane = tl & 63;
#pragma unroll
                for (int k = 0; k < NE; ++k) {
                    T a = T(0);
                    uint32_t ix = static_cast<uint32_t>(own);
                    if (k < W) {
                        const int64_t at = base + (k < 4 * ng ? 4 * (64 * (k >> 2) + lane) + (k & 3)
                                                              : 256 * ng + 64 * (k - 4 * ng) + lane);
                        a = A.val[at];
                        ix = A.sidx[at];
                    }
                    v[j][k] = a;
                    pk[j][k / 2] = (k & 1) ? pk[j][k / 2] | ix << 16 : ix;
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int32_t e = tl + u * BLOCK;
                hrow[u] = e < nh ? A.halo[h0 + e] : -1;
            }
        } else if constexpr (BRICK) {
            // the planes below and above in full, then both ends of the own planes
            const int32_t w2 = 2 * A.reach, many = 2 * A.S + BZ * w2;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int32_t e = tl + u * BLOCK, f = e - 2 * A.S, q = f < 0 ? 0 : f / w2, r = f - q * w2;
                const int32_t slot = f >= 0 ? 1 + q : e < A.S ? 0 : BZ + 1;
                const int32_t in = f >= 0 ? (r < A.reach ? r : blen + r) : e < A.S ? e : e - A.S;
                const int32_t row = hbase + slot * A.P + in;
                const bool have = e < many && row >= 0 && row < n;
                hrow[u] = (e < many ? slot * A.S + in : A.spare) | (have ? slot << 16 : INT32_MIN);
            }
        } else {
#pragma unroll
            for (int j = 0; j < NK; ++j) load_row(i0 + j * BLOCK + tl, v[j]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int32_t row;
            const int32_t li = element(u, tl, row);
            zw[u] = rows.load(tag, row);
            if (restart) win[li] = zw[u];
        }
        __syncthreads();
        // a brick's values: NK rows in flight, also over the end of an iteration
        if constexpr (BRICK) {
#pragma unroll
            for (int j = 0; j < NK; ++j) load_row(own_row(j, tl), v[j]);
        }
        [[maybe_unused]] bool moved = false;  // an iteration done in this run
        // FP64, converged: 1 the round of q = A z, 2 that of the residual after the step
        [[maybe_unused]] int closing = 0;
        [[maybe_unused]] bool undo = false;
        constexpr T third = T(1.0 / 3.0);
        [[maybe_unused]] int act = 0;         // why it ended: 1 replace r, 2 drop x and restart
        while (true) {
            ++tag;
            // q = A p in difference form; w = D^-1 q
#pragma unroll
            for (int k = 0; k < 5; ++k) s[k] = 0.0;
            if constexpr (BRICK) {
#pragma unroll
                for (int j = 0; j < RPT; ++j) {
                    const int32_t t = fresh(tid), in = (j % TP) * BLOCK + t, row = own_row(j, t);
                    // the seven offsets are 1, a, a + 1, P, P + 1, P + a, P + a + 1:
                    // adjacent neighbours come with one LDS instruction
                    const T *c = win + own_lds(j, t);
                    const int32_t a = A.lf[1] - lown, sa = A.S + a;
                    const T *fa = c + a, *ba = c - a, *fs = c + A.S, *bs = c - A.S, *fsa = c + sa, *bsa = c - sa;
                    const T nb[E] = {c[1],  fa[0], fa[1],  fs[0], fs[1],  fsa[0], fsa[1],
                                     c[-1], ba[0], ba[-1], bs[0], bs[-1], bsa[0], bsa[-1]};
                    const T pj = c[0];
                    T a0 = T(0), a1 = T(0);
#pragma unroll
                    for (int k = 0; k < K; ++k) {
                        a0 += v[j % NK][k] * (nb[k] - pj);
                        a1 += v[j % NK][K + k] * (nb[K + k] - pj);
                    }
                    const T q = d[j] != T(0) ? a0 + a1 : T(0);
                    w[j] = d[j] * q;
                    // only the rows that other blocks reach go out
                    const bool inner = j >= TP && j < RPT - TP && in >= A.reach && in < blen - A.reach;
                    rows.store(tag, inner ? kNoRow : row, w[j]);
                    load_row(own_row((j + NK) % RPT, t), v[j % NK]);
                    const double zd = static_cast<double>(z[j]), qd = static_cast<double>(q);
                    const double rd = static_cast<double>(reciprocal(d[j]) * z[j]);
                    // past a run pj is any LDS word
                    s[0] += static_cast<double>(d[j] != T(0) ? pj : T(0)) * qd;
                    s[1] += rd * zd;
                    s[2] += qd * zd;
                    s[3] += qd * static_cast<double>(w[j]);
                    s[4] += rd * rd;
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
            [[maybe_unused]] T sv[E];  // values of the streamed row at hand
            if constexpr (NK < RPT) load_row(i0 + NK * BLOCK + fresh(tid), sv);
            // the neighbours of a row are loaded together, and where registers
            // allow a row ahead: one LDS latency per row, not one per neighbour
            T nb[E];
            const auto neighbours = [&](int j, T(&o)[E]) {
                if constexpr (GEN) {
#pragma unroll
                    for (int k = 0; k < NE; ++k)
                        o[k] = win[(k & 1) ? pk[j][k / 2] >> 16 : pk[j][k / 2] & 0xffffu];
                } else {
                    const int32_t l = j * BLOCK + fresh(tid);
#pragma unroll
                    for (int k = 0; k < K; ++k) {
                        o[k] = win[A.lf[k] + l];
                        o[K + k] = win[A.lb[k] + l];
                    }
                }
            };
            if constexpr (AHEAD) neighbours(0, nb);
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                const int32_t row = i0 + j * BLOCK + fresh(tid);
                T next[E], nv[E];
                if (AHEAD && j + 1 < RPT) neighbours(j + 1, next);
                if (!AHEAD) neighbours(j, nb);
                if (NK < RPT && j >= NK && j + 1 < RPT) load_row(row + BLOCK, nv);
                __builtin_amdgcn_sched_barrier(0);
                T a0 = T(0), a1 = T(0);
                const int jk = j < NK ? j : 0;
#pragma unroll
                for (int k = 0; k < E / 2; ++k) {
                    a0 += (j < NK ? v[jk][k] : sv[k]) * (nb[k] - p[j]);
                    a1 += (j < NK ? v[jk][E / 2 + k] : sv[E / 2 + k]) * (nb[E / 2 + k] - p[j]);
                }
                if (AHEAD && j + 1 < RPT) {
#pragma unroll
                    for (int k = 0; k < E; ++k) nb[k] = next[k];
                }
                if (NK < RPT && j >= NK && j + 1 < RPT) {
#pragma unroll
                    for (int k = 0; k < E; ++k) sv[k] = nv[k];
                }
                const T q = d[j] != T(0) ? a0 + a1 : T(0);
                w[j] = d[j] * q;
                rows.store(tag, row, w[j]);  // 0 past the last row
                const double zd = static_cast<double>(z[j]), qd = static_cast<double>(q);
                const double rd = static_cast<double>(g[j] * z[j]);
                s[0] += static_cast<double>(p[j]) * qd;
                s[1] += rd * zd;
                s[2] += qd * zd;
                s[3] += qd * static_cast<double>(w[j]);
                s[4] += rd * rd;
                __builtin_amdgcn_sched_barrier(0);
            }
            }
            alive = all_reduce5<BLOCK>(s, A.slots, me, A.nb, tag, sh);
            T ww[U];
            const int32_t ft = fresh(tid);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                int32_t row;
                (void)element(u, ft, row);
                ww[u] = rows.load(tag, row);
            }
            const double pq = s[0], rz = s[1];
            T alpha = static_cast<T>(rz / pq);
            const double al = static_cast<double>(alpha), inv_rz = 1.0 / rz;
            T beta = static_cast<T>(fmax(rz - al * (2.0 * s[2] - al * s[3]), 0.0) * inv_rz);
            rr = s[4];
            if constexpr (REFINE) {
                act = !alive                                                   ? 3
                      : moved && rr < A.target2                                ? 1
                      : !isfinite(rr)                                          ? 2
                      : it >= A.max_iter                                       ? 1
                      : until_check == 0 && moved && rr < A.delta2 * rr_last   ? 1
                      : !(pq > 0.0) || !isfinite(pq)                           ? 2
                                                                               : 0;
                act = __builtin_amdgcn_readfirstlane(act);
                if (until_check == 0) until_check = A.G;
                if (act) break;
                --until_check;
                moved = true;
            } else {
                if (it == 0) {
                    if (!(bb >= 0.0)) bb = rr;
                    thresh = A.rtol * A.rtol * bb;
                }
                code = !alive                                  ? FK_ERR_HIP
                       : rr < thresh || (it == 0 && rr == 0.0) ? FK_OK
                       : !isfinite(rr)                         ? FK_ERR_NONFINITE
                       : it >= A.max_iter                      ? FK_ERR_NOT_CONVERGED
                       : !(pq > 0.0) || !isfinite(pq)          ? FK_ERR_SINGULAR  // not positive definite on the space
                                                               : -1;
                code = __builtin_amdgcn_readfirstlane(code);
                if (code >= 0) {
                    // a converged recursion that has moved x goes two rounds more. One
                    // loop body for all rounds (fresh): copies of it for the last two
                    // cost every FP64 shape 7 to 40 registers
                    const int phase = __builtin_amdgcn_readfirstlane(fresh(closing));
                    if (!alive) break;
                    if (phase == 2) {  // r after the step
                        it -= kClosing;
                        undo = !(rr < thresh);
                        if (undo && tid == 0) rr = before;
                        code = FK_OK;
                        break;
                    }
                    if (phase == 1) {  // p = z, w = D^-1 A z: the step; p stays, to take it back
#pragma unroll
                        for (int j = 0; j < RPT; ++j) {
                            if constexpr (BRICK) {
                                if ((j % TP) * BLOCK + ft < blen) xj(j, ft) += third * win[own_lds(j, ft)];
                            } else {
                                xj(j, ft) += third * p[j];
                            }
                            z[j] -= third * w[j];
                        }
                        if (tid == 0) before = rr;
                        it += kClosing;  // the next round ends here whatever r is
                        closing = 2;
                        continue;
                    }
                    if (code != FK_OK || it == 0 || !(pq > 0.0) || !isfinite(pq) || !isfinite(s[3])) break;
                    closing = 1;
                    alpha = beta = T(0);
                    --it;
                }
            }
            ++it;
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                if constexpr (BRICK) {
                    if ((j % TP) * BLOCK + ft < blen) {
                        T &pj = win[own_lds(j, ft)];
                        const T old = pj;
                        xj(j, ft) += alpha * old;
                        z[j] -= alpha * w[j];
                        pj = z[j] + beta * old;
                    }
                    if (j % TP == TP - 1) __builtin_amdgcn_sched_barrier(0);
                } else {
                    xj(j, ft) += alpha * p[j];
                    z[j] -= alpha * w[j];
                    p[j] = z[j] + beta * p[j];
                    win[lown + j * BLOCK + ft] = p[j];
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                int32_t row;
                const int32_t li = element(u, ft, row);
                zw[u] -= alpha * ww[u];
                win[li] = zw[u] + beta * win[li];
            }
            __syncthreads();
        }
        if constexpr (!REFINE) {
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                const int32_t row = own_row(j, tid);
                // One Jacobi step of 1/3 was done on the way out. The largest eigenvalues
                // of D^-1 A are those of slivers, 2 to 4 (4: flat, four nodes; the
                // scaled matrix of an element with parallel gradients has rank one
                // and trace 4). Rounding brings their modes back late in the
                // recursion; the residual norm hardly sees them, H inside the
                // sliver does. The step takes two thirds or more off them and
                // lengthens no other mode of D^-1/2 r. Largest error of H at rtol
                // 1e-10 over its rms, 8 jittered meshes of 63^3 cells (jitter 0.2
                // to 0.26): 2.4e-9 to 1.6e-7 with the step, 1.9e-9 to 3.1e-7 after
                // the three kernels. ||r|| itself mostly falls by 0.7 but may rise
                // (1.25 times on a graded Delaunay mesh), so a round of its own
                // measures it after the step, which is taken back where it does
                // not stay below the tolerance; the residual reported is that of
                // the x returned. Weighing the sums of one round instead (r.q and
                // q.q) cost two selects a row in all rounds, 1% of a solve.
                if (row < n) {
                    const T xr = xj(j, tid);
                    T pj;
                    if constexpr (BRICK)
                        pj = win[own_lds(j, tid)];
                    else
                        pj = p[j];
                    A.x[row] = undo ? xr - third * pj : xr;
                }
            }
            break;
        } else {
            // ---- replacement: nothing but x and p leaves the registers
            if (act == 3) {
                code = FK_ERR_HIP;
                break;
            }
            restart = act == 2;
            const int32_t tc = fresh(tid);
            const AgentRows<double> sol(A.u, n * A.us);
            const auto at = [&](int32_t row) { return static_cast<int64_t>(row) * A.us; };
            if (act == 1) {
                const double inv_s = 1.0 / A.s;
#pragma unroll
                for (int j = 0; j < RPT; ++j) {
                    const int32_t row = own_row(j, tc);
                    if (row < n) {
                        sol.store(0, row * A.us, A.u[at(row)] + inv_s * static_cast<double>(xj(j, tc)));
                        if constexpr (!BRICK) A.p[row] = p[j];
                    }
                    if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                }
                ++tag;
                alive = all_reduce5<BLOCK>(s, A.slots, me, A.nb, tag, sh);
                // the other blocks' u through this CU's caches: one wave's
                // acquire serves the block (a fence in every wave takes 16
                // times as long)
                if (tid < 64) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                __syncthreads();
            } else {
                if (++restarts > kResRestarts || it >= A.max_iter) {
                    code = it >= A.max_iter ? FK_ERR_NOT_CONVERGED : isfinite(rr) ? FK_ERR_SINGULAR : FK_ERR_NONFINITE;
                    break;
                }
                ++it;
            }
            ++tag;
            s[0] = 0.0;
            if (!GEN && act == 1) {
                // all loads of two rows in flight together, without a branch: rows
                // and neighbours that do not exist read zero
                constexpr int Q = RPT > 1 ? 2 : 1;
                const ValueColumns<double> val64(A.val64, A.K, A.ld), u64s(A.u, 1, n * A.us);
#pragma unroll 1
                for (int j0 = 0; j0 < RPT; j0 += Q) {
                    int32_t row[Q];
                    double a[Q][2 * K], y[Q][2 * K], yc[Q], dg[Q], bv[Q];
                    T dj[Q];
#pragma unroll
                    for (int q = 0; q < Q; ++q) {
                        row[q] = j0 + q < RPT ? own_row(j0 + q, tc) : kNoRow;
                        const int32_t in = min(row[q], n - 1);
                        row[q] = row[q] < n ? row[q] : kNoRow;
                        const int32_t c = row[q] < n ? row[q] * A.us : kNoRow;
#pragma unroll
                        for (int k = 0; k < K; ++k) {
                            a[q][k] = a[q][K + k] = y[q][k] = y[q][K + k] = 0.0;
                            if (BRICK || k < A.K) {
                                a[q][k] = val64.load(k, row[q]);
                                a[q][K + k] = val64.load(k, row[q] - A.off[k]);
                                y[q][k] = u64s.load(0, c + A.off[k] * A.us);
                                y[q][K + k] = u64s.load(0, c - A.off[k] * A.us);
                            }
                        }
                        yc[q] = u64s.load(0, c);
                        dg[q] = A.diag64[in];
                        dj[q] = A.dinv[in];
                        bv[q] = A.b ? A.b[in] : 0.0;
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int q = 0; q < Q; ++q) {
                        double y0 = 0.0, y1 = 0.0;
#pragma unroll
                        for (int k = 0; k < K; ++k) {
                            y0 += a[q][k] * y[q][k];
                            y1 += a[q][K + k] * y[q][K + k];
                        }
                        const double sum = (y0 + y1) + dg[q] * yc[q];
                        const double v = dj[q] != T(0) && row[q] < n ? bv[q] - sum : 0.0;
                        if (row[q] < n) A.r64[at(row[q])] = v;
                        s[0] += v * v;
                        rows.store(tag, row[q], dj[q] * static_cast<T>(A.s * v));
                    }
                }
            } else {
#pragma unroll 1
                for (int j = 0; j < RPT; ++j) {
                    const int32_t row = own_row(j, tc);
                    if (row >= n) continue;
                    const T dj = A.dinv[row];
                    double v = dj != T(0) ? A.r64[at(row)] : 0.0;
                    if constexpr (GEN) {
                        if (act == 1) {
                            double y0 = 0.0;
                            const int32_t sl = i0 / 64 + j * (BLOCK / 64) + wave, lane = tc & 63;
                            const int64_t base = A.sptr[sl];
                            const int32_t W = abs(A.swidth[sl]), ng = W >> 2;
#pragma unroll 4
                            for (int k = 0; k < W; ++k) {
                                const int64_t e = base + (k < 4 * ng ? 4 * (64 * (k >> 2) + lane) + (k & 3)
                                                                     : 256 * ng + 64 * (k - 4 * ng) + lane);
                                const int32_t ix = A.sidx[e];
                                y0 += A.val64[e] * A.u[at(ix < R ? i0 + ix : A.halo[h0 + ix - R])];
                            }
                            const double y = y0 + A.diag64[row] * A.u[at(row)];
                            v = dj != T(0) ? (A.b ? A.b[row] - y : -y) : 0.0;
                            A.r64[at(row)] = v;
                            s[0] += v * v;
                        }
                    }
                    rows.store(tag, row, dj * static_cast<T>(A.s * v));
                }
            }
            alive = alive && all_reduce5<BLOCK>(s, A.slots, me, A.nb, tag, sh);
            if (!alive) {
                code = FK_ERR_HIP;
                break;
            }
            if (act == 1) {
                rr64 = s[0];
                ++nrep;
                rr_last = rr64 * A.s * A.s;
                restart = rr_last > 4.0 * rr;  // the recursion drifted below the true residual
                if (restart && !(rr64 < A.thresh64)) ++restarts;
                code = rr64 < A.thresh64                             ? FK_OK
                       : !isfinite(rr64)                             ? FK_ERR_NONFINITE
                       : it >= A.max_iter || restarts > kResRestarts ? FK_ERR_NOT_CONVERGED
                                                                     : -1;
                code = __builtin_amdgcn_readfirstlane(code);
                restart = __builtin_amdgcn_readfirstlane(restart);
            }
        }
    }
    // Block 0 may have seen the last round whole where another block gave up on
    // it. A refined solve has stored u by then; x of FP64 differs by the step.
    if (!REFINE && code == FK_ERR_HIP && tid == 0)
        __hip_atomic_store(&A.state->timed_out, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (me == 0 && tid == 0) {
        if constexpr (REFINE) {
            A.ru->nrep = nrep;
            A.ru->restarts = restarts;
            A.ru->rr64 = rr64;
            A.ru->status = code;
        }
        A.state->iters = it;
        A.state->rr = rr;
        A.state->bb = bb;
        A.state->thresh = thresh;
        A.state->status = code;
        A.state->done_at[0] = A.state->done_at[1] = 1;
    }
}

template <typename T, int BLOCK, int RPT, int NK, int U, bool REFINE, int NE>
__global__ __launch_bounds__(BLOCK) void k_resident_pcg(const ResidentArgs<T> A) {
    const int32_t lb = logical_block(A.nb);
    if constexpr (NE < 0) {
        // a block past the last plane owns nothing
        const int32_t z0 = lb / A.groups * (RPT / -NE), t0 = lb % A.groups * A.len;
        const int32_t last = (A.n - 1) / A.P + 1;
        resident_solve<T, BLOCK, RPT, NK, U, REFINE, NE>(A, static_cast<int>(blockIdx.x), min(z0, last) * A.P + t0);
    } else {
        resident_solve<T, BLOCK, RPT, NK, U, REFINE, NE>(A, static_cast<int>(blockIdx.x), lb * (BLOCK * RPT));
    }
}

// Several systems in one launch: block b is block first[b].y of system
// first[b].x. The arguments are read as constants, as kernel arguments are.
template <typename T, int BLOCK, int RPT, int NK, int U>
__global__ __launch_bounds__(BLOCK) void k_resident_batch(const ResidentArgs<T> *__restrict__ all,
                                                          const int2 *__restrict__ first) {
    using Const = const __attribute__((address_space(4))) ResidentArgs<T>;
    const int2 b = first[blockIdx.x];
    const int sys = __builtin_amdgcn_readfirstlane(b.x), me = __builtin_amdgcn_readfirstlane(b.y);
    Const &A = *((Const *)(all + sys));
    resident_solve<T, BLOCK, RPT, NK, U, true, 0>(A, me, me * (BLOCK * RPT));
}

// slots, the rows n..stride of the two exchange arrays and the time-out flag
template <typename T>
__global__ void k_resident_clear(u64 *__restrict__ slots, int words, T *__restrict__ w, int32_t n, int32_t stride,
                                 CgState *__restrict__ state) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x, step = gridDim.x * blockDim.x;
    if (t == 0) state->timed_out = 0;
    for (int i = t; i < words; i += step) slots[i] = 0;
    for (int i = n + t; i < stride; i += step) w[i] = w[stride + i] = T(0);
}

__global__ void k_resident_zero(u64 *__restrict__ a, int64_t na, float *__restrict__ b, int64_t nb) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int64_t step = static_cast<int64_t>(gridDim.x) * blockDim.x;
    for (int64_t i = t; i < na; i += step) a[i] = 0;
    for (int64_t i = t; i < nb; i += step) b[i] = 0.f;
}

// ---------------------------------------------------------------------------
// host side

// The windows of a block of R rows, in LDS one after another. False when they
// are too many or too long.
template <typename T>
static bool place_windows(const int32_t *off, int K, int R, ResidentArgs<T> &A, int32_t *elements) {
    std::vector<std::pair<int64_t, int64_t>> iv{{0, R}};
    for (int k = 0; k < K; ++k) {
        const int64_t o = off[k];
        iv.push_back({o, o + R});
        iv.push_back({-o, R - o});
    }
    std::sort(iv.begin(), iv.end());
    std::vector<std::pair<int64_t, int64_t>> u;  // disjoint, ascending
    for (const auto &v : iv) {
        if (!u.empty() && v.first <= u.back().second)
            u.back().second = std::max(u.back().second, v.second);
        else
            u.push_back(v);
    }
    if (u.size() > static_cast<size_t>(kResWindows)) return false;
    int64_t total = 0;
    for (int k = 0; k < kResWindows; ++k) {
        const bool have = static_cast<size_t>(k) < u.size();
        A.wbeg[k] = static_cast<int32_t>(have ? total : INT32_MAX);
        A.wrow[k] = static_cast<int32_t>(have ? u[k].first - total : 0);
        if (have) total += u[k].second - u[k].first;
        if (total > kResLdsMax) return false;
    }
    A.wbeg[kResWindows] = *elements = static_cast<int32_t>(total);
    auto place = [&](int64_t o) {
        int k = 0;
        while (o >= u[k].second) ++k;
        return static_cast<int32_t>(A.wbeg[k] + o - u[k].first);
    };
    A.lown = place(0);
    for (int k = 0; k < kResK; ++k) {
        A.off[k] = k < K ? off[k] : 0;
        A.lf[k] = place(A.off[k]);
        A.lb[k] = place(-static_cast<int64_t>(A.off[k]));
    }
    return true;
}

// The bricks of BZ planes whose runs fill TP x BLOCK threads, at most `most` of
// them, for the offsets 1, a, a + 1, P, P + 1, P + a, P + a + 1 of a grid of
// boxes cut along their diagonals. Nothing else is asked of the numbering: a
// row is z P + t by definition, and t may run past a plane's end into the next.
template <typename T>
static bool place_bricks(const int32_t *off, int K, int64_t n, int most, int BZ, int run, ResidentArgs<T> &A, int *nb,
                         int32_t *elements, int32_t *halo) {
    if (K != 7) return false;
    const int64_t a = off[1], P = off[3], reach = a + 1;
    if (off[0] != 1 || off[2] != a + 1 || off[4] != P + 1 || off[5] != P + a || off[6] != P + a + 1) return false;
    const int64_t planes = (n + P - 1) / P, layers = (planes + BZ - 1) / BZ;
    if (layers > most) return false;
    const int64_t groups = most / layers, len = (P + groups - 1) / groups;
    const int64_t S = len + 2 * reach, total = (BZ + 2) * S + run - len;
    if (len > run || 2 * reach >= P || total > 0xffff) return false;
    A.P = static_cast<int32_t>(P);
    A.len = static_cast<int32_t>(len);
    A.reach = static_cast<int32_t>(reach);
    A.S = static_cast<int32_t>(S);
    A.groups = static_cast<int32_t>((P + len - 1) / len);
    A.lown = static_cast<int32_t>(S + reach);
    for (int k = 0; k < kResK; ++k) {
        const int64_t o = k < 3 ? off[k] : off[k] - P + S;
        A.off[k] = off[k];
        A.lf[k] = static_cast<int32_t>(A.lown + o);
        A.lb[k] = static_cast<int32_t>(A.lown - o);
    }
    A.spare = *elements = static_cast<int32_t>(total);
    *halo = static_cast<int32_t>(2 * S + 2 * reach * BZ);
    *nb = static_cast<int>(layers * A.groups);
    // neighbouring bricks on one XCD: n = 160 FP32 32.9 -> 31.7 us an iteration, n = 100 FP64 14.6 -> 13.7
    if (*nb > kNumXcd) *nb = std::min((*nb + kNumXcd - 1) / kNumXcd * kNumXcd, most);
    return true;
}

// Scratch that the three kernels do without: false where there is no memory for it.
template <typename F>
static bool have_memory(F reserve) {
    try {
        reserve();
        return true;
    } catch (const Error &e) {
        if (e.code != FK_ERR_OOM) throw;
        (void)hipGetLastError();
        return false;
    }
}

// halo elements per thread of a brick at most: its two outer planes, and the
// ends of the inner ones up to a reach of 170 (FP64: 128)
template <typename T>
constexpr int brick_halo(int BZ, int TP) {
    return 2 * TP + (sizeof(T) == 4 ? (2 * BZ + 6) / 3 : (BZ + 3) / 2);
}

template <typename T, int BLOCK, int RPT, int NK, bool REFINE = false, int NE = 0>
static bool launch_resident(fk_mesh *m, ResidentArgs<T> &A) {
    constexpr int R = BLOCK * RPT;
    constexpr int U = NE > 0   ? (RPT <= 2 ? 4 * RPT : 3 * RPT)
                      : NE < 0 ? brick_halo<T>(RPT / (NE < 0 ? -NE : 1), -NE)
                               : 2 * RPT + 2;
    const int most = std::min(m->ctx->num_cus, kMaxResidentBlocks);
    int nb = static_cast<int>((m->nv + R - 1) / R);
    if (nb > most) return false;
    int32_t elements = 0;
    if constexpr (NE < 0) {
        int32_t halo = 0;
        if (!place_bricks<T>(m->st_off, m->st_K, m->nv, most, RPT / -NE, BLOCK * -NE, A, &nb, &elements, &halo) ||
            halo > U * BLOCK)
            return false;
    }
    // streamed values: one band of rows per XCD
    if (NE == 0 && NK < RPT && nb > kNumXcd) nb = std::min((nb + kNumXcd - 1) / kNumXcd * kNumXcd, most);
    if constexpr (NE > 0) {
        if (m->res_R != R || m->res_halo_max > U * BLOCK) return false;
        elements = R + m->res_halo_max;
        A.spare = elements;
        A.sptr = m->sell_ptr.get();
        A.swidth = m->sell_width.get();
        A.sidx = m->res_sidx.get();
        A.halo_ptr = m->res_halo_ptr.get();
        A.halo = m->res_halo.get();
        A.nslices = static_cast<int32_t>(m->nslices);
    } else if constexpr (NE == 0) {
        if (!place_windows<T>(m->st_off, m->st_K, R, A, &elements) || elements - R > U * BLOCK) return false;
    }
    const size_t lds = (static_cast<size_t>(elements) + 1 + x_in_lds<T>(RPT, NE < 0) * BLOCK) * sizeof(T);
    if (lds > static_cast<size_t>(kResLdsMax)) return false;
    A.nb = nb;
    A.first = 0u - m->ctx->resident_rounds;
    // rows past the last, as far as the last block's windows reach, read zero
    const int64_t reach = NE < 0 ? m->nv : static_cast<int64_t>(nb) * R + (NE > 0 ? 0 : m->st_off[m->st_K - 1] + R);
    const int64_t stride = (reach + 63) / 64 * 64;
    hipStream_t st = m->ctx->stream;
    if (!have_memory([&] {
            m->res_slots.ensure(reduce_words(kMaxResidentBlocks));
            m->res_w.ensure(static_cast<size_t>(2 * stride));
        }))
        return false;
    A.stride = static_cast<int32_t>(stride);
    A.slots = m->res_slots.get();
    A.w = reinterpret_cast<T *>(m->res_w.get());
    auto kern = k_resident_pcg<T, BLOCK, RPT, NK, U, REFINE, NE>;
    FK_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                               static_cast<int>(lds)));
    k_resident_clear<T><<<64, 256, 0, st>>>(A.slots, reduce_words(nb), A.w, A.n, A.stride, A.state);
    FK_HIP(hipGetLastError());
    void *args[] = {&A};
    const hipError_t e = hipLaunchCooperativeKernel(reinterpret_cast<const void *>(kern), dim3(nb), dim3(BLOCK),
                                                    args, static_cast<unsigned>(lds), st);
    if (e == hipErrorCooperativeLaunchTooLarge) {  // not all blocks fit at once on this device
        (void)hipGetLastError();
        return false;
    }
    FK_HIP(e);
    m->launch_layout = NE < 0 ? FK_SOLVE_BRICKS : NE > 0 ? FK_SOLVE_SELL : FK_SOLVE_WINDOWS;
    m->launch_rows = R;
    m->launch_blocks = nb;
    return true;
}

static std::mutex &resident_mutex(int device) {
    static std::mutex all[64];
    return all[device & 63];
}

static int64_t rows_per_block(const fk_mesh *m) {
    const int most = std::min(m->ctx->num_cus, kMaxResidentBlocks);
    return (m->nv + most - 1) / most;
}

// Bricks of BZ planes and runs of up to TP x 512 rows in a plane, the values
// streamed one row ahead: the first shape of the list, by slots per thread,
// whose threads, halo registers and LDS cover the mesh with one brick per CU.
// The shapes are those that leave few slots empty on some mesh: an m^3 grid
// wastes 1 to 20% of them. Measured per iteration (us; in
// brackets the windows or, for FP64 n > 100 and FP32 n > 126, the three kernels),
// Kuhn meshes of n cells per side:
//   FP64  n = 80  8.9 (10.9)   n = 90 11.0 (14.1)   n = 95 11.7 (18.5)   n = 100 13.9 (22.2)
//         n = 105 15.9 (41.5)  n = 118 19.7 (52.7)  n = 125 25.9 (60.0)  n = 130 33.2 (67.5)
//   FP32  n = 80  7.8 (8.7)    n = 95 9.0 (11.5)    n = 100 10.6 (13.5)  n = 118 14.5 (20.5)
//         n = 126 16.1 (28.8)  n = 140 22.2 (45.6)  n = 150 25.3 (53.8)  n = 160 29.7 (61.8)
// More rows in flight (2 or 3 per thread) were no faster at any size: n = 160
// 40.0 us with 3, where they spill, n = 115 14.9 with 2 or 3. What bounds the
// larger ones is the value stream from the MALL: of 29 us at n = 160, 12.3 go
// away when the values (7 columns, 117 MB) are not loaded and 3.0 without the
// exchange; 3.2 are the residual replacements, one in 63 iterations.
//
// Up to four rows per thread the windows, which keep the values in registers,
// are faster: FP64 n = 76 6.8 us against 7.8, n = 70 6.0 against 7.9.
constexpr int64_t kBrickRows = 2048;

template <typename T, int BZ, int TP>
static bool brick(fk_mesh *m, ResidentArgs<T> &A) {
    return launch_resident<T, 512, BZ * TP, 1, sizeof(T) == 4, -TP>(m, A);
}
static bool launch_bricks(fk_mesh *m, ResidentArgs<double> &A) {
    return brick<double, 5, 1>(m, A) || brick<double, 6, 1>(m, A) || brick<double, 7, 1>(m, A) ||
           brick<double, 8, 1>(m, A) || brick<double, 9, 1>(m, A) || brick<double, 5, 2>(m, A) ||
           brick<double, 11, 1>(m, A) || brick<double, 6, 2>(m, A) || brick<double, 7, 2>(m, A) ||
           brick<double, 8, 2>(m, A) || brick<double, 9, 2>(m, A);
}
static bool launch_bricks(fk_mesh *m, ResidentArgs<float> &A) {
    return brick<float, 5, 1>(m, A) || brick<float, 6, 1>(m, A) || brick<float, 7, 1>(m, A) ||
           brick<float, 9, 1>(m, A) || brick<float, 5, 2>(m, A) || brick<float, 6, 2>(m, A) ||
           brick<float, 7, 2>(m, A) || brick<float, 8, 2>(m, A) || brick<float, 9, 2>(m, A) ||
           brick<float, 7, 3>(m, A) || brick<float, 8, 3>(m, A) || brick<float, 9, 3>(m, A) ||
           brick<float, 10, 3>(m, A) || brick<float, 11, 3>(m, A) || brick<float, 12, 3>(m, A);
}

// Rows per block by the number of rows: the smallest shape of the list with
// which at most one block per CU covers them. Few rows per thread leave room
// for all their matrix values in registers (NK = RPT) and shorten every step
// between two exchanges. Measured per iteration (us; three-kernel iteration in
// brackets), Kuhn meshes of n cells per side:
//   n = 20  512 x 1   3.1 (14.7)     n = 40  512 x 1   3.6 (15.9)
//   n = 63  512 x 2   4.5 (21.5)     n = 70  512 x 3   6.0 (23.7)
//   n = 79  512 x 4   7.3 (26.9)     n = 84  512 x 5   8.8 (29.4)
//   n = 90  512 x 6  13.4 (31.5)     n = 95  512 x 7  16.1 (34)
//   n = 99  512 x 8  18.5 (36.8)
// The last four shapes serve stencils that are cut into no bricks (measured on
// boxes cut along their other diagonal).
// One shape up costs (when the shape taken was at 4.8, 7.6 and 11.3): n = 63 on 512 x 3 5.8, n = 79 on 512 x 5 10.9, n = 85 on
// 512 x 6 13.6. More rows than 256 blocks of 4096 keep the three-kernel
// iteration: the windows of more rows per block exceed the LDS.
static bool launch_by_rows(fk_mesh *m, ResidentArgs<double> &A) {
    const int64_t per = rows_per_block(m);
    if (per > kBrickRows && launch_bricks(m, A)) return true;
    if (per <= 512) return launch_resident<double, 512, 1, 1>(m, A);
    if (per <= 1024) return launch_resident<double, 512, 2, 2>(m, A);
    if (per <= 1536) return launch_resident<double, 512, 3, 3>(m, A);
    if (per <= 2048) return launch_resident<double, 512, 4, 4>(m, A);
    if (per <= 2560) return launch_resident<double, 512, 5, 2>(m, A);
    if (per <= 3072) return launch_resident<double, 512, 6, 1>(m, A);
    if (per <= 3584) return launch_resident<double, 512, 7, 0>(m, A);
    if (per <= 4096) return launch_resident<double, 512, 8, 0>(m, A);
    return false;
}

// The same for the FP32 recursion with residual replacement, half the
// registers and LDS per row. Measured as above, replacements included:
//   n = 20  512 x 1   3.8 (14.5)     n = 48  512 x 1   4.9 (15.7)
//   n = 63  512 x 2   5.0 (19.0)     n = 75  512 x 4   6.4 (20.7)
//   n = 85 1024 x 3   9.4 (22.8)     n = 98  512 x 8  12.9 (25.2)
//   n = 110 512 x 12 19.9 (31)       n = 125 512 x 16 27.5 (35.6)
// The last four shapes serve stencils that are cut into no bricks. Below 400k
// rows an iteration takes longer than in FP64 (the replacements); who asks for
// FP32 there gets it.
static bool launch_by_rows(fk_mesh *m, ResidentArgs<float> &A) {
    const int64_t per = rows_per_block(m);
    if (per > kBrickRows && launch_bricks(m, A)) return true;
    if (per <= 512) return launch_resident<float, 512, 1, 1, true>(m, A);
    if (per <= 1024) return launch_resident<float, 512, 2, 2, true>(m, A);
    if (per <= 1536) return launch_resident<float, 512, 3, 3, true>(m, A);
    if (per <= 2048) return launch_resident<float, 512, 4, 4, true>(m, A);
    if (per <= 3072) return launch_resident<float, 1024, 3, 3, true>(m, A);
    if (per <= 4096) return launch_resident<float, 512, 8, 8, true>(m, A);
    if (per <= 6144) return launch_resident<float, 512, 12, 4, true>(m, A);
    if (per <= 8192) return launch_resident<float, 512, 16, 0, true>(m, A);
    return false;
}

// Rows per block of the SELL shapes (0: none): the same for both precisions.
static int sell_rows_per_block(const fk_mesh *m, int width) {
    const int64_t per = rows_per_block(m);
    const int most = width <= 20 ? 2048 : width <= 32 ? 1024 : 0;
    const int R = static_cast<int>((per + 511) / 512 * 512);
    return R <= most ? R : 0;
}

// By the longest row (up to 16 entries: a numbering of a structured mesh; 20:
// the same with slices padded to a common offset set; 32: Delaunay meshes of
// some hundred nodes) and the rows per block. One longer row keeps the whole
// mesh on the three kernels: so do Delaunay meshes of 4k nodes and more, where
// one row in 500 has 33 to 65. The values, LDS indices and halo of more rows do
// not fit the registers. Measured per iteration (us; three-kernel iteration in
// brackets), randomly numbered Kuhn meshes:
//   FP64  n = 20 2.8 (14.0)  n = 41 3.4 (15.9)  n = 55 4.5 (24.4)  n = 70 7.5 (29.6)
//   FP32  n = 20 3.8 (15.3)  n = 41 4.7 (17.4)  n = 55 6.4 (21.2)  n = 70 6.5 (24.8)
static bool launch_sell(fk_mesh *m, ResidentArgs<double> &A) {
    const int w = m->res_width;
    switch (m->res_R) {
        case 512:
            return w <= 16   ? launch_resident<double, 512, 1, 1, false, 16>(m, A)
                   : w <= 20 ? launch_resident<double, 512, 1, 1, false, 20>(m, A)
                             : launch_resident<double, 512, 1, 1, false, 32>(m, A);
        case 1024:
            return w <= 16   ? launch_resident<double, 512, 2, 2, false, 16>(m, A)
                   : w <= 20 ? launch_resident<double, 512, 2, 2, false, 20>(m, A)
                             : false;
        case 1536: return w <= 16 && launch_resident<double, 512, 3, 3, false, 16>(m, A);
        default: return false;
    }
}

static bool launch_sell(fk_mesh *m, ResidentArgs<float> &A) {
    const int w = m->res_width;
    switch (m->res_R) {
        case 512:
            return w <= 16   ? launch_resident<float, 512, 1, 1, true, 16>(m, A)
                   : w <= 20 ? launch_resident<float, 512, 1, 1, true, 20>(m, A)
                             : launch_resident<float, 512, 1, 1, true, 32>(m, A);
        case 1024:
            return w <= 16   ? launch_resident<float, 512, 2, 2, true, 16>(m, A)
                   : w <= 20 ? launch_resident<float, 512, 2, 2, true, 20>(m, A)
                             : launch_resident<float, 512, 2, 2, true, 32>(m, A);
        case 1536:
            return w <= 16 ? launch_resident<float, 512, 3, 3, true, 16>(m, A)
                           : launch_resident<float, 512, 3, 3, true, 20>(m, A);
        case 2048:
            return w <= 16 ? launch_resident<float, 512, 4, 4, true, 16>(m, A)
                           : launch_resident<float, 512, 4, 4, true, 20>(m, A);
        default: return false;
    }
}

// The lists of resident_lists.h on the device. No lists (res_R = 0: the three
// kernels) where the mesh is too large or its rows too long for the resident
// launch, or where the lists cannot be had: the solves do not need them.
void build_resident_sell(fk_mesh *m, const std::vector<int32_t> &rp, const std::vector<int32_t> &ci,
                         const std::vector<int32_t> &width, const std::vector<std::vector<int32_t>> &shared,
                         const std::vector<int64_t> &vptr) {
    m->res_R = 0;
    int32_t most = 0;
    for (int32_t w : width) most = std::max(most, w < 0 ? -w : w);
    const int R = sell_rows_per_block(m, most);
    if (!R || most == 0) return;
    try {
        ResidentLists l;
        if (!resident_lists(m->nv, R, rp, ci, width, shared, vptr, l)) return;
        m->res_sidx.alloc(l.idx.size());
        m->res_halo_ptr.alloc(l.ptr.size());
        m->res_halo.alloc(std::max<size_t>(l.halo.size(), 1));
        hipStream_t st = m->ctx->stream;
        const auto send = [&](auto &to, const auto &from) {
            FK_HIP(hipMemcpyAsync(to.get(), from.data(), from.size() * sizeof(from[0]), hipMemcpyHostToDevice, st));
        };
        send(m->res_sidx, l.idx);
        send(m->res_halo_ptr, l.ptr);
        if (!l.halo.empty()) send(m->res_halo, l.halo);
        FK_HIP(hipStreamSynchronize(st));
        m->res_R = R;
        m->res_width = most;
        m->res_halo_max = l.halo_max;
    } catch (const Error &e) {
        if (e.code != FK_ERR_OOM) throw;
        (void)hipGetLastError();
    } catch (const std::bad_alloc &) {
    }
}

bool resident_allowed(fk_context *c) {
    if (c->timing.enabled || !c->resident) return false;
    if (c->resident_skip == 0) return true;
    --c->resident_skip;
    return false;
}

// A wait that runs out costs about a second. Another process that keeps the
// CUs does so for longer than one solve: the solves that follow it, 8 and after
// every further time-out in a row twice as many up to 1024, run on the three
// kernels before one is tried again.
static bool timed_out(fk_context *c, bool yes) {
    c->resident_pause = yes ? std::min(std::max(2 * c->resident_pause, 8), 1024) : 0;
    c->resident_skip = c->resident_pause;
    return yes;
}

// the copy of the matrix a resident launch can run on, with fresh values
static bool resident_kind(const fk_mesh *m) {
    if (m->kind == FK_SPMV_STENCIL) return m->st_K <= kResK;
    return m->kind == FK_SPMV_SELL64 && m->format != FK_SPMV_CSR && m->have_sell && m->res_R > 0;
}

bool resident_pcg_f64(fk_mesh *m, double rtol, int64_t max_iter, double bb_ref, CgState *out) {
    if (!resident_kind(m) || !resident_allowed(m->ctx)) return false;
    const bool stencil = m->kind == FK_SPMV_STENCIL;
    PcgWork<double> &w = m->w64;
    ResidentArgs<double> A{};
    A.val = stencil ? m->st_val64.get() : m->sell_val64.get();
    A.dinv = w.dinv.get();
    A.r0 = w.r.get();
    A.x = w.x.get();
    A.state = w.state.get();
    A.ld = static_cast<int32_t>(m->st_ld);
    A.n = static_cast<int32_t>(m->nv);
    A.K = m->st_K;
    A.bb_ref = bb_ref;
    A.rtol = rtol;
    A.max_iter = std::min(max_iter, kClosing / 2);
    // one resident launch of this process at a time on the device: the blocks
    // of two would take each other's CUs and wait for blocks not yet started
    const std::lock_guard<std::mutex> alone(resident_mutex(m->ctx->device));
    if (!(stencil ? launch_by_rows(m, A) : launch_sell(m, A))) return false;
    hipStream_t st = m->ctx->stream;
    CgState *hs = m->hstate.ptr;
    FK_HIP(hipMemcpyAsync(hs, w.state.get(), sizeof(CgState), hipMemcpyDeviceToHost, st));
    FK_HIP(hipStreamSynchronize(st));
    // a wait ran out (another process's launch); r0 is unchanged
    if (timed_out(m->ctx, hs->status == FK_ERR_HIP || hs->timed_out)) return false;
    *out = *hs;
    return true;
}

// The FP32-refined solve of solve.hip's solve_f32_replace from the FP64
// residual in r64 (its norm^2 rr): false when this mesh or moment does not
// allow a resident launch; u and r64 may then have changed if one was started.
bool resident_refined(fk_mesh *m, double *u, const double *b, double rr, double thresh, double delta, int64_t max_iter,
                      int chunk, int64_t *iters, int32_t *nrep, double *rr_out, int *status, bool *started) {
    *started = false;
    if (!resident_kind(m) || !resident_allowed(m->ctx)) return false;
    const bool stencil = m->kind == FK_SPMV_STENCIL;
    PcgWork<float> &w = m->w32;
    if (!m->ru) {
        m->ru.alloc(1);
        m->hru.alloc(2);
    }
    ResidentArgs<float> A{};
    A.val = stencil ? m->st_val32.get() : m->sell_val32.get();
    A.dinv = w.dinv.get();
    A.state = w.state.get();
    A.ld = static_cast<int32_t>(m->st_ld);
    A.n = static_cast<int32_t>(m->nv);
    A.K = m->st_K;
    A.max_iter = max_iter;
    A.u = u;
    A.b = b;
    A.r64 = m->r64.get();
    A.val64 = stencil ? m->st_val64.get() : m->sell_val64.get();
    A.diag64 = m->sell_diag64.get();
    A.ru = m->ru.get();
    A.p = w.p.get();
    A.us = 1;
    A.s = 1.0 / std::sqrt(rr);
    A.target2 = thresh * A.s * A.s;
    A.thresh64 = thresh;
    A.delta2 = delta * delta;
    A.G = chunk;
    const std::lock_guard<std::mutex> alone(resident_mutex(m->ctx->device));
    if (!(stencil ? launch_by_rows(m, A) : launch_sell(m, A))) return false;
    *started = true;
    hipStream_t st = m->ctx->stream;
    CgState *hs = m->hstate.ptr;
    RuState *hr = m->hru.ptr;
    FK_HIP(hipMemcpyAsync(hs, w.state.get(), sizeof(CgState), hipMemcpyDeviceToHost, st));
    FK_HIP(hipMemcpyAsync(hr, m->ru.get(), sizeof(RuState), hipMemcpyDeviceToHost, st));
    FK_HIP(hipStreamSynchronize(st));
    if (timed_out(m->ctx, hr->status == FK_ERR_HIP)) return false;  // a wait ran out (another process's launch)
    *iters = hs->iters;
    *nrep = hr->nrep;
    *rr_out = hr->rr64;
    *status = hr->status;
    return true;
}

// ---- batches ----------------------------------------------------------------
// Every system (mesh, right-hand side) is a group of blocks of its own that
// solves and stops by itself; a launch holds as many systems as fit the chip at
// once, so no group ever waits for a block that has not started. Systems are
// packed into launches largest first: those of one launch take about equally
// many iterations.
//
// Rows per block: the fewest with which one launch holds the batch (an
// iteration takes 4.6, 5.2 and 6.2 us with 512, 1024 and 2048 rows a block),
// else 2048, and no more than kResBatchLaunches launches: a launch ends with
// its slowest system, and with many of them the three kernels per iteration,
// which read a matrix value once for all right-hand sides of its mesh, win.
// Solve of 3 right-hand sides per mesh, three kernels against launches of 2048
// rows a block: 10 meshes of 10..20 cells 3.89 to 1.05 ms (0.80 with 512 rows),
// 20 of 10..40 (3 launches) 15.5 to 5.4, 6 of 40..50 (4) 19.6 to 10.2, 40 of
// 10..44 (7) 21.7 to 14.6, 50 of 10..50 (12) 36.1 to 29.3, 100 of 10..40 (15)
// 30.1 to 28.0, 16 of 50..60 (17) 55.4 to 65.2, 64 of 10..60 (27) 67.1 to 71.3.
constexpr size_t kResBatchLaunches = 12;

template <int BLOCK, int RPT, int NK>
static bool launch_batch(ResidentBatch &B, const std::vector<ResidentSystem> &sys, double delta, int64_t max_iter,
                         int chunk, size_t most) {
    constexpr int R = BLOCK * RPT, U = 2 * RPT + 2;
    if (B.started) return false;  // an earlier shape did not fit the device after all
    fk_context *ctx = B.ctx;
    hipStream_t st = ctx->stream;
    const int S = static_cast<int>(sys.size());
    std::vector<ResidentArgs<float>> args(static_cast<size_t>(S));
    size_t lds = 0;
    int64_t words = 0, floats = 0;
    for (int s = 0; s < S; ++s) {
        const ResidentSystem &q = sys[s];
        ResidentArgs<float> &A = args[s];
        int32_t elements = 0;
        if (q.K < 1 || q.K > kResK || !place_windows<float>(q.off, q.K, R, A, &elements) || elements - R > U * BLOCK) return false;
        lds = std::max(lds, (static_cast<size_t>(elements) + 1) * sizeof(float));
        A.nb = (q.n + R - 1) / R;
        if (A.nb > kMaxResidentBlocks) return false;
        A.stride = static_cast<int32_t>((static_cast<int64_t>(A.nb) * R + q.off[q.K - 1] + R + 63) / 64 * 64);
        words += reduce_words(A.nb);
        floats += 2 * static_cast<int64_t>(A.stride);
    }
    if (lds > static_cast<size_t>(kResLdsMax)) return false;
    auto kern = k_resident_batch<float, BLOCK, RPT, NK, U>;
    FK_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                               static_cast<int>(lds)));
    int per_cu = 0;
    FK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(kern), BLOCK, lds));
    const int room = std::min(per_cu, 2) * ctx->num_cus;
    if (room < 1) return false;
    for (const ResidentArgs<float> &A : args)
        if (A.nb > room) return false;
    // launches: first fit, largest systems first
    std::vector<int> order(static_cast<size_t>(S));
    for (int s = 0; s < S; ++s) order[s] = s;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return sys[a].n > sys[b].n; });
    std::vector<std::vector<int2>> rounds;
    for (int s : order) {
        size_t k = 0;
        while (k < rounds.size() && static_cast<int>(rounds[k].size()) + args[s].nb > room) ++k;
        if (k == rounds.size()) rounds.emplace_back();
        for (int b = 0; b < args[s].nb; ++b) rounds[k].push_back(make_int2(s, b));
    }
    if (rounds.size() > most) return false;
    std::vector<int2> table;
    for (const auto &r : rounds) table.insert(table.end(), r.begin(), r.end());
    if (!have_memory([&] {
            B.words.ensure(words);
            B.w.ensure(floats);
            B.args.ensure(S * sizeof(ResidentArgs<float>));
            B.state.ensure(S);
            B.ru.ensure(S);
            B.table.ensure(table.size());
        }))
        return false;
    words = floats = 0;
    for (int s = 0; s < S; ++s) {
        const ResidentSystem &q = sys[s];
        ResidentArgs<float> &A = args[s];
        A.val = q.val32;
        A.dinv = q.dinv;
        A.w = B.w.get() + floats;
        A.slots = B.words.get() + words;
        A.state = B.state.get() + s;
        A.ld = q.n;
        A.n = q.n;
        A.K = q.K;
        A.max_iter = max_iter;
        A.u = q.u;
        A.us = q.us;
        A.r64 = q.r64;
        A.val64 = q.val64;
        A.diag64 = q.diag64;
        A.p = q.p;
        A.ru = B.ru.get() + s;
        A.s = q.s;
        A.target2 = q.target2;
        A.thresh64 = q.thresh64;
        A.delta2 = delta * delta;
        A.G = chunk;
        A.first = 0u - ctx->resident_rounds;
        words += reduce_words(A.nb);
        floats += 2 * static_cast<int64_t>(A.stride);
    }
    FK_HIP(hipMemcpyAsync(B.args.get(), args.data(), S * sizeof(ResidentArgs<float>), hipMemcpyHostToDevice, st));
    FK_HIP(hipMemcpyAsync(B.table.get(), table.data(), table.size() * sizeof(int2), hipMemcpyHostToDevice, st));
    k_resident_zero<<<256, 256, 0, st>>>(B.words.get(), words, B.w.get(), floats);
    FK_HIP(hipGetLastError());
    const auto *dargs = reinterpret_cast<const ResidentArgs<float> *>(B.args.get());
    const int2 *at = B.table.get();
    B.started = true;
    for (const auto &r : rounds) {
        void *params[] = {&dargs, &at};
        const hipError_t e = hipLaunchCooperativeKernel(reinterpret_cast<const void *>(kern),
                                                        dim3(static_cast<unsigned>(r.size())), dim3(BLOCK), params,
                                                        static_cast<unsigned>(lds), st);
        if (e == hipErrorCooperativeLaunchTooLarge) {  // not all blocks fit at once on this device
            (void)hipGetLastError();
            FK_HIP(hipStreamSynchronize(st));
            return false;
        }
        FK_HIP(e);
        at += r.size();
    }
    FK_HIP(hipStreamSynchronize(st));  // args and table go out of scope
    B.rows = R;
    B.launches = static_cast<int32_t>(rounds.size());
    return true;
}

bool resident_batch(ResidentBatch &B, const std::vector<ResidentSystem> &sys, double delta, int64_t max_iter, int chunk,
                    std::vector<CgState> &state, std::vector<RuState> &ru) {
    B.rows = B.launches = 0;
    if (sys.empty()) return true;
    const std::lock_guard<std::mutex> alone(resident_mutex(B.ctx->device));
    B.started = false;
    if (!launch_batch<512, 1, 1>(B, sys, delta, max_iter, chunk, 1) &&
        !launch_batch<512, 2, 2>(B, sys, delta, max_iter, chunk, 1) &&
        !launch_batch<512, 4, 4>(B, sys, delta, max_iter, chunk, kResBatchLaunches))
        return false;
    hipStream_t st = B.ctx->stream;
    const size_t S = sys.size();
    state.resize(S);
    ru.resize(S);
    FK_HIP(hipMemcpyAsync(state.data(), B.state.get(), S * sizeof(CgState), hipMemcpyDeviceToHost, st));
    FK_HIP(hipMemcpyAsync(ru.data(), B.ru.get(), S * sizeof(RuState), hipMemcpyDeviceToHost, st));
    FK_HIP(hipStreamSynchronize(st));
    const bool late = std::any_of(ru.begin(), ru.end(), [](const RuState &r) { return r.status == FK_ERR_HIP; });
    if (timed_out(B.ctx, late)) {  // a wait ran out (another process's launch)
        B.rows = B.launches = 0;
        return false;
    }
    return true;
}

}  // namespace fk
