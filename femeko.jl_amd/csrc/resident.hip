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
#include <algorithm>
#include <cmath>
#include <mutex>
#include <utility>
#include <vector>

#include "device.h"
#include "internal.h"
#include "resident.h"

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
    double bb_ref, rtol;
    int64_t max_iter;
};

// A copy of v that the compiler takes for a new value: addresses computed from
// it inside the iteration loop are not hoisted out of it, where the 14 LDS
// and 8 value offsets of each row would occupy registers for the whole solve.
__device__ __forceinline__ int32_t fresh(int32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}

// row of window element li (LDS index)
template <typename T>
__device__ __forceinline__ int32_t window_row(const ResidentArgs<T> &A, int32_t i0, int32_t li) {
    int32_t d = A.wrow[0];
#pragma unroll
    for (int k = 1; k < kResWindows; ++k) d = li >= A.wbeg[k] ? A.wrow[k] : d;
    return li < A.wbeg[kResWindows] ? i0 + li + d : -1;
}

// RPT rows per thread, the values of the first NK of them in registers (the
// others are streamed from L2 / MALL, a row ahead of their use); U window
// elements per thread at most.
template <typename T, int BLOCK, int RPT, int NK, int U>
__global__ __launch_bounds__(BLOCK) void k_resident_pcg(const ResidentArgs<T> A) {
    extern __shared__ char lds_raw[];
    T *win = reinterpret_cast<T *>(lds_raw);
    __shared__ double sh[5 * (BLOCK / 64 + 1) + 1];
    constexpr int K = kResK, R = BLOCK * RPT;
    const int32_t i0 = logical_block(A.nb) * R;
    const int32_t tid = threadIdx.x;
    const AgentRows<T> rows(A.w, A.stride);
    const ValueColumns<T> vals(A.val, A.K, A.ld);
    const int32_t n = A.n;
    uint32_t tag = 0;
    if (tid == 0) sh[5 * (BLOCK / 64 + 1)] = 0.0;

    T d[RPT], g[RPT], x[RPT], z[RPT], p[RPT], w[RPT];
    T zw[U];
    int32_t li[U];  // LDS index of this thread's window elements (one spare element past the windows)
    T vf[NK > 0 ? NK : 1][K], vb[NK > 0 ? NK : 1][K];
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const int32_t row = i0 + j * BLOCK + tid;
        const bool in = row < n;
        d[j] = in ? A.dinv[row] : T(0);
        const bool free = d[j] != T(0);
        g[j] = free ? T(1) / d[j] : T(0);
        x[j] = T(0);
        z[j] = free ? d[j] * A.r0[row] : T(0);
        p[j] = z[j];
        if (in) rows.store(1, row, z[j]);
        win[A.lown + j * BLOCK + tid] = p[j];
    }
#pragma unroll
    for (int j = 0; j < NK; ++j)
#pragma unroll
        for (int k = 0; k < K; ++k) {
            vf[j][k] = vb[j][k] = T(0);
            if (k < A.K) {
                vf[j][k] = vals.load(k, i0 + j * BLOCK + tid);
                vb[j][k] = vals.load(k, i0 + j * BLOCK + tid - A.off[k]);
            }
        }
    double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    bool alive = all_reduce5<BLOCK>(s, A.slots, A.nb, ++tag, sh);  // every z is out
#pragma unroll
    for (int u = 0; u < U; ++u) {
        // the windows' elements in LDS order, the own rows left out
        const int32_t e = tid + u * BLOCK;
        li[u] = min(e < A.lown ? e : e + R, A.wbeg[kResWindows]);
        zw[u] = rows.load(1, window_row(A, i0, li[u]));
        win[li[u]] = zw[u];
    }
    __syncthreads();

    double rr = 0.0, thresh = 0.0, bb = A.bb_ref;
    int64_t it = 0;
    int code = alive ? -1 : FK_ERR_HIP;  // -1: running
    while (code < 0) {
        ++tag;
        // q = A p in difference form; w = D^-1 q
#pragma unroll
        for (int k = 0; k < 5; ++k) s[k] = 0.0;
        T sf[K], sb[K];
        [[maybe_unused]] const int32_t t0 = fresh(tid);
        if constexpr (NK < RPT) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                sf[k] = sb[k] = T(0);
                if (k < A.K) {
                    sf[k] = vals.load(k, i0 + NK * BLOCK + t0);
                    sb[k] = vals.load(k, i0 + NK * BLOCK + t0 - A.off[k]);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            const int32_t l = j * BLOCK + fresh(tid), row = i0 + l;
            T a0 = T(0), a1 = T(0);
            if (j < NK) {
                const int jk = j < NK ? j : 0;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    a0 += vf[jk][k] * (win[A.lf[k] + l] - p[j]);
                    a1 += vb[jk][k] * (win[A.lb[k] + l] - p[j]);
                }
            } else {
                T nf[K], nbk[K];
                if (j + 1 < RPT) {
#pragma unroll
                    for (int k = 0; k < K; ++k) {
                        nf[k] = nbk[k] = T(0);
                        if (k < A.K) {
                            nf[k] = vals.load(k, row + BLOCK);
                            nbk[k] = vals.load(k, row + BLOCK - A.off[k]);
                        }
                    }
                }
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    a0 += sf[k] * (win[A.lf[k] + l] - p[j]);
                    a1 += sb[k] * (win[A.lb[k] + l] - p[j]);
                }
                if (j + 1 < RPT) {
#pragma unroll
                    for (int k = 0; k < K; ++k) {
                        sf[k] = nf[k];
                        sb[k] = nbk[k];
                    }
                }
            }
            const T q = d[j] != T(0) ? a0 + a1 : T(0);
            w[j] = d[j] * q;
            if (row < n) rows.store(tag, row, w[j]);
            const double zd = static_cast<double>(z[j]), qd = static_cast<double>(q);
            const double rd = static_cast<double>(g[j] * z[j]);
            s[0] += static_cast<double>(p[j]) * qd;
            s[1] += rd * zd;
            s[2] += qd * zd;
            s[3] += qd * static_cast<double>(w[j]);
            s[4] += rd * rd;
            __builtin_amdgcn_sched_barrier(0);
        }
        alive = all_reduce5<BLOCK>(s, A.slots, A.nb, tag, sh);
        T ww[U];
#pragma unroll
        for (int u = 0; u < U; ++u) ww[u] = rows.load(tag, window_row(A, i0, fresh(li[u])));
        const double pq = s[0], rz = s[1];
        const T alpha = static_cast<T>(rz / pq);
        const double al = static_cast<double>(alpha), inv_rz = 1.0 / rz;
        const T beta = static_cast<T>(fmax(rz - al * (2.0 * s[2] - al * s[3]), 0.0) * inv_rz);
        rr = s[4];
        if (it == 0) {
            if (!(bb >= 0.0)) bb = rr;
            thresh = A.rtol * A.rtol * bb;
        }
        code = !alive                                      ? FK_ERR_HIP
               : rr < thresh || (it == 0 && rr == 0.0)     ? FK_OK
               : !isfinite(rr)                             ? FK_ERR_NONFINITE
               : it >= A.max_iter                          ? FK_ERR_NOT_CONVERGED
               : !(pq > 0.0) || !isfinite(pq)              ? FK_ERR_SINGULAR  // not positive definite on the space
                                                           : -1;
        code = __builtin_amdgcn_readfirstlane(code);
        if (code >= 0) break;
        ++it;
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            x[j] += alpha * p[j];
            z[j] -= alpha * w[j];
            p[j] = z[j] + beta * p[j];
            win[A.lown + j * BLOCK + tid] = p[j];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            zw[u] -= alpha * ww[u];
            win[li[u]] = zw[u] + beta * win[li[u]];
        }
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const int32_t row = i0 + j * BLOCK + tid;
        if (row < n) A.x[row] = x[j];
    }
    if (blockIdx.x == 0 && tid == 0) {
        A.state->iters = it;
        A.state->rr = rr;
        A.state->bb = bb;
        A.state->thresh = thresh;
        A.state->status = code;
        A.state->done_at[0] = A.state->done_at[1] = 1;
    }
}

// slots, and the rows n..stride of the two exchange arrays
template <typename T>
__global__ void k_resident_clear(u64 *__restrict__ slots, int words, T *__restrict__ w, int32_t n, int32_t stride) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x, step = gridDim.x * blockDim.x;
    for (int i = t; i < words; i += step) slots[i] = 0;
    for (int i = n + t; i < stride; i += step) w[i] = w[stride + i] = T(0);
}

// ---------------------------------------------------------------------------
// host side

// The windows of a block of R rows, in LDS one after another. False when they
// are too many or too long.
template <typename T>
static bool place_windows(const fk_mesh *m, int R, ResidentArgs<T> &A, int32_t *elements) {
    const int K = m->st_K;
    std::vector<std::pair<int64_t, int64_t>> iv{{0, R}};
    for (int k = 0; k < K; ++k) {
        const int64_t o = m->st_off[k];
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
        A.off[k] = k < K ? m->st_off[k] : 0;
        A.lf[k] = place(A.off[k]);
        A.lb[k] = place(-static_cast<int64_t>(A.off[k]));
    }
    return true;
}

template <typename T, int BLOCK, int RPT, int NK>
static bool launch_resident(fk_mesh *m, ResidentArgs<T> &A) {
    constexpr int R = BLOCK * RPT, U = 2 * RPT + 2;
    const int most = std::min(m->ctx->num_cus, kMaxResidentBlocks);
    int nb = static_cast<int>((m->nv + R - 1) / R);
    // streamed values: one band of rows per XCD
    if (NK < RPT && nb > kNumXcd) nb = std::min((nb + kNumXcd - 1) / kNumXcd * kNumXcd, most);
    int32_t elements = 0;
    if (!place_windows<T>(m, R, A, &elements) || elements - R > U * BLOCK) return false;
    const size_t lds = (static_cast<size_t>(elements) + 1) * sizeof(T);
    if (lds > static_cast<size_t>(kResLdsMax)) return false;
    A.nb = nb;
    // rows past the last, as far as the last block's windows reach, read zero
    const int64_t reach = static_cast<int64_t>(nb) * R + m->st_off[m->st_K - 1] + R;
    const int64_t stride = (reach + 63) / 64 * 64;
    hipStream_t st = m->ctx->stream;
    m->res_slots.ensure(reduce_words(5));
    m->res_w.ensure(static_cast<size_t>(2 * stride));
    A.stride = static_cast<int32_t>(stride);
    A.slots = m->res_slots.get();
    A.w = reinterpret_cast<T *>(m->res_w.get());
    auto kern = k_resident_pcg<T, BLOCK, RPT, NK, U>;
    FK_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                               static_cast<int>(lds)));
    k_resident_clear<T><<<64, 256, 0, st>>>(A.slots, reduce_words(5), A.w, A.n, A.stride);
    FK_HIP(hipGetLastError());
    void *args[] = {&A};
    const hipError_t e = hipLaunchCooperativeKernel(reinterpret_cast<const void *>(kern), dim3(nb), dim3(BLOCK),
                                                    args, static_cast<unsigned>(lds), st);
    if (e == hipErrorCooperativeLaunchTooLarge) {  // not all blocks fit at once on this device
        (void)hipGetLastError();
        return false;
    }
    FK_HIP(e);
    return true;
}

static std::mutex &resident_mutex(int device) {
    static std::mutex all[64];
    return all[device & 63];
}

// Rows per block R by the number of rows: the smallest of the list with which
// at most one block per CU covers them. Few rows per thread leave room for all
// their matrix values in registers (NK = RPT) and shorten every step between
// two exchanges; beyond 5 per thread the values are streamed. Measured per
// iteration (us; three-kernel iteration in brackets), Kuhn meshes of n cells
// per side:
//   n = 20  512 x 1   4.1 (14.7)     n = 40  512 x 1   4.3 (15.9)
//   n = 60 1024 x 1   5.2 (21.0)     n = 70  512 x 4  10.5 (23.7)
//   n = 79  512 x 4  11.9 (26.9)     n = 85  512 x 5  14.6 (29.4)
//   n = 92  512 x 8  20.6 (32.6)     n = 100 512 x 8  25.1 (36.8)
// More rows than 256 blocks of 4096 keep the three-kernel iteration: the
// windows of more rows per block exceed the LDS.
static bool launch_by_rows(fk_mesh *m, ResidentArgs<double> &A) {
    const int64_t per = (m->nv + std::min(m->ctx->num_cus, kMaxResidentBlocks) - 1) /
                        std::min(m->ctx->num_cus, kMaxResidentBlocks);
    if (per <= 512) return launch_resident<double, 512, 1, 1>(m, A);
    if (per <= 1024) return launch_resident<double, 1024, 1, 1>(m, A);
    if (per <= 1536) return launch_resident<double, 512, 3, 3>(m, A);
    if (per <= 2048) return launch_resident<double, 512, 4, 3>(m, A);
    if (per <= 2560) return launch_resident<double, 512, 5, 3>(m, A);
    if (per <= 3072) return launch_resident<double, 512, 6, 1>(m, A);
    if (per <= 3584) return launch_resident<double, 512, 7, 0>(m, A);
    if (per <= 4096) return launch_resident<double, 512, 8, 0>(m, A);
    return false;
}

bool resident_pcg_f64(fk_mesh *m, double rtol, int64_t max_iter, double bb_ref, CgState *out) {
    if (m->kind != FK_SPMV_STENCIL || m->st_K > kResK || m->ctx->timing.enabled) return false;
    PcgWork<double> &w = m->w64;
    ResidentArgs<double> A{};
    A.val = m->st_val64.get();
    A.dinv = w.dinv.get();
    A.r0 = w.r.get();
    A.x = w.x.get();
    A.state = w.state.get();
    A.ld = static_cast<int32_t>(m->st_ld);
    A.n = static_cast<int32_t>(m->nv);
    A.K = m->st_K;
    A.bb_ref = bb_ref;
    A.rtol = rtol;
    A.max_iter = max_iter;
    // one resident launch of this process at a time on the device: the blocks
    // of two would take each other's CUs and wait for blocks not yet started
    const std::lock_guard<std::mutex> alone(resident_mutex(m->ctx->device));
    if (!launch_by_rows(m, A)) return false;
    hipStream_t st = m->ctx->stream;
    CgState *hs = m->hstate.ptr;
    FK_HIP(hipMemcpyAsync(hs, w.state.get(), sizeof(CgState), hipMemcpyDeviceToHost, st));
    FK_HIP(hipStreamSynchronize(st));
    if (hs->status == FK_ERR_HIP) return false;  // a wait ran out (another process's launch); r0 is unchanged
    *out = *hs;
    return true;
}

}  // namespace fk
