// Device helpers of the register-resident PCG kernels (gfx950, wave64): one
// cooperative launch whose blocks stay on the chip for a whole solve and
// exchange data through memory at agent scope.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace fk {

using u64 = unsigned long long;

// ---- 64-lane sums with DPP moves ------------------------------------------
// Fixed order: pairs, quads, halves and rows of 16 by DPP, then the four rows.
// A DPP step costs a few cycles where the ds_bpermute of __shfl_xor costs
// over a hundred.
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
    const u64 b = static_cast<u64>(__double_as_longlong(v));
    const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double(static_cast<long long>((static_cast<u64>(static_cast<uint32_t>(hi)) << 32) |
                                                       static_cast<uint32_t>(lo)));
}
__device__ __forceinline__ double lane_value(double v, int lane) {
    const u64 b = static_cast<u64>(__double_as_longlong(v));
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<int>(b), lane);
    const uint32_t hi = __builtin_amdgcn_readlane(static_cast<int>(b >> 32), lane);
    return __longlong_as_double(static_cast<long long>((static_cast<u64>(hi) << 32) | lo));
}
// every lane: the sum over its row of 16 lanes
__device__ __forceinline__ double row16_sum(double v) {
    v += dpp_move<0xB1>(v);   // quad_perm [1,0,3,2]
    v += dpp_move<0x4E>(v);   // quad_perm [2,3,0,1]
    v += dpp_move<0x141>(v);  // row_half_mirror
    v += dpp_move<0x140>(v);  // row_mirror
    return v;
}
__device__ __forceinline__ double wave64_sum(double v) {
    v = row16_sum(v);
    return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}
// a in one half of the lanes and b in the other, each the sum of its halves
// (SWAP 32), or the same for the rows of 16 within each half (SWAP 16): one
// swap and one add for two values
template <int SWAP>
__device__ __forceinline__ double fold_pair(double a, double b) {
    const uint32_t alo = __double2loint(a), ahi = __double2hiint(a), blo = __double2loint(b), bhi = __double2hiint(b);
    if constexpr (SWAP == 32) {
        const auto lo = __builtin_amdgcn_permlane32_swap(alo, blo, false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(ahi, bhi, false, false);
        return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
    } else {
        const auto lo = __builtin_amdgcn_permlane16_swap(alo, blo, false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(ahi, bhi, false, false);
        return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
    }
}
// the wave sums of a, b, c, d in the lane rows 0, 2, 1, 3
__device__ __forceinline__ double fold4(double a, double b, double c, double d) {
    return row16_sum(fold_pair<16>(fold_pair<32>(a, b), fold_pair<32>(c, d)));
}

// ---- all-reduce between the blocks of a cooperative launch -------------------
// Five sums. A block leaves its partial sums in a line of ten 64-bit words that
// carry half a double and a 32-bit tag each; readers poll until every word
// shows the tag of this round, so no counter, flag or fence is needed for the
// sums, and every block adds them in the same order. Lines alternate by the
// tag's parity: a block can write round t + 2 only after it has seen the sums
// of round t + 1, which exist only once every block has read round t. Tags
// start at 1 on lines cleared before the launch.
//
// Every block polls all lines of its copy: a block writes kReduceCopies copies
// of its line, each with one store instruction, and the blocks read the copy of
// their number modulo that, since loads of one line from many blocks are
// served one after another. Measured for 256 blocks of 512 threads (us per
// round): 2.9; with the words of one value from all blocks side by side, one
// 8-byte store per block each, 3.9; one copy 5.6 (16 blocks: 1.6, 1.5, 1.6).
// Sums by groups of 16 blocks and then of the groups took two trips through
// memory and 12 us: all blocks polling the few group sums wait for each other.
//
// Waits are bounded: after kSpinLimit polls (about a second; a co-resident
// block answers in microseconds) the round fails and the kernel ends. The round
// with tag 0, which tags counted up from a first one of 1 do not reach, fails
// at its first poll.
constexpr int kSpinLimit = 1 << 20;
constexpr int kMaxResidentBlocks = 256;
constexpr int kReduceCopies = 8;
constexpr int kReduceLine = 16;   // words of a line, ten used
constexpr int kReduceWaves = 8;   // polling waves of a block
constexpr int reduce_words(int nb) { return 2 * kReduceCopies * nb * kReduceLine; }
constexpr int kReduceShared = 5 * 16 + 5 * kReduceWaves + 1;  // doubles of LDS

// Sum of v[0..5) over all threads of the nb blocks of a group (block `me` of
// it), the same bits in every thread; false when the wait ran out. Before the blocks' partials leave, every
// wave waits for its earlier stores, so agent-scope stores made before the
// call are visible to agent-scope loads made after it. sh: kReduceShared
// doubles, the last one 0 before the first call; lines: reduce_words(nb) words.
template <int BLOCK>
__device__ __forceinline__ bool all_reduce5(double (&v)[5], u64 *__restrict__ lines, int me, int nb, uint32_t tag,
                                            double *sh) {
    constexpr int W = BLOCK / 64, P = kReduceWaves;
    static_assert(W >= P && W <= 16, "one row of lanes adds the wave sums");
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, row = l >> 4, c = l & 15;
    double *part = sh + 5 * 16, *failed = part + 5 * P;
    const double f = fold4(v[0], v[2], v[1], v[3]);  // value k in lane row k
    const double f4 = row16_sum(fold_pair<16>(fold_pair<32>(v[4], 0.0), 0.0));
    if (c == 0) sh[row * 16 + w] = f;
    if (l == 0) sh[4 * 16 + w] = f4;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    u64 *base = lines + (tag & 1) * (kReduceCopies * kReduceLine * nb);
    if (w == 0) {
        // lane 16 k + 2 copy + half writes that half of value k
        const u64 a = static_cast<u64>(__double_as_longlong(row16_sum(c < W ? sh[row * 16 + c] : 0.0)));
        const u64 b = static_cast<u64>(__double_as_longlong(row16_sum(c < W ? sh[4 * 16 + c] : 0.0)));
        const int copy = c >> 1, half = c & 1;
        static_assert(kReduceCopies == 8, "16 lanes write two halves to each copy");
        u64 *line = base + (copy * nb + me) * kReduceLine;
        const u64 high = 0xffffffff00000000ull;
        __hip_atomic_store(line + 2 * row + half, (half ? a & high : a << 32) | tag, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        if (row == 0)
            __hip_atomic_store(line + 8 + half, (half ? b & high : b << 32) | tag, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
    if (w < P) {
        // a row of lanes polls a line; block 4 P i + 4 w + row
        const u64 *mine = base + (me % kReduceCopies) * (nb * kReduceLine);
        constexpr int PER = kMaxResidentBlocks / (4 * P);
        u64 a[PER];
#pragma unroll
        for (int i = 0; i < PER; ++i) a[i] = tag;  // a lane without a word holds the tag over zero
        int spin = tag == 0 ? kSpinLimit : 0;
        uint32_t miss;
        do {
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int b = 4 * P * i + 4 * w + row;
                if (b < nb && c < 10)
                    a[i] = __hip_atomic_load(mine + b * kReduceLine + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            miss = 0;
#pragma unroll
            for (int i = 0; i < PER; ++i) miss |= static_cast<uint32_t>(a[i]) ^ tag;
        } while (__any(miss != 0) && ++spin < kSpinLimit);
        double s = 0.0;  // even lanes: value c / 2, the high half from the next lane
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int lo = static_cast<int>(a[i] >> 32);
            s += __hiloint2double(__builtin_amdgcn_update_dpp(0, lo, 0xB1, 0xf, 0xf, true), lo);
        }
        s = fold_pair<32>(s, s);
        s = fold_pair<16>(s, s);
        if (l < 10 && !(l & 1)) part[(l >> 1) * P + w] = s;
        if (spin >= kSpinLimit && l == 0) *failed = 1.0;
    }
    __syncthreads();
    double t = part[l < 5 * P ? l : 0];
    t += dpp_move<0xB1>(t);
    t += dpp_move<0x4E>(t);
    t += dpp_move<0x141>(t);  // all 8 lanes of value l / 8: its sum
    static_assert(P == 8, "eight partial sums per value");
#pragma unroll
    for (int k = 0; k < 5; ++k) v[k] = lane_value(t, k * P);
    return __builtin_amdgcn_readfirstlane(__double2hiint(*failed)) == 0;
}

// ---- agent-scope row values ----------------------------------------------------
// A value per row, written by the row's owner and read by the blocks that hold
// its neighbours, past the caches of either (cache policy sc1: agent scope).
// Two arrays of `stride` rows used by turns; rows n..stride of both hold zero,
// and a negative row reads zero.
constexpr int kAgentScope = 16;  // sc1

template <typename T>
struct AgentRows {
    __amdgpu_buffer_rsrc_t rsrc;
    int32_t stride;  // bytes
    __device__ __forceinline__ AgentRows(T *base, int32_t stride_rows)
        : rsrc(__builtin_amdgcn_make_buffer_rsrc(base, 0, 2 * stride_rows * static_cast<int32_t>(sizeof(T)),
                                                 0x00020000)),
          stride(stride_rows * static_cast<int32_t>(sizeof(T))) {}
    static __device__ __forceinline__ int32_t offset(int32_t row) {
        return static_cast<int32_t>(static_cast<uint32_t>(row) * static_cast<uint32_t>(sizeof(T)));
    }
    __device__ __forceinline__ T load(uint32_t turn, int32_t row) const {
        const int32_t half = (turn & 1) ? stride : 0;
        if constexpr (sizeof(T) == 8) {
            using V = uint32_t __attribute__((ext_vector_type(2)));
            const V v = __builtin_amdgcn_raw_buffer_load_b64(rsrc, offset(row), half, kAgentScope);
            return __hiloint2double(static_cast<int>(v.y), static_cast<int>(v.x));
        } else {
            return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, offset(row), half, kAgentScope));
        }
    }
    __device__ __forceinline__ void store(uint32_t turn, int32_t row, T v) const {
        const int32_t half = (turn & 1) ? stride : 0;
        if constexpr (sizeof(T) == 8) {
            using V = uint32_t __attribute__((ext_vector_type(2)));
            V w;
            w.x = static_cast<uint32_t>(__double2loint(v));
            w.y = static_cast<uint32_t>(__double2hiint(v));
            __builtin_amdgcn_raw_buffer_store_b64(w, rsrc, offset(row), half, kAgentScope);
        } else {
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rsrc, offset(row), half, kAgentScope);
        }
    }
};

// ---- value columns of the stencil copy ------------------------------------------
// Element (k, row) of the K x ld columns by a buffer load: one 32-bit offset
// per load and no branch. A negative row reads zero; a row past the column
// reads zero or another column's value (rows without a node multiply it by
// D^-1 = 0).
template <typename T>
struct ValueColumns {
    __amdgpu_buffer_rsrc_t rsrc;
    int32_t ld;
    __device__ __forceinline__ ValueColumns(const T *base, int32_t K, int32_t ld_)
        : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(base), 0,
                                                 K * ld_ * static_cast<int32_t>(sizeof(T)), 0x00020000)),
          ld(ld_) {}
    __device__ __forceinline__ T load(int32_t k, int32_t row) const {
        const int32_t at = static_cast<int32_t>(static_cast<uint32_t>(row) * static_cast<uint32_t>(sizeof(T)));
        const int32_t col = k * ld * static_cast<int32_t>(sizeof(T));
        if constexpr (sizeof(T) == 8) {
            using V = uint32_t __attribute__((ext_vector_type(2)));
            const V v = __builtin_amdgcn_raw_buffer_load_b64(rsrc, at, col, 0);
            return __hiloint2double(static_cast<int>(v.y), static_cast<int>(v.x));
        } else {
            return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, at, col, 0));
        }
    }
};

}  // namespace fk
