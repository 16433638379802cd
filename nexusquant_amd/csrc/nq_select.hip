// Keep-mask construction on gfx950: BOS + recent window + top-k of the
// evictable prefix + protected positions, and the ascending kept-index list.
//
// One 1024-thread block per batch row.  What bounds it is one CU's chain of
// block-wide steps, so the design has few of them and keeps the row's
// order-preserving 32-bit keys in registers, 16384 positions (a window) at a
// time: a row of one window is loaded once, a longer one streams through every
// pass with the next window's loads in flight (the first window's of the next
// pass among them).  Lane l of wave v holds positions base + 1024 v + 64 j + l,
// so loads and stores are coalesced and the order of positions is the order of
// (window, wave, j, lane): ranks come from ballots.
//  1. The candidates' smallest and largest key, then a 2048-bin LDS histogram
//     over exactly that range: the bins follow the row's own spread, so few
//     lanes of an atomic meet on one bin (the top byte of a float has a handful
//     of values, and an atomic on it serialises most of a wave) and the bin that
//     holds the k-th key is small.
//  2. That bin's keys, at most 256 of them, are collected in LDS and each is
//     ranked against all by four threads; a fuller bin is split again (at most
//     two more times: 11 of 32 bits a pass).  Rows of at most 256 candidates
//     start here.  (Ranking up to 1024 keys, one thread each, took 36 us at 512
//     positions against 20 for four radix passes.)
//  3. Keys above the threshold are kept, and of those equal to it the first
//     (lowest-position) ones.  Per-wave counts are scanned once and every lane
//     writes its flags and list entries: kept positions ascending from the
//     front, evicted positions descending from the back.
// Ties at the threshold therefore keep the lowest positions; torch.topk leaves
// their order unspecified.
// Measured, one row, between events (us; a 4-pass 8-bit radix select that
// staged the keys in LDS before): 512 positions 20.2 -> 15.6, 8191 26.0 -> 16.8,
// 16384 33.7 -> 19.3, 65521 159 -> 52, 131072 310 -> 82.
#include "nq_common.h"

namespace nq {

constexpr int kSelThreads = 1024;
constexpr int kSelWaves = kSelThreads / 64;
constexpr int kPer = 16;                   // positions per thread in a window
constexpr int kWin = kSelThreads * kPer;   // positions per window
constexpr int kBins = 2048;                // histogram bins, 11 bits a pass
constexpr int kList = 256;                 // keys ranked directly, four threads each

__device__ __forceinline__ uint32_t order_key(float f) {
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Inclusive block scan of one value per thread.  Uses lds[0 .. kSelWaves - 1] and ends
// without a barrier: the caller puts one before lds is written again.
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* lds) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) lds[wave] = x;
    __syncthreads();
    uint32_t before = 0;
#pragma unroll
    for (int w = 0; w < kSelWaves; ++w) before += w < wave ? lds[w] : 0u;
    return x + before;
}

struct SelectArgs {
    const float* importance;  // [batch, seq]
    uint8_t* keep;            // [batch, seq]
    int32_t* kept_idx;        // [batch, seq] kept positions ascending, then evicted descending
    int32_t* n_kept;          // [batch]
    const int32_t* protected_pos;
    int32_t n_protected;
    int32_t seq, prefix, k, window;
};

__global__ __launch_bounds__(kSelThreads) void keep_mask_kernel(SelectArgs a) {
    __shared__ uint32_t s_bins[kBins];                 // histogram, then the protected positions' bitmap
    __shared__ __align__(16) uint32_t s_list[kList];
    __shared__ uint32_t s_scan[kSelWaves];
    __shared__ uint32_t s_mm[2][kSelWaves];
    __shared__ uint32_t s_cnt[2][kSelWaves];           // per wave: threshold-equal keys, kept positions
    __shared__ uint32_t s_sel[4];                      // bin or key, keys above it, keys in it, list length
    const int row = blockIdx.x;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const float* imp = a.importance + (size_t)row * a.seq;
    const int n_cand = a.prefix > 1 ? a.prefix - 1 : 0;  // candidates: positions 1 .. prefix - 1
    const int n_win = (a.seq + kWin - 1) / kWin;
    const int first = wave * (kPer * 64) + lane;         // this lane's first position of a window
    auto cand = [&](int p) { return (uint32_t)(p - 1) < (uint32_t)n_cand; };
    float v[kPer];     // the raw values of the window loaded next
    uint32_t u[kPer];  // the keys of the current window
    auto load = [&](int win) {
        const float* src = imp + (size_t)win * kWin + first;
        if ((win + 1) * (int64_t)kWin <= a.seq) {
#pragma unroll
            for (int j = 0; j < kPer; ++j) v[j] = src[64 * j];
        } else {
            const int left = a.seq - (win * kWin + first);  // positions past the row are no candidates
#pragma unroll
            for (int j = 0; j < kPer; ++j) v[j] = 64 * j < left ? src[64 * j] : 0.0f;
        }
    };
    // the keys of window win (its loads are in flight), the next window's loads issued
    auto take = [&](int win) {
#pragma unroll
        for (int j = 0; j < kPer; ++j) u[j] = order_key(v[j]);
        if (n_win > 1) load(win + 1 < n_win ? win + 1 : 0);
    };
    // body(j, is position j of this lane a candidate), without the test in
    // windows that lie inside the candidates
    auto each = [&](int win, auto body) {
        if (win > 0 && (win + 1) * (int64_t)kWin <= n_cand) {
#pragma unroll
            for (int j = 0; j < kPer; ++j) body(j, true);
        } else {
            const int p0 = win * kWin + first;
#pragma unroll
            for (int j = 0; j < kPer; ++j) body(j, cand(p0 + 64 * j));
        }
    };
    uint32_t want = (uint32_t)a.k, thr = 0, n_eq = 0;
    if (want > 0) {
        if (t == 0) s_sel[3] = 0;
        uint32_t lo = 0, range = 0xffffffffu, in_bin = (uint32_t)n_cand;
        load(0);
        if (n_win == 1) take(0);
        if (in_bin > (uint32_t)kList) {
            uint32_t kmin = 0xffffffffu, kmax = 0;
            for (int win = 0; win < n_win; ++win) {
                if (n_win > 1) take(win);
                each(win, [&](int j, bool c) {
                    if (c) {
                        kmin = min(kmin, u[j]);
                        kmax = max(kmax, u[j]);
                    }
                });
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                kmin = min(kmin, (uint32_t)__shfl_xor(kmin, o, 64));
                kmax = max(kmax, (uint32_t)__shfl_xor(kmax, o, 64));
            }
            if (lane == 0) {
                s_mm[0][wave] = kmin;
                s_mm[1][wave] = kmax;
            }
            __syncthreads();
#pragma unroll
            for (int w = 0; w < kSelWaves; ++w) {
                kmin = min(kmin, s_mm[0][w]);
                kmax = max(kmax, s_mm[1][w]);
            }
            lo = kmin;
            range = kmax - kmin;
        }
        // split the range until its k-th key's bin can be ranked directly, or
        // holds a single key value (11 bits a pass: at most three passes)
        while (in_bin > (uint32_t)kList && range > 0) {
            const int bits = 32 - __builtin_clz(range);
            const int shift = bits > 11 ? bits - 11 : 0;
            s_bins[t] = 0;
            s_bins[t + kSelThreads] = 0;
            __syncthreads();
            for (int win = 0; win < n_win; ++win) {
                if (n_win > 1) take(win);
                each(win, [&](int j, bool c) {
                    const uint32_t d = u[j] - lo;
                    if (c && d <= range) atomicAdd(&s_bins[d >> shift], 1u);
                });
            }
            __syncthreads();
            // bins from the top, two a thread: the one where the running count
            // reaches want (unique: the range holds at least want >= 1 keys)
            const uint32_t h0 = s_bins[kBins - 1 - 2 * t], h1 = s_bins[kBins - 2 - 2 * t];
            const uint32_t above = block_scan(h0 + h1, s_scan) - (h0 + h1);
            if (above < want && want <= above + h0 + h1) {
                const bool second = want > above + h0;
                s_sel[0] = (uint32_t)(kBins - 1 - 2 * t) - (second ? 1u : 0u);
                s_sel[1] = above + (second ? h0 : 0u);
                s_sel[2] = second ? h1 : h0;
            }
            __syncthreads();
            lo += s_sel[0] << shift;
            range = (1u << shift) - 1u;
            want -= s_sel[1];
            in_bin = s_sel[2];
        }
        if (range == 0) {  // every key left is the threshold
            thr = lo;
            n_eq = in_bin;
        } else {
            __syncthreads();  // s_sel[3] is cleared
            for (int win = 0; win < n_win; ++win) {
                if (n_win > 1) take(win);
                each(win, [&](int j, bool c) {
                    if (c && u[j] - lo <= range) s_list[atomicAdd(&s_sel[3], 1u)] = u[j];
                });
            }
            __syncthreads();
            // thread t ranks key t / 4 against every fourth run of four keys
            const uint32_t n4 = (in_bin + 3) / 4;
            const uint32_t mine = s_list[min((uint32_t)t >> 2, in_bin - 1)];
            uint32_t gt = 0, eq = 0;
            if (t < 4 * (int)in_bin) {
#pragma unroll 4
                for (uint32_t i = t & 3; i < n4; i += 4) {
                    const uint4 o = *reinterpret_cast<const uint4*>(s_list + 4 * i);
                    const uint32_t ov[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
                    for (uint32_t q = 0; q < 4; ++q) {
                        const bool in = 4 * i + q < in_bin;
                        gt += in && ov[q] > mine ? 1u : 0u;
                        eq += in && ov[q] == mine ? 1u : 0u;
                    }
                }
            }
#pragma unroll
            for (int o = 1; o < 4; o <<= 1) {
                gt += __shfl_xor(gt, o, 64);
                eq += __shfl_xor(eq, o, 64);
            }
            if (t < 4 * (int)in_bin && gt < want && want <= gt + eq) {  // equal keys write the same values
                s_sel[0] = mine;
                s_sel[1] = gt;
                s_sel[2] = eq;
            }
            __syncthreads();
            thr = s_sel[0];
            want -= s_sel[1];
            n_eq = s_sel[2];
        }
    }
    // want = number of threshold-equal keys to keep (lowest positions first)
    const bool all_eq = n_eq == want;
    uint32_t eq_before = 0, kept_before = 0;
    uint8_t* krow = a.keep + (size_t)row * a.seq;
    int32_t* idx = a.kept_idx + (size_t)row * a.seq;
    // counts before this wave's positions of the window, and the window's total
    auto wave_base = [&](int which, uint32_t& total) {
        uint32_t before = 0, sum = 0;
#pragma unroll
        for (int w = 0; w < kSelWaves; ++w) {
            const uint32_t c = s_cnt[which][w];
            before += w < wave ? c : 0u;
            sum += c;
        }
        total = sum;
        return before;
    };
    auto below = [&](uint64_t m) {  // set bits of m in lanes below this one
        return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    };
    for (int win = 0; win < n_win; ++win) {
        const int w0 = win * kWin, p0 = w0 + first;
        if (a.k > 0 && n_win > 1) take(win);
        if (a.n_protected > 0) {  // protected positions never reduce the set
            __syncthreads();  // the bins (or the previous window's bitmap) are read
            if (t < kWin / 32) s_bins[t] = 0;
            __syncthreads();
            for (int j = t; j < a.n_protected; j += kSelThreads) {
                const int p = a.protected_pos[j] - w0;
                if (p >= 0 && p < kWin) atomicOr(&s_bins[p >> 5], 1u << (p & 31));
            }
            __syncthreads();
        }
        uint64_t kept[kPer];  // lane masks of the kept positions
        if (win > 0 && (win + 1) * (int64_t)kWin <= n_cand && (win + 1) * (int64_t)kWin <= a.seq - a.window &&
            all_eq && a.k > 0 && a.n_protected == 0) {
            // inside the candidates: the threshold alone decides
#pragma unroll
            for (int j = 0; j < kPer; ++j) kept[j] = __ballot(u[j] >= thr);
        } else {
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                const int p = p0 + 64 * j;
                bool keep = p == 0 || (a.window > 0 && p >= a.seq - a.window);
                if (a.k > 0 && cand(p)) keep = keep || u[j] > thr || (u[j] == thr && all_eq);
                if (a.n_protected > 0) keep = keep || ((s_bins[(p - w0) >> 5] >> (p & 31)) & 1u);
                kept[j] = __ballot(keep && p < a.seq);
            }
            if (!all_eq) {  // rank the threshold-equal keys: the first `want` of the row stay
                uint32_t n = 0;
#pragma unroll
                for (int j = 0; j < kPer; ++j)
                    n += (uint32_t)__builtin_popcountll(__ballot(cand(p0 + 64 * j) && u[j] == thr));
                if (lane == 0) s_cnt[0][wave] = n;
                __syncthreads();
                uint32_t tot;
                uint32_t rank = eq_before + wave_base(0, tot);
#pragma unroll
                for (int j = 0; j < kPer; ++j) {
                    const bool eq = cand(p0 + 64 * j) && u[j] == thr;
                    const uint64_t m = __ballot(eq);
                    kept[j] |= __ballot(eq && rank + below(m) < want);
                    rank += (uint32_t)__builtin_popcountll(m);
                }
                eq_before += tot;
            }
        }
        uint32_t n = 0;
#pragma unroll
        for (int j = 0; j < kPer; ++j) n += (uint32_t)__builtin_popcountll(kept[j]);
        if (lane == 0) s_cnt[1][wave] = n;
        __syncthreads();
        uint32_t tot;
        uint32_t out = kept_before + wave_base(1, tot);
        // kept positions ascending from the front; an evicted position p has
        // p - o evicted positions before it and goes to seq - 1 - (p - o), so
        // the evicted ones fill the tail descending
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int p = p0 + 64 * j;
            const bool keep = __builtin_amdgcn_inverse_ballot_w64(kept[j]);
            const int o = (int)(out + below(kept[j]));
            if (p < a.seq) {
                krow[p] = keep ? 1 : 0;
                idx[keep ? o : a.seq - 1 - (p - o)] = p;
            }
            out += (uint32_t)__builtin_popcountll(kept[j]);
        }
        kept_before += tot;
        if (n_win > 1) __syncthreads();  // s_cnt is read before the next window writes it
    }
    if (t == 0) a.n_kept[row] = (int32_t)kept_before;
}

}  // namespace nq

extern "C" int nq_keep_mask(const float* importance, int32_t batch, int32_t seq, int32_t sliding_window,
                            int32_t prefix, int32_t k, const int32_t* protected_pos, int32_t n_protected,
                            uint8_t* keep, int32_t* kept_idx, int32_t* n_kept, void* stream) {
    using namespace nq;
    NQ_CHECK_ARG(importance && keep && kept_idx && n_kept, "nq_keep_mask: NULL pointer");
    NQ_CHECK_ARG(batch > 0 && batch <= 65535 && seq >= 0, "nq_keep_mask: bad shape");
    NQ_CHECK_ARG(prefix >= 0 && prefix <= seq, "nq_keep_mask: prefix %d outside [0, %d]", prefix, seq);
    NQ_CHECK_ARG(k >= 0 && k <= (prefix > 1 ? prefix - 1 : 0), "nq_keep_mask: k %d exceeds the prefix", k);
    NQ_CHECK_ARG(sliding_window >= 0, "nq_keep_mask: negative window");
    NQ_CHECK_ARG(n_protected == 0 || protected_pos, "nq_keep_mask: protected list is NULL");
    if (seq == 0) return NQ_OK;
    SelectArgs a;
    a.importance = importance;
    a.keep = keep;
    a.kept_idx = kept_idx;
    a.n_kept = n_kept;
    a.protected_pos = protected_pos;
    a.n_protected = n_protected;
    a.seq = seq;
    a.prefix = prefix;
    a.k = k;
    a.window = sliding_window;
    hipLaunchKernelGGL(keep_mask_kernel, dim3(batch), dim3(kSelThreads), 0, (hipStream_t)stream, a);
    NQ_CHECK_HIP(hipGetLastError());
    return NQ_OK;
}
