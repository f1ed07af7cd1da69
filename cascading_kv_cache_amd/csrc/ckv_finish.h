// The last step of a chunk's scores: per-head sums -> dtype -> head reduction -> EMA / new-token scores
// (cascade_attention.py:231-248, 319-330).
#pragma once
#include "ckv_attn_internal.h"

#include <type_traits>

namespace ckv {

template <typename T>
__device__ inline float round_t(float v) {
    return Elem<T>::to_float(Elem<T>::from_float(v));
}

// Median: lower median (torch.median), element (nh - 1) / 2 of the sorted values.  Up to eight heads stay in registers, without a branch
// a head: a plan works its scores out in code that is cold at every launch.  More heads' values are kept in scratch memory, which the
// launches of the others would pay for.
constexpr int kFewHeads = 8;
enum Reduction { kMeanOfFew, kMaxOfFew, kMedianOfFew, kMeanOrMaxOfMany, kMedianOfMany };

// Eight heads' sums are on their way at a time; they are taken in the order of the heads.  first: that of the first head.
template <typename T, int kHow>
__device__ inline float reduce_heads(const float* first, int nh, int64_t N, int64_t n, int mode) {
    float r = 0.f, x[kFewHeads];
    auto request = [&](int g0) {
#pragma unroll
        for (int u = 0; u < kFewHeads; u++) {
            const float* row = first + (g0 + u < nh ? g0 + u : nh - 1) * N;
            x[u] = row[(uint32_t)n];
        }
    };
    if constexpr (kHow <= kMedianOfFew) {
        [[maybe_unused]] float vals[kFewHeads];
        request(0);
#pragma unroll
        for (int u = 0; u < kFewHeads; u++) {
            const float v = round_t<T>(x[u]);
            const bool in = u < nh;
            if constexpr (kHow == kMeanOfFew) {
                r = in ? __fadd_rn(r, v) : r;
            } else if constexpr (kHow == kMaxOfFew) {
                r = u == 0 ? v : in ? fmaxf(r, v) : r;
            } else {   // sorted in, every place known to the compiler
                bool moves = in;
#pragma unroll
                for (int i = u; i > 0; i--) {
                    const bool on = moves && vals[i - 1] > v;
                    vals[i] = on ? vals[i - 1] : moves || i == u ? v : vals[i];
                    moves = on;
                }
                vals[0] = moves ? v : vals[0];
            }
        }
        if constexpr (kHow == kMeanOfFew) return round_t<T>(r / (float)nh);
        if constexpr (kHow == kMedianOfFew) {
            r = vals[0];
#pragma unroll
            for (int i = 1; i < kFewHeads / 2; i++) r = i == (nh - 1) / 2 ? vals[i] : r;
        }
        return r;
    } else {
        [[maybe_unused]] float vals[kHow == kMedianOfMany ? 128 : 1];
        for (int g0 = 0; g0 < nh; g0 += kFewHeads) {
            request(g0);
#pragma unroll
            for (int u = 0; u < kFewHeads; u++) {
                const int g = g0 + u;
                if (g >= nh) break;
                const float v = round_t<T>(x[u]);
                if constexpr (kHow == kMedianOfMany) {
                    int i = g;
                    while (i > 0 && vals[i - 1] > v) {
                        vals[i] = vals[i - 1];
                        i--;
                    }
                    vals[i] = v;
                } else if (mode == CKV_REDUCE_MAX) {
                    r = g == 0 ? v : fmaxf(r, v);
                } else {
                    r = __fadd_rn(r, v);
                }
            }
        }
        if constexpr (kHow == kMedianOfMany) return vals[(nh - 1) / 2];
        return mode == CKV_REDUCE_MAX ? r : round_t<T>(r / (float)nh);
    }
}

template <typename T, int kHow>
__device__ inline float reduced_sum(const FinishProblem& p, int64_t b, int64_t kvh, int64_t n) {
    return reduce_heads<T, kHow>(p.colsum + (b * p.H + (p.homogeneous ? 0 : kvh * p.heads)) * p.N, p.heads, p.N, n, p.head_reduction);
}

// a slot's score after the call, from that before it
template <typename T, int kHow>
__device__ inline T slot_score(const FinishProblem& p, int64_t b, int64_t kvh, int64_t slot, T old) {
    const float red = reduced_sum<T, kHow>(p, b, kvh, p.num_sink + slot);
    const float decayed = round_t<T>(__fmul_rn(p.beta_pow_q, Elem<T>::to_float(old)));
    return Elem<T>::from_float(__fadd_rn(decayed, red));
}

template <typename T, int kHow>
__device__ inline T token_score(const FinishProblem& p, int64_t b, int64_t kvh, int64_t token) {
    return Elem<T>::from_float(reduced_sum<T, kHow>(p, b, kvh, p.num_sink + p.S + token));
}

// item i of a kv head: its slots, then the call's tokens
template <typename T, int kHow>
__device__ inline void finish_score(const FinishProblem& p, int64_t b, int64_t kvh, int64_t i) {
    if (i < p.S) {
        T* cs = (T*)p.cache_s + b * p.cache_s_stride[0] + kvh * p.cache_s_stride[1] + i * p.cache_s_stride[2];
        const T old = *cs;
        *cs = slot_score<T, kHow>(p, b, kvh, i, old);
    } else {
        const int64_t m = i - p.S;
        ((T*)p.new_scores)[b * p.new_scores_stride[0] + kvh * p.new_scores_stride[1] + m * p.new_scores_stride[2]] =
            token_score<T, kHow>(p, b, kvh, m);
    }
}

// calls `launch` with the kernel's way to reduce
template <typename F>
inline auto with_reduction(const FinishProblem& p, const F& launch) {
    const bool few = p.heads <= kFewHeads;
    if (p.head_reduction == CKV_REDUCE_MAX && few) return launch(std::integral_constant<int, kMaxOfFew>{});
    if (p.head_reduction == CKV_REDUCE_MEAN && few) return launch(std::integral_constant<int, kMeanOfFew>{});
    if (p.head_reduction == CKV_REDUCE_MAX || p.head_reduction == CKV_REDUCE_MEAN) return launch(std::integral_constant<int, kMeanOrMaxOfMany>{});
    return few ? launch(std::integral_constant<int, kMedianOfFew>{}) : launch(std::integral_constant<int, kMedianOfMany>{});
}

}  // namespace ckv
