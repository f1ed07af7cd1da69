// The cache update of a single incoming token, as far as it hangs on the trackers alone, for the kernels that do the whole
// update (ckv_update.hip) and for the ones of a decoding step that do it beside the scores (ckv_attn_decode.hip).
#pragma once
#include "ckv_common.h"

namespace ckv {
namespace {

// What lane i of a wavefront needs of cascade i, and all lanes of the call: one trip to memory.
struct TokenTrackers {
    int64_t index;       // 0-based global index of the token
    int64_t sinks, per;  // sinks stored before the call; lane: acceptance period
    int32_t st, sx;      // lane: trackers before the call
    __device__ inline void request(const ckv_update_args& A, int64_t n, int64_t h, int64_t token, int lane) {
        index = *A.real_token_idx + token;
        sinks = A.stored_sinks[n * A.stored_sinks_stride[0] + h * A.stored_sinks_stride[1]];
        st = sx = 0;
        per = 1;
        if (lane < A.cascades) {
            const int64_t at = n * A.tracker_stride[0] + h * A.tracker_stride[1] + lane * A.tracker_stride[2];
            st = (int32_t)A.stored_tokens[at];
            sx = (int32_t)A.start_indices[at];
            per = A.do_cache_every_n[lane];
        }
    }
};

// Where a row that comes to a cascade may land, and the trackers after the call: no score has a say in either.  The token
// passes through the full cascades that accept it, pushing their oldest entries on, up to the first cascade that is not full
// or does not accept: a count of trailing ones.  There it is appended, or it challenges the newest entry.
struct TokenPath {
    int stop;                // full, accepting cascades from the front
    int slot;                // lane i < stop: where the row that comes to cascade i lands; lane stop: where it may land; else -1
    int32_t st_new, sx_new;  // lane: trackers after the call
    bool sink;               // the token is a sink: slot is S + index, in every lane
    bool ends, takes;        // there is a cascade `stop`; it appends (else the newest entry, in lane stop's slot, is challenged)
};

__device__ inline int token_lead(int lane, int32_t W, int32_t st, int32_t sx) {   // lane: the newest slot of a cascade with tokens
    return lane * W + (sx > 0 && sx <= st ? sx - 1 : (sx - 1 + st) % st);
}

__device__ inline TokenPath token_path(const ckv_update_args& A, const TokenTrackers& t, int lane) {
    const int C = A.cascades;
    const int32_t W = (int32_t)A.window_size;
    TokenPath w;
    w.stop = 0;
    w.slot = -1;
    w.st_new = t.st;
    w.sx_new = t.sx;
    w.ends = w.takes = false;
    w.sink = t.sinks < A.num_sink;
    if (w.sink) {  // cascading_cache.py:399-431
        w.slot = (int)(A.max_seq_len + t.sinks);
        return w;
    }
    const int64_t rel = t.index - A.num_sink;
    bool on_period;
    if (rel >= 0 && rel < (1ll << 32) && __builtin_amdgcn_ballot_w64(t.per <= 0 || t.per >= (1ll << 32)) == 0) {
        on_period = (uint32_t)rel % (uint32_t)t.per == 0;
    } else {
        on_period = lane < C && rel % t.per == 0;
    }
    const bool takes = lane < C && ((A.eager_fill && t.index <= A.max_seq_len + A.num_sink) || on_period || t.st == 0);
    const uint32_t ahead = (uint32_t)t.sx + (uint32_t)t.st;  // W: the ring's slots; both at most W
    const int phys = lane * W + (int)(ahead < (uint32_t)W ? ahead : ahead < 2u * (uint32_t)W ? ahead - (uint32_t)W : ahead % (uint32_t)W);
    const unsigned long long stays = ~__builtin_amdgcn_ballot_w64(takes && t.st >= W);
    w.stop = stays ? __builtin_ctzll(stays) : CKV_WAVE;  // at most C: the lanes past it take nothing
    w.ends = w.stop < C;
    w.takes = w.ends && (__builtin_amdgcn_ballot_w64(takes) >> w.stop & 1) != 0;
    if (lane < w.stop) {
        w.slot = phys;
        w.sx_new = t.sx + 1 < W ? t.sx + 1 : (t.sx + 1) % W;
    } else if (lane == w.stop && w.ends) {
        w.slot = w.takes ? phys : token_lead(lane, W, t.st, t.sx);
        if (w.takes) w.st_new = t.st + 1;
    }
    return w;
}

// What a cascade's position ids are made of, from the trackers after the call (cascading_cache.py:728-774, 129-142): slot j
// gets ((j + seg - start) mod seg) + ub - seg, where seg is the number of stored tokens and ub the ids still to hand out (all
// stored tokens, less a window per earlier cascade).  Lane i of a wavefront holds cascade i.
struct PosRange {
    bool write;     // every earlier cascade holds tokens and ids are left
    uint32_t seg, add;
    int32_t base;
    __device__ int64_t id_of(uint32_t j) const {
        uint32_t x = j + add;
        if (x >= seg) x -= seg;
        if (x >= seg) x %= seg;  // slots past the stored tokens of a cascade that is not full
        return (int64_t)((int32_t)x + base);
    }
};

__device__ inline PosRange pos_range(int lane, int C, int32_t W, int32_t st, int32_t sx) {   // by every lane: it sums over them
    int32_t tot = C * W;   // ids are indices below max_seq_len: they fit 32 bits
    const unsigned long long below = __builtin_amdgcn_ballot_w64(lane < C && st < W);
    int first_empty = C;
    if (below) {
        tot = lane < C ? st : 0;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) tot += __shfl_xor(tot, off);
        const unsigned long long empty = __builtin_amdgcn_ballot_w64(lane < C && st <= 0);
        if (empty) first_empty = __builtin_ctzll(empty);
    }
    const int32_t ub = tot - lane * W;
    PosRange r;
    r.seg = (uint32_t)(st < W ? st : W);
    r.write = lane <= first_empty && (lane == 0 || ub > 0) && r.seg != 0;
    r.add = r.seg - (uint32_t)sx;  // start < seg or start == 0
    r.base = ub - (int32_t)r.seg;
    return r;
}

}  // namespace
}  // namespace ckv
