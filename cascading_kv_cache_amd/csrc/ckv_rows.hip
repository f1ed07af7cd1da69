// out = x W^T of a few rows x: the products of a decoding step, with what surrounds them in a decoder layer.  In front: RMSNorm of
// the rows; behind: bias, the gate of a fused MLP, the residual.
//
// Bound by the weights, each of which is read once.  W (N, K) is cut into groups of 16 rows, one v_mfma_f32_16x16x32 operand high;
// the rows of x are the other operand's columns, so up to 16 rows cost what one does.  A wavefront streams its group through a ring
// of 2 KiB stages in LDS (64 elements of 16 rows: two copies of 1 KiB, whole 128-byte lines, past the caches), several stages ahead
// and without a barrier.  A group is shared by kParts wavefronts where N alone has too few groups to keep enough of them in flight.
// One bf16 row, us, torch's operations (product, norm, gate, residual) and this, weights out of memory:
//   6144 x 4096 norm 20 + 6 -> 11        4096 x 4096 residual 20 + 3 -> 8.2    28672 x 4096 norm, gate 60 + 6 + 4 -> 41 (5.7 TB/s)
//   4096 x 14336 residual 26 + 3 -> 22   128256 x 4096 norm 185 + 6 -> 151 (7.0 TB/s)   3584 x 18944 residual 48 + 3 -> 23.5
// Stretches of W by XCD (rows_kernel): the five products above in turn over four layers and a head of 2.8 GB, 491 -> 477 us.
// Ring stages of four parts: 6 and 7 are level (12 with the norm at 6144 x 4096) and leave room for two workgroups, 8 do not (14.3);
// stages of 128 elements are level with two of 64.  Copies through the L2 160 -> 190 us at 128256 x 4096.  How many wavefronts and
// stages a workgroup gets: run_rows below.
//
// The order of a sum is the caller's (kParts, kUnit): part p takes the stretches of kUnit * 64 elements p, p + kParts, ..., one chain
// of matrix instructions each, and the parts are added up in order.  Another order is as good, but flips the rounding of a few
// outputs in ten thousand, which a decoder of random weights turns into a percent of its logits; so a decoder that has used a library's
// products before keeps their order (row_products.py finds it).  Where the library cuts the sums of some tiles, so does kCut: heads of
// 128256 x 4096 and 152064 x 3584, norm, a row, 150.5 and 156 us with it, 150.7 and 154 without (torch's operations 190 and 226).
#include "ckv_common.h"

#include <algorithm>

namespace ckv {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 rows_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 rows_f16x8 __attribute__((ext_vector_type(8)));

struct RowsParams {
    const void* x;          // (rows, K), row_stride elements apart
    const void* w;          // (N, K); gated: gate rows, then N / 2 up rows
    const void* bias;       // (N) or null
    const void* residual;   // (rows, N) or null
    const void* norm;       // (K) weights of the RMSNorm in front, or null
    void* out;              // (rows, N); gated: (rows, N / 2)
    float eps;
    int rows, N, K;
    int64_t x_stride;
    // kCut: tiles of cut_groups groups from tile cut_first on are cut, see cut_of
    int cut_groups, cut_first, cut_span, cut_length;
};

constexpr int kChunk = 64;             // elements of a stage
constexpr int kStageBytes = 2048;      // of 16 rows
constexpr int kMaxRows = 16;
constexpr int kMaxRuns = 1024;

template <typename T>
__device__ inline f32x4 rows_mma(uint4 a, uint4 b, f32x4 c) {
    if constexpr (std::is_same<T, __hip_bfloat16>::value)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(rows_bf16x8, a), __builtin_bit_cast(rows_bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(rows_f16x8, a), __builtin_bit_cast(rows_f16x8, b), c, 0, 0, 0);
}

__host__ __device__ inline int rows_pitch(int K) { return 2 * K + 16; }   // bytes between the rows of x in LDS; the pad spreads the banks

// A library that deals its tiles out over a fixed number of workgroups lays the last ones, which do not come out even, end to end and
// cuts the line of their cut_span stretches into runs of cut_length: a sum whose tile holds the end of a run is two sums, added up.
// Returns how many stretches of `group` lie before that end, 0 for none.  A run is no shorter than a tile, so there is one end at most.
__device__ inline int cut_of(const RowsParams& p, int group) {
    const int tile = group / p.cut_groups - p.cut_first;
    if (tile < 0) return 0;
    const int from = tile * p.cut_span, end = (from + p.cut_length - 1) / p.cut_length * p.cut_length;
    return end < from + p.cut_span ? end - from : 0;
}

// wavefronts of a workgroup, at most: with one part any number, else one per part
template <int kParts>
constexpr int kMostWaves = kParts == 1 ? 8 : kParts;

// RMSNorm of the rows in LDS, in place.  The sum of squares is that of 256 threads of four elements at a time, whatever the workgroup:
// the order (and the bits) of torch's kernel.
template <typename T>
__device__ inline void rows_norm(unsigned char* xs, const unsigned char* weights, float (*part)[4], int waves, const RowsParams& p) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int pieces = p.K / 4, pitch = rows_pitch(p.K);
    struct alignas(8) Piece {
        T v[4];
    };
    for (int j = 0; j < p.rows; j++)
        for (int vw = wave; vw < 4; vw += waves) {
            float s = 0.f;
            for (int i = vw * 64 + lane; i < pieces; i += 256) {
                const Piece a = *reinterpret_cast<const Piece*>(xs + j * pitch + 8 * i);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float v = Elem<T>::to_float(a.v[e]);
                    s = fmaf(v, v, s);
                }
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o);
            if (lane == 0) part[j][vw] = s;
        }
    __syncthreads();
    for (int j = 0; j < p.rows; j++) {
        const float sum = (part[j][0] + part[j][2]) + (part[j][1] + part[j][3]);
        const float r = rsqrtf(sum / (float)p.K + p.eps);
        for (int i = threadIdx.x; i < pieces; i += 64 * waves) {
            Piece* at = reinterpret_cast<Piece*>(xs + j * pitch + 8 * i);
            const Piece a = *at, w = *reinterpret_cast<const Piece*>(weights + 8 * i);
            Piece o;
#pragma unroll
            for (int e = 0; e < 4; e++) o.v[e] = Elem<T>::from_float(Elem<T>::to_float(w.v[e]) * (r * Elem<T>::to_float(a.v[e])));
            *at = o;
        }
    }
    __syncthreads();
}

template <typename T, int kParts, int kUnit, bool kGated, bool kCut, int kStages>
__global__ void __launch_bounds__(64 * kMostWaves<kParts>) rows_kernel(RowsParams p) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ float norm_part[kMaxRows][4];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = kParts > 1 ? kParts : blockDim.x >> 6;
    const int part = wave % kParts;
    const int groups = p.N / 16;
    // Workgroups go round the eight XCDs: each gets a stretch of W of its own, and meets an eighth of its pages.
    const int xcd = blockIdx.x % 8, many = gridDim.x / 8, over = gridDim.x % 8;
    const int block = xcd * many + min(xcd, over) + blockIdx.x / 8;
    int group = kParts > 1 ? block : block * waves + wave;
    const bool live = group < groups;
    if (!live) group = groups - 1;   // reads what another wavefront does and writes nothing
    const int64_t row_bytes = 2 * (int64_t)p.K;
    unsigned char* ring = smem + wave * (kStages * kStageBytes);
    unsigned char* xs = smem + waves * (kStages * kStageBytes);
    const int pitch = rows_pitch(p.K);
    const uint32_t ring_addr = lds_address(ring), xs_addr = lds_address(xs);

    // rows of x, and the norm's weights behind them, go first: 1 KiB a copy, dealt out over the wavefronts
    {
        const int blocks = (p.K + 511) / 512, all = (p.rows + (p.norm ? 1 : 0)) * blocks;
        for (int i = wave; i < all; i += waves) {
            const int j = i / blocks, blk = i - j * blocks;
            const char* src = j < p.rows ? (const char*)p.x + 2 * j * p.x_stride : (const char*)p.norm;
            const int at = blk * 1024 + lane * 16;
            if (at < 2 * p.K) async_copy16(src + blk * 1024, lane * 16, xs_addr + j * pitch + blk * 1024);
        }
    }
    // 64-element stretch i of this part
    auto chunk_of = [&](int i) {
        if constexpr (kParts == 1) return i;
        else return kUnit == 1 ? part + kParts * i : kUnit * (part + kParts * (i / kUnit)) + i % kUnit;
    };
    const int chunks = p.K / kChunk;
    int n = 0;   // stretches of this part
    if constexpr (kParts == 1) n = chunks;
    else {
        const int round = kUnit * kParts, rest = chunks % round - kUnit * part;
        n = chunks / round * kUnit + (rest < 0 ? 0 : rest < kUnit ? rest : kUnit);
    }
    // Lane (r, s) of a copy brings piece s ^ r (^ 1 in the lower half) of row r: an operand read of 16 rows then meets every bank once.
    const int cr = lane >> 3, cs = lane & 7;
    const uint32_t voff0 = cr * (uint32_t)row_bytes + ((cs ^ cr) << 4), voff1 = cr * (uint32_t)row_bytes + ((cs ^ cr ^ 1) << 4);
    const char* rows0 = (const char*)p.w + (int64_t)group * (kGated ? 8 : 16) * row_bytes;
    const char* rows1 = rows0 + (kGated ? (int64_t)(p.N / 2) : 8) * row_bytes;
    auto issue = [&](int chunk, int slot) {
        const int64_t at = (int64_t)chunk * (2 * kChunk);
        async_copy16_once(rows0 + at, voff0, ring_addr + slot * kStageBytes);
        async_copy16_once(rows1 + at, voff1, ring_addr + slot * kStageBytes + 1024);
    };
    // Every wavefront issues the same number of copies here (the row's first stretch again where it has fewer), so that the count
    // below is one number.
#pragma unroll
    for (int i = 0; i < kStages; i++) issue(i < n ? chunk_of(i) : 0, i);
    wait_copies<2 * kStages>();
    __syncthreads();
    if (p.norm) rows_norm<T>(xs, xs + p.rows * pitch, norm_part, waves, p);

    const int r = lane & 15, q = lane >> 4;
    const int flip = (r & 7) ^ (r >> 3);
    const unsigned char* a_at = ring + (r >> 3) * 1024 + (r & 7) * 128;
    const unsigned char* b_at = xs + (r < p.rows ? r : 0) * pitch + q * 16;   // columns that stand for no row repeat the first
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    [[maybe_unused]] f32x4 before = {0.f, 0.f, 0.f, 0.f};   // the sum up to the cut
    const int cut = kCut ? kUnit * cut_of(p, group) : 0;
    auto step = [&](int i, int slot) {
        if constexpr (kCut) {
            if (i == cut) {   // not cut: nothing is in it yet
                before = acc;
                acc = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
        const unsigned char* b = b_at + chunk_of(i) * (2 * kChunk);
        const uint4 a0 = *reinterpret_cast<const uint4*>(a_at + slot * kStageBytes + ((q ^ flip) << 4));
        const uint4 a1 = *reinterpret_cast<const uint4*>(a_at + slot * kStageBytes + (((q + 4) ^ flip) << 4));
        const uint4 b0 = *reinterpret_cast<const uint4*>(b), b1 = *reinterpret_cast<const uint4*>(b + 64);
        acc = rows_mma<T>(a0, b0, acc);
        acc = rows_mma<T>(a1, b1, acc);
    };
    int i = 0, slot = 0;
    for (; i + kStages < n; i++) {
        wait_copies<2 * (kStages - 1)>();
        step(i, slot);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the operands are in registers: their place may be filled again
        issue(chunk_of(i + kStages), slot);
        slot = slot + 1 == kStages ? 0 : slot + 1;
    }
    wait_copies<0>();
    for (; i < n; i++) {
        step(i, slot);
        slot = slot + 1 == kStages ? 0 : slot + 1;
    }

    if constexpr (kParts > 1) {   // the parts in order
        float4* mine = reinterpret_cast<float4*>(ring);
        mine[lane] = make_float4(acc[0], acc[1], acc[2], acc[3]);
        if constexpr (kCut) mine[CKV_WAVE + lane] = make_float4(before[0], before[1], before[2], before[3]);
        __syncthreads();
        if (part != 0) return;
#pragma unroll
        for (int w = 1; w < kParts; w++) {
            const float4* others = reinterpret_cast<const float4*>(ring + w * (kStages * kStageBytes));
            const float4 o = others[lane];
            acc[0] += o.x; acc[1] += o.y; acc[2] += o.z; acc[3] += o.w;
            if constexpr (kCut) {
                const float4 b = others[CKV_WAVE + lane];
                before[0] += b.x; before[1] += b.y; before[2] += b.z; before[3] += b.w;
            }
        }
    }
    if constexpr (kCut) acc += before;
    // lane: row r of x, outputs 4 q + 0..3 of the group
    struct alignas(8) Out {
        T v[4];
    };
    if constexpr (kGated) {
        Out o;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float up = __shfl_xor(acc[e], 32);
            o.v[e] = gated<T>(Elem<T>::from_float(acc[e]), Elem<T>::from_float(up));
        }
        if (live && r < p.rows && q < 2) *reinterpret_cast<Out*>((T*)p.out + (int64_t)r * (p.N / 2) + group * 8 + 4 * q) = o;
    } else {
        if (!live || r >= p.rows) return;
        const int at = group * 16 + 4 * q;
        Out o;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float v = acc[e];
            if (p.bias) v += Elem<T>::to_float(((const T*)p.bias)[at + e]);
            o.v[e] = Elem<T>::from_float(v);
        }
        if (p.residual) {   // rounded before and after it joins, as the two operations are
            const Out res = *reinterpret_cast<const Out*>((const T*)p.residual + (int64_t)r * p.N + at);
#pragma unroll
            for (int e = 0; e < 4; e++) o.v[e] = Elem<T>::from_float(Elem<T>::to_float(res.v[e]) + Elem<T>::to_float(o.v[e]));
        }
        *reinterpret_cast<Out*>((T*)p.out + (int64_t)r * p.N + at) = o;
    }
}

template <typename T, int kParts, int kUnit, bool kGated, bool kCut, int kStages>
int launch_rows(const RowsParams& p, int waves, int lds, hipStream_t stream) {
    auto kernel = rows_kernel<T, kParts, kUnit, kGated, kCut, kStages>;
    if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), lds)) return rc;
    const int groups = p.N / 16, per = waves / kParts;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((groups + per - 1) / per)), dim3(64 * waves), lds, stream, p);
    CKV_HIP_TRY(hipGetLastError());
    return CKV_OK;
}

// A launch lasts as long as the compute unit with the most groups, and a workgroup brings the rows and normalises them for itself: with
// one part a compute unit's even share of the groups is one workgroup of up to eight wavefronts, or a few of the same size (28672 x 4096:
// 448 workgroups of four lay two on most compute units and one on the others; 256 of seven 43.6 -> 39.4 us, in turn with the other products
// of a step 43.1 -> 42.0.  37888 x 3584: 44.8 -> 42.0).  Where one workgroup has a compute unit to itself its rings have twice the
// stages (39.4 -> 38.5, in turn with the others 45 -> 42.0; 10 stages are level).  Two parts: the longer ring where two
// workgroups still fit (6144 x 4096, norm, a row: 11.6 with 12 stages, 11.9 with 8; four rows, one workgroup on a unit or two: 29.8, 18.0).
// Four parts: the shorter ring where the longer does not fit.
template <typename T, int kParts, int kUnit, bool kGated, bool kCut>
int run_rows(const RowsParams& p, hipStream_t stream) {
    DeviceInfo di;
    if (int rc = current_device_info(&di)) return rc;
    constexpr int kLong = kParts == 1 ? 8 : kParts == 2 ? 12 : 6, kShort = kParts == 2 ? 8 : 4;
    const int rest = p.rows * rows_pitch(p.K) + (p.norm ? 2 * p.K : 0);
    auto lds = [&](int waves, int stages) { return waves * stages * kStageBytes + rest; };
    auto fits = [&](int bytes) { return bytes + 256 <= di.lds_max; };
    int waves = kParts;
    bool longer = fits(lds(waves, kLong) * (kParts == 2 ? 2 : 1));
    if constexpr (kParts == 1) {
        constexpr int kMany = 4;   // rounds of workgroups: the last one no longer counts, and four wavefronts are the better workgroup
        const int share = (p.N / 16 + di.cus - 1) / di.cus, most = share > kMany * kMostWaves<1> ? 4 : kMostWaves<1>;
        const int shares = (share + most - 1) / most;
        waves = (share + shares - 1) / shares;
        longer = shares == 1 && fits(lds(waves, kLong));
        while (waves > 1 && !fits(lds(waves, kShort))) waves--;   // long rows
    }
    if (!longer && !fits(lds(waves, kShort))) return CKV_ERR_UNSUPPORTED;
    return longer ? launch_rows<T, kParts, kUnit, kGated, kCut, kLong>(p, waves, lds(waves, kLong), stream)
                  : launch_rows<T, kParts, kUnit, kGated, kCut, kShort>(p, waves, lds(waves, kShort), stream);
}

// Fills in how sums are cut whose tiles are dealt out over `runs` workgroups: as many whole tiles as come out even, less one round, go
// first.  Tiles are of 256 rows and 64 elements, or (four parts) of 32 rows and 256 elements.
inline void cut_into_runs(RowsParams& p, int parts, int runs) {
    p.cut_groups = parts == 1 ? 16 : 2;
    p.cut_span = p.K / (kChunk * parts);
    const int tiles = (p.N / 16 + p.cut_groups - 1) / p.cut_groups, shared = tiles % runs ? tiles % runs + runs : 0;
    p.cut_first = tiles - shared;   // negative: fewer tiles than runs
    p.cut_length = std::max(1, (shared * p.cut_span + runs - 1) / runs);
}

template <typename T>
int run_rows(RowsParams p, bool gated, int parts, int unit, int runs, hipStream_t stream) {
    if (runs) {
        if (gated || unit != 1 || (parts != 1 && parts != 4) || p.K % (kChunk * parts)) return CKV_ERR_UNSUPPORTED;
        cut_into_runs(p, parts, runs);
        if (p.cut_first < 0) return CKV_ERR_UNSUPPORTED;
        return parts == 1 ? run_rows<T, 1, 1, false, true>(p, stream) : run_rows<T, 4, 1, false, true>(p, stream);
    }
    if (parts == 1) return gated ? run_rows<T, 1, 1, true, false>(p, stream) : run_rows<T, 1, 1, false, false>(p, stream);
    if (gated) return CKV_ERR_UNSUPPORTED;
    if (parts == 2 && unit == 2) return run_rows<T, 2, 2, false, false>(p, stream);
    if (parts == 4 && unit == 1) return run_rows<T, 4, 1, false, false>(p, stream);
    if (parts == 4 && unit == 2) return run_rows<T, 4, 2, false, false>(p, stream);
    return CKV_ERR_UNSUPPORTED;
}

}  // namespace
}  // namespace ckv

extern "C" int ckv_linear_rows(const void* x, const void* w, const void* bias, const void* residual, const void* norm, float eps, void* out,
                               int64_t rows, int64_t n, int64_t k, int64_t x_stride, int32_t gated, int32_t parts, int32_t unit, int32_t dtype,
                               void* stream) {
    using namespace ckv;
    if (rows < 0 || n <= 0 || k <= 0 || x_stride < k) return CKV_ERR_SHAPE;
    if (dtype != CKV_F16 && dtype != CKV_BF16) return CKV_ERR_DTYPE;
    if (rows == 0) return CKV_OK;
    if (!x || !w || !out) return CKV_ERR_NULL;
    const int runs = unit >= 256 ? unit >> 8 : 0;
    if (runs > kMaxRuns) return CKV_ERR_UNSUPPORTED;
    if (rows > kMaxRows || n % 16 || k % kChunk || n > 0x7fffffff || k > (1 << 20) || (gated && (bias || residual))) return CKV_ERR_UNSUPPORTED;
    // copies and operands are pieces of 16 bytes, outputs of 8
    if (((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(norm)) & 15) || x_stride % 8 ||
        ((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(residual)) & 7))
        return CKV_ERR_STRIDE;
    RowsParams p;
    p.x = x; p.w = w; p.bias = bias; p.residual = residual; p.norm = norm; p.out = out;
    p.eps = eps;
    p.rows = (int)rows; p.N = (int)n; p.K = (int)k;
    p.x_stride = x_stride;
    p.cut_groups = 1; p.cut_first = 0; p.cut_span = 0; p.cut_length = 1;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (runs) unit &= 255;
    return dtype == CKV_F16 ? run_rows<__half>(p, gated != 0, parts, unit, runs, s) : run_rows<__hip_bfloat16>(p, gated != 0, parts, unit, runs, s);
}
