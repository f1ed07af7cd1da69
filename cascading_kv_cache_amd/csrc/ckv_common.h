// Shared device/host helpers for libckv (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include "../../include/ckv.h"

#define CKV_WAVE 64

#define CKV_HIP_TRY(expr)                          \
    do {                                           \
        hipError_t err__ = (expr);                 \
        if (err__ != hipSuccess) {                 \
            (void)hipGetLastError();               \
            return CKV_ERR_LAUNCH;                 \
        }                                          \
    } while (0)

namespace ckv {

__host__ __device__ inline int64_t elem_bytes(int dtype) { return dtype == CKV_F32 ? 4 : 2; }

// exact widening of one stored score to fp32
__device__ inline float load_as_float(const void* base, int64_t idx, int dtype) {
    if (dtype == CKV_F32) return reinterpret_cast<const float*>(base)[idx];
    const uint16_t h = reinterpret_cast<const uint16_t*>(base)[idx];
    if (dtype == CKV_BF16) return __uint_as_float(static_cast<uint32_t>(h) << 16);
    return __half2float(__ushort_as_half(h));
}

__device__ inline float bf16_bits_to_float(uint16_t h) { return __uint_as_float(static_cast<uint32_t>(h) << 16); }

// round-to-nearest-even fp32 -> bf16 bits (NaN kept quiet)
__device__ inline uint16_t float_to_bf16_bits(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return static_cast<uint16_t>((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return static_cast<uint16_t>(u >> 16);
}

template <typename T>
struct Elem;
template <>
struct Elem<float> {
    static constexpr int code = CKV_F32;
    __device__ static float to_float(float v) { return v; }
    __device__ static float from_float(float v) { return v; }
};
template <>
struct Elem<__hip_bfloat16> {
    static constexpr int code = CKV_BF16;
    __device__ static float to_float(__hip_bfloat16 v) { return __bfloat162float(v); }
    __device__ static __hip_bfloat16 from_float(float v) { return __float2bfloat16(v); }
};
template <>
struct Elem<__half> {
    static constexpr int code = CKV_F16;
    __device__ static float to_float(__half v) { return __half2float(v); }
    __device__ static __half from_float(float v) { return __float2half(v); }
};

// silu(gate) * up, rounded as the two operations are that it stands for
template <typename T>
__device__ inline T gated(T gate, T up) {
    const float x = Elem<T>::to_float(gate), s = Elem<T>::to_float(Elem<T>::from_float(x / (1.f + expf(-x))));
    return Elem<T>::from_float(s * Elem<T>::to_float(up));
}

// stage timing hooks (ckv_profile_enable / ckv_profile_read); no-ops while disabled
void prof_begin(int stage, hipStream_t stream);
void prof_end(int stage, hipStream_t stream);
void prof_empty(int stage);   // counted, of no length
// Timing of a single kernel by events attached to its own dispatch (hipExtLaunchKernelGGL): unlike an
// event record in the stream, this puts nothing between the kernel and its neighbours.  Used when only
// the attention main kernels are timed.
bool prof_kernel_events_wanted(int stage);
void prof_kernel_events(int stage, hipEvent_t* start, hipEvent_t* stop);  // both null unless wanted
struct StageScope {
    int stage;
    hipStream_t stream;
    bool own;
    // kernel_events: the stage is a single kernel whose launch site takes its start / stop events from
    // prof_kernel_events; the scope then records nothing itself when only main kernels are timed
    StageScope(int s, hipStream_t st, bool kernel_events = false)
        : stage(s), stream(st), own(!(kernel_events && prof_kernel_events_wanted(s))) {
        if (own) prof_begin(s, st);
    }
    ~StageScope() {
        if (own) prof_end(stage, stream);
    }
};

// Quotient and remainder of indices, which nearly always fit 32 bits: 64-bit division is a long chain of instructions.
__device__ inline int64_t div_index(int64_t x, int64_t y, int64_t& rem) {
    if ((((uint64_t)x | (uint64_t)y) >> 32) == 0) {
        const uint32_t q = (uint32_t)x / (uint32_t)y;
        rem = (int64_t)((uint32_t)x - q * (uint32_t)y);
        return (int64_t)q;
    }
    rem = x % y;
    return x / y;
}

inline int64_t align_up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }

// Facts about the current device, asked of the runtime once per device and process.
struct DeviceInfo {
    int device;        // ordinal of the current device
    int cus;           // compute units
    int lds_max;       // bytes of LDS one workgroup may use
};
int current_device_info(DeviceInfo* info);  // CKV_OK or CKV_ERR_LAUNCH
// Raises the dynamic LDS limit of `func` on the current device to at least `bytes`; the runtime is asked
// only when the limit this process has already set for (device, func) is smaller.
int ensure_dynamic_lds(const void* func, int bytes);


// sin and cos of an fp32 angle for the 16-bit cache paths: exact range reduction in double (the
// angle is position * frequency, tens of thousands of radians for long contexts), then the hardware
// sin / cos of the remainder, which take revolutions.  Absolute error about 1e-6: three orders below
// the rounding of the rotated values to bf16 / fp16.  The fp32 paths keep sincosf.
__device__ inline void fast_sincos(float x, float* sn, float* cs) {
    const double xd = (double)x;
    const double n = __builtin_rint(xd * 0.15915494309189535);     // x / (2 pi)
    const double r = __builtin_fma(-n, 6.283185307179586, xd);     // |r| <= pi, error ~ n * 2^-52
    const float rev = (float)(r * 0.15915494309189535);
    *sn = __builtin_amdgcn_sinf(rev);
    *cs = __builtin_amdgcn_cosf(rev);
}

// ---------------------------------------------------------------------------------------------
// Rotary embedding on packed 16-bit words with the roundings of the reference's eager path, which evaluates
// x*cos + rotate_half(x)*sin in the tensor dtype (cascade_attention.py:31-35; cos and sin cast to the dtype,
// modeling_llama.py:219-220) and then multiplies queries and keys alike by sqrt(softmax scale)
// (cascade_attention.py:284-291).  w1 holds elements (j, j+1) of a row, w2 their rotation partners (j+64, j+65);
// RopeWord carries the rounded cos / sin of the two pairs in the form the arithmetic consumes.  Every product of
// two 16-bit values and every sum of two 16-bit values is exact in fp32, so each conversion to the tensor dtype
// is one of the reference's roundings: the four products, the two sums, and the products with `post`.
// ---------------------------------------------------------------------------------------------
typedef __bf16 ckv_bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 ckv_f16x2 __attribute__((ext_vector_type(2)));
typedef float ckv_f32x2 __attribute__((ext_vector_type(2)));

template <typename T>
struct RopeWord;
// bfloat16 has no packed arithmetic on this chip, but v_dot2_f32_bf16 multiplies both halves of a word without
// unpacking them: with (c, 0) or (0, c) as the other operand it returns one exact product, with (1, -1) or (1, 1)
// the exact difference or sum of a packed pair.
template <>
struct RopeWord<__hip_bfloat16> {
    static constexpr uint32_t kOneMinusOne = 0xbf803f80u, kOneOne = 0x3f803f80u;  // (1, -1), (1, 1)
    uint32_t c_lo, c_hi, s_lo, s_hi;  // (c0, 0), (0, c1), (s0, 0), (0, s1)
    __device__ static uint32_t pack2(float a, float b) {
        ckv_f32x2 f = {a, b};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, ckv_bf16x2));
    }
    __device__ static float lo(uint32_t w) { return __uint_as_float(w << 16); }
    __device__ static float hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
    __device__ static RopeWord make(float c0, float s0, float c1, float s1) {
        return RopeWord{pack2(c0, 0.f), pack2(0.f, c1), pack2(s0, 0.f), pack2(0.f, s1)};
    }
    __device__ static RopeWord of(uint2 w) {  // w: pack2(c0, c1), pack2(s0, s1)
        return RopeWord{w.x & 0xffffu, w.x & 0xffff0000u, w.y & 0xffffu, w.y & 0xffff0000u};
    }
    __device__ static float dot(uint32_t a, uint32_t b) {
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(ckv_bf16x2, a), __builtin_bit_cast(ckv_bf16x2, b), 0.f, false);
    }
    // scaled == false: the rotation alone
    __device__ void rotate(uint32_t w1, uint32_t w2, float post, bool scaled, uint32_t& o1, uint32_t& o2) const {
        const uint32_t p0 = pack2(dot(w1, c_lo), dot(w2, s_lo)), q0 = pack2(dot(w2, c_lo), dot(w1, s_lo));
        const uint32_t p1 = pack2(dot(w1, c_hi), dot(w2, s_hi)), q1 = pack2(dot(w2, c_hi), dot(w1, s_hi));
        o1 = pack2(dot(p0, kOneMinusOne), dot(p1, kOneMinusOne));
        o2 = pack2(dot(q0, kOneOne), dot(q1, kOneOne));
        if (scaled) {
            o1 = pack2(lo(o1) * post, hi(o1) * post);
            o2 = pack2(lo(o2) * post, hi(o2) * post);
        }
    }
    // Two words, rotated and scaled: the same bits.  The compiler takes the two-operand form of the dot product for the
    // builtin, whose accumulator it has to clear first, and parts each one from its conversion with wait states: of its 40
    // instructions and 8 or so waits a word 12 are such clears.  The three-operand form starts from a literal zero, and two
    // words at a time put three instructions between a dot product and whoever reads it (what the hardware asks for where
    // the reader is another opcode; the block ends on conversions).  A sum is rounded into the upper half of a register,
    // where it is the float that the multiplication takes.  Eight words of one wavefront beside another's: 574 -> 384 ns.
    __device__ static void rotate_scaled2(const RopeWord& x, const RopeWord& y, uint32_t x1, uint32_t x2, uint32_t y1, uint32_t y2,
                                          float post, uint32_t& ox1, uint32_t& ox2, uint32_t& oy1, uint32_t& oy2) {
        float t0, t1, t2, t3, t4, t5, t6, t7, u0, u1, u2, u3, u4, u5, u6, u7;
        asm("v_dot2_f32_bf16 %[t0], %[x1], %[xcl], 0\n\t"
            "v_dot2_f32_bf16 %[t1], %[x2], %[xsl], 0\n\t"
            "v_dot2_f32_bf16 %[t2], %[x2], %[xcl], 0\n\t"
            "v_dot2_f32_bf16 %[t3], %[x1], %[xsl], 0\n\t"
            "v_dot2_f32_bf16 %[t4], %[x1], %[xch], 0\n\t"
            "v_dot2_f32_bf16 %[t5], %[x2], %[xsh], 0\n\t"
            "v_dot2_f32_bf16 %[t6], %[x2], %[xch], 0\n\t"
            "v_dot2_f32_bf16 %[t7], %[x1], %[xsh], 0\n\t"
            "v_cvt_pk_bf16_f32 %[t0], %[t0], %[t1]\n\t"
            "v_dot2_f32_bf16 %[u0], %[y1], %[ycl], 0\n\t"
            "v_dot2_f32_bf16 %[u1], %[y2], %[ysl], 0\n\t"
            "v_cvt_pk_bf16_f32 %[t2], %[t2], %[t3]\n\t"
            "v_dot2_f32_bf16 %[u2], %[y2], %[ycl], 0\n\t"
            "v_dot2_f32_bf16 %[u3], %[y1], %[ysl], 0\n\t"
            "v_cvt_pk_bf16_f32 %[t4], %[t4], %[t5]\n\t"
            "v_dot2_f32_bf16 %[u4], %[y1], %[ych], 0\n\t"
            "v_dot2_f32_bf16 %[u5], %[y2], %[ysh], 0\n\t"
            "v_cvt_pk_bf16_f32 %[t6], %[t6], %[t7]\n\t"
            "v_dot2_f32_bf16 %[u6], %[y2], %[ych], 0\n\t"
            "v_dot2_f32_bf16 %[u7], %[y1], %[ysh], 0\n\t"
            "v_dot2_f32_bf16 %[t0], %[t0], %[om], 0\n\t"
            "v_dot2_f32_bf16 %[t2], %[t2], %[oo], 0\n\t"
            "v_dot2_f32_bf16 %[t4], %[t4], %[om], 0\n\t"
            "v_dot2_f32_bf16 %[t6], %[t6], %[oo], 0\n\t"
            "v_cvt_pk_bf16_f32 %[u0], %[u0], %[u1]\n\t"
            "v_cvt_pk_bf16_f32 %[u2], %[u2], %[u3]\n\t"
            "v_cvt_pk_bf16_f32 %[u4], %[u4], %[u5]\n\t"
            "v_cvt_pk_bf16_f32 %[u6], %[u6], %[u7]\n\t"
            "v_dot2_f32_bf16 %[u0], %[u0], %[om], 0\n\t"
            "v_dot2_f32_bf16 %[u2], %[u2], %[oo], 0\n\t"
            "v_dot2_f32_bf16 %[u4], %[u4], %[om], 0\n\t"
            "v_dot2_f32_bf16 %[u6], %[u6], %[oo], 0\n\t"
            "v_cvt_pk_bf16_f32 %[t0], 0, %[t0]\n\t"
            "v_cvt_pk_bf16_f32 %[t2], 0, %[t2]\n\t"
            "v_cvt_pk_bf16_f32 %[t4], 0, %[t4]\n\t"
            "v_cvt_pk_bf16_f32 %[t6], 0, %[t6]\n\t"
            "v_cvt_pk_bf16_f32 %[u0], 0, %[u0]\n\t"
            "v_cvt_pk_bf16_f32 %[u2], 0, %[u2]\n\t"
            "v_cvt_pk_bf16_f32 %[u4], 0, %[u4]\n\t"
            "v_cvt_pk_bf16_f32 %[u6], 0, %[u6]"
            : [t0] "=&v"(t0), [t1] "=&v"(t1), [t2] "=&v"(t2), [t3] "=&v"(t3), [t4] "=&v"(t4), [t5] "=&v"(t5), [t6] "=&v"(t6),
              [t7] "=&v"(t7), [u0] "=&v"(u0), [u1] "=&v"(u1), [u2] "=&v"(u2), [u3] "=&v"(u3), [u4] "=&v"(u4), [u5] "=&v"(u5),
              [u6] "=&v"(u6), [u7] "=&v"(u7)
            : [x1] "v"(x1), [x2] "v"(x2), [y1] "v"(y1), [y2] "v"(y2), [xcl] "v"(x.c_lo), [xch] "v"(x.c_hi), [xsl] "v"(x.s_lo),
              [xsh] "v"(x.s_hi), [ycl] "v"(y.c_lo), [ych] "v"(y.c_hi), [ysl] "v"(y.s_lo), [ysh] "v"(y.s_hi),
              [om] "s"(kOneMinusOne), [oo] "s"(kOneOne));
        ox1 = pack2(t0 * post, t4 * post);
        ox2 = pack2(t2 * post, t6 * post);
        oy1 = pack2(u0 * post, u4 * post);
        oy2 = pack2(u2 * post, u6 * post);
    }
};
// float16: the packed multiply, subtract and add round each result to float16, which is the reference's arithmetic
template <>
struct RopeWord<__half> {
    uint32_t c, s;  // (c0, c1), (s0, s1)
    __device__ static uint32_t pack2(float a, float b) {
        ckv_f32x2 f = {a, b};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, ckv_f16x2));
    }
    __device__ static float lo(uint32_t w) { return (float)__builtin_bit_cast(ckv_f16x2, w)[0]; }
    __device__ static float hi(uint32_t w) { return (float)__builtin_bit_cast(ckv_f16x2, w)[1]; }
    __device__ static RopeWord make(float c0, float s0, float c1, float s1) { return RopeWord{pack2(c0, c1), pack2(s0, s1)}; }
    __device__ static RopeWord of(uint2 w) { return RopeWord{w.x, w.y}; }  // w: pack2(c0, c1), pack2(s0, s1)
    __device__ void rotate(uint32_t w1, uint32_t w2, float post, bool scaled, uint32_t& o1, uint32_t& o2) const {
#pragma clang fp contract(off)  // a fused multiply-add would skip the rounding of the product
        const ckv_f16x2 x1 = __builtin_bit_cast(ckv_f16x2, w1), x2 = __builtin_bit_cast(ckv_f16x2, w2);
        const ckv_f16x2 cc = __builtin_bit_cast(ckv_f16x2, c), ss = __builtin_bit_cast(ckv_f16x2, s);
        const ckv_f16x2 a1 = x1 * cc, b1 = x2 * ss, a2 = x2 * cc, b2 = x1 * ss;
        const ckv_f16x2 r1 = a1 - b1, r2 = a2 + b2;
        o1 = __builtin_bit_cast(uint32_t, r1);
        o2 = __builtin_bit_cast(uint32_t, r2);
        if (scaled) {
            o1 = pack2(lo(o1) * post, hi(o1) * post);
            o2 = pack2(lo(o2) * post, hi(o2) * post);
        }
    }
    __device__ static void rotate_scaled2(const RopeWord& x, const RopeWord& y, uint32_t x1, uint32_t x2, uint32_t y1, uint32_t y2,
                                          float post, uint32_t& ox1, uint32_t& ox2, uint32_t& oy1, uint32_t& oy2) {
        x.rotate(x1, x2, post, true, ox1, ox2);
        y.rotate(y1, y2, post, true, oy1, oy2);
    }
};

__device__ inline const void* uniform_ptr(const void* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<const void*>(((uint64_t)hi << 32) | lo);
}

// Asynchronous global -> LDS copy of one 16-byte piece per lane (gfx950 global_load_lds_dwordx4):
// the wavefront's 64 pieces land contiguously at LDS byte address `lds_wave_base` (uniform, goes
// to M0), lane i at +16*i; the source is `sbase` (uniform, SGPR pair) + `voff` (per lane).
// Inline assembly on purpose: the compiler keeps no scoreboard entry for the copy, so it cannot
// force it to complete before unrelated LDS reads; completion is awaited explicitly with
// s_waitcnt vmcnt(n) (copies retire in issue order).  M0 is written without being declared: the compiler
// reserves it and loads it itself right before each of its own instructions that read it.
__device__ inline void async_copy16(const void* sbase, uint32_t voff, uint32_t lds_wave_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds_wave_base)), "v"(voff), "s"(uniform_ptr(sbase))
                 : "memory");
}

// One 4-byte piece per lane, lane i at +4*i; lanes that are switched off leave their piece alone.
__device__ inline void async_copy4(const void* sbase, uint32_t voff, uint32_t lds_wave_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds_wave_base)), "v"(voff), "s"(uniform_ptr(sbase))
                 : "memory");
}

// Waits until at most kLeft of this wavefront's copies (and other vector memory operations) are on their way.  Reads of what
// landed may follow at once where the wavefront copied it itself.
template <int kLeft>
__device__ inline void wait_copies() {
    static_assert(kLeft < 64, "vmcnt has six bits");
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(kLeft) : "memory");
}

// The same from an address of the lane's own, for sources more than 4 GiB apart.
__device__ inline void async_copy16_from(const void* src, uint32_t lds_wave_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds_wave_base)), "v"(src)
                 : "memory");
}

// Both again for rows that are read once: non-temporal, so that the stream passes through the L2 without driving out what is
// written beside it.  The results of 0.27 GB of cache rows (9 MB) or of 2.2 GB (69 MB) then leave the L2 in long bursts
// instead of between the reads: streaming decode over 8 x 65601 keys 60.7 -> 56.8 us, over 128 x 32833 keys 430 -> 403;
// caches that would stay in the L2 or the last-level cache from call to call are read as fast as before (8 x 2053 keys 9.3,
// 8 x 8257 17.8 -> 17.4, 8 x 32833 34.3 -> 33.2).
__device__ inline void async_copy16_once(const void* sbase, uint32_t voff, uint32_t lds_wave_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds_wave_base)), "v"(voff), "s"(uniform_ptr(sbase))
                 : "memory");
}
__device__ inline void async_copy16_once_from(const void* src, uint32_t lds_wave_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds_wave_base)), "v"(src)
                 : "memory");
}

__device__ inline uint32_t lds_address(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

}  // namespace ckv
