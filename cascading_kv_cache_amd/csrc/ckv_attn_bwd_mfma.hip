// Backward of the dense-input attention operator on the matrix cores (cascade/models/flash_attention.py:279-537):
// bf16 / fp16, head_dim 64 or 128 (template parameter kHD), v_mfma_f32_32x32x16.  Two kernels, as in the reference (_attn_bwd_dq, _attn_bwd_dkdv),
// so that no gradient is accumulated with atomics; both recompute the probabilities from the row normalisers of
// the forward pass and take delta[m] = sum_d out[m, d] dout[m, d] from the caller.
//
//   dq     a wavefront owns 32 query rows, a workgroup 128; 32-key blocks of K and V stream through LDS.
//          S^T = K Q^T and dP^T = V dO^T keep a query in one lane (its normaliser and delta are one value per
//          lane), dS^T = P^T (dP^T - delta) scale is, packed, directly the B operand of dQ^T += K^T dS^T.
//   dkdv   a wavefront owns 32 keys, a workgroup 128; 32-row blocks of Q and dO stream through LDS.
//          S = Q K^T and dP = dO V^T keep a key in one lane; P and dS are the B operands of
//          dV^T += dO^T P and dK^T += Q^T dS.
//
// Precision.  With 128 dims P and dS enter those products rounded to the tensor dtype.  With 64 dims nothing but the operands
// is held in 16 bits: P and dS enter as three bfloat16 terms that add up to the float32 value, one matrix instruction each
// (Weights).  A float16 operand of such a product is two bfloat16 numbers (Halves), so that it takes six.  Float16 terms would
// need three, but resolve 2^-24 of a value that has to be scaled into their range: a dS 2^-25 times its row's largest would keep
// half of its bits, and where that row's largest meet zeros in a dim of K or Q the sum is what was lost.  Blocks that no terms
// hold (infinite dS or gradients) take v_mfma_f32_32x32x2 on the values themselves.  That instruction for every block never runs
// beside a vector instruction: 8 heads x 1000 rows x 5095 keys in float16 dq 55 and dk/dv 91 us, six products 45 and 74 (three
// float16 ones 35 and 49; the vector kernels 2520 and 1838).  Against float64 over 50 random shapes dq, dk and dv are 2.0956e-4,
// 2.0816e-4 and 2.0747e-4 off (relative), which is the rounding of the result; float32 products 2.0956e-4, 2.0816e-4, 2.0747e-4.
// Before that rounding dq is 2.99e-7 off (8 shapes), bfloat16 3.11e-7; with float32 products 3.69e-7 and 3.61e-7.
//
// What bounds them (64 heads x 1024 rows x 8704 visible keys, 128 dims, bf16: dq 386 us, dk/dv 590).  Vector work
// beside the matrix work: both take most of a block's time and overlap only where a wavefront alternates them, so an
// element costs one fused multiply-add, one exponential, one multiplication and half a conversion per product (no
// subtraction of delta, no scale, no mask in a block that every row sees, no addresses), where it was twice that.  The
// copies: 100 to 170 cycles each at the issue, whatever else the wavefront does (let out one by one between matrix
// instructions: dq 514 us, dk/dv level); dq has them 64 keys ahead.  Waiting for them where the work does not need them yet: the
// compiler put a wait for everything in flight before the first use of registers loaded in front of the loop (arrived; without
// it dq 436 us, with it 401, by eight wavefronts 389, with everything a workgroup starts from requested at once 386).  Reads from LDS are not it: operands of dK / dV 4 instead of 2 matrix
// instructions ahead, and of dP 2 instead of 1, dk/dv level; dk/dv by eight wavefronts and 64 rows a barrier 628 us instead of 590.
//
// The A operands K^T, Q^T and dO^T are read from the row-major tiles in LDS with the transposing read
// ds_read_b64_tr_b16: lane i of a 16-lane group receives element [4e + i/4][i%4] (e = 0..3) of the 16 x 4 matrix
// whose row r is the 8 bytes lane r points at; with lane r pointing at dims 4 (r%4) .. +3 of row r/4 of a
// 4-row group, lane i receives dim i of the four rows.  The 16-byte piece c of row r sits in slot c ^ f(r) of its row
// (swz), with f chosen so that both the 16-byte row reads (32 rows, one piece) and the transposing reads (4 rows x 64
// bytes) stay off each other's banks.
//
// Masked keys: the caller sorts the keys, the visible ones first (launch_dense_prologue), and both kernels take key
// block i from the rows key_order names, so a masked key costs no work at all; the dk/dv kernel writes its zeros.
// Without an order (a caller whose workspace has no room for it) the keys are taken as they lie and masked one by one.
#include "ckv_attn_internal.h"

#include <type_traits>

namespace ckv {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));

constexpr int kBlk = 32;              // rows of a streamed block
constexpr int kWaves = 4;             // wavefronts of a workgroup, 32 stationary rows each
constexpr int kThreads = kWaves * CKV_WAVE;
constexpr int kOwn = kWaves * 32;     // stationary rows of a workgroup
constexpr int kAhead = 3, kKvAhead = 3;  // matrix instructions between an operand's read from LDS and its use
// Workgroups of the dq kernel: four wavefronts with a block of keys per barrier, two workgroups on a compute unit, or eight with
// two blocks, one workgroup (wide_dq).  Either way a wavefront copies as much per barrier, 64 keys ahead of their use.
template <int kDqWaves>
struct Team {
    static constexpr int kThreads = kDqWaves * CKV_WAVE, kOwn = kDqWaves * 32, kPerCu = 8 / kDqWaves;
    static constexpr int kSub = kDqWaves / 4, kRows = kSub * kBlk, kStages = kSub == 1 ? 3 : 2;   // blocks and keys of a stage, stages
};
constexpr float kLog2e = 1.4426950408889634f;
// kSplit: the A operands of the products that P and dS enter come from two bfloat16 tiles beside the tile itself, see Halves
template <int kHD, bool kSplit = false>
struct Geo {
    static constexpr int kRowBytes = kHD * 2;
    static constexpr int kTile = kBlk * kRowBytes;  // 8 KiB with 128 dims
    static constexpr int kPieces = kHD / 8;         // 16-byte pieces of a row
    // dynamic LDS of the dk/dv kernel: two stages of (Q, dO) tiles, with kSplit their halves, the per-row scalars of both
    // stages, V^T operands
    static constexpr int kDkdvHalves = 2 * 2 * kTile;
    static constexpr int kDkdvRowv = kDkdvHalves + (kSplit ? 2 * 2 * 2 * kTile : 0);
    static constexpr int kDkdvOdd = kDkdvRowv + 2 * 2 * kBlk * (int)sizeof(float);   // 64 dims: a word per stage
    static constexpr int kDkdvV = kDkdvOdd + (kHD == 64 ? 16 : 0);
    static constexpr int kParked = kHD == 128 ? 3 : 0;   // K^T operands that are kept there too: 12 registers that would spill
    static constexpr int kDkdvLds = kDkdvV + kWaves * (kHD / 16 + kParked) * CKV_WAVE * 16;
};

template <typename T>
struct Mma;
template <>
struct Mma<__hip_bfloat16> {
    __device__ static f32x16 mma(uint4 a, uint4 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
    }
    __device__ static uint32_t pack2(float lo, float hi) {
        f32x2 f = {lo, hi};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
    }
    // the two elements of a packed pair as floats
    __device__ static float lo_f(uint32_t w) { return __uint_as_float(w << 16); }
    __device__ static float hi_f(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
    // x less an element of a packed pair, exact where the element is x rounded
    __device__ static float less_lo(float x, uint32_t w) { return x - lo_f(w); }
    __device__ static float less_hi(float x, uint32_t w) { return x - hi_f(w); }
};
template <>
struct Mma<__half> {
    __device__ static f32x16 mma(uint4 a, uint4 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                      0, 0);
    }
    __device__ static uint32_t pack2(float lo, float hi) {
        f32x2 f = {lo, hi};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2));
    }
    __device__ static float lo_f(uint32_t w) { return (float)__builtin_bit_cast(f16x2, w)[0]; }
    __device__ static float hi_f(uint32_t w) { return (float)__builtin_bit_cast(f16x2, w)[1]; }
};

struct BwdMfmaParams {
    ckv_dense_bwd_args a;
    const float* delta;  // (B, H, n_ctx)
    const int* key_order;  // null: keys as they lie
    const int* n_visible;
    float* part_dq;      // dq in shares of the keys, see dq_splits; null with one share
    int n_split;
    int dq_per_head, dkdv_per_head;        // workgroups of a (batch, head)
    int dq_by_xcd, dkdv_by_xcd;            // see unit_of
    int dkdv_blocks;     // of a launch of both: the workgroups behind them do dq
};

// Workgroup ids go round the 8 XCDs, each with an L2 of its own.  With 8 | B * H all workgroups of a head can run on one
// XCD, so that the rows they all stream (K and V for dq, Q and dO for dk / dv) are fetched into one L2 instead of eight.
// dq always does (64 heads x 1024 rows x 8704 visible keys x 128: 555 -> 529 us); dk / dv only while the launch is one round
// of workgroups (8 heads x 5095 keys x 64: 45.5 -> 39 us; 64 heads x 17408 keys, seventeen rounds: 760 -> 988 us, all compute
// units of an XCD on the same few rows).
struct Unit {
    int x;          // workgroup of the head
    int64_t bh;
};
__device__ inline Unit unit_of(int id, int per_head, bool by_xcd) {   // id: workgroup of the tensor
    const int j = by_xcd ? id >> 3 : id;
    return Unit{j % per_head, by_xcd ? (int64_t)(id & 7) + 8 * (j / per_head) : (int64_t)(j / per_head)};
}

// 128 dims: a row is all 64 banks, so 16 consecutive rows need 16 different slots for one piece, and the four rows of a
// transposing read different 64-byte quarters.  64 dims: two rows share the banks, eight slots each, and rows r, r + 2 of
// a transposing read need different halves.
template <int kHD>
__device__ inline int swz(int row, int piece) {
    if constexpr (kHD == 128) return piece ^ (((row & 3) << 2) | ((row >> 2) & 3));
    else return piece ^ ((((row >> 1) & 1) << 2) | ((row >> 2) & 3));
}

// The keys of a launch: `n` of them can be seen (cached ones first), position i is row row_of(i) of K and V.
struct Keys {
    const int* order;
    const uint8_t* mask;
    int64_t n_cached;   // cached keys in front of the chunk keys
    int64_t n_seen;     // positions below it hold keys some query may see
    int64_t n_kv;
    __device__ Keys(const BwdMfmaParams& p) {
        const int64_t nc = p.a.n_kv - p.a.n_ctx;
        order = p.key_order;
        mask = p.a.mask;
        n_cached = order ? *p.n_visible : nc;
        n_seen = n_cached + p.a.n_ctx;
        n_kv = p.a.n_kv;
    }
    __device__ int64_t row_of(int64_t i) const { return order ? order[i] : i; }
    __device__ bool visible(int64_t i) const { return i < n_seen && (order || i >= n_cached || mask[i] == 0); }
};

// A block of a (rows, kHD) tensor, eight rows a wavefront, into a tile, global -> LDS without registers, 1 KiB per instruction; a
// wavefront copies kRowBytes / 128 of them, lane i of copy j one slot of row block_row(wave, lane, j).  Rows past row `last`
// of the block repeat it (finite values; whatever is computed from them is masked).  The caller waits with vmcnt(0)
// before the barrier that publishes the tile.
template <int kHD>
__device__ inline int block_row(int wave, int lane, int j) {
    constexpr int kPer = CKV_WAVE / Geo<kHD>::kPieces;   // rows per instruction
    return kPer * (kHD / 64 * wave + j) + lane / Geo<kHD>::kPieces;
}
template <int kHD>
__device__ inline void copy_block(const char* blk, uint32_t row_bytes, int last, uint32_t tile_lds, int wave, int lane) {
#pragma unroll
    for (int j = 0; j < kHD / 64; j++) {
        const int row = block_row<kHD>(wave, lane, j), rr = row < last ? row : last;
        const uint32_t voff = (uint32_t)rr * row_bytes + (uint32_t)(swz<kHD>(row, lane % Geo<kHD>::kPieces) << 4);
        async_copy16(blk, voff, tile_lds + (uint32_t)((kHD / 64 * wave + j) * 1024));
    }
}
// The same for rows given by number (one per copy of this lane).  kWide: the rows of a head span 4 GiB or more.
template <int kHD, bool kWide>
__device__ inline void copy_rows(const char* base, uint32_t row_bytes, const uint32_t (&rows)[kHD / 64], uint32_t tile_lds, int wave,
                                 int lane) {
#pragma unroll
    for (int j = 0; j < kHD / 64; j++) {
        const uint32_t piece = (uint32_t)(swz<kHD>(block_row<kHD>(wave, lane, j), lane % Geo<kHD>::kPieces) << 4);
        const uint32_t to = tile_lds + (uint32_t)((kHD / 64 * wave + j) * 1024);
        if constexpr (kWide) async_copy16_from(base + (uint64_t)rows[j] * row_bytes + piece, to);
        else async_copy16(base, rows[j] * row_bytes + piece, to);
    }
}

// Where a lane's operands lie inside a tile; the tile itself is a constant offset of the instruction, so that a read costs no
// address arithmetic (an addition per read was a seventh of the vector work of a block).
//   row[ds]    A operand of a product that contracts over the head dims: row lane%32, dims 16 ds + 8 (lane/32) .. +7
//   col[db][a] A operand of a product that contracts over the rows of the tile: dim 32 db + lane%32 of rows
//              16 s + 8 a + 4 (lane/32) + e (elements 4 a + e), the order in which the packed B operand holds them;
//              blocks of 32 dims flip bits 2-3 of the slot, step s is 16 rows further
// kTight: registers are kept for 64 dims of columns only, those of the other 64 are worked out at the read.
template <int kHD, bool kTight>
struct Operands {
    static constexpr int kCols = kTight && kHD == 128 ? 2 : kHD / 32;
    uint32_t row[kHD / 16], col[kCols][2];
    __device__ Operands(uint32_t lds0, int lane) {
        const int r = lane & 31, h = lane >> 5, g16 = (lane >> 4) & 1, rl = lane & 15;
#pragma unroll
        for (int ds = 0; ds < kHD / 16; ds++) row[ds] = lds0 + (uint32_t)(r * Geo<kHD>::kRowBytes + swz<kHD>(r, 2 * ds + h) * 16);
#pragma unroll
        for (int a = 0; a < 2; a++) {
            const int cr = 8 * a + 4 * h + (rl >> 2);              // + 16 s
            const int piece = 2 * g16 + ((rl & 3) >> 1);           // + 4 db
            const uint32_t base = (uint32_t)(cr * Geo<kHD>::kRowBytes + swz<kHD>(cr, piece) * 16 + 8 * (rl & 1));
#pragma unroll
            for (int db = 0; db < kCols; db++) col[db][a] = lds0 + (base ^ (uint32_t)(db << 6));
        }
#pragma unroll
        for (int ds = 0; ds < kHD / 16; ds++) asm("" : "+v"(row[ds]));   // kept, not worked out again at every read
#pragma unroll
        for (int db = 0; db < kCols; db++) asm("" : "+v"(col[db][0]), "+v"(col[db][1]));
    }
    __device__ uint4 row_op(uint32_t tile, int ds) const { const u32x4 v = *(const __attribute__((address_space(3))) u32x4*)(uintptr_t)(row[ds] + tile);
        return make_uint4(v[0], v[1], v[2], v[3]); }
    __device__ uint4 col_op(uint32_t tile, int s, int db) const {
        uint2 u[2];
#pragma unroll
        for (int a = 0; a < 2; a++) {
            uint32_t at = col[db % kCols][a];
            if (db >= kCols) asm volatile("v_xor_b32 %0, 0x80, %1" : "=v"(at) : "v"(at));   // volatile: not kept in a register
            u[a] = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(uintptr_t)(
                                                 at + tile + (uint32_t)(s * 16 * Geo<kHD>::kRowBytes))));
        }
        return make_uint4(u[0].x, u[0].y, u[1].x, u[1].y);
    }
};

// The loads of these registers end here.  The compiler does not see what wait_copies waits for: to it a load in front of a loop
// may be in flight in every turn, and it waits at the first use there, for the copies issued since as well.
template <int kN>
__device__ inline void arrived(uint4 (&regs)[kN]) {
#pragma unroll
    for (int i = 0; i < kN; i++) asm volatile("" : "+v"(regs[i].x), "+v"(regs[i].y), "+v"(regs[i].z), "+v"(regs[i].w));
}

__device__ inline f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; i++) z[i] = 0.f;
    return z;
}

template <typename T>
__device__ inline uint4 pack8(const f32x16& v, int s) {
    return make_uint4(Mma<T>::pack2(v[8 * s + 0], v[8 * s + 1]), Mma<T>::pack2(v[8 * s + 2], v[8 * s + 3]),
                      Mma<T>::pack2(v[8 * s + 4], v[8 * s + 5]), Mma<T>::pack2(v[8 * s + 6], v[8 * s + 7]));
}

// The B operand of the two products that contract over a block's 32 rows, element 8 s + i of `v` belonging to step s, and the
// product of a step with the A operand of Operands::col_op.  Element 4 a + e of that holds rows 16 s + 8 a + 4 (lane/32) + e,
// the row of accumulator register 8 s + 4 a + e in the same lane half.  `accumulate` is product k, step k / kDB into
// accumulator k % kDB with A operand `op`.  128 dims: packed in the tensor dtype; 64 dims: three bfloat16 terms that add up
// to the float32 value (24 bits in three times 8, and bfloat16 has float32's range), one matrix instruction each.
template <typename T, int kHD>
struct Weights {
    static constexpr int kDB = kHD / 32, kTerms = kHD == 64 ? 3 : 1;
    typedef typename std::conditional<kHD == 64, __hip_bfloat16, T>::type Term;
    typedef Mma<Term> M;
    uint4 w[kTerms][2];
    __device__ void set(const f32x16& v, int s) {
        w[0][s] = pack8<Term>(v, s);
        if constexpr (kTerms == 3) {
            f32x16 rest = v;
#pragma unroll
            for (int t = 1; t < 3; t++) {
                const uint32_t p[4] = {w[t - 1][s].x, w[t - 1][s].y, w[t - 1][s].z, w[t - 1][s].w};
#pragma unroll
                for (int i = 0; i < 8; i++) rest[8 * s + i] -= i & 1 ? M::hi_f(p[i >> 1]) : M::lo_f(p[i >> 1]);   // exact
                w[t][s] = pack8<Term>(rest, s);
            }
        }
    }
    __device__ void accumulate(const uint4& op, int k, f32x16 (&c)[kDB]) const {
#pragma unroll
        for (int t = 0; t < kTerms; t++) c[k % kDB] = M::mma(op, w[t][k / kDB], c[k % kDB]);
    }
};

// Float16 operands of those products with 64 dims: a float16 number is the sum of two bfloat16 ones, itself rounded to 8 bits
// and the rest, which has three (infinity: the rest is NaN, but a product of P or dS with an infinite row of K or Q is NaN in
// any arithmetic, and blocks with an infinite row of dO take float32 products).  Every wavefront splits the rows that it copied
// itself, its lanes the 16 bytes that they copied, into two tiles laid out like the first (`split`: kTiles of them from byte
// `tile` on, two each from byte `halves` on).
template <typename T, int kHD>
struct Halves {
    static constexpr bool kSplit = kHD == 64 && std::is_same<T, __half>::value;
    static constexpr int kOps = kSplit ? 2 : 1;   // A operands of a product
    // Product k with all of its operands.  Of a split one the instructions are added up from zero in `block`, which joins the
    // accumulator when the block is done: one rounding of the large sum per block instead of twelve (dq before it is rounded
    // 2.99e-7 off instead of 3.49e-7, for 1.5 us of 74 in dk/dv and none in dq).
    __device__ static void accumulate(const Weights<T, kHD>& w, const uint4 (&ops)[kOps][kHD / 16], int k, f32x16 (&c)[kHD / 32], f32x16 (&block)[kHD / 32]) {
        constexpr int kDB = kHD / 32;
        if constexpr (kSplit) {
            if (k < kDB) block[k] = zero16();
#pragma unroll
            for (int o = 0; o < kOps; o++) w.accumulate(ops[o][k], k, block);
            if (k > kDB) join(k - kDB - 1, c, block);   // a product behind its last instruction
        } else {
            w.accumulate(ops[0][k], k, c);
        }
    }
    // the last accumulator's, once there is other work to do behind its last instruction
    __device__ static void finish(f32x16 (&c)[kHD / 32], const f32x16 (&block)[kHD / 32]) {
        if constexpr (kSplit) join(kHD / 32 - 1, c, block);
    }
    __device__ static void join(int db, f32x16 (&c)[kHD / 32], const f32x16 (&block)[kHD / 32]) {
#pragma unroll
        for (int i = 0; i < 16; i++) c[db][i] += block[db][i];
    }
    template <int kTiles, int kTile>
    __device__ static void split(unsigned char* lds, uint32_t tile, uint32_t halves, int wave, int lane) {
        if constexpr (kSplit) {
            const uint32_t at = (uint32_t)(wave * 1024 + lane * 16);
#pragma unroll
            for (int i = 0; i < kTiles; i++) {
                const uint4 v = *reinterpret_cast<const uint4*>(lds + tile + (uint32_t)(i * kTile) + at);
                const uint32_t in[4] = {v.x, v.y, v.z, v.w};
                uint32_t hi[4], lo[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    typedef Mma<__hip_bfloat16> M;
                    const float x0 = Mma<__half>::lo_f(in[j]), x1 = Mma<__half>::hi_f(in[j]);
                    hi[j] = M::pack2(x0, x1);
                    lo[j] = M::pack2(x0 - M::lo_f(hi[j]), x1 - M::hi_f(hi[j]));   // exact
                }
                unsigned char* to = lds + halves + (uint32_t)(2 * i * kTile) + at;
                *reinterpret_cast<uint4*>(to) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
                *reinterpret_cast<uint4*>(to + kTile) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
            }
        }
    }
};

// The same product with the float32 values themselves, all of it (64 dims): v_mfma_f32_32x32x2, whose B operand is an
// accumulator register as it stands and whose A operand is the same transposed read, widened.  For what the terms cannot
// hold: infinity less its first term is NaN.
template <typename T>
__device__ inline void accumulate_f32(const uint4 (&ops)[4], const f32x16& v, f32x16 (&c)[2]) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
        float a[2][8];
#pragma unroll
        for (int db = 0; db < 2; db++) {
            const uint4& o = ops[2 * s + db];
            const uint32_t p[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
            for (int i = 0; i < 8; i++) a[db][i] = i & 1 ? Mma<T>::hi_f(p[i >> 1]) : Mma<T>::lo_f(p[i >> 1]);
        }
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int db = 0; db < 2; db++) c[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[db][i], v[8 * s + i], c[db], 0, 0, 0);
    }
}

// 64 dims: some dS of the wavefront's block is infinite or so large that its terms could be
__device__ inline bool beyond_terms(const f32x16& ds) {
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) m = fmaxf(m, fabsf(ds[i]));
    return __ballot(m > 0x1p120f) != 0ull;
}

// bits [0, n) set, for 0 <= n <= 32
__device__ inline uint32_t low_bits(int n) { return n >= 32 ? 0xffffffffu : ((1u << n) - 1u); }

// dk: the softmax scale multiplies dS, so that float16 dS stays in range, or the finished sum, which leaves a multiplication per
// element out.  With 128 dims dS is rounded before the scale then instead of behind it, one rounding of 8 bits either way: dk in
// bfloat16 2.351e-3 off float64 (relative, 16 random shapes), 2.361e-3 with the scale on every dS.
template <typename T, int kHD>
constexpr bool kScaleInside = kHD == 128 && std::is_same<T, __half>::value;

// v if bit `bit` of `word` is set, else +0: a sign-extended one-bit field and a bitwise and
__device__ inline float keep_if_bit(float v, uint32_t word, int bit) {
    const int32_t m = __builtin_amdgcn_sbfe((int32_t)word, bit, 1);
    return __uint_as_float(__float_as_uint(v) & (uint32_t)m);
}

// ---------------------------------------------------------------------------------------------
// dq
// ---------------------------------------------------------------------------------------------
template <typename T, int kHD, bool kWide, int kWaves>
__device__ __forceinline__ void dq_workgroup(const BwdMfmaParams& p, const Unit& unit, unsigned char* const smem) {   // dq_lds of it
    constexpr int kOwn = Team<kWaves>::kOwn, kSub = Team<kWaves>::kSub, kRows = Team<kWaves>::kRows, kDqStages = Team<kWaves>::kStages;
    constexpr int kBlkBytes = Geo<kHD>::kTile, kTile = kSub * kBlkBytes, kStage = 2 * kTile;   // K, V
    constexpr int kCopies = 2 * (kHD / 64);                      // of a wavefront and stage
    constexpr int kMine = kRows / kWaves;                        // rows of a stage that a wavefront copies
    typedef Halves<T, kHD> Half;                                 // of K: two tiles per stage
    constexpr uint32_t kHalves = kDqStages * kStage, kRowNumbers = kHalves + (Half::kSplit ? kDqStages * 2 * kTile : 0);
    const ckv_dense_bwd_args& a = p.a;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / CKV_WAVE), lane = tid % CKV_WAVE, h = lane >> 5;
    const Keys keys(p);
    const int64_t n_ctx = a.n_ctx;
    const int n_cached = (int)keys.n_cached, n_seen = (int)keys.n_seen;   // below 2^31, see bwd_mfma_supported
    const int64_t bh = unit.bh, b = bh / a.H, hd = bh % a.H;
    const int share = unit.x % p.n_split;
    const int m_wg = unit.x / p.n_split * kOwn;
    const int m_lane = m_wg + wave * 32 + (lane & 31);  // this lane's query
    const char* kb = reinterpret_cast<const char*>(a.k) + (b * a.kv_stride[0] + hd * a.kv_stride[1]) * 2;
    const char* vb = reinterpret_cast<const char*>(a.v) + (b * a.kv_stride[0] + hd * a.kv_stride[1]) * 2;
    const uint32_t row_bytes = (uint32_t)(a.kv_stride[2] * 2);

    const uint32_t lds0 = lds_address(smem);
    const Operands<kHD, false> op(lds0, lane);

    // keys past the diagonal of the workgroup's last row are visible to none of its rows
    int m_last = m_wg + kOwn - 1;
    if (m_last > (int)n_ctx - 1) m_last = (int)n_ctx - 1;
    const int nblk_all = (int)(((int64_t)n_cached + m_last + kRows) / kRows);   // stages of them
    // this workgroup's share of them: an equal stretch (an empty one leaves zeros)
    const int per_share = (nblk_all + p.n_split - 1) / p.n_split;
    const int blk0 = share * per_share, nblk = blk0 + per_share < nblk_all ? blk0 + per_share : nblk_all;

    // Stages are copied 64 rows ahead.  With an order the row numbers of a wavefront's eight rows of a stage
    // come to LDS the same way, one stage earlier, so that no load in the loop is one whose result the compiler would
    // wait for together with the copies behind it.
    const uint32_t mine = lds0 + kRowNumbers + (uint32_t)(wave * kMine * (int)sizeof(int));
    constexpr uint32_t kSlot = kRows * sizeof(int);
    const int mine_lane = kHD == 128 ? lane / 16 : lane / 8;   // of copy 0; copy j takes row 4 j + this one
    auto clamped = [&](int i) { return i < n_seen ? i : n_seen - 1; };   // a chunk key: finite values, and no query looks at this copy
    auto request_rows = [&](int blk, int slot) {
        if (keys.order && lane < kMine)
            async_copy4(keys.order, (uint32_t)clamped(blk * kRows + wave * kMine + lane) * 4u, mine + (uint32_t)slot * kSlot);
    };
    auto rows_of = [&](int blk, int slot, uint32_t(&r)[kHD / 64]) {
#pragma unroll
        for (int j = 0; j < kHD / 64; j++)
            r[j] = keys.order ? *(const __attribute__((address_space(3))) uint32_t*)(uintptr_t)(mine + (uint32_t)slot * kSlot + (uint32_t)(4 * j + mine_lane) * 4u)
                              : (uint32_t)clamped(blk * kRows + wave * kMine + 4 * j + mine_lane);
    };
    auto copy = [&](const uint32_t(&r)[kHD / 64], int st) {
        copy_rows<kHD, kWide>(kb, row_bytes, r, lds0 + (uint32_t)(st * kStage), wave, lane);
        copy_rows<kHD, kWide>(vb, row_bytes, r, lds0 + (uint32_t)(st * kStage + kTile), wave, lane);
    };
    uint32_t rows_next[kHD / 64];   // of the block that is copied next
    // All that does not hang on the row numbers is requested with them, in one go: as loads of one operand at a time, each behind
    // the last one's, these were four (64 dims) or eight (128) trips to memory in a row and two more for the scalars (64 heads x 1024 rows x
    // 8704 visible keys, 128 dims: 389 -> 386 us; the same for dk/dv, whose workgroups come in rounds, level).
    if (blk0 < nblk) {
#pragma unroll
        for (int i = 0; i < kDqStages; i++) request_rows(blk0 + i, i);
    }
    // stationary B operands: Q^T and dO^T of this lane's query, dims 16 ds + 8 h .. +7
    uint4 qreg[kHD / 16], greg[kHD / 16];
    const bool row_ok = m_lane < n_ctx;
    float lse = 0.f, delta = 0.f;
#pragma unroll
    for (int ds = 0; ds < kHD / 16; ds++) qreg[ds] = greg[ds] = make_uint4(0u, 0u, 0u, 0u);
    if (row_ok) {
        const char* qrow = reinterpret_cast<const char*>(a.q) +
                           (b * a.q_stride[0] + hd * a.q_stride[1] + m_lane * a.q_stride[2]) * 2;
        const char* grow = reinterpret_cast<const char*>(a.dout) +
                           (b * a.dout_stride[0] + hd * a.dout_stride[1] + m_lane * a.dout_stride[2]) * 2;
#pragma unroll
        for (int ds = 0; ds < kHD / 16; ds++) {
            qreg[ds] = *reinterpret_cast<const uint4*>(qrow + (16 * ds + 8 * h) * 2);
            greg[ds] = *reinterpret_cast<const uint4*>(grow + (16 * ds + 8 * h) * 2);
        }
        lse = a.lse[bh * n_ctx + m_lane];
        delta = p.delta[bh * n_ctx + m_lane];
    }
    arrived(qreg);
    arrived(greg);
    // The magnitude of the softmax scale rides on the exponent (nothing here needs P without it), its sign on the result;
    // the products of V and dO start from -delta.  That leaves one multiplication per element beside the exponential.
    float nl = row_ok ? fmaf(-lse, kLog2e, __builtin_amdgcn_logf(fabsf(a.scale))) : 0.f;
    const float c2 = a.scale * kLog2e;
    f32x16 neg_delta;
    {
        const float d = -delta;
#pragma unroll
        for (int i = 0; i < 16; i++) neg_delta[i] = d;
        asm volatile("" : "+v"(neg_delta));   // 16 registers to start from, not 16 moves a block
    }
    f32x16 dq[kHD / 32];
#pragma unroll
    for (int db = 0; db < kHD / 32; db++) dq[db] = zero16();
    if (blk0 < nblk) {
        wait_copies<0>();
        rows_of(blk0, 0, rows_next);
        copy(rows_next, 0);
        if constexpr (kDqStages == 3) {
            rows_of(blk0 + 1, 1, rows_next);
            if (blk0 + 1 < nblk) copy(rows_next, 1);
        }
        rows_of(blk0 + kDqStages - 1, kDqStages - 1, rows_next);
        if (kDqStages == 3 && blk0 + 1 < nblk) wait_copies<kCopies>();
        else wait_copies<0>();
        Half::template split<1, kTile>(smem, 0, kHalves, wave, lane);
    }
    __syncthreads();
    // 32 keys from position n0 on, whose tiles begin at byte kt of the stages (K) and vt (V)
    auto block = [&](auto tile_tag, auto halves_tag, int n0) {
        constexpr uint32_t kt = decltype(tile_tag)::value, vt = kt + kTile;
        // Which keys of the block any query may see: all of them in front of the chunk when they were sorted.
        uint32_t vis = 0xffffffffu;
        if (!keys.order) vis = (uint32_t)__ballot(keys.visible(n0 + (lane & 31)));
        __builtin_amdgcn_sched_barrier(0);
        // keys of this block that are chunk keys past this wavefront's last row: nothing to do for it
        const bool dead = vis == 0u || (n0 >= n_cached && n0 - n_cached > m_wg + wave * 32 + 31);
        // Written in issue order: an operand is read from LDS kAhead matrix instructions before the one that takes it, the
        // exponentials run beside the products of V and dO, the second half of dS beside the products of the first.
        constexpr int kRow = kHD / 16, kDB = kHD / 32;
        if (!dead) {
            f32x16 s = zero16(), dp = neg_delta;
            constexpr uint32_t ct = Half::kSplit ? decltype(halves_tag)::value : kt;
            uint4 ops[2 * kRow], cops[Half::kOps][2 * kDB];
            auto row_op = [&](int k) { return op.row_op(k < kRow ? kt : vt, k % kRow); };
            auto col_op = [&](int k) {
#pragma unroll
                for (int o = 0; o < Half::kOps; o++) cops[o][k] = op.col_op(ct + o * kTile, k / kDB, k % kDB);
            };
            auto weight = [&](int i) {
                s[i] = __builtin_amdgcn_exp2f(fmaf(s[i], c2, nl));
            };
#pragma unroll
            for (int k = 0; k < kAhead; k++) ops[k] = row_op(k);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < 2 * kRow; k++) {
                if (k + kAhead < 2 * kRow) ops[k + kAhead] = row_op(k + kAhead);
                else col_op(k + kAhead - 2 * kRow);
                if (k < kRow) s = Mma<T>::mma(ops[k], qreg[k], s);
                else dp = Mma<T>::mma(ops[k], greg[k - kRow], dp);
                if (k > kRow) {   // not beside the first, which the last logits are only just behind
                    constexpr int kPer = (16 + kRow - 2) / (kRow - 1);
#pragma unroll
                    for (int i = (k - kRow - 1) * kPer; i < (k - kRow) * kPer && i < 16; i++) weight(i);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            // A cached block with every key visible tests nothing.  A lane is a query: a row past the end spoils only its own
            // accumulators, which are never stored, so no element tests its row.
            if (vis != 0xffffffffu || n0 + kBlk > n_cached) {
                // cached key r of the block is visible to all, chunk key r to this lane's query iff it is no later
                const int cached = n_cached - n0, seen = cached + m_lane + 1;
                const uint32_t allow = (vis & (low_bits(cached > 0 ? cached : 0) | low_bits(seen > 0 ? seen : 0))) >> (4 * h);
#pragma unroll
                for (int i = 0; i < 16; i++) s[i] = keep_if_bit(s[i], allow, 8 * (i / 4) + (i % 4));
            }
            f32x16 dsv;
            bool outside = false;
#pragma unroll
            for (int i = 0; i < (kHD == 64 ? 16 : 8); i++) dsv[i] = s[i] * dp[i];
            if constexpr (kHD == 64) {
                outside = beyond_terms(dsv);
                if (outside) {
                    uint4 kops[2 * kDB];
#pragma unroll
                    for (int k = 0; k < 2 * kDB; k++) kops[k] = op.col_op(kt, k / kDB, k % kDB);
                    accumulate_f32<T>(kops, dsv, dq);
                }
                asm volatile("");
            }
            if (!outside) {
                Weights<T, kHD> bop;
                f32x16 sums[kDB];
                bop.set(dsv, 0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < 2 * kDB; k++) {
                    if (k + kAhead < 2 * kDB) col_op(k + kAhead);
                    Half::accumulate(bop, cops, k, dq, sums);
                    if (kHD == 128 && k < kDB) {
#pragma unroll
                        for (int i = 8 + k * (8 / kDB); i < 8 + (k + 1) * (8 / kDB); i++) dsv[i] = s[i] * dp[i];
                    }
                    if (k == (kHD == 128 ? kDB - 1 : 0)) bop.set(dsv, 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                Half::finish(dq, sums);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto step = [&](auto stage_tag, int blk) {
        constexpr int st = decltype(stage_tag)::value;
        const bool more = blk + kDqStages - 1 < nblk;
        if (more) {  // the stage was last read before the barrier that ended the step before
            request_rows(blk + kDqStages, st);
            copy(rows_next, (st + kDqStages - 1) % kDqStages);
        }
        __builtin_amdgcn_sched_barrier(0);
        block(std::integral_constant<uint32_t, st * kStage>{}, std::integral_constant<uint32_t, kHalves + st * 2 * kTile>{}, blk * kRows);
        if constexpr (kSub == 2)
            block(std::integral_constant<uint32_t, st * kStage + kBlkBytes>{}, std::integral_constant<uint32_t, kHalves + st * 2 * kTile + kBlkBytes>{},
                  blk * kRows + kBlk);
        if (more) {   // this wavefront's copies of the next block have landed, and the row numbers requested above
            wait_copies<(kDqStages - 2) * kCopies>();
            rows_of(blk + kDqStages, st, rows_next);
        } else {
            wait_copies<0>();
        }
        // the halves of that stage were last read in the step before (two stages) or in the one before it: at least one barrier ago
        if (blk + 1 < nblk) Half::template split<1, kTile>(smem, (st + 1) % kDqStages * kStage, kHalves + (st + 1) % kDqStages * 2 * kTile, wave, lane);
        __syncthreads();
    };
    for (int blk = blk0; blk < nblk; blk += kDqStages) {
        step(std::integral_constant<int, 0>{}, blk);
        if (blk + 1 < nblk) step(std::integral_constant<int, 1>{}, blk + 1);
        if constexpr (kDqStages == 3)
            if (blk + 2 < nblk) step(std::integral_constant<int, 2>{}, blk + 2);
    }
    if (a.scale < 0.f) {
#pragma unroll
        for (int db = 0; db < kHD / 32; db++)
#pragma unroll
            for (int i = 0; i < 16; i++) dq[db][i] = -dq[db][i];
    }
    if (row_ok && p.n_split > 1) {
        float* out = p.part_dq + ((int64_t)share * a.B * a.H * n_ctx + bh * n_ctx + m_lane) * kHD;
#pragma unroll
        for (int db = 0; db < kHD / 32; db++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                *reinterpret_cast<float4*>(out + 32 * db + 8 * j + 4 * h) =
                    make_float4(dq[db][4 * j], dq[db][4 * j + 1], dq[db][4 * j + 2], dq[db][4 * j + 3]);
    } else if (row_ok) {
        char* out = reinterpret_cast<char*>(a.dq) + (b * a.dq_stride[0] + hd * a.dq_stride[1] + m_lane * a.dq_stride[2]) * 2;
#pragma unroll
        for (int db = 0; db < kHD / 32; db++) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int d = 32 * db + 8 * j + 4 * h;
                *reinterpret_cast<uint2*>(out + d * 2) = make_uint2(Mma<T>::pack2(dq[db][4 * j], dq[db][4 * j + 1]),
                                                                    Mma<T>::pack2(dq[db][4 * j + 2], dq[db][4 * j + 3]));
            }
        }
    }
}

template <typename T, int kHD, bool kWide, int kWaves>
__global__ void __launch_bounds__(Team<kWaves>::kThreads, Team<kWaves>::kPerCu) bwd_mfma_dq_kernel(BwdMfmaParams p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char dyn_smem[];
    dq_workgroup<T, kHD, kWide, kWaves>(p, unit_of((int)blockIdx.x, p.dq_per_head, p.dq_by_xcd), dyn_smem);
}

// the shares of dq added up in order and rounded once; a thread takes four dims of a row
template <typename T, int kHD>
__global__ void __launch_bounds__(kThreads) bwd_dq_sum_kernel(BwdMfmaParams p) {
    const ckv_dense_bwd_args& a = p.a;
    const int64_t rows = a.B * a.H * a.n_ctx, i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    const int64_t row = i / (kHD / 4);
    const int d = (int)(i % (kHD / 4)) * 4;
    if (row >= rows) return;
    float4 sum = *reinterpret_cast<const float4*>(p.part_dq + row * kHD + d);
    for (int s = 1; s < p.n_split; s++) {
        const float4 v = *reinterpret_cast<const float4*>(p.part_dq + (s * rows + row) * kHD + d);
        sum.x += v.x; sum.y += v.y; sum.z += v.z; sum.w += v.w;
    }
    const int64_t bh = row / a.n_ctx, m = row % a.n_ctx, b = bh / a.H, hd = bh % a.H;
    char* out = reinterpret_cast<char*>(a.dq) + (b * a.dq_stride[0] + hd * a.dq_stride[1] + m * a.dq_stride[2] + d) * 2;
    *reinterpret_cast<uint2*>(out) = make_uint2(Mma<T>::pack2(sum.x, sum.y), Mma<T>::pack2(sum.z, sum.w));
}

// ---------------------------------------------------------------------------------------------
// dk, dv
// ---------------------------------------------------------------------------------------------
template <typename T, int kHD>
__device__ __forceinline__ void dkdv_workgroup(const BwdMfmaParams& p, const Unit& unit, unsigned char* const dyn_smem) {   // kDkdvLds of it
    typedef Halves<T, kHD> Half;   // of Q and dO
    typedef Geo<kHD, Half::kSplit> G;
    constexpr int kTile = G::kTile;
    typedef float (*RowPtr)[2][kBlk];
    RowPtr rowv = reinterpret_cast<RowPtr>(dyn_smem + G::kDkdvRowv);                        // [stage][-lse log2 e, -delta]
    int* odd_rows = reinterpret_cast<int*>(dyn_smem + G::kDkdvOdd);               // [stage] some row's delta is not finite
    // the V^T operands of a wavefront's 32 keys and the first of K^T, in operand order: [wave][ds][lane] 16 bytes each
    uint4* vstat = reinterpret_cast<uint4*>(dyn_smem + G::kDkdvV) + __builtin_amdgcn_readfirstlane(threadIdx.x / CKV_WAVE) * (kHD / 16 + G::kParked) * CKV_WAVE;
    const ckv_dense_bwd_args& a = p.a;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / CKV_WAVE), lane = tid % CKV_WAVE, h = lane >> 5;
    const Keys keys(p);
    const int n_ctx = (int)a.n_ctx, n_cached = (int)keys.n_cached;   // below 2^31, see bwd_mfma_supported
    const int64_t bh = unit.bh, b = bh / a.H, hd = bh % a.H;
    const int n_wg = unit.x * kOwn;
    const int n_lane = n_wg + wave * 32 + (lane & 31);  // this lane's key
    const bool key_ok = keys.visible(n_lane);
    const char* qb = reinterpret_cast<const char*>(a.q) + (b * a.q_stride[0] + hd * a.q_stride[1]) * 2;
    const char* gb = reinterpret_cast<const char*>(a.dout) + (b * a.dout_stride[0] + hd * a.dout_stride[1]) * 2;
    const int64_t q_row = a.q_stride[2] * 2, g_row = a.dout_stride[2] * 2;
    const float* lse = a.lse + bh * n_ctx;
    const float* dl = p.delta + bh * n_ctx;

    // stationary B operands: K^T of this lane's key in registers but for what is parked in LDS, V^T in LDS (the registers go to the accumulators)
    constexpr int kParked = G::kParked;
    uint4 kreg[kHD / 16 - kParked];   // of ds >= kParked
    {
        const int64_t off = (b * a.kv_stride[0] + hd * a.kv_stride[1] + (key_ok ? keys.row_of(n_lane) : 0) * a.kv_stride[2]) * 2;
        const char* krow = reinterpret_cast<const char*>(a.k) + off;
        const char* vrow = reinterpret_cast<const char*>(a.v) + off;
#pragma unroll
        for (int ds = 0; ds < kHD / 16; ds++) {
            uint4 kk = make_uint4(0u, 0u, 0u, 0u), vv = kk;
            if (key_ok) {
                kk = *reinterpret_cast<const uint4*>(krow + (16 * ds + 8 * h) * 2);
                vv = *reinterpret_cast<const uint4*>(vrow + (16 * ds + 8 * h) * 2);
            }
            vstat[ds * CKV_WAVE + lane] = vv;
            if (ds < kParked) vstat[(kHD / 16 + ds) * CKV_WAVE + lane] = kk;
            else kreg[ds - kParked] = kk;
        }
    }
    const int first_row = n_lane < n_cached ? 0 : n_lane - n_cached;  // the first query that sees this key
    const float c2 = a.scale * kLog2e;

    const uint32_t lds0 = lds_address(dyn_smem);
    const Operands<kHD, true> op(lds0, lane);

    f32x16 dk[kHD / 32], dv[kHD / 32];
#pragma unroll
    for (int db = 0; db < kHD / 32; db++) dk[db] = dv[db] = zero16();

    // the first query block any key of the workgroup can be seen from
    const int blk0 = (n_wg < n_cached ? 0 : n_wg - n_cached) / kBlk;
    // keys sorted behind the visible ones: nothing but the zeros at the end
    const int nblk = n_wg < keys.n_seen ? (n_ctx + kBlk - 1) / kBlk : 0;
    // does any key of this wavefront exist and pass its mask?
    const bool wave_alive = __ballot(key_ok) != 0ull;
    const int wave_first_key = n_wg + wave * 32;

    // the copies of block m0 / 32 into a stage; rows past the end repeat the last one
    auto copy = [&](int m0, int st) {
        copy_block<kHD>(qb + m0 * q_row, (uint32_t)q_row, n_ctx - 1 - m0, lds0 + (uint32_t)(st * 2 * kTile), wave, lane);
        copy_block<kHD>(gb + m0 * g_row, (uint32_t)g_row, n_ctx - 1 - m0, lds0 + (uint32_t)(st * 2 * kTile + kTile), wave, lane);
    };
    // Per-row scalars of a block, one per lane of wavefront 0.  Rows of dout that are not finite show in their delta (a sum of
    // products with out): in their blocks the products with 64 dims take P and dS as they are, zero terms times infinity are NaN.
    constexpr bool kTerms = kHD == 64;
    auto row_scalar = [&](int m0) {
        const int m = m0 + (lane & 31);
        return m < n_ctx ? (h ? dl[m] : lse[m]) : 0.f;
    };
    auto park = [&](float v, int st) {
        rowv[st][h][lane & 31] = h ? -v : -v * kLog2e;
        if constexpr (kTerms) {
            const bool odd = __ballot(h && !(fabsf(v) < INFINITY)) != 0ull;
            if (lane == 0) odd_rows[st] = odd ? 1 : 0;
        }
    };
    if (blk0 < nblk) {
        copy(blk0 * kBlk, 0);
        if (wave == 0) park(row_scalar(blk0 * kBlk), 0);
    }
    wait_copies<0>();
    if (blk0 < nblk) Half::template split<2, kTile>(dyn_smem, 0, G::kDkdvHalves, wave, lane);
    __syncthreads();
    auto step = [&](auto stage_tag, int blk) {
        constexpr int st = decltype(stage_tag)::value;
        constexpr uint32_t qt = st * 2 * kTile, gt = qt + kTile;
        const int m0 = blk * kBlk;
        const bool more = blk + 1 < nblk;
        float rv_next = 0.f;  // a per-row scalar of the next block: requested first, parked in LDS last
        if (more) {  // the other stage was last read before the barrier that ended the step before
            if (wave == 0) rv_next = row_scalar(m0 + kBlk);
            __builtin_amdgcn_sched_barrier(0);
            copy(m0 + kBlk, st ^ 1);
        }
        // rows before the first chunk key of the wavefront's keys see none of them when all its keys are chunk keys
        const bool dead = !wave_alive || (wave_first_key >= n_cached && wave_first_key - n_cached > m0 + kBlk - 1);
        if (!dead) {
            // Rows r of the block with r_lo <= r < r_hi see this lane's key.  A lane is a key: a masked or absent key spoils only
            // its own accumulators, which are stored as zeros.
            const int r_lo = first_row - m0 < 0 ? 0 : first_row - m0 > kBlk ? kBlk : first_row - m0;
            const int r_hi = n_ctx - m0 > kBlk ? kBlk : n_ctx - m0;
            const bool plain = __ballot(r_lo > 0) == 0ull && r_hi == kBlk;  // every row of the block sees every key
            // bit r of `allow`: row r of the block sees this lane's key; element i looks at row 8 (i / 4) + 4 h + i % 4
            const uint32_t allow = (low_bits(r_hi) & ~low_bits(r_lo)) >> (4 * h);
            // Phases S, dP with P, dV with dS, dK, each in issue order: an operand is read from LDS kKvAhead matrix
            // instructions before the one that takes it, the first ones of a phase in the phase before.
            constexpr int kRow = kHD / 16, kDB = kHD / 32;
            static_assert(kParked <= kKvAhead, "parked operands are read with the first ones");
            constexpr uint32_t qc = Half::kSplit ? G::kDkdvHalves + st * 4 * kTile : qt, gc = Half::kSplit ? qc + 2 * kTile : gt;
            uint4 kops[kKvAhead], qops[kRow], gops[Half::kOps][2 * kDB], rops[kRow], vops[kRow], cops[Half::kOps][2 * kDB];
            auto g_col = [&](int k) {
#pragma unroll
                for (int o = 0; o < Half::kOps; o++) gops[o][k] = op.col_op(gc + o * kTile, k / kDB, k % kDB);
            };
            auto q_col = [&](int k) {
#pragma unroll
                for (int o = 0; o < Half::kOps; o++) cops[o][k] = op.col_op(qc + o * kTile, k / kDB, k % kDB);
            };
            f32x16 block[kDB];
            f32x16 pv = zero16(), dp;
            float nls[16];
            auto row_scalars = [&](int which, int j, auto& to) {
                const float4 v = *reinterpret_cast<const float4*>(&rowv[st][which][8 * j + 4 * h]);
                to[4 * j] = v.x; to[4 * j + 1] = v.y; to[4 * j + 2] = v.z; to[4 * j + 3] = v.w;
            };
#pragma unroll
            for (int k = 0; k < kKvAhead; k++) {
                qops[k] = op.row_op(qt, k);
                if (k < kParked) kops[k] = vstat[(kRow + k) * CKV_WAVE + lane];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < kRow; k++) {
                if (k + kKvAhead < kRow) qops[k + kKvAhead] = op.row_op(qt, k + kKvAhead);
                else if (k == kRow - 1) {
                    rops[0] = op.row_op(gt, 0);
                    vops[0] = vstat[lane];
                }
                if (k >= kRow - 4) row_scalars(1, k - (kRow - 4), dp);
                pv = Mma<T>::mma(qops[k], k < kParked ? kops[k] : kreg[k - kParked], pv);
                __builtin_amdgcn_sched_barrier(0);
            }
            constexpr int kPer = (16 + kRow - 2) / (kRow - 1);   // exponentials beside a matrix instruction
            auto weight = [&](int i) { pv[i] = __builtin_amdgcn_exp2f(fmaf(pv[i], c2, nls[i])); };
#pragma unroll
            for (int k = 0; k < kRow; k++) {
                if (k + 1 < kRow) {
                    rops[k + 1] = op.row_op(gt, k + 1);
                    vops[k + 1] = vstat[(k + 1) * CKV_WAVE + lane];
                }
                if (k >= kRow - kKvAhead) g_col(k + kKvAhead - kRow);
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (k == 4 * j / kPer) row_scalars(0, j, nls);   // a slot before the first exponential that takes one
                dp = Mma<T>::mma(rops[k], vops[k], dp);
                if (k > 0) {   // not beside the first, which the last logits are only just behind
#pragma unroll
                    for (int i = (k - 1) * kPer; i < k * kPer && i < 16; i++) weight(i);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (!plain) {
#pragma unroll
                for (int i = 0; i < 16; i++) pv[i] = keep_if_bit(pv[i], allow, 8 * (i / 4) + (i % 4));
            }
            if constexpr (!kTerms) {
                Weights<T, kHD> pw, dw;
                pw.set(pv, 0);
                pw.set(pv, 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < 2 * kDB; k++) {
                    if (k + kKvAhead < 2 * kDB) g_col(k + kKvAhead);
                    else q_col(k + kKvAhead - 2 * kDB);
                    Half::accumulate(pw, gops, k, dv, block);
#pragma unroll
                    for (int i = k * (8 / kDB); i < (k + 1) * (8 / kDB); i++) dp[i] = kScaleInside<T, kHD> ? pv[i] * dp[i] * a.scale : pv[i] * dp[i];
                    if (k == kDB - 1) dw.set(dp, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
                dw.set(dp, 1);
#pragma unroll
                for (int k = 0; k < 2 * kDB; k++) {
                    if (k + kKvAhead < 2 * kDB) q_col(k + kKvAhead);
                    Half::accumulate(dw, cops, k, dk, block);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                // the rare sides are branches of their own: as the other sides of one they spill registers of the common one
                const bool odd = __builtin_amdgcn_readfirstlane(odd_rows[st]) != 0;
                auto product_f32 = [&](uint32_t tile, const f32x16& v, f32x16(&c)[kDB]) {
                    uint4 ops[2 * kDB];
#pragma unroll
                    for (int k = 0; k < 2 * kDB; k++) ops[k] = op.col_op(tile, k / kDB, k % kDB);
                    accumulate_f32<T>(ops, v, c);
                };
                if (odd) {
                    product_f32(gt, pv, dv);
#pragma unroll
                    for (int i = 0; i < 16; i++) dp[i] *= pv[i];
                    product_f32(qt, dp, dk);
                }
                asm volatile("");
                if (!odd) {
                    Weights<T, kHD> w;
                    w.set(pv, 0);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int k = 0; k < 2 * kDB; k++) {
                        if (k + kKvAhead < 2 * kDB) g_col(k + kKvAhead);
                        else q_col(k + kKvAhead - 2 * kDB);
                        Half::accumulate(w, gops, k, dv, block);
                        if (k == 0) w.set(pv, 1);
                        if (k > 0) {
#pragma unroll
                            for (int i = (k - 1) * 6; i < k * 6 && i < 16; i++) dp[i] *= pv[i];
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    const bool outside = beyond_terms(dp);
                    Half::finish(dv, block);
                    if (outside) product_f32(qt, dp, dk);
                    asm volatile("");
                    if (!outside) {
                        w.set(dp, 0);
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int k = 0; k < 2 * kDB; k++) {
                            if (k + kKvAhead < 2 * kDB) q_col(k + kKvAhead);
                            Half::accumulate(w, cops, k, dk, block);
                            if (k == 0) w.set(dp, 1);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        Half::finish(dk, block);
                    }
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        wait_copies<0>();  // this wavefront's copies of the next block have landed
        if (more) {
            if (wave == 0) park(rv_next, st ^ 1);
            Half::template split<2, kTile>(dyn_smem, (st ^ 1) * 2 * kTile, G::kDkdvHalves + (st ^ 1) * 4 * kTile, wave, lane);
        }
        __syncthreads();
    };
    for (int blk = blk0; blk < nblk; blk += 2) {
        step(std::integral_constant<int, 0>{}, blk);
        if (blk + 1 < nblk) step(std::integral_constant<int, 1>{}, blk + 1);
    }
    if constexpr (!kScaleInside<T, kHD>) {
#pragma unroll
        for (int db = 0; db < kHD / 32; db++)
#pragma unroll
            for (int i = 0; i < 16; i++) dk[db][i] *= a.scale;
    }
    if (!key_ok) {
#pragma unroll
        for (int db = 0; db < kHD / 32; db++) dk[db] = dv[db] = zero16();
    }
    // The rows leave through LDS (the stages: nobody reads them any more), so that a store is whole rows of 16-byte pieces, 1 KiB
    // an instruction; 8-byte pieces of 32 rows apiece cost a workgroup of 32 blocks an eighth of its time.
    constexpr int kPieces = G::kPieces, kPer = CKV_WAVE / kPieces, kOut = 32 / kPer;   // rows of a store, stores of a tensor
    unsigned char* mine = dyn_smem + wave * 32 * G::kRowBytes;
    int64_t out_off[kOut];
#pragma unroll
    for (int i = 0; i < kOut; i++) {
        const int64_t n = n_wg + wave * 32 + kPer * i + lane / kPieces;
        out_off[i] = n < a.n_kv ? (b * a.dkv_stride[0] + hd * a.dkv_stride[1] + keys.row_of(n) * a.dkv_stride[2]) * 2 + (lane % kPieces) * 16 : -1;
    }
    auto store = [&](const f32x16(&acc)[kHD / 32], void* to) {
#pragma unroll
        for (int db = 0; db < kHD / 32; db++) {
#pragma unroll
            for (int j = 0; j < 4; j++)   // dims 32 db + 8 j + 4 h .. +3 of this lane's key
                *reinterpret_cast<uint2*>(mine + (lane & 31) * G::kRowBytes + (((4 * db + j) ^ (lane & (kPieces - 1))) << 4) + 8 * h) =
                    make_uint2(Mma<T>::pack2(acc[db][4 * j], acc[db][4 * j + 1]), Mma<T>::pack2(acc[db][4 * j + 2], acc[db][4 * j + 3]));
        }
#pragma unroll
        for (int i = 0; i < kOut; i++) {
            const int row = kPer * i + lane / kPieces, piece = lane % kPieces;
            const uint4 v = *reinterpret_cast<const uint4*>(mine + row * G::kRowBytes + ((piece ^ (row & (kPieces - 1))) << 4));
            if (out_off[i] >= 0) *reinterpret_cast<uint4*>(reinterpret_cast<char*>(to) + out_off[i]) = v;
        }
    };
    store(dk, a.dk);
    store(dv, a.dv);
}

template <typename T, int kHD>
__global__ void __launch_bounds__(kThreads, 2) bwd_mfma_dkdv_kernel(BwdMfmaParams p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char dyn_smem[];
    dkdv_workgroup<T, kHD>(p, unit_of((int)blockIdx.x, p.dkdv_per_head, p.dkdv_by_xcd), dyn_smem);
}

// dk / dv and dq in one launch, the longer workgroups first.
template <typename T, int kHD>
__global__ void __launch_bounds__(kThreads, 2) bwd_mfma_both_kernel(BwdMfmaParams p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char dyn_smem[];
    const int id = (int)blockIdx.x - p.dkdv_blocks;
    if (id < 0) dkdv_workgroup<T, kHD>(p, unit_of((int)blockIdx.x, p.dkdv_per_head, p.dkdv_by_xcd), dyn_smem);
    else dq_workgroup<T, kHD, false, kWaves>(p, unit_of(id, p.dq_per_head, p.dq_by_xcd), dyn_smem);
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
// unit stride along the head dim, 16-byte addressable rows, and 32 rows apart still within a 32-bit byte offset
inline bool rows_ok(const int64_t* st) {
    return st[3] == 1 && st[2] % 8 == 0 && st[1] % 8 == 0 && st[0] % 8 == 0 && st[2] > 0 && st[2] < (1 << 24);
}

template <typename T, int kHD, int kWaves>
constexpr int dq_lds() {
    constexpr int kTile = Team<kWaves>::kSub * Geo<kHD>::kTile;
    return Team<kWaves>::kStages * (2 * kTile + (Halves<T, kHD>::kSplit ? 2 * kTile : 0) + Team<kWaves>::kRows * (int)sizeof(int));
}

// Eight wavefronts where their workgroups leave no more rows empty than those of four, run all at once, and those of four would
// share compute units two by two.  K and V then reach a unit's LDS once instead of twice, and a barrier comes every 64 keys.
// units: heads of the batch x shares of the keys.  Time of the wide kernel over that of the narrow one, by the number of wide
// workgroups on 256 compute units (1024 rows x 1536 visible cached keys; 128 dims bf16 / 64 dims f16 / 64 dims bf16):
//   128 (a narrow one has a unit to itself)   1.25 / 1.17 / 1.20
//   144 to 248   0.92 to 0.95 / 0.88 to 0.91 / 0.88 to 0.91        256   0.96 / 0.91 / 0.92   (114, 150 and 107 us)
//   272   1.14 / 1.11 / 1.34     384   1.08 / 1.06 / 1.26     512   0.97 / 0.95 / 0.98
//   576   1.18 / 1.17 / 1.32     768   1.00 / 0.96 / 1.04    1536   1.03 / 1.03 / 1.12
// Past one round a unit stands idle while a wide workgroup ends or fetches its first keys, and a last round of few takes as long
// as a full one; two full rounds still gain here and lose elsewhere (1000 rows of chunk keys alone 1.00 / 0.95 / 1.15, 2048
// rows 1.13 / 1.08 / 1.33).  Within one round the other shapes are 0.88 to 1.00 too (256 rows x 768 cached keys, chunk keys
// alone, 512 rows x 3072 in shares), 2048 rows of chunk keys in 128 dims 0.95 to 1.02, and the launches of shares at few heads (32
// or 40 workgroups in 8 or 6 shares) 0.93 to 1.03.
inline bool wide_dq(int64_t n_ctx, int64_t units, int64_t cus) {
    const int64_t wide = (n_ctx + Team<8>::kOwn - 1) / Team<8>::kOwn, narrow = (n_ctx + Team<4>::kOwn - 1) / Team<4>::kOwn;
    return 2 * wide == narrow && wide * units <= cus && narrow * units > cus;
}

// dk / dv and dq in one launch (dq by workgroups of four wavefronts) while the workgroups of dk / dv are few: one launch after the other
// leaves units idle at the end of each, and with fewer workgroups than places half of every unit throughout.  Time of one launch over
// that of two (and of wide dq where wide_dq takes it), by the number of dk / dv's workgroups, heads x rows x cached keys, 128 dims bf16 / 64
// dims f16:
//   4 (2 x 64 x 128)  0.55 / 0.59        272 (2 x 1024 x 16384)  0.69 / 0.67       320 (8 x 1000 x 4095, a quarter masked)  0.81 / 0.76
//   576 (8 x 1024 x 8192)  0.92 / 0.93   640 (16 x 1024 x 4096)  0.88 / 0.92       768 (32 x 1024 x 2048)  0.91 / 0.92
//   1216 (64 x 300 x 2048)  0.93 / 0.93  1280 (32 x 1024 x 4096, half masked)  0.99 / 0.97
//   1536 (64 x 1024 x 2048)  1.02 / 0.99   4352 (32 x 1024 x 16384)  1.10 / 1.08   8256 (64 x 100 x 16384)  1.06 / 1.04
// (8 heads x 1000 rows x 5095 keys of 64 dims in float16: 123.8 -> 94.1 us.)  Many rounds of dk / dv run better by themselves.
inline bool both_at_once(int64_t dkdv_blocks, int64_t cus) { return dkdv_blocks <= 5 * cus; }

template <typename T, int kHD>
int run(const BwdMfmaParams& p_in, hipStream_t stream) {
    BwdMfmaParams p = p_in;
    const ckv_dense_bwd_args& a = p.a;
    const int64_t heads = a.B * a.H, cus = mfma_device_cus();
    auto by_xcd = [&](int64_t blocks, int64_t most) { return heads % 8 == 0 && blocks <= most ? 1 : 0; };
    const int64_t dkdv_blocks = (a.n_kv + kOwn - 1) / kOwn * heads;
    p.dkdv_per_head = (int)((a.n_kv + kOwn - 1) / kOwn);
    p.dkdv_by_xcd = by_xcd(dkdv_blocks, 2 * cus);
    p.dkdv_blocks = (int)dkdv_blocks;
    constexpr int kDkdvLds = Geo<kHD, Halves<T, kHD>::kSplit>::kDkdvLds;
    auto dq_blocks = [&](int own) -> int64_t {
        p.dq_per_head = (int)((a.n_ctx + own - 1) / own * p.n_split);
        p.dq_by_xcd = heads % 8 == 0;
        return heads * p.dq_per_head;
    };
    if (dkdv_blocks > 0x3fffffff || (a.n_ctx + kOwn - 1) / kOwn * p.n_split * heads > 0x3fffffff) return CKV_ERR_UNSUPPORTED;
    auto launch_dq = [&](auto waves_tag, auto wide_rows_tag) -> int {
        constexpr int kWaves = decltype(waves_tag)::value;
        constexpr int kLds = dq_lds<T, kHD, kWaves>();
        auto* kernel = bwd_mfma_dq_kernel<T, kHD, decltype(wide_rows_tag)::value, kWaves>;
        if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), kLds)) return rc;
        const int64_t blocks = dq_blocks(Team<kWaves>::kOwn);
        hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(Team<kWaves>::kThreads), kLds, stream, p);
        CKV_HIP_TRY(hipGetLastError());
        return CKV_OK;
    };
    auto sum_shares = [&]() -> int {
        if (p.n_split > 1) {
            const int64_t threads = heads * a.n_ctx * (kHD / 4);
            hipLaunchKernelGGL((bwd_dq_sum_kernel<T, kHD>), dim3((unsigned)((threads + kThreads - 1) / kThreads)), dim3(kThreads), 0,
                               stream, p);
            CKV_HIP_TRY(hipGetLastError());
        }
        return CKV_OK;
    };
    constexpr std::integral_constant<int, 4> narrow{};
    constexpr std::integral_constant<int, 8> wide{};
    const bool far_rows = a.n_kv * a.kv_stride[2] * 2 >= (int64_t)1 << 32;
    if (!far_rows && both_at_once(dkdv_blocks, cus)) {
        constexpr int kLds = kDkdvLds > dq_lds<T, kHD, kWaves>() ? kDkdvLds : dq_lds<T, kHD, kWaves>();
        if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(bwd_mfma_both_kernel<T, kHD>), kLds)) return rc;
        const int64_t blocks = dkdv_blocks + dq_blocks(kOwn);
        hipLaunchKernelGGL((bwd_mfma_both_kernel<T, kHD>), dim3((unsigned)blocks), dim3(kThreads), kLds, stream, p);
        CKV_HIP_TRY(hipGetLastError());
        return sum_shares();
    }
    if (far_rows) {
        if (int rc = launch_dq(narrow, std::true_type{})) return rc;
    } else if (wide_dq(a.n_ctx, heads * p.n_split, cus)) {
        if (int rc = launch_dq(wide, std::false_type{})) return rc;
    } else if (int rc = launch_dq(narrow, std::false_type{})) {
        return rc;
    }
    if (int rc = sum_shares()) return rc;
    if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(bwd_mfma_dkdv_kernel<T, kHD>), kDkdvLds)) return rc;
    hipLaunchKernelGGL((bwd_mfma_dkdv_kernel<T, kHD>), dim3((unsigned)dkdv_blocks), dim3(kThreads), kDkdvLds, stream, p);
    CKV_HIP_TRY(hipGetLastError());
    return CKV_OK;
}

}  // namespace

bool bwd_mfma_supported(const ckv_dense_bwd_args& a) {
    if (a.dtype != CKV_F16 && a.dtype != CKV_BF16) return false;
    if (a.D != 64 && a.D != 128) return false;
    if (a.n_kv > 0x7fffff00) return false;   // keys and rows are numbered in 32 bits
    if (!rows_ok(a.q_stride) || !rows_ok(a.kv_stride) || !rows_ok(a.dout_stride) || !rows_ok(a.dq_stride) ||
        !rows_ok(a.dkv_stride))
        return false;
    return aligned16(a.q) && aligned16(a.k) && aligned16(a.v) && aligned16(a.dout) && aligned16(a.dq) &&
           aligned16(a.dk) && aligned16(a.dv);
}

// Shares of the keys for dq (1: no sharing), counted in workgroups of four wavefronts, one per 128 rows of a head, two of which
// fit a compute unit: with fewer than one per compute unit the keys are dealt out over up to 8 of them, at least 8 blocks of 32
// keys each, about two workgroups per compute unit in all (as many rows and keys as one wide workgroup, which wide_dq may then
// take in their place), and the shares (float32) are added up by a kernel behind.  8 heads x 1000 rows are 64 workgroups, a
// quarter of the chip.
int bwd_mfma_dq_splits(int64_t B, int64_t H, int64_t n_ctx, int64_t n_kv, int cus) {
    constexpr int kDqRows = Team<4>::kOwn;
    const int64_t wgs = (n_ctx + kDqRows - 1) / kDqRows * B * H, blocks = (n_kv + kBlk - 1) / kBlk;
    if (wgs >= cus) return 1;
    int64_t s = 2 * (int64_t)cus / wgs;
    if (s > blocks / 8) s = blocks / 8;
    if (s > 8) s = 8;
    return s < 1 ? 1 : (int)s;
}

int launch_bwd_mfma(const ckv_dense_bwd_args& a, const float* delta, const int* key_order, const int* n_visible, float* part_dq,
                    int n_split, hipStream_t stream) {
    BwdMfmaParams p;
    p.dq_per_head = p.dkdv_per_head = p.dkdv_blocks = 1;
    p.dq_by_xcd = p.dkdv_by_xcd = 0;
    p.part_dq = part_dq;
    p.n_split = part_dq ? n_split : 1;
    p.a = a;
    p.delta = delta;
    p.key_order = key_order;
    p.n_visible = n_visible;
    if (a.D == 64) return a.dtype == CKV_F16 ? run<__half, 64>(p, stream) : run<__hip_bfloat16, 64>(p, stream);
    return a.dtype == CKV_F16 ? run<__half, 128>(p, stream) : run<__hip_bfloat16, 128>(p, stream);
}

}  // namespace ckv

// For tests that aim at one kernel (cus 0: the current device's): are dk / dv and dq one launch; where not, and for rows
// addressed in 32 bits, the wavefronts of dq's workgroups
extern "C" int ckv_dense_bwd_one_launch(int64_t n_kv, int64_t heads, int64_t cus) {
    return ckv::both_at_once((n_kv + ckv::kOwn - 1) / ckv::kOwn * heads, cus > 0 ? cus : ckv::mfma_device_cus());
}
extern "C" int ckv_dense_bwd_dq_wavefronts(int64_t n_ctx, int64_t units, int64_t cus) {
    return ckv::wide_dq(n_ctx, units, cus > 0 ? cus : ckv::mfma_device_cus()) ? 8 : 4;
}
