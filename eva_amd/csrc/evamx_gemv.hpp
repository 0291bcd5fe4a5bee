// Wave-level decode GEMV and Hadamard helpers shared by the MoE and the single-linear kernels.
//
// GEMV lane layout (wave64): lane = 8*i + q streams tile (kt, 8*cg + i) words q*K..q*K+K-1 with
// one vector load per k-slice and owns output columns 16i+q and 16i+q+8 of the 128-column group
// for all 16 k of the tile, so the k-loop needs no cross-lane reduction and a wave's 128 columns
// are exactly one Hadamard chunk. The 16 decoded k of a column pair up as (k, k+1). The MoE
// decode path multiplies them on the matrix cores with fp32 accumulation (gemv_wave_m4: each lane
// quad is one v_mfma_f32_4x4x4_16b_f16 block). The single linear and the MFMA tiles take the same
// decode with the lanes 2 tiles across by 4 k-slices down (evamx_mfma.hpp).
#pragma once
#include "evamx_device.hpp"

#include <type_traits>

namespace evamx {

__device__ __forceinline__ float h2f(half_t h) { return (float)h; }
__device__ __forceinline__ half_t f2h(float f) { return (half_t)f; }

// ---------------------------------------------------------------------------------------------
// Wave Hadamard over a 128-chunk held as two values per lane at element e = 16*(lane>>3) +
// 8*h + (lane&7): stages on e bits 0..6 in order (lane xor 1,2,4; in-lane; lane xor 8,16,32),
// which is the reference's order (hadamard_inner.cuh:17-44, exl3_moe_coop_kernel.cuh:131-147).

__device__ __forceinline__ int lane_col(int lane, int h) { return 16 * (lane >> 3) + 8 * h + (lane & 7); }

__device__ __forceinline__ void had128_lane(float& v0, float& v1, int lane)
{
    v0 = bfly_x<1>(v0, lane);  v1 = bfly_x<1>(v1, lane);
    v0 = bfly_x<2>(v0, lane);  v1 = bfly_x<2>(v1, lane);
    v0 = bfly_x<4>(v0, lane);  v1 = bfly_x<4>(v1, lane);
    {
        const float a = v0, c = v1;
        v0 = a + c;
        v1 = a - c;
    }
    v0 = bfly_x<8>(v0, lane);  v1 = bfly_x<8>(v1, lane);
    v0 = bfly_x<16>(v0, lane); v1 = bfly_x<16>(v1, lane);
    v0 = bfly_x<32>(v0, lane); v1 = bfly_x<32>(v1, lane);
    v0 *= R_SCALE;
    v1 *= R_SCALE;
}

// The same transform for a chunk held as consecutive pairs, element e = 2*lane + h: stage 0 is
// in-lane, stages 1..6 pair lanes xor 1..32. Same stage order and operand pairs as had128_lane,
// so the results are bit-identical.
__device__ __forceinline__ void had128_pair(float& v0, float& v1, int lane)
{
    {
        const float a = v0, c = v1;
        v0 = a + c;
        v1 = a - c;
    }
    v0 = bfly_x<1>(v0, lane);  v1 = bfly_x<1>(v1, lane);
    v0 = bfly_x<2>(v0, lane);  v1 = bfly_x<2>(v1, lane);
    v0 = bfly_x<4>(v0, lane);  v1 = bfly_x<4>(v1, lane);
    v0 = bfly_x<8>(v0, lane);  v1 = bfly_x<8>(v1, lane);
    v0 = bfly_x<16>(v0, lane); v1 = bfly_x<16>(v1, lane);
    v0 = bfly_x<32>(v0, lane); v1 = bfly_x<32>(v1, lane);
    v0 *= R_SCALE;
    v1 *= R_SCALE;
}

// The same Hadamard with a chunk on 16 lanes, 8 consecutive elements a lane (a wave holds four chunks):
// element bits 0-2 are in the lane; bits 3-6 pair lanes xor 1, 2, 7 and 8, each one DPP pattern of a
// 16-lane row (xor 4 would take two and a select), so lane l holds the elements from 8 * oct_piece(l)
// on. Same stages in the same order, so the results are bit-identical; 12 instructions an element
// instead of 17, and a chunk's values move as 16-byte pieces.
__device__ __forceinline__ int oct_piece(int lane)
{
    const int b2 = (lane >> 2) & 1;
    return (((lane & 3) ^ (3 * b2)) | (lane & 12));
}

template <int CTRL>
__device__ __forceinline__ void oct_stage(float (&v)[8], bool upper)
{
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = dpp_f<CTRL>(v[i]) + (upper ? -v[i] : v[i]);
}

__device__ __forceinline__ void had128_oct(float (&v)[8], int lane)
{
    const int e = oct_piece(lane);
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        const float a = v[i], c = v[i + 1];
        v[i] = a + c;
        v[i + 1] = a - c;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int i = (j & 1) + 4 * (j >> 1);
        const float a = v[i], c = v[i + 2];
        v[i] = a + c;
        v[i + 2] = a - c;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = v[i], c = v[i + 4];
        v[i] = a + c;
        v[i + 4] = a - c;
    }
    oct_stage<0xB1>(v, e & 1);             // quad_perm [1,0,3,2]: lane xor 1
    oct_stage<0x4E>(v, e & 2);             // quad_perm [2,3,0,1]: lane xor 2
    oct_stage<0x141>(v, e & 4);            // row_half_mirror: lane xor 7
    oct_stage<0x128>(v, e & 8);            // row_ror:8: lane xor 8
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] *= R_SCALE;
}

// Sum of a chunk's 8 values a lane after their rounding to fp16, in every lane of its 16.
__device__ __forceinline__ float oct_sum(const half2_t (&r)[4])
{
    const half2_t one = {(half_t)1.0f, (half_t)1.0f};
    float t = dot2(r[3], one, dot2(r[2], one, dot2(r[1], one, dot2(r[0], one, 0.0f))));
    t += dpp_f<0xB1>(t);
    t += dpp_f<0x4E>(t);
    t += dpp_f<0x141>(t);
    t += dpp_f<0x128>(t);
    return t;
}

// 16-byte pieces of rows whose alignment is only that of their elements or of a dword (caller's
// pointers); the compiler emits wide accesses where the hardware takes them.
typedef uint32_t u32x4w __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4h __attribute__((ext_vector_type(4), aligned(2)));
typedef float f32x4w __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ void oct_halves(const uint32_t (&w)[4], float (&v)[8])
{
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const half2_t h = __builtin_bit_cast(half2_t, w[i]);
        v[2 * i] = h2f(h.x);
        v[2 * i + 1] = h2f(h.y);
    }
}

// 8 fp16 values at p (2-byte aligned) as floats.
__device__ __forceinline__ void oct_load_half(const half_t* p, float (&v)[8])
{
    const u32x4h w = *(const __attribute__((address_space(1))) u32x4h*)p;
    const uint32_t u[4] = {w.x, w.y, w.z, w.w};
    oct_halves(u, v);
}

// The codebook's affine map applied to a column's sums: sum_k x_k w_k = 0x1eee * sum_k x_k h_k +
// 0xc931 * sum_k x_k, with one explicit fused multiply-add, so that no kernel's row count can change
// how the compiler contracts it (a row's bits must not depend on its call's row count).
__device__ __forceinline__ float mul1_affine(float acc, float xs)
{
    return __builtin_fmaf(MUL1_K_INV, acc, MUL1_K_BIAS * xs);
}

// ---------------------------------------------------------------------------------------------
// Streaming loads.

typedef uint32_t u32x2a __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t u32x3a __attribute__((ext_vector_type(3), aligned(4)));
typedef uint32_t u32x4a __attribute__((ext_vector_type(4), aligned(4)));

// Global-address-space view of a pointer. Loads through a generic pointer become flat loads,
// which also count against the LDS/scalar counter: every wait for a scalar activation load
// would then drain the whole weight prefetch ring.
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(1))) T* gptr(const void* p)
{
    return (const __attribute__((address_space(1))) T*)p;
}

// A lane's words of one k-slice: its K words with one non-temporal 64/96/128-bit buffer load
// (+1 dword at K=5). The word before them in the tile's circular bit string comes from the lane
// that owns it (prev_word): a second load from the same cache lines cost more than the two
// instructions of the exchange, since the vector memory path is as busy as the vector ALU here
// (16 tokens at 4 bpw, MFMA tiles: 361 -> 327 us; 400 tokens at 3 bpw: 1850 -> 1719 us). Buffer
// loads take the wave-uniform slice offset in a scalar register and the per-lane offsets as
// constant vector offsets, so a step spends no vector instructions on addresses.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int BUF_NT = 2;                          // cache policy: non-temporal
constexpr int BUF_WORD3 = 0x00020000;              // raw 32-bit buffer resource on gfx9-family parts

// Resource of a wave-uniform base (the pointer is made provably uniform, so the descriptor lives
// in scalar registers and no load needs a per-lane loop over descriptors).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t weight_rsrc(const uint32_t* base)
{
    const uint64_t v = (uint64_t)(uintptr_t)base;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    uint32_t* u = (uint32_t*)(uintptr_t)(((uint64_t)hi << 32) | lo);
    return __builtin_amdgcn_make_buffer_rsrc(u, (short)0, 0x7fffffff, BUF_WORD3);
}

template <int K>
__device__ __forceinline__ void load_slice(LaneWords<K>& w, __amdgpu_buffer_rsrc_t rsrc, uint32_t soff, uint32_t lane_off)
{
    if constexpr (K == 1) {
        w.b[1] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, lane_off, soff, BUF_NT);
    } else if constexpr (K == 2) {
        const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, lane_off, soff, BUF_NT));
        w.b[1] = v.x; w.b[2] = v.y;
    } else if constexpr (K == 3) {
        const u32x3 v = __builtin_bit_cast(u32x3, __builtin_amdgcn_raw_buffer_load_b96(rsrc, lane_off, soff, BUF_NT));
        w.b[1] = v.x; w.b[2] = v.y; w.b[3] = v.z;
    } else {
        const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane_off, soff, BUF_NT));
        w.b[1] = v.x; w.b[2] = v.y; w.b[3] = v.z; w.b[4] = v.w;
#pragma unroll
        for (int i = 4; i < K; ++i) w.b[i + 1] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, lane_off + 4 * i, soff, BUF_NT);
    }
}

// The word before a lane's own: the last word of the lane before it among the tile's 8 lanes,
// circularly. A row of 16 lanes holds two tiles: rotated by one it gives every lane but each tile's
// first its word, rotated by nine those two. (At half rates only the even lanes' windows reach into
// the word before their own, and for them it is the previous lane's last word too.)
template <int K>
__device__ __forceinline__ uint32_t prev_word(const LaneWords<K>& w)
{
    const int r9 = __builtin_amdgcn_update_dpp(0, (int)w.b[K], 0x129, 0xf, 0xf, true);     // row_ror:9
    const int r1 = __builtin_amdgcn_update_dpp(0, (int)w.b[K], 0x121, 0xf, 0xf, true);     // row_ror:1
    return (uint32_t)((threadIdx.x & 7) == 0 ? r9 : r1);
}

// ---------------------------------------------------------------------------------------------
// Waves sharing a SIMD issue oldest-first, so without help the oldest races ahead, the youngest
// finishes last, and the SIMD's last stretch runs one wave that cannot hide its own load
// latency. A streaming loop sets its wave's priority from its progress (done of n steps): 3
// below half, 2 to 3/4, 1 to 9/10, then 0, so a wave that is ahead yields to the ones behind
// and the SIMD's waves reach each mark together; only the last tenth is issued oldest-first.
__device__ __forceinline__ void progress_priority(int done, int n)
{
    if (10 * done >= 9 * n) __builtin_amdgcn_s_setprio(0);
    else if (4 * done >= 3 * n) __builtin_amdgcn_s_setprio(1);
    else if (2 * done >= n) __builtin_amdgcn_s_setprio(2);
    else __builtin_amdgcn_s_setprio(3);
}

// ---------------------------------------------------------------------------------------------
// Rate geometry and per-slice decode of the lane layout (lane = 8*i + q owns tile i's columns q
// and q + 8 for the 16 k of a k-slice), shared by the decode GEMV and the MFMA path.

// K2 = 2 x bits: even for integer rates (K = K2/2 words per lane), odd for rates b + 0.5.
template <int K2>
struct Rate {
    static constexpr bool HALF = (K2 & 1) != 0;
    static constexpr int B = K2 / 2;                          // whole bits (half rates)
    static constexpr int K = HALF ? B + 1 : K2 / 2;           // words loaded per lane besides b[0]
    static constexpr int TW = HALF ? 4 * (2 * B + 1) : 8 * K; // words per tile
};

// Byte offset of a lane's K words within its tile group and, at half rates, the normalising shift.
template <int K2>
__device__ __forceinline__ void lane_offsets(int lane, uint32_t& lane_off, uint32_t& sh)
{
    using R = Rate<K2>;
    const int q = lane & 7;
    sh = 0;
    if constexpr (!R::HALF) {
        lane_off = 4u * (uint32_t)((lane >> 3) * R::TW + q * R::K);
    } else {
        // the words from the one that holds the lane's first bit: 16 q (2 B + 1) bits into the tile
        lane_off = 4u * (uint32_t)((lane >> 3) * R::TW + q * (2 * R::B + 1) / 2);
        sh = (q & 1) ? 0u : 16u;
    }
}

// The (1024 + bytesum) pairs of the lane's 32 positions of one k-slice:
// wp[4u + 2c + kh] = column q + 8c, k = 8kh + 2u and 8kh + 2u + 1 (low half: even k).
// FENCED: no matrix instruction runs among this decode's (see Mul1).
template <int K2, bool FENCED>
__device__ __forceinline__ void decode_slice(LaneWords<Rate<K2>::K>& w, uint32_t sh, half2_t (&wp)[16])
{
    using R = Rate<K2>;
    constexpr int K = R::K, B = R::B;
    w.b[0] = prev_word<K>(w);
    Mul1<FENCED> m;
    if constexpr (!R::HALF) {
        lane_pairs<K, FENCED>(w, m, wp);
    } else {
        uint32_t N[B + 1];
#pragma unroll
        for (int k = 0; k <= B; ++k) N[k] = __builtin_amdgcn_alignbit(w.b[k], w.b[k + 1], sh);
        half_pairs<B, FENCED>(N, m, wp);
    }
}

// ---------------------------------------------------------------------------------------------
// Activation rows of the MFMA tiles: the k-vector of each slot, which a tile's lanes read as their A
// operands, together with its per-128-chunk sums (fp32) that the affine codebook map needs.

struct GlobalRows {
    const half_t* A;
    size_t stride;          // elements per row
    const float* sums;      // [row][chunk] sums of the fp16 row values over 128-element chunks
    int sums_stride;        // chunks per row
};

// Orders a wave's LDS writes before its later LDS reads of other lanes' data (and its reads
// before later overwrites): LDS instructions of one wave execute in order, the fence keeps the
// compiler from moving them across.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------------------------
// The decode GEMV's products on the matrix cores: v_mfma_f32_4x4x4_16b_f16 runs 16
// independent 4x4x4 blocks, block b on lanes 4b..4b+3, and the decode layout's lane quads are
// exactly such blocks (the four lanes of a quad own four columns of one tile at the same k).
// Lane 4b + j supplies column j of its block as the B operand (the four k of a k-group from its
// decoded pairs) and row j of the block's A operand (the activations of row 4g + j of its 4-row
// group at those k); the block's D holds the four rows of the lane's column in four registers.
// One MFMA thus takes the products of 4 rows x 4 k per lane where v_dot2 takes 1 row x 2 k:
// a k-slice costs 8 MFMAs per 4-row group instead of 16 v_dot2 per row. Rows of a group past the
// call's rows read a copy of the group's first row (their outputs are dropped); a row's result
// does not depend on the other rows of its group.

typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float f32x4v_t __attribute__((ext_vector_type(4)));

// Activation rows of the MFMA-product GEMV, staged in LDS: row m at base + m * row_words (a
// padded stride, so that the four rows a lane quad reads sit in different banks), k-slice kt at
// word 8 * (kt - kt0). Lane l reads row 4g + (l & 3) of group g.
template <int NG>
struct XLds4 {
    const uint32_t* base;
    int off[NG];            // this lane's row offset (words) in each group
    int kt0;
    __device__ __forceinline__ void init(const uint32_t* b, int row_words, int k0, int tm)
    {
        base = b;
        kt0 = k0;
        const int j = threadIdx.x & 3;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int m = 4 * g + j;
            off[g] = (m < tm ? m : 4 * g < tm ? 4 * g : 0) * row_words;
        }
    }
    __device__ __forceinline__ void load(int g, int kt, uint32_t (&d)[8]) const
    {
        const uint32_t* xp = (const uint32_t*)__builtin_assume_aligned(base + off[g] + 8 * (kt - kt0), 32);
#pragma unroll
        for (int i = 0; i < 8; ++i) d[i] = xp[i];
    }
};

// B operand of one MFMA: column c (0: q, 1: q + 8) of the lane, k-group kg (k = 4 kg .. 4 kg + 3)
// of the slice's decoded pairs (wp[4u + 2c + kh] holds k = 8 kh + 2u, 8 kh + 2u + 1).
__device__ __forceinline__ half4_t m4_b(const half2_t (&wp)[16], int c, int kg)
{
    const int kh = kg >> 1, u = 2 * (kg & 1);
    const half2_t lo = wp[4 * u + 2 * c + kh], hi = wp[4 * (u + 1) + 2 * c + kh];
    return half4_t{lo.x, lo.y, hi.x, hi.y};
}

__device__ __forceinline__ half4_t m4_a(const uint32_t (&a)[8], int kg)
{
    const half2_t lo = __builtin_bit_cast(half2_t, a[2 * kg]), hi = __builtin_bit_cast(half2_t, a[2 * kg + 1]);
    return half4_t{lo.x, lo.y, hi.x, hi.y};
}

// acc[g][c][i] += sum_k X[4g + i][k] * h_k over the wave's k-range [kt0, kt1) for the lane's column
// c, for tm >= 1 rows; groups g with 4g >= tm are skipped. prologue.issue() runs
// before the first weight loads (loads issued there return first: vector memory loads return in
// order), prologue.finish() once they are in flight.
template <int K2, int NG, int PF = 4, typename Pro>
__device__ __forceinline__ void gemv_wave_m4(const uint32_t* __restrict__ trellis, int nt_n, int cg, int kt0, int kt1,
                                             const XLds4<NG>& xs, int tm, f32x4v_t (&acc)[NG][2], Pro& prologue)
{
    using R = Rate<K2>;
    constexpr int K = R::K;
    constexpr int TW = R::TW;
    const int lane = threadIdx.x & 63;
    kt0 = __builtin_amdgcn_readfirstlane(kt0);
    kt1 = __builtin_amdgcn_readfirstlane(kt1);
    const uint32_t slice = __builtin_amdgcn_readfirstlane(4u * (uint32_t)(nt_n * TW));
    const uint32_t cbase = __builtin_amdgcn_readfirstlane(4u * (uint32_t)(cg * 8 * TW));
    const __amdgpu_buffer_rsrc_t rsrc = weight_rsrc(trellis);
    uint32_t lane_off, sh;
    lane_offsets<K2>(lane, lane_off, sh);

    prologue.issue();
    LaneWords<K> ring[PF];
    const int last = kt1 - 1;
#pragma unroll
    for (int d = 0; d < PF; ++d) load_slice<K>(ring[d], rsrc, cbase + (uint32_t)min(kt0 + d, last) * slice, lane_off);
    __builtin_amdgcn_sched_barrier(0);
    prologue.finish();

    // The loop over the k-slices for NA active groups (the groups holding rows), with no branch
    // inside a step: a per-group test in the step splits it into blocks that serialise the
    // decode and the products.
    auto run = [&](auto na) {
        constexpr int NA = decltype(na)::value;
        // a step reads its slice's activations from LDS first: the decode hides their latency
        auto step = [&](int kt, LaneWords<K>& w) {
            uint32_t xa[NA][8];
#pragma unroll
            for (int g = 0; g < NA; ++g) xs.load(g, kt, xa[g]);
            half2_t wp[16];
            decode_slice<K2, true>(w, sh, wp);
            load_slice<K>(w, rsrc, cbase + (uint32_t)min(kt + PF, last) * slice, lane_off);
            mfma_begin();
#pragma unroll
            for (int kg = 0; kg < 4; ++kg)
#pragma unroll
                for (int g = 0; g < NA; ++g) {
                    const half4_t a = m4_a(xa[g], kg);
#pragma unroll
                    for (int c = 0; c < 2; ++c)
                        acc[g][c] = __builtin_amdgcn_mfma_f32_4x4x4f16(a, m4_b(wp, c, kg), acc[g][c], 0, 0, 0);
                }
            mfma_end<2>();
        };

        const int n_kt = kt1 - kt0;
        int kt = kt0;
        for (; kt + PF <= kt1; kt += PF) {
            progress_priority(kt - kt0, n_kt);
#pragma unroll
            for (int d = 0; d < PF; ++d) step(kt + d, ring[d]);
        }
        progress_priority(n_kt, n_kt);
#pragma unroll
        for (int d = 0; d < PF - 1; ++d)
            if (kt + d < kt1) step(kt + d, ring[d]);
    };
    static_assert(NG == 1 || NG == 2 || NG == 4, "decode path row groups: 1, 2 or 4");
    if constexpr (NG == 1) {
        run(std::integral_constant<int, 1>{});
    } else if constexpr (NG == 2) {
        if (tm > 4) run(std::integral_constant<int, 2>{});
        else run(std::integral_constant<int, 1>{});
    } else {
        // four groups: 9 to 16 rows (9-12 rows too: the fourth group's products are dropped)
        run(std::integral_constant<int, 4>{});
    }
}

// sum of sp[c0], sp[c0 + d], ... below c1, added in that order from 0 (as a sequential loop
// does), the loads of up to B terms issued before their adds: one memory round trip per B terms
// instead of one per term (a loop that adds each load before issuing the next waits a full round
// trip per term).
template <int B>
__device__ __forceinline__ float strided_sum(const float* sp, int c0, int c1, int d = 1)
{
    float xs = 0.0f;
    for (int c = c0; c < c1; c += B * d) {
        float t[B];
#pragma unroll
        for (int j = 0; j < B; ++j) t[j] = gptr<float>(sp)[c + j * d < c1 ? c + j * d : c];
#pragma unroll
        for (int j = 0; j < B; ++j)
            if (c + j * d < c1) xs += t[j];
    }
    return xs;
}

// Sum over the wave of one value per lane (order fixed by the butterfly).
__device__ __forceinline__ float wave_sum(float v)
{
    const int lane = threadIdx.x & 63;
    v = pair_sum<1>(v, lane);
    v = pair_sum<2>(v, lane);
    v = pair_sum<4>(v, lane);
    v = pair_sum<8>(v, lane);
    v = pair_sum<16>(v, lane);
    v = pair_sum<32>(v, lane);
    return v;
}

}  // namespace evamx
