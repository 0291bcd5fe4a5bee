// Wide tiles: a workgroup of WIDE_WAVES waves multiplies up to 16 MB rows a wave by 128 columns with every
// weight decoded once for all of them.
//
// Per stage of 128 k (8 k-slices) each wave decodes one unit (a pair of the column group's tiles over
// 4 k-slices) into its four B operands (evamx_mfma.hpp: the decode's own register layout) and stores
// them to LDS as they are, 16 bytes a lane; all waves then multiply all the operands by their own rows'
// A operands, read straight from global memory. Operands alternate between two LDS buffers, so a stage needs one
// barrier, and the next stage's decode (vector ALU) runs beside this stage's products (matrix cores).
#pragma once
#include "evamx_mfma.hpp"

namespace evamx {

constexpr int WIDE_WAVES = 8;

struct WideLds {
    u32x4_t b[2][4 * WIDE_WAVES][64];       // [buffer][4 unit + 2 c + h][lane]; unit 4 i + j: pair j at k64 step i
};

// LDS stores before the barrier are visible after it; loads from global memory stay in flight.
__device__ __forceinline__ void wide_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A unit decoded into its four operands (2 c + h).
struct WideOps {
    u32x4_t o0, o1, o2, o3;
};

template <int K2>
__device__ __forceinline__ WideOps wide_decode(LaneWords<Rate<K2>::K>& w, uint32_t sh)
{
    half2_t wp[16];
    decode_slice<K2, false>(w, sh, wp);
    return WideOps{__builtin_bit_cast(u32x4_t, mfma_b(wp, 0, 0)), __builtin_bit_cast(u32x4_t, mfma_b(wp, 0, 1)),
                   __builtin_bit_cast(u32x4_t, mfma_b(wp, 1, 0)), __builtin_bit_cast(u32x4_t, mfma_b(wp, 1, 1))};
}

__device__ __forceinline__ void wide_put(WideLds& lds, int buf, int unit, int lane, const WideOps& o)
{
    lds.b[buf][4 * unit][lane] = o.o0;
    lds.b[buf][4 * unit + 1][lane] = o.o1;
    lds.b[buf][4 * unit + 2][lane] = o.o2;
    lds.b[buf][4 * unit + 3][lane] = o.o3;
}

// acc[mb][nb][r] += sum_k x_k h_k over `chunks` 128-chunks of k from k-slice kt0 on, for row 4 g + r of
// the 16-row block mb (its A operands at arow[mb], a_operand_offset) and column mfma_col(lane, nb).
// end(c) runs after chunk c.
template <int K2, int MB, typename End>
__device__ __forceinline__ void wide_accumulate(const uint32_t* __restrict__ trellis, int nt_n, int cg, int kt0, int chunks,
                                                const __attribute__((address_space(1))) u32x4_t* const (&arow)[MB],
                                                WideLds& lds, f32x4_t (&acc)[MB][8], End&& end)
{
    using R = Rate<K2>;
    constexpr int K = R::K;
    constexpr int TW = R::TW;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int g = lane >> 4;
    const int last = chunks - 1, last_step = 2 * chunks - 1;       // a stage is a chunk, of two k64 steps
    const uint32_t slice = __builtin_amdgcn_readfirstlane(4u * (uint32_t)(nt_n * TW));
    const uint32_t cbase = __builtin_amdgcn_readfirstlane(4u * (uint32_t)((cg * 8 + 2 * (wave & 3)) * TW) +
                                                          (uint32_t)(kt0 + 4 * (wave >> 2)) * slice);
    const __amdgpu_buffer_rsrc_t rsrc = weight_rsrc(trellis);
    uint32_t lane_off, sh;
    lane_offsets<K2>(lane & 15, lane_off, sh);
    lane_off += (uint32_t)g * slice;

    LaneWords<K> ring[2];
    u32x4_t a[2][MB][2];                          // activations of alternate k64 steps
    auto load_a = [&](u32x4_t (&d)[MB][2], int t) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int h = 0; h < 2; ++h) d[mb][h] = arow[mb][128 * min(t, last_step) + 64 * h];
    };
    auto load_w = [&](LaneWords<K>& w, int s) {
        load_slice<K>(w, rsrc, cbase + (uint32_t)(8 * min(s, last)) * slice, lane_off);
    };
    load_w(ring[0], 0);
    load_w(ring[1], 1);
    load_a(a[0], 0);
    {
        const WideOps o = wide_decode<K2>(ring[0], sh);
        load_w(ring[0], 2);
        wide_put(lds, 0, wave, lane, o);
        wide_barrier();
    }
    // the products of k64 step i of a stage
    auto products = [&](int buf, int i, const u32x4_t (&x)[MB][2]) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const half8_t b = __builtin_bit_cast(half8_t, lds.b[buf][16 * i + j][lane]);
            const int nb = 2 * (j >> 2) + ((j >> 1) & 1);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
                acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, x[mb][j & 1]), b, acc[mb][nb], 0, 0, 0);
        }
    };
    // stage s from buffer buf, while the next stage's unit w is decoded into the other buffer (past the
    // end: a repeat, unused); activations are loaded one k64 step ahead, weights two stages
    auto stage = [&](int s, int buf, LaneWords<K>& w) {
        load_a(a[1], 2 * s + 1);
        const WideOps o = wide_decode<K2>(w, sh);
        load_w(w, s + 3);
        products(buf, 0, a[0]);
        load_a(a[0], 2 * s + 2);
        products(buf, 1, a[1]);
        wide_put(lds, buf ^ 1, wave, lane, o);
        wide_barrier();
    };
    for (int s = 0; s < chunks; s += 2) {
        stage(s, 0, ring[1]);
        end(s);
        if (s + 1 >= chunks) break;
        stage(s + 1, 1, ring[0]);
        end(s + 1);
    }
}

}  // namespace evamx
