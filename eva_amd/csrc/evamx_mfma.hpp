// The MFMA core shared by the prefill-shaped expert GEMMs and the large-row EXL3 linear:
// trellis decode feeding fp16 MFMA on gfx950, in registers.
//
//   - the 64 lanes of a wave take 8 trellis tiles at a time, 8 lanes a tile as in the decode GEMV
//     (lane q of a tile owns its columns q, q + 8 for all 16 k), but 2 tiles across by 4 k-slices
//     down: lane = q + 8 t + 16 g has tile t of a pair at k-slice g. That is the B operand of
//     v_mfma_f32_16x16x32_f16 as it stands (lane n + 16 g holds column n at the k group g): the
//     columns q of both tiles are one operand's 16 columns, the columns q + 8 another's, and the
//     k of an operand is any 8 of a lane's 16 as long as A takes the same. So the decoded
//     (1024 + bytesum) fp16 values of the affine codebook map (w = 0x1eee * h + 0xc931) go from
//     the decode to the matrix cores with no exchange between lanes;
//   - the rotated activations of its rows are the A operands (lane m + 16 g holds row m, 32
//     contiguous bytes of k-slice g), straight from global memory;
//   - MB x 8 accumulators (16 MB rows x 128 columns, fp32) take sum_k x_k h_k; the caller
//     applies the codebook map per column with the rows' activation sums.
#pragma once
#include "evamx_gemv.hpp"

namespace evamx {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// B operand of column c (0: q, 1: q + 8) and k half h of a decoded slice: its pairs hold
// k = 8 h + 2 u, 8 h + 2 u + 1 in wp[4 u + 2 c + h].
__device__ __forceinline__ half8_t mfma_b(const half2_t (&wp)[16], int c, int h)
{
    const u32x4_t v = {__builtin_bit_cast(uint32_t, wp[h + 2 * c]), __builtin_bit_cast(uint32_t, wp[h + 2 * c + 4]),
                       __builtin_bit_cast(uint32_t, wp[h + 2 * c + 8]), __builtin_bit_cast(uint32_t, wp[h + 2 * c + 12])};
    return __builtin_bit_cast(half8_t, v);
}

// Column (of the item's 128) of accumulator nb in a lane: accumulator 2 j + c takes column c (0: q,
// 1: q + 8) of the tiles 2 j and 2 j + 1.
__device__ __forceinline__ int mfma_col(int lane, int nb)
{
    return 32 * (nb >> 1) + 16 * ((lane >> 3) & 1) + 8 * (nb & 1) + (lane & 7);
}

// had128_lane for a row's 128 values in the accumulator layout, value nb at column mfma_col(lane, nb):
// bits 0-2 and 4 of the column are lane bits 0-3, bits 3, 5 and 6 are bits of nb. Same stages in the
// same order, so the results are bit-identical.
__device__ __forceinline__ void had128_acc(float (&v)[8], int lane)
{
#pragma unroll
    for (int nb = 0; nb < 8; ++nb) v[nb] = bfly_x<4>(bfly_x<2>(bfly_x<1>(v[nb], lane), lane), lane);
#pragma unroll
    for (int nb = 0; nb < 8; nb += 2) {
        const float a = v[nb], c = v[nb + 1];
        v[nb] = a + c;
        v[nb + 1] = a - c;
    }
#pragma unroll
    for (int nb = 0; nb < 8; ++nb) v[nb] = bfly_x<8>(v[nb], lane);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int nb = (i & 1) + 4 * (i >> 1);               // nb bit 1: column bit 5
        const float a = v[nb], c = v[nb + 2];
        v[nb] = a + c;
        v[nb + 2] = a - c;
    }
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {                         // nb bit 2: column bit 6
        const float a = v[nb], c = v[nb + 4];
        v[nb] = a + c;
        v[nb + 4] = a - c;
    }
#pragma unroll
    for (int nb = 0; nb < 8; ++nb) v[nb] *= R_SCALE;
}

// Accumulators of one work item: rows [0, rows) (slots slot_of[0..rows)) of activations src
// (fp16 [slot][K] with 128-chunk sums) times the (1024 + bytesum) values of tiles 8*cg .. 8*cg+7
// of a projection over the k-slices [kt0, kt1) (whole 128-chunks): acc[mb][nb][r] = sum_k x_k h_k
// for row 16 mb + 4 g + r and column mfma_col(lane, nb) (lane = m16 + 16 g).
// One row block decodes apart from the products, more interleaved with them (Mul1): fenced, a unit's four
// operands and four blocks' rows are all live at once and spill (3001 tokens 5404 against 5193 us), interleaved
// one block is slower (100 tokens at 3 bpw 1454 against 1410).
template <int K2, int MB>
__device__ __forceinline__ void mfma_accumulate(const uint32_t* __restrict__ trellis, int nt_n, int cg, int kt0, int kt1,
                                                const GlobalRows& src, const int* __restrict__ slot_of, int rows,
                                                f32x4_t (&acc)[MB][8])
{
    using R = Rate<K2>;
    constexpr int K = R::K;
    constexpr int TW = R::TW;
    const int lane = threadIdx.x & 63;
    const int m16 = lane & 15, g = lane >> 4;     // MFMA layout: row/column m16, k group g
    kt0 = __builtin_amdgcn_readfirstlane(kt0);
    const int steps = (__builtin_amdgcn_readfirstlane(kt1) - kt0) >> 2;
    const uint32_t slice = __builtin_amdgcn_readfirstlane(4u * (uint32_t)(nt_n * TW));
    const uint32_t cbase = __builtin_amdgcn_readfirstlane(4u * (uint32_t)(cg * 8 * TW) + (uint32_t)kt0 * slice);
    const __amdgpu_buffer_rsrc_t rsrc = weight_rsrc(trellis);
    uint32_t lane_off, sh;
    lane_offsets<K2>(lane & 15, lane_off, sh);     // tile (lane >> 3) & 1 of the pair
    lane_off += (uint32_t)g * slice;

    // A rows of this lane: m16 + 16 mb (rows past the tile read row 0; their results are dropped)
    const __attribute__((address_space(1))) u32x4_t* arow[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const int r = m16 + 16 * mb;
        const int s = slot_of[r < rows ? r : 0];
        arow[mb] = (const __attribute__((address_space(1))) u32x4_t*)(src.A + (size_t)s * src.stride + 16 * kt0) + 2 * g;
    }

#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) acc[mb][nb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    LaneWords<K> ring[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) load_slice<K>(ring[j], rsrc, cbase + (uint32_t)(8 * j * TW), lane_off);

    u32x4_t a[MB][2];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int h = 0; h < 2; ++h) a[mb][h] = arow[mb][h];

    for (int kk = 0; kk < steps; ++kk) {
        progress_priority(kk, steps);
        // the next step's A operands and weights, clamped to the last step (in bounds, unused)
        const int kn = kk + 1 < steps ? kk + 1 : kk;
        u32x4_t an[MB][2];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int h = 0; h < 2; ++h) an[mb][h] = arow[mb][8 * kn + h];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            half2_t wp[16];
            decode_slice<K2, MB == 1>(ring[j], sh, wp);
            load_slice<K>(ring[j], rsrc, cbase + (uint32_t)(4 * kn) * slice + (uint32_t)(8 * j * TW), lane_off);
            if constexpr (MB == 1) mfma_begin();
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const half8_t b = mfma_b(wp, c, h);
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb)
                        acc[mb][2 * j + c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a[mb][h]), b,
                                                                                    acc[mb][2 * j + c], 0, 0, 0);
                }
            if constexpr (MB == 1) mfma_end<4>();
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int h = 0; h < 2; ++h) a[mb][h] = an[mb][h];
    }
    progress_priority(1, 1);
}

// Activations laid out as A operands: a block of 16 rows is, for each k64 step t and k half h, the 64
// lanes' 16 bytes in lane order (row m16, k = 64 t + 16 g + 8 h ..), 1 KiB a load. Read from plain rows
// instead, the lanes of a load lie in 16 rows and each takes an address cycle of its own, four times the
// load's data cycles (64 rows, 7168 x 2048: 115 us a call, all of it these loads). Byte offset of the
// block with row 16 b, K columns.
__host__ __device__ __forceinline__ size_t a_operand_offset(int b, int K) { return (size_t)b * 16 * K * 2; }

// The same products for one pair of tiles (32 columns) over `chunks` 128-chunks of k: acc[mb][c][r] +=
// for row 16 mb + 4 g + r and column mfma_col(lane, c) of the pair, rows at arow[mb] (the lane's k-slice
// group g). pair: the pair's index among the projection's column tiles. Weights three steps of 64 k in
// flight, activations two. end(i) runs after chunk i.
template <int K2, int MB, typename End>
__device__ __forceinline__ void mfma_pair(const uint32_t* __restrict__ trellis, int nt_n, int pair, int kt0, int chunks,
                                          const __attribute__((address_space(1))) u32x4_t* const (&arow)[MB], f32x4_t (&acc)[MB][2],
                                          End&& end)
{
    using R = Rate<K2>;
    constexpr int K = R::K;
    constexpr int TW = R::TW;
    const int lane = threadIdx.x & 63;
    const int last = 2 * chunks - 1;
    const uint32_t slice = __builtin_amdgcn_readfirstlane(4u * (uint32_t)(nt_n * TW));
    const uint32_t cbase = __builtin_amdgcn_readfirstlane(4u * (uint32_t)(2 * pair * TW) + (uint32_t)kt0 * slice);
    const __amdgpu_buffer_rsrc_t rsrc = weight_rsrc(trellis);
    uint32_t lane_off, sh;
    lane_offsets<K2>(lane & 15, lane_off, sh);
    lane_off += (uint32_t)(lane >> 4) * slice;
    LaneWords<K> ring[3];
    u32x4_t a[3][MB][2];
    auto load_w = [&](LaneWords<K>& w, int t) { load_slice<K>(w, rsrc, cbase + (uint32_t)(4 * min(t, last)) * slice, lane_off); };
    auto load_a = [&](u32x4_t (&d)[MB][2], int t) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int h = 0; h < 2; ++h) d[mb][h] = arow[mb][128 * min(t, last) + 64 * h];
    };
    auto step = [&](int t, LaneWords<K>& w, const u32x4_t (&x)[MB][2], u32x4_t (&y)[MB][2]) {
        load_a(y, t + 2);
        __builtin_amdgcn_sched_barrier(0);        // the loads first
        half2_t wp[16];
        decode_slice<K2, false>(w, sh, wp);
        load_w(w, t + 3);
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const half8_t b = mfma_b(wp, c, h);
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
                    acc[mb][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, x[mb][h]), b, acc[mb][c], 0, 0, 0);
            }
    };
#pragma unroll
    for (int d = 0; d < 3; ++d) load_w(ring[d], d);
    load_a(a[0], 0);
    load_a(a[1], 1);
    for (int i = 0; i < chunks; i += 3) {
        step(2 * i, ring[0], a[0], a[2]);
        step(2 * i + 1, ring[1], a[1], a[0]);
        end(i);
        if (i + 1 >= chunks) break;
        step(2 * i + 2, ring[2], a[2], a[1]);
        step(2 * i + 3, ring[0], a[0], a[2]);
        end(i + 1);
        if (i + 2 >= chunks) break;
        step(2 * i + 4, ring[1], a[1], a[0]);
        step(2 * i + 5, ring[2], a[2], a[1]);
        end(i + 2);
    }
}

// Activation sums over the k-slices [kt0, kt0 + nk) of the rows whose accumulators a lane holds:
// xs[mb][r] for row 16 mb + 4 g + r (lane = m16 + 16 g). Lane (m16, g) first sums chunks c0 + g,
// c0 + g + 4, ... of row m16 + 16 mb; the four k groups are summed across lanes; then each
// lane fetches the sums of its output rows.
template <int MB>
__device__ __forceinline__ void mfma_row_sums(const GlobalRows& src, const int* __restrict__ slot_of, int rows, int kt0,
                                              int nk, float (&xs)[MB][4])
{
    const int lane = threadIdx.x & 63;
    const int m16 = lane & 15, g = lane >> 4;
    const int c0 = kt0 >> 3, c1 = c0 + (nk >> 3);
    float v[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const int r = m16 + 16 * mb;
        const int s = slot_of[r < rows ? r : 0];
        float t = strided_sum<8>(src.sums + (size_t)s * src.sums_stride, c0 + g, c1, 4);
        t = pair_sum<16>(t, lane);
        t = pair_sum<32>(t, lane);
        v[mb] = t;
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int r = 0; r < 4; ++r) xs[mb][r] = __shfl(v[mb], 4 * g + r, WAVE);
}

// One work item with its partials stored: part[slot * part_stride + 128 * cg + column] =
// 0x1eee * acc + 0xc931 * (row's activation sum), for rows < rows.
template <int K2, int MB>
__device__ __forceinline__ void mfma_item(const uint32_t* __restrict__ trellis, int nt_n, int cg, int kt0, int kt1,
                                          const GlobalRows& src, const int* __restrict__ slot_of, int rows,
                                          float* __restrict__ part, size_t part_stride)
{
    f32x4_t acc[MB][8];
    mfma_accumulate<K2, MB>(trellis, nt_n, cg, kt0, kt1, src, slot_of, rows, acc);
    kt0 = __builtin_amdgcn_readfirstlane(kt0);
    const int nk = __builtin_amdgcn_readfirstlane(kt1) - kt0;
    float xs[MB][4];
    mfma_row_sums<MB>(src, slot_of, rows, kt0, nk, xs);
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * mb + 4 * g + r;
            if (row < rows) {
                float* dst = part + (size_t)slot_of[row] * part_stride + 128 * cg;
#pragma unroll
                for (int nb = 0; nb < 8; ++nb) dst[mfma_col(lane, nb)] = mul1_affine(acc[mb][nb][r], xs[mb][r]);
            }
        }
    }
}

}  // namespace evamx
