// EXL3 trellis -> fp16 W[k][n] (bit-exact decode).
//
// Reference: exl3_dq.cuh:15-31 (windows), codebook.cuh:86-99 (MUL1), the tile layout of
// exl3_moe_coop_kernel.cuh:377,404 and the fragment map of rocm/ptx_rocm.cuh:11-14.
#include "evamx_gemv.hpp"
#include "evamx_internal.hpp"

namespace evamx {

// Lane-structured decode (the same code the decode GEMV runs), every rate: one wave = 8 consecutive
// tiles of one k-slice; lane = (tile i, q) decodes columns q, q + 8 of tile i for all 16 k. A pair holds
// (k, k + 1) of a column; neighbour lanes swap halves into pairs of columns, which meet in the wave's LDS
// as the slice's 16 rows and leave as 16-byte pieces. Bound by the launch and the rows written
// (7168 x 2048 at 2.5 bpw: 48.4 -> 8.8 us, 3.9 TB/s; one thread a weight at half rates and 2-byte stores at
// the others before).
constexpr int DQ_ROW = 68;            // dwords per staged row: 128 columns, padded

template <int K2>
__global__ __launch_bounds__(256) void dequant_kernel(const uint32_t* __restrict__ trellis, int kt_n, int nt_n,
                                                      half_t* __restrict__ w)
{
    using R = Rate<K2>;
    __shared__ uint32_t rows[4][16 * DQ_ROW];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    const int groups = (nt_n + 7) / 8;
    const int kt = wave / groups, nt0 = 8 * (wave - kt * groups);
    if (kt >= kt_n) return;
    const int q = lane & 7, ti = lane >> 3;
    uint32_t lane_off, sh;
    lane_offsets<K2>(nt0 + ti < nt_n ? lane : q, lane_off, sh);      // past the last tile: tile 0 again, not stored
    LaneWords<R::K> lw;
    load_slice<R::K>(lw, weight_rsrc(trellis + ((size_t)kt * nt_n + nt0) * R::TW), 0, lane_off);
    half2_t wp[16];
    decode_slice<K2, true>(lw, sh, wp);
    uint32_t* dst = rows[threadIdx.x >> 6];
    // wp[4 u + 2 c + kh]: column q + 8 c, k = 8 kh + 2 u and + 1; even lanes keep k of columns q, q + 1,
    // odd lanes k + 1 of columns q - 1, q
    const half2_t k = {__builtin_bit_cast(half_t, (uint16_t)0x1eee), __builtin_bit_cast(half_t, (uint16_t)0x1eee)};
    const half2_t b = {__builtin_bit_cast(half_t, (uint16_t)0xc931), __builtin_bit_cast(half_t, (uint16_t)0xc931)};
    const uint32_t sel = (q & 1) ? 0x03020706u : 0x05040100u;         // (other.hi, own.hi) or (own.lo, other.lo)
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int kh = 0; kh < 2; ++kh) {
                const uint32_t own = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(wp[4 * u + 2 * c + kh], k, b));
                const uint32_t other = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)own, 0xB1, 0xf, 0xf, true);     // lane xor 1
                dst[(8 * kh + 2 * u + (q & 1)) * DQ_ROW + 8 * ti + 4 * c + (q >> 1)] = __builtin_amdgcn_perm(other, own, sel);
            }
    wave_lds_fence();
    const size_t n_out = (size_t)nt_n * 16;
    half_t* base = w + (size_t)(16 * kt) * n_out + 16 * nt0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 4 * i + (lane >> 4), piece = lane & 15;
        const u32x4 v = *(const u32x4*)(dst + r * DQ_ROW + 4 * piece);
        if (nt0 + (piece >> 1) < nt_n) *(u32x4h*)(base + r * n_out + 8 * piece) = u32x4h{v.x, v.y, v.z, v.w};
    }
}

int launch_dequant(const void* trellis, int in, int out, int k2, void* w, hipStream_t stream)
{
    const int kt_n = in / 16, nt_n = out / 16;
    const uint32_t* t = (const uint32_t*)trellis;
    half_t* o = (half_t*)w;
    const long waves = (long)kt_n * ((nt_n + 7) / 8);
    const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
#define EVAMX_DQ_RATE(K2) \
    case K2: hipLaunchKernelGGL(dequant_kernel<K2>, grid, block, 0, stream, t, kt_n, nt_n, o); break
    switch (k2) {
        EVAMX_DQ_RATE(2);
        EVAMX_DQ_RATE(3);
        EVAMX_DQ_RATE(4);
        EVAMX_DQ_RATE(5);
        EVAMX_DQ_RATE(6);
        EVAMX_DQ_RATE(7);
        EVAMX_DQ_RATE(8);
        EVAMX_DQ_RATE(10);
        EVAMX_DQ_RATE(12);
        EVAMX_DQ_RATE(14);
        EVAMX_DQ_RATE(16);
        default: return -1;             // the rate is validated by the caller
    }
#undef EVAMX_DQ_RATE
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace evamx
