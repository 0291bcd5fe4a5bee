// Single EXL3 linear, fp16 in / fp16 out (the config-1 layer).
//
// Reference: ELinear.forward -> LinearEXL3 (runtime/ds41/exl3_linear.py:97-131), kernel
// exl3_gemv_kernel.cuh:217-234 (input: fp16 x*suh, Hadamard, fp16), 295-459 (GEMV, fp16 C),
// 463-490 with hadamard_inner.cuh:93-147 (output Hadamard to fp16, fp16 product with svh).
// Up to 2 rows, one launch: a k-split decode GEMV whose waves rotate their own input chunks
// (fp16(H128(fp16(x * suh)))) into LDS while their first weight loads are in flight, writing fp32
// partials; the workgroup that arrives last at its column group's counter then runs that group's
// output epilogue (the partials summed in fixed split order, fp16 C, Hadamard, fp16 svh product).
// 3 to 16 rows, three launches: the input rotation, the same GEMV on the rotated rows, and the
// same epilogue in a launch of its own.
// More rows: the input rotation, written as MFMA operands, then one of three MFMA kernels by size
// (linear_kind): 256-row workgroups that share each decoded weight (lin_wide_kernel), 64-row
// workgroups over the whole k range, or over one k-range each with the output epilogue in a launch
// of its own. All add the same k-ranges' sums in the same order. In both paths (up to
// LIN_GEMV_ROWS rows, and beyond) a row's arithmetic depends on in/out only, not on how many rows
// share the call.
#include "evamx_internal.hpp"
#include "evamx_wide.hpp"

namespace evamx {


__constant__ int k_iota64[64] = {0,  1,  2,  3,  4,  5,  6,  7,  8,  9,  10, 11, 12, 13, 14, 15,
                                 16, 17, 18, 19, 20, 21, 22, 23, 24, 25, 26, 27, 28, 29, 30, 31,
                                 32, 33, 34, 35, 36, 37, 38, 39, 40, 41, 42, 43, 44, 45, 46, 47,
                                 48, 49, 50, 51, 52, 53, 54, 55, 56, 57, 58, 59, 60, 61, 62, 63};

constexpr int LIN_GEMV_ROWS = 16;     // decode GEMV up to this many rows, MFMA tiles beyond
constexpr int LIN_ROT_ROWS = 2;       // the GEMV rotates its own inputs up to this many rows
// Weight prefetch depth of the 1-2 row GEMV: its waves stream 8 k-slices each at 2048 x 7168,
// one wave per SIMD; 3 slices in flight measured best (2: 7.58, 3: 6.84, 4: 6.98,
// 5: 7.07 us per call; the MoE's longer items keep 4).
constexpr int LIN_PF = 3;

struct LinParams {
    const half_t* x;
    int rows, in, out, k2, ks;
    const uint32_t* trellis;
    const half_t* suh;
    const half_t* svh;
    half_t* y;
    half_t* xr;        // [rows][in]
    float* xsum;       // [rows][in/128]
    float* part;       // [ks][rows][out]
    unsigned long long* arrive;   // arrival counters of the decode path, one per ARRIVE_STRIDE words
};

// Rotated inputs of tm rows (rows r0 .. r0 + tm - 1 of x) over the 128-chunks [w0, w1) into
// the wave's LDS rows (row m at dst + m * LIN_CW * 64 words, chunk w0 + j at word 64 j), with
// each row's chunk sums added in chunk order; the same operations as lin_rotate_kernel, so the
// rows are bit-identical to its output. issue() loads the x and suh words before the weight
// prefetch ring, finish() rotates them once the ring is in flight.
constexpr int LIN_CW = 4;             // 128-chunks per LDS window

template <int TM>
struct LinRot {
    static constexpr bool kWork = true;
    const LinParams& p;
    int tm, w0, w1, lane;
    __amdgpu_buffer_rsrc_t xrs[TM], srs;
    uint32_t* dst;
    float (&xs)[TM];
    uint32_t xv[TM][LIN_CW], sv[LIN_CW];

    __device__ __forceinline__ void issue()
    {
        // chunks past the window reload its last one (in bounds, unused): no branches
#pragma unroll
        for (int j = 0; j < LIN_CW; ++j)
            sv[j] = __builtin_amdgcn_raw_buffer_load_b32(srs, 4 * lane, 256 * min(w0 + j, w1 - 1), 0);
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
            for (int j = 0; j < LIN_CW; ++j)
                xv[m][j] = __builtin_amdgcn_raw_buffer_load_b32(xrs[m], 4 * lane, 256 * min(w0 + j, w1 - 1), 0);
    }
    __device__ __forceinline__ void finish()
    {
#pragma unroll
        for (int m = 0; m < TM; ++m) {
            if (m >= tm) continue;
#pragma unroll
            for (int j = 0; j < LIN_CW; ++j) {
                if (w0 + j < w1) {
                    const half2_t xx = __builtin_bit_cast(half2_t, xv[m][j]);
                    const half2_t su = __builtin_bit_cast(half2_t, sv[j]);
                    float v0 = h2f(f2h(h2f(xx.x) * h2f(su.x)));      // fp16 product
                    float v1 = h2f(f2h(h2f(xx.y) * h2f(su.y)));
                    had128_pair(v0, v1, lane);
                    const half2_t r = {f2h(v0), f2h(v1)};
                    dst[m * LIN_CW * 64 + j * 64 + lane] = __builtin_bit_cast(uint32_t, r);
                    xs[m] += wave_sum(h2f(r.x) + h2f(r.y));
                }
            }
        }
        wave_lds_fence();
    }
};

template <int K2, int TM>
__device__ __forceinline__ void lin_rows(const LinParams& p, int r0, int tm, int cg, int ks, int c0, int c1, uint32_t* lds)
{
    const int lane = threadIdx.x & 63;
    __amdgpu_buffer_rsrc_t xrs[TM];
#pragma unroll
    for (int m = 0; m < TM; ++m) xrs[m] = weight_rsrc((const uint32_t*)(p.x + (size_t)(r0 + (m < tm ? m : 0)) * p.in));
    const __amdgpu_buffer_rsrc_t srs = weight_rsrc((const uint32_t*)p.suh);
    float acc[TM][2], xs[TM];
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[m][0] = acc[m][1] = xs[m] = 0.0f;
    auto window = [&](int w0, int w1) {
        const XLds src{lds, LIN_CW * 64, 8 * w0};
        LinRot<TM> stage{p, tm, w0, w1, lane, {}, srs, lds, xs};
#pragma unroll
        for (int m = 0; m < TM; ++m) stage.xrs[m] = xrs[m];
        gemv_wave<K2, TM, LIN_PF>(p.trellis, p.out / 16, cg, 8 * w0, 8 * w1, src, tm, acc, stage);
    };
    if (c1 - c0 <= LIN_CW) {
        window(c0, c1);
    } else {
        for (int w0 = c0; w0 < c1; w0 += LIN_CW) {
            window(w0, min(c1, w0 + LIN_CW));
            wave_lds_fence();           // this window's reads before the next window's writes
        }
    }
    const int col0 = cg * 128 + lane_col(lane, 0), col1 = cg * 128 + lane_col(lane, 1);
#pragma unroll
    for (int m = 0; m < TM; ++m) {
        if (m < tm) {
            float* dst = p.part + ((size_t)ks * p.rows + r0 + m) * p.out;
            store_wt(dst + col0, mul1_affine(acc[m][0], xs[m]));
            store_wt(dst + col1, mul1_affine(acc[m][1], xs[m]));
        }
    }
}

template <int K2, int TM>
__device__ __forceinline__ void lin_item(const LinParams& p, int cg, int ks, int c0, int c1, uint32_t* lds)
{
    if constexpr (TM == 1) lin_rows<K2, 1>(p, 0, 1, cg, ks, c0, c1, lds);
    else lin_rows<K2, 2>(p, 0, p.rows, cg, ks, c0, c1, lds);
}

// Partials of 16 splits for the lane's two columns (byte offsets vo and vo + 32 in rs, splits sb
// bytes apart from split q0 on), the loads all issued before the adds; splits from `valid` on are
// loaded clamped and not added. POL LD_SC1: the loads read the memory side, where the other
// workgroups' write-through stores went; buffer loads take the split offsets in scalar registers,
// so no vector instruction computes an address.

template <bool FULL, int POL>
__device__ __forceinline__ void lin_sum16(__amdgpu_buffer_rsrc_t rs, uint32_t vo, uint32_t sb, int q0, int valid,
                                          float& v0, float& v1)
{
    float t0[16], t1[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const uint32_t so = sb * (uint32_t)(q0 + (FULL ? i : min(i, valid - 1)));
        t0[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, vo, so, POL));
        t1[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, vo + 32, so, POL));
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
        if (FULL || i < valid) {
            v0 += t0[i];
            v1 += t1[i];
        }
}

// Output epilogue of row m of a column group: the row's k-split partials summed in split order
// (one memory round trip per 16 splits), C to fp16, Hadamard, fp16 svh product. POL: LD_SC1 in
// the launch that wrote the partials (run by the group's last workgroup after its arrival, where
// every instruction is on the call's critical path), 0 in a launch of its own.
template <int POL>
__device__ __forceinline__ void lin_epilogue_row(const LinParams& p, int cg, int m, const float (&sv)[2])
{
    const int lane = threadIdx.x & 63;
    const __amdgpu_buffer_rsrc_t rs = weight_rsrc((const uint32_t*)p.part);
    const uint32_t vo = 4u * (uint32_t)(m * p.out + cg * 128 + lane_col(lane, 0));   // column 1: + 32 bytes
    const uint32_t sb = 4u * (uint32_t)(p.rows * p.out);
    float v0 = 0.0f, v1 = 0.0f;
    for (int q0 = 0; q0 < p.ks; q0 += 16) {
        if (q0 + 16 <= p.ks) lin_sum16<true, POL>(rs, vo, sb, q0, 16, v0, v1);
        else lin_sum16<false, POL>(rs, vo, sb, q0, p.ks - q0, v0, v1);
    }
    v0 = h2f(f2h(v0));                  // C in fp16
    v1 = h2f(f2h(v1));
    had128_lane(v0, v1, lane);
    half_t* y = p.y + (size_t)m * p.out + cg * 128 + lane_col(lane, 0);
    y[0] = f2h(h2f(f2h(v0)) * sv[0]);
    y[8] = f2h(h2f(f2h(v1)) * sv[1]);
}

// After a workgroup's waves stored their partials: wait until every store is acknowledged, arrive
// at the column group's counter, and run the epilogue if last (the stores of every workgroup of
// the group then precede the loads). One row: wave 0 arrives and runs the epilogue alone, with no
// second barrier; two: the arrival is shared through LDS and wave m runs row m.
template <int TM>
__device__ __forceinline__ void lin_arrive(const LinParams& p, int cg, int n, const float (&sv)[2])
{
    unsigned long long* word = p.arrive + (size_t)cg * ARRIVE_STRIDE;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if constexpr (TM == 1) {
        if (wave != 0) return;
        int l = 0;
        if (threadIdx.x == 0) l = arrive_last(word, (unsigned)n);
        if (__builtin_amdgcn_readfirstlane(l)) lin_epilogue_row<LD_SC1>(p, cg, 0, sv);
    } else {
        __shared__ int last;
        if (threadIdx.x == 0) last = arrive_last(word, (unsigned)n);
        __syncthreads();
        if (last && wave < p.rows) lin_epilogue_row<LD_SC1>(p, cg, wave, sv);
    }
}

// The lane's two svh values, loaded at the start of the launch (the epilogue needs them only in
// the last workgroup, but then without waiting for them).
__device__ __forceinline__ void lin_load_sv(const LinParams& p, int cg, float (&sv)[2])
{
    const int lane = threadIdx.x & 63;
    sv[0] = h2f(p.svh[cg * 128 + lane_col(lane, 0)]);
    sv[1] = h2f(p.svh[cg * 128 + lane_col(lane, 1)]);
}

// Decode path: one workgroup of four waves per (128 output columns, quarter q of the k-splits),
// wave w taking split 4q + w (waves past the last split only arrive); each row's reduction order
// depends only on in/out, never on how many rows share the call. One kernel per rate (the host
// picks it). TM (1 or 2) rows: inputs rotated in the wave.
template <int K2, int TM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void lin_gemv_kernel(LinParams p)
{
    __shared__ uint32_t xl[4][TM * LIN_CW * 64];
    const int nq = (p.ks + 3) >> 2;
    const int cg = blockIdx.x / nq, q = blockIdx.x % nq;
    const int ks = __builtin_amdgcn_readfirstlane(4 * q + (threadIdx.x >> 6));
    float sv[2];
    lin_load_sv(p, cg, sv);
    if (ks < p.ks) {
        const int nch = p.in / 128;
        const int c0 = nch * ks / p.ks, c1 = nch * (ks + 1) / p.ks;
        lin_item<K2, TM>(p, cg, ks, c0, c1, xl[threadIdx.x >> 6]);
    }
    lin_arrive<TM>(p, cg, nq, sv);
}

// 3 to LIN_GEMV_ROWS rows: the rows rotated beforehand (lin_rotate_kernel), read through
// scalar loads (wider row blocks in LDS would not fit the register budget); one wave per (128
// output columns, k-split), the output epilogue in a launch of its own (lin_epilogue_kernel). At
// these row counts the last workgroup of a column group would run many rows' epilogues one after
// another (16 rows at 2048 x 7168: 38.6 us per call, against 32.1 us with the epilogue launch).
template <int K2, int TMAX>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void lin_gemv_rows_kernel(LinParams p)
{
    const int wid = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    const int ncg = p.out / 128;
    if (wid >= ncg * p.ks) return;
    const int cg = __builtin_amdgcn_readfirstlane(wid / p.ks), ks = __builtin_amdgcn_readfirstlane(wid % p.ks);
    const int nch = p.in / 128;
    const int c0 = nch * ks / p.ks, c1 = nch * (ks + 1) / p.ks;
    gemv_chunk<K2, TMAX>(p.trellis, p.out / 16, cg, c0, c1, GlobalRows{p.xr, (size_t)p.in, p.xsum, nch}, k_iota64,
                         p.rows, p.part + (size_t)ks * p.rows * p.out, (size_t)p.out);
}

// One wave per (row, 128 output columns).
__global__ __launch_bounds__(256) void lin_epilogue_kernel(LinParams p)
{
    const int wid = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    const int ncg = p.out / 128;
    if (wid >= ncg * p.rows) return;
    const int m = wid / ncg, cg = wid % ncg;
    float sv[2];
    lin_load_sv(p, cg, sv);
    lin_epilogue_row<0>(p, cg, m, sv);
}

// Decode path launches of one rate: up to 2 rows one launch (workgroups per (column group, 4
// splits)); 3 to 16 rows the GEMV (a wave per (column group, split)) and the epilogue.
template <int K2>
void launch_gemv_rate(const LinParams& p, hipStream_t stream)
{
    const int ncg = p.out / 128;
    if (p.rows <= LIN_ROT_ROWS) {
        const dim3 grid((unsigned)(ncg * ((p.ks + 3) / 4)));
        if (p.rows == 1) hipLaunchKernelGGL((lin_gemv_kernel<K2, 1>), grid, dim3(256), 0, stream, p);
        else hipLaunchKernelGGL((lin_gemv_kernel<K2, 2>), grid, dim3(256), 0, stream, p);
        return;
    }
    const dim3 grid((unsigned)((ncg * p.ks + 3) / 4));
    if (p.rows <= 4) hipLaunchKernelGGL((lin_gemv_rows_kernel<K2, 4>), grid, dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((lin_gemv_rows_kernel<K2, 8>), grid, dim3(256), 0, stream, p);
    hipLaunchKernelGGL(lin_epilogue_kernel, dim3((unsigned)((ncg * p.rows + 3) / 4)), dim3(256), 0, stream, p);
}

// ---------------------------------------------------------------------------------------------
// More than LIN_GEMV_ROWS rows (and the rotation of 3 to LIN_GEMV_ROWS rows).

constexpr int LIN_RANGES = 8;         // k-ranges whose sums are added in order

// fp16(H128(fp16(x * suh))) of every (row, 128-chunk) with the chunk's sum: one wave each.
__global__ __launch_bounds__(256) void lin_rotate_kernel(LinParams p)
{
    const int lane = threadIdx.x & 63;
    const int item = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    const int nch = p.in / 128;
    if (item >= p.rows * nch) return;
    const int r = item / nch, c = item % nch;
    const uint32_t xw = ((const uint32_t*)(p.x + (size_t)r * p.in + c * 128))[lane];
    const uint32_t sw = ((const uint32_t*)(p.suh + c * 128))[lane];
    const half2_t xx = __builtin_bit_cast(half2_t, xw), su = __builtin_bit_cast(half2_t, sw);
    float v0 = h2f(f2h(h2f(xx.x) * h2f(su.x)));        // fp16 product
    float v1 = h2f(f2h(h2f(xx.y) * h2f(su.y)));
    had128_pair(v0, v1, lane);
    const half2_t o = {f2h(v0), f2h(v1)};
    ((uint32_t*)(p.xr + (size_t)r * p.in + c * 128))[lane] = __builtin_bit_cast(uint32_t, o);
    const float sum = wave_sum(h2f(o.x) + h2f(o.y));
    if (lane == 0) p.xsum[(size_t)r * nch + c] = sum;
}

// The same rotations for calls of more than LIN_GEMV_ROWS rows, written as A operands
// (a_operand_offset): one workgroup per (16 rows, 128-chunk), each wave four rows, which meet in LDS and
// leave as the chunk's 4 KiB. Rows past the call's are zero.
__global__ __launch_bounds__(256) void lin_rotate16_kernel(LinParams p)
{
    __shared__ half_t sh[16][136];                       // padded rows
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nch = p.in / 128;
    const int b = blockIdx.x / nch, c = blockIdx.x % nch;
    const half2_t su = __builtin_bit_cast(half2_t, ((const uint32_t*)(p.suh + c * 128))[lane]);
    uint32_t xw[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        xw[i] = ((const uint32_t*)(p.x + (size_t)min(16 * b + 4 * wave + i, p.rows - 1) * p.in + c * 128))[lane];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 16 * b + 4 * wave + i;
        const half2_t xx = __builtin_bit_cast(half2_t, xw[i]);
        float v0 = h2f(f2h(h2f(xx.x) * h2f(su.x)));      // fp16 product
        float v1 = h2f(f2h(h2f(xx.y) * h2f(su.y)));
        had128_pair(v0, v1, lane);
        const half2_t o = {f2h(v0), f2h(v1)};
        *(uint32_t*)&sh[4 * wave + i][2 * lane] = r < p.rows ? __builtin_bit_cast(uint32_t, o) : 0u;
        const float sum = wave_sum(h2f(o.x) + h2f(o.y));
        if (lane == 0 && r < p.rows) p.xsum[(size_t)r * nch + c] = sum;
    }
    __syncthreads();
    // thread -> operand (k64 step wave >> 1, half wave & 1), lane
    const int m16 = lane & 15, g = lane >> 4;
    const u32x4_t v = *(const u32x4_t*)&sh[m16][64 * (wave >> 1) + 16 * g + 8 * (wave & 1)];
    ((u32x4_t*)((char*)p.xr + a_operand_offset(b, p.in)))[(4 * c + wave) * 64 + lane] = v;
}

// Activation sum of a row: its 128-chunk sums, lane l those of chunks l, l + 64, ..., then the wave's
// butterfly. Every kernel for more than LIN_GEMV_ROWS rows takes it (and the k-ranges' sums in range
// order), so a row's result does not depend on which of them its call runs.
__device__ __forceinline__ float lin_row_total(const LinParams& p, int row)
{
    const int nch = p.in / 128;
    return wave_sum(strided_sum<2>(p.xsum + (size_t)row * nch, threadIdx.x & 63, nch, 64));
}

// Output epilogue of a row's 128 accumulated columns (the lane's two): codebook map, C in fp16, Hadamard,
// fp16 svh product.
__device__ __forceinline__ void lin_store_row(const LinParams& p, int row, int cg, float v0, float v1, float xs, const float (&sv)[2])
{
    const int lane = threadIdx.x & 63;
    v0 = h2f(f2h(mul1_affine(v0, xs)));
    v1 = h2f(f2h(mul1_affine(v1, xs)));
    had128_lane(v0, v1, lane);
    half_t* y = p.y + (size_t)row * p.out + cg * 128 + lane_col(lane, 0);
    y[0] = f2h(h2f(f2h(v0)) * sv[0]);
    y[8] = f2h(h2f(f2h(v1)) * sv[1]);
}

// Calls of more than LIN_GEMV_ROWS rows with too few wide tiles to fill the device: one workgroup per
// tile of up to 64 rows and 128 output columns, wave j taking the pair j of the group's tiles, whose
// decoded weights stay in its registers. The waves read the same activations, which the CU's cache
// serves. SPLIT: a workgroup takes one k-range and stores its accumulators as partials
// (lin_mid_epilogue_kernel adds the ranges); otherwise all of them, added in order, and the output
// epilogue meets in LDS.
constexpr int LM_ROWS = 64;
constexpr int LM_WAVES = 4;

template <int K2, int MB, bool SPLIT>
__device__ __forceinline__ void lin_mid_tile(const LinParams& p, int r0, int rows, int cg, int range, float (*red)[132])
{
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int g = lane >> 4;
    const int nch = p.in / 128;
    const int c0 = SPLIT ? nch * range / p.ks : 0, c1 = SPLIT ? nch * (range + 1) / p.ks : nch;
    const __attribute__((address_space(1))) u32x4_t* arow[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
        arow[mb] = (const __attribute__((address_space(1))) u32x4_t*)((const char*)p.xr + a_operand_offset(r0 / 16 + mb, p.in)) + 256 * c0 + lane;
    f32x4_t acc[MB][2], tot[MB][2];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int c = 0; c < 2; ++c) acc[mb][c] = tot[mb][c] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    int n = 0, stop = nch / p.ks;                                // the chunk after the range's last
    mfma_pair<K2, MB>(p.trellis, p.out / 16, 4 * cg + wave, 8 * c0, c1 - c0, arow, acc, [&](int i) {
        if (SPLIT || i + 1 != stop) return;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                tot[mb][c] += acc[mb][c];
                acc[mb][c] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            }
        ++n;
        stop = nch * (n + 1) / p.ks;
    });
    float* part = SPLIT ? p.part + ((size_t)range * p.rows + r0) * p.out + 128 * cg + 32 * wave : nullptr;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * mb + 4 * g + r;
            if (row < rows) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    if constexpr (SPLIT) part[(size_t)row * p.out + mfma_col(lane, c)] = acc[mb][c][r];
                    else red[row][32 * wave + mfma_col(lane, c)] = tot[mb][c][r];
                }
            }
        }
    if constexpr (!SPLIT) {
        __syncthreads();
        float sv[2];
        lin_load_sv(p, cg, sv);
        for (int row = wave; row < rows; row += LM_WAVES) {
            const float xs = lin_row_total(p, r0 + row);
            lin_store_row(p, r0 + row, cg, red[row][lane_col(lane, 0)], red[row][lane_col(lane, 1)], xs, sv);
        }
    }
}

template <int K2, bool SPLIT>
__global__ __launch_bounds__(64 * LM_WAVES) __attribute__((amdgpu_waves_per_eu(2))) void lin_mid_kernel(LinParams p)
{
    __shared__ float red[SPLIT ? 1 : LM_ROWS][132];              // padded rows
    // ranges fastest: the workgroups of a tile and column group run side by side
    const int nr = SPLIT ? p.ks : 1;
    const int range = blockIdx.x % nr, rest = blockIdx.x / nr, ncg = p.out / 128;
    const int r0 = rest / ncg * LM_ROWS, cg = rest % ncg;
    const int rows = min(LM_ROWS, p.rows - r0);
    switch (__builtin_amdgcn_readfirstlane((rows + 15) >> 4)) {
        case 1: lin_mid_tile<K2, 1, SPLIT>(p, r0, rows, cg, range, red); break;
        case 2: lin_mid_tile<K2, 2, SPLIT>(p, r0, rows, cg, range, red); break;
        case 3: lin_mid_tile<K2, 3, SPLIT>(p, r0, rows, cg, range, red); break;
        default: lin_mid_tile<K2, 4, SPLIT>(p, r0, rows, cg, range, red); break;
    }
}

// One wave per (row, 128 output columns): the ranges' accumulators added in range order, the codebook
// map, C in fp16, Hadamard, fp16 svh product.
__global__ __launch_bounds__(256) void lin_mid_epilogue_kernel(LinParams p)
{
    const int wid = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    const int ncg = p.out / 128;
    if (wid >= ncg * p.rows) return;
    const int m = wid / ncg, cg = wid % ncg, lane = threadIdx.x & 63;
    float sv[2];
    lin_load_sv(p, cg, sv);
    const float* src = p.part + (size_t)m * p.out + cg * 128 + lane_col(lane, 0);
    const size_t stride = (size_t)p.rows * p.out;
    float t[LIN_RANGES][2];
#pragma unroll
    for (int i = 0; i < LIN_RANGES; ++i) {
        const float* q = src + (size_t)min(i, p.ks - 1) * stride;
        t[i][0] = q[0];
        t[i][1] = q[8];
    }
    const float xs = lin_row_total(p, m);
    float v0 = t[0][0], v1 = t[0][1];
#pragma unroll
    for (int i = 1; i < LIN_RANGES; ++i)
        if (i < p.ks) {
            v0 += t[i][0];
            v1 += t[i][1];
        }
    lin_store_row(p, m, cg, v0, v1, xs, sv);
}

// Calls of many rows: one workgroup per (256 rows, 128 output columns) over the whole k range, its
// weights decoded once for the 256 rows (evamx_wide.hpp). Bound by the matrix cores and what feeds them:
// the products alone take two thirds of its time at 8192 rows, without the decode it is 5% faster.
// 2048 -> 7168 at 4 bpw, 8192 rows: 950 -> 356 us a call with its rotation (256 -> 676 TFLOP/s). The accumulators of the k-ranges that
// lin_mid_kernel splits over workgroups are added in the same order, so the two give a row the same bits.
// The epilogue runs on the accumulators where they are: a row's 128 columns lie on 16 lanes, whose
// exchanges stay in a DPP row; the fp16 rows leave through LDS as whole 16-byte pieces.
// Workgroup -> (row tile, column group). Workgroups are dispatched to the 8 XCDs round robin; each XCD
// takes a contiguous share of the items, ordered by blocks of LW_GROUP row tiles with the tiles
// fastest, so that the workgroups resident together on an XCD share LW_GROUP tiles' activations and a
// few column groups' weights in its L2.
constexpr int LW_GROUP = 4;
__device__ __forceinline__ void lin_wide_item(int b, int nb, int tiles, int ncg, int& tile, int& cg)
{
    const int per = nb >> 3, rest = nb & 7, x = b & 7;
    const int item = x * per + min(x, rest) + (b >> 3);
    const int blk = item / (LW_GROUP * ncg), r = item - blk * LW_GROUP * ncg;
    const int n = min(LW_GROUP, tiles - blk * LW_GROUP);
    cg = r / n;
    tile = blk * LW_GROUP + r % n;
}

constexpr int LW_MB = 2;
constexpr int LW_WAVES = 8;
constexpr int LW_ROWS = 16 * LW_MB * LW_WAVES;
constexpr int LW_STRIDE = 136;                       // halves per staged output row (padded)

template <int K2>
__global__ __launch_bounds__(64 * LW_WAVES) __attribute__((amdgpu_waves_per_eu(2))) void lin_wide_kernel(LinParams p)
{
    __shared__ union {
        WideLds<LW_WAVES> w;
        half_t y[LW_WAVES][16 * LW_MB][LW_STRIDE];
    } lds;
    __shared__ float xs[LW_WAVES][16 * LW_MB];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int g = lane >> 4;
    const int ncg = p.out / 128, nch = p.in / 128;
    int tile, cg;
    lin_wide_item(blockIdx.x, gridDim.x, (p.rows + LW_ROWS - 1) / LW_ROWS, ncg, tile, cg);
    const int r0 = tile * LW_ROWS + 16 * LW_MB * wave;
    const __attribute__((address_space(1))) u32x4_t* arow[LW_MB];
#pragma unroll
    for (int mb = 0; mb < LW_MB; ++mb)                           // blocks past the call's: not stored
        arow[mb] = (const __attribute__((address_space(1))) u32x4_t*)((const char*)p.xr + a_operand_offset(min(r0 / 16 + mb, (p.rows - 1) / 16), p.in)) + lane;
    f32x4_t acc[LW_MB][8], tot[LW_MB][8];
#pragma unroll
    for (int mb = 0; mb < LW_MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) acc[mb][nb] = tot[mb][nb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    int range = 0, stop = nch / p.ks;                            // the chunk after the range's last
    wide_accumulate<K2, LW_MB, LW_WAVES>(p.trellis, p.out / 16, cg, 0, nch, arow, lds.w, acc, [&](int c) {
        if (c + 1 != stop) return;
#pragma unroll
        for (int mb = 0; mb < LW_MB; ++mb)
#pragma unroll
            for (int nb = 0; nb < 8; ++nb) {
                tot[mb][nb] += acc[mb][nb];
                acc[mb][nb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            }
        ++range;
        stop = nch * (range + 1) / p.ks;
    });
    for (int i = 0; i < 16 * LW_MB; ++i) {
        const float t = lin_row_total(p, min(r0 + i, p.rows - 1));
        if (lane == 0) xs[wave][i] = t;
    }
    float sv[8];
#pragma unroll
    for (int nb = 0; nb < 8; ++nb) sv[nb] = h2f(p.svh[cg * 128 + mfma_col(lane, nb)]);
    wave_lds_fence();
#pragma unroll
    for (int mb = 0; mb < LW_MB; ++mb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * mb + 4 * g + r;
            float v[8];
#pragma unroll
            for (int nb = 0; nb < 8; ++nb) v[nb] = h2f(f2h(mul1_affine(tot[mb][nb][r], xs[wave][row])));     // C in fp16
            had128_acc(v, lane);
#pragma unroll
            for (int nb = 0; nb < 8; ++nb) lds.y[wave][row][mfma_col(lane, nb)] = f2h(h2f(f2h(v[nb])) * sv[nb]);
        }
    wave_lds_fence();
    for (int i = lane; i < 16 * LW_MB * 16; i += 64) {
        const int row = i >> 4, piece = i & 15;
        if (r0 + row < p.rows)
            *(u32x4_t*)(p.y + (size_t)(r0 + row) * p.out + cg * 128 + 8 * piece) = *(const u32x4_t*)&lds.y[wave][row][8 * piece];
    }
}

// Kernel of a call of more than LIN_GEMV_ROWS rows. Wide tiles pay off once they fill the device, the
// earlier the longer k is (a wide workgroup's fixed cost is its epilogue); below that the 64-row
// workgroups over all ranges, and, when those are few, the ones of a range each (their partials cost
// more the more tiles there are, the others' latency the longer k). us per call split / all ranges /
// wide at 4 bpw, 2048 -> 7168: 64 rows 22 / 30 / 48, 256 rows 48 / 32 / 49, 512 rows 84 / 45 / 52, 1024
// rows 161 / 79 / 58; 7168 -> 2048 (3.5 bpw): 256 rows 37 / 82 / 117, 512 rows 66 / 84 / 119, 1024 rows
// 125 / 88 / 121, 2048 rows 241 / 141 / 128; 1024 -> 1024: 512 rows 20 / 24 / 38, 2048 rows 47 / 30 / 40,
// 8192 rows 153 / 68 / 54.
enum { LIN_SPLIT, LIN_FULL, LIN_WIDE };
static int linear_kind(int rows, int in, int out)
{
    const long ncg = out / 128;
    if ((rows + LW_ROWS - 1) / LW_ROWS * ncg >= 80 + 114688 / in) return LIN_WIDE;
    // up to 32 rows and 1024 inputs the call is launches: one less (17.0 against 19.0 us)
    if (rows <= 32 && in <= 1024) return LIN_FULL;
    return (rows + LM_ROWS - 1) / LM_ROWS * ncg >= 80 + in / 76 ? LIN_FULL : LIN_SPLIT;
}

template <int K2>
static void launch_rows_rate(const LinParams& p, int kind, hipStream_t stream)
{
    const long ncg = p.out / 128;
    const long tiles = (p.rows + LM_ROWS - 1) / LM_ROWS * ncg;
    if (kind == LIN_WIDE) {
        const dim3 grid((unsigned)((p.rows + LW_ROWS - 1) / LW_ROWS * ncg));
        hipLaunchKernelGGL(lin_wide_kernel<K2>, grid, dim3(64 * LW_WAVES), 0, stream, p);
    } else if (kind == LIN_FULL) {
        hipLaunchKernelGGL((lin_mid_kernel<K2, false>), dim3((unsigned)tiles), dim3(64 * LM_WAVES), 0, stream, p);
    } else {
        hipLaunchKernelGGL((lin_mid_kernel<K2, true>), dim3((unsigned)(tiles * p.ks)), dim3(64 * LM_WAVES), 0, stream, p);
        hipLaunchKernelGGL(lin_mid_epilogue_kernel, dim3((unsigned)((ncg * p.rows + 3) / 4)), dim3(256), 0, stream, p);
    }
}

// k-split of a call: decode path, enough splits to fill the device once; beyond it the k-ranges. Both
// depend on in/out only.
int linear_ksplit(int rows, int in, int out)
{
    const int ncg = out / 128, nch = in / 128;
    if (rows > LIN_GEMV_ROWS) return nch < LIN_RANGES ? nch : LIN_RANGES;
    int ks = (4096 + ncg - 1) / ncg;
    if (ks > nch) ks = nch;
    if (ks < 1) ks = 1;
    return ks;
}

// Workspace: the column groups' arrival counters (out/128 of them, 128 bytes apart, at offset 0
// for every row count, so that no other layout overwrites them); from 3 rows the rotated rows
// [rows][in] fp16 and their 128-chunk sums [rows][in/128]; up to 16 rows the fp32 partials
// [ks][rows][out].
static size_t arrive_bytes(int out) { return (size_t)(out / 128) * ARRIVE_STRIDE * 8; }

size_t linear_workspace(int rows, int in, int out, size_t* off_part, size_t* off_sum)
{
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    size_t o = al(arrive_bytes(out));
    if (off_sum) *off_sum = 0;
    if (off_part) *off_part = 0;
    if (rows > LIN_ROT_ROWS) {
        o = al(o + (size_t)(rows > LIN_GEMV_ROWS ? (rows + 15) & ~15 : rows) * in * 2);
        if (off_sum) *off_sum = o;
        o = al(o + (size_t)rows * (in / 128) * 4);
    }
    if (rows <= LIN_GEMV_ROWS || linear_kind(rows, in, out) == LIN_SPLIT) {
        if (off_part) *off_part = o;
        o = al(o + (size_t)linear_ksplit(rows, in, out) * rows * out * 4);
    }
    return o;
}

int launch_linear(const void* x, int rows, int in, int out, const void* trellis, const void* suh,
                  const void* svh, int k2, void* y, void* ws, hipStream_t stream)
{
    LinParams p;
    size_t off_part, off_sum;
    linear_workspace(rows, in, out, &off_part, &off_sum);
    p.x = (const half_t*)x;
    p.rows = rows; p.in = in; p.out = out; p.k2 = k2;
    p.ks = linear_ksplit(rows, in, out);
    p.trellis = (const uint32_t*)trellis;
    p.suh = (const half_t*)suh;
    p.svh = (const half_t*)svh;
    p.y = (half_t*)y;
    const size_t off_xr = (arrive_bytes(out) + 255) & ~(size_t)255;
    p.arrive = (unsigned long long*)ws;
    p.xr = rows > LIN_ROT_ROWS ? (half_t*)((char*)ws + off_xr) : nullptr;
    p.xsum = rows > LIN_ROT_ROWS ? (float*)((char*)ws + off_sum) : nullptr;
    p.part = rows <= LIN_GEMV_ROWS || linear_kind(rows, in, out) == LIN_SPLIT ? (float*)((char*)ws + off_part) : nullptr;
    if (rows > LIN_GEMV_ROWS) {
        hipLaunchKernelGGL(lin_rotate16_kernel, dim3((unsigned)((rows + 15) / 16 * (in / 128))), dim3(256), 0, stream, p);
    } else if (rows > LIN_ROT_ROWS) {
        const long waves = (long)rows * (in / 128);
        hipLaunchKernelGGL(lin_rotate_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, stream, p);
    }
    int kind = rows > LIN_GEMV_ROWS ? linear_kind(rows, in, out) : -1;
    if (kind == LIN_WIDE && ((uintptr_t)y & 15)) kind = LIN_FULL;      // its stores are 16 bytes wide
#define EVAMX_LIN_RATE(K2)                                   \
    case K2:                                                 \
        if (kind >= 0) launch_rows_rate<K2>(p, kind, stream); \
        else launch_gemv_rate<K2>(p, stream);                \
        break
    switch (k2) {
        EVAMX_LIN_RATE(3);
        EVAMX_LIN_RATE(4);
        EVAMX_LIN_RATE(5);
        EVAMX_LIN_RATE(6);
        EVAMX_LIN_RATE(7);
        EVAMX_LIN_RATE(8);
        EVAMX_LIN_RATE(10);
        default: return -1;             // the rate is validated by the caller
    }
#undef EVAMX_LIN_RATE
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace evamx
