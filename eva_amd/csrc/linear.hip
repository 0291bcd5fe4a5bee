// Single EXL3 linear, fp16 in / fp16 out (the config-1 layer).
//
// Reference: ELinear.forward -> LinearEXL3 (runtime/ds41/exl3_linear.py:97-131), kernel
// exl3_gemv_kernel.cuh:217-234 (input: fp16 x*suh, Hadamard, fp16), 295-459 (GEMV, fp16 C),
// 463-490 with hadamard_inner.cuh:93-147 (output Hadamard to fp16, fp16 product with svh).
// Up to LIN_GEMV_ROWS rows, one launch: a k-split GEMV whose waves rotate their own input chunks
// (fp16(H128(fp16(x * suh)))) into LDS while their first weight loads are in flight and multiply the
// decoded weights by the rows as 16-row matrix operands; a workgroup adds its four splits in LDS and
// writes them as fp32 partials; the workgroup that arrives last at its column group's counter then runs
// that group's output epilogue (the partials summed in fixed order, fp16 C, Hadamard, fp16 svh product).
// More rows: the input rotation, written as MFMA operands, then one of three MFMA kernels by size
// (linear_kind): 256-row workgroups that share each decoded weight (lin_wide_kernel), 64-row
// workgroups over the whole k range, or over one k-range each with the output epilogue in a launch
// of its own. All add the same k-ranges' sums in the same order. In both paths (up to
// LIN_GEMV_ROWS rows, and beyond) a row's arithmetic depends on in/out only, not on how many rows
// share the call.
#include <algorithm>

#include "evamx_internal.hpp"
#include "evamx_wide.hpp"

namespace evamx {


constexpr int LIN_GEMV_ROWS = 16;     // lin_gemv_kernel up to this many rows
constexpr int LIN_GRID_Y = 32768;     // column groups along y of its grid

struct LinParams {
    const half_t* x;
    int rows, in, out, ks;
    int per;           // 128-chunks of a k-split, or 0 where they differ by one
    const uint32_t* trellis;
    const half_t* suh;
    const half_t* svh;
    half_t* y;
    half_t* xr;        // rotated rows as A operands (a_operand_offset), beyond LIN_GEMV_ROWS rows
    float* xsum;       // [rows][in/128]
    float* part;       // decode path: [quarters of ks][rows][out]; k-range partials: [ks][rows][out]
    unsigned long long* arrive;   // arrival counters of the decode path, one per ARRIVE_STRIDE words
};

// The lane's two svh values, loaded at the start of the launch (the epilogue needs them only in
// the last workgroup, but then without waiting for them).
__device__ __forceinline__ void lin_load_sv(const LinParams& p, int cg, float (&sv)[2])
{
    const int lane = threadIdx.x & 63;
    sv[0] = h2f(p.svh[cg * 128 + lane_col(lane, 0)]);
    sv[1] = h2f(p.svh[cg * 128 + lane_col(lane, 1)]);
}

// ---------------------------------------------------------------------------------------------
// Up to LIN_GEMV_ROWS rows: one launch. A workgroup of eight waves takes 128 output columns and four of
// the ks k-splits, two waves a split with 64 columns each (two waves a SIMD hide each other's latency).
// The rows are rotated over the split's k-range into LDS while the first weights are in flight; a wave
// multiplies the decoded weights, as the B operands they are, by the rows as one 16-row A operand; a
// further operand of ones gives the rows' sums for the codebook map. So one row and sixteen take the same
// instructions, and a row's bits do not depend on how many share the call. The
// four splits' results are added in LDS in order; the quarters meet through memory, and the last
// workgroup to arrive at the column group's counter adds them in order and runs the output epilogue.
// Bound by latency: the launch, the first weights, the arrival. So nothing is computed or loaded on the way
// to the first weights that the call can do without: no division (the workgroup's place is its grid index,
// equal splits need none), and where a split is one 128-chunk, as up to 2^26 weights, one chunk's loads
// and nothing past them. (Against a v_dot2 kernel up to two rows, and three launches from three rows on;
// 2048 -> 7168 at 4 bpw, 64 copies in a graph, us per call, that / this with divisions and loads past the
// chunk / this: 1 row 6.84 / 7.16 / 6.27, 2 rows 8.44 / 8.05 / 7.25, 8 rows 21.0 / 8.9 / 7.7, 16 rows 35.7 / 11.3
// / 9.3; 5120 -> 5120 at 3.5 bpw, 1 row 10.2 / 9.5 / 9.0; 1024 -> 18432 at 4 bpw, 1 row 8.5 / 9.4 / 7.9.)

// 128-chunks of rotated rows in LDS at a time, and words of a row there (padded, so that the 16 rows an
// operand reads lie in different banks). One row: each wave rotates it for itself; more: the waves of a
// split share the rows (LinRot).
template <int TM>
struct LinStage {
    static constexpr int CW = TM == 1 ? 4 : 2;
    static constexpr int ROW = CW * 64 + 4;
    static constexpr int WORDS = TM == 1 ? ROW : TM * ROW;
};

// fp16(H128(fp16(x * suh))) of the call's rows over the 128-chunks [w0, w1) into LDS, NC of them at most.
// issue() loads ahead of the weight prefetch, finish() rotates behind it. One row: a chunk on the whole
// wave; more: 16 lanes a chunk, four (row, chunk) pairs at a time, the split's HV waves taking turns. The
// same bits either way.
template <int TM, int NC, int HV>
struct LinRot;

template <int NC, int HV>
struct LinRot<1, NC, HV> {
    uint32_t xv[NC], sv[NC];
    __device__ __forceinline__ void issue(const LinParams& p, int w0, int w1, int)
    {
        const int lane = threadIdx.x & 63;
        const __amdgpu_buffer_rsrc_t xrs = weight_rsrc((const uint32_t*)p.x), srs = weight_rsrc((const uint32_t*)p.suh);
        // chunks past the window reload its last one (in bounds, unused): no branches
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const uint32_t off = 256u * (uint32_t)min(w0 + j, w1 - 1);
            sv[j] = __builtin_amdgcn_raw_buffer_load_b32(srs, 4 * lane, off, 0);
            xv[j] = __builtin_amdgcn_raw_buffer_load_b32(xrs, 4 * lane, off, 0);
        }
    }
    __device__ __forceinline__ void finish(const LinParams&, int w0, int w1, int, uint32_t* dst)
    {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            if (w0 + j < w1) {
                const half2_t xx = __builtin_bit_cast(half2_t, xv[j]), su = __builtin_bit_cast(half2_t, sv[j]);
                float v0 = h2f(f2h(h2f(xx.x) * h2f(su.x)));      // fp16 product
                float v1 = h2f(f2h(h2f(xx.y) * h2f(su.y)));
                had128_pair(v0, v1, lane);
                const half2_t r = {f2h(v0), f2h(v1)};
                dst[64 * j + lane] = __builtin_bit_cast(uint32_t, r);
            }
        }
    }
};

template <int NC, int HV>
struct LinRot<16, NC, HV> {
    static_assert(NC <= 2, "a pair's row and chunk by a shift");
    static constexpr int NG = LIN_GEMV_ROWS * NC / (4 * HV);     // groups of four pairs a wave at most
    static constexpr int NL = NG < 4 ? NG : 4;                   // of them loaded at a time
    u32x4w xv[NL], sv[NL];
    // pair it: row it >> (nw - 1), chunk w0 + (it & (nw - 1)), for a window of nw (1 or 2) chunks
    __device__ __forceinline__ void load(const LinParams& p, int w0, int w1, int half, int g0)
    {
        const int lane = threadIdx.x & 63, sh = NC == 1 ? 0 : w1 - w0 - 1, n = p.rows << sh;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int b = 4 * (HV * (g0 + i) + half);
            if (b >= n) break;
            const int it = min(b + (lane >> 4), n - 1);
            const size_t k = 128 * (w0 + (it & sh)) + 8 * oct_piece(lane);
            xv[i] = *(const __attribute__((address_space(1))) u32x4w*)(p.x + (size_t)(it >> sh) * p.in + k);
            sv[i] = *(const __attribute__((address_space(1))) u32x4w*)(p.suh + k);
        }
    }
    __device__ __forceinline__ void issue(const LinParams& p, int w0, int w1, int half) { load(p, w0, w1, half, 0); }
    __device__ __forceinline__ void finish(const LinParams& p, int w0, int w1, int half, uint32_t* dst)
    {
        const int lane = threadIdx.x & 63, sh = NC == 1 ? 0 : w1 - w0 - 1, n = p.rows << sh;
        for (int g0 = 0; g0 < NG && 4 * (HV * g0 + half) < n; g0 += NL) {
            if (g0 > 0) load(p, w0, w1, half, g0);
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                const int b = 4 * (HV * (g0 + i) + half), it = b + (lane >> 4);
                if (b >= n) break;
                const uint32_t xu[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w}, su[4] = {sv[i].x, sv[i].y, sv[i].z, sv[i].w};
                float x[8], h[8];
                oct_halves(xu, x);
                oct_halves(su, h);
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = h2f(f2h(x[e] * h[e]));       // fp16 product
                had128_oct(x, lane);
                u32x4 r;
#pragma unroll
                for (int e = 0; e < 4; ++e) r[e] = __builtin_bit_cast(uint32_t, half2_t{f2h(x[2 * e]), f2h(x[2 * e + 1])});
                if (it < n) *(u32x4*)(dst + (it >> sh) * LinStage<16>::ROW + 64 * (it & sh) + 4 * oct_piece(lane)) = r;
            }
        }
    }
};

// The wave's share of the columns (128 / HV from 128 / HV * half on) over its split's k-range [c0, c1)
// (128-chunks, none for a wave past the splits): acc[nb][r] = sum_k x_k h_k, ones[r] = sum_k x_k for row
// 4 g + r and column 128 / HV * half + mfma_col(lane, nb), in windows of NC chunks (TM > 1: every wave of
// the workgroup runs as many), HV steps of weights in flight. NC 1: every split is one chunk, and
// nothing past it is loaded.
template <int K2, int TM, int HV, int NC>
__device__ __forceinline__ void lin_gemv_range(const LinParams& p, int cg, int half, int c0, int c1, int windows, uint32_t* lds,
                                               f32x4_t (&acc)[8 / HV], f32x4_t& ones)
{
    using R = Rate<K2>;
    constexpr int K = R::K;
    constexpr int TW = R::TW;
    constexpr int NU = 4 / HV;                            // units (pairs of tiles) a step
    const int lane = threadIdx.x & 63, m16 = lane & 15, g = lane >> 4, nt_n = p.out / 16;
    const uint32_t slice = __builtin_amdgcn_readfirstlane(4u * (uint32_t)(nt_n * TW));
    const uint32_t cbase = __builtin_amdgcn_readfirstlane(4u * (uint32_t)((cg * 8 + 2 * NU * half) * TW));
    const __amdgpu_buffer_rsrc_t rsrc = weight_rsrc(p.trellis);
    uint32_t lane_off, sh;
    lane_offsets<K2>(lane & 15, lane_off, sh);
    lane_off += (uint32_t)g * slice;
    // rows past the call's read row 0 (their results are dropped)
    const uint32_t* xrow = lds + (m16 < p.rows ? m16 : 0) * LinStage<TM>::ROW + 8 * g;
    const half_t o1 = (half_t)1.0f;
    const half8_t bones = {o1, o1, o1, o1, o1, o1, o1, o1};
#pragma unroll
    for (int nb = 0; nb < 2 * NU; ++nb) acc[nb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    ones = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    for (int i = 0; i < windows; ++i) {
        const int w0 = c0 + i * NC, w1 = min(c1, w0 + NC), steps = NC == 1 ? 2 : 2 * (w1 - w0);
        const uint32_t wbase = cbase + (uint32_t)(8 * w0) * slice;
        const bool work = w0 < w1;                        // wave-uniform
        LaneWords<K> ring[HV][NU];                        // HV steps
        auto load_w = [&](LaneWords<K>& w, int t, int j) {
            load_slice<K>(w, rsrc, wbase + (uint32_t)(4 * min(t, steps - 1)) * slice + (uint32_t)(8 * j * TW), lane_off);
        };
        if (work) {
            LinRot<TM, NC, HV> rot;
            rot.issue(p, w0, w1, half);
#pragma unroll
            for (int t = 0; t < HV; ++t)
#pragma unroll
                for (int j = 0; j < NU; ++j) load_w(ring[t][j], t, j);
            __builtin_amdgcn_sched_barrier(0);
            rot.finish(p, w0, w1, half, lds);
        }
        if constexpr (TM == 1) wave_lds_fence();
        else __syncthreads();
        auto step = [&](int t, LaneWords<K> (&w)[NU]) {
            const half8_t a0 = __builtin_bit_cast(half8_t, *(const u32x4_t*)(xrow + 32 * t));
            const half8_t a1 = __builtin_bit_cast(half8_t, *(const u32x4_t*)(xrow + 32 * t + 4));
#pragma unroll
            for (int j = 0; j < NU; ++j) {
                half2_t wp[16];
                decode_slice<K2, true>(w[j], sh, wp);
                if (NC > 1 || t + HV < steps) load_w(w[j], t + HV, j);
                mfma_begin();
                if (j == 0) {
                    ones = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, bones, ones, 0, 0, 0);
                    ones = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, bones, ones, 0, 0, 0);
                }
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    acc[2 * j + c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, mfma_b(wp, c, 0), acc[2 * j + c], 0, 0, 0);
                    acc[2 * j + c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, mfma_b(wp, c, 1), acc[2 * j + c], 0, 0, 0);
                }
                mfma_end<4>();
            }
        };
        if (work)
            for (int t = 0; t < steps; t += 2) {
                step(t, ring[0]);
                step(t + 1, ring[HV - 1]);
            }
        // this window's reads before the next window's writes (or the results)
        if constexpr (TM == 1) wave_lds_fence();
        else __syncthreads();
    }
}

// Output epilogue of a row's 128 columns (the lane's two), their codebook map applied: C in fp16,
// Hadamard, fp16 svh product.
__device__ __forceinline__ void lin_finish_row(const LinParams& p, int row, int cg, float v0, float v1, const float (&sv)[2])
{
    const int lane = threadIdx.x & 63;
    v0 = h2f(f2h(v0));
    v1 = h2f(f2h(v1));
    had128_lane(v0, v1, lane);
    half_t* y = p.y + (size_t)row * p.out + cg * 128 + lane_col(lane, 0);
    y[0] = f2h(h2f(f2h(v0)) * sv[0]);
    y[8] = f2h(h2f(f2h(v1)) * sv[1]);
}

// The rows r0, r0 + d, .. (NR of them at most, below p.rows) of a column group: the nq quarters' partials
// added in order, read from the memory side, where the other workgroups' write-through stores went; the
// loads of a batch of quarters of every row are issued before any add. Buffer loads take the quarters'
// offsets in scalar registers.
template <int NR, int QB>
__device__ __forceinline__ void lin_last_rows(const LinParams& p, int cg, int r0, int d, int nq, const float (&sv)[2])
{
    const int lane = threadIdx.x & 63;
    const __amdgpu_buffer_rsrc_t rs = weight_rsrc((const uint32_t*)p.part);
    const uint32_t vo = 4u * (uint32_t)(cg * 128 + lane_col(lane, 0));           // column 1: + 32 bytes
    float v[NR][2];
#pragma unroll
    for (int i = 0; i < NR; ++i) v[i][0] = v[i][1] = 0.0f;
    for (int q0 = 0; q0 < nq; q0 += QB) {
        float t[NR][QB][2];
#pragma unroll
        for (int i = 0; i < NR; ++i)
#pragma unroll
            for (int q = 0; q < QB; ++q) {
                const uint32_t so = 4u * (uint32_t)p.out * (uint32_t)(min(q0 + q, nq - 1) * p.rows + min(r0 + i * d, p.rows - 1));
                t[i][q][0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, vo, so, LD_SC1));
                t[i][q][1] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, vo + 32, so, LD_SC1));
            }
#pragma unroll
        for (int i = 0; i < NR; ++i)
#pragma unroll
            for (int q = 0; q < QB; ++q)
                if (q0 + q < nq) {
                    v[i][0] += t[i][q][0];
                    v[i][1] += t[i][q][1];
                }
    }
#pragma unroll
    for (int i = 0; i < NR; ++i)
        if (r0 + i * d < p.rows) lin_finish_row(p, r0 + i * d, cg, v[i][0], v[i][1], sv);
}

// One row: every quarter in flight up to 16 (a second round trip cost 0.3 us at 10 quarters, clamped loads
// 0.4 us at 4).
__device__ __forceinline__ void lin_last_one(const LinParams& p, int cg, int row, int nq, const float (&sv)[2])
{
    if (nq <= 4) lin_last_rows<1, 4>(p, cg, row, 1, nq, sv);
    else if (nq <= 8) lin_last_rows<1, 8>(p, cg, row, 1, nq, sv);
    else lin_last_rows<1, 16>(p, cg, row, 1, nq, sv);
}

// TM: 1, or 16 (2 to LIN_GEMV_ROWS rows).
template <int K2, int TM, int HV>
__global__ __launch_bounds__(256 * HV) __attribute__((amdgpu_waves_per_eu(TM == 1 ? 4 : 3))) void lin_gemv_kernel(LinParams p)
{
    __shared__ uint32_t lds[TM == 1 ? 4 * HV : 4][LinStage<TM>::WORDS];
    __shared__ float res1[TM == 1 ? 4 : 1][128];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63, g = lane >> 4;
    const int split = wave / HV, half = wave % HV;
    // q fastest: the workgroups of a column group side by side
    const int nq = (p.ks + 3) >> 2, q = blockIdx.x, cg = blockIdx.y + LIN_GRID_Y * blockIdx.z;
    if (cg >= p.out / 128) return;
    const int ks = 4 * q + split, nv = min(4, p.ks - 4 * q);     // the workgroup's splits
    float sv[2];
    lin_load_sv(p, cg, sv);
    f32x4_t acc[8 / HV], ones;
    uint32_t* const stage = lds[TM == 1 ? wave : split];
    if (p.per == 1) {
        lin_gemv_range<K2, TM, HV, 1>(p, cg, half, ks, split < nv ? ks + 1 : ks, 1, stage, acc, ones);
    } else {
        constexpr int CW = LinStage<TM>::CW;
        const int nch = p.in / 128;
        const int c0 = split < nv ? nch * ks / p.ks : 0, c1 = split < nv ? nch * (ks + 1) / p.ks : 0;
        const int most = TM == 1 ? c1 - c0 : (nch + p.ks - 1) / p.ks;
        lin_gemv_range<K2, TM, HV, CW>(p, cg, half, c0, c1, (most + CW - 1) / CW, stage, acc, ones);
    }
    auto res = [&](int w) { return TM == 1 ? res1[w] : (float*)lds[w]; };        // split w's results [row][128]
    if (split < nv) {
        float* d = res(split) + 128 / HV * half;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 4 * g + r;
            if (TM == 1 ? lane < 16 && r == 0 : row < p.rows) {
#pragma unroll
                for (int nb = 0; nb < 8 / HV; ++nb) d[128 * row + mfma_col(lane, nb)] = mul1_affine(acc[nb][r], ones[r]);
            }
        }
    }
    __syncthreads();
    auto sum = [&](int i) {                                      // the splits' result i, in split order
        const float t0 = res(0)[i], t1 = res(min(1, nv - 1))[i], t2 = res(min(2, nv - 1))[i], t3 = res(nv - 1)[i];
        float t = t0;
        if (nv > 1) t += t1;
        if (nv > 2) t += t2;
        if (nv > 3) t += t3;
        return t;
    };
    if (nq == 1) {
        // the only quarter: nothing to meet
        for (int row = wave; row < p.rows; row += 4 * HV)
            lin_finish_row(p, row, cg, 0.0f + sum(128 * row + lane_col(lane, 0)), 0.0f + sum(128 * row + lane_col(lane, 1)), sv);
        return;
    }
    // store, wait until every store is acknowledged, arrive, and run the epilogue if last (the stores of
    // every workgroup of the group then precede the loads); one row: wave 0 alone
    unsigned long long* word = p.arrive + (size_t)cg * ARRIVE_STRIDE;
    if constexpr (TM == 1) {
        if (wave != 0) return;
        float* dst = p.part + (size_t)q * p.out + cg * 128;
#pragma unroll
        for (int h = 0; h < 2; ++h) store_wt(dst + lane_col(lane, h), sum(lane_col(lane, h)));
        if (wave_arrive_last(word, (unsigned)nq)) lin_last_one(p, cg, 0, nq, sv);
    } else {
        __shared__ int last;
        for (int i = threadIdx.x; i < 128 * p.rows; i += 256 * HV)
            store_wt(p.part + ((size_t)q * p.rows + (i >> 7)) * p.out + cg * 128 + (i & 127), sum(i));
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (threadIdx.x == 0) last = arrive_last(word, (unsigned)nq);
        __syncthreads();
        if (last && wave < p.rows) {
            if (p.rows <= 4 * HV) lin_last_one(p, cg, wave, nq, sv);
            else lin_last_rows<4 / HV, 4 * HV>(p, cg, wave, 4 * HV, nq, sv);
        }
    }
}

// Decode path launch of one rate: workgroups per (column group, four splits), of eight waves while one
// workgroup a CU leaves the SIMDs a wave each otherwise, of four beyond (four waves against eight: 5120 ->
// 5120 at 5 bpw, 400 workgroups, one row 9.8 against 10.0 us, 13 rows 14.9 against 18.4; 7168 -> 2048 at 2.5
// bpw, 224, one row 6.9 against 6.6, 8 rows 10.8 against 8.8).
template <int K2>
void launch_gemv_rate(const LinParams& p, hipStream_t stream)
{
    const int ncg = p.out / 128, nq = (p.ks + 3) / 4, blocks = ncg * nq;
    const dim3 grid((unsigned)nq, (unsigned)std::min(ncg, LIN_GRID_Y), (unsigned)((ncg + LIN_GRID_Y - 1) / LIN_GRID_Y));
    if (blocks <= 256) {
        if (p.rows == 1) hipLaunchKernelGGL((lin_gemv_kernel<K2, 1, 2>), grid, dim3(512), 0, stream, p);
        else hipLaunchKernelGGL((lin_gemv_kernel<K2, 16, 2>), grid, dim3(512), 0, stream, p);
    } else {
        if (p.rows == 1) hipLaunchKernelGGL((lin_gemv_kernel<K2, 1, 1>), grid, dim3(256), 0, stream, p);
        else hipLaunchKernelGGL((lin_gemv_kernel<K2, 16, 1>), grid, dim3(256), 0, stream, p);
    }
}

// ---------------------------------------------------------------------------------------------
// More than LIN_GEMV_ROWS rows.

constexpr int LIN_RANGES = 8;         // k-ranges whose sums are added in order

// fp16(H128(fp16(x * suh))) of the rows with each 128-chunk's sum, written as A operands
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

// lin_finish_row of a row's accumulated columns: the codebook map first.
__device__ __forceinline__ void lin_store_row(const LinParams& p, int row, int cg, float v0, float v1, float xs, const float (&sv)[2])
{
    lin_finish_row(p, row, cg, mul1_affine(v0, xs), mul1_affine(v1, xs), sv);
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
constexpr int LW_WAVES = WIDE_WAVES;
constexpr int LW_ROWS = 16 * LW_MB * LW_WAVES;
constexpr int LW_STRIDE = 136;                       // halves per staged output row (padded)

template <int K2>
__global__ __launch_bounds__(64 * LW_WAVES) __attribute__((amdgpu_waves_per_eu(2))) void lin_wide_kernel(LinParams p)
{
    __shared__ union {
        WideLds w;
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
    wide_accumulate<K2, LW_MB>(p.trellis, p.out / 16, cg, 0, nch, arow, lds.w, acc, [&](int c) {
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

// Whether a call's 64-row workgroups take one k-range each: while their 16-row blocks are few (the ranges'
// partials and products grow with them, the others' latency with k). us per call split / all ranges at 4
// bpw in a graph: 2048 -> 7168, 64 rows 23 / 30, 128 rows 32 / 31; 7168 -> 2048, 512 rows 52 / 69, 768 rows 78 /
// 75; 7168 -> 18432, 65 rows 76 / 86, 129 rows 125 / 117; 18432 -> 7168, 224 rows 156 / 156, 256 rows 175 / 162.
// By size only: the workspace depends on it.
static bool linear_splits(int rows, int in, int out)
{
    // up to 32 rows and 1024 inputs an eager call is launches: one less (17.0 against 19.0 us)
    if (rows <= 32 && in <= 1024) return false;
    return (long)((rows + 15) / 16) * (out / 128) < 240 + in / 14;
}

// Kernel of a call of more than LIN_GEMV_ROWS rows. Wide tiles pay off once they fill the device, the
// earlier the longer k is (a wide workgroup's fixed cost is its epilogue), if their rows are there: a wide
// workgroup of a few rows takes as long as a full one, so the 64-row workgroups, which count the rows that
// there are, have to fill the device (256 workgroups) about twice for each time the wide ones do; somewhat
// less from 7168 inputs on, where two of the former on a CU take as long as one wide one. us per call split /
// all ranges / wide in a graph: 7168 -> 18432 at 4 bpw, 17 rows 41 / 53 / 111, 128 rows 108 / 114 / 117, 257
// rows - / 173 / 229, 512 rows - / 298 / 246, at 5 bpw 17 rows 51 / 60 / 118, 128 rows 127 / 145 / 122, 512 rows
// - / 374 / 259; 4096 -> 14336 at 3.5 bpw, 64 rows 40 / 46 / 76, 320 rows - / 104 / 86; 7168 -> 7168 at 4 bpw, 257
// rows 91 / 82 / 117, 384 rows 121 / 114 / 118, 640 rows - / 168 / 121; 2048 -> 12288, 640 rows - / 78 / 102;
// 7168 -> 2048, 1024 rows 103 / 79 / 121, 2048 rows - / 145 / 139; 384 -> 40960 at 2.5 bpw, 257 rows - / 44 / 70;
// 1024 -> 1024, 2048 rows 52 / 33 / 44.
enum { LIN_SPLIT, LIN_FULL, LIN_WIDE };
static int linear_kind(int rows, int in, int out)
{
    const long ncg = out / 128, wide = (rows + LW_ROWS - 1) / LW_ROWS * ncg, mid = (rows + LM_ROWS - 1) / LM_ROWS * ncg;
    const float rounds = (float)((wide + 255) / 256);
    const float fill = rounds * (2.0f + 300.0f / in) - (in >= 7168 ? 0.75f : 0.0f);
    if (wide >= 80 + 114688 / in && (float)mid >= 256.0f * fill) return LIN_WIDE;
    return linear_splits(rows, in, out) ? LIN_SPLIT : LIN_FULL;
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
// for every row count, so that no other layout overwrites them); beyond LIN_GEMV_ROWS rows the rotated
// rows in blocks of 16 and their 128-chunk sums [rows][in/128]; the fp32 partials of the decode path's
// quarters or of the k-ranges.
static size_t arrive_bytes(int out) { return (size_t)(out / 128) * ARRIVE_STRIDE * 8; }

size_t linear_workspace(int rows, int in, int out, size_t* off_part, size_t* off_sum)
{
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    size_t o = al(arrive_bytes(out));
    if (off_sum) *off_sum = 0;
    if (off_part) *off_part = 0;
    const bool decode = rows <= LIN_GEMV_ROWS;
    if (!decode) {
        o = al(o + (size_t)((rows + 15) & ~15) * in * 2);
        if (off_sum) *off_sum = o;
        o = al(o + (size_t)rows * (in / 128) * 4);
    }
    if (decode || linear_splits(rows, in, out)) {
        if (off_part) *off_part = o;
        const int ks = linear_ksplit(rows, in, out);
        o = al(o + (size_t)(decode ? (ks + 3) / 4 : ks) * rows * out * 4);
    }
    return o;
}

// What a program is told to keep for calls of up to `rows` rows. The k-ranges' partials go only with the
// row counts between the decode path and the unsplit kernels, so a smaller call can need more than a
// larger one: the largest need of any row count up to this, so that a workspace made for the largest call
// (and captured with it) serves the smaller ones too.
size_t linear_workspace_upto(int rows, int in, int out)
{
    size_t n = linear_workspace(rows, in, out, nullptr, nullptr);
    if (rows <= LIN_GEMV_ROWS) return n;
    auto most = [&](int r) {
        const size_t v = linear_workspace(r < rows ? r : rows, in, out, nullptr, nullptr);
        if (v > n) n = v;
    };
    most(LIN_GEMV_ROWS);
    // the last row count that may be split (linear_splits' line)
    const long ncg = out / 128, full = 240 + in / 14, last = ((full + ncg - 1) / ncg - 1) * 16;
    if (last > LIN_GEMV_ROWS) most((int)std::min(last, 65536L));
    return n;
}

// Whether the decode path takes the shape: its limit is 2 GiB of one partial a split and the rows. The
// path keeps a quarter of the partials and no rows, but what it refuses stays what it is.
bool linear_decode_fits(int rows, int in, int out)
{
    return (size_t)linear_ksplit(rows, in, out) * rows * out * 4 + (size_t)rows * in * 2 + arrive_bytes(out) < ((size_t)1 << 31);
}

int launch_linear(const void* x, int rows, int in, int out, const void* trellis, const void* suh,
                  const void* svh, int k2, void* y, void* ws, hipStream_t stream)
{
    LinParams p;
    size_t off_part, off_sum;
    linear_workspace(rows, in, out, &off_part, &off_sum);
    const int kind_ws = rows > LIN_GEMV_ROWS ? linear_kind(rows, in, out) : -1;
    p.x = (const half_t*)x;
    p.rows = rows; p.in = in; p.out = out;
    p.ks = linear_ksplit(rows, in, out);
    p.per = in / 128 % p.ks == 0 ? in / 128 / p.ks : 0;
    p.trellis = (const uint32_t*)trellis;
    p.suh = (const half_t*)suh;
    p.svh = (const half_t*)svh;
    p.y = (half_t*)y;
    p.arrive = (unsigned long long*)ws;
    p.xr = kind_ws >= 0 ? (half_t*)((char*)ws + ((arrive_bytes(out) + 255) & ~(size_t)255)) : nullptr;
    p.xsum = kind_ws >= 0 ? (float*)((char*)ws + off_sum) : nullptr;
    p.part = off_part ? (float*)((char*)ws + off_part) : nullptr;
    // the wide kernel's stores are 16 bytes wide
    const int kind = kind_ws == LIN_WIDE && ((uintptr_t)y & 15) ? (int)LIN_FULL : kind_ws;
    if (kind >= 0)
        hipLaunchKernelGGL(lin_rotate16_kernel, dim3((unsigned)((rows + 15) / 16 * (in / 128))), dim3(256), 0, stream, p);
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
