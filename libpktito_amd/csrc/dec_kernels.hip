/* The decoder's per-token work on the device (core/decoder.c:54-101 in
 * peterheb/libpktito): its products are T = 1 GEMVs, each a quantize of one
 * row and a product, latency-bound at a few microseconds of work. Each
 * launch here fuses what the reference runs as separate calls: the row's
 * quantize with its product (gemv), an LSTM layer's two products, their add
 * and its cell (lstm), and the joint's ReLU, quantize, product and argmax.
 *
 * Bits: the reference's ref backend's. The quantize is
 * backend/ref/kernels.c:24-58 with one block of the whole row; the sums are
 * exact int32 (v_dot4 over the repacked units, any order); the epilogue,
 * the cell (backend/ref/kernels.c:203-213) and the argmax (the first of
 * equal values) are the reference's operations in its order. Built with
 * -ffp-contract=off.
 */
#include "q8_device.h"
#include "q8_internal.h"

#pragma clang fp contract(off)

namespace pkq8 {

constexpr uint32_t kDecMaxCols = 4096;

/* Chunk i (elements 4i .. 4i + 3, 4i < n) of a row of n floats: one float4
 * load when the row is 16-byte aligned and n a multiple of 4 (AL), else
 * four loads with zeros past n. */
template <bool AL>
__device__ __forceinline__ float4 row4(const float *__restrict__ x, uint32_t i, uint32_t n) {
    if (AL)
        return ((const float4 *)x)[i];
    const uint32_t k = 4 * i;
    return make_float4(x[k], k + 1 < n ? x[k + 1] : 0.0f, k + 2 < n ? x[k + 2] : 0.0f, k + 3 < n ? x[k + 3] : 0.0f);
}

/* One row of n <= 256 CH values, quantized whole by one wave into q (LDS,
 * bytes, zero to 64 kr, kr <= 4 CH) in two steps. load_row: every lane
 * issues the loads of its chunks i + 64 c (value4(i) gives chunk i, zeros
 * past n), so the row costs one memory round trip, and the caller may
 * issue other loads behind them before it uses the row. */
template <int CH, typename F>
__device__ __forceinline__ void load_row(F value4, uint32_t n, int lane, float4 (&v)[CH]) {
    const uint32_t n4 = (n + 3) >> 2;
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const uint32_t i = lane + 64 * c;
        v[c] = i < n4 ? value4(i) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
}

/* quant_loaded: the loaded row quantized into q. Returns d (the block rule
 * on magnitude bits: a NaN or an infinity, or an amax below 2^-121, makes
 * the row zero). */
template <int CH>
__device__ __forceinline__ float quant_loaded(const float4 (&v)[CH], uint32_t n, uint32_t kr, int8_t *q, int lane) {
    const uint32_t n4 = (n + 3) >> 2;
    const WaveScales<CH, 0> sc(v);
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const uint32_t i = lane + 64 * c;
        if (i < 16 * kr)
            ((int *)q)[i] = i < n4 && !sc.zero[0] ? pack4(v[c], sc.id[0]) : 0;
    }
    return sc.dv[0];
}

/* The exact int32 sums of the 16 rows of panel p over units [0, kr), kr <=
 * KU, in two steps. panel_load: lane l loads the unit's bytes 16 l .. 16 l
 * + 15 of each unit (the wave reads each 1 KB unit whole, every unit's load
 * issued before the first sum). panel_sum: lane l takes row l % 16 and
 * inputs 16 (l / 16) .. + 15 of each unit, and the four lanes of a row add
 * up by shuffles; every lane returns its row's sum. */
template <int KU>
__device__ __forceinline__ void panel_load(const int8_t *__restrict__ w, uint64_t wstride, uint32_t p, uint32_t kr,
                                           int lane, v4i (&wv)[KU]) {
    const int8_t *wp = w + (size_t)p * kUnitBytes + lane * 16;
#pragma unroll
    for (int u = 0; u < KU; u++)
        if (u < (int)kr)
            wv[u] = *(const v4i *)(wp + (size_t)u * wstride);
}

template <int KU>
__device__ __forceinline__ int panel_sum(const v4i (&wv)[KU], uint32_t kr, const int8_t *q, int lane) {
    const int8_t *qp = q + (lane >> 4) * 16;
    int s = 0;
#pragma unroll
    for (int u = 0; u < KU; u++)
        if (u < (int)kr) {
            const v4i av = *(const v4i *)(qp + 64 * u);
            s = __builtin_amdgcn_sdot4(wv[u][0], av[0], s, false);
            s = __builtin_amdgcn_sdot4(wv[u][1], av[1], s, false);
            s = __builtin_amdgcn_sdot4(wv[u][2], av[2], s, false);
            s = __builtin_amdgcn_sdot4(wv[u][3], av[3], s, false);
        }
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
    return s;
}

/* Whether a kernel of KU units a panel loads its panels behind its row,
 * before the quantize (one memory round trip instead of two): where the
 * panels fit the registers beside the row (the 64-unit kernels load them
 * after). */
template <int KU>
constexpr bool kEarly = KU <= 16;

template <int KU>
__device__ __forceinline__ int panel_dot(const int8_t *__restrict__ w, uint64_t wstride, uint32_t p, uint32_t kr,
                                         const int8_t *q, int lane) {
    v4i wv[KU];
    panel_load<KU>(w, wstride, p, kr, lane, wv);
    return panel_sum<KU>(wv, kr, q, lane);
}

/* gemm_q8's epilogue for one output of a one-block row
 * (backend/ref/kernels.c:75-84): fmaf((float)s, d, +0), times ws, plus the
 * bias br where there is a bias */
__device__ __forceinline__ float gemv_out(int s, float d, float ws, const float *bias, float br) {
    float v = __builtin_fmaf((float)s, d, 0.0f) * ws;
    if (bias)
        v = v + br;
    return v;
}

/* gemv: a wave a 16-row panel, the row quantized by every wave. CH float4
 * chunks a lane hold the row (n <= 256 CH), KU units the panel (kr <= KU);
 * AL as row4's. */
template <int CH, int KU, bool AL>
__global__ __launch_bounds__(64) void gemv_kernel(float *__restrict__ out, const int8_t *__restrict__ w,
                                                  uint64_t wstride, const float *__restrict__ ws,
                                                  const float *__restrict__ bias, const float *__restrict__ x,
                                                  uint32_t n, uint32_t kr, int add) {
    __shared__ __attribute__((aligned(16))) int8_t q[64 * KU];
    const int lane = threadIdx.x;
    const uint32_t p = blockIdx.x;
    float4 v[CH];
    load_row<CH>([&](uint32_t i) { return row4<AL>(x, i, n); }, n, lane, v);
    v4i wv[KU];
    if constexpr (kEarly<KU>)
        panel_load<KU>(w, wstride, p, kr, lane, wv);
    const uint32_t r = 16 * p + (lane & 15);
    const float wsr = ws[r], br = bias ? bias[r] : 0.0f, old = add ? out[r] : 0.0f;
    const float d = quant_loaded<CH>(v, n, kr, q, lane);
    __syncthreads();
    if constexpr (!kEarly<KU>)
        panel_load<KU>(w, wstride, p, kr, lane, wv);
    const int s = panel_sum<KU>(wv, kr, q, lane);
    if (lane < 16) {
        const float o = gemv_out(s, d, wsr, bias, br);
        out[r] = add ? old + o : o;
    }
}

/* An LSTM layer's step (core/decoder.c:68-75): a workgroup 16 units j0 ..
 * j0 + 15, wave w their gate w (rows w P + j), each gate wx x + b and then +
 * wh h as the reference's two calls make it, then the cell
 * (backend/ref/kernels.c:203-213). h_in is read, h_out written (other
 * workgroups still read h_in); c is stepped in place, each unit by one
 * thread. */
template <int CH, int KU, bool AL>
__global__ __launch_bounds__(256) void lstm_kernel(float *__restrict__ h_out, float *__restrict__ c,
                                                   const float *__restrict__ h_in, const float *__restrict__ x,
                                                   const int8_t *__restrict__ wx, const float *__restrict__ wxs,
                                                   const int8_t *__restrict__ wh, const float *__restrict__ whs,
                                                   uint64_t wstride, const float *__restrict__ b, uint32_t P,
                                                   uint32_t kr) {
    __shared__ __attribute__((aligned(16))) int8_t qx[64 * KU], qh[64 * KU];
    __shared__ float dq[2], gates[4][16];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint32_t j0 = 16 * blockIdx.x;
    /* every load the step needs is issued before the first use: the row
     * (waves 0 and 1), the gate's two panels, the scales, the bias, c */
    float4 v[CH];
    if (wv == 0)
        load_row<CH>([&](uint32_t i) { return row4<AL>(x, i, P); }, P, lane, v);
    else if (wv == 1)
        load_row<CH>([&](uint32_t i) { return row4<AL>(h_in, i, P); }, P, lane, v);
    const uint32_t p = (wv * P + j0) / 16;
    constexpr int KE = kEarly<KU> ? KU : 1;       /* late: one panel's registers at a time */
    v4i wxv[KE], whv[KE];
    if constexpr (kEarly<KU>) {
        panel_load<KU>(wx, wstride, p, kr, lane, wxv);
        panel_load<KU>(wh, wstride, p, kr, lane, whv);
    }
    const uint32_t r = wv * P + j0 + (lane & 15);
    const float wxsr = wxs[r], whsr = whs[r], br = b ? b[r] : 0.0f;
    const float cold = threadIdx.x < 16 ? c[j0 + threadIdx.x] : 0.0f;
    if (wv == 0) {
        const float d = quant_loaded<CH>(v, P, kr, qx, lane);
        if (lane == 0)
            dq[0] = d;
    } else if (wv == 1) {
        const float d = quant_loaded<CH>(v, P, kr, qh, lane);
        if (lane == 0)
            dq[1] = d;
    }
    __syncthreads();
    int sx, sh;
    if constexpr (kEarly<KU>) {
        sx = panel_sum<KU>(wxv, kr, qx, lane);
        sh = panel_sum<KU>(whv, kr, qh, lane);
    } else {
        sx = panel_dot<KU>(wx, wstride, p, kr, qx, lane);
        sh = panel_dot<KU>(wh, wstride, p, kr, qh, lane);
    }
    if (lane < 16) {
        const float g = gemv_out(sx, dq[0], wxsr, b, br);
        gates[wv][lane] = g + gemv_out(sh, dq[1], whsr, nullptr, 0.0f);
    }
    __syncthreads();
    if (threadIdx.x < 16) {
        const uint32_t t = threadIdx.x, j = j0 + t;
        const float i = pk_sigmoidf(gates[0][t]);
        const float f = pk_sigmoidf(gates[1][t]);
        const float u = pk_tanhf(gates[2][t]);
        const float o = pk_sigmoidf(gates[3][t]);
        const float cj = f * cold + i * u;
        c[j] = cj;
        h_out[j] = o * pk_tanhf(cj);
    }
}

/* The joint's logits (core/decoder.c:83-89): z = relu(f + gp) quantized by
 * every wave, a wave a 16-row panel of jout */
__device__ __forceinline__ float relu_sum(float a, float b) {
    const float v = a + b;
    return v > 0 ? v : 0.0f;
}

template <int CH, int KU, bool AL>
__global__ __launch_bounds__(64) void joint_kernel(float *__restrict__ logit, const int8_t *__restrict__ w,
                                                   uint64_t wstride, const float *__restrict__ ws,
                                                   const float *__restrict__ bias, const float *__restrict__ f,
                                                   const float *__restrict__ gp, uint32_t J, uint32_t kr) {
    __shared__ __attribute__((aligned(16))) int8_t q[64 * KU];
    const int lane = threadIdx.x;
    const uint32_t p = blockIdx.x;
    float4 vf[CH], vg[CH];
    load_row<CH>([&](uint32_t i) { return row4<AL>(f, i, J); }, J, lane, vf);
    load_row<CH>([&](uint32_t i) { return row4<AL>(gp, i, J); }, J, lane, vg);
    v4i wv[KU];
    if constexpr (kEarly<KU>)
        panel_load<KU>(w, wstride, p, kr, lane, wv);
    const uint32_t r = 16 * p + (lane & 15);
    const float wsr = ws[r], br = bias ? bias[r] : 0.0f;
#pragma unroll
    for (int c = 0; c < CH; c++)
        vf[c] = make_float4(relu_sum(vf[c].x, vg[c].x), relu_sum(vf[c].y, vg[c].y), relu_sum(vf[c].z, vg[c].z),
                            relu_sum(vf[c].w, vg[c].w));
    const float d = quant_loaded<CH>(vf, J, kr, q, lane);
    __syncthreads();
    if constexpr (!kEarly<KU>)
        panel_load<KU>(w, wstride, p, kr, lane, wv);
    const int s = panel_sum<KU>(wv, kr, q, lane);
    if (lane < 16)
        logit[r] = gemv_out(s, d, wsr, bias, br);
}

/* core/decoder.c:90-98: the first best token of [0, V] and the first best
 * duration of the n_dur after them. The scan's rule, best = i when
 * logit[i] > logit[best] from best = 0, picks the first index of the
 * maximum over the values that are not NaN, unless logit[0] is NaN (nothing
 * is greater than it). So a lane takes a contiguous run of at most RUN
 * (loaded at once) and keeps its first maximum over non-NaN values, the runs
 * meet in order (ties to the earlier run, +0 and -0 equal as the comparison
 * has them), and a NaN at 0 wins. The durations are few: lane 0 scans them. */
template <int RUN, typename L>
__device__ __forceinline__ void argmax_wave(L logit_at, uint32_t V, uint32_t n_dur, int lane, uint32_t &tok,
                                            uint32_t &dur) {
    const uint32_t n = V + 1, run = (n + 63) / 64, a = lane * run;
    float lv[RUN];
#pragma unroll
    for (int k = 0; k < RUN; k++)
        lv[k] = k < (int)run && a + k < n ? logit_at(a + k) : 0.0f;
    /* the durations' logits, lane i the i-th (up to 64), loaded with the run */
    const float dv = lane < (int)n_dur ? logit_at(V + 1 + lane) : 0.0f;
    float bv = 0.0f;
    int bi = -1;
#pragma unroll
    for (int k = 0; k < RUN; k++) {
        const float v = lv[k];
        if (k < (int)run && a + k < n && v == v && (bi < 0 || v > bv)) {
            bv = v;
            bi = (int)(a + k);
        }
    }
    for (int off = 1; off < 64; off <<= 1) {
        const float ov = __shfl_down(bv, off);
        const int oi = __shfl_down(bi, off);
        if (lane + off < 64 && oi >= 0 && (bi < 0 || ov > bv)) {
            bv = ov;
            bi = oi;
        }
    }
    /* the scan over the durations, each compared with the best so far */
    uint32_t bd = 0;
    if (n_dur <= 64) {
        float bdv = __shfl(dv, 0);
        for (uint32_t i = 1; i < n_dur; i++) {
            const float x = __shfl(dv, (int)i);
            if (x > bdv) {
                bd = i;
                bdv = x;
            }
        }
    } else {
        if (lane == 0)
            for (uint32_t i = 1; i < n_dur; i++)
                if (logit_at(V + 1 + i) > logit_at(V + 1 + bd))
                    bd = i;
        bd = __shfl(bd, 0);
    }
    const float l0 = __shfl(lv[0], 0);          /* lane 0's run starts at token 0 */
    const int b0 = __shfl(bi, 0);
    tok = l0 != l0 || b0 < 0 ? 0u : (uint32_t)b0;
    dur = bd;
}

template <int RUN>
__global__ __launch_bounds__(64) void argmax_kernel(uint32_t *__restrict__ tok_dur, const float *__restrict__ logit,
                                                    uint32_t V, uint32_t n_dur) {
    uint32_t tok, dur;
    argmax_wave<RUN>([&](uint32_t i) { return logit[i]; }, V, n_dur, threadIdx.x, tok, dur);
    if (threadIdx.x == 0) {
        tok_dur[0] = tok;
        tok_dur[1] = dur;
    }
}

/* ------------------------------------------------------- the search -- *
 *
 * TDT's greedy search (core/decoder.c:121-147) over a segment's frames in one
 * launch: the prediction (the label's embedding through the LSTM layers and
 * jpred, :65-79), the joint and its argmax (:81-101), the duration step, the
 * max_symbols rule and the token list, with every state (h, c of each layer,
 * gp, the logits, the frame, the tokens) in HBM and registers, so the host
 * reads nothing between frames.
 *
 * Every workgroup runs the same control flow. A phase (an LSTM layer's step,
 * jpred, the joint's logits) splits its rows over the workgroups as the
 * one-launch kernels above split them, and ends at a grid barrier; after the
 * joint's barrier every workgroup reads all the logits and makes the same
 * argmax, so all of them take the same branch of the search and meet at the
 * same barriers. What one workgroup writes and another reads (h, gp, the
 * logits) goes through agent-scope atomic stores and loads, coherent across
 * the XCDs' L2s, and so does c, which the workgroup that steps it reads
 * back a token later. The launch is
 * cooperative (every workgroup resident at once), and every barrier's wait is
 * bounded: past its iteration limit a workgroup raises the error flag and
 * leaves, and the others see the flag in their waits and leave too, so a
 * launch always ends; the host reads the flag. The bits are the one-launch
 * kernels' (the same helpers in the same order), so the reference's. */

__device__ __forceinline__ float cload(const float *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void cstore(float *p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* chunk i of a row of n floats read coherently, zeros past n */
__device__ __forceinline__ float4 crow4(const float *x, uint32_t i, uint32_t n) {
    const uint32_t k = 4 * i;
    return make_float4(k < n ? cload(x + k) : 0.0f, k + 1 < n ? cload(x + k + 1) : 0.0f,
                       k + 2 < n ? cload(x + k + 2) : 0.0f, k + 3 < n ? cload(x + k + 3) : 0.0f);
}

template <int CH, int KU>
__global__ __launch_bounds__(256) void search_kernel(SearchArgs a) {
    __shared__ __attribute__((aligned(16))) int8_t q0[64 * KU], q1[64 * KU];
    __shared__ float dq[2], gates[4][16];
    __shared__ uint32_t shared_u[3];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint32_t G = gridDim.x, wg = blockIdx.x;
    const uint32_t P = a.P, J = a.J;
    uint32_t nbar = 0;

    /* the grid barrier: this workgroup's stores have landed, then it counts
     * itself in and waits for the G arrivals of barrier nbar; false (leave)
     * on the error flag or past the iteration limit */
    auto barrier = [&]() -> bool {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        nbar++;
        if (wv == 0) {
            /* each workgroup stores the barrier's number to its own slot;
             * wave 0 reads every slot in one load (lane i slot i, G <= 64)
             * until all of them hold it: no two workgroups update one word */
            uint32_t *slot = a.sync + 64;
            if (lane == 0)
                __hip_atomic_store(slot + wg, nbar, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            uint32_t it = 0, bad = 0;
            while (true) {
                const uint32_t v = lane < (int)G ? __hip_atomic_load(slot + lane, __ATOMIC_RELAXED,
                                                                     __HIP_MEMORY_SCOPE_AGENT) : nbar;
                if (__builtin_amdgcn_read_exec() == __ballot(v >= nbar))
                    break;
                if (++it >= a.spin || ((it & 15) == 0 &&
                                       __hip_atomic_load(a.sync + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
                    bad = 1;
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            if (bad && lane == 0)
                __hip_atomic_store(a.sync + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (lane == 0)
                shared_u[2] = bad;
        }
        __syncthreads();
        return shared_u[2] == 0;
    };

    /* one LSTM layer's step on units 16 wg .. + 15 (lstm_kernel's steps):
     * x, h_in and c read, c and h_out stored, all through the coherent
     * accessors (c is this workgroup's own, read back a token later) */
    auto lstm = [&](uint32_t l, const float *x, const float *h_in, float *h_out) {
        if (wg >= P / 16)
            return;
        float *c = a.c + (size_t)l * P;
        const uint32_t j0 = 16 * wg;
        float4 v[CH];
        if (wv == 0)
            load_row<CH>([&](uint32_t i) { return crow4(x, i, P); }, P, lane, v);
        else if (wv == 1)
            load_row<CH>([&](uint32_t i) { return crow4(h_in, i, P); }, P, lane, v);
        const uint32_t pn = (wv * P + j0) / 16;
        v4i wxv[KU], whv[KU];
        panel_load<KU>(a.wx[l], a.lstm_stride, pn, a.kr_p, lane, wxv);
        panel_load<KU>(a.wh[l], a.lstm_stride, pn, a.kr_p, lane, whv);
        const uint32_t r = wv * P + j0 + (lane & 15);
        const float wxsr = a.wxs[l][r], whsr = a.whs[l][r], br = a.b[l] ? a.b[l][r] : 0.0f;
        const float cold = threadIdx.x < 16 ? cload(c + j0 + threadIdx.x) : 0.0f;
        if (wv == 0) {
            const float d = quant_loaded<CH>(v, P, a.kr_p, q0, lane);
            if (lane == 0)
                dq[0] = d;
        } else if (wv == 1) {
            const float d = quant_loaded<CH>(v, P, a.kr_p, q1, lane);
            if (lane == 0)
                dq[1] = d;
        }
        __syncthreads();
        const int sx = panel_sum<KU>(wxv, a.kr_p, q0, lane), sh = panel_sum<KU>(whv, a.kr_p, q1, lane);
        if (lane < 16) {
            const float g = gemv_out(sx, dq[0], wxsr, a.b[l], br);
            gates[wv][lane] = g + gemv_out(sh, dq[1], whsr, nullptr, 0.0f);
        }
        __syncthreads();
        if (threadIdx.x < 16) {
            const uint32_t t = threadIdx.x, j = j0 + t;
            const float i = pk_sigmoidf(gates[0][t]);
            const float f = pk_sigmoidf(gates[1][t]);
            const float u = pk_tanhf(gates[2][t]);
            const float o = pk_sigmoidf(gates[3][t]);
            const float cj = f * cold + i * u;
            cstore(c + j, cj);
            cstore(h_out + j, o * pk_tanhf(cj));
        }
    };

    /* a row of n inputs (value4 gives its chunks) quantized once by wave 0,
     * then one 16-row panel of w a wave (panel 4 wg + wave, those below
     * panels): gemv_out into out, stored coherently */
    auto gemv = [&](auto value4, uint32_t n, uint32_t kr, const int8_t *w, uint64_t stride, const float *ws,
                    const float *bias, uint32_t panels, float *out) {
        const uint32_t pn = 4 * wg + wv;
        const bool mine = pn < panels;
        float4 v[CH];
        if (wv == 0)
            load_row<CH>(value4, n, lane, v);
        v4i wvv[KU];
        if (mine)
            panel_load<KU>(w, stride, pn, kr, lane, wvv);
        const uint32_t r = 16 * pn + (lane & 15);
        const float wsr = mine ? ws[r] : 0.0f, br = mine && bias ? bias[r] : 0.0f;
        if (wv == 0) {
            const float d = quant_loaded<CH>(v, n, kr, q0, lane);
            if (lane == 0)
                dq[0] = d;
        }
        __syncthreads();
        if (mine) {
            const int s = panel_sum<KU>(wvv, kr, q0, lane);
            if (lane < 16)
                cstore(out + r, gemv_out(s, dq[0], wsr, bias, br));
        }
    };

    uint32_t cur = 0;                               /* bit l: which of layer l's two h buffers is current */
    auto predict = [&](uint32_t label) -> bool {
        const float *x = a.embed + (size_t)label * P;
        for (uint32_t l = 0; l < a.L; l++) {
            const uint32_t c0 = (cur >> l) & 1;
            const float *h_in = a.h + ((size_t)l * 2 + c0) * P;
            float *h_out = a.h + ((size_t)l * 2 + (c0 ^ 1)) * P;
            lstm(l, x, h_in, h_out);
            cur ^= 1u << l;
            if (!barrier())
                return false;
            x = h_out;
        }
        const float *hl = x;
        gemv([&](uint32_t i) { return crow4(hl, i, P); }, P, a.kr_p, a.jpred, a.jpred_stride, a.jpred_s, a.jpred_b,
             J / 16, a.gp);
        return barrier();
    };

    /* the joint at frame t: relu(f + gp) quantized, jout's panels, then every
     * workgroup's wave 0 takes the argmax of all the logits */
    auto joint = [&](uint32_t t, uint32_t &k, uint32_t &di) -> bool {
        const float *ft = a.f + (size_t)t * J;
        auto zrow = [&](uint32_t i) {
            const float4 fv = row4<false>(ft, i, J), gv = crow4(a.gp, i, J);
            return make_float4(relu_sum(fv.x, gv.x), relu_sum(fv.y, gv.y), relu_sum(fv.z, gv.z),
                               relu_sum(fv.w, gv.w));
        };
        gemv(zrow, J, a.kr_j, a.jout, a.jout_stride, a.jout_s, a.jout_b, a.rows_out / 16, a.logit);
        if (!barrier())
            return false;
        if (wv == 0) {
            uint32_t tk, dd;
            argmax_wave<32>([&](uint32_t i) { return cload(a.logit + i); }, a.V, a.n_dur, lane, tk, dd);
            if (lane == 0) {
                shared_u[0] = tk;
                shared_u[1] = dd;
            }
        }
        __syncthreads();
        k = shared_u[0];
        di = shared_u[1];
        __syncthreads();
        return true;
    };

    const uint32_t T = a.T, blank = a.blank;
    uint32_t ntoks = 0, status = 0;
    if (!predict(blank))
        return;
    uint32_t t = 0, last = 0xffffffffu, lasts = 0;
    while (t < T) {
        uint32_t k, di, d, at;
        do {
            at = t;
            if (!joint(t, k, di))
                return;
            d = (uint32_t)a.dur[di];
            if (k == blank && d == 0)
                d = 1;
            t += d;
        } while (k == blank && t < T);
        if (k == blank)
            break;
        if (ntoks == a.cap) {
            status = 2;
            break;
        }
        if (wg == 0 && threadIdx.x == 0) {
            a.toks[3 * ntoks] = (int32_t)k;
            a.toks[3 * ntoks + 1] = (int32_t)at;
            a.toks[3 * ntoks + 2] = a.dur[di];
        }
        ntoks++;
        lasts = last == at ? lasts + 1 : 1;
        last = at;
        if (!predict(k))
            return;
        if (lasts >= a.max_symbols && last == t)
            t++;
    }
    if (wg == 0 && threadIdx.x == 0) {
        a.out[0] = ntoks;
        a.out[1] = status;
    }
}

/* The resident search: the same search where every panel fits the chip's
 * registers (a.L <= kResLayers, panels of kResUnits units), each workgroup of
 * eight waves holding its rows of every matrix for the whole segment: waves
 * 0 to 3 a gate each of 16 units' wx rows of every layer, waves 4 to 7 their
 * wh rows; wave 4 a jpred panel too, waves 5 and 6 a jout panel each. What
 * bounds it is the exchange between workgroups, four of them a token (each
 * layer's h, gp, the joint's best), so an exchange is one trip through
 * memory: every value travels as one 64-bit word with the number of the step
 * it belongs to (agent scope, coherent across the XCDs' L2s), and its readers
 * poll the values themselves. A barrier and a load after it, as the streaming
 * kernel above has them, are three trips.
 *
 * Words are never overwritten while someone may still read them: each h and
 * gp word changes once a prediction, and between two predictions lies a
 * joint, whose words every workgroup writes (its two panels' bests, empty
 * where it has none) only after it has read h and gp, and reads whole before
 * it goes on; the joint's own words alternate between two sets. Words start
 * at zero and steps count from 1.
 *
 * The joint's logits do not travel: a panel's wave reduces its 16 to the
 * best (argmax_wave's rule: a key ordered as the values are, both zeros
 * alike, NaN below all, a NaN at token 0 above all; the first of equal keys),
 * the durations' travel as keys. Between two exchanges wave 0 polls and
 * quantizes and nothing else: the wh half of a layer's step needs only the h
 * that the prediction before made, so waves 4 to 7 sum it while the h moves
 * on, and wave 7 keeps frames in a ring in LDS up to kRingFrames ahead.
 * Waits are bounded as above.
 *
 * Measured, the model's shapes (40 workgroups), 384 frames with 123 tokens
 * and 133 joints: 1.29 ms a launch where the same panels resident with a
 * barrier an exchange took 2.89 ms; of an exchange's 2.6 us, 1.55 us is the
 * wait for the words, 0.35 us the row's quantize, 0.45 us the sums and the
 * activations (with v_dot4 chains and one lane a whole cell: 1.4 us). */
constexpr int kRingFrames = 8;

/* (non-NaN) values as unsigned keys in the order of the values, +0 and -0
 * one key, above 0; NaN: 0 */
__device__ __forceinline__ uint32_t order_key(float v) {
    const uint32_t b = __float_as_uint(v + 0.0f);
    return v == v ? ((b & 0x80000000u) ? ~b : b | 0x80000000u) : 0u;
}

/* the largest of the wave's, all lanes active (wave_max_nonneg's steps) */
__device__ __forceinline__ uint32_t wave_max_u(uint32_t v) {
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

/* chunk i of a row of whole chunks, from any float's address (one 16-byte
 * load: the hardware takes it at 4-byte alignment) */
typedef float v4fu __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ float4 row4u(const float *x, uint32_t i) {
    const v4fu v = *(const v4fu *)(x + 4 * i);
    return make_float4(v.x, v.y, v.z, v.w);
}

/* The resident panels have KU units always, those past the matrix zero, so
 * their sums have no branches (whatever bytes q holds there meet zeros). */
template <int KU>
__device__ __forceinline__ void panel_load_whole(const int8_t *__restrict__ w, uint64_t wstride, uint32_t p,
                                                 uint32_t kr, int lane, v4i (&wv)[KU]) {
    const int8_t *wp = w + (size_t)p * kUnitBytes + lane * 16;
#pragma unroll
    for (int u = 0; u < KU; u++)
        wv[u] = u < (int)kr ? *(const v4i *)(wp + (size_t)u * wstride) : v4i{ 0, 0, 0, 0 };
}

/* The sums of a panel's 16 rows on the matrix cores: the unit's 16 rows by
 * 64 inputs are an operand as they are, the vector is the other one's every
 * column (lane l holds inputs 16 (l / 16) .. + 15, whatever its column), so
 * lane l gets rows 4 (l / 16) + 0 .. 3 with no exchange between lanes, and
 * keeps row_of(l). Exact int32 sums, two chains. */
__device__ __forceinline__ int row_of(int lane) { return 4 * (lane >> 4) + (lane & 3); }

template <int KU>
__device__ __forceinline__ int panel_sum_whole(const v4i (&wv)[KU], const int8_t *q, int lane) {
    const int8_t *qp = q + (lane >> 4) * 16;
    v4i s[2] = { { 0, 0, 0, 0 }, { 0, 0, 0, 0 } };
#pragma unroll
    for (int u = 0; u < KU; u++)
        s[u & 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wv[u], *(const v4i *)(qp + 64 * u), s[u & 1], 0, 0, 0);
    s[0] += s[1];
    const int lo = lane & 1 ? s[0][1] : s[0][0], hi = lane & 1 ? s[0][3] : s[0][2];
    return lane & 2 ? hi : lo;
}

__device__ __forceinline__ uint64_t wload(const uint64_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void wstore(uint64_t *p, uint32_t hi, uint32_t lo) {
    __hip_atomic_store(p, (uint64_t)hi << 32 | lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ __launch_bounds__(512) void search_resident_kernel(SearchArgs a) {
    constexpr int KU = kResUnits, RL = kResLayers, CH = (16 * KU + 63) / 64;
    __shared__ __attribute__((aligned(16))) int8_t qx[64 * KU], qh[RL][64 * KU];
    __shared__ float dx, dh[RL], gates[4][16], hsum[RL][4][16];
    __shared__ uint32_t s_tok, s_dur, s_bad;
    __shared__ __attribute__((aligned(16))) float ring[kRingFrames][64 * KU];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t G = gridDim.x, wg = blockIdx.x, P = a.P, J = a.J, T = a.T;
    const bool has_units = wg < P / 16;
    const int row = row_of(lane);                   /* this lane's row of a panel; */
    const bool own = (lane & 12) == 0;              /* four lanes have it, the first speaks for it */

    /* everything this workgroup keeps, loaded once: wr the wave's gate panel
     * of each layer's wx or wh with its rows' scales and wx's biases, wj its
     * jpred or jout panel */
    v4i wr[RL][KU], wj[KU];
    float rs[RL], rb[RL], creg[RL], jsr = 0.0f, jbr = 0.0f;
#pragma unroll
    for (int l = 0; l < RL; l++) {
        rs[l] = rb[l] = creg[l] = 0.0f;
        if (has_units && l < (int)a.L) {
            const uint32_t pn = ((wv & 3) * P) / 16 + wg, r = 16 * pn + row;
            panel_load_whole<KU>(wv < 4 ? a.wx[l] : a.wh[l], a.lstm_stride, pn, a.kr_p, lane, wr[l]);
            rs[l] = (wv < 4 ? a.wxs[l] : a.whs[l])[r];
            rb[l] = wv < 4 && a.b[l] ? a.b[l][r] : 0.0f;
        }
    }
    const bool jp = wv == 4, jo = wv == 5 || wv == 6;
    const uint32_t my_panel = jp ? wg : wg + (wv - 5) * G;
    const bool mine = (jp && my_panel < J / 16) || (jo && my_panel < a.rows_out / 16);
    if (mine) {
        const uint32_t r = 16 * my_panel + row;
        panel_load_whole<KU>(jp ? a.jpred : a.jout, jp ? a.jpred_stride : a.jout_stride, my_panel,
                             jp ? a.kr_p : a.kr_j, lane, wj);
        const float *bb = jp ? a.jpred_b : a.jout_b;
        jsr = (jp ? a.jpred_s : a.jout_s)[r];
        jbr = bb ? bb[r] : 0.0f;
    }
    if (threadIdx.x == 0)
        s_bad = 0;

    /* wave 0: load() until it finds every word it wants (a lane's ok); s_bad
     * past the iteration limit or where another workgroup has given up */
    auto poll = [&](auto load) {
        for (uint32_t it = 0;;) {
            if (__ballot(load()) == __builtin_amdgcn_read_exec())
                return;
            if (++it >= a.spin || ((it & 63) == 0 && __hip_atomic_load(a.sync + 1, __ATOMIC_RELAXED,
                                                                       __HIP_MEMORY_SCOPE_AGENT))) {
                if (lane == 0) {
                    __hip_atomic_store(a.sync + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    s_bad = 1;
                }
                return;
            }
        }
    };
    /* wave 0: n words (a multiple of 16, at most 64 KU) of step tag into v,
     * a lane's chunks as load_row has them */
    auto poll_row = [&](const uint64_t *w, uint32_t n, uint32_t tag, float4 (&v)[CH]) {
        poll([&]() {
            uint64_t x[CH][4];
#pragma unroll
            for (int c = 0; c < CH; c++) {
                const uint32_t i = lane + 64 * c;
#pragma unroll
                for (int e = 0; e < 4; e++)
                    x[c][e] = 4 * i < n ? wload(w + 4 * i + e) : (uint64_t)tag;
            }
            bool ok = true;
#pragma unroll
            for (int c = 0; c < CH; c++) {
                v[c] = make_float4(__uint_as_float((uint32_t)(x[c][0] >> 32)), __uint_as_float((uint32_t)(x[c][1] >> 32)),
                                   __uint_as_float((uint32_t)(x[c][2] >> 32)), __uint_as_float((uint32_t)(x[c][3] >> 32)));
#pragma unroll
                for (int e = 0; e < 4; e++)
                    ok = ok && (uint32_t)x[c][e] == tag;
            }
            return ok;
        });
    };

    /* the ring holds frames max(lo, hi - kRingFrames) .. hi - 1; wave 7 adds
     * the next four at most of frames from .. from + kRingFrames - 1 (a zero
     * duration comes back to frame from, which stays) */
    uint32_t lo = 0, hi = 0;
    auto ring_fill = [&](uint32_t from) {
        if (from > hi)
            lo = hi = from;
        const uint32_t end = min(min(from + (uint32_t)kRingFrames, T), hi + 4);
        if (wv == 7) {
            float4 v[4][CH];
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (hi + k < end) {
                    const float *fr = a.f + (size_t)(hi + k) * J;
                    load_row<CH>([&](uint32_t i) { return row4u(fr, i); }, J, lane, v[k]);
                }
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (hi + k < end)
#pragma unroll
                    for (int c = 0; c < CH; c++)
                        if (4 * (lane + 64 * c) < J)
                            *(float4 *)&ring[(hi + k) % kRingFrames][4 * (lane + 64 * c)] = v[k][c];
        }
        hi = hi > end ? hi : end;
    };
    ring_fill(0);
    /* the first prediction's h is zero: a row quantized to d = 0 and sums 0 */
    if (wv >= 4 && own)
#pragma unroll
        for (int l = 0; l < RL; l++)
            hsum[l][wv - 4][row] = gemv_out(0, 0.0f, rs[l], nullptr, 0.0f);
    __syncthreads();

    uint32_t step = 0, jstep = 0;                   /* predictions and joints so far */
    bool fresh = false;                             /* gp not read since the last prediction */
    float4 vg[CH];

    /* layer l's step of units 16 wg .. + 15 from the quantized x and the wh
     * half at hand: wave w's gate with its activation, then, the gates met in
     * LDS, the cell and the word of each unit's h; l is a constant at every
     * call */
    auto gate = [&](int l, const int8_t *q, float d) {
        float g = gemv_out(panel_sum_whole<KU>(wr[l], q, lane), d, rs[l], a.b[l], rb[l]);
        g = g + hsum[l][wv][row];
        g = wv == 2 ? pk_tanhf(g) : pk_sigmoidf(g);
        if (own)
            gates[wv][row] = g;
    };
    auto cell = [&](int l) {
        if (threadIdx.x < 16) {
            const uint32_t t = threadIdx.x;
            const float cj = gates[1][t] * creg[l] + gates[0][t] * gates[2][t];
            creg[l] = cj;
            wstore(a.hw + (size_t)l * P + 16 * wg + t, __float_as_uint(gates[3][t] * pk_tanhf(cj)), step);
        }
    };

    auto predict = [&](uint32_t label) -> bool {
        step++;
        fresh = true;
        if (wv == 0 && has_units) {
            float4 v[CH];
            const float *x = a.embed + (size_t)label * P;
            load_row<CH>([&](uint32_t i) { return row4u(x, i); }, P, lane, v);
            const float d = quant_loaded<CH>(v, P, a.kr_p, qx, lane);
            if (lane == 0)
                dx = d;
        }
        __syncthreads();
        if (has_units && wv < 4)
            gate(0, qx, dx);
        __syncthreads();
#pragma unroll
        for (int l = 0; l < RL; l++)
            if (l < (int)a.L) {
                /* h of layer l whole: the next layer's x (or jpred's row) and
                 * this layer's h_in of the next prediction */
                const bool last = l + 1 == (int)a.L;
                if (wv == 0) {
                    if (has_units)
                        cell(l);
                    float4 v[CH];
                    poll_row(a.hw + (size_t)l * P, P, step, v);
                    const float d = quant_loaded<CH>(v, P, a.kr_p, qh[l], lane);
                    if (lane == 0)
                        dh[l] = d;
                }
                __syncthreads();
                if (s_bad)
                    return false;
                if (last && jp && mine) {
                    const float o = gemv_out(panel_sum_whole<KU>(wj, qh[l], lane), dh[l], jsr, a.jpred_b, jbr);
                    if (own)
                        wstore(a.gpw + 16 * my_panel + row, __float_as_uint(o), step);
                }
                if (has_units) {
                    if (wv >= 4) {
                        const float o = gemv_out(panel_sum_whole<KU>(wr[l], qh[l], lane), dh[l], rs[l], nullptr, 0.0f);
                        if (own)
                            hsum[l][wv - 4][row] = o;
                    } else if (!last && l + 1 < RL) {
                        gate(l + 1 < RL ? l + 1 : l, qh[l], dh[l]);
                    }
                }
                if (!last)
                    __syncthreads();
            }
        return true;
    };

    /* the joint at frame t: every panel's best out, all of them in */
    auto joint = [&](uint32_t t, uint32_t &k, uint32_t &di) -> bool {
        jstep++;
        const uint32_t tag = jstep & 0xfffffu;
        uint64_t *tw = a.jw + (size_t)(jstep & 1) * kJointWords, *dw = tw + 128;
        if (wv == 0) {
            float4 v[CH];
            if (t >= lo && t < hi && hi - t <= (uint32_t)kRingFrames)
                load_row<CH>([&](uint32_t i) { return *(const float4 *)&ring[t % kRingFrames][4 * i]; }, J, lane, v);
            else
                load_row<CH>([&](uint32_t i) { return row4u(a.f + (size_t)t * J, i); }, J, lane, v);
            if (fresh)
                poll_row(a.gpw, J, step, vg);
#pragma unroll
            for (int c = 0; c < CH; c++)
                v[c] = 4 * (lane + 64 * c) < J
                           ? make_float4(relu_sum(v[c].x, vg[c].x), relu_sum(v[c].y, vg[c].y),
                                         relu_sum(v[c].z, vg[c].z), relu_sum(v[c].w, vg[c].w))
                           : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            const float d = quant_loaded<CH>(v, J, a.kr_j, qx, lane);
            if (lane == 0)
                dx = d;
        }
        fresh = false;
        __syncthreads();
        if (s_bad)
            return false;
        if (jo) {
            uint32_t best = 0, at = 0;
            if (mine) {
                const float v = gemv_out(panel_sum_whole<KU>(wj, qx, lane), dx, jsr, a.jout_b, jbr);
                const uint32_t r = 16 * my_panel + row;
                const uint32_t key = (r == 0 || r == a.V + 1) && v != v ? ~0u : order_key(v);
                const uint32_t tk = r <= a.V ? key : 0u;
                best = wave_max_u(tk);
                at = 16 * my_panel + (uint32_t)row_of(__builtin_ctzll(__ballot(tk == best)));
                if (own && r > a.V && r <= a.V + a.n_dur)
                    wstore(dw + (r - a.V - 1), key, tag);
            }
            if (lane == 0)
                wstore(tw + wg + (wv - 5) * G, best, (best ? at : 0u) << 20 | tag);
        }
        ring_fill(t);
        if (wv == 0) {
            uint64_t xa, xb, xd;
            poll([&]() {
                xa = lane < (int)(2 * G) ? wload(tw + lane) : (uint64_t)tag;
                xb = 64 + lane < (int)(2 * G) ? wload(tw + 64 + lane) : (uint64_t)tag;
                xd = lane < (int)a.n_dur ? wload(dw + lane) : (uint64_t)tag;
                return ((uint32_t)xa & 0xfffffu) == tag && ((uint32_t)xb & 0xfffffu) == tag && (uint32_t)xd == tag;
            });
            const uint32_t ka = (uint32_t)(xa >> 32), kb = (uint32_t)(xb >> 32), kd = (uint32_t)(xd >> 32);
            const uint32_t ma = wave_max_u(ka), mb = wave_max_u(kb), md = wave_max_u(kd);
            const int la = __builtin_ctzll(__ballot(ka == ma)), lb = __builtin_ctzll(__ballot(kb == mb));
            const uint32_t ta = (uint32_t)__builtin_amdgcn_readlane((int)((uint32_t)xa >> 20), la);
            const uint32_t tb = (uint32_t)__builtin_amdgcn_readlane((int)((uint32_t)xb >> 20), lb);
            const uint32_t ld = (uint32_t)__builtin_ctzll(__ballot(kd == md));
            if (lane == 0) {
                s_tok = mb > ma ? tb : ta;
                s_dur = ld;
            }
        }
        __syncthreads();
        if (s_bad)
            return false;
        k = s_tok;
        di = s_dur;
        return true;
    };

    /* one copy of each phase's code: the first prediction is the blank's */
    const uint32_t blank = a.blank;
    uint32_t ntoks = 0, status = 0, k = blank, t = 0, last = 0xffffffffu, lasts = 0;
    while (true) {
        if (!predict(k))
            return;
        if (lasts >= a.max_symbols && last == t)
            t++;
        if (t >= T)
            break;
        uint32_t di, d, at;
        do {
            at = t;
            if (!joint(t, k, di))
                return;
            d = (uint32_t)a.dur[di];
            if (k == blank && d == 0)
                d = 1;
            t += d;
        } while (k == blank && t < T);
        if (k == blank)
            break;
        if (ntoks == a.cap) {
            status = 2;
            break;
        }
        if (wg == 0 && threadIdx.x == 0) {
            a.toks[3 * ntoks] = (int32_t)k;
            a.toks[3 * ntoks + 1] = (int32_t)at;
            a.toks[3 * ntoks + 2] = a.dur[di];
        }
        ntoks++;
        lasts = last == at ? lasts + 1 : 1;
        last = at;
    }
    if (wg == 0 && threadIdx.x == 0) {
        a.out[0] = ntoks;
        a.out[1] = status;
    }
}

/* ---------------------------------------------------------- launchers -- */

static bool al16(const void *p) { return ((uintptr_t)p & 15) == 0; }

/* The row's float4 chunks a lane and the panel's units a wave: up to 1024
 * inputs in 16 units, or 4096 in 64; float4 loads when the rows are 16-byte
 * aligned and n a multiple of 4 (al). */
#define PK_DEC_SIZE(n, kr, al, CALL)                        \
    do {                                                    \
        if ((n) <= 1024 && (kr) <= 16) {                    \
            constexpr int CH = 4, KU = 16;                  \
            if (al) {                                       \
                constexpr bool AL = true;                   \
                CALL;                                       \
            } else {                                        \
                constexpr bool AL = false;                  \
                CALL;                                       \
            }                                               \
        } else {                                            \
            constexpr int CH = 16, KU = 64;                 \
            if (al) {                                       \
                constexpr bool AL = true;                   \
                CALL;                                       \
            } else {                                        \
                constexpr bool AL = false;                  \
                CALL;                                       \
            }                                               \
        }                                                   \
    } while (0)

int launch_gemv(float *out, const int8_t *w, uint64_t wstride, const float *ws, const float *bias, const float *x,
                uint32_t rows, uint32_t n, uint32_t kr, int add, hipStream_t s) {
    if (n == 0 || n > kDecMaxCols || rows % 16 || 64 * kr > kDecMaxCols || 64 * kr < n)
        return -2;
    const bool al = n % 4 == 0 && al16(x);
    PK_DEC_SIZE(n, kr, al,
                (gemv_kernel<CH, KU, AL><<<rows / 16, 64, 0, s>>>(out, w, wstride, ws, bias, x, n, kr, add)));
    return hipPeekAtLastError() == hipSuccess ? 0 : -1;
}

int launch_lstm(float *h_out, float *c, const float *h_in, const float *x, const int8_t *wx, const float *wxs,
                const int8_t *wh, const float *whs, uint64_t wstride, const float *b, uint32_t P, uint32_t kr,
                hipStream_t s) {
    if (P == 0 || P % 16 || P > kDecMaxCols || 64 * kr > kDecMaxCols || 64 * kr < P)
        return -2;
    const bool al = al16(x) && al16(h_in);
    PK_DEC_SIZE(P, kr, al,
                (lstm_kernel<CH, KU, AL><<<P / 16, 256, 0, s>>>(h_out, c, h_in, x, wx, wxs, wh, whs, wstride, b, P,
                                                                kr)));
    return hipPeekAtLastError() == hipSuccess ? 0 : -1;
}

int launch_joint(float *logit, uint32_t *tok_dur, const int8_t *w, uint64_t wstride, const float *ws,
                 const float *bias, const float *f, const float *gp, uint32_t rows, uint32_t J, uint32_t kr,
                 uint32_t V, uint32_t n_dur, hipStream_t s) {
    if (J == 0 || J > kDecMaxCols || rows % 16 || 64 * kr > kDecMaxCols || 64 * kr < J || V + 1 + n_dur > rows ||
        n_dur == 0 || V + 1 > 64 * 64)
        return -2;
    const bool al = J % 4 == 0 && al16(f) && al16(gp);
    PK_DEC_SIZE(J, kr, al,
                (joint_kernel<CH, KU, AL><<<rows / 16, 64, 0, s>>>(logit, w, wstride, ws, bias, f, gp, J, kr)));
    if (V + 1 <= 64 * 32)
        argmax_kernel<32><<<1, 64, 0, s>>>(tok_dur, logit, V, n_dur);
    else
        argmax_kernel<64><<<1, 64, 0, s>>>(tok_dur, logit, V, n_dur);
    return hipPeekAtLastError() == hipSuccess ? 0 : -1;
}

static bool g_search_resident = true;

bool set_search_resident(bool on) {
    const bool was = g_search_resident;
    g_search_resident = on;
    return was;
}

/* The workspace: the flags, the tokens, then what the kernel's workgroups
 * exchange: h, c, gp and the logits of the streaming kernel, or the resident
 * kernel's words (h's and gp's, and the joint's two sets). */
static size_t up256(size_t x) { return (x + 255) & ~(size_t)255; }

size_t search_workspace_bytes(uint32_t L, uint32_t P, uint32_t J, uint32_t rows_out, uint32_t cap) {
    const size_t loaded = up256((size_t)L * P * 4) + up256((size_t)J * 4) + up256((size_t)rows_out * 4);
    const size_t words = up256((size_t)J * 8) + up256((size_t)2 * kJointWords * 8);
    return up256(512) + up256((size_t)cap * 12) + up256((size_t)L * P * 8) + (loaded > words ? loaded : words) + 256;
}

int launch_search(SearchArgs &a, void *ws, hipStream_t s, const char **name) {
    if (a.P == 0 || a.P % 16 || a.P > 1024 || a.J == 0 || a.J % 16 || a.J > 1024 || a.L == 0 ||
        a.L > (uint32_t)kMaxDecLayers || a.rows_out % 16 || a.V + 1 + a.n_dur > a.rows_out || a.n_dur == 0 ||
        a.n_dur > 64 || a.V + 1 > 64 * 32 || 64 * a.kr_p < a.P || a.kr_p > 16 || 64 * a.kr_j < a.J || a.kr_j > 16)
        return -2;
    /* resident: every panel's units and every layer's gate panels fit
     * (kr <= kResUnits, L <= kResLayers) and at most 64 workgroups have a
     * jpred panel and two jout panels each at most (the jout panels' words
     * are read two a lane of one wave); else the panels are loaded each token */
    uint32_t Gr = a.P / 16;
    Gr = Gr > a.J / 16 ? Gr : a.J / 16;
    Gr = Gr > (a.rows_out / 16 + 1) / 2 ? Gr : (a.rows_out / 16 + 1) / 2;
    const bool res = g_search_resident && a.L <= (uint32_t)kResLayers && a.kr_p <= (uint32_t)kResUnits &&
                     a.kr_j <= (uint32_t)kResUnits && Gr <= 64;
    uint32_t G = a.P / 16;
    G = G > (a.rows_out / 16 + 3) / 4 ? G : (a.rows_out / 16 + 3) / 4;
    G = G > (a.J / 16 + 3) / 4 ? G : (a.J / 16 + 3) / 4;
    if (res)
        G = Gr;
    if (G > 64)
        return -2;                              /* the barrier reads every workgroup's slot in one wave */
    char *p = (char *)ws;
    a.sync = (uint32_t *)p;
    a.out = a.sync + 2;
    p += up256(512);
    a.toks = (int32_t *)p;
    p += up256((size_t)a.cap * 12);
    char *state = p;
    size_t zero = up256((size_t)a.L * a.P * 8);
    a.h = (float *)p;
    a.hw = (uint64_t *)p;
    p += zero;
    a.c = (float *)p;
    a.gpw = (uint64_t *)p;
    if (res) {
        a.jw = (uint64_t *)(p + up256((size_t)a.J * 8));
        zero += up256((size_t)a.J * 8) + up256((size_t)2 * kJointWords * 8);
    } else {
        zero += up256((size_t)a.L * a.P * 4);
        p += up256((size_t)a.L * a.P * 4);
        a.gp = (float *)p;
        a.logit = (float *)(p + up256((size_t)a.J * 4));
    }
    /* the arrivals, the flag, the counts and the state (or the words' step
     * numbers) start at zero (c and h: the reference zeroes them a segment,
     * core/decoder.c:158-165); the streaming kernel's logits and gp and the
     * tokens are written before they are read */
    if (hipMemsetAsync(a.sync, 0, 512, s) != hipSuccess || hipMemsetAsync(state, 0, zero, s) != hipSuccess)
        return -1;
    void *args[] = { &a };
    const void *k = res ? (const void *)search_resident_kernel : (const void *)search_kernel<4, 16>;
    const hipError_t e = hipLaunchCooperativeKernel(k, dim3(G), dim3(res ? 512 : 256), args, 0, s);
    *name = res ? "search_resident" : "search";
    return e == hipSuccess ? 0 : -1;
}

}  // namespace pkq8
