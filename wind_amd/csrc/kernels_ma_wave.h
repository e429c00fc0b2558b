// Exact-mode SIE for table-driven mass-action networks with N <= 64: the
// matrix in registers, lane c of a wave owning stored column c (equation c).
//
// The one-workgroup kernel (kernels_mass_action.h) keeps the matrix and its
// inverse in LDS and crosses two barriers per pivot; at N = 32 a sub-step
// took 60 to 70 us of that latency.  Here one wave inverts a matrix without
// a barrier: the pivot column's multipliers come from its lane by v_readlane
// and every lane updates its whole column, three instructions per element
// (readlane, multiply, subtract).  A workgroup of two waves integrates one
// system: both evaluate the network, then one wave takes the full step while
// the other takes the first half step, and the second half step follows.
// Bound by the waves' own instruction streams (the elimination is unrolled
// over all pivots: rolled in groups of four it took 1.7 times as long at
// N = 37 to 64) and the divisions' latency.  512 systems, t = 10^7,
// adaptive, one-workgroup kernel against this one: N = 8 23.0 / 5.6 ms,
// N = 16 46.8 / 11.8, N = 32 97.7 / 19.0, N = 45 301 / 40.5, N = 64 691 /
// 87; 4096 systems N = 32 373 / 32, N = 37 780 / 43; one system 2.8 to 8
// times faster.
//
// The elimination is in place, as in gje_row_exact (kernels_row.h): rows
// below c hold the matrix's column until pivot c and the inverse's
// afterwards.  Every element sees the reference's operations in order
// (gje_gold.c:56-144, matrix_ops.c:6-27), so results are bit-identical to
// the one-workgroup kernel's.
#pragma once
#include "kernels_mass_action.h"
#include "kernels_row.h"

namespace wind {

__device__ inline float lane_value(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// op(q, lane r's W[q]) for q = B .. E - 1, eight reads ahead of their uses (a
// read's result may not be used by the next instruction).
template <int B, int E, int NP, class F>
__device__ inline void column_values(const float (&W)[NP], int r, F &&op) {
#pragma unroll
    for (int q0 = B; q0 < E; q0 += 8) {
        float s[8];
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (q0 + u < E) s[u] = lane_value(W[q0 + u], r);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (q0 + u < E) op(q0 + u, s[u]);
    }
}

// g = inverse(W) f, component `lane`; W[q] = row q of the lane's stored
// column, f in LDS.  N <= NP, a multiple of 8 with NP - N < 8; rows and
// lanes from N on are never read by others.
template <int NP>
__device__ inline float gje_wave_exact(float (&W)[NP], const float *f, int lane, int N) {
    // the lane index made opaque, so that the compiler derives the per-pivot
    // lane masks here instead of keeping NP of them across the passes
    asm volatile("" : "+v"(lane));
    static_for<0, NP>([&](auto r) {
        if (r >= NP - 8 && r >= N) return;
        const bool own = lane == r;
        const float X = (own ? 1.0f : W[r]) / lane_value(W[r], r);
        // the inverse's column starts from 0 below its pivot: 0 - t, as
        // W * 0 - t (the rounding of W * m - t, m = 0 or 1, is the
        // subtraction's)
        const float m = own ? 0.0f : 1.0f;
        W[r] = X;
        column_values<r + 1, NP>(W, r, [&](int q, float sq) { W[q] = fmaf(W[q], m, -(sq * X)); });
    });
    float Inv[NP];
#pragma unroll
    for (int q = 0; q < NP; q++) Inv[q] = q < lane ? 0.0f : W[q];
    static_for<0, NP - 1>([&](auto i) {
        constexpr int b = NP - 1 - i;
        if (b >= NP - 8 && b >= N) return;
        column_values<0, b>(W, b, [&](int q, float sq) { Inv[q] = Inv[q] - sq * Inv[b]; });
    });
    float acc = 0.0f;
#pragma unroll
    for (int c = 0; c < NP; c++)
        if (c < NP - 7 || c < N) acc = acc + Inv[c] * f[c];
    return acc;
}

// LDS of ma_wave_integrate in floats: y, yh, y1, f, the reactions' rate
// terms and the Jacobian (NP x NP, stored columns).
__host__ __device__ constexpr int ma_wave_lds_floats(int NP, int R) { return 4 * NP + NP * NP + 3 * R; }

// Words a thread loads at a time of its term stream (mass_action_build): the
// terms of f and of the Jacobian's elements, dealt to the 128 threads.
constexpr int kMaWaveBatch = 8;

template <int NP>
__global__ void __launch_bounds__(128) ma_wave_integrate(IntegrateArgs a, MassActionDevice net) {
    constexpr int B = kMaWaveBatch;
    extern __shared__ float lds[];
    float *J = lds, *y = J + NP * NP, *yh = y + NP, *y1 = yh + NP, *f = y1 + NP;
    float *w = f + NP, *da = w + net.R, *db = da + net.R;
    __shared__ int s_flag, s_sid;
    __shared__ double s_err;
    const int N = net.N, R = net.R, t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int col = lane < N ? lane : 0;
    const int *__restrict__ sp = net.ex_ent + t;
    unsigned int *head = reinterpret_cast<unsigned int *>(a.counters);
    unsigned long long steps = 0;
    int sid = blockIdx.x;
    while (sid < a.nsys) {
        if (t < N) y[t] = a.equations[(size_t)sid * N + t];
        const float scale = a.constants[(size_t)sid * a.const_stride];
        __syncthreads();
        float tnow = a.tnow, h = a.h0;
        int unsolved = 0, attempts = 0, status = WIND_STATUS_OK;
        while (tnow < a.tend) {
            const float hh = fminf(a.tend - tnow, h);
            const float tb = tnow + hh;
            const float hs_full = tb - tnow, hs_half = (tb - tnow) / 2.0f;
            float y2 = 0.0f;
#pragma unroll 1
            for (int pass = 0; pass < 2; pass++) {
                // rates, f and J at yv: every sum in the order of ma_eval's
                const float *yv = pass ? yh : y;
                int en[B];
#pragma unroll
                for (int u = 0; u < B; u++) en[u] = sp[u * 128];
                for (int r = t; r < R; r += 128) {
                    const float ks = net.k[r] * scale;
                    const float ya = yv[net.rx[4 * r]], yb = yv[net.rx[4 * r + 1]];
                    w[r] = (ks * ya) * yb;
                    da[r] = ks * yb;
                    db[r] = ks * ya;
                }
                for (int e = 4 * t; e < NP * NP; e += 512)
                    *reinterpret_cast<float4 *>(J + e) = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (t < N) f[t] = 0.0f;
                __syncthreads();
                float acc = 0.0f;
                for (int j = 0;;) {
                    float v[B];
                    int e[B];
#pragma unroll
                    for (int u = 0; u < B; u++) {
                        e[u] = en[u];
                        v[u] = lds[(unsigned)e[u] >> 16];
                    }
                    j += B;
                    if (j < net.ex_len)
#pragma unroll
                        for (int u = 0; u < B; u++) en[u] = sp[(j + u) * 128];
#pragma unroll
                    for (int u = 0; u < B; u++) {
                        acc = (e[u] & 1) ? acc - v[u] : acc + v[u];
                        if (e[u] & 2) {
                            lds[(e[u] >> 3) & 8191] = acc;
                            acc = 0.0f;
                        }
                    }
                    if (j >= net.ex_len) break;
                }
                __syncthreads();
                if (pass == 0 || wave == 0) {
                    const float hs = pass == 0 && wave == 1 ? hs_full : hs_half;
                    const float nh = -hs;
                    float W[NP];
                    int own = lane;
                    asm volatile("" : "+v"(own));  // as in gje_wave_exact
#pragma unroll
                    for (int q = 0; q < NP; q++) {
                        const float v = nh * J[q * NP + col];
                        W[q] = q == own ? v + 1.0f : v;
                    }
                    const float g = gje_wave_exact<NP>(W, f, lane, N);
                    const float v = yv[col] + hs * g;
                    if (pass == 0 && lane < N) (wave == 1 ? y1 : yh)[lane] = v;
                    y2 = v;
                }
                if (pass == 0) __syncthreads();
            }
            if (wave == 0) {
                bool flag = false;
                double err = 0.0;
                if (a.controller == WIND_CTRL_REFERENCE) {
                    flag = __any(lane < N && species_fails<WIND_SIE, true>(y1[col], y2, a.ABS, a.REL));
                } else {
                    if (lane < N) err = err_term(y1[col], y2, a.ABS, a.REL);
#pragma unroll
                    for (int off = 32; off > 0; off >>= 1) err = err_max(err, __shfl_xor(err, off));
                }
                if (lane == 0) {
                    s_flag = flag;
                    s_err = err;
                }
            }
            __syncthreads();
            attempts++;
            const bool acc = control_step<WIND_SIE>(a.controller, a.tend, hh, s_flag != 0, s_err, tnow, h, unsolved, status);
            if (acc && t < N) y[t] = a.controller != WIND_CTRL_REFERENCE ? 2.0f * y2 - y1[t] : y2;
            __syncthreads();
            if (status != WIND_STATUS_OK) break;
            if (attempts >= a.max_attempts && tnow < a.tend) {
                status = WIND_STATUS_EXHAUSTED;
                break;
            }
        }
        if (t < N) a.equations[(size_t)sid * N + t] = y[t];
        if (t == 0) {
            if (a.steps_out) a.steps_out[sid] = 3 * attempts;
            if (a.status_out) a.status_out[sid] = status;
            steps += 3ull * (unsigned long long)attempts;
            s_sid = gridDim.x + (int)atomicAdd(head, 1u);
        }
        __syncthreads();
        sid = s_sid;
    }
    if (t == 0 && steps) atomicAdd(a.counters + 1, steps);
}

}  // namespace wind
