// Integrators that give a system several lanes: one 16-lane DPP row per
// system (or per tile of a tiled network), lane i of the row owning equation
// i and column i of the stored matrix.  A lane-per-system attempt
// (kernels_small.h) is one long dependent instruction stream - the three
// Gauss-Jordan inversions and the error test dominate it - so a batch too
// small to fill the device, and the last systems of a large one, run at the
// latency of that stream.  Here the elimination works on all columns at once
// (the pivot column's multipliers reach the other lanes through DPP row
// broadcasts, part of the multiply), so the stream is a third as long (hhe6:
// 1,560 vector instructions against 4,700, and 2.9 us per attempt in a wave
// alone on its SIMD against 10 to 15).  It stays bound by the latency of that
// stream; 6 of a row's 16 lanes work at N = 6.
//
// Exact mode only: each element sees the reference's operations in the
// reference's order (gje_gold.c:56-144, matrix_ops.c:6-27, skipping the
// structurally zero operands as gje_solve_exact does), so results are
// bit-identical to the lane-per-system kernels.
#pragma once
#include <type_traits>

#include "kernels_small.h"

namespace wind {

// f(integral_constant<B>) ... f(integral_constant<E - 1>)
template <int B, int E, class F>
__device__ inline void static_for(F &&f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// The value of lane K of this lane's 16-lane row.
template <int K>
__device__ inline float row_get(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + K, 0xF, 0xF, true));
}
template <int K>
__device__ inline int row_get_i(int v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x150 + K, 0xF, 0xF, true);
}

// out[i] = lane i's v, i < N.
template <int N>
__device__ inline void row_gather(float v, float (&out)[N]) {
    static_for<0, N>([&](auto i) { out[i] = row_get<i>(v); });
}

// v[i] with i the lane's index (selects: registers cannot be indexed.  Constant
// indices from the start: of a loop over v the compiler made a load by index,
// v went to LDS by thread, and the workgroup's sizes for that came from the
// launch packet in host memory, 10 us at the start of every RK2 kernel).
template <int N>
__device__ inline float lane_pick(const float (&v)[N], int li) {
    float r = v[0];
    static_for<1, N>([&](auto i) { r = li == i ? v[i] : r; });
    return r;
}

// The largest err of the row's lanes, a NaN kept (err_max), in every lane:
// rotations by 8, 4, 2, 1 within the row.
template <int CTRL>
__device__ inline double row_ror_d(double v) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ inline double row_err_max(double e) {
    e = err_max(e, row_ror_d<0x128>(e));
    e = err_max(e, row_ror_d<0x124>(e));
    e = err_max(e, row_ror_d<0x122>(e));
    e = err_max(e, row_ror_d<0x121>(e));
    return e;
}

// K independent solves g = inverse(W_k) f by the reference's Gauss-Jordan,
// lane li holding stored column li of each matrix (W[k][q] = row q) and
// receiving component li of g.  In place during the forward sweep: rows below
// li hold the matrix's column until pivot li is taken, and the inverse's
// afterwards.  K > 1 interleaves the solves' dependent chains.
template <int N, int K>
__device__ inline void gje_row_exact(float (&W)[K][N], const float (&f)[N], int li, float (&g)[K]) {
    static_for<0, N>([&](auto r) {
        const bool own = li == r;
        float X[K];
#pragma unroll
        for (int k = 0; k < K; k++) X[k] = (own ? 1.0f : W[k][r]) / row_get<r>(W[k][r]);
#pragma unroll
        for (int q = r + 1; q < N; q++)
#pragma unroll
            for (int k = 0; k < K; k++) {
                const float t = row_get<r>(W[k][q]) * X[k];
                W[k][q] = (own ? 0.0f : W[k][q]) - t;
            }
#pragma unroll
        for (int k = 0; k < K; k++) W[k][r] = X[k];
    });
    float Inv[K][N];
#pragma unroll
    for (int k = 0; k < K; k++)
#pragma unroll
        for (int q = 0; q < N; q++) Inv[k][q] = q < li ? 0.0f : W[k][q];
    static_for<0, N - 1>([&](auto r) {
        constexpr int b = N - 1 - r;
#pragma unroll
        for (int q = b - 1; q >= 0; q--)
#pragma unroll
            for (int k = 0; k < K; k++) Inv[k][q] = Inv[k][q] - row_get<b>(W[k][q]) * Inv[k][b];
    });
#pragma unroll
    for (int k = 0; k < K; k++) {
        float acc = 0.0f;
#pragma unroll
        for (int c = 0; c < N; c++) acc = acc + Inv[k][c] * f[c];
        g[k] = acc;
    }
}

// A network (or one tile of a tiled one) as the row kernels evaluate it: the
// generated networks' tile functions, or a compiled-in network as one tile.
template <class Net, class = void>
struct TileOf {
    static constexpr int NB = Net::N, NTILE = 1;
    static constexpr bool kFirstTile = false;
    template <class M>
    __device__ static inline void rhs(const typename Net::Params &p, const float *c, const float *, const float *y,
                                      float *f) {
        Net::template rhs<M>(p, c, y, f);
    }
    template <class M>
    __device__ static inline void jac(const typename Net::Params &p, const float *c, const float *, const float *y,
                                      float *J) {
        Net::template jac<M>(p, c, y, J);
    }
};
template <class Net>
struct TileOf<Net, std::void_t<decltype(Net::NTILE)>> {
    static constexpr int NB = Net::NB, NTILE = Net::NTILE;
    static constexpr bool kFirstTile = Net::kFirstTile && Net::NTILE > 1;
    template <class M>
    __device__ static inline void rhs(const typename Net::Params &, const float *c, const float *y0, const float *y,
                                      float *f) {
        Net::template rhs_at<M>(c, y0, y, f);
    }
    template <class M>
    __device__ static inline void jac(const typename Net::Params &, const float *c, const float *y0, const float *y,
                                      float *J) {
        Net::template jac_at<M, NB>(c, y0, y, J);
    }
};

// Network evaluation by a row: y (and the first tile's y0) in every lane; f
// in every lane, Jr[k] = d f_li / d y_k of the lane's own equation.  The
// general form evaluates everything in every lane and picks the lane's row.
template <class Net, class M>
struct RowEval {
    using T = TileOf<Net>;
    static constexpr int N = T::NB;
    const typename Net::Params &p;
    int li;
    __device__ RowEval(const typename Net::Params &p_, int li_) : p(p_), li(li_) {}
    template <bool JAC>
    __device__ inline void operator()(const float *c, const float (&y0)[N], const float (&y)[N], float (&f)[N],
                                      float (&Jr)[N]) {
        T::template rhs<M>(p, c, y0, y, f);
        if constexpr (JAC) {
            float J[N * N];
#pragma unroll
            for (int e = 0; e < N * N; e++) J[e] = 0.0f;
            T::template jac<M>(p, c, y0, y, J);
#pragma unroll
            for (int k = 0; k < N; k++) {
                Jr[k] = J[k * N];
#pragma unroll
                for (int i = 1; i < N; i++) Jr[k] = li == i ? J[k * N + i] : Jr[k];
            }
        }
    }
};

// hhe6: lane j takes rate j (lane 7 the square root's exponential), lane k
// the Jacobian column of species k; the columns become rows through the
// row's slice of LDS (a wave's LDS accesses stay in order).
template <>
struct RowEval<NetHHe6, MathExact> {
    static constexpr int N = 6;
    const NetHHe6::Params &p;
    int li;
    float lnA, b, C, dmu, dxe, dion, heat;
    float *buf;  // this row's columns, 8 floats each
    __device__ RowEval(const NetHHe6::Params &p_, int li_) : p(p_), li(li_) {
        __shared__ float rowbuf[16][144];  // rows 16 banks apart
        buf = rowbuf[threadIdx.x >> 4];
        lnA = lane_pick<7>(p.lnA, li);
        b = lane_pick<7>(p.b, li);
        C = lane_pick<7>(p.C, li);
        dmu = li == 4 ? 3.0f : li == 1 || li == 3 ? 2.0f : 1.0f;
        dxe = li == 4 ? 2.0f : li == 1 || li == 3 ? 1.0f : 0.0f;
        dion = li == 4 ? 4.0f : li == 1 || li == 3 ? 1.0f : 0.0f;
        heat = li == 0   ? (p.Gamma[0] * NetHHe6::YR) * NetHHe6::E0
               : li == 2 ? (p.Gamma[1] * NetHHe6::YR) * NetHHe6::E1
               : li == 3 ? (p.Gamma[2] * NetHHe6::YR) * NetHHe6::E2
                         : 0.0f;
    }
    template <bool JAC>
    __device__ inline void operator()(const float *c, const float (&)[N], const float (&y)[N], float (&f)[N],
                                      float (&Jr)[N]) {
        using M = MathExact;
        NetHHe6::State s;
        s.xe = (y[1] + y[3]) + (y[4] + y[4]);
        s.mu = (((y[0] + y[1]) + (y[2] + y[3])) + y[4]) + s.xe;
        const float dTde = M::div(NetHHe6::TUNIT, 1.5f * s.mu);
        const float Traw = y[5] * dTde;
        const bool clamped = !(Traw > NetHHe6::TFLOOR);
        s.T = clamped ? NetHHe6::TFLOOR : Traw;
        s.phi = clamped ? Traw * 0.1f : 1.0f;
        s.invT = M::div(1.0f, s.T);
        s.nHyr = c[0] * NetHHe6::YR;
        s.lnT = M::lg(s.T);
        const float arg = (lnA + b * s.lnT) - C * s.invT;
        const float ev = M::ex(li == 7 ? 0.5f * s.lnT : arg);
        s.sqT = row_get<7>(ev);
        const float R = ev * s.nHyr;
        static_for<0, 7>([&](auto j) { s.Rj[j] = row_get<j>(R); });
#pragma unroll
        for (int j = 0; j < 3; j++) s.G[j] = p.Gamma[j] * NetHHe6::YR;
        NetHHe6::rhs_of(s, y, f);
        if constexpr (JAC) {
            const float gl = R * ((b + C * s.invT) * s.invT);
            static_for<0, 7>([&](auto j) { s.gj[j] = row_get<j>(gl); });
            const float Tmu = M::div(Traw, s.mu);
            const float dTraw = li == 5 ? dTde : -(Tmu * dmu);
            const float dT = clamped ? 0.0f : dTraw;
            const float dphi = clamped ? dTraw * 0.1f : 0.0f;
            float col[6];
            NetHHe6::jac_col(s, y, li, dT, dphi, dxe, dion, heat, col);
            *reinterpret_cast<float4 *>(buf + 8 * li) = make_float4(col[0], col[1], col[2], col[3]);
            *reinterpret_cast<float2 *>(buf + 8 * li + 4) = make_float2(col[4], col[5]);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int k = 0; k < N; k++) Jr[k] = buf[8 * k + li];
            __builtin_amdgcn_wave_barrier();
        }
    }
};

// The two sub-steps of an attempt that start from the same state (full step
// hs1, first half step hs2): own components y1, yh from own component yo.
template <class Net, int METHOD, class Ev, int N>
__device__ inline void row_pair(Ev &ev, const float *c, const float (&y0)[N], const float (&y)[N], float yo, float hs1,
                                float hs2, int li, float &y1, float &yh) {
    float f[N], Jr[N];
    ev.template operator()<METHOD == WIND_SIE>(c, y0, y, f, Jr);
    if constexpr (METHOD == WIND_SIE) {
        float W[2][N], g[2];
        const float nh1 = -hs1, nh2 = -hs2;
#pragma unroll
        for (int q = 0; q < N; q++) {
            const float a = nh1 * Jr[q], b = nh2 * Jr[q];
            W[0][q] = li == q ? a + 1.0f : a;
            W[1][q] = li == q ? b + 1.0f : b;
        }
        gje_row_exact<N, 2>(W, f, li, g);
        y1 = yo + hs1 * g[0];
        yh = yo + hs2 * g[1];
    } else {
        const float fo = lane_pick<N>(f, li);
        y1 = yo + hs1 * fo;
        yh = yo + hs2 * fo;
    }
}

// The second half step: own component of y + hs x.
template <class Net, int METHOD, class Ev, int N>
__device__ inline float row_half(Ev &ev, const float *c, const float (&y0)[N], const float (&y)[N], float yo, float hs,
                                 int li) {
    float f[N], Jr[N];
    ev.template operator()<METHOD == WIND_SIE>(c, y0, y, f, Jr);
    if constexpr (METHOD == WIND_SIE) {
        float W[1][N], g[1];
        const float nh = -hs;
#pragma unroll
        for (int q = 0; q < N; q++) {
            const float a = nh * Jr[q];
            W[0][q] = li == q ? a + 1.0f : a;
        }
        gje_row_exact<N, 1>(W, f, li, g);
        return yo + hs * g[0];
    } else {
        return yo + hs * lane_pick<N>(f, li);
    }
}

// Networks the row kernel is built for: one tile, and few enough equations
// for a row's registers.
template <class Net>
constexpr bool row_network() {
    return TileOf<Net>::NTILE == 1 && Net::N <= 8;
}

// Systems per CU up to which rows are the faster form whatever the systems'
// lengths: the largest batch that the row kernel takes whole, and the number
// of unfinished systems at which a larger one's go on on rows.  At 16 every
// SIMD has one row wave (4 systems).  Kernel times, lane against row kernel:
// hhe6 SIE 1000 systems 338 / 60 ms, 4096 375 / 68, all of 400 attempts 3.1 /
// 1.0; katz96 SIE 80 systems 0.75 / 0.26; katz96 RK2 4096 0.152 / 0.082; NR_test
// SIE 4096 0.162 / 0.117, adaptive 0.073 / 0.069.  More rows than that only pay
// where few systems are long (SIE, 16,384 systems, hhe6 411 / 131, but of one
// length 3.1 / 3.2, katz96 1.2 / 1.6).  Adaptive calls of five equations make too
// few attempts for 16 (katz96 to t = 2, 4096 systems, lanes / rows 36 / 40 us).
constexpr int row_limit_per_cu(int N, int controller) { return N == 5 && controller == WIND_CTRL_ADAPTIVE ? 8 : 16; }

// Equations from which on a call's last systems are handed over (IntegrateArgs::spill).
constexpr int kSpillMinN = 5;

// Where nothing can be handed over (handover false: batches, the server, the
// output-step driver) an implicit method on five or more equations takes 32:
// lanes throughout are the only other choice, and at 32 rows are faster whatever
// the systems' lengths (8192 systems, hhe6 1.7 to 3.6 times, katz96 1.2 to 1.3; at
// 64 per CU, 0.98 and 0.73 times where all are of one length).
inline int row_max_systems(int N, int method, int controller, int num_cu, bool handover) {
    return (!handover && method == WIND_SIE && N >= kSpillMinN ? 32 : row_limit_per_cu(N, controller)) * num_cu;
}

// Threads that give each of nsys systems a row.
inline int row_threads(int nsys) { return 16 * (nsys < (1 << 26) ? nsys : 1 << 26); }

// v = lane src's value where take is set.
template <class T>
__device__ inline void row_take(bool take, int src, T &v) {
    const T x = __shfl(v, src);
    v = take ? x : v;
}

// One system per row, four per wave, taken from the device queue; or (TAIL)
// the systems that the lane kernels before it handed over (a.spill), a row each.
template <class Net, int METHOD, bool TAIL = false>
__global__ void __launch_bounds__(256) row_integrate(IntegrateArgs a, typename Net::Params p) {
    constexpr int N = Net::N, NC = Net::NCONST;
    static_assert(N <= 16, "one equation per lane of a 16-lane row");
    const int li = threadIdx.x & 15;
    const bool mine = li < N;
    unsigned int *const words = reinterpret_cast<unsigned int *>(a.counters);
    unsigned int *head = words + (TAIL ? SPILL_ROW_HEAD : 0);
    const bool second = TAIL && (int)words[SPILL_FIRST] > a.spill_rows;
    const int count = !TAIL ? a.nsys : (int)words[second ? SPILL_SECOND : SPILL_FIRST];
    RowEval<Net, MathExact> ev(p, li);
    float y[N], c[NC > 0 ? NC : 1], yo = 0.0f, tnow = 0.0f, h = 0.0f;
    int sid = 0, unsolved = 0, attempts = 0, status = WIND_STATUS_OK;
    // fill: the queue is empty and the row repeats another row's system,
    // storing nothing: a wave with idle lanes runs slower (lane_integrate_body).
    // hhe6 SIE 100,003 systems, reference controller, 136 -> 127 ms; Katz96, 80
    // systems, 263 -> 238 us; NR_test, 1,024, 121 -> 114 us.
    bool active = false, need = true, fill = false;
    unsigned long long steps = 0;
    // The first system of a row is its own index in the grid; the queue
    // counts on from there, and is not asked where it is empty (its atomics
    // are serial: 40 of 76 us for 4096 systems of NR_test that way).
    const int rows = gridDim.x * (blockDim.x >> 4);
    int next = (blockIdx.x * blockDim.x + threadIdx.x) >> 4;
    for (;;) {
        if (__any(need)) {
            const int got = next >= 0 ? next : rows + row_get_i<0>(queue_fetch(head, need && li == 0 && rows < count));
            next = -1;
            if (need) {
                need = false;
                active = got < count;
                if (active) {
                    if constexpr (TAIL) {
                        const float *r = a.spill + (size_t)(got + (second ? a.spill_cap : 0)) * spill_record_words(N);
                        yo = r[mine ? li : 0];
                        tnow = r[N];
                        h = r[N + 1];
                        unsolved = __float_as_int(r[N + 2]);
                        attempts = __float_as_int(r[N + 3]);
                        sid = __float_as_int(r[N + 4]);
                    } else {
                        sid = a.index ? a.index[got] : got;
                        yo = a.equations[(size_t)sid * N + (mine ? li : 0)];
                        tnow = a.tnow;
                        h = a.h0;
                        unsolved = attempts = 0;
                    }
                    status = WIND_STATUS_OK;
                    row_gather<N>(yo, y);
#pragma unroll
                    for (int k = 0; k < NC; k++) c[k] = a.constants[(size_t)sid * a.const_stride + k];
                }
            }
            const unsigned long long busy = __ballot(active);
            if (busy == 0ull) break;
            if (__ballot(active || fill) != ~0ull) {
                const int src = (__ffsll((long long)busy) - 1) + li;  // the lane's counterpart in the first active row
                const bool take = !active && !fill;
                row_take(take, src, yo);
#pragma unroll
                for (int i = 0; i < N; i++) row_take(take, src, y[i]);
#pragma unroll
                for (int k = 0; k < NC; k++) row_take(take, src, c[k]);
                row_take(take, src, tnow);
                row_take(take, src, h);
                row_take(take, src, unsolved);
                row_take(take, src, attempts);
                if (take) status = WIND_STATUS_OK;
                fill = fill || take;
            }
        }
        const float hh = fminf(a.tend - tnow, h);
        const float tb = tnow + hh;
        const float hs1 = tb - tnow, hs2 = (tb - tnow) / 2.0f;
        float y1, yh, yv[N];
        row_pair<Net, METHOD>(ev, c, y, y, yo, hs1, hs2, li, y1, yh);
        row_gather<N>(yh, yv);
        const float y2 = row_half<Net, METHOD>(ev, c, yv, yv, yh, hs2, li);
        bool flag = false;
        double err = 0.0;
        if (a.controller == WIND_CTRL_REFERENCE) {
            const bool fail = mine && species_fails<METHOD, true>(y1, y2, a.ABS, a.REL);
            flag = ((__ballot(fail) >> (__lane_id() & 48)) & 0xFFFFull) != 0;
        } else {
            err = row_err_max(mine ? err_term(y1, y2, a.ABS, a.REL) : 0.0);
        }
        attempts++;
        if (control_step<METHOD>(a.controller, a.tend, hh, flag, err, tnow, h, unsolved, status)) {
            const bool extrap = METHOD == WIND_RK2 || a.controller != WIND_CTRL_REFERENCE;
            yo = extrap ? 2.0f * y2 - y1 : y2;
            row_gather<N>(yo, y);
        }
        if (status == WIND_STATUS_OK && tnow < a.tend) {
            if (attempts < a.max_attempts) continue;
            status = WIND_STATUS_EXHAUSTED;
        }
        if (active && mine) a.equations[(size_t)sid * N + li] = yo;
        if (active && li == 0) {
            if (a.steps_out) a.steps_out[sid] = 3 * attempts;
            if (a.status_out) a.status_out[sid] = status;
            steps += 3ull * (unsigned long long)attempts;
        }
        // (a row without a system asks again too, to take another to repeat)
        active = fill = false;
        need = true;
    }
    wave_add_steps(a.counters + 1, steps);
}

// Tiled networks in exact mode: the workgroup integrates one system, a row
// per tile.  I - hJ is block-diagonal in the tiles (each tile's Jacobian
// entries lie in its own block), so each row inverts its own NB x NB block:
// the dense Gauss-Jordan's other operations multiply by, or subtract, exact
// zeros, which changes no non-zero bit, and a zero's sign cannot reach the
// result (the mat-vec's sums start at +0).  That holds for finite values; in
// the dense elimination an infinity or a NaN of one tile reaches the others
// through those zeros.  A non-finite f or inverse entry makes its tile's
// sub-step result non-finite, and so does a non-finite matrix entry, through
// the pivot that it meets, but for an infinite diagonal alone: it scales its
// own row to zeros, in the dense elimination as here.  So a system with a
// non-finite result is integrated again, from its start, by the dense path
// (dense(sid)).
// The tiles share the step control, and the first tile's state where the
// network's temporaries read it; both go through LDS, with one barrier per
// attempt for each.
template <class Net>
constexpr int row_tile_threads() {
    return (TileOf<Net>::NTILE * 16 + 63) / 64 * 64;
}

// Networks the tile kernel is built for: at least two tiles, at most 64 (a
// workgroup's 1024 lanes), and few enough equations per tile for a row's
// registers.
template <class Net>
constexpr bool row_tile_network() {
    return TileOf<Net>::NTILE > 1 && TileOf<Net>::NTILE <= 64 && TileOf<Net>::NB <= 8;
}

template <class Net, int METHOD, class Dense>
__device__ inline void row_tile_integrate(const IntegrateArgs &a, const typename Net::Params &p, Dense &&dense) {
    using TT = TileOf<Net>;
    constexpr int NB = TT::NB, T = TT::NTILE, N = NB * T, NC = Net::NCONST, WV = row_tile_threads<Net>() / 64;
    __shared__ float s_mid[NB], s_new[NB];
    __shared__ unsigned s_vote[2][WV];
    __shared__ double s_err[2][WV];
    const int t = threadIdx.x, li = t & 15, wave = t >> 6;
    const bool mine = li < NB && (t >> 4) < T;
    const int tile = (t >> 4) < T ? t >> 4 : T - 1;
    const int own = tile * NB + (li < NB ? li : 0);
    RowEval<Net, MathExact> ev(p, li);
    unsigned long long steps = 0;
    int slot = 0;
    for (int sid = blockIdx.x; sid < a.nsys; sid += gridDim.x) {
        const float *ys = a.equations + (size_t)sid * N;
        float y[NB], y0[NB], c[NC > 0 ? NC : 1], yo = ys[own];
        row_gather<NB>(yo, y);
#pragma unroll
        for (int i = 0; i < NB; i++) y0[i] = TT::kFirstTile ? ys[i] : 0.0f;
#pragma unroll
        for (int k = 0; k < NC; k++) c[k] = a.constants[(size_t)sid * a.const_stride + k];
        float tnow = a.tnow, h = a.h0;
        int unsolved = 0, attempts = 0, status = WIND_STATUS_OK;
        bool finite = true;
        while (tnow < a.tend) {
            const float hh = fminf(a.tend - tnow, h);
            const float tb = tnow + hh;
            const float hs1 = tb - tnow, hs2 = (tb - tnow) / 2.0f;
            float y1, yh, yv[NB], y0v[NB];
            row_pair<Net, METHOD>(ev, c, y0, y, yo, hs1, hs2, li, y1, yh);
            if constexpr (TT::kFirstTile) {
                if (t < NB) s_mid[t] = yh;
                __syncthreads();
            }
#pragma unroll
            for (int i = 0; i < NB; i++) y0v[i] = TT::kFirstTile ? s_mid[i] : 0.0f;
            row_gather<NB>(yh, yv);
            const float y2 = row_half<Net, METHOD>(ev, c, y0v, yv, yh, hs2, li);
            const bool extrap = METHOD == WIND_RK2 || a.controller != WIND_CTRL_REFERENCE;
            const float ynew = extrap ? 2.0f * y2 - y1 : y2;
            if (TT::kFirstTile && t < NB) s_new[t] = ynew;
            bool fail = false;
            if (a.controller == WIND_CTRL_REFERENCE) {
                fail = mine && species_fails<METHOD, true>(y1, y2, a.ABS, a.REL);
            } else {
                double e = row_err_max(mine ? err_term(y1, y2, a.ABS, a.REL) : 0.0);
                e = err_max(e, __shfl_xor(e, 16));
                e = err_max(e, __shfl_xor(e, 32));
                if ((t & 63) == 0) s_err[slot][wave] = e;
            }
            const bool odd = METHOD == WIND_SIE && mine &&
                             !(__builtin_isfinite(y1) && __builtin_isfinite(yh) && __builtin_isfinite(y2));
            const unsigned vote = (__any(fail) ? 1u : 0u) | (__any(odd) ? 2u : 0u);
            if ((t & 63) == 0) s_vote[slot][wave] = vote;
            __syncthreads();
            unsigned all = 0;
            double err = 0.0;
#pragma unroll
            for (int w = 0; w < WV; w++) {
                all |= s_vote[slot][w];
                if (a.controller != WIND_CTRL_REFERENCE) err = err_max(err, s_err[slot][w]);
            }
            slot ^= 1;  // (the next attempt writes while slower waves still read)
            finite = (all & 2u) == 0;
            if (!finite) break;
            attempts++;
            if (control_step<METHOD>(a.controller, a.tend, hh, (all & 1u) != 0, err, tnow, h, unsolved, status)) {
                yo = ynew;
                row_gather<NB>(yo, y);
                if constexpr (TT::kFirstTile)
#pragma unroll
                    for (int i = 0; i < NB; i++) y0[i] = s_new[i];
            }
            if (status != WIND_STATUS_OK) break;
            if (attempts >= a.max_attempts && tnow < a.tend) {
                status = WIND_STATUS_EXHAUSTED;
                break;
            }
        }
        if (finite) {
            if (mine) a.equations[(size_t)sid * N + own] = yo;
            if (t == 0) {
                if (a.steps_out) a.steps_out[sid] = 3 * attempts;
                if (a.status_out) a.status_out[sid] = status;
            }
        } else {
            __syncthreads();
            attempts = dense(sid);
        }
        steps += 3ull * (unsigned long long)attempts;
    }
    if (t == 0 && steps) atomicAdd(a.counters + 1, steps);
}

}  // namespace wind
