// Register-resident dense SIE solver for mass-action networks with
// 16 NT - 15 <= N <= 16 NT (fast mode).  One workgroup of WR x WC waves
// (2 x 2, or 4 x 2 for few systems, dense.hip) owns one system at a time,
// systems taken from a device queue, and the matrix A = I - hJ lives in the
// waves' registers instead of LDS: wave (wi, wj) holds the 16x16 tiles (i, j)
// with i = wi (mod WR), j = wj (mod WC), each in the MFMA accumulator layout
// (lane l holds rows 4(l/16) + q, q = 0..3, of column l % 16).  Without the
// matrix in LDS a workgroup needs a third to an eighth of a CU's LDS and
// registers (dense_reg_wgs_for), so three to eight systems share a CU and each
// one's serial parts (the pivot chain of a diagonal block, the barriers)
// overlap with the others' work.
//
// Per pass (step-doubling sub-step) of an attempt:
// * assembly: the per-reaction rate terms and f as in the LDS solver
//   (kernels_dense.h, dense_eval, same order, so f and every matrix element
//   round identically); f and the matrix elements with Jacobian terms are
//   summed into a compact LDS buffer (dealt to all threads on the host,
//   each element its terms in sweep order, one branch-free stream of term
//   words per thread), and the owner lanes of the tiles read them into
//   registers through per-lane offset and mask words (1 on the diagonal, 0
//   elsewhere where absent), loaded ahead while the tiles' registers are
//   free.  Against f summed from lists of its own by the first N threads,
//   words loaded a tile row at a time and tile addresses and conditions kept
//   in (spilled) registers across the phases, a sub-step went from 21.7 to
//   19.1 us per CU at N = 157, 3.37 to 3.30 at N = 64 and 1.84 to 1.72 at
//   N = 32 with the CU full, and from 51.5 / 12.4 / 7.4 to 46.8 / 10.5 /
//   5.7 us for a system alone on it;
// * block LU without pivoting, A = [I 0; A21 G I][A11 A12; 0 A22 - A21 G A12],
//   G = A11^-1, per 16-column panel k, with two barriers:
//     B: W_kj = G_k A_kj for the row panel (G_k from LDS, A_kj in the
//        owner's registers; W replaces A_kj and goes to LDS), the column
//        panel A_ik to LDS, and the forward sweep: A_ik c_k is added to the
//        row's sums, a lane's columns in the lane; row k + 1, complete, is
//        summed over its lanes;
//     C: the trailing update A_ij -= A_ik W_kj on the matrix cores
//        (v_mfma_f32_16x16x4f32, operands from LDS, accumulator in place);
//        the owner of the next diagonal tile updates it first, inverts it in
//        registers (Gauss-Jordan on its transpose, which the accumulator
//        layout holds as rows), publishes G_{k+1} and forms c_{k+1} =
//        G_{k+1} r_{k+1};
// * backward sweep x_k = c_k - sum_{j>k} W_kj x_j by columns, its sums kept the
//   same way, one barrier per block, the W tiles still in registers;
// * y += h x.
// The sweeps' sums live in the registers of tiles that are no longer needed
// and are reduced (DPP shifts over the 16 lanes of a row, then one partial sum
// per wave column through LDS) once per block row.  Reduced and subtracted in
// LDS per tile instead, a sub-step took 19.1 instead of 17.6 us per CU at
// N = 157 with four systems on it and 37.0 instead of 34.0 us alone, 3.92 /
// 3.81 (four on the CU) and 9.8 / 9.5 (alone) at N = 64, and whole batches 630
// / 579 ms (1,024 systems, N = 157) and 812 / 719 (4,096, N = 100).  Every
// result is deterministic and independent of the grid and of the waves'
// number.  The step control is the LDS solver's.
#pragma once
#include "kernels_dense.h"

namespace wind {

// Workgroups per CU (WGS) the solver is built for: four from seven tiles per
// dimension (N > 96), five at five and six, six at three and four, eight
// below, when the network's LDS footprint allows it (dense_reg_wgs_for); else
// three.  Built for more than three, the kernel reads the rate constants from
// global memory instead of LDS and the compiler keeps it within 512 / WGS
// VGPRs (spilling up to 38 of them).  Measured, whole batches, the
// three-per-CU build (which may leave room for more) against this choice:
// 2,048 systems, N = 112 270 / 249 ms, 128 364 / 320, 144 431 / 421, N = 157 3%
// faster; 8,192 systems, N = 40 117 / 112 (five per CU 119), 80 376 / 344, 96
// 449 / 419; 64 six per CU 193, five 209.  Where the CU is not full the builds
// are within 2% of each other.

// Assembly stream words a thread loads at a time (streams are padded to a
// multiple of it).
constexpr int kDenseRegBatch = 8;

// Row-panel tiles a wave holds at a time in the trailing update: two from
// eight tiles per dimension (N = 157: 2.26 k -> 2.31 k systems/s; N = 64,
// four tiles, 1.5% slower with two), one below.
template <int NT>
constexpr int kDenseRegGW = NT >= 8 ? 2 : 1;

// Wave columns of every shape.
constexpr int kDenseRegWC = 2;

// LDS layout of the register-resident solver (offsets in floats, 16-byte
// aligned): per-system vectors, per-reaction rate terms (the sweeps' partial
// sums in the same place later), reactant indices and rate constants, and a work
// area shared by the assembly's compact element buffer (cap floats) with f
// behind it, and the factorisation's panel buffers.  The term lists stay in
// global memory.
struct DenseRegOffsets {
    int y, yw, y1, r, part, w, hda, hdb, k, ab, work, total;
};

__host__ __device__ inline DenseRegOffsets dense_reg_offsets(int NT, int R, int WGS, int cap) {
    const int NP = 16 * NT;
    auto up = [](int x) { return (x + 3) & ~3; };
    DenseRegOffsets o;
    int p = 0;
    o.y = p;
    p = up(p + NP);
    o.yw = p;
    p = up(p + NP);
    o.y1 = p;
    p = up(p + NP);
    o.r = p;
    p = up(p + NP);
    o.w = p;
    p = up(p + R);
    o.hda = p;
    p = up(p + R);
    o.hdb = p;
    p = up(p + R);
    // the sweeps' partial sums, in the rate terms' place where it is large
    // enough: the terms are read for the last time two barriers before the first
    // of the sums is written, and written again after the sums' last barrier
    constexpr int sums = 3 * kDenseRegWC * 16;
    o.part = p - o.w >= sums ? o.w : p;
    if (p - o.w < sums) p = up(p + sums);
    o.k = p;
    if (WGS == 3) p = up(p + R);  // rate constants in LDS
    o.ab = p;
    p = up(p + 2 * R);
    o.work = p;
    const int lu = (2 * NT + 1) * 256, el = cap + NP;
    p = up(p + (el > lu ? el : lu));
    o.total = p;
    return o;
}

template <int CTRL>
__device__ inline float dpp_f(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}

// Sum over the 16 lanes of each DPP row (lanes 16m .. 16m + 15), as a
// prefix sum: lane 15 of the row ends with the row's total.
__device__ inline float row_sum16(float v) {
    v += dpp_f<0x111>(v);  // row_shr:1
    v += dpp_f<0x112>(v);  // row_shr:2
    v += dpp_f<0x114>(v);  // row_shr:4
    v += dpp_f<0x118>(v);  // row_shr:8
    return v;
}

// Inverts a 16x16 tile held in the accumulator layout (lane (c, g) holds
// T[4g + q][c]) in place.  Read as rows, those registers are T^T in the
// layout diag_block_invert works on (lane (r, g) holds row r, columns
// 4g .. 4g + 3); Gauss-Jordan on T^T gives (T^T)^-1 = (T^-1)^T, which read
// back in the accumulator layout is T^-1.  No pivoting: the leading
// principal minors of T^T are those of T.
__device__ inline void tile_invert_acc(f32x4 &m, int lane) {
    // the lane index made opaque, so that the compiler derives the per-step
    // lane masks here instead of keeping 32 of them live across the kernel
    asm volatile("" : "+v"(lane));
    const int r = lane & 15, g = lane >> 4;
    float a[4] = {m[0], m[1], m[2], m[3]};
#pragma unroll
    for (int k = 0; k < 16; k++) {
        const int kg = k >> 2, kc = k & 3;
        float pv[4];
#pragma unroll
        for (int c = 0; c < 4; c++) pv[c] = row_bcast(a[c], k);
        const float f = row_to_all(a[kc], kg);
        const float rp = __builtin_amdgcn_rcpf(bcast(a[kc], k + 16 * kg));
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const float prow = pv[c] * rp;
            const bool pc = 4 * g + c == k;
            if (r == k)
                a[c] = pc ? rp : prow;
            else
                a[c] = pc ? -f * rp : fmaf(-f, prow, a[c]);
        }
    }
    m = f32x4{a[0], a[1], a[2], a[3]};
}

// dst[4g + q] (q = 0..3, lanes with c = 15 store) = the sum of m[q] over the
// 16 lanes of the lane's DPP row (the columns).
__device__ inline void tile_rowsum_store(const f32x4 &m, float *dst, int lane) {
    const int c = lane & 15, g = lane >> 4;
    f32x4 p;
#pragma unroll
    for (int q = 0; q < 4; q++) p[q] = row_sum16(m[q]);
    if (c == 15) *reinterpret_cast<f32x4 *>(dst + 4 * g) = p;
}

__device__ inline float uniform(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// TRACE: per-attempt trace and replay through a.trace, as in the other
// kernels.
template <int NT, int WGS, int WR, int WC, bool TRACE = false>
__global__ void __launch_bounds__(64 * WR * WC, WGS *WR *WC / 4)
    ma_dense_reg_integrate(IntegrateArgs a, MassActionDevice net) {
    static_assert(WC == kDenseRegWC, "the sweeps' partial sums are laid out for this");
    constexpr int NP = 16 * NT, T = 64 * WR * WC, NR = (NT + WR - 1) / WR, NC = (NT + WC - 1) / WC;
    extern __shared__ float lds[];
    const int N = net.N, R = net.R, t = threadIdx.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wi = wave / WC, wj = wave % WC;
    const int lr = lane & 15, g = lane >> 4;
    const DenseRegOffsets o = dense_reg_offsets(NT, R, WGS, net.sc_cap);
    float *y = lds + o.y, *yw = lds + o.yw, *y1 = lds + o.y1, *rv = lds + o.r;
    float *w = lds + o.w, *hda = lds + o.hda, *hdb = lds + o.hdb, *kk = lds + o.k;
    int2 *ab = reinterpret_cast<int2 *>(lds + o.ab);
    const int *__restrict__ scent = T == 256 ? net.sc_ent : net.sc_ent2;
    const unsigned *__restrict__ sctile = net.sc_tile;
    float *work = lds + o.work, *f = work + net.sc_cap;
    float *Gbuf = work, *Cbuf = work + 256, *Wbuf = work + 256 * (NT + 1);
    // Per-lane bases of this wave's tiles (tile row i = WR ta + wi, column
    // j = WC tb + wj): the accesses below add compile-time offsets.
    constexpr int RS = 256 * WR, CS = 256 * WC;
    float *const cA = Cbuf + wi * 256 + lr * 16 + 4 * g;  // A-operand reads of Cbuf tile i: + ta * RS
    float *const cS = Cbuf + wi * 256 + 64 * g + lr;      // stores to Cbuf tile i: + ta * RS + q * 16
    float *const wB = Wbuf + wj * 256 + lane * 4;          // Wbuf tile j: + tb * CS
    float *const fp = lds + o.part, *const bp = fp + 16 * WC;  // partial sums, by wave column: forward; backward, twice
    float *const xv = work;                                    // the solution (no panel buffer is in use by then)
    for (int r = t; r < R; r += T) {
        ab[r] = make_int2(net.rx[4 * r], net.rx[4 * r + 1]);
        if (WGS == 3) kk[r] = net.k[r];
    }
    __shared__ int s_flag, s_sid, s_rec;
    __shared__ int s_done;
    __shared__ double s_err[WR * WC];
    f32x4 M[NR][NC];
    unsigned long long steps = 0;
    unsigned int *head = reinterpret_cast<unsigned int *>(a.counters);
    __syncthreads();

    // f and A = I - hs J at yv into f and the register tiles (ends with a
    // barrier).
    auto assemble = [&](const float *yv, float scale, float hs) __attribute__((always_inline)) {
        constexpr int B = kDenseRegBatch;
        // (the wave's place made opaque, so that the compiler derives the
        // tiles' conditions and offsets here instead of keeping them all)
        int wv = wave;
        asm volatile("" : "+s"(wv));
        const int wi = wv / WC, wj = wv % WC;
        // the tiles' old values are dead (every tile is stored again below,
        // under conditions the compiler cannot prove cover all of them)
#pragma unroll
        for (int ta = 0; ta < NR; ta++)
#pragma unroll
            for (int tb = 0; tb < NC; tb++) M[ta][tb] = __builtin_nondeterministic_value(M[ta][tb]);
        // This lane's word of each tile: offset << 4 | the mask of its q
        // present; loaded here, the tiles' registers being free, and used
        // after the elements are summed.  (An opaque offset per pass, so that
        // the compiler does not keep them across passes.)
        int tsel = 0;
        asm volatile("" : "+s"(tsel));
        const unsigned *tpass = sctile + tsel + lane;
        unsigned wt[NR][NC];
#pragma unroll
        for (int ta = 0; ta < NR; ta++)
#pragma unroll
            for (int tb = 0; tb < NC; tb++) {
                const int i = WR * ta + wi, jb = WC * tb + wj;
                wt[ta][tb] = (i < NT && jb < NT) ? tpass[(i * NT + jb) * 64] : 0u;
            }
        // the first words of the term stream, loaded while the rate terms
        // and f are formed
        int en[B];
        const int *sp = scent + t;
#pragma unroll
        for (int u = 0; u < B; u++) en[u] = sp[u * T];
        for (int r = t; r < R; r += T) {
            const int2 x = ab[r];
            const float ks = (WGS == 3 ? kk[r] : net.k[r]) * scale;
            const float ya = yv[x.x], yb = yv[x.y];
            w[r] = (ks * ya) * yb;
            hda[r] = hs * (ks * yb);
            hdb[r] = hs * (ks * ya);
        }
        if (t < NP) f[t] = 0.0f;  // species without reactions, and the padding
        __syncthreads();
        // f and the matrix's non-zero elements through a compact buffer: each
        // thread walks its term stream (the elements dealt to the
        // threads on the host, interleaved so that a batch of words is one
        // coalesced load per word); an element is its terms summed in order
        // in a register (from 1 on the diagonal), stored at its offset.
        // The owner lane of each tile element then reads it from the buffer
        // through its per-lane offset and mask word (1 on the diagonal, 0
        // elsewhere where the element is absent).
        {
            const int len = T == 256 ? net.sc_len : net.sc_len2;
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
                if (j < len)
#pragma unroll
                    for (int u = 0; u < B; u++) en[u] = sp[(j + u) * T];
#pragma unroll
                for (int u = 0; u < B; u++) {
                    // the running sum is stored at every term (the element's
                    // last store stays); padding stores where nothing reads
                    acc = (e[u] & 2) ? ((e[u] & 4) ? 1.0f : 0.0f) : acc;
                    acc += __uint_as_float(__float_as_uint(v[u]) ^ ((unsigned)e[u] << 31));
                    work[(e[u] >> 3) & 8191] = acc;
                }
                if (j >= len) break;
            }
        }
        __syncthreads();
#pragma unroll
        for (int ta = 0; ta < NR; ta++) {
            const int i = WR * ta + wi;
#pragma unroll
            for (int tb = 0; tb < NC; tb++) {
                const int jb = WC * tb + wj;
                if (i >= NT || jb >= NT) continue;
                const unsigned wd = wt[ta][tb];
                unsigned p = wd >> 4;
                f32x4 m;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const bool has = ((wd >> q) & 1u) != 0;
                    const float x = work[p];
                    m[q] = has ? x : (i == jb && 4 * g + q == lr ? 1.0f : 0.0f);
                    p += has ? 1u : 0u;
                }
                M[ta][tb] = m;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // Diagonal tile (k, k) of its owner: invert, publish G_k, c_k = G_k r_k.
    auto diag_step = [&](f32x4 m, int k) __attribute__((always_inline)) {
        tile_invert_acc(m, lane);
#pragma unroll
        for (int q = 0; q < 4; q++) Gbuf[(4 * g + q) * 16 + lr] = m[q];
        float v = rv[16 * k + lr];
#pragma unroll
        for (int u = 0; u < WC; u++)
            if (u < k) v -= fp[16 * u + lr];
#pragma unroll
        for (int q = 0; q < 4; q++) m[q] *= v;
        tile_rowsum_store(m, rv + 16 * k, lane);
    };

    // the last tile column of wave column u (-1: it has none)
    auto last_col = [](int u) __attribute__((always_inline)) { return u < NT ? NT - 1 - (NT - 1 - u) % WC : -1; };

    // Block LU without pivoting with the forward sweep on rv (= f on entry),
    // per 16-column panel k (two barriers): B) the row panel W_kj = G_k A_kj
    // (G_k from LDS; W replaces A_kj and goes to LDS), the column panel A_ik
    // (i > k) to LDS and the sums of A_ik c_k; C) A_ij -= A_ik W_kj on the matrix
    // cores, the owner of the next diagonal tile updating it first, inverting
    // it and forming c_{k+1} = G_{k+1} r_{k+1}.  Leaves c in rv.
    auto factor = [&]() __attribute__((always_inline)) {
        int wv = wave;
        asm volatile("" : "+s"(wv));
        const int wi = wv / WC, wj = wv % WC;
        if (t < NP) rv[t] = f[t];
        __syncthreads();
        if (wave == 0) diag_step(M[0][0], 0);
        __syncthreads();
        for (int k = 0; k < NT - 1; k++) {
            if (wi == k % WR) {
                const f32x4 gr = *reinterpret_cast<const f32x4 *>(Gbuf + lr * 16 + 4 * g);
#pragma unroll
                for (int ta = 0; ta < NR; ta++) {
                    if (WR * ta + wi != k) continue;
#pragma unroll
                    for (int tb = 0; tb < NC; tb++) {
                        const int j = WC * tb + wj;
                        if (j <= k || j >= NT) continue;
                        f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int q = 0; q < 4; q++) z = __builtin_amdgcn_mfma_f32_16x16x4f32(gr[q], M[ta][tb][q], z, 0, 0, 0);
                        M[ta][tb] = z;
                        *reinterpret_cast<f32x4 *>(wB + tb * CS) = z;
                    }
                }
            }
            if (wj == k % WC) {
                const float ck = rv[16 * k + lr];
#pragma unroll
                for (int tb = 0; tb < NC; tb++) {
                    if (WC * tb + wj != k) continue;
#pragma unroll
                    for (int ta = 0; ta < NR; ta++) {
                        const int i = WR * ta + wi;
                        if (i <= k || i >= NT) continue;
                        const f32x4 m = M[ta][tb];
#pragma unroll
                        for (int q = 0; q < 4; q++) {
                            cS[ta * RS + q * 16] = -m[q];
                            // the row's sum of A_ik c_k over this wave's
                            // columns, a lane's columns in the lane, in the
                            // registers of the first of these tiles (each is
                            // in the panel buffer from here on)
                            M[ta][0][q] = tb == 0 ? m[q] * ck : fmaf(m[q], ck, M[ta][0][q]);
                        }
                    }
                }
            }
            // row k + 1 has all its columns
            if (wi == (k + 1) % WR && wj <= k) {
#pragma unroll
                for (int ta = 0; ta < NR; ta++)
                    if (WR * ta + wi == k + 1) tile_rowsum_store(M[ta][0], fp + 16 * wj, lane);
            }
            __syncthreads();
            const int k1 = k + 1;
            if (wi == k1 % WR && wj == k1 % WC) {
                // in a copy, so that the inversion's code exists once; the
                // tile itself is not read again
                f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int ta = 0; ta < NR; ta++)
#pragma unroll
                    for (int tb = 0; tb < NC; tb++) {
                        if (WR * ta >= WC * (tb + 1) || WC * tb >= WR * (ta + 1)) continue;  // no diagonal tile
                        if (WR * ta + wi != k1 || WC * tb + wj != k1) continue;
                        const f32x4 xa = *reinterpret_cast<const f32x4 *>(cA + ta * RS);
                        const f32x4 wv = *reinterpret_cast<const f32x4 *>(wB + tb * CS);
                        d = M[ta][tb];
#pragma unroll
                        for (int q = 0; q < 4; q++) d = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[q], wv[q], d, 0, 0, 0);
                    }
                diag_step(d, k1);
            }
            // GW row-panel tiles W_kj held at a time, each A_ik read once
            // per group (fewer LDS reads than one W read per tile update)
#pragma unroll
            for (int tb0 = 0; tb0 < NC; tb0 += kDenseRegGW<NT>) {
                constexpr int GW = kDenseRegGW<NT>;
                f32x4 wv[GW];
                bool vv[GW], any = false;
#pragma unroll
                for (int u = 0; u < GW; u++) {
                    const int j = WC * (tb0 + u) + wj;
                    vv[u] = tb0 + u < NC && j > k && j < NT;
                    any = any || vv[u];
                    wv[u] = vv[u] ? *reinterpret_cast<const f32x4 *>(wB + (tb0 + u) * CS) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                }
                if (!any) continue;
#pragma unroll
                for (int ta = 0; ta < NR; ta++) {
                    const int i = WR * ta + wi;
                    if (i <= k || i >= NT) continue;
                    const f32x4 xa = *reinterpret_cast<const f32x4 *>(cA + ta * RS);
#pragma unroll
                    for (int u = 0; u < GW; u++) {
                        const int tb = tb0 + u < NC ? tb0 + u : NC - 1;
                        const int j = WC * (tb0 + u) + wj;
                        if (!vv[u] || (i == k1 && j == k1)) continue;
#pragma unroll
                        for (int q = 0; q < 4; q++)
                            M[ta][tb] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[q], wv[u][q], M[ta][tb], 0, 0, 0);
                    }
                }
            }
            __syncthreads();
        }
    };

    // Backward sweep by columns: x_k = c_k - sum_j W_kj x_j, the sums kept as
    // in the forward sweep, in the registers of the last of a row's tiles.
    // Leaves x_k in xv for k > 0 and the partial sums of row 0 in bp.
    auto back = [&]() __attribute__((always_inline)) {
        int wv = wave;
        asm volatile("" : "+s"(wv));
        const int wi = wv / WC, wj = wv % WC;
        for (int k = NT - 1; k >= 1; k--) {
            if (wj == k % WC) {
                float xk = rv[16 * k + lr];
#pragma unroll
                for (int u = 0; u < WC; u++)
                    if (last_col(u) > k) xk -= bp[16 * (WC * (k & 1) + u) + lr];
                if (wi == 0 && g == 0) xv[16 * k + lr] = xk;
#pragma unroll
                for (int tb = 0; tb < NC; tb++) {
                    if (WC * tb + wj != k) continue;
#pragma unroll
                    for (int ta = 0; ta < NR; ta++) {
                        if (WR * ta + wi >= k) continue;
                        const bool first = k + WC >= NT;
#pragma unroll
                        for (int q = 0; q < 4; q++)
                            M[ta][NC - 1][q] = first ? M[ta][tb][q] * xk : fmaf(M[ta][tb][q], xk, M[ta][NC - 1][q]);
                    }
                }
            }
            // row k - 1 has all its columns
            if (wi == (k - 1) % WR && last_col(wj) >= k) {
#pragma unroll
                for (int ta = 0; ta < NR; ta++)
                    if (WR * ta + wi == k - 1)
                        tile_rowsum_store(M[ta][NC - 1], bp + 16 * (WC * ((k - 1) & 1) + wj), lane);
            }
            __syncthreads();
        }
    };
    auto solution = [&](int i) __attribute__((always_inline)) {
        if (i >= 16) return xv[i];
        float x = rv[i];
#pragma unroll
        for (int u = 0; u < WC; u++)
            if (last_col(u) > 0) x -= bp[16 * u + i];
        return x;
    };

    unsigned *const words = reinterpret_cast<unsigned *>(a.counters);
    float *const hand = TRACE || NT < 4 ? nullptr : a.spill;  // (eight waves from four tiles on)
    for (;;) {
        if (t == 0) {
            if (WR > 2 && hand) {
                const unsigned q = atomicAdd(words + DENSE_TAIL_HEAD, 1u);
                s_rec = (int)q;
                s_sid = q < words[DENSE_HANDED] ? __float_as_int(hand[(size_t)q * kDenseHandWords]) : a.nsys;
            } else {
                const unsigned q = atomicAdd(head, 1u);
                s_sid = q < (unsigned)a.nsys ? (a.index ? a.index[q] : (int)q) : a.nsys;
            }
        }
        __syncthreads();
        const int sid = __builtin_amdgcn_readfirstlane(s_sid);
        if (sid >= a.nsys) break;
        for (int i = t; i < N; i += T) y[i] = a.equations[(size_t)sid * N + i];
        const float scale = a.constants[(size_t)sid * a.const_stride];
        __syncthreads();
        float tnow = a.tnow, h = a.h0;
        int unsolved = 0, attempts = 0, status = WIND_STATUS_OK;
        bool handed = false;
        if (WR > 2 && hand) {
            const float *r = hand + (size_t)__builtin_amdgcn_readfirstlane(s_rec) * kDenseHandWords;
            tnow = uniform(r[1]);
            h = uniform(r[2]);
            unsolved = __builtin_amdgcn_readfirstlane(__float_as_int(r[3]));
            attempts = __builtin_amdgcn_readfirstlane(__float_as_int(r[4]));
        }
        const bool replay = TRACE && a.trace.h != nullptr;
        const int rcount = replay ? min(a.trace.count[sid], a.trace.capacity) : 0;
        while (replay ? attempts < rcount : tnow < a.tend) {
            const size_t slot = TRACE ? (size_t)sid * a.trace.capacity + attempts : 0;
            if (replay && a.trace.y_start) {
                for (int i = t; i < N; i += T) y[i] = a.trace.y_start[slot * N + i];
                __syncthreads();
            }
            const float hh = replay ? a.trace.h[slot] : fminf(a.tend - tnow, h);
            const float tb = tnow + hh;
            const float hs_full = tb - tnow, hs_half = (tb - tnow) / 2.0f;
            for (int pass = 0; pass < 3; pass++) {
                const float hs = pass == 0 ? hs_full : hs_half;
                if (pass != 2) {
                    for (int i = t; i < N; i += T) yw[i] = y[i];
                    __syncthreads();
                }
                assemble(yw, scale, hs);
                factor();
                back();
                for (int i = t; i < N; i += T) yw[i] = fmaf(hs, solution(i), yw[i]);
                __syncthreads();
                if (pass == 0)
                    for (int i = t; i < N; i += T) y1[i] = yw[i];
            }
            // every eighth attempt: how many systems are finished (the read's
            // latency would show if it were every one)
            const bool look = WR == 2 && hand && (attempts & 7) == 7;
            if (t == 0) {
                s_flag = 0;
                if (look) s_done = (int)__hip_atomic_load(words + DENSE_DONE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __syncthreads();
            bool flag = false;
            double err = 0.0;
            if (a.controller == WIND_CTRL_REFERENCE) {
                bool fail = false;
                for (int i = t; i < N; i += T) fail = fail || species_fails<WIND_SIE>(y1[i], yw[i], a.ABS, a.REL);
                if (fail) s_flag = 1;
            } else {
                for (int i = t; i < N; i += T) err = err_max(err, err_term(y1[i], yw[i], a.ABS, a.REL));
#pragma unroll
                for (int off = 32; off > 0; off >>= 1) err = err_max(err, __shfl_xor(err, off));
                if (lane == 0) s_err[wave] = err;
            }
            __syncthreads();
            flag = s_flag != 0;
            if (a.controller != WIND_CTRL_REFERENCE) {
                err = s_err[0];
                for (int wv = 1; wv < WR * WC; wv++) err = err_max(err, s_err[wv]);
            }
            const bool extrap = a.controller != WIND_CTRL_REFERENCE;
            if constexpr (TRACE) {
                if (attempts < a.trace.capacity) {
                    for (int i = t; i < N; i += T) {
                        if (a.trace.y1) a.trace.y1[slot * N + i] = y1[i];
                        if (a.trace.y2) a.trace.y2[slot * N + i] = yw[i];
                    }
                    if (t == 0 && a.trace.flag)
                        a.trace.flag[slot] = a.controller == WIND_CTRL_REFERENCE ? (int)flag : !(err <= 1.0);
                }
                if (replay) {
                    attempts++;
                    if (a.trace.accept[slot]) {
                        tnow = tnow + hh;
                        for (int i = t; i < N; i += T) y[i] = extrap ? 2.0f * yw[i] - y1[i] : yw[i];
                    }
                    __syncthreads();
                    continue;
                }
            }
            attempts++;
            const bool acc = control_step<WIND_SIE, true>(a.controller, a.tend, hh, flag, err, tnow, h, unsolved, status);
            // (the same in every lane: kept in scalar registers)
            tnow = uniform(tnow);
            h = uniform(h);
            unsolved = __builtin_amdgcn_readfirstlane(unsolved);
            status = __builtin_amdgcn_readfirstlane(status);
            if (acc)
                for (int i = t; i < N; i += T) y[i] = extrap ? 2.0f * yw[i] - y1[i] : yw[i];
            __syncthreads();
            if (status != WIND_STATUS_OK) break;
            if (attempts >= a.max_attempts && tnow < a.tend) {
                status = WIND_STATUS_EXHAUSTED;
                break;
            }
            if (look && tnow < a.tend &&
                a.nsys - __builtin_amdgcn_readfirstlane(s_done) <= a.spill_cap) {
                handed = true;
                break;
            }
        }
        __syncthreads();
        for (int i = t; i < N; i += T) a.equations[(size_t)sid * N + i] = y[i];
        if (WR == 2 && hand && t == 0) {
            if (handed) {
                // at most spill_cap systems are unfinished, so the list holds them
                float *r = hand + (size_t)atomicAdd(words + DENSE_HANDED, 1u) * kDenseHandWords;
                r[0] = __int_as_float(sid);
                r[1] = tnow;
                r[2] = h;
                r[3] = __int_as_float(unsolved);
                r[4] = __int_as_float(attempts);
            } else {
                atomicAdd(words + DENSE_DONE, 1u);
            }
        }
        if (t == 0 && !handed) {
            if (a.steps_out) a.steps_out[sid] = 3 * attempts;
            if (a.status_out) a.status_out[sid] = status;
            steps += 3ull * (unsigned long long)attempts;
        }
        __syncthreads();
    }
    if (t == 0 && steps) atomicAdd(a.counters + 1, steps);
}

// LDS bytes of ma_dense_reg_integrate (dynamic part) for a network.
inline size_t dense_reg_lds_bytes(int NT, int R, int WGS, int cap) {
    return sizeof(float) * (size_t)dense_reg_offsets(NT, R, WGS, cap).total;
}

// The workgroups per CU to build for where their LDS fits.
constexpr int dense_reg_wgs_want(int NT) { return NT >= 7 ? 4 : NT >= 5 ? 5 : NT >= 3 ? 6 : 8; }

// The workgroups per CU to build for: dense_reg_wgs_want when they fit the
// CU's LDS (max_lds bytes), else three when three fit, else 0 (the solver
// does not apply).  cap: the network's compact element buffer (floats).
inline int dense_reg_wgs_for(int NT, int R, int cap, size_t max_lds) {
    const int want = dense_reg_wgs_want(NT);
    if (want * (dense_reg_lds_bytes(NT, R, want, cap) + 256) <= max_lds) return want;
    return 3 * (dense_reg_lds_bytes(NT, R, 3, cap) + 256) <= max_lds ? 3 : 0;
}

}  // namespace wind
