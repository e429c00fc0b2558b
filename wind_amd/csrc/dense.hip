// Launchers of the dense LDS/MFMA solver (kernels_dense.h).  A translation
// unit of its own, compiled with fused multiply-add contraction: the dense
// solver exists only in fast mode, which promises no operation order.
#include <hip/hip_runtime.h>

#include "kernels_dense.h"
#include "kernels_dense_reg.h"
#include "wind_internal.h"

using namespace wind;

template <int METHOD, int PREC>
int launch_dense(int num_cu, const MassActionDevice &d, const IntegrateArgs &a, int ir, size_t lds, int T,
                 const SolverChoice &sc, hipStream_t st) {
    auto kfn = a.trace.capacity > 0 ? ma_dense_integrate<METHOD, PREC, true> : ma_dense_integrate<METHOD, PREC>;
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute((const void *)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return wind_fail(WIND_ERR_DEVICE, hipGetErrorString(e));
    }
    int per_cu = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kfn, T, lds);
    if (e != hipSuccess) return wind_fail(WIND_ERR_DEVICE, hipGetErrorString(e));
    const int grid = scaled_grid(num_cu, per_cu, sc, a.nsys);
    hipLaunchKernelGGL(kfn, dim3(grid), dim3(T), lds, st, a, d, ir);
    e = hipGetLastError();
    if (e != hipSuccess) return wind_fail(WIND_ERR_DEVICE, hipGetErrorString(e));
    return WIND_OK;
}

#define WIND_DENSE(M, P)                                                                                     \
    template int launch_dense<M, P>(int, const MassActionDevice &, const IntegrateArgs &, int, size_t, int,    \
                                    const SolverChoice &, hipStream_t);
WIND_DENSE(WIND_SIE, PREC_VALU)
WIND_DENSE(WIND_SIE, PREC_MFMA_F32)
WIND_DENSE(WIND_SIE, PREC_MFMA_BF16)
WIND_DENSE(WIND_SIE, PREC_MFMA_BF16X3)
WIND_DENSE(WIND_RK2, PREC_VALU)
WIND_DENSE(WIND_RK2, PREC_MFMA_F32)
WIND_DENSE(WIND_RK2, PREC_MFMA_BF16)
WIND_DENSE(WIND_RK2, PREC_MFMA_BF16X3)

// ---------------------------------------------------------------------------
// Register-resident solver (kernels_dense_reg.h).

// Workgroups per CU the register solver runs with on the current device for
// network d (dense_reg_wgs_for), or 0 where it does not fit.
static int dense_reg_wgs_dev(const MassActionDevice &d) {
    int dev = 0, max_lds = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) != hipSuccess)
        return 0;
    return dense_reg_wgs_for((d.N + 15) / 16, d.R, d.sc_cap, (size_t)max_lds);
}

bool dense_reg_eligible(const MassActionDevice &d, const SolverChoice &sc) {
    if (sc.dense_kernel == 1 || !d.sc_ent) return false;
    if (sc.pivot || sc.ir_sweeps != 0) return false;
    if (sc.solver != WIND_SOLVER_AUTO && sc.solver != WIND_SOLVER_MFMA_F32) return false;
    const int NT = (d.N + 15) / 16;
    if (!dense_reg_tiles(NT)) return false;
    // three workgroups per CU must fit, else the LDS-resident solver is the better shape
    return dense_reg_wgs_dev(d) != 0;
}

template <int NT, int WGS, int WR = 2, int WC = 2>
int launch_dense_reg_nt(int num_cu, const MassActionDevice &d, const IntegrateArgs &a, const SolverChoice &sc,
                        hipStream_t st) {
    auto kfn = a.trace.capacity > 0 ? ma_dense_reg_integrate<NT, WGS, WR, WC, true>
                                      : ma_dense_reg_integrate<NT, WGS, WR, WC>;
    const size_t lds = dense_reg_lds_bytes(NT, d.R, WGS, d.sc_cap);
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute((const void *)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return wind_fail(WIND_ERR_DEVICE, hipGetErrorString(e));
    }
    int per_cu = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kfn, 64 * WR * WC, lds);
    if (e != hipSuccess) return wind_fail(WIND_ERR_DEVICE, hipGetErrorString(e));
    const int grid = scaled_grid(num_cu, per_cu, sc, WR > 2 && a.spill ? a.spill_cap : a.nsys);
    hipLaunchKernelGGL(kfn, dim3(grid), dim3(64 * WR * WC), lds, st, a, d);
    e = hipGetLastError();
    if (e != hipSuccess) return wind_fail(WIND_ERR_DEVICE, hipGetErrorString(e));
    return WIND_OK;
}

// The four-wave build for as many workgroups per CU as fit (dense_reg_wgs_for).
template <int NT>
int launch_dense_reg_wgs(int num_cu, const MassActionDevice &d, const IntegrateArgs &a, const SolverChoice &sc,
                         hipStream_t st) {
    constexpr int want = dense_reg_wgs_want(NT);
    return dense_reg_wgs_dev(d) == want ? launch_dense_reg_nt<NT, want>(num_cu, d, a, sc, st)
                                        : launch_dense_reg_nt<NT, 3>(num_cu, d, a, sc, st);
}

// Few systems: eight waves each, two workgroups per CU, no register
// spilled.  Four waves against eight, us per sub-step of a system alone on its
// CU: N = 160 42.0 / 31.7, 128 24.6 / 21.0, 96 15.6 / 14.8, 64 9.5 / 9.1; two per CU:
// 49.5 / 39.7, 29.1 / 26.3, 18.0 / 18.5 (512 systems to the end 144 ms in either
// form), 10.8 / 11.6; three: 56.7 / 67.3, 33.4 / 44.0, 20.4 / 34.0, 12.2 / 20.0.
//
// The largest number of systems that the eight-wave form takes; 0: it is not built.
static int dense_reg_few(int NT, int num_cu) { return NT >= 6 ? 2 * num_cu : NT >= kDenseRegMinNT8 ? num_cu : 0; }

static int launch_dense_reg_few(int num_cu, const MassActionDevice &d, const IntegrateArgs &a, const SolverChoice &sc,
                         hipStream_t st) {
    switch ((d.N + 15) / 16) {
    case 4: return launch_dense_reg_nt<4, 2, 4, 2>(num_cu, d, a, sc, st);
    case 5: return launch_dense_reg_nt<5, 2, 4, 2>(num_cu, d, a, sc, st);
    case 6: return launch_dense_reg_nt<6, 2, 4, 2>(num_cu, d, a, sc, st);
    case 7: return launch_dense_reg_nt<7, 2, 4, 2>(num_cu, d, a, sc, st);
    case 8: return launch_dense_reg_nt<8, 2, 4, 2>(num_cu, d, a, sc, st);
    case 9: return launch_dense_reg_nt<9, 2, 4, 2>(num_cu, d, a, sc, st);
    case 10: return launch_dense_reg_nt<10, 2, 4, 2>(num_cu, d, a, sc, st);
    default: return wind_fail(WIND_ERR_UNSUPPORTED, "register-resident dense solver: N out of range");
    }
}

static int launch_dense_reg_many(int num_cu, const MassActionDevice &d, const IntegrateArgs &a, const SolverChoice &sc,
                          hipStream_t st) {
    switch ((d.N + 15) / 16) {
    case 1: return launch_dense_reg_wgs<1>(num_cu, d, a, sc, st);
    case 2: return launch_dense_reg_wgs<2>(num_cu, d, a, sc, st);
    case 3: return launch_dense_reg_wgs<3>(num_cu, d, a, sc, st);
    case 4: return launch_dense_reg_wgs<4>(num_cu, d, a, sc, st);
    case 5: return launch_dense_reg_wgs<5>(num_cu, d, a, sc, st);
    case 6: return launch_dense_reg_wgs<6>(num_cu, d, a, sc, st);
    case 7: return launch_dense_reg_wgs<7>(num_cu, d, a, sc, st);
    case 8: return launch_dense_reg_wgs<8>(num_cu, d, a, sc, st);
    case 9: return launch_dense_reg_wgs<9>(num_cu, d, a, sc, st);
    case 10: return launch_dense_reg_wgs<10>(num_cu, d, a, sc, st);
    default: return wind_fail(WIND_ERR_UNSUPPORTED, "register-resident dense solver: N out of range");
    }
}

int dense_reg_hand_cap(const wind_network *net, const wind_options &o, const SolverChoice &sc, int nsys, int num_cu) {
    if (net->builtin != WIND_NET_MASS_ACTION || o.mode != WIND_MODE_FAST || o.method != WIND_SIE || o.trace) return 0;
    const int few = dense_reg_few((net->N + 15) / 16, num_cu);
    return nsys > few && dense_reg_eligible(net->ma, sc) ? few : 0;
}

// More systems than that: four waves each until no more than that are
// unfinished; where the caller has a list for them (a.spill), those go on
// on eight waves each, spread over the CUs again (a system's last attempts
// otherwise run at the pace that its CU's other long systems leave it).
// Whole batches, ms, handed over never / at 128 / 256 / 384 / 512 / 768 unfinished:
// N = 157, 1,021 systems, 354 / 334 / 327 / 322 / 308 / 310; 112, 2,000, 221 /
// 215 / 211 / 211 / 206 / 211; 64, 4,099, 113 / 109 / 106 / 107 / 105 / 109; 80,
// 1,500, 105 / 103 / 105 / 101 / 101 / 102.
int launch_dense_reg(int num_cu, const MassActionDevice &d, const IntegrateArgs &a, const SolverChoice &sc,
                     hipStream_t st) {
    if (a.nsys <= dense_reg_few((d.N + 15) / 16, num_cu)) return launch_dense_reg_few(num_cu, d, a, sc, st);
    const int rc = launch_dense_reg_many(num_cu, d, a, sc, st);
    return rc || !a.spill ? rc : launch_dense_reg_few(num_cu, d, a, sc, st);
}
