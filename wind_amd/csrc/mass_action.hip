// Host side of the mass-action networks: gather-list construction, device
// upload, and kernel launch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <functional>
#include <string>
#include <vector>

#include "kernels_dense.h"
#include "kernels_dense_reg.h"
#include "kernels_ma_wave.h"
#include "kernels_mass_action.h"
#include "wind_internal.h"

using namespace wind;

namespace {

// The tables of a network, in one device allocation (each on a 256-byte
// boundary) and one copy: the first table's address is the allocation's.
struct Table {
    void **dst;
    const void *src;
    size_t bytes;
};
int upload(const std::vector<Table> &tables) {
    auto part = [](size_t b) { return (b + 255) & ~(size_t)255; };
    size_t total = 256;
    for (const Table &t : tables) total += part(t.bytes);
    std::vector<char> host(total);
    size_t at = 0;
    for (const Table &t : tables) {
        if (t.bytes) std::memcpy(host.data() + at, t.src, t.bytes);
        at += part(t.bytes);
    }
    char *dev = nullptr;
    hipError_t e = hipMalloc((void **)&dev, total);
    if (e != hipSuccess) return wind_fail(WIND_ERR_DEVICE, hipGetErrorString(e));
    e = hipMemcpy(dev, host.data(), total, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipFree(dev);
        return wind_fail(WIND_ERR_DEVICE, hipGetErrorString(e));
    }
    at = 0;
    for (const Table &t : tables) {
        *t.dst = dev + at;
        at += part(t.bytes);
    }
    return WIND_OK;
}

struct Scratch {
    float *ptr = nullptr;
    size_t bytes = 0;
};
Scratch g_scratch;  // per-process matrix scratch; callers hold the context lock

}  // namespace

// The exact register kernel (ma_wave_integrate): N <= 64, its LDS within the
// default limit.
static bool ma_wave_fits(int N, int R) {
    return N <= 64 && sizeof(float) * ma_wave_lds_floats((N + 7) & ~7, R) <= 65536 - 64;
}

// Lists of words, list z the words ptr[z] .. ptr[z + 1] - 1.
struct WordLists {
    std::vector<int32_t> key, ptr = {0};
    std::vector<uint32_t> word;
    size_t size() const { return ptr.size() - 1; }
    void close() { ptr.push_back((int32_t)word.size()); }
};

// The words of each key (< nkeys) in their order in `word`, the non-empty keys ascending.
static WordLists lists_by_key(int nkeys, const std::vector<int32_t> &key, const std::vector<uint32_t> &word) {
    std::vector<int32_t> at(nkeys + 1, 0);
    for (int32_t k : key) at[k + 1]++;
    WordLists l;
    for (int k = 0; k < nkeys; k++) {
        if (at[k + 1]) {
            l.key.push_back(k);
            l.ptr.push_back(at[k] + at[k + 1]);
        }
        at[k + 1] += at[k];
    }
    l.word.resize(word.size());
    for (size_t i = 0; i < word.size(); i++) l.word[at[key[i]]++] = word[i];
    return l;
}

// Deals elements (their terms' words) to `threads` streams, most terms first
// to the least-loaded thread (the first of equals); streams padded with `pad`
// to the longest, rounded up to `batch`, and interleaved: word j of thread t at
// [j * threads + t].
static std::vector<int32_t> deal_streams(const WordLists &items, int threads, int batch, uint32_t pad, int *len) {
    auto terms = [&](int z) { return items.ptr[z + 1] - items.ptr[z]; };
    int most = 0;
    for (size_t z = 0; z < items.size(); z++) most = std::max(most, terms((int)z));
    // by falling number of terms, equals in order (a counting sort)
    std::vector<int32_t> start(most + 2, 0), order(items.size());
    for (size_t z = 0; z < items.size(); z++) start[most - terms((int)z) + 1]++;
    for (int c = 0; c <= most; c++) start[c + 1] += start[c];
    for (size_t z = 0; z < items.size(); z++) order[start[most - terms((int)z)]++] = (int32_t)z;
    // the threads with their loads, the least-loaded on top
    using Load = std::pair<int32_t, int32_t>;
    std::vector<Load> heap(threads);
    for (int th = 0; th < threads; th++) heap[th] = {0, th};
    std::vector<Load> place(items.size());  // first word's place in the stream, thread
    int longest = 1;
    for (int32_t z : order) {
        std::pop_heap(heap.begin(), heap.end(), std::greater<Load>());
        Load &top = heap.back();
        place[z] = top;
        top.first += terms(z);
        longest = std::max(longest, top.first);
        std::push_heap(heap.begin(), heap.end(), std::greater<Load>());
    }
    *len = (longest + batch - 1) / batch * batch;
    std::vector<int32_t> out((size_t)*len * threads, (int32_t)pad);
    for (size_t z = 0; z < items.size(); z++)
        for (int j = 0; j < terms((int)z); j++)
            out[(size_t)(place[z].first + j) * threads + place[z].second] = (int32_t)items.word[items.ptr[z] + j];
    return out;
}

int mass_action_build(wind_network *n, int N, int R, const int32_t *rx, const float *k) {
    n->rx.assign(rx, rx + 4 * (size_t)R);
    n->k.assign(k, k + R);
    // Contribution lists in the order of a serial sweep over reactions.
    std::vector<std::vector<int32_t>> flist(N);
    WordLists jlist;
    {
        std::vector<int32_t> key;
        std::vector<uint32_t> ent;
        key.reserve(8 * (size_t)R);
        ent.reserve(8 * (size_t)R);
        for (int r = 0; r < R; r++) {
            const int32_t *x = rx + 4 * r;
            for (int slot = 0; slot < 4; slot++) {
                const int neg = slot < 2 ? 1 : 0;
                flist[x[slot]].push_back(r * 2 + neg);
                for (int which = 0; which < 2; which++) {
                    key.push_back(x[which] * N + x[slot]);
                    ent.push_back((uint32_t)(((r * 2 + which) * 2) + neg));
                }
            }
        }
        jlist = lists_by_key(N * N, key, ent);
    }
    std::vector<int32_t> f_ptr(N + 1, 0), f_ent;
    for (int i = 0; i < N; i++) {
        f_ent.insert(f_ent.end(), flist[i].begin(), flist[i].end());
        f_ptr[i + 1] = (int32_t)f_ent.size();
    }
    const std::vector<int32_t> &j_pos = jlist.key, &j_ptr = jlist.ptr;
    const std::vector<int32_t> j_ent(jlist.word.begin(), jlist.word.end());
    std::vector<std::vector<int32_t>> rows(N);
    for (size_t z = 0; z < j_pos.size(); z++) rows[j_pos[z] % N].push_back((int32_t)z);
    std::vector<int32_t> r_ptr(N + 1, 0), r_z;
    for (int i = 0; i < N; i++) {
        r_z.insert(r_z.end(), rows[i].begin(), rows[i].end());
        r_ptr[i + 1] = (int32_t)r_z.size();
    }
    // Assembly of the register-resident dense solver.  The matrix elements
    // (row, col) with Jacobian terms live, once summed, in a compact LDS
    // buffer (the others are 1 on the diagonal, 0 elsewhere), ordered by
    // 16x16 tile (row-major over tiles), then by lane
    // l = 16 ((row % 16) / 4) + col % 16 of the MFMA accumulator layout, then
    // by that lane's accumulator register q = row % 4.  Per tile and lane,
    // sc_tile[tile * 64 + l] = (offset of the lane's first element) << 4 |
    // (mask of the q present), so that the owner lane finds element q at
    // that offset plus the present q below it.  An element is its terms in
    // the order dense_eval applies them (the row's reactions in sweep order,
    // the reaction's first reactant before its second), summed from 1 on the
    // diagonal; the elements are dealt to the workgroup's 256 or
    // 512 threads (deal_streams), and a thread's stream is its elements' terms,
    // one word each:
    //   (LDS float index of the term's h dJ value) << 16 | (buffer offset of
    //   the element) << 3 | (element on the diagonal) << 2 | (element's first
    //   term) << 1 | (the term is subtracted: a product row)
    // f's elements (from 0, their terms w) follow the matrix's in the buffer,
    // at sc_cap + row; padding words go to a place that nothing reads.
    const int NT = (N + 15) / 16;
    std::vector<int32_t> sc_ent, sc_ent2;
    std::vector<uint32_t> sc_tile;
    int sc_len = 0, sc_len2 = 0, sc_cap = 0;
    if (dense_reg_tiles(NT)) {
        const DenseRegOffsets lo = dense_reg_offsets(NT, R, 3, 0);
        bool ok = lo.hdb + R < 65536;
        WordLists elem;  // by row * N + col
        if (ok) {
            std::vector<int32_t> key;
            std::vector<uint32_t> word;
            key.reserve(8 * (size_t)R);
            word.reserve(8 * (size_t)R);
            for (int i = 0; i < N; i++)
                for (int32_t e : flist[i]) {
                    const int r = e >> 1, neg = e & 1;
                    const int32_t *x = rx + 4 * r;
                    for (int which = 0; which < 2; which++) {
                        const uint32_t hd = (uint32_t)((which ? lo.hdb : lo.hda) + r);
                        key.push_back(i * N + x[which]);
                        word.push_back((hd << 16) | ((x[which] == i ? 1u : 0u) << 2) | (uint32_t)!neg);
                    }
                }
            elem = lists_by_key(N * N, key, word);
        }
        // the q present per (tile, lane), then the offsets
        std::vector<uint32_t> mask4((size_t)NT * NT * 64, 0);
        auto slot = [&](int row, int col, int *tl, int *q) {
            *tl = ((row >> 4) * NT + (col >> 4)) * 64 + 16 * ((row & 15) >> 2) + (col & 15);
            *q = row & 3;
        };
        for (int32_t key : elem.key) {
            int tl, q;
            slot(key / N, key % N, &tl, &q);
            mask4[tl] |= 1u << q;
        }
        sc_tile.resize(mask4.size());
        uint32_t nnz = 0;
        for (size_t u = 0; u < mask4.size(); u++) {
            sc_tile[u] = nnz << 4 | mask4[u];
            nnz += (uint32_t)__builtin_popcount(mask4[u]);
        }
        // (+1: an owner lane reads one place past its elements, unused)
        sc_cap = (int)((nnz + 1 + 3) & ~3u);
        ok = ok && sc_cap + 16 * NT <= 8192;
        if (ok) {
            for (size_t z = 0; z < elem.size(); z++) {
                int tl, q;
                slot(elem.key[z] / N, elem.key[z] % N, &tl, &q);
                const uint32_t dest = (sc_tile[tl] >> 4) + (uint32_t)__builtin_popcount(mask4[tl] & ((1u << q) - 1));
                for (int32_t j = elem.ptr[z]; j < elem.ptr[z + 1]; j++) elem.word[j] |= dest << 3;
                elem.word[elem.ptr[z]] |= 2u;
            }
            for (int i = 0; i < N; i++) {
                if (flist[i].empty()) continue;
                const size_t first = elem.word.size();
                for (int32_t e : flist[i])
                    elem.word.push_back((uint32_t)(lo.w + (e >> 1)) << 16 | (uint32_t)(sc_cap + i) << 3 |
                                        (uint32_t)(e & 1));
                elem.word[first] |= 2u;
                elem.close();
            }
            sc_ent = deal_streams(elem, 256, kDenseRegBatch, nnz << 3, &sc_len);
            if (NT >= kDenseRegMinNT8) sc_ent2 = deal_streams(elem, 512, kDenseRegBatch, nnz << 3, &sc_len2);
        } else {
            sc_tile.clear();
            sc_cap = 0;
        }
    }
    // Assembly of the exact register kernel (ma_wave_integrate): f's and the
    // Jacobian's elements, each its terms in sweep order, one word per term:
    //   (LDS float index of the term's w, da or db) << 16 | (LDS float index
    //   of the element) << 3 | (element's last term) << 1 | (subtracted)
    std::vector<int32_t> ex_ent;
    int ex_len = 0;
    if (ma_wave_fits(N, R)) {
        const int NP = (N + 7) & ~7;
        const uint32_t f0 = NP * NP + 3 * NP, w0 = f0 + NP;
        WordLists items;
        for (int i = 0; i < N; i++) {
            if (flist[i].empty()) continue;
            for (int32_t e : flist[i])
                items.word.push_back((w0 + (uint32_t)(e >> 1)) << 16 | (f0 + i) << 3 | (uint32_t)(e & 1));
            items.word.back() |= 2u;
            items.close();
        }
        for (size_t z = 0; z < jlist.size(); z++) {
            const uint32_t dest = (uint32_t)(j_pos[z] / N * NP + j_pos[z] % N);
            for (int32_t j = j_ptr[z]; j < j_ptr[z + 1]; j++) {
                const int32_t e = j_ent[j];
                items.word.push_back((w0 + (uint32_t)(R * ((e & 2) ? 2 : 1) + (e >> 2))) << 16 | dest << 3 |
                                     (uint32_t)(e & 1));
            }
            items.word.back() |= 2u;
            items.close();
        }
        ex_ent = deal_streams(items, 128, kMaWaveBatch, 0, &ex_len);
    }
    MassActionDevice &d = n->ma;
    d.N = N;
    d.R = R;
    d.nnz = (int)j_pos.size();
    d.sc_len = sc_len;
    d.sc_cap = sc_cap;
    d.sc_len2 = sc_len2;
    d.ex_len = ex_len;
    std::vector<Table> tables = {{(void **)&d.rx, rx, sizeof(int32_t) * 4 * R}, {(void **)&d.k, k, sizeof(float) * R}};
    auto add = [&](auto &dst, const auto &v) { tables.push_back({(void **)&dst, v.data(), sizeof(v[0]) * v.size()}); };
    add(d.f_ptr, f_ptr);
    add(d.f_ent, f_ent);
    add(d.j_pos, j_pos);
    add(d.j_ptr, j_ptr);
    add(d.j_ent, j_ent);
    add(d.r_ptr, r_ptr);
    add(d.r_z, r_z);
    if (!sc_ent.empty()) {
        add(d.sc_ent, sc_ent);
        add(d.sc_tile, sc_tile);
    }
    if (!sc_ent2.empty()) add(d.sc_ent2, sc_ent2);
    if (!ex_ent.empty()) add(d.ex_ent, ex_ent);
    return upload(tables);
}

void mass_action_release(wind_network *n) {
    MassActionDevice &d = n->ma;
    if (d.rx) (void)hipFree(d.rx);  // the allocation of all tables (upload)
    d = MassActionDevice();
}

// Which kernel launch_mass_action picks, and whether it needs the
// process-wide matrix scratch (only callers holding the context lock may
// use that).
struct MassActionPlan {
    bool dense = false;      // ma_dense_integrate
    bool in_lds = true;      // ma_block_integrate: matrices in LDS
    size_t lds = 0;
};

// PIVOT (fast mode, WIND_FLAG_PIVOT) takes the LDS LU with partial pivoting
// instead of the dense solver, whose diagonal blocks are unpivoted.
static MassActionPlan mass_action_plan(const MassActionDevice &d, int mode, bool pivot = false) {
    MassActionPlan p;
    int dev = 0, max_lds = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
    const int N = d.N;
    const bool fast = mode == WIND_MODE_FAST;
    if (fast && !pivot && (N + 15) / 16 * 16 <= 192) {
        const size_t lds = dense_lds_bytes(N, d.R);
        if (lds + 128 <= (size_t)max_lds) {
            p.dense = true;
            p.lds = lds;
            return p;
        }
    }
    const size_t base = sizeof(float) * (5 * (size_t)N + 3 * (size_t)d.R);
    const size_t mats = sizeof(float) * (fast ? 1 : 2) * (size_t)N * N;
    p.in_lds = base + mats + 64 <= (size_t)max_lds;
    p.lds = base + (p.in_lds ? mats : 0);
    return p;
}

bool mass_action_needs_scratch(const wind_network *net, int mode) {
    const MassActionPlan p = mass_action_plan(net->ma, mode);
    return !p.dense && !p.in_lds;
}

namespace {

// Launch shape of the one-workgroup-per-system kernel (ma_block_integrate).
struct BlockShape {
    int T = 0, grid = 0;
    size_t lds = 0;
    bool in_lds = true;
};

template <int METHOD>
auto block_kernel(bool fast, bool pivot) {
    return fast ? (pivot ? ma_block_integrate<METHOD, true, true> : ma_block_integrate<METHOD, true>)
                : ma_block_integrate<METHOD, false>;
}

template <int METHOD>
int block_shape(int num_cu, const MassActionDevice &d, const MassActionPlan &plan, bool fast, const SolverChoice &sc,
                int nsys, BlockShape *s) {
    s->T = block_threads(d.N, nsys, num_cu);
    s->in_lds = plan.in_lds;
    s->lds = plan.lds;
    int max_lds = 0, dev = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
    if (s->lds + 64 > (size_t)max_lds) return wind_fail(WIND_ERR_UNSUPPORTED, "network too large for LDS");
    auto kfn = block_kernel<METHOD>(fast, sc.pivot != 0);
    if (s->lds > 65536) {
        hipError_t e = hipFuncSetAttribute((const void *)kfn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)s->lds);
        if (e != hipSuccess) return wind_fail(WIND_ERR_DEVICE, hipGetErrorString(e));
    }
    int per_cu = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kfn, s->T, s->lds);
    if (e != hipSuccess) return wind_fail(WIND_ERR_DEVICE, hipGetErrorString(e));
    s->grid = scaled_grid(num_cu, per_cu, sc, nsys);
    return WIND_OK;
}

size_t scratch_bytes(const MassActionDevice &d, const BlockShape &s) {
    return s.in_lds ? 0 : sizeof(float) * 2 * (size_t)d.N * d.N * s.grid;
}

template <int NP>
int launch_ma_wave(int num_cu, const MassActionDevice &d, const IntegrateArgs &a, const SolverChoice &sc, hipStream_t st) {
    const size_t lds = sizeof(float) * ma_wave_lds_floats(NP, d.R);
    int per_cu = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, ma_wave_integrate<NP>, 128, lds);
    if (e != hipSuccess) return wind_fail(WIND_ERR_DEVICE, hipGetErrorString(e));
    hipLaunchKernelGGL(ma_wave_integrate<NP>, dim3(scaled_grid(num_cu, per_cu, sc, a.nsys)), dim3(128), lds, st, a, d);
    e = hipGetLastError();
    if (e != hipSuccess) return wind_fail(WIND_ERR_DEVICE, hipGetErrorString(e));
    return WIND_OK;
}

}  // namespace

template <int METHOD>
int mass_action_scratch_bytes(int num_cu, const wind_network *net, int mode, const SolverChoice &sc, int nsys,
                              size_t *bytes) {
    *bytes = 0;
    if (net->builtin != WIND_NET_MASS_ACTION) return WIND_OK;
    const MassActionPlan plan = mass_action_plan(net->ma, mode, sc.pivot != 0);
    if (plan.dense || plan.in_lds) return WIND_OK;
    BlockShape s;
    const int rc = block_shape<METHOD>(num_cu, net->ma, plan, mode == WIND_MODE_FAST, sc, nsys, &s);
    if (rc) return rc;
    *bytes = scratch_bytes(net->ma, s);
    return WIND_OK;
}

// Grows the scratch; a growth frees the old buffer, so anything that kept
// its address (a captured batch graph) must key on mass_action_scratch_ptr().
int mass_action_scratch_reserve(size_t need) {
    if (need <= g_scratch.bytes) return WIND_OK;
    if (g_scratch.ptr) (void)hipFree(g_scratch.ptr);
    g_scratch.ptr = nullptr;
    g_scratch.bytes = 0;
    hipError_t e = hipMalloc((void **)&g_scratch.ptr, need);
    if (e != hipSuccess) return wind_fail(WIND_ERR_DEVICE, hipGetErrorString(e));
    g_scratch.bytes = need;
    return WIND_OK;
}

const void *mass_action_scratch_ptr() { return g_scratch.ptr; }

template <int METHOD>
int launch_mass_action(int num_cu, const wind_network *net, const IntegrateArgs &a, int mode,
                       int kernel, const SolverChoice &sc, hipStream_t st) {
    if (kernel == WIND_KERNEL_LANE)
        return wind_fail(WIND_ERR_UNSUPPORTED, "mass-action networks run on the block kernel");
    const MassActionDevice &d = net->ma;
    const int N = d.N;
    const bool fast = mode == WIND_MODE_FAST;
    const MassActionPlan plan = mass_action_plan(d, mode, sc.pivot != 0);
    if (plan.dense) {
        if (METHOD == WIND_SIE && dense_reg_eligible(d, sc)) return launch_dense_reg(num_cu, d, a, sc, st);
        const size_t lds = plan.lds;
        int T = ((N + 15) & ~15) <= 64 ? 64 : 512;
        if (sc.block == 64 || sc.block == 128 || sc.block == 256 || sc.block == 512) T = sc.block;
        const int solver = sc.solver == WIND_SOLVER_AUTO ? WIND_SOLVER_MFMA_F32 : sc.solver;
        switch (solver) {
        case WIND_SOLVER_VALU: return launch_dense<METHOD, PREC_VALU>(num_cu, d, a, sc.ir_sweeps, lds, T, sc, st);
        case WIND_SOLVER_MFMA_F32:
            return launch_dense<METHOD, PREC_MFMA_F32>(num_cu, d, a, sc.ir_sweeps, lds, T, sc, st);
        case WIND_SOLVER_MFMA_BF16:
            return launch_dense<METHOD, PREC_MFMA_BF16>(num_cu, d, a, sc.ir_sweeps, lds, T, sc, st);
        default:
            return launch_dense<METHOD, PREC_MFMA_BF16X3>(num_cu, d, a, sc.ir_sweeps, lds, T, sc, st);
        }
    }
    if (a.trace.capacity > 0)
        return wind_fail(WIND_ERR_UNSUPPORTED, "trace: mass-action networks are traced by the dense solver "
                                               "(fast mode, N <= 176) only");
    if (METHOD == WIND_SIE && !fast && kernel == WIND_KERNEL_AUTO && d.ex_ent) {
        switch ((N + 7) / 8) {
        case 1: return launch_ma_wave<8>(num_cu, d, a, sc, st);
        case 2: return launch_ma_wave<16>(num_cu, d, a, sc, st);
        case 3: return launch_ma_wave<24>(num_cu, d, a, sc, st);
        case 4: return launch_ma_wave<32>(num_cu, d, a, sc, st);
        case 5: return launch_ma_wave<40>(num_cu, d, a, sc, st);
        case 6: return launch_ma_wave<48>(num_cu, d, a, sc, st);
        case 7: return launch_ma_wave<56>(num_cu, d, a, sc, st);
        default: return launch_ma_wave<64>(num_cu, d, a, sc, st);
        }
    }
    BlockShape s;
    int rc = block_shape<METHOD>(num_cu, d, plan, fast, sc, a.nsys, &s);
    if (rc) return rc;
    // Matrices beyond LDS live in the process-wide scratch, one slice per
    // workgroup.  Launches that use it must not overlap: callers hold the
    // context lock, and batches reserve it up front and put every bucket
    // that uses it on one stream.
    float *scratch = nullptr;
    if (!s.in_lds) {
        rc = mass_action_scratch_reserve(scratch_bytes(d, s));
        if (rc) return rc;
        scratch = g_scratch.ptr;
    }
    auto kfn = block_kernel<METHOD>(fast, sc.pivot != 0);
    hipLaunchKernelGGL(kfn, dim3(s.grid), dim3(s.T), s.lds, st, a, d, scratch, s.in_lds ? 1 : 0);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return wind_fail(WIND_ERR_DEVICE, hipGetErrorString(e));
    return WIND_OK;
}

template int launch_mass_action<WIND_SIE>(int, const wind_network *, const IntegrateArgs &, int, int,
                                          const SolverChoice &, hipStream_t);
template int launch_mass_action<WIND_RK2>(int, const wind_network *, const IntegrateArgs &, int, int,
                                          const SolverChoice &, hipStream_t);
template int mass_action_scratch_bytes<WIND_SIE>(int, const wind_network *, int, const SolverChoice &, int, size_t *);
template int mass_action_scratch_bytes<WIND_RK2>(int, const wind_network *, int, const SolverChoice &, int, size_t *);
