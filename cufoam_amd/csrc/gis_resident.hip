// CG and BiCG of one system that fits the chip: a whole solve in one launch.
//
// A small or mid-size system spends its iterations on launches and on the
// first-use latency of kernels too small to fill the chip (CG per iteration:
// 14 us at 16^3, 18 us at 64^3, 27 us at 63^3 renumbered, against a few us of
// work).  Here every workgroup owns one or two consecutive tiles for the whole
// solve: its matrix slots, r and x stay in registers, p in LDS, and only what
// another workgroup refers to travels through memory.  The two reductions of an
// iteration are also its two grid barriers: each workgroup publishes its
// subtree sum, and one wave of every workgroup reads and folds all of them.
// What bounds an iteration then is the latency of those two exchanges (about
// 1.2 us each between 4 workgroups, 3 us between 256); a single workgroup needs
// none and takes 1.0 us (one tile) or 1.7 us (two).  Measured per CG iteration:
// 5.4 us at 16^3, 9.3 us at 64^3, 9.3 us at 63^3 renumbered, 13.1 us at 80^3
// (23.5 before).
//
// Same arithmetic as the launch-per-stage kernels (p = fma(beta, p, r), rounded
// products summed in storage order, the pairwise reduction tree of
// gis_device.hpp), so every iterate has their bits.
//
// The workgroups of one launch wait for each other, so all of them must be
// resident.  A launch therefore starts with a handshake: it goes ahead only
// once every workgroup has arrived, and gives up (having changed nothing) when
// that takes too long, for instance because another program's kernel holds
// compute units.  The caller then runs the launch-per-stage loop, and the next
// solves go there without waiting.
#include <algorithm>
#include <climits>
#include <cmath>
#include <mutex>
#include <vector>

#include "gis_kernels.hpp"

namespace gis {

namespace {

constexpr int kResWG = 1024;          // 16 waves: one workgroup per CU
constexpr int kResEntries = 8;        // matrix entries per row it holds
constexpr int kResMaxGrid = 256;      // workgroups a reduction reads (4 slots per lane)
constexpr int kResSets = kResQ;       // slot sets and q buffers in rotation
// Every workgroup reads every slot, so a set is published in 8 copies on other
// memory channels, each read by every 8th workgroup (64^3: 12.6 us per iteration
// with one copy, 11.3 with 4, 11.1 with 8, 10.9 with 16).
constexpr int kResCopies = 8;
constexpr int kCopyStride = 1056;     // doubles between copies, 2 sums per workgroup
constexpr int kResSlots = kResCopies * kCopyStride;

struct ResWs {
    double* slot;         // kResSets x kResSlots published sums
    int* sync;            // [0] workgroups arrived, [1] verdict (kRes*)
    long long patience;   // wall-clock ticks to wait for the grid
};

enum : int { kResWait = 0, kResGo = 1, kResLate = 2, kResNoFit = 3 };

// A workgroup's place: workgroup g of the G that share one system, whose rows end
// at row_end; row0 is the workgroup's first.
struct ResPlace {
    int row0, row_end, g, G;
};

template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

constexpr int kHalfMirror = 0x141, kMirror = 0x140;   // lane i -> 7 - i of 8, 15 - i of 16
constexpr int kXor1 = 0xB1, kXor2 = 0x4E;             // within quads

// The sum of the 16-lane row's 4 leaves (one row of the matrix per lane): each
// leaf of 4 lanes accumulates fma(a, b, .) from +0.0 in lane order, rows that do
// not exist are skipped; the leaves are folded pairwise.  Every lane of the 16
// gets it.
__device__ __forceinline__ double leaf_tree16(double a, double b, bool valid) {
    double s = 0.0, t;
    t = valid ? fma(a, b, s) : s;
    s = dpp<0x00>(t);
    t = valid ? fma(a, b, s) : s;
    s = dpp<0x55>(t);
    t = valid ? fma(a, b, s) : s;
    s = dpp<0xAA>(t);
    t = valid ? fma(a, b, s) : s;
    s = dpp<0xFF>(t);
    s = s + dpp<kHalfMirror>(s);
    s = s + dpp<kMirror>(s);
    return s;
}

// wave_tree of one value without LDS traffic
__device__ __forceinline__ double wave_total(double v) {
    v = v + dpp<kXor1>(v);
    v = v + dpp<kXor2>(v);
    v = v + dpp<kHalfMirror>(v);
    v = v + dpp<kMirror>(v);
    // every 16-lane row is uniform here: swapping odd rows of one copy with even
    // rows of the other leaves both partners' values in the lane
    {
        const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v),
                                                         false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v),
                                                         false, false);
        v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
    }
    {
        const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v),
                                                         false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v),
                                                         false, false);
        v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
    }
    return v;
}

// All workgroups of the launch, or none: true once gridDim.x have arrived.  A
// workgroup that cannot take part (fits = false) gives up for all.  The verdict
// of a launch that does not go ahead is left in *verdict.
__device__ __forceinline__ bool arrive_all(const ResWs& ws, bool fits, int* verdict, int* sh) {
    if (threadIdx.x == 0) {
        auto settle = [&](int to) {
            int expect = kResWait;
            (void)__hip_atomic_compare_exchange_strong(&ws.sync[1], &expect, to, __ATOMIC_RELAXED,
                                                       __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT);
        };
        if (!fits) settle(kResNoFit);
        else if (__hip_atomic_fetch_add(&ws.sync[0], 1, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1)
            settle(kResGo);
        const long long t0 = wall_clock64();
        int s;
        while ((s = __hip_atomic_load(&ws.sync[1], __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT)) == kResWait) {
            if (wall_clock64() - t0 > ws.patience) settle(kResLate);
            __builtin_amdgcn_s_sleep(1);
        }
        if (s != kResGo) *verdict = s;
        *sh = s;
    }
    __syncthreads();
    return *sh == kResGo;
}

// Wave 0, with the workgroup's 64 x RPT sums of 16 rows in part[v]: the totals
// over the grid, in every lane.  Slot sets rotate: whoever has completed
// reduction s knows that every workgroup has published s and so has finished
// reading s - 1; it then empties its own slots of s - 1, which are published
// again by reduction s + 2 (the caller waits for the emptying before the next
// publication).  ok = false when the bounded wait ran out.
template <int RPT, int NV>
__device__ __forceinline__ void allreduce(const double (*part)[64 * RPT], const ResWs& ws,
                                          const ResPlace& at, unsigned phase, int fault, double (&t)[NV], bool& ok) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        double e[RPT];
#pragma unroll
        for (int i = 0; i < RPT; ++i) e[i] = part[v][lane * RPT + i];
#pragma unroll
        for (int h = 1; h < RPT; h <<= 1)
#pragma unroll
            for (int i = 0; i + h < RPT; i += 2 * h) e[i] = e[i] + e[i + h];
        t[v] = wave_total(e[0]);
    }
    const int G = at.G;
    ok = true;
    if (G == 1) return;
    double* set = ws.slot + (size_t)(phase % kResSets) * kResSlots;
    double* own = set + (size_t)lane * kCopyStride + at.g;   // lane < kResCopies
    if (lane < kResCopies) {
#pragma unroll
        for (int v = 0; v < NV; ++v) st_agent(own + v * kResMaxGrid, t[v]);
    }
    const double* mine = set + (size_t)(at.g % kResCopies) * kCopyStride;
    const int limit = fault > 0 ? fault : kSlotSpins;
    double x[NV][4];
    for (int spins = 0;; ++spins) {
        int miss = fault > 0 ? 1 : 0;
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int s = j * 64 + lane;
                x[v][j] = 0.0;
                if (j * 64 < G) {
                    if (s < G) x[v][j] = ld_agent(mine + v * kResMaxGrid + s);
                    miss |= slot_empty(x[v][j]) ? 1 : 0;
                }
            }
        if (!__any(miss)) break;
        if (spins >= limit) {
            ok = false;
            break;
        }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {   // groups of 64, then pairwise: the tree's upper levels
        t[v] = wave_total(x[v][0]);
        if (G > 64) t[v] = t[v] + wave_total(x[v][1]);
        if (G > 128) t[v] = t[v] + (wave_total(x[v][2]) + wave_total(x[v][3]));
    }
    if (lane < kResCopies) {
        double* old = ws.slot + (size_t)((phase + 2) % kResSets) * kResSlots +
                      (size_t)lane * kCopyStride + at.g;
        slot_clear(old);
        slot_clear(old + kResMaxGrid);
    }
}

// Geometry of a workgroup of RPT tiles that exchanges M vectors (CG: q; BiCG: q and
// q*).  Each LDS vector: its own rows, the halo (the other workgroups' rows its
// rows refer to, each once), and one zero that absent entries read.
template <int RPT, int M, bool ALONE>
struct ResGeom {
    static constexpr int kRows = kResWG * RPT;
    static constexpr int kHpt = ALONE ? 0 : M == 2 ? 4 : RPT == 1 ? 8 : 5;   // halo rows a thread
    static constexpr int kHalo = kHpt * kResWG;
    static constexpr int kZero = kRows + kHalo;
    static constexpr int kHash = ALONE ? 0 : 16384;   // set-up: hash table of the halo columns
    static constexpr int kHashBits = 14;
    static constexpr size_t kBytesP = sizeof(double) * M * (kZero + 1);
    static constexpr size_t kBytesSetup = sizeof(int) * (size_t)(kHash + kHalo);
    static constexpr size_t kBytes = kBytesP > kBytesSetup ? kBytesP : kBytesSetup;
};

// A value the compiler may not derive others from ahead of the loop: decoding it
// again every iteration costs less than the registers to keep the results (80^3:
// 15.1 -> 13.1 us per iteration).
__device__ __forceinline__ unsigned fresh(unsigned v) {
    asm volatile("" : "+v"(v));
    return v;
}

// What a thread holds of the matrix: RPT rows' slots (rows 64 apart), where each
// entry's vector value lies in the LDS vectors (two places a word), and its halo
// columns.
template <int RPT, int M, bool ALONE>
struct ResRows {
    static constexpr int H = ResGeom<RPT, M, ALONE>::kHpt;
    unsigned addr[RPT][kResEntries / 2];
    int hcol[H > 0 ? H : 1];   // -1: none
    unsigned pub;              // bit i: row i is read by other workgroups
    int nh;                    // the workgroup's halo rows
};

// TAB: the slots of the column-offset tables (every slice tabled); else the int32
// slot columns.  val / valT: the slot values of A, and of A^T (M = 2) from mt.
// Ends with a workgroup barrier, the LDS vectors free.
template <int RPT, int M, bool TAB, bool ALONE>
__device__ __forceinline__ void res_rows(const Mat<double>& m, const Mat<double>& mt,
                                         const ResPlace& place, unsigned char* lds, int* n_halo, int* wsum,
                                         ResRows<RPT, M, ALONE>& rows,
                                         double (&val)[RPT][kResEntries],
                                         double (&valT)[M == 2 ? RPT : 1][kResEntries]) {
    using G = ResGeom<RPT, M, ALONE>;
    constexpr int K = kResEntries;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row0 = place.row0, N = place.row_end;
    const int nloc = min(G::kRows, N - row0);
    const int nslices = (N + kSlice - 1) / kSlice;
    int* hash = reinterpret_cast<int*>(lds);
    int* list = hash + G::kHash;
    for (int i = tid; i < G::kHash; i += kResWG) hash[i] = -1;
    if (tid == 0) *n_halo = 0;
    __syncthreads();
    rows.pub = 0;
    int at[RPT][K];
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        const int s = min(row0 / kSlice + w * RPT + i, nslices - 1);
        const int row = row0 + (w * RPT + i) * kSlice + lane;
        const int o = TAB ? m.ooff[s] : m.soff[s];
        const int len = TAB ? m.ooff[s + 1] - o : (m.soff[s + 1] - o) / kSlice;
        unsigned mask = 0;
        if constexpr (TAB) mask = row_mask(m.dmask, m.dmask8, len, row, N);   // 0 past the end
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int kk = min(k, len - 1);
            bool on;
            int c;
            if constexpr (TAB) {
                const size_t slot = ((size_t)o + kk) * kSlice + lane;
                on = k < len && ((mask >> k) & 1u);
                c = row + m.doffs[o + kk];
                val[i][k] = on ? m.dval[slot] : 0.0;
                if constexpr (M == 2) valT[i][k] = on ? mt.dval[slot] : 0.0;
            } else {
                const int slot = o + kk * kSlice + lane;
                c = m.scol[slot];
                on = k < len && c >= 0 && row < N;
                val[i][k] = on ? m.sval[slot] : 0.0;
                if constexpr (M == 2) valT[i][k] = on ? mt.sval[slot] : 0.0;
            }
            int a = G::kZero;
            if (on) {
                a = c - row0;
                if (!ALONE && (unsigned)a >= (unsigned)nloc) {   // insert c into the halo
                    rows.pub |= 1u << i;
                    unsigned pos = ((unsigned)c * 2654435761u) >> (32 - G::kHashBits);
                    for (int tries = 0; tries < G::kHash; ++tries) {
                        const int old = atomicCAS(&hash[pos], -1, c);
                        if (old == -1 || old == c) break;
                        pos = (pos + 1) & (G::kHash - 1);
                    }
                    a = -1 - (int)pos;
                }
            }
            at[i][k] = a;
        }
    }
    if constexpr (!ALONE) {
        __syncthreads();
        // halo index of each occupied table position, in table order
        constexpr int kPer = G::kHash / kResWG;
        int cnt = 0;
#pragma unroll
        for (int j = 0; j < kPer; ++j) cnt += hash[tid * kPer + j] >= 0 ? 1 : 0;
        int incl = cnt;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(incl, o, 64);
            if (lane >= o) incl += y;
        }
        if (lane == 63) wsum[w] = incl;
        __syncthreads();
        int base = incl - cnt;
        for (int j = 0; j < w; ++j) base += wsum[j];
        if (tid == kResWG - 1) *n_halo = base + cnt;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int c = hash[tid * kPer + j];
            if (c >= 0) {
                if (base < G::kHalo) list[base] = c;
                hash[tid * kPer + j] = base++;
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < RPT; ++i)
#pragma unroll
        for (int k = 0; k < K; k += 2) {
            const int a = at[i][k], b = at[i][k + 1];
            rows.addr[i][k / 2] =
                (unsigned)(a < 0 ? G::kRows + hash[-1 - a] : a) |
                ((unsigned)(b < 0 ? G::kRows + hash[-1 - b] : b) << 16);
        }
    rows.nh = ALONE ? 0 : __builtin_amdgcn_readfirstlane(*n_halo);
    if constexpr (!ALONE) {
#pragma unroll
        for (int j = 0; j < G::kHpt; ++j) {
            const int h = j * kResWG + tid;
            rows.hcol[j] = h < min(rows.nh, G::kHalo) ? list[h] : -1;
        }
    }
    __syncthreads();
}

// Row i's product with the LDS vector v: rounded products in storage order.  An
// absent entry adds 0 * 0 (it reads the zero), which leaves the sum as it is.
template <int RPT, int M, bool ALONE>
__device__ __forceinline__ double res_row(const ResRows<RPT, M, ALONE>& rows, int i,
                                          const double (&val)[kResEntries], const double* v) {
    constexpr int K = kResEntries;
    double g[K];
#pragma unroll
    for (int e = 0; e < K; e += 2) {
        const unsigned ab = RPT > 1 ? fresh(rows.addr[i][e / 2]) : rows.addr[i][e / 2];
        g[e] = v[ab & 0xffffu];
        g[e + 1] = v[ab >> 16];
    }
    double acc = 0.0;
#pragma unroll
    for (int e = 0; e < K; ++e) acc = acc + val[e] * g[e];
    return acc;
}

// The halo rows' values of M exchanged vectors (buffers M n apart in qx), polled
// until written; false when the bounded wait ran out.
template <int RPT, int M, bool ALONE, class Use>
__device__ __forceinline__ bool poll_halo(const ResRows<RPT, M, ALONE>& rows, const double* qx,
                                          size_t n, int fault, Use&& use) {
    constexpr int H = ResRows<RPT, M, ALONE>::H;
    const int limit = fault > 0 ? fault : kSlotSpins;
    double q[M][H > 0 ? H : 1];
    bool got = true;
    for (int spins = 0;; ++spins) {
        int miss = fault > 0 ? 1 : 0;
#pragma unroll
        for (int v = 0; v < M; ++v)
#pragma unroll
            for (int j = 0; j < H; ++j)
                if (j * kResWG < rows.nh) {
                    q[v][j] = rows.hcol[j] >= 0 ? ld_agent(qx + v * n + rows.hcol[j]) : 0.0;
                    miss |= slot_empty(q[v][j]) ? 1 : 0;
                }
        if (!__any(miss)) break;
        if (spins >= limit) {
            got = false;
            break;
        }
    }
#pragma unroll
    for (int j = 0; j < H; ++j)
        if (j * kResWG < rows.nh) {
            double qj[M];
#pragma unroll
            for (int v = 0; v < M; ++v) qj[v] = q[v][j];
            use(j, qj);
        }
    return got;
}

// The workgroup's slots and exchanged rows emptied, then the handshake.
template <int RPT, int M, bool ALONE>
__device__ __forceinline__ bool res_start(const ResRows<RPT, M, ALONE>& rows, const ResWs& ws,
                                          const ResPlace& at, double* qx, size_t n, int row,
                                          int* verdict, int* sh) {
    using G = ResGeom<RPT, M, ALONE>;
    if constexpr (ALONE) {
        __syncthreads();
        return true;
    }
#pragma unroll
    for (int i = 0; i < RPT; ++i)
        if ((rows.pub >> i) & 1u)
#pragma unroll
            for (int b = 0; b < M * kResSets; ++b) slot_clear(qx + b * n + row + i * kSlice);
    const int tid = threadIdx.x;
    if (tid < kResSets * kResCopies) {
        double* s = ws.slot + (size_t)(tid / kResCopies) * kResSlots +
                    (size_t)(tid % kResCopies) * kCopyStride + at.g;
        slot_clear(s);
        slot_clear(s + kResMaxGrid);
    }
    order_release();
    __syncthreads();
    return arrive_all(ws, rows.nh <= G::kHalo, verdict, sh);
}

__device__ __forceinline__ void res_hist(const KState* st, const ResPlace& at, double* hist,
                                         int hist_cap, int detail, int k, double norm) {
    if (at.g == 0 && k < hist_cap)
        hist[k] = detail ? (double)(wall_clock64() - st->t0) * st->tick : norm;
}

// CG (k_cg1, k_cg2).  A workgroup follows the p and r of its halo rows itself
// (the same fma as their owners), so the one thing exchanged is q: the owner of a
// row that others refer to stores q with an agent-scope store, and they poll for
// it while the second reduction of the iteration is under way (q buffers hold
// kSlotEmpty until written).  Structural symmetry tells the owner which rows those
// are: the rows that themselves refer to another workgroup's row.  Three q
// buffers rotate: whoever has completed the first reduction of iteration k knows
// that every workgroup is done with q of k - 1, and empties its rows there; they
// are written again in iteration k + 2.
//
// n: the vectors' length (q buffers lie n apart).  verdict: arrive_all's.
template <int RPT, bool TAB, bool ALONE>
__device__ __forceinline__ void cg_res(const Mat<double>& m, const ResPlace& at, size_t n,
                                       double* __restrict__ r, double* __restrict__ p,
                                       double* __restrict__ qx, double* __restrict__ x,
                                       KState* st, const ResWs& ws, int chunk, int* verdict) {
    using G = ResGeom<RPT, 1, ALONE>;
    constexpr int H = G::kHpt;
    __shared__ __attribute__((aligned(16))) unsigned char lds[G::kBytes];
    __shared__ double part[1][64 * RPT];
    __shared__ double bc[2];
    __shared__ int bci, n_halo, wsum[kResWG / 64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row0 = at.row0, N = at.row_end;
    const int nloc = min(G::kRows, N - row0);
    const int li0 = w * RPT * kSlice + lane;   // the thread's rows: li0, li0 + 64, ...
    const int k0 = st->k, fault = st->slot_fault;
    const double error = st->error;
    const long long max_steps = st->max_steps, min_steps = st->min_steps;
    double* const hist = st->hist;
    const int hist_cap = st->hist_cap, detail = st->detail;
    double beta = st->beta, alpha = st->alpha;
    double rho = st->rho0, rho1 = st->rho1, norm = st->norm;

    ResRows<RPT, 1, ALONE> rows;
    double val[RPT][kResEntries], none[1][kResEntries];
    res_rows<RPT, 1, TAB, ALONE>(m, m, at, lds, &n_halo, wsum, rows, val, none);
    double* sp = reinterpret_cast<double*>(lds);
    if (tid == 0) sp[G::kZero] = 0.0;
    double rv[RPT], xv[RPT], rh[H > 0 ? H : 1];
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        const int li = li0 + i * kSlice;
        const bool in = li < nloc;
        rv[i] = in ? r[row0 + li] : 0.0;
        xv[i] = in ? x[row0 + li] : 0.0;
        sp[li] = in && k0 > 0 ? p[row0 + li] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < H; ++j) {
        rh[j] = rows.hcol[j] >= 0 ? r[rows.hcol[j]] : 0.0;
        if (j * kResWG < rows.nh)
            sp[G::kRows + j * kResWG + tid] =
                rows.hcol[j] >= 0 && k0 > 0 ? p[rows.hcol[j]] : 0.0;
    }
    if (!res_start(rows, ws, at, qx, n, row0 + li0, verdict, &bci)) return;

    unsigned phase = 0;
    bool stop = false, ok = true;
    int k = k0, qb = 0;
    for (int it = 0; it < chunk && !stop; ++it) {
        ++k;
        const bool first = k == 1;
        double* q_new = qx + (size_t)qb * n;
        qb = qb == kResSets - 1 ? 0 : qb + 1;
        double* q_old = qx + (size_t)(qb == kResSets - 1 ? 0 : qb + 1) * n;   // of k - 1
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            const int li = li0 + i * kSlice;
            sp[li] = first ? rv[i] : fma(beta, sp[li], rv[i]);
        }
#pragma unroll
        for (int j = 0; j < H; ++j)
            if (j * kResWG < rows.nh) {
                const int h = G::kRows + j * kResWG + tid;
                sp[h] = first ? rh[j] : fma(beta, sp[h], rh[j]);
            }
        __syncthreads();
        if (w == 0) order_release();   // the slots it emptied in the last reduction
        double q[RPT];
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            const int li = li0 + i * kSlice;
            q[i] = res_row(rows, i, val[i], sp);
            if ((rows.pub >> i) & 1u) st_agent(q_new + row0 + li, q[i]);
            const double t = leaf_tree16(sp[li], q[i], li < nloc);
            if ((lane & 15) == 0) part[0][(w * RPT + i) * 4 + (lane >> 4)] = t;
        }
        __syncthreads();
        if (w == 0) {
            double t[1];
            allreduce<RPT, 1>(part, ws, at, phase, fault, t, ok);
            alpha = rho / t[0];
            if (lane == 0) {
                bc[0] = alpha;
                bci = ok ? 0 : 1;
            }
        }
        ++phase;
        __syncthreads();
        const double al = bc[0];
        if (bci) {
            ok = false;
            break;
        }
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            rv[i] = fma(-al, q[i], rv[i]);
            const double t = leaf_tree16(rv[i], rv[i], li0 + i * kSlice < nloc);
            if ((lane & 15) == 0) part[0][(w * RPT + i) * 4 + (lane >> 4)] = t;
        }
        order_release();   // q, and the rows emptied before, are in memory
        __syncthreads();
        if (w == 0) {
            double t[1];
            allreduce<RPT, 1>(part, ws, at, phase, fault, t, ok);
            rho1 = rho;
            rho = t[0];
            beta = rho / rho1;
            norm = sqrt(t[0]);
            if (lane == 0) {
                bc[1] = beta;
                bci = !ok ? 2
                          : ((!(norm > error) || k >= max_steps) && k >= min_steps) ? 1 : 0;
                if (ok) res_hist(st, at, hist, hist_cap, detail, k, norm);
            }
        }
        ++phase;
        bool got = true;
        if (!ALONE && rows.nh > 0) {
            // a moment's pause lets wave 0's publication go first (64^3: 11.1 -> 9.9
            // us per iteration; 8 and 2 instead of 4: 10.4 and 10.7)
            if (w) __builtin_amdgcn_s_sleep(4);
            got = poll_halo(rows, q_new, n, fault, [&](int j, const double (&qj)[1]) {
                rh[j] = fma(-al, qj[0], rh[j]);
            });
        }
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            const int li = li0 + i * kSlice;
            xv[i] = fma(al, sp[li], xv[i]);
            if ((rows.pub >> i) & 1u) slot_clear(q_old + row0 + li);
        }
        if (!__syncthreads_and(got)) {
            ok = false;
            break;
        }
        beta = bc[1];
        stop = bci != 0;
        if (bci == 2) ok = false;
    }
    if (!ok) {   // some workgroup never came: the solve has failed
        if (tid == 0) slot_fail(st, 1);
        return;
    }
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        const int li = li0 + i * kSlice;
        if (li < nloc) {
            x[row0 + li] = xv[i];
            r[row0 + li] = rv[i];
            p[row0 + li] = sp[li];
        }
    }
    if (at.g == 0 && tid == 0) {
        st->k = k;
        st->norm = norm;
        st->rho0 = rho;
        st->rho1 = rho1;
        st->alpha = alpha;
        st->beta = beta;
        if (stop) st->done = 1;
    }
}

template <int RPT, bool TAB, bool ALONE>
__global__ __launch_bounds__(kResWG) void k_cg_res(Mat<double> m, int N, double* __restrict__ r,
                                                   double* __restrict__ p, double* __restrict__ qx,
                                                   double* __restrict__ x, KState* st, ResWs ws,
                                                   int chunk) {
    if (st->done) return;
    const ResPlace at{(int)blockIdx.x * kResWG * RPT, N, (int)blockIdx.x, (int)gridDim.x};
    cg_res<RPT, TAB, ALONE>(m, at, (size_t)N, r, p, qx, x, st, ws, chunk, &st->flag);
}

// Several systems of a batch in one launch: block b's place, system and slots.
struct ResBlock {
    ResPlace at;
    int sys, slot;
};

template <int RPT>
__global__ __launch_bounds__(kResWG) void k_bcg_res(Mat<double> m, size_t n,
                                                    double* __restrict__ r,
                                                    double* __restrict__ p,
                                                    double* __restrict__ qx,
                                                    double* __restrict__ x, KState* states,
                                                    const ResBlock* __restrict__ blocks, ResWs ws,
                                                    int chunk) {
    const ResBlock b = blocks[blockIdx.x];
    KState* st = states + b.sys;
    if (st->done) {   // the others wait for this workgroup too
        __shared__ int verdict;
        (void)arrive_all(ws, true, &ws.sync[2], &verdict);
        return;
    }
    ws.slot += (size_t)b.slot * kResSets * kResSlots;
    cg_res<RPT, false, false>(m, b.at, n, r, p, qx, x, st, ws, chunk, &ws.sync[2]);
    // x is complete: nothing is left to k_bcg_flush
    if (b.at.g == 0 && threadIdx.x == 0 && st->k > 0) st->flag = 1;
}

// BiCG (k_bicg1, k_bicg2<P, 0>) in the same way, with A's slots from m and A^T's
// from mt: q = A p and q* = A^T p* are exchanged together, and the second
// reduction carries (r, r) and (r, r*).
template <bool TAB, bool ALONE>
__global__ __launch_bounds__(kResWG) void k_bicg_res(Mat<double> m, Mat<double> mt, int N,
                                                     double* __restrict__ r,
                                                     double* __restrict__ rs,
                                                     double* __restrict__ p,
                                                     double* __restrict__ ps,
                                                     double* __restrict__ qx,
                                                     double* __restrict__ x, KState* st, ResWs ws,
                                                     int chunk) {
    using G = ResGeom<1, 2, ALONE>;
    constexpr int H = G::kHpt;
    __shared__ __attribute__((aligned(16))) unsigned char lds[G::kBytes];
    __shared__ double part[2][64];
    __shared__ double bc[2];
    __shared__ int bci, n_halo, wsum[kResWG / 64];
    if (st->done) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const ResPlace at{(int)blockIdx.x * G::kRows, N, (int)blockIdx.x, (int)gridDim.x};
    const int row0 = at.row0;
    const int nloc = min(G::kRows, N - row0);
    const bool in = tid < nloc;
    const int row = row0 + tid;
    const size_t n = (size_t)N;
    const int k0 = st->k, fault = st->slot_fault;
    const double error = st->error, bound = st->int_bound;
    const long long max_steps = st->max_steps, min_steps = st->min_steps;
    double* const hist = st->hist;
    const int hist_cap = st->hist_cap, detail = st->detail;
    double beta = st->beta, xi = st->alpha;
    double rho = st->rho0, rho1 = st->rho1, norm = st->norm;

    ResRows<1, 2, ALONE> rows;
    double val[1][kResEntries], valT[1][kResEntries];
    res_rows<1, 2, TAB, ALONE>(m, mt, at, lds, &n_halo, wsum, rows, val, valT);
    double* sp = reinterpret_cast<double*>(lds);
    double* sps = sp + G::kZero + 1;
    if (tid == 0) sp[G::kZero] = sps[G::kZero] = 0.0;
    double rv = in ? r[row] : 0.0, rsv = in ? rs[row] : 0.0, xv = in ? x[row] : 0.0;
    double rh[H > 0 ? H : 1], rsh[H > 0 ? H : 1];
    sp[tid] = in && k0 > 0 ? p[row] : 0.0;
    sps[tid] = in && k0 > 0 ? ps[row] : 0.0;
#pragma unroll
    for (int j = 0; j < H; ++j) {
        const int c = rows.hcol[j];
        rh[j] = c >= 0 ? r[c] : 0.0;
        rsh[j] = c >= 0 ? rs[c] : 0.0;
        if (j * kResWG < rows.nh) {
            const int h = G::kRows + j * kResWG + tid;
            sp[h] = c >= 0 && k0 > 0 ? p[c] : 0.0;
            sps[h] = c >= 0 && k0 > 0 ? ps[c] : 0.0;
        }
    }
    if (!res_start(rows, ws, at, qx, n, row, &st->flag, &bci)) return;

    unsigned phase = 0;
    bool stop = false, ok = true, broke = false;
    int k = k0, qb = 0;
    for (int it = 0; it < chunk && !stop; ++it) {
        const bool first = k == 0;
        double* q_new = qx + (size_t)(2 * qb) * n;
        qb = qb == kResSets - 1 ? 0 : qb + 1;
        double* q_old = qx + (size_t)(2 * (qb == kResSets - 1 ? 0 : qb + 1)) * n;   // last one's
        sp[tid] = first ? rv : fma(beta, sp[tid], rv);
        sps[tid] = first ? rsv : fma(beta, sps[tid], rsv);
#pragma unroll
        for (int j = 0; j < H; ++j)
            if (j * kResWG < rows.nh) {
                const int h = G::kRows + j * kResWG + tid;
                sp[h] = first ? rh[j] : fma(beta, sp[h], rh[j]);
                sps[h] = first ? rsh[j] : fma(beta, sps[h], rsh[j]);
            }
        __syncthreads();
        if (w == 0) order_release();   // the slots it emptied in the last reduction
        const double q = res_row(rows, 0, val[0], sp);
        const double qs = res_row(rows, 0, valT[0], sps);
        if (rows.pub) {
            st_agent(q_new + row, q);
            st_agent(q_new + n + row, qs);
        }
        {
            const double t = leaf_tree16(sps[tid], q, in);
            if ((lane & 15) == 0) part[0][w * 4 + (lane >> 4)] = t;
        }
        __syncthreads();
        if (w == 0) {
            double t[1];
            allreduce<1, 1>(part, ws, at, phase, fault, t, ok);
            xi = rho / t[0];
            if (lane == 0) {
                bc[0] = xi;
                bci = !ok ? 2 : (xi > -bound && xi < bound) ? 1 : 0;
            }
        }
        ++phase;
        __syncthreads();
        const double a = bc[0];
        if (bci) {
            ok = bci != 2;
            broke = bci == 1;
            break;
        }
        rv = fma(-a, q, rv);
        rsv = fma(-a, qs, rsv);
        {
            const double t0 = leaf_tree16(rv, rv, in);
            const double t1 = leaf_tree16(rv, rsv, in);
            if ((lane & 15) == 0) {
                part[0][w * 4 + (lane >> 4)] = t0;
                part[1][w * 4 + (lane >> 4)] = t1;
            }
        }
        ++k;
        order_release();   // q, q*, and the rows emptied before, are in memory
        __syncthreads();
        if (w == 0) {
            double t[2];
            allreduce<1, 2>(part, ws, at, phase, fault, t, ok);
            norm = sqrt(t[0]);
            const bool end = (norm < error || k >= max_steps) && k >= min_steps;
            if (!end) {
                rho1 = rho;
                rho = t[1];
                beta = rho / rho1;
            }
            if (lane == 0) {
                bc[1] = beta;
                bci = !ok ? 2 : end ? 1 : 0;
                if (ok) res_hist(st, at, hist, hist_cap, detail, k, norm);
            }
        }
        ++phase;
        bool got = true;
        if (!ALONE && rows.nh > 0) {
            if (w) __builtin_amdgcn_s_sleep(4);   // as k_cg_res
            got = poll_halo(rows, q_new, n, fault, [&](int j, const double (&qj)[2]) {
                rh[j] = fma(-a, qj[0], rh[j]);
                rsh[j] = fma(-a, qj[1], rsh[j]);
            });
        }
        xv = fma(a, sp[tid], xv);
        if (rows.pub) {
            slot_clear(q_old + row);
            slot_clear(q_old + n + row);
        }
        if (!__syncthreads_and(got)) {
            ok = false;
            break;
        }
        beta = bc[1];
        stop = bci != 0;
        if (bci == 2) ok = false;
    }
    if (!ok) {
        if (tid == 0) slot_fail(st, 1);
        return;
    }
    if (in) {
        x[row] = xv;
        r[row] = rv;
        rs[row] = rsv;
        p[row] = sp[tid];
        ps[row] = sps[tid];
    }
    if (blockIdx.x == 0 && tid == 0) {
        st->k = k;
        st->norm = norm;
        st->rho0 = rho;
        st->rho1 = rho1;
        st->alpha = xi;
        st->beta = beta;
        if (broke) st->status = kBreakdown;
        if (stop || broke) st->done = 1;
    }
}

// verdict: kResWait, or kResLate for a launch that is to find its grid late; fault
// > 0 (gis_set_resident_fault): the waits inside the launch are to run out
__global__ void k_res_reset(ResWs ws, KState* st, int verdict, int fault) {
    if (threadIdx.x == 0) ws.sync[0] = 0;
    if (threadIdx.x == 1) ws.sync[1] = verdict;
    if (threadIdx.x == 2) st->flag = 0;
    if (threadIdx.x == 3 && fault > 0) st->slot_fault = fault;
}

// One waiting grid per GPU in this process: two that share the chip could each
// hold what the other waits for (their handshakes would end that, late).
constexpr int kResDevices = 16;
std::mutex g_resident[kResDevices];

// Iterations per launch: the host looks at the state in between.
constexpr int kResChunk = 2048;

// How long a launch waits for its grid.  A solve that is under way has nothing
// else to do, so its later launches wait up to 16 times as long, and are tried
// again until about 80 s have gone.
constexpr double kResPatience = 5e-3;
constexpr int kResRetries = 1000;

// After a launch whose grid came late (another program's kernels hold compute
// units), the next 1, 3, 7, .. 63 solves of the handle go stage by stage without
// waiting for theirs: at most one solve in 64 then pays the 5 ms.  A launch that
// runs ends it.
constexpr int kResMaxBackoff = 63;

bool held_back(gis_context* h) {
    if (h->res_skip == 0) return false;
    --h->res_skip;
    ++h->res_count[kResSkipped];
    return true;
}

void hold_back_next(gis_context* h, bool late) {
    h->res_backoff = late ? std::min(2 * h->res_backoff + 1, kResMaxBackoff) : 0;
    h->res_skip = h->res_backoff;
}

long long patience_ticks(const gis_context* h, int late) {
    const double tick = h->wall_tick > 0.0 ? h->wall_tick : 1e-8;
    return (long long)(kResPatience / tick) << std::min(late, 4);
}

// gis_set_late_launches: which of the next n launches find their grid late
struct LateLaunches {
    int first, end;
};

LateLaunches late_launches(gis_context* h, int n) {
    const int first = std::min(h->late_after, n), end = first + std::min(h->late_n, n - first);
    h->late_after -= first;
    h->late_n -= end - first;
    return {first, end};
}

// A launch's verdict (0: it ran) into the handle's counts.
void count_launch(gis_context* h, int verdict) {
    ++h->res_count[verdict == 0           ? kResRan
                   : verdict == kResNoFit ? kResUnfit
                                          : kResTooLate];
}

// Launches chunks until the solve is done.  launch(ws) enqueues one.  *ran =
// false: nothing was done.
template <class Launch>
int run_resident(gis_context* h, int form, Launch&& launch, bool* ran) {
    *ran = false;
    if (held_back(h)) return kOK;
    std::unique_lock<std::mutex> lock(g_resident[h->device], std::try_to_lock);
    if (!lock.owns_lock()) {
        ++h->res_count[kResSkipped];
        return kOK;
    }
    const size_t n_slot = (size_t)kResSets * kResSlots;
    GIS_HIP(h, h->res_mem.ensure(sizeof(double) * n_slot + 64));
    double* s = h->res_mem.as<double>();
    for (int late = 0;;) {
        const ResWs ws{s, reinterpret_cast<int*>(s + n_slot), patience_ticks(h, late)};
        const LateLaunches f = late_launches(h, 1);
        hipLaunchKernelGGL(k_res_reset, dim3(1), dim3(64), 0, h->stream, ws, h->st,
                           f.first < f.end ? kResLate : kResWait, h->res_fault);
        launch(ws);
        GIS_HIP(h, hipGetLastError());
        GIS_TRY(read_state(h));
        const KState& st = *h->st_host;
        if (st.flag == kResNoFit) h->res_unfit[form] = true;   // the pattern's halo is too large
        count_launch(h, st.flag);
        if (!*ran) hold_back_next(h, st.flag == kResLate);
        if (st.flag != 0 && !*ran) return kOK;
        // a later chunk that could not start is tried again: its r and p are the
        // resident form's
        if (st.flag != 0 && ++late > kResRetries)
            return fail(h, kErrSync, "the solve's grid could not be made resident again");
        *ran = true;
        if (st.done) return kOK;
    }
}

// 4 words a launch; launches [late0, late1) are to find their grid late; fault as
// k_res_reset, for the S systems
__global__ void k_res_reset_all(int* sync, int n, int late0, int late1, KState* st, int S,
                                int fault) {
    if (fault > 0)
        for (int i = threadIdx.x; i < S; i += blockDim.x) st[i].slot_fault = fault;
    for (int i = threadIdx.x; i < 4 * n; i += blockDim.x)
        sync[i] = i % 4 == 1 && i / 4 >= late0 && i / 4 < late1 ? kResLate : 0;
}

// TAB form of the pattern; false: it takes no resident form.  The int32 slots
// serve where some slice has no offset table, or a long one.
bool res_form(const gis_context* h, int form, bool* tab) {
    // iteration timers count the stages' launches; a chosen schedule is a choice of them
    if (h->sched_pinned || (h->timer.mask & 0x13) || h->res_unfit[form] ||
        h->device >= kResDevices)
        return false;
    *tab = h->lay_table_slices == h->lay_slices && h->lay_max_table <= kResEntries;
    return *tab || h->lay_max_row <= kResEntries;
}

// Tiles per workgroup of a resident CG, 0: none.  One tile as long as the chip
// has a CU for each (a second costs 0.7 us more per iteration than the smaller
// grid saves: 64^3 9.3 against 10.1 us), and two tiles as a single workgroup, which
// exchanges nothing (12^3: 3.3 against 5.5 us).
int res_cg_tiles(const gis_context* h) {
    const int T = tiles_of(h->N), G = std::min(h->n_cu, kResMaxGrid);
    return T <= 2 ? T : T <= G ? 1 : T <= 2 * G ? 2 : 0;
}

}  // namespace

bool resident_cg_fits(const gis_context* h) {
    bool tab;
    return res_form(h, kResCg, &tab) && res_cg_tiles(h) != 0;
}

bool resident_bicg_fits(const gis_context* h) {
    bool tab;
    return res_form(h, kResBicg, &tab) && tiles_of(h->N) <= std::min(h->n_cu, kResMaxGrid);
}

int resident_cg(gis_context* h, const Mat<double>& m, double* r, double* p, double* qx, double* x,
                bool* ran) {
    *ran = false;
    bool tab;
    const int rpt = res_cg_tiles(h);
    if (!res_form(h, kResCg, &tab) || rpt == 0 || iteration_budget(h) < kResMinSteps) return kOK;
    const dim3 g((unsigned)((tiles_of(h->N) + rpt - 1) / rpt));
    return run_resident(h, kResCg, [&](const ResWs& ws) {
        const auto go = [&](auto k) {
            hipLaunchKernelGGL(k, g, dim3(kResWG), 0, h->stream, m, h->N, r, p, qx, x, h->st, ws,
                               kResChunk);
        };
        if (g.x == 1) {
            if (rpt == 1) tab ? go(k_cg_res<1, true, true>) : go(k_cg_res<1, false, true>);
            else tab ? go(k_cg_res<2, true, true>) : go(k_cg_res<2, false, true>);
        } else {
            if (rpt == 1) tab ? go(k_cg_res<1, true, false>) : go(k_cg_res<1, false, false>);
            else tab ? go(k_cg_res<2, true, false>) : go(k_cg_res<2, false, false>);
        }
    }, ran);
}

int resident_bicg(gis_context* h, const Mat<double>& m, const Mat<double>& mt, double* r,
                  double* rs, double* p, double* ps, double* qx, double* x, bool* ran) {
    *ran = false;
    bool tab;
    if (!resident_bicg_fits(h) || !res_form(h, kResBicg, &tab) ||
        iteration_budget(h) < kResMinSteps)
        return kOK;
    const dim3 g((unsigned)tiles_of(h->N));
    return run_resident(h, kResBicg, [&](const ResWs& ws) {
        const auto go = [&](auto k) {
            hipLaunchKernelGGL(k, g, dim3(kResWG), 0, h->stream, m, mt, h->N, r, rs, p, ps, qx, x,
                               h->st, ws, kResChunk);
        };
        if (g.x == 1) tab ? go(k_bicg_res<true, true>) : go(k_bicg_res<false, true>);
        else tab ? go(k_bicg_res<true, false>) : go(k_bicg_res<false, false>);
    }, ran);
}

// Measured against one launch per stage for the whole batch (edges, tiles in all):
// 64 systems of 8-24, 364: 4.67 -> 1.43 ms; 8 of 16-64, 422: 9.9 -> 4.3; 64 of 20-40,
// 1980: 18.3 -> 9.2; 32 of 16-64, 2994: 35.3 -> 31.0; 64 of 16-64, 5735: 60.2 -> 57.7;
// 20 of 50-64, 3657: 44.0 -> 44.7, where both run at the chip's rate.
// A batch's systems as resident launches, each of as many systems as fit the chip
// together (largest first, so that those of one launch take about as long).
// Systems that are not done afterwards have not been started: the caller's loop
// takes them.
int resident_batch(gis_context* h, const Mat<double>& m, double* r, double* p, double* qx,
                   double* x) {
    BatchInfo& B = h->batch;
    if (!resident_batch_fits(h)) return kOK;
    const int n_cu = std::min(h->n_cu, kResMaxGrid), S = B.S;
    if (B.res_first.empty()) {   // once per pattern
        std::vector<int> sys(S);
        long long tiles = 0;
        for (int i = 0; i < S; ++i) {
            sys[i] = i;
            tiles += B.tile0[i + 1] - B.tile0[i];
        }
        B.res_tiles = tiles <= n_cu ? 1 : 2;
        const auto groups = [&](int i) {
            return (B.tile0[i + 1] - B.tile0[i] + B.res_tiles - 1) / B.res_tiles;
        };
        std::stable_sort(sys.begin(), sys.end(),
                         [&](int a, int b) { return groups(a) > groups(b); });
        std::vector<ResBlock> blocks;
        std::vector<int> first;
        int slot = 0, slots = 0;
        for (int i : sys) {
            const int G = groups(i);
            if (first.empty() || (int)blocks.size() - first.back() + G > n_cu) {
                first.push_back((int)blocks.size());
                slot = 0;
            }
            for (int g = 0; g < G; ++g)
                blocks.push_back(ResBlock{{B.pad_off[i] + g * B.res_tiles * kTile,
                                           B.pad_off[i] + B.n[i], g, G}, i, slot});
            slots = std::max(slots, ++slot);
        }
        first.push_back((int)blocks.size());
        GIS_HIP(h, B.res_blocks.ensure(sizeof(ResBlock) * blocks.size()));
        GIS_HIP(h, hipMemcpyAsync(B.res_blocks.p, blocks.data(), sizeof(ResBlock) * blocks.size(),
                                  hipMemcpyHostToDevice, h->stream));
        GIS_HIP(h, hipStreamSynchronize(h->stream));   // blocks is a host temporary
        B.res_slots = slots;
        B.res_first = first;
    }
    if (held_back(h)) return kOK;
    std::unique_lock<std::mutex> lock(g_resident[h->device], std::try_to_lock);
    if (!lock.owns_lock()) {
        ++h->res_count[kResSkipped];
        return kOK;
    }
    const int L = (int)B.res_first.size() - 1;
    const size_t n_slot = (size_t)B.res_slots * kResSets * kResSlots;
    GIS_HIP(h, h->res_mem.ensure(sizeof(double) * n_slot + sizeof(int) * 4 * (size_t)L));
    double* slot = h->res_mem.as<double>();
    int* sync = reinterpret_cast<int*>(slot + n_slot);
    std::vector<int> verdict(4 * (size_t)L);
    bool first = true;
    for (int late = 0;;) {
        const LateLaunches f = late_launches(h, L);
        hipLaunchKernelGGL(k_res_reset_all, dim3(1), dim3(kWG), 0, h->stream, sync, L, f.first,
                           f.end, B.st.as<KState>(), S, h->res_fault);
        for (int l = 0; l < L; ++l) {
            const ResWs ws{slot, sync + 4 * l, patience_ticks(h, late)};
            const dim3 g((unsigned)(B.res_first[l + 1] - B.res_first[l]));
            const auto go = [&](auto k) {
                hipLaunchKernelGGL(k, g, dim3(kResWG), 0, h->stream, m, (size_t)h->N, r, p, qx, x,
                                   B.st.as<KState>(), B.res_blocks.as<ResBlock>() + B.res_first[l],
                                   ws, kResChunk);
            };
            B.res_tiles == 1 ? go(k_bcg_res<1>) : go(k_bcg_res<2>);
        }
        GIS_HIP(h, hipGetLastError());
        GIS_HIP(h, hipMemcpyAsync(B.st_host, B.st.p, sizeof(KState) * S, hipMemcpyDeviceToHost,
                                  h->stream));
        GIS_HIP(h, hipMemcpyAsync(verdict.data(), sync, sizeof(int) * 4 * (size_t)L,
                                  hipMemcpyDeviceToHost, h->stream));
        GIS_HIP(h, hipStreamSynchronize(h->stream));
        bool any_late = false;
        for (int l = 0; l < L; ++l) {
            if (verdict[4 * l + 2] == kResNoFit) h->res_unfit[kResBatch] = true;
            count_launch(h, verdict[4 * l + 2]);
            any_late = any_late || verdict[4 * l + 2] == kResLate;
        }
        if (first) hold_back_next(h, any_late);
        first = false;
        // a system that a chunk left unfinished goes on in its resident form
        bool open = false;
        for (int i = 0; i < S; ++i) open = open || (!B.st_host[i].done && B.st_host[i].k > 0);
        if (!open) return kOK;
        if (any_late && ++late > kResRetries)
            return fail(h, kErrSync, "the batch's grid could not be made resident again");
    }
}

bool resident_batch_fits(const gis_context* h) {
    bool tab;
    if (!res_form(h, kResBatch, &tab) || h->lay_max_row > kResEntries) return false;
    const BatchInfo& B = h->batch;
    const int n_cu = std::min(h->n_cu, kResMaxGrid);
    int most = 0;
    for (int i = 0; i < B.S; ++i) most = std::max(most, B.tile0[i + 1] - B.tile0[i]);
    return most <= 2 * n_cu;
}

}  // namespace gis
