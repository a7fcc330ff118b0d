// A whole preconditioned flexible BiCGSTAB solve in one launch: the two-level
// solve of a p' system and the smoothed solves of the momentum systems, for
// systems of up to a few thousand cells per compute unit.
//
// What bounds it.  The launch-per-stage iteration of km_twolevel.hip costs the
// latency of four launches (three for the momentum systems), 45-50 us per
// iteration at 1282 x 258 cells (22 us here; 13 us at 320 x 64), however few
// bytes it moves.  Here one
// workgroup per tile stays on its compute unit for the whole solve: the five
// coefficients, r, p and v of the tile and its halo and x, r~ of the tile live
// in registers, z in LDS, and only what other workgroups need goes through
// memory: the tile's edge cells of v and t, the restriction pieces of P^T v and
// P^T t, the partial sums and, on the larger coarse levels, the coarse values.
// What is left is the exchange: two rounds per iteration (four with shared
// coarse values), each a store, a flag and a load through the memory side.
//
// The recurrences, the preconditioner and the stopping test are those of
// km_twolevel.hip; every workgroup sums the same partial sums in the same order,
// so all take the same decisions.  A workgroup holds r, p and v on its halo
// too and advances them by the same expressions as their owner.
//
// Exchange.  Values other workgroups read are stored and loaded as relaxed
// agent-scope atomics (they bypass the caches that are not coherent between
// the eight dies).  A round: every wave waits until its stores are complete
// (vmcnt 0), the workgroup meets, one thread stores the round's number into
// the workgroup's flag, then every workgroup reads all flags until they have
// it.  Round numbers only grow, over all launches of a context, so a flag is
// never cleared.  A flag has a 64-byte line of its own: 1.65 us a round for 256
// workgroups, against 4.5 us with the flags in neighbouring words and 3.9 us
// for a central counter.  The few shared coarse values carry the round's number
// in each 64-bit word instead (half a double beside a 32-bit tag): their
// readers need no round, 1.5 us instead of 3.2.  The same for the partial sums
// and the halo took longer (5-11 us a round: more words to ask for again and
// again, and registers spilled).
//
// All workgroups must be resident at once: the host admits at most one per
// compute unit and orders these launches of a process one after another
// (Gate).  A wait is bounded in time; on the limit (another process holding
// compute units, say) every workgroup leaves, and the host solves by launches.
#include "km_persist.h"
#include "km_coarse.h"

#include <algorithm>
#include <mutex>
#include <type_traits>

// Per-context exchange buffers (allocated at the first such solve).
struct km_persist {
    char* arena = nullptr;
    unsigned* flags = nullptr;   // [2 systems][kMaxWg] lines of kFlagStride words
    unsigned* abort = nullptr;   // set by a wait that ran into its limit
    uint64_t* Y = nullptr;       // [2][kMaxM][2] shared coarse values Y(p), Y(s) with their round
    double* part = nullptr;      // [2 systems][2 half-iterations][kMaxWg][4] partial sums
    double* rc = nullptr;        // [2][kMaxSlots][kMaxM] restriction pieces of P^T v, P^T t
    unsigned round = 0;          // the last round's number
    bool clean = false;          // flags and Y hold numbers up to ``round`` only
};

namespace {

constexpr int kMaxWg = 256;
constexpr int kFlagStride = 16;
constexpr int kMaxSlots = 16;
constexpr int kMaxM = 2048;
constexpr int kMaxF = 64;                // aggregates under one tile's z frame
constexpr size_t kLdsBytes = 160 * 1024;
constexpr int kEpt = 4;                  // restricted values per thread: m <= kEpt NT
constexpr int kStallWindow = 300;        // as km_twolevel.hip
constexpr long long kWaitTicks = 200000000LL;   // 2 s of the 100 MHz clock
constexpr int kUnsupported = 100;        // status words of a launch that gave up
constexpr int kAborted = 101;

// Tile shapes (interior rows x columns of a workgroup) and threads, smallest
// first: a solve takes the first shape whose tiles number at most one per
// compute unit.  Threads: as many as the register frame (tile plus halo 4) has
// pairs of cells, or half or a third of them.
constexpr int kNumShapes = 7;
constexpr int kTI[kNumShapes] = {16, 16, 32, 40, 48, 48, 64};
constexpr int kTJ[kNumShapes] = {16, 32, 32, 32, 32, 48, 56};
constexpr int kNT[kNumShapes] = {320, 512, 512, 512, 512, 512, 512};

// What of a tile's own cells lies where (vectors of size vec): v and t of the
// slots that hold own cells only in LDS beside z and the restriction's y; then,
// as long as the LDS lasts (keeping 20 KB for the restricted vector and the
// tables), r~, x, and p^ until x takes it.  What does not fit: t takes y's
// place in yb (and the free-cell mask a byte per cell), x stays in memory (the
// die's L2: 5 us per iteration at 64 x 56 cells), and without p^ x takes
// alpha p^ while z still is p^.  r~ always fits: read from memory it cost 5 us
// per half-iteration.
struct Plan {
    bool t_in_yb, x_in_lds, p_in_lds;
    size_t bytes;
};
__host__ __device__ constexpr Plan plan(int TI, int TJ, int NT, int sweeps, bool coarse, size_t vec) {
    const size_t h = 2 * (2 * sweeps + 1), QI = (TI * TJ / 2 + NT - 1) / NT, QF = TI * TJ / 2 / NT;
    const size_t own = 2 * QI * NT * vec, full = 2 * QF * NT * vec;
    const size_t room = 160 * 1024 - (coarse ? 20 : 4) * 1024;
    Plan p{};
    p.bytes = (TI + h) * (TJ + h) * vec + (coarse ? (size_t)TI * TJ * 8 : 0) + full + own;
    p.t_in_yb = coarse && vec == 8 && p.bytes + full > room;
    p.bytes += p.t_in_yb ? (size_t)TI * TJ : full;
    p.x_in_lds = p.bytes + own <= room;
    if (p.x_in_lds) p.bytes += own;
    p.p_in_lds = p.x_in_lds && p.bytes + own <= room;
    if (p.p_in_lds) p.bytes += own;
    return p;
}

template <typename T>
struct PSys {
    int NX, NY, tiles_j, G;
    const void* c;        // five coefficient planes
    const T* b;
    T* x;
    T* v;                 // edge cells of v and t for the neighbours
    T* t;
    unsigned* flags;
    unsigned* abort;
    unsigned round;       // the last round before this launch
    double* pa;           // partial sums of the two half-iterations
    double* pb;
    double eps;
    int max_iter;
    T om;
    int* hw;              // the host's words
    // coarse level
    int B, mJ, m, SJ;
    int R;                // > 0: each workgroup computes R coarse values and shares them; 0: all it needs
    int cached;           // rows of A_c^-1 kept in LDS
    const uint8_t* mask;
    const double* inv;
    double* rcv;
    double* rct;
    uint64_t* Yp;         // shared coarse values (R > 0)
    uint64_t* Ys;
};

__device__ __forceinline__ bool fin(double v) { return v == v && v - v == 0.0; }

// 1 / d refined as in km_twolevel.hip
__device__ __forceinline__ double recip(double d) {
    double x = __builtin_amdgcn_rcp(d);
    x = __builtin_fma(x, __builtin_fma(-d, x, 1.0), x);
    x = __builtin_fma(x, __builtin_fma(-d, x, 1.0), x);
    return x;
}
__device__ __forceinline__ float recip(float d) { return 1.0f / d; }

template <typename V>
__device__ __forceinline__ void put(V* p, V v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename V>
__device__ __forceinline__ V get(const V* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// base[k], base the same in all lanes: a 32-bit offset per lane
template <typename V>
__device__ __forceinline__ V get_at(const V* base, int k) {
    return get(reinterpret_cast<const V*>(reinterpret_cast<const char*>(base) + (uint32_t)k * (uint32_t)sizeof(V)));
}

template <typename V>
__device__ __forceinline__ void put_at(V* base, int k, V v) {
    put(reinterpret_cast<V*>(reinterpret_cast<char*>(base) + (uint32_t)k * (uint32_t)sizeof(V)), v);
}

// One round: false when the wait ran into its limit here or elsewhere.
template <int NT>
__device__ __forceinline__ bool meet(unsigned* flags, int L, int G, unsigned round, unsigned* abort, int* bad) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) put(flags + L * kFlagStride, round);
    if ((int)threadIdx.x < G) {
        const unsigned* f = flags + threadIdx.x * kFlagStride;
        if (get(f) < round) {
            const long long t0 = wall_clock64();
            int spin = 0;
            while (get(f) < round) {
                if ((++spin & 63) == 0 && (wall_clock64() - t0 > kWaitTicks || get(abort)) && get(f) < round) {
                    put(abort, 1u);
                    *bad = 1;
                    break;
                }
            }
        }
    }
    __syncthreads();
    return *bad == 0;
}

// Totals over the workgroups' partial sums P[G][4], in a fixed order: thread t
// holds workgroup t's values.
template <int NV, int NT>
__device__ __forceinline__ void totals(const double (&mine)[NV], int G, double (&out)[NV], double* red) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int nw = (G + 63) >> 6;
    if (w < nw) {
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            const double a = wave_sum(mine[q]);
            if (lane == 0) red[w * NV + q] = a;
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        double a = red[q];
        for (int k = 1; k < nw; ++k) a += red[k * NV + q];
        out[q] = a;
    }
}

// The workgroup's sums of NV values, published as its partial sums.
template <int NV, int NT>
__device__ __forceinline__ void publish(const double (&v)[NV], double* P, double* red) {
    constexpr int NW = NT / 64;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        const double a = wave_sum(v[q]);
        if (lane == 0) red[w * NV + q] = a;
    }
    __syncthreads();
    if (threadIdx.x < NV) {
        double a = red[threadIdx.x];
        for (int k = 1; k < NW; ++k) a += red[k * NV + threadIdx.x];
        put(P + threadIdx.x, a);
    }
}

// Part of an aggregate in a tile: first cell in yb, width, cells, the steps of
// 64 cells in rows and columns, 65536 / width rounded up, its slot's value.
struct Piece {
    int at, wdt, cnt, dr, dc, inv, dst;
};

// A row of the cached A_c^-1, by its offset in the dynamic LDS (a plain
// pointer would turn its loads into flat ones).
struct LdsRow {
    int at;
    __device__ __forceinline__ double operator[](int k) const {
        extern __shared__ double dyn[];
        return dyn[at + k];
    }
};

// v, as a value the compiler knows nothing about: what is computed from it in
// the iteration is computed there, not kept in a register over all of it (the
// predicates and addresses so kept cost 90 registers, and spills from 32 x 32
// cells on).
__device__ __forceinline__ int fresh(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// SW red-black sweeps (halo NS = 2 SW); COARSE: the two-level preconditioner.
// CT: coefficient and arithmetic type (FP64 for the two-level solve of FP32
// vectors, see k_tl_tile's C64).
template <typename T, typename CT, int TI, int TJ, int NT, int SW, bool COARSE>
__device__ __forceinline__ void solve_body(const PSys<T>& s, int L) {
#pragma clang fp contract(fast)
    constexpr int NS = 2 * SW;
    constexpr int WZ = TJ + 2 * (NS + 1), HZ = TI + 2 * (NS + 1);
    constexpr int WR = TJ + 2 * NS, HR = TI + 2 * NS;
    constexpr int NPI = TI * TJ / 2, NP = HR * WR / 2;
    constexpr int QI = (NPI + NT - 1) / NT, Q = (NP + NT - 1) / NT;
    constexpr int BAND = NS * (WR / 2);
    constexpr int QZ = (HZ * WZ + NT - 1) / NT;
    constexpr int NW = NT / 64;
    constexpr int QF = NPI / NT;     // slots that hold own cells only: their v and t lie in LDS
    constexpr Plan PL = plan(TI, TJ, NT, SW, COARSE, sizeof(T));
    static_assert(TJ % 2 == 0 && TI >= NS && TJ >= NS && NT % 64 == 0 && NT >= kMaxWg, "tile");
    extern __shared__ double dyn[];            // COARSE: m restricted values, then the cached rows of A_c^-1
    __shared__ T za[HZ * WZ];
    __shared__ double yb[COARSE ? TI * TJ : 1];
    // Y(r), Y(p), Y(v), Y(s) of the coarse rows computed here; yl: shared
    // values of the aggregates under the z frame
    __shared__ double yr[COARSE ? kMaxF : 1], yp[COARSE ? kMaxF : 1], yv[COARSE ? kMaxF : 1], ysv[COARSE ? kMaxF : 1];
    __shared__ double yl[COARSE ? kMaxF : 1];
    __shared__ Piece piece[COARSE ? kMaxF : 1];
    __shared__ double red[4 * (NW > 4 ? NW : 4)];
    __shared__ double red2[4 * 4];
    // x, r~ and p^ of the own cells: each thread reads back what it wrote
    __shared__ T xs[PL.x_in_lds ? 2 * QI * NT : 1], rts[2 * QI * NT], hps[PL.p_in_lds ? 2 * QI * NT : 1];
    __shared__ T vs[QF ? 2 * QF * NT : 1], ts[QF && !PL.t_in_yb ? 2 * QF * NT : 1];
    __shared__ uint8_t mk[PL.t_in_yb ? TI * TJ : 1];   // free own cells
    __shared__ int bad;

    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int NX = s.NX, NY = s.NY, nx = NX - 2, ny = NY - 2, G = s.G;
    const int64_t n = (int64_t)NX * NY;
    const CT* __restrict__ c = static_cast<const CT*>(s.c);
    const CT om = (CT)s.om;
    const int ta = L / s.tiles_j, tb = L - ta * s.tiles_j;
    const int ti0 = 1 + ta * TI, tj0 = 1 + tb * TJ;
    unsigned round = s.round;
    // raised before this launch (by the one before it, say): leave at the first
    // round instead of waiting too.  In flight while the frame is loaded (waited
    // for here it was 1 us per solve).
    unsigned raised = 0;
    if (t == 0) raised = get(s.abort);

    // boundary cells of the system next to this tile: x = 0, and their rows
    // must be empty (checked: otherwise the launch gives up)
    double odd = 0.0;
    {
        const int j0 = tb == 0 ? 0 : tj0, j1 = tj0 + TJ > ny ? NY : tj0 + TJ;
        const int i0 = ta == 0 ? 0 : ti0, i1 = ti0 + TI > nx ? NX : ti0 + TI;
        auto check = [&](int i, int j) {
            const int64_t k = (int64_t)i * NY + j;
            bool any = s.b[k] != T(0);
            for (int e = 0; e < 5; ++e) any = any || c[e * n + k] != CT(0);
            if (any) odd += 1.0;
            s.x[k] = T(0);
        };
        if (ta == 0)
            for (int j = j0 + t; j < j1; j += NT) check(0, j);
        if (ti0 + TI > nx)
            for (int j = j0 + t; j < j1; j += NT) check(NX - 1, j);
        if (tb == 0)
            for (int i = i0 + t; i < i1; i += NT) check(i, 0);
        if (tj0 + TJ > ny)
            for (int i = i0 + t; i < i1; i += NT) check(i, NY - 1);
    }

    // the frame: pair slots as k_tl_tile's, the tile's own block first
    CT cr[Q][2][5], wd[Q][2];
    T r[Q][2], p[Q][2], v[Q - QF][2];
    int kq[Q][2];
    auto rtv = [&](int q, int cc) { return rts[(2 * q + cc) * NT + t]; };   // r~ of an own cell
    short dq[Q][2], pz[Q][2];   // distance outside the tile (99: not in the system), z index
    uint32_t own = 0, edge = 0, fm = 0;   // bit 2 q + c: own cell; read by a neighbour; free cell
    auto yb_at = [&](int q, int cc) {        // place of a pair cell of the tile's own block in yb
        const int P = fresh(t) + q * NT, lr = P / (TJ / 2);
        return lr * TJ + pz[q][cc] - (lr + NS + 1) * WZ - (NS + 1);
    };
    const int par0 = (ti0 + tj0) & 1;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int P = t + q * NT;
        int a, b0;
        if (P < NPI) {
            a = NS + P / (TJ / 2);
            b0 = NS + 2 * (P - (P / (TJ / 2)) * (TJ / 2));
        } else {
            const int u0 = P - NPI;
            if (u0 < BAND) {
                a = u0 / (WR / 2);
                b0 = 2 * (u0 - a * (WR / 2));
            } else if (u0 < 2 * BAND) {
                const int u = u0 - BAND;
                a = NS + TI + u / (WR / 2);
                b0 = 2 * (u - (u / (WR / 2)) * (WR / 2));
            } else {
                const int u = u0 - 2 * BAND, e = u - (u / NS) * NS;
                a = NS + u / NS;
                b0 = e < NS / 2 ? 2 * e : TJ + NS + 2 * (e - NS / 2);
            }
        }
        const int par = (par0 + a) & 1;
#pragma unroll
        for (int cc = 0; cc < 2; ++cc) {
            const int b = b0 + (par ^ cc);
            const int i = ti0 - NS + a, j = tj0 - NS + b;
            const bool in = P < NP && i >= 1 && i <= nx && j >= 1 && j <= ny;
            const int k = in ? i * NY + j : 0;
            kq[q][cc] = k;
            pz[q][cc] = (short)(P < NP ? (a + 1) * WZ + b + 1 : 0);
            const int di = NS - a > a - (TI + NS - 1) ? NS - a : a - (TI + NS - 1);
            const int dj = NS - b > b - (TJ + NS - 1) ? NS - b : b - (TJ + NS - 1);
            const int d = di > dj ? di : dj;
            dq[q][cc] = (short)(in ? d : 99);
            const uint32_t bit = 1u << (2 * q + cc);
            if (q < QI && in && P < NPI) {
                own |= bit;
                if (a < 2 * NS || a >= TI || b < 2 * NS || b >= TJ) edge |= bit;
            }
#pragma unroll
            for (int e = 0; e < 5; ++e) cr[q][cc][e] = c[e * n + k];
            r[q][cc] = s.b[k];
        }
    }
    double rr = 0.0;
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int cc = 0; cc < 2; ++cc) {
            const bool in = dq[q][cc] != 99;
            if (!in) r[q][cc] = T(0);
            wd[q][cc] = cr[q][cc][0] != CT(0) ? om * recip(cr[q][cc][0]) : CT(0);
            p[q][cc] = r[q][cc];
            if (q >= QF) v[q >= QF ? q - QF : 0][cc] = T(0);
            else vs[(2 * q + cc) * NT + t] = T(0);
            if (q < QI) {
                const bool o = (own >> (2 * q + cc)) & 1u;
                const T b = o ? r[q][cc] : T(0);
                rts[(2 * q + cc) * NT + t] = b;
                if constexpr (PL.x_in_lds) xs[(2 * q + cc) * NT + t] = T(0);
                else if (o) s.x[kq[q][cc]] = T(0);
                rr += (double)b * (double)b;
                if (COARSE && o && s.mask[kq[q][cc]]) fm |= 1u << (2 * q + cc);
                if constexpr (PL.t_in_yb)
                    if (t + q * NT < NPI) mk[yb_at(q, cc)] = (fm >> (2 * q + cc)) & 1u;
            }
        }
    // z frame: which cells take a coarse value, and from which aggregate
    uint32_t zm = 0;
    short zi[COARSE ? QZ : 1];
    int I0 = 0, J0 = 0, nI = 0, nJ = 0;
    uint32_t slots[COARSE ? kEpt : 1];
    if (COARSE) {
        const int ilo = ti0 - NS - 1 < 1 ? 1 : ti0 - NS - 1, ihi = ti0 + TI + NS > nx ? nx : ti0 + TI + NS;
        const int jlo = tj0 - NS - 1 < 1 ? 1 : tj0 - NS - 1, jhi = tj0 + TJ + NS > ny ? ny : tj0 + TJ + NS;
        I0 = (ilo - 1) / s.B;
        J0 = (jlo - 1) / s.B;
        nI = (ihi - 1) / s.B - I0 + 1;
        nJ = (jhi - 1) / s.B - J0 + 1;
#pragma unroll
        for (int q = 0; q < QZ; ++q) {
            const int idx = t + q * NT;
            const int a = idx / WZ, b = idx - (idx / WZ) * WZ;
            const int i = ti0 - NS - 1 + a, j = tj0 - NS - 1 + b;
            const bool in = idx < HZ * WZ && i >= 1 && i <= nx && j >= 1 && j <= ny;
            zi[q] = in ? (short)(((i - 1) / s.B - I0) * nJ + (j - 1) / s.B - J0) : (short)0;
            if (in && s.mask[(int64_t)i * NY + j]) zm |= 1u << q;
        }
        // the slots of each restricted value this thread sums that a tile writes
#pragma unroll
        for (int e = 0; e < kEpt; ++e) {
            const int k = t + e * NT;
            uint32_t u = 0;
            if (k < s.m) {
                const int I = k / s.mJ, J = k - I * s.mJ;
                const int ie = ((I + 1) * s.B < nx ? (I + 1) * s.B : nx) - 1;
                const int je = ((J + 1) * s.B < ny ? (J + 1) * s.B : ny) - 1;
                const int ni = ie / TI - (I * s.B) / TI + 1, nj = je / TJ - (J * s.B) / TJ + 1;
                for (int a = 0; a < ni; ++a)
                    for (int b = 0; b < nj; ++b) u |= 1u << (a * s.SJ + b);
            }
            slots[e] = u;
        }
    }
    // coarse rows computed here: local row f is coarse unknown unknown(f)
    const bool shared = COARSE && s.R > 0;
    const int row0 = L * s.R;
    const int nF = !COARSE ? 0 : shared ? (row0 + s.R <= s.m ? s.R : (row0 < s.m ? s.m - row0 : 0)) : nI * nJ;
    auto unknown = [&](int f) { return shared ? row0 + f : (I0 + f / nJ) * s.mJ + J0 + f % nJ; };
    const int nc = COARSE ? (s.cached < nF ? s.cached : nF) : 0;
    if (COARSE) {
        for (int f = w; f < nc; f += NW) {
            const double* __restrict__ a = s.inv + (int64_t)unknown(f) * s.m;
            for (int k = lane; k < s.m; k += 64) dyn[(int64_t)(f + 1) * s.m + k] = a[k];
        }
    }

    // P^T of the values in yb, one wave per piece (the part of an aggregate in
    // this tile), published in the tile's slots
    const int np = !COARSE ? 0 : [&]() {
        const int r0 = ti0 - 1, c0 = tj0 - 1;
        const int r1 = r0 + TI < nx ? r0 + TI : nx, c1 = c0 + TJ < ny ? c0 + TJ : ny;
        const int B = s.B, A0 = r0 / B, C0 = c0 / B;
        const int mJt = (c1 - 1) / B - C0 + 1, cnt = ((r1 - 1) / B - A0 + 1) * mJt;
        for (int u = t; u < cnt; u += NT) {
            const int I = A0 + u / mJt, J = C0 + u % mJt;
            const int ra = I * B > r0 ? I * B : r0, rb = (I + 1) * B < r1 ? (I + 1) * B : r1;
            const int ca = J * B > c0 ? J * B : c0, cb = (J + 1) * B < c1 ? (J + 1) * B : c1;
            const int wdt = cb - ca;
            Piece q;
            q.at = (ra - r0) * TJ + (ca - c0);
            q.wdt = wdt;
            q.cnt = (rb - ra) * wdt;
            q.dr = 64 / wdt;
            q.dc = 64 % wdt;
            q.inv = 65536 / wdt + 1;
            q.dst = ((ta - (I * B) / TI) * s.SJ + (tb - (J * B) / TJ)) * s.m + I * s.mJ + J;
            piece[COARSE ? u : 0] = q;
        }
        return cnt;
    }();
    auto restrict_yb = [&](double* rcs) {
        __syncthreads();
        for (int u = w; u < np; u += NW) {
            const Piece q = piece[COARSE ? u : 0];
            const int er = (lane * q.inv) >> 16;          // lane / wdt
            int ec = lane - er * q.wdt, at = q.at + er * TJ + ec;
            double acc = 0.0;
            for (int e = lane; e < q.cnt; e += 64) {
                acc += PL.t_in_yb && !mk[PL.t_in_yb ? at : 0] ? 0.0 : yb[at];
                ec += q.dc;
                at += q.dr * TJ + q.dc;
                if (ec >= q.wdt) {
                    ec -= q.wdt;
                    at += TJ - q.wdt;
                }
            }
            acc = wave_sum(acc);
            if (lane == 0) put(rcs + q.dst, acc);
        }
    };
    // A_c^-1 times the gathered restricted values: g(f, value) by lane 0.
    // Where the rows of all aggregates under the
    // frame fit the LDS, every workgroup computes the values it needs (an
    // aggregate's value has the same bits wherever it is computed: no further
    // round of exchange; 320 x 64 cells 13.3 us per iteration against 19 with
    // two more rounds).  Where they do not, reading them from the L2 twice an
    // iteration costs more than to share them (1280 x 256: 4 us and as much again
    // waiting for the workgroups with more rows, against 3 us), so each
    // workgroup computes R rows and shares them (R > 0).
    // rows [f1, f2), row f at at(f)[k], from wave w0 = 0 on, NR rows per wave and U
    // loads of each at a time
    auto some_rows = [&](auto NRc, auto Uc, int w0, int f1, int f2, auto at, auto g) {
        constexpr int NR = decltype(NRc)::value, U = decltype(Uc)::value;
        for (int f0 = f1 + w0; f0 < f2; f0 += NR * NW) {
            decltype(at(0)) a[NR];
            double acc[NR];
#pragma unroll
            for (int u = 0; u < NR; ++u) {
                a[u] = at(f0 + u * NW < f2 ? f0 + u * NW : f0);
                acc[u] = 0.0;
            }
            int k = lane;
            for (; k + 64 * (U - 1) < s.m; k += 64 * U) {
                double av[NR][U];
#pragma unroll
                for (int u = 0; u < NR; ++u)
#pragma unroll
                    for (int e = 0; e < U; ++e) av[u][e] = a[u][k + 64 * e];
#pragma unroll
                for (int e = 0; e < U; ++e) {
                    const double d = dyn[k + 64 * e];
#pragma unroll
                    for (int u = 0; u < NR; ++u) acc[u] += av[u][e] * d;
                }
            }
            for (; k < s.m; k += 64) {
                const double d = dyn[k];
#pragma unroll
                for (int u = 0; u < NR; ++u) acc[u] += a[u][k] * d;
            }
#pragma unroll
            for (int u = 0; u < NR; ++u) {
                const double y = wave_sum(acc[u]);
                if (lane == 0 && f0 + u * NW < f2) g(f0 + u * NW, y);
            }
        }
    };
    auto rows = [&](auto g) {
        using std::integral_constant;
        const auto mem = [&](int f) -> const double* { return s.inv + (int64_t)unknown(f) * s.m; };
        const auto lds = [&](int f) { return LdsRow{(f + 1) * s.m}; };
        // rows from memory on the first waves, those from LDS on the others
        if (nc < nF) some_rows(integral_constant<int, 1>(), integral_constant<int, 16>(), w, nc, nF, mem, g);
        const int w1 = (w + NW - (nF - nc) % NW) % NW;
        if (nc <= NW) some_rows(integral_constant<int, 1>(), integral_constant<int, 8>(), w1, 0, nc, lds, g);
        else some_rows(integral_constant<int, 3>(), integral_constant<int, 4>(), w1, 0, nc, lds, g);
    };
    // the restricted vector from its pieces, added in slot order; the loads of
    // a thread's first two pieces per value are in flight together
    auto gather = [&](const double* rcs) {
        double g0[kEpt], g1[kEpt];
        const int tt = fresh(t);
#pragma unroll
        for (int e = 0; e < kEpt; ++e) {
            const uint32_t u = (uint32_t)fresh((int)slots[e]), u1 = u & (u - 1);
            const int k = tt + e * NT;
            g0[e] = u ? get_at(rcs, (__ffs(u) - 1) * s.m + k) : 0.0;
            g1[e] = u1 ? get_at(rcs, (__ffs(u1) - 1) * s.m + k) : 0.0;
        }
#pragma unroll
        for (int e = 0; e < kEpt; ++e) {
            const int k = tt + e * NT;
            const uint32_t u = (uint32_t)fresh((int)slots[e]), u1 = u & (u - 1);
            double acc = g0[e] + g1[e];
            for (uint32_t w2 = u1 & (u1 - 1); w2; w2 &= w2 - 1) acc += get_at(rcs, (__ffs(w2) - 1) * s.m + k);
            if (k < s.m) dyn[k] = acc;
        }
    };
    // the frame's coarse values from the workgroups that computed them
    auto share = [&](const double* y, uint64_t* Y, unsigned tag) {
        const uint64_t hi = (uint64_t)tag << 32;
        for (int f = t; f < nF; f += NT) {
            uint64_t* q = Y + 2 * (row0 + f);
            put(q, hi | (uint32_t)__double2loint(y[f]));
            put(q + 1, hi | (uint32_t)__double2hiint(y[f]));
        }
        if (t < nI * nJ) {
            const uint64_t* q = Y + 2 * ((I0 + t / nJ) * s.mJ + J0 + t % nJ);
            uint64_t a = get(q), b = get(q + 1);
            if ((unsigned)(a >> 32) != tag || (unsigned)(b >> 32) != tag) {
                const long long t0 = wall_clock64();
                for (int spin = 1;; ++spin) {
                    a = get(q);
                    b = get(q + 1);
                    if ((unsigned)(a >> 32) == tag && (unsigned)(b >> 32) == tag) break;
                    if ((spin & 63) == 0 && (wall_clock64() - t0 > kWaitTicks || get(s.abort))) {
                        put(s.abort, 1u);
                        bad = 1;
                        break;
                    }
                }
            }
            yl[COARSE ? t : 0] = __hiloint2double((int)(uint32_t)b, (int)(uint32_t)a);
        }
        __syncthreads();
    };
    // z = z1 from the frame's coarse values y, or 0
    auto start_z = [&](const double* y) {
        const int tt = fresh(t);
        const uint32_t zz = (uint32_t)fresh((int)zm);
#pragma unroll
        for (int q = 0; q < QZ; ++q) {
            const int idx = tt + q * NT;
            if (idx < HZ * WZ) za[idx] = COARSE && ((zz >> q) & 1u) ? (T)y[fresh(zi[COARSE ? q : 0])] : T(0);
        }
        __syncthreads();
    };
    auto sweep = [&](const T (&src)[Q][2]) {
#pragma unroll
        for (int hs = 0; hs < NS; ++hs) {
            const int h = NS - hs, cc = hs & 1;
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                if (fresh(dq[q][cc]) > h) continue;
                const int z0 = pz[q][cc];
                const CT zc = za[z0];
                CT az = cr[q][cc][0] * zc;
                az = az + cr[q][cc][1] * (CT)za[z0 - WZ];
                az = az + cr[q][cc][2] * (CT)za[z0 + WZ];
                az = az + cr[q][cc][3] * (CT)za[z0 + 1];
                az = az + cr[q][cc][4] * (CT)za[z0 - 1];
                za[z0] = (T)(zc + wd[q][cc] * ((CT)src[q][cc] - az));
            }
            __syncthreads();
        }
    };
    // y = A z of an own cell
    auto matvec = [&](int q, int cc) {
        const int z0 = pz[q][cc];
        CT y = cr[q][cc][0] * (CT)za[z0];
        y = y + cr[q][cc][1] * (CT)za[z0 - WZ];
        y = y + cr[q][cc][2] * (CT)za[z0 + WZ];
        y = y + cr[q][cc][3] * (CT)za[z0 + 1];
        y = y + cr[q][cc][4] * (CT)za[z0 - 1];
        return y;
    };
    auto into_yb = [&](int q, int cc, double y) {
        yb[yb_at(q, cc)] = PL.t_in_yb || (((uint32_t)fresh((int)fm) >> (2 * q + cc)) & 1u) ? y : 0.0;
    };

    double rho = 0.0, alpha = 0.0, omega = 1.0, r0 = 0.0, best = 1e300;
    int it = 0, best_it = 0, status = -1;
    if (t == 0) bad = (int)raised;
    __syncthreads();
    if (COARSE) {
        // Y(r) = Y(p) = A_c^-1 P^T rhs
#pragma unroll
        for (int q = 0; q < QI; ++q)
#pragma unroll
            for (int cc = 0; cc < 2; ++cc)
                if (t + q * NT < NPI) into_yb(q, cc, ((own >> (2 * q + cc)) & 1u) ? (double)rtv(q, cc) : 0.0);
        // (through the second buffer, whose next words follow another round)
        restrict_yb(s.rct);
        if (!meet<NT>(s.flags, L, G, ++round, s.abort, &bad)) status = kAborted;
        gather(s.rct);
        __syncthreads();
        rows([&](int k, double y) {
            yr[k] = y;
            yp[k] = y;
        });
        __syncthreads();
    }
    while (status < 0) {
        // ---- p^ = M(p), v = A p^; <r~,v>, <r,r>
        if (shared) share(yp, s.Yp, round + 1);
        start_z(shared ? yl : yp);
        sweep(p);
        {
            double sum[3] = {0.0, rr, it == 0 ? odd : 0.0};
#pragma unroll
            for (int q = 0; q < QI; ++q)
#pragma unroll
                for (int cc = 0; cc < 2; ++cc) {
                    const uint32_t bit = 1u << (2 * q + cc);
                    CT y = CT(0);
                    if ((uint32_t)fresh((int)own) & bit) {
                        y = matvec(q, cc);
                        if (q >= QF) v[q >= QF ? q - QF : 0][cc] = (T)y;
                        else vs[(2 * q + cc) * NT + t] = (T)y;
                        if constexpr (PL.p_in_lds) hps[(2 * q + cc) * NT + t] = za[pz[q][cc]];
                        if ((uint32_t)fresh((int)edge) & bit) put_at(s.v, kq[q][cc], (T)y);
                        sum[0] += (double)rtv(q, cc) * (double)y;
                    }
                    if (COARSE && t + q * NT < NPI) into_yb(q, cc, (double)y);
                }
            if (COARSE) restrict_yb(s.rcv);
            publish<3, NT>(sum, s.pa + 4 * L, red);
        }
        if (!meet<NT>(s.flags, L, G, ++round, s.abort, &bad)) { status = kAborted; break; }
        double tot[3];
        {
            double mine[3] = {0.0, 0.0, 0.0};
            if (t < G)
#pragma unroll
                for (int q = 0; q < 3; ++q) mine[q] = get_at(s.pa, 4 * t + q);
#pragma unroll
            for (int q = QF; q < Q; ++q)
#pragma unroll
                for (int cc = 0; cc < 2; ++cc) {
                    const int d = fresh(dq[q][cc]);
                    if (d > 0 && d <= NS) v[q - QF][cc] = get_at(s.v, kq[q][cc]);
                }
            if (COARSE) gather(s.rcv);
            totals<3, NT>(mine, G, tot, red2);   // its barrier covers dyn
        }
        // the stopping test and alpha (cv_scalars of km_twolevel.hip)
        const double rvv = tot[0];
        rr = tot[1];
        if (it == 0) {
            rho = rr;
            r0 = rr;
        }
        if (it == 0 && tot[2] != 0.0) status = kUnsupported;
        else if (!fin(rr)) status = KM_NONFINITE;
        else if (it == 0 && rr == 0.0) status = KM_OK;
        else if (it > 0 && sqrt(rr / r0) < s.eps) status = KM_OK;      // bicgsolver.py:130
        else if (it > 0 && omega == 0.0) status = KM_BREAKDOWN;
        else if (it >= s.max_iter) status = KM_MAXITER;
        else if (!fin(rho)) status = KM_NONFINITE;
        else if (rho == 0.0) status = KM_BREAKDOWN;
        else if (!fin(rvv)) status = KM_NONFINITE;
        else if (rvv == 0.0) status = KM_BREAKDOWN;
        const bool better = rr < 0.81 * best;
        if (status < 0 && !better && it - best_it >= kStallWindow) status = KM_STALL;
        if (status >= 0) break;
        if (better) {
            best = rr;
            best_it = it;
        }
        alpha = rho / rvv;                                              // bicgsolver.py:108
        if (COARSE) {
            rows([&](int k, double y) {
                yv[k] = y;                      // Y(v)
                ysv[k] = yr[k] - alpha * y;     // Y(s)
            });
        }
        {
            const T fa = (T)alpha;
#pragma unroll
            for (int q = 0; q < Q; ++q)
#pragma unroll
                for (int cc = 0; cc < 2; ++cc) {
                    const T vq = q >= QF ? v[q >= QF ? q - QF : 0][cc] : vs[(2 * q + cc) * NT + t];
                    r[q][cc] = r[q][cc] - fa * vq;                      // s (bicgsolver.py:110)
                    if constexpr (!PL.p_in_lds)
                        if (q < QI && (((uint32_t)fresh((int)own) >> (2 * q + cc)) & 1u)) {
                            const T dx = (T)(alpha * (double)za[pz[q][cc]]);
                            if constexpr (PL.x_in_lds) xs[(2 * q + cc) * NT + t] += dx;
                            else s.x[kq[q][cc]] += dx;
                        }
                }
        }
        if (COARSE || !PL.p_in_lds) __syncthreads();   // ysv, and z, which start_z writes
        // ---- s^ = M(s), t = A s^; <t,s>, <t,t>, <s,r~>, <t,r~>
        if (shared) share(ysv, s.Ys, round + 1);
        start_z(shared ? yl : ysv);
        sweep(r);
        T th[Q - QF][2];
        {
            double sum[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < QI; ++q)
#pragma unroll
                for (int cc = 0; cc < 2; ++cc) {
                    const uint32_t bit = 1u << (2 * q + cc);
                    CT y = CT(0);
                    if (q >= QF) th[q >= QF ? q - QF : 0][cc] = T(0);
                    if ((uint32_t)fresh((int)own) & bit) {
                        y = matvec(q, cc);
                        if (q >= QF) th[q >= QF ? q - QF : 0][cc] = (T)y;
                        else if constexpr (!PL.t_in_yb) ts[(2 * q + cc) * NT + t] = (T)y;
                        if ((uint32_t)fresh((int)edge) & bit) put_at(s.t, kq[q][cc], (T)y);
                        const double sk = (double)r[q][cc], rk = (double)rtv(q, cc);
                        sum[0] += (double)y * sk;
                        sum[1] += (double)y * (double)y;
                        sum[2] += sk * rk;
                        sum[3] += (double)y * rk;
                    }
                    if (COARSE && t + q * NT < NPI) into_yb(q, cc, (double)y);
                }
            if (COARSE) restrict_yb(s.rct);
            publish<4, NT>(sum, s.pb + 4 * L, red);
        }
        if (!meet<NT>(s.flags, L, G, ++round, s.abort, &bad)) { status = kAborted; break; }
        double pt[4];
        {
            double mine[4] = {0.0, 0.0, 0.0, 0.0};
            if (t < G)
#pragma unroll
                for (int q = 0; q < 4; ++q) mine[q] = get_at(s.pb, 4 * t + q);
#pragma unroll
            for (int q = QF; q < Q; ++q)
#pragma unroll
                for (int cc = 0; cc < 2; ++cc) {
                    if (q >= QI) th[q - QF][cc] = T(0);
                    const int d = fresh(dq[q][cc]);
                    if (d > 0 && d <= NS) th[q - QF][cc] = get_at(s.t, kq[q][cc]);
                }
            if (COARSE) gather(s.rct);
            totals<4, NT>(mine, G, pt, red2);
        }
        // omega, rho, beta (ct_scalars of km_twolevel.hip)
        omega = pt[1] != 0.0 ? pt[0] / pt[1] : 0.0;                          // bicgsolver.py:118
        const double rho1 = pt[2] - omega * pt[3];                           // bicgsolver.py:95
        const double beta = omega != 0.0 ? (rho1 / rho) * (alpha / omega) : 0.0;   // bicgsolver.py:102
        rho = rho1;
        if (COARSE) {
            rows([&](int k, double y) {
                const double v1 = ysv[k] - omega * y;                        // Y(r)
                yr[k] = v1;
                yp[k] = v1 + beta * (yp[k] - omega * yv[k]);                 // Y(p)
            });
        }
        const T fo = (T)omega, fb = (T)beta;
        rr = 0.0;
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
            for (int cc = 0; cc < 2; ++cc) {
                T tq;
                if (q >= QF) tq = th[q >= QF ? q - QF : 0][cc];
                else if constexpr (PL.t_in_yb) tq = (T)yb[yb_at(q, cc)];
                else tq = ts[(2 * q + cc) * NT + t];
                const T vq = q >= QF ? v[q >= QF ? q - QF : 0][cc] : vs[(2 * q + cc) * NT + t];
                const T rn = r[q][cc] - fo * tq;                             // bicgsolver.py:134
                r[q][cc] = rn;
                p[q][cc] = rn + fb * (p[q][cc] - fo * vq);                   // bicgsolver.py:103
                if (q < QI && (((uint32_t)fresh((int)own) >> (2 * q + cc)) & 1u)) {
                    // s^ is still in za
                    const int o = (2 * q + cc) * NT + t;
                    const double dx = omega * (double)za[pz[q][cc]];
                    if constexpr (PL.p_in_lds) xs[o] = xs[o] + (T)(alpha * (double)hps[o] + dx);
                    else if constexpr (PL.x_in_lds) xs[o] += (T)dx;
                    else s.x[kq[q][cc]] += (T)dx;
                    rr += (double)rn * (double)rn;
                }
            }
        ++it;
        __syncthreads();   // za is read above and written by the next start_z, yp the other way round
    }
#pragma unroll
    for (int q = 0; q < QI; ++q)
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
            if ((own >> (2 * q + cc)) & 1u) {
                if constexpr (PL.x_in_lds) s.x[kq[q][cc]] = status < kUnsupported ? xs[(2 * q + cc) * NT + t] : T(0);
                else if (status >= kUnsupported) s.x[kq[q][cc]] = T(0);
            }
    if (t == 0 && (L == 0 || status == kAborted)) {
        // the host's words (read after the stream has been waited for)
        if (L == 0) {
            __hip_atomic_store(s.hw + 1, it, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(s.hw + 2, status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(reinterpret_cast<double*>(s.hw + 4), r0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(reinterpret_cast<double*>(s.hw + 6), rr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        if (status == kAborted) __hip_atomic_store(s.hw + 3, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (L == 0) __hip_atomic_store(s.hw, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

template <typename T, typename CT, int TI, int TJ, int NT, int SW, bool COARSE>
__global__ void __launch_bounds__(NT) k_solve(PSys<T> s) {
    solve_body<T, CT, TI, TJ, NT, SW, COARSE>(s, xcd_remap(blockIdx.x, s.G));
}

// Two independent systems: workgroups [0, a.G) the first, the rest the second.
template <typename T, typename CT, int TI, int TJ, int NT, int SW>
__global__ void __launch_bounds__(NT) k_solve2(PSys<T> a, PSys<T> b) {
    const bool first = (int)blockIdx.x < a.G;
    const PSys<T>& s = first ? a : b;
    solve_body<T, CT, TI, TJ, NT, SW, false>(s, xcd_remap(first ? blockIdx.x : blockIdx.x - a.G, s.G));
}

// ------------------------------------------------------------ plain solves
//
// The reference's BiCGSTAB (bicgsolver.py:88-136) and CG (cgsolver.py:83-114) of
// a whole system in one launch, with the scalars, order of tests and
// recurrences of km_krylov.hip.  A thread holds coefficients and vectors of
// its tile's cells in registers; the stencil's input lies in LDS with a one-cell
// halo, whose cells (at most one per thread) advance like the tile's.  An
// iteration is two or three rounds (one per reduction).  A system of one tile
// needs none: 16 us per iteration by launches at 34 x 34 cells is three
// launches' latency, whatever they do.
struct PPlain {
    int NX, NY, tiles_j, G;
    const double* c;
    const double* rin;    // the first residual: b, or b - A x0
    double* x;
    int from_x;           // 1: x holds x0
    double* v;            // edge cells of v (A p), t
    double* t;
    unsigned* flags;
    unsigned* abort;
    unsigned round;
    double* part[3];      // partial sums of the rounds in turn
    double eps, ref;      // ref > 0: the stopping test's denominator
    int max_iter;
    int* hw;
};

constexpr int kNumPlain = 5;
constexpr int kPlainOne = 2;     // shapes that a whole system may fill alone
constexpr int kPTI[kNumPlain] = {16, 32, 40, 48, 64};
constexpr int kPTJ[kNumPlain] = {16, 32, 32, 48, 64};
constexpr int kPNT[kNumPlain] = {256, 512, 640, 768, 1024};

template <int TI, int TJ, int NT, bool CG>
__global__ void __launch_bounds__(NT) k_plain(PPlain s) {
    constexpr int W = TJ + 2, Q = (TI * TJ + NT - 1) / NT, NW = NT / 64;
    constexpr int RING = 2 * (TI + TJ);
    static_assert(RING <= NT && NT >= kMaxWg, "one halo cell per thread, one flag per thread");
    __shared__ double z[(TI + 2) * W];
    __shared__ double red[2][2][NW], red2[2 * 4];   // two buffers: a sum's reads may overlap the next one's writes
    __shared__ int bad;
    const int t = threadIdx.x;
    const int L = xcd_remap(blockIdx.x, s.G), G = s.G;
    const int NX = s.NX, NY = s.NY, nx = NX - 2, ny = NY - 2;
    const int64_t n = (int64_t)NX * NY;
    const int ta = L / s.tiles_j, tb = L - ta * s.tiles_j;
    const int ti0 = 1 + ta * TI, tj0 = 1 + tb * TJ;
    unsigned round = s.round, raised = 0;
    if (t == 0) raised = get(s.abort);   // as in solve_body
    for (int k = t; k < (TI + 2) * W; k += NT) z[k] = 0.0;
    // boundary rows must be empty (see solve_body)
    const int j0 = tb == 0 ? 0 : tj0, j1 = tj0 + TJ > ny ? NY : tj0 + TJ;
    const int i0 = ta == 0 ? 0 : ti0, i1 = ti0 + TI > nx ? NX : ti0 + TI;
    auto boundary = [&](auto f) {
        if (ta == 0)
            for (int j = j0 + t; j < j1; j += NT) f((int64_t)j);
        if (ti0 + TI > nx)
            for (int j = j0 + t; j < j1; j += NT) f((int64_t)(NX - 1) * NY + j);
        if (tb == 0)
            for (int i = i0 + t; i < i1; i += NT) f((int64_t)i * NY);
        if (tj0 + TJ > ny)
            for (int i = i0 + t; i < i1; i += NT) f((int64_t)i * NY + NY - 1);
    };
    double odd = 0.0;
    boundary([&](int64_t k) {
        bool any = s.rin[k] != 0.0;
        for (int e = 0; e < 5; ++e) any = any || s.c[e * n + k] != 0.0;
        if (any) odd += 1.0;
    });
    double c[Q][5], r[Q], rt[Q], p[Q], v[Q], x[Q];
    int kq[Q], lz[Q];
    uint32_t own = 0, edge = 0;
    double rr = 0.0;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int u = t + q * NT, a = u / TJ, b = u - a * TJ;
        const int i = ti0 + a, j = tj0 + b;
        const bool in = u < TI * TJ && i <= nx && j <= ny;
        kq[q] = in ? i * NY + j : 0;
        lz[q] = u < TI * TJ ? (a + 1) * W + b + 1 : 0;
        if (in) own |= 1u << q;
        if (in && (a == 0 || a == TI - 1 || b == 0 || b == TJ - 1)) edge |= 1u << q;
#pragma unroll
        for (int e = 0; e < 5; ++e) c[q][e] = in ? s.c[e * n + kq[q]] : 0.0;
        r[q] = in ? s.rin[kq[q]] : 0.0;
        x[q] = in && s.from_x ? s.x[kq[q]] : 0.0;
        rt[q] = r[q];
        p[q] = 0.0;
        v[q] = 0.0;
        rr += r[q] * r[q];
    }
    // the halo cell of this thread
    int hk = -1, hz = 0;
    if (t < RING) {
        const int a = t < TJ ? -1 : t < 2 * TJ ? TI : (t - 2 * TJ) % TI;
        const int b = t < TJ ? t : t < 2 * TJ ? t - TJ : t < 2 * TJ + TI ? -1 : TJ;
        const int i = ti0 + a, j = tj0 + b;
        if (i >= 1 && i <= nx && j >= 1 && j <= ny) hk = i * NY + j;
        hz = (a + 1) * W + b + 1;
    }
    double hr = hk >= 0 ? s.rin[hk] : 0.0, hp = 0.0, hv = 0.0;
    // everyone's totals of (a, b): false when the launch gave up
    double T0 = 0.0, T1 = 0.0;
    int buf = 0;
    auto sum = [&](double a, double b, double* P) {
        const int lane = t & 63, w = t >> 6;
        const double sa = wave_sum(a), sb = wave_sum(b);
        buf ^= 1;
        if (lane == 0) {
            red[buf][0][w] = sa;
            red[buf][1][w] = sb;
        }
        __syncthreads();
        // pairwise, all loads first
        auto waves = [&](const double* q) {
            double y[NW];
#pragma unroll
            for (int k = 0; k < NW; ++k) y[k] = q[k];
#pragma unroll
            for (int d = 1; d < NW; d *= 2)
#pragma unroll
                for (int k = 0; k + d < NW; k += 2 * d) y[k] += y[k + d];
            return y[0];
        };
        if (G == 1) {
            T0 = waves(red[buf][0]);
            T1 = waves(red[buf][1]);
            return true;
        }
        if (t < 2) put(P + 2 * L + t, waves(red[buf][t]));
        return meet<NT>(s.flags, L, G, ++round, s.abort, &bad);
    };
    // the totals after a round (G > 1), with this thread's halo value of h
    auto total = [&](const double* P, const double* h, double* out) {
        if (G == 1) return;
        double mine[2] = {0.0, 0.0};
        if (t < G) {
            mine[0] = get_at(P, 2 * t);
            mine[1] = get_at(P, 2 * t + 1);
        }
        if (h && hk >= 0) *out = get_at(h, hk);
        double y[2];
        totals<2, NT>(mine, G, y, red2);
        T0 = y[0];
        T1 = y[1];
    };
    auto apply = [&](int q) {
        const int k = lz[q];
        double y = c[q][0] * z[k];
        y += c[q][1] * z[k - W];
        y += c[q][2] * z[k + W];
        y += c[q][3] * z[k + 1];
        y += c[q][4] * z[k - 1];
        return y;
    };
    int it = 0, status = -1;
    double r0 = 0.0, rho = 0.0, rho0 = 1.0, alpha = 0.0, omega = 0.0, rTr = 0.0;
    if (t == 0) bad = (int)raised;   // before the sum's barrier
    // <r,r> (and <r,r~>, the same at the start); the count of odd boundary cells first
    bool ok = sum(odd, 0.0, s.part[1]);
    if (ok) total(s.part[1], nullptr, nullptr);
    if (!ok) status = kAborted;
    else if (T0 != 0.0) status = kUnsupported;
    if (status < 0) {
        ok = sum(rr, rr, s.part[2]);
        if (ok) total(s.part[2], nullptr, nullptr);
        else status = kAborted;
    }
    while (status < 0) {
        rTr = T0;
        rho = CG ? T0 : T1;
        if (it == 0) r0 = s.ref > 0.0 ? s.ref : rTr;
        if (!fin(rTr)) status = KM_NONFINITE;
        else if (it == 0 && rTr == 0.0) status = KM_OK;
        else if (it > 0 && (CG ? sqrt(rTr) < sqrt(r0) * s.eps : sqrt(rTr / r0) < s.eps)) status = KM_OK;   // bicgsolver.py:130, cgsolver.py:240
        else if (!CG && it > 0 && omega == 0.0) status = KM_BREAKDOWN;
        else if (it >= s.max_iter) status = KM_MAXITER;
        else if (!CG && !fin(rho)) status = KM_NONFINITE;
        else if (!CG && rho == 0.0) status = KM_BREAKDOWN;                                     // bicgsolver.py:96-98
        if (status >= 0) break;
        const double beta = it == 0 ? 0.0 : CG ? rho / rho0 : (rho / rho0) * (alpha / omega);   // :102, cgsolver.py:245
        const double om = it == 0 ? 0.0 : omega;
        rho0 = rho;
        // p = r + beta (p - omega v) (bicgsolver.py:43-46; CG: r + beta p)
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            p[q] = r[q] + beta * (CG ? p[q] : p[q] - om * v[q]);
            if ((own >> q) & 1u) z[lz[q]] = p[q];
        }
        hp = hr + beta * (CG ? hp : hp - om * hv);
        if (hk >= 0) z[hz] = hp;
        __syncthreads();
        double d0 = 0.0, d1 = 0.0;
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if ((own >> q) & 1u) {
                v[q] = apply(q);
                if (G > 1 && ((edge >> q) & 1u)) put(s.v + kq[q], v[q]);
                d0 += (CG ? p[q] : rt[q]) * v[q];
            }
        if (!sum(d0, 0.0, s.part[0])) { status = kAborted; break; }
        if (G > 1) total(s.part[0], s.v, &hv);
        if (!fin(T0)) status = KM_NONFINITE;
        else if (T0 == 0.0) status = KM_BREAKDOWN;
        if (status >= 0) break;
        alpha = rho / T0;                                     // bicgsolver.py:108, cgsolver.py:234
        if (CG) {
            rr = 0.0;
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                x[q] = x[q] + alpha * p[q];                   // cgsolver.py:206-209
                r[q] = r[q] - alpha * v[q];                   // cgsolver.py:211-214
                rr += r[q] * r[q];
            }
            if (G == 1) hv = 0.0;
            hr = hr - alpha * hv;
            d0 = d1 = rr;
        } else {
            // s = r - alpha v (bicgsolver.py:60-63)
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                r[q] = r[q] - alpha * v[q];
                if ((own >> q) & 1u) z[lz[q]] = r[q];
            }
            hr = hr - alpha * hv;
            if (hk >= 0) z[hz] = hr;
            __syncthreads();
            double th = 0.0, tq[Q];
            d0 = d1 = 0.0;
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                tq[q] = 0.0;
                if ((own >> q) & 1u) {
                    tq[q] = apply(q);
                    if (G > 1 && ((edge >> q) & 1u)) put(s.t + kq[q], tq[q]);
                    d0 += tq[q] * r[q];                       // <t,s>, <t,t> (:116-117)
                    d1 += tq[q] * tq[q];
                }
            }
            if (!sum(d0, d1, s.part[1])) { status = kAborted; break; }
            if (G > 1) total(s.part[1], s.t, &th);
            omega = T1 != 0.0 ? T0 / T1 : 0.0;                // bicgsolver.py:118
            d0 = d1 = 0.0;
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                x[q] = x[q] + (alpha * p[q] + omega * r[q]);  // bicgsolver.py:78-81
                r[q] = r[q] - omega * tq[q];                  // :83-86
                d0 += r[q] * r[q];
                d1 += r[q] * rt[q];
            }
            hr = hr - omega * th;
        }
        if (!sum(d0, d1, s.part[2])) { status = kAborted; break; }
        if (G > 1) total(s.part[2], nullptr, nullptr);
        ++it;
    }
    if (status < kUnsupported) {
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if ((own >> q) & 1u) s.x[kq[q]] = x[q];
        if (!s.from_x) boundary([&](int64_t k) { s.x[k] = 0.0; });
    }
    if (t == 0 && (L == 0 || status == kAborted)) {
        if (L == 0) {
            __hip_atomic_store(s.hw + 1, it, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(s.hw + 2, status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(reinterpret_cast<double*>(s.hw + 4), r0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(reinterpret_cast<double*>(s.hw + 6), rTr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        if (status == kAborted) __hip_atomic_store(s.hw + 3, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (L == 0) __hip_atomic_store(s.hw, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Launches of one device in one process follow each other: two of them side
// by side could each hold compute units the other waits for.  (Letting those run
// together whose workgroups fit the device at once gained 2% on 12 cases of 13k
// to 210k cells on three streams, which is within its spread.)
struct Gate {
    std::mutex m;
    hipEvent_t last = nullptr;
    hipStream_t stream = nullptr;
    bool any = false;
};
constexpr int kMaxDevices = 64;
Gate g_gate[kMaxDevices];

int admit(km_ctx* ctx, const std::function<void()>& launch) {
    Gate& g = g_gate[ctx->device];
    std::lock_guard<std::mutex> lk(g.m);
    KM_REQUIRE(ctx, g.last, "device %d has no launch gate", ctx->device);
    if (g.any && g.stream != ctx->stream) KM_HIP(ctx, hipStreamWaitEvent(ctx->stream, g.last, 0));
    launch();
    KM_CHECK_LAUNCH(ctx);
    KM_HIP(ctx, hipEventRecord(g.last, ctx->stream));
    g.any = true;
    g.stream = ctx->stream;
    return KM_OK;
}

int tiles_of(int n, int T) { return (n + T - 1) / T; }

int slots_along(int n, int B, int Tt) {
    int most = 1;
    for (int I = 0; I * B < n; ++I) {
        const int e = ((I + 1) * B < n ? (I + 1) * B : n) - 1;
        most = std::max(most, e / Tt - (I * B) / Tt + 1);
    }
    return most;
}

// At most this many aggregates of size B lie under a tile's z frame.
int frame_rows(int B, int shape) {
    const int h = 2 * (2 * kmcoarse::kSweeps + 1);
    return ((kTI[shape] + h - 2) / B + 2) * ((kTJ[shape] + h - 2) / B + 2);
}

// Bytes of solve_body's LDS arrays with a coarse level, rounded up.
size_t solve_lds(int TI, int TJ, int NT, int sweeps, size_t vec) {
    return plan(TI, TJ, NT, sweeps, true, vec).bytes + kMaxF * (5 * 8 + sizeof(Piece)) + 2048;
}

int compute_units(km_ctx* ctx) {
    static std::mutex m;
    static int cus[kMaxDevices] = {};
    if (ctx->device < 0 || ctx->device >= kMaxDevices) return 0;
    std::lock_guard<std::mutex> lk(m);
    if (!cus[ctx->device]) {
        int v = 0;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, ctx->device) != hipSuccess) v = 0;
        cus[ctx->device] = v > 0 ? v : -1;
    }
    return std::max(0, cus[ctx->device]);
}

// The words that hold round numbers: flags, the abort word, Y.
constexpr size_t kFlagBytes = (size_t)2 * kMaxWg * kFlagStride * sizeof(unsigned);
constexpr size_t kWords = kFlagBytes + 256 + (size_t)4 * kMaxM * sizeof(uint64_t);

// km_one_launch_give_up: this launch finds its abort word raised.
int raise_abort(km_ctx* ctx, unsigned* abort) {
    if (ctx->one_raise <= 0) return KM_OK;
    ctx->one_raise--;
    KM_HIP(ctx, hipMemsetAsync(abort, 1, sizeof(unsigned), ctx->stream));
    return KM_OK;
}

int ensure(km_ctx* ctx) {
    if (km_persist* K = ctx->persist) {
        if (!K->clean || K->round > 0xe0000000u) {
            KM_HIP(ctx, hipMemsetAsync(K->arena, 0, kWords, ctx->stream));
            K->round = 0;
        }
        K->clean = false;   // until the launch has ended well
        return raise_abort(ctx, K->abort);
    }
    km_persist* K = new km_persist();
    const size_t pt = (size_t)4 * kMaxWg * 4 * sizeof(double);
    const size_t rc = (size_t)2 * kMaxSlots * kMaxM * sizeof(double);
    void* q = nullptr;
    hipError_t e;
    {
        KmHostLock lk(km_host_mutex());
        e = hipSetDevice(ctx->device);
        if (e == hipSuccess) e = hipMalloc(&q, kWords + pt + rc);
    }
    if (e == hipSuccess) e = hipMemsetAsync(q, 0, kWords, ctx->stream);
    if (e != hipSuccess) {
        (void)hipGetLastError();     // not the caller's error: the solve runs by launches
        if (q) (void)hipFree(q);
        delete K;
        return KM_ENOMEM;
    }
    char* a = K->arena = static_cast<char*>(q);
    K->flags = reinterpret_cast<unsigned*>(a);
    K->abort = reinterpret_cast<unsigned*>(a + kFlagBytes);
    K->Y = reinterpret_cast<uint64_t*>(a + kFlagBytes + 256);
    K->part = reinterpret_cast<double*>(a + kWords);
    K->rc = reinterpret_cast<double*>(a + kWords + pt);
    ctx->persist = K;
    return raise_abort(ctx, K->abort);
}

template <typename T>
PSys<T> system(km_ctx* ctx, int slot, int shape, int NX, int NY, const void* c, const T* b, T* x, T* ws, double eps,
               int max_iter, double om) {
    km_persist* K = ctx->persist;
    const int64_t n = (int64_t)NX * NY;
    PSys<T> s{};
    s.NX = NX;
    s.NY = NY;
    s.tiles_j = tiles_of(NY - 2, kTJ[shape]);
    s.G = tiles_of(NX - 2, kTI[shape]) * s.tiles_j;
    s.c = c;
    s.b = b;
    s.x = x;
    s.v = ws;
    s.t = ws + n;
    s.flags = K->flags + (size_t)(slot * kMaxWg) * kFlagStride;
    s.abort = K->abort;
    s.round = K->round;
    s.pa = K->part + (size_t)(slot * 2) * kMaxWg * 4;
    s.pb = s.pa + (size_t)kMaxWg * 4;
    s.eps = eps;
    s.max_iter = max_iter;
    s.om = (T)om;
    s.hw = ctx->d_flag + KM_HW * slot;
    return s;
}

// A refused system costs its launch, the tail behind it and a wait before its
// solve by launches begins (24 to 41 us on solves of 190 to 370 us, 34 x 34 to
// 515 x 130 cells), and a program that writes identity rows on the rim of its
// systems does so every time.  So a size that was refused rests: its next kRest
// solves of that family go straight to the launches (100 x 71 cells 336 us
// with plain BiCGSTAB against 362, 236 with the coarse level against 266), then one
// is tried again (a program may have several kinds of systems of one size).
// Only the path is chosen by it: the kernel checks every system it is given.
enum Family { kPlainFamily, kTwoLevelFamily, kSmoothFamily };
constexpr int kRest = 31;

void refused(km_ctx* ctx, Family f, int NX, int NY) {
    if (ctx->one_rest.size() >= 64) ctx->one_rest.clear();
    ctx->one_rest[std::make_tuple((int)f, NX, NY)] = kRest;
}

bool rests(km_ctx* ctx, Family f, int NX, int NY) {
    const auto it = ctx->one_rest.find(std::make_tuple((int)f, NX, NY));
    if (it == ctx->one_rest.end()) return false;
    if (it->second-- > 0) return true;
    ctx->one_rest.erase(it);
    return false;
}

// Launch, the tail, and the final states; *ran = false if it gave up.
int finish(km_ctx* ctx, Family fam, int nsys, const int* NX, const int* NY, const std::function<void()>& launch, KState* out, const std::function<int()>* tail,
           bool* ran, km_persist* K, int rounds) {
    volatile int* hf = ctx->h_flag;
    for (int q = 0; q < nsys; ++q)
        for (int k = 0; k < 4; ++k) hf[KM_HW * q + k] = 0;
    std::atomic_thread_fence(std::memory_order_seq_cst);
    if (int rc = admit(ctx, launch)) return rc;
    if (tail)
        if (int rc = (*tail)()) return rc;
    KM_HIP_SYNC(ctx, hipStreamSynchronize(ctx->stream));
    std::atomic_thread_fence(std::memory_order_acquire);
    *ran = true;
    bool aborted = false;
    for (int q = 0; q < nsys; ++q) {
        volatile int* w = hf + KM_HW * q;
        KState& f = out[q];
        f = KState{};
        f.done = w[0];
        f.iter = w[1];
        f.status = w[2];
        f.r0 = *reinterpret_cast<volatile double*>(w + 4);
        f.rTr = *reinterpret_cast<volatile double*>(w + 6);
        aborted = aborted || w[3];
        if (!f.done) return km_fail(ctx, KM_EHIP, "solver stopped without reporting completion");
        if (f.status >= kUnsupported) *ran = false;
        if (f.status == kUnsupported) refused(ctx, fam, NX[q], NY[q]);
    }
    if (aborted) {
        *ran = false;
        ctx->one_count[2]++;
        return KM_OK;
    }
    ctx->one_count[*ran ? 0 : 1] += nsys;
    int most = 0;
    for (int q = 0; q < nsys; ++q) most = std::max(most, out[q].iter);
    if (K) {
        K->round += (unsigned)rounds * (unsigned)most + 8;
        K->clean = true;
    }
    return KM_OK;
}

}  // namespace

namespace kmpersist {

// Preconditioned systems with a longer side stay with the launches, so that
// their results stay what they were: the kernel itself takes any system whose
// tiles fit, and is faster there too.  The two paths add their sums in another
// order, a solve may stop an iteration earlier or later, and a step's fields
// differ by about the tolerance, at every size.  Measured over three outer steps
// at eps 1e-8: v by 1.0e-8 of its norm at 1280 x 256, 1.3e-8 at 1400 x 280, 8e-9
// at 640 x 640, 8e-10 at 1999 x 401 (at eps 1e-10 by 1.6e-10); p' by 1e-12 to 1e-10
// where it takes up to 60 iterations, by up to 1.6e-9 where it takes 134 (900 x
// 900).  That is taken below the line, where a step of a 5 : 1 channel is twice
// as fast (2.0x at 1024 x 205, 2.1x at 1280 x 256), and not above it, where the
// gain falls (1.6x at 1400 x 280, 1.5x at 1500 x 300, 1.4x at 1999 x 401: tiles of
// more than 48 x 32 cells).  The line looks at the longer side only: 1400 x 60
// (1.9x) lies outside it, 900 x 900 (1.2x) inside.  Plain solves, two to four
// times as fast at any size, have no such line.
constexpr int kMaxSide = 1300;

// Two launches that waited out their limit, of any entry: something holds the
// compute units, and each further try would cost two seconds.
bool closed(const km_ctx* ctx) { return ctx->one_count[2] >= 2; }

bool fits_twolevel(km_ctx* ctx, const km_coarse* C, int NX, int NY, int* shape) {
    if (!C || C->m > kMaxM || closed(ctx) || rests(ctx, kTwoLevelFamily, NX, NY)) return false;
    const int cus = std::min(kMaxWg, compute_units(ctx));
    const int nx = NX - 2, ny = NY - 2;
    if (nx > kMaxSide || ny > kMaxSide) return false;
    for (int k = 0; k < kNumShapes; ++k) {
        const int64_t G = (int64_t)tiles_of(nx, kTI[k]) * tiles_of(ny, kTJ[k]);
        if (G > cus) continue;
        const int B = C->B;
        if (C->m > kEpt * kNT[k]) return false;
        if (slots_along(nx, B, kTI[k]) * slots_along(ny, B, kTJ[k]) > kMaxSlots) return false;
        if (frame_rows(B, k) > kMaxF || (C->m + G - 1) / G > kMaxF) return false;
        *shape = k;
        return true;
    }
    return false;
}

// A system that fits half of the compute units with one of the first
// kHalfShapes shapes takes the smallest that does, so that u and v share a
// launch; a larger one takes the smallest that fits all of them.  The rule
// looks at one system only: a pair's results are those of two solves.
constexpr int kHalfShapes = 4;

bool smooth_shape(km_ctx* ctx, int NX, int NY, int* shape) {
    if (std::max(NX, NY) - 2 > kMaxSide + 1) return false;
    const int cus = std::min(kMaxWg, compute_units(ctx));
    for (int half = 1; half >= 0; --half)
        for (int k = 0; k < (half ? kHalfShapes : kNumShapes); ++k) {
            const int64_t G = (int64_t)tiles_of(NX - 2, kTI[k]) * tiles_of(NY - 2, kTJ[k]);
            if (G > (half ? cus / 2 : cus)) continue;
            *shape = k;
            return true;
        }
    return false;
}

bool fits_smooth(km_ctx* ctx, int NX, int NY, int* shape) {
    return !closed(ctx) && !rests(ctx, kSmoothFamily, NX, NY) && smooth_shape(ctx, NX, NY, shape);
}

#define KM_SHAPES(X) X(0) X(1) X(2) X(3) X(4) X(5) X(6)

template <typename T>
int twolevel(km_ctx* ctx, int shape, int NX, int NY, const double* coef, const T* rhs, T* xd, T* ws, double eps,
             int max_iter, KState* out, const std::function<int()>* tail, bool* ran) {
    if (int rc = ensure(ctx)) {
        *ran = false;
        return rc == KM_ENOMEM ? KM_OK : rc;
    }
    const km_coarse* C = ctx->coarse;
    km_persist* K = ctx->persist;
    PSys<T> s = system<T>(ctx, 0, shape, NX, NY, coef, rhs, xd, ws, eps, max_iter, kmcoarse::kOmega);
    s.B = C->B;
    s.mJ = C->mJ;
    s.m = C->m;
    s.SJ = slots_along(NY - 2, C->B, kTJ[shape]);
    s.mask = C->mask;
    s.inv = C->inv;
    s.rcv = K->rc;
    s.rct = K->rc + (size_t)kMaxSlots * kMaxM;
    // the restricted vector, then as many rows of A_c^-1 as fit
    const size_t row = (size_t)C->m * sizeof(double);
    const size_t fixed = solve_lds(kTI[shape], kTJ[shape], kNT[shape], kmcoarse::kSweeps, sizeof(T));
    const int room = fixed + row < kLdsBytes ? (int)((kLdsBytes - fixed) / row) - 1 : 0;
    const int under = std::min(frame_rows(C->B, shape), C->m);
    s.R = room >= under ? 0 : (C->m + s.G - 1) / s.G;
    s.cached = std::min(room, s.R > 0 ? s.R : under);
    s.Yp = K->Y;
    s.Ys = K->Y + 2 * kMaxM;
    const size_t lds = row * (1 + s.cached);
    auto launch = [&]() {
        switch (shape) {
#define KM_CASE(I)                                                                                                 \
    case I:                                                                                                        \
        hipLaunchKernelGGL((k_solve<T, double, kTI[I], kTJ[I], kNT[I], kmcoarse::kSweeps, true>), dim3(s.G),       \
                           dim3(kNT[I]), lds, ctx->stream, s);                                                     \
        break;
            KM_SHAPES(KM_CASE)
#undef KM_CASE
        }
    };
    return finish(ctx, kTwoLevelFamily, 1, &NX, &NY, launch, out, tail, ran, K, 2);
}

template <typename T>
int smooth(km_ctx* ctx, int nsys, const int* NX, const int* NY, const T* const* coef, const T* const* rhs,
           T* const* xd, T* const* ws, double eps, const int* max_iter, int sweeps, KState* out,
           const std::function<int()>* tail, bool* ran) {
    if (int rc = ensure(ctx)) {
        *ran = false;
        return rc == KM_ENOMEM ? KM_OK : rc;
    }
    PSys<T> s[2] = {};
    int shape[2] = {0, 0};
    for (int q = 0; q < nsys; ++q) {
        KM_REQUIRE(ctx, smooth_shape(ctx, NX[q], NY[q], &shape[q]), "system %d does not fit one launch", q);
        s[q] = system<T>(ctx, q, shape[q], NX[q], NY[q], coef[q], rhs[q], xd[q], ws[q], eps, max_iter[q], 1.0);
    }
    const bool together = nsys == 2 && shape[0] == shape[1] && s[0].G + s[1].G <= std::min(kMaxWg, compute_units(ctx));
    auto one = [&](int sh, const PSys<T>& a, const PSys<T>& b) {
        switch (sh * 2 + (sweeps == 2 ? 1 : 0)) {
#define KM_CASE(I)                                                                                                 \
    case 2 * I:                                                                                                    \
        hipLaunchKernelGGL((k_solve2<T, T, kTI[I], kTJ[I], kNT[I], 1>), dim3(a.G + b.G), dim3(kNT[I]), 0,          \
                           ctx->stream, a, b);                                                                     \
        break;                                                                                                     \
    case 2 * I + 1:                                                                                                \
        hipLaunchKernelGGL((k_solve2<T, T, kTI[I], kTJ[I], kNT[I], 2>), dim3(a.G + b.G), dim3(kNT[I]), 0,          \
                           ctx->stream, a, b);                                                                     \
        break;
            KM_SHAPES(KM_CASE)
#undef KM_CASE
        }
    };
    auto launch = [&]() {
        const PSys<T> none{};
        if (together) {
            one(shape[0], s[0], s[1]);
        } else {
            for (int q = 0; q < nsys; ++q) one(shape[q], s[q], none);
        }
    };
    return finish(ctx, kSmoothFamily, nsys, NX, NY, launch, out, tail, ran, ctx->persist, 2);
}

int gate(int device) {
    if (device < 0 || device >= kMaxDevices) return KM_OK;   // no path on that device (fits_*)
    Gate& g = g_gate[device];
    std::lock_guard<std::mutex> lk(g.m);
    if (!g.last && hipEventCreateWithFlags(&g.last, hipEventDisableTiming) != hipSuccess) return KM_EHIP;
    return KM_OK;
}

// One workgroup where the system fits one (no exchange: 2-3 us per iteration
// against 16 by launches), else the smallest tiles that number at most one per
// compute unit.  A tile chosen by km_set_tile asks for the launches.
bool fits_plain(km_ctx* ctx, int NX, int NY, int* shape) {
    if (closed(ctx) || NX < 3 || NY < 3 || ctx->tile_override.count(std::make_tuple(NX, NY, KM_F64)) ||
        rests(ctx, kPlainFamily, NX, NY))
        return false;
    const int cus = std::min(kMaxWg, compute_units(ctx));
    for (int one = 1; one >= 0; --one)
        for (int k = 0; k < (one ? kPlainOne : kNumPlain); ++k) {
            const int64_t G = (int64_t)tiles_of(NX - 2, kPTI[k]) * tiles_of(NY - 2, kPTJ[k]);
            if (G > (one ? 1 : cus)) continue;
            *shape = k;
            return true;
        }
    return false;
}

size_t plain_words_bytes() { return kFlagBytes + 256 + (size_t)3 * kMaxWg * 2 * sizeof(double); }

int plain(km_ctx* ctx, int shape, bool cg, int NX, int NY, const double* coef, const double* rin, double* x, bool from_x,
          double* ws, void* words, double eps, int max_iter, double ref, KState* out, const std::function<int()>* tail,
          bool* ran) {
    km_persist* K = nullptr;
    PPlain s{};
    if (words) {
        // the caller's memory: flags from zero
        char* w = static_cast<char*>(words);
        KM_HIP(ctx, hipMemsetAsync(w, 0, kFlagBytes + 256, ctx->stream));
        s.flags = reinterpret_cast<unsigned*>(w);
        s.abort = reinterpret_cast<unsigned*>(w + kFlagBytes);
        if (int rc = raise_abort(ctx, s.abort)) return rc;
        for (int k = 0; k < 3; ++k)
            s.part[k] = reinterpret_cast<double*>(w + kFlagBytes + 256) + (size_t)k * kMaxWg * 2;
    } else {
        if (int rc = ensure(ctx)) {
            *ran = false;
            return rc == KM_ENOMEM ? KM_OK : rc;
        }
        K = ctx->persist;
        s.flags = K->flags;
        s.abort = K->abort;
        s.round = K->round;
        for (int k = 0; k < 3; ++k) s.part[k] = K->part + (size_t)k * kMaxWg * 2;
    }
    s.NX = NX;
    s.NY = NY;
    s.tiles_j = tiles_of(NY - 2, kPTJ[shape]);
    s.G = tiles_of(NX - 2, kPTI[shape]) * s.tiles_j;
    s.c = coef;
    s.rin = rin;
    s.x = x;
    s.from_x = from_x ? 1 : 0;
    s.v = ws;
    s.t = ws + (size_t)NX * NY;
    s.eps = eps;
    s.ref = ref;
    s.max_iter = max_iter;
    s.hw = ctx->d_flag;
    auto launch = [&]() {
        switch (shape * 2 + (cg ? 1 : 0)) {
#define KM_CASE(I)                                                                                                 \
    case 2 * I:                                                                                                    \
        hipLaunchKernelGGL((k_plain<kPTI[I], kPTJ[I], kPNT[I], false>), dim3(s.G), dim3(kPNT[I]), 0, ctx->stream, s); \
        break;                                                                                                     \
    case 2 * I + 1:                                                                                                \
        hipLaunchKernelGGL((k_plain<kPTI[I], kPTJ[I], kPNT[I], true>), dim3(s.G), dim3(kPNT[I]), 0, ctx->stream, s); \
        break;
            KM_CASE(0) KM_CASE(1) KM_CASE(2) KM_CASE(3) KM_CASE(4)
#undef KM_CASE
        }
    };
    return finish(ctx, kPlainFamily, 1, &NX, &NY, launch, out, tail, ran, K, 3);
}

template int twolevel<double>(km_ctx*, int, int, int, const double*, const double*, double*, double*, double, int,
                              KState*, const std::function<int()>*, bool*);
template int twolevel<float>(km_ctx*, int, int, int, const double*, const float*, float*, float*, double, int, KState*,
                             const std::function<int()>*, bool*);
template int smooth<double>(km_ctx*, int, const int*, const int*, const double* const*, const double* const*,
                            double* const*, double* const*, double, const int*, int, KState*,
                            const std::function<int()>*, bool*);
template int smooth<float>(km_ctx*, int, const int*, const int*, const float* const*, const float* const*,
                           float* const*, float* const*, double, const int*, int, KState*,
                           const std::function<int()>*, bool*);

}  // namespace kmpersist

void km_persist_free(km_ctx* ctx) {
    if (!ctx->persist) return;
    KmHostLock lk(km_host_mutex());
    if (ctx->persist->arena) (void)hipFree(ctx->persist->arena);
    delete ctx->persist;
    ctx->persist = nullptr;
}

extern "C" {

int km_one_launch_counts(const km_ctx* ctx, int64_t* run, int64_t* refused, int64_t* gave_up) {
    if (!ctx) return KM_EINVAL;
    if (run) *run = ctx->one_count[0];
    if (refused) *refused = ctx->one_count[1];
    if (gave_up) *gave_up = ctx->one_count[2];
    return KM_OK;
}

int km_one_launch_give_up(km_ctx* ctx, int n) {
    if (!ctx) return KM_EINVAL;
    KM_REQUIRE(ctx, n >= 0, "%d launches", n);
    ctx->one_raise = n;
    return KM_OK;
}

}  // extern "C"
