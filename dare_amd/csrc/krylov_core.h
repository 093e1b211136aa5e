// Krylov building blocks shared by the single-system solver (krylov.hip) and the batched
// solver (batch.hip): device-resident BiCGStab(2) scalars and their update rules, the
// block part of the two-kernel deterministic reductions, the operator traversals (CSR and the
// tiled diagonal view) with their fused epilogues, and the vector-update kernels.
#pragma once

#include <cmath>
#include <cstring>

#include <type_traits>

#include "common.h"

namespace dare_hip {
namespace {

constexpr int kThreads = 256;
constexpr int kGridMax = 2048;      // work-groups of the grid-stride launches
constexpr int kTileI = 16;          // planes per tile of the diagonal-view traversals
constexpr int kXcd = 8;             // MI355X: 8 accelerator complex dies, blocks dealt round robin

// Device-resident BiCGStab2 state (BiCGStab2.inl:180-196 scalars).
struct KState {
    double alpha, beta, gamma, rho0, rho1;
    double om1, om2, mu, nu, tau;
    double alpha1;     // alpha of step 7, applied to x in the pass's last kernel
    double rnorm;      // ||r|| after the last update
    double dots[kMaxDots];
    int status;        // breakdown inside the pass (step number), 0 = none
    int next_status;   // breakdown in the prelude of the next pass (steps 3-4)
    int x_due;         // step 10 (x += alpha1 u) has been reached and waits for the pass's last kernel
};

enum TailOp : int {
    TAIL_NONE = 0,
    TAIL_STORE = 1,     // store the dots only
    TAIL_INIT = 2,      // ||r0||, prelude of pass 1 (steps 1, 3, 4)
    TAIL_GAMMA = 3,     // gamma = <v, r0>, alpha = rho0 / gamma (steps 7 / 14)
    TAIL_RHO = 4,       // rho1 = <r0, s>, beta, rho0 = rho1 (step 11)
    TAIL_GCR = 5,       // omega_1,2 (steps 19-23)
    TAIL_END = 6,       // ||r||, prelude of the next pass (steps 3-4)
    TAIL_START = 7,     // TAIL_INIT from <r,r>, <b,b> (rh = r, so <rh,r> = <r,r>); dots[1] = <b,b>
};

__device__ void apply_tail(int op, KState* st, const double* d) {
    switch (op) {
    case TAIL_STORE:
        for (int j = 0; j < kMaxDots; j++) st->dots[j] = d[j];
        break;
    case TAIL_START: st->dots[1] = d[1]; [[fallthrough]];
    case TAIL_INIT: {
        st->rnorm = sqrt(d[0]);
        st->x_due = 0;
        st->alpha = 0.;
        st->rho0 = 1.;
        st->om1 = st->om2 = 1.;
        st->status = 0;
        st->next_status = 0;
        st->rho0 = -st->om2 * st->rho0;                     // (3)
        if (st->rho0 == 0.0) {
            st->next_status = 3;
            break;
        }
        st->rho1 = op == TAIL_START ? d[0] : d[1];           // (4)
        st->beta = st->alpha * st->rho1 / st->rho0;
        st->rho0 = st->rho1;
        if (st->rho0 == 0.0) st->next_status = 4;
        break;
    }
    case TAIL_GAMMA:
        st->gamma = d[0];
        if (st->gamma == 0.0) {
            st->status = 7;
            break;
        }
        st->alpha = st->rho0 / st->gamma;
        break;
    case TAIL_RHO:
        st->alpha1 = st->alpha;
        st->x_due = 1;
        st->rho1 = d[0];
        st->beta = st->alpha * st->rho1 / st->rho0;
        st->rho0 = st->rho1;
        break;
    case TAIL_GCR: {
        // omega/mu/nu/tau are long double in the reference; FP64 here (they are cast to
        // double before use there as well, :545-568)
        double om1 = d[0], mu = d[1], nu = d[2], tau = d[3], om2 = d[4];
        st->mu = mu;
        st->nu = nu;
        if (mu == 0.) {
            st->status = 20;
            break;
        }
        tau -= nu * nu / mu;
        st->tau = tau;
        if (tau == 0.0) {
            st->status = 21;
            break;
        }
        om2 = (om2 - (nu * om1) / mu) / tau;
        om1 = (om1 - nu * om2) / mu;
        st->om1 = om1;
        st->om2 = om2;
        break;
    }
    case TAIL_END: {
        st->rnorm = sqrt(d[0]);
        st->x_due = 0;
        st->next_status = 0;
        st->rho0 = -st->om2 * st->rho0;
        if (st->rho0 == 0.0) {
            st->next_status = 3;
            break;
        }
        st->rho1 = d[1];
        st->beta = st->alpha * st->rho1 / st->rho0;
        st->rho0 = st->rho1;
        if (st->rho0 == 0.0) st->next_status = 4;
        break;
    }
    default: break;
    }
}

// Block-level part of a grid reduction: each work-group writes its NDOT partial sums with
// plain stores. No fence or arrival counter here: on MI355X the eight XCD L2 caches are not
// coherent, and an agent-scope release fence in every work-group writes the L2 back each time.
// The kernel boundary publishes the partials; k_finish (one work-group) sums them in block
// order — deterministic — and applies the BiCGStab2 scalar update on the device.
// block_partials_at writes dot j of this work-group to partial[j * stride + slot]; a work-group
// that calls it more than once (persistent loops) separates the calls with a barrier.
template <int NDOT>
__device__ inline void block_partials_at(double (&acc)[NDOT], double* partial, long long stride, long long slot) {
    __shared__ double red[NDOT][kThreads / 64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int j = 0; j < NDOT; j++) {
        const double v = wave_sum(acc[j]);
        if (lane == 0) red[j][wid] = v;
    }
    __syncthreads();
    if (threadIdx.x < NDOT) {     // dot-major: the finish kernel reads each dot's partials contiguously
        double s = 0.;
        for (int w = 0; w < kThreads / 64; w++) s += red[threadIdx.x][w];
        partial[threadIdx.x * stride + slot] = s;
    }
}

template <int NDOT>
__device__ inline void block_partials(double (&acc)[NDOT], ReduceWs ws) {
    block_partials_at<NDOT>(acc, ws.partial, kReduceBlocks, blockIdx.x);
}

// The scalars as the host reads them: pinned memory the finish kernel writes itself (seq last,
// released to the system), so that a readback is neither a copy on the stream nor a stream
// synchronisation. The host waits for its sequence number (wait_state).
struct HostState {
    KState k;
    unsigned long long seq;
};
static_assert(sizeof(HostState) <= 64 * sizeof(double), "pinned readback block too small");

__device__ inline void publish_state(HostState* host, const KState& k, unsigned long long seq) {
    host->k = k;
    __threadfence_system();
    __hip_atomic_store(&host->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

constexpr int kFinishThreads = 1024;

// sin / sout: the state before and after the tail (the same where no other kernel reads sin);
// host != NULL: the new state is published to the host under seq
template <int NDOT>
__global__ __launch_bounds__(kFinishThreads) void k_finish(ReduceWs ws, unsigned nblocks, const KState* sin, KState* sout,
                                                           int tail, int check_status, HostState* host,
                                                           unsigned long long seq) {
    if (check_status && sin->status) {            // the pass has broken down: keep its state
        if (threadIdx.x == 0) {
            if (sout != sin) *sout = *sin;
            if (host) publish_state(host, *sin, seq);
        }
        return;
    }
    __shared__ double red[kMaxDots][kFinishThreads / 64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    double tot[NDOT];
#pragma unroll
    for (int j = 0; j < NDOT; j++) {
        // fixed order: thread t owns blocks t, t + 1024, ...; loads issued before the adds
        const double* p = ws.partial + j * kReduceBlocks;
        double v[kReduceBlocks / kFinishThreads];
#pragma unroll
        for (int q = 0; q < kReduceBlocks / kFinishThreads; q++) {
            const unsigned b = threadIdx.x + q * kFinishThreads;
            v[q] = b < nblocks ? p[b] : 0.;
        }
        double s = 0.;
#pragma unroll
        for (int q = 0; q < kReduceBlocks / kFinishThreads; q++) s += v[q];
        s = wave_sum(s);
        if (lane == 0) red[j][wid] = s;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NDOT; j++) {
        double t = 0.;
        for (int w = 0; w < kFinishThreads / 64; w++) t += red[j][w];
        tot[j] = t;
    }
    if (threadIdx.x == 0) {
        double d[kMaxDots];
        for (int j = 0; j < kMaxDots; j++) d[j] = j < NDOT ? tot[j] : 0.;
        if (sout != sin) *sout = *sin;
        apply_tail(tail, sout, d);
        if (host) publish_state(host, *sout, seq);
    }
}

// grid_reduce keeps the call sites of the kernels: the block part only.
template <int NDOT>
__device__ inline void grid_reduce(double (&acc)[NDOT], ReduceWs ws, KState*, int) {
    block_partials<NDOT>(acc, ws);
}

// Where a finish kernel publishes the state, if at all.
struct Publish {
    HostState* host = nullptr;
    unsigned long long seq = 0;
};

template <int NDOT>
inline void launch_finish(hipStream_t sm, ReduceWs ws, unsigned nblocks, KState* st, int tail, int check,
                          Publish pub = {}, const KState* sin = nullptr) {
    hipLaunchKernelGGL((k_finish<NDOT>), dim3(1), dim3(kFinishThreads), 0, sm, ws, nblocks, sin ? sin : st, st, tail,
                       check, pub.host, pub.seq);
}

// ------------------------------------------------------------------------------ operators
template <typename VT>
struct CsrOp {
    const int* rp;
    const int* col;
    const VT* val;
    long long n;
};

template <typename VT>
struct DiaOp {
    DiaView V;
    const VT* D;
    int tiles_k, tiles_j, tiles_i;
    int lk_log2;        // lanes along k of a tile (16, 32 or 64); the other 256 / lanes go along j
    int tile_i;         // planes per tile
    int per_xcd;        // tiles owned by each XCD (grid = kXcd * per_xcd)
    int pair;           // cells per lane along k (2, or 4 for FP32: one component, n2 a multiple)
    bool sym = false;            // the view is exactly symmetric: the four-slot pair / quad traversals
    bool unit_c = false;         // every C coefficient is 1 and not stored (FP32 quads, column-scaled view)
};

// Lanes along k of a tile (2^lk, the other kThreads / 2^lk along j) for nk lanes' worth of k
// extent. Small systems take the split with the fewest idle lanes (the widest on a tie): at n2 = 64
// the paired traversal fills 32 lanes, and 64 x 4 tiles left half of every wave idle. Large ones
// are bound by memory, not by lanes, and a row of a narrow tile is a short piece of every array, so
// a narrower split must save a fifth of the tiles, and 16 lanes are for k extents of 16 only (seven
// slots, FP64, us a sweep with 64, 32 and 16 lanes: pairs, 2 M rows, n2 = 66: 34, 40, 38; n2 =
// 150, a quarter fewer tiles of 32: 33, 30, 33; one row, 6 M rows, n2 = 161: 110, 117, 164). The
// line lies at 1.6 M rows, of one row a lane at 2.6 M (0.9 M rows, n2 = 97, two tiles against 1.75:
// a four-pass solve 0.83 and 0.74 ms; 2 M, n2 = 33: 1.24 and 1.10).
struct LaneSplit {
    int lk_log2, tiles_k, tiles_j;
    long long tiles() const { return static_cast<long long>(tiles_k) * tiles_j; }
};
inline LaneSplit lane_split(int nk, int nj, bool large) {
    const auto split = [&](int lk) {
        return LaneSplit{lk, (nk + (1 << lk) - 1) >> lk, (nj + (kThreads >> lk) - 1) / (kThreads >> lk)};
    };
    LaneSplit best = split(6);
    for (int lk = 5; lk >= 4; lk--) {
        const LaneSplit L = split(lk);
        const bool fewer = lk == 5 && large ? 5 * L.tiles() <= 4 * best.tiles() : L.tiles() < best.tiles();
        if (fewer && (lk == 5 || !large || nk <= 16)) best = L;
    }
    return best;
}
inline LaneSplit lane_split(const DiaView& V, int pair) {
    return lane_split((V.n[2] + pair - 1) / pair, V.n[1], V.nrows >= (pair == 1 ? 5LL << 19 : 3LL << 19));
}

// Tile of a work-group: lane_split's lanes, pair cells each, marched over tile_i planes. 16 planes
// read x about once; shorter marches make more work-groups of the launch. A march is a chain of
// dependent loads, so small systems need them spread out: 512 work-groups below a million rows
// (64^3: 15.2 us per sweep as 64 of 16 planes, 4.9 as 256, 4.5 as 512), of one row a lane 1024 up
// to 2.6 M (206 x 207 x 33: 18.4 us as 507, 15.4 as 1014). Above, a work-group for each of the
// kFullGrid CUs, and of the marches of 16, 8, 4 and 2 planes that give that, the one with the fewest
// planes on the busiest CU, a march counting 0.7 of a plane for its start (seven slots, FP64: 128^3,
// 256 work-groups of 16 planes 27.7 us, 512 of 8 28.8; 112^3, 196 of 16 17.5, 392 of 8 16.3; 134 x
// 135 x 66, 306 of 16 21.9, 1156 of 4 19.8; four slots, one row a lane: 145 x 128 x 121, 640 of 16
// 32.8, 1216 of 8 29.3).
// tile_i grows past 16 only where the reduction slots would not hold the grid.
constexpr int kFullGrid = 256;
template <typename VT>
DiaOp<VT> make_dia(const DiaView& V, const VT* D, bool allow_pair = false) {
    DiaOp<VT> A;
    A.V = V;
    A.D = D;
    A.pair = (allow_pair && V.N == 1 && V.n[2] % 2 == 0) ? 2 : 1;
    if (allow_pair && std::is_same_v<VT, float> && V.N == 1 && V.n[2] % 4 == 0) A.pair = 4;
    const LaneSplit L = lane_split(V, A.pair);
    A.lk_log2 = L.lk_log2;
    A.tiles_k = L.tiles_k;
    A.tiles_j = L.tiles_j;
    auto tiles = [&](int ti) { return L.tiles() * ((V.n[0] + ti - 1) / ti); };
    A.tile_i = kTileI;
    if (V.nrows < (A.pair == 1 ? 5LL << 19 : 1LL << 20)) {
        const int want = kFullGrid * (V.nrows < (1LL << 20) ? 2 : 4);
        while (A.tile_i > 1 && tiles(A.tile_i) < want) A.tile_i /= 2;
    } else {
        const auto cost = [&](int ti) { return (tiles(ti) + kFullGrid - 1) / kFullGrid * (10 * ti + 7); };
        while (A.tile_i > 2 && tiles(A.tile_i) < kFullGrid) A.tile_i /= 2;
        for (int ti = A.tile_i / 2; ti >= 2; ti /= 2)
            if (cost(ti) < cost(A.tile_i)) A.tile_i = ti;
    }
    while (kXcd * ((tiles(A.tile_i) + kXcd - 1) / kXcd) > kReduceBlocks && A.tile_i < V.n[0]) A.tile_i *= 2;
    A.tiles_i = (V.n[0] + A.tile_i - 1) / A.tile_i;
    A.per_xcd = static_cast<int>((tiles(A.tile_i) + kXcd - 1) / kXcd);
    return A;
}

// ------------------------------------------------------------------------------ epilogues
// load(i) fetches the row's vector operands (issued together with the matrix loads);
// operator() gets y = (A x)_i, xc = x_i and the loaded operands, stores results and adds to
// the per-thread dot accumulators.
template <typename XT, bool NT = false>
struct EpiDot {         // out = A p; <out, w>                   (6)-(7), (9)+(11), (13)-(14)
    static constexpr int NDOT = 1;
    static constexpr bool kNT = NT;
    XT* out;
    const XT* w;
    __device__ double load(long long i) const { return static_cast<double>(w[i]); }
    __device__ void operator()(long long i, double y, double, double wi, double* acc) const {
        const XT yi = static_cast<XT>(y);
        put<NT>(out + i, yi);
        acc[0] += static_cast<double>(yi) * wi;
    }
};

// Epilogues that need a scalar of the device state read it once per work-item, in begin().
template <class Epi>
__device__ inline auto epi_begin(Epi& e, int) -> decltype(e.begin()) { return e.begin(); }
template <class Epi>
__device__ inline void epi_begin(Epi&, long) {}
// the same where the state is not the epilogue's own (the batched solver's, one per system)
template <class Epi>
__device__ inline auto epi_begin(Epi& e, const KState& k, int) -> decltype(e.begin(k)) { return e.begin(k); }
template <class Epi>
__device__ inline void epi_begin(Epi&, const KState&, long) {}

// r = b - A x into rh alone; <r,r>, <b,b>. The shadow residual never changes, so the first pass
// reads it as r and as u (u = r - beta u with u = 0) and writes both vectors itself: nothing
// else needs a value here, and ||b|| costs no sweep of its own.
template <typename XT, bool NT = false>
struct EpiStart {
    static constexpr int NDOT = 2;
    static constexpr bool kNT = NT;
    const XT* b;
    XT* rh;
    __device__ double load(long long i) const { return static_cast<double>(b[i]); }
    __device__ void operator()(long long i, double y, double, double bi, double* acc) const {
        const XT ri = static_cast<XT>(bi - y);
        put<NT>(rh + i, ri);
        const double rd = static_cast<double>(ri);
        acc[0] += rd * rd;
        acc[1] += bi * bi;
    }
};

// (16) and (18)-(20) in one: t = A s with r = r - alpha v formed here for the dots and again in
// k_pass_end, never stored in between
template <typename XT, bool NT = false>
struct EpiGcrL {
    static constexpr int NDOT = 5;
    static constexpr bool kNT = NT;
    XT* t;
    const XT* r;
    const XT* v;
    const KState* st;
    double alpha = 0.;
    __device__ void begin() { begin(*st); }
    __device__ void begin(const KState& k) { alpha = k.alpha; }
    __device__ double load(long long i) const {
        return static_cast<double>(static_cast<XT>(static_cast<double>(r[i]) - alpha * static_cast<double>(v[i])));
    }
    __device__ void operator()(long long i, double y, double sc, double rd, double* acc) const {
        const XT ti = static_cast<XT>(y);
        put<NT>(t + i, ti);
        const double td = static_cast<double>(ti);
        acc[0] += rd * sc;
        acc[1] += sc * sc;
        acc[2] += sc * td;
        acc[3] += td * td;
        acc[4] += rd * td;
    }
};

// the same step when a right preconditioner sits between s and the operator: t = A (M^-1 s),
// with s read from its own vector (the operand of the traversal is M^-1 s)
template <typename XT, bool NT = false>
struct EpiGcrP : EpiGcrL<XT, NT> {
    const XT* s;
    __device__ EpiGcrP() = default;
    __host__ __device__ EpiGcrP(XT* t_, const XT* r_, const XT* v_, const KState* st_, const XT* s_)
        : EpiGcrL<XT, NT>{t_, r_, v_, st_}, s(s_) {}
    __device__ void operator()(long long i, double y, double, double rd, double* acc) const {
        EpiGcrL<XT, NT>::operator()(i, y, static_cast<double>(s[i]), rd, acc);
    }
};

template <bool NT = false>
struct EpiResid {       // refinement: r = b - A x in FP64, r32 = float(r), <r,r>
    static constexpr int NDOT = 1;
    static constexpr bool kNT = NT;
    const double* b;
    float* r32;
    __device__ double load(long long i) const { return b[i]; }
    __device__ void operator()(long long i, double y, double, double bi, double* acc) const {
        const double ri = bi - y;
        put<NT>(r32 + i, static_cast<float>(ri));
        acc[0] += ri * ri;
    }
};

template <bool NT = false>
struct EpiResidB {      // the first refinement residual: as EpiResid, and <b,b> from the same read of b
    static constexpr int NDOT = 2;
    static constexpr bool kNT = NT;
    const double* b;
    float* r32;
    __device__ double load(long long i) const { return b[i]; }
    __device__ void operator()(long long i, double y, double, double bi, double* acc) const {
        const double ri = bi - y;
        put<NT>(r32 + i, static_cast<float>(ri));
        acc[0] += ri * ri;
        acc[1] += bi * bi;
    }
};

template <bool NT = false>
struct EpiResid64 {     // r = b - A x in FP64, <r,r>
    static constexpr int NDOT = 1;
    static constexpr bool kNT = NT;
    const double* b;
    double* r;
    __device__ double load(long long i) const { return b[i]; }
    __device__ void operator()(long long i, double y, double, double bi, double* acc) const {
        const double ri = bi - y;
        put<NT>(r + i, ri);
        acc[0] += ri * ri;
    }
};

template <typename XT, bool NT = false>
struct EpiStore {
    static constexpr int NDOT = 1;
    static constexpr bool kNT = NT;
    XT* out;
    __device__ double load(long long) const { return 0.; }
    __device__ void operator()(long long i, double y, double, double, double*) const {
        put<NT>(out + i, static_cast<XT>(y));
    }
};

// The epilogue of a lane's two adjacent rows i, i+1 (paired traversal): two calls, whose single
// stores land next to each other and merge into one wide store.
template <class Epi>
__device__ __forceinline__ void epi_pair(const Epi& e, long long i, double y0, double y1, double x0, double x1,
                                         double p0, double p1, double* acc) {
    e(i, y0, x0, p0, acc);
    e(i + 1, y1, x1, p1, acc);
}
// The epilogue of four adjacent rows (the FP32 quad traversal): four calls.
template <class Epi>
__device__ __forceinline__ void epi_quad(const Epi& e, long long i, const double* y, const double* xc,
                                         const double* pre, double* acc) {
#pragma unroll
    for (int m = 0; m < 4; m++) e(i + m, y[m], xc[m], pre[m], acc);
}
// ------------------------------------------------------------------------------ operands
// Element offsets within one system's slot or vector, 32 or 64 bits. 32 (also in bytes, so up to
// kWideRows rows): a load takes a scalar base and one register of offset instead of a 64-bit
// address per access, which leaves room for another wave per SIMD. The traversal of one row a lane
// takes them wherever it does not stream (odd extents, 0.7-1.3 M rows, FP64, five-slot start to end
// 2-3 % faster), and so do the fused steps, whose operand reads two vectors (128^3, seven slots:
// 37.9 -> 31.1 us; pairs in FP32 115 x 116 x 150: a four-pass solve 1.3 of 1.6 ms). The other
// sweeps of pairs and quads keep 64 bits: their waves already fill the memory's queues, and one more
// per SIMD evicts the lines that the next plane or the partner row is about to read again (FP64
// pairs, 115 x 116 x 150: four slots 28.4 us with 32 bits, 19.2 with 64, seven 32.8 and 26.7; 256^3
// 192 and 179; level at 128^3). So do the five-dot sweep of step 18, which reads two vectors more
// (128^3: 33.5 us, with 32 bits 40.2), everything from kStreamRows rows on, and a batch with a
// system of more rows than kWideRows (Wide).
constexpr long long kWideRows = 1LL << 29;
template <class Epi>
struct Wide : Epi {};
template <class Epi>
struct SweepIndexOf {
    using type = std::conditional_t<Epi::kNT || Epi::NDOT == 5, long long, unsigned>;
};
template <class Epi>
struct SweepIndexOf<Wide<Epi>> {
    using type = long long;
};
template <class Epi>
using SweepIndex = typename SweepIndexOf<Epi>::type;
// of the pairs and quads: 32 bits in the epilogues of the fused steps (kStep) alone
template <class Epi, class = void>
struct PairIndexOf {
    using type = long long;
};
template <class Epi>
struct PairIndexOf<Epi, std::enable_if_t<Epi::kStep>> {
    using type = SweepIndex<Epi>;
};
template <class Epi>
using PairIndex = typename PairIndexOf<Epi>::type;
template <typename T>
__device__ __forceinline__ const T* at_off(const T* base, unsigned e) {
    return reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + e * static_cast<unsigned>(sizeof(T)));
}
template <typename T>
__device__ __forceinline__ const T* at_off(const T* base, long long e) { return base + e; }
template <typename T>
__device__ __forceinline__ const T* at_off(const T* base, int e) { return base + e; }      // CSR columns

// What a traversal multiplies: a vector, or the combination a - c b formed where it is read
// (rounded to the vector type, as the vector it stands for would hold it). 1, 2 or 4 entries.
typedef float f32x4 __attribute__((ext_vector_type(4)));
template <typename XT>
struct Comb {
    const XT* a;
    const XT* b;
    double c;
    __device__ XT of(XT av, XT bv) const {
        return static_cast<XT>(static_cast<double>(av) - c * static_cast<double>(bv));
    }
};
template <typename XT, typename Ix>
__device__ __forceinline__ XT src1(const XT* x, Ix i) { return *at_off(x, i); }
template <typename XT, typename Ix>
__device__ __forceinline__ XT src1(const Comb<XT>& x, Ix i) { return x.of(*at_off(x.a, i), *at_off(x.b, i)); }
template <typename XT, typename Ix>
__device__ __forceinline__ void src2(const XT* x, Ix i, double* o) {      // i even, x 2-element aligned
    typedef XT x2 __attribute__((ext_vector_type(2)));
    const x2 v = *reinterpret_cast<const x2*>(at_off(x, i));
    o[0] = static_cast<double>(v.x);
    o[1] = static_cast<double>(v.y);
}
template <typename XT, typename Ix>
__device__ __forceinline__ void src2(const Comb<XT>& x, Ix i, double* o) {
    typedef XT x2 __attribute__((ext_vector_type(2)));
    const x2 a = *reinterpret_cast<const x2*>(at_off(x.a, i)),
             b = *reinterpret_cast<const x2*>(at_off(x.b, i));
    o[0] = static_cast<double>(x.of(a.x, b.x));
    o[1] = static_cast<double>(x.of(a.y, b.y));
}
template <typename Ix>
__device__ __forceinline__ f32x4 src4(const float* x, Ix i) { return *reinterpret_cast<const f32x4*>(at_off(x, i)); }
template <typename Ix>
__device__ __forceinline__ f32x4 src4(const Comb<float>& x, Ix i) {
    const f32x4 a = src4(x.a, i), b = src4(x.b, i);
    return f32x4{x.of(a.x, b.x), x.of(a.y, b.y), x.of(a.z, b.z), x.of(a.w, b.w)};
}

// ------------------------------------------------------------------------------ traversals
// Generic CSR, one wave per 64 consecutive rows. The wave walks its rows' run of the CSR
// arrays -- one contiguous range -- with coalesced loads (lane l takes entries l, l + 64, ...),
// forms each product val * x[col] (rounded to double, as the row loop rounds it) and stages it
// in its own slice of LDS; then lane l sums row r0 + l from LDS in column order, starting from
// +0.0: the sequential row sum of the reference's row loop, so y is bit-identical to it. A wave
// whose rows hold more than kCsrWaveNnz entries sums them from global memory instead. Wave
// tiles are dealt so that each XCD (blocks b = x mod 8) owns one contiguous eighth of the rows.
// Only the wave that wrote a slice reads it, so the phases need no work-group barrier.
constexpr int kCsrWaveRows = 64;
constexpr int kCsrWaveNnz = 8 * 64;   // eight entries per lane
constexpr int kCsrWaves = kThreads / kCsrWaveRows;

__device__ inline void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// row bounds of wave tile t: the run [B, E) of the CSR arrays and this lane's row [b, e)
struct CsrTileRp {
    int B, E, b, e;
};
template <typename VT>
__device__ inline CsrTileRp csr_tile_rp(const CsrOp<VT>& A, long long t, int lane) {
    const long long r0 = t * kCsrWaveRows;
    const long long r1 = (r0 + kCsrWaveRows < A.n) ? r0 + kCsrWaveRows : A.n;
    const long long i = r0 + lane;
    CsrTileRp R;
    R.B = A.rp[r0];
    R.E = A.rp[r1];
    R.b = i < r1 ? A.rp[i] : R.E;
    R.e = i < r1 ? A.rp[i + 1] : R.E;
    return R;
}

// columns and values of a staged wave tile: eight entries per lane, entries past the tile's run
// repeating its last one; streamed with non-temporal loads so that x keeps the caches
template <typename VT>
__device__ inline void csr_tile_cv(const CsrOp<VT>& A, const CsrTileRp& R, int lane, int* c, double* v) {
    const int nnz = R.E - R.B;
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const int k = u * kCsrWaveRows + lane;
        const int kk = R.B + (k < nnz ? k : nnz - 1);
        c[u] = __builtin_nontemporal_load(A.col + kk);
        v[u] = static_cast<double>(__builtin_nontemporal_load(A.val + kk));
    }
}

template <typename VT, class Src, class Epi>
__device__ inline void csr_sweep(const CsrOp<VT>& A, const Src x, const Epi& epi, double* acc) {
    __shared__ double s_prod[kCsrWaves][kCsrWaveNnz];
    {
        const int lane = threadIdx.x % kCsrWaveRows, wv = threadIdx.x / kCsrWaveRows;
        double* prod = s_prod[wv];
        const long long ntiles = (A.n + kCsrWaveRows - 1) / kCsrWaveRows;
        const int xcd = static_cast<int>(blockIdx.x % kXcd);
        const long long t0 = ntiles * xcd / kXcd, t1 = ntiles * (xcd + 1) / kXcd;
        const long long stride = static_cast<long long>(gridDim.x / kXcd) * kCsrWaves;
        long long tile = t0 + static_cast<long long>(blockIdx.x / kXcd) * kCsrWaves + wv;
        // software pipeline: the next tile's columns and values, and the row bounds of the one
        // after it, are loaded while this tile's x entries are gathered and summed
        CsrTileRp R0{}, R1{};
        int c[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        double v[8] = {0., 0., 0., 0., 0., 0., 0., 0.};
        if (tile < t1) {
            R0 = csr_tile_rp(A, tile, lane);
            if (R0.E - R0.B > 0 && R0.E - R0.B <= kCsrWaveNnz) csr_tile_cv(A, R0, lane, c, v);
        }
        if (tile + stride < t1) R1 = csr_tile_rp(A, tile + stride, lane);
        for (; tile < t1; tile += stride) {
            const long long i = tile * kCsrWaveRows + lane;
            const bool own = i < A.n;
            const long long ic = own ? i : A.n - 1;      // a valid address for every lane
            const double xi = static_cast<double>(src1(x, ic));
            const double pre = epi.load(ic);
            const int nnz = R0.E - R0.B, b = R0.b - R0.B, e = R0.e - R0.B;
            const bool staged = nnz <= kCsrWaveNnz;
            int cn[8] = {0, 0, 0, 0, 0, 0, 0, 0};
            double vn[8] = {0., 0., 0., 0., 0., 0., 0., 0.};
            CsrTileRp R2{};
            if (tile + stride < t1 && R1.E - R1.B > 0 && R1.E - R1.B <= kCsrWaveNnz) csr_tile_cv(A, R1, lane, cn, vn);
            if (tile + 2 * stride < t1) R2 = csr_tile_rp(A, tile + 2 * stride, lane);
            double s = 0.;
            if (staged) {
                // every slot of the slice is written (entries past nnz repeat the last one and
                // are never read), so no lane branches
                if (nnz > 0) {
                    double xv[8];
#pragma unroll
                    for (int u = 0; u < 8; u++) xv[u] = static_cast<double>(src1(x, c[u]));
#pragma unroll
                    for (int u = 0; u < 8; u++) prod[u * kCsrWaveRows + lane] = v[u] * xv[u];
                }
                wave_lds_sync();
                for (int k = b; k < e; k += 8) {
                    double pv[8];
#pragma unroll
                    for (int u = 0; u < 8; u++) pv[u] = prod[(k + u < e) ? k + u : b];
#pragma unroll
                    for (int u = 0; u < 8; u++)
                        if (k + u < e) s += pv[u];
                }
                wave_lds_sync();   // the slice is rewritten by the wave's next tile
            } else {
                for (int k = R0.B + b; k < R0.B + e; k++)
                    s += static_cast<double>(A.val[k]) * static_cast<double>(src1(x, A.col[k]));
            }
            if (own) epi(i, s, xi, pre, acc);
            R0 = R1;
            R1 = R2;
#pragma unroll
            for (int u = 0; u < 8; u++) {
                c[u] = cn[u];
                v[u] = vn[u];
            }
        }
    }
}

template <typename VT, typename XT, class Epi>
__global__ __launch_bounds__(kThreads) void k_apply_csr(CsrOp<VT> A, const XT* __restrict__ x, Epi epi, ReduceWs ws,
                                                       KState* st, int tail, int check_status) {
    double acc[Epi::NDOT];
#pragma unroll
    for (int j = 0; j < Epi::NDOT; j++) acc[j] = 0.;
    const bool run = !(check_status && st->status);
    if (run) {
        epi_begin(epi, 0);
        csr_sweep<VT>(A, x, epi, acc);
    }
    if (tail >= 0) grid_reduce<Epi::NDOT>(acc, ws, st, run ? tail : TAIL_NONE);
}

// y_row = sum over the row's slots in the order W,S,B,[X],C,[X],T,N,E (the sorted column
// order of a non-wrapped row; X is the cross entry, before C for component 1, after it for 0).
// Every load of a plane is issued before the multiply-adds; entries removed by a boundary
// edit read a valid in-range address and contribute +0.0 (the partial sum starts at +0.0 and
// so is never -0.0: adding +0.0 leaves it bit-identical to skipping the term).
//
// dia_column runs one (j, k) column of a tile over the planes i0 <= i < i1 with the i-1/i/i+1
// values of x rolled through registers. x and D belong to one system; row0 is that system's
// first row in the epilogue's vectors (0 for a single system).
// COPY: each slot value is also written to D32 in FP32 (every row is visited once per sweep).
// SYM (one component): the view is exactly symmetric, and a row's E, N and T are read as the W, S
// and B of its east, north and top neighbours, as in dia_column_pair_sym: four slots' bytes instead
// of seven where an odd k extent keeps the pairs out (145 x 128 x 121, FP64: 28.7 -> 22.5 us).
template <int NC, typename VT, bool COPY = false, bool SYM = false, class Src, class Epi>
__device__ inline void dia_column(const DiaView& V, const VT* __restrict__ D, const Src x,
                                  long long row0, int k, int j, int i0, int i1, const Epi& epi, double* acc,
                                  float* __restrict__ D32 = nullptr) {
    using Ix = SweepIndex<Epi>;
    const int n0 = V.n[0], n1 = V.n[1], n2 = V.n[2];
    const Ix sI = static_cast<Ix>(n1) * n2, sJ = n2, one = 1;
    const long long nr = V.nrows;
    // j and k neighbours: presence (boundary edits) and wrap
    const bool hasS = !(j == 0 && V.rm_lo[1]);
    const bool hasN = !(j == n1 - 1 && V.rm_hi[1] && !(j == 0 && V.rm_lo[1]));
    const bool hasB = !(k == 0 && V.rm_lo[2]);
    const bool hasT = !(k == n2 - 1 && V.rm_hi[2] && !(k == 0 && V.rm_lo[2]));
    const Ix dS = !hasS ? 0 : (j == 0) ? (n1 - 1) * sJ : 0 - sJ;
    const Ix dN = !hasN ? 0 : (j == n1 - 1) ? 0 - (n1 - 1) * sJ : sJ;
    const Ix dB = !hasB ? 0 : (k == 0) ? sJ - one : 0 - one;
    const Ix dT = !hasT ? 0 : (k == n2 - 1) ? one - sJ : one;
    Ix node = (static_cast<Ix>(i0) * n1 + j) * n2 + k;
    double xp[NC], xc[NC];
    static_assert(!SYM || (NC == 1 && !COPY), "symmetric views have one component");
    const auto ldnt = [](const VT* p) {
        if constexpr (Epi::kNT) return ld_nt(p);
        else return *p;
    };
    VT wv = VT(0);             // SYM: W of this plane's row, the E of the plane before
    if constexpr (SYM) wv = ldnt(at_off(D, node));
    {
        const bool need = !(i0 == 0 && V.rm_lo[0]);
        const Ix nprev = !need ? node : (i0 == 0) ? node + (n0 - 1) * sI : node - sI;
#pragma unroll
        for (int c = 0; c < NC; c++) {
            xc[c] = static_cast<double>(src1(x, node * NC + c));
            xp[c] = static_cast<double>(src1(x, nprev * NC + c));
        }
    }
    for (int i = i0; i < i1; i++) {
        const bool hasW = !(i == 0 && V.rm_lo[0]);
        const bool hasE = !(i == n0 - 1 && V.rm_hi[0] && !(i == 0 && V.rm_lo[0]));
        const Ix nnext = !hasE ? node : (i == n0 - 1) ? node - (n0 - 1) * sI : node + sI;
        double xn[NC], xs[NC], xnn[NC], xb[NC], xt[NC], pre[NC];
        VT dv[NC][8];      // converted where they are used: FP32 slots take half the registers
        if constexpr (NC == 2) {
            // the two component rows of a cell are adjacent (row = 2 node + c, nrows even, the
            // arrays start on 2-element boundaries): one 2-wide load per slot and per x entry
            typedef VT v2 __attribute__((ext_vector_type(2)));
            auto ldx = [&](Ix nd, double* o) { src2(x, nd * 2, o); };
            ldx(nnext, xn);
            ldx(node + dS, xs);
            ldx(node + dN, xnn);
            ldx(node + dB, xb);
            ldx(node + dT, xt);
            const int nsl = V.cross ? 8 : 7;
#pragma unroll
            for (int sl = 0; sl < 8; sl++) {
                v2 d = v2{VT(0), VT(0)};
                if (sl < nsl) {
                    const v2* p = reinterpret_cast<const v2*>(at_off(D + sl * nr, node * 2));
                    if constexpr (Epi::kNT) d = __builtin_nontemporal_load(p);
                    else d = *p;
                }
                dv[0][sl] = d.x;
                dv[1][sl] = d.y;
                if constexpr (COPY) {
                    typedef float f2 __attribute__((ext_vector_type(2)));
                    if (sl < nsl)
                        *reinterpret_cast<f2*>(D32 + sl * nr + node * 2) = f2{static_cast<float>(d.x), static_cast<float>(d.y)};
                }
            }
#pragma unroll
            for (int c = 0; c < NC; c++) pre[c] = epi.load(row0 + node * NC + c);
        } else {
#pragma unroll
            for (int c = 0; c < NC; c++) {
                const Ix row = node * NC + c;
                xn[c] = static_cast<double>(src1(x, nnext * NC + c));
                xs[c] = static_cast<double>(src1(x, (node + dS) * NC + c));
                xnn[c] = static_cast<double>(src1(x, (node + dN) * NC + c));
                xb[c] = static_cast<double>(src1(x, (node + dB) * NC + c));
                xt[c] = static_cast<double>(src1(x, (node + dT) * NC + c));
                if constexpr (SYM) {      // S and B are read again as partners: no hint
                    dv[c][0] = wv;
                    dv[c][1] = *at_off(D + nr, row);
                    dv[c][2] = *at_off(D + 2 * nr, row);
                    dv[c][3] = ldnt(at_off(D + 3 * nr, row));
                    dv[c][4] = *at_off(D + 2 * nr, row + dT);
                    dv[c][5] = *at_off(D + nr, row + dN);
                    dv[c][6] = wv = ldnt(at_off(D, nnext));
                }
#pragma unroll
                for (int sl = 0; sl < (SYM ? 0 : 7); sl++) {
                    dv[c][sl] = ldnt(at_off(D + sl * nr, row));
                    if constexpr (COPY) D32[sl * nr + row] = static_cast<float>(dv[c][sl]);
                }
                dv[c][7] = VT(0);
                pre[c] = epi.load(row0 + row);
            }
        }
        // straight-line per component (no loop around the epilogue's stores: LLVM's loop
        // invariant code motion promotes a store out of a one-trip loop and drops its
        // non-temporal hint on the way)
        auto row_out = [&](const int c) {
            const auto d = [&](int sl) { return static_cast<double>(dv[c][sl]); };
            double s = 0.;
            s += hasW ? d(0) * xp[c] : 0.;
            s += hasS ? d(1) * xs[c] : 0.;
            s += hasB ? d(2) * xb[c] : 0.;
            if (NC == 2 && V.cross && c == 1) s += d(7) * xc[0];
            s += d(3) * xc[c];
            if (NC == 2 && V.cross && c == 0) s += d(7) * xc[NC - 1];
            s += hasT ? d(4) * xt[c] : 0.;
            s += hasN ? d(5) * xnn[c] : 0.;
            s += hasE ? d(6) * xn[c] : 0.;
            epi(row0 + node * NC + c, s, xc[c], pre[c], acc);
        };
        row_out(0);
        if constexpr (NC == 2) row_out(1);
#pragma unroll
        for (int c = 0; c < NC; c++) {
            xp[c] = xc[c];
            xc[c] = xn[c];
        }
        node += sI;   // a tile never runs past plane n0 - 1, so xc is always a real plane
    }
}

// dia_column_pair: one component, the two cells k (even) and k+1 of a lane. Their slot values,
// x entries along i and j and epilogue operands are adjacent in memory, so each pair is one
// access twice as wide (a wave moves twice the bytes per memory instruction). Within the pair
// the top neighbour of cell k and the bottom neighbour of cell k+1 are the pair itself; only
// k-1 (cell k) and k+2 (cell k+1) are single loads. Each cell's sum keeps the order of
// dia_column, so y is bit-identical; the per-lane dot accumulation order differs.
template <typename VT, class Src, class Epi>
__device__ inline void dia_column_pair(const DiaView& V, const VT* __restrict__ D, const Src x,
                                       int k, int j, int i0, int i1, const Epi& epi, double* acc) {
    using Ix = PairIndex<Epi>;
    const int n0 = V.n[0], n1 = V.n[1], n2 = V.n[2];
    const Ix sI = static_cast<Ix>(n1) * n2, sJ = n2, one = 1;
    const long long nr = V.nrows;
    const bool hasS = !(j == 0 && V.rm_lo[1]);
    const bool hasN = !(j == n1 - 1 && V.rm_hi[1] && !(j == 0 && V.rm_lo[1]));
    const bool hasB = !(k == 0 && V.rm_lo[2]);               // cell k   (its top is cell k+1)
    const bool hasT = !(k + 1 == n2 - 1 && V.rm_hi[2]);      // cell k+1 (its bottom is cell k; n2 >= 2)
    const Ix dS = !hasS ? 0 : (j == 0) ? (n1 - 1) * sJ : 0 - sJ;
    const Ix dN = !hasN ? 0 : (j == n1 - 1) ? 0 - (n1 - 1) * sJ : sJ;
    const Ix dB = !hasB ? 0 : (k == 0) ? sJ - one : 0 - one;            // from cell k
    const Ix dT = !hasT ? 0 : (k + 1 == n2 - 1) ? one - sJ : one;   // from cell k+1
    Ix node = (static_cast<Ix>(i0) * n1 + j) * n2 + k;
    double xp0, xp1, xc0, xc1;
    {
        const bool need = !(i0 == 0 && V.rm_lo[0]);
        const Ix nprev = !need ? node : (i0 == 0) ? node + (n0 - 1) * sI : node - sI;
        xc0 = static_cast<double>(src1(x, node));
        xc1 = static_cast<double>(src1(x, node + 1));
        xp0 = static_cast<double>(src1(x, nprev));
        xp1 = static_cast<double>(src1(x, nprev + 1));
    }
    for (int i = i0; i < i1; i++) {
        const bool hasW = !(i == 0 && V.rm_lo[0]);
        const bool hasE = !(i == n0 - 1 && V.rm_hi[0] && !(i == 0 && V.rm_lo[0]));
        const Ix nnext = !hasE ? node : (i == n0 - 1) ? node - (n0 - 1) * sI : node + sI;
        const double xn0 = static_cast<double>(src1(x, nnext)), xn1 = static_cast<double>(src1(x, nnext + 1));
        const double xs0 = static_cast<double>(src1(x, node + dS)), xs1 = static_cast<double>(src1(x, node + dS + 1));
        const double xq0 = static_cast<double>(src1(x, node + dN)), xq1 = static_cast<double>(src1(x, node + dN + 1));
        const double xb = static_cast<double>(src1(x, node + dB));
        const double xt = static_cast<double>(src1(x, node + 1 + dT));
        double d0[7], d1[7];
#pragma unroll
        for (int sl = 0; sl < 7; sl++) {
            if constexpr (Epi::kNT) {
                d0[sl] = static_cast<double>(ld_nt(at_off(D + sl * nr, node)));
                d1[sl] = static_cast<double>(ld_nt(at_off(D + sl * nr, node) + 1));
            } else {
                d0[sl] = static_cast<double>(*at_off(D + sl * nr, node));
                d1[sl] = static_cast<double>(at_off(D + sl * nr, node)[1]);
            }
        }
        const double pre0 = epi.load(node), pre1 = epi.load(node + 1);
        double s0 = 0.;
        s0 += hasW ? d0[0] * xp0 : 0.;
        s0 += hasS ? d0[1] * xs0 : 0.;
        s0 += hasB ? d0[2] * xb : 0.;
        s0 += d0[3] * xc0;
        s0 += d0[4] * xc1;
        s0 += hasN ? d0[5] * xq0 : 0.;
        s0 += hasE ? d0[6] * xn0 : 0.;
        double s1 = 0.;
        s1 += hasW ? d1[0] * xp1 : 0.;
        s1 += hasS ? d1[1] * xs1 : 0.;
        s1 += d1[2] * xc0;
        s1 += d1[3] * xc1;
        s1 += hasT ? d1[4] * xt : 0.;
        s1 += hasN ? d1[5] * xq1 : 0.;
        s1 += hasE ? d1[6] * xn1 : 0.;
        epi_pair(epi, node, s0, s1, xc0, xc1, pre0, pre1, acc);
        xp0 = xc0;
        xp1 = xc1;
        xc0 = xn0;
        xc1 = xn1;
        node += sI;
    }
}

// dia_column_pair for an exactly symmetric view (symmetric by construction, or found so by
// k_dia_asym): the E, N and T coefficients of a row are read as the W, S and B coefficients
// of its east, north and top neighbours, so four slots stream from HBM instead of seven. The
// partner values are the same numbers and each sum keeps dia_column_pair's order, so y is
// bit-identical. The east neighbour's W is the next plane's own W: it is loaded once and kept
// in registers. S and B are read again as partners of the rows south and below (from the
// caches), so they carry no non-temporal hint; C and the east W do.
template <typename VT, class Src, class Epi>
__device__ inline void dia_column_pair_sym(const DiaView& V, const VT* __restrict__ D, const Src x,
                                           int k, int j, int i0, int i1, const Epi& epi, double* acc) {
    using Ix = PairIndex<Epi>;
    const int n0 = V.n[0], n1 = V.n[1], n2 = V.n[2];
    const Ix sI = static_cast<Ix>(n1) * n2, sJ = n2, one = 1;
    const long long nr = V.nrows;
    const bool hasS = !(j == 0 && V.rm_lo[1]);
    const bool hasN = !(j == n1 - 1 && V.rm_hi[1] && !(j == 0 && V.rm_lo[1]));
    const bool hasB = !(k == 0 && V.rm_lo[2]);
    const bool hasT = !(k + 1 == n2 - 1 && V.rm_hi[2]);
    const Ix dS = !hasS ? 0 : (j == 0) ? (n1 - 1) * sJ : 0 - sJ;
    const Ix dN = !hasN ? 0 : (j == n1 - 1) ? 0 - (n1 - 1) * sJ : sJ;
    const Ix dB = !hasB ? 0 : (k == 0) ? sJ - one : 0 - one;
    const Ix dT = !hasT ? 0 : (k + 1 == n2 - 1) ? one - sJ : one;
    const VT* DW = D;
    const VT* DS = D + nr;
    const VT* DB = D + 2 * nr;
    const VT* DC = D + 3 * nr;
    auto ldnt = [](const VT* p) {
        if constexpr (Epi::kNT) return static_cast<double>(ld_nt(p));
        else return static_cast<double>(*p);
    };
    Ix node = (static_cast<Ix>(i0) * n1 + j) * n2 + k;
    double xp0, xp1, xc0, xc1;
    {
        const bool need = !(i0 == 0 && V.rm_lo[0]);
        const Ix nprev = !need ? node : (i0 == 0) ? node + (n0 - 1) * sI : node - sI;
        xc0 = static_cast<double>(src1(x, node));
        xc1 = static_cast<double>(src1(x, node + 1));
        xp0 = static_cast<double>(src1(x, nprev));
        xp1 = static_cast<double>(src1(x, nprev + 1));
    }
    double w0 = ldnt(at_off(DW, node)), w1 = ldnt(at_off(DW, node) + 1);
    for (int i = i0; i < i1; i++) {
        const bool hasW = !(i == 0 && V.rm_lo[0]);
        const bool hasE = !(i == n0 - 1 && V.rm_hi[0] && !(i == 0 && V.rm_lo[0]));
        // a following plane of this tile is always node + sI (i < n0 - 1 there), so the east
        // W loaded here is that plane's own W
        const Ix nnext = !hasE ? node : (i == n0 - 1) ? node - (n0 - 1) * sI : node + sI;
        const double xn0 = static_cast<double>(src1(x, nnext)), xn1 = static_cast<double>(src1(x, nnext + 1));
        const double xs0 = static_cast<double>(src1(x, node + dS)), xs1 = static_cast<double>(src1(x, node + dS + 1));
        const double xq0 = static_cast<double>(src1(x, node + dN)), xq1 = static_cast<double>(src1(x, node + dN + 1));
        const double xb = static_cast<double>(src1(x, node + dB));
        const double xt = static_cast<double>(src1(x, node + 1 + dT));
        const double sv0 = static_cast<double>(*at_off(DS, node)), sv1 = static_cast<double>(*at_off(DS, node + 1));
        const double bv0 = static_cast<double>(*at_off(DB, node)), bv1 = static_cast<double>(*at_off(DB, node + 1));
        const double cv0 = ldnt(at_off(DC, node)), cv1 = ldnt(at_off(DC, node) + 1);
        const double ev0 = ldnt(at_off(DW, nnext)), ev1 = ldnt(at_off(DW, nnext) + 1);        // W of the east neighbour
        const double nv0 = static_cast<double>(*at_off(DS, node + dN)), nv1 = static_cast<double>(*at_off(DS, node + dN + 1));
        const double tv1 = static_cast<double>(*at_off(DB, node + 1 + dT));              // B of cell k+1's top neighbour
        const double pre0 = epi.load(node), pre1 = epi.load(node + 1);
        double s0 = 0.;
        s0 += hasW ? w0 * xp0 : 0.;
        s0 += hasS ? sv0 * xs0 : 0.;
        s0 += hasB ? bv0 * xb : 0.;
        s0 += cv0 * xc0;
        s0 += bv1 * xc1;              // T of cell k = B of cell k+1
        s0 += hasN ? nv0 * xq0 : 0.;
        s0 += hasE ? ev0 * xn0 : 0.;
        double s1 = 0.;
        s1 += hasW ? w1 * xp1 : 0.;
        s1 += hasS ? sv1 * xs1 : 0.;
        s1 += bv1 * xc0;
        s1 += cv1 * xc1;
        s1 += hasT ? tv1 * xt : 0.;
        s1 += hasN ? nv1 * xq1 : 0.;
        s1 += hasE ? ev1 * xn1 : 0.;
        epi_pair(epi, node, s0, s1, xc0, xc1, pre0, pre1, acc);
        xp0 = xc0;
        xp1 = xc1;
        xc0 = xn0;
        xc1 = xn1;
        w0 = ev0;
        w1 = ev1;
        node += sI;
    }
}

// dia_column_quad: the FP32 operator of the inner solves (one component, FP32 slots and
// vectors), four k-adjacent rows per lane, so every slot, x and vector access is one 16-byte
// float4 and a wave moves 1 KB per memory instruction. The products and sums are FP32 (the
// precision of the inner iterations; the slot order of each row is dia_column's), the dot
// accumulators stay FP64. Rows k..k+3 with k a multiple of 4 and n2 % 4 == 0.
// UNIT: the C slot is 1 in every row and not read (36 instead of 40 bytes a row).
template <bool UNIT, class Src, class Epi>
__device__ inline void dia_column_quad(const DiaView& V, const float* __restrict__ D, const Src x,
                                       int k, int j, int i0, int i1, const Epi& epi, double* acc) {
    using Ix = PairIndex<Epi>;
    const int n0 = V.n[0], n1 = V.n[1], n2 = V.n[2];
    const Ix sI = static_cast<Ix>(n1) * n2, sJ = n2, one = 1;
    const long long nr = V.nrows;
    const bool hasS = !(j == 0 && V.rm_lo[1]);
    const bool hasN = !(j == n1 - 1 && V.rm_hi[1] && !(j == 0 && V.rm_lo[1]));
    const bool hasB = !(k == 0 && V.rm_lo[2]);               // cell k   (its top is cell k+1)
    const bool hasT = !(k + 3 == n2 - 1 && V.rm_hi[2]);      // cell k+3 (n2 >= 4)
    const Ix dS = !hasS ? 0 : (j == 0) ? (n1 - 1) * sJ : 0 - sJ;
    const Ix dN = !hasN ? 0 : (j == n1 - 1) ? 0 - (n1 - 1) * sJ : sJ;
    const Ix dB = !hasB ? 0 : (k == 0) ? sJ - one : 0 - one;            // from cell k
    const Ix dT = !hasT ? 0 : (k + 3 == n2 - 1) ? one - sJ : one;   // from cell k+3
    typedef f32x4 f4;
    auto ld4 = [](const float* p) { return *reinterpret_cast<const f4*>(p); };
    auto ld4nt = [](const float* p) {
        if constexpr (Epi::kNT) return __builtin_nontemporal_load(reinterpret_cast<const f4*>(p));
        else return *reinterpret_cast<const f4*>(p);
    };
    Ix node = (static_cast<Ix>(i0) * n1 + j) * n2 + k;
    f4 xp, xc;
    {
        const bool need = !(i0 == 0 && V.rm_lo[0]);
        const Ix nprev = !need ? node : (i0 == 0) ? node + (n0 - 1) * sI : node - sI;
        xc = src4(x, node);
        xp = src4(x, nprev);
    }
    for (int i = i0; i < i1; i++) {
        const bool hasW = !(i == 0 && V.rm_lo[0]);
        const bool hasE = !(i == n0 - 1 && V.rm_hi[0] && !(i == 0 && V.rm_lo[0]));
        const Ix nnext = !hasE ? node : (i == n0 - 1) ? node - (n0 - 1) * sI : node + sI;
        const f4 xn = src4(x, nnext), xs = src4(x, node + dS), xq = src4(x, node + dN);
        const float xb = src1(x, node + dB), xt = src1(x, node + 3 + dT);
        f4 d[7];
#pragma unroll
        for (int sl = 0; sl < 7; sl++)
            if (!(UNIT && sl == 3)) d[sl] = ld4nt(at_off(D + sl * nr, node));
        const double p0 = epi.load(node), p1 = epi.load(node + 1), p2 = epi.load(node + 2), p3 = epi.load(node + 3);
        const float xcv[4] = {xc.x, xc.y, xc.z, xc.w}, xpv[4] = {xp.x, xp.y, xp.z, xp.w};
        const float xsv[4] = {xs.x, xs.y, xs.z, xs.w}, xqv[4] = {xq.x, xq.y, xq.z, xq.w};
        const float xnv[4] = {xn.x, xn.y, xn.z, xn.w};
        double y[4];
#pragma unroll
        for (int m = 0; m < 4; m++) {
            auto dv = [&](int sl) { return m == 0 ? d[sl].x : m == 1 ? d[sl].y : m == 2 ? d[sl].z : d[sl].w; };
            float s = 0.f;
            s += hasW ? dv(0) * xpv[m] : 0.f;
            s += hasS ? dv(1) * xsv[m] : 0.f;
            if (m == 0) s += hasB ? dv(2) * xb : 0.f;
            else s += dv(2) * xcv[m - 1];
            s += UNIT ? xcv[m] : dv(3) * xcv[m];
            if (m == 3) s += hasT ? dv(4) * xt : 0.f;
            else s += dv(4) * xcv[m + 1];
            s += hasN ? dv(5) * xqv[m] : 0.f;
            s += hasE ? dv(6) * xnv[m] : 0.f;
            y[m] = static_cast<double>(s);
        }
        const double xcd[4] = {xcv[0], xcv[1], xcv[2], xcv[3]}, pre[4] = {p0, p1, p2, p3};
        epi_quad(epi, node, y, xcd, pre, acc);
        xp = xc;
        xc = xn;
        node += sI;
    }
}

// dia_column_quad for an exactly symmetric FP32 view (the FP32 copy of a symmetric FP64 view): the E, N and T
// coefficients of a row are read as the W, S and B coefficients of its east, north and top
// neighbours, so four slots stream from HBM instead of seven. The partner values are the same
// floats and the arithmetic is that of dia_column_quad, so the results are bit-identical. The
// W, S and B slots are read twice (as a row's own and as its neighbour's partner), the second
// time from the caches, so they carry no non-temporal hint.
template <class Src, class Epi>
__device__ inline void dia_column_quad_sym(const DiaView& V, const float* __restrict__ D, const Src x,
                                           int k, int j, int i0, int i1, const Epi& epi, double* acc) {
    using Ix = PairIndex<Epi>;
    const int n0 = V.n[0], n1 = V.n[1], n2 = V.n[2];
    const Ix sI = static_cast<Ix>(n1) * n2, sJ = n2, one = 1;
    const long long nr = V.nrows;
    const bool hasS = !(j == 0 && V.rm_lo[1]);
    const bool hasN = !(j == n1 - 1 && V.rm_hi[1] && !(j == 0 && V.rm_lo[1]));
    const bool hasB = !(k == 0 && V.rm_lo[2]);
    const bool hasT = !(k + 3 == n2 - 1 && V.rm_hi[2]);
    const Ix dS = !hasS ? 0 : (j == 0) ? (n1 - 1) * sJ : 0 - sJ;
    const Ix dN = !hasN ? 0 : (j == n1 - 1) ? 0 - (n1 - 1) * sJ : sJ;
    const Ix dB = !hasB ? 0 : (k == 0) ? sJ - one : 0 - one;
    const Ix dT = !hasT ? 0 : (k + 3 == n2 - 1) ? one - sJ : one;
    typedef f32x4 f4;
    auto ld4 = [](const float* p) { return *reinterpret_cast<const f4*>(p); };
    auto ld4nt = [](const float* p) {
        if constexpr (Epi::kNT) return __builtin_nontemporal_load(reinterpret_cast<const f4*>(p));
        else return *reinterpret_cast<const f4*>(p);
    };
    const float* DW = D;
    const float* DS = D + nr;
    const float* DB = D + 2 * nr;
    const float* DC = D + 3 * nr;
    // everything a plane reads, loaded one plane ahead (the next plane's loads are in flight
    // while this plane's sums are formed)
    struct Plane {
        f4 xn, xs, xq, cW, cS, cB, cC, cN, cE;
        float xb, xt, cT3;
        double pre[4];
        bool hasW, hasE;
    };
    auto load = [&](int i, Ix node, Plane& P) {
        P.hasW = !(i == 0 && V.rm_lo[0]);
        P.hasE = !(i == n0 - 1 && V.rm_hi[0] && !(i == 0 && V.rm_lo[0]));
        const Ix nnext = !P.hasE ? node : (i == n0 - 1) ? node - (n0 - 1) * sI : node + sI;
        P.xn = src4(x, nnext);
        P.xs = src4(x, node + dS);
        P.xq = src4(x, node + dN);
        P.xb = src1(x, node + dB);
        P.xt = src1(x, node + 3 + dT);
        P.cW = ld4(at_off(DW, node));
        P.cS = ld4(at_off(DS, node));
        P.cB = ld4(at_off(DB, node));
        P.cC = ld4nt(at_off(DC, node));
        P.cN = ld4(at_off(DS, node + dN));          // S of the north neighbour (unused without it)
        P.cE = ld4(at_off(DW, nnext));              // W of the east neighbour
        P.cT3 = *at_off(DB, node + 3 + dT);           // B of the top neighbour of cell k + 3
#pragma unroll
        for (int m = 0; m < 4; m++) P.pre[m] = epi.load(node + m);
    };
    Ix node = (static_cast<Ix>(i0) * n1 + j) * n2 + k;
    f4 xp, xc;
    {
        const bool need = !(i0 == 0 && V.rm_lo[0]);
        const Ix nprev = !need ? node : (i0 == 0) ? node + (n0 - 1) * sI : node - sI;
        xc = src4(x, node);
        xp = src4(x, nprev);
    }
    Plane cur;
    load(i0, node, cur);
    for (int i = i0; i < i1; i++) {
        Plane nxt;
        const int inext = i + 1 < i1 ? i + 1 : i;            // the last plane reloads itself
        load(inext, node + (i + 1 < i1 ? sI : 0), nxt);
        const float xcv[4] = {xc.x, xc.y, xc.z, xc.w}, xpv[4] = {xp.x, xp.y, xp.z, xp.w};
        const float xsv[4] = {cur.xs.x, cur.xs.y, cur.xs.z, cur.xs.w};
        const float xqv[4] = {cur.xq.x, cur.xq.y, cur.xq.z, cur.xq.w};
        const float xnv[4] = {cur.xn.x, cur.xn.y, cur.xn.z, cur.xn.w};
        const float wv[4] = {cur.cW.x, cur.cW.y, cur.cW.z, cur.cW.w}, sv[4] = {cur.cS.x, cur.cS.y, cur.cS.z, cur.cS.w};
        const float bv[4] = {cur.cB.x, cur.cB.y, cur.cB.z, cur.cB.w}, cv[4] = {cur.cC.x, cur.cC.y, cur.cC.z, cur.cC.w};
        const float tv[4] = {cur.cB.y, cur.cB.z, cur.cB.w, cur.cT3};
        const float nv[4] = {cur.cN.x, cur.cN.y, cur.cN.z, cur.cN.w}, ev[4] = {cur.cE.x, cur.cE.y, cur.cE.z, cur.cE.w};
        double y[4];
#pragma unroll
        for (int m = 0; m < 4; m++) {
            float s = 0.f;
            s += cur.hasW ? wv[m] * xpv[m] : 0.f;
            s += hasS ? sv[m] * xsv[m] : 0.f;
            if (m == 0) s += hasB ? bv[m] * cur.xb : 0.f;
            else s += bv[m] * xcv[m - 1];
            s += cv[m] * xcv[m];
            if (m == 3) s += hasT ? tv[m] * cur.xt : 0.f;
            else s += tv[m] * xcv[m + 1];
            s += hasN ? nv[m] * xqv[m] : 0.f;
            s += cur.hasE ? ev[m] * xnv[m] : 0.f;
            y[m] = static_cast<double>(s);
        }
        const double xcd[4] = {xcv[0], xcv[1], xcv[2], xcv[3]};
        epi_quad(epi, node, y, xcd, cur.pre, acc);
        xp = xc;
        xc = cur.xn;
        cur = nxt;
        node += sI;
    }
}

// Symmetry check of a one-component view (FP32 or FP64 slots): flag = 1 if the E, N or T
// coefficient of any row differs (bit for bit) from the W, S or B coefficient of the neighbour
// it couples to, with the neighbour and presence rules of dia_column. flag must be 0 before the
// launch.
template <typename VT>
__global__ __launch_bounds__(kThreads) void k_dia_asym(DiaView V, const VT* __restrict__ D, int* __restrict__ flag) {
    const long long nr = V.nrows;
    const int n0 = V.n[0], n1 = V.n[1], n2 = V.n[2];
    const long long sI = static_cast<long long>(n1) * n2, sJ = n2;
    auto bits = [](VT v) {
        if constexpr (std::is_same_v<VT, float>) return __float_as_uint(v);
        else return static_cast<unsigned long long>(__double_as_longlong(v));
    };
    bool bad = false;
    for (long long row = static_cast<long long>(blockIdx.x) * kThreads + threadIdx.x; row < nr;
         row += static_cast<long long>(gridDim.x) * kThreads) {
        const int k = static_cast<int>(row % n2), j = static_cast<int>((row / n2) % n1), i = static_cast<int>(row / sI);
        if (!(i == n0 - 1 && V.rm_hi[0] && !(i == 0 && V.rm_lo[0]))) {
            const long long nb = (i == n0 - 1) ? row - (long long)(n0 - 1) * sI : row + sI;
            bad |= bits(D[6 * nr + row]) != bits(D[nb]);
        }
        if (!(j == n1 - 1 && V.rm_hi[1] && !(j == 0 && V.rm_lo[1]))) {
            const long long nb = (j == n1 - 1) ? row - (long long)(n1 - 1) * sJ : row + sJ;
            bad |= bits(D[5 * nr + row]) != bits(D[nr + nb]);
        }
        if (!(k == n2 - 1 && V.rm_hi[2])) {
            const long long nb = (k == n2 - 1) ? row - (n2 - 1) : row + 1;
            bad |= bits(D[4 * nr + row]) != bits(D[2 * nr + nb]);
        }
    }
    if (bad) flag[0] = 1;
}

__global__ void k_set_int(int* __restrict__ p, int v) { p[0] = v; }

// One work-group's tile of the view. PAIR: cells per lane along k (1, 2, or 4 for FP32); SYM
// (pairs and quads): the symmetric traversal.
template <int NC, int PAIR, bool SYM, bool UNIT = false, typename VT, class Src, class Epi>
__device__ inline void dia_tile(const DiaOp<VT>& A, const Src x, const Epi& epi, double* acc) {
    const int tile = static_cast<int>(blockIdx.x % kXcd) * A.per_xcd + static_cast<int>(blockIdx.x / kXcd);
    if (tile >= A.tiles_k * A.tiles_j * A.tiles_i) return;
    const int tk = tile % A.tiles_k;
    const int t2 = tile / A.tiles_k;
    const int tj = t2 % A.tiles_j;
    const int ti = t2 / A.tiles_j;
    const int lane_k = threadIdx.x & ((1 << A.lk_log2) - 1);
    const int k = ((tk << A.lk_log2) + lane_k) * PAIR;
    const int j = tj * (kThreads >> A.lk_log2) + (threadIdx.x >> A.lk_log2);
    if (k >= A.V.n[2] || j >= A.V.n[1]) return;
    const int i0 = ti * A.tile_i;
    const int i1 = (i0 + A.tile_i < A.V.n[0]) ? i0 + A.tile_i : A.V.n[0];
    if constexpr (PAIR == 4) {
        static_assert(std::is_same_v<VT, float>, "quad traversal is FP32");
        if constexpr (SYM) dia_column_quad_sym(A.V, A.D, x, k, j, i0, i1, epi, acc);
        else dia_column_quad<UNIT>(A.V, A.D, x, k, j, i0, i1, epi, acc);
    } else if constexpr (PAIR == 2 && SYM) {
        dia_column_pair_sym<VT>(A.V, A.D, x, k, j, i0, i1, epi, acc);
    } else if constexpr (PAIR == 2) {
        dia_column_pair<VT>(A.V, A.D, x, k, j, i0, i1, epi, acc);
    } else {
        dia_column<NC, VT, false, SYM>(A.V, A.D, x, 0, k, j, i0, i1, epi, acc);
    }
}

// the symmetric traversal is a separate instantiation so that the seven-slot one keeps its own
// register count
template <int NC, typename VT, typename XT, class Epi, int PAIR = 1, bool SYM = false, bool UNIT = false>
__global__ __launch_bounds__(kThreads) void k_apply_dia(DiaOp<VT> A, const XT* __restrict__ x, Epi epi, ReduceWs ws,
                                                       KState* st, int tail, int check_status) {
    double acc[Epi::NDOT];
#pragma unroll
    for (int j = 0; j < Epi::NDOT; j++) acc[j] = 0.;
    const bool run = !(check_status && st->status);
    if (run) {
        epi_begin(epi, 0);
        dia_tile<NC, PAIR, SYM, UNIT>(A, x, epi, acc);
    }
    if (tail >= 0) grid_reduce<Epi::NDOT>(acc, ws, st, run ? tail : TAIL_NONE);
}

// ------------------------------------------------------------------------------ fused steps
// Passes of SolveOp::fused: five launches and a finish instead of nine launches and five finish
// kernels. Each operator application forms its operand a - c b where it reads it (steps 5, 8, 12,
// 17) and writes it out once; and each kernel sums the previous one's partials itself and applies
// the scalar update (every work-group alike; the first one stores the new state for the next
// kernel, which reads another slot), so the four finish kernels between them are gone. A small
// kernel is a few microseconds of latency whatever it does: a 64^3 implicit step went from 233 to
// 156 us (with the readback through pinned memory), a 160 x 120 two-component one from 200 to 123.
// At 128^3 a step of seven slots takes 31 us; update, sweep and finish took 9.0 + 24.3 + 4.5. Where
// the two forms are level stands beside SolveOp::fused; where sweeps stream, the streaming form is
// not given up. The vector operations round as the separate kernels do.
template <typename XT>
struct StepVecs {
    const XT *a, *b;     // the operand is a - c b
    XT* xo;              // where it goes
    XT* y;               // A times it
    const XT* w;         // <y, w>; for step 18: r before step 16
    const XT* v;         // step 18: v
};
struct StepRed {
    const double* pin;   // partials of the previous kernel, dot-major with stride kReduceBlocks
    unsigned npin;
    double* pout;
    const KState* sin;
    KState* sout;
    int tail;            // TAIL_NONE: no partials to sum, the state is sin
    int alpha;           // c = alpha, else beta
};

// The state at this kernel's start, the same in every work-group: sin after the tail with the
// sums of pin. st: one per work-group, in LDS. Ends with a barrier; true unless broken down.
template <int NIN>
__device__ inline bool step_state(const StepRed& R, KState* st) {
    __shared__ double red[NIN][kThreads / 64];
    if (R.tail != TAIL_NONE) {
        const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
        double s[NIN];
#pragma unroll
        for (int j = 0; j < NIN; j++) s[j] = 0.;
        for (unsigned b0 = 0; b0 < R.npin; b0 += 4 * kThreads) {
            double v[NIN][4];
#pragma unroll
            for (int j = 0; j < NIN; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const unsigned b = b0 + q * kThreads + threadIdx.x;
                    v[j][q] = b < R.npin ? R.pin[j * kReduceBlocks + b] : 0.;
                }
#pragma unroll
            for (int j = 0; j < NIN; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) s[j] += v[j][q];
        }
#pragma unroll
        for (int j = 0; j < NIN; j++) {
            const double t = wave_sum(s[j]);
            if (lane == 0) red[j][wid] = t;
        }
    }
    KState k = *R.sin;
    __syncthreads();
    if (threadIdx.x == 0) {
        if (R.tail != TAIL_NONE && !k.status) {
            double d[kMaxDots] = {};
            for (int j = 0; j < NIN; j++)
                for (int w = 0; w < kThreads / 64; w++) d[j] += red[j][w];
            apply_tail(R.tail, &k, d);
        }
        *st = k;
        if (blockIdx.x == 0 && R.sout) *R.sout = k;
    }
    __syncthreads();
    return st->status == 0;
}

template <typename XT>
struct EpiStepDot {      // the operand and out = A p; <out, w>
    static constexpr bool kStep = true;
    static constexpr int NDOT = 1;
    static constexpr bool kNT = false;
    XT* xo;
    XT* out;
    const XT* w;
    __device__ double load(long long i) const { return static_cast<double>(w[i]); }
    __device__ void operator()(long long i, double y, double xc, double wi, double* acc) const {
        const XT yi = static_cast<XT>(y);
        xo[i] = static_cast<XT>(xc);
        out[i] = yi;
        acc[0] += static_cast<double>(yi) * wi;
    }
};
template <typename XT>
struct EpiStepGcr {      // the operand s, t = A s, and step 18's five dots with r - alpha v
    static constexpr int NDOT = 5;
    static constexpr bool kNT = false;
    XT* xo;
    XT* t;
    const XT* r;
    const XT* v;
    double alpha;
    __device__ double load(long long i) const {
        return static_cast<double>(static_cast<XT>(static_cast<double>(r[i]) - alpha * static_cast<double>(v[i])));
    }
    __device__ void operator()(long long i, double y, double sc, double rd, double* acc) const {
        const XT ti = static_cast<XT>(y);
        xo[i] = static_cast<XT>(sc);
        t[i] = ti;
        const double td = static_cast<double>(ti);
        acc[0] += rd * sc;
        acc[1] += sc * sc;
        acc[2] += sc * td;
        acc[3] += td * td;
        acc[4] += rd * td;
    }
};

// GCR: steps 17-20, else one of steps 5-7, 8-11 (its two parts) or 12-14; APPLY runs the sweep
// over the work-group's rows
template <bool GCR, typename XT, class Apply>
__device__ inline void step_body(const StepVecs<XT>& S, const StepRed& R, Apply&& apply) {
    __shared__ KState st;
    constexpr int NDOT = GCR ? 5 : 1;
    double acc[NDOT] = {};
    if (step_state<1>(R, &st)) {
        const Comb<XT> x{S.a, S.b, R.alpha ? st.alpha : st.beta};
        if constexpr (GCR) apply(x, EpiStepGcr<XT>{S.xo, S.y, S.w, S.v, st.alpha}, acc);
        else apply(x, EpiStepDot<XT>{S.xo, S.y, S.w}, acc);
    }
    block_partials_at<NDOT>(acc, R.pout, kReduceBlocks, blockIdx.x);
}
template <int NC, typename VT, typename XT, bool GCR, int PAIR, bool SYM>
__global__ __launch_bounds__(kThreads) void k_step_dia(DiaOp<VT> A, StepVecs<XT> S, StepRed R) {
    step_body<GCR>(S, R, [&](const Comb<XT>& x, const auto& epi, double* acc) {
        dia_tile<NC, PAIR, SYM>(A, x, epi, acc);
    });
}
template <typename VT, typename XT, bool GCR>
__global__ __launch_bounds__(kThreads) void k_step_csr(CsrOp<VT> A, StepVecs<XT> S, StepRed R) {
    step_body<GCR>(S, R, [&](const Comb<XT>& x, const auto& epi, double* acc) { csr_sweep<VT>(A, x, epi, acc); });
}

// ------------------------------------------------------------------------------ vector updates
// Grid-stride over chunks of kU * kThreads elements; all loads of a chunk are issued before
// its arithmetic so that every wave keeps several independent HBM requests in flight.
// (status != 0 => the pass has broken down: every launch is a no-op)
constexpr int kU = 4;

#define DARE_CHUNK_LOOP(n)                                                                        \
    for (long long base_ = blockIdx.x * (long long)(kThreads * kU); base_ < (n);                  \
         base_ += (long long)gridDim.x * (kThreads * kU))
#define DARE_IDX(u) (base_ + (long long)(u) * kThreads + threadIdx.x)

// Steps 5, 8, 12 and 17: out = a - c b with c = beta or alpha. (out may be a or b.)
template <typename XT, bool NT, bool ALPHA>
__global__ __launch_bounds__(kThreads) void k_comb(long long n, const XT* a, const XT* b, XT* out,
                                                   const KState* __restrict__ st) {
    if (st->status) return;
    const double c = ALPHA ? st->alpha : st->beta;
    DARE_CHUNK_LOOP(n) {
        double av[kU], bv[kU];
#pragma unroll
        for (int q = 0; q < kU; q++) {
            const long long i = DARE_IDX(q) < n ? DARE_IDX(q) : 0;
            av[q] = static_cast<double>(a[i]);
            bv[q] = static_cast<double>(b[i]);
        }
#pragma unroll
        for (int q = 0; q < kU; q++)
            if (DARE_IDX(q) < n) put<NT>(out + DARE_IDX(q), static_cast<XT>(av[q] - c * bv[q]));
    }
}

// The pass's last kernel: every update of x, r and u that no operator application of the pass
// waits for, from the vectors as the applications left them.
//   (15) u' = r - beta u    (16) r' = r - alpha v    (10) x' = x + alpha1 u
//   x = x' + om1 r' + om2 s + alpha u'; r = r' - om1 s - om2 t; u = u' - om1 v - om2 w;
//   <r,r>, <rh,r>
// Steps 10, 15 and 16 took 64 B/row of their own (FP64) and r', u' were written only to be read
// back here: a pass moves 416 B/row instead of 472, with the same rounding at every step
// (256^3 FP64: steps 8, 10 and 15-17 took 135 + 184 us, steps 8 and 17 alone 65 + 65; t's sweep
// reads one vector more, 210 -> 212 us; this kernel 272 -> 256).
// ro, uo: r and u before the pass's last updates (the shadow residual in a first pass, which
// reads u = r); XZERO: x was never written and counts as 0. A breakdown after step 10 leaves
// x = x + alpha1 u, as the reference's order of the updates does.
template <typename XT>
struct EndVecs {
    XT* x;
    const XT *ro, *s, *t, *uo, *v, *w, *rh;
    XT *r, *u;           // written: r may be ro or w, u may be uo or t
};
template <typename XT, bool NT, bool XZERO>
__device__ inline void pass_end(long long n, const EndVecs<XT>& E, const KState* st, bool run, double (&acc)[2]) {
    XT* x = E.x;
    const XT *ro = E.ro, *s = E.s, *t = E.t, *uo = E.uo, *v = E.v, *w = E.w, *rh = E.rh;
    XT *r = E.r, *u = E.u;
    const double a1 = st->alpha1;
    if (run) {
        const double o1 = st->om1, o2 = st->om2, a = st->alpha, beta = st->beta;
        DARE_CHUNK_LOOP(n) {
            double xv[kU], rv[kU], sv[kU], tv[kU], uv[kU], vv[kU], wv[kU], hv[kU];
#pragma unroll
            for (int q = 0; q < kU; q++) {
                const long long i = DARE_IDX(q) < n ? DARE_IDX(q) : 0;
                xv[q] = XZERO ? 0. : static_cast<double>(x[i]);
                rv[q] = static_cast<double>(ro[i]);
                sv[q] = static_cast<double>(s[i]);
                tv[q] = static_cast<double>(t[i]);
                uv[q] = static_cast<double>(uo[i]);
                vv[q] = static_cast<double>(v[i]);
                wv[q] = static_cast<double>(w[i]);
                hv[q] = static_cast<double>(rh[i]);
            }
#pragma unroll
            for (int q = 0; q < kU; q++) {
                const long long i = DARE_IDX(q);
                if (i < n) {
                    const double x1 = static_cast<double>(static_cast<XT>(1. * xv[q] + a1 * uv[q]));      // (10)
                    const double u1 = static_cast<double>(static_cast<XT>(rv[q] - beta * uv[q]));         // (15)
                    const double r1 = static_cast<double>(static_cast<XT>(rv[q] - a * vv[q]));            // (16)
                    double xi = 1. * x1 + o1 * r1 + o2 * sv[q];                                           // (24)
                    xi = 1. * xi + a * u1;
                    put<NT>(x + i, static_cast<XT>(xi));
                    const XT rn = static_cast<XT>(1. * r1 + (-o1) * sv[q] + (-o2) * tv[q]);               // (25)
                    put<NT>(r + i, rn);
                    put<NT>(u + i, static_cast<XT>(1. * u1 + (-o1) * vv[q] + (-o2) * wv[q]));
                    const double rd = static_cast<double>(rn);
                    acc[0] += rd * rd;
                    acc[1] += hv[q] * rd;
                }
            }
        }
    } else if (st->x_due || XZERO) {
        const double c = st->x_due ? a1 : 0.;
        for (long long i = blockIdx.x * (long long)kThreads + threadIdx.x; i < n; i += (long long)gridDim.x * kThreads)
            put<NT>(x + i, c == 0. ? (XZERO ? XT(0) : x[i])
                                   : static_cast<XT>((XZERO ? 0. : 1. * static_cast<double>(x[i])) +
                                                     c * static_cast<double>(uo[i])));
    }
}

template <typename XT, bool NT, bool XZERO>
__global__ __launch_bounds__(kThreads) void k_pass_end(long long n, EndVecs<XT> E, ReduceWs ws, KState* st) {
    double acc[2] = {0., 0.};
    pass_end<XT, NT, XZERO>(n, E, st, st->status == 0, acc);
    block_partials<2>(acc, ws);
}

// the same as the last of the fused steps: the scalars of step 19 from the partials first
template <typename XT, bool XZERO>
__global__ __launch_bounds__(kThreads) void k_step_end(long long n, EndVecs<XT> E, StepRed R) {
    __shared__ KState st;
    double acc[2] = {0., 0.};
    const bool run = step_state<5>(R, &st);
    pass_end<XT, false, XZERO>(n, E, &st, run, acc);
    block_partials_at<2>(acc, R.pout, kReduceBlocks, blockIdx.x);
}

template <typename XT>
__global__ __launch_bounds__(kThreads) void k_dot(long long n, const XT* __restrict__ a, const XT* __restrict__ b,
                                                  ReduceWs ws, KState* st) {
    double acc[1] = {0.};
    DARE_CHUNK_LOOP(n) {
        double av[kU], bv[kU];
#pragma unroll
        for (int q = 0; q < kU; q++) {
            const long long i = DARE_IDX(q) < n ? DARE_IDX(q) : 0;
            av[q] = static_cast<double>(a[i]);
            bv[q] = static_cast<double>(b[i]);
        }
#pragma unroll
        for (int q = 0; q < kU; q++)
            if (DARE_IDX(q) < n) acc[0] += av[q] * bv[q];
    }
    grid_reduce<1>(acc, ws, st, TAIL_STORE);
}

// Initialisation (0)-(2) for a zero initial guess: A x0 is +0 in every row, so r = b - A x0 = b
// bit for bit, and <r,r>, <rh,r> go to the reduction. Nothing is written: the
// first pass reads b where it would read r or u and 0 where it would read x, and writes them.
// rh = r0 is never written again, so the caller reads b itself as rh (b stays untouched during
// the solve); v and w are written before they are read.
template <typename XT>
__global__ __launch_bounds__(kThreads) void k_init_zero(long long n, const XT* __restrict__ b, ReduceWs ws, KState* st) {
    double acc[2] = {0., 0.};
    DARE_CHUNK_LOOP(n) {
        XT bv[kU];
#pragma unroll
        for (int q = 0; q < kU; q++) bv[q] = b[DARE_IDX(q) < n ? DARE_IDX(q) : 0];
#pragma unroll
        for (int q = 0; q < kU; q++) {
            if (DARE_IDX(q) < n) {
                const double rd = static_cast<double>(bv[q]);
                acc[0] += rd * rd;
                acc[1] += rd * rd;
            }
        }
    }
    grid_reduce<2>(acc, ws, st, TAIL_INIT);
}

__global__ __launch_bounds__(kThreads) void k_axpby(long long n, double a, const double* __restrict__ x, double b,
                                                    double* __restrict__ y) {
    for (long long i = blockIdx.x * (long long)kThreads + threadIdx.x; i < n; i += (long long)gridDim.x * kThreads)
        y[i] = a * x[i] + b * y[i];
}

__global__ __launch_bounds__(kThreads) void k_add_correction(long long n, double* __restrict__ x,
                                                             const float* __restrict__ d) {
    for (long long i = blockIdx.x * (long long)kThreads + threadIdx.x; i < n; i += (long long)gridDim.x * kThreads)
        x[i] = x[i] + static_cast<double>(d[i]);
}

template <typename T>
__global__ __launch_bounds__(kThreads) void k_zero(long long n, T* __restrict__ p) {
    for (long long i = blockIdx.x * (long long)kThreads + threadIdx.x; i < n; i += (long long)gridDim.x * kThreads)
        p[i] = T(0);
}

__global__ __launch_bounds__(kThreads) void k_to_f32(long long n, const double* __restrict__ a, float* __restrict__ b) {
    for (long long i = blockIdx.x * (long long)kThreads + threadIdx.x; i < n; i += (long long)gridDim.x * kThreads)
        b[i] = static_cast<float>(a[i]);
}

__global__ void k_clear_state(KState* st) {
    if (threadIdx.x == 0) {
        st->status = 0;
        st->next_status = 0;
    }
}

// The fused steps: never from kFusedRows rows on, where sweeps stream; below by the traversal
// (SolveOp::fused in krylov.hip).
constexpr long long kFusedRows = kStreamRows;
constexpr unsigned kStepCsrGrid = 1024;      // ... on CSR, whose waves loop over their rows
constexpr unsigned kFusedEndBlocks = 512;    // k_step_end: every work-group sums all of step 18's partials
constexpr int kStates = 5;                   // state slots of a solve, one per kernel of a fused pass
constexpr int kPassVecs = 8;                 // work vectors of a pass (seven without the fused steps)

inline unsigned grid_rows(long long n) {      // CSR traversal: kThreads rows (one per wave and 64 rows) per block and sweep
    long long g = (n + kThreads - 1) / kThreads;
    if (g > kReduceBlocks) g = kReduceBlocks;
    g = (g + kXcd - 1) / kXcd * kXcd;             // every XCD gets the same number of blocks
    return static_cast<unsigned>(g);
}

inline unsigned grid_for(long long n) {
    long long g = (n + kThreads * kU - 1) / (kThreads * kU);
    if (g > kGridMax) g = kGridMax;
    if (g < 1) g = 1;
    return static_cast<unsigned>(g);
}

}  // namespace
}  // namespace dare_hip
