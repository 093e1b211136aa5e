// Aggregation multigrid on the Cartesian diagonal view: the right preconditioner of
// BiCGStab2 that stands in for MueLu's AMG (MatrixSystem/TrilinosSolver.inl:180-246, used as
// PreCondPackage::MueLu "AMG" in test_TrilinosSolver.cpp:214-231). Included by krylov.hip.
//
// Hierarchy: each level aggregates 2x2x2 cells of the finer one (an odd extent leaves a last
// layer of one cell; a periodic axis keeps its wrap). With P the piecewise-constant
// prolongation, the coarse operator is P^T E P + beta P^T L P, where A = E + L splits each row
// into its excess E_ii = sum of the row (mass, boundary and convection terms) and the
// zero-row-sum coupling part L. beta = 1/2 corrects the known factor two by which piecewise
// constant aggregation overweights diffusive couplings (the sum of four fine faces across a
// coarse face against one coarse face of twice the width). The coarse operator is again a
// seven-point diagonal view, held in the vector type CT of the solve: FP64 for the FP64
// solve, so that M^-1 is linear to FP64 rounding and the recurrence residual tracks the true
// one as closely as without preconditioning; FP32 for the inner solve of mixed refinement,
// whose outer loop recomputes the true residual in FP64.
//
// V-cycle (a fixed linear operator, as BiCGStab needs), with W = omega / C the damped-Jacobi
// weight of each level:
//   z0 = W r (pre-smoothing from zero)                              t = r - A z0
//   rc = P^T t (the sum over each aggregate, in a fixed order)      zc = coarse cycle of rc
//   z  = z0 + P zc                                                  out = z + W (r - A z)
// Each level runs as two kernels: k_mg_down forms rc straight from r (z0 and t are formed per
// cell and never stored; the eight cells of an aggregate sit in two lanes) and k_mg_up forms out
// with z evaluated at each neighbour on the fly. The coarsest level (at most 1024 rows) runs its
// sweeps inside one work-group (taking the level above it into that work-group as well cost 38 us
// against 15 for the three launches at 19 x 16 x 16). Work is dealt so that each XCD (blocks b =
// x mod 8) owns one contiguous eighth of a level, keeping the neighbour planes of a row in that
// XCD's L2.
#pragma once

namespace dare_hip {
namespace {

constexpr int kMgMaxLevels = 12;
constexpr long long kMgCoarsestRows = 1024;

// coarse-level arrays are of the hierarchy's coarse type CT (double or float), set up by
// mg_setup<VT, XT> with CT = XT; they are typed at each use with mg_ptr<CT>
struct MgLevel {
    DiaView V{};
    long long rows = 0;
    void* D = nullptr;         // seven slots (coarse levels)
    void* W = nullptr;         // omega / C (coarse levels)
    void *r = nullptr, *z = nullptr;   // right-hand side and cycle result (coarse levels)
};
template <typename CT>
inline CT* mg_ptr(void* p) { return static_cast<CT*>(p); }

struct MgHierarchy {
    int nlev = 0;              // levels including the fine one
    MgLevel lev[kMgMaxLevels];
    void* coarse = nullptr;    // one allocation for every coarse level's arrays
    size_t coarse_bytes = 0;
    void* fine = nullptr;      // fine level: W (VT) and the cycle result (XT)
    size_t fine_bytes = 0;
    const void* D0 = nullptr;  // fine-level slots (VT) of the last set-up
    bool sym = false;          // ... which were exactly symmetric: E, N, T are not read
    double omega = 0.8;
    int coarse_sweeps = 12;
};

// Neighbour of cell p[3] through slot s (0 W, 1 S, 2 B, 4 T, 5 N, 6 E) with the diagonal
// view's presence and wrap rules (dia_column): false when the boundary edit removed it, else
// its coordinates in q.
__device__ inline bool mg_nb(const DiaView& V, const int p[3], int s, int q[3]) {
    const int d = s < 3 ? s : 6 - s;
    const int n = V.n[d];
    int c = p[d];
    if (s < 3) {
        if (c == 0 && V.rm_lo[d]) return false;
        c = (c == 0) ? n - 1 : c - 1;
    } else {
        if (c == n - 1 && V.rm_hi[d] && !(c == 0 && V.rm_lo[d])) return false;
        c = (c == n - 1) ? 0 : c + 1;
    }
    q[0] = p[0];
    q[1] = p[1];
    q[2] = p[2];
    q[d] = c;
    return true;
}
__device__ inline long long mg_row(const DiaView& V, const int q[3]) {
    return (static_cast<long long>(q[0]) * V.n[1] + q[1]) * V.n[2] + q[2];
}
__device__ inline void mg_cell(const DiaView& V, long long row, int p[3]) {
    p[2] = static_cast<int>(row % V.n[2]);
    p[1] = static_cast<int>((row / V.n[2]) % V.n[1]);
    p[0] = static_cast<int>(row / (static_cast<long long>(V.n[1]) * V.n[2]));
}
// this lane's rows of an n-row level: XCD x (blocks b = x mod 8) owns rows [n x / 8, n (x+1) / 8)
struct MgSlab {
    long long first, end, step;
};
__device__ inline MgSlab mg_slab(long long n) {
    const int xcd = static_cast<int>(blockIdx.x % kXcd);
    const long long per = gridDim.x / kXcd;
    MgSlab S;
    S.first = n * xcd / kXcd + static_cast<long long>(blockIdx.x / kXcd) * kThreads + threadIdx.x;
    S.end = n * (xcd + 1) / kXcd;
    S.step = per * kThreads;
    return S;
}

// W = omega / C of the fine level
template <typename VT>
__global__ __launch_bounds__(kThreads) void k_mg_weight(long long n, const VT* __restrict__ C, VT* __restrict__ W,
                                                       double omega) {
    const MgSlab S = mg_slab(n);
    for (long long i = S.first; i < S.end; i += S.step) W[i] = static_cast<VT>(omega / static_cast<double>(C[i]));
}

// ---- the level kernels. One lane holds the four cells (2 i x 2 j at one k) of an aggregate's
// half; the lane of the other k is its neighbour in the wave, so an aggregate's sum is three adds
// in the lane and one exchange. A wave is 2^lk lanes along k times 64 >> lk pairs of rows along j
// on one pair of planes, and XCD x (blocks b = x mod 8) owns one contiguous eighth of the tiles.
// What bounds the fine level is the slots' and vectors' bytes; before, with a lane per cell, 28
// (up) and 21 (down) loads a cell in runs of 16 k cells kept it above that. Here a run is up to 64
// cells, the four cells share their neighbours, and the seven values of zc serve all four (18 and
// 16 loads a cell). 145 x 128 x 121, FP64, four slots: down 28.8 -> 25.7 us, up 34.3 -> 27.5 (seven
// slots and 64-bit rows: down 35, up 38).
struct MgTiles {
    int lk;                    // log2 of the lanes along k
    unsigned tk, tj;           // tiles along k and along j
    long long total;
};
inline MgTiles mg_tiles(const DiaView& V) {
    // the longest run whose padding of the k extent is within 1/8 of the least, at least a pair
    const auto padded = [&](int lk) { return (static_cast<long long>(V.n[2]) + (1 << lk) - 1) >> lk << lk; };
    MgTiles T;
    T.lk = 6;
    while (T.lk > 4 && (V.n[2] <= 1 << (T.lk - 1) || 8 * padded(T.lk) > 9 * padded(4))) T.lk--;
    while (T.lk > 1 && V.n[2] <= 1 << (T.lk - 1)) T.lk--;
    const int rows = 64 >> T.lk;
    T.tk = static_cast<unsigned>(padded(T.lk) >> T.lk);
    T.tj = static_cast<unsigned>(((V.n[1] + 1) / 2 + rows - 1) / rows);
    T.total = static_cast<long long>(T.tk) * T.tj * ((V.n[0] + 1) / 2);
    return T;
}
inline unsigned mg_tile_grid(const MgTiles& T) {      // one wave per work-group, a multiple of kXcd
    const long long g = T.total < (1LL << 20) ? T.total : (1LL << 20);
    return static_cast<unsigned>((g + kXcd - 1) / kXcd * kXcd);
}
struct MgTileIter {
    long long first, end, step;
};
__device__ inline MgTileIter mg_tile_iter(const MgTiles& T) {
    const int xcd = static_cast<int>(blockIdx.x % kXcd);
    MgTileIter it;
    it.first = T.total * xcd / kXcd + blockIdx.x / kXcd;
    it.end = T.total * (xcd + 1) / kXcd;
    it.step = gridDim.x / kXcd;
    return it;
}

// Rows, in 32 bits, that a lane reads: its cells c[a][b] (plane 2I + a, row 2J + b) and their
// neighbours. A neighbour that the boundary edit removed (mg_nb) counts as the cell itself: its
// slot holds 0, so the term it feeds is +0.0 and every load can be issued unconditionally. Cells
// outside the level (an odd extent's last pair, lanes beyond the tile's end) stand on a valid cell
// and are dropped by the caller.
struct MgQuad {
    unsigned c[2][2], loI[2], hiI[2], loJ[2], hiJ[2];
    unsigned dlo, dhi;         // to the neighbours along k, added mod 2^32
    bool in, i1, j1;           // the lane's cells 0, its second plane and its second row exist
    unsigned gone;             // axes (bit d) whose removed higher neighbour the last cell would have
    int I[3];                  // aggregate
    int lo[3], hi[3];          // aggregate coordinate of the neighbours along each axis
};
__device__ inline MgQuad mg_quad(const DiaView& V, const MgTiles& T, long long w) {
    MgQuad q;
    const int lane = threadIdx.x % 64;
    const unsigned wu = static_cast<unsigned>(w);     // tiles < 2^32 (mg_setup)
    const unsigned ij = wu / T.tk;
    const unsigned ti = ij / T.tj;
    int p[3] = {2 * static_cast<int>(ti), static_cast<int>(ij - ti * T.tj) * (64 >> T.lk) + (lane >> T.lk),
                static_cast<int>(wu - ij * T.tk) << T.lk | (lane & ((1 << T.lk) - 1))};
    p[1] *= 2;
    q.in = p[1] < V.n[1] && p[2] < V.n[2];
    p[1] = p[1] < V.n[1] ? p[1] : 0;
    p[2] = p[2] < V.n[2] ? p[2] : V.n[2] - 1;
    q.i1 = p[0] + 1 < V.n[0];
    q.j1 = p[1] + 1 < V.n[1];
    const unsigned stride[3] = {static_cast<unsigned>(V.n[1]) * static_cast<unsigned>(V.n[2]),
                                static_cast<unsigned>(V.n[2]), 1u};
    const int last[3] = {p[0] + (q.i1 ? 1 : 0), p[1] + (q.j1 ? 1 : 0), p[2]};
    unsigned dlo[3], dhi[3];   // from the first cell of the axis
    q.gone = 0u;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const int n = V.n[d];
        const bool lo_gone = p[d] == 0 && V.rm_lo[d];
        const bool hi_gone = last[d] == n - 1 && V.rm_hi[d] && !(last[d] == 0 && V.rm_lo[d]);
        const int lo = lo_gone ? p[d] : p[d] == 0 ? n - 1 : p[d] - 1;
        const int hi = hi_gone ? last[d] : last[d] == n - 1 ? 0 : last[d] + 1;
        q.gone |= static_cast<unsigned>(hi_gone) << d;
        dlo[d] = static_cast<unsigned>(lo - p[d]) * stride[d];
        dhi[d] = static_cast<unsigned>(hi - p[d]) * stride[d];
        q.I[d] = p[d] >> 1;
        q.lo[d] = lo >> 1;
        q.hi[d] = hi >> 1;
    }
    const unsigned c0 = p[0] * stride[0] + p[1] * stride[1] + p[2];
    const unsigned si = q.i1 ? stride[0] : 0u, sj = q.j1 ? stride[1] : 0u;
#pragma unroll
    for (int a = 0; a < 2; a++) {
#pragma unroll
        for (int b = 0; b < 2; b++) q.c[a][b] = c0 + (a ? si : 0u) + (b ? sj : 0u);
        q.loI[a] = c0 + dlo[0] + (a ? sj : 0u);
        q.hiI[a] = c0 + dhi[0] + (a ? sj : 0u);
        q.loJ[a] = c0 + dlo[1] + (a ? si : 0u);
        q.hiJ[a] = c0 + dhi[1] + (a ? si : 0u);
    }
    q.dlo = dlo[2];
    q.dhi = dhi[2];
    return q;
}

// The slots of a lane's four cells. SYM: the view is exactly symmetric, and its E, N, T slots,
// which a fill may have left out, are read as the W, S, B slots of the neighbours.
template <bool SYM, typename Ix, typename DT>
__device__ inline void mg_slots(const DT* __restrict__ D, long long nr, const MgQuad& q, DT a[2][2][7]) {
    const auto at = [&](int s, unsigned row) { return *at_off(D + s * nr, static_cast<Ix>(row)); };
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int s = 0; s < (SYM ? 4 : 7); s++) a[i][j][s] = at(s, q.c[i][j]);
    if constexpr (SYM) {
        const DT z = static_cast<DT>(0);
#pragma unroll
        for (int m = 0; m < 2; m++) {
            const DT e = at(0, q.hiI[m]), n = at(1, q.hiJ[m]);
            a[1][m][6] = q.gone & 1u ? z : e;
            a[0][m][6] = q.i1 ? a[1][m][0] : a[1][m][6];
            a[m][1][5] = q.gone & 2u ? z : n;
            a[m][0][5] = q.j1 ? a[m][1][1] : a[m][1][5];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const DT t = at(2, q.c[m][j] + q.dhi);
                a[m][j][4] = q.gone & 4u ? z : t;
            }
        }
    }
}

// The value at a row of the operand, by what of(row, aggregate's part) gives, at the lane's cells
// and their neighbours; y(i, j) is then the row's product, in the order C W S B T N E.
struct MgPoints {
    double c[2][2], loI[2], hiI[2], loJ[2], hiJ[2], loK[2][2], hiK[2][2];
    bool i1, j1;
    template <typename DT>
    __device__ double product(const DT a[2][2][7], int i, int j) const {
        const auto f = [&](int s) { return static_cast<double>(a[i][j][s]); };
        double y = f(3) * c[i][j];
        y += f(0) * (i ? c[0][j] : loI[j]);
        y += f(1) * (j ? c[i][0] : loJ[i]);
        y += f(2) * loK[i][j];
        y += f(4) * hiK[i][j];
        y += f(5) * (j == 0 && j1 ? c[i][1] : hiJ[i]);
        y += f(6) * (i == 0 && i1 ? c[1][j] : hiI[j]);
        return y;
    }
};
// of(row, n): n is 0 for the lane's own aggregate, 1..6 for its W S B T N E neighbour
template <class F>
__device__ inline MgPoints mg_points(const MgQuad& q, const F& of) {
    MgPoints z;
    z.i1 = q.i1;
    z.j1 = q.j1;
#pragma unroll
    for (int m = 0; m < 2; m++) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            z.c[m][j] = of(q.c[m][j], 0);
            z.loK[m][j] = of(q.c[m][j] + q.dlo, 3);
            z.hiK[m][j] = of(q.c[m][j] + q.dhi, 4);
        }
        z.loI[m] = of(q.loI[m], 1);
        z.hiI[m] = of(q.hiI[m], 6);
        z.loJ[m] = of(q.loJ[m], 2);
        z.hiJ[m] = of(q.hiJ[m], 5);
    }
    return z;
}

// coarse slots and W of level l+1 from the slots of level l. On a symmetric view they are
// symmetric too: a face's coefficients are summed in the same order from both sides.
template <bool SYM, typename Ix, typename VT, typename CT>
__global__ __launch_bounds__(64) void k_mg_coarsen(DiaView Vf, MgTiles Tf, const VT* __restrict__ Df, DiaView Vc,
                                                  CT* __restrict__ Dc, CT* __restrict__ Wc, double beta, double omega) {
    const long long nrf = Vf.nrows, nrc = Vc.nrows;
    const MgTileIter it = mg_tile_iter(Tf);
    for (long long w = it.first; w < it.end; w += it.step) {
        const MgQuad q = mg_quad(Vf, Tf, w);
        VT a[2][2][7];
        mg_slots<SYM, Ix>(Df, nrf, q, a);
        double excess = 0., cpl[7] = {0., 0., 0., 0., 0., 0., 0.};
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                if (!q.in || (i && !q.i1) || (j && !q.j1)) continue;
                const bool out[7] = {i == 0 && q.lo[0] != q.I[0], j == 0 && q.lo[1] != q.I[1], q.lo[2] != q.I[2], false,
                                     q.hi[2] != q.I[2], (j || !q.j1) && q.hi[1] != q.I[1],
                                     (i || !q.i1) && q.hi[0] != q.I[0]};
                excess += static_cast<double>(a[i][j][3]);
#pragma unroll
                for (int s = 0; s < 7; s++) {
                    if (s == 3) continue;
                    const double v = static_cast<double>(a[i][j][s]);
                    excess += v;
                    if (out[s]) cpl[s] += beta * v;            // coupling to a neighbour aggregate
                }
            }
        excess += __shfl_xor(excess, 1);
        double c = excess;
#pragma unroll
        for (int s = 0; s < 7; s++)
            if (s != 3) {
                cpl[s] += __shfl_xor(cpl[s], 1);
                c -= cpl[s];
            }
        if (q.in && (threadIdx.x & 1) == 0) {
            const long long row = mg_row(Vc, q.I);
#pragma unroll
            for (int s = 0; s < 7; s++) Dc[s * nrc + row] = static_cast<CT>(s == 3 ? c : cpl[s]);
            Wc[row] = static_cast<CT>(omega / c);
        }
    }
}

// rc = P^T (r - A W r), an aggregate's eight values summed in a fixed order
template <bool SYM, typename Ix, typename DT, typename XT, typename CT>
__global__ __launch_bounds__(64) void k_mg_down(DiaView Vf, MgTiles Tf, const DT* __restrict__ Df,
                                               const DT* __restrict__ Wf, const XT* __restrict__ r, DiaView Vc,
                                               CT* __restrict__ rc) {
    const MgTileIter it = mg_tile_iter(Tf);
    for (long long w = it.first; w < it.end; w += it.step) {
        const MgQuad q = mg_quad(Vf, Tf, w);
        DT a[2][2][7];
        mg_slots<SYM, Ix>(Df, Vf.nrows, q, a);
        const MgPoints z = mg_points(q, [&](unsigned row, int) {
            return static_cast<double>(*at_off(Wf, static_cast<Ix>(row))) *
                   static_cast<double>(*at_off(r, static_cast<Ix>(row)));
        });
        double t = 0.;
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const double d = static_cast<double>(*at_off(r, static_cast<Ix>(q.c[i][j]))) - z.product(a, i, j);
                if (q.in && (!i || q.i1) && (!j || q.j1)) t += d;
            }
        t += __shfl_xor(t, 1);
        if (q.in && (threadIdx.x & 1) == 0) rc[mg_row(Vc, q.I)] = static_cast<CT>(t);
    }
}

// out = z + W (r - A z) with z = W r + P zc evaluated at each neighbour
template <bool SYM, typename Ix, typename DT, typename XT, typename CT>
__global__ __launch_bounds__(64) void k_mg_up(DiaView Vf, MgTiles Tf, const DT* __restrict__ Df,
                                             const DT* __restrict__ Wf, const XT* __restrict__ r, DiaView Vc,
                                             const CT* __restrict__ zc, XT* __restrict__ out) {
    const MgTileIter it = mg_tile_iter(Tf);
    for (long long w = it.first; w < it.end; w += it.step) {
        const MgQuad q = mg_quad(Vf, Tf, w);
        DT a[2][2][7];
        mg_slots<SYM, Ix>(Df, Vf.nrows, q, a);
        const unsigned stride[3] = {static_cast<unsigned>(Vc.n[1]) * static_cast<unsigned>(Vc.n[2]),
                                    static_cast<unsigned>(Vc.n[2]), 1u};
        const unsigned own = q.I[0] * stride[0] + q.I[1] * stride[1] + q.I[2];
        double zn[7];
        zn[0] = static_cast<double>(*at_off(zc, static_cast<Ix>(own)));
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const unsigned lo = own + static_cast<unsigned>(q.lo[d] - q.I[d]) * stride[d];
            const unsigned hi = own + static_cast<unsigned>(q.hi[d] - q.I[d]) * stride[d];
            zn[1 + d] = static_cast<double>(*at_off(zc, static_cast<Ix>(lo)));
            zn[6 - d] = static_cast<double>(*at_off(zc, static_cast<Ix>(hi)));
        }
        const MgPoints z = mg_points(q, [&](unsigned row, int n) {
            return static_cast<double>(*at_off(Wf, static_cast<Ix>(row))) *
                       static_cast<double>(*at_off(r, static_cast<Ix>(row))) +
                   zn[n];
        });
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const double wr = static_cast<double>(*at_off(Wf, static_cast<Ix>(q.c[i][j])));
                const double rr = static_cast<double>(*at_off(r, static_cast<Ix>(q.c[i][j])));
                const double o = z.c[i][j] + wr * (rr - z.product(a, i, j));
                if (q.in && (!i || q.i1) && (!j || q.j1)) out[q.c[i][j]] = static_cast<XT>(o);
            }
    }
}

// the coarsest level: z = W r, then sweeps - 1 damped-Jacobi sweeps, all in one work-group
// (rows <= 1024) with z held in LDS. A chain of sweeps bounds it: the seven reads of a row go out
// together, a removed neighbour's as the row itself times 0 (640 rows: 7.2 -> 5.6 us).
template <typename CT>
__global__ __launch_bounds__(1024) void k_mg_coarsest(DiaView V, const CT* __restrict__ D, const CT* __restrict__ W,
                                                     const CT* __restrict__ r, CT* __restrict__ z, int sweeps) {
    __shared__ CT za[kMgCoarsestRows], zb[kMgCoarsestRows];
    const long long nr = V.nrows;
    const int row = threadIdx.x;
    CT a[7] = {0, 0, 0, 0, 0, 0, 0};
    int nb[7] = {row, row, row, row, row, row, row};
    CT rv = 0, wv = 0;
    if (row < nr) {
        int p[3];
        mg_cell(V, row, p);
#pragma unroll
        for (int s = 0; s < 7; s++) {
            a[s] = D[s * nr + row];
            int q[3];
            if (s != 3 && mg_nb(V, p, s, q)) nb[s] = static_cast<int>(mg_row(V, q));
        }
        rv = r[row];
        wv = W[row];
        za[row] = wv * rv;
    }
    __syncthreads();
    CT* cur = za;
    CT* nxt = zb;
    for (int it = 1; it < sweeps; it++) {
        if (row < nr) {
            CT v[7], y = 0;
#pragma unroll
            for (int s = 0; s < 7; s++) v[s] = cur[nb[s]];
#pragma unroll
            for (int s = 0; s < 7; s++) y += a[s] * v[s];
            nxt[row] = cur[row] + wv * (rv - y);
        }
        __syncthreads();
        CT* tmp = cur;
        cur = nxt;
        nxt = tmp;
    }
    if (row < nr) z[row] = cur[row];
}

// out = x + z (x may be NULL: out = z); out may alias x
template <typename XT>
__global__ __launch_bounds__(kThreads) void k_mg_combine(long long n, const XT* x, const XT* __restrict__ z, XT* out) {
    for (long long i = blockIdx.x * (long long)kThreads + threadIdx.x; i < n; i += (long long)gridDim.x * kThreads)
        out[i] = x ? static_cast<XT>(x[i] + z[i]) : z[i];
}

inline unsigned mg_grid(long long n) {   // a multiple of kXcd (mg_slab)
    long long g = (n + kThreads - 1) / kThreads;
    if (g > 4096) g = 4096;
    g = (g + kXcd - 1) / kXcd * kXcd;
    return static_cast<unsigned>(g);
}

// f(symmetric view?, type of the row offsets) for a level
template <class F>
void mg_level(bool sym, long long rows, const F& f) {
    if (sym && rows > kWideRows) f(std::true_type{}, 0LL);
    else if (sym) f(std::true_type{}, 0u);
    else if (rows > kWideRows) f(std::false_type{}, 0LL);
    else f(std::false_type{}, 0u);
}

// Builds (or refreshes) the hierarchy of a one-component 3-D diagonal view whose level-0 slots
// D0 are of type VT; XT is the vector type of the solve and of the coarse levels.
template <typename VT, typename XT>
int mg_setup(dare_ctx* ctx, MgHierarchy* H, const DiaView& V0, const VT* D0, bool sym) {
    using CT = XT;
    if (V0.N != 1 || V0.cross) {
        set_error("the multigrid preconditioner needs a one-component operator without cross entries");
        return DARE_ERR_UNSUPPORTED;
    }
    MgLevel lv[kMgMaxLevels];
    lv[0].V = V0;
    lv[0].rows = V0.nrows;
    int nlev = 1;
    while (nlev < kMgMaxLevels && (nlev == 1 || lv[nlev - 1].rows > kMgCoarsestRows)) {
        const DiaView& F = lv[nlev - 1].V;
        DiaView C = F;
        for (int d = 0; d < 3; d++) C.n[d] = (F.n[d] + 1) / 2;
        C.nrows = static_cast<long long>(C.n[0]) * C.n[1] * C.n[2];
        if (C.nrows == F.nrows) break;
        lv[nlev].V = C;
        lv[nlev].rows = C.nrows;
        nlev++;
    }
    if (nlev < 2 || lv[nlev - 1].rows > kMgCoarsestRows) {
        set_error("multigrid needs a grid that coarsens (at least two cells along an axis) to at most 1024 rows");
        return DARE_ERR_UNSUPPORTED;
    }
    if (mg_tiles(V0).total >= (1LL << 32)) {
        set_error("grid too large for the multigrid preconditioner");
        return DARE_ERR_UNSUPPORTED;
    }
    long long need = 0;
    for (int l = 1; l < nlev; l++) need += 10 * lv[l].rows;            // 7 slots, W, r, z
    const size_t coarse_need = sizeof(CT) * static_cast<size_t>(need);
    const size_t fine_need = (sizeof(VT) + sizeof(XT)) * static_cast<size_t>(V0.nrows);
    if (H->coarse_bytes < coarse_need) {
        if (H->coarse) (void)hipFree(H->coarse);
        H->coarse = nullptr;
        H->coarse_bytes = 0;
        if (hipMalloc(&H->coarse, coarse_need) != hipSuccess) {
            (void)hipGetLastError();
            set_error("multigrid hierarchy allocation failed");
            return DARE_ERR_OOM;
        }
        H->coarse_bytes = coarse_need;
    }
    if (H->fine_bytes < fine_need) {
        if (H->fine) (void)hipFree(H->fine);
        H->fine = nullptr;
        H->fine_bytes = 0;
        if (hipMalloc(&H->fine, fine_need) != hipSuccess) {
            (void)hipGetLastError();
            set_error("multigrid work vector allocation failed");
            return DARE_ERR_OOM;
        }
        H->fine_bytes = fine_need;
    }
    CT* p = static_cast<CT*>(H->coarse);
    for (int l = 1; l < nlev; l++) {
        const long long n = lv[l].rows;
        lv[l].D = p;
        p += 7 * n;
        lv[l].W = p;
        p += n;
        lv[l].r = p;
        p += n;
        lv[l].z = p;
        p += n;
    }
    lv[0].W = H->fine;
    lv[0].z = static_cast<char*>(H->fine) + sizeof(VT) * V0.nrows;
    H->nlev = nlev;
    H->sym = sym;
    H->D0 = D0;
    for (int l = 0; l < nlev; l++) H->lev[l] = lv[l];
    hipLaunchKernelGGL((k_mg_weight<VT>), dim3(mg_grid(V0.nrows)), dim3(kThreads), 0, ctx->stream, V0.nrows,
                       D0 + 3 * V0.nrows, mg_ptr<VT>(lv[0].W), H->omega);
    // every level's kernels by the view's symmetry and the width of its row offsets
    for (int l = 0; l + 1 < nlev; l++)
        mg_level(sym, lv[l].rows, [&](auto sc, auto ix) {
            const MgTiles T = mg_tiles(lv[l].V);
            const auto run = [&](const auto* D) {
                using DT = std::remove_const_t<std::remove_pointer_t<decltype(D)>>;
                hipLaunchKernelGGL((k_mg_coarsen<decltype(sc)::value, decltype(ix), DT, CT>), dim3(mg_tile_grid(T)),
                                   dim3(64), 0, ctx->stream, lv[l].V, T, D, lv[l + 1].V, mg_ptr<CT>(lv[l + 1].D),
                                   mg_ptr<CT>(lv[l + 1].W), 0.5, H->omega);
            };
            if (l == 0) run(D0);
            else run(static_cast<const CT*>(lv[l].D));
        });
    DARE_LAUNCH_CHECK();
    return DARE_OK;
}

// z = M^-1 r on the fine level (slots of type VT, vectors XT, coarse levels of type XT, as set
// up by mg_setup<VT, XT>); returns the device vector that holds z (the hierarchy's fine result
// vector, rewritten by the next call)
template <typename VT, typename XT>
XT* mg_apply(hipStream_t sm, const MgHierarchy& H, const XT* r) {
    using CT = XT;
    const VT* D0 = static_cast<const VT*>(H.D0);
    const int L = H.nlev - 1;
    const MgLevel& F = H.lev[0];
    const VT* W0 = static_cast<const VT*>(F.W);
    // restriction from level l to l + 1, and correction of level l by l + 1
    const auto down = [&](int l, auto sc, auto ix, const auto* D, const auto* W, const XT* rl) {
        using DT = std::remove_const_t<std::remove_pointer_t<decltype(D)>>;
        const MgTiles T = mg_tiles(H.lev[l].V);
        hipLaunchKernelGGL((k_mg_down<decltype(sc)::value, decltype(ix), DT, XT, CT>), dim3(mg_tile_grid(T)), dim3(64),
                           0, sm, H.lev[l].V, T, D, W, rl, H.lev[l + 1].V, mg_ptr<CT>(H.lev[l + 1].r));
    };
    const auto up = [&](int l, auto sc, auto ix, const auto* D, const auto* W, const XT* rl) {
        using DT = std::remove_const_t<std::remove_pointer_t<decltype(D)>>;
        const MgTiles T = mg_tiles(H.lev[l].V);
        hipLaunchKernelGGL((k_mg_up<decltype(sc)::value, decltype(ix), DT, XT, CT>), dim3(mg_tile_grid(T)), dim3(64), 0,
                           sm, H.lev[l].V, T, D, W, rl, H.lev[l + 1].V, static_cast<const CT*>(H.lev[l + 1].z),
                           mg_ptr<XT>(H.lev[l].z));
    };
    const auto level = [&](int l, const auto& step) {
        const MgLevel& A = H.lev[l];
        mg_level(H.sym, A.rows, [&](auto sc, auto ix) {
            if (l == 0) step(l, sc, ix, D0, W0, r);
            else step(l, sc, ix, static_cast<const CT*>(A.D), static_cast<const CT*>(A.W), static_cast<const CT*>(A.r));
        });
    };
    const MgLevel& Z = H.lev[L];
    for (int l = 0; l < L; l++) level(l, down);
    hipLaunchKernelGGL((k_mg_coarsest<CT>), dim3(1), dim3(1024), 0, sm, Z.V, static_cast<const CT*>(Z.D),
                       static_cast<const CT*>(Z.W), static_cast<const CT*>(Z.r), mg_ptr<CT>(Z.z), H.coarse_sweeps);
    for (int l = L - 1; l >= 0; l--) level(l, up);
    return mg_ptr<XT>(F.z);
}

}  // namespace
}  // namespace dare_hip
