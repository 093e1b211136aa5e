// Field-wide FV stencils for gfx950: ghost fill, face gradient, value divergence, TVD face
// flux and the fused explicit TVD step. One work-item per internal cell; wave64 lanes run
// along the fastest (last) axis so every plane-neighbour load is a coalesced row.
// Floating-point operation order follows the reference per-cell code exactly (the file is
// built with -ffp-contract=off), so results are bit-identical to the per-cell evaluation.
#include "common.h"

namespace dare_hip {

struct FaceGeo {            // strides of the three face arrays (axis d has n[d]+1 faces)
    long long fs[3][3];
};

static FaceGeo make_face_geo(const Geo& G) {
    FaceGeo F;
    for (int ax = 0; ax < 3; ax++) {
        long long nf[3];
        for (int e = 0; e < 3; e++) nf[e] = G.n[e] + (e == ax ? 1 : 0);
        for (int d = 0; d < 3; d++) {
            long long s = 1;
            for (int e = d + 1; e < G.dim; e++) s *= nf[e];
            F.fs[ax][d] = d < G.dim ? s : 0;
        }
    }
    return F;
}

// Launch shape of the kernels for any dimension and component count: one lane per (cell,
// component), or per two of them (`each`), x along axis dim-1 with the components innermost, y along
// axis dim-2, z along axis dim-3; 64 x 4 lanes, or 32 x 8 where that saves an eighth of the
// work-groups, or 16 x 16 where that saves a quarter more (the shorter rows cost otherwise: 112^3,
// an eighth fewer of 16 lanes, face interpolation 11.2 -> 13.6 us, flux 20.9 -> 24.8). A lane per
// cell that looped over its N components made every access of a wave N doubles apart: TVD step,
// two components on 130 x 131 x 90 cells, 74 -> 47 us.
struct Launch {
    dim3 grid, block;
};

static Launch cell_launch(const Geo& G, int each = 1) {
    Launch L;
    const int ax_x = G.dim - 1, ax_y = G.dim - 2, ax_z = G.dim - 3;
    const long long nx = ceil_div(static_cast<long long>(G.n[ax_x]) * G.N, each);
    if (ax_y < 0) {
        L.block = dim3(64);
        L.grid = dim3(ceil_div(nx, 64));
        return L;
    }
    unsigned lanes = 64;
    const auto tiles = [&](unsigned l) { return static_cast<long long>(ceil_div(nx, l)) * ceil_div(G.n[ax_y], 256 / l); };
    for (unsigned l = 32; l >= 16; l /= 2)
        if (l == 32 ? 8 * tiles(l) <= 7 * tiles(lanes) : 4 * tiles(l) <= 3 * tiles(lanes)) lanes = l;
    L.block = dim3(lanes, 256 / lanes);
    L.grid = dim3(ceil_div(nx, lanes), ceil_div(G.n[ax_y], 256 / lanes), ax_z >= 0 ? G.n[ax_z] : 1);
    return L;
}

constexpr unsigned kGridYZ = 65535;      // work-groups along y and z that a launch takes
// The same for line_pairs: two entries a lane, any number of rows and planes. From kDieEntries
// entries on, the tiles of a 3-D plane (at least 28) are dealt in eight runs, one for each die
// (work-groups b = x mod 8, along the grid's x, per_xcd slots a run), so that what the next plane
// reads again comes from the die's own L2; the planes follow one another, which keeps the pages of
// the arrays few. The runs move on by a die every eight planes: their lengths differ by one tile,
// and without it 57 tiles a plane left seven dies waiting for the eighth (152^3 on arrays in turn
// 54.8 us with tiles in order, 59 with fixed runs, 53.0 now). Gradient and divergence, us, tiles in
// order and dealt: 161^3 on the same arrays 61.4 and 46.2, on arrays in turn 66.0 and 62.0; 112^3
// 21.5 and 18.6, 25.6 and 24.4; 224^3 154 and 137, 156 and 143; level from 256^3 on and below a
// million entries; 300 x 100 x 101, 25 tiles a plane, in turn 49.2 and 55.1.
constexpr long long kDieEntries = 1LL << 20;
struct PairTiles {
    unsigned tiles_x, tiles, per_xcd;
};
struct PairLaunch : Launch {
    PairTiles P{1, 0, 0};
};
static PairLaunch pair_launch(const Geo& G) {
    PairLaunch L;
    static_cast<Launch&>(L) = cell_launch(G, 2);
    const unsigned long long tiles = static_cast<unsigned long long>(L.grid.x) * L.grid.y, per = (tiles + 7) / 8;
    if (G.dim == 3 && G.ncell_int * G.N >= kDieEntries && tiles >= 28 && tiles <= (1ULL << 20)) {
        L.P = PairTiles{L.grid.x, static_cast<unsigned>(tiles), static_cast<unsigned>(per)};
        L.grid.x = 8 * L.P.per_xcd;
        L.grid.y = 1;
    }
    L.grid.y = L.grid.y < kGridYZ ? L.grid.y : kGridYZ;
    L.grid.z = L.grid.z < kGridYZ ? L.grid.z : kGridYZ;
    return L;
}

template <int DIM>
__device__ inline bool cell_coord(const Geo& G, int q[3], int& c) {
    q[0] = q[1] = q[2] = 0;
    const unsigned a = blockIdx.x * blockDim.x + threadIdx.x;
    const unsigned N = static_cast<unsigned>(G.N), k = N == 1 ? a : a / N;
    c = static_cast<int>(a - k * N);
    q[DIM - 1] = static_cast<int>(k);
    if (k >= static_cast<unsigned>(G.n[DIM - 1])) return false;
    if (DIM >= 2) {
        const int b = blockIdx.y * blockDim.y + threadIdx.y;
        if (b >= G.n[DIM - 2]) return false;
        q[DIM - 2] = b;
    }
    if (DIM == 3) q[0] = blockIdx.z;
    return true;
}

template <int DIM>
__device__ inline long long pad_ord(const Geo& G, const int q[3]) {   // internal q -> padded ordinal
    long long o = 0;
#pragma unroll
    for (int d = 0; d < DIM; d++) o += G.sl[d] * (q[d] + G.g);
    return o;
}

template <int DIM>
__device__ inline long long face_ord(const FaceGeo& F, int ax, const int q[3]) {
    long long o = 0;
#pragma unroll
    for (int d = 0; d < DIM; d++) o += F.fs[ax][d] * q[d];
    return o;
}

// Limiter Psi(r): FluxLimiter.h:41-173 with std::min/std::max as comparisons; van Leer from
// its closed form with the same NaN -> 0 convention and limits 2 / 0 at +inf / -inf.
__device__ inline double limiter(int id, double r) {
    switch (id) {
    case DARE_LIMITER_CDS: return 1.;
    case DARE_LIMITER_UPWIND: return 0.;
    case DARE_LIMITER_VANALBADA: {
        r = isnan(r) ? 0. : r;
        const double r2 = r * r;
        return (r + r2) / (1. + r2);
    }
    case DARE_LIMITER_MINMOD: {
        r = isnan(r) ? 0. : r;
        const double m = (1. < r) ? 1. : r;       // std::min(r, 1)
        return (0. < m) ? m : 0.;                 // std::max(0, m)
    }
    case DARE_LIMITER_VANLEER: {
        // branch-free: the quotient is formed for every r (inf/inf for infinite r) and the
        // special cases are selected over it, so a wave never splits and the loads of the
        // stencil can all be in flight before the first division
        const double a = fabs(r);
        double q = (r + a) / (1. + a);
        asm volatile("" : "+v"(q));   // keeps the division unconditional (not sunk into a branch)
        const double psi = isinf(r) ? (r > 0. ? 2. : 0.) : q;
        return isnan(r) ? 0. : psi;
    }
    default: return 0.;
    }
}

// Face value between L and L+1 given the four cells a = L-1, b = L, c = L+1, d = L+2
// (TVD_Cartesian.inl:133-157), times the face velocity.
__device__ inline double tvd_flux4(double a, double b, double c, double d, int lim, double u) {
    double pUU, pU, pD;
    if (u >= 0.) {
        pUU = a;
        pU = b;
        pD = c;
    } else {
        pUU = d;
        pU = c;
        pD = b;
    }
    const double r = (pU - pUU) / (pD - pU);
    const double psi = limiter(lim, r);
    return (pU + (psi * 0.5) * (pD - pU)) * u;
}

// The same for a limiter of one value psi (CDS, UPWIND), which needs L and L+1 alone.
__device__ inline double tvd_flux2(double b, double c, double psi, double u) {
    const bool up = u >= 0.;
    const double pU = up ? b : c, pD = up ? c : b;
    return (pU + (psi * 0.5) * (pD - pU)) * u;
}
constexpr bool one_psi(int lim) { return lim == DARE_LIMITER_CDS || lim == DARE_LIMITER_UPWIND; }

// ------------------------------------------------------------------------------ ghost fill
struct GhostSlabs {
    long long start[7];      // prefix offsets of the 6 slabs (W,E,S,N,B,T)
    int mode[6];
    double value[6];
};

// One lane per ghost value (slab by slab, components innermost); I: 32-bit indices where they hold
// the count, whose divisions by the extents are a fraction of the 64-bit ones (2-D 128 x 128
// periodic 3.5 -> 3.1 us, three components on 97 x 131 x 115 cells 7.5 -> 6.3).
template <int DIM, typename I>
__global__ __launch_bounds__(256) void k_ghost_fill(Geo G, GhostSlabs S, double* __restrict__ phi) {
    I r = static_cast<I>(blockIdx.x) * 256 + threadIdx.x;
    if (r >= static_cast<I>(S.start[2 * DIM] * G.N)) return;
    const I N = static_cast<I>(G.N);
    int c = 0;
    if (G.N > 1) {
        const I t = r / N;
        c = static_cast<int>(r - t * N);
        r = t;
    }
    int f = 0;
#pragma unroll
    for (int e = 1; e < 2 * DIM; e++) f = r >= static_cast<I>(S.start[e]) ? e : f;
    const int mode = S.mode[f];
    if (mode == DARE_GHOST_LEAVE) return;
    r -= static_cast<I>(S.start[f]);
    const int d = f / 2;
    const bool low = (f % 2) == 0;
    int p[3] = {0, 0, 0};       // padded index
    // decompose r over (layer, other axes) with the last other axis fastest
#pragma unroll
    for (int e = DIM - 1; e >= 0; e--) {
        if (e == d) continue;
        const I n = static_cast<I>(G.n[e]), t = r / n;
        p[e] = static_cast<int>(r - t * n) + G.g;
        r = t;
    }
    const int l = static_cast<int>(r) + 1;   // ghost layer 1..g
    const int n = G.n[d];
    const int to = low ? G.g - l : G.g + n - 1 + l;
    const int from = mode == DARE_GHOST_PERIODIC ? G.g + (low ? n - l : l - 1) : G.g + (low ? l - 1 : n - l);
    long long o = 0;
#pragma unroll
    for (int e = 0; e < DIM; e++) o += G.sl[e] * p[e];
    double* line = phi + o * G.N + c;
    const long long sd = G.sl[d] * G.N;
    const double s = line[from * sd];
    line[to * sd] = mode == DARE_GHOST_DIRICHLET ? 2. * S.value[f] - s : mode == DARE_GHOST_CONSTANT ? S.value[f] : s;
}

// Two adjacent entries (cell, component) of a line in fastest order. A line of entries is
// contiguous in phi and in every face array, whatever the components, and starts on 8 bytes.
typedef double pair2 __attribute__((ext_vector_type(2), aligned(8)));
template <int DIM>
struct LinePair {
    int q[3];          // the line's cell 0
    int e;             // first entry
    bool two, high0, high1;   // a second entry; entries in the line's last cell
};
// f(LinePair) for this lane's entries of every line it owns: one, but for grids of more than 65535
// planes or work-groups of rows
template <int DIM, bool DIES, class F>
__device__ __forceinline__ void line_pairs(const Geo& G, const PairTiles& P, F&& f) {
    const int len = G.n[DIM - 1] * G.N;
    unsigned bx = blockIdx.x, by = blockIdx.y;
    if constexpr (DIES) {
        const unsigned d = (bx + (blockIdx.z >> 3)) & 7, t = (P.tiles * d >> 3) + (bx >> 3);
        if (t >= P.tiles * (d + 1) >> 3) return;
        by = t / P.tiles_x;
        bx = t - by * P.tiles_x;
    }
    const unsigned e = 2 * (bx * blockDim.x + threadIdx.x);
    if (e >= static_cast<unsigned>(len)) return;
    LinePair<DIM> L;
    L.e = static_cast<int>(e);
    L.two = L.e + 1 < len;
    L.high0 = L.e >= len - G.N;
    L.high1 = L.two && L.e + 1 >= len - G.N;
    const int n0 = DIM == 3 ? G.n[0] : 1, n1 = DIM >= 2 ? G.n[DIM - 2] : 1;
    for (int i = blockIdx.z; i < n0; i += gridDim.z)
        for (int j = by * blockDim.y + threadIdx.y; j < n1; j += gridDim.y * blockDim.y) {
            L.q[0] = L.q[1] = L.q[2] = 0;
            if (DIM >= 2) L.q[DIM - 2] = j;
            if (DIM == 3) L.q[0] = i;
            f(L);
            if (DIES) break;
        }
}
__device__ inline pair2 ld_pair(const double* p, bool two) {
    if (two) return *reinterpret_cast<const pair2*>(p);
    return pair2{p[0], 0.};
}
template <bool NT>
__device__ inline void st_pair(double* p, pair2 v, bool two) {
    if (!two) p[0] = v.x;
    else if constexpr (NT) __builtin_nontemporal_store(v, reinterpret_cast<pair2*>(p));
    else *reinterpret_cast<pair2*>(p) = v;
}

// --------------------------------------------------------------------------- face gradient
// Gradient_Cartesian.inl:62-96: W = (phiC - phiW) dn_r, E = (phiE - phiC) dn_r, ... Bytes bound it.
// 16-byte accesses move more per instruction than one entry a lane: 97 x 131 x 115 cells of three
// components 37.9 -> 34.4 us (divergence 32.7 -> 29.5), 64^3 of three 7.5 -> 6.5 (5.5 -> 4.4),
// 1024^2 6.6 -> 5.8 (5.2 -> 4.3), level at 10^5 entries. And entries in the order of memory keep
// the pages of the four arrays few: a march along i in persistent work-groups, which re-reads
// nothing, took 277 us for gradient and divergence of 256^3 on arrays in turn, this form 194 (128^3
// 40.8 and 31.9; on one set of arrays over and over 268 and 194, 161^3 54 and 46). NT: stores past
// the caches from kStreamRows entries on (256^3 without 230; 128^3 with 26.9 against 26.7).
template <int DIM, bool NT, bool DIES>
__global__ __launch_bounds__(256) void k_grad_faces(Geo G, FaceGeo F, PairTiles P, const double* __restrict__ phi,
                                                    double* __restrict__ f0, double* __restrict__ f1,
                                                    double* __restrict__ f2) {
    double* out[3] = {f0, f1, f2};
    const int N = G.N;
    line_pairs<DIM, DIES>(G, P, [&](const LinePair<DIM>& L) {
        const double* b = phi + pad_ord<DIM>(G, L.q) * N + L.e;
        const pair2 pc = ld_pair(b, L.two);
        pair2 lo[DIM];
#pragma unroll
        for (int d = 0; d < DIM; d++) lo[d] = ld_pair(b - G.sl[d] * N, L.two);
#pragma unroll
        for (int d = 0; d < DIM; d++) {
            double* o = out[d] + face_ord<DIM>(F, d, L.q) * N + L.e;
            st_pair<NT>(o, (pc - lo[d]) * G.dnr[d], L.two);
            if (d < DIM - 1) {
                if (L.q[d] == G.n[d] - 1)
                    st_pair<NT>(o + F.fs[d][d] * N, (ld_pair(b + G.sl[d] * N, L.two) - pc) * G.dnr[d], L.two);
            } else {
                if (L.high0) o[N] = (b[N] - pc.x) * G.dnr[d];
                if (L.high1) o[N + 1] = (b[N + 1] - pc.y) * G.dnr[d];
            }
        }
    });
}

// ---------------------------------------------------------------------- value divergence
// Divergence_Cartesian.inl:211-235: A0 E - A0 W + A1 N - A1 S + A2 T - A2 B, in that order.
template <int DIM, bool NT, bool DIES>
__global__ __launch_bounds__(256) void k_div_faces(Geo G, FaceGeo F, PairTiles P, const double* __restrict__ f0,
                                                   const double* __restrict__ f1, const double* __restrict__ f2,
                                                   double* __restrict__ out) {
    const double* in[3] = {f0, f1, f2};
    const int N = G.N;
    line_pairs<DIM, DIES>(G, P, [&](const LinePair<DIM>& L) {
        pair2 lo[DIM], hi[DIM];
#pragma unroll
        for (int d = 0; d < DIM; d++) {
            const double* f = in[d] + face_ord<DIM>(F, d, L.q) * N + L.e;
            lo[d] = ld_pair(f, L.two);
            hi[d] = ld_pair(f + F.fs[d][d] * N, L.two);
        }
        pair2 v = G.A[0] * hi[0];
        v -= G.A[0] * lo[0];
#pragma unroll
        for (int d = 1; d < DIM; d++) {
            v += G.A[d] * hi[d];
            v -= G.A[d] * lo[d];
        }
        st_pair<NT>(out + pad_ord<DIM>(G, L.q) * N + L.e, v, L.two);
    });
}

// ------------------------------------------------------------ cell-centred velocity -> faces
// InterpolateToFace of a cell-centred one-component field (Interpolation_Cartesian.h:203-219,
// 298-354), as the TVD constructor evaluates it for every face (TVD_Cartesian.inl:27-38): the
// neighbour's value plus the cell's, times Divisor<2> = 0.5. Face m along axis d is shared by
// cells m-1 and m; both orders of the sum give the same bits, so each face is written once.
template <int DIM>
__global__ __launch_bounds__(256) void k_interp_faces(Geo G, FaceGeo F, const double* __restrict__ u0,
                                                      const double* __restrict__ u1, const double* __restrict__ u2,
                                                      double* __restrict__ f0, double* __restrict__ f1,
                                                      double* __restrict__ f2) {
    int q[3], c;
    if (!cell_coord<DIM>(G, q, c)) return;
    const double* in[3] = {u0, u1, u2};
    double* out[3] = {f0, f1, f2};
    const long long lp = pad_ord<DIM>(G, q);
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        const long long s = G.sl[d];
        const long long fo = face_ord<DIM>(F, d, q);
        const double uc = in[d][lp];
        double v = in[d][lp - s];
        v += uc;
        out[d][fo] = v * 0.5;
        if (q[d] == G.n[d] - 1) {
            double w = uc;
            w += in[d][lp + s];
            out[d][fo + F.fs[d][d]] = w * 0.5;
        }
    }
}

// -------------------------------------------------------------------------- TVD face flux
template <int DIM>
__global__ __launch_bounds__(256) void k_tvd_flux(Geo G, FaceGeo F, int lim, const double* __restrict__ phi,
                                                  const double* __restrict__ u0,
                                                  const double* __restrict__ u1,
                                                  const double* __restrict__ u2, double* __restrict__ f0,
                                                  double* __restrict__ f1, double* __restrict__ f2) {
    int q[3], c;
    if (!cell_coord<DIM>(G, q, c)) return;
    const double* vel[3] = {u0, u1, u2};
    double* out[3] = {f0, f1, f2};
    const int N = G.N;
    const double* b = phi + pad_ord<DIM>(G, q) * N + c;
    double p[DIM][5], ulo[DIM], uhi[DIM];       // every load first: the five cells of each axis
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        const long long s = G.sl[d] * N, fi = face_ord<DIM>(F, d, q);
#pragma unroll
        for (int m = 0; m < 5; m++) p[d][m] = b[(m - 2) * s];
        ulo[d] = vel[d][fi];
        uhi[d] = vel[d][q[d] == G.n[d] - 1 ? fi + F.fs[d][d] : fi];
    }
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        double* o = out[d] + face_ord<DIM>(F, d, q) * N + c;
        o[0] = tvd_flux4(p[d][0], p[d][1], p[d][2], p[d][3], lim, ulo[d]);
        if (q[d] == G.n[d] - 1) o[F.fs[d][d] * N] = tvd_flux4(p[d][1], p[d][2], p[d][3], p[d][4], lim, uhi[d]);
    }
}

// ------------------------------------------------------------------ fused explicit TVD step
// phi_out = phi - (dt/V) * div(phi_f * u_f); reads phi (13-point star) + 2 face velocities per
// axis, writes one value per cell.
// ONE: a limiter of one value: neither the second neighbours nor the ratio (88^3, upwind: 12.8 us
// with them).
template <int DIM, bool ONE>
__global__ __launch_bounds__(256) void k_tvd_step(Geo G, FaceGeo F, int lim, const double* __restrict__ phi,
                                                  const double* __restrict__ u0,
                                                  const double* __restrict__ u1,
                                                  const double* __restrict__ u2, double fac,
                                                  double* __restrict__ phi_out) {
    int q[3], c;
    if (!cell_coord<DIM>(G, q, c)) return;
    const double* vel[3] = {u0, u1, u2};
    const int N = G.N;
    const long long at = pad_ord<DIM>(G, q) * N + c;
    const double* b = phi + at;
    double p[DIM][5], ulo[DIM], uhi[DIM];
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        const long long s = G.sl[d] * N, fi = face_ord<DIM>(F, d, q);
#pragma unroll
        for (int m = ONE; m < 5 - ONE; m++) p[d][m] = b[(m - 2) * s];
        ulo[d] = vel[d][fi];
        uhi[d] = vel[d][fi + F.fs[d][d]];
    }
    const double psi = ONE && lim == DARE_LIMITER_CDS ? 1. : 0.;      // of ONE
    double v = 0.;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        double flo, fhi;
        if constexpr (ONE) {
            flo = tvd_flux2(p[d][1], p[d][2], psi, ulo[d]);
            fhi = tvd_flux2(p[d][2], p[d][3], psi, uhi[d]);
        } else {
            flo = tvd_flux4(p[d][0], p[d][1], p[d][2], p[d][3], lim, ulo[d]);
            fhi = tvd_flux4(p[d][1], p[d][2], p[d][3], p[d][4], lim, uhi[d]);
        }
        if (d == 0) v = G.A[0] * fhi;
        else v += G.A[d] * fhi;
        v -= G.A[d] * flo;
    }
    phi_out[at] = p[0][2] - fac * v;
}

constexpr int kStepTileK = 64, kStepXcd = 8, kStepMinPlanes = 8;

// LDS-staged march of a 64 (k) x TJ (j) tile over the planes [i0, i1) (all 64 TJ threads active,
// so the block can synchronise). The planes i-2..i+2 of phi at a cell stay in registers and the
// x-face flux at (i, i+1) is carried to the next plane as its low face. Plane i of phi is staged
// with two ghost rows and columns (rows j0-2..j0+TJ+1, columns k0-2..k0+65), each y and z face
// flux of the plane is computed once, by one lane, and shared through LDS (the face between rows
// j-1 and j by the lane of cell j; the top face row by the last wave; the right face column by
// lanes 0..TJ-1 of wave 0): (3 + 2/TJ) fluxes and five loads per cell and plane instead of five
// and fourteen. Waves 0, 1 stage the two ghost rows below the tile, waves 2, 3 the two above. NT
// streams the x-face velocities in and the result out with the non-temporal hint.
// In a tile cut by the grid's edge the lanes past the last cell take the coordinates of the
// nearest ghost cell (of phi) or face: the first two of them stage the high ghost layers and
// compute the last faces like any other lane, and none of them stores. (Such tiles used to march
// without LDS, five fluxes and fourteen loads per cell: 150 x 161 x 173, a third of whose tiles
// are cut, 57.5 -> 54.3 us.)
constexpr int kTvdRow = 68;   // staged row: 2 + 64 + 2 doubles
template <bool NT, int TJ, bool AHEAD>
__device__ __forceinline__ void tvd_march3_lds(const Geo& G, int lim, const double* __restrict__ phi,
                                               const double* __restrict__ ux, const double* __restrict__ uy,
                                               const double* __restrict__ uz, double fac, double* __restrict__ out,
                                               int k0, int j0, int i0, int i1, double* T, double* Fy, double* Fz) {
    static_assert(TJ >= 4 && TJ <= 16, "ghost rows are staged by waves 0..3, ghost columns by wave 1");
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int n1 = G.n[1], n2 = G.n[2];
    const bool own = k0 + lane < n2 && j0 + w < n1;
    // this lane's cell of phi (ghost layers n, n + 1 at most), its x face and its low y, z faces
    const auto upto = [](int v, int most) { return v < most ? v : most; };
    const int k = upto(k0 + lane, n2 + 1), j = upto(j0 + w, n1 + 1);
    const int kx = upto(k0 + lane, n2 - 1), jx = upto(j0 + w, n1 - 1);
    const int jy = upto(j0 + w, n1), kz = upto(k0 + lane, n2);
    const long long sI = G.sl[0], sJ = G.sl[1];
    long long lp = (static_cast<long long>(i0 + G.g) * G.np[1] + (j + G.g)) * G.np[2] + (k + G.g);
    const long long fxs = static_cast<long long>(n1) * n2;
    long long fx = static_cast<long long>(i0) * fxs + static_cast<long long>(jx) * n2 + kx;
    long long fy = (static_cast<long long>(i0) * (n1 + 1) + jy) * n2 + kx;
    const long long fys = static_cast<long long>(n1 + 1) * n2;
    long long fz = (static_cast<long long>(i0) * n1 + jx) * (n2 + 1) + kz;
    const long long fzs = static_cast<long long>(n1) * (n2 + 1);
    // ghost row staged by waves 0..3: j0-2, j0-1, j0+TJ, j0+TJ+1 (staged rows 0, 1, TJ+2, TJ+3)
    const bool hload = w < 4;
    const int hj = w < 2 ? w - 2 : TJ + w - 2;                  // tile-relative row
    const long long hoff = static_cast<long long>(upto(j0 + hj, n1 + 1) - j) * sJ;
    const int hrow = hj + 2;
    // ghost columns (wave 1, lanes 0..4 TJ-1): rows j0..j0+TJ-1 x columns k0-2, k0-1, k0+64, k0+65
    const int gr = lane >> 2, gq = lane & 3;
    const int gdk = gq < 2 ? gq - 2 : 62 + gq;                  // -2, -1, 64, 65
    const long long goff = static_cast<long long>(upto(j0 + gr, n1 + 1) - j) * sJ + (upto(k0 + gdk, n2 + 1) - k);
    const int gslot = (2 + gr) * kTvdRow + (gdk + 2);
    const bool gload = w == 1 && lane < 4 * TJ;
    // top face row (last wave): face j0 + TJ; right face column (wave 0, lanes 0..TJ-1): row
    // j0 + lane, face k0 + 64; both only meet cells of a tile that is full along their axis
    const long long ty_off = static_cast<long long>(upto(j0 + TJ, n1) - jy) * n2;
    const long long zx_off = static_cast<long long>(upto(j0 + lane, n1 - 1) - jx) * (n2 + 1) + (upto(k0 + 64, n2) - kz);
    double pm2 = phi[lp - 2 * sI], pm1 = phi[lp - sI], p0 = phi[lp], pp1 = phi[lp + sI];
    // the march's first flux: before the loads of its first plane for van Leer (150 x 161 x 173 53.7 us
    // after them, 52.9 before; 128^3 23.6 and 23.1), after them for the others (minmod 128^3 19.3, 19.6
    // before)
    const bool flux_first = lim == DARE_LIMITER_VANLEER;
    const double u_lo = ux[fx];
    double f_lo = flux_first ? tvd_flux4(pm2, pm1, p0, pp1, lim, u_lo) : 0.;
    const double row0 = hload ? phi[lp + hoff] : 0., col0 = gload ? phi[lp + goff] : 0.;
    const double A0 = G.A[0], A1 = G.A[1], A2 = G.A[2];
    // Plane i + 1 is staged while plane i is computed from the other buffer, and the fluxes are shared
    // through two buffers too, so a plane has one barrier. nx: what the next plane reads, and the
    // ghost rows and columns of the one after it, loaded a plane ahead (161^3, van Leer: 63.2 -> 60.6
    // us a step). The divisions of the limiter are most of what remains: the vector units are busy
    // for 60 % of the time; three blocks a CU instead of two would have to spill (73.5 us).
    constexpr int kT = (TJ + 4) * kTvdRow, kY = (TJ + 1) * 64, kZ = TJ * 65;
    const int own_slot = (2 + w) * kTvdRow + 2 + lane, row_slot = hrow * kTvdRow + 2 + lane;
    double nx[8];
    const auto load = [&](long long at, long long ax, long long ay, long long az) {
        nx[0] = phi[at + 2 * sI];
        if constexpr (NT) nx[1] = ld_nt(ux + ax + fxs);
        else nx[1] = ux[ax + fxs];
        nx[2] = uy[ay];
        nx[3] = uz[az];
        nx[4] = w == TJ - 1 ? uy[ay + ty_off] : 0.;
        nx[5] = (w == 0 && lane < TJ) ? uz[az + zx_off] : 0.;
        nx[6] = hload ? phi[at + sI + hoff] : 0.;
        nx[7] = gload ? phi[at + sI + goff] : 0.;
    };
    if constexpr (AHEAD) load(lp, fx, fy, fz);
    T[own_slot] = p0;
    if (hload) T[row_slot] = row0;
    if (gload) T[gslot] = col0;
    if (!flux_first) f_lo = tvd_flux4(pm2, pm1, p0, pp1, lim, u_lo);
    __syncthreads();
    for (int i = i0; i < i1; i++) {
        const int buf = (i - i0) & 1;
        if constexpr (!AHEAD) load(lp, fx, fy, fz);
        const double pp2 = nx[0], u_hi = nx[1], vy = nx[2], wz = nx[3], vyt = nx[4], wzr = nx[5];
        double* Tn = T + (buf ? 0 : kT);
        Tn[own_slot] = pp1;
        if (hload) Tn[row_slot] = nx[6];
        if (gload) Tn[gslot] = nx[7];
        if (AHEAD && i + 1 < i1) load(lp + sI, fx + fxs, fy + fys, fz + fzs);
        const double* Ti = T + (buf ? kT : 0);
        double* Y = Fy + (buf ? kY : 0);
        double* Z = Fz + (buf ? kZ : 0);
        const double f_hi = tvd_flux4(pm1, p0, pp1, pp2, lim, u_hi);
        const double* Tc = Ti + w * kTvdRow + 2 + lane;            // column k, rows j-2 ..
        const double gy_lo = tvd_flux4(Tc[0], Tc[kTvdRow], Tc[2 * kTvdRow], Tc[3 * kTvdRow], lim, vy);
        const double* Tr = Ti + (2 + w) * kTvdRow + lane;          // row j, columns k-2 ..
        const double hz_lo = tvd_flux4(Tr[0], Tr[1], Tr[2], Tr[3], lim, wz);
        Y[w * 64 + lane] = gy_lo;
        Z[w * 65 + lane] = hz_lo;
        if (w == TJ - 1) {                                        // top face row j0+TJ
            const double* Tt = Ti + TJ * kTvdRow + 2 + lane;
            Y[TJ * 64 + lane] = tvd_flux4(Tt[0], Tt[kTvdRow], Tt[2 * kTvdRow], Tt[3 * kTvdRow], lim, vyt);
        }
        if (w == 0 && lane < TJ) {                                // right face column k0+64
            const double* Te = Ti + (2 + lane) * kTvdRow + 64;
            Z[lane * 65 + 64] = tvd_flux4(Te[0], Te[1], Te[2], Te[3], lim, wzr);
        }
        __syncthreads();
        const double gy_hi = Y[(w + 1) * 64 + lane];
        const double hz_hi = Z[w * 65 + lane + 1];
        double v = A0 * f_hi;
        v -= A0 * f_lo;
        v += A1 * gy_hi;
        v -= A1 * gy_lo;
        v += A2 * hz_hi;
        v -= A2 * hz_lo;
        if (own) put<NT>(out + lp, p0 - fac * v);
        pm2 = pm1;
        pm1 = p0;
        p0 = pp1;
        pp1 = pp2;
        f_lo = f_hi;
        lp += sI;
        fx += fxs;
        fy += fys;
        fz += fzs;
    }
}

// 3-D, one component, persistent and balanced TVD step over 64 (k) x kStepTvdJ (j) tiles.
// Logical block L takes the column-plane range [L*chunk, (L+1)*chunk): columns ordered k-tile
// fastest, planes along i; blocks are dealt XCD by XCD (blocks b = x mod 8 own a contiguous run). The limiter is a template parameter so that each instantiation carries only its
// own branch.
constexpr int kStepTvdJ = 8;
template <bool NT, int LIM, bool AHEAD>
__global__ __launch_bounds__(64 * kStepTvdJ) void k_tvd_step3(Geo G, const double* __restrict__ phi,
                                                              const double* __restrict__ ux,
                                                              const double* __restrict__ uy,
                                                              const double* __restrict__ uz, double fac,
                                                              double* __restrict__ out, int tiles_k, long long total,
                                                              long long chunk, int per_xcd) {
    __shared__ double T[2 * (kStepTvdJ + 4) * kTvdRow];
    __shared__ double Fy[2 * (kStepTvdJ + 1) * 64];
    __shared__ double Fz[2 * kStepTvdJ * 65];
    const long long L = static_cast<long long>(blockIdx.x % kStepXcd) * per_xcd + blockIdx.x / kStepXcd;
    const int n0 = G.n[0];
    long long c = L * chunk;
    const long long cend = (c + chunk < total) ? c + chunk : total;
    while (c < cend) {
        const long long col = c / n0;
        const int i0 = static_cast<int>(c - col * n0);
        const int i1 = (cend - c < n0 - i0) ? i0 + static_cast<int>(cend - c) : n0;
        const int k0 = static_cast<int>(col % tiles_k) * kStepTileK;
        const int j0 = static_cast<int>(col / tiles_k) * kStepTvdJ;
        tvd_march3_lds<NT, kStepTvdJ, AHEAD>(G, LIM, phi, ux, uy, uz, fac, out, k0, j0, i0, i1, T, Fy, Fz);
        c += i1 - i0;
    }
}

__global__ void k_fill(double* __restrict__ p, long long n, double v) {
    const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Read + write stream, the attainable-bandwidth probe of the measurements: each lane reads R
// 16-byte chunks (non-temporal, all in flight before the store) and writes their sum, one
// 16-byte chunk; a work-group covers 256 consecutive chunks per read, so every access is
// coalesced. R = 1 is a copy; larger R gives the read-heavy mixes of the solver kernels
// (the FP64 SpMV moves 9 bytes read per byte written).
typedef double dvec2 __attribute__((ext_vector_type(2)));
// LAYOUT 0: XCD x (blocks b = x mod 8) owns one contiguous eighth of the chunks and each chunk
// reads R consecutive 4 KiB pieces of src; 1: the same pieces with the grid striding over all
// chunks; 2: XCD slabs, piece u of a chunk read from the u-th of R separate arrays (src + u *
// n_dst: the per-slot arrays of the diagonal view); 3: layout 2 read-only, each lane adding its
// chunks' sums and writing the total once, to dst[block * 256 + lane].
template <int R, int LAYOUT>
__global__ __launch_bounds__(256) void k_stream_probe(const dvec2* __restrict__ src, dvec2* __restrict__ dst,
                                                      long long n2_dst) {
    const long long nblk = n2_dst / 256;
    long long b0 = blockIdx.x, b1 = nblk, step = gridDim.x;
    if (LAYOUT != 1) {
        const int xcd = static_cast<int>(blockIdx.x % 8);
        b0 = nblk * xcd / 8 + blockIdx.x / 8;
        b1 = nblk * (xcd + 1) / 8;
        step = gridDim.x / 8;
    }
    dvec2 total = {0., 0.};
    for (long long blk = b0; blk < b1; blk += step) {
        const long long j = blk * 256 + threadIdx.x;
        dvec2 v[R];
#pragma unroll
        for (int u = 0; u < R; u++)
            v[u] = __builtin_nontemporal_load(LAYOUT >= 2 ? src + u * n2_dst + j : src + (blk * R + u) * 256 + threadIdx.x);
        dvec2 sum = v[0];
#pragma unroll
        for (int u = 1; u < R; u++) sum += v[u];
        if (LAYOUT == 3) total += sum;
        else __builtin_nontemporal_store(sum, dst + j);
    }
    if (LAYOUT == 3) dst[static_cast<long long>(blockIdx.x) * 256 + threadIdx.x] = total;
}

template <int DIM>
__global__ __launch_bounds__(256) void k_copy_to_field(Geo G, const double* __restrict__ x, double* __restrict__ phi) {
    int q[3], c;
    if (!cell_coord<DIM>(G, q, c)) return;
    long long nd = 0;
#pragma unroll
    for (int d = 0; d < DIM; d++) nd += G.si[d] * q[d];
    phi[pad_ord<DIM>(G, q) * G.N + c] = x[nd * G.N + c];
}

// Cells from which the 3-D one-component TVD step marches along i in persistent work-groups. Below,
// a launch of one lane per cell is over before a march of eight planes (its shortest): van Leer
// 24^3 10.6 us marched, 4.6 not; 64^3 14.6 and 6.7; 96^3 22.8 and 17.5; level at 1.3 M cells;
// 150 x 161 x 173 50 and 66.
constexpr long long kMarchCells = 1LL << 20;

// Balanced persistent schedule of the 3-D marching kernels: as many of their work-groups (512
// threads for the TVD step) as stay resident at once (per_cu, queried once per kernel), each with at
// least kStepMinPlanes planes.
struct MarchPlan {
    int tiles_k, per_xcd;
    long long total, chunk;
    unsigned grid;
};

inline MarchPlan march_plan(const dare_ctx* ctx, const Geo& G, int per_cu, int tile_j) {
    MarchPlan P;
    P.tiles_k = static_cast<int>(ceil_div(G.n[2], kStepTileK));
    P.total = static_cast<long long>(P.tiles_k) * ceil_div(G.n[1], tile_j) * G.n[0];
    long long nb = static_cast<long long>(ctx->num_cu) * per_cu;
    const long long by_work = ceil_div(P.total, kStepMinPlanes);
    if (nb > by_work) nb = by_work;
    P.per_xcd = static_cast<int>(ceil_div(nb, kStepXcd));
    P.chunk = ceil_div(P.total, static_cast<long long>(P.per_xcd) * kStepXcd);
    P.grid = static_cast<unsigned>(kStepXcd * P.per_xcd);
    return P;
}

template <class K>
int resident_per_cu(K kernel, int threads = 256) {
    int n = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, 0);
    return (e == hipSuccess && n > 0) ? n : 2;
}

// A short march of a limiter without divisions has nothing to hide the loads of the next plane
// behind, and the extra ones before its first plane cost it: 128^3, upwind, 8 planes 16.9 us with
// them, 16.2 without; 200^3, 32 planes 70.9 and 74.0. Minmod has one division and no special cases:
// where it streams, loads ahead only fill the memory's queues (arrays in turn, 256^3 150-154 us with
// them, 147-150 without; 200^3 88.5 and 87; level below), and so does the third work-group a CU that
// fits without them (256^3 174).
constexpr long long kShortMarch = 12;
template <bool NT, int LIM>
void launch_step3(dare_ctx* ctx, const Geo& G, const double* phi, const double* ux, const double* uy,
                  const double* uz, double fac, double* out) {
    const auto run = [&](auto ahead, const MarchPlan& P) {
        hipLaunchKernelGGL((k_tvd_step3<NT, LIM, decltype(ahead)::value>), dim3(P.grid), dim3(64 * kStepTvdJ), 0,
                           ctx->stream, G, phi, ux, uy, uz, fac, out, P.tiles_k, P.total, P.chunk, P.per_xcd);
    };
    constexpr bool kAhead = !(NT && LIM == DARE_LIMITER_MINMOD);
    static const int fit = resident_per_cu(k_tvd_step3<NT, LIM, kAhead>, 64 * kStepTvdJ);
    const int per_cu = kAhead || fit < 2 ? fit : 2;
    const MarchPlan P = march_plan(ctx, G, per_cu, kStepTvdJ);
    if constexpr (!NT && one_psi(LIM)) {
        if (P.chunk <= kShortMarch) {
            run(std::false_type{}, P);
            return;
        }
    }
    run(std::integral_constant<bool, kAhead>{}, P);
}

template <bool NT>
void launch_step3_lim(dare_ctx* ctx, const Geo& G, int lim, const double* phi, const double* ux,
                      const double* uy, const double* uz, double fac, double* out) {
    switch (lim) {
    case DARE_LIMITER_CDS: launch_step3<NT, DARE_LIMITER_CDS>(ctx, G, phi, ux, uy, uz, fac, out); break;
    case DARE_LIMITER_UPWIND: launch_step3<NT, DARE_LIMITER_UPWIND>(ctx, G, phi, ux, uy, uz, fac, out); break;
    case DARE_LIMITER_VANALBADA: launch_step3<NT, DARE_LIMITER_VANALBADA>(ctx, G, phi, ux, uy, uz, fac, out); break;
    case DARE_LIMITER_MINMOD: launch_step3<NT, DARE_LIMITER_MINMOD>(ctx, G, phi, ux, uy, uz, fac, out); break;
    default: launch_step3<NT, DARE_LIMITER_VANLEER>(ctx, G, phi, ux, uy, uz, fac, out); break;
    }
}

#define DARE_DISPATCH_DIM(G, KERNEL, L, ...)                                                       \
    do {                                                                                         \
        switch ((G).dim) {                                                                       \
        case 1: hipLaunchKernelGGL(KERNEL<1>, (L).grid, (L).block, 0, ctx->stream, __VA_ARGS__); break; \
        case 2: hipLaunchKernelGGL(KERNEL<2>, (L).grid, (L).block, 0, ctx->stream, __VA_ARGS__); break; \
        default: hipLaunchKernelGGL(KERNEL<3>, (L).grid, (L).block, 0, ctx->stream, __VA_ARGS__); break; \
        }                                                                                        \
    } while (0)

// a kernel over line pairs: by dimension, streaming stores, planes dealt to the dies
template <class F>
void dispatch_pairs(const Geo& G, const PairLaunch& L, F&& f) {
    using D1 = std::integral_constant<int, 1>;
    using D2 = std::integral_constant<int, 2>;
    using D3 = std::integral_constant<int, 3>;
    using Yes = std::true_type;
    using No = std::false_type;
    const auto nt = [&](auto dim, auto dies) {
        if (G.ncell_int * G.N >= kStreamRows) f(dim, Yes{}, dies);
        else f(dim, No{}, dies);
    };
    if (G.dim == 1) nt(D1{}, No{});
    else if (G.dim == 2) nt(D2{}, No{});
    else if (L.P.per_xcd) nt(D3{}, Yes{});
    else nt(D3{}, No{});
}

}  // namespace dare_hip

using namespace dare_hip;

extern "C" {

int dare_fill_f64(dare_ctx* ctx, double* p, int64_t n, double v) {
    DARE_CHECK_ARG(ctx && (p || n == 0) && n >= 0, "invalid fill arguments");
    if (n == 0) return DARE_OK;
    hipLaunchKernelGGL(k_fill, dim3(ceil_div(n, 256)), dim3(256), 0, ctx->stream, p, static_cast<long long>(n), v);
    DARE_LAUNCH_CHECK();
    return DARE_OK;
}

int dare_stream_probe(dare_ctx* ctx, int64_t n_dst, const double* src, double* dst, int32_t ratio, int32_t grid,
                      int32_t layout) {
    DARE_CHECK_ARG(ctx && src && dst && n_dst >= 0 && n_dst % 512 == 0,
                   "invalid stream-probe arguments (n_dst a multiple of 512)");
    DARE_CHECK_ARG(ratio == 1 || ratio == 2 || ratio == 4 || ratio == 8, "ratio must be 1, 2, 4 or 8");
    DARE_CHECK_ARG(layout >= 0 && layout <= 3,
                   "layout must be 0 (XCD slabs), 1 (grid stride), 2 (separate arrays) or 3 (read-only)");
    DARE_CHECK_ARG((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) % 16 == 0,
                   "stream probe needs 16-byte aligned vectors");
    if (n_dst == 0) return DARE_OK;
    const long long n2 = n_dst / 2;
    long long gr = grid > 0 ? grid : 8 * ctx->num_cu;
    if (gr > n2 / 256) gr = n2 / 256;
    if (layout != 1) gr = (gr + 7) / 8 * 8;
    DARE_CHECK_ARG(layout != 3 || 512 * gr <= n_dst, "read-only probe: dst holds 512 doubles per work-group");
    const dim3 g(static_cast<unsigned>(gr)), b(256);
    const dvec2* s2 = reinterpret_cast<const dvec2*>(src);
    dvec2* d2 = reinterpret_cast<dvec2*>(dst);
#define DARE_PROBE(R)                                                                                   \
    if (layout == 0) hipLaunchKernelGGL((k_stream_probe<R, 0>), g, b, 0, ctx->stream, s2, d2, n2);     \
    else if (layout == 1) hipLaunchKernelGGL((k_stream_probe<R, 1>), g, b, 0, ctx->stream, s2, d2, n2); \
    else if (layout == 2) hipLaunchKernelGGL((k_stream_probe<R, 2>), g, b, 0, ctx->stream, s2, d2, n2); \
    else hipLaunchKernelGGL((k_stream_probe<R, 3>), g, b, 0, ctx->stream, s2, d2, n2);
    switch (ratio) {
    case 1: DARE_PROBE(1) break;
    case 2: DARE_PROBE(2) break;
    case 4: DARE_PROBE(4) break;
    default: DARE_PROBE(8) break;
    }
#undef DARE_PROBE
    DARE_LAUNCH_CHECK();
    return DARE_OK;
}

int dare_ghost_fill(dare_ctx* ctx, const dare_grid* g, const int32_t* mode6, const double* value6,
                    double* phi) {
    DARE_CHECK_ARG(ctx && g && mode6 && phi, "NULL argument");
    Geo G;
    int rc = make_geo(g, &G);
    if (rc) return rc;
    GhostSlabs S;
    S.start[0] = 0;
    for (int f = 0; f < 6; f++) {
        const int d = f / 2;
        S.mode[f] = f < 2 * G.dim ? mode6[f] : DARE_GHOST_LEAVE;
        S.value[f] = value6 ? value6[f] : 0.;
        DARE_CHECK_ARG(S.mode[f] >= 0 && S.mode[f] <= DARE_GHOST_CONSTANT, "invalid ghost mode");
        DARE_CHECK_ARG(!(S.mode[f] == DARE_GHOST_PERIODIC && !G.per[d]), "periodic ghost fill on a non-periodic axis");
        long long cnt = 0;
        if (f < 2 * G.dim) {
            cnt = G.g;
            for (int e = 0; e < G.dim; e++)
                if (e != d) cnt *= G.n[e];
        }
        S.start[f + 1] = S.start[f] + cnt;
    }
    const long long total = S.start[2 * G.dim] * G.N;
    if (total == 0) return DARE_OK;
    const dim3 grid(ceil_div(total, 256)), block(256);
    const auto launch = [&](auto index) {
        using I = decltype(index);
        switch (G.dim) {
        case 1: hipLaunchKernelGGL((k_ghost_fill<1, I>), grid, block, 0, ctx->stream, G, S, phi); break;
        case 2: hipLaunchKernelGGL((k_ghost_fill<2, I>), grid, block, 0, ctx->stream, G, S, phi); break;
        default: hipLaunchKernelGGL((k_ghost_fill<3, I>), grid, block, 0, ctx->stream, G, S, phi); break;
        }
    };
    if (total < (1LL << 31)) launch(0u);
    else launch(0ULL);
    DARE_LAUNCH_CHECK();
    return DARE_OK;
}

int dare_grad_faces(dare_ctx* ctx, const dare_grid* g, const double* phi, double* fx, double* fy,
                    double* fz) {
    DARE_CHECK_ARG(ctx && g && phi && fx, "NULL argument");
    Geo G;
    int rc = make_geo(g, &G);
    if (rc) return rc;
    DARE_CHECK_ARG(G.g >= 1, "face gradient needs >= 1 ghost layer");
    DARE_CHECK_ARG(G.dim < 2 || fy, "fy is NULL");
    DARE_CHECK_ARG(G.dim < 3 || fz, "fz is NULL");
    const FaceGeo F = make_face_geo(G);
    const PairLaunch L = pair_launch(G);
    dispatch_pairs(G, L, [&](auto dim, auto nt, auto dies) {
        hipLaunchKernelGGL((k_grad_faces<decltype(dim)::value, decltype(nt)::value, decltype(dies)::value>), L.grid, L.block, 0,
                           ctx->stream, G, F, L.P, phi, fx, fy, fz);
    });
    DARE_LAUNCH_CHECK();
    return DARE_OK;
}

int dare_interpolate_to_faces(dare_ctx* ctx, const dare_grid* g, const double* ux, const double* uy,
                              const double* uz, double* fx, double* fy, double* fz) {
    DARE_CHECK_ARG(ctx && g && ux && fx, "NULL argument");
    dare_grid g1 = *g;
    g1.ncomp = 1;              // velocity fields carry one component
    Geo G;
    int rc = make_geo(&g1, &G);
    if (rc) return rc;
    DARE_CHECK_ARG(G.g >= 1, "face interpolation needs >= 1 ghost layer");
    DARE_CHECK_ARG(G.dim < 2 || (uy && fy), "y arrays are NULL");
    DARE_CHECK_ARG(G.dim < 3 || (uz && fz), "z arrays are NULL");
    const FaceGeo F = make_face_geo(G);
    const Launch L = cell_launch(G);
    DARE_DISPATCH_DIM(G, k_interp_faces, L, G, F, ux, uy, uz, fx, fy, fz);
    DARE_LAUNCH_CHECK();
    return DARE_OK;
}

int dare_div_faces(dare_ctx* ctx, const dare_grid* g, const double* fx, const double* fy,
                   const double* fz, double* out) {
    DARE_CHECK_ARG(ctx && g && fx && out, "NULL argument");
    Geo G;
    int rc = make_geo(g, &G);
    if (rc) return rc;
    DARE_CHECK_ARG(G.dim < 2 || fy, "fy is NULL");
    DARE_CHECK_ARG(G.dim < 3 || fz, "fz is NULL");
    const FaceGeo F = make_face_geo(G);
    const PairLaunch L = pair_launch(G);
    dispatch_pairs(G, L, [&](auto dim, auto nt, auto dies) {
        hipLaunchKernelGGL((k_div_faces<decltype(dim)::value, decltype(nt)::value, decltype(dies)::value>), L.grid, L.block, 0,
                           ctx->stream, G, F, L.P, fx, fy, fz, out);
    });
    DARE_LAUNCH_CHECK();
    return DARE_OK;
}

int dare_tvd_face_flux(dare_ctx* ctx, const dare_grid* g, int32_t limiter, const double* phi,
                       const double* ux, const double* uy, const double* uz, double* fx,
                       double* fy, double* fz) {
    DARE_CHECK_ARG(ctx && g && phi && ux && fx, "NULL argument");
    Geo G;
    int rc = make_geo(g, &G);
    if (rc) return rc;
    DARE_CHECK_ARG(G.g >= 2, "TVD needs >= 2 ghost layers");
    DARE_CHECK_ARG(limiter >= 0 && limiter <= DARE_LIMITER_VANLEER, "unknown limiter");
    DARE_CHECK_ARG(G.dim < 2 || (uy && fy), "y arrays are NULL");
    DARE_CHECK_ARG(G.dim < 3 || (uz && fz), "z arrays are NULL");
    const FaceGeo F = make_face_geo(G);
    const Launch L = cell_launch(G);
    DARE_DISPATCH_DIM(G, k_tvd_flux, L, G, F, limiter, phi, ux, uy, uz, fx, fy, fz);
    DARE_LAUNCH_CHECK();
    return DARE_OK;
}

int dare_tvd_explicit_step(dare_ctx* ctx, const dare_grid* g, int32_t limiter, const double* phi,
                           const double* ux, const double* uy, const double* uz, double dt,
                           double* phi_out) {
    DARE_CHECK_ARG(ctx && g && phi && ux && phi_out && phi != phi_out, "invalid arguments");
    Geo G;
    int rc = make_geo(g, &G);
    if (rc) return rc;
    DARE_CHECK_ARG(G.g >= 2, "TVD needs >= 2 ghost layers");
    DARE_CHECK_ARG(limiter >= 0 && limiter <= DARE_LIMITER_VANLEER, "unknown limiter");
    DARE_CHECK_ARG(G.dim < 2 || uy, "uy is NULL");
    DARE_CHECK_ARG(G.dim < 3 || uz, "uz is NULL");
    const FaceGeo F = make_face_geo(G);
    const Launch L = cell_launch(G);
    const double fac = dt / G.V;
    // (the march takes any number of rows and planes)
    const bool march = G.ncell_int >= kMarchCells || L.grid.y > kGridYZ || L.grid.z > kGridYZ;
    if (G.dim == 3 && G.N == 1 && march) {
        if (G.ncell_int >= kStreamRows) launch_step3_lim<true>(ctx, G, limiter, phi, ux, uy, uz, fac, phi_out);
        else launch_step3_lim<false>(ctx, G, limiter, phi, ux, uy, uz, fac, phi_out);
        DARE_LAUNCH_CHECK();
        return DARE_OK;
    }
    const auto step = [&](auto dim, auto one) {
        hipLaunchKernelGGL((k_tvd_step<decltype(dim)::value, decltype(one)::value>), L.grid, L.block, 0, ctx->stream, G, F,
                           limiter, phi, ux, uy, uz, fac, phi_out);
    };
    const auto by_dim = [&](auto one) {
        if (G.dim == 1) step(std::integral_constant<int, 1>{}, one);
        else if (G.dim == 2) step(std::integral_constant<int, 2>{}, one);
        else step(std::integral_constant<int, 3>{}, one);
    };
    if (one_psi(limiter)) by_dim(std::true_type{});
    else by_dim(std::false_type{});
    DARE_LAUNCH_CHECK();
    return DARE_OK;
}

int dare_copy_to_field(dare_ctx* ctx, const dare_grid* g, const double* x, double* phi) {
    DARE_CHECK_ARG(ctx && g && x && phi, "NULL argument");
    Geo G;
    int rc = make_geo(g, &G);
    if (rc) return rc;
    const Launch L = cell_launch(G);
    DARE_DISPATCH_DIM(G, k_copy_to_field, L, G, x, phi);
    DARE_LAUNCH_CHECK();
    return DARE_OK;
}

}  // extern "C"
