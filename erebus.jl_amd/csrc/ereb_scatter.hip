// ereb_scatter.hip -- step 2 of the transfer pipeline: the bilinear
// marker->node scatter onto the basic, Vx, Vy and P grids
// (marker_to_{basic,vx,vy,p}_nodes!, E:1605-1863, loop E:6419-6517).  Step 1,
// the marker properties (compute_marker_properties!, E:700-750), is evaluated
// in storage order by the sort's key pass (k_fine_count in ereb_sort.hip),
// where the property vectors are written with coalesced stores; the scatter
// reads them through the sort order.
//
// Geometry of the reduction:
//   - A marker's four stencils follow from two cells: basic (ib, jb) and
//     P (ip, jp); Vx uses (ip, jb), Vy uses (ib, jp), because the staggered
//     axes (C:40-64) and clamps (C:66-101) coincide that way.  The pair
//     (ip-ib, jp-jb) is in {0,1}^2, so a marker's "fine cell" (a quarter of
//     its basic cell) fixes all 16 nodes it touches, and every marker of a
//     tile of TILE x TILE basic cells lands in a (TILE+2)^2 = 64-node window
//     of each grid.
//   - Markers arrive sorted by fine key (ereb_sort.hip): a tile's markers are
//     contiguous and grouped by fine cell in ascending marker index.
//
// One workgroup per tile.  The sums of one fine cell are a contraction over
// its markers: (corner weights)^T x (property values), 4 corners by up to 10
// values for each of the four grids.  They run on the FP64 matrix cores
// (v_mfma_f64_4x4x4_4b: four independent 4x4x4 products an instruction, each
// element the chain of fmas over its k in ascending order): the four blocks b
// are four fine cells, k four markers of a block's fine cell, the rows the four
// corners and the columns four property values.
//   Lane l of the operands: t = l & 3, block b = l >> 2 & 3, k = l >> 4 (A row
// t, B column t); lane l of the result: column l & 3, block l >> 2 & 3, row
// l >> 4.
//   The four blocks are four fine cells on top of each other, whose markers are
// one run of the sort order; a wavefront walks its four fine rows across a
// segment of fine columns, its markers in groups of up to four a block (a fine
// column has as many groups as its fullest cell needs).  A chunk is four
// consecutive groups, of one fine column or of several: lane t of a quad loads
// the values of its block's k-th marker of group t (neighbouring lanes take
// neighbouring markers, so a load's lanes read the few cache lines of the
// cells' marker columns), a 4x4 transpose inside each quad of lanes turns them
// into the products' B operands (no marker value goes through LDS), and the
// marker's four stencil fractions reach the A operands by quad broadcasts.  The
// next chunk's values are loaded before this chunk's products, the marker
// numbers of the one after that too; no barrier separates the chunks.
//   The blocks lie on top of each other because a cache line holds 16 markers of
// one marker column: with the blocks side by side, walking down, every line was
// fetched five times (15 against 3.5 million L2 requests at 2.8M markers, 215
// against 150 us).  Staging the values in LDS with the sums in vector
// instructions, two barriers a chunk, took 173 us (2.8M markers, Float64; mixed
// form 131) and 1,426 us (20M, 16 markers a fine cell); this takes 134 (110) and
// 604 us, 3.5 TB/s of the 160 algorithmic bytes a marker at 2.8M.  What bounds
// it: about half vector and matrix issue (timed with the loads left out 98 us),
// half the loads' latency, three wavefronts a SIMD (five in the mixed form).
//   Row q of A and of the result: node column parity q >> 1, node row side
// q & 1.  The parity, not left/right, so that the node column shared by two
// neighbouring grid cells stays in its accumulator lanes: walking on, a
// finished grid cell's left node column is complete for these rows; its lanes
// are written to LDS and cleared, and become the next right node column.
//   At the end the workgroup adds, per window node and value, the at most four
// fine rows (two where a pair of fine rows was added in registers) and two
// column segments that touch it, in a fixed order.
// No atomics: every sum has exactly one owner and a fixed order, so results
// are identical run to run.  Tile windows overlap by two node rows/columns;
// k_combine adds the at most 2 x 2 window partials of each node in a fixed
// tile order.  Sums accumulate with fused multiply-add, which changes the
// rounding of the sequential sums only.
#include <cmath>
#include <type_traits>

#include "ereb_internal.h"

namespace ereb {

constexpr int NSEG = 2;              // column segments of a tile, a wavefront each per 4 fine rows
constexpr int SEGC = FINE / NSEG;    // fine columns of a segment (even)
constexpr int NRB = FINE / 4;        // wavefronts on top of each other (4 fine rows each)
constexpr int SCAT_NW = NSEG * NRB;  // wavefronts of a workgroup
// wavefronts a SIMD whose registers fit (no spills: a spilled value's reload
// waits for every load in flight)
constexpr int scat_waves(bool mixed, bool typed) {
    return typed && mixed ? 5 : 4;
}
static_assert(SEGC % 2 == 0 && FINE % 4 == 0, "segment shape");

// Quads of property values (B operands):
//   N1 etatotal etavp sxy -(1)   N2 rhototal ktotal etafkphi phi
//   N3 sxx tkrhocp rhocptotal hrtotal
// typed markers (ScatterArgs::typed): I, the indicators of the three types;
// the seven type-derived values' sums and the weight sum are combinations of
// the three indicators' sums.  Otherwise
//   T1 tens frict 1/G cohes      T2 rhof alphas alphaf 1
// Accumulator a (one double a lane) sums quad QUAD[a] on grid GRID[a]; column
// j is slot SLOT[a] >> 4 j & 15 of that grid's sums in LDS (15: none).  The
// slots are the SUM order without the typed values, then the three
// indicators; for untyped markers the SUM order.
enum { N1 = 0, N2, N3, T1, T2, I = T1 };
template <bool TYPED> struct Plan;
template <> struct Plan<true> {
    static constexpr int nquad = 4, nacc = 9;
    static constexpr int nsum[4] = {6, 7, 7, 9};
    static constexpr int GRID[nacc] = {0, 0, 1, 1, 2, 2, 3, 3, 3};
    static constexpr int QUAD[nacc] = {N1, I, N2, I, N2, I, N2, N3, I};
    // basic eta etavp sxy | Vx, Vy rho k etafk phi | P rho phi sxx tk rhocp hr
    static constexpr uint32_t SLOT[nacc] = {0xf210, 0xf543, 0x3210, 0xf654, 0x3210,
                                            0xf654, 0x1ff0, 0x5432, 0xf876};
};
template <> struct Plan<false> {
    static constexpr int nquad = 5, nacc = 10;
    static constexpr int nsum[4] = {8, 6, 6, 10};
    static constexpr int GRID[nacc] = {0, 0, 1, 1, 2, 2, 3, 3, 3, 3};
    static constexpr int QUAD[nacc] = {N1, T1, N2, T2, N2, T2, N2, N3, T1, T2};
    static constexpr uint32_t SLOT[nacc] = {0x7310, 0x4265, 0x3420, 0x5ff1, 0x3420,
                                            0x5ff1, 0x8ff0, 0x4176, 0xf5ff, 0x932f};
};

// Per-row sums in LDS, slot v of grid G for row c (a basic row on the grids
// with basic y, whose two fine rows are added in registers; a fine row on the
// others), side, node column slot: off + v*SV + side*SS + c*SC + slot.  Column
// slots of segment s: SC / NSEG from s * SC / NSEG, the first for node column
// s * SEGC / 2.  The strides spread a write (4 values, 4 rows, 2 sides) and a
// read (8 columns, 4 rows) over the LDS banks.
constexpr bool grid_prow(int G) { return G & 1; }   // staggered rows: Vx, P
constexpr bool grid_pcol(int G) { return G >> 1; }  // staggered columns: Vy, P
constexpr int SUM0[4] = {0, 8, 14, 20};             // first SUM of each grid
constexpr int seg_cols(bool pcol) { return SEGC / 2 + (pcol ? 2 : 1); }
template <bool TYPED, int G> struct PartShape {
    static constexpr int cols = seg_cols(grid_pcol(G));
    static constexpr int SC = NSEG * cols;
    static constexpr int NR = grid_prow(G) ? FINE : TILE;
    static constexpr int SS = NR * SC + 4, SV = 2 * SS + 1;
    static constexpr int size = SV * Plan<TYPED>::nsum[G];
    static constexpr int off() {
        if constexpr (G == 0) return 0;
        else return PartShape<TYPED, G - 1>::off() + PartShape<TYPED, G - 1>::size;
    }
};

// Per-type values of the seven material vectors (E:659-665): 1/G (inv),
// cohesion, tension, friction, fluid density, solid and fluid expansivity
struct TypedTab {
    double v[7][3];
};

__host__ static TypedTab typed_tab(const ereb_materials& M) {
    TypedTab T;
    for (int k = 0; k < 3; ++k) {
        T.v[0][k] = 1.0 / M.gggsolidm[k];  // inv(gggsolidm[tm]), E:659
        T.v[1][k] = M.cohessolidm[k];
        T.v[2][k] = M.tenssolidm[k];
        T.v[3][k] = M.frictsolidm[k];
        T.v[4][k] = M.rhofluidm[k];
        T.v[5][k] = M.alphasolidm[k];
        T.v[6][k] = M.alphafluidm[k];
    }
    return T;
}

// every value finite in the vectors' precision: a combination of the types'
// weight sums then equals the sum over the markers also where a type's weight
// is zero
template <class R>
static bool tab_finite(const TypedTab& T) {
    for (const auto& row : T.v)
        for (double v : row)
            if (!std::isfinite((R)v)) return false;
    return true;
}

// row q of the table at type index t (0..2), by selects (no dynamic
// indexing of the kernel argument)
__device__ __forceinline__ double typed_at(const TypedTab& T, int q, int t) {
    return t == 0 ? T.v[q][0] : (t == 1 ? T.v[q][1] : T.v[q][2]);
}

// R is the type of the property vectors: double in the Float64 form, float in
// the mixed form.  The marker state (coordinates, temperature, porosity,
// stresses), the weights and the sums are double in both.
template <class R>
struct ScatterArgs {
    GeomK g;
    int nty;
    const uint32_t* __restrict__ perm;
    const int32_t* __restrict__ fstart;
    const double *xm, *ym, *phim, *sxx, *sxy;
    const R *etavp, *invggg, *frict, *cohes, *tens, *rhof, *alphas, *alphaf;
    const R *rhototal, *rhocptotal, *etatotal, *hrtotal, *ktotal, *tkrhocp, *etafkphi;
    double* part;
    // typed: 1/G, cohesion, tension, friction, fluid density and the two
    // expansivities are the material table values of the marker's type, as
    // the reference sets them (E:659-665, checked on the device by
    // typed_refresh), all of them finite: tm is read instead of the seven
    // vectors, whose sums follow from the types' weight sums and `tab`
    int typed;
    const int32_t* tm;
    TypedTab tab;
};

template <bool TYPED> struct ScatterLDS {
    double part[PartShape<TYPED, 3>::off() + PartShape<TYPED, 3>::size];
    double typed[7][3];  // the typed material table, in the vectors' precision
    double ax[4][WIN];   // the window's x, xp, y and yp nodes
    // where result lane l of accumulator a of row strip r goes in part, without
    // the column slot; -1: nowhere
    int32_t addr[NRB][Plan<TYPED>::nacc][64];
    int32_t fs[NFINE + 1];
};

// lane G of the quad, in every lane of it
template <int G>
__device__ __forceinline__ int quad_bcast(int x) {
    return __builtin_amdgcn_update_dpp(0, x, G * 0x55, 0xf, 0xf, true);
}
template <int G>
__device__ __forceinline__ double quad_bcast(double x) {
    const uint64_t u = (uint64_t)__double_as_longlong(x);
    const uint32_t lo = (uint32_t)quad_bcast<G>((int)(uint32_t)u);
    const uint32_t hi = (uint32_t)quad_bcast<G>((int)(uint32_t)(u >> 32));
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

constexpr int QP_XOR1 = 0xB1, QP_XOR2 = 0x4E;  // quad_perm [1,0,3,2], [2,3,0,1]
template <int CTRL>
__device__ __forceinline__ double quad_swap(double x) {
    const uint64_t u = (uint64_t)__double_as_longlong(x);
    const uint32_t lo =
        (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xf, 0xf, true);
    const uint32_t hi =
        (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

template <int CTRL>
__device__ __forceinline__ float quad_swap(float x) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}

// r[f] at lane t of a quad -> r[g] at lane j: the old r[j] of lane g
template <class V>
__device__ __forceinline__ void quad_transpose(V (&r)[4], bool odd, bool high) {
#pragma unroll
    for (int f = 0; f < 4; f += 2) {
        const V a = r[f], b = r[f + 1];
        const V ax = quad_swap<QP_XOR1>(a), bx = quad_swap<QP_XOR1>(b);
        r[f] = odd ? bx : a;
        r[f + 1] = odd ? b : ax;
    }
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        const V a = r[f], b = r[f + 2];
        const V ax = quad_swap<QP_XOR2>(a), bx = quad_swap<QP_XOR2>(b);
        r[f] = high ? bx : a;
        r[f + 2] = high ? b : ax;
    }
}

// A chunk's loaded values: the lane's marker's, by quad
template <class R, bool TYPED> struct ChunkData {
    double sxy, sxx, phi, x, y;
    R etatotal, etavp, rhototal, ktotal, etafkphi, tkrhocp, rhocptotal, hrtotal;
    R tens, frict, invggg, cohes, rhof, alphas, alphaf;  // untyped
    int32_t tm;                                          // typed
    int32_t fj;                                          // fine column, -1: no marker
};

// loads of the lane's marker, without the material vectors of untyped markers
template <class R, bool TYPED>
__device__ __forceinline__ void load_marker(const ScatterArgs<R>& A, uint32_t mk, int fj,
                                            ChunkData<R, TYPED>& D) {
    D = ChunkData<R, TYPED>{};
    D.fj = fj;
    if (fj < 0) return;
    const size_t m = mk;
    D.x = A.xm[m];
    D.y = A.ym[m];
    if constexpr (TYPED) D.tm = A.tm[m];
    D.etatotal = A.etatotal[m];
    D.etavp = A.etavp[m];
    D.sxy = A.sxy[m];
    D.rhototal = A.rhototal[m];
    D.ktotal = A.ktotal[m];
    D.etafkphi = A.etafkphi[m];
    D.phi = A.phim[m];
    D.sxx = A.sxx[m];
    D.tkrhocp = A.tkrhocp[m];
    D.rhocptotal = A.rhocptotal[m];
    D.hrtotal = A.hrtotal[m];
}
template <class R>
__device__ __forceinline__ void load_material(const ScatterArgs<R>& A, uint32_t mk,
                                              ChunkData<R, false>& D) {
    if (D.fj < 0) return;
    const size_t m = mk;
    D.tens = A.tens[m];
    D.frict = A.frict[m];
    D.invggg = A.invggg[m];
    D.cohes = A.cohes[m];
    D.rhof = A.rhof[m];
    D.alphas = A.alphas[m];
    D.alphaf = A.alphaf[m];
}

// addresses of strip rb's results (ScatterLDS::addr)
template <bool TYPED, int A0 = 0>
__device__ __forceinline__ void result_addr(ScatterLDS<TYPED>& L, int lane, int rb) {
    using P = Plan<TYPED>;
    if constexpr (A0 < P::nacc) {
        using PS = PartShape<TYPED, P::GRID[A0]>;
        constexpr bool prow = grid_prow(P::GRID[A0]);
        const int j = lane & 3, b = lane >> 2 & 3, side = lane >> 4 & 1;
        const int s = (int)(P::SLOT[A0] >> (4 * j)) & 15;
        const int c = prow ? 4 * rb + b : 2 * rb + (b >> 1);
        const bool used = s != 15 && (prow || !(b & 1));
        L.addr[rb][A0][lane] =
            used ? PS::off() + s * PS::SV + side * PS::SS + c * PS::SC : -1;
        result_addr<TYPED, A0 + 1>(L, lane, rb);
    }
}

// node column slot `slot` of the accumulators of the grids with column kind
// PCOL: the lanes of its parity (mine) write their sums and start over.  All
// LDS reads first, so that one wait covers them.
template <bool TYPED, bool PCOL>
__device__ __forceinline__ void write_col(ScatterLDS<TYPED>& L, double (&acc)[Plan<TYPED>::nacc],
                                          int lane, int rb, int slot, bool mine) {
    using P = Plan<TYPED>;
    int at[P::nacc];
    int2 other[P::nacc];
#pragma unroll
    for (int a = 0; a < P::nacc; ++a) {
        if (grid_pcol(P::GRID[a]) != PCOL) continue;
        at[a] = L.addr[rb][a][lane];
        if (grid_prow(P::GRID[a])) continue;
        // the basic row's other fine row (lane ^ 4)
        const uint64_t u = (uint64_t)__double_as_longlong(acc[a]);
        other[a].x = __builtin_amdgcn_ds_swizzle((int)(uint32_t)u, 0x101F);
        other[a].y = __builtin_amdgcn_ds_swizzle((int)(uint32_t)(u >> 32), 0x101F);
    }
#pragma unroll
    for (int a = 0; a < P::nacc; ++a) {
        if (grid_pcol(P::GRID[a]) != PCOL) continue;
        double v = acc[a];
        if (!grid_prow(P::GRID[a]))
            v += __longlong_as_double(
                (long long)(((uint64_t)(uint32_t)other[a].y << 32) | (uint32_t)other[a].x));
        if (mine && at[a] >= 0) L.part[at[a] + slot] = v;
        acc[a] = mine ? 0.0 : acc[a];
    }
}

// Where the sums of window node (r, c) of grid G lie in part: the rows above
// (their side 1) and below (side 0) the node, the segments that hold its
// column, in this order; out-of-range terms point at a term in range, unused
template <bool TYPED, int G> struct NodeTerms {
    using PS = PartShape<TYPED, G>;
    static constexpr int n = grid_prow(G) ? 2 : 1;  // rows a side
    static constexpr int N = 2 * n * NSEG;
    int at[N];
    bool ok[N];
    __device__ __forceinline__ NodeTerms(int r, int c) {
        const int r1 = grid_prow(G) ? 2 * r - 3 : r - 1;
#pragma unroll
        for (int d = 0; d < 2 * n; ++d) {
            const int row = r1 + d, side = d < n ? 1 : 0;
#pragma unroll
            for (int g = 0; g < NSEG; ++g) {
                const int slot = c - g * (SEGC / 2), i = d * NSEG + g;
                ok[i] = row >= 0 && row < PS::NR && slot >= 0 && slot < PS::cols;
                at[i] = PS::off() + (ok[i] ? side * PS::SS + row * PS::SC + g * PS::cols + slot : 0);
            }
        }
    }
    __device__ __forceinline__ double sum(const ScatterLDS<TYPED>& L, int v) const {
        double t[N], s = 0.0;
#pragma unroll
        for (int i = 0; i < N; ++i) t[i] = L.part[at[i] + v * PS::SV];
#pragma unroll
        for (int i = 0; i < N; ++i) s += ok[i] ? t[i] : 0.0;
        return s;
    }
};

// one node's sums of one grid: value v (the grid's own numbering) of `out`
// from slot s; from the three indicators' sums w
template <bool TYPED, int G> struct NodeOut {
    const ScatterLDS<TYPED>& L;
    const NodeTerms<TYPED, G> T;
    double* out;
    __device__ __forceinline__ NodeOut(const ScatterLDS<TYPED>& L_, double* o, int r, int c)
        : L(L_), T(r, c), out(o + (size_t)SUM0[G] * 64) {}
    __device__ __forceinline__ void put(int v, int s) const { out[v * 64] = T.sum(L, s); }
    // the weight sum (value v) and the typed values of table rows q: the
    // indicators' sums are in slots s..s+2
    double w[3];
    __device__ __forceinline__ void types(int v, int s) {
#pragma unroll
        for (int e = 0; e < 3; ++e) w[e] = T.sum(L, s + e);
        out[v * 64] = (w[0] + w[1]) + w[2];
    }
    __device__ __forceinline__ void typed(int v, int q) const {
        out[v * 64] = fma(L.typed[q][2], w[2], fma(L.typed[q][1], w[1], L.typed[q][0] * w[0]));
    }
};

// the window's 30 sums, split over the workgroup's wavefronts by the LDS terms
// they add
template <bool TYPED>
__device__ __forceinline__ void window_sums(const ScatterLDS<TYPED>& L, double* out, int wave,
                                            int lane) {
    static_assert(SCAT_NW == 6, "the split below");
    // the lane's node: neighbouring lanes read neighbouring column slots
    const int c = lane & 7, r = lane >> 3;
    out += 8 * c + r;
    if constexpr (TYPED) {
        // typed table rows: 1/G, cohesion, tension, friction, rhof, alphas, alphaf
        if (wave == 0) {  // basic ETA0 ETA (GGG) SXY (COH TEN FRI) WT
            NodeOut<true, 0> o(L, out, r, c);
            o.put(0, 0);
            o.put(1, 1);
            o.put(3, 2);
            o.types(7, 3);
            o.typed(2, 0);
            o.typed(4, 1);
            o.typed(5, 2);
            o.typed(6, 3);
        } else if (wave == 1) {  // Vx RHOX (RHOFX) KX PHIX RX WTX
            NodeOut<true, 1> o(L, out, r, c);
            o.put(0, 0);
            o.put(2, 1);
            o.put(3, 3);
            o.put(4, 2);
        } else if (wave == 2) {
            NodeOut<true, 1> o(L, out, r, c);
            o.types(5, 4);
            o.typed(1, 4);
        } else if (wave == 3) {  // Vy
            NodeOut<true, 2> o(L, out, r, c);
            o.put(0, 0);
            o.put(2, 1);
            o.put(3, 3);
            o.put(4, 2);
            o.types(5, 4);
            o.typed(1, 4);
        } else if (wave == 4) {  // P RHO RHOCP (ALPHA ALPHAF) HR (GGGP) SXX TK PHI WTP
            NodeOut<true, 3> o(L, out, r, c);
            o.put(0, 0);
            o.put(8, 1);
            o.put(6, 2);
            o.put(7, 3);
        } else {
            NodeOut<true, 3> o(L, out, r, c);
            o.put(1, 4);
            o.put(4, 5);
            o.types(9, 6);
            o.typed(2, 5);
            o.typed(3, 6);
            o.typed(5, 0);
        }
    } else {
        auto all = [&](auto o, int v0, int v1) {
            for (int v = v0; v < v1; ++v) o.put(v, v);
        };
        if (wave == 0) all(NodeOut<false, 0>(L, out, r, c), 0, 8);
        else if (wave == 1) all(NodeOut<false, 1>(L, out, r, c), 0, 3);
        else if (wave == 2) all(NodeOut<false, 1>(L, out, r, c), 3, 6);
        else if (wave == 3) all(NodeOut<false, 2>(L, out, r, c), 0, 6);
        else if (wave == 4) all(NodeOut<false, 3>(L, out, r, c), 0, 5);
        else all(NodeOut<false, 3>(L, out, r, c), 5, 10);
    }
}

template <class R, bool TYPED>
__global__ __launch_bounds__(SCAT_NW * 64, scat_waves(sizeof(R) == 4, TYPED)) void k_scatter(ScatterArgs<R> A) {
    using P = Plan<TYPED>;
    __shared__ ScatterLDS<TYPED> L;
    // XCD-contiguous: vertically neighbouring tiles (consecutive numbers)
    // read adjacent runs of the same marker columns
    const int tile = (int)xcd_block();
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rb = wave % NRB, seg = wave / NRB;
    const int t = lane & 3, b = lane >> 2 & 3, k = lane >> 4;
    const int j0 = (tile / A.nty) * TILE, i0 = (tile % A.nty) * TILE;
    for (int i = tid; i <= NFINE; i += SCAT_NW * 64)
        L.fs[i] = A.fstart[(size_t)tile * NFINE + i];
    if (TYPED && tid < 21) L.typed[tid / 3][tid % 3] = (double)(R)A.tab.v[tid / 3][tid % 3];
    if (tid < 4 * WIN) {
        const int e = tid / WIN, w = tid % WIN;
        const double* axis = e == 0 ? A.g.x : e == 1 ? A.g.xp : e == 2 ? A.g.y : A.g.yp;
        const int n = e == 0 ? A.g.Nx : e == 1 ? A.g.Nx1 : e == 2 ? A.g.Ny : A.g.Ny1;
        L.ax[e][w] = axis[min((e < 2 ? j0 : i0) + w, n - 1)];
    }
    if (seg == 0) result_addr<TYPED>(L, lane, rb);
    __syncthreads();

    const int fi = 4 * rb + b;  // the block's fine row
    const double dx = A.g.dx, dy = A.g.dy, rdx = A.g.idx, rdy = A.g.idy;
    const bool ls = !(t & 1);  // the A row's node row: upper (weight 1 - f) or lower (f)
    double acc[P::nacc];
#pragma unroll
    for (int a = 0; a < P::nacc; ++a) acc[a] = 0.0;

    const int f0 = seg * SEGC, f1 = f0 + SEGC;
    // groups of the segment's fine columns before its column q: pre[q]; all
    // wave-uniform
    int pre[SEGC + 1];
    pre[0] = 0;
#pragma unroll
    for (int q = 0; q < SEGC; ++q) {
        const int n = L.fs[(f0 + q) * FINE + fi + 1] - L.fs[(f0 + q) * FINE + fi];
        const int nmax =
            max(max(__builtin_amdgcn_readlane(n, 0), __builtin_amdgcn_readlane(n, 4)),
                max(__builtin_amdgcn_readlane(n, 8), __builtin_amdgcn_readlane(n, 12)));
        pre[q + 1] = pre[q] + ((nmax + 3) >> 2);
    }
    // the lane's marker of the chunk at group s0: its fine column in fj (-1:
    // none).  A chunk takes a run of each cell's markers, 4 a group; it is dealt
    // so that the lanes of a quad (one a group) take neighbouring markers.
    auto marker = [&](int s0, int& fj) {
        const int s = s0 + t;
        int q = 0, p = 0, pn = pre[1];
#pragma unroll
        for (int e = 1; e < SEGC; ++e) {
            q = s >= pre[e] ? e : q;
            p = s >= pre[e] ? pre[e] : p;
            pn = s >= pre[e] ? pre[e + 1] : pn;
        }
        // the chunk's groups of this column: first g0 of it, ng of them
        const int g0 = max(p, s0), ng = min(pn, s0 + 4) - g0;
        const int a = L.fs[(f0 + q) * FINE + fi], o = 4 * (g0 - p) + k * ng + (s - g0);
        const bool on = s < pre[SEGC] && o < L.fs[(f0 + q) * FINE + fi + 1] - a;
        fj = on ? f0 + q : -1;
        return on ? A.perm[a + o] : 0u;
    };
    // fine column `col` is done: the grid cells that end with it
    int col = f0, end = pre[1];  // end: the group after col's last
    auto next_col = [&]() {
        const int pb = col >> 1, c = pb - seg * (SEGC / 2);
        const bool mine = (lane >> 5) == (pb & 1);
        if (col & 1)
            write_col<TYPED, false>(L, acc, lane, rb, seg * seg_cols(false) + c, mine);
        else
            write_col<TYPED, true>(L, acc, lane, rb, seg * seg_cols(true) + c, mine);
        ++col;
        int e = 0;
#pragma unroll
        for (int q = 1; q <= SEGC; ++q) e = col - f0 == q - 1 ? pre[q] : e;
        end = e;
    };
    while (col < f1 && end == 0) next_col();  // empty columns before the first marker
    ChunkData<R, TYPED> D;
    int fjx;
    {
        const uint32_t m = marker(0, fjx);
        load_marker<R, TYPED>(A, m, fjx, D);
        if constexpr (!TYPED) load_material<R>(A, m, D);
    }
    uint32_t mx = marker(4, fjx);
    for (int s0 = 0; s0 < pre[SEGC]; s0 += 4) {
        // this chunk's values out of the load registers, the next one's into
        // them, then this chunk's products
        const int cj = max(D.fj, 0);
        const double xb = L.ax[0][cj >> 1], xp = L.ax[1][(cj + 1) >> 1];
        // read here, not held in registers across the chunks
        int ci = fi;
        asm volatile("" : "+v"(ci));
        const double yb = L.ax[2][ci >> 1], yp = L.ax[3][(ci + 1) >> 1];
        double fxb = div_by(D.x - xb, dx, rdx), fxp = div_by(D.x - xp, dx, rdx);
        double fyb = div_by(D.y - yb, dy, rdy), fyp = div_by(D.y - yp, dy, rdy);
        int tm = 0;
        // done here, before the loads below (as the transposes)
        if constexpr (TYPED) {
            tm = D.fj >= 0 ? min(max(D.tm, 1), 3) : 0;
            asm volatile("" : "+v"(fxb), "+v"(fxp), "+v"(fyb), "+v"(fyp), "+v"(tm));
        } else {
            asm volatile("" : "+v"(fxb), "+v"(fxp), "+v"(fyb), "+v"(fyp));
        }
        double q[P::nquad][4];
        R qt[2][4];  // T1, T2: in the vectors' type until a product takes them
        {
            const R one = D.fj >= 0 ? R(1) : R(0);
            // done here: the selects would otherwise move into the groups
            // below and hold twice the registers until then
            auto turn = [&](auto& r) {
                quad_transpose(r, t & 1, t & 2);
#pragma unroll
                for (int f = 0; f < 4; ++f) asm volatile("" : "+v"(r[f]));
            };
            const double raw[3][4] = {
                {(double)D.etatotal, (double)D.etavp, D.sxy, TYPED ? 0.0 : (double)one},
                {(double)D.rhototal, (double)D.ktotal, (double)D.etafkphi, D.phi},
                {D.sxx, (double)D.tkrhocp, (double)D.rhocptotal, (double)D.hrtotal}};
#pragma unroll
            for (int u = 0; u < 3; ++u) {
#pragma unroll
                for (int f = 0; f < 4; ++f) q[u][f] = raw[u][f];
                turn(q[u]);
            }
            if constexpr (!TYPED) {
                const R rawt[2][4] = {{D.tens, D.frict, D.invggg, D.cohes},
                                      {D.rhof, D.alphas, D.alphaf, one}};
#pragma unroll
                for (int u = 0; u < 2; ++u) {
#pragma unroll
                    for (int f = 0; f < 4; ++f) qt[u][f] = rawt[u][f];
                    turn(qt[u]);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        load_marker<R, TYPED>(A, mx, fjx, D);
        const uint32_t m1 = mx;
        mx = marker(s0 + 8, fjx);
        __builtin_amdgcn_sched_barrier(0);
        auto group = [&](auto gc) {
            constexpr int g = decltype(gc)::value;
            if (s0 + g >= pre[SEGC]) return;
            // 1 - f or f: the A row's node column, of the left one's parity or
            // not, and its node row, upper or lower
            const double axb = quad_bcast<g>(fxb), axp = quad_bcast<g>(fxp);
            const double ayb = quad_bcast<g>(fyb), ayp = quad_bcast<g>(fyp);
            const bool lb = ((t >> 1 ^ col >> 1) & 1) == 0, lp = ((t >> 1 ^ (col + 1) >> 1) & 1) == 0;
            const double wxb = lb ? 1.0 - axb : axb, wxp = lp ? 1.0 - axp : axp;
            const double wyb = ls ? 1.0 - ayb : ayb, wyp = ls ? 1.0 - ayp : ayp;
            const double w[4] = {wyb * wxb, wyp * wxb, wyb * wxp, wyp * wxp};
            if constexpr (TYPED) {
                q[I][g] = quad_bcast<g>(tm) == t + 1 ? 1.0 : 0.0;
            } else {
                q[T1][g] = (double)qt[0][g];
                q[T2][g] = (double)qt[1][g];
            }
#pragma unroll
            for (int e = 0; e < P::nacc; ++e)
                acc[e] = __builtin_amdgcn_mfma_f64_4x4x4f64(w[P::GRID[e]], q[P::QUAD[e]][g],
                                                            acc[e], 0, 0, 0);
            while (col < f1 && s0 + g + 1 == end) next_col();
        };
        group(std::integral_constant<int, 0>{});
        if constexpr (!TYPED) {
            // once the first group's registers are free: with all loads ahead
            // of it the Float64 form spilled one of 128 (176 us at 2.8M
            // markers, 163 so; two workgroups a CU need at most 128), the
            // mixed form took 141, 134 with its float quads
            __builtin_amdgcn_sched_barrier(0);
            load_material<R>(A, m1, D);
            __builtin_amdgcn_sched_barrier(0);
        }
        group(std::integral_constant<int, 1>{});
        group(std::integral_constant<int, 2>{});
        group(std::integral_constant<int, 3>{});
    }
    {   // the columns still open at the segment's end: the right column of the
        // last basic column cell, both columns of the last P column cell
        const bool even = (lane >> 5) == (f1 >> 1 & 1);  // parity of column f1 / 2
        const int c = SEGC / 2;
        write_col<TYPED, false>(L, acc, lane, rb, seg * seg_cols(false) + c, even);
        write_col<TYPED, true>(L, acc, lane, rb, seg * seg_cols(true) + c + (even ? 0 : 1), true);
    }
    __syncthreads();
    window_sums<TYPED>(L, A.part + (size_t)tile * NSUM * 64, wave, lane);
}

struct SumPtrs {
    double* p[NSUM];
};

// SUM[s][node] = 0 + sum of the window partials covering the node, tiles in
// ascending (tx, ty) order
__global__ __launch_bounds__(256) void k_combine(const double* __restrict__ part, int nty, int ntx,
                                                 int Ny, int Nx, SumPtrs out) {
    const int s = blockIdx.y;
    const bool basic = s < 8;
    const int rows = basic ? Ny : Ny + 1, cols = basic ? Nx : Nx + 1;
    // node counts stay far below 2^31: 32-bit index arithmetic
    const int n = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (n >= rows * cols) return;
    const int i0 = n % rows, j0 = n / rows;
    out.p[s][n] = win_sum(part, nty, win_tiles(i0, j0, nty, ntx), s, i0, j0);
}

static const int kSumGrid[NSUM] = {
    EREB_G_ETA0SUM, EREB_G_ETASUM, EREB_G_GGGSUM, EREB_G_SXYSUM, EREB_G_COHSUM,
    EREB_G_TENSUM, EREB_G_FRISUM, EREB_G_WTSUM,
    EREB_G_RHOXSUM, EREB_G_RHOFXSUM, EREB_G_KXSUM, EREB_G_PHIXSUM, EREB_G_RXSUM, EREB_G_WTXSUM,
    EREB_G_RHOYSUM, EREB_G_RHOFYSUM, EREB_G_KYSUM, EREB_G_PHIYSUM, EREB_G_RYSUM, EREB_G_WTYSUM,
    EREB_G_RHOSUM, EREB_G_RHOCPSUM, EREB_G_ALPHASUM, EREB_G_ALPHAFSUM, EREB_G_HRSUM,
    EREB_G_GGGPSUM, EREB_G_SXXSUM, EREB_G_TKSUM, EREB_G_PHISUM, EREB_G_WTPSUM};

int sum_grid_field(int s) { return kSumGrid[s]; }

// flag[0] := 1 if any marker's seven material values differ (bitwise) from
// its type's table values (in the vectors' precision)
__device__ __forceinline__ bool same_bits(double a, double b) {
    return __double_as_longlong(a) == __double_as_longlong(b);
}
__device__ __forceinline__ bool same_bits(float a, double b) {
    return __float_as_uint(a) == __float_as_uint((float)b);
}

template <class R>
__global__ __launch_bounds__(256) void k_typed_check(ScatterArgs<R> A, int64_t M,
                                                     int32_t* __restrict__ flag) {
    const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= M) return;
    const int t = min(max(A.tm[m], 1), 3) - 1;
    const R* v[7] = {A.invggg, A.cohes, A.tens, A.frict, A.rhof, A.alphas, A.alphaf};
    bool ok = true;
#pragma unroll
    for (int q = 0; q < 7; ++q) ok = ok && same_bits(v[q][m], typed_at(A.tab, q, t));
    if (!ok) flag[0] = 1;
}

template <class R>
static int typed_check_t(ereb_ctx* c) {
    auto P = [&](int f) { return (const R*)c->d_m[f]; };
    ScatterArgs<R> A{};
    A.invggg = P(EREB_M_INV_GGGTOTALM);
    A.cohes = P(EREB_M_COHESTOTALM);
    A.tens = P(EREB_M_TENSTOTALM);
    A.frict = P(EREB_M_FRICTTOTALM);
    A.rhof = P(EREB_M_RHOFLUIDCUR);
    A.alphas = P(EREB_M_ALPHASOLIDCUR);
    A.alphaf = P(EREB_M_ALPHAFLUIDCUR);
    A.tm = tm_ptr(c);
    A.tab = typed_tab(c->mat);
    int rc = fill_i32(c, c->d_typed, 0, 1);
    if (rc) return rc;
    const int64_t M = c->marknum;
    if (M > 0)
        hipLaunchKernelGGL(k_typed_check<R>, dim3((unsigned)((M + 255) / 256)), dim3(256), 0,
                           c->stream, A, M, c->d_typed);
    EREB_HIP(c, hipGetLastError());
    int32_t flag = 1;
    EREB_HIP(c, hipMemcpyAsync(&flag, c->d_typed, sizeof flag, hipMemcpyDeviceToHost,
                               c->stream));
    EREB_HIP(c, hipStreamSynchronize(c->stream));
    c->typed = flag ? 0 : 1;
    return EREB_OK;
}

int typed_refresh(ereb_ctx* c) {
    if (c->typed >= 0) return EREB_OK;
    if (c->capturing) return fail(c, EREB_ERR_STATE, "material check inside a captured step");
    // the vectors are float exactly when the context is in the mixed form
    if (marker_is_f32(c->precision, EREB_M_INV_GGGTOTALM)) return typed_check_t<float>(c);
    return typed_check_t<double>(c);
}

template <class R>
static int launch_scatter_t(ereb_ctx* c) {
    auto P = [&](int f) { return (const R*)c->d_m[f]; };
    ScatterArgs<R> A;
    A.g = geomk(c);
    A.nty = c->nty;
    A.perm = c->d_perm;
    A.fstart = c->d_fstart;
    A.xm = mptr(c, EREB_M_XM);
    A.ym = mptr(c, EREB_M_YM);
    A.phim = mptr(c, EREB_M_PHIM);
    A.sxx = mptr(c, EREB_M_SXXM);
    A.sxy = mptr(c, EREB_M_SXYM);
    A.etavp = P(EREB_M_ETAVPM);
    A.invggg = P(EREB_M_INV_GGGTOTALM);
    A.frict = P(EREB_M_FRICTTOTALM);
    A.cohes = P(EREB_M_COHESTOTALM);
    A.tens = P(EREB_M_TENSTOTALM);
    A.rhof = P(EREB_M_RHOFLUIDCUR);
    A.alphas = P(EREB_M_ALPHASOLIDCUR);
    A.alphaf = P(EREB_M_ALPHAFLUIDCUR);
    A.rhototal = P(EREB_M_RHOTOTALM);
    A.rhocptotal = P(EREB_M_RHOCPTOTALM);
    A.etatotal = P(EREB_M_ETATOTALM);
    A.hrtotal = P(EREB_M_HRTOTALM);
    A.ktotal = P(EREB_M_KTOTALM);
    A.tkrhocp = P(EREB_M_TKM_RHOCPTOTALM);
    A.etafkphi = P(EREB_M_ETAFLUIDCUR_INV_KPHIM);
    A.part = c->d_part;
    if (c->typed < 0 && !c->capturing) {
        const int rc = typed_refresh(c);
        if (rc) return rc;
    }
    A.tm = tm_ptr(c);
    A.tab = typed_tab(c->mat);
    A.typed = c->typed == 1 && tab_finite<R>(A.tab) ? 1 : 0;
    hipEvent_t ev;
    prof_begin(c, EREB_K_SCATTER, &ev);
    // the scatter's completion as ev_scatter when asked (rec_scatter)
    const dim3 grid((unsigned)c->ntiles), block(SCAT_NW * 64);
    auto* kern = A.typed ? k_scatter<R, true> : k_scatter<R, false>;
    if (c->rec_scatter)
        hipExtLaunchKernelGGL(kern, grid, block, 0, c->stream, nullptr, c->ev_scatter, 0, A);
    else
        hipLaunchKernelGGL(kern, grid, block, 0, c->stream, A);
    c->rec_scatter = false;
    EREB_HIP(c, hipGetLastError());
    prof_end(c, EREB_K_SCATTER, ev);
    return EREB_OK;
}

int launch_scatter(ereb_ctx* c, const double* hrs, const double* hrf, int mode) {
    // compute_marker_properties! (E:700-750) in the sort's pass over the markers
    const PropsReq req{hrs, hrf, mode};
    int rc = launch_fine_sort(c, &req);
    if (rc) return rc;
    // the property vectors are float exactly when the context is in the mixed form
    if (marker_is_f32(c->precision, EREB_M_ETATOTALM)) return launch_scatter_t<float>(c);
    return launch_scatter_t<double>(c);
}

int launch_combine(ereb_ctx* c) {
    SumPtrs o;
    for (int s = 0; s < NSUM; ++s) o.p[s] = gptr(c, kSumGrid[s]);
    const int64_t nmax = (int64_t)(c->Ny + 1) * (c->Nx + 1);
    hipEvent_t ev;
    prof_begin(c, EREB_K_COMBINE, &ev);
    hipLaunchKernelGGL(k_combine, dim3((unsigned)((nmax + 255) / 256), NSUM), dim3(256), 0,
                       c->stream, c->d_part, c->nty, c->ntx, c->Ny, c->Nx, o);
    EREB_HIP(c, hipGetLastError());
    prof_end(c, EREB_K_COMBINE, ev);
    return EREB_OK;
}

}  // namespace ereb
