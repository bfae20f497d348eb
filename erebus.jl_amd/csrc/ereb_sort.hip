// ereb_sort.hip -- stable counting sort of marker indices by fine key.
//
// The fine key of a marker is its "fine cell": the basic cell (ib, jb)
// (fix with the basic clamps, E:1456) refined by the P cell offsets
// (ip-ib, jp-jb) in {0,1}^2, numbered tile-major: tiles of TILE x TILE
// basic cells in column-major order, then FINE x FINE fine cells inside a
// tile, column-major.  All markers of one fine cell share the same four
// stencils on every grid.  The result perm[] lists marker indices in
// ascending key and, inside a key, ascending marker index -- exactly a
// stable counting sort, which makes every later summation order canonical.
//
//   1. k_fine_count : key per marker and its rank among the markers of its
//                     key in arrival order (one returning integer atomic per
//                     run of equal keys in a wavefront: the counts do not
//                     depend on order); before a scatter also the marker
//                     properties
//   2. scan         : key starts
//   3. k_fine_place : perm[start of the key + rank] = marker, no atomics
//                     (in the transfer step also the RK4 coefficient tables,
//                     by workgroups of their own);
//   4. k_fine_order : each key segment (about 9 markers) is sorted by marker
//                     index in place, removing the arrival order of step 3: up
//                     to 32 markers by a thread in registers, up to 1,024 by a
//                     wavefront in registers, the longer ones (listed by step 2)
//                     by a workgroup each (bitonic in LDS up to 16384, global
//                     memory beyond).
#include <algorithm>

#include "ereb_internal.h"
#include "ereb_rkcoef.h"

namespace ereb {

// Lanes of a wavefront grouped into runs: maximal stretches of consecutive
// active lanes with equal keys (markers in storage order come in runs of a
// few per fine cell).  The first lane of a run is its leader; every lane
// learns its leader and its rank in the run, a leader the run length.  A key
// split over several runs gets one count per run, which the counts and the
// slot reservations below allow (k_fine_order fixes the order within a key
// afterwards).  Two ballots and a shuffle, no loop.
struct KeyGroup {
    int leader, rank, count;  // count is non-zero on leaders only
};
__device__ __forceinline__ KeyGroup wave_group(uint32_t key, bool active) {
    const int lane = __lane_id();
    const uint32_t prev = __shfl_up(key, 1, 64);
    const uint64_t act = __ballot(active);
    const bool prev_active = lane > 0 && ((act >> (lane - 1)) & 1ull);
    const bool head = active && (!prev_active || prev != key);
    const uint64_t heads = __ballot(head);
    const uint64_t le = lanemask_lt() | (1ull << lane);
    // my run's leader: the highest head at or below this lane
    const uint64_t below = heads & le;
    KeyGroup g{lane, 0, 0};
    if (active) {
        g.leader = 63 - __clzll((long long)below);
        g.rank = lane - g.leader;
    }
    if (head) {
        // the run ends at the next head or at the next inactive lane
        const uint64_t stop = (heads | ~act) & ~le;
        const int next = stop ? __ffsll((unsigned long long)stop) - 1 : 64;
        g.count = next - lane;
    }
    return g;
}

// For every active lane: reserve one slot in counters[key]; returns the slot
// index.  All leaders issue their atomic together (one round trip per
// wavefront); within a run the slots follow lane order.
__device__ __forceinline__ int32_t wave_reserve(int32_t* counters, uint32_t key, bool active) {
    const KeyGroup g = wave_group(key, active);
    int32_t base = 0;
    if (g.count > 0) base = atomicAdd(&counters[key], g.count);
    base = __shfl(base, g.leader);
    return base + g.rank;
}

// fine key of a marker (see the file header); sets *bad when the P cell is
// not within one cell of the basic cell (coordinates beyond ~1e15 m)
__device__ __forceinline__ uint32_t fine_key(const Cells& c, int nty, bool* bad) {
    int di = c.ip - c.ib, dj = c.jp - c.jb;
    *bad = di < 0 || di > 1 || dj < 0 || dj > 1;
    di = min(max(di, 0), 1);
    dj = min(max(dj, 0), 1);
    const int ty = (c.ib - 1) / TILE, tx = (c.jb - 1) / TILE;
    const int fi = 2 * (c.ib - 1 - ty * TILE) + di;
    const int fj = 2 * (c.jb - 1 - tx * TILE) + dj;
    return (uint32_t)((tx * nty + ty) * NFINE + fj * FINE + fi);
}

// fine key, rank within the key (arrival order) and count of every marker;
// with PropArgs also the marker properties, in the same pass over the markers
// in storage order
template <class P>
__global__ __launch_bounds__(256) void k_fine_count(GeomK g, int nty, const double* __restrict__ xm,
                                                    const double* __restrict__ ym, int64_t M,
                                                    uint32_t* __restrict__ key,
                                                    int32_t* __restrict__ rank,
                                                    int32_t* __restrict__ count,
                                                    int32_t* __restrict__ flags, P props) {
    const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = m < M;
    uint32_t k = 0;
    if (active) {
        bool bad;
        k = fine_key(marker_cells(g, xm[m], ym[m]), nty, &bad);
        if (bad) flags[0] = 1;
        key[m] = k;
    }
    const int32_t r = wave_reserve(count, k, active);
    if (active) rank[m] = r;
    if (active) props.apply(m);
    // last, where nothing else is live: the step scalars, when they come with
    // this launch, to the device block for the kernels after it
    if (m == 0) props.publish();
}

template <class R>
static PropArgs<R> prop_args(ereb_ctx* c, const PropsReq& q) {
    PropArgs<R> P;
    P.M = c->d_mat;
    P.S = c->d_scal;  // hrs, hrf written there by set_heating
    // the step's scalars with this launch when they ride with the key pass
    P.Sv = c->scal;
    P.Sw = c->scal_ride && c->marknum > 0 ? c->d_scal : nullptr;
    P.mode = q.mode;
    P.tm = tm_ptr(c);
    P.tkm = mptr(c, EREB_M_TKM);
    P.phim = mptr(c, EREB_M_PHIM);
    auto f = [&](int field) { return (R*)c->d_m[field]; };
    P.XW = f(EREB_M_XWSOLIDM0);
    P.rhototal = f(EREB_M_RHOTOTALM);
    P.rhocptotal = f(EREB_M_RHOCPTOTALM);
    P.etatotal = f(EREB_M_ETATOTALM);
    P.hrtotal = f(EREB_M_HRTOTALM);
    P.ktotal = f(EREB_M_KTOTALM);
    P.tkrhocp = f(EREB_M_TKM_RHOCPTOTALM);
    P.etafkphi = f(EREB_M_ETAFLUIDCUR_INV_KPHIM);
    return P;
}

// each marker to its sorted slot: the key's start plus its rank.  The
// workgroups are numbered XCD-contiguously, so that neighbouring marker
// columns, whose markers fill the same key segments, write through one L2.
__device__ __forceinline__ void fine_place(int64_t m, const uint32_t* __restrict__ key,
                                           const int32_t* __restrict__ rank, int64_t M,
                                           const int32_t* __restrict__ start,
                                           uint32_t* __restrict__ perm) {
    if (m < M) perm[start[key[m]] + rank[m]] = (uint32_t)m;
}
__global__ __launch_bounds__(256) void k_fine_place(const uint32_t* __restrict__ key,
                                                    const int32_t* __restrict__ rank, int64_t M,
                                                    const int32_t* __restrict__ start,
                                                    uint32_t* __restrict__ perm) {
    fine_place((int64_t)xcd_block() * blockDim.x + threadIdx.x, key, rank, M, start, perm);
}

// The placement and, in the workgroups from nplace on, the RK4 coefficient
// tables, which depend on the velocities only: in a launch of their own on the
// second stream they cost the step a launch and two event calls (~15 us of
// host time; the step of a 15 x 15 grid is its launches).  Only in the steps
// that run on one stream: the tables' writes slow the placement down (35 us
// together at 2.8M markers, where they take 14 and 12 apart; 203 at 20M, 77 and
// 35), and beside the node pass and the assemblies they cost nothing.
__global__ __launch_bounds__(256) void k_fine_place_tables(const uint32_t* __restrict__ key,
                                                           const int32_t* __restrict__ rank,
                                                           int64_t M,
                                                           const int32_t* __restrict__ start,
                                                           uint32_t* __restrict__ perm,
                                                           uint32_t nplace, uint32_t ntab,
                                                           RKCoefArgs A) {
    static_assert(RKCOEF_CELLS == 256, "one workgroup size for both");
    __shared__ double sh[RKCOEF_CELLS * RKC];
    if (blockIdx.x < nplace) {
        fine_place((int64_t)xcd_block(nplace, blockIdx.x) * 256 + threadIdx.x, key, rank, M, start,
                   perm);
        return;
    }
    const uint32_t b = blockIdx.x - nplace;
    rk4_coef_block(A, (int)(b % ntab), (int)(b / ntab), sh);
}

constexpr int SEG_REG = 32;     // longest segment ordered by one thread, in registers
static_assert(SEG_WAVE == 16 * 64, "16 registers a lane");  // longest of one wavefront
constexpr int SEG_BIG = 16384;  // longest segment ordered in LDS (64 KB)
constexpr int ORD_T = 1024;     // threads of a workgroup, and its most keys
constexpr int ORD_MIN = 16;     // its fewest keys: one a wavefront

// Bitonic sorting network on N registers, ascending (Batcher 1968; every merge
// begins with the flip, so all comparators point the same way): 80 comparators
// of a minimum and a maximum for 16 values, 240 for 32.
template <int N, int K, bool FLIP>
__device__ __forceinline__ void net_stage(uint32_t (&v)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int l = FLIP ? i ^ (K - 1) : i ^ K;
        if (l > i) {
            const uint32_t lo = min(v[i], v[l]), hi = max(v[i], v[l]);
            v[i] = lo;
            v[l] = hi;
        }
    }
    if constexpr (FLIP ? K > 2 : K > 1) net_stage<N, FLIP ? K / 4 : K / 2, false>(v);
}
template <int N, int K = 2>
__device__ __forceinline__ void net_sort(uint32_t (&v)[N]) {
    net_stage<N, K, true>(v);
    if constexpr (K < N) net_sort<N, 2 * K>(v);
}
template <int N>
__device__ __forceinline__ void order_regs(uint32_t* __restrict__ seg, int n) {
    uint32_t v[N];
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = i < n ? seg[i] : 0xffffffffu;
    net_sort<N>(v);
#pragma unroll
    for (int i = 0; i < N; ++i)
        if (i < n) seg[i] = v[i];
}

// The same network over a wavefront, E values a lane (value i in lane i / E):
// each lane's values, then merges of 2, 4, .. 64 lanes, whose comparators
// across lanes are shuffles
template <int E>
__device__ __forceinline__ void wave_sort(uint32_t (&v)[E], int lane) {
    if constexpr (E > 1) net_sort<E>(v);
#pragma unroll 1
    for (int w = 2; w <= 64; w <<= 1) {
        uint32_t o[E];
        const bool up = lane & (w >> 1);  // this lane keeps the maxima
#pragma unroll
        for (int e = 0; e < E; ++e) o[e] = __shfl_xor(v[E - 1 - e], w - 1, 64);
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = up ? max(v[e], o[e]) : min(v[e], o[e]);
#pragma unroll 1
        for (int d = w >> 2; d > 0; d >>= 1) {
            const bool u = lane & d;
#pragma unroll
            for (int e = 0; e < E; ++e) o[e] = __shfl_xor(v[e], d, 64);
#pragma unroll
            for (int e = 0; e < E; ++e) v[e] = u ? max(v[e], o[e]) : min(v[e], o[e]);
        }
        if constexpr (E > 1) net_stage<E, E / 2, false>(v);
    }
}
template <int E>
__device__ __forceinline__ void order_wave(uint32_t* __restrict__ seg, int n, int lane) {
    uint32_t v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = lane * E + e < n ? seg[lane * E + e] : 0xffffffffu;
    wave_sort<E>(v, lane);
#pragma unroll
    for (int e = 0; e < E; ++e)
        if (lane * E + e < n) seg[lane * E + e] = v[e];
}

// keys of a workgroup of the ordering pass: at most one a thread; fewer where
// that leaves the 256 CUs without a workgroup each (a small grid's wavefronts
// then share its crowded keys), and fewer the more markers a key holds, so that
// a workgroup has about 16,384 markers
static int order_keys(int64_t nkeys, int64_t M) {
    const int64_t chip = nkeys / 256;
    const int64_t load = (int64_t)SEG_BIG * nkeys / std::max<int64_t>(M, 1);
    return (int)std::clamp<int64_t>(std::min(chip, load), ORD_MIN, ORD_T);
}

// One thread per key of the workgroup's nper; the longer segments are then
// dealt to its wavefronts, and those of more than SEG_WAVE markers, listed in
// big, to the workgroups of the launch (a launch of its own for them, with
// nothing to do in most steps, cost 5 us).  tmp: scratch of 2 M words.
// What bounds it: the keys' dependent memory accesses; 64 registers, so that a
// CU holds two workgroups.  The sort with every key crowded (16 x 16 markers a
// cell) took 3,072 us at 15 x 15 nodes and 4,408 at 141 x 141 with such segments
// ordered one after another by the workgroup that holds their 1,024 keys; 18 and
// 189 now.
__global__ __launch_bounds__(ORD_T, 8) void k_fine_order(const int32_t* __restrict__ start,
                                                         int64_t nkeys, int nper,
                                                         uint32_t* __restrict__ perm,
                                                         const int32_t* __restrict__ big,
                                                         uint32_t* __restrict__ tmp) {
    extern __shared__ uint32_t sdyn[];
    __shared__ int32_t left[ORD_T], nleft;  // keys left to the wavefronts
    if (threadIdx.x == 0) nleft = 0;
    __syncthreads();
    const int64_t k = (int64_t)blockIdx.x * nper + threadIdx.x;
    const bool mine = (int)threadIdx.x < nper && k < nkeys;
    const int32_t a = mine ? start[k] : 0, n = mine ? start[k + 1] - a : 0;
    if (n > SEG_REG) {
        if (n <= SEG_WAVE) left[atomicAdd(&nleft, 1)] = (int32_t)k;
    } else if (n > SEG_REG / 2) {
        order_regs<SEG_REG>(perm + a, n);
    } else if (n > 1) {
        order_regs<SEG_REG / 2>(perm + a, n);
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    for (int q = threadIdx.x >> 6; q < nleft; q += ORD_T / 64) {
        const int32_t a = start[left[q]], n = start[left[q] + 1] - a;
        if (n <= 64) order_wave<1>(perm + a, n, lane);
        else if (n <= 128) order_wave<2>(perm + a, n, lane);
        else if (n <= 256) order_wave<4>(perm + a, n, lane);
        else if (n <= 512) order_wave<8>(perm + a, n, lane);
        else order_wave<16>(perm + a, n, lane);
    }
    for (int q = blockIdx.x; q < big[0]; q += gridDim.x) {
        const int32_t a = start[big[1 + q]], L = start[big[1 + q] + 1] - a;
        int n = 1;
        while (n < L) n <<= 1;
        // LDS when it fits, else the scratch region [2a, 2a + n) of tmp,
        // disjoint between segments because n < 2L
        uint32_t* s = n <= SEG_BIG ? sdyn : tmp + 2 * (int64_t)a;
        for (int i = threadIdx.x; i < n; i += ORD_T) s[i] = i < L ? perm[a + i] : 0xFFFFFFFFu;
        __syncthreads();
        bitonic(s, n);
        for (int i = threadIdx.x; i < L; i += ORD_T) perm[a + i] = s[i];
        __syncthreads();
    }
}

int launch_fine_sort(ereb_ctx* c, const PropsReq* props) {
    const int64_t M = c->marknum;
    const int64_t nk = c->nkeys;
    int rc;
    hipEvent_t ev;
    if (props && (rc = set_heating(c, props->hrs, props->hrf))) return rc;
    // perm is rewritten below: it orders no marker set until the sort completes
    c->have_sort = false;
    prof_begin(c, EREB_K_SORT, &ev);
    // the key counts are zero here (left so by the previous sort's scan)
    // unless a sort stopped half-way; a domain error flag stays set until
    // the host reads it (check_flags)
    if (c->fcount_dirty && (rc = fill_i32(c, c->d_fcount, 0, nk))) return rc;
    // ranks live in the first M words of the oversize-segment scratch, which
    // k_fine_order uses only after the placement
    int32_t* rank = (int32_t*)c->d_tmp;
    int32_t* big = rank + 2 * c->cap;  // sort_list_words(cap) words
    if (M > 0) {
        c->fcount_dirty = true;
        const unsigned nb = (unsigned)((M + 255) / 256);
        const GeomK g = geomk(c);
        const double *xm = mptr(c, EREB_M_XM), *ym = mptr(c, EREB_M_YM);
        // the property vectors are float exactly when the context is in the mixed form
        if (!props)
            hipLaunchKernelGGL(k_fine_count<NoProps>, dim3(nb), dim3(256), 0, c->stream, g,
                               c->nty, xm, ym, M, c->d_key, rank, c->d_fcount, c->d_flags,
                               NoProps{});
        else {
            auto keys = [&](auto kern, auto P) {
                hipLaunchKernelGGL(kern, dim3(nb), dim3(256), 0, c->stream, g, c->nty, xm, ym, M,
                                   c->d_key, rank, c->d_fcount, c->d_flags, P);
            };
            if (marker_is_f32(c->precision, EREB_M_ETATOTALM))
                keys(k_fine_count<PropArgs<float>>, prop_args<float>(c, *props));
            else
                keys(k_fine_count<PropArgs<double>>, prop_args<double>(c, *props));
        }
        if (props && c->scal_ride) {  // the device block now follows this launch
            c->scal_ride = false;
            c->scal_dev = c->scal;
            c->scal_written = true;
        }
    }
    // key starts; the counts are cleared for the next sort
    if ((rc = scan_exclusive(c, c->d_fcount, c->d_fstart, nk, big, SEG_WAVE, true))) return rc;
    c->fcount_dirty = false;
    if (M > 0) {
        const unsigned nb = (unsigned)((M + 255) / 256);
        if (c->tables_ride) {
            const unsigned nt = rk4_coef_blocks(c);
            hipLaunchKernelGGL(k_fine_place_tables, dim3(nb + 4 * nt), dim3(256), 0, c->stream,
                               c->d_key, (const int32_t*)rank, M, c->d_fstart, c->d_perm, nb, nt,
                               rk4_coef_args(c));
            c->tables_ride = false;
        } else
            hipLaunchKernelGGL(k_fine_place, dim3(nb), dim3(256), 0, c->stream, c->d_key,
                               (const int32_t*)rank, M, c->d_fstart, c->d_perm);
        const int nper = order_keys(nk, M);
        hipLaunchKernelGGL(k_fine_order, dim3((unsigned)((nk + nper - 1) / nper)), dim3(ORD_T),
                           SEG_BIG * sizeof(uint32_t), c->stream, c->d_fstart, nk, nper,
                           c->d_perm, (const int32_t*)big, c->d_tmp);
    }
    EREB_HIP(c, hipGetLastError());
    prof_end(c, EREB_K_SORT, ev);
    c->have_sort = true;
    c->sort_gen = c->pos_gen;
    c->sort_m = M;
    return EREB_OK;
}

int ensure_sort(ereb_ctx* c) {
    if (c->have_sort && c->sort_gen == c->pos_gen) return EREB_OK;
    return launch_fine_sort(c);
}

}  // namespace ereb
