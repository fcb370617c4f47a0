// The fused bundle + chain-growth kernel of double maps (k_curvelets) and the
// small kernels that feed it.  Included by cvg_pipeline.hip inside its
// namespace, after the wave helpers.
//
// The reference decides everything by comparing bundle bounds lo < hi
// (cpu_curvelet.hpp:821-854), each bound a quotient of the transport formulas.
// Four IEEE divisions are ~270 of the ~430 SIMD cycles one pair's 63 cells take
// that way (66.8 cycles per wave division against 5 for a multiply, measured),
// and their per-pair sines another pass over memory.  Here the bounds are first
// formed approximately, with a proven error bound: sines by rotating the edges'
// correctly rounded sin/cos, one reciprocal for the three denominators, the
// result in 32-bit fixed point.  A comparison whose margin exceeds the error
// bound is decided by it.  An anchor with any closer comparison is done again
// on the reference's own bounds (its operands and rounding points, correctly
// rounded math, IEEE divisions, doubles).  The results are the reference's bit
// for bit.
//
// Measured on the 1080p map (207,326 edges, 2.04M pairs, G = 7): 1,000 us for
// the kernel on exact bounds and 141 us for its sines pass (345 MB) before; now
// 432 us, and 32 us for the four anchors left open, which is one wave's time for
// one of them.  The same map at whole pixels and 16 orientations leaves 9,162 of
// 184,425 anchors open: 350 us in all.
#ifndef CVG_FUSED_HPP
#define CVG_FUSED_HPP

// The grid and edges of exact_bound.
struct ExactGrid {
    const double *x, *y, *th;
    const double *off_x, *off_t;  // delta_x2, delta_t2 (cpu_curvelet.hpp:697-698)
    double dt, dx, dx2, close_thr, max_k;
    int kt;
};

// One bound of a pair's bundle at one grid cell, exactly as
// compute_curve_bundle leaves it (cpu_curvelet.hpp:636-819): lo, or hi with
// `upper`.  Angles are below 2^20 here (fused_limits), so the sines need no
// Payne-Hanek reduction.  (sa, ca) = sin/cos of theta_a, (s2, c2) of
// T2t = theta_a + delta_t2; ox = delta_x2; b the neighbour.  The two branches
// (:711-751, :774-806) differ in a factor of two on the curvature fraction and
// in which of theta_n -+ dt bounds which side.
__device__ inline double exact_bound(const ExactGrid &E, bool upper, double ax, double ay, double sa, double ca,
                                     double T2t, double s2, double c2, double ox, int b)
{
    const double DX = ax - E.x[b], DY = ay - E.y[b], nt = E.th[b];
    const double DX2 = DX * DX, DY2 = DY * DY;
    double v = upper ? E.max_k : -E.max_k;
    if (DX2 + DY2 < E.close_thr) return v;  // :682
    const bool branch_a = (DX * ca + DY * sa) < 0;  // :690
    const double tt = s2 * DX - c2 * DY;
    const double ttm = tt - ox;
    // (:711; :774 negates the sum, so that an exact zero is -0 there)
    const double u = 2.0 * ox * tt - DX2 - DY2 + E.dx2 - ox * ox;
    const double x = upper ? ttm + E.dx : ttm - E.dx;
    const double kx = (branch_a ? 2.0 * x : x) / (branch_a ? 0.0 - u : -u / 2.0);
    const double T0 = branch_a == upper ? nt + E.dt : nt - E.dt;
    double s0, c0;
    cvg::cr_sincos<false>(T0, c_sincos_tab, &s0, &c0);
    const double s = cvg::cr_sin<false>(T2t - T0, c_sincos_tab);  // :728-729
    const double kt = s / (-s * ox + DX * c0 + DY * s0);
    // the reference's compare-and-assign, which ignores NaN
    if (upper) {
        if (v > kx) v = kx;
        if (v > kt) v = kt;
    } else {
        if (v < kx) v = kx;
        if (v < kt) v = kt;
    }
    return v;
}

// Correctly rounded, of any finite angle; out of line: the direct kernel's
// anchors are often few, and then spend much of their time on instruction fetch.
__device__ __noinline__ double2 direct_sincos(double x)
{
    double s, c;
    cvg::cr_sincos(x, c_sincos_tab, &s, &c);
    return make_double2(s, c);
}
__device__ __noinline__ double direct_sin(double x) { return cvg::cr_sin(x, c_sincos_tab); }
__device__ __noinline__ int direct_class(double ax, double ay, double ca, double sa, double nx, double ny)
{
    return cvg::direction_class(ax, ay, ca, sa, nx, ny, c_sincos_tab, c_atan_tab);
}

// Per edge: (x, y, sin theta, cos theta), the correctly rounded pair.  Block 0
// also clears the curvelet stage's counters (the graph stage's words are left
// alone, so this may run before its last host read).
__global__ __launch_bounds__(kBlock) void k_edge_rec(int n, const double *__restrict__ x, const double *__restrict__ y,
                                                     const double *__restrict__ th, double4 *__restrict__ rec,
                                                     unsigned *__restrict__ scal)
{
    if (blockIdx.x == 0) {
        const int t = static_cast<int>(threadIdx.x);
        if (t == 0) scal[S_VALID] = 0u;
        if (t == 1) scal[S_COUNT] = 0u;
        if (t == 2) scal[S_COUNT + 1] = 0u;
        for (int w = kBucketBase + t; w < kScalarBufWords; w += static_cast<int>(blockDim.x)) scal[w] = 0u;
    }
    const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n) return;
    double s, c;
    cvg::cr_sincos(th[i], c_sincos_tab, &s, &c);
    rec[i] = make_double4(x[i], y[i], s, c);
}

// Anchors in spatial (cell) order in lists by falling degree: first those of
// more than 64 neighbours (for k_curvelets_direct), then k_curvelets': its waves
// take entries round robin over those concatenated lists, so each gets its
// share of long and short anchors, and the kernel's tail consists of the
// shortest.  Narrow lists keep the shares alike: with 14 of them in place of
// four the 720p map's kernel takes 239 us against 268, the 1080p map's 455
// against 472.  The open list is k_curvelets' own.  Anchors without neighbours get
// their zero count here.  Each entry carries (anchor, CSR base, degree).
constexpr int kOrderBlock = 1024;  // few workgroups: one list-length atomic each per list
enum { L_OPEN = 0, L_WIDE = 1, L_FIRST = 2, kLists = 16 };

// The open list has n places, and so has the wide one, last (a double map
// without lists of more than 64 does not use it).  An anchor is in one degree
// list, so two of those share n, one from the front and one from the back.
constexpr int kListRegions = L_FIRST + (kLists - L_FIRST) / 2;
__host__ __device__ __forceinline__ long long entry_place(int list, long long i, int n)
{
    const int region = list == L_OPEN ? 0 : (list == L_WIDE ? kListRegions - 1 : 1 + (list - L_FIRST) / 2);
    const bool back = list > L_FIRST && ((list - L_FIRST) & 1) != 0;
    return static_cast<long long>(region) * n + (back ? n - 1 - i : i);
}

__device__ __forceinline__ int degree_list(unsigned deg)
{
    constexpr unsigned kAbove[kLists - 1 - L_FIRST] = {48, 40, 32, 28, 24, 20, 17, 14, 12, 10, 8, 6, 4};
    int list = L_FIRST;
#pragma unroll
    for (unsigned bound : kAbove) list += deg <= bound ? 1 : 0;
    return deg > 64u ? L_WIDE : list;
}

__global__ __launch_bounds__(kOrderBlock) void k_order(int n, const int *__restrict__ sorted,
                                                       const unsigned *__restrict__ off, int4 *__restrict__ lists,
                                                       unsigned *__restrict__ acc_count, unsigned *__restrict__ scal)
{
    __shared__ unsigned s_count[kLists];
    __shared__ unsigned s_base[kLists];
    // a guessed size that did not hold (this may run before the host knows):
    // the graph is built again
    if (scal[S_MISS] | scal[S_BAD]) return;
    const int p = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (threadIdx.x < kLists) s_count[threadIdx.x] = 0;
    __syncthreads();
    int a = -1, b = -1;
    unsigned o0 = 0, o1 = 0;
    if (p < n) {
        a = sorted[p];
        o0 = off[a];
        o1 = off[a + 1];
        const unsigned deg = o1 - o0;
        if (deg == 0)
            acc_count[a] = 0u;
        else
            b = degree_list(deg);
    }
    // a place in the block's share of the list, then one global atomic per
    // block and list
    const unsigned my_off = b >= 0 ? atomicAdd(&s_count[b], 1u) : 0u;
    __syncthreads();
    if (threadIdx.x < kLists && s_count[threadIdx.x] > 0)
        s_base[threadIdx.x] = atomicAdd(&scal[kBucketBase + threadIdx.x * kBucketStride], s_count[threadIdx.x]);
    __syncthreads();
    if (b >= 0)
        lists[entry_place(b, static_cast<long long>(s_base[b]) + my_off, n)] =
            make_int4(a, static_cast<int>(o0), static_cast<int>(o1 - o0), 0);
}

// Load from a wave-uniform address through the scalar data cache (read only).
template <typename T>
__device__ __forceinline__ T uload(const T *p)
{
    return *(const __attribute__((address_space(4))) T *)p;
}

using cvg::kFixOne;
using cvg::kFixTol;

// v_cvt_i32_f64: truncates and saturates (NaN gives 0), where the C++ cast is
// undefined out of range.
__device__ __forceinline__ int fix(double v)
{
    int r;
    asm("v_cvt_i32_f64 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

// One instruction each (fmax and fmin quiet their operands first; bounds are NaN
// all or none, with max_k).
__device__ __forceinline__ double larger(double a, double b)
{
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double smaller(double a, double b)
{
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ int larger(int a, int b) { return max(a, b); }
__device__ __forceinline__ int smaller(int a, int b) { return min(a, b); }

__device__ __forceinline__ int sub_sat(int a, int b) { return __builtin_elementwise_sub_sat(a, b); }

__device__ __forceinline__ unsigned long long perm64(int src_lane, unsigned long long v)
{
    const int lo = __builtin_amdgcn_ds_bpermute(src_lane << 2, static_cast<int>(v));
    const int hi = __builtin_amdgcn_ds_bpermute(src_lane << 2, static_cast<int>(v >> 32));
    return static_cast<unsigned long long>(static_cast<unsigned>(hi)) << 32 | static_cast<unsigned>(lo);
}

// v with lane `l` (uniform) replaced by the uniform value s.
__device__ __forceinline__ unsigned long long set_lane64(unsigned long long v, unsigned long long s, int l)
{
    const unsigned lo = static_cast<unsigned>(
        lane_write(static_cast<int>(s), l, static_cast<int>(v)));
    const unsigned hi = static_cast<unsigned>(
        lane_write(static_cast<int>(s >> 32), l, static_cast<int>(v >> 32)));
    return static_cast<unsigned long long>(hi) << 32 | lo;
}

__device__ __forceinline__ unsigned long long get_lane64(unsigned long long v, int l)
{
    const unsigned lo = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(v), l));
    const unsigned hi = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(v >> 32), l));
    return static_cast<unsigned long long>(hi) << 32 | lo;
}

// Staged row of an accepted seed: the run's hypotheses as bits over the
// anchor's neighbour list, the chain as bits over the hypotheses, and this
// word: the best cell's rank, the direction, whether the masks have four words, and
// the seed (a hypothesis; its bundle belongs to the running one even when the
// chain filled up before its turn).  The record forms k_min and k_max.
__host__ __device__ inline unsigned row_meta(int rank, bool fwd, bool wide, int seed)
{
    return static_cast<unsigned>(rank) | (fwd ? 1u << 8 : 0u) | (wide ? 1u << 9 : 0u) |
           static_cast<unsigned>(seed) << 10;
}

struct FusedArgs {
    const double4 *rec;  // per edge (x, y, sin, cos)
    const double *th;
    const double2 *compass;  // cosine and sine of the eight neighbours' directions, 3 (sign of y) + sign of x
    ExactGrid exact;
    const int *ids;
    const unsigned *off;  // CSR offsets
    int4 *lists;         // (anchor, CSR base, degree, -), at entry_place
    unsigned *list_len;  // entry counts, kBucketStride words apart (device; k_order's, and the open list's)
    int n;
    int K, G;
    // per cell in rank order: delta_x2, delta_t2, sin and cos of delta_t2,
    // whether it can be a best cell
    const double *rank_ox, *rank_ot, *rank_so, *rank_co;
    const int *rank_elig;
    const int *rank_cell;
    float inv_kt;  // 1 / exact.kt
    int rank_of_cell0;
    double sin_dt, cos_dt, dx, four_dx, dx2, close_thr, max_k;
    double scale;                    // kFixOne / max_k
    double min_den, num_err, den_err;  // fused_limits
    double min_prod;                 // below it a product of the three denominators may have a small one
    int slots;                       // bundle slots in LDS; a run's other bundles go to `spill`
    char *spill;
    size_t spill_stride;             // bytes per wave
    ulonglong2 *st_mask;             // (hypotheses, chain) per row
    size_t mask_plane;               // entries between the 64-bit planes of st_mask
    unsigned *st_meta;
    // float maps: the reference's float operands, and rows as the general
    // kernel stages them
    float dt_f, dx_f, max_k_f, close_f;
    int *st_ids;
    int st_stride;
    double *st_k;
    unsigned *acc_count;
    unsigned *partial;               // per wave: valid pairs, then two words of the intersection count
};

constexpr int kFusedWaves = 4;  // anchor streams (waves) per workgroup
// What LDS lets stay resident (double maps at one cell per lane: five).
__host__ __device__ constexpr int waves_per_simd(int cpl, bool flt) { return cpl == 4 ? 2 : (cpl == 1 && !flt ? 5 : 4); }
constexpr int kFusedSlots = 12;  // bundle slots at one cell per lane
// pair records in LDS at a time, as a power of two (with two cells per lane 16
// of them would cost a resident wave per SIMD)
__host__ __device__ constexpr int batch_log(int cpl) { return cpl == 1 ? 4 : 3; }
constexpr int kSmallRun = 8;    // runs up to here grow on cell masks

constexpr int kLeftOpen = 16;   // a wave's anchors waiting to be appended to another list

struct SliceCarve {
    int bun, rec, pm, sines, left, bytes;
};

// One wave's LDS slice: bundle slots (lo, hi per lane), the pair records of
// one batch (80 B each), the mask matrix of a small run, and the anchors left
// open.  With 12 slots that is 8,000 B, four of them the 25 blocks of 1,280 B that
// let a fifth workgroup onto a CU.
__host__ __device__ inline SliceCarve slice_carve(int slots, int cpl)
{
    SliceCarve c{};
    c.bun = 0;
    c.rec = c.bun + slots * cpl * 64 * 8;
    c.pm = c.rec + (80 << batch_log(cpl));
    c.left = c.pm + 64 * cpl * 8;
    c.bytes = c.left + kLeftOpen * 4;
    return c;
}

// The same with bounds in doubles, 16 pair records of 64 B at a time, and the
// transport sines of a group of pairs, one to a lane as far as they go: at the
// default grid 10,176 B, a sixteenth of a CU's.
constexpr int kDirectSlots = 8;
__host__ __device__ inline int direct_pairs_log(int kt)
{
    int log = 4;
    while (log > 0 && (2 * kt << log) > 64) --log;
    return log;
}
__host__ __device__ inline SliceCarve direct_carve(int slots, int cpl, int kt)
{
    SliceCarve c{};
    c.bun = 0;
    c.rec = c.bun + slots * cpl * 64 * 16;
    c.pm = c.rec + 16 * 64;
    c.sines = c.pm + 64 * cpl * 8;
    c.bytes = c.sines + (2 * kt << direct_pairs_log(kt)) * 8;
    return c;
}

// A lane's cells: lanes without one repeat the first.
template <int CPL>
struct WaveCells {
    double ox[CPL], oxp2[CPL], so[CPL], co[CPL];
    double m2ox[CPL], ox2[CPL];  // (float maps)
    double ot[CPL];
    int j[CPL];  // (direct) the cell's orientation offset
    unsigned long long emask[CPL];  // cells that can be a best one
};

// LDS and device memory, told apart by type: one pointer for both would make
// every bundle access a flat one.
template <typename T>
using lds_ptr = __attribute__((address_space(3))) T *;
template <typename T>
using mem_ptr = __attribute__((address_space(1))) T *;

template <typename V>
struct alignas(2 * sizeof(V)) BoundsOf {
    V lo, hi;
};

// Float maps (the reference's float instantiation).  Its bounds are formed by
// its own float operations, which take a lane no division longer than the
// approximations above; only the correctly rounded float sines come from
// doubles: rotations, as above, corrected for the angle's rounding to float,
// and certain unless within kSineErr of where the float changes.  Bounds are
// compared as integers of the same order.  720p float map (92,070 edges): 4,860
// us on the general kernel, whose two correctly rounded sines a cell are some
// 600 instructions; 322 us so, and 56 us for the anchors left open (346 us when
// those went to the general kernel).
// M_FLOAT leaves an anchor with an uncertain sine or direction open;
// M_FLOAT_EXACT takes the correctly rounded ones there.
enum { M_FAST = 0, M_DIRECT = 1, M_FLOAT = 2, M_FLOAT_EXACT = 3 };

__device__ inline int direction_class_f(float ax, float ay, float at, float nx, float ny, float cos_at, float sin_at);

// (out of line, as direct_sin)
__device__ __noinline__ float exact_sine(float x, bool cosine)
{
    float s, c;
    cvg::cr_sincosf(x, c_sincos_tab, &s, &c);
    return cosine ? c : s;
}
__device__ __noinline__ int exact_direction(float ax, float ay, float at, float nx, float ny, float ca, float sa)
{
    return direction_class_f(ax, ay, at, nx, ny, ca, sa);
}

// Beyond what the rotations are off by: sums of an orientation (up to 64) and
// an offset 2^-47, their sines and cosines 2^-51 each, the products 2^-50.
constexpr double kSineErr = 0x1p-44;

// v as float; `bad` gets a bit where v + kSineErr or v - kSineErr rounds
// differently.
__device__ __forceinline__ float sure_float(double v, unsigned &bad)
{
    const float f = static_cast<float>(v + kSineErr);
    bad |= __float_as_uint(f) ^ __float_as_uint(static_cast<float>(v - kSineErr));
    return f;
}

// Floats as integers of the same order, and back (no -0.0f).
__device__ __forceinline__ int float_key(float v)
{
    const int b = __float_as_int(v);
    return b ^ ((b >> 31) & INT_MAX);
}
__device__ __forceinline__ float key_float(int k) { return __int_as_float(k ^ ((k >> 31) & INT_MAX)); }

// One anchor on one wave.  M_FAST and M_FLOAT return true, with nothing
// counted, when something is closer than they can decide; M_DIRECT forms the
// reference's own bounds, and M_FLOAT_EXACT returns true only for a bound or
// denominator of zero, whose sign is lost.
//
// M_DIRECT: correctly rounded sines and four IEEE divisions a cell, bounds in
// doubles.  A pair's transport sines depend on the cell's orientation offset
// alone (sin(T2t - T0), :728-729): the lanes take (pair, side, offset) items,
// 7 to a side in place of 63 cells, and the cells read them in LDS.
//
// Lane = neighbour forms the pairs' direction class, flags and
// cell-independent terms (16 records in LDS at a time, in run order).  Then,
// lane = bundle cell in "rank" order (cells sorted by (ox^2 + ot^2, index), so
// that fill_curvelet_info's cell, cpu_curvelet.hpp:202-219, is the lowest
// valid one; CPL cells per lane), each run's bundles: forward neighbours,
// backward, neither (validity only, for the count).  A valid (or close) pair
// is a hypothesis and takes the next slot; its cells with hi <= lo are stored
// as (largest, smallest), so that they compare as invalid from then on (M_DIRECT:
// as they are).
//
// Growth.  A chain's running bundle is max lo, min hi over its members, so it
// is valid at a cell exactly where every member's lo lies below every member's
// hi.  For a run of up to 8 hypotheses one 64-bit mask per pair of them says
// at which cells that holds; the seeds' chains then grow together, lane
// (j, h) holding the cells where seed j's chain and hypothesis h are
// compatible: step h is one ballot and two ANDs for all seeds at once.  (A
// step per seed and hypothesis, lane = cell, is a chain of LDS reads,
// compares, ballots and branches: 34% of the kernel's wave time before.)
// Longer runs walk seed by seed.
//
// Rows.  Chains are sets of slots, so equal chains are equal masks
// (check_curvelet_exist, :876-916: the first of equal chains is kept).  The
// best cell is the lowest eligible bit of the seed's final mask.  k_min and
// k_max are left to the record, where a lane has a row of its own.
//
// NW: 64-bit words of a slot or neighbour mask (64 NW neighbours at most).
//
// nid, nb, nth: lane's neighbour (of the first 64), its record and orientation.
template <int CPL, int NW, int MODE>
__device__ __forceinline__ bool do_anchor(const FusedArgs &A, const WaveCells<CPL> &W, char *sl, char *spill, int a,
                                          unsigned base, int deg, int nid, const double4 nb, double nth,
                                          unsigned &vp_sum, unsigned long long &isect_sum)
{
    typedef unsigned long long u64;
    constexpr bool DIRECT = MODE == M_DIRECT, FLT = MODE >= M_FLOAT, SINES = MODE == M_FLOAT_EXACT;
    constexpr bool CLASSES = DIRECT || SINES;  // exact directions, with the third class
    static_assert(!FLT || NW == 1, "float maps: up to 64 neighbours");
    using V = typename std::conditional<DIRECT, double, int>::type;
    using Bounds = BoundsOf<V>;
    constexpr int kTol = FLT ? 0 : kFixTol;
    constexpr int kLog = DIRECT ? 4 : batch_log(CPL), kLast = (1 << kLog) - 1;
    constexpr int NC = NW;  // 64-seed (64-neighbour) chunks
    const int lane = threadIdx.x & 63;
    const int G = A.G;
    const int slots = A.slots;
    const SliceCarve cv = DIRECT ? direct_carve(A.slots, CPL, A.exact.kt) : slice_carve(A.slots, CPL);
    const lds_ptr<Bounds> bun = (lds_ptr<Bounds>)(sl + cv.bun) + lane;
    const lds_ptr<double2> rec = (lds_ptr<double2>)(sl + cv.rec);
    const lds_ptr<u64> pm = (lds_ptr<u64>)(sl + cv.pm);
    const mem_ptr<Bounds> spl = (mem_ptr<Bounds>)spill + lane;
    auto get_bundle = [&](int s, int m) -> Bounds {
        Bounds v;
        if (s < slots) {
            v.lo = bun[(s * CPL + m) * 64].lo;
            v.hi = bun[(s * CPL + m) * 64].hi;
        } else {
            v.lo = spl[((s - slots) * CPL + m) * 64].lo;
            v.hi = spl[((s - slots) * CPL + m) * 64].hi;
        }
        return v;
    };
    auto load_rec = [&](int c) -> double4 {  // neighbours 64 c + lane
        double4 v = make_double4(0.0, 0.0, 0.0, 1.0);
        if (64 * c + lane < deg) v = A.rec[A.ids[base + 64 * c + lane]];
        return v;
    };
    // M_FAST, each comparison's t = hi - lo: true above kFixTol, false below
    // -kFixTol, and in between open.  A lane's smallest open_key says at the
    // end whether any of its comparisons was open.
    unsigned closest = ~0u;
    auto note = [&](int t) {
        if (MODE == M_FAST) closest = min(closest, cvg::open_key(t));
    };
    unsigned bad = 0u;        // M_FLOAT: nonzero where a float sine is uncertain
    // the float of v, an approximation of x's sine or cosine, in the lanes `in`
    auto sure = [&](double v, float x, bool cosine, bool in) -> float {
        unsigned u = 0u;
        float f = sure_float(v, u);
        u = in ? u : 0u;
        if constexpr (SINES) {
            if (__builtin_amdgcn_ballot_w64(u != 0u) != 0ULL) {
                if (u != 0u) f = exact_sine(x, cosine);
            }
        } else {
            bad |= u;
        }
        return f;
    };
    // float maps: the smallest magnitude of a bound or of its first denominator
    // (a zero's sign would be lost: :774 makes it -0)
    float least = A.max_k_f;
    u64 open = 0ULL;  // (not CLASSES) neighbours whose direction class is uncertain

    const double *ar = reinterpret_cast<const double *>(A.rec + a);
    const double ax = uload(ar), ay = uload(ar + 1), sa = uload(ar + 2), ca = uload(ar + 3);
    // sin/cos of theta_a + delta_t2 (by rotation)
    double sT[CPL], cT[CPL];
    float T2[CPL], sf[CPL], cf[CPL];  // float maps: the angle, its sine and cosine
#pragma unroll
    for (int m = 0; m < CPL; ++m) {
        if constexpr (DIRECT) {
            sT[m] = cT[m] = 0.0;
            if (A.exact.kt > 32) {  // (fewer: with the first pairs' below)
                const double2 t = direct_sincos(uload(A.th + a) + W.ot[m]);  // :702
                sT[m] = t.x;
                cT[m] = t.y;
            }
            continue;
        }
        sT[m] = __builtin_fma(sa, W.co[m], ca * W.so[m]);
        cT[m] = __builtin_fma(ca, W.co[m], -(sa * W.so[m]));
        if constexpr (FLT) {
            const double th = uload(A.th + a);
            T2[m] = static_cast<float>(th) + static_cast<float>(W.ot[m]);  // :702
            const double e = static_cast<double>(T2[m]) - (th + W.ot[m]);
            const double s = sT[m], c = cT[m];
            sT[m] = __builtin_fma(e, __builtin_fma(-0.5 * e, s, c), s);
            cT[m] = __builtin_fma(-e, __builtin_fma(0.5 * e, c, s), c);
            sf[m] = sure(sT[m], T2[m], false, true);
            cf[m] = sure(cT[m], T2[m], true, true);
        }
    }

    [[maybe_unused]] float fth = 0.0f, fsa = 0.0f, fca = 0.0f;
    if constexpr (FLT) {
        fth = static_cast<float>(uload(A.th + a));
        fsa = sure(sa, fth, false, true);
        fca = sure(ca, fth, true, true);
    }

    // direction classes (:459-461), lane = neighbour; a neighbour's place in
    // run order (forward, backward, neither; CSR order within)
    int pos[NC];
    u64 closep[NC];  // close pairs, as bits over the places
    int n1 = 0, n2 = 0;
    {
        int cls[NC];
        bool cl[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            cls[c] = 3;
            cl[c] = false;
            if (NC > 1 && 64 * c >= deg) continue;
            const double4 q = c > 0 ? load_rec(c) : nb;
            const bool in = 64 * c + lane < deg;
            const double vx = q.x - ax, vy = q.y - ay;
            cl[c] = in && vx * vx + vy * vy < A.close_thr;  // :682 (DX^2 + DY^2, the same squares)
            if constexpr (FLT) {
                const float fx = static_cast<float>(ax) - static_cast<float>(q.x);
                const float fy = static_cast<float>(ay) - static_cast<float>(q.y);
                cl[c] = in && fx * fx + fy * fy < A.close_f;
            }
            int k;
            if constexpr (DIRECT) {
                k = 3;
                if (in) k = direct_class(ax, ay, ca, sa, q.x, q.y);
            } else if constexpr (SINES) {
                k = 3;
                if (in)
                    k = exact_direction(static_cast<float>(ax), static_cast<float>(ay), fth, static_cast<float>(q.x),
                                        static_cast<float>(q.y), fca, fsa);
            } else {
                // (direction_class's projection and a bound at least as strict)
                const double p = vx * ca + vy * sa;
                bool unsure = in && !(fabs(p) > (FLT ? 1e-5 : 1e-12) * (fabs(vx) + fabs(vy)));
                k = p > 0 ? 1 : 2;
                if constexpr (!FLT) {
                    // on whole pixels, neighbours along an axis or a diagonal:
                    // the reference's angle is one of eight, and its dot
                    // product (:459-461) is formed as it is
                    if (__builtin_amdgcn_ballot_w64(unsure) != 0ULL) {
                        if (unsure && (vx == 0.0 || vy == 0.0 || fabs(vx) == fabs(vy))) {
                            const double2 d = A.compass[4 + 3 * ((vy > 0.0) - (vy < 0.0)) + (vx > 0.0) - (vx < 0.0)];
                            const double dot = d.x * ca + d.y * sa;
                            k = dot > 0 ? 1 : 2;
                            unsure = dot == 0.0;  // (there is no third class here)
                        }
                    }
                }
                open |= __ballot(unsure);
            }
            cls[c] = in ? k : 3;
            n1 += __popcll(__ballot(cls[c] == 1));
            if (CLASSES) n2 += __popcll(__ballot(cls[c] == 2));
        }
        if (!CLASSES) {
            if (open != 0ULL) return true;  // (a neighbour across the anchor's direction)
            n2 = deg - n1;
        }
        int b1 = 0, b2 = n1, b0 = n1 + n2;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            auto below = [&](u64 m) {
                return static_cast<int>(__builtin_amdgcn_mbcnt_hi(
                    static_cast<unsigned>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(m), 0u)));
            };
            const u64 m1 = __ballot(cls[c] == 1);
            if constexpr (CLASSES) {
                const u64 m2 = __ballot(cls[c] == 2), m0 = __ballot(cls[c] == 0);
                pos[c] = cls[c] == 1 ? b1 + below(m1) : cls[c] == 2 ? b2 + below(m2) : b0 + below(m0);
                b2 += __popcll(m2);
                b0 += __popcll(m0);
            } else {
                const int f = below(m1);  // (no third class without exact directions)
                pos[c] = cls[c] == 1 ? b1 + f : b2 + lane - f;
                b2 += 64 - __popcll(m1);
            }
            pos[c] = cls[c] == 3 ? -1 : pos[c];
            b1 += __popcll(m1);
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) closep[c] = 0ULL;
#pragma unroll
        for (int c = 0; c < NC; ++c)
            for (u64 m = __ballot(cl[c]); m != 0ULL; m &= m - 1ULL) {  // (few: within 2 dx)
                const int at = __builtin_amdgcn_readlane(pos[c], __builtin_ctzll(m));
#pragma unroll
                for (int w = 0; w < NC; ++w)
                    if (NC == 1 || (at >> 6) == w) closep[w] |= 1ULL << (at & 63);
            }
    }

    // the pair records of batch b (that many places from its number times as many) into LDS: DX, DY,
    // DX^2 + DY^2 - dx^2, and for the lower and the upper orientation
    // constraint (theta_n -+ dt, by branch, :736, :799) the sine and cosine of
    // the angle and DX cos + DY sin
    auto fill_batch = [&](int b) {
        wave_sync();  // the last batch's reads are done
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            if (NC > 1 && 64 * c >= deg) continue;
            const double4 q = c > 0 ? load_rec(c) : nb;
            if constexpr (FLT) {
                // M_FLOAT: the sines and cosines, DX^2 and DY^2, DX, DY and
                // the angles, DX cos and DY sin
                const float fx = static_cast<float>(ax) - static_cast<float>(q.x);
                const float fy = static_cast<float>(ay) - static_cast<float>(q.y);
                const bool branch_a = (fx * fca + fy * fsa) < 0;  // :690
                double s[2], co[2];
                float T0[2], cx[2], sy[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const bool minus = (k == 0) == branch_a;
                    const float fn = static_cast<float>(nth);
                    const double d = minus ? -static_cast<double>(A.dt_f) : static_cast<double>(A.dt_f);
                    const double sd = minus ? -A.sin_dt : A.sin_dt;
                    T0[k] = minus ? fn - A.dt_f : fn + A.dt_f;
                    const double e = static_cast<double>(T0[k]) - (nth + d);
                    const double s0 = __builtin_fma(q.z, A.cos_dt, q.w * sd);
                    const double c0 = __builtin_fma(q.w, A.cos_dt, -(q.z * sd));
                    s[k] = __builtin_fma(e, __builtin_fma(-0.5 * e, s0, c0), s0);
                    co[k] = __builtin_fma(-e, __builtin_fma(0.5 * e, c0, s0), c0);
                    cx[k] = fx * sure(co[k], T0[k], true, pos[c] >= 0);  // :730-733
                    sy[k] = fy * sure(s[k], T0[k], false, pos[c] >= 0);
                }
                if (pos[c] >= 0 && (pos[c] >> kLog) == b) {
                    const lds_ptr<double2> o = rec + (pos[c] & kLast) * 5;
                    o[0].x = s[0];
                    o[0].y = co[0];
                    o[1].x = s[1];
                    o[1].y = co[1];
                    o[2].x = static_cast<double>(fx * fx);
                    o[2].y = static_cast<double>(fy * fy);
                    const lds_ptr<float4> f = (lds_ptr<float4>)(o + 3);
                    f[0].x = fx;
                    f[0].y = fy;
                    f[0].z = T0[0];
                    f[0].w = T0[1];
                    f[1].x = cx[0];
                    f[1].y = sy[0];
                    f[1].z = cx[1];
                    f[1].w = sy[1];
                }
                continue;
            }
            const double DX = ax - q.x, DY = ay - q.y;
            const bool branch_a = (DX * ca + DY * sa) < 0;  // :690
            if constexpr (DIRECT) {
                // DX, DY, the angles; below: DX cos and DY sin
                if (pos[c] >= 0 && (pos[c] >> kLog) == b) {
                    const double th = c > 0 ? A.th[A.ids[base + 64 * c + lane]] : nth;
                    const lds_ptr<double2> o = rec + (pos[c] & kLast) * 4;
                    o[0].x = DX;
                    o[0].y = DY;
                    o[3].x = branch_a ? th - A.exact.dt : th + A.exact.dt;
                    o[3].y = branch_a ? th + A.exact.dt : th - A.exact.dt;
                }
                continue;
            }
            const double sd = branch_a ? -A.sin_dt : A.sin_dt;
            const double s0 = __builtin_fma(q.z, A.cos_dt, q.w * sd), c0 = __builtin_fma(q.w, A.cos_dt, -(q.z * sd));
            const double s1 = __builtin_fma(q.z, A.cos_dt, -(q.w * sd)), c1 = __builtin_fma(q.w, A.cos_dt, q.z * sd);
            if (pos[c] >= 0 && (pos[c] >> kLog) == b) {
                const lds_ptr<double2> o = rec + (pos[c] & kLast) * 5;
                o[0].x = DX;
                o[0].y = DY;
                o[1].x = __builtin_fma(DX, DX, __builtin_fma(DY, DY, -A.dx2));
                o[1].y = __builtin_fma(DX, c0, DY * s0);
                o[2].x = __builtin_fma(DX, c1, DY * s1);
                o[2].y = s0;
                o[3].x = c0;
                o[3].y = s1;
                o[4].x = c1;
            }
        }
        wave_sync();
        if constexpr (DIRECT) {
            // lanes 0-31: the batch's angles; 32 on: with the first batch, the
            // anchor's with each offset (:702)
            const int kt = A.exact.kt;
            const bool mine = lane < 32 && (b << kLog) + (lane >> 1) < deg;
            const bool with_t2 = b == 0 && kt <= 32;
            const lds_ptr<double2> o = rec + (lane >> 1) * 4;
            double x = 0.0;
            if (mine) x = (lane & 1) != 0 ? o[3].y : o[3].x;
            if (with_t2 && lane >= 32) x = uload(A.th + a) + A.exact.off_t[min(lane - 32, kt - 1)];
            const double2 t = direct_sincos(x);
            if (mine) {
                o[1 + (lane & 1)].x = o[0].x * t.y;  // :730-733
                o[1 + (lane & 1)].y = o[0].y * t.x;
            }
            if (with_t2) {
#pragma unroll
                for (int m = 0; m < CPL; ++m) {
                    sT[m] = __shfl(t.x, 32 + W.j[m], 64);
                    cT[m] = __shfl(t.y, 32 + W.j[m], 64);
                }
            }
            wave_sync();
        }
    };

    // M_DIRECT: the transport sines of one group of pairs of the batch in LDS
    const int slog = DIRECT ? direct_pairs_log(A.exact.kt) : 0;
    const lds_ptr<double> sines = (lds_ptr<double>)(sl + cv.sines);
    auto fill_sines = [&](int group) {
        const int kt = A.exact.kt;
        const int items = 2 * kt * min(1 << slog, deg - (group << slog));
        const double th = uload(A.th + a);
        wave_sync();  // the last group's reads are done
#pragma unroll 1
        for (int t = lane; t < items; t += 64) {
            const int side = static_cast<int>((static_cast<float>(t) + 0.5f) * A.inv_kt);  // 2 pair + side
            const lds_ptr<double2> o = rec + (((group << slog) + (side >> 1)) & kLast) * 4;
            sines[t] = direct_sin(th + A.exact.off_t[t - side * kt] - ((side & 1) != 0 ? o[3].y : o[3].x));
        }
        wave_sync();
    };

    int batch = -1, group = -1;
    unsigned nacc = 0, vp = 0, isect_u = 0;  // isect_u: the wave's, isect: the lane's
    unsigned isect = 0;
    for (int run = 0; run < (CLASSES ? 3 : 2); ++run) {
        const int p0 = run == 0 ? 0 : (run == 1 ? n1 : n1 + n2);
        const int p1 = run == 0 ? n1 : (run == 1 ? n1 + n2 : deg);
        int R = 0;      // hypotheses of the run
        u64 place[NW];  // as bits over the places
#pragma unroll
        for (int w = 0; w < NW; ++w) place[w] = 0ULL;

        // the bundle of the pair at place p (record q, not close): the lane's
        // cells and, as bits, those with hi > lo (compute_curve_bundle, :636-819)
        auto bundle = [&](int p, lds_ptr<double2> q, Bounds (&v)[CPL]) __attribute__((always_inline)) -> u64 {
            if constexpr (FLT) {
                // compute_curve_bundle<float>; its branches differ (a
                // power of two on both sides of a quotient apart) in the
                // angles' order only
                const lds_ptr<float4> f = (lds_ptr<float4>)(q + 3);
                const float DX = f[0].x, DY = f[0].y;
                const double DX2 = q[2].x, DY2 = q[2].y;
                u64 any = 0ULL;
#pragma unroll
                for (int m = 0; m < CPL; ++m) {
                    const float o = static_cast<float>(W.ox[m]);
                    const float tt = sf[m] * DX - cf[m] * DY;  // :705
                    const float ttm = tt - o;
                    // :711 (the first product is exact)
                    const float den = static_cast<float>(
                        __builtin_fma(W.m2ox[m], static_cast<double>(tt), DX2) + DY2 - A.dx2 + W.ox2[m]);
                    const float kx0 = 2.0f * (ttm - A.dx_f) / den, kx1 = 2.0f * (ttm + A.dx_f) / den;
                    float kt[2];
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        const double s0 = q[k].x, c0 = q[k].y;
                        const float T0 = k == 0 ? f[0].z : f[0].w;
                        const float cx = k == 0 ? f[1].x : f[1].z, sy = k == 0 ? f[1].y : f[1].w;
                        const double e = static_cast<double>(T2[m] - T0) -
                                         (static_cast<double>(T2[m]) - static_cast<double>(T0));
                        const double s = __builtin_fma(sT[m], c0, -(cT[m] * s0));
                        const double c = __builtin_fma(cT[m], c0, sT[m] * s0);
                        const float sn = sure(__builtin_fma(e, __builtin_fma(-0.5 * e, s, c), s), T2[m] - T0, false, true);
                        kt[k] = sn / (-sn * o + cx + sy);
                    }
                    // the reference's compare-and-assign, which ignores NaN
                    const float lo = __builtin_fmaxf(__builtin_fmaxf(-A.max_k_f, kx0), kt[0]);
                    const float hi = __builtin_fminf(__builtin_fminf(A.max_k_f, kx1), kt[1]);
                    least = __builtin_fminf(__builtin_fminf(least, __builtin_fabsf(den)),
                                            __builtin_fminf(__builtin_fabsf(lo), __builtin_fabsf(hi)));
                    const bool ok = hi > lo;
                    v[m].lo = ok ? float_key(lo) : INT_MAX;
                    v[m].hi = ok ? float_key(hi) : INT_MIN;
                    any |= __builtin_amdgcn_ballot_w64(ok);
                }
                return any;
            } else if constexpr (DIRECT) {
                const double DX = q[0].x, DY = q[0].y, DX2 = DX * DX, DY2 = DY * DY;
                const double cx0 = q[1].x, sy0 = q[1].y, cx1 = q[2].x, sy1 = q[2].y;
                const bool branch_a = (DX * ca + DY * sa) < 0;  // :690
                const lds_ptr<double> sn = sines + 2 * A.exact.kt * (p & ((1 << slog) - 1));
                u64 any = 0ULL;
#pragma unroll
                for (int m = 0; m < CPL; ++m) {
                    double lo, hi;
                    cvg::bundle_cell(DX, DY, DX2, DY2, branch_a, W.ox[m], sT[m], cT[m], sn[W.j[m]], cx0, sy0,
                                     sn[W.j[m] + A.exact.kt], cx1, sy1, A.exact.dx, A.exact.dx2, A.exact.max_k, lo, hi);
                    v[m].lo = lo;
                    v[m].hi = hi;
                    any |= __builtin_amdgcn_ballot_w64(hi > lo);
                }
                return any;
            } else {
                const double DX = q[0].x, DY = q[0].y, r2 = q[1].x, C0 = q[1].y, C1 = q[2].x;
                const double s0n = q[2].y, c0n = q[3].x, s1n = q[3].y, c1n = q[4].x;
                u64 any = 0ULL;  // cells with hi > lo
#pragma unroll
                for (int m = 0; m < CPL; ++m) {
                    const double tt = __builtin_fma(sT[m], DX, -(cT[m] * DY));
                    const double den = __builtin_fma(W.ox[m], __builtin_fma(-2.0, tt, W.ox[m]), r2);
                    const double x0 = __builtin_fma(2.0, tt, -W.oxp2[m]);  // :712's numerator
                    const double s0 = __builtin_fma(sT[m], c0n, -(cT[m] * s0n));
                    const double s1 = __builtin_fma(sT[m], c1n, -(cT[m] * s1n));
                    const double d0 = __builtin_fma(-s0, W.ox[m], C0);
                    const double d1 = __builtin_fma(-s1, W.ox[m], C1);
                    // 1 / den, 1 / d0 and 1 / d1 (times scale) from one reciprocal
                    const double pp = den * d0, ppp = pp * d1;
                    double y = __builtin_amdgcn_rcp(ppp);
                    y = __builtin_fma(y, __builtin_fma(-ppp, y, 1.0), y);
                    y *= A.scale;
                    const double yd1 = y * pp, w = y * d1;
                    const double yd0 = w * den, yx = w * d0;
                    const double k0 = x0 * yx, k1 = __builtin_fma(A.four_dx, yx, k0);
                    // (clamped to +-max_k as the reference's: a bundle beyond the
                    // fixed-point range on both sides is not within the tolerance
                    // of an invalid cell's values)
                    const int lo = max(max(fix(k0), fix(s0 * yd0)), -kFixOne);
                    const int hi = min(min(fix(k1), fix(s1 * yd1)), kFixOne);
                    const int t = sub_sat(hi, lo);
                    note(t);
                    const bool ok = t > kFixTol;
                    // a small denominator (then the product is small as well)
                    // settles nothing unless its sign is certain and its
                    // quotients lie well beyond max_k, where they stay either way
                    if (__builtin_amdgcn_ballot_w64(!(fabs(ppp) >= A.min_prod)) != 0ULL) {
                        auto weak = [&](double n, double d) {
                            return !(fabs(d) >= A.min_den) &&
                                   !(fabs(d) > A.den_err && fabs(n) > 4.0 * A.max_k * fabs(d) + A.num_err);
                        };
                        const bool bad = weak(x0, den) || weak(x0 + A.four_dx, den) ||
                                         weak(s0, d0) || weak(s1, d1);
                        closest = bad ? 0u : closest;
                    }
                    v[m].lo = ok ? lo : INT_MAX;
                    v[m].hi = ok ? hi : INT_MIN;
                    any |= __builtin_amdgcn_ballot_w64(ok);
                }
                return any;
            }
        };
        V def_lo, def_hi;
        if constexpr (DIRECT) {
            def_lo = -A.exact.max_k;
            def_hi = A.exact.max_k;
        } else {
            def_lo = FLT ? float_key(-A.max_k_f) : -kFixOne;
            def_hi = FLT ? float_key(A.max_k_f) : kFixOne;
        }

        // the run's bundles, a batch of records at a time
        lds_ptr<Bounds> bp = bun;  // the next slot
        // (without a positive max_k no cell is valid, and only close pairs count)
        const bool barren = DIRECT && !(A.exact.max_k > 0.0);
        for (int p = p0; p < p1;) {
            if (!barren && (p >> kLog) != batch) {
                batch = p >> kLog;
                fill_batch(batch);
            }
            if (DIRECT && !barren && (p >> slog) != group) {
                group = p >> slog;
                fill_sines(group);
            }
            const int pe = min(p1, (DIRECT ? p | ((1 << slog) - 1) : p | kLast) + 1);
            constexpr int kRec = DIRECT ? 4 : 5;
            lds_ptr<double2> q = rec + (p & kLast) * kRec;
            if (!CLASSES && R + pe - p <= slots && ((closep[0] >> (p & 63)) & ((1ULL << (pe - p)) - 1ULL)) == 0ULL) {
                // (most batches: no close pair, and slots for all)
                for (; p < pe; ++p, q += kRec) {
                    Bounds v[CPL];
                    if (bundle(p, q, v) == 0ULL) continue;  // bundle_valid_check, :821-830
#pragma unroll
                    for (int m = 0; m < CPL; ++m) {
                        bp[m * 64].lo = v[m].lo;
                        bp[m * 64].hi = v[m].hi;
                    }
                    bp += CPL * 64;
                    place[0] |= 1ULL << (p & 63);
                }
                R = __popcll(place[0]);
                continue;
            }
            for (; p < pe; ++p, q += kRec) {
                bool close = false;
#pragma unroll
                for (int c = 0; c < NC; ++c)
                    if (NC == 1 || (p >> 6) == c) close = (closep[c] >> (p & 63)) & 1ULL;
                Bounds v[CPL];
                if (close) {
                    // the default bundle [-max_k, max_k]
#pragma unroll
                    for (int m = 0; m < CPL; ++m) {
                        v[m].lo = def_lo;
                        v[m].hi = def_hi;
                    }
                } else if (barren || bundle(p, q, v) == 0ULL) {
                    continue;
                }
                if (CLASSES) ++vp;
                if (CLASSES && run == 2) continue;
                if (R < slots) {
#pragma unroll
                    for (int m = 0; m < CPL; ++m) {
                        bp[m * 64].lo = v[m].lo;
                        bp[m * 64].hi = v[m].hi;
                    }
                    bp += CPL * 64;
                } else {
#pragma unroll
                    for (int m = 0; m < CPL; ++m) {
                        spl[((R - slots) * CPL + m) * 64].lo = v[m].lo;
                        spl[((R - slots) * CPL + m) * 64].hi = v[m].hi;
                    }
                }
#pragma unroll
                for (int w = 0; w < NW; ++w)
                    if (NW == 1 || (p >> 6) == w) place[w] |= 1ULL << (p & 63);
                ++R;
            }
        }
        if (!CLASSES) vp += static_cast<unsigned>(R);
        // a chain longer than 2 takes two hypotheses and G >= 3
        if ((CLASSES && run == 2) || R < 2 || G < 3) continue;

        u64 hyp[NW];  // the run's hypotheses as bits over the neighbour list
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            u64 word = place[0];
#pragma unroll
            for (int w = 1; w < NW; ++w)
                if ((pos[c] >> 6) == w) word = place[w];
            hyp[c] = __builtin_amdgcn_ballot_w64(pos[c] >= 0 && ((word >> (pos[c] & 63)) & 1ULL) != 0ULL);
        }
        auto put_row = [&](unsigned rank, const u64 (&chain)[NW], int best, int seed) {
            const size_t q = static_cast<size_t>(base) + rank;
            if constexpr (FLT) {
                // the slots' edges are in `pm`; k_max and k_min over the
                // members' and the seed's bundles at the best cell
                const lds_ptr<int> slot_id = (lds_ptr<int>)pm;
                const lds_ptr<Bounds> at = (lds_ptr<Bounds>)(sl + cv.bun) + best;
                const mem_ptr<Bounds> far = (mem_ptr<Bounds>)spill + best;
                const mem_ptr<int> ids = (mem_ptr<int>)A.st_ids + q * A.st_stride;
                int len = 0, lo = INT_MIN, hi = INT_MAX;
                ids[len++] = a;
                for (u64 set = chain[0] | 1ULL << seed; set != 0ULL; set &= set - 1ULL) {
                    const int s = __builtin_ctzll(set);
                    if ((chain[0] >> s) & 1ULL) ids[len++] = slot_id[s];
                    int l, h;
                    if (s < slots) {
                        l = at[s * CPL * 64].lo;
                        h = at[s * CPL * 64].hi;
                    } else {
                        l = far[(s - slots) * CPL * 64].lo;
                        h = far[(s - slots) * CPL * 64].hi;
                    }
                    lo = max(lo, l);
                    hi = min(hi, h);
                }
                ((mem_ptr<unsigned>)A.st_meta)[q] = static_cast<unsigned>(len) | (run == 0 ? 0x8000u : 0u) |
                                                    static_cast<unsigned>(A.rank_cell[best]) << 16;
                ((mem_ptr<double>)A.st_k)[2 * q] = static_cast<double>(key_float(hi));
                ((mem_ptr<double>)A.st_k)[2 * q + 1] = static_cast<double>(key_float(lo));
                return;
            }
#pragma unroll
            for (int w = 0; w < NW; ++w)
                if (w == 0 || deg > 64) {
                    const mem_ptr<ulonglong2> o = (mem_ptr<ulonglong2>)A.st_mask + w * A.mask_plane + q;
                    o->x = hyp[w];
                    o->y = chain[w];
                }
            ((mem_ptr<unsigned>)A.st_meta)[q] = row_meta(best, run == 0, deg > 64, seed);
            if constexpr (DIRECT) {
                if (A.st_k == nullptr) return;  // (the record forms them)
                // the running bundle at the best cell, the seed's first (:838-841)
                const lds_ptr<Bounds> at = (lds_ptr<Bounds>)(sl + cv.bun) + best;
                const mem_ptr<Bounds> far = (mem_ptr<Bounds>)spill + best;
                double lo = 0.0, hi = 0.0;
                int s = seed;
                u64 set[NW];
#pragma unroll
                for (int w = 0; w < NW; ++w) set[w] = chain[w];
                for (bool first = true;; first = false) {
                    double l, h;
                    if (s < slots) {
                        l = at[s * CPL * 64].lo;
                        h = at[s * CPL * 64].hi;
                    } else {
                        l = far[(s - slots) * CPL * 64].lo;
                        h = far[(s - slots) * CPL * 64].hi;
                    }
                    lo = first || lo < l ? l : lo;
                    hi = first || hi > h ? h : hi;
                    s = -1;
#pragma unroll
                    for (int w = 0; w < NW; ++w)
                        if (s < 0 && set[w] != 0ULL) {
                            s = 64 * w + __builtin_ctzll(set[w]);
                            set[w] &= set[w] - 1ULL;
                        }
                    if (s < 0) break;
                }
                ((mem_ptr<double>)A.st_k)[2 * q] = hi;
                ((mem_ptr<double>)A.st_k)[2 * q + 1] = lo;
            }
        };
        auto best_cell = [&](const u64 (&valid)[CPL]) -> int {  // fill_curvelet_info, :202-226
            int best = -1;
#pragma unroll
            for (int m = 0; m < CPL; ++m) {
                const u64 e = valid[m] & W.emask[m];
                if (best < 0 && e != 0ULL) best = 64 * m + __builtin_ctzll(e);
            }
            return best < 0 ? A.rank_of_cell0 : best;
        };
        auto slot_ids = [&]() {  // M_FLOAT: the slots' edges into `pm`
            if constexpr (FLT) {
                wave_sync();  // the last reads there are done, and every bundle is written
                if (__builtin_amdgcn_inverse_ballot_w64(hyp[0]))
                    ((lds_ptr<int>)pm)[__builtin_amdgcn_mbcnt_hi(
                        static_cast<unsigned>(hyp[0] >> 32),
                        __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(hyp[0]), 0u))] = nid;
                wave_sync();
            }
        };
        auto rank_of = [&](u64 acc) -> unsigned {
            return nacc + static_cast<unsigned>(__builtin_amdgcn_mbcnt_hi(
                              static_cast<unsigned>(acc >> 32),
                              __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(acc), 0u)));
        };

        if (R <= kSmallRun) {
            // the compatibility masks of every two slots: lane 8 i + k, the
            // cells where slots i and k are valid together
            Bounds b[kSmallRun][CPL];
            u64 own[kSmallRun][CPL];  // M_DIRECT: the slots' own valid cells
            u64 P[CPL];
#pragma unroll
            for (int m = 0; m < CPL; ++m) P[m] = 0ULL;
            auto meet = [&](auto slot) -> bool {
                constexpr int i = decltype(slot)::value;
                if (i >= R) return false;
                asm volatile("");  // (a branch: runs of 2 to 4 slots would do the work of 8)
#pragma unroll
                for (int m = 0; m < CPL; ++m) {
                    b[i][m].lo = bun[(i * CPL + m) * 64].lo;
                    b[i][m].hi = bun[(i * CPL + m) * 64].hi;
                    own[i][m] = __builtin_amdgcn_ballot_w64(b[i][m].hi > b[i][m].lo);
                    P[m] = set_lane64(P[m], own[i][m], 9 * i);
                }
#pragma unroll
                for (int k = 0; k < i; ++k) {
#pragma unroll
                    for (int m = 0; m < CPL; ++m) {
                        if constexpr (DIRECT) {
                            const u64 both = __builtin_amdgcn_ballot_w64(b[k][m].hi > b[i][m].lo) &
                                             __builtin_amdgcn_ballot_w64(b[i][m].hi > b[k][m].lo);
                            P[m] = set_lane64(P[m], both & own[i][m] & own[k][m], 8 * i + k);
                        } else {
                            const int t = min(sub_sat(b[k][m].hi, b[i][m].lo), sub_sat(b[i][m].hi, b[k][m].lo));
                            note(t);
                            P[m] = set_lane64(P[m], __builtin_amdgcn_ballot_w64(t > kTol), 8 * i + k);
                        }
                    }
                }
                return true;
            };
            each(meet, std::make_integer_sequence<int, kSmallRun>{});
            // the upper triangle, and the rows in LDS
            u64 C[CPL];
            wave_sync();  // (the last matrix's reads are done)
#pragma unroll
            for (int m = 0; m < CPL; ++m) {
                C[m] = P[m] | perm64((lane & 7) << 3 | lane >> 3, P[m]);
                pm[m * 64 + lane] = C[m];
            }
            wave_sync();
            // growth (:479-536): step h offers slot h to every seed's chain.
            // Lane (j, h'): C = the cells where seed j's running bundle and
            // slot h' are valid together; taking h leaves of them those where
            // h is valid with the chain and with h'.
            const bool limited = R > G - 1;  // a chain can fill up
            const u64 ones = 0x0101010101010101ULL;
            u64 count = 0ULL, stop = 0ULL;  // per seed, one byte each
            u64 chain = 0ULL;               // byte j: seed j's chain, as slots
            auto grow = [&](auto slot, auto full) -> bool {
                constexpr int h = decltype(slot)::value;
                constexpr bool limited = decltype(full)::value;
                if (h >= R) return false;
                u64 nz = 0ULL;
#pragma unroll
                for (int m = 0; m < CPL; ++m) nz |= C[m];
                const u64 okb = __builtin_amdgcn_ballot_w64(
                    (static_cast<unsigned>(nz) | static_cast<unsigned>(nz >> 32)) != 0u);
                // the seed joins at its own distance rank (:496-510)
                u64 rows = ((okb >> h) & ones) | 1ULL << (8 * h);
                if (limited) rows &= ~stop;
                const bool take = __builtin_amdgcn_inverse_ballot_w64((rows << 8) - rows);
#pragma unroll
                for (int m = 0; m < CPL; ++m) {
                    // (lane & 56) | h's value: ds_swizzle, within 8 lanes
                    const unsigned lo = static_cast<unsigned>(
                        __builtin_amdgcn_ds_swizzle(static_cast<int>(C[m]), h << 5 | 0x18));
                    const unsigned hi = static_cast<unsigned>(
                        __builtin_amdgcn_ds_swizzle(static_cast<int>(C[m] >> 32), h << 5 | 0x18));
                    const u64 n = C[m] & (static_cast<u64>(hi) << 32 | lo) & pm[m * 64 + 8 * h + (lane & 7)];
                    C[m] = take ? n : C[m];
                }
                chain |= rows << h;
                if (limited) {
                    count += rows;
                    stop = ((count + (128ULL - static_cast<u64>(G - 1)) * ones) >> 7) & ones;
                }
                return true;
            };
            if (limited) {
                auto step = [&](auto slot) -> bool { return grow(slot, std::true_type{}); };
                each(step, std::make_integer_sequence<int, kSmallRun>{});
            } else {
                auto step = [&](auto slot) -> bool { return grow(slot, std::false_type{}); };
                each(step, std::make_integer_sequence<int, kSmallRun>{});
            }
            // rows, lane 9 j = seed j: kept with more than 2 edges (:549) and
            // no earlier seed with the same chain (lane 8 j + k compares j's
            // with k's)
            const int j = lane >> 3, k = lane & 7;
            const unsigned cj = static_cast<unsigned>(chain >> (lane & 56)) & 0xffu;
            const unsigned ck = static_cast<unsigned>(chain >> (8 * k)) & 0xffu;
            const u64 dup = __builtin_amdgcn_ballot_w64(cj == ck && k < j);
            const int members = __popc(cj);
            if (!limited) {
                isect_u += static_cast<unsigned>(R * (R - 1));  // every seed meets every other hypothesis
            } else if (j == k && j < R) {
                // the slots the reference's loop visits, without the seed's own step
                const int visited = members + 1 >= G ? 32 - __clz(static_cast<int>(cj)) : R;
                isect += static_cast<unsigned>(visited - (j < visited ? 1 : 0));
            }
            const bool keep = j == k && j < R && members >= 2 && ((dup >> (lane & 56)) & 0xffULL) == 0ULL;
            const u64 acc = __builtin_amdgcn_ballot_w64(keep);
            if (FLT && acc != 0ULL) slot_ids();
            if (keep) {
                u64 row[NW];
#pragma unroll
                for (int w = 0; w < NW; ++w) row[w] = w == 0 ? static_cast<u64>(cj) : 0ULL;
                put_row(rank_of(acc), row, best_cell(C), j);
            }
            nacc += static_cast<unsigned>(__popcll(acc));
            continue;
        }

        auto valid_lanes = [&](const Bounds &b) -> u64 {
            if constexpr (DIRECT)
                return __builtin_amdgcn_ballot_w64(b.hi > b.lo);
            else
                return __builtin_amdgcn_ballot_w64(sub_sat(b.hi, b.lo) > kTol);
        };
        // longer runs: seed by seed, lane = cell: the running bundle over the
        // hypotheses in CSR order
        u64 sm[NC][NW];   // lane = seed (of chunk c): the chain's slots
        u64 sM[NC][CPL];  // and the running bundle's valid cells
#pragma unroll
        for (int c = 0; c < NC; ++c) {
#pragma unroll
            for (int w = 0; w < NW; ++w) sm[c][w] = 0ULL;
#pragma unroll
            for (int m = 0; m < CPL; ++m) sM[c][m] = 0ULL;
        }
        for (int j = 0; j < R; ++j) {
            Bounds cur[CPL], nx[CPL];
#pragma unroll
            for (int m = 0; m < CPL; ++m) {
                cur[m] = get_bundle(j, m);
                nx[m] = get_bundle(0, m);
            }
            u64 S[NW];
#pragma unroll
            for (int w = 0; w < NW; ++w) S[w] = 0ULL;
            int len = 1, h = 0;
            for (; h < R && len < G; ++h) {
                Bounds n[CPL];
                u64 T = 0ULL;
#pragma unroll
                for (int m = 0; m < CPL; ++m) {
                    n[m].lo = larger(cur[m].lo, nx[m].lo);
                    n[m].hi = smaller(cur[m].hi, nx[m].hi);
                    T |= valid_lanes(n[m]);
                }
                const int hn = h + 1 < R ? h + 1 : h;
#pragma unroll
                for (int m = 0; m < CPL; ++m) nx[m] = get_bundle(hn, m);
                if constexpr (MODE == M_FAST) {
                    if (T == 0ULL && h != j) {
                        // (a step with a certainly valid cell is settled by it)
#pragma unroll
                        for (int m = 0; m < CPL; ++m) note(sub_sat(n[m].hi, n[m].lo));
                    }
                }
                if (h == j || T != 0ULL) {
#pragma unroll
                    for (int m = 0; m < CPL; ++m) cur[m] = n[m];
#pragma unroll
                    for (int w = 0; w < NW; ++w)
                        if (NW == 1 || (h >> 6) == w) S[w] |= 1ULL << (h & 63);
                    ++len;
                }
            }
#pragma unroll
            for (int m = 0; m < CPL; ++m) {
                if constexpr (MODE == M_FAST) note(sub_sat(cur[m].hi, cur[m].lo));
                const u64 T = valid_lanes(cur[m]);
#pragma unroll
                for (int c = 0; c < NC; ++c)
                    if (NC == 1 || (j >> 6) == c) sM[c][m] = set_lane64(sM[c][m], T, j & 63);
            }
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int w = 0; w < NW; ++w)
                    if (NC == 1 || (j >> 6) == c) sm[c][w] = set_lane64(sm[c][w], S[w], j & 63);
        }
        // rows, lane = seed (as above)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            if (NC > 1 && 64 * c >= R) break;
            const int j = 64 * c + lane;
            const bool in = j < R;
            int members = 0, top = -1;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                members += __popcll(sm[c][w]);
                if (sm[c][w] != 0ULL) top = 64 * w + 63 - __clzll(static_cast<long long>(sm[c][w]));
            }
            if (in) {
                const int visited = members + 1 >= G ? top + 1 : R;
                isect += static_cast<unsigned>(visited - (j < visited ? 1 : 0));
            }
            u64 acc = __builtin_amdgcn_ballot_w64(in && members >= 2);
#pragma unroll
            for (int cc = 0; cc <= c; ++cc) {
                const int kend = min(64, R - 64 * cc);
                for (int k = 0; k < kend; ++k) {
                    u64 same = cc < c ? ~0ULL : ~1ULL << k;  // the later seeds
#pragma unroll
                    for (int w = 0; w < NW; ++w)
                        same &= __builtin_amdgcn_ballot_w64(get_lane64(sm[cc][w], k) == sm[c][w]);
                    acc &= ~same;
                }
            }
            if (FLT && acc != 0ULL) slot_ids();
            if (__builtin_amdgcn_inverse_ballot_w64(acc)) put_row(rank_of(acc), sm[c], best_cell(sM[c]), j);
            nacc += static_cast<unsigned>(__popcll(acc));
        }
    }
    if (MODE == M_FAST && __builtin_amdgcn_ballot_w64(closest <= 2u * kFixTol) != 0ULL) return true;
    if (FLT && __builtin_amdgcn_ballot_w64(bad != 0u || least == 0.0f) != 0ULL) return true;
    if (lane == 0) ((mem_ptr<unsigned>)A.acc_count)[a] = nacc;
    vp_sum += vp;
    isect_sum += isect + (lane == 0 ? isect_u : 0u);
    return false;
}

// A wave's anchors for another list, kept in LDS and appended several at a
// time: an atomic each, ~11 ns on the one counter, took 2 ms where most anchors
// of a 1080p map were left open.
struct LeftOpen {
    const FusedArgs &A;
    lds_ptr<int> buf;
    int list, count = 0;
    __device__ void put(int a)
    {
        if ((threadIdx.x & 63) == 0) buf[count] = a;
        if (++count == kLeftOpen) flush();
    }
    __device__ void flush()
    {
        if (count == 0) return;
        wave_sync();
        const int lane = threadIdx.x & 63;
        unsigned at = 0;
        if (lane == 0) at = atomicAdd(A.list_len + list * kBucketStride, static_cast<unsigned>(count));
        at = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(at)));
        if (lane < count) {
            const int a = buf[lane];
            const unsigned o0 = A.off[a], o1 = A.off[a + 1];
            A.lists[entry_place(list, static_cast<long long>(at) + lane, A.n)] =
                make_int4(a, static_cast<int>(o0), static_cast<int>(o1 - o0), 0);
        }
        wave_sync();
        count = 0;
    }
};

// One wave's sums into its place (k_record adds the places up).
__device__ __forceinline__ void put_sums(unsigned *partial, int g, unsigned vp, unsigned long long isect)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        isect += static_cast<unsigned long long>(__shfl_xor(static_cast<long long>(isect), o, 64));
    if ((threadIdx.x & 63) == 0) {
        partial[3 * g] = vp;
        partial[3 * g + 1] = static_cast<unsigned>(isect);
        partial[3 * g + 2] = static_cast<unsigned>(isect >> 32);
    }
}

template <int CPL>
__device__ __forceinline__ WaveCells<CPL> wave_cells(const FusedArgs &A)
{
    WaveCells<CPL> W;
#pragma unroll
    for (int m = 0; m < CPL; ++m) {
        const int rho = static_cast<int>(threadIdx.x & 63) + 64 * m;
        const bool live = rho < A.K;
        const int r = live ? rho : 0;
        W.ox[m] = A.rank_ox[r];
        W.m2ox[m] = -2.0 * W.ox[m];
        W.ox2[m] = static_cast<double>(static_cast<float>(W.ox[m]) * static_cast<float>(W.ox[m]));
        W.oxp2[m] = 2.0 * (W.ox[m] + A.dx);
        W.ot[m] = A.rank_ot[r];
        W.j[m] = A.rank_cell[r] % A.exact.kt;
        W.so[m] = A.rank_so[r];
        W.co[m] = A.rank_co[r];
        W.emask[m] = __ballot(live && A.rank_elig[r] != 0);
    }
    return W;
}

__device__ __forceinline__ void load_entry(const int4 *p, int &a, unsigned &base, int &deg)
{
    const int *e = reinterpret_cast<const int *>(p);
    a = uload(e);
    base = static_cast<unsigned>(uload(e + 1));
    deg = uload(e + 2);
}

// build_curvelets_greedy (cpu_curvelet.hpp:437-591) plus the
// form_pairwise_bundles valid-pair count (:305-361), in one pass, for anchors
// of up to 64 neighbours.
//
// Persistent: one wave per anchor (do_anchor), wave g takes entries g,
// g + waves, ... of the concatenated lists.  The neighbours' records of the
// next anchor, the ids of the one after it and the list entry of the third are
// in flight while an anchor is worked on.  Bound by instruction issue and
// latency together: on the 1080p map one to four waves per SIMD take 1,145,
// 723, 574 and 516 us, five 473 (432 with bounds clamped as they are formed, in
// place of two differences a cell; 752 vector, 475 scalar and 90 LDS
// instructions an anchor).  Anchors with a comparison too close
// for the approximate bounds go to the open list.  (Done again here, their
// code costs the main loop its registers: 1,272 us against 720 on the 1080p
// map.)
template <int CPL, bool FLT>
__global__ __launch_bounds__(64 * kFusedWaves, waves_per_simd(CPL, FLT))
void k_curvelets(FusedArgs A)
{
    extern __shared__ double lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int g = static_cast<int>(blockIdx.x) * kFusedWaves + wave;
    const int streams = static_cast<int>(gridDim.x) * kFusedWaves;
    unsigned vp = 0;               // valid or close pairs of this wave's anchors
    unsigned long long isect = 0;  // bundle intersections the reference tests (per lane)
    char *sl = reinterpret_cast<char *>(lds) + static_cast<size_t>(wave) * slice_carve(A.slots, CPL).bytes;
    char *spill = A.spill + static_cast<size_t>(g) * A.spill_stride;
    const WaveCells<CPL> W = wave_cells<CPL>(A);

    // the wave's entries: a cursor into the current list
    int list = L_FIRST - 1, left = 0, at = g;
    auto next = [&](int &ea, unsigned &eb, int &ed) {
        ed = -1;
        while (at >= left) {
            at -= left;
            if (list == kLists - 1) return;
            ++list;
            left = static_cast<int>(uload(A.list_len + list * kBucketStride));
        }
        load_entry(A.lists + entry_place(list, at, A.n), ea, eb, ed);
        at += streams;
    };
    auto load_id = [&](unsigned b0, int d0) -> int { return lane < d0 ? A.ids[b0 + lane] : -1; };
    auto load_rec = [&](int id) -> double4 {
        double4 v = make_double4(0.0, 0.0, 0.0, 1.0);
        if (id >= 0) v = A.rec[id];
        return v;
    };
    auto load_th = [&](int id) -> double { return FLT && id >= 0 ? A.th[id] : 0.0; };
    int a = 0, deg, na = 0, ndeg = -1;
    unsigned base = 0, nbase = 0;
    next(a, base, deg);
    int id = load_id(base, deg);
    double4 nb = load_rec(id);
    double nth = load_th(id);
    if (deg >= 0) next(na, nbase, ndeg);
    int nid = load_id(nbase, ndeg);
    LeftOpen open{A, (lds_ptr<int>)(sl + slice_carve(A.slots, CPL).left), L_OPEN};
    // (where most anchors turn out open, the rest go there at once: their work
    // here would be done twice)
    int lead = -6;  // the open anchors' over the others
    while (deg >= 0 && lead < 0) {
        // start the next anchor's loads
        const double4 nnb = load_rec(nid);
        const double nnth = load_th(nid);
        int nna = 0, nndeg = -1;
        unsigned nnbase = 0;
        if (ndeg >= 0) next(nna, nnbase, nndeg);
        const int nnid = load_id(nnbase, nndeg);
        --lead;
        if (do_anchor<CPL, 1, FLT ? M_FLOAT : M_FAST>(A, W, sl, spill, a, base, deg, id, nb, nth, vp, isect)) {
            lead += 2;
            open.put(a);
        }
        a = na;
        base = nbase;
        deg = ndeg;
        nb = nnb;
        nth = nnth;
        id = nid;
        na = nna;
        nbase = nnbase;
        ndeg = nndeg;
        nid = nnid;
    }
    if (deg >= 0) open.put(a);
    if (ndeg >= 0) open.put(na);
    open.flush();
    while (ndeg >= 0) {
        // the wave's next 64 entries, one to a lane
        int l = list, rest = left;
        long long i = at + static_cast<long long>(lane) * streams;
        while (l < kLists && i >= rest) {
            i -= rest;
            ++l;
            rest = l < kLists ? static_cast<int>(A.list_len[l * kBucketStride]) : 0;
        }
        const bool some = l < kLists;
        const unsigned long long m = __ballot(some);
        if (m == 0ULL) break;
        unsigned to = 0;
        if (lane == 0)
            to = atomicAdd(A.list_len + L_OPEN * kBucketStride, static_cast<unsigned>(__popcll(m)));
        to = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(to)));
        if (some) A.lists[entry_place(L_OPEN, static_cast<long long>(to) + lane, A.n)] = A.lists[entry_place(l, i, A.n)];
        if (m != ~0ULL) break;
        // (on from the last lane's place)
        list = __builtin_amdgcn_readlane(l, 63);
        left = __builtin_amdgcn_readlane(rest, 63);
        at = __builtin_amdgcn_readlane(static_cast<int>(i), 63) + streams;
    }
    put_sums(A.partial, g, vp, isect);
}

// A wave's entries of lists first .. last: numbers at, at + step, ... of their
// concatenation.
struct ListCursor {
    const FusedArgs &A;
    int list, last, left, at, step;
    __device__ ListCursor(const FusedArgs &a, int first, int last_, int g, int step_)
        : A(a), list(first - 1), last(last_), left(0), at(g), step(step_)
    {
    }
    // deg = -1 at the end
    __device__ __forceinline__ void next(int &a, unsigned &base, int &deg)
    {
        deg = -1;
        while (at >= left) {
            at -= left;
            if (list == last) {
                left = 0;
                return;
            }
            ++list;
            left = static_cast<int>(uload(A.list_len + list * kBucketStride));
        }
        load_entry(A.lists + entry_place(list, at, A.n), a, base, deg);
        at += step;
    }
};

// The anchors of some lists on their own bounds: those k_curvelets left open,
// those of 65 to 256 neighbours, or all of a map that k_curvelets' error bound
// does not cover.  One wave per workgroup; the grid is what stays resident, since
// on whole-pixel maps most anchors can be open, and waves without an anchor leave
// at once (k_record adds up the others' sums).  Three waves a SIMD for lists of
// more than 64, whose masks four leave no registers for: 30,000 edges of 200
// neighbours each 4.56 ms against 4.80.  Bound by instruction issue: all
// 207,326 anchors of the 1080p map take 1,090 us, 2,100 vector and 912 scalar
// instructions each.  (Fourteen waves a CU in place of sixteen, with 80 B records
// and 112 sines at a time, and the anchor's and pairs' sines in two calls: 1,370.
// Quotients of one denominator on one refined reciprocal: 1,070.)
template <int CPL, int NW>
__global__ __launch_bounds__(64, CPL == 1 ? (NW == 1 ? 4 : 3) : 2) void k_curvelets_direct(FusedArgs A, int first, int last)
{
    extern __shared__ double lds[];
    const int lane = threadIdx.x & 63;
    const int g = static_cast<int>(blockIdx.x);
    ListCursor entries(A, first, last, g, static_cast<int>(gridDim.x));
    int a = 0, deg;
    unsigned base = 0;
    entries.next(a, base, deg);
    if (deg < 0 && first == last) return;
    unsigned vp = 0;
    unsigned long long isect = 0;
    const WaveCells<CPL> W = wave_cells<CPL>(A);
    char *spill = A.spill + static_cast<size_t>(g) * A.spill_stride;
    int id = lane < deg ? A.ids[base + lane] : -1;
    while (deg >= 0) {
        const double4 nb = id >= 0 ? A.rec[id] : make_double4(0.0, 0.0, 0.0, 1.0);
        const double nth = id >= 0 ? A.th[id] : 0.0;
        int na = 0, ndeg;
        unsigned nbase = 0;
        entries.next(na, nbase, ndeg);
        id = lane < ndeg ? A.ids[nbase + lane] : -1;
        (void)do_anchor<CPL, NW, M_DIRECT>(A, W, reinterpret_cast<char *>(lds), spill, a, base, deg, 0, nb, nth, vp,
                                           isect);
        a = na;
        base = nbase;
        deg = ndeg;
    }
    put_sums(A.partial, g, vp, isect);
}

// Float maps: the anchors k_curvelets left open.  Those with a zero bound or
// denominator join the wide ones, for the general kernel.
template <int CPL>
__global__ __launch_bounds__(64, waves_per_simd(CPL, true)) void k_curvelets_float_open(FusedArgs A)
{
    extern __shared__ double lds[];
    const int lane = threadIdx.x & 63;
    const int g = static_cast<int>(blockIdx.x);
    const int total = static_cast<int>(uload(A.list_len + L_OPEN * kBucketStride));
    if (g >= total) return;
    unsigned vp = 0;
    unsigned long long isect = 0;
    const WaveCells<CPL> W = wave_cells<CPL>(A);
    char *spill = A.spill + static_cast<size_t>(g) * A.spill_stride;
    char *sl = reinterpret_cast<char *>(lds);
    LeftOpen zero{A, (lds_ptr<int>)(sl + slice_carve(A.slots, CPL).left), L_WIDE};
    for (int L = g; L < total; L += static_cast<int>(gridDim.x)) {
        int a, deg;
        unsigned base;
        load_entry(A.lists + entry_place(L_OPEN, L, A.n), a, base, deg);
        const int id = lane < deg ? A.ids[base + lane] : -1;
        const double4 nb = id >= 0 ? A.rec[id] : make_double4(0.0, 0.0, 0.0, 1.0);
        const double nth = id >= 0 ? A.th[id] : 0.0;
        if (do_anchor<CPL, 1, M_FLOAT_EXACT>(A, W, sl, spill, a, base, deg, id, nb, nth, vp, isect)) zero.put(a);
    }
    zero.flush();
    put_sums(A.partial, g, vp, isect);
}

using FusedKernel = void (*)(FusedArgs);
using DirectKernel = void (*)(FusedArgs, int, int);

// by cells per lane
template <bool FLT>
inline FusedKernel fused_kernel(int cpl)
{
    return cpl == 1 ? k_curvelets<1, FLT> : (cpl == 2 ? k_curvelets<2, FLT> : k_curvelets<4, FLT>);
}
inline FusedKernel float_open_kernel(int cpl)
{
    return cpl == 1 ? k_curvelets_float_open<1> : (cpl == 2 ? k_curvelets_float_open<2> : k_curvelets_float_open<4>);
}
template <int NW>
inline DirectKernel direct_kernel(int cpl)
{
    return cpl == 1 ? k_curvelets_direct<1, NW> : (cpl == 2 ? k_curvelets_direct<2, NW> : k_curvelets_direct<4, NW>);
}

#endif
