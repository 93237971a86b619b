// resident.hip -- the x and y sweeps of whole z planes held in LDS, and the FP64 x sweep of strips of
// rows where planes do not fit (k_strip).
//
// The kernels of lod.hip stream a line through a ring of rows and keep of it what fits on chip;
// they are made for lines and fields far larger than a CU's storage.  Where a z plane of one
// substrate fits into a CU's LDS (FP64 up to about 139 x 139, FP32 200 x 200), k_plane applies the
// cell sources and sinks, the x sweep and the y sweep to it there: both sweeps stay inside the
// plane, so the field crosses the memory system once instead of twice, the agents' voxels are
// updated without a pass of their own, and a step is two launches (planes, z sweep).
//
// What bounds it is the recurrence, one line per lane: at most ceil(lines / 64) wavefronts of a
// workgroup are at work, and a single wavefront issues about one operation per 6 clocks, dependent
// or not (LDS latency: 90 clocks).  So what counts is operations per row: a forward row divides by
// a reciprocal pair (2 operations, div_corr takes 5), a backward row is one operation, and the
// Thomas tables of a line are staged in LDS beside it and read by broadcast.  (Read by scalar
// loads, as in lod.hip, they arrived one memory latency per batch late, since a launch starts
// with cold scalar caches and the compiler sinks such loads to their use: 94 and 90 clocks per
// forward and backward row of a 128 x 128 FP64 plane instead of 67 and 43.)
//
// Microseconds per step of sweeps (separate sweeps -> planes and z sweep; in brackets x + y ->
// planes): FP64 50^3 x 1 34 -> 20, 97 x 61 x 83 x 3 66 -> 32, 128^3 x 2 79 -> 44 (53 -> 25),
// 128^3 x 8 193 -> 128 (138 -> 77, 3.5 TB/s of the 5.0 a copy reaches), 139^3 x 8 317 -> 195; FP32
// 64^3 x 4 33 -> 22, 160^3 x 4 127 -> 100, 200^3 x 2 150 -> 100, 200^3 x 8 448 -> 296.  Every shape
// tried whose planes fit (16^3 to 200^3, 16 x 16 x 512) was at least as fast.
//
// The tables of settled rows (forward_line) are kept in registers; read from LDS for every row:
// 128^3 x 2 FP64 46, 128^3 x 8 137, 200^3 x 8 FP32 313.
//
// Tried and dropped: whole z lines in LDS, 64 or 32 per workgroup (slower than the z sweep of
// lod.hip at every size: 128^3 x 2 FP64 step 55 against 49 us); the next plane's loads issued by
// the solving threads (24 us per 128 x 128 FP64 plane, with loading wavefronts 21); one element
// per load (k_plane's loaders then overflow the instruction cache in FP32, 190 x 190 planes twice
// as slow); the last sweep's results to LDS and out by all wavefronts instead of a row at a time by
// the solvers (200^3 x 8 FP32 340 instead of 296).
#include <algorithm>
#include <type_traits>

#include "bfvmb_internal.hpp"

namespace bfvmb {
namespace {

typedef const __attribute__((address_space(4))) double *ctab;
__device__ __forceinline__ ctab as_ctab(const double *p) { return (ctab)p; }

// Field values go through the global address space: a generic (flat) access also counts on the
// LDS counter, so every wait for LDS would drain the next plane's loads.
template <class T>
using gmem = __attribute__((address_space(1))) T *;
template <class T>
__device__ __forceinline__ gmem<T> as_global(T *p)
{
    return (gmem<T>)p;
}

__device__ __forceinline__ int find_domain(const long long *prefix, int ndom, long long t)
{
    int lo = 0, hi = ndom - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (prefix[mid] <= t)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// Workgroup barrier that orders LDS only: __syncthreads() also waits for every global access in
// flight, and with it for the next plane's loads.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// How a forward row divides by its denominator (FP64 storage; FP32 storage multiplies by rden).
// All three give the correctly rounded quotient for the numerators they are used on.
enum Division {
    kPair,  // fma(a, rden, a*rlow): rows with a reciprocal pair (reciprocal_pair, thomas.cpp)
    kCorr,  // a*rden and two corrections (Markstein): a substrate with a row that has no pair
    kTrue   // IEEE division: tiny, infinite or NaN numerators
};

// Key of a numerator that kPair and kCorr must not divide: with h = the upper 32 bits of its
// pattern, (h << 1) - (kTinyHi << 1) (mod 2^32; the shift drops the sign) is below kKeyBad
// exactly when 2^-900 <= |a| < inf (below, the low product or the correction's residual may
// underflow).  A line keeps the largest key it met.
constexpr unsigned kTinyHi = (1023u - 900u) << 20;
constexpr unsigned kKeyBad = (0x7ff00000u << 1) - (kTinyHi << 1);
__device__ __forceinline__ unsigned num_key(double a)
{
    unsigned k;  // one operation; from C++ the compiler makes three of it (align, mask, add)
    asm("v_lshl_add_u32 %0, %1, 1, %2" : "=v"(k) : "v"(__double2hiint(a)), "s"(0u - (kTinyHi << 1)));
    return k;
}

// a / den; d1 = rlow (kPair) or den (kCorr, kTrue)
template <class T, int DIV>
__device__ __forceinline__ double divide(double a, double d1, double rden)
{
    if constexpr (sizeof(T) == 4)
        return a * rden;
    else if constexpr (DIV == kPair)
        return fma(a, rden, a * d1);
    else if constexpr (DIV == kCorr) {
        double q = a * rden;
        q = fma(fma(-q, d1, a), rden, q);
        return fma(fma(-q, d1, a), rden, q);
    } else
        return a / d1;
}

// Tables of one axis and substrate, staged in LDS: what a forward row divides by ({rlow or den,
// rden}; FP32 storage: rden) and the back-substitution factor.
template <class T>
using FwdRow = std::conditional_t<sizeof(T) == 8, double2, double>;
template <class T>
__host__ __device__ constexpr size_t table_bytes()  // per row
{
    return sizeof(FwdRow<T>) + sizeof(double);
}
template <class T>
__device__ __forceinline__ void load_row(const AxisTables &tab, size_t off, int n, bool pair, int i, FwdRow<T> &f,
                                         double &c)
{
    const int k = (int)min(i, n - 1);
    if constexpr (sizeof(T) == 8)
        f = make_double2(as_global((pair ? tab.rlow : tab.den) + off)[k], as_global(tab.rden + off)[k]);
    else
        f = as_global(tab.rden + off)[k];
    c = as_global(tab.cc + off)[k];
}

// Rows are taken in batches of kBatch from two buffers, each refilled as soon as its batch is
// computed, so a batch's rows and table entries are requested one batch of arithmetic before
// their use, and no more LDS accesses are in flight than the wait counter tells apart (15).
// Requests past the last batch repeat it.
template <class T, int kBatch>
struct Rows {
    T *q[kBatch];  // where they are
    T v[kBatch];
    FwdRow<T> f[kBatch];
};

// LDS offsets of a line's rows: the columns of a plane (y lines) lie pitch elements apart, plus, in a
// SKEWed plane, one element every 2^shift rows; x lines are contiguous.  The extra element never
// falls inside a batch (batches start at multiples of 4, shift >= 2).
template <bool SKEW>
struct Columns {
    int pitch, shift;
    __host__ __device__ int operator()(int k) const { return SKEW ? k * pitch + (k >> shift) : k * pitch; }
    __device__ int step() const { return pitch; }
};
struct Contiguous {
    __device__ int operator()(int k) const { return k; }
    __device__ constexpr int step() const { return 1; }
};

// One Thomas line in LDS, row k at p[at(k)], swept forward in place.  Returns the last row's value
// in double; `key` collects num_key (FP64, not kTrue).  The first row of a line may be +0 (a
// Dirichlet value of 0): every division gives +0 for it, so its numerator is not flagged.
//
// The recursion behind the tables settles on one value after some rows (D = 1e3 to 1e5 um^2/min,
// dt = 0.01, dx = 20: 6 to 30 rows): rows [settled, n - 2] share their entries, which then stay in
// registers.
template <class T, int DIV, int kBatch, class At>
__device__ __forceinline__ double forward_line(T *p, At at, int n, int settled, double c1, const FwdRow<T> *f, ctab den,
                                               unsigned &key)
{
    if constexpr (sizeof(T) == 8 && DIV == kTrue) {  // rare: row by row, few registers
        double y = -0.0;
#pragma unroll 1
        for (int k = 0; k < n; ++k) {
            y = fma(c1, y, (double)p[at(k)]) / den[k];
            p[at(k)] = (T)y;
        }
        return y;
    }
    auto request = [&](int k, Rows<T, kBatch> &r, bool table) {
        r.q[0] = p + at(k);
#pragma unroll
        for (int j = 1; j < kBatch; ++j)
            r.q[j] = r.q[j - 1] + at.step();
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            r.v[j] = *r.q[j];
            if (table)
                r.f[j] = f[k + j];
        }
        asm volatile("" ::: "memory");  // requested here, not where the values are used
    };
    double y = -0.0;  // fma(c1, -0.0, v) is v, signed zeros included
    unsigned kb = 0u;
    auto row = [&](T *q, T v, const FwdRow<T> &d) {
        const double num = fma(c1, y, (double)v);
        if constexpr (sizeof(T) == 8) {
            kb = max(kb, num_key(num));
            y = divide<T, DIV>(num, d.x, d.y);
        } else
            y = num * d;
        *q = (T)y;
    };
    auto batch = [&](const Rows<T, kBatch> &r) {
#pragma unroll
        for (int j = 0; j < kBatch; ++j)
            row(r.q[j], r.v[j], r.f[j]);
    };
    auto few = [&](int k, Rows<T, kBatch> &r) {
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            r.q[j] = p + at(min(k + j, n - 1));
            r.v[j] = *r.q[j];
            r.f[j] = f[min(k + j, n - 1)];
        }
    };
    auto some = [&](int k, const Rows<T, kBatch> &r) {  // the rows of a batch that exist
#pragma unroll
        for (int j = 0; j < kBatch; ++j)
            if (k + j < n)
                row(r.q[j], r.v[j], r.f[j]);
    };
    // the first batch, pairs of batches up to the settled rows, pairs of those, then the rest
    Rows<T, kBatch> r0, r1;
    few(0, r0);
    const int pairs = n > kBatch ? (n - kBatch) / (2 * kBatch) : 0;
    const int early = min(pairs, max(settled - kBatch + 2 * kBatch - 1, 0) / (2 * kBatch));
    const int same = kBatch + early * 2 * kBatch;  // first settled row taken as one
    const int late = max(n - 1 - same, 0) / (2 * kBatch), end = same + late * 2 * kBatch;
    if (early > 0)
        request(kBatch, r1, true);
    row(r0.q[0], r0.v[0], r0.f[0]);
    if constexpr (sizeof(T) == 8)
        kb = __double_as_longlong((double)r0.v[0]) == 0 ? 0u : kb;
#pragma unroll
    for (int j = 1; j < kBatch; ++j)
        if (j < n)
            row(r0.q[j], r0.v[j], r0.f[j]);
    if (early > 0) {
        request(2 * kBatch, r0, true);
        for (int k = kBatch; k < same; k += 2 * kBatch) {
            batch(r1);
            request(min(k + 2 * kBatch, same - kBatch), r1, true);
            batch(r0);
            request(min(k + 3 * kBatch, same - kBatch), r0, true);
        }
    }
    if (late > 0) {
        const FwdRow<T> d = f[same];
        request(same, r1, false);
        request(same + kBatch, r0, false);
        for (int k = same; k < end; k += 2 * kBatch) {
#pragma unroll
            for (int j = 0; j < kBatch; ++j)
                row(r1.q[j], r1.v[j], d);
            request(min(k + 2 * kBatch, end - kBatch), r1, false);
#pragma unroll
            for (int j = 0; j < kBatch; ++j)
                row(r0.q[j], r0.v[j], d);
            request(min(k + 3 * kBatch, end - kBatch), r0, false);
        }
    }
    if (end < n) {
        few(end, r0);
        few(end + kBatch, r1);
        some(end, r0);
        some(end + kBatch, r1);
    }
    if constexpr (sizeof(T) == 8)
        key = max(key, kb);
    return y;
}

// Back substitution of the same line from its last row's value xv: rows n-2 .. 0 go to out(k, x),
// in that order (k is wave-uniform).  Settled rows go in longer batches: two operations a row, a
// batch of four would be shorter than the latency of its requests.
template <class T, int kBatch, class At, class Out>
__device__ __forceinline__ void back_line(const T *p, At at, int n, int settled, double xv, const double *c, Out out)
{
    struct {
        T v[kBatch];
        double c[kBatch];
    } r0, r1;
    auto request = [&](int k, auto &r) {  // rows k .. k + kBatch - 1
        const T *q = p + at(k);
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            r.v[j] = *q;
            r.c[j] = c[k + j];
            q += at.step();
        }
        asm volatile("" ::: "memory");
    };
    auto batch = [&](int k, auto &r) {
#pragma unroll
        for (int j = kBatch - 1; j >= 0; --j) {
            xv = fma(-r.c[j], xv, (double)r.v[j]);
            out(k + j, xv);
        }
    };
    // rows [0, full) in pairs of batches, [full, n - 1) first
    const int full = (n - 1) / (2 * kBatch) * (2 * kBatch);
    auto few = [&](int k, auto &r) {
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            r.v[j] = p[at(min(k + j, n - 1))];
            r.c[j] = c[min(k + j, n - 1)];
        }
    };
    few(full + kBatch, r1);
    few(full, r0);
#pragma unroll
    for (int j = kBatch - 2; j >= 0; --j)
        if (full + kBatch + j < n - 1) {
            xv = fma(-r1.c[j], xv, (double)r1.v[j]);
            out(full + kBatch + j, xv);
        }
#pragma unroll
    for (int j = kBatch - 1; j >= 0; --j)
        if (full + j < n - 1) {
            xv = fma(-r0.c[j], xv, (double)r0.v[j]);
            out(full + j, xv);
        }
    // pairs of long batches while all their rows are settled
    constexpr int kLong = 2 * kBatch;
    const int late = max(full - settled, 0) / (2 * kLong), low = full - late * 2 * kLong;
    if (late > 0) {
        const double cs = c[full - 1];
        T l0[kLong], l1[kLong];
        auto ask = [&](int k, T *l) {
#pragma unroll
            for (int h = 0; h < kLong; h += kBatch) {
                const T *q = p + at(k + h);
#pragma unroll
                for (int j = 0; j < kBatch; ++j) {
                    l[h + j] = *q;
                    q += at.step();
                }
            }
            asm volatile("" ::: "memory");
        };
        auto go = [&](int k, const T *l) {
#pragma unroll
            for (int j = kLong - 1; j >= 0; --j) {
                xv = fma(-cs, xv, (double)l[j]);
                out(k + j, xv);
            }
        };
        ask(full - kLong, l1);
        ask(full - 2 * kLong, l0);
        for (int k = full - 2 * kLong; k >= low; k -= 2 * kLong) {
            go(k + kLong, l1);
            ask(max(k - kLong, 0), l1);
            go(k, l0);
            ask(max(k - 2 * kLong, 0), l0);
        }
    }
    if (low > 0) {
        request(low - kBatch, r1);
        request(low - 2 * kBatch, r0);
    }
    for (int k = low - 2 * kBatch; k >= 0; k -= 2 * kBatch) {
        batch(k + kBatch, r1);
        request(max(k - kBatch, 0), r1);
        batch(k, r0);
        request(max(k - 2 * kBatch, 0), r0);
    }
}

// results are stored plainly: the z sweep reads them next, often from the 256 MB memory-side cache
template <class T>
__device__ __forceinline__ void store_result(gmem<T> p, T v)
{
    *p = v;
}

// n / d with inv = ceil(2^32 / d), d >= 2: exact while n*d < 2^32 (planes in LDS hold at most 2^15.4
// values)
__device__ __forceinline__ int quot(int n, unsigned inv) { return (int)__umulhi((unsigned)n, inv); }
__device__ __forceinline__ unsigned quot_inv(int d) { return 0xffffffffu / (unsigned)d + 1u; }

// Layout of a plane in LDS: row y at y*pitch, or (SKEW) y*nx + (y >> shift).  64 rows read at one
// column (x sweep) have to fall on distinct banks, 32 of 4 bytes for each group of lanes served at
// once (32 lanes of 4 bytes, 16 of 8): an odd pitch does that.  Where rows of nx + 1 do not fit, one
// element more every group/g rows does too, g = gcd(nx, group) the number of rows apart by a
// multiple of all banks; a 200 x 200 FP32 plane fits that way.  It is not the rule because the
// column sweep then forms longer addresses (128 x 128 FP64 planes: 4% slower).
template <bool SKEW>
__host__ __device__ __forceinline__ Columns<SKEW> plane_layout(int nx, size_t elem)
{
    if (!SKEW)
        return Columns<SKEW>{nx | 1, 0};
    const int group = elem == 8 ? 16 : 32;
    int g = 1, shift = elem == 8 ? 4 : 5;
    while (g < group && nx % (2 * g) == 0) {
        g *= 2;
        --shift;
    }
    return Columns<SKEW>{nx, shift};
}

constexpr int kVoteBytes = 16;  // before the tile in LDS

constexpr int kMaxThreads = 512;

// The kernel comes in two sizes.  BIG, planes above 80 KB: one workgroup per CU, 256 registers per
// lane.  Otherwise 128 (FP64) or 96 registers, so that several workgroups share a CU, with smaller
// batches of rows.  Pairs of a plane's elements per loading thread, all of them in registers at
// once (pairs, aligned like one element, so that the unrolled loads fit the instruction cache: a
// 76 KB kernel of single FP32 loads ran at half the speed):
template <class T, bool BIG>
constexpr int plane_loads()
{
    return (BIG ? (sizeof(T) == 8 ? 31 : 80) : (sizeof(T) == 8 ? 15 : 24));
}
template <class T>
struct PairOf;
template <>
struct PairOf<double> {
    typedef double type __attribute__((ext_vector_type(2), aligned(8)));
};
template <>
struct PairOf<float> {
    typedef float type __attribute__((ext_vector_type(2), aligned(4)));
};
template <class T, bool BIG>
constexpr int plane_waves_per_simd()
{
    return BIG ? 2 : sizeof(T) == 8 ? 4 : 5;
}

// What a workgroup needs to know of one plane.
template <class T>
struct Plane {
    const DomainDesc<T> *D;
    int di, s, z;
};

template <class T>
__device__ __forceinline__ Plane<T> locate(const DomainDesc<T> *descs, const long long *prefix, int ndom, int t)
{
    Plane<T> p;
    long long lt = t;
    p.di = 0;
    if (ndom > 1) {
        p.di = __builtin_amdgcn_readfirstlane(find_domain(prefix, ndom, lt));
        lt -= prefix[p.di];
    }
    p.D = descs + p.di;
    const int nz = p.D->nz;
    p.s = __builtin_amdgcn_readfirstlane((int)((unsigned)lt / (unsigned)nz));
    p.z = __builtin_amdgcn_readfirstlane((int)lt - p.s * nz);
    return p;
}

// Workgroups stride over the z planes of a size class; a plane of one substrate is held in LDS,
// (rows as plane_layout places them), and swept in place there: x then y, or y then x for the adjoint's
// reverse order (YX).  AG: the cell sources and sinks first, on the plane in LDS (segments
// [zseg[z], zseg[z+1]) of the voxel-sorted agent list), agents of a voxel in list order, as the
// separate agent kernel applies them.  The plane is written back where it was read.
//
// The first `solvers` threads (whole wavefronts, at least as many lanes as the plane has rows or
// columns) sweep; the other wavefronts load: they read the next plane into registers while this
// one is swept, and put it into LDS when it is done.  (Registers, because LDS is full; wavefronts
// of their own, because the solvers' registers and instruction slots are what a plane waits
// for.)  Both run through the same sequence of barriers.
template <class T, bool BIG, bool SKEW, bool YX, bool AG>
__global__ __launch_bounds__(kMaxThreads, (plane_waves_per_simd<T, BIG>())) void k_plane(const DomainDesc<T> *__restrict__ descs,
                                                                    const long long *__restrict__ prefix, int ndom,
                                                                    int planes, int solvers, int parity)
{
    constexpr int kLoads = plane_loads<T, BIG>(), B = BIG || sizeof(T) == 4 ? 4 : 2;
    extern __shared__ unsigned char smem[];
    int *vote = reinterpret_cast<int *>(smem);  // set by a lane that met a flagged numerator
    const int tid = threadIdx.x, nt = blockDim.x;
    const int wave_first = __builtin_amdgcn_readfirstlane(tid);  // uniform: this wavefront's role

    // LDS: vote, tables of the axis being swept, plane
    auto lds_tables = [&](const DomainDesc<T> &) { return reinterpret_cast<FwdRow<T> *>(smem + kVoteBytes); };
    auto lds_factors = [&](const DomainDesc<T> &D) {
        return reinterpret_cast<double *>(lds_tables(D) + max(D.nx, D.ny));
    };
    auto lds_plane = [&](const DomainDesc<T> &D) { return reinterpret_cast<T *>(lds_factors(D) + max(D.nx, D.ny)); };
    // LDS index of the plane's element e
    auto at = [](int e, int nx, const Columns<SKEW> &lay, unsigned inv) {
        if (lay.pitch == nx && !SKEW)
            return e;
        const int y = quot(e, inv);
        return e + (SKEW ? y >> lay.shift : y);
    };
    auto active = [&](const DomainDesc<T> &D, int s) {
        return __builtin_amdgcn_readfirstlane((int)as_global(D.dact)[s]) != 0;
    };
    // results that went to LDS, out by all threads
    auto copy_out = [&](const DomainDesc<T> &D, int s, int z) {
        const int nel = D.nx * D.ny;
        const Columns<SKEW> lay = plane_layout<SKEW>(D.nx, sizeof(T));
        const unsigned inv = quot_inv(max(D.nx, 2));
        const T *P = lds_plane(D);
        const gmem<T> f = as_global(D.field[parity] + ((size_t)s * D.nz + z) * nel);
        for (int e = tid; e < nel; e += nt)
            store_result<T>(f + e, P[at(e, D.nx, lay, inv)]);
    };

    if (wave_first >= solvers) {
        // ------------------------------------------------------------------ loading wavefronts
        const int lid = tid - solvers, ln = nt - solvers;
        typedef typename PairOf<T>::type Pair;
        Pair r[kLoads];  // the next plane's values
        // first element of pair lid + j*ln, the last pair's for lanes past the end (n >= 2)
        auto first = [&](int j, int n) { return min(2 * (lid + j * ln), n - 2); };
        auto request = [&](const Plane<T> &p) {
            const int n = p.D->nx * p.D->ny;
            const gmem<const T> src = as_global<const T>(p.D->field[parity] + ((size_t)p.s * p.D->nz + p.z) * n);
#pragma unroll
            for (int j = 0; j < kLoads; ++j)
                if (2 * j * ln < n)
                    r[j] = *(gmem<const Pair>)(src + (unsigned)first(j, n));
        };
        int t = blockIdx.x;
        Plane<T> p = locate(descs, prefix, ndom, t);
        request(p);
        for (;;) {
            const DomainDesc<T> &D = *p.D;
            const int s = p.s, z = p.z, nel = D.nx * D.ny;
            const bool act = active(D, s), voxels = D.dface != nullptr;
            const bool zface = act && (z == 0 || z == D.nz - 1);
            {
                T *P = lds_plane(D);
                const Columns<SKEW> lay = plane_layout<SKEW>(D.nx, sizeof(T));
                const unsigned inv = quot_inv(max(D.nx, 2));
#pragma unroll
                for (int j = 0; j < kLoads; ++j)
                    if (2 * j * ln < nel) {
                        int e = first(j, nel);
                        asm("" : "+v"(e));  // so many LDS addresses are cheaper to form than to keep
                        // the pair stays together: rows are padded where nx is even, and then a
                        // pair does not cross a row's end
                        T *q = P + at(e, D.nx, lay, inv);
                        q[0] = r[j].x;
                        q[1] = r[j].y;
                    }
                // a launch over uneven members may have more solvers, and so fewer loaders, than this
                // plane alone would: what their registers could not hold
                const gmem<const T> src = as_global<const T>(D.field[parity] + ((size_t)s * D.nz + z) * nel);
                for (int e = 2 * kLoads * ln + lid; e < nel; e += ln)
                    P[at(e, D.nx, lay, inv)] = src[e];
            }
            lds_barrier();  // plane and first tables in LDS
            t += gridDim.x;
            if (t < planes) {
                p = locate(descs, prefix, ndom, t);
                request(p);
            }
            if (!zface) {
                if (AG && D.zseg != nullptr)
                    lds_barrier();  // agents
                for (bool exact = false;;) {
                    if (act)
                        lds_barrier();  // Dirichlet values
                    lds_barrier();      // first axis
                    lds_barrier();      // Dirichlet values, second tables
                    if constexpr (sizeof(T) == 8) {
                        if (!exact) {
                            lds_barrier();  // vote
                            if (*vote) {
                                exact = true;
                                lds_barrier();  // vote read
                                lds_barrier();  // plane reloaded
                                if (AG && D.zseg != nullptr)
                                    lds_barrier();
                                continue;
                            }
                        }
                    }
                    if (YX || (act && voxels)) {
                        lds_barrier();  // second axis
                        if (act)
                            lds_barrier();
                        copy_out(D, s, z);
                    }
                    break;
                }
            }
            if (t >= planes)
                return;
            lds_barrier();  // the plane's LDS is free
        }
    }

    // ---------------------------------------------------------------------- solving wavefronts
    FwdRow<T> xf, yf;  // row tid of the tables
    double xc = 0.0, yc = 0.0;
    if (tid == 0)
        *vote = 0;
    int t = blockIdx.x, di_had = -1, s_had = -1;
    for (;;) {
        const Plane<T> p = locate(descs, prefix, ndom, t);
        const DomainDesc<T> &D = *p.D;
        const int s = p.s, z = p.z;
        const int nx = D.nx, ny = D.ny, nz = D.nz;
        const int nel = nx * ny;
        const Columns<SKEW> lay = plane_layout<SKEW>(nx, sizeof(T));
        const unsigned inv = quot_inv(max(nx, 2));
        const double c1 = as_ctab(D.c1)[s];
        const bool pairx = sizeof(T) == 4 || as_ctab(D.tab[0].nopair)[s] == 0.0;
        const bool pairy = sizeof(T) == 4 || as_ctab(D.tab[1].nopair)[s] == 0.0;
        const int setx = (int)as_ctab(D.tab[0].settled)[s], sety = (int)as_ctab(D.tab[1].settled)[s];
        const bool act = active(D, s);
        const T dv = ((const __attribute__((address_space(4))) T *)D.dval)[s];
        const gmem<const T> fv = as_global(D.dface);  // per-voxel Dirichlet values
        const bool voxels = D.dface != nullptr;
        const gmem<T> f = as_global(D.field[parity] + ((size_t)s * nz + z) * nel);
        if (p.di != di_had || s != s_had) {
            load_row<T>(D.tab[0], (size_t)s * nx, nx, pairx, tid, xf, xc);
            load_row<T>(D.tab[1], (size_t)s * ny, ny, pairy, tid, yf, yc);
            di_had = p.di;
            s_had = s;
        }
        FwdRow<T> *tf = lds_tables(D);
        double *tc = lds_factors(D);
        T *P = lds_plane(D);
        auto put_table = [&](bool x) {
            if (tid < (x ? nx : ny)) {
                tf[tid] = x ? xf : yf;
                tc[tid] = x ? xc : yc;
            }
        };
        // the plane's face voxels take their Dirichlet values (apply_dirichlet_conditions)
        auto dirichlet = [&]() {
            if (!act)
                return;
            // low or high face of y (k < nx) or x, position k along it
            auto place = [&](int e, int k) {
                return P + (k < nx ? lay(e ? ny - 1 : 0) + k : lay(k - nx) + (e ? nx - 1 : 0));
            };
            if (voxels)
                for (int i = tid; i < 2 * (nx + ny); i += solvers) {
                    const int e = i & 1, k = i >> 1;
                    *place(e, k) = fv[k < nx ? face_y(nx, ny, nz, D.nsub, e, s, k, z)
                                             : face_x(ny, nz, D.nsub, e, s, k - nx, z)];
                }
            else
                for (int i = tid; i < 2 * (nx + ny); i += solvers)
                    *place(i & 1, i >> 1) = dv;
        };
        auto agents = [&]() {
            const auto zs = (const __attribute__((address_space(4))) int *)D.zseg;
            const int lo = zs[z], hi = zs[z + 1];
            const gmem<const double> a1 = as_global(D.t1 + (size_t)s * D.nact), a2 = as_global(D.t2 + (size_t)s * D.nact);
            for (int k = lo + tid; k < hi; k += solvers) {
                const int e = at((int)(as_global(D.seg_off)[k] - (long long)z * nel), nx, lay, inv);
                const int b1 = as_global(D.seg_start)[k + 1];
                double v = (double)P[e];
                for (int a = as_global(D.seg_start)[k]; a < b1; ++a) {
                    v = v + a1[a];
                    v = v / a2[a];
                }
                P[e] = (T)v;
            }
        };
        const bool zface = act && (z == 0 || z == nz - 1);  // such a plane ends as its Dirichlet values
        put_table(!YX);
        lds_barrier();  // plane and first tables in LDS
        if (zface) {
            const size_t fz = face_z(nx, ny, nz, D.nsub, z == 0 ? 0 : 1, s, 0, 0);
            if (voxels)
                for (int e = tid; e < nel; e += solvers)
                    f[e] = fv[fz + e];
            else
                for (int e = tid; e < nel; e += solvers)
                    f[e] = dv;
        } else {
            if (AG && D.zseg != nullptr) {
                agents();
                lds_barrier();
            }
            for (bool exact = false;;) {
                if (act) {
                    dirichlet();
                    lds_barrier();
                }
                unsigned key = 0u;
                auto forward = [&](T *q, auto rows, int n, int settled, bool pair, const double *den) {
                    if constexpr (sizeof(T) == 4)
                        return forward_line<T, kPair, B>(q, rows, n, settled, c1, tf, nullptr, key);
                    else
                        return exact ? forward_line<T, kTrue, B>(q, rows, n, settled, c1, tf, as_ctab(den), key)
                                     : pair ? forward_line<T, kPair, B>(q, rows, n, settled, c1, tf, nullptr, key)
                                            : forward_line<T, kCorr, B>(q, rows, n, settled, c1, tf, nullptr, key);
                };
                const Contiguous row;
                // a line on a Dirichlet face is overwritten whole, whatever its numerators were
                auto x_forward = [&]() {
                    const unsigned k0 = key;
                    const double y = forward(P + lay(tid), row, nx, setx, pairx, D.tab[0].den + (size_t)s * nx);
                    if (act && (tid == 0 || tid == ny - 1))
                        key = k0;
                    return y;
                };
                auto x_back = [&](double y) {
                    T *q = P + lay(tid);
                    back_line<T, B>(q, row, nx, setx, y, tc, [&](int k, double x) { q[k] = (T)x; });
                };
                auto y_forward = [&]() {
                    const unsigned k0 = key;
                    const double y = forward(P + tid, lay, ny, sety, pairy, D.tab[1].den + (size_t)s * ny);
                    if (act && (tid == 0 || tid == nx - 1))
                        key = k0;
                    return y;
                };
                auto y_back = [&](double y) {
                    T *q = P + tid;
                    back_line<T, B>(q, lay, ny, sety, y, tc, [&](int k, double x) { q[lay(k)] = (T)x; });
                };
                double last = 0.0;
                if constexpr (!YX) {
                    if (tid < ny)
                        x_back(x_forward());
                } else {
                    if (tid < nx)
                        y_back(y_forward());
                }
                lds_barrier();  // first axis
                dirichlet();
                put_table(YX);
                lds_barrier();
                if constexpr (!YX) {
                    if (tid < nx)
                        last = y_forward();
                } else {
                    if (tid < ny)
                        last = x_forward();
                }
                if constexpr (sizeof(T) == 8) {
                    // a numerator outside the fast divisions' range somewhere in the plane: the
                    // whole plane again from memory (nothing is stored yet) with true divisions
                    if (!exact) {
                        if (key >= kKeyBad)
                            *vote = 1;
                        lds_barrier();
                        if (*vote) {
                            exact = true;
                            lds_barrier();
                            if (tid == 0)
                                *vote = 0;
                            for (int e = tid; e < nel; e += solvers)
                                P[at(e, nx, lay, inv)] = f[e];
                            put_table(!YX);
                            lds_barrier();
                            if (AG && D.zseg != nullptr) {
                                agents();
                                lds_barrier();
                            }
                            continue;
                        }
                    }
                }
                if (!YX && !(act && voxels)) {  // results go out as they are found, one row of columns at a time
                    if (tid < nx) {
                        const bool face = act && (tid == 0 || tid == nx - 1);
                        gmem<T> q = f + tid + (size_t)(ny - 1) * nx;  // rows are stored from the last to the first
                        store_result<T>(q, act ? dv : (T)last);
                        back_line<T, B>(P + tid, lay, ny, sety, last, tc, [&](int k, double x) {
                            q -= nx;
                            store_result<T>(q, face || (act && k == 0) ? dv : (T)x);
                        });
                    }
                    break;
                }
                if constexpr (YX) {
                    if (tid < ny)
                        x_back(last);
                } else {
                    if (tid < nx)
                        y_back(last);
                }
                lds_barrier();  // second axis
                if (act) {
                    dirichlet();
                    lds_barrier();
                }
                copy_out(D, s, z);
                break;
            }
        }
        t += gridDim.x;
        if (t >= planes)
            return;
        lds_barrier();  // the plane's LDS is free
    }
}

// ---- strips: the FP64 x sweep of rows in LDS, for planes that do not fit there

constexpr int kStripLoads = 31;  // pairs per loading thread

// One strip: `rows` consecutive rows (z*ny + y) of one substrate from row r0, strip i of it.
template <class T>
struct Strip {
    const DomainDesc<T> *D;
    int di, s, i, r0, rows;
};

template <class T>
__device__ __forceinline__ Strip<T> locate_strip(const DomainDesc<T> *descs, const long long *prefix, int ndom, int t)
{
    Strip<T> p;
    long long lt = t;
    p.di = 0;
    if (ndom > 1) {
        p.di = __builtin_amdgcn_readfirstlane(find_domain(prefix, ndom, lt));
        lt -= prefix[p.di];
    }
    p.D = descs + p.di;
    const unsigned R = (unsigned)p.D->strip, all = (unsigned)p.D->ny * (unsigned)p.D->nz, n = (all + R - 1) / R;
    p.s = __builtin_amdgcn_readfirstlane((int)((unsigned)lt / n));
    p.i = __builtin_amdgcn_readfirstlane((int)((unsigned)lt - (unsigned)p.s * n));
    p.r0 = p.i * (int)R;
    p.rows = (int)min(R, all - (unsigned)p.r0);
    return p;
}

// What bounds it: the solvers need 68 + 36 clocks per column forward and back (64 rows of 256: 10 us),
// then 128 KB go out and the next strip goes in, during which no row is solved; a CU has LDS for one
// strip of such rows, so the memory system idles in the solve and queues in between (256^3 x 4 FP64:
// 0.31 ms, 3.5 TB/s).  It still beats lod.hip's x sweep (0.37 ms) in FP64, which reads most of each line
// twice.  Tried: results out in column segments during back substitution (256^3 x 4 783 -> 834 us per
// step), a staggered start of the workgroups and contiguous strips per XCD (no change).
//
// Workgroups stride over the strips; the first `solvers` threads sweep, a row per lane, the other
// wavefronts hold the next strip in registers meanwhile, as k_plane's do.  Reads field[parity],
// writes field[parity ^ 1].  AG: the cell sources and sinks first, on the strip in LDS; the loaders
// also fetch the next strip's (one voxel each; what a denser strip has more is fetched when applied).
// NT: non-temporal loads and stores.
template <class T, bool AG, bool NT>
__global__ __launch_bounds__(kMaxThreads, 2) void k_strip(const DomainDesc<T> *__restrict__ descs,
                                                          const long long *__restrict__ prefix, int ndom, int strips,
                                                          int solvers, int parity)
{
    constexpr int kLoads = kStripLoads, B = 4;
    typedef typename PairOf<T>::type Pair;
    extern __shared__ unsigned char smem[];
    const int tid = threadIdx.x, nt = blockDim.x;
    const int wave_first = __builtin_amdgcn_readfirstlane(tid);

    auto lds_tables = [&]() { return reinterpret_cast<FwdRow<T> *>(smem); };
    auto lds_factors = [&](const DomainDesc<T> &D) { return reinterpret_cast<double *>(lds_tables() + D.nx); };
    auto lds_strip = [&](const DomainDesc<T> &D) { return reinterpret_cast<T *>(lds_factors(D) + D.nx); };
    // LDS index of the strip's element e: rows lie nx | 1 apart
    auto at = [](int e, int nx, unsigned inv) { return nx & 1 ? e : e + quot(e, inv); };
    auto source = [&](const Strip<T> &p, int par) {
        return as_global(p.D->field[par] + ((size_t)p.s * ((size_t)p.D->ny * p.D->nz) + p.r0) * p.D->nx);
    };
    auto copy_out = [&](const Strip<T> &p) {
        const int nx = p.D->nx, n = p.rows * nx;
        const unsigned inv = quot_inv(nx);
        const T *P = lds_strip(*p.D);
        const gmem<T> f = source(p, parity ^ 1);
        int e = 2 * tid;
        for (; e < n - 1; e += 2 * nt) {
            const T *q = P + at(e, nx, inv);
            Pair v;
            v.x = q[0];
            v.y = q[1];
            if constexpr (NT)
                __builtin_nontemporal_store(v, (gmem<Pair>)(f + (unsigned)e));
            else
                *(gmem<Pair>)(f + (unsigned)e) = v;
        }
        if (e == n - 1)
            f[e] = P[at(e, nx, inv)];
    };
    auto update = [](T *q, const gmem<const double> a1, const gmem<const double> a2, int b0, int b1) {
        double v = (double)*q;
        for (int a = b0; a < b1; ++a) {
            v = v + a1[a];
            v = v / a2[a];
        }
        *q = (T)v;
    };

    if (wave_first >= solvers) {
        // ------------------------------------------------------------------ loading wavefronts
        const int lid = tid - solvers, ln = nt - solvers;
        Pair r[kLoads];
        auto first = [&](int j, int n) { return min(2 * (lid + j * ln), n - 2); };
        int ag_e = -1, ag_b0 = 0, ag_b1 = 0;  // this thread's voxel with agents in the next strip
        double ag_1 = 0.0, ag_2 = 1.0;
        auto request = [&](const Strip<T> &p) {
            const DomainDesc<T> &D = *p.D;
            if (AG && D.sseg != nullptr) {
                const auto ss = (const __attribute__((address_space(4))) int *)D.sseg;
                const int k = ss[p.i] + lid;
                ag_e = -1;
                if (k < ss[p.i + 1]) {
                    ag_e = (int)(as_global(D.seg_off)[k] - (long long)p.r0 * D.nx);
                    ag_b0 = as_global(D.seg_start)[k];
                    ag_b1 = as_global(D.seg_start)[k + 1];
                    ag_1 = as_global(D.t1 + (size_t)p.s * D.nact)[ag_b0];
                    ag_2 = as_global(D.t2 + (size_t)p.s * D.nact)[ag_b0];
                }
            }
            const int n = p.rows * D.nx;
            const gmem<const T> src = source(p, parity);
#pragma unroll
            for (int j = 0; j < kLoads; ++j)
                if (2 * j * ln < n)
                    if constexpr (NT)
                        r[j] = __builtin_nontemporal_load((gmem<const Pair>)(src + (unsigned)first(j, n)));
                    else
                        r[j] = *(gmem<const Pair>)(src + (unsigned)first(j, n));
        };
        int t = blockIdx.x;
        Strip<T> p = locate_strip(descs, prefix, ndom, t);
        request(p);
        for (;;) {
            const Strip<T> now = p;
            const DomainDesc<T> &D = *now.D;
            T *P = lds_strip(D);
            const int nx = D.nx, n = now.rows * nx;
            const unsigned inv = quot_inv(nx);
#pragma unroll
            for (int j = 0; j < kLoads; ++j)
                if (2 * j * ln < n) {
                    int e = first(j, n);
                    asm("" : "+v"(e));  // so many LDS addresses are cheaper to form than to keep
                    T *q = P + at(e, nx, inv);  // a pair stays in its row where rows are padded (nx even)
                    q[0] = r[j].x;
                    q[1] = r[j].y;
                }
            lds_barrier();  // strip and tables in LDS
            if (AG && D.sseg != nullptr) {
                const gmem<const double> a1 = as_global<const double>(D.t1 + (size_t)now.s * D.nact);
                const gmem<const double> a2 = as_global<const double>(D.t2 + (size_t)now.s * D.nact);
                if (ag_e >= 0) {
                    T *q = P + at(ag_e, nx, inv);
                    double v = ((double)*q + ag_1) / ag_2;
                    for (int a = ag_b0 + 1; a < ag_b1; ++a) {
                        v = v + a1[a];
                        v = v / a2[a];
                    }
                    *q = (T)v;
                }
                const auto ss = (const __attribute__((address_space(4))) int *)D.sseg;
                for (int k = ss[now.i] + lid + ln; k < ss[now.i + 1]; k += ln)
                    update(P + at((int)(as_global(D.seg_off)[k] - (long long)now.r0 * nx), nx, inv), a1, a2,
                           as_global(D.seg_start)[k], as_global(D.seg_start)[k + 1]);
                lds_barrier();  // agents
            }
            t += gridDim.x;
            if (t < strips) {
                p = locate_strip(descs, prefix, ndom, t);
                request(p);
            }
            lds_barrier();  // solved
            copy_out(now);
            if (t >= strips)
                return;
            lds_barrier();  // the strip's LDS is free
        }
    }

    // ---------------------------------------------------------------------- solving wavefronts
    int t = blockIdx.x, di_had = -1, s_had = -1;
    for (;;) {
        const Strip<T> p = locate_strip(descs, prefix, ndom, t);
        const DomainDesc<T> &D = *p.D;
        const int s = p.s, nx = D.nx, ny = D.ny, nz = D.nz;
        const unsigned inv = quot_inv(nx);
        const double c1 = as_ctab(D.c1)[s];
        const bool pair = as_ctab(D.tab[0].nopair)[s] == 0.0;
        const int settled = (int)as_ctab(D.tab[0].settled)[s];
        const bool act = __builtin_amdgcn_readfirstlane((int)as_global(D.dact)[s]) != 0;
        const T dv = ((const __attribute__((address_space(4))) T *)D.dval)[s];
        const gmem<const T> fv = as_global(D.dface);  // per-voxel Dirichlet values
        const bool voxels = D.dface != nullptr;
        FwdRow<T> *tf = lds_tables();
        double *tc = lds_factors(D);
        T *P = lds_strip(D);
        if (p.di != di_had || s != s_had) {
            for (int k = tid; k < nx; k += solvers) {
                FwdRow<T> f;
                double c;
                load_row<T>(D.tab[0], (size_t)s * nx, nx, pair, k, f, c);
                tf[k] = f;
                tc[k] = c;
            }
            di_had = p.di;
            s_had = s;
        }
        const bool mine = tid < p.rows;
        const int row = p.r0 + (mine ? tid : 0), z = row / ny, y = row - z * ny;
        const bool face = act && (y == 0 || y == ny - 1 || z == 0 || z == nz - 1);
        T *q = P + (mine ? tid : 0) * (nx | 1);
        auto ends = [&]() {  // the row's voxels on the x faces
            if (act && mine) {
                q[0] = voxels ? fv[face_x(ny, nz, D.nsub, 0, s, y, z)] : dv;
                q[nx - 1] = voxels ? fv[face_x(ny, nz, D.nsub, 1, s, y, z)] : dv;
            }
        };
        lds_barrier();  // strip and tables in LDS
        if (AG && D.sseg != nullptr)
            lds_barrier();  // agents
        ends();
        double last = 0.0;
        unsigned key = 0u;
        const Contiguous cols;
        auto forward = [&](auto div) {
            if (mine)
                last = forward_line<T, decltype(div)::value, B>(q, cols, nx, settled, c1, tf,
                                                                as_ctab(D.tab[0].den + (size_t)s * nx), key);
        };
        if (pair)
            forward(std::integral_constant<int, kPair>());
        else
            forward(std::integral_constant<int, kCorr>());
        // a numerator outside the fast divisions' range: this wavefront's rows again from
        // memory (which still holds them) with true divisions.  A row on a face is overwritten.
        if (__ballot(mine && !face && key >= kKeyBad) != 0) {
            const int l0 = wave_first / kWave * kWave, l1 = min(l0 + kWave, p.rows), lane = tid - l0;
            const gmem<const T> src = source(p, parity);
            for (int e = l0 * nx + lane; e < l1 * nx; e += kWave)
                P[at(e, nx, inv)] = src[e];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
            if (AG && D.sseg != nullptr) {
                const auto ss = (const __attribute__((address_space(4))) int *)D.sseg;
                for (int k = ss[p.i] + lane; k < ss[p.i + 1]; k += kWave) {
                    const int e = (int)(as_global(D.seg_off)[k] - (long long)p.r0 * nx);
                    if (e >= l0 * nx && e < l1 * nx)
                        update(P + at(e, nx, inv), as_global<const double>(D.t1 + (size_t)s * D.nact),
                               as_global<const double>(D.t2 + (size_t)s * D.nact), as_global(D.seg_start)[k],
                               as_global(D.seg_start)[k + 1]);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
            }
            ends();
            forward(std::integral_constant<int, kTrue>());
        }
        if (mine) {
            q[nx - 1] = (T)last;
            back_line<T, B>(q, cols, nx, settled, last, tc, [&](int k, double x) { q[k] = (T)x; });
        }
        ends();
        unsigned long long faces = __ballot(mine && face);
        while (faces != 0) {  // whole rows on the y and z faces
            const int l = __builtin_amdgcn_readfirstlane(__ffsll((long long)faces) - 1);
            faces &= faces - 1;
            const int fl = wave_first / kWave * kWave + l, fr = p.r0 + fl, fz = fr / ny, fy = fr - fz * ny;
            const bool zf = fz == 0 || fz == nz - 1;
            const size_t base = !voxels ? 0
                                : zf    ? face_z(nx, ny, nz, D.nsub, fz == 0 ? 0 : 1, s, 0, fy)
                                        : face_y(nx, ny, nz, D.nsub, fy == 0 ? 0 : 1, s, 0, fz);
            for (int x = tid % kWave; x < nx; x += kWave)
                P[fl * (nx | 1) + x] = voxels ? fv[base + x] : dv;
        }
        lds_barrier();  // solved
        copy_out(p);
        t += gridDim.x;
        if (t >= strips)
            return;
        lds_barrier();  // the strip's LDS is free
    }
}

size_t strip_bytes(int nx, int rows, size_t elem)
{
    return (size_t)nx * (elem == 8 ? table_bytes<double>() : table_bytes<float>()) +
           ((size_t)rows * (nx | 1) + 1) * elem;
}

// Fields up to this size stay in the 256 MB memory-side cache for the y sweep; larger ones are read
// and written non-temporally (250 x 230 x 210 x 2 FP64, 193 MB: 322 -> 299 us per step, 256^3 x 4 806 ->
// 783; 160^3 x 4, 131 MB: 190 -> 200).
constexpr size_t kStripCached = 160u << 20;
constexpr size_t kStripSmall = 192u << 20;  // "large fields" of strips_pay

template <bool SKEW>
size_t plane_bytes(const Domain &d, size_t elem)
{
    const size_t row = elem == 8 ? table_bytes<double>() : table_bytes<float>();
    return kVoteBytes + (size_t)std::max(d.nx, d.ny) * row + (size_t)(plane_layout<SKEW>(d.nx, elem)(d.ny) + 1) * elem;
}

int size_class(size_t bytes)
{
    int c = 0;
    while (c < 3 && bytes > (kLdsBytes >> (3 - c)))
        ++c;
    return c;
}

// loading threads for planes of `el` elements, at most `loads` pairs each (whole wavefronts)
size_t plane_loaders(size_t el, int loads) { return ((el + 2 * loads - 1) / (2 * loads) + kWave - 1) / kWave * kWave; }

constexpr int kSmallClasses = 3;  // classes of the small kernel: planes up to 80 KB
constexpr int kSkewClass = 4;     // planes that fit only skewed
static_assert(kClasses == kSkewClass + 1, "size classes");

template <class T, bool BIG, bool SKEW, bool YX, bool AG>
void launch_plane_kernel(const Group *g, int c, unsigned grid, int planes, unsigned threads, int solvers, size_t lds)
{
    const DomainDesc<T> *d = static_cast<const DomainDesc<T> *>(g->d_desc);
    const int ndom = (int)g->doms.size();
    const long long *pre = g->d_prefix + (size_t)(kPlane0 + c) * (ndom + 1);
    hipLaunchKernelGGL((k_plane<T, BIG, SKEW, YX, AG>), dim3(grid), dim3(threads), lds, g->stream, d, pre, ndom, planes,
                       solvers, g->cur);
}

template <class T, bool BIG, bool SKEW>
int launch_planes_class(Group *g, int c, bool yx, bool agents)
{
    const long long planes = g->prefix[kPlane0 + c][g->doms.size()];
    size_t lds = 0, el = 0;
    int lines = 0;
    for (const Domain &d : g->doms)
        if (d.plane_class == c) {
            lds = std::max(lds, plane_bytes<SKEW>(d, sizeof(T)));
            el = std::max(el, (size_t)d.nx * d.ny);
            lines = std::max(lines, std::max(d.nx, d.ny));
        }
    const int solvers = (lines + kWave - 1) / kWave * kWave;
    // (resident_class leaves each member a wavefront of loaders at least)
    const unsigned th = BIG ? kMaxThreads
                            : (unsigned)std::min<size_t>(solvers + plane_loaders(el, plane_loads<T, BIG>()), kMaxThreads);
    // as many workgroups as the CUs hold, each striding over the planes
    const int waves = 4 * plane_waves_per_simd<T, BIG>() / (int)(th / kWave);
    const long long percu = std::max(1, std::min(waves, (int)(kLdsBytes / lds)));
    const unsigned grid = (unsigned)std::min<long long>(planes, percu * std::max(g->cu_count, 1));
    if (yx)
        launch_plane_kernel<T, BIG, SKEW, true, false>(g, c, grid, (int)planes, th, solvers, lds);
    else if (agents)
        launch_plane_kernel<T, BIG, SKEW, false, true>(g, c, grid, (int)planes, th, solvers, lds);
    else
        launch_plane_kernel<T, BIG, SKEW, false, false>(g, c, grid, (int)planes, th, solvers, lds);
    return hip_check(g, hipGetLastError(), "plane launch");
}

template <class T>
int launch_planes_t(Group *g, bool yx, bool agents)
{
    for (int c = 0; c < kClasses; ++c) {
        if (g->prefix[kPlane0 + c].back() == 0)
            continue;
        const int rc = c < kSmallClasses ? launch_planes_class<T, false, false>(g, c, yx, agents)
                       : c < kSkewClass  ? launch_planes_class<T, true, false>(g, c, yx, agents)
                                         : launch_planes_class<T, true, true>(g, c, yx, agents);
        if (rc)
            return rc;
    }
    return BFVMB_OK;
}

template <class T, bool BIG, bool SKEW>
hipError_t attributes(int bytes)
{
    const void *k[3] = {(const void *)k_plane<T, BIG, SKEW, false, false>, (const void *)k_plane<T, BIG, SKEW, false, true>,
                        (const void *)k_plane<T, BIG, SKEW, true, false>};
    hipError_t e = hipSuccess;
    for (int i = 0; i < 3 && e == hipSuccess; ++i)
        e = hipFuncSetAttribute(k[i], hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    return e;
}

template <class T>
hipError_t attributes_all(int bytes)
{
    hipError_t e = attributes<T, false, false>(bytes);
    if (e == hipSuccess)
        e = attributes<T, true, false>(bytes);
    if (e == hipSuccess)
        e = attributes<T, true, true>(bytes);
    return e;
}

}  // namespace

int strip_rows(const Domain &d, size_t elem, size_t limit)
{
    limit = std::min(limit, kLdsBytes);
    const size_t tables = strip_bytes(d.nx, 0, elem), row = (size_t)(d.nx | 1) * elem;
    const size_t loads = 2 * (size_t)kStripLoads;
    if (elem != 8 || d.nx < 2 || tables + row > limit)
        return 0;
    // two workgroups of 64 rows per CU, or one of as many rows as fit, 128 at most
    if (tables + kWave * row <= limit / 2 && (size_t)d.nx * kWave <= loads * (kMaxThreads / 2 - kWave))
        return kWave;
    size_t r = std::min<size_t>((limit - tables) / row, 2 * kWave);
    r = std::min(r, loads * (kMaxThreads - 2 * kWave) / d.nx);
    return r >= 32 ? (int)r : 0;
}

// Whether its x sweep goes by `strips` strips, `before` of other domains in the launch.  FP64 only:
// lod.hip's FP32 kernel holds whole lines on chip and streams better (400 x 400 x 40, three simulations on
// a stream each: 49 against 57 us per step).  FP64 where 32 rows fit (28 rows of 640 columns: 1597 ->
// 1685), except large fields of rows of whole 128-byte lines below 320 columns, which lod.hip stores
// non-temporally and reads again least.  Microseconds per step of one simulation, lod.hip's x sweep ->
// strips (in brackets: of three in turn, on a stream each): 250 x 230 x 210 x 2 400 -> 297 (351 -> 286),
// 300^3 x 2 829 -> 677 (756 -> 638), 200^3 x 2 208 -> 198 (203 -> 183), 192^3 x 3 280 -> 245 (245 -> 223),
// 160^3 x 4 217 -> 185 (168 -> 169), 400^3 x 2 1552 -> 1478 (1331 -> 1306), 512 x 512 x 128 480 -> 455
// (385 -> 386); 256^3 x 4, with its agents, 862 -> 815, but (696 -> 715).
bool strips_pay(const Group *g, const Domain &d, long long strips, long long before)
{
    if (g->elem != 8 || strips == 0 || before + strips > (1 << 30))
        return false;
    return d.nx * sizeof(double) % 128 != 0 || d.nx >= 320 || d.nvox * d.nsub * sizeof(double) <= kStripSmall;
}

int launch_strips(Group *g, bool agents)
{
    int rc = sync_descriptors(g);
    if (rc)
        return rc;
    const int ndom = (int)g->doms.size();
    const long long strips = g->prefix[kStrip0][ndom];
    if (strips == 0)
        return BFVMB_OK;
    size_t lds = 0, bytes = 0;
    int rows = 0;
    for (const Domain &d : g->doms)
        if (d.strips) {
            lds = std::max(lds, strip_bytes(d.nx, d.strip, sizeof(double)));
            bytes += d.nvox * d.nsub * sizeof(double);
            rows = std::max(rows, d.strip);
        }
    const int solvers = (rows + kWave - 1) / kWave * kWave;
    const bool two = 2 * lds <= kLdsBytes;  // two workgroups per CU share its wavefronts
    const unsigned th = two ? kMaxThreads / 2 : kMaxThreads;
    const unsigned grid = (unsigned)std::min<long long>(strips, (two ? 2 : 1) * std::max(g->cu_count, 1));
    const DomainDesc<double> *d = static_cast<const DomainDesc<double> *>(g->d_desc);
    const long long *pre = g->d_prefix + (size_t)kStrip0 * (ndom + 1);
    const bool nt = bytes > kStripCached;
    const auto k = agents ? (nt ? k_strip<double, true, true> : k_strip<double, true, false>)
                          : (nt ? k_strip<double, false, true> : k_strip<double, false, false>);
    hipLaunchKernelGGL(k, dim3(grid), dim3(th), lds, g->stream, d, pre, ndom, (int)strips, solvers, g->cur);
    return hip_check(g, hipGetLastError(), "strip launch");
}

void resident_class(const Group *g, Domain &d)
{
    const size_t limit = std::min(kLdsBytes, g->max_lds_per_block), el = (size_t)d.nx * d.ny;
    const size_t plain = plane_bytes<false>(d, g->elem), skewed = plane_bytes<true>(d, g->elem);
    const bool skewable = plane_layout<true>(d.nx, g->elem).shift >= 2;
    int c = plain <= limit ? size_class(plain) : skewed <= limit && skewable ? kSkewClass : -1;
    if (c >= 0) {
        const int loads = g->elem == 8 ? (c < kSmallClasses ? plane_loads<double, false>() : plane_loads<double, true>())
                                       : (c < kSmallClasses ? plane_loads<float, false>() : plane_loads<float, true>());
        const size_t solvers = (std::max(d.nx, d.ny) + kWave - 1) / kWave * kWave;
        if (el < 2 || solvers + plane_loaders(el, loads) > kMaxThreads || (long long)d.nz * d.nsub >= (1LL << 30))
            c = -1;
    }
    d.plane_class = c;
}

int launch_planes(Group *g, bool yx, bool agents)
{
    int rc = sync_descriptors(g);
    if (rc)
        return rc;
    return g->precision == BFVMB_FP64 ? launch_planes_t<double>(g, yx, agents) : launch_planes_t<float>(g, yx, agents);
}

int resident_lds_attributes(size_t lds_bytes)
{
    const int bytes = (int)std::min(lds_bytes, kLdsBytes);
    hipError_t e = attributes_all<double>(bytes);
    const void *strip[4] = {(const void *)k_strip<double, false, false>, (const void *)k_strip<double, false, true>,
                            (const void *)k_strip<double, true, false>, (const void *)k_strip<double, true, true>};
    for (int i = 0; i < 4 && e == hipSuccess; ++i)
        e = hipFuncSetAttribute(strip[i], hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess)
        e = attributes_all<float>(bytes);
    return (int)e;
}

}  // namespace bfvmb
