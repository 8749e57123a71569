// Thermophysical-property state shared by the table lookup (props.hip) and
// the learned surrogate (mlp.hip).
#pragma once

#include <type_traits>

#include "chs_common.hpp"

namespace chs {
struct Mlp;
}

// The property handle of the C ABI (declared opaque in chapsim_gpu.h).
struct chs_props {
    int n = 0;                 // knots of the scaled table
    int nbh = 0, nbt = 0;      // buckets of the H and T interval searches
    int kwalk = 0;             // fixed walk steps that make both searches exact (0: walk to the end)
    double h_lo = 0, h_hi = 0, t_lo = 0, t_hi = 0;
    double hbi = 0, tbi = 0;   // 1 / bucket width
    double rhoh_max = 0;       // RHOHmax of NIST_SPLINE_H (the limiter of the energy update)
    hipStream_t stream = nullptr;
    bool own_stream = false;
    int lds_max = 65536;       // LDS bytes a block may use on the table's device
    int ncu = 256;             // compute units of that device
    // device table: knots, bucket starts, per-interval coefficient records
    double* xh = nullptr;      // H knots [n]
    double* xt = nullptr;      // T knots [n]
    int* sh = nullptr;         // H bucket -> first candidate interval [nbh]
    int* st = nullptr;         // T bucket -> first candidate interval [nbt]
    double* rh = nullptr;      // [n][4]: T, b, c, d of the H -> T spline
    double* rt = nullptr;      // [n][16]: (y, b, c, d) of T -> D, M, K, CP
    unsigned long long* counters = nullptr;   // device counters: [4] training and certification, [4] ecnt, [4] ucnt; the tables follow
    unsigned long long* ucnt = nullptr;       // those of chs_therm_prop_update, zero between calls
    // host copies used by the surrogate's certification
    std::vector<double> hH, hT, hrh, hrt;
    // learned surrogate (mlp.hip)
    chs::Mlp* mlp = nullptr;
    // the THERM_PROP_UPDATE form of chs_energy_substep (CHS_PROPS_TABLE or
    // CHS_PROPS_SURROGATE) and the cells its last call handed to the table
    int mode = 0;
    long long last_fallback = 0;
    // the energy substep's range check, read without a stream sync: its
    // device counters, their pinned host
    // copy (ecnt_host[0..1]; [2..3]: that of ucnt), the event that follows the copy, and a resolved count not yet
    // reported
    unsigned long long* ecnt = nullptr;
    unsigned long long* ecnt_host = nullptr;
    hipEvent_t ecnt_ev = nullptr;
    bool ecnt_pending = false, ecnt_sur = false;
    unsigned long long ecnt_bad = 0;
};

namespace chs {

// Rows of cells: row r holds rowlen consecutive values starting at r*stride
// (the interior j-block of one k plane of a ghost-aware array, or one flat run).
struct Rows {
    long long nrow, rowlen, stride;
};

// The range check of the last chs_energy_substep on p (props.hip):
// energy_range_resolve waits for its pending copy; energy_range_check also
// reports cells outside the table, once, as CHS_E_RANGE.
void energy_range_resolve(chs_props* p);
int energy_range_check(chs_props* p, const char* who);
// two device counts to pinned host memory (kernel, no copy), and zeros in their place
int props_counts_out(unsigned long long* c, unsigned long long* host, hipStream_t s);

// LDS bytes of the staged search tables of one lookup block
inline size_t props_lds_bytes(const chs_props* p) {
    return sizeof(double) * 2 * (size_t)p->n + sizeof(int) * ((size_t)p->nbh + p->nbt);
}
// and with the H -> T and T -> D coefficient records staged too (LdsTab<true>)
inline size_t props_lds_wide(const chs_props* p) {
    return sizeof(double) * 9 * (size_t)p->n + sizeof(unsigned short) * ((size_t)p->nbh + p->nbt);
}

// Blocks of a persistent lookup kernel of `threads` threads with the staged
// tables in LDS: as many as are resident at once on the device (registers and
// LDS), at most `want`.
inline int props_grid_occ(const chs_props* p, const void* kernel, int threads, size_t lds, long long want) {
    int per = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, threads, lds) != hipSuccess || per < 1)
        per = 1;
    const long long g = (long long)p->ncu * per;
    return (int)(want < g ? want : g);
}

// Allow a lookup kernel the staged tables' LDS when they exceed the default
// 64 KB per block (props_create has checked them against the device limit).
inline int props_lds_attr(const void* kernel, size_t b) {
    if (b > 65536) {
        hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)b);
        if (e != hipSuccess) {
            set_error(std::string("hipFuncSetAttribute (property tables in LDS): ") + hipGetErrorString(e));
            return CHS_E_HIP;
        }
    }
    return CHS_OK;
}

// Interval i (0-based) with x[i] <= u < x[i+1], for x[0] < u < x[n-1]: the
// result of the reference's bisection (NIST_SLEVAL_*, src/Flow_State.f90:
// 1050-1061).  A bucket gives the first candidate; short walks make it exact
// whatever the rounding of the bucket index.
template <class Ix>
__device__ __forceinline__ int find_interval(const double* x, const Ix* start, int n, int nb, double lo,
                                             double bi, double u) {
    int b = (int)((u - lo) * bi);
    b = b < 0 ? 0 : (b >= nb ? nb - 1 : b);
    int i = start[b];
    while (i < n - 2 && x[i + 1] <= u) ++i;
    while (i > 0 && x[i] > u) --i;
    return i;
}

// find_interval with a fixed number of steps and no branch: at most one step
// back (the rounding of the bucket index) and K forward, K being one more
// than the most knots any bucket holds (props_create checks it), so that the
// searches of several cells interleave.
template <int K, class Ix>
__device__ __forceinline__ int find_interval_k(const double* x, const Ix* start, int n, int nb, double lo,
                                               double bi, double u) {
    int b = (int)((u - lo) * bi);
    b = b < 0 ? 0 : (b >= nb ? nb - 1 : b);
    int i = start[b];
    i -= (i > 0 && x[i] > u) ? 1 : 0;
#pragma unroll
    for (int s = 0; s < K; ++s) i += (i < n - 2 && x[i + 1] <= u) ? 1 : 0;
    return i;
}

template <int K, class Ix>
__device__ __forceinline__ int find_iv(const double* x, const Ix* start, int n, int nb, double lo, double bi,
                                       double u) {
    if constexpr (K > 0)
        return find_interval_k<K>(x, start, n, nb, lo, bi, u);
    else
        return find_interval(x, start, n, nb, lo, bi, u);
}

// y + dx*(b + dx*(c + dx*d)) evaluated as written, without contraction into
// fused multiply-adds (the same roundings as the reference's FP64 code).
__device__ __forceinline__ double cubic_nc(double y, double b, double c, double d, double dx) {
#pragma clang fp contract(off)
    return y + dx * (b + dx * (c + dx * d));
}

// device view of the table
struct PropTab {
    int n, nbh, nbt;
    double h_lo, h_hi, t_lo, t_hi, hbi, tbi;
    const double *xh, *xt, *rh, *rt;
    const int *sh, *st;
};

inline PropTab tab_of(const chs_props* p) {
    PropTab t;
    t.n = p->n;
    t.nbh = p->nbh;
    t.nbt = p->nbt;
    t.h_lo = p->h_lo;
    t.h_hi = p->h_hi;
    t.t_lo = p->t_lo;
    t.t_hi = p->t_hi;
    t.hbi = p->hbi;
    t.tbi = p->tbi;
    t.xh = p->xh;
    t.xt = p->xt;
    t.rh = p->rh;
    t.rt = p->rt;
    t.sh = p->sh;
    t.st = p->st;
    return t;
}

// The table as a lookup block holds it in LDS: the knots and bucket starts of
// both searches and, WIDE, the coefficient records of H -> T (its values are
// the T knots) and T -> D.  A record read from L2 is two 16-byte gathers whose
// 64 lanes touch 64 cache lines, one line a cycle: ten of them a cell (H -> T,
// D, M, K, CP) took 271 us of texture addressing at 12.6 M cells.  LDS serves
// 64 scattered doubles in some ten cycles, and 2048 knots leave room for two of
// the five records (156 KB, one block of 1024 threads per CU).
template <bool WIDE>
struct LdsTab {
    using Ix = std::conditional_t<WIDE, unsigned short, int>;
    const double *xh, *xt;       // knots
    const double *hb, *ty, *tb;  // WIDE: b, c, d of H -> T; values and b, c, d of T -> D
    const Ix *sh, *st;
    // record i of H -> T, record k of T -> D: (y, b, c, d)
    __device__ __forceinline__ double4 ht(const PropTab& t, int i) const {
        if constexpr (WIDE)
            return make_double4(xt[i], hb[3 * i], hb[3 * i + 1], hb[3 * i + 2]);
        else
            return reinterpret_cast<const double4*>(t.rh)[i];
    }
    __device__ __forceinline__ double4 td(const PropTab& t, int k) const {
        if constexpr (WIDE)
            return make_double4(ty[k], tb[3 * k], tb[3 * k + 1], tb[3 * k + 2]);
        else
            return reinterpret_cast<const double4*>(t.rt)[4 * (size_t)k];
    }
};

// Stage the table (all threads of the block; ends with a barrier):
// props_lds_wide() or props_lds_bytes() bytes.
template <bool WIDE>
__device__ __forceinline__ LdsTab<WIDE> stage_tab(const PropTab& t, unsigned char* smem) {
    using Ix = typename LdsTab<WIDE>::Ix;
    double* a = reinterpret_cast<double*>(smem);
    double *b = a + t.n, *e = b + t.n;
    double *hb = nullptr, *ty = nullptr, *tb = nullptr;
    if constexpr (WIDE) {
        hb = e;
        ty = hb + 3 * t.n;
        tb = ty + t.n;
        e = tb + 3 * t.n;
    }
    Ix *c = reinterpret_cast<Ix*>(e), *d = c + t.nbh;
    // SB entries of every array in flight per thread (entries past the last:
    // that one again): the staging is a chain of L2 latencies otherwise, 13 us
    // of a call of k_energy_props (1024 threads), 7 batched; k_energy_wall (256
    // threads) 11.5 -> 6.8 us
    constexpr int SB = 4;
    const int bd = blockDim.x;
    for (int q0 = threadIdx.x; q0 < t.n; q0 += SB * bd) {
        double vh[SB], vt[SB];
        double4 r[SB], s[SB];
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            const int q = min(q0 + u * bd, t.n - 1);
            vh[u] = t.xh[q];
            vt[u] = t.xt[q];
            if constexpr (WIDE) {
                r[u] = reinterpret_cast<const double4*>(t.rh)[q];
                s[u] = reinterpret_cast<const double4*>(t.rt)[4 * (size_t)q];
            }
        }
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            const int q = min(q0 + u * bd, t.n - 1);
            a[q] = vh[u];
            b[q] = vt[u];
            if constexpr (WIDE) {
                hb[3 * q] = r[u].y, hb[3 * q + 1] = r[u].z, hb[3 * q + 2] = r[u].w;
                ty[q] = s[u].x;
                tb[3 * q] = s[u].y, tb[3 * q + 1] = s[u].z, tb[3 * q + 2] = s[u].w;
            }
        }
    }
    const int nbm = max(t.nbh, t.nbt);
    for (int q0 = threadIdx.x; q0 < nbm; q0 += SB * bd) {
        int vc[SB], vd[SB];
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            vc[u] = t.sh[min(q0 + u * bd, t.nbh - 1)];
            vd[u] = t.st[min(q0 + u * bd, t.nbt - 1)];
        }
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            c[min(q0 + u * bd, t.nbh - 1)] = (Ix)vc[u];
            d[min(q0 + u * bd, t.nbt - 1)] = (Ix)vd[u];
        }
    }
    __syncthreads();
    return LdsTab<WIDE>{a, b, hb, ty, tb, c, d};
}

// The T intervals k of N cells whose T came out of the H intervals i.  The T
// knots are the H -> T spline's values at the H knots, so k = i unless the
// spline overshoots or rounds past a knot, or T was set: the search is left to
// those cells, in one branch for all N so that their chains still interleave.
template <int KW, int N, class Ix>
__device__ __forceinline__ void t_intervals(const PropTab& t, const double* xt, const Ix* st, const int (&i)[N],
                                            const double (&tq)[N], int (&k)[N]) {
    bool miss = false;
#pragma unroll
    for (int u = 0; u < N; ++u) {
        k[u] = i[u];
        miss |= !(xt[i[u]] <= tq[u] && tq[u] < xt[i[u] + 1]);
    }
    if (miss) {
#pragma unroll
        for (int u = 0; u < N; ++u) k[u] = find_iv<KW>(xt, st, t.n, t.nbt, t.t_lo, t.tbi, tq[u]);
    }
}

// A DPP move of a double2 (CTRL: quad_perm)
template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ double2 dpp_d2(double2 v) {
    const double x = __hiloint2double(dpp_i<CTRL>(__double2hiint(v.x)), dpp_i<CTRL>(__double2loint(v.x)));
    const double y = __hiloint2double(dpp_i<CTRL>(__double2hiint(v.y)), dpp_i<CTRL>(__double2loint(v.y)));
    return make_double2(x, y);
}

// One step of a transpose between lanes l and l ^ 1 (CTRL 0xB1) or l ^ 2
// (0x4E): the lane with the bit set gives a and takes the other's b for it,
// the other gives b.
template <int CTRL>
__device__ __forceinline__ void lane_swap(bool bit, double2& a, double2& b) {
    const double2 send = make_double2(bit ? a.x : b.x, bit ? a.y : b.y), got = dpp_d2<CTRL>(send);
    a = make_double2(bit ? got.x : a.x, bit ? got.y : a.y);
    b = make_double2(bit ? b.x : got.x, bit ? b.y : got.y);
}

// The records of interval k from global memory, by the lanes of a quad
// together (every lane of the wave takes part): a lane's own 16-byte loads
// touch 64 cache lines an instruction, one line a cycle, while four lanes that
// load the four 16-byte pieces of one cell's M and K records touch 16.  The
// pieces then change lanes (DPP).  D and CP by quads as well: 212 us a call of
// k_props_table with cp, 189 without, against 214 and 177.
__device__ __forceinline__ void quad_mk(const double* rt, int k, double4& cm, double4& ck) {
    const int p = threadIdx.x & 3;
    const int k0 = dpp_i<0x00>(k), k1 = dpp_i<0x55>(k), k2 = dpp_i<0xAA>(k), k3 = dpp_i<0xFF>(k);
    const double2* b = reinterpret_cast<const double2*>(rt) + 2 + p;   // 8 double2 a record of four; M and K: 2 to 5
    double2 v0 = b[8 * (size_t)k0], v1 = b[8 * (size_t)k1], v2 = b[8 * (size_t)k2], v3 = b[8 * (size_t)k3];
    lane_swap<0xB1>(p & 1, v0, v1);
    lane_swap<0xB1>(p & 1, v2, v3);
    lane_swap<0x4E>(p & 2, v0, v2);
    lane_swap<0x4E>(p & 2, v1, v3);
    cm = make_double4(v0.x, v0.y, v1.x, v1.y);
    ck = make_double4(v2.x, v2.y, v3.x, v3.y);
}
// the CP record, by pairs of lanes
__device__ __forceinline__ double4 pair_cp(const double* rt, int k) {
    const int p = threadIdx.x & 1;
    const int k0 = dpp_i<0xA0>(k), k1 = dpp_i<0xF5>(k);   // of the pair's even and odd lane
    const double2* b = reinterpret_cast<const double2*>(rt) + 6 + p;
    double2 v0 = b[8 * (size_t)k0], v1 = b[8 * (size_t)k1];
    lane_swap<0xB1>(p, v0, v1);
    return make_double4(v0.x, v0.y, v1.x, v1.y);
}

// S_HT (NIST_SLEVAL_HT, src/Flow_State.f90:1015-1070): false when h leaves
// the table (the reference STOPs); hack: |h| < 1e-10 gives T = 1.  A NaN
// passes the range tests and gives NaN, as there.
template <int KW = 0>
__device__ __forceinline__ bool spline_ht(const PropTab& t, const double* xh, const int* sh, double hv, double& T,
                                          bool hack) {
    if (hv != hv) {
        T = hv;
        return true;
    }
    if (hv <= t.h_lo || hv >= t.h_hi) return false;
    const int i = find_iv<KW>(xh, sh, t.n, t.nbh, t.h_lo, t.hbi, hv);
    const double4 r = reinterpret_cast<const double4*>(t.rh)[i];
    T = cubic_nc(r.x, r.y, r.z, r.w, hv - xh[i]);
    if (hack && fabs(hv) < 1.0e-10) T = 1.0;
    return true;
}

// S_TD, S_TM, S_TK, S_TCp at T (NIST_SLEVAL_TD/TM/TK/TCp, src/Flow_State.f90:
// 1415-1692): one interval search for all four; |T - 1| < 1e-10 gives
// D = M = K = CP = 1 (each evaluator's own rule, :1470, :1524, :1578, :1686).
template <int KW = 0>
__device__ __forceinline__ bool spline_t(const PropTab& t, const double* xt, const int* st, double tv, double& D,
                                         double& Mu, double& K, double& CP) {
    if (tv != tv) {
        D = Mu = K = CP = tv;
        return true;
    }
    if (tv <= t.t_lo || tv >= t.t_hi) return false;
    const int k = find_iv<KW>(xt, st, t.n, t.nbt, t.t_lo, t.tbi, tv);
    const double4* q = reinterpret_cast<const double4*>(t.rt) + 4 * (size_t)k;
    const double4 cd = q[0], cm = q[1], ck = q[2], cc = q[3];
    const double dt = tv - xt[k];
    D = cubic_nc(cd.x, cd.y, cd.z, cd.w, dt);
    Mu = cubic_nc(cm.x, cm.y, cm.z, cm.w, dt);
    K = cubic_nc(ck.x, ck.y, ck.z, ck.w, dt);
    CP = cubic_nc(cc.x, cc.y, cc.z, cc.w, dt);
    if (fabs(tv - 1.0) < 1.0e-10) D = Mu = K = CP = 1.0;
    return true;
}

// THERM_PROP_UPDATE of one cell (the caller skips |h| < 1e-10); false
// (outputs untouched) when h or T leaves the table.
// S_TD alone (DENSITY_UPDATE needs only the density): the same interval
// search and the same evaluation as spline_t, reading only the density's
// coefficients of the interval's record.
template <int KW = 0>
__device__ __forceinline__ bool spline_t_density(const PropTab& t, const double* xt, const int* st, double tv,
                                                 double& D) {
    if (tv != tv) {
        D = tv;
        return true;
    }
    if (tv <= t.t_lo || tv >= t.t_hi) return false;
    const int k = find_iv<KW>(xt, st, t.n, t.nbt, t.t_lo, t.tbi, tv);
    const double4 cd = reinterpret_cast<const double4*>(t.rt)[4 * (size_t)k];
    D = cubic_nc(cd.x, cd.y, cd.z, cd.w, tv - xt[k]);
    if (fabs(tv - 1.0) < 1.0e-10) D = 1.0;
    return true;
}

template <int KW = 0>
__device__ __forceinline__ bool lookup_cell(const PropTab& t, const double* xh, const double* xt, const int* sh,
                                            const int* st, double hv, double& T, double& D, double& Mu, double& K,
                                            double& CP) {
    double tv;
    if (!spline_ht<KW>(t, xh, sh, hv, tv, false)) return false;
    if (!spline_t<KW>(t, xt, st, tv, D, Mu, K, CP)) return false;
    T = tv;
    return true;
}

}  // namespace chs
