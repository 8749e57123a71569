// Standalone batched tridiagonal solves: the C-ABI chs_tdma_batched, which
// stands in for the reference's four line solvers
//   TDMAIJJ_nonCYC (src/TDMAIJJ_nonCYC.f90:67-123)   TDMAIJI_nonCYC (src/TDMAIJI_nonCYC.f90:67-123)
//   TDMAIJJ_CYC    (src/TDMAIJJ_CYC.f90:67-157)      TDMAIJI_CYC    (src/TDMAIJI_CYC.f90:67-157)
// on arbitrary line/element strides.
#include "chs_common.hpp"
#include "tdma_dev.hpp"

namespace chs {

// Segmented solver: LPB lines per block, P = ceil(n / MS) segments per line.
// Consecutive lanes take consecutive lines (also where the rows are the
// contiguous ones: non-cyclic 65536 x 192, 0.203 ms, 0.319 with consecutive
// segments of a line), or with ROWC consecutive segments of one line (short
// cyclic lines with contiguous rows: 65536 x 32, 8 lines a block, 26.4 against
// 30.6 us).  SERIAL (cyclic): one thread per line sweeps the reduced system.
template <int MS, bool CYC, bool ROWC = false, bool SERIAL = false>
__global__ void __launch_bounds__(1024) k_tdma_seg(const double* __restrict__ A, const double* __restrict__ B,
                                                   const double* __restrict__ Cc, double* __restrict__ Rr,
                                                   const double* __restrict__ bc, int n, int nlines,
                                                   long long es, long long ls, int LPB, int P) {
    extern __shared__ unsigned char smem[];
    const int tid = threadIdx.x;
    int ll = ROWC ? tid / P : tid % LPB, seg = ROWC ? tid % P : tid / LPB;
    // hides that ll and seg come from one division: with that known the loads'
    // addresses are kept apart in registers (126 instead of 92 at MS = 8)
    asm("" : "+v"(ll), "+v"(seg));
    const long long line = (long long)blockIdx.x * LPB + ll;
    const bool valid = line < nlines;
    double a[MS], b[MS], c[MS], d[MS];
    const long long base = valid ? line * ls : 0;
    // branch-free loads (rows past n read row n - 1 of a valid line), all
    // issued before the first wait; padding rows become identity rows
#pragma unroll
    for (int l = 0; l < MS; ++l) {
        const long long o = base + (long long)min(seg * MS + l, n - 1) * es;
        a[l] = A[o];
        b[l] = B[o];
        c[l] = Cc[o];
        d[l] = Rr[o];
    }
#pragma unroll
    for (int l = 0; l < MS; ++l) {
        if (!(valid && seg * MS + l < n)) {   // padding rows: identity, decoupled
            a[l] = 0.0;
            b[l] = 1.0;
            c[l] = 0.0;
            d[l] = 0.0;
        }
    }
    if (!CYC && valid) {
        // the end rows take the boundary values BC(line,1:2) (TDMAIJJ_nonCYC.f90:93-97,108-113)
        if (seg == 0) {
            if (bc) d[0] = d[0] - a[0] * bc[line];
            a[0] = 0.0;
        }
        const int jl = n - 1;
        if (jl / MS == seg) {
            const int l = jl % MS;
#pragma unroll
            for (int q = 0; q < MS; ++q)
                if (q == l) {
                    if (bc) d[q] = d[q] - c[q] * bc[nlines + line];
                    c[q] = 0.0;
                }
        }
    }
    seg_solve<MS, double, SERIAL>(a, b, c, d, LPB, P, ll, seg, valid, CYC, smem);
    if (valid) {
#pragma unroll
        for (int l = 0; l < MS; ++l) {
            const int j = seg * MS + l;
            if (j < n) Rr[base + (long long)j * es] = d[l];
        }
    }
}

// Cyclic lines of any length (k_tdma_seg's cyclic form needs n to be a whole
// number of segments, since the wrap couples the last real row): the last
// unknown is split off, the n-1 rows left are a non-cyclic line, padded with
// identity rows like any other, with two right-hand sides held as one double2:
// r, and minus the couplings to x_{n-1}, so that x_i = y_i + z_i x_{n-1} and
// the line's last equation gives x_{n-1}.  The reduced systems go through the
// parallel cyclic reduction of all segment threads.  At most 512 threads: the
// double2 rows need more than the 128 registers of a 1024-thread block.
// Bound by the latency of its load - eliminate - reduce chain on few lines,
// by HBM on many (40 B a row).  Replaces one thread per line with a device
// workspace (k_tdma_seq): 1500 lines of 135 rows,
// rows contiguous, 230 -> 8.4 us.
template <int MS>
__global__ void __launch_bounds__(512) k_tdma_cyc(const double* __restrict__ A, const double* __restrict__ B,
                                                  const double* __restrict__ Cc, double* __restrict__ Rr, int n,
                                                  int nlines, long long es, long long ls, int LPB, int P) {
    extern __shared__ unsigned char smem[];
    const int tid = threadIdx.x, ni = n - 1;
    // rows contiguous: consecutive lanes take consecutive segments of a line
    const bool rowc = es == 1;
    const int ll = rowc ? tid / P : tid % LPB, seg = rowc ? tid % P : tid / LPB;
    const long long line = (long long)blockIdx.x * LPB + ll;
    const bool valid = line < nlines;
    const long long base = valid ? line * ls : 0;
    double a[MS], b[MS], c[MS];
    double2 d[MS];
#pragma unroll
    for (int l = 0; l < MS; ++l) {
        const long long o = base + (long long)min(seg * MS + l, ni - 1) * es;
        a[l] = A[o];
        b[l] = B[o];
        c[l] = Cc[o];
        d[l].x = Rr[o];
    }
    const long long on = base + (long long)ni * es;   // the line's last row
    const double an = A[on], bn = B[on], cn = Cc[on], rn = Rr[on];
#pragma unroll
    for (int l = 0; l < MS; ++l) {
        const int j = seg * MS + l;
        d[l].y = (j == 0 ? -a[l] : 0.0) + (j == ni - 1 ? -c[l] : 0.0);
        if (j == 0) a[l] = 0.0;
        if (j == ni - 1) c[l] = 0.0;
        if (!(valid && j < ni)) {   // padding rows: identity, decoupled
            a[l] = 0.0;
            b[l] = 1.0;
            c[l] = 0.0;
            d[l] = make_double2(0.0, 0.0);
        }
    }
    seg_solve<MS, double2>(a, b, c, d, LPB, P, ll, seg, valid, false, smem);
    // the reduced systems are dead (seg_solve's last barrier): the line's end
    // values (y_0, z_0), (y_{n-2}, z_{n-2}) take their place
    double2* ends = reinterpret_cast<double2*>(smem);
    if (seg == 0) ends[2 * ll] = d[0];
    if ((ni - 1) / MS == seg) {
#pragma unroll
        for (int l = 0; l < MS; ++l)
            if (l == (ni - 1) % MS) ends[2 * ll + 1] = d[l];
    }
    __syncthreads();
    if (!valid) return;
    const double2 e0 = ends[2 * ll], e1 = ends[2 * ll + 1];
    const double xn = (rn - cn * e0.x - an * e1.x) / (bn + cn * e0.y + an * e1.y);
#pragma unroll
    for (int l = 0; l < MS; ++l) {
        const int j = seg * MS + l;
        if (j < ni) Rr[base + (long long)j * es] = d[l].x + d[l].y * xn;
    }
    if (seg == 0) Rr[on] = xn;
}

// Fallback for shapes the segmented kernels do not cover: one thread per
// line, the reference recurrences, H/G in a device workspace.
__global__ void k_tdma_seq(const double* __restrict__ A, const double* __restrict__ B,
                           const double* __restrict__ Cc, double* __restrict__ Rr, const double* __restrict__ bc,
                           int n, int nlines, long long es, long long ls, int cyclic, double* __restrict__ ws) {
    const long long line = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (line >= nlines) return;
    const double* a = A + line * ls;
    const double* b = B + line * ls;
    const double* c = Cc + line * ls;
    double* r = Rr + line * ls;
    // workspace rows are interleaved over lines: coalesced
    double* H = ws + line;
    double* G = ws + (long long)n * nlines + line;
    double* G2 = ws + 2LL * n * nlines + line;
    const long long wst = nlines;
    if (!cyclic) {
        const double blo = bc ? bc[line] : 0.0, bhi = bc ? bc[nlines + line] : 0.0;
        H[0] = c[0] / b[0];
        G[0] = (r[0] - a[0] * blo) / b[0];
        for (int j = 1; j < n - 1; ++j) {
            const double pp = 1.0 / (b[j * es] - H[(j - 1) * wst] * a[j * es]);
            H[j * wst] = c[j * es] * pp;
            G[j * wst] = (r[j * es] - a[j * es] * G[(j - 1) * wst]) * pp;
        }
        const int j = n - 1;
        const double pp = 1.0 / (b[j * es] - H[(j - 1) * wst] * a[j * es]);
        double x = (r[j * es] - c[j * es] * bhi - a[j * es] * G[(j - 1) * wst]) * pp;
        r[j * es] = x;
        for (int jj = n - 2; jj >= 0; --jj) {
            x = G[jj * wst] - H[jj * wst] * x;
            r[jj * es] = x;
        }
        return;
    }
    H[(n - 2) * wst] = 0.0;
    H[0] = c[0] / b[0];
    G[0] = r[0] / b[0];
    G2[0] = -a[0] / b[0];
    for (int i = 1; i <= n - 3; ++i) {
        const double pp = 1.0 / (b[i * es] - H[(i - 1) * wst] * a[i * es]);
        const double q1 = G[(i - 1) * wst] * a[i * es], q2 = G2[(i - 1) * wst] * a[i * es];
        H[i * wst] = c[i * es] * pp;
        G[i * wst] = (r[i * es] - q1) * pp;
        G2[i * wst] = -q2 * pp;
    }
    {
        const int i = n - 2;
        const double pp = 1.0 / (b[i * es] - H[(i - 1) * wst] * a[i * es]);
        const double q1 = G[(i - 1) * wst] * a[i * es], q2 = G2[(i - 1) * wst] * a[i * es];
        G[i * wst] = (r[i * es] - q1) * pp;
        G2[i * wst] = (-c[i * es] - q2) * pp;
    }
    for (int i = n - 3; i >= 0; --i) {
        G[i * wst] = -H[i * wst] * G[(i + 1) * wst] + G[i * wst];
        G2[i * wst] = -H[i * wst] * G2[(i + 1) * wst] + G2[i * wst];
    }
    const int i = n - 1;
    const double pp = r[i * es] - c[i * es] * G[0] - a[i * es] * G[(i - 1) * wst];
    const double qq = b[i * es] + c[i * es] * G2[0] + a[i * es] * G2[(i - 1) * wst];
    const double xn = pp / qq;
    r[i * es] = xn;
    for (int k = n - 2; k >= 0; --k) r[k * es] = G[k * wst] + G2[k * wst] * xn;
}

// Choose the segmented configuration for (n, cyclic) within maxthr threads per
// block, or return false.  8-row segments keep the solver within 128 VGPRs.
// lpb_small: blocks of 8 lines (several blocks per CU overlap their load,
// reduce and store phases; measured faster for the complex-valued Poisson
// lines, slower for the real batched solver)
#ifndef CHS_TDMA_LPB
#define CHS_TDMA_LPB 64
#endif
bool tdma_seg_config(int n, bool cyclic, int* MS, int* P, int* LPB, int maxthr, bool lpb_small) {
    const int cand[4] = {8, 12, 16, 4};
    const int lpbs_big[2] = {CHS_TDMA_LPB, CHS_TDMA_LPB == 64 ? 32 : CHS_TDMA_LPB}, lpbs_small[2] = {8, 8};
    const int* lpbs = lpb_small ? lpbs_small : lpbs_big;
    for (int ms : cand) {
        for (int q = 0; q < 2; ++q) {
            const int lpb = lpbs[q];
            const int p = (n + ms - 1) / ms;
            if (p * lpb > maxthr) continue;
            // cyclic lines cannot be padded (the wrap couples the last real row)
            if (cyclic && (n % ms != 0 || p < 2)) continue;
            *MS = ms;
            *P = p;
            *LPB = lpb;
            return true;
        }
    }
    return false;
}

// Lines per block of lpb0 (a power of two), halved to at least lo while the
// block of p threads per line has more than thr threads.
static int lines_per_block(int p, int lpb0, int lo, int thr) {
    int lpb = lpb0;
    while (lpb > lo && p * lpb > thr) lpb /= 2;
    return lpb;
}

// The kernel of a batch of lines: k_tdma_seg with its reduced systems by
// parallel cyclic reduction (Pcr) or, cyclic, by one thread per line (Serial);
// k_tdma_cyc (Split); k_tdma_seq (Seq), the only one with a workspace.
enum class TdmaKind { Pcr, Serial, Split, Seq };
struct TdmaPlan {
    TdmaKind kind;
    int ms, lpb;   // rows per segment, lines per block
    bool rowc;     // consecutive lanes take consecutive segments of a line
};

// Rows per segment and lines per block by the number of lines and rows, from a
// sweep of all of them on an MI355X: 42 lengths from 8 to 512 rows x 20 to 23
// counts from 16 to 65536 lines, both layouts.  Over the sweep the choice is on
// average 2% (lines contiguous), 11% and 7% (rows contiguous, non-cyclic and
// cyclic) behind the fastest candidate of each point; what it loses most at:
// 30% to 2 lines a block (64 lines of 512 rows, 11.5 against 8.9 us), 20% to 2
// lines of 4-row segments (65536x192, rows contiguous, 181 against 145).  What
// decides:
//   fullest CU    on_cu(lpb): the lines of the CU with the most, in whole
//     blocks.  Where 32 lines a block leave it no more than 16 do, the larger
//     accesses win (non-cyclic 65536x128 72 us with 32, 85 with 16; 14000x144,
//     12 x 32, 21.6, 8 x 16 23.1), otherwise the evener split (20000x128 22.5,
//     21.3).
//   straddled     16 lines are one 128-byte line only where the row pitch is a
//     multiple of 16 values; elsewhere they touch two, 64 lines five for four
//     (8500x64 16 lines 11.6 us, 32 10.5, 64 9.7; 32767x64 26.4, 21.0, 19.7)
//   resident      above 4096 lines a block of at most 8 waves, so that two on
//     a CU overlap their phases: 12-row segments for 257 to 384 rows (10000x360
//     12 x 16 40.9 us, 8 x 16 50.5, 8 x 8 51.5), 8 lines beyond (10000x504 61.8
//     against 71.1)
//   few lines     fewer lines a block, so that no CU is idle: 16 up to 4096
//     lines (2000x192 8.9 us; 8 lines 10.8, 32 12.1), 8 below 1280 (1000x192
//     8.0, 16 lines 9.1)
//   rows contiguous  blocks of about 128 threads: 10000x360 58 us (8 lines 69,
//     16 80); 4-row segments (8 waves to a SIMD for the 5 of 8-row ones) for
//     17 to 128 rows from 14000 lines on (65536x28 20 us, 8 x 16 26; 45000x56
//     27, 8 x 16 37; 32768x120 48, 8 x 16 58)
//   cyclic        short lines of whole segments: the serial sweep of a reduced
//     system of up to 20 rows (32 at most) has two barriers where the cyclic
//     reduction has two a step (10000x16 3.9 us, Split 4.9; 65536x96 12 x 32
//     57, Split 68; rows contiguous 65536x8 6.9, Split 10.9); whole 12-row
//     segments of 132 to 192 rows (65536x192 121 us, Split 150) and of 257 to
//     384 (10000x360 42, Split 60); everything else Split
static TdmaPlan tdma_plan(int n, int nlines, long long es, long long ls, bool cyclic) {
    constexpr int CUS = 256;
    const int p8 = (n + 7) / 8, p12 = (n + 11) / 12, ps = (n + 6) / 8;   // segments; ps: of the n - 1 rows of Split
    const bool whole8 = n % 8 == 0, whole12 = n % 12 == 0;
    auto on_cu = [&](long lpb) { return ((nlines + lpb - 1) / lpb + CUS - 1) / CUS * lpb; };
    const bool wide = on_cu(32) <= on_cu(16), straddled = es % 16 != 0, few = nlines <= 4096;
    const bool at_once = nlines <= 64 * CUS;   // every block of 64 lines on a CU of its own
    auto split = [&](int lpb) {
        lpb = lines_per_block(ps, lpb, 2, 512);
        return TdmaPlan{ps * lpb <= 512 ? TdmaKind::Split : TdmaKind::Seq, 8, lpb, es == 1};
    };
    auto pcr = [&](int ms, int lpb) {
        const int p = (n + ms - 1) / ms;
        lpb = lines_per_block(p, lpb, 4, 1024);
        return TdmaPlan{p * lpb <= 1024 ? TdmaKind::Pcr : TdmaKind::Seq, ms, lpb, false};
    };
    auto serial = [&](int ms, int lpb) { return TdmaPlan{TdmaKind::Serial, ms, lpb, es == 1}; };
    // 16, 32 or 64 of more than 4096 contiguous lines, in blocks of p threads a line
    auto lines = [&](int p) { return straddled && nlines > 8192 && (at_once || p <= 8) ? 64 : wide ? 32 : 16; };

    if (!cyclic && ls == 1) {
        if (p8 <= 2) return pcr(8, 64);
        if (nlines < 1280) return pcr(8, p8 <= 6 ? 16 : 8);
        if (few) return pcr(8, 16);
        if (p8 <= 4) return pcr(8, straddled && nlines > 8192 ? 64 : 32);
        if (p8 <= 16) return p12 == 8 && wide && !at_once ? pcr(12, 32) : pcr(8, lines(p8));
        if (p8 <= 32 && nlines <= 8192 && wide) return pcr(8, 32);
        if (p12 <= 16 && wide) return pcr(12, 32);
        if (p8 <= 32) return pcr(8, 16);
        if (p12 <= 32) return pcr(12, wide ? 32 : 16);
        return pcr(8, 8);
    }
    if (!cyclic) {
        if (p8 >= 3 && p8 <= 16 && nlines >= 14000) return pcr(4, 8);
        if (p8 <= 2) return pcr(8, p8 == 2 && nlines >= 30000 ? 16 : 32);
        return pcr(8, lines_per_block(p8, 16, 4, 128));
    }
    if (ls == 1) {
        const int ms = whole12 && n >= 24 ? 12 : whole8 && n >= 16 ? 8 : n % 4 == 0 && n >= 8 && n <= 20 ? 4 : 0;
        const int p = ms ? n / ms : n;
        if (ms && few && p <= (ms == 12 ? 4 : 6)) return serial(ms, p <= 3 && ms < 12 ? 32 : 16);
        if (ms && !few && p <= (ms == 12 ? 8 : 10)) {
            const bool l64 = on_cu(64) <= on_cu(32) && (at_once || (p <= 8 && (straddled || nlines <= 32768)));
            return serial(ms, l64 ? 64 : 32);
        }
        if (whole8 && p8 <= 16 && straddled && at_once && nlines > 8192) return serial(8, 64);
        if (whole12 && !few && p12 >= 11 && p12 <= 16) return pcr(12, wide ? 32 : 16);
        if (n > 256 && n <= 384 && nlines >= 1280) {
            if (whole12) return pcr(12, 16);
            if (whole8) return pcr(8, 16);
        }
        return split(nlines < 1280 ? (ps <= 4 ? 16 : 8) : few ? 16 : lines(ps));
    }
    if (whole8 && p8 >= 2 && p8 <= 8 && (p8 <= 6 || !few))
        return serial(8, p8 == 2 ? 32 : p8 == 3 && nlines <= 8192 ? 16 : 8);
    if (n % 4 == 0 && n >= 8 && n <= 28 && (n <= 12 || nlines >= 14000)) return serial(4, n == 12 || n == 28 ? 16 : 32);
    return split(lines_per_block(ps, 64, 2, 64));
}

// ws: the workspace of k_tdma_seq, 3 n nlines doubles, or nullptr to take it
// from the stream-ordered pool for this launch
int tdma_launch(const double* a, const double* b, const double* c, double* r, const double* bc, int n, int nlines,
                long long es, long long ls, int cyclic, hipStream_t s, double* ws_given = nullptr) {
    const TdmaPlan t = tdma_plan(n, nlines, es, ls, cyclic != 0);
    const int LPB = t.lpb;
    if (t.kind == TdmaKind::Split) {
        const int P = (n - 1 + t.ms - 1) / t.ms;
        const size_t sm = std::max(seg_smem_bytes<double2>(LPB, P), 2 * sizeof(double2) * (size_t)LPB);
        CHS_LAUNCH(k_tdma_cyc<8>, dim3((nlines + LPB - 1) / LPB), dim3(LPB * P), sm, s, a, b, c, r, n, nlines, es, ls,
                   LPB, P);
        return CHS_OK;
    }
    if (t.kind != TdmaKind::Seq) {
        const int P = (n + t.ms - 1) / t.ms;
        const dim3 grid((nlines + LPB - 1) / LPB), block(LPB * P);
        const size_t sm = seg_smem_bytes<double>(LPB, P, cyclic && t.kind == TdmaKind::Pcr);   // at most 64 KiB
#define CHS_SEG(...) \
    CHS_LAUNCH((k_tdma_seg<__VA_ARGS__>), grid, block, sm, s, a, b, c, r, bc, n, nlines, es, ls, LPB, P)
        if (t.kind == TdmaKind::Serial) {
            if (t.ms == 12) CHS_SEG(12, true, false, true);
            else if (t.ms == 8 && t.rowc) CHS_SEG(8, true, true, true);
            else if (t.ms == 8) CHS_SEG(8, true, false, true);
            else if (t.rowc) CHS_SEG(4, true, true, true);
            else CHS_SEG(4, true, false, true);
        } else if (cyclic) {
            if (t.ms == 12) CHS_SEG(12, true);
            else CHS_SEG(8, true);
        } else {
            if (t.ms == 12) CHS_SEG(12, false);
            else if (t.ms == 4) CHS_SEG(4, false);
            else CHS_SEG(8, false);
        }
#undef CHS_SEG
        return CHS_OK;
    }
    const int bs = 256;
    if (ws_given) {
        CHS_LAUNCH(k_tdma_seq, dim3((nlines + bs - 1) / bs), dim3(bs), 0, s, a, b, c, r, bc, n, nlines, es, ls, cyclic,
                   ws_given);
        return CHS_OK;
    }
    double* ws = nullptr;
    CHS_HIP(hipMallocAsync((void**)&ws, sizeof(double) * 3 * (size_t)n * nlines, s));
    CHS_LAUNCH(k_tdma_seq, dim3((nlines + bs - 1) / bs), dim3(bs), 0, s, a, b, c, r, bc, n, nlines, es, ls, cyclic, ws);
    CHS_HIP(hipFreeAsync(ws, s));
    return CHS_OK;
}

// Workspace of the allocation-free entry point: one copy per GPU, held until
// the process ends.  Host code never passes `scratch` itself to a kernel (its
// host-side name is not a device address); it uses the address that
// hipGetSymbolAddress returns on each device, kept in scratch_dev[].
constexpr size_t TDMA_SCRATCH_DOUBLES = size_t(4) << 20;   // 32 MiB
static __device__ __align__(256) double scratch[TDMA_SCRATCH_DOUBLES];

static std::mutex scratch_mu;
static double* scratch_dev[64] = {};

// The current device's scratch address, looked up once per device.
static int scratch_address(double** out) {
    int dev = 0;
    CHS_HIP(hipGetDevice(&dev));
    CHS_CHECK(dev >= 0 && dev < 64, CHS_E_ARG, "chs_tdma_batched_noalloc: device ordinal above 63");
    std::lock_guard<std::mutex> lk(scratch_mu);
    if (!scratch_dev[dev]) {
        void* p = nullptr;
        CHS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        scratch_dev[dev] = static_cast<double*>(p);
    }
    *out = scratch_dev[dev];
    return CHS_OK;
}

}  // namespace chs

extern "C" int chs_tdma_batched(const double* a_dev, const double* b_dev, const double* c_dev, double* r_dev,
                                const double* bc_dev, int n, int nlines, long long elem_stride,
                                long long line_stride, int cyclic, void* stream) {
    CHS_CHECK(a_dev && b_dev && c_dev && r_dev, CHS_E_ARG, "chs_tdma_batched: null array");
    CHS_CHECK(n >= 3, CHS_E_ARG, "chs_tdma_batched: n must be >= 3 (the reference reads outside its arrays below that)");
    CHS_CHECK(nlines >= 0, CHS_E_ARG, "chs_tdma_batched: nlines < 0");
    CHS_CHECK(elem_stride != 0 || n == 1, CHS_E_ARG, "chs_tdma_batched: zero element stride");
    if (nlines == 0) return CHS_OK;
    return chs::tdma_launch(a_dev, b_dev, c_dev, r_dev, cyclic ? nullptr : bc_dev, n, nlines, elem_stride,
                            line_stride, cyclic, (hipStream_t)stream);
}

// chs_tdma_batched without any allocation: of its kernels only k_tdma_seq has a
// workspace, this GPU's static scratch array.  Lines that no segments of a
// block of 32 divide (tdma_seg_config) are held to the size of that array,
// whichever kernel takes them: the limit callers are promised does not move
// with tdma_plan.
extern "C" int chs_tdma_batched_noalloc(const double* a_dev, const double* b_dev, const double* c_dev, double* r_dev,
                                        const double* bc_dev, int n, int nlines, long long elem_stride,
                                        long long line_stride, int cyclic, void* stream) {
    CHS_CHECK(a_dev && b_dev && c_dev && r_dev, CHS_E_ARG, "chs_tdma_batched_noalloc: null array");
    CHS_CHECK(n >= 3, CHS_E_ARG, "chs_tdma_batched_noalloc: n must be >= 3 (the reference reads outside its arrays below that)");
    CHS_CHECK(nlines >= 0, CHS_E_ARG, "chs_tdma_batched_noalloc: nlines < 0");
    CHS_CHECK(elem_stride != 0, CHS_E_ARG, "chs_tdma_batched_noalloc: zero element stride");
    if (nlines == 0) return CHS_OK;
    int MS = 0, P = 0, LPB = 0;
    double* ws = nullptr;
    CHS_CHECK(chs::tdma_seg_config(n, cyclic != 0, &MS, &P, &LPB, 1024, false) ||
                  3 * (size_t)n * (size_t)nlines <= chs::TDMA_SCRATCH_DOUBLES,
              CHS_E_ARG,
              "chs_tdma_batched_noalloc: lines of this length are held to 3*n*nlines <= 4194304, the doubles of the "
              "static scratch array (use chs_tdma_batched)");
    if (chs::tdma_plan(n, nlines, elem_stride, line_stride, cyclic != 0).kind == chs::TdmaKind::Seq) {
        const int st = chs::scratch_address(&ws);
        if (st != CHS_OK) return st;
    }
    return chs::tdma_launch(a_dev, b_dev, c_dev, r_dev, cyclic ? nullptr : bc_dev, n, nlines, elem_stride,
                            line_stride, cyclic, (hipStream_t)stream, ws);
}

// Host-array form for a drop-in of the reference subroutines called on host
// (Fortran) arrays: copies the lines to the device, solves, copies r back.
// Element (l, j) at l*line_stride + j*elem_stride within each host array of
// span = (nlines-1)*line_stride + (n-1)*elem_stride + 1 doubles.
extern "C" int chs_tdma_batched_host(const double* a, const double* b, const double* c, double* r,
                                     const double* bc, int n, int nlines, long long elem_stride,
                                     long long line_stride, int cyclic) {
    CHS_CHECK(a && b && c && r, CHS_E_ARG, "chs_tdma_batched_host: null array");
    CHS_CHECK(n >= 3 && nlines >= 0 && elem_stride > 0 && line_stride > 0, CHS_E_ARG,
              "chs_tdma_batched_host: need n >= 3 and positive strides");
    if (nlines == 0) return CHS_OK;
    const size_t span = (size_t)(nlines - 1) * line_stride + (size_t)(n - 1) * elem_stride + 1;
    double* d = nullptr;
    const size_t nb = bc && !cyclic ? 2 * (size_t)nlines : 0;
    CHS_HIP(hipMalloc((void**)&d, sizeof(double) * (4 * span + nb)));
    int st = CHS_OK;
    const double* src[4] = {a, b, c, r};
    for (int q = 0; q < 4 && st == CHS_OK; ++q)
        if (hipMemcpy(d + q * span, src[q], span * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) st = CHS_E_HIP;
    if (st == CHS_OK && nb && hipMemcpy(d + 4 * span, bc, nb * sizeof(double), hipMemcpyHostToDevice) != hipSuccess)
        st = CHS_E_HIP;
    if (st == CHS_OK)
        st = chs::tdma_launch(d, d + span, d + 2 * span, d + 3 * span, nb ? d + 4 * span : nullptr, n, nlines,
                              elem_stride, line_stride, cyclic, nullptr);
    if (st == CHS_OK && hipMemcpy(r, d + 3 * span, span * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess)
        st = CHS_E_HIP;
    (void)hipFree(d);
    if (st == CHS_E_HIP) chs::set_error("chs_tdma_batched_host: HIP copy or launch failed");
    return st;
}
