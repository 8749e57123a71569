// Standalone batched tridiagonal solves: the C-ABI chs_tdma_batched, which
// stands in for the reference's four line solvers
//   TDMAIJJ_nonCYC (src/TDMAIJJ_nonCYC.f90:67-123)   TDMAIJI_nonCYC (src/TDMAIJI_nonCYC.f90:67-123)
//   TDMAIJJ_CYC    (src/TDMAIJJ_CYC.f90:67-157)      TDMAIJI_CYC    (src/TDMAIJI_CYC.f90:67-157)
// on arbitrary line/element strides.
#include "chs_common.hpp"
#include "tdma_dev.hpp"

namespace chs {

// Segmented solver: LPB lines per block, P = ceil(n / MS) segments per line.
template <int MS, bool CYC>
__global__ void __launch_bounds__(1024) k_tdma_seg(const double* __restrict__ A, const double* __restrict__ B,
                                                   const double* __restrict__ Cc, double* __restrict__ Rr,
                                                   const double* __restrict__ bc, int n, int nlines,
                                                   long long es, long long ls, int LPB, int P) {
    extern __shared__ unsigned char smem[];
    const int tid = threadIdx.x;
    // consecutive lanes take consecutive lines, also where the rows are the
    // contiguous ones (measured at 65536 x 192, es = 1, with consecutive
    // segments of a line instead: 0.203 -> 0.319 ms)
    int ll = tid % LPB, seg = tid / LPB;
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
    seg_solve<MS, double>(a, b, c, d, LPB, P, ll, seg, valid, CYC, smem);
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

// ws: the sequential fallback's workspace of 3 n nlines doubles, or nullptr to
// take it from the stream-ordered pool for this launch
int tdma_launch(const double* a, const double* b, const double* c, double* r, const double* bc, int n, int nlines,
                long long es, long long ls, int cyclic, hipStream_t s, double* ws_given = nullptr) {
    // Rows per segment and lines per block, swept on an MI355X for both
    // layouts (lines x rows: best of the sweep; before: one configuration per
    // layout, 12 x 32 for lines contiguous, 8 x 16 for rows contiguous):
    //   lines contiguous   500x192 7.7 (11.4) us, 4000x192 11.0 (12.9),
    //     2000x504 16.7 (37.3), 20000x504 113 (150): 8-row segments, 16 lines
    //     (a 128-byte access) or 8 where few lines leave CUs idle; only a whole
    //     grid's lines (65536x192) keep 12 x 32: 113 against 129 us
    //   rows contiguous    500x192 7.2 (12.9), 10000x360 52.8 (75.3),
    //     20000x504 131 (214): blocks of about 128 threads, whose phases
    //     overlap; 65536x192 182 (189)
    //   cyclic             through the split-off unknown (k_tdma_cyc), whose
    //     reduced systems have no serial sweep: 500x192 8.3 (15.2), 2000x504
    //     20.0 (20.1), rows contiguous 500x192 6.9 (20.3), 20000x504 144 (287);
    //     only a whole grid's contiguous lines of whole 12-row segments stay
    //     with k_tdma_seg: 65536x192 110 against 148 us, 40000x360 at 12 x 16
    //     (two blocks per CU; 12 x 32: 170) 132 us
    const bool grid_lines = nlines >= 32768, lines_contig = ls == 1;
    int MS = 8, LPB = 0;
    const int p12 = (n + 11) / 12;   // 12 x 32: blocks whose waves fill a CU's 16 (one block of 9 would leave 7 idle)
    if (lines_contig && grid_lines && ((p12 >= 4 && p12 <= 16) || (p12 >= 28 && p12 <= 32)) &&
        (!cyclic || n % 12 == 0)) {
        MS = 12;
        LPB = cyclic && p12 > 16 ? 16 : 32;
    } else if (cyclic) {
        const int p = (n - 1 + MS - 1) / MS;
        LPB = es == 1 ? lines_per_block(p, 64, 2, 64)
                      : lines_per_block(p, p <= 4 ? 32 : nlines < 2048 ? 8 : 16, 2, 512);
        if (p * LPB <= 512) {
            const size_t sm = std::max(seg_smem_bytes<double2>(LPB, p), 2 * sizeof(double2) * (size_t)LPB);
            CHS_LAUNCH(k_tdma_cyc<8>, dim3((nlines + LPB - 1) / LPB), dim3(LPB * p), sm, s, a, b, c, r, n, nlines, es,
                       ls, LPB, p);
            return CHS_OK;
        }
        LPB = 0;
    } else if (lines_contig) {
        const int p = (n + MS - 1) / MS;
        LPB = lines_per_block(p, p <= 4 ? 32 : nlines < 2048 ? 8 : 16, 4, 1024);
    } else {
        LPB = lines_per_block((n + MS - 1) / MS, 32, 4, 128);
    }
    const int P = (n + MS - 1) / MS;
    if (LPB > 0 && P * LPB <= 1024) {
        const dim3 grid((nlines + LPB - 1) / LPB), block(LPB * P);
        const size_t sm = seg_smem_bytes<double>(LPB, P, cyclic != 0);
        if (cyclic)
            CHS_LAUNCH((k_tdma_seg<12, true>), grid, block, sm, s, a, b, c, r, bc, n, nlines, es, ls, LPB, P);
        else if (MS == 12)
            CHS_LAUNCH((k_tdma_seg<12, false>), grid, block, sm, s, a, b, c, r, bc, n, nlines, es, ls, LPB, P);
        else
            CHS_LAUNCH((k_tdma_seg<8, false>), grid, block, sm, s, a, b, c, r, bc, n, nlines, es, ls, LPB, P);
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

// chs_tdma_batched without any allocation: the segmented kernel needs only
// LDS; the sequential fallback (lines the segmented kernel cannot split) takes
// its 3 n nlines-double workspace from this GPU's static scratch array.
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
    if (!chs::tdma_seg_config(n, cyclic != 0, &MS, &P, &LPB, 1024, false)) {
        CHS_CHECK(3 * (size_t)n * (size_t)nlines <= chs::TDMA_SCRATCH_DOUBLES, CHS_E_ARG,
                  "chs_tdma_batched_noalloc: these lines need a workspace of 3*n*nlines doubles, above the "
                  "4194304 of the static scratch array (use chs_tdma_batched)");
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
