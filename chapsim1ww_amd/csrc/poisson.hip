// Pressure Poisson solve, the MI355X form of FFT99_POIS3D_periodicxz
// (src/possion3d_FFT99.f90:254-488):
//
//   x: real FFT of every (j,k) row          k_reg_x_fwd, k_fft256_x_fwd  (2 rows per complex FFT)
//   z: complex FFT along k for every (j,kx) k_reg_z, k_fft256_z          (tile of 8 kx columns)
//   y: tridiagonal solve per (kx,kz) line   k_poisson_y   (segmented Thomas, FP64, complex RHS)
//   z, x inverse transforms                 k_reg_z, k_reg_x_inv, k_fft256_*
// (k_fft_x_fwd, k_fft_z, k_fft_x_inv: LDS Stockham, the FP32 spectra of other
// lengths than 256 and FP64 lengths without a register plan)
//
// The spectral array S is complex, layout S[(kz*M + j)*LHP + kx], so rows of
// kx are contiguous: the x transform writes whole rows, the z transform reads
// 128-byte column tiles and the y solve reads 64 consecutive kx per wave.
// The reference's two separate Re/Im line solves with the same real matrix
// (:331-443) become one solve with a complex right-hand side.  The transposes
// TRASP23_Y2Z/Z2Y (src/TRASP23.f90) disappear: on one GPU every direction is
// addressed in place.
//
// Precision: the FFT kernels are templated on the real type (FP64 for the
// plain form, FP32 for the mixed form); the y elimination is always FP64.
#include "chs_common.hpp"
#include "fft_dev.hpp"
#include "tdma_dev.hpp"

namespace chs {

constexpr int XROWS = 8;   // rows per block in the x transforms (4 complex FFTs)
constexpr int ZTX = 8;     // kx columns per block in the z transform

// ---- x forward: f rows (real, FP64 input) -> S rows (half spectrum) -------
// mode 0: input f; mode 1: input = f - L_h(phi) (FP64 residual, for refinement)
// TI: the input type (double: f; float: the refinement's FP32 residual)
template <typename Rl, typename TI = double>
__global__ void __launch_bounds__(256) k_fft_x_fwd(const TI* __restrict__ f, cpx_t<Rl>* __restrict__ S, int L,
                                                   int nrows, int LHP, FftPlan plan, const cpx_t<Rl>* __restrict__ tw) {
    using C = cpx_t<Rl>;
    extern __shared__ unsigned char smem_raw[];
    C* b0 = reinterpret_cast<C*>(smem_raw);
    C* b1 = b0 + (XROWS / 2) * L;
    const int row0 = blockIdx.x * XROWS;
    const int npair = XROWS / 2;
    for (int e = threadIdx.x; e < npair * L; e += blockDim.x) {
        const int p = e / L, i = e - p * L;
        const int ra = row0 + 2 * p, rb = ra + 1;
        const Rl va = ra < nrows ? (Rl)f[(size_t)ra * L + i] : Rl(0);
        const Rl vb = rb < nrows ? (Rl)f[(size_t)rb * L + i] : Rl(0);
        b0[p * L + i] = C{va, vb};
    }
    __syncthreads();
    C* Z = fft_lds<Rl>(b0, b1, npair, L, plan, tw, -1);
    const int LH = L / 2 + 1;
    for (int e = threadIdx.x; e < npair * LH; e += blockDim.x) {
        const int p = e / LH, kx = e - p * LH;
        const C z = Z[p * L + kx];
        const C zc = Z[p * L + (kx == 0 ? 0 : L - kx)];
        // A = (z + conj(zc))/2, B = (z - conj(zc))/(2i)
        const C A = C{Rl(0.5) * (z.x + zc.x), Rl(0.5) * (z.y - zc.y)};
        const C B = C{Rl(0.5) * (z.y + zc.y), Rl(-0.5) * (z.x - zc.x)};
        const int ra = row0 + 2 * p, rb = ra + 1;
        if (ra < nrows) S[(size_t)ra * LHP + kx] = A;
        if (rb < nrows) S[(size_t)rb * LHP + kx] = B;
    }
}

// ---- z transform, in place on S: block (j, kx tile) --------------------------
template <typename Rl>
__global__ void __launch_bounds__(256) k_fft_z(cpx_t<Rl>* __restrict__ S, int N, int M, int LH, int LHP, int dir,
                                               FftPlan plan, const cpx_t<Rl>* __restrict__ tw) {
    using C = cpx_t<Rl>;
    extern __shared__ unsigned char smem_raw[];
    C* b0 = reinterpret_cast<C*>(smem_raw);
    C* b1 = b0 + ZTX * N;
    const int j = blockIdx.y;
    const int kx0 = blockIdx.x * ZTX;
    const int tx = min(ZTX, LH - kx0);
    const size_t kst = (size_t)M * LHP;
    for (int e = threadIdx.x; e < N * ZTX; e += blockDim.x) {
        const int k = e / ZTX, c = e - k * ZTX;
        if (c < tx) b0[c * N + k] = S[(size_t)j * LHP + k * kst + kx0 + c];
    }
    __syncthreads();
    C* Z = fft_lds<Rl>(b0, b1, tx, N, plan, tw, dir);
    for (int e = threadIdx.x; e < N * ZTX; e += blockDim.x) {
        const int k = e / ZTX, c = e - k * ZTX;
        if (c < tx) S[(size_t)j * LHP + k * kst + kx0 + c] = Z[c * N + k];
    }
}

// ---------------------------------------------------------------------------
// 256-point transforms as 16 x 16 (x and z lengths of 256).  A transform is
// held by 16 threads: pass A gives each thread 16 values x[16 n1 + n2]
// (n2 = its index) in registers for a 16-point DFT over n1 (4 x 4 radix-4),
// multiplies by W256^(n2 k1) and writes to LDS transposed (row stride 17
// against bank conflicts); pass B gives thread k1 the values of its k1 for a
// 16-point DFT over n2, producing X[k1 + 16 k2].  One LDS exchange per
// transform instead of one per radix-4 stage, shifts instead of index
// divisions, and global loads/stores straight from/to registers.
// ---------------------------------------------------------------------------
constexpr int F16S = 17;            // LDS row stride of the 16 x 16 exchange
constexpr int F16T = 16 * F16S;     // LDS complex values per transform

// 16-point DFT in registers, natural order in and out; dir -1 forward, +1 inverse
template <typename C, typename Rl>
__device__ __forceinline__ void dft16(C (&v)[16], int dir) {
    // W16^m = cos(pi m/8) + dir i sin(pi m/8) for the m = n2 k1 that occur
    const Rl c8 = Rl(0.92387953251128675613), s8 = Rl(0.38268343236508977173), h2 = Rl(0.70710678118654752440);
    const Rl wc[10] = {Rl(1), c8, h2, s8, Rl(0), Rl(0), -h2, Rl(0), Rl(0), -c8};
    const Rl ws[10] = {Rl(0), s8, h2, c8, Rl(1), Rl(0), h2, Rl(0), Rl(0), -s8};
    C y[16];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {   // n = 4 n1 + n2: DFT-4 over n1
        C t[5] = {v[n2], v[4 + n2], v[8 + n2], v[12 + n2], v[0]};
        dft_small<4, C, Rl>(t, dir);
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) {
            const int m = n2 * k1;
            C z = t[k1];
            if (m != 0) {
                const C w = C{wc[m], dir > 0 ? ws[m] : -ws[m]};
                z = cmul(z, w);
            }
            y[4 * n2 + k1] = z;
        }
    }
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {   // DFT-4 over n2: X[k1 + 4 k2]
        C t[5] = {y[k1], y[4 + k1], y[8 + k1], y[12 + k1], y[0]};
        dft_small<4, C, Rl>(t, dir);
#pragma unroll
        for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = t[k2];
    }
}

// pass A tail + exchange + pass B for one transform held by 16 threads:
// v = x[16 n1 + n2] on entry (n2 = q), X[q + 16 k2] on exit.  buf: this
// transform's F16T values of LDS; all threads of the block must call it.
template <typename C, typename Rl>
__device__ __forceinline__ void fft256_regs(C (&v)[16], int q, C* buf, const C* __restrict__ tw, int dir) {
    // the twiddles W256^(n2 k1) (n2 k1 <= 225) are loaded before the first
    // 16-point DFT so their latency hides behind it (loaded where they are
    // used, each load waited on its own)
    C w[16];
#pragma unroll
    for (int k1 = 1; k1 < 16; ++k1) w[k1] = tw[q * k1];
    asm volatile("" ::: "memory");
    dft16<C, Rl>(v, dir);
#pragma unroll
    for (int k1 = 0; k1 < 16; ++k1) {
        if (k1 == 0) {
            buf[q] = v[0];
            continue;
        }
        C wk = w[k1];
        if (dir > 0) wk.y = -wk.y;
        buf[k1 * F16S + q] = cmul(v[k1], wk);
    }
    __syncthreads();
#pragma unroll
    for (int n2 = 0; n2 < 16; ++n2) v[n2] = buf[q * F16S + n2];
    dft16<C, Rl>(v, dir);
}

// x forward, L = 256: 16 rows (8 complex transforms) per block of 128 threads
template <typename Rl, typename TI = double>
__global__ void __launch_bounds__(128) k_fft256_x_fwd(const TI* __restrict__ f, cpx_t<Rl>* __restrict__ S,
                                                      int nrows, int LHP, const cpx_t<Rl>* __restrict__ tw) {
    using C = cpx_t<Rl>;
    extern __shared__ unsigned char smem_raw[];
    C* sh = reinterpret_cast<C*>(smem_raw);
    const int g = threadIdx.x >> 4, q = threadIdx.x & 15;
    const int ra = blockIdx.x * 16 + 2 * g, rb = ra + 1;
    // all 32 loads are issued before any is converted: for FP32 the compiler
    // would otherwise convert as it loads, a few loads in flight at a time
    TI la[16], lb[16];
#pragma unroll
    for (int n1 = 0; n1 < 16; ++n1) {
        const int i = 16 * n1 + q;
        la[n1] = ra < nrows ? f[(size_t)ra * 256 + i] : TI(0);
        lb[n1] = rb < nrows ? f[(size_t)rb * 256 + i] : TI(0);
    }
    asm volatile("" ::: "memory");
    C v[16];
#pragma unroll
    for (int n1 = 0; n1 < 16; ++n1) {
        asm volatile("" : "+v"(la[n1]), "+v"(lb[n1]));   // conversions stay behind every load
        v[n1] = C{(Rl)la[n1], (Rl)lb[n1]};
    }
    C* buf = sh + g * F16T;
    fft256_regs<C, Rl>(v, q, buf, tw, -1);
    __syncthreads();   // every thread has read its exchange column
    C* Z = sh + g * 256;   // the transform in natural order (fits inside the exchange space)
#pragma unroll
    for (int k2 = 0; k2 < 16; ++k2) Z[q + 16 * k2] = v[k2];
    __syncthreads();
    // split the two real rows: A = (Z_k + conj Z_{L-k}) / 2, B = (Z_k - conj Z_{L-k}) / (2i)
    for (int e = threadIdx.x; e < 8 * 129; e += blockDim.x) {
        const int p = e / 129, kx = e - p * 129;
        const C z = sh[p * 256 + kx];
        const C zc = sh[p * 256 + ((256 - kx) & 255)];
        const C A = C{Rl(0.5) * (z.x + zc.x), Rl(0.5) * (z.y - zc.y)};
        const C B = C{Rl(0.5) * (z.y + zc.y), Rl(-0.5) * (z.x - zc.x)};
        const int r0 = blockIdx.x * 16 + 2 * p;
        if (r0 < nrows) S[(size_t)r0 * LHP + kx] = A;
        if (r0 + 1 < nrows) S[(size_t)(r0 + 1) * LHP + kx] = B;
    }
}

// z transform, N = 256, in place on S: CB kx columns of one j per block of
// 16 CB threads; CB columns span 128 bytes of a row (8 FP64, 16 FP32 values)
template <typename Rl, int CB>
__global__ void __launch_bounds__(16 * CB) k_fft256_z(cpx_t<Rl>* __restrict__ S, int M, int LH, int LHP, int dir,
                                                      const cpx_t<Rl>* __restrict__ tw) {
    using C = cpx_t<Rl>;
    extern __shared__ unsigned char smem_raw[];
    C* sh = reinterpret_cast<C*>(smem_raw);
    const int c = threadIdx.x % CB, q = threadIdx.x / CB;
    const int j = blockIdx.y;
    const int kx = blockIdx.x * CB + c;
    const bool ok = kx < LH;
    const size_t kst = (size_t)M * LHP;
    C* col = S + (size_t)j * LHP + (ok ? kx : 0);
    C v[16];
#pragma unroll
    for (int n1 = 0; n1 < 16; ++n1) v[n1] = ok ? col[(size_t)(16 * n1 + q) * kst] : C{Rl(0), Rl(0)};
    fft256_regs<C, Rl>(v, q, sh + c * (F16T + 1), tw, dir);
    if (ok) {
#pragma unroll
        for (int k2 = 0; k2 < 16; ++k2) col[(size_t)(q + 16 * k2) * kst] = v[k2];
    }
}

// x inverse, L = 256: 16 rows per block of 128 threads; ghost as k_fft_x_inv,
// and three modes of the mixed form's refinement, on phf (FP32, interior rows,
// the layout of f): 3 = write phf only (the first pass's solution), 4 = dph
// = phf + the transform (the correction added to it), ghost planes as
// Neumann copies, 5 = as 4 with the ghost planes zeroed
template <typename Rl>
__global__ void __launch_bounds__(128) k_fft256_x_inv(const cpx_t<Rl>* __restrict__ S, double* __restrict__ dph,
                                                      int M, int nrows, int LHP, int ghost,
                                                      const cpx_t<Rl>* __restrict__ tw, float* __restrict__ phf) {
    using C = cpx_t<Rl>;
    extern __shared__ unsigned char smem_raw[];
    C* sh = reinterpret_cast<C*>(smem_raw);
    const int g = threadIdx.x >> 4, q = threadIdx.x & 15;
    const int ra = blockIdx.x * 16 + 2 * g, rb = ra + 1;
    C v[16];
#pragma unroll
    for (int n1 = 0; n1 < 16; ++n1) {
        const int n = 16 * n1 + q;
        const int m = n <= 128 ? n : 256 - n;
        C A = ra < nrows ? S[(size_t)ra * LHP + m] : C{Rl(0), Rl(0)};
        C B = rb < nrows ? S[(size_t)rb * LHP + m] : C{Rl(0), Rl(0)};
        if (m == 0 || m == 128) {   // b_0 = b_{L/2} = 0 (FFT99 ordering)
            A.y = Rl(0);
            B.y = Rl(0);
        }
        // Z[m] = A + iB; Z[L-m] = conj(A) + i conj(B)
        v[n1] = n <= 128 ? C{A.x - B.y, A.y + B.x} : C{A.x + B.y, B.x - A.y};
    }
    fft256_regs<C, Rl>(v, q, sh + g * F16T, tw, +1);
    const size_t plane = (size_t)256 * (M + 2);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int row = h ? rb : ra;
        if (row >= nrows) continue;
        const int jj = row % M, k = row / M;
        double* base = dph + (size_t)k * plane + q;     // column q of plane k
        double* rowp = base + (size_t)(jj + 1) * 256;
        const bool lo = jj == 0, hi = jj == M - 1;
        if (ghost == 3) {
            float* fr = phf + (size_t)row * 256 + q;
#pragma unroll
            for (int k2 = 0; k2 < 16; ++k2) fr[16 * k2] = (float)(h ? v[k2].y : v[k2].x);
            continue;
        }
        if (ghost == 4 || ghost == 5) {   // all 16 FP32 values loaded before the first store
            const float* fr = phf + (size_t)row * 256 + q;
            float old[16];
#pragma unroll
            for (int k2 = 0; k2 < 16; ++k2) old[k2] = fr[16 * k2];
#pragma unroll
            for (int k2 = 0; k2 < 16; ++k2) {
                const double val = (double)old[k2] + (h ? (double)v[k2].y : (double)v[k2].x);
                rowp[16 * k2] = val;
                // the ghost planes as Neumann copies (BC_WALL_DPH) or zero
                if (lo) base[16 * k2] = ghost == 4 ? val : 0.0;
                if (hi) base[(size_t)(M + 1) * 256 + 16 * k2] = ghost == 4 ? val : 0.0;
            }
            continue;
        }
        if (ghost == 2) {   // add to phi: all 16 old values loaded before the first add
            double old[16];
#pragma unroll
            for (int k2 = 0; k2 < 16; ++k2) old[k2] = rowp[16 * k2];
#pragma unroll
            for (int k2 = 0; k2 < 16; ++k2) rowp[16 * k2] = old[k2] + (h ? (double)v[k2].y : (double)v[k2].x);
            continue;
        }
#pragma unroll
        for (int k2 = 0; k2 < 16; ++k2) {
            const double val = h ? (double)v[k2].y : (double)v[k2].x;
            rowp[16 * k2] = val;
            if (lo) base[16 * k2] = ghost == 1 ? val : 0.0;
            if (hi) base[(size_t)(M + 1) * 256 + 16 * k2] = ghost == 1 ? val : 0.0;
        }
    }
}

// ---------------------------------------------------------------------------
// FP64 transforms of any length with a register plan (fft_dev.hpp): the x and
// z passes of k_fft_x_fwd, k_fft_z and k_fft_x_inv with the stages' radices
// chosen at run time by one switch per stage, and no integer division per
// element.  Bound: HBM, each pass reading and writing its array once.  Against
// the Stockham stages, which cross LDS once per radix up to 5 with two runtime
// divisions per butterfly: at 320x150x240 z 79.8 -> 32.5 us (5.7 TB/s), x
// 64.1 -> 41.0 and 67.1 -> 39.6 us; at 512x256x384 z 603 -> 160, x 416 -> 144
// and 420 -> 207 us; a solve 338 -> 193 us and 2186 -> 830 us.  Length 256
// keeps its own kernels: 43 + 37 (x), 37 us (z) against 41 + 42, 38 us here
// at 256x192x256.
// ---------------------------------------------------------------------------
// f(R) for the radix of a stage (uniform over the block)
template <int NST, class F>
__device__ __forceinline__ void reg_radix(int rad, F f) {
    switch (rad) {
        case 4: f(std::integral_constant<int, 4>{}); return;
        case 5: f(std::integral_constant<int, 5>{}); return;
        case 6: f(std::integral_constant<int, 6>{}); return;
        case 8: f(std::integral_constant<int, 8>{}); return;
        case 9: f(std::integral_constant<int, 9>{}); return;
        case 10: f(std::integral_constant<int, 10>{}); return;
        default: break;
    }
    if constexpr (NST == 2) {
        switch (rad) {
            case 2: f(std::integral_constant<int, 2>{}); return;
            case 3: f(std::integral_constant<int, 3>{}); return;
            case 12: f(std::integral_constant<int, 12>{}); return;
            case 15: f(std::integral_constant<int, 15>{}); return;
            case 16: f(std::integral_constant<int, 16>{}); return;
            default: break;
        }
    }
}

// A transform's elements in LDS, mul apart: after the first stage element
// q r0 + k at q sA + k, after the middle one q r0 r1 + k at q sB + k.  In x
// (mul = 1, lanes along the transform) odd strides keep the stages' stores
// off each other's banks; in z (mul = 8, lanes along kx) any stride does.
struct RegLds {
    double2* b;
    int mul, sA, sB;
    __device__ __forceinline__ double2& at(int s, int q, int k) const { return b[(q * s + k) * mul]; }
};

// v = the twiddled inputs of butterfly t (clamped) of the stage of radix R
// whose inputs are n/R = nb apart: place(r) is the LDS place of input r, step
// the twiddle exponent of r = 1.  The twiddles are loaded before the barrier
// that makes the stage before visible.
template <int R, int DIR, class P>
__device__ __forceinline__ void reg_gather(double2 (&v)[R], const double2* __restrict__ tw, int step, P place) {
    double2 w[R];
#pragma unroll
    for (int r = 1; r < R; ++r) w[r] = tw[r * step];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = place(r);
#pragma unroll
    for (int r = 1; r < R; ++r) v[r] = cmul(v[r], DIR > 0 ? cconj(w[r]) : w[r]);
    dft_reg<R, DIR>(v);
}

// The stages of one transform held by T threads (t = the thread's number; all
// threads of the block call it: barriers).  load(i) gives input element i,
// last(v, t, nb, R) takes the outputs t + r nb, r < R, of the threads with
// t < nb (the others hold a copy of the last butterfly's).
template <int NST, int DIR, class Ld, class Last>
__device__ __forceinline__ void reg_fft(const RegPlan& p, int t, const RegLds& x, const double2* __restrict__ tw,
                                        Ld load, Last last) {
    reg_radix<NST>(p.r[0], [&](auto rc) {
        constexpr int R = decltype(rc)::value;
        if (t < p.nb[0]) {
            double2 v[R];
#pragma unroll
            for (int r = 0; r < R; ++r) v[r] = load(t + r * p.nb[0]);
            dft_reg<R, DIR>(v);
#pragma unroll
            for (int r = 0; r < R; ++r) x.at(x.sA, t, r) = v[r];
        }
    });
    if constexpr (NST == 3) {
        reg_radix<NST>(p.r[1], [&](auto rc) {
            constexpr int R = decltype(rc)::value;
            const int tc = min(t, p.nb[1] - 1), q = tc / p.r[0], k = tc - q * p.r[0];
            double2 v[R];
            reg_gather<R, DIR>(v, tw, k * p.r[2], [&](int r) { return x.at(x.sA, q + r * p.r[2], k); });
            __syncthreads();   // every input of this stage has been read
            if (t < p.nb[1]) {
#pragma unroll
                for (int r = 0; r < R; ++r) x.at(x.sB, q, k + r * p.r[0]) = v[r];
            }
        });
    }
    reg_radix<NST>(p.r[NST - 1], [&](auto rc) {
        constexpr int R = decltype(rc)::value;
        const int nb = p.nb[NST - 1], tc = min(t, nb - 1);
        double2 v[R];
        reg_gather<R, DIR>(v, tw, tc, [&](int r) { return x.at(NST == 2 ? x.sA : x.sB, r, tc); });
        last(v, nb, rc);
    });
}

// z: 8 kx columns (128 bytes of a row of S) of JB rows j per block
template <int NST, int DIR>
__global__ void __launch_bounds__(NST == 2 ? 256 : 1024) k_reg_z(double2* __restrict__ S, int M, int LH, int LHP,
                                                                RegPlan p, int JB, const double2* __restrict__ tw) {
    extern __shared__ unsigned char smem_raw[];
    const int c = threadIdx.x & 7, u = threadIdx.x >> 3;
    const int jj = (int)(((float)u + 0.5f) * p.Tinv), t = u - jj * p.T;
    const int j = blockIdx.y * JB + jj, kx = blockIdx.x * 8 + c;   // kx < LHP, a multiple of 8
    const size_t kst = (size_t)M * LHP;
    double2* col = S + (size_t)min(j, M - 1) * LHP + kx;
    const bool ok = j < M && kx < LH;
    const RegLds x{reinterpret_cast<double2*>(smem_raw) + (size_t)jj * p.n * 8 + c, 8, p.r[0], p.r[0] * p.r[1]};
    reg_fft<NST, DIR>(p, t, x, tw, [&](int i) { return col[i * kst]; },
                      [&](auto& v, int nb, auto rc) {
                          if (!ok || t >= nb) return;
#pragma unroll
                          for (int r = 0; r < decltype(rc)::value; ++r) col[(size_t)(t + r * nb) * kst] = v[r];
                      });
}

// x forward: pairs of real rows, blockDim.x / T pairs per block
template <int NST>
__global__ void __launch_bounds__(256) k_reg_x_fwd(const double* __restrict__ f, double2* __restrict__ S, int nrows,
                                                   int LHP, RegPlan p, const double2* __restrict__ tw) {
    extern __shared__ unsigned char smem_raw[];
    const int T = p.T, L = p.n, PB = blockDim.x / T;
    const int pr = (int)(((float)threadIdx.x + 0.5f) * p.Tinv), t = threadIdx.x - pr * T;
    const int ra = (blockIdx.x * PB + pr) * 2;
    const double* fa = f + (size_t)min(ra, nrows - 1) * L;
    const double* fb = f + (size_t)min(ra + 1, nrows - 1) * L;
    double2* Z = reinterpret_cast<double2*>(smem_raw) + (size_t)pr * (L + T);
    const RegLds x{Z, 1, p.r[0] | 1, (p.r[0] * p.r[1]) | 1};
    reg_fft<NST, -1>(p, t, x, tw, [&](int i) { return make_double2(fa[i], fb[i]); },
                     [&](auto& v, int nb, auto rc) {
                         __syncthreads();   // every input has been read: the outputs in natural order
                         if (t < nb) {
#pragma unroll
                             for (int r = 0; r < decltype(rc)::value; ++r) Z[t + r * nb] = v[r];
                         }
                     });
    __syncthreads();
    // split the two real rows: A = (Z_k + conj Z_{L-k}) / 2, B = (Z_k - conj Z_{L-k}) / (2i)
    const int LH = L / 2 + 1;
    double2* Sa = S + (size_t)ra * LHP;
    for (int kx = t; kx < LH; kx += T) {
        const double2 z = Z[kx], zc = Z[kx == 0 ? 0 : L - kx];
        if (ra < nrows) Sa[kx] = make_double2(0.5 * (z.x + zc.x), 0.5 * (z.y - zc.y));
        if (ra + 1 < nrows) Sa[LHP + kx] = make_double2(0.5 * (z.y + zc.y), -0.5 * (z.x - zc.x));
    }
}

// x inverse: as k_fft_x_inv, ghost planes zero (ghost = 0) or Neumann copies (1)
template <int NST>
__global__ void __launch_bounds__(256) k_reg_x_inv(const double2* __restrict__ S, double* __restrict__ dph, int M,
                                                   int nrows, int LHP, int ghost, RegPlan p,
                                                   const double2* __restrict__ tw) {
    extern __shared__ unsigned char smem_raw[];
    const int T = p.T, L = p.n, PB = blockDim.x / T;
    const int pr = (int)(((float)threadIdx.x + 0.5f) * p.Tinv), t = threadIdx.x - pr * T;
    const int ra = (blockIdx.x * PB + pr) * 2;
    const double2* Sa = S + (size_t)min(ra, nrows - 1) * LHP;
    const double2* Sb = S + (size_t)min(ra + 1, nrows - 1) * LHP;
    const RegLds x{reinterpret_cast<double2*>(smem_raw) + (size_t)pr * (L + T), 1, p.r[0] | 1,
                   (p.r[0] * p.r[1]) | 1};
    const size_t plane = (size_t)L * (M + 2);
    reg_fft<NST, 1>(
        p, t, x, tw,
        [&](int n) {
            const bool up = 2 * n > L;
            const int m = up ? L - n : n;
            double2 A = Sa[m], B = Sb[m];
            if (m == 0 || 2 * m == L) A.y = B.y = 0.0;   // b_0 = b_{L/2} = 0 (FFT99 ordering)
            // Z[m] = A + iB; Z[L-m] = conj(A) + i conj(B)
            return up ? make_double2(A.x + B.y, B.x - A.y) : make_double2(A.x - B.y, A.y + B.x);
        },
        [&](auto& v, int nb, auto rc) {
            if (t >= nb) return;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int row = ra + h;
                if (row >= nrows) continue;
                const int k = row / M, j = row - k * M;
                double* base = dph + (size_t)k * plane + t;
                double* o = base + (size_t)(j + 1) * L;
#pragma unroll
                for (int r = 0; r < decltype(rc)::value; ++r) o[r * nb] = h ? v[r].y : v[r].x;
                if (j == 0) {
#pragma unroll
                    for (int r = 0; r < decltype(rc)::value; ++r) base[r * nb] = ghost == 1 ? (h ? v[r].y : v[r].x) : 0.0;
                }
                if (j == M - 1) {
                    double* g = base + (size_t)(M + 1) * L;
#pragma unroll
                    for (int r = 0; r < decltype(rc)::value; ++r) g[r * nb] = ghost == 1 ? (h ? v[r].y : v[r].x) : 0.0;
                }
            }
        });
}

// ---- y: tridiagonal solve per (kx, kz) line, FP64 --------------------------
// Matrix of TDMA_PHI_COEF (src/possion3d_FFT99.f90:185-220):
//   a_j = AMPH(j), c_j = APPH(j), b_j = ACPH(j) + (-AK1(kx)/RCCI2(j) - AK3(kz)),
// and on the (0,0) line row 1 pinned: a = c = 0, f = 0 (:206-212, :324-327, :370-372).
template <int MS, typename Rl>
__global__ void __launch_bounds__(768) k_poisson_y(cpx_t<Rl>* __restrict__ S, int M, int LH, int LHP, int nlines,
                                                    int LPB, int P, double scale, const double* __restrict__ amph,
                                                    const double* __restrict__ acph, const double* __restrict__ apph,
                                                    const double* __restrict__ ak1, const double* __restrict__ ak3) {
    extern __shared__ unsigned char smem[];
    const int tid = threadIdx.x;
    const int ll = tid % LPB, seg = tid / LPB;
    // lines run over the padded rows (LHP per kz), so that a block's LPB
    // consecutive kx start on a 128-byte line of S and no two blocks share
    // one; the padding lines (kx >= LH) solve a dummy system
    const int line = blockIdx.x * LPB + ll;
    const int kz0 = line / LHP, kx0 = line - kz0 * LHP;
    const bool valid = line < nlines && kx0 < LH;
    const int kz = valid ? kz0 : 0, kx = valid ? kx0 : 0;
    const size_t base = (size_t)kz * M * LHP + kx;
    const double lam = -ak1[kx] - ak3[kz];
    double a[MS], b[MS], c[MS];
    double2 d[MS];
    // branch-free: rows past M (and dummy lines) load row M - 1 of a valid
    // line and are replaced by identity rows, so all the segment's loads are
    // issued before the first wait (a branch per row serialised them)
    cpx_t<Rl> sv[MS];
    double av[MS], bv[MS], cv[MS];
#pragma unroll
    for (int l = 0; l < MS; ++l) {
        const int jc = min(seg * MS + l, M - 1);
        sv[l] = S[base + (size_t)jc * LHP];
        av[l] = amph[jc];
        cv[l] = apph[jc];
        bv[l] = acph[jc];
    }
#pragma unroll
    for (int l = 0; l < MS; ++l) {
        const bool ok = valid && seg * MS + l < M;
        d[l] = ok ? make_double2((double)sv[l].x * scale, (double)sv[l].y * scale) : make_double2(0.0, 0.0);
        a[l] = ok ? av[l] : 0.0;
        c[l] = ok ? cv[l] : 0.0;
        b[l] = ok ? bv[l] + lam : 1.0;
    }
    if (seg == 0) {
        a[0] = 0.0;
        if (kx == 0 && kz == 0) {
            c[0] = 0.0;
            d[0] = make_double2(0.0, 0.0);
        }
    }
    seg_solve<MS, double2>(a, b, c, d, LPB, P, ll, seg, valid, false, smem);
    if (valid) {
#pragma unroll
        for (int l = 0; l < MS; ++l) {
            const int j = seg * MS + l;
            if (j < M) S[base + (size_t)j * LHP] = cpx_t<Rl>{(Rl)d[l].x, (Rl)d[l].y};
        }
    }
}

// ---- x inverse: S rows -> DPH rows ------------------------------------------
// ghost: 0 = zero the ghost planes (reference FFT99_POIS3D), 1 = Neumann copy
// (BC_WALL_DPH), 2 = accumulate into dph (refinement: phi += delta), no ghosts.
template <typename Rl>
__global__ void __launch_bounds__(256) k_fft_x_inv(const cpx_t<Rl>* __restrict__ S, double* __restrict__ dph, int L,
                                                   int M, int nrows, int LHP, int ghost, FftPlan plan,
                                                   const cpx_t<Rl>* __restrict__ tw) {
    using C = cpx_t<Rl>;
    extern __shared__ unsigned char smem_raw[];
    C* b0 = reinterpret_cast<C*>(smem_raw);
    C* b1 = b0 + (XROWS / 2) * L;
    const int row0 = blockIdx.x * XROWS;
    const int npair = XROWS / 2;
    const int LH = L / 2 + 1;
    for (int e = threadIdx.x; e < npair * LH; e += blockDim.x) {
        const int p = e / LH, kx = e - p * LH;
        const int ra = row0 + 2 * p, rb = ra + 1;
        C A = ra < nrows ? S[(size_t)ra * LHP + kx] : C{Rl(0), Rl(0)};
        C B = rb < nrows ? S[(size_t)rb * LHP + kx] : C{Rl(0), Rl(0)};
        if (kx == 0 || 2 * kx == L) {  // b_0 = b_{L/2} = 0 (FFT99 ordering)
            A.y = Rl(0);
            B.y = Rl(0);
        }
        // Z[kx] = A + iB ; Z[L-kx] = conj(A) + i conj(B)
        b0[p * L + kx] = C{A.x - B.y, A.y + B.x};
        if (kx != 0 && 2 * kx != L) b0[p * L + (L - kx)] = C{A.x + B.y, B.x - A.y};
    }
    __syncthreads();
    C* Z = fft_lds<Rl>(b0, b1, npair, L, plan, tw, +1);
    const size_t plane = (size_t)L * (M + 2);
    for (int e = threadIdx.x; e < XROWS * L; e += blockDim.x) {
        const int r = e / L, i = e - r * L;
        const int row = row0 + r;
        if (row >= nrows) continue;
        const int p = r >> 1;
        const double v = (r & 1) ? (double)Z[p * L + i].y : (double)Z[p * L + i].x;
        const int j = row % M, k = row / M;
        double* col = dph + (size_t)k * plane + i;
        if (ghost == 2) {
            col[(size_t)(j + 1) * L] += v;
            continue;
        }
        col[(size_t)(j + 1) * L] = v;
        if (j == 0) col[0] = ghost == 1 ? v : 0.0;
        if (j == M - 1) col[(size_t)(M + 1) * L] = ghost == 1 ? v : 0.0;
    }
}

// ---- FP64 residual of the discrete operator (CHECK_FFT_SOLVER,
// src/PRESSURE_CORRECTION.f90:169-199): r = f - L_h(phi), with the Neumann
// wall rule for the y ghosts; also the block max of |r| and |f|.  Tiles of
// 64 i x 4 k x RJ rows of j; the grid (a multiple of 8 blocks) splits the
// tiles into 8 contiguous ranges, one per XCD, whose blocks walk them in j
// order so the j +- 1 rows of phi are read from that XCD's L2.  A thread takes
// RJ rows of its (i, k) column per tile, sharing the y neighbours, and issues
// the tile's loads together.  STORE = false only checks
// (no r written).  32-bit offsets (chs_create bounds the arrays below 2^31).
// NaN-propagating maximum: a NaN in phi or f makes the refinement check fail
// (and the solve report that it did not converge) instead of being skipped
__device__ __forceinline__ double pmax(double a, double b) { return a != a ? a : (b != b ? b : fmax(a, b)); }

template <bool STORE>
__global__ void __launch_bounds__(256) k_poisson_residual(const double* __restrict__ phi, const double* __restrict__ f,
                                                          float* __restrict__ r, int L, int M, int N, double dxqi,
                                                          double dzqi, const double* __restrict__ amph,
                                                          const double* __restrict__ acph,
                                                          const double* __restrict__ apph, double* __restrict__ part) {
    constexpr int RJ = 4;   // rows of j per thread and tile
    __shared__ double red[2][4];
    const int ni = (L + 63) / 64, nk = (N + 3) / 4, ng = (M + RJ - 1) / RJ;
    const int nt = ni * ng * nk, per = (nt + 7) / 8;
    const int xcd = blockIdx.x % 8, nq = gridDim.x / 8;
    const int t1 = min(nt, (xcd + 1) * per);
    const int li = threadIdx.x & 63, lk = threadIdx.x >> 6;
    const int LP = L * (M + 2);
    double mr = 0.0, mf = 0.0;
    for (int t = xcd * per + (int)blockIdx.x / 8; t < t1; t += nq) {
        const int it = t % ni, rr = t / ni;
        const int jg = rr % ng, kt = rr / ng;
        const int i0 = it * 64 + li, k0 = kt * 4 + lk;
        const bool okc = i0 < L && k0 < N;
        // cells outside the grid and rows past M evaluate a valid cell and are masked
        const int i = min(i0, L - 1), k = min(k0, N - 1);
        const int ip = i == L - 1 ? 1 - L : 1, im = i == 0 ? L - 1 : -1;
        const int kp = k == N - 1 ? (1 - N) * LP : LP, km = k == 0 ? (N - 1) * LP : -LP;
        const int j0 = jg * RJ;
        const int c0 = i + L * (j0 + 1) + LP * k;   // stored row j0 + 1 (interior row j0)
        // the column's stored rows j0 .. j0 + RJ + 1 (row M + 1 is the ghost
        // row): each cell's j - 1, j, j + 1, shared with its neighbours
        double py[RJ + 2], pe[RJ], pw[RJ], pt[RJ], pb[RJ], fv[RJ];
#pragma unroll
        for (int q = 0; q < RJ + 2; ++q) py[q] = phi[c0 + L * (min(j0 + q, M + 1) - j0 - 1)];
#pragma unroll
        for (int u = 0; u < RJ; ++u) {
            const int jc = min(j0 + u, M - 1);
            const int c = c0 + L * (jc - j0);
            pe[u] = phi[c + ip];
            pw[u] = phi[c + im];
            pt[u] = phi[c + kp];
            pb[u] = phi[c + km];
            fv[u] = f[i + L * (jc + M * k)];
        }
#pragma unroll
        for (int u = 0; u < RJ; ++u) {
            const int j = j0 + u;
            const double pc = py[u + 1];
            // the wall rule for the y ghosts
            const double pjp = j == M - 1 ? pc : py[u + 2];
            const double pjm = j == 0 ? pc : py[u];
            const int jl = min(j, M - 1);
            const double lx = (pe[u] - 2.0 * pc + pw[u]) * dxqi;
            const double ly = pjp * ldc(apph, jl) + pc * ldc(acph, jl) + pjm * ldc(amph, jl);
            const double lz = (pt[u] - 2.0 * pc + pb[u]) * dzqi;
            const double rv = fv[u] - (lx + ly + lz);
            if (okc && j < M) {
                if (STORE) r[i + L * (j + M * k)] = float(rv);   // the correction is an FP32 solve
                mr = pmax(mr, fabs(rv));
                mf = pmax(mf, fabs(fv[u]));
            }
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        mr = pmax(mr, __shfl_xor(mr, o));
        mf = pmax(mf, __shfl_xor(mf, o));
    }
    if (li == 0) {
        red[0][lk] = mr;
        red[1][lk] = mf;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = pmax(pmax(red[0][0], red[0][1]), pmax(red[0][2], red[0][3]));
        part[2 * blockIdx.x + 1] = pmax(pmax(red[1][0], red[1][1]), pmax(red[1][2], red[1][3]));
    }
}

// The residual r = f - L_h(phi) of k_poisson_residual, formed row by row and
// transformed in x at once (L = 256): the refinement pass's first step, with
// no r array written and read back.  Rows and threads as k_fft256_x_fwd: 16
// rows (row = j + M k) per block of 128 threads, thread (g, q) holding
// elements i = 16 n1 + q of rows 2g and 2g + 1.
// v of lane (q - R) mod 16 of the lane's 16-lane row (DPP row_ror:R)
template <int R>
__device__ __forceinline__ float row_rot(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + R, 0xF, 0xF, false));
}

template <typename Rl>
__global__ void __launch_bounds__(128) k_fft256_x_fwd_res(const float* __restrict__ phi,
                                                          const double* __restrict__ f, cpx_t<Rl>* __restrict__ S,
                                                          int M, int nrows, int LHP, const cpx_t<Rl>* __restrict__ tw,
                                                          double dxqi, double dzqi, const double* __restrict__ amph,
                                                          const double* __restrict__ acph,
                                                          const double* __restrict__ apph) {
    using C = cpx_t<Rl>;
    extern __shared__ unsigned char smem_raw[];
    C* sh = reinterpret_cast<C*>(smem_raw);
    const int g = threadIdx.x >> 4, q = threadIdx.x & 15;
    const int N = nrows / M;
    const int LP = 256 * M;   // phi: interior rows only, the layout of f
    // XCD-aware order of the 16-row tiles (a grid of whole groups of 8
    // blocks): each XCD transforms a contiguous range of rows, so the k +- 1
    // rows of phi a tile reads (M rows away) were read by its XCD's L2
    const int tb = xcd_tile(blockIdx.x, gridDim.x);
    if (tb * 16 >= nrows) return;
    // per row: centre offset, y and z neighbour offsets (the wall rule as
    // k_poisson_residual: the y neighbour of a wall row is the row itself)
    int cc[2], jp[2], jm[2], kp[2], km[2];
    double ap[2], ac[2], am[2];
    bool ok[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int r = tb * 16 + 2 * g + s;
        ok[s] = r < nrows;
        const int rr = ok[s] ? r : nrows - 1;
        const int j = rr % M, k = rr / M;
        cc[s] = 256 * rr;
        jp[s] = j == M - 1 ? 0 : 256;
        jm[s] = j == 0 ? 0 : -256;
        kp[s] = k == N - 1 ? (1 - N) * LP : LP;
        km[s] = k == 0 ? (N - 1) * LP : -LP;
        ap[s] = ldc(apph, j);
        ac[s] = ldc(acph, j);
        am[s] = ldc(amph, j);
    }
    // rows 2g and 2g + 1 in one plane (always when M is even): each is the
    // other's y neighbour
    const bool pair = ok[1] && jp[0] != 0;
    // the centre values of both rows, a window of two n1 at a time; the x
    // neighbours come from the other lanes of the 16-lane row by DPP
    // rotations (lane q holds i = 16 n1 + q: i - 1 is lane q - 1, or lane 15
    // at n1 - 1 for q = 0; i + 1 is lane q + 1, or lane 0 at n1 + 1 for q = 15)
    float cn[2], dprev[2], u0[2], ucur[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        cn[s] = phi[cc[s] + q];
        dprev[s] = row_rot<1>(phi[cc[s] + 240 + q]);
        u0[s] = row_rot<15>(cn[s]);
        ucur[s] = u0[s];
    }
    C v[16];
#pragma unroll
    for (int n1 = 0; n1 < 16; ++n1) {
        const int i = 16 * n1 + q;
        float nx[2];
        double rv[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) nx[s] = n1 < 15 ? phi[cc[s] + i + 16] : 0.0f;
        const float pn0 = pair ? cn[1] : phi[cc[0] + jp[0] + i];
        const float ps1 = pair ? cn[0] : phi[cc[1] + jm[1] + i];
        const float ps0 = phi[cc[0] + jm[0] + i];
        const float pn1 = phi[cc[1] + jp[1] + i];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const double pc = cn[s];
            const float dcur = row_rot<1>(cn[s]);
            const double pw = q == 0 ? dprev[s] : dcur;
            dprev[s] = dcur;
            const float unext = n1 < 15 ? row_rot<15>(nx[s]) : u0[s];
            const double pe = q == 15 ? unext : ucur[s];
            ucur[s] = unext;
            const double pjp = s == 0 ? pn0 : pn1, pjm = s == 0 ? ps0 : ps1;
            const double lx = (pe - 2.0 * pc + pw) * dxqi;
            const double ly = pjp * ap[s] + pc * ac[s] + pjm * am[s];
            const double lz = ((double)phi[cc[s] + kp[s] + i] - 2.0 * pc + (double)phi[cc[s] + km[s] + i]) * dzqi;
            rv[s] = ok[s] ? f[cc[s] + i] - (lx + ly + lz) : 0.0;
        }
        cn[0] = nx[0];
        cn[1] = nx[1];
        v[n1] = C{(Rl)rv[0], (Rl)rv[1]};
    }
    C* buf = sh + g * F16T;
    fft256_regs<C, Rl>(v, q, buf, tw, -1);
    __syncthreads();   // every thread has read its exchange column
    C* Z = sh + g * 256;
#pragma unroll
    for (int k2 = 0; k2 < 16; ++k2) Z[q + 16 * k2] = v[k2];
    __syncthreads();
    for (int e = threadIdx.x; e < 8 * 129; e += blockDim.x) {
        const int p = e / 129, kx = e - p * 129;
        const C z = sh[p * 256 + kx];
        const C zc = sh[p * 256 + ((256 - kx) & 255)];
        const C A = C{Rl(0.5) * (z.x + zc.x), Rl(0.5) * (z.y - zc.y)};
        const C B = C{Rl(0.5) * (z.y + zc.y), Rl(-0.5) * (z.x - zc.x)};
        const int r0 = tb * 16 + 2 * p;
        if (r0 < nrows) S[(size_t)r0 * LHP + kx] = A;
        if (r0 + 1 < nrows) S[(size_t)(r0 + 1) * LHP + kx] = B;
    }
}

// Max over the block partials written by k_poisson_residual -> out[0..1]
__global__ void k_reduce_max2(const double* __restrict__ part, int nb, double* __restrict__ out) {
    __shared__ double red[2][256];
    double a = 0.0, b = 0.0;
    for (int i = threadIdx.x; i < nb; i += blockDim.x) {
        a = pmax(a, part[2 * i]);
        b = pmax(b, part[2 * i + 1]);
    }
    red[0][threadIdx.x] = a;
    red[1][threadIdx.x] = b;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            red[0][threadIdx.x] = pmax(red[0][threadIdx.x], red[0][threadIdx.x + s]);
            red[1][threadIdx.x] = pmax(red[1][threadIdx.x], red[1][threadIdx.x + s]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = red[0][0];
        out[1] = red[1][0];
    }
}

__global__ void k_zero(double* __restrict__ p, size_t n) {
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x)
        p[t] = 0.0;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
bool tdma_seg_config(int n, bool cyclic, int* MS, int* P, int* LPB, int maxthr, bool lpb_small = false);

// rows j per block of k_reg_z: 8 T threads a row, 72 to 128 a block for the
// two-stage lengths (T up to 16), one row of up to 1024 for the others
inline int reg_z_rows(const RegPlan& p) { return std::max(1, 16 / p.T); }

// LDS bytes of a block of the z transforms of h (NCL3 = 256 and lengths with a
// register plan need less than the Stockham stages' two buffers).
size_t poisson_z_lds(const chs_handle* h) {
    const bool f64 = h->precision == CHS_FP64;
    RegPlan rz;
    if (h->N == 256) return sizeof(double2) * (size_t)8 * (F16T + 1);
    if (f64 && reg_plan(h->N, false, &rz)) return sizeof(double2) * (size_t)8 * reg_z_rows(rz) * h->N;
    return (f64 ? sizeof(double2) : sizeof(float2)) * (size_t)2 * ZTX * h->N;
}

template <typename Rl, typename TI = double>
static int poisson_pass(chs_handle* h, const TI* f, double* dph, int ghost, cpx_t<Rl>* S, const cpx_t<Rl>* twx,
                        const cpx_t<Rl>* twz, const float* rphi = nullptr, float* phf = nullptr) {
    // L = 256 only: rphi transforms the residual f - L_h(rphi) instead of f
    // (rphi: FP32 values of the interior rows); phf is the FP32 solution of
    // ghost modes 3, 4 and 5 (k_fft256_x_inv)
    // FP32 spectra use rows of a multiple of 16 values (128-byte aligned rows)
    constexpr bool f32 = sizeof(Rl) == 4;
    constexpr int ZCB = f32 ? 16 : 8;   // kx columns per z block: 128 bytes
    const int L = h->L, M = h->M, N = h->N, LH = h->LH, LHP = f32 ? h->LHP32 : h->LHP;
    const hipStream_t s = h->stream;
    FftPlan px, pz;
    fft_plan(L, &px);
    fft_plan(N, &pz);
    const int nrows = M * N;
    const dim3 gx((nrows + XROWS - 1) / XROWS);
    const size_t smx = sizeof(cpx_t<Rl>) * (size_t)XROWS * L;  // two buffers of XROWS/2 vectors
    hipEvent_t ev;
    // 256-point lengths use the 16 x 16 register transforms
    const bool x256 = L == 256, z256 = N == 256;
    const dim3 gx16((nrows + 15) / 16);
    const size_t sm16x = sizeof(cpx_t<Rl>) * (size_t)8 * F16T;
    const size_t sm16z = sizeof(cpx_t<Rl>) * (size_t)ZCB * (F16T + 1);
    const dim3 gz16((LH + ZCB - 1) / ZCB, M);
    if ((rphi != nullptr || ghost >= 3) && !x256) {
        set_error("poisson: the fused residual transform needs NCL1 = 256");
        return CHS_E_ARG;
    }
    // FP64, other lengths: register transforms where the length has a plan
    // (FP32 spectra still run the Stockham stages there)
    RegPlan rx, rxi, rz;
    const bool xr = !f32 && !x256 && reg_plan(L, true, &rx) && reg_plan(L, false, &rxi);
    const bool zr = !f32 && !z256 && reg_plan(N, false, &rz);
    const int pb = xr ? std::max(1, (rx.nst == 2 ? 128 : 256) / rx.T) : 1;   // row pairs per block
    const dim3 gxr((nrows + 2 * pb - 1) / (2 * pb)), bxr(pb * (xr ? rx.T : 1));
    const size_t smxr = xr ? sizeof(double2) * (size_t)pb * (L + rx.T) : 0;
    const int jb = zr ? reg_z_rows(rz) : 1;
    const dim3 gzr(LHP / 8, (M + jb - 1) / jb), bzr(8 * jb * (zr ? rz.T : 1));
    const size_t smzr = zr ? sizeof(double2) * (size_t)8 * jb * N : 0;
    auto fft_z_reg = [&](int dir) -> int {
        if constexpr (!f32) {
            if (rz.nst == 2 && dir < 0)
                CHS_LAUNCH((k_reg_z<2, -1>), gzr, bzr, smzr, s, S, M, LH, LHP, rz, jb, twz);
            else if (rz.nst == 2)
                CHS_LAUNCH((k_reg_z<2, 1>), gzr, bzr, smzr, s, S, M, LH, LHP, rz, jb, twz);
            else if (dir < 0)
                CHS_LAUNCH((k_reg_z<3, -1>), gzr, bzr, smzr, s, S, M, LH, LHP, rz, jb, twz);
            else
                CHS_LAUNCH((k_reg_z<3, 1>), gzr, bzr, smzr, s, S, M, LH, LHP, rz, jb, twz);
        }
        return CHS_OK;
    };
    auto fft_x_reg = [&](int dir) -> int {
        if constexpr (!f32) {
            if (rx.nst == 2 && dir < 0)
                CHS_LAUNCH((k_reg_x_fwd<2>), gxr, bxr, smxr, s, f, S, nrows, LHP, rx, twx);
            else if (dir < 0)
                CHS_LAUNCH((k_reg_x_fwd<3>), gxr, bxr, smxr, s, f, S, nrows, LHP, rx, twx);
            else if (rx.nst == 2)
                CHS_LAUNCH((k_reg_x_inv<2>), gxr, bxr, smxr, s, S, dph, M, nrows, LHP, ghost, rxi, twx);
            else
                CHS_LAUNCH((k_reg_x_inv<3>), gxr, bxr, smxr, s, S, dph, M, nrows, LHP, ghost, rxi, twx);
        }
        return CHS_OK;
    };
    h->timer.begin(rphi ? "resid_fft_x" : "fft_x_fwd", s, &ev);
    if (xr)
        CHS_TRY(fft_x_reg(-1));
    else if (rphi != nullptr)
        CHS_LAUNCH((k_fft256_x_fwd_res<Rl>), dim3(8 * ((gx16.x + 7) / 8)), dim3(128), sm16x, s, rphi, (const double*)f, S, M, nrows, LHP,
                   twx, h->dxqi, h->dzqi, h->amph, h->acph, h->apph);
    else if (x256)
        CHS_LAUNCH((k_fft256_x_fwd<Rl, TI>), gx16, dim3(128), sm16x, s, f, S, nrows, LHP, twx);
    else
        CHS_LAUNCH((k_fft_x_fwd<Rl, TI>), gx, dim3(256), smx, s, f, S, L, nrows, LHP, px, twx);
    h->timer.end(ev, rphi ? "resid_fft_x" : "fft_x_fwd", s);
    const dim3 gz((LH + ZTX - 1) / ZTX, M);
    const size_t smz = sizeof(cpx_t<Rl>) * (size_t)2 * ZTX * N;
    h->timer.begin("fft_z", s, &ev);
    if (zr)
        CHS_TRY(fft_z_reg(-1));
    else if (z256)
        CHS_LAUNCH((k_fft256_z<Rl, ZCB>), gz16, dim3(16 * ZCB), sm16z, s, S, M, LH, LHP, -1, twz);
    else
        CHS_LAUNCH(k_fft_z<Rl>, gz, dim3(256), smz, s, S, N, M, LH, LHP, -1, pz, twz);
    h->timer.end(ev, "fft_z", s);
    // FP32 spectra: segments of 12 rows and 16 lines per block (measured
    // fastest at NCL2 = 192: 16-row segments spill registers, 8-row segments
    // double the reduced system; 8 lines of 16-row segments above NCL2 = 576).
    // FP64: the segmentation of the batched TDMA with 8 lines per block, whose
    // roundings the FP64 parity tests pin.
    int MS = 0, P = 0, LPB = 0;
    if (f32) {
        const int cfg[4][2] = {{12, 16}, {8, 16}, {16, 8}, {16, 4}};
        for (const auto& c : cfg) {
            if ((M + c[0] - 1) / c[0] * c[1] <= 768) {
                MS = c[0];
                P = (M + c[0] - 1) / c[0];
                LPB = c[1];
                break;
            }
        }
    } else if (!tdma_seg_config(M, false, &MS, &P, &LPB, 768, true)) {
        MS = 0;
    }
    if (MS == 0) {
        set_error("poisson: unsupported NCL2");
        return CHS_E_ARG;
    }
    const int nlines = LHP * N;  // padded rows: see k_poisson_y
    const dim3 gy((nlines + LPB - 1) / LPB), by(LPB * P);
    const size_t smy = seg_smem_bytes<double2>(LPB, P);
    const double scale = 1.0 / ((double)L * (double)N);
    h->timer.begin("poisson_y", s, &ev);
    switch (MS) {
        case 16: CHS_LAUNCH((k_poisson_y<16, Rl>), gy, by, smy, s, S, M, LH, LHP, nlines, LPB, P, scale, h->amph, h->acph, h->apph, h->ak1, h->ak3); break;
        case 12: CHS_LAUNCH((k_poisson_y<12, Rl>), gy, by, smy, s, S, M, LH, LHP, nlines, LPB, P, scale, h->amph, h->acph, h->apph, h->ak1, h->ak3); break;
        case 4: CHS_LAUNCH((k_poisson_y<4, Rl>), gy, by, smy, s, S, M, LH, LHP, nlines, LPB, P, scale, h->amph, h->acph, h->apph, h->ak1, h->ak3); break;
        default: CHS_LAUNCH((k_poisson_y<8, Rl>), gy, by, smy, s, S, M, LH, LHP, nlines, LPB, P, scale, h->amph, h->acph, h->apph, h->ak1, h->ak3); break;
    }
    h->timer.end(ev, "poisson_y", s);
    h->timer.begin("fft_z", s, &ev);
    if (zr)
        CHS_TRY(fft_z_reg(1));
    else if (z256)
        CHS_LAUNCH((k_fft256_z<Rl, ZCB>), gz16, dim3(16 * ZCB), sm16z, s, S, M, LH, LHP, +1, twz);
    else
        CHS_LAUNCH(k_fft_z<Rl>, gz, dim3(256), smz, s, S, N, M, LH, LHP, +1, pz, twz);
    h->timer.end(ev, "fft_z", s);
    h->timer.begin("fft_x_inv", s, &ev);
    if (xr)
        CHS_TRY(fft_x_reg(1));
    else if (x256)
        CHS_LAUNCH(k_fft256_x_inv<Rl>, gx16, dim3(128), sm16x, s, S, dph, M, nrows, LHP, ghost, twx, phf);
    else
        CHS_LAUNCH(k_fft_x_inv<Rl>, gx, dim3(256), smx, s, S, dph, L, M, nrows, LHP, ghost, px, twx);
    h->timer.end(ev, "fft_x_inv", s);
    return CHS_OK;
}

// Ghost planes of DPH after a refinement (mode 0: zero, 1: Neumann copy).
__global__ void k_dph_ghost(double* __restrict__ dph, int L, int M, int N, int mode) {
    const size_t plane = (size_t)L * (M + 2);
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < (size_t)L * N; t += (size_t)gridDim.x * blockDim.x) {
        const int i = t % L, k = t / L;
        double* col = dph + (size_t)k * plane + i;
        col[0] = mode == 1 ? col[L] : 0.0;
        col[(size_t)(M + 1) * L] = mode == 1 ? col[(size_t)M * L] : 0.0;
    }
}

// Mixed form inside the substep: the FP32 pass and one refinement, with no
// check here and no wait; the substep's projection checks the residual of the
// result (k_update<true>) and the host reads the verdict later.
int poisson_solve_unchecked(chs_handle* h, const double* f, double* dph, int ghost) {
    const hipStream_t s = h->stream;
    float* rf = reinterpret_cast<float*>(h->resid);   // the FP32 residual (first half of the buffer)
    if (h->L == 256 && ghost == 1) {
        // the first pass's solution phi1 kept in FP32 (interior rows, in the
        // residual buffer); the residual f - L_h(phi1) formed in FP64 inside
        // the refinement pass's x transform; DPH = phi1 + the correction
        CHS_TRY(poisson_pass<float>(h, f, dph, 3, h->spec32, h->twx32, h->twz32, nullptr, rf));
        CHS_TRY((poisson_pass<float, double>(h, f, dph, 4, h->spec32, h->twx32, h->twz32, rf, rf)));
    } else {
        CHS_TRY(poisson_pass<float>(h, f, dph, ghost, h->spec32, h->twx32, h->twz32));
        hipEvent_t ev;
        h->timer.begin("poisson_residual", s, &ev);
        CHS_LAUNCH(k_poisson_residual<true>, dim3(2048), dim3(256), 0, s, dph, f, rf, h->L, h->M, h->N, h->dxqi,
                   h->dzqi, h->amph, h->acph, h->apph, h->partials);
        h->timer.end(ev, "poisson_residual", s);
        CHS_TRY(poisson_pass<float>(h, rf, dph, 2, h->spec32, h->twx32, h->twz32));
        if (ghost != 2) CHS_LAUNCH(k_dph_ghost, dim3(256), dim3(256), 0, s, dph, h->L, h->M, h->N, ghost);
    }
    h->last_refine_iters = 1;
    h->last_refine_resid = -1.0;   // known once the substep's check has been read
    return CHS_OK;
}

// FP64 form: one pass.  Mixed form: FP32 pass on f, then FP32 passes on the
// FP64 residual (at least one) until max|f - L phi| <= abs_tol or
// max|f - L phi| <= rel_tol * max|f|.
int poisson_solve(chs_handle* h, const double* f, double* dph, int ghost, double abs_tol) {
    if (h->precision == CHS_FP64) return poisson_pass<double>(h, f, dph, ghost, h->spec, h->twx, h->twz);
    const hipStream_t s = h->stream;
    float* rf = reinterpret_cast<float*>(h->resid);   // the FP32 residual (first half of the buffer)
    // NCL1 = 256 and a first refinement allowed: the pair of the substep (the
    // FP32 pass keeping phi1 in FP32, the refinement forming the residual
    // inside its x transform), then the checks below
    const bool fused = h->refine_max > 0 && h->L == 256 && (ghost == 0 || ghost == 1);
    if (fused) {
        CHS_TRY(poisson_pass<float>(h, f, dph, 3, h->spec32, h->twx32, h->twz32, nullptr, rf));
        CHS_TRY((poisson_pass<float, double>(h, f, dph, ghost == 1 ? 4 : 5, h->spec32, h->twx32, h->twz32, rf, rf)));
    } else {
        CHS_TRY(poisson_pass<float>(h, f, dph, ghost, h->spec32, h->twx32, h->twz32));
    }
    // 2048 blocks of row tiles (a multiple of 8: one contiguous tile range per XCD)
    const int nb = 2048;
    hipEvent_t ev;
    h->last_refine_iters = 0;
    h->last_refine_resid = -1.0;
    double host[2] = {0.0, 0.0};
    bool stored = false;   // h->resid holds the residual of the current dph
    auto residual = [&](bool store) -> int {
        h->timer.begin("poisson_residual", s, &ev);
        if (store)
            CHS_LAUNCH(k_poisson_residual<true>, dim3(nb), dim3(256), 0, s, dph, f, rf, h->L, h->M, h->N,
                       h->dxqi, h->dzqi, h->amph, h->acph, h->apph, h->partials);
        else
            CHS_LAUNCH(k_poisson_residual<false>, dim3(nb), dim3(256), 0, s, dph, f, rf, h->L, h->M, h->N,
                       h->dxqi, h->dzqi, h->amph, h->acph, h->apph, h->partials);
        h->timer.end(ev, "poisson_residual", s);
        stored = store;
        return CHS_OK;
    };
    // One refinement always (when any is allowed): an FP32 pass leaves a
    // relative residual near 1e-7, far above the tolerances this form serves,
    // so checking it first would only cost a round trip to the host.  Then
    // check-only residuals (r is formed again in the rare case that one more
    // refinement is needed) until the tolerance holds.
    int it0 = 0;
    if (fused) {
        h->last_refine_iters = 1;
        it0 = 1;
    } else if (h->refine_max > 0) {
        CHS_TRY(residual(true));
        CHS_TRY(poisson_pass<float>(h, rf, dph, 2, h->spec32, h->twx32, h->twz32));
        h->last_refine_iters = 1;
        it0 = 1;
    }
    for (int it = it0; it <= h->refine_max; ++it) {
        CHS_TRY(residual(false));
        CHS_LAUNCH(k_reduce_max2, dim3(1), dim3(256), 0, s, h->partials, nb, h->scalars + 4);
        CHS_HIP(hipMemcpyAsync(host, h->scalars + 4, 2 * sizeof(double), hipMemcpyDeviceToHost, s));
        CHS_HIP(hipStreamSynchronize(s));
        if (host[0] != host[0] || host[1] != host[1]) {
            h->last_refine_resid = host[0] + host[1];
            set_error("poisson: NaN in the mixed-precision residual (phi or the right-hand side)");
            return CHS_E_NOTCONV;
        }
        const double rel = host[1] > 0.0 ? host[0] / host[1] : 0.0;
        h->last_refine_resid = rel;
        if (host[0] <= abs_tol || rel <= h->refine_tol) break;
        if (it == h->refine_max) {
            set_error("poisson: mixed-precision refinement did not reach its tolerance");
            return CHS_E_NOTCONV;
        }
        if (!stored) CHS_TRY(residual(true));
        CHS_TRY(poisson_pass<float>(h, rf, dph, 2, h->spec32, h->twx32, h->twz32));
        h->last_refine_iters = it + 1;
    }
    // ghost planes after the accumulating refinements (the fused pair writes its own)
    if (h->last_refine_iters > (fused ? 1 : 0) && ghost != 2)
        CHS_LAUNCH(k_dph_ghost, dim3(256), dim3(256), 0, s, dph, h->L, h->M, h->N, ghost);
    return CHS_OK;
}

}  // namespace chs
