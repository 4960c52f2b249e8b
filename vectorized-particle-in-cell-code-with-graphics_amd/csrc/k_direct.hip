// k_direct.hip -- direct FP64 Poisson solve by fast sine transforms.
//
// The 5-point Laplacian with zero walls is diagonal in the type-I discrete
// sine transform: u = S^-1 (S f S / lambda) S^-1.  With n = N - 1 a power of
// two, a DST-I of a row x[1..n-1] is the complex FFT of length 2n of its odd
// extension (x[0] = x[n] = 0, x[2n-q] = -x[q]), which is purely imaginary; a
// second row rides in the imaginary part of the input and comes out in the
// real part.  Three launches: rows (k_dst_rows), columns there and back with
// the eigenvalue scale between (k_dst_cols), rows back; grids up to 65^2 in
// one workgroup (k_dst_small).  All arithmetic FP64: one solve leaves a
// residual of rounding size, where the FP32 V-cycles with FP64 refinement
// took 2 (65^2) to 5 (1025^2) cycles of 2 to 9 launches each.
//
// Methods: the Fourier solution of the 5-point problem is Hockney's (J. ACM 12,
// 1965), the sine transform through the FFT of the odd extension Cooley, Lewis
// and Welch's (J. Sound Vib. 12, 1970), the self-sorting FFT Stockham's
// (Cochran et al., Proc. IEEE 55, 1967).
//
// The FFT (fft_fwd) keeps eight points per thread in registers and exchanges
// them through LDS between radix-8 passes: thread t holds the points t + NT s,
// s = 0..7, NT = L/8, before the first pass, and the same points of the
// spectrum after the last, so the columns go from the forward to the
// backward transform without touching LDS or memory.
//
// What bounds it: latency.  The three passes move 3 x 2 x 8 N^2 bytes (50 MB
// at 1025^2, held by the last-level cache) and 4 x 5 L log2(L) flops per row
// pair; a launch's blocks all run at once up to 1025^2.
#include <cmath>
#include <vector>

#include "pic_internal.h"

namespace pic {

// --------------------------------------------------------------- the FFT

__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return {a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return {a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return {fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x)};
}
__device__ __forceinline__ double2 mul_mi(double2 a) { return {a.y, -a.x}; }  // times -i

__device__ __forceinline__ void fft2(double2 &a, double2 &b) {
    const double2 t = csub(a, b);
    a = cadd(a, b);
    b = t;
}

__device__ __forceinline__ void fft4(double2 &a, double2 &b, double2 &c, double2 &d) {
    const double2 s0 = cadd(a, c), s1 = csub(a, c), s2 = cadd(b, d), s3 = mul_mi(csub(b, d));
    a = cadd(s0, s2);
    b = cadd(s1, s3);
    c = csub(s0, s2);
    d = csub(s1, s3);
}

__device__ __forceinline__ void fft8(double2 (&v)[8]) {
    const double r = 0.70710678118654752440;
    double2 a[4], b[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        a[k] = cadd(v[k], v[k + 4]);
        b[k] = csub(v[k], v[k + 4]);
    }
    b[1] = double2{(b[1].x + b[1].y) * r, (b[1].y - b[1].x) * r};   // (1 - i) / sqrt 2
    b[2] = mul_mi(b[2]);
    b[3] = double2{(b[3].y - b[3].x) * r, -(b[3].x + b[3].y) * r};  // -(1 + i) / sqrt 2
    fft4(a[0], a[1], a[2], a[3]);
    fft4(b[0], b[1], b[2], b[3]);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        v[2 * k] = a[k];
        v[2 * k + 1] = b[k];
    }
}

// one complex of padding after every eight: the first pass's stores (stride
// 8) then fall on different banks
__device__ __forceinline__ int fpad(int i) { return i + (i >> 3); }
constexpr int fft_lds(int logl) { return (1 << logl) + (1 << (logl - 3)); }  // double2 per FFT

// thread t's twiddles, loaded beside the data (a load between two exchanges
// would put the cache's latency on the chain of every pass; with the barriers
// that fft_sync saves a 65^2 step takes 743 us for eight frames, it took 761):
// w[p-1] of the radix-8 pass p, l[m] of butterfly m of the last pass
template <int LOGL> struct Twid {
    static constexpr int A = LOGL / 3, B = LOGL % 3, M = B ? 8 >> B : 0;
    double2 w[A > 1 ? A - 1 : 1], l[M ? M : 1];
    __device__ __forceinline__ void load(int t, const double2 *__restrict__ tw) {
        constexpr int L = 1 << LOGL;
#pragma unroll
        for (int p = 1; p < A; p++) w[p - 1] = tw[(t & ((1 << (3 * p)) - 1)) * (L >> (3 * p + 3))];
#pragma unroll
        for (int m = 0; m < M; m++) l[m] = tw[t + L / 8 * m];
    }
    __device__ __forceinline__ double2 pass(int p) const { return w[p - 1]; }
    __device__ __forceinline__ double2 last(int m) const { return l[m]; }
};
// the longest transform has 1024 threads and 128 registers for each: its
// twiddles are loaded where they are used
template <> struct Twid<13> {
    const double2 *tw;
    int t;
    __device__ __forceinline__ void load(int t_, const double2 *tw_) { t = t_, tw = tw_; }
    __device__ __forceinline__ double2 pass(int p) const {
        return tw[(t & ((1 << (3 * p)) - 1)) << (10 - 3 * p)];
    }
    __device__ __forceinline__ double2 last(int m) const { return tw[t + 1024 * m]; }
};

// the threads of an FFT meet: its NT threads lie in one wavefront, whose LDS
// operations complete in order (the compiler must keep them so), or the
// workgroup waits
template <bool WAVE>
__device__ __forceinline__ void fft_sync() {
    if (WAVE) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}

// forward FFT of length L = 2^LOGL (Stockham, radix 8 with a last pass of 2
// or 4), thread t of its NT = L/8 threads; buf: fft_lds(LOGL) of LDS; tw[k] =
// exp(-2 pi i k / L).  Every thread of the workgroup calls it.  For NT up to
// 64 a wavefront holds whole FFTs and no exchange takes a barrier.
template <int LOGL>
__device__ __forceinline__ void fft_fwd(double2 (&v)[8], int t, double2 *buf,
                                        const Twid<LOGL> &tw) {
    constexpr int L = 1 << LOGL, NT = L / 8, A = LOGL / 3, B = LOGL % 3;
    constexpr bool WAVE = NT <= 64;
#pragma unroll
    for (int p = 0; p < A; p++) {
        const int ns = 1 << (3 * p), k = t & (ns - 1);
        if (p > 0) {
            const double2 w1 = tw.pass(p), w2 = cmul(w1, w1), w3 = cmul(w2, w1),
                          w4 = cmul(w2, w2);
            v[1] = cmul(v[1], w1);
            v[2] = cmul(v[2], w2);
            v[3] = cmul(v[3], w3);
            v[4] = cmul(v[4], w4);
            v[5] = cmul(v[5], cmul(w4, w1));
            v[6] = cmul(v[6], cmul(w4, w2));
            v[7] = cmul(v[7], cmul(w4, w3));
        }
        fft8(v);
        if (p == A - 1 && B == 0) break;  // natural order: t + NT s
        const int base = (t - k) * 8 + k;
        if (p > 0) fft_sync<WAVE>();  // the last exchange has been read
#pragma unroll
        for (int r = 0; r < 8; r++) buf[fpad(base + r * ns)] = v[r];
        fft_sync<WAVE>();
#pragma unroll
        for (int s = 0; s < 8; s++) v[s] = buf[fpad(t + NT * s)];
    }
    if constexpr (B > 0) {
        constexpr int R = 1 << B, M = 8 / R;
#pragma unroll
        for (int m = 0; m < M; m++) {
            const double2 w1 = tw.last(m);
            v[m + M] = cmul(v[m + M], w1);
            if constexpr (R == 4) {
                const double2 w2 = cmul(w1, w1);
                v[m + 2 * M] = cmul(v[m + 2 * M], w2);
                v[m + 3 * M] = cmul(v[m + 3 * M], cmul(w2, w1));
                fft4(v[m], v[m + M], v[m + 2 * M], v[m + 3 * M]);
            } else {
                fft2(v[m], v[m + M]);
            }
        }
    }
}

// ------------------------------------------------------- rows and columns
// T, the transform between the launches: row i, frequency or column k at
// T[(i-1) n + k-1] (n columns, the last unused: aligned pairs).

// the value at q = t + NT s of the odd extension of a pair (load(q), 0 < q < n)
template <int LOGN, class Load>
__device__ __forceinline__ void load_odd(double2 (&v)[8], int t, Load load) {
    constexpr int n = 1 << LOGN, NT = n / 4;
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const int q = t + NT * s, m = q < n ? q : 2 * n - q;
        double2 z = {0.0, 0.0};
        if (m > 0 && m < n) z = load(m);
        v[s] = s < 4 ? z : double2{-z.x, -z.y};
    }
}

// DST-I of row pairs (2p+1, 2p+2), FPB pairs per workgroup.  BACK false: rows
// of src (row stride N) to T; true: rows of T to dst (row stride N), added to
// it when add.  Each application gives 2 S x, so there and back is 2n x: the
// columns' scale carries the factor.
template <int LOGN, int FPB, bool BACK>
__global__ void __launch_bounds__(FPB * (1 << LOGN) / 4)
    k_dst_rows(const double *__restrict__ src, double *__restrict__ dst,
               const double2 *__restrict__ tw, int add) {
    constexpr int n = 1 << LOGN, N = n + 1, NT = n / 4;
    __shared__ double2 buf[FPB * fft_lds(LOGN + 1)];
    const int f = (int)threadIdx.x / NT, t = (int)threadIdx.x % NT;
    const int ra = 2 * ((int)blockIdx.x * FPB + f) + 1;
    const bool two = ra + 1 < n;
    double2 v[8];
    Twid<LOGN + 1> w;
    w.load(t, tw);
    const double *__restrict__ a = BACK ? src + (long)(ra - 1) * n - 1 : src + (long)ra * N;
    constexpr int ls = BACK ? n : N;
    load_odd<LOGN>(v, t, [&](int q) { return double2{a[q], two ? a[q + ls] : 0.0}; });
    fft_fwd<LOGN + 1>(v, t, buf + f * fft_lds(LOGN + 1), w);
    double *__restrict__ o = BACK ? dst + (long)ra * N : dst + (long)(ra - 1) * n - 1;
    constexpr int os = BACK ? N : n;
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int q = t + NT * s;
        if (q == 0) continue;
        double x = -v[s].y, y = v[s].x;
        if (BACK && add) {
            x += o[q];
            if (two) y += o[q + os];
        }
        o[q] = x;
        if (two) o[q + os] = y;
    }
}

// columns of T (pairs 2p+1, 2p+2, FPB pairs per workgroup): DST, times
// scale / (lam[k] + lam[column]), DST back, in place.  Neighbouring pairs
// share cache lines: the pair index is dealt so that an XCD's workgroups
// (blockIdx mod 8) take neighbouring pairs.
template <int LOGN, int FPB>
__global__ void __launch_bounds__(FPB * (1 << LOGN) / 4)
    k_dst_cols(double *__restrict__ T, const double2 *__restrict__ tw,
               const double *__restrict__ lam, double scale) {
    constexpr int n = 1 << LOGN, NT = n / 4, NB = n / 2 / FPB, XCD = 8;
    static_assert(NB % XCD == 0, "pairs per XCD");
    __shared__ double2 buf[FPB * fft_lds(LOGN + 1)];
    // neighbouring threads take neighbouring pairs of one row
    const int f = (int)threadIdx.x % FPB, t = (int)threadIdx.x / FPB;
    const int b = ((int)blockIdx.x % XCD) * (NB / XCD) + (int)blockIdx.x / XCD;
    const int p = b * FPB + f;
    const bool two = 2 * p + 2 < n;
    double2 v[8];
    Twid<LOGN + 1> w;
    w.load(t, tw);
    const double la = lam[2 * p + 1], lb = lam[2 * p + 2];
    double2 *__restrict__ c = reinterpret_cast<double2 *>(T) + p;
    load_odd<LOGN>(v, t, [&](int q) {
        double2 z = c[(long)(q - 1) * (n / 2)];
        if (!two) z.y = 0.0;
        return z;
    });
    double2 *bf = buf + f * fft_lds(LOGN + 1);
    fft_fwd<LOGN + 1>(v, t, bf, w);
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const int k = t + NT * s;
        const double lk = lam[k <= n ? k : 2 * n - k];
        v[s].y *= scale / (lk + la);  // the imaginary part is the first column's
        v[s].x *= scale / (lk + lb);
    }
    fft_sync<NT <= 64>();  // the forward transform's last exchange has been read
    fft_fwd<LOGN + 1>(v, t, bf, w);
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int q = t + NT * s;
        if (q > 0) c[(long)(q - 1) * (n / 2)] = double2{v[s].x, two ? v[s].y : 0.0};
    }
}

// the whole solve of a grid up to 65^2 in one workgroup: the matrix in LDS
// (row i, column j at X[i LD + j]) between the passes
template <int LOGN>
__global__ void __launch_bounds__((1 << (2 * LOGN)) / 8 < 64 ? 64 : (1 << (2 * LOGN)) / 8)
    k_dst_small(const double *__restrict__ f, double *__restrict__ u,
                const double2 *__restrict__ tw, const double *__restrict__ lam, double scale,
                int add) {
    constexpr int n = 1 << LOGN, N = n + 1, NT = n / 4, LD = n + 1, W = n / 2 * NT;
    constexpr int BLK = W < 64 ? 64 : W;
    __shared__ double X[N * LD];
    __shared__ double2 buf[n / 2 * fft_lds(LOGN + 1)];
    const int tid = (int)threadIdx.x;
    const bool on = tid < W;  // the smallest grids fill less than a wavefront
    const int p = on ? tid / NT : 0, t = on ? tid % NT : 0;
    for (int k = tid; k < N * N; k += BLK) {
        const int i = k / N, j = k - i * N;
        X[i * LD + j] = (i > 0 && j > 0 && i < n && j < n) ? f[k] : 0.0;
    }
    __syncthreads();
    double2 v[8];
    double2 *bf = buf + p * fft_lds(LOGN + 1);
    Twid<LOGN + 1> w;
    w.load(t, tw);
    const double la = lam[2 * p + 1], lb = lam[2 * p + 2];
    double lk[8];
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const int k = t + NT * s;
        lk[s] = lam[k <= n ? k : 2 * n - k];
    }
    auto rows = [&]() {  // the zero column and row n of X stay zero
        load_odd<LOGN>(v, t, [&](int q) {
            return double2{X[(2 * p + 1) * LD + q], X[(2 * p + 2) * LD + q]};
        });
        fft_fwd<LOGN + 1>(v, t, bf, w);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int q = t + NT * s;
            if (on && q > 0) {
                X[(2 * p + 1) * LD + q] = -v[s].y;
                if (2 * p + 2 < n) X[(2 * p + 2) * LD + q] = v[s].x;
            }
        }
        __syncthreads();
    };
    rows();
    load_odd<LOGN>(v, t, [&](int q) {
        return double2{X[q * LD + 2 * p + 1], X[q * LD + 2 * p + 2]};
    });
    fft_fwd<LOGN + 1>(v, t, bf, w);
#pragma unroll
    for (int s = 0; s < 8; s++) {
        v[s].y *= scale / (lk[s] + la);
        v[s].x *= scale / (lk[s] + lb);
    }
    fft_sync<true>();
    fft_fwd<LOGN + 1>(v, t, bf, w);
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int q = t + NT * s;
        if (on && q > 0) {
            X[q * LD + 2 * p + 1] = v[s].x;
            if (2 * p + 2 < n) X[q * LD + 2 * p + 2] = v[s].y;
        }
    }
    __syncthreads();
    rows();
    for (int k = tid; k < N * N; k += BLK) {
        const int i = k / N, j = k - i * N;
        if (i > 0 && j > 0 && i < n && j < n) u[k] = add ? u[k] + X[i * LD + j] : X[i * LD + j];
    }
}

// ------------------------------------------------ phi, E and the residual

// phi with its boundary values (fields.cpp:209-219), E from it when ex64 is
// given (fields.cpp:230-268: central differences inside, linear
// extrapolation at the walls, never-written entries 0), the FP64 residual of
// the solver's iterate u, and with r64 the residual itself.  The node
// expressions are those of k_phi_efield and resid_node.  phi null: residual
// only.  Each block leaves its sums of r^2 and f^2 in parts; the host adds
// them when the relative residual is asked for (published from the launch
// itself, by arrival counters and a system-scope store, it cost 10 us a step).
// One node per thread: the wall nodes' dependent loads follow the inner ones'
// in a wavefront that has both, four nodes per thread took 10.2 us instead of
// 5.1 at 257^2.
struct PhiBc4 {
    double x0, xR, y0, yL;
};
__global__ void __launch_bounds__(256)
    k_phi_resid(const double *__restrict__ u, const double *__restrict__ f, int N, PhiBc4 b,
                double twoDX, double h2i, double *__restrict__ phi, double *__restrict__ ex64,
                double *__restrict__ ey64, float2 *__restrict__ E32, double *__restrict__ r64,
                double *__restrict__ parts) {
    const unsigned tot = ex64 ? (unsigned)(N + 1) * (N + 1) : (unsigned)N * N;
    const unsigned nn = (unsigned)N * N, tot32 = (unsigned)(N + 1) * N + 1;
    auto at = [&](int j, int i) {
        double v = u[(long)j * N + i];
        if (i == 0) v = b.x0;
        if (i == N - 1) v = b.xR;
        if (j == 0) v = b.y0;
        if (j == N - 1) v = b.yL;
        return v;
    };
    auto exn = [&](int j, int i) {
        if (j < 1 || j > N - 2 || i < 1 || i > N - 2) return 0.0;
        return (at(j, i - 1) - at(j, i + 1)) / twoDX;
    };
    auto eyn = [&](int j, int i) {
        if (j < 1 || j > N - 2 || i < 1 || i > N - 2) return 0.0;
        return (at(j - 1, i) - at(j + 1, i)) / twoDX;
    };
    double rr = 0.0, ff = 0.0;
    const unsigned k = blockIdx.x * 256u + threadIdx.x;
    const int j = (int)(k / (unsigned)N), i = (int)(k - (unsigned)j * N);
    if (k >= nn && k < tot) {
        if (k < tot32) E32[k] = make_float2(0.0f, 0.0f);
        ex64[k] = 0.0;
        ey64[k] = 0.0;
    } else if (k < nn && i > 0 && j > 0 && i < N - 1 && j < N - 1) {
        const double c = u[k], n_ = u[k + N], s_ = u[k - N], e_ = u[k + 1], w_ = u[k - 1];
        const double fk = f[k];
        const double r = -h2i * (n_ + s_ + e_ + w_ - 4.0 * c) + fk;
        rr = r * r;
        ff = fk * fk;
        if (r64) r64[k] = r;
        if (phi) phi[k] = c;
        if (ex64) {
            const double pw = i == 1 ? b.x0 : w_, pe = i == N - 2 ? b.xR : e_;
            const double ps = j == 1 ? b.y0 : s_, pn = j == N - 2 ? b.yL : n_;
            const double ex = (pw - pe) / twoDX, ey = (ps - pn) / twoDX;
            ex64[k] = ex;
            ey64[k] = ey;
            E32[k] = make_float2((float)ex, (float)ey);
        }
    } else if (k < nn) {
        if (phi) phi[k] = at(j, i);
        if (ex64) {
            double ex, ey;
            if (i == 0)
                ex = 2.0 * exn(j, 1) - exn(j, 2);
            else if (i == N - 1)
                ex = 2.0 * exn(j, N - 2) - exn(j, N - 3);
            else
                ex = exn(j, i);
            if (j == 0)
                ey = 2.0 * eyn(1, i) - eyn(2, i);
            else if (j == N - 1)
                ey = 2.0 * eyn(N - 2, i) - eyn(N - 3, i);
            else
                ey = eyn(j, i);
            ex64[k] = ex;
            ey64[k] = ey;
            E32[k] = make_float2((float)ex, (float)ey);
        }
    }
    __shared__ double ws[8];
    for (int o = 32; o > 0; o >>= 1) {
        rr += __shfl_xor(rr, o, 64);
        ff += __shfl_xor(ff, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        ws[threadIdx.x >> 6] = rr;
        ws[4 + (threadIdx.x >> 6)] = ff;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const double *w = ws + 4 * threadIdx.x;
        parts[2 * blockIdx.x + threadIdx.x] = ((w[0] + w[1]) + w[2]) + w[3];
    }
}

// ------------------------------------------------------------------ driver

bool direct_ok(int N) {
    const int n = N - 1;
    return n >= 4 && n <= 4096 && (n & (n - 1)) == 0;
}

// One direct solve leaves ||f - Au|| <= C eps kappa ||f||, kappa = 4 n^2 /
// pi^2 the Laplacian's condition number (the error of u is a few eps, A
// amplifies it by at most ||A|| and ||u|| <= ||f|| / lambda_min); the largest
// measured C is 1.3 (the lowest mode alone, 5^2 to 4097^2; charge noise 0.3
// at 5^2 to 0.001 at 1025^2).  A tolerance of at least 8 eps kappa (7.5e-10 at
// 1025^2) is met by the first solve and needs no verdict.
bool direct_always_meets(int N, double tol) {
    const double n = N - 1, eps = 2.220446049250313e-16;
    return tol >= 8.0 * eps * (4.0 * n * n / (3.14159265358979323846 * 3.14159265358979323846));
}

static unsigned resid_blocks(int N) { return ((unsigned)(N + 1) * (N + 1) + 255) / 256; }

// the plan's arrays: tables (twiddles, eigenvalues), the transform, the
// residual's block sums.  alloc(p, doubles) allocates device memory.
int direct_plan(DirectPlan &D, int N, const std::function<int(double **, size_t)> &alloc) {
    const int n = N - 1, L = 2 * n;
    D.n = n;
    const double pi = 3.14159265358979323846;
    std::vector<double> t(2 * (size_t)L + n + 1);
    // one quadrant's arguments only, so the table is symmetric to the bit
    auto cosk = [&](long k) {  // cos(2 pi k / L), L a multiple of 8
        k %= L;
        if (k > L / 2) k = L - k;
        const bool neg = k > L / 4;
        if (neg) k = L / 2 - k;
        const double v = k <= L / 8 ? std::cos(2.0 * pi * k / L) : std::sin(2.0 * pi * (L / 4 - k) / L);
        return neg ? -v : v;
    };
    for (long k = 0; k < L; k++) {
        t[2 * k] = cosk(k);
        t[2 * k + 1] = -cosk(k + 3L * L / 4);  // -sin
    }
    for (int k = 0; k <= n; k++) {
        const double s = std::sin(pi * k / (2.0 * n));
        t[2 * (size_t)L + k] = 4.0 * s * s;
    }
    D.nparts = (int)resid_blocks(N);
    int rc;
    if ((rc = alloc(&D.table, t.size())) || (n > 64 && (rc = alloc(&D.T, (size_t)n * n))) ||
        (rc = alloc(&D.parts, 2 * (size_t)D.nparts)))
        return rc;
    if (hipHostMalloc((void **)&D.parts_host, 2 * sizeof(double) * D.nparts, 0) != hipSuccess ||
        hipMemcpy(D.table, t.data(), t.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess)
        return DIRECT_DEVICE;
    return 0;
}

void direct_free(DirectPlan &D) {
    void *p[] = {D.table, D.T, D.parts, D.r64};
    for (void *x : p)
        if (x) hipFree(x);
    if (D.parts_host) hipHostFree(D.parts_host);
    D = DirectPlan();
}

template <int LOGN, int FR, int FC>
static void solve_pow(hipStream_t st, const DirectPlan &D, const double *f, double *u,
                      double scale, int add) {
    constexpr int n = 1 << LOGN, NT = n / 4;
    const double2 *tw = reinterpret_cast<const double2 *>(D.table);
    const double *lam = D.table + 4 * n;
    hipLaunchKernelGGL((k_dst_rows<LOGN, FR, false>), dim3(n / 2 / FR), dim3(FR * NT), 0, st, f,
                       D.T, tw, 0);
    hipLaunchKernelGGL((k_dst_cols<LOGN, FC>), dim3(n / 2 / FC), dim3(FC * NT), 0, st, D.T, tw,
                       lam, scale);
    hipLaunchKernelGGL((k_dst_rows<LOGN, FR, true>), dim3(n / 2 / FR), dim3(FR * NT), 0, st, D.T,
                       u, tw, add);
}

template <int LOGN>
static void solve_small(hipStream_t st, const DirectPlan &D, const double *f, double *u,
                        double scale, int add) {
    constexpr int n = 1 << LOGN, W = n * n / 8;
    hipLaunchKernelGGL((k_dst_small<LOGN>), dim3(1), dim3(W < 64 ? 64 : W), 0, st, f, u,
                       reinterpret_cast<const double2 *>(D.table), D.table + 4 * n, scale, add);
}

void direct_solve(hipStream_t st, const DirectPlan &D, const double *f, double *u, double length,
                  bool add) {
    const double n = D.n, h = length / n, scale = h * h / (4.0 * n * n);
    const int a = add ? 1 : 0;
    switch (D.n) {
    case 4: solve_small<2>(st, D, f, u, scale, a); break;
    case 8: solve_small<3>(st, D, f, u, scale, a); break;
    case 16: solve_small<4>(st, D, f, u, scale, a); break;
    case 32: solve_small<5>(st, D, f, u, scale, a); break;
    case 64: solve_small<6>(st, D, f, u, scale, a); break;
    // pairs per workgroup: a wavefront at least; the columns of 1025^2 take
    // two pairs, a 32-byte sector of each row
    case 128: solve_pow<7, 2, 2>(st, D, f, u, scale, a); break;
    case 256: solve_pow<8, 1, 1>(st, D, f, u, scale, a); break;
    case 512: solve_pow<9, 1, 1>(st, D, f, u, scale, a); break;
    case 1024: solve_pow<10, 1, 2>(st, D, f, u, scale, a); break;
    case 2048: solve_pow<11, 1, 1>(st, D, f, u, scale, a); break;
    case 4096: solve_pow<12, 1, 1>(st, D, f, u, scale, a); break;
    }
}

void launch_phi_resid(hipStream_t st, const DirectPlan &D, const double *u, const double *f,
                      double phi0X, double phiR, double phi0Y, double phiLY, double length,
                      double dx, double *phi, double *ex64, double *ey64, float2 *E32,
                      double *r64) {
    const int N = D.n + 1;
    const double h = length / D.n;
    hipLaunchKernelGGL(k_phi_resid, dim3(D.nparts), dim3(256), 0, st, u, f, N,
                       PhiBc4{phi0X, phiR, phi0Y, phiLY}, 2.0 * dx, 1.0 / (h * h), phi, ex64, ey64,
                       E32, r64, D.parts);
}

int direct_relres(hipStream_t st, const DirectPlan &D, double *relres) {
    if (hipMemcpyAsync(D.parts_host, D.parts, 2 * sizeof(double) * D.nparts, hipMemcpyDeviceToHost,
                       st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
        return -1;
    double rr = 0.0, ff = 0.0;
    for (int b = 0; b < D.nparts; b++) {
        rr += D.parts_host[2 * b];
        ff += D.parts_host[2 * b + 1];
    }
    *relres = ff > 0.0 ? std::sqrt(rr / ff) : std::sqrt(rr);
    return 0;
}

}  // namespace pic
