// k_fmg.hip -- the reference's FP64 full multigrid (Mglin, mglin.cpp:21-196):
// ncycle V(1,1) cycles per level, red-black Gauss-Seidel, half-weighting
// restriction, bilinear prolongation.  Every per-node expression keeps the
// reference's association and every sweep its colour order, so the result is
// Mglin's bit for bit, whatever is fused.
//
// Levels up to 65^2 are visited inside one workgroup (k_fmg_coarse); above,
// one launch takes a leg of a V-cycle (k_fmg_leg): the smoothing before the
// coarse correction with the restricted residual, the prolongation-add with
// the smoothing after it, or both where one cycle follows another.
#include <vector>

#include "pic_internal.h"

namespace pic {

static __host__ __device__ inline int lvl_size(int l) { return (1 << (l + 1)) + 1; }

// ------------------------------------------------------------ node rules

__device__ __forceinline__ double rstrct_node(const double *uf, int nc, int ic, int jc) {
    const int nf = 2 * nc - 1, ncc = 2 * nc - 2;
    if (jc == 0) return uf[(2 * ic) * nf + 0];
    if (jc == nc - 1 && ic != 0 && ic != nc - 1) return uf[(2 * ic) * nf + ncc];
    if (ic == 0) return uf[0 * nf + 2 * jc];
    if (ic == nc - 1) return uf[ncc * nf + 2 * jc];
    const int i = 2 * ic, j = 2 * jc;
    return 0.5 * uf[i * nf + j] + 0.125 * (uf[(i + 1) * nf + j] + uf[(i - 1) * nf + j] +
                                           uf[i * nf + j + 1] + uf[i * nf + j - 1]);
}

// bilinear prolongation value at fine (i,j) (mglin.cpp:70-82)
__device__ __forceinline__ double interp_even_col(const double *uc, int nc, int i, int j) {
    if ((i & 1) == 0) return uc[(i >> 1) * nc + (j >> 1)];
    return 0.5 * (uc[((i + 1) >> 1) * nc + (j >> 1)] + uc[((i - 1) >> 1) * nc + (j >> 1)]);
}
__device__ __forceinline__ double interp_node(const double *uc, int nc, int i, int j) {
    if ((j & 1) == 0) return interp_even_col(uc, nc, i, j);
    return 0.5 * (interp_even_col(uc, nc, i, j + 1) + interp_even_col(uc, nc, i, j - 1));
}

// the right-hand side restricted to the next coarser grid
__global__ void __launch_bounds__(128)
    k_fmg_rstrct(double *__restrict__ uc, int nc, const double *__restrict__ uf) {
    const int jc = blockIdx.x * blockDim.x + threadIdx.x, ic = blockIdx.y;
    if (jc < nc) uc[ic * nc + jc] = rstrct_node(uf, nc, ic, jc);
}

// ------------------------------------------- levels up to 65^2, one workgroup
// A level l has n = 2^(l+1) intervals; thread (b, c) of its 2^l x 2^l owns the
// block of nodes A = (2b, 2c), B = (2b, 2c+1), C = (2b+1, 2c), D = (2b+1,
// 2c+1): A and D are red, B and C black, so a sweep updates two nodes of every
// thread and reads two neighbours of each from LDS (the other two are the
// thread's own).  Each kind of node has a plane of its own ((2^l + 1)^2, the
// wall row and column zero): consecutive threads read consecutive doubles.
// The black nodes' residuals need only values the black sweep has read, so a
// leg before the coarse correction takes three barriers, one after it three.
// Levels up to 17^2 (64 threads) are visited by the first wavefront alone,
// without barriers.
//
// What bounds it: latency, a serial chain of about 6 dependent LDS round trips
// per level visit.  Before this form (one node per thread and sweep, index
// divisions, all five operands from LDS) a V-cycle from 65^2 took 45 us and
// the full multigrid 170 us.
#define FMG_TOP 5

struct CoarseMem {
    double planes[4 * (33 * 33 + 17 * 17 + 9 * 9 + 5 * 5 + 3 * 3) + 40];
    double res[2 * 33 * 33 + 40];             // black residuals of the visited level
    double cres[33 * 33 + 17 * 17 + 9 * 9 + 5 * 5 + 3 * 3];  // V-cycle rhs, levels 0..4
    double sol[33 * 33 + 17 * 17 + 9 * 9 + 5 * 5 + 3 * 3];   // solutions, levels 0..4
    double rhs[65 * 65 + 33 * 33 + 17 * 17 + 9 * 9 + 5 * 5 + 3 * 3];  // levels 0..5
    double h2[FMG_TOP + 1], h2i[FMG_TOP + 1];
};

// sum of (2^k + 1)^2 for k = 1 .. l-1, the start of level l's plane quartet / 4
__device__ __forceinline__ int plane_start(int l) {
    return ((1 << (2 * l)) - 4) / 3 + 2 * ((1 << l) - 2) + (l - 1);
}
// sum of lvl_size(k)^2 for k < l
__device__ __forceinline__ int flat_start(int l) { return plane_start(l + 1); }

template <bool WAVE>
__device__ __forceinline__ void level_sync() {
    if (WAVE) {
        // one wavefront: its LDS operations complete in order, the compiler
        // must keep them so
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}

// thread's place on a level
struct Blk {
    int nb, ld, k;   // blocks per side, plane row, own plane index
    bool on, ia, ib, ic;  // owns a block; A, B, C are inside (D always is)
    double *pA, *pB, *pC, *pD;
};
__device__ __forceinline__ Blk blk_of(CoarseMem &m, int l) {
    Blk q;
    q.nb = 1 << l;
    q.ld = q.nb + 1;
    const int t = (int)threadIdx.x, b = t >> l, c = t & (q.nb - 1);
    q.on = b < q.nb;
    q.k = q.on ? b * q.ld + c : 0;
    q.ia = q.on && b > 0 && c > 0;
    q.ib = q.on && b > 0;
    q.ic = q.on && c > 0;
    // 34 doubles ahead: index -1 and -ld of a wall block are never used but
    // stay inside the array
    q.pA = m.planes + 34 + 4 * plane_start(l);
    const int s = q.ld * q.ld;
    q.pB = q.pA + s;
    q.pC = q.pB + s;
    q.pD = q.pC + s;
    return q;
}

// own four nodes of a row-major array of level l
__device__ __forceinline__ void own4(const double *f, int l, double &a, double &b, double &c,
                                     double &d) {
    const int n = lvl_size(l), t = (int)threadIdx.x, nb = 1 << l;
    const double *p = f + (2 * (t >> l)) * n + 2 * (t & (nb - 1));
    a = p[0];
    b = p[1];
    c = p[n];
    d = p[n + 1];
}

// smoothing of level l on f (zero: from a zero iterate, else from the planes),
// the residual restricted into cres of level l - 1
template <bool WAVE>
__device__ __forceinline__ void coarse_pre(CoarseMem &m, int l, const double *f, bool zero) {
    const Blk q = blk_of(m, l);
    const double h2 = m.h2[l], h2i = m.h2i[l];
    double fa = 0, fb = 0, fc = 0, fd = 0, a = 0, b = 0, c = 0, d = 0;
    double cu = 0, bl = 0, bd = 0, cr = 0;
    const int k = q.k;
    if (q.on) {
        own4(f, l, fa, fb, fc, fd);
        if (!zero) {
            a = q.pA[k];
            b = q.pB[k];
            c = q.pC[k];
            d = q.pD[k];
            cu = q.pC[k - q.ld];
            bl = q.pB[k - 1];
            bd = q.pB[k + q.ld];
            cr = q.pC[k + 1];
        }
        // red: south, north, east, west of A are C, C above, B, B left
        if (q.ia) a = 0.25 * (c + cu + b + bl - h2 * fa);
        d = 0.25 * (bd + b + cr + c - h2 * fd);
        q.pA[k] = a;
        q.pD[k] = d;
    }
    level_sync<WAVE>();
    double rb = 0, rc = 0;
    double *rB = m.res + 34, *rC = rB + q.ld * q.ld;
    if (q.on) {
        const double du = q.pD[k - q.ld], ar = q.pA[k + 1], ad = q.pA[k + q.ld], dl = q.pD[k - 1];
        if (q.ib) {
            b = 0.25 * (d + du + ar + a - h2 * fb);
            rb = -h2i * (d + du + ar + a - 4.0 * b) + fb;
        }
        if (q.ic) {
            c = 0.25 * (ad + a + d + dl - h2 * fc);
            rc = -h2i * (ad + a + d + dl - 4.0 * c) + fc;
        }
        q.pB[k] = b;
        q.pC[k] = c;
        rB[k] = rb;
        rC[k] = rc;
    }
    level_sync<WAVE>();
    if (q.ia) {
        const double ra = -h2i * (c + q.pC[k - q.ld] + b + q.pB[k - 1] - 4.0 * a) + fa;
        const int t = (int)threadIdx.x;
        m.cres[flat_start(l - 1) + (t >> l) * q.ld + (t & (q.nb - 1))] =
            0.5 * ra + 0.125 * (rc + rC[k - q.ld] + rb + rB[k - 1]);
    }
    level_sync<WAVE>();
}

// prolongation of level l - 1's solution to the planes of level l: added to
// the iterate, or (start) as the iterate
template <bool WAVE>
__device__ __forceinline__ void coarse_interp(CoarseMem &m, int l, bool start, double &a,
                                              double &b, double &c, double &d, const Blk &q) {
    const double *s = m.sol + flat_start(l - 1) + q.k;  // its rows are ld long too
    const double c00 = s[0], c01 = s[1], c10 = s[q.ld], c11 = s[q.ld + 1];
    const double vc = 0.5 * (c10 + c00), vb = 0.5 * (c01 + c00);
    const double vd = 0.5 * (0.5 * (c11 + c01) + vc);
    if (start) {
        a = q.ia ? c00 : 0.0;
        b = q.ib ? vb : 0.0;
        c = q.ic ? vc : 0.0;
        d = vd;
    } else {
        a = q.ia ? q.pA[q.k] + c00 : 0.0;
        b = q.ib ? q.pB[q.k] + vb : 0.0;
        c = q.ic ? q.pC[q.k] + vc : 0.0;
        d = q.pD[q.k] + vd;
    }
}

// prolongation-add and smoothing of level l; the result to the planes and to
// sol (out null) or to the row-major array out
template <bool WAVE>
__device__ __forceinline__ void coarse_post(CoarseMem &m, int l, const double *f, double *out) {
    const Blk q = blk_of(m, l);
    const double h2 = m.h2[l];
    double fa = 0, fb = 0, fc = 0, fd = 0, a = 0, b = 0, c = 0, d = 0;
    const int k = q.k;
    if (q.on) {
        own4(f, l, fa, fb, fc, fd);
        coarse_interp<WAVE>(m, l, false, a, b, c, d, q);
        q.pB[k] = b;
        q.pC[k] = c;
    }
    level_sync<WAVE>();
    if (q.on) {
        if (q.ia) a = 0.25 * (c + q.pC[k - q.ld] + b + q.pB[k - 1] - h2 * fa);
        d = 0.25 * (q.pB[k + q.ld] + b + q.pC[k + 1] + c - h2 * fd);
        q.pA[k] = a;
        q.pD[k] = d;
    }
    level_sync<WAVE>();
    if (q.on) {
        const double du = q.pD[k - q.ld], ar = q.pA[k + 1], ad = q.pA[k + q.ld], dl = q.pD[k - 1];
        if (q.ib) b = 0.25 * (d + du + ar + a - h2 * fb);
        if (q.ic) c = 0.25 * (ad + a + d + dl - h2 * fc);
        q.pB[k] = b;
        q.pC[k] = c;
        const int n = lvl_size(l), t = (int)threadIdx.x;
        double *o = (out ? out : m.sol + flat_start(l)) + (2 * (t >> l)) * n + 2 * (t & (q.nb - 1));
        o[0] = a;
        o[1] = b;
        o[n] = c;
        o[n + 1] = d;
    }
    level_sync<WAVE>();
}

// the 3 x 3 level: h = length / 2, one unknown (mglin.cpp:103-110); one thread
__device__ __forceinline__ void coarse_slvsml(CoarseMem &m, double rhs, double length) {
    const double h = 0.5 * length;
    m.sol[4] = -h * h * rhs / 4.0;
}

// one V(1,1) cycle at level j >= 1 on f (mglin.cpp:176-196)
__device__ __forceinline__ void coarse_vcycle(CoarseMem &m, int j, const double *f, bool zero,
                                              double length, double *out) {
    int l = j;
    for (; l > 3; l--) coarse_pre<false>(m, l, l == j ? f : m.cres + flat_start(l), zero || l < j);
    if (threadIdx.x < 64) {
        for (int w = l; w >= 1; w--)
            coarse_pre<true>(m, w, w == j ? f : m.cres + flat_start(w), zero || w < j);
        if (threadIdx.x == 0) coarse_slvsml(m, m.cres[4], length);
        level_sync<true>();
        for (int w = 1; w <= l; w++)
            coarse_post<true>(m, w, w == j ? f : m.cres + flat_start(w), w == j ? out : nullptr);
    }
    __syncthreads();
    for (l++; l <= j; l++)
        coarse_post<false>(m, l, l == j ? f : m.cres + flat_start(l), l == j ? out : nullptr);
}

// full: full multigrid from rhs_in (level lc) -> u_out; else one V-cycle from
// a zero iterate (the coarse correction of a finer V-cycle).  max(64, 4^lc)
// threads.
__global__ void __launch_bounds__(1024)
    k_fmg_coarse(const double *__restrict__ rhs_in, double *__restrict__ u_out, int lc, int full,
                 int ncycle, double length) {
    __shared__ CoarseMem m;
    const int tid = (int)threadIdx.x, nt = (int)blockDim.x, n = lvl_size(lc), nn = n * n;
    double *top = m.rhs + flat_start(lc);
    for (int k = tid; k < nn; k += nt) top[k] = rhs_in[k];
    for (int k = tid; k < (int)(sizeof(m.planes) / 8); k += nt) m.planes[k] = 0.0;
    for (int k = tid; k < (int)(sizeof(m.sol) / 8); k += nt) m.sol[k] = 0.0;
    for (int k = tid; k < (int)(sizeof(m.res) / 8); k += nt) m.res[k] = 0.0;
    if (tid <= lc) {
        const double h = length / (lvl_size(tid) - 1), h2 = h * h;
        m.h2[tid] = h2;
        m.h2i[tid] = 1.0 / h2;
    }
    // the walls of u_out; the blocks write the rest (and the first row and
    // column again)
    for (int k = tid; k < n; k += nt) u_out[k * n + n - 1] = u_out[(n - 1) * n + k] = 0.0;
    __syncthreads();
    if (lc == 0) {
        const double h = 0.5 * length;
        for (int k = tid; k < nn; k += nt) u_out[k] = k == 4 ? -h * h * top[4] / 4.0 : 0.0;
        return;
    }
    if (!full) {
        coarse_vcycle(m, lc, top, true, length, u_out);
        return;
    }
    for (int l = lc - 1; l >= 0; l--) {
        const int nc = lvl_size(l);
        for (int t = tid; t < 1 << (2 * l + 2); t += nt) {  // rows and columns 1 .. nc - 2
            const int ic = t >> (l + 1), jc = t & ((1 << (l + 1)) - 1);
            if (ic > 0 && jc > 0)
                m.rhs[flat_start(l) + ic * nc + jc] =
                    rstrct_node(m.rhs + flat_start(l + 1), nc, ic, jc);
        }
        __syncthreads();
    }
    if (tid == 0) coarse_slvsml(m, m.rhs[4], length);
    __syncthreads();
    for (int j = 1; j <= lc; j++) {
        const Blk q = blk_of(m, j);
        if (q.on) {
            double a, b, c, d;
            coarse_interp<false>(m, j, true, a, b, c, d, q);
            q.pA[q.k] = a;
            q.pB[q.k] = b;
            q.pC[q.k] = c;
            q.pD[q.k] = d;
        }
        __syncthreads();
        for (int c = 0; c < ncycle; c++)
            coarse_vcycle(m, j, m.rhs + flat_start(j), false, length, j == lc ? u_out : nullptr);
    }
}

// ------------------------------------------------- levels above 65^2: legs
// A workgroup owns a T x T tile of fine nodes and recomputes the halo it needs
// in LDS (each sweep of one colour uses up a ring, the residual one more), so
// no other tile's output is read.  POST: the iterate is us plus the
// prolongation of cv, smoothed; PRE: the iterate (POST's, or u_in, or the
// prolongation of uc, or zero) is smoothed, written to u_out and its
// restricted residual to cres.  POST without PRE writes u_out.
template <int T, bool POST, bool PRE> struct Leg {
    static constexpr int H = (POST ? 2 : 0) + (PRE ? 4 : 0), W = T + 2 * H;
};

template <int T>
__device__ __forceinline__ void leg_sweep(double *s, const double *f, int W, int H, int x0, int y0,
                                          int ring, int n, double h2, int color) {
    const int lo = H - ring, w = T + 2 * ring;
    for (int k = threadIdx.x; k < w * w; k += 256) {
        const int ly = lo + k / w, lx = lo + k % w;
        const int i = y0 - H + ly, j = x0 - H + lx;
        if (i < 1 || j < 1 || i > n - 2 || j > n - 2 || ((i + j) & 1) != color) continue;
        const int c = ly * W + lx;
        s[c] = 0.25 * (s[c + W] + s[c - W] + s[c + 1] + s[c - 1] - h2 * f[c]);
    }
    __syncthreads();
}

template <int T, bool POST, bool PRE>
__global__ void __launch_bounds__(256)
    k_fmg_leg(const double *__restrict__ u_in, const double *__restrict__ uc,
              const double *__restrict__ cv, const double *__restrict__ rhs, int n, double h2,
              double h2i, double *__restrict__ u_out, double *__restrict__ cres) {
    constexpr int H = Leg<T, POST, PRE>::H, W = Leg<T, POST, PRE>::W;
    __shared__ double su[W * W], sf[W * W];
    const int x0 = blockIdx.x * T, y0 = blockIdx.y * T, nc = (n + 1) / 2;
    for (int k = threadIdx.x; k < W * W; k += 256) {
        const int i = y0 - H + k / W, j = x0 - H + k % W;
        double u = 0.0, f = 0.0;
        if (i >= 0 && j >= 0 && i < n && j < n) {
            f = rhs[i * n + j];
            if (u_in) u = u_in[i * n + j];
            if (POST) u += interp_node(cv, nc, i, j);
            if (uc) u = interp_node(uc, nc, i, j);
        }
        su[k] = u;
        sf[k] = f;
    }
    __syncthreads();
    constexpr int R = PRE ? 4 : 0;  // rings still valid after POST's sweeps
    if (POST) {
        leg_sweep<T>(su, sf, W, H, x0, y0, R + 1, n, h2, 0);
        leg_sweep<T>(su, sf, W, H, x0, y0, R, n, h2, 1);
    }
    if (PRE) {
        leg_sweep<T>(su, sf, W, H, x0, y0, 3, n, h2, 0);
        leg_sweep<T>(su, sf, W, H, x0, y0, 2, n, h2, 1);
    }
    for (int k = threadIdx.x; k < T * T; k += 256) {
        const int ly = k / T, lx = k % T, i = y0 + ly, j = x0 + lx;
        if (i < n && j < n) u_out[i * n + j] = su[(ly + H) * W + lx + H];
    }
    if (PRE) {
        auto resid = [&](int c) {
            return -h2i * (su[c + W] + su[c - W] + su[c + 1] + su[c - 1] - 4.0 * su[c]) + sf[c];
        };
        for (int k = threadIdx.x; k < (T / 2) * (T / 2); k += 256) {
            const int ic = y0 / 2 + k / (T / 2), jc = x0 / 2 + k % (T / 2);
            if (ic >= nc || jc >= nc) continue;
            double v = 0.0;
            if (ic > 0 && jc > 0 && ic < nc - 1 && jc < nc - 1) {
                const int c = (2 * ic - y0 + H) * W + (2 * jc - x0 + H);
                v = 0.5 * resid(c) +
                    0.125 * (resid(c + W) + resid(c - W) + resid(c + 1) + resid(c - 1));
            }
            cres[ic * nc + jc] = v;
        }
    }
}

// ------------------------------------------------------------------ driver

static void coarse_launch(hipStream_t st, int lc, const double *rhs, double *u, bool full,
                          int ncycle, double length) {
    const int t = 1 << (2 * lc);
    hipLaunchKernelGGL(k_fmg_coarse, dim3(1), dim3(t < 64 ? 64 : t), 0, st, rhs, u, lc,
                       full ? 1 : 0, ncycle, length);
}

// the legs' tile edge: 16 keeps more workgroups in flight where a leg is bound
// by its latency, 32 above 513^2 rereads less halo
template <bool POST, bool PRE>
static void leg_launch(hipStream_t st, const double *u_in, const double *uc, const double *cv,
                       const double *rhs, int l, double length, double *u_out, double *cres) {
    const int n = lvl_size(l), T = n <= 513 ? 16 : 32, tiles = (n + T - 1) / T;
    const double h = length / (n - 1), h2 = h * h, h2i = 1.0 / (h * h);
    const dim3 g(tiles, tiles), b(256);
    if (T == 16)
        hipLaunchKernelGGL((k_fmg_leg<16, POST, PRE>), g, b, 0, st, u_in, uc, cv, rhs, n, h2, h2i,
                           u_out, cres);
    else
        hipLaunchKernelGGL((k_fmg_leg<32, POST, PRE>), g, b, 0, st, u_in, uc, cv, rhs, n, h2, h2i,
                           u_out, cres);
}

// the coarse correction of a V-cycle at level j: A.cv[j-1] from A.cres[j-1]
static void correction(hipStream_t st, MgArrays<double> &A, int lc, int j, double length) {
    const int l = j - 1;
    if (l == lc) {
        coarse_launch(st, lc, A.cres[l], A.cv[l], false, 1, length);
        return;
    }
    // below the cycles' own level its full-multigrid iterate is spent: u[l]
    // holds the smoothed iterate between the legs
    leg_launch<false, true>(st, nullptr, nullptr, nullptr, A.cres[l], l, length, A.u[l],
                            A.cres[l - 1]);
    correction(st, A, lc, l, length);
    leg_launch<true, false>(st, A.u[l], nullptr, A.cv[l - 1], A.cres[l], l, length, A.cv[l],
                            nullptr);
}

// ncycle V(1,1) cycles at level j > lc on u[j], which starts as the
// prolongation of u[j-1] (from_coarse) or is what it holds.  The iterate
// alternates between u[j] and cv[j] (free at the cycles' own level) and ends
// in u[j].
static void cycles(hipStream_t st, MgArrays<double> &A, int lc, int j, int ncycle, double length,
                   bool from_coarse) {
    double *a = A.cv[j], *b = A.u[j];
    if (from_coarse && ncycle % 2 == 0) std::swap(a, b);
    leg_launch<false, true>(st, from_coarse ? nullptr : A.u[j], from_coarse ? A.u[j - 1] : nullptr,
                            nullptr, A.rhsF[j], j, length, a, A.cres[j - 1]);
    for (int c = 1; c < ncycle; c++) {
        correction(st, A, lc, j, length);
        leg_launch<true, true>(st, a, nullptr, A.cv[j - 1], A.rhsF[j], j, length, b, A.cres[j - 1]);
        std::swap(a, b);
    }
    correction(st, A, lc, j, length);
    leg_launch<true, false>(st, a, nullptr, A.cv[j - 1], A.rhsF[j], j, length, A.u[j], nullptr);
}

int mg_coarse_level_for(int ng) { return ng - 1 < FMG_TOP ? ng - 1 : FMG_TOP; }

// FP64 full multigrid (mglin.cpp:21-55) on the device.  rhs = M.d.rhsF[ng-1]
// (finest) on entry; the solution is written to M.d.u[ng-1].
void mg_fixed_solve(hipStream_t st, MgLevels &M, int ncycle, double length) {
    MgArrays<double> &A = M.d;
    const int lf = M.ng - 1, lc = M.lc;
    for (int l = lf - 1; l >= lc; l--) {
        const int nc = lvl_size(l);
        hipLaunchKernelGGL(k_fmg_rstrct, dim3((nc + 127) / 128, nc), dim3(128), 0, st, A.rhsF[l],
                           nc, A.rhsF[l + 1]);
    }
    coarse_launch(st, lc, A.rhsF[lc], A.u[lc], true, ncycle, length);
    for (int j = lc + 1; j <= lf; j++) cycles(st, A, lc, j, ncycle, length, true);
}

void mg_fixed_vcycle(hipStream_t st, MgLevels &M, double length) {
    cycles(st, M.d, M.lc, M.ng - 1, 1, length, false);
}

}  // namespace pic
