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
// What bounds it: latency, per level visit some 100 instructions of one
// wavefront and 6 dependent LDS round trips.  So the level is a template
// argument (a thread's plane index is its own plus its block row, and every
// LDS address that plus a constant), its nodes and right-hand side stay in
// registers between the two legs, and the grid spacings are exact powers of
// four apart: 9.5 us for a V-cycle from 65^2 and 35 us for the full multigrid
// there.  With runtime levels (the index arithmetic of every visit) they took
// 11.5 and 50 us, with one node per thread and sweep 45 and 170 us.
#define FMG_TOP 5

struct CoarseMem {
    double planes[4 * (33 * 33 + 17 * 17 + 9 * 9 + 5 * 5 + 3 * 3) + 40];
    double res[2 * 33 * 33 + 40];  // black residuals of the visited level
    double cres[33 * 33 + 17 * 17 + 9 * 9 + 5 * 5 + 3 * 3];  // V-cycle rhs, levels 0..4
    double sol[33 * 33 + 17 * 17 + 9 * 9 + 5 * 5 + 3 * 3];   // solutions, levels 0..4
    double rhs[65 * 65 + 33 * 33 + 17 * 17 + 9 * 9 + 5 * 5 + 3 * 3];  // levels 0..5
};

// sum of (2^k + 1)^2 for k = 1 .. l-1, the start of level l's plane quartet / 4
__host__ __device__ constexpr int plane_start(int l) {
    return ((1 << (2 * l)) - 4) / 3 + 2 * ((1 << l) - 2) + (l - 1);
}
// sum of lvl_size(k)^2 for k < l
__host__ __device__ constexpr int flat_start(int l) { return plane_start(l + 1); }

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

struct Node4 {
    double a, b, c, d;
};

// a level and the thread's place on it
template <int L>
struct Lvl {
    static constexpr int NB = 1 << L;       // blocks per side
    static constexpr int LD = NB + 1;       // plane row (and row of the level below)
    static constexpr int S = LD * LD;       // plane
    static constexpr int N = 2 * NB + 1;    // row of a row-major array
    static constexpr double H = 1.0 / (1 << (2 * L));  // (spacing / level 0's)^2
    int k, o;             // place in a plane, of node A in a row-major array
    bool on, ia, ib, ic;  // owns a block; A, B, C are inside (D always is)
    __device__ __forceinline__ Lvl() {
        const int t = (int)threadIdx.x;
        on = t < NB * NB;
        const int u = on ? t : 0, b = u >> L, c = u & (NB - 1);
        k = u + b;
        o = 2 * (k + (u & ~(NB - 1)));
        ia = on && b > 0 && c > 0;
        ib = on && b > 0;
        ic = on && c > 0;
    }
    // 34 doubles ahead: index -1 and -LD of a wall block are never used but
    // stay inside the array
    __device__ __forceinline__ double *plane(CoarseMem &m, int p) const {
        return m.planes + 34 + 4 * plane_start(L) + p * S + k;
    }
    __device__ __forceinline__ Node4 own4(const double *f) const {
        return Node4{f[o], f[o + 1], f[o + N], f[o + N + 1]};
    }
};

struct Spacing {
    double h2, h2i;  // level 0's squared spacing and its reciprocal
    double length;
};

// smoothing of level L on rhs (zero: from a zero iterate, else from the
// planes), the thread's nodes in u, the residual restricted into cres of level
// L - 1
template <int L, bool WAVE>
__device__ __forceinline__ void coarse_pre(CoarseMem &m, const Spacing &sp, const double *rhs,
                                           Node4 &u, bool zero) {
    constexpr int LD = Lvl<L>::LD;
    const Lvl<L> q;
    const double h2 = sp.h2 * Lvl<L>::H, h2i = sp.h2i * (1.0 / Lvl<L>::H);
    double *pA = q.plane(m, 0), *pB = q.plane(m, 1), *pC = q.plane(m, 2), *pD = q.plane(m, 3);
    double *rB = m.res + 34 + q.k, *rC = rB + Lvl<L>::S;
    double cu = 0, bl = 0, bd = 0, cr = 0;
    const Node4 f = q.own4(rhs);
    u = Node4{0, 0, 0, 0};
    if (!zero && q.on) {
        u = Node4{*pA, *pB, *pC, *pD};
        cu = pC[-LD];
        bl = pB[-1];
        bd = pB[LD];
        cr = pC[1];
    }
    if (q.on) {
        // red: south, north, east, west of A are C, C above, B, B left
        const double a = 0.25 * (u.c + cu + u.b + bl - h2 * f.a);
        u.a = q.ia ? a : u.a;
        u.d = 0.25 * (bd + u.b + cr + u.c - h2 * f.d);
        *pA = u.a;
        *pD = u.d;
    }
    level_sync<WAVE>();
    double rb = 0, rc = 0;
    if (q.on) {
        const double du = pD[-LD], ar = pA[1], ad = pA[LD], dl = pD[-1];
        const double sb = u.d + du + ar + u.a, sc = ad + u.a + u.d + dl;
        const double b = 0.25 * (sb - h2 * f.b), c = 0.25 * (sc - h2 * f.c);
        u.b = q.ib ? b : u.b;
        u.c = q.ic ? c : u.c;
        rb = q.ib ? -h2i * (sb - 4.0 * b) + f.b : 0.0;
        rc = q.ic ? -h2i * (sc - 4.0 * c) + f.c : 0.0;
        *pB = u.b;
        *pC = u.c;
        *rB = rb;
        *rC = rc;
    }
    level_sync<WAVE>();
    if (q.ia) {
        const double ra = -h2i * (u.c + pC[-LD] + u.b + pB[-1] - 4.0 * u.a) + f.a;
        m.cres[flat_start(L - 1) + q.k] = 0.5 * ra + 0.125 * (rc + rC[-LD] + rb + rB[-1]);
    }
    level_sync<WAVE>();
}

// prolongation of level L - 1's solution to the thread's nodes
template <int L>
__device__ __forceinline__ Node4 coarse_interp(CoarseMem &m, const Lvl<L> &q) {
    constexpr int LD = Lvl<L>::LD;
    const double *s = m.sol + flat_start(L - 1) + q.k;  // its rows are LD long too
    const double c00 = s[0], c01 = s[1], c10 = s[LD], c11 = s[LD + 1];
    const double vc = 0.5 * (c10 + c00), vb = 0.5 * (c01 + c00);
    return Node4{c00, vb, vc, 0.5 * (0.5 * (c11 + c01) + vc)};
}

// level L's iterate from level L - 1's solution, to the planes
template <int L>
__device__ __forceinline__ void coarse_start(CoarseMem &m) {
    const Lvl<L> q;
    if (q.on) {
        const Node4 v = coarse_interp<L>(m, q);
        *q.plane(m, 0) = q.ia ? v.a : 0.0;
        *q.plane(m, 1) = q.ib ? v.b : 0.0;
        *q.plane(m, 2) = q.ic ? v.c : 0.0;
        *q.plane(m, 3) = v.d;
    }
    __syncthreads();
}

// prolongation-add to the nodes u and smoothing of level L; the result to the
// planes and to sol (out null) or the row-major array out
template <int L, bool WAVE>
__device__ __forceinline__ void coarse_post(CoarseMem &m, const Spacing &sp, const double *rhs,
                                            Node4 u, double *out) {
    constexpr int LD = Lvl<L>::LD, N = Lvl<L>::N;
    const Lvl<L> q;
    const double h2 = sp.h2 * Lvl<L>::H;
    double *pA = q.plane(m, 0), *pB = q.plane(m, 1), *pC = q.plane(m, 2), *pD = q.plane(m, 3);
    const Node4 f = q.own4(rhs);
    if (q.on) {
        const Node4 v = coarse_interp<L>(m, q);
        u = Node4{q.ia ? u.a + v.a : 0.0, q.ib ? u.b + v.b : 0.0, q.ic ? u.c + v.c : 0.0,
                  u.d + v.d};
        *pB = u.b;
        *pC = u.c;
    }
    level_sync<WAVE>();
    if (q.on) {
        const double a = 0.25 * (u.c + pC[-LD] + u.b + pB[-1] - h2 * f.a);
        u.a = q.ia ? a : u.a;
        u.d = 0.25 * (pB[LD] + u.b + pC[1] + u.c - h2 * f.d);
        *pA = u.a;
        *pD = u.d;
    }
    level_sync<WAVE>();
    if (q.on) {
        const double du = pD[-LD], ar = pA[1], ad = pA[LD], dl = pD[-1];
        const double b = 0.25 * (u.d + du + ar + u.a - h2 * f.b);
        const double c = 0.25 * (ad + u.a + u.d + dl - h2 * f.c);
        u.b = q.ib ? b : u.b;
        u.c = q.ic ? c : u.c;
        *pB = u.b;
        *pC = u.c;
        if (out) {
            out[q.o] = u.a;
            out[q.o + 1] = u.b;
            out[q.o + N] = u.c;
            out[q.o + N + 1] = u.d;
        } else {
            double *s = m.sol + flat_start(L) + q.o;
            s[0] = u.a;
            s[1] = u.b;
            s[N] = u.c;
            s[N + 1] = u.d;
        }
    }
    level_sync<WAVE>();
}

// the 3 x 3 level: h = length / 2, one unknown (mglin.cpp:103-110); one thread
__device__ __forceinline__ void coarse_slvsml(CoarseMem &m, double rhs, double length) {
    const double h = 0.5 * length;
    m.sol[4] = -h * h * rhs / 4.0;
}

// one V(1,1) cycle at level j >= 1 (mglin.cpp:176-196) on rhs, from a zero
// iterate (zero) or the planes; the levels below follow in line, those above j
// are skipped
__device__ __forceinline__ void coarse_vcycle(CoarseMem &m, int j, const Spacing &sp, bool zero,
                                              double *out) {
    Node4 u5, u4;
#define FMG_RHS(L) ((j == L ? m.rhs : m.cres) + flat_start(L))
#define FMG_DOWN(L, WAVE, U) \
    if (j >= L) coarse_pre<L, WAVE>(m, sp, FMG_RHS(L), U, zero || j > L);
#define FMG_UP(L, WAVE, U) \
    if (j >= L) coarse_post<L, WAVE>(m, sp, FMG_RHS(L), U, j == L ? out : nullptr);
    FMG_DOWN(5, false, u5)
    FMG_DOWN(4, false, u4)
    if (threadIdx.x < 64) {
        Node4 u3, u2, u1;
        FMG_DOWN(3, true, u3)
        FMG_DOWN(2, true, u2)
        FMG_DOWN(1, true, u1)
        if (threadIdx.x == 0) coarse_slvsml(m, m.cres[4], sp.length);
        level_sync<true>();
        FMG_UP(1, true, u1)
        FMG_UP(2, true, u2)
        FMG_UP(3, true, u3)
    }
    __syncthreads();
    FMG_UP(4, false, u4)
    FMG_UP(5, false, u5)
#undef FMG_RHS
#undef FMG_DOWN
#undef FMG_UP
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
    // level l's spacing is 2^-l of level 0's: its square and the square's
    // reciprocal are those of level 0 times a power of four, exactly
    const double h0 = length / 2.0, h00 = h0 * h0;
    const Spacing sp{h00, 1.0 / h00, length};
    // the walls of u_out; the blocks write the rest (and the first row and
    // column again)
    for (int k = tid; k < n; k += nt) u_out[k * n + n - 1] = u_out[(n - 1) * n + k] = 0.0;
    __syncthreads();
    if (lc == 0) {
        const double h = 0.5 * length;
        for (int k = tid; k < nn; k += nt) u_out[k] = k == 4 ? -h * h * top[4] / 4.0 : 0.0;
        return;
    }
    if (full) {
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
    }
    for (int j = full ? 1 : lc; j <= lc; j++) {
        if (full) switch (j) {
            case 1: coarse_start<1>(m); break;
            case 2: coarse_start<2>(m); break;
            case 3: coarse_start<3>(m); break;
            case 4: coarse_start<4>(m); break;
            default: coarse_start<5>(m); break;
            }
        for (int c = 0; c < (full ? ncycle : 1); c++)
            coarse_vcycle(m, j, sp, !full, j == lc ? u_out : nullptr);
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
