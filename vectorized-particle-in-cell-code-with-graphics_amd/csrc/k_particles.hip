// k_particles.hip -- particle kernels.
//
// Sort pass of one species (a timestep that also reorders the store):
//   pass 1  k_key_count:    histogram of the sort keys of the particles'
//                           cells at the start of the step (counting-sort
//                           key, aggregated per block in LDS); holes of the
//                           store are not counted, so they are dropped;
//   scan    k_scan_*:       exclusive scan of the histogram -> bin starts;
//   pass 2  k_push_scatter: collisions + gather + push + wall test, the
//                           particle written to its key's slot of the other
//                           buffer (one claim per key per block; a particle
//                           lost in this step leaves a hole there), per-wall
//                           loss counts, and the fixed-point CIC deposit
//                           accumulated in an LDS window around the block's
//                           cells, flushed with one 64-bit atomic per touched
//                           node.
// Between sort passes, k_push_inplace advances a species in its own slots.
// Per-phase kernels for the reference-shaped entry points (gather, move,
// collect_charge, wall pass) reuse the same device functions.
#include "mcc.h"
#include "pic_internal.h"

namespace pic {

__device__ __forceinline__ PState load_state(const SpView &v, uint32_t i, bool need_vz) {
    PState s;
    uint32_t c = v.cell[i];
    s.jx = cell_jx(c);
    s.jy = cell_jy(c);
    s.ox = v.ox[i];
    s.oy = v.oy[i];
    s.vx = v.vx[i];
    s.vy = v.vy[i];
    s.vz = need_vz ? v.vz[i] : 0.0f;
    return s;
}

__device__ __forceinline__ void store_state(const SpView &v, uint32_t i, const PState &s,
                                            uint32_t id) {
    v.cell[i] = cell_pack(s.jx, s.jy);
    v.ox[i] = s.ox;
    v.oy[i] = s.oy;
    v.vx[i] = s.vx;
    v.vy[i] = s.vy;
    v.vz[i] = s.vz;
    v.id[i] = id;
}


// ------------------------------------------------------------ pass 1

// e_collisions.cpp:507-511 / ion_collisions.cpp:273-277: collide only while
// (int)(x/dx) and (int)(y/dy) are in [0, N), i.e. x in (-dx, N*dx)
__device__ __forceinline__ bool ref_mcc_inside(const PState &s, int N) {
    return s.jx >= -1 && s.jx <= N - 1 && !(s.jx == -1 && s.ox == 0.0f) && s.jy >= -1 &&
           s.jy <= N - 1 && !(s.jy == -1 && s.oy == 0.0f);
}

// collision (if enabled and not already settled by block_collide_n) then push;
// returns the particle's status.  `ev` and `ch` report the collision.
__device__ __forceinline__ int advance_one(PState &s, uint32_t id, const float2 *__restrict__ E,
                                           const PushConst &pc, const mcc::MccConst &mc,
                                           uint32_t step, int do_push, int &ev, mcc::Child &ch,
                                           bool mcc_done = false) {
    if (!mcc_done) ev = mcc::EV_NONE;
    if (s.jx == CELL_HOLE) return ST_HOLE;
    if (mc.on && !mcc_done) {
        if (mc.electron) {
            ev = mcc::collide_electron(mc, s.vx, s.vy, s.vz, id, step, ref_mcc_inside(s, pc.N), ch);
            if (EV_KIND(ev) == mcc::EV_IONIZE && mc.mode == PIC_DEV_MODE_REF) {
                s.jx = s.jy = CELL_DEAD;  // e_collisions.cpp:377-381: the parent does not survive
                return ST_DEAD;
            }
        } else {
            ev = mcc::collide_ion(mc, s.vx, s.vy, s.vz, id, step);
        }
    }
    if (do_push) push_one(s, E, pc);
    return classify(s, pc.N, pc.mode);
}


// LDS shared by the block-level collision queue and the deposit window
#define BLOCK_LDS_U64 2048
#define CQ_CAP 256  // collision queue entries per block (11 words each)

// Block-level null-collision step (physical mode) for the P particles of every
// thread.  Every particle makes its candidate test (mcc::candidate); the
// candidates -- about 13% of the electrons in the argon discharge, some 130 of
// a block's 1024 particles -- go into one LDS queue so the collision
// kinematics run once per block on dense lanes.  qs[r] returns the particle's
// queue entry (>= 0), -1 (no candidate) or -2 (queue full: the particle
// collides on its own lane in advance_one).  The results stay in the queue
// until every round has read them (collide_take): the caller leaves the LDS
// alone until a barrier after the last round.  The draws are the per-particle
// Philox streams of collide_electron / collide_ion, so every result is the
// per-lane one bit for bit.  Every thread of the block must call this (uniform
// condition: mc.on in physical mode).
template <int P>
__device__ __forceinline__ void block_collide_n(const bool (&active)[P], const PState (&s)[P],
                                                const uint32_t (&id)[P], const mcc::MccConst &mc,
                                                uint32_t step, int (&qs)[P],
                                                unsigned long long *lds, const float2 *tab) {
    static_assert(11 * CQ_CAP * 4 <= BLOCK_LDS_U64 * 8, "collision queue size");
    __shared__ uint32_t wcnt[4];
    float *q = reinterpret_cast<float *>(lds);  // SoA: v (3), id, event, child (6)
    uint32_t *qid = reinterpret_cast<uint32_t *>(q + 3 * CQ_CAP);
    int *qev = reinterpret_cast<int *>(q + 4 * CQ_CAP);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    uint32_t pos[P];
    uint32_t wtot = 0;
#pragma unroll
    for (int r = 0; r < P; r++) {
        const bool cand =
            active[r] && mcc::candidate(mc, id[r], step,
                                        s[r].vx * s[r].vx + s[r].vy * s[r].vy + s[r].vz * s[r].vz,
                                        tab);
        const uint64_t bal = __ballot(cand);
        pos[r] = cand ? wtot + (uint32_t)__popcll(bal & below) : 0xFFFFFFFFu;
        wtot += (uint32_t)__popcll(bal);
    }
    if (lane == 0) wcnt[w] = wtot;
    __syncthreads();
    uint32_t base = 0, total = 0;
    for (int k = 0; k < (int)(blockDim.x >> 6); k++) {
        if (k < w) base += wcnt[k];
        total += wcnt[k];
    }
#pragma unroll
    for (int r = 0; r < P; r++) {
        qs[r] = -1;
        if (pos[r] != 0xFFFFFFFFu) {
            const uint32_t slot = base + pos[r];
            if (slot < CQ_CAP) {
                q[slot] = s[r].vx;
                q[CQ_CAP + slot] = s[r].vy;
                q[2 * CQ_CAP + slot] = s[r].vz;
                qid[slot] = id[r];
                qs[r] = (int)slot;
            } else {
                qs[r] = -2;
            }
        }
    }
    __syncthreads();
    const uint32_t nq = min(total, (uint32_t)CQ_CAP);
    for (uint32_t t = threadIdx.x; t < nq; t += blockDim.x) {
        float vx = q[t], vy = q[CQ_CAP + t], vz = q[2 * CQ_CAP + t];
        mcc::Child c{};
        const int e = mc.electron ? mcc::collide_electron(mc, vx, vy, vz, qid[t], step, true, c, tab)
                                  : mcc::collide_ion(mc, vx, vy, vz, qid[t], step);
        q[t] = vx;
        q[CQ_CAP + t] = vy;
        q[2 * CQ_CAP + t] = vz;
        qev[t] = e;
        if (EV_KIND(e) == mcc::EV_IONIZE) {  // the only event with children
            q[5 * CQ_CAP + t] = c.vx;
            q[6 * CQ_CAP + t] = c.vy;
            q[7 * CQ_CAP + t] = c.vz;
            q[8 * CQ_CAP + t] = c.ivx;
            q[9 * CQ_CAP + t] = c.ivy;
            q[10 * CQ_CAP + t] = c.ivz;
        }
    }
    __syncthreads();
}

// A round's collision after block_collide_n: a queued particle takes its
// result.  Returns whether the collision is settled (false: not in physical
// mode, or the queue was full and advance_one collides the particle itself).
__device__ __forceinline__ bool collide_take(bool blk, int qs, PState &s, int &ev, mcc::Child &ch,
                                             const unsigned long long *lds) {
    if (!blk) return false;
    if (qs >= 0) {
        const float *q = reinterpret_cast<const float *>(lds);
        s.vx = q[qs];
        s.vy = q[CQ_CAP + qs];
        s.vz = q[2 * CQ_CAP + qs];
        ev = reinterpret_cast<const int *>(q + 4 * CQ_CAP)[qs];
        if (EV_KIND(ev) == mcc::EV_IONIZE) {
            ch.vx = q[5 * CQ_CAP + qs];
            ch.vy = q[6 * CQ_CAP + qs];
            ch.vz = q[7 * CQ_CAP + qs];
            ch.ivx = q[8 * CQ_CAP + qs];
            ch.ivy = q[9 * CQ_CAP + qs];
            ch.ivz = q[10 * CQ_CAP + qs];
        }
    }
    return qs != -2;
}

// Block-level key aggregation for the sort pass: the keys of the block's
// 256 x IPP particles go into an LDS hash table (open addressing, at most half
// full); each distinct key then costs one global atomic per block, and the
// block's particles of one key take consecutive slots.  Every particle's rank
// within its key comes from the LDS counter of its entry.
#define IPP (PASS_BLOCK / 256)
// The in-place passes of a store with room for at most INPL_SMALL_MAX particles
// (its capacity, which the grid covers: half as much again as the initial count
// where particles are created) take IPP_SMALL per thread: with IPP there are
// fewer blocks than 256 CUs, and a pass is the latency of one block's chain,
// not throughput.  A step with one and with four per thread, by capacity:
//                              131 k       200 k       262 k       410-420 k
//   257^2, reference mode   193 / 221   197 / 223   204 / 225   219 / 244 us
//   257^2, collisionless     36 / 41     36 / 43     40 / 41     43 / 49
//   65^2, collisionless      29 / 30     31 / 31     34 / 32     37 / 34
//   65^2, argon              46 / 51     49 / 54     52 / 56     54 / 56
// Dense cells cross over near 200 k (one particle per thread flushes four
// windows where one would do), sparse ones above 420 k; 33^2 gains 148 -> 144 us.
#define IPP_SMALL 1
#define INPL_SMALL_MAX (256 * PASS_BLOCK)
#define HASH_BITS 11
#define HASH_SIZE (1 << HASH_BITS)  // >= 2 x 256 x IPP
#define HASH_EMPTY 0xFFFFFFFFu
// direct key table of the scatter pass: key ranges up to SCAT_WIN entries,
// SCAT_EPT entries per thread of the 256
#define SCAT_WIN 1024
#define SCAT_EPT (SCAT_WIN / 256)

struct BlockHash {
    uint32_t key[HASH_SIZE];   // pass 2, after the claims: slot of the entry's rank-0 particle
    uint32_t cnt[HASH_SIZE];   // pass 2, after the claims: lowest rank with a valid slot
};

__device__ __forceinline__ void hash_clear(BlockHash &H) {
    for (int e = threadIdx.x; e < HASH_SIZE; e += blockDim.x) {
        H.key[e] = HASH_EMPTY;
        H.cnt[e] = 0u;
    }
}

// Wavefront key grouping: lanes holding the same key form one group (one per
// distinct key in the wavefront; leader = lowest lane).  Sorted input keeps
// the number of groups per wavefront small.
struct WaveGroup {
    int leader;      // lane of this lane's group leader (-1 if inactive)
    uint32_t rank;   // position of this lane within its group
    uint32_t count;  // group size (meaningful on the leader)
};

__device__ __forceinline__ WaveGroup wave_group(uint32_t key, bool active) {
    const int lane = threadIdx.x & 63;
    const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    WaveGroup g{-1, 0u, 0u};
    uint64_t pending = __ballot(active);
    while (pending) {
        const int leader = __ffsll((unsigned long long)pending) - 1;  // wave-uniform
        const uint32_t lkey = (uint32_t)__builtin_amdgcn_readlane((int)key, leader);
        const uint64_t grp = __ballot(active && key == lkey) & pending;
        if ((grp >> lane) & 1ull) {
            g.leader = leader;
            g.rank = (uint32_t)__popcll(grp & below);
            g.count = (uint32_t)__popcll(grp);
        }
        pending &= ~grp;
    }
    return g;
}

// entry of `key` in the table (inserted if new)
__device__ __forceinline__ uint32_t hash_entry(BlockHash &H, uint32_t key) {
    uint32_t e = (key * 0x9E3779B1u) >> (32 - HASH_BITS);
    for (;;) {  // the table never fills: at most 256 x IPP keys in 2x as many entries
        const uint32_t old = atomicCAS(&H.key[e], HASH_EMPTY, key);
        if (old == HASH_EMPTY || old == key) break;
        e = (e + 1u) & (HASH_SIZE - 1);
    }
    return e;
}

// Called by every lane of the wavefront.  Active lanes get the entry of their
// key and their rank among the block's particles of that key: the lanes of
// one key in a wavefront take consecutive ranks in lane order (one LDS
// atomic per distinct key per wavefront), so their slots are contiguous.
__device__ __forceinline__ uint32_t hash_insert(BlockHash &H, uint32_t key, bool active,
                                                uint32_t &rank) {
    const WaveGroup g = wave_group(key, active);
    uint32_t e = 0u, b = 0u;
    if (active && g.rank == 0) {
        e = hash_entry(H, key);
        b = atomicAdd(&H.cnt[e], g.count);
    }
    const int src = g.leader < 0 ? 0 : g.leader;
    e = (uint32_t)__shfl((int)e, src, 64);
    b = (uint32_t)__shfl((int)b, src, 64);
    rank = b + g.rank;
    return e;
}

// Variants of the particle passes.  The generic kernel takes every option at
// run time; the others pin options that the host has checked (physical mode,
// no magnetic field, no pair sampling in the pass, per-particle weights with
// PV_W and none without; then: no collisions and nothing staged (PLAIN); no
// collisions and lost particles queuing for re-injection or the surface pass
// (SPAWN); or the block-queued collisions of one species (COLL_E, COLL_I)),
// so the compiler drops the code and registers of everything else.  A pinned value always equals the one
// passed in, so every variant computes what the generic kernel computes.
// The argon ions (0.5 % candidates) used to leave theirs to a pass of their
// own, to keep the collision code's registers out of the ions' pass; with the
// products settled on the queue's lanes COLL_I takes 72 VGPRs like SPAWN, and
// that pass (18 us at 257^2, 125 us at 1025^2) is gone.
enum PassVariant {
    PV_GENERIC = 0,
    PV_PLAIN = 1,
    PV_COLL_E = 2,
    PV_COLL_I = 3,
    PV_SPAWN = 4,
    PV_COMPACT = 5,  // sort pass without a push (drops holes): the generic body, pinned
    PV_W = 8         // flag on PLAIN, SPAWN, COLL_E, COLL_I: per-particle weights
};
constexpr int pv_base(int v) { return v & 7; }
constexpr bool pv_weighted(int v) { return (v & PV_W) != 0; }
constexpr bool pv_coll_e(int v) { return pv_base(v) == PV_COLL_E; }
constexpr bool pv_coll_i(int v) { return pv_base(v) == PV_COLL_I; }

template <int V>
__device__ __forceinline__ void pin_variant(PushConst &pc, mcc::MccConst &mc, SpView &sp) {
    if (V == PV_GENERIC) return;
    pc.mode = PIC_DEV_MODE_PHYS;
    pc.bfield = 0;
    if (!pv_weighted(V)) sp.w = nullptr;
    if (!pv_coll_e(V) && !pv_coll_i(V)) {
        mc.on = 0;
    } else {
        mc.on = 1;
        mc.mode = PIC_DEV_MODE_PHYS;
        mc.electron = pv_coll_e(V) ? 1 : 0;
    }
}
// no variant but the generic one samples re-injected pairs in the pass (the
// fused step queues lost ions for the commit); PLAIN stages nothing at all
template <int V>
__device__ __forceinline__ void pin_spawn(Spawn &spn) {
    if (V != PV_GENERIC) spn.plop = 0;
    if (pv_base(V) == PV_PLAIN || V == PV_COMPACT) spn.wall = spn.lost_ids = 0;
}

// a particle lost through a wall queues its id and weight for the commit
__device__ __forceinline__ void queue_lost(const Spawn &spn, uint32_t id, float w) {
    const uint32_t slot = atomicAdd(&spn.cw->wall_count, 1u);
    if (slot >= spn.wq.cap) {
        atomicAdd(&spn.cw->overflow, 1u);
        return;
    }
    spn.wq.key[slot] = id;
    if (spn.wq.w) spn.wq.w[slot] = w;
}

// wavefront reductions of the device library (DPP row shifts and lane reads:
// no LDS round trips); every lane gets the result.  Called with all lanes
// active.
extern "C" __device__ int __ockl_wfred_min_i32(int);
extern "C" __device__ int __ockl_wfred_max_i32(int);
extern "C" __device__ int __ockl_wfred_add_i32(int);
__device__ __forceinline__ int wave_min(int v) { return __ockl_wfred_min_i32(v); }
__device__ __forceinline__ int wave_max(int v) { return __ockl_wfred_max_i32(v); }
__device__ __forceinline__ int wave_sum(int v) { return __ockl_wfred_add_i32(v); }

#define KC_WIN (2 * HASH_SIZE)  // direct-histogram range: the hash table's LDS

// Adds the block's keys (those with in[r]) to binCount, one global atomic
// per distinct key.  The keys of a block of a sorted store lie in a narrow
// range (a few rows of tiles): then the block counts them in a direct LDS
// histogram over that range (one LDS atomic per particle); a range of
// KC_WIN keys or more (an unsorted store) takes the LDS hash table.  `hist` is KC_WIN words of LDS, free on entry; every
// thread of the block calls this.
template <int P>
__device__ __forceinline__ void block_key_hist(const bool (&in)[P], const uint32_t (&key)[P],
                                               uint32_t *__restrict__ binCount, uint32_t *hist) {
    static_assert(sizeof(BlockHash) == KC_WIN * sizeof(uint32_t), "histogram size");
    __shared__ int wmin[4], wmax[4];
    int kmin = 0x7FFFFFFF, kmax = -1;
#pragma unroll
    for (int r = 0; r < P; r++)
        if (in[r]) {
            kmin = min(kmin, (int)key[r]);
            kmax = max(kmax, (int)key[r]);
        }
    kmin = wave_min(kmin);
    kmax = wave_max(kmax);
    if ((threadIdx.x & 63) == 0) {
        wmin[threadIdx.x >> 6] = kmin;
        wmax[threadIdx.x >> 6] = kmax;
    }
    __syncthreads();
    kmin = min(min(wmin[0], wmin[1]), min(wmin[2], wmin[3]));
    kmax = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
    if (kmax < kmin) return;  // no particle counted (uniform)
    if (kmax - kmin < KC_WIN) {
        const int span = kmax - kmin + 1;
        for (int e = threadIdx.x; e < span; e += blockDim.x) hist[e] = 0u;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < P; r++)
            if (in[r]) atomicAdd(&hist[key[r] - (uint32_t)kmin], 1u);
        __syncthreads();
        for (int e = threadIdx.x; e < span; e += blockDim.x) {
            const uint32_t c = hist[e];
            if (c) atomicAdd(&binCount[(size_t)(kmin + e) * BIN_STRIDE], c);
        }
        return;
    }
    BlockHash &H = *reinterpret_cast<BlockHash *>(hist);
    hash_clear(H);
    __syncthreads();  // table cleared
#pragma unroll
    for (int r = 0; r < P; r++) {
        uint32_t rank;
        hash_insert(H, key[r], in[r], rank);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < HASH_SIZE; e += blockDim.x) {
        const uint32_t k = H.key[e];
        if (k != HASH_EMPTY) atomicAdd(&binCount[(size_t)k * BIN_STRIDE], H.cnt[e]);
    }
}

// Pass 1 of the sort pass: the histogram of the sort keys of the particles'
// current cells (block_key_hist).  In a timestep's sort pass (do_push) every
// particle that is not a hole takes a slot, keyed by its cell before the
// step: one that leaves during the step leaves a hole in its slot, which the
// next sort pass drops.  Without a push (compaction) only the particles
// inside the domain are counted, so the output is compact.  Reads 4 B per
// particle (12 B without a push).  An in-place pass ahead of a sort pass
// makes this histogram itself (k_push_inplace, `hist`).
__global__ void __launch_bounds__(256)
    k_key_count(SpView sp, const uint32_t *__restrict__ nptr, PushConst pc,
                uint32_t *__restrict__ binCount, int do_push) {
    const uint32_t n = *nptr;
    if (blockIdx.x * (blockDim.x * IPP) >= n) return;  // past the live count
    __shared__ uint32_t hist[KC_WIN];  // the direct histogram or the hash table
    const uint32_t base = blockIdx.x * (blockDim.x * IPP) + threadIdx.x;
    uint32_t key[IPP];
    bool in[IPP];
#pragma unroll
    for (int r = 0; r < IPP; r++) {
        const uint32_t i = base + r * blockDim.x;
        key[r] = 0u;
        in[r] = false;
        if (i < n) {
            const uint32_t c = sp.cell[i];
            PState s{};
            s.jx = cell_jx(c);
            s.jy = cell_jy(c);
            if (do_push) {
                in[r] = s.jx != CELL_HOLE;
            } else if (s.jx != CELL_HOLE) {
                s.ox = sp.ox[i];
                s.oy = sp.oy[i];
                in[r] = classify(s, pc.N, pc.mode) == ST_KEPT;
            }
            if (in[r]) key[r] = bin_key(s.jx, s.jy, pc.tilesX) >> pc.keyshift;
        }
    }
    block_key_hist<IPP>(in, key, binCount, hist);
}

// ------------------------------------------------------------ scan
// exclusive scan of SCAN_TILE-element tiles: partial sums, top-level scan in
// one block, then per-tile scan plus offset.
#define SCAN_THREADS 256
#define SCAN_PER_THREAD 16
#define SCAN_TILE (SCAN_THREADS * SCAN_PER_THREAD)

__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t *total) {
    __shared__ uint32_t wsum[SCAN_THREADS / 64];
    int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t x = v;
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    uint32_t pre = 0, tot = 0;
    for (int k = 0; k < SCAN_THREADS / 64; k++) {
        if (k < w) pre += wsum[k];
        tot += wsum[k];
    }
    __syncthreads();
    *total = tot;
    return pre + x - v;
}

// exclusive scan over a 1024-thread block
__device__ __forceinline__ uint32_t block_excl_scan_1024(uint32_t v, uint32_t *total) {
    __shared__ uint32_t wsum[16];
    int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t x = v;
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    uint32_t pre = 0, tot = 0;
    for (int k = 0; k < (int)(blockDim.x >> 6); k++) {
        if (k < w) pre += wsum[k];
        tot += wsum[k];
    }
    __syncthreads();
    *total = tot;
    return pre + x - v;
}

// the counts are S words apart (BIN_STRIDE for the sort histogram, 1 for
// the compaction's block counts)
template <int S>
__global__ void __launch_bounds__(SCAN_THREADS)
    k_scan_partial(const uint32_t *__restrict__ in, uint32_t *__restrict__ partial) {
    const uint32_t *p =
        in + ((size_t)blockIdx.x * SCAN_TILE + threadIdx.x * SCAN_PER_THREAD) * S;
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < SCAN_PER_THREAD; k++) s += p[k * S];
    uint32_t tot;
    block_excl_scan(s, &tot);
    if (threadIdx.x == 0) partial[blockIdx.x] = tot;
}

__global__ void __launch_bounds__(SCAN_THREADS)
    k_scan_top(uint32_t *__restrict__ partial, int nparts, uint32_t *__restrict__ start_total,
               uint32_t *__restrict__ n_out) {
    uint32_t carry = 0;
    for (int base = 0; base < nparts; base += SCAN_THREADS) {
        int k = base + threadIdx.x;
        uint32_t v = (k < nparts) ? partial[k] : 0u;
        uint32_t tot;
        uint32_t ex = block_excl_scan(v, &tot);
        if (k < nparts) partial[k] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) {
        *start_total = carry;
        *n_out = carry;
    }
}

template <int S>
__global__ void __launch_bounds__(SCAN_THREADS)
    k_scan_final(const uint32_t *__restrict__ in, const uint32_t *__restrict__ partial,
                 uint32_t *__restrict__ out) {
    size_t base = (size_t)blockIdx.x * SCAN_TILE + threadIdx.x * SCAN_PER_THREAD;
    uint32_t v[SCAN_PER_THREAD];
    const uint32_t *p = in + base * S;
#pragma unroll
    for (int k = 0; k < SCAN_PER_THREAD; k++) v[k] = p[k * S];
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < SCAN_PER_THREAD; k++) s += v[k];
    uint32_t tot;
    uint32_t run = partial[blockIdx.x] + block_excl_scan(s, &tot);
    uint4 *o = reinterpret_cast<uint4 *>(out + base);
#pragma unroll
    for (int k = 0; k < SCAN_PER_THREAD / 4; k++) {
        uint4 q;
        q.x = run;
        run += v[4 * k];
        q.y = run;
        run += v[4 * k + 1];
        q.z = run;
        run += v[4 * k + 2];
        q.w = run;
        run += v[4 * k + 3];
        o[k] = q;
    }
}

// The whole scan of a few tiles of adjacent counts in one workgroup, a tile a
// round
__global__ void __launch_bounds__(1024)
    k_scan_one(const uint32_t *__restrict__ in, uint32_t *__restrict__ out, int nparts,
               uint32_t *__restrict__ n_out) {
    static_assert(SCAN_TILE == 4 * 1024, "four counts a thread");
    uint32_t carry = 0;
    for (int t = 0; t < nparts; t++) {
        const size_t k = (size_t)t * (SCAN_TILE / 4) + threadIdx.x;
        const uint4 v = reinterpret_cast<const uint4 *>(in)[k];
        uint32_t tot;
        const uint32_t x = carry + block_excl_scan_1024(v.x + v.y + v.z + v.w, &tot);
        reinterpret_cast<uint4 *>(out)[k] = uint4{x, x + v.x, x + v.x + v.y, x + v.x + v.y + v.z};
        carry += tot;
    }
    if (threadIdx.x == 0) {
        out[(size_t)nparts * SCAN_TILE] = carry;
        *n_out = carry;
    }
}

// Up to SCAN_ONE tiles of adjacent counts take one launch: 3.3 us for a tile
// against 7.4 for three launches.  (The sort histogram's counters, a line each,
// are too much for one CU: 31 us for three tiles, 20 for three launches.)
#define SCAN_ONE 4
template <int S>
static void launch_scan_s(hipStream_t st, const uint32_t *count, uint32_t *start,
                          uint32_t nbins_pad, uint32_t *partial, uint32_t *n_out) {
    int nparts = (int)(nbins_pad / SCAN_TILE);
    if (S == 1 && nparts <= SCAN_ONE) {
        hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(1024), 0, st, count, start, nparts, n_out);
        return;
    }
    hipLaunchKernelGGL(k_scan_partial<S>, dim3(nparts), dim3(SCAN_THREADS), 0, st, count, partial);
    hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(SCAN_THREADS), 0, st, partial, nparts,
                       start + nbins_pad, n_out);
    hipLaunchKernelGGL(k_scan_final<S>, dim3(nparts), dim3(SCAN_THREADS), 0, st, count, partial,
                       start);
}

void launch_scan(hipStream_t st, const uint32_t *count, uint32_t *start, uint32_t nbins_pad,
                 uint32_t *partial, uint32_t *n_out) {
    launch_scan_s<BIN_STRIDE>(st, count, start, nbins_pad, partial, n_out);
}

uint32_t scan_pad(uint32_t nbins) { return (nbins + SCAN_TILE - 1) / SCAN_TILE * SCAN_TILE; }

// ------------------------------------------------------------ pass 2
#define DEP_WCAP BLOCK_LDS_U64  // LDS window capacity (nodes), 16 KB of uint64


// Deposit the block's particles (dep true) through an LDS window spanning the
// bounding box of their cells (block reduction), flushed with one 64-bit
// atomic per touched node.  Sorted particles put most lanes of a
// wavefront on the same four nodes, and LDS atomics to one address serialise,
// so the window is replicated (up to DEP_COPIES copies, as many as fit) and
// lane l adds into copy l mod copies; the flush sums the copies.  Integer
// sums: the result does not depend on the split.  Every thread of the block
// must call this.
#define DEP_COPIES 8
// block_deposit_n for P particles per thread (dep[r] true: deposit s[r]); one
// window and one flush for the whole block.  When the bounding box of the
// block's cells exceeds the window (a few fast particles far from the rest),
// the window is a fixed square around the block's mean cell: the particles
// inside it go through LDS, the others deposit with global atomics.
// The window holds WCAP nodes (DEP_WCAP by default); the fallback square has
// edge 2 half + 2 with half = (floor(sqrt(WCAP)) - 2) / 2 (21 for 2048 nodes:
// 44 x 44 = 1936; 31 for 4096: 64 x 64).
constexpr int dep_half(int wcap) {
    int r = 0;
    while ((r + 1) * (r + 1) <= wcap) r++;
    return (r - 2) / 2;
}
template <int P, int WCAP = DEP_WCAP>
__device__ __forceinline__ void block_deposit_n(const bool (&dep)[P], const PState (&s)[P],
                                                const float (&pw)[P],
                                                unsigned long long *__restrict__ q, int N,
                                                unsigned long long *sq) {
    constexpr int DEP_HALF = dep_half(WCAP);
    static_assert((2 * DEP_HALF + 2) * (2 * DEP_HALF + 2) <= WCAP, "fallback window size");
    __shared__ int red[4][4];
    const int big = 1 << 30;
    int mnx = big, mny = big, mxx = -big, mxy = -big;
#pragma unroll
    for (int r = 0; r < P; r++) {
        mnx = min(mnx, dep[r] ? s[r].jx : big);
        mny = min(mny, dep[r] ? s[r].jy : big);
        mxx = max(mxx, dep[r] ? s[r].jx : -big);
        mxy = max(mxy, dep[r] ? s[r].jy : -big);
    }
    mnx = wave_min(mnx);
    mny = wave_min(mny);
    mxx = wave_max(mxx);
    mxy = wave_max(mxy);
    const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        red[w][0] = mnx;
        red[w][1] = mny;
        red[w][2] = mxx;
        red[w][3] = mxy;
    }
    __syncthreads();
    for (int k = 0; k < nw; k++) {
        mnx = min(mnx, red[k][0]);
        mny = min(mny, red[k][1]);
        mxx = max(mxx, red[k][2]);
        mxy = max(mxy, red[k][3]);
    }
    if (mxx < mnx) {  // nothing to deposit (uniform: all threads)
        __syncthreads();  // red[] is reused by the next call in the same kernel
        return;
    }
    // a depositing particle has jx in [0, N-2]: its nodes jx, jx+1 <= N-1
    int x0 = mnx, y0 = mny, ww = mxx - mnx + 2, wh = mxy - mny + 2;
    if (ww * wh > WCAP) {  // uniform: the block's mean cell is needed only here
        int sx = 0, sy = 0, cnt = 0;
#pragma unroll
        for (int r = 0; r < P; r++)
            if (dep[r]) {
                sx += s[r].jx;
                sy += s[r].jy;
                cnt++;
            }
        sx = wave_sum(sx);
        sy = wave_sum(sy);
        cnt = wave_sum(cnt);
        __syncthreads();  // red[] has been read
        if ((threadIdx.x & 63) == 0) {
            red[w][0] = sx;
            red[w][1] = sy;
            red[w][2] = cnt;
        }
        __syncthreads();
        sx = sy = cnt = 0;
        for (int k = 0; k < nw; k++) {
            sx += red[k][0];
            sy += red[k][1];
            cnt += red[k][2];
        }
        x0 = sx / cnt - DEP_HALF;
        y0 = sy / cnt - DEP_HALF;
        ww = wh = 2 * DEP_HALF + 2;
    }
    const int area = ww * wh;
    int copies = DEP_COPIES;
    while (copies > 1 && copies * area > WCAP) copies >>= 1;
    for (int k = threadIdx.x; k < copies * area; k += blockDim.x) sq[k] = 0ull;
    __syncthreads();
    const int cb = (int)(threadIdx.x & (copies - 1)) * area;
#pragma unroll
    for (int r = 0; r < P; r++)
        if (dep[r]) {
            const FxW fw = fx_weights_w(s[r].ox, s[r].oy, pw[r]);
            const int dx = s[r].jx - x0, dy = s[r].jy - y0;
            if ((unsigned)dx <= (unsigned)(ww - 2) && (unsigned)dy <= (unsigned)(wh - 2)) {
                const int b = cb + dy * ww + dx;
                atomicAdd(&sq[b], fw.a4);
                atomicAdd(&sq[b + 1], fw.a3);
                atomicAdd(&sq[b + ww], fw.a2);
                atomicAdd(&sq[b + ww + 1], fw.a1);
            } else {
                dep_global(q, N, s[r].jx, s[r].jy, fw);
            }
        }
    __syncthreads();
    // window nodes outside the grid (fallback window at an edge) stay zero.
    // The row of node k is k / ww in fp32: (k + 1/2) / ww is at least 1 / 2ww
    // off every integer and its rounding error below area 2^-23 / ww.
    const float inv = 1.0f / (float)ww;
    for (int k = threadIdx.x; k < area; k += blockDim.x) {
        unsigned long long v = 0ull;
        for (int c = 0; c < copies; c++) v += sq[c * area + k];
        if (v) {
            const int row = (int)(((float)k + 0.5f) * inv);
            atomicAdd(&q[(long)(y0 + row) * N + (x0 + k - row * ww)], v);
        }
    }
}

__device__ __forceinline__ void block_deposit(bool dep, const PState &s,
                                              unsigned long long *__restrict__ q, int N,
                                              unsigned long long *sq, float pw = 1.0f) {
    const bool d[1] = {dep};
    const PState ss[1] = {s};
    const float ww[1] = {pw};
    block_deposit_n<1>(d, ss, ww, q, N, sq);
}

// staging of a created particle (slot order is arbitrary; the commit pass
// sorts by key)
__device__ __forceinline__ void stage_put(const StageView &sv, uint32_t *__restrict__ count,
                                          uint32_t *__restrict__ overflow, const PState &s,
                                          unsigned long long key, float w = 1.0f) {
    uint32_t slot = atomicAdd(count, 1u);
    if (slot >= sv.cap) {
        atomicAdd(overflow, 1u);
        return;
    }
    sv.cell[slot] = cell_pack(s.jx, s.jy);
    sv.ox[slot] = s.ox;
    sv.oy[slot] = s.oy;
    sv.vx[slot] = s.vx;
    sv.vy[slot] = s.vy;
    sv.vz[slot] = s.vz;
    sv.key[slot] = key;
    if (sv.w) sv.w[slot] = w;
}

__device__ __forceinline__ void count_events(int ev, unsigned long long *__restrict__ events) {
    __shared__ uint32_t se[8];
    if (threadIdx.x < 8) se[threadIdx.x] = 0;
    __syncthreads();
    if (EV_KIND(ev) > 0) atomicAdd(&se[EV_KIND(ev)], 1u);
    if (ev & EV_OVER_BOUND) atomicAdd(&se[6], 1u);
    __syncthreads();
    if (threadIdx.x < 8 && se[threadIdx.x])
        atomicAdd(&events[cnt_slot() * 8 + threadIdx.x], (unsigned long long)se[threadIdx.x]);
}

// Products of a physical-mode ionisation of particle pid at `pre` (its state
// before the push), weight w
__device__ __forceinline__ void stage_ionisation(const mcc::Child &ch, const PState &pre,
                                                 uint32_t pid, const float2 *__restrict__ E,
                                                 const PushConst &pc, const Spawn &sp,
                                                 uint32_t *__restrict__ lost6, float w) {
    // ejected electron: born at the parent's position, pushed this step
    // as the reference pushes particles appended before move_particles
    PState ce = pre;
    ce.vx = ch.vx;
    ce.vy = ch.vy;
    ce.vz = ch.vz;
    push_one(ce, E, pc);
    const int cst = classify(ce, pc.N, pc.mode);
    if (cst != ST_KEPT) {
        // left the domain during its first push: it still takes its id
        // (as it does when created before the push), but is not stored
        atomicAdd(&lost6[cnt_slot() * 6 + cst - 1], 1u);
        ce.jx = ce.jy = CELL_DEAD;
    }
    stage_put(sp.se, &sp.ce->stage_count, &sp.ce->overflow, ce, (unsigned long long)pid, w);
    // new ion at the same place; the ion pass of this step moves it
    PState ci = pre;
    ci.vx = ch.ivx;
    ci.vy = ch.ivy;
    ci.vz = ch.ivz;
    // products take the parent's weight (e_collisions.cpp:413,441)
    stage_put(sp.si, &sp.ci->stage_count, &sp.ci->overflow, ci, (unsigned long long)pid, w);
}

// Products of one particle's step: the ejected electron and the new ion of a
// physical-mode ionisation, and the electron-ion pair re-injected for an ion
// lost through a wall (sp.plop).  `pre` is the state before the push.
__device__ __forceinline__ void stage_products(int ev, const mcc::Child &ch, const PState &pre,
                                               int st, bool valid, uint32_t pid,
                                               const float2 *__restrict__ E, const PushConst &pc,
                                               const mcc::MccConst &mc, uint32_t step,
                                               const Spawn &sp, uint32_t *__restrict__ lost6,
                                               float w, const PState &post) {
    if (EV_KIND(ev) == mcc::EV_IONIZE && mc.mode == PIC_DEV_MODE_PHYS)
        stage_ionisation(ch, pre, pid, E, pc, sp, lost6, w);
    if (sp.plop && valid && st >= ST_LEFT && st <= ST_TOP) {
        PState pe, pi;
        mcc::plop_pair(mc, pid, step, pc.N, sp.se_sigma, sp.si_sigma, sp.plop_ref, pe, pi);
        unsigned long long k = (1ull << 32) | pid;
        // the re-injected pair replaces the lost ion: it carries its weight
        stage_put(sp.se, &sp.ce->stage_count, &sp.ce->overflow, pe, k, w);
        stage_put(sp.si, &sp.ci->stage_count, &sp.ci->overflow, pi, k, w);
    }
    // a particle that reached a wall waits for the surface pass
    if (sp.wall && valid && st >= ST_LEFT && st <= ST_TOP)
        stage_put(sp.wq, &sp.cw->wall_count, &sp.cw->overflow, post, (unsigned long long)pid, w);
}

// one particle of k_push_scatter (before the claims)
__device__ __forceinline__ void scatter_round(PState &s, uint32_t pid, float w, bool valid,
                                              bool claim, bool &kept, bool &dep,
                                              const float2 *__restrict__ E, const PushConst &pc,
                                              const mcc::MccConst &mc, uint32_t step, int do_push,
                                              bool blk, int qs, uint32_t *se, uint32_t *sl,
                                              uint32_t *shole, const unsigned long long *lds,
                                              const Spawn &sp, uint32_t *__restrict__ lost6) {
    const PState pre = s;
    int ev = mcc::EV_NONE, st = -1;
    mcc::Child ch{};
    const bool done = collide_take(blk, qs, s, ev, ch, lds);
    if (valid) st = advance_one(s, pid, E, pc, mc, step, do_push, ev, ch, done);
    kept = st == ST_KEPT;
    dep = kept && deposit_ok(s, pc.N, pc.mode);
    if (valid && st != ST_KEPT && st != ST_HOLE) atomicAdd(&sl[st - 1], 1u);
    if (claim && !kept) atomicAdd(shole, 1u);
    if (sp.lost_ids && valid && st >= ST_LEFT && st <= ST_TOP) queue_lost(sp, pid, w);
    if (mc.on) {
        if (EV_KIND(ev) > 0) atomicAdd(&se[EV_KIND(ev)], 1u);
        if (ev & EV_OVER_BOUND) atomicAdd(&se[6], 1u);
    }
    stage_products(ev, ch, pre, st, valid, pid, E, pc, mc, step, sp, lost6, w, s);
}

// Pass 2 of the sort pass: the collide + push of IPP particles per thread,
// one claim (atomicSub on the bin count, which runs back to zero) per
// distinct key of the block, the deposit through one LDS window, the products
// staged.  The keys are the cells before the step, so the ranks and the
// claims come first and the claims' latency overlaps the collisions and the
// push.  A block of a sorted store ranks its particles in a direct LDS table
// over its narrow key range (up to SCAT_WIN keys); a block with a wider range
// (an unsorted store, or the particles appended since the last sort) ranks
// them in an LDS hash table and makes its claims before the collisions.  The
// slots a direct-table block claimed (survivors, and holes for the particles
// lost in this step) are staged in LDS in slot order (each key's claimed
// range contiguous) and written out by consecutive threads, so every store
// instruction covers consecutive slots; a wide block writes its particles
// directly.
//
// LDS: one arena serves three phases -- the rank table (8 KB) beside the
// collision queue (20 KB), or the hash table alone; then the deposit window
// (as many nodes as the arena holds, a 62 x 62 fallback window); then the
// write staging.  31 KB let five blocks share a CU, as the variants' 89-93
// VGPRs do (5 waves per SIMD).  Measured, 20 steps at 257^2 and 10 at 1025^2
// of the argon discharge: 5 waves 7.19 and 35.1 ms; collisionless variants at
// 6 in 25 KB 7.22 and 35.1; collisional ones at 4 7.20 and 35.4.
#define SCAT_WAVES 5
#define SCAT_ARENA 3900
template <int V>
constexpr int scat_arena_u64() {
    return V == PV_GENERIC ? 4096 : V == PV_COMPACT ? 3200 : SCAT_ARENA;
}
static_assert(SCAT_WIN + (11 * CQ_CAP * 4) / 8 <= 3200, "table + queue");
static_assert(8 * (256 * IPP / 2) * 4 <= 3200 * 8, "staging half");
static_assert(sizeof(BlockHash) <= 3200 * 8, "hash table");
#define PUSH_SCATTER_PARAMS                                                                   \
    SpView src, SpView dst, const uint32_t *__restrict__ nptr, uint32_t cap,                  \
        const float2 *__restrict__ E, PushConst pc, mcc::MccConst mc, uint32_t step,          \
        uint32_t *__restrict__ binCount, const uint32_t *__restrict__ binStart,               \
        unsigned long long *__restrict__ q, int do_push, int deposit, Spawn sp,               \
        unsigned long long *__restrict__ events, uint32_t *__restrict__ lost6,                \
        uint32_t *__restrict__ holes
#define PUSH_SCATTER_ARGS                                                                     \
    src, dst, nptr, cap, E, pc, mc, step, binCount, binStart, q, do_push, deposit, sp, events, \
        lost6, holes
template <int V>
__device__ __forceinline__ void push_scatter_body(PUSH_SCATTER_PARAMS) {
    pin_variant<V>(pc, mc, src);
    pin_spawn<V>(sp);
    if (V == PV_COMPACT) {
        dst.w = nullptr;
        do_push = deposit = 0;
    }
    if (blockIdx.x * (blockDim.x * IPP) >= *nptr) return;  // past the live count
    constexpr int ARENA = scat_arena_u64<V>();
    __shared__ unsigned long long arena[ARENA];
    __shared__ uint32_t se[8], sl[6], s_total, shole;
    uint32_t *tcnt = reinterpret_cast<uint32_t *>(arena);  // per key: count, then staging base
    uint32_t *tkey = tcnt + SCAT_WIN;                      // per key: slot of its rank 0
    unsigned long long *cq = arena + SCAT_WIN;             // collision queue behind the table
    if (threadIdx.x < 8) se[threadIdx.x] = 0;
    if (threadIdx.x < 6) sl[threadIdx.x] = 0;
    if (threadIdx.x == 0) s_total = shole = 0;
    __shared__ int wmin[4], wmax[4];
    const uint32_t n = *nptr;
    const uint32_t base = blockIdx.x * (blockDim.x * IPP) + threadIdx.x;
    const bool blk = mc.on && mc.mode == PIC_DEV_MODE_PHYS;
    PState s[IPP];
    uint32_t pid[IPP], ent[IPP], rank[IPP];
    float w[IPP];
    bool claim[IPP], kept[IPP], dep[IPP];
    int kmin = 0x7FFFFFFF, kmax = -1;
#pragma unroll
    for (int r = 0; r < IPP; r++) {  // every load first
        const uint32_t i = base + r * blockDim.x;
        s[r] = PState{};
        pid[r] = 0u;
        w[r] = 1.0f;
        if (i < n) {
            s[r] = load_state(src, i, true);
            pid[r] = src.id[i];
            w[r] = load_w(src, i);
        }
        // the slot k_key_count counted, keyed by the cell before the step
        // (without a push nothing moves: the particles inside keep slots)
        claim[r] = i < n && s[r].jx != CELL_HOLE &&
                   (do_push || classify(s[r], pc.N, pc.mode) == ST_KEPT);
        ent[r] = claim[r] ? bin_key(s[r].jx, s[r].jy, pc.tilesX) >> pc.keyshift : 0u;
        if (claim[r]) {
            kmin = min(kmin, (int)ent[r]);
            kmax = max(kmax, (int)ent[r]);
        }
    }
    kmin = wave_min(kmin);
    kmax = wave_max(kmax);
    if ((threadIdx.x & 63) == 0) {
        wmin[threadIdx.x >> 6] = kmin;
        wmax[threadIdx.x >> 6] = kmax;
    }
    // the electrons' null-collision bounds in LDS (loaded beside the state)
    __shared__ float2 sbins[MCC_BINS];
    if (mc.bins && threadIdx.x < MCC_BINS) sbins[threadIdx.x] = mc.bins[threadIdx.x];
    __syncthreads();  // counters cleared, key range known, bounds staged
    kmin = min(min(wmin[0], wmin[1]), min(wmin[2], wmin[3]));
    kmax = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
    const int span = kmax - kmin + 1;  // <= 0: no claims
    const bool direct = span <= SCAT_WIN;  // uniform over the block
    if (direct)
        for (int e = threadIdx.x; e < span; e += blockDim.x) tcnt[e] = 0u;
    __syncthreads();
    // table block: rank of each particle within its key; wide block: one
    // claim per particle, its slot start(k) + old - 1 (old = 0 on a corrupt
    // histogram gives a slot >= cap, which is skipped)
    uint32_t slot[IPP];
#pragma unroll
    for (int r = 0; r < IPP; r++) {
        rank[r] = 0u;
        slot[r] = 0xFFFFFFFFu;
        if (direct) {
            ent[r] -= (uint32_t)kmin;
            if (claim[r]) rank[r] = atomicAdd(&tcnt[ent[r]], 1u);
        }
    }
    if (!direct) {
        // wide block: ranks in the LDS hash table, one claim per distinct
        // key, and every slot known before the collision queue takes the
        // LDS (the claims' latency is not hidden: such blocks are few once
        // the store has been sorted)
        BlockHash &H = *reinterpret_cast<BlockHash *>(arena);
        hash_clear(H);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < IPP; r++) ent[r] = hash_insert(H, ent[r], claim[r], rank[r]);
        __syncthreads();
        constexpr int EPT = HASH_SIZE / 256;
        uint32_t kk[EPT], cc[EPT], ho[EPT], hs[EPT];
#pragma unroll
        for (int j = 0; j < EPT; j++) {
            kk[j] = H.key[threadIdx.x + j * 256];
            cc[j] = H.cnt[threadIdx.x + j * 256];
        }
#pragma unroll
        for (int j = 0; j < EPT; j++) {
            ho[j] = hs[j] = 0u;
            if (kk[j] != HASH_EMPTY) {
                ho[j] = atomicSub(&binCount[(size_t)kk[j] * BIN_STRIDE], cc[j]);
                hs[j] = binStart[kk[j]];
            }
        }
#pragma unroll
        for (int j = 0; j < EPT; j++)
            if (kk[j] != HASH_EMPTY) H.key[threadIdx.x + j * 256] = hs[j] + ho[j] - cc[j];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < IPP; r++)
            if (claim[r]) slot[r] = H.key[ent[r]] + rank[r];
    }
    __syncthreads();
    // one claim per distinct key of a table block: the bin count runs down
    // from its total, so the block's c particles of key k take the slots
    // start(k) + old - c + rank, rank < c.  The claims are issued here and
    // their results used after the push.
    uint32_t old[SCAT_EPT], st0[SCAT_EPT];
#pragma unroll
    for (int j = 0; j < SCAT_EPT; j++) {
        const int e = threadIdx.x + j * 256;
        old[j] = st0[j] = 0u;
        if (direct && e < span) {
            const uint32_t c = tcnt[e];
            if (c) {
                old[j] = atomicSub(&binCount[(size_t)(kmin + e) * BIN_STRIDE], c);
                st0[j] = binStart[kmin + e];
            }
        }
    }
    int qs[IPP];
    if (blk) {
        bool act[IPP];
#pragma unroll
        for (int r = 0; r < IPP; r++) act[r] = base + r * blockDim.x < n && s[r].jx != CELL_HOLE;
        block_collide_n<IPP>(act, s, pid, mc, step, qs, cq, mc.bins ? sbins : nullptr);
    }
    // the rounds are spelled out so every array index is a compile-time constant
    scatter_round(s[0], pid[0], w[0], base + 0 * blockDim.x < n, claim[0], kept[0],
                  dep[0], E, pc, mc, step, do_push, blk, qs[0], se, sl, &shole, cq, sp, lost6);
    scatter_round(s[1], pid[1], w[1], base + 1 * blockDim.x < n, claim[1], kept[1],
                  dep[1], E, pc, mc, step, do_push, blk, qs[1], se, sl, &shole, cq, sp, lost6);
    scatter_round(s[2], pid[2], w[2], base + 2 * blockDim.x < n, claim[2], kept[2],
                  dep[2], E, pc, mc, step, do_push, blk, qs[2], se, sl, &shole, cq, sp, lost6);
    scatter_round(s[3], pid[3], w[3], base + 3 * blockDim.x < n, claim[3], kept[3],
                  dep[3], E, pc, mc, step, do_push, blk, qs[3], se, sl, &shole, cq, sp, lost6);
    __syncthreads();  // every round has read its collision result
    if (direct) {
#pragma unroll
        for (int j = 0; j < SCAT_EPT; j++) {
            const int e = threadIdx.x + j * 256;
            if (e < span) {
                const uint32_t c = tcnt[e];
                if (c) {
                    tkey[e] = st0[j] + old[j] - c;
                    tcnt[e] = atomicAdd(&s_total, c);
                }
            }
        }
    }
    __syncthreads();
    uint32_t lidx[IPP];
#pragma unroll
    for (int r = 0; r < IPP; r++) {
        lidx[r] = 0u;
        if (direct && claim[r]) {
            slot[r] = tkey[ent[r]] + rank[r];
            lidx[r] = tcnt[ent[r]] + rank[r];
        }
        // weighted stores stay direct
        if (dst.w && claim[r] && slot[r] < cap) dst.w[slot[r]] = w[r];
    }
    __syncthreads();  // the table is read; the deposit window reuses the LDS
    if (deposit) block_deposit_n<IPP, ARENA>(dep, s, w, q, pc.N, arena);
    __syncthreads();
    if (direct) {
        // the claimed slots staged in slot order, half of the block's at a
        // time (a claimed slot of a particle that left holds a hole)
        uint32_t *stg = reinterpret_cast<uint32_t *>(arena);  // 8 words x SH, SoA
        constexpr uint32_t SH = 256 * IPP / 2;
        const uint32_t tot = s_total;
        for (uint32_t lo = 0; lo < tot; lo += SH) {  // uniform: tot is the block's
#pragma unroll
            for (int r = 0; r < IPP; r++) {
                if (claim[r] && lidx[r] >= lo && lidx[r] < lo + SH) {
                    const uint32_t l = lidx[r] - lo;
                    stg[l] = slot[r];
                    stg[SH + l] =
                        kept[r] ? cell_pack(s[r].jx, s[r].jy) : cell_pack(CELL_HOLE, CELL_HOLE);
                    stg[2 * SH + l] = __float_as_uint(s[r].ox);
                    stg[3 * SH + l] = __float_as_uint(s[r].oy);
                    stg[4 * SH + l] = __float_as_uint(s[r].vx);
                    stg[5 * SH + l] = __float_as_uint(s[r].vy);
                    stg[6 * SH + l] = __float_as_uint(s[r].vz);
                    stg[7 * SH + l] = pid[r];
                }
            }
            __syncthreads();
            const uint32_t m = min(SH, tot - lo);
            for (uint32_t l = threadIdx.x; l < m; l += blockDim.x) {
                const uint32_t sl = stg[l];
                if (sl < cap) {
                    dst.cell[sl] = stg[SH + l];
                    dst.ox[sl] = __uint_as_float(stg[2 * SH + l]);
                    dst.oy[sl] = __uint_as_float(stg[3 * SH + l]);
                    dst.vx[sl] = __uint_as_float(stg[4 * SH + l]);
                    dst.vy[sl] = __uint_as_float(stg[5 * SH + l]);
                    dst.vz[sl] = __uint_as_float(stg[6 * SH + l]);
                    dst.id[sl] = stg[7 * SH + l];
                }
            }
            __syncthreads();  // the half is written out before the next fills it
        }
    } else {
#pragma unroll
        for (int r = 0; r < IPP; r++) {
            if (claim[r] && slot[r] < cap) {
                PState o = s[r];
                if (!kept[r]) o.jx = o.jy = CELL_HOLE;
                store_state(dst, slot[r], o, pid[r]);
            }
        }
    }
    if (mc.on) {
        if (threadIdx.x < 8 && se[threadIdx.x])
            atomicAdd(&events[cnt_slot() * 8 + threadIdx.x], (unsigned long long)se[threadIdx.x]);
    }
    if (threadIdx.x < 6 && sl[threadIdx.x])
        atomicAdd(&lost6[cnt_slot() * 6 + threadIdx.x], sl[threadIdx.x]);
    if (threadIdx.x == 0 && shole) atomicAdd(&holes[cnt_slot()], shole);
}

// ---- the passes with pinned options (physical mode, no magnetic field)

// A copy of the collision constants the compiler takes for new: expressions of
// them are then evaluated where they are used.  (Hoisted out of the queue's
// loop they are uniform floats in some 40 VGPRs, held across it.)
__device__ __forceinline__ mcc::MccConst fresh(mcc::MccConst c) {
    asm volatile("" : "+s"(c.mass), "+s"(c.M), "+s"(c.q), "+s"(c.ng), "+s"(c.opal_B), "+s"(c.vtn));
    asm volatile("" : "+s"(c.e_exc), "+s"(c.e_iz), "+s"(c.kev_amu_div), "+s"(c.nu_max), "+s"(c.gas));
    return c;
}

// mcc's block-level collisions on the pinned passes (COLL_E, COLL_I): the
// candidates of the block's P x 256 particles are queued in LDS and collide
// on dense lanes; vx and vy (and vz: VZ_BACK) come back to the particles'
// lanes, everything else -- vz into the store, the event counts, the products of an ionisation -- is
// settled by the lane that made the collision, so none of it takes code or
// registers in the particles' rounds.  The queue holds every particle of the
// block (5 words each): it cannot overflow.  Without VZ_IN (no energy bins, tab
// null: the bound does not depend on the speed) only candidates' vz is read.  q: free on entry and again after
// the next barrier.  The store's words of the block are not yet overwritten.
#define CQ_WORDS 5
template <int P, bool VZ_IN, bool VZ_BACK>
__device__ __forceinline__ void collide_queue(const bool (&live)[P], float (&vx)[P],
                                              float (&vy)[P], float (&vz)[P],
                                              const uint32_t (&id)[P], const SpView &sp,
                                              uint32_t blk0, const float2 *__restrict__ E,
                                              const PushConst &pc, const mcc::MccConst &mc0,
                                              uint32_t step, const Spawn &spn,
                                              uint32_t *__restrict__ lost6, uint32_t *se,
                                              const float2 *tab, float *q) {
    constexpr uint32_t CAP = P * 256;
    __shared__ uint32_t wcnt[4];
    uint32_t *qu = reinterpret_cast<uint32_t *>(q);  // v (3), id, slot
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    uint32_t pos[P], wtot = 0;
#pragma unroll
    for (int r = 0; r < P; r++) {
        const float v2 = VZ_IN ? vx[r] * vx[r] + vy[r] * vy[r] + vz[r] * vz[r] : 0.0f;
        const bool cand = live[r] && mcc::candidate(mc0, id[r], step, v2, tab);
        const uint64_t bal = __ballot(cand);
        pos[r] = cand ? wtot + (uint32_t)__popcll(bal & below) : 0xFFFFFFFFu;
        wtot += (uint32_t)__popcll(bal);
    }
    if (lane == 0) wcnt[w] = wtot;
    __syncthreads();
    uint32_t base = 0, total = 0;
    for (int k = 0; k < 4; k++) {
        if (k < w) base += wcnt[k];
        total += wcnt[k];
    }
    if (total == 0) return;  // uniform
#pragma unroll
    for (int r = 0; r < P; r++) {
        if (pos[r] != 0xFFFFFFFFu) {
            const uint32_t t = pos[r] += base;
            q[t] = vx[r];
            q[CAP + t] = vy[r];
            if (VZ_IN) q[2 * CAP + t] = vz[r];
            qu[3 * CAP + t] = id[r];
            qu[4 * CAP + t] = blk0 + threadIdx.x + r * 256;
        }
    }
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < total; t += 256) {
        const mcc::MccConst mc = fresh(mc0);
        const uint32_t pid = qu[3 * CAP + t], i = qu[4 * CAP + t];
        float ux = q[t], uy = q[CAP + t], uz = VZ_IN ? q[2 * CAP + t] : sp.vz[i];
        mcc::Child ch{};
        const int ev = mc.electron
                           ? mcc::collide_electron<true>(mc, ux, uy, uz, pid, step, true, ch, tab)
                           : mcc::collide_ion<true>(mc, ux, uy, uz, pid, step);
        q[t] = ux;
        q[CAP + t] = uy;
        if (VZ_BACK)
            q[2 * CAP + t] = uz;
        else
            sp.vz[i] = uz;
        if (EV_KIND(ev) > 0) atomicAdd(&se[EV_KIND(ev)], 1u);
        if (ev & EV_OVER_BOUND) atomicAdd(&se[6], 1u);
        if (EV_KIND(ev) == mcc::EV_IONIZE)
            stage_ionisation(ch, load_state(sp, i, false), pid, E, pc, spn, lost6, load_w(sp, i));
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < P; r++)
        if (pos[r] != 0xFFFFFFFFu) {
            vx[r] = q[pos[r]];
            vy[r] = q[CAP + pos[r]];
            if (VZ_BACK) vz[r] = q[2 * CAP + pos[r]];
        }
}

// gather_one's field of G particles, every load issued before the first is
// used; a particle that cannot move (ok false) reads node 0
template <int G>
__device__ __forceinline__ void gather_field(const PState (&s)[G], const bool (&ok)[G],
                                           const float2 *__restrict__ E, int N, float (&ex)[G],
                                           float (&ey)[G]) {
    float2 e00[G], e01[G], e10[G], e11[G];
#pragma unroll
    for (int r = 0; r < G; r++) {
        const uint32_t b = ok[r] ? (uint32_t)(s[r].jy * N + s[r].jx) : 0u;
        const float2 *lo = E + b, *hi = E + (b + (uint32_t)N);
        e00[r] = lo[0];
        e01[r] = lo[1];
        e10[r] = hi[0];
        e11[r] = hi[1];
    }
#pragma unroll
    for (int r = 0; r < G; r++) {
        const float wj = s[r].ox, wk = s[r].oy;
        const float a4 = (1.0f - wj) * (1.0f - wk), a3 = wj * (1.0f - wk);
        const float a2 = wk * (1.0f - wj), a1 = wj * wk;
        ex[r] = a4 * e00[r].x + a3 * e01[r].x + a2 * e10[r].x + a1 * e11[r].x;
        ey[r] = a4 * e00[r].y + a3 * e01[r].y + a2 * e10[r].y + a1 * e11[r].y;
    }
}

// reposition without branches
__device__ __forceinline__ void reposition_sel(int j, float t, int &jn, float &on) {
    const float k0 = floorf(t), f0 = t - k0;
    const bool up = f0 >= 1.0f;  // t just below an integer: t - k rounded up to 1
    const int jj = min(max(j + (int)(up ? k0 + 1.0f : k0), -CELL_FAR), CELL_FAR);
    const bool in = t > -POS_GUARD && t < POS_GUARD;  // false for NaN
    jn = in ? jj : (t > 0.0f ? CELL_FAR : -CELL_FAR);
    on = (in && !up) ? f0 : 0.0f;
}

// move_one without a magnetic field; ok false: unchanged
__device__ __forceinline__ void move_sel(PState &s, bool ok, float ex, float ey,
                                         const PushConst &pc) {
    float ux = s.vx + pc.cE * ex, uy = s.vy + pc.cE * ey;
    ux = ux + pc.cE * ex;
    uy = uy + pc.cE * ey;
    int jx, jy;
    float ox, oy;
    reposition_sel(s.jx, s.ox + ux * pc.dtdx, jx, ox);
    reposition_sel(s.jy, s.oy + uy * pc.dtdy, jy, oy);
    s.jx = ok ? jx : s.jx;
    s.jy = ok ? jy : s.jy;
    s.ox = ok ? ox : s.ox;
    s.oy = ok ? oy : s.oy;
    s.vx = ok ? ux : s.vx;
    s.vy = ok ? uy : s.vy;
}

__device__ __forceinline__ bool inside_cells(const PState &s, int N) {
    return (unsigned)s.jx <= (unsigned)(N - 2) && (unsigned)s.jy <= (unsigned)(N - 2);
}

// The sort pass's pinned variants, with the push: push_scatter_body's plan in
// push_inplace_body's form (every load first, field loads of two particles at
// a time, straight-line rounds, collisions settled on the queue's lanes).
// Bound by the scattered writes (1025^2, a sort every 3rd pass: 5.5 GB written
// for 2.9 GB of particles, runs of about 16 particles per tile) and the flush
// atomics; 2.93 -> 2.57 ms at 104.9 M electrons over the one-particle rounds.
template <int V>
__device__ __forceinline__ void push_scatter_fast(PUSH_SCATTER_PARAMS) {
    pin_variant<V>(pc, mc, src);
    pin_spawn<V>(sp);
    constexpr bool COLL = pv_coll_e(V) || pv_coll_i(V), WGT = pv_weighted(V);
    const uint32_t n = *nptr, blk0 = blockIdx.x * (256 * IPP);
    if (blk0 >= n) return;  // past the live count
    constexpr int ARENA = scat_arena_u64<V>();
    __shared__ unsigned long long arena[ARENA];
    __shared__ uint32_t se[8], sl[6], s_total, shole;
    __shared__ int wmin[4], wmax[4];
    __shared__ float2 sbins[MCC_BINS];
    uint32_t *tcnt = reinterpret_cast<uint32_t *>(arena);  // per key: count, then staging base
    uint32_t *tkey = tcnt + SCAT_WIN;                      // per key: slot of its rank 0
    float *cq = reinterpret_cast<float *>(arena + SCAT_WIN);  // collision queue behind the table
    static_assert(!COLL || SCAT_WIN + CQ_WORDS * IPP * 256 / 2 <= ARENA, "table + queue");
    const uint32_t tid = threadIdx.x;
    if (tid < 8) se[tid] = 0;
    if (tid < 6) sl[tid] = 0;
    if (tid == 0) s_total = shole = 0;
    uint32_t c0[IPP], pid[IPP];
    float ox[IPP], oy[IPP], vx[IPP], vy[IPP], vz[IPP], w[IPP];
    {
        const uint32_t *pc_ = src.cell + blk0, *pi = src.id + blk0;
        const float *px = src.ox + blk0, *py = src.oy + blk0, *pu = src.vx + blk0,
                    *pv = src.vy + blk0, *pz = src.vz + blk0;
#pragma unroll
        for (int r = 0; r < IPP; r++) {  // every load first
            c0[r] = pc_[tid + r * 256];
            pid[r] = pi[tid + r * 256];
            vx[r] = pu[tid + r * 256];
            vy[r] = pv[tid + r * 256];
            vz[r] = pz[tid + r * 256];
            ox[r] = px[tid + r * 256];
            oy[r] = py[tid + r * 256];
            w[r] = WGT ? src.w[blk0 + tid + r * 256] : 1.0f;
        }
    }
    if (COLL && mc.bins && tid < MCC_BINS) sbins[tid] = mc.bins[tid];
    bool claim[IPP];  // the slots k_key_count counted, keyed by the cell before the step
    uint32_t ent[IPP], rank[IPP];
    int kmin = 0x7FFFFFFF, kmax = -1;
#pragma unroll
    for (int r = 0; r < IPP; r++) {
        const int jx = cell_jx(c0[r]);
        claim[r] = blk0 + tid + r * 256 < n && jx != CELL_HOLE;
        ent[r] = bin_key(jx, cell_jy(c0[r]), pc.tilesX) >> pc.keyshift;
        kmin = min(kmin, claim[r] ? (int)ent[r] : 0x7FFFFFFF);
        kmax = max(kmax, claim[r] ? (int)ent[r] : -1);
    }
    kmin = wave_min(kmin);
    kmax = wave_max(kmax);
    if ((tid & 63) == 0) {
        wmin[tid >> 6] = kmin;
        wmax[tid >> 6] = kmax;
    }
    __syncthreads();  // counters cleared, key range known, bounds staged
    kmin = min(min(wmin[0], wmin[1]), min(wmin[2], wmin[3]));
    kmax = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
    const int span = kmax - kmin + 1;      // <= 0: no claims
    const bool direct = span <= SCAT_WIN;  // uniform over the block
    // `late`: each of the first threads holds one key's claim in flight over
    // the collisions and the push; a wider table claims at once
    const bool late = span <= 256;
    uint32_t cnt0 = 0u, old0 = 0u, st0 = 0u;
    if (direct) {
        for (int e = tid; e < span; e += 256) tcnt[e] = 0u;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < IPP; r++) {
            ent[r] -= (uint32_t)kmin;
            rank[r] = 0u;
            if (claim[r]) rank[r] = atomicAdd(&tcnt[ent[r]], 1u);
        }
        __syncthreads();
        // one claim per distinct key: the bin count runs down from its total,
        // so the block's c particles of key k take the slots start(k) + old -
        // c + rank, rank < c
        for (int e = tid; e < span; e += 256) {
            const uint32_t c = tcnt[e];
            if (!c) continue;
            const uint32_t old = atomicSub(&binCount[(size_t)(kmin + e) * BIN_STRIDE], c);
            const uint32_t st = binStart[kmin + e];
            if (late) {
                cnt0 = c;
                old0 = old;
                st0 = st;
            } else {
                tkey[e] = st + old - c;
                tcnt[e] = atomicAdd(&s_total, c);
            }
        }
    } else {
        // wide block (an unsorted store, or the particles appended since the
        // last sort): ranks in the LDS hash table, one claim per distinct key,
        // every slot (in rank) known before the collision queue takes the LDS
        BlockHash &H = *reinterpret_cast<BlockHash *>(arena);
        hash_clear(H);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < IPP; r++) ent[r] = hash_insert(H, ent[r], claim[r], rank[r]);
        __syncthreads();
        for (int e = tid; e < HASH_SIZE; e += 256) {
            const uint32_t k = H.key[e], c = H.cnt[e];
            if (k != HASH_EMPTY)
                H.key[e] = binStart[k] + atomicSub(&binCount[(size_t)k * BIN_STRIDE], c) - c;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < IPP; r++)
            if (claim[r]) rank[r] += H.key[ent[r]];
        __syncthreads();
    }
    if (COLL)
        collide_queue<IPP, true, true>(claim, vx, vy, vz, pid, src, blk0, E, pc, mc, step, sp, lost6, se,
                                 mc.bins ? sbins : nullptr, cq);
    PState s[IPP];
    bool kept[IPP];
#pragma unroll
    for (int h = 0; h < IPP; h += 2) {
        PState t[2];
        bool ok[2];
        float ex[2], ey[2];
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const int r = h + g;
            t[g] = PState{cell_jx(c0[r]), cell_jy(c0[r]), ox[r], oy[r], vx[r], vy[r], vz[r]};
            ok[g] = claim[r] && inside_cells(t[g], pc.N);
        }
        gather_field<2>(t, ok, E, pc.N, ex, ey);
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const int r = h + g;
            s[r] = t[g];
            move_sel(s[r], ok[g], ex[g], ey[g], pc);
            kept[r] = claim[r] && inside_cells(s[r], pc.N);
            if (claim[r] && !kept[r]) {
                const int st = classify(s[r], pc.N, pc.mode);
                atomicAdd(&sl[st - 1], 1u);
                atomicAdd(&shole, 1u);
                // (an uploaded CELL_DEAD particle has reached no wall; the
                // first pass after an upload sorts, so no in-place pass meets one)
                if (sp.lost_ids && st <= ST_TOP) queue_lost(sp, pid[r], w[r]);
                if (sp.wall && st <= ST_TOP)  // waits for the surface pass
                    stage_put(sp.wq, &sp.cw->wall_count, &sp.cw->overflow, s[r],
                              (unsigned long long)pid[r], w[r]);
            }
        }
    }
    if (direct) {
        if (late && cnt0) {
            tkey[tid] = st0 + old0 - cnt0;
            tcnt[tid] = atomicAdd(&s_total, cnt0);
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < IPP; r++) {  // the slot, and the place in slot order
            const uint32_t e = claim[r] ? ent[r] : 0u;
            ent[r] = tcnt[e] + rank[r];
            rank[r] = tkey[e] + rank[r];
        }
    }
    __syncthreads();  // the table is read; the deposit window reuses the LDS
    if (deposit) block_deposit_n<IPP, ARENA>(kept, s, w, q, pc.N, arena);
    __syncthreads();
    if (direct) {
        // the claimed slots staged in slot order, SH at a time (a claimed
        // slot of a particle that left holds a hole)
        constexpr uint32_t SW = WGT ? 9 : 8;  // words of a slot, SoA
        constexpr uint32_t SH = 2 * ARENA / SW < 256 * IPP ? 2 * ARENA / SW : 256 * IPP;
        uint32_t *stg = reinterpret_cast<uint32_t *>(arena);
        const uint32_t tot = s_total;
        for (uint32_t lo = 0; lo < tot; lo += SH) {  // uniform: tot is the block's
#pragma unroll
            for (int r = 0; r < IPP; r++) {
                const uint32_t l = ent[r] - lo;
                if (claim[r] && l < SH) {
                    stg[l] = rank[r];
                    stg[SH + l] =
                        kept[r] ? cell_pack(s[r].jx, s[r].jy) : cell_pack(CELL_HOLE, CELL_HOLE);
                    stg[2 * SH + l] = __float_as_uint(s[r].ox);
                    stg[3 * SH + l] = __float_as_uint(s[r].oy);
                    stg[4 * SH + l] = __float_as_uint(s[r].vx);
                    stg[5 * SH + l] = __float_as_uint(s[r].vy);
                    stg[6 * SH + l] = __float_as_uint(s[r].vz);
                    stg[7 * SH + l] = pid[r];
                    if (WGT) stg[8 * SH + l] = __float_as_uint(w[r]);
                }
            }
            __syncthreads();
            const uint32_t m = min(SH, tot - lo);
            for (uint32_t l = tid; l < m; l += 256) {
                const uint32_t d = stg[l];
                if (d < cap) {
                    dst.cell[d] = stg[SH + l];
                    dst.ox[d] = __uint_as_float(stg[2 * SH + l]);
                    dst.oy[d] = __uint_as_float(stg[3 * SH + l]);
                    dst.vx[d] = __uint_as_float(stg[4 * SH + l]);
                    dst.vy[d] = __uint_as_float(stg[5 * SH + l]);
                    dst.vz[d] = __uint_as_float(stg[6 * SH + l]);
                    dst.id[d] = stg[7 * SH + l];
                    if (WGT) dst.w[d] = __uint_as_float(stg[8 * SH + l]);
                }
            }
            __syncthreads();  // written out before the next part fills it
        }
    } else {
#pragma unroll
        for (int r = 0; r < IPP; r++)
            if (claim[r] && rank[r] < cap) {
                PState o = s[r];
                if (!kept[r]) o.jx = o.jy = CELL_HOLE;
                store_state(dst, rank[r], o, pid[r]);
                if (WGT) dst.w[rank[r]] = w[r];
            }
    }
    if (COLL && tid < 8 && se[tid])
        atomicAdd(&events[cnt_slot() * 8 + tid], (unsigned long long)se[tid]);
    if (tid < 6 && sl[tid]) atomicAdd(&lost6[cnt_slot() * 6 + tid], sl[tid]);
    if (tid == 0 && shole) atomicAdd(&holes[cnt_slot()], shole);
}

template <int V>
__global__ void __launch_bounds__(256) k_push_scatter(PUSH_SCATTER_PARAMS) {
    push_scatter_body<V>(PUSH_SCATTER_ARGS);
}
#define SCATTER_FAST(V)                                                        \
    template <>                                                                \
    __global__ void __launch_bounds__(256)                                     \
        __attribute__((amdgpu_waves_per_eu(SCAT_WAVES, SCAT_WAVES)))           \
        k_push_scatter<V>(PUSH_SCATTER_PARAMS) {                               \
        push_scatter_fast<V>(PUSH_SCATTER_ARGS);                               \
    }
SCATTER_FAST(PV_PLAIN)
SCATTER_FAST(PV_SPAWN)
SCATTER_FAST(PV_COLL_E)
SCATTER_FAST(PV_COLL_I)
SCATTER_FAST((PV_PLAIN | PV_W))
SCATTER_FAST((PV_SPAWN | PV_W))
SCATTER_FAST((PV_COLL_E | PV_W))
SCATTER_FAST((PV_COLL_I | PV_W))

// one particle of the generic k_push_inplace: collide (block-wide when blk), push, store
// in place or leave a hole, count, stage products; dep = deposit it
__device__ __forceinline__ void inplace_round(const SpView &sp, uint32_t i, uint32_t n, PState &s,
                                              uint32_t pid, bool live, bool &dep, bool &kept_out,
                                              const float2 *__restrict__ E, const PushConst &pc,
                                              const mcc::MccConst &mc, uint32_t step,
                                              const Spawn &spn, uint32_t *__restrict__ lost6,
                                              bool need_vz, bool blk, int qs, uint32_t *sl,
                                              uint32_t *shole, uint32_t *se,
                                              const unsigned long long *lds, float w) {
    const PState pre = s;
    int ev = mcc::EV_NONE;
    mcc::Child ch{};
    const bool done = collide_take(blk, qs, s, ev, ch, lds);
    int st = ST_HOLE;
    if (live) st = advance_one(s, pid, E, pc, mc, step, 1, ev, ch, done);
    const bool kept = (st == ST_KEPT);
    kept_out = kept;
    dep = kept && deposit_ok(s, pc.N, pc.mode);
    if (kept) {
        // the slot holds this particle's previous state: a word whose bits
        // did not change (the cell of a particle that stayed in its cell, vz
        // without a collision or rotation) is not written again, and a
        // wavefront with no changed lane issues no store
        const uint32_t c1 = cell_pack(s.jx, s.jy);
        if (c1 != cell_pack(pre.jx, pre.jy)) sp.cell[i] = c1;
        sp.ox[i] = s.ox;
        sp.oy[i] = s.oy;
        sp.vx[i] = s.vx;
        sp.vy[i] = s.vy;
        if (need_vz && __float_as_uint(s.vz) != __float_as_uint(pre.vz)) sp.vz[i] = s.vz;
    } else if (live) {
        sp.cell[i] = cell_pack(CELL_HOLE, CELL_HOLE);
        atomicAdd(&sl[st - 1], 1u);
        atomicAdd(shole, 1u);
        // the id is read only here: a pass that needs it for nothing else
        // does not load it for every particle
        if (spn.lost_ids && st >= ST_LEFT && st <= ST_TOP) queue_lost(spn, sp.id[i], w);
    }
    if (mc.on) {
        if (EV_KIND(ev) > 0) atomicAdd(&se[EV_KIND(ev)], 1u);
        if (ev & EV_OVER_BOUND) atomicAdd(&se[6], 1u);
    }
    stage_products(ev, ch, pre, st, i < n, pid, E, pc, mc, step, spn, lost6, w, s);
}

// The in-place pass with every option taken at run time (push_inplace_body's
// comment says what an in-place pass is).
template <int P>
__device__ __forceinline__ void push_inplace_generic(
    SpView sp, const uint32_t *__restrict__ nptr, const float2 *__restrict__ E, PushConst pc,
    mcc::MccConst mc, uint32_t step, unsigned long long *__restrict__ q, int deposit, Spawn spn,
    unsigned long long *__restrict__ events, uint32_t *__restrict__ lost6,
    uint32_t *__restrict__ holes, uint32_t *__restrict__ hist, uint32_t bid) {
    const uint32_t n = *nptr;
    // the grid covers the capacity: blocks past the live count leave at once
    // (uniformly, before any barrier); bid: this block's index in the species
    if (bid * (blockDim.x * P) >= n) return;
    __shared__ uint32_t sl[6];
    __shared__ uint32_t shole;
    __shared__ uint32_t se[8];
    constexpr int LDS_U64 = BLOCK_LDS_U64;
    __shared__ unsigned long long lds[LDS_U64];
    if (threadIdx.x < 6) sl[threadIdx.x] = 0;
    if (threadIdx.x < 8) se[threadIdx.x] = 0;
    if (threadIdx.x == 0) shole = 0;
    const uint32_t base = bid * (blockDim.x * P) + threadIdx.x;
    // vz and the id are read only where something uses them: the magnetic
    // rotation, collisions, re-injection keyed by the id, and the wall
    // queue (surface physics needs the full velocity and the id's draws)
    const bool need_vz = pc.bfield != 0 || mc.on || spn.wall;
    const bool need_id = mc.on || spn.plop || spn.wall;
    const bool blk = mc.on && mc.mode == PIC_DEV_MODE_PHYS;
    PState s[P];
    uint32_t pid[P];
    bool live[P];
    float w[P];
#pragma unroll
    for (int r = 0; r < P; r++) {  // every load first
        const uint32_t i = base + r * blockDim.x;
        s[r] = PState{};
        pid[r] = 0u;
        live[r] = false;
        w[r] = 1.0f;
        if (i < n) {
            s[r] = load_state(sp, i, need_vz);
            live[r] = s[r].jx != CELL_HOLE;
            if (live[r] && need_id) pid[r] = sp.id[i];
            if (live[r]) w[r] = load_w(sp, i);
        }
    }
    // the electrons' null-collision bounds in LDS (loaded beside the state)
    __shared__ float2 sbins[MCC_BINS];
    if (blk && mc.bins && threadIdx.x < MCC_BINS) sbins[threadIdx.x] = mc.bins[threadIdx.x];
    __syncthreads();  // counters initialised, bounds staged
    int qs[P];
    if (blk) block_collide_n<P>(live, s, pid, mc, step, qs, lds, mc.bins ? sbins : nullptr);
    bool dep[P], kept[P];
#pragma unroll
    for (int r = 0; r < P; r++)
        inplace_round(sp, base + r * blockDim.x, n, s[r], pid[r], live[r], dep[r], kept[r], E, pc,
                      mc, step, spn, lost6, need_vz, blk, qs[r], sl, &shole, se, lds, w[r]);
    // block_deposit_n passes a barrier before it writes the window, so every
    // round has read its collision result from the shared LDS by then
    if (deposit) block_deposit_n<P, LDS_U64>(dep, s, w, q, pc.N, lds);
    __syncthreads();
    // ahead of a sort pass: the histogram of the cells the particles end the
    // step in, the keys that pass claims by (no k_key_count then)
    if (hist) {
        uint32_t key[P];
#pragma unroll
        for (int r = 0; r < P; r++)
            key[r] = kept[r] ? bin_key(s[r].jx, s[r].jy, pc.tilesX) >> pc.keyshift : 0u;
        block_key_hist<P>(kept, key, hist, reinterpret_cast<uint32_t *>(lds));
    }
    if (threadIdx.x < 6 && sl[threadIdx.x])
        atomicAdd(&lost6[cnt_slot() * 6 + threadIdx.x], sl[threadIdx.x]);
    if (threadIdx.x < 8 && se[threadIdx.x])
        atomicAdd(&events[cnt_slot() * 8 + threadIdx.x], (unsigned long long)se[threadIdx.x]);
    if (threadIdx.x == 0 && shole) atomicAdd(&holes[cnt_slot()], shole);
}

// LDS of an in-place pass (u64 words): the collision queue, then the deposit
// window, then the sort histogram (which needs 16 KB).  The electrons'
// collisional variant takes a 58 x 58 fallback window (28 KB, five blocks per
// CU) for particles that moved up to three steps since their store was
// sorted.
template <int V>
constexpr int inplace_lds_u64() {
    return pv_coll_e(V) ? 3584 : pv_coll_i(V) ? 2560 : BLOCK_LDS_U64;
}

// In-place timestep of one species between sort passes: the same collide +
// push as the sort pass, the state written back to its own slot, the
// deposit through one LDS window per block.  A particle that leaves (or that
// a collision removes) becomes a hole; the next sort pass compacts the store.
// Each thread handles P particles (strided by the block size, so every
// load and store stays coalesced): one deposit window and one flush of the
// block's counters then serve 256 * P particles.  Reads 20-28 B and writes
// 20-24 B per particle, with no histogram or slot claims.
//
// Bound by HBM (257^2, 13.1 M particles: 129 us the ions, 149 us the
// electrons, against 122 us for a copy of their 48 B) and by VALU issue about
// equally.  The loads of all four particles are issued before the first is
// decoded (the arrays are padded to whole blocks: no bounds test before a
// load), the field loads of two at a time, and the rounds are straight-line
// selects: only particles that leave take a branch, and the collisions'
// products are settled on the queue's lanes.  Before, each particle waited
// for its own cell and then its own field loads, and the collision code was
// inlined once more in every round (queue overflow): 269 VALU instructions
// per ion and 374 per electron instead of 196 and 261, 158 and 210 us.
template <int V, int P>
__device__ __forceinline__ void push_inplace_body(
    SpView sp, const uint32_t *__restrict__ nptr, const float2 *__restrict__ E, PushConst pc,
    mcc::MccConst mc, uint32_t step, unsigned long long *__restrict__ q, int deposit, Spawn spn,
    unsigned long long *__restrict__ events, uint32_t *__restrict__ lost6,
    uint32_t *__restrict__ holes, uint32_t *__restrict__ hist, uint32_t bid) {
    pin_variant<V>(pc, mc, sp);
    pin_spawn<V>(spn);
    constexpr bool COLL = pv_coll_e(V) || pv_coll_i(V), WGT = pv_weighted(V);
    const uint32_t n = *nptr, blk0 = bid * (256 * P);
    // the grid covers the capacity: blocks past the live count leave at once
    // (uniformly, before any barrier); bid: this block's index in the species
    if (blk0 >= n) return;
    __shared__ uint32_t sl[6];
    __shared__ uint32_t shole;
    __shared__ uint32_t se[8];
    constexpr int LDS_U64 = inplace_lds_u64<V>();
    __shared__ unsigned long long lds[LDS_U64];
    static_assert(!COLL || CQ_WORDS * P * 256 * 4 <= LDS_U64 * 8, "collision queue size");
    const uint32_t tid = threadIdx.x;
    if (tid < 6) sl[tid] = 0;
    if (tid < 8) se[tid] = 0;
    if (tid == 0) shole = 0;
    uint32_t c0[P], pid[P];
    float ox[P], oy[P], vx[P], vy[P], vz[P], w[P];
    {
        const uint32_t *pc_ = sp.cell + blk0, *pi = sp.id + blk0;
        const float *px = sp.ox + blk0, *py = sp.oy + blk0, *pu = sp.vx + blk0,
                    *pv = sp.vy + blk0, *pz = sp.vz + blk0;
#pragma unroll
        for (int r = 0; r < P; r++) {  // every load first
            c0[r] = pc_[tid + r * 256];
            if (COLL) pid[r] = pi[tid + r * 256];
            vx[r] = pu[tid + r * 256];
            vy[r] = pv[tid + r * 256];
            if (pv_coll_e(V)) vz[r] = pz[tid + r * 256];
            ox[r] = px[tid + r * 256];
            oy[r] = py[tid + r * 256];
            w[r] = WGT ? sp.w[blk0 + tid + r * 256] : 1.0f;
        }
    }
    // the electrons' null-collision bounds in LDS (loaded beside the state)
    __shared__ float2 sbins[MCC_BINS];
    if (pv_coll_e(V) && mc.bins && tid < MCC_BINS) sbins[tid] = mc.bins[tid];
    bool live[P];
#pragma unroll
    for (int r = 0; r < P; r++) {
        live[r] = blk0 + tid + r * 256 < n && cell_jx(c0[r]) != CELL_HOLE;
    }
    __syncthreads();  // counters initialised, bounds staged
    if (COLL)
        collide_queue<P, pv_coll_e(V), false>(live, vx, vy, vz, pid, sp, blk0, E, pc, mc, step,
                                                spn, lost6, se,
                                                pv_coll_e(V) && mc.bins ? sbins : nullptr,
                                                reinterpret_cast<float *>(lds));
    PState s[P];
    bool dep[P];
    uint32_t *pc_ = sp.cell + blk0;
    float *px = sp.ox + blk0, *py = sp.oy + blk0, *pu = sp.vx + blk0, *pv = sp.vy + blk0;
    constexpr int G = P > 1 ? 2 : 1;
#pragma unroll
    for (int h = 0; h < P; h += G) {  // the field loads of two particles at a time
        PState t[G];
        bool ok[G];
        float ex[G], ey[G];
#pragma unroll
        for (int g = 0; g < G; g++) {
            const int r = h + g;
            t[g] = PState{cell_jx(c0[r]), cell_jy(c0[r]), ox[r], oy[r], vx[r], vy[r], 0.0f};
            ok[g] = live[r] && inside_cells(t[g], pc.N);
        }
        gather_field<G>(t, ok, E, pc.N, ex, ey);
#pragma unroll
        for (int g = 0; g < G; g++) {
            const int r = h + g;
            s[r] = t[g];
            move_sel(s[r], ok[g], ex[g], ey[g], pc);
            dep[r] = live[r] && inside_cells(s[r], pc.N);
            if (dep[r]) {
                // a word whose bits did not change (the cell of a particle
                // that stayed in its cell) is not written again, and a
                // wavefront with no changed lane issues no store
                const uint32_t c1 = cell_pack(s[r].jx, s[r].jy);
                if (c1 != c0[r]) pc_[tid + r * 256] = c1;
                px[tid + r * 256] = s[r].ox;
                py[tid + r * 256] = s[r].oy;
                pu[tid + r * 256] = s[r].vx;
                pv[tid + r * 256] = s[r].vy;
            } else if (live[r]) {
                pc_[tid + r * 256] = cell_pack(CELL_HOLE, CELL_HOLE);
                const int st = classify(s[r], pc.N, pc.mode);
                atomicAdd(&sl[st - 1], 1u);
                atomicAdd(&shole, 1u);
                // the id and vz are read again only here
                const uint32_t i = blk0 + tid + r * 256;
                if (spn.lost_ids) queue_lost(spn, sp.id[i], w[r]);
                if (spn.wall) {  // waits for the surface pass
                    PState post = s[r];
                    post.vz = sp.vz[i];
                    stage_put(spn.wq, &spn.cw->wall_count, &spn.cw->overflow, post,
                              (unsigned long long)sp.id[i], w[r]);
                }
            }
        }
    }
    // block_deposit_n passes a barrier before it writes the window, so every
    // lane has read its collision result from the shared LDS by then
    if (deposit) block_deposit_n<P, LDS_U64>(dep, s, w, q, pc.N, lds);
    __syncthreads();
    // ahead of a sort pass: the histogram of the cells the particles end the
    // step in, the keys that pass claims by (no k_key_count then)
    if (hist) {
        uint32_t key[P];
#pragma unroll
        for (int r = 0; r < P; r++)
            key[r] = dep[r] ? bin_key(s[r].jx, s[r].jy, pc.tilesX) >> pc.keyshift : 0u;
        block_key_hist<P>(dep, key, hist, reinterpret_cast<uint32_t *>(lds));
    }
    if (tid < 6 && sl[tid]) atomicAdd(&lost6[cnt_slot() * 6 + tid], sl[tid]);
    if (COLL && tid < 8 && se[tid])
        atomicAdd(&events[cnt_slot() * 8 + tid], (unsigned long long)se[tid]);
    if (tid == 0 && shole) atomicAdd(&holes[cnt_slot()], shole);
}

#define PUSH_INPLACE_PARAMS                                                                    \
    SpView sp, const uint32_t *__restrict__ nptr, const float2 *__restrict__ E, PushConst pc, \
        mcc::MccConst mc, uint32_t step, unsigned long long *__restrict__ q, int deposit,     \
        Spawn spn, unsigned long long *__restrict__ events, uint32_t *__restrict__ lost6,     \
        uint32_t *__restrict__ holes, uint32_t *__restrict__ hist
template <int V, int P>
__global__ void __launch_bounds__(256) k_push_inplace(PUSH_INPLACE_PARAMS);
#define INPLACE_GENERIC(P)                                                                      \
    template <>                                                                                \
    __global__ void __launch_bounds__(256) k_push_inplace<PV_GENERIC, P>(PUSH_INPLACE_PARAMS) { \
        push_inplace_generic<P>(sp, nptr, E, pc, mc, step, q, deposit, spn, events, lost6, holes, \
                                hist, blockIdx.x);                                             \
    }
INPLACE_GENERIC(IPP)
INPLACE_GENERIC(IPP_SMALL)
// Waves per SIMD, measured over 4 to 8 at 257^2 and 1025^2 (20 and 10 steps
// of the argon discharge): 7 for the collisionless variants (66-72 VGPRs) and
// 5 for the collisional ones (87), 7.37 and 36.3 ms; 6 and 4: 7.58 and 37.0; 8
// and 6 (a few spills): 7.63 and 37.0; 8 and 7 (ten): 8.05 and 37.9.
#define INPL_WAVES_PLAIN 7
#define INPL_WAVES_COLL 5
#define INPL_WAVES_COLL_I 7
#define INPL_WAVES_W 6  // four weights more in registers
#define INPLACE_FAST_P(V, P, WAVES)                                                            \
    template <>                                                                                \
    __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES)))  \
        k_push_inplace<V, P>(PUSH_INPLACE_PARAMS) {                                            \
        push_inplace_body<V, P>(sp, nptr, E, pc, mc, step, q, deposit, spn, events, lost6,     \
                                holes, hist, blockIdx.x);                                      \
    }
#define INPLACE_FAST(V, WAVES)    \
    INPLACE_FAST_P(V, IPP, WAVES) \
    INPLACE_FAST_P(V, IPP_SMALL, WAVES)
INPLACE_FAST(PV_PLAIN, INPL_WAVES_PLAIN)
INPLACE_FAST(PV_SPAWN, INPL_WAVES_PLAIN)
INPLACE_FAST(PV_COLL_E, INPL_WAVES_COLL)
INPLACE_FAST(PV_COLL_I, INPL_WAVES_COLL_I)
INPLACE_FAST((PV_PLAIN | PV_W), INPL_WAVES_W)
INPLACE_FAST((PV_SPAWN | PV_W), INPL_WAVES_W)
INPLACE_FAST((PV_COLL_E | PV_W), INPL_WAVES_COLL)
INPLACE_FAST((PV_COLL_I | PV_W), INPL_WAVES_W)

// Both species' collisionless in-place passes in one launch (the first nba
// blocks advance a, the rest b): the kernel of each species pass as it is,
// one launch's fixed cost instead of two on the small grids
template <int P>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(INPL_WAVES_PLAIN, INPL_WAVES_PLAIN)))
    k_push_inplace_pair(InplaceArgs a, InplaceArgs b, uint32_t nba,
                        const float2 *__restrict__ E, uint32_t step, int deposit) {
    if (blockIdx.x < nba)
        push_inplace_body<PV_PLAIN, P>(a.sp, a.n, E, a.pc, a.mc, step, a.q, deposit, a.spn,
                                    a.events, a.lost6, a.holes, a.hist, blockIdx.x);
    else
        push_inplace_body<PV_PLAIN, P>(b.sp, b.n, E, b.pc, b.mc, step, b.q, deposit, b.spn,
                                    b.events, b.lost6, b.holes, b.hist, blockIdx.x - nba);
}

// ------------------------------------------------------- per-phase path
__global__ void __launch_bounds__(256)
    k_gather(SpView sp, const uint32_t *__restrict__ nptr, const float2 *__restrict__ E,
             PushConst pc, float *__restrict__ exp_, float *__restrict__ eyp) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= *nptr) return;
    PState s = load_state(sp, i, false);
    float ex = 0.0f, ey = 0.0f;  // pic.cl:70-71
    if (can_move(s, pc)) gather_one(s, E, pc, ex, ey);
    exp_[i] = ex;
    eyp[i] = ey;
}

__global__ void __launch_bounds__(256)
    k_move(SpView sp, const uint32_t *__restrict__ nptr, const float *__restrict__ exp_,
           const float *__restrict__ eyp, PushConst pc) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= *nptr) return;
    PState s = load_state(sp, i, true);
    if (!can_move(s, pc)) return;
    move_one(s, exp_[i], eyp[i], pc);
    sp.cell[i] = cell_pack(s.jx, s.jy);
    sp.ox[i] = s.ox;
    sp.oy[i] = s.oy;
    sp.vx[i] = s.vx;
    sp.vy[i] = s.vy;
    sp.vz[i] = s.vz;
}

__global__ void __launch_bounds__(256)
    k_deposit(SpView sp, const uint32_t *__restrict__ nptr, int N, int mode,
              unsigned long long *__restrict__ q) {
    uint32_t n = *nptr;
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    bool valid = i < n;
    PState s{};
    float w = 1.0f;
    if (valid) {
        s = load_state(sp, i, false);
        w = load_w(sp, i);
    }
    bool dep = valid && deposit_ok(s, N, mode);
    __shared__ unsigned long long lds[BLOCK_LDS_U64];
    block_deposit(dep, s, q, N, lds, w);
}

// e_collisions::collision / ion_collisions::collision as a phase of its own
// (e_collisions.cpp:480-597, ion_collisions.cpp:255-308): velocities are
// updated in place; created particles are staged at the parent's position.
__global__ void __launch_bounds__(256)
    k_mcc(SpView sp, const uint32_t *__restrict__ nptr, PushConst pc, mcc::MccConst mc,
          uint32_t step, Spawn spn, unsigned long long *__restrict__ events) {
    uint32_t n = *nptr;
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    int ev = mcc::EV_NONE;
    mcc::Child ch{};
    PState s{};
    uint32_t pid = 0;
    if (i < n) s = load_state(sp, i, true);
    if (i < n && s.jx != CELL_HOLE) {
        pid = sp.id[i];
        if (mc.electron)
            ev = mcc::collide_electron(mc, s.vx, s.vy, s.vz, pid, step, ref_mcc_inside(s, pc.N), ch);
        else
            ev = mcc::collide_ion(mc, s.vx, s.vy, s.vz, pid, step);
        sp.vx[i] = s.vx;
        sp.vy[i] = s.vy;
        sp.vz[i] = s.vz;
        if (EV_KIND(ev) == mcc::EV_IONIZE && mc.mode == PIC_DEV_MODE_REF)
            sp.cell[i] = cell_pack(CELL_DEAD, CELL_DEAD);
    }
    count_events(ev, events);
    if (EV_KIND(ev) == mcc::EV_IONIZE && mc.mode == PIC_DEV_MODE_PHYS) {
        PState ce = s, ci = s;
        ce.vx = ch.vx;
        ce.vy = ch.vy;
        ce.vz = ch.vz;
        ci.vx = ch.ivx;
        ci.vy = ch.ivy;
        ci.vz = ch.ivz;
        const float w = load_w(sp, i);
        stage_put(spn.se, &spn.ce->stage_count, &spn.ce->overflow, ce, (unsigned long long)pid, w);
        stage_put(spn.si, &spn.ci->stage_count, &spn.ci->overflow, ci, (unsigned long long)pid, w);
    }
}

// Wall pass of the absorbing walls (pic_run's pre-loop pass, pic_boundary;
// boundary.cpp:581-677, 765-824 with zero yields): the particles inside are
// kept, in store order, the others counted as losses (and, with spn.plop,
// re-injected as pairs, or queued for the surface pass).  An
// order-preserving compaction in three launches: k_absorb_count counts each
// block's survivors (12 B per particle read), a scan gives every block its
// output offset, k_absorb writes the survivors there in order (the store
// stays sorted if it was).
#define ABS_IPP 4
__device__ __forceinline__ int absorb_class(const SpView &src, uint32_t i, int N, int mode) {
    PState s{};
    const uint32_t c = src.cell[i];
    s.jx = cell_jx(c);
    s.jy = cell_jy(c);
    if (s.jx == CELL_HOLE) return ST_HOLE;
    s.ox = src.ox[i];
    s.oy = src.oy[i];
    return classify(s, N, mode);
}

// the grid covers every count the scan reads (blocks past the live count
// write 0)
__global__ void __launch_bounds__(256)
    k_absorb_count(SpView src, const uint32_t *__restrict__ nptr, int N, int mode,
                   uint32_t *__restrict__ bcount) {
    const uint32_t n = *nptr;
    const uint32_t base = blockIdx.x * (256 * ABS_IPP) + threadIdx.x;
    int c = 0;
#pragma unroll
    for (int r = 0; r < ABS_IPP; r++) {
        const uint32_t i = base + r * 256;
        if (i < n && absorb_class(src, i, N, mode) == ST_KEPT) c++;
    }
    c = wave_sum(c);
    __shared__ int wc[4];
    if ((threadIdx.x & 63) == 0) wc[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) bcount[blockIdx.x] = (uint32_t)(wc[0] + wc[1] + wc[2] + wc[3]);
}

__global__ void __launch_bounds__(256)
    k_absorb(SpView src, SpView dst, const uint32_t *__restrict__ nptr,
             const uint32_t *__restrict__ bstart, int N, int mode, uint32_t *__restrict__ lost6,
             mcc::MccConst mc, uint32_t step, Spawn spn) {
    const uint32_t n = *nptr;
    if (blockIdx.x * (256 * ABS_IPP) >= n) return;  // past the live count
    __shared__ uint32_t sl[6];
    __shared__ uint32_t cnt[ABS_IPP][4];
    if (threadIdx.x < 6) sl[threadIdx.x] = 0;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const uint32_t base = blockIdx.x * (256 * ABS_IPP) + threadIdx.x;
    PState s[ABS_IPP];
    uint32_t pid[ABS_IPP], rank[ABS_IPP];
    float wt[ABS_IPP];
    int st[ABS_IPP];
#pragma unroll
    for (int r = 0; r < ABS_IPP; r++) {
        const uint32_t i = base + r * 256;
        s[r] = PState{};
        pid[r] = 0u;
        wt[r] = 1.0f;
        st[r] = ST_HOLE;
        if (i < n) {
            s[r] = load_state(src, i, true);
            pid[r] = src.id[i];
            wt[r] = load_w(src, i);
            st[r] = classify(s[r], N, mode);
        }
        const uint64_t bal = __ballot(st[r] == ST_KEPT);
        rank[r] = (uint32_t)__popcll(bal & below);
        if (lane == 0) cnt[r][w] = (uint32_t)__popcll(bal);
    }
    __syncthreads();
    // store order: round r's particles follow round r-1's, waves in order
#pragma unroll
    for (int r = 0; r < ABS_IPP; r++) {
        uint32_t pre = bstart[blockIdx.x];
        for (int k = 0; k < ABS_IPP * 4; k++)
            if (k < r * 4 + w) pre += cnt[k >> 2][k & 3];
        if (st[r] == ST_KEPT) {
            const uint32_t o = pre + rank[r];
            store_state(dst, o, s[r], pid[r]);
            if (dst.w) dst.w[o] = wt[r];
        } else if (st[r] != ST_HOLE) {
            atomicAdd(&sl[st[r] - 1], 1u);
            if (spn.plop && st[r] >= ST_LEFT && st[r] <= ST_TOP) {
                PState pe, pi;
                mcc::plop_pair(mc, pid[r], step, N, spn.se_sigma, spn.si_sigma, spn.plop_ref, pe,
                               pi);
                const unsigned long long k = (1ull << 32) | pid[r];
                stage_put(spn.se, &spn.ce->stage_count, &spn.ce->overflow, pe, k, wt[r]);
                stage_put(spn.si, &spn.ci->stage_count, &spn.ci->overflow, pi, k, wt[r]);
            }
            if (spn.wall && st[r] >= ST_LEFT && st[r] <= ST_TOP)
                stage_put(spn.wq, &spn.cw->wall_count, &spn.cw->overflow, s[r],
                          (unsigned long long)pid[r], wt[r]);
        }
    }
    __syncthreads();
    if (threadIdx.x < 6 && sl[threadIdx.x])
        atomicAdd(&lost6[cnt_slot() * 6 + threadIdx.x], sl[threadIdx.x]);
}

// ---- commit of the staged particles
// v of the lane J away (a power of two below 64; every lane is active)
template <int J>
__device__ __forceinline__ unsigned long long lane_xor(unsigned long long v) {
    int lo = (int)(uint32_t)v, hi = (int)(uint32_t)(v >> 32);
#define DPP2(ctrl)                                               \
    lo = __builtin_amdgcn_mov_dpp(lo, ctrl, 0xF, 0xF, true);     \
    hi = __builtin_amdgcn_mov_dpp(hi, ctrl, 0xF, 0xF, true)
    if (J == 1) {
        DPP2(0xB1);  // quad_perm 1 0 3 2
    } else if (J == 2) {
        DPP2(0x4E);  // quad_perm 2 3 0 1
    } else if (J == 4) {
        DPP2(0x141);  // row_half_mirror: lane ^ 7
        DPP2(0x1B);   // quad_perm 3 2 1 0: lane ^ 3
    } else if (J == 8) {
        DPP2(0x128);  // row_ror 8
    } else {
        return __shfl_xor(v, J, 64);
    }
#undef DPP2
    return (unsigned long long)(uint32_t)hi << 32 | (uint32_t)lo;
}

// one step of a bitonic network between lanes: the lower element keeps the
// smaller key where `up`
template <int J>
__device__ __forceinline__ void lane_step(unsigned long long &v, bool up) {
    const unsigned long long o = lane_xor<J>(v);
    const bool low = (threadIdx.x & J) == 0;
    v = (low == up) == (o < v) ? o : v;
}
template <int J>
__device__ __forceinline__ void lane_merge(unsigned long long &v, bool up) {
    lane_step<J>(v, up);
    if constexpr (J > 1) lane_merge<J / 2>(v, up);
}
template <int K>
__device__ __forceinline__ void lane_sort(unsigned long long &v) {
    if constexpr (K > 2) lane_sort<K / 2>(v);
    lane_merge<K / 2>(v, (threadIdx.x & K) == 0);
}

// Sort the P <= 1024 M values (a power of two, at least 64; distinct but for
// padding) ascending, thread t of 1024 holding values t + 1024 m: a bitonic
// network whose steps below 64 are lane exchanges, between 64 and 512 LDS
// exchanges (x: P words) and from 1024 on in registers.
template <int M>
__device__ __forceinline__ void block_sort_regs(unsigned long long (&v)[M], uint32_t P,
                                                unsigned long long *x) {
    const uint32_t t = threadIdx.x;
    const bool on = (t & ~63u) < P;  // whole waves
    if (on)
#pragma unroll
        for (int m = 0; m < M; m++) {
            lane_sort<32>(v[m]);
            lane_merge<32>(v[m], (t & 64u) == 0);
        }
    for (uint32_t k = 128; k <= P; k <<= 1) {
#pragma unroll
        for (uint32_t j = 512u * M; j >= 1024; j >>= 1) {
            if (j >= k) continue;
#pragma unroll
            for (int m = 0; m < M; m++) {
                const int o = m ^ (int)(j >> 10);
                if (o < M && o > m) {
                    const bool up = ((t + 1024u * m) & k) == 0;
                    const unsigned long long a = v[m], b = v[o];
                    v[m] = (a < b) == up ? a : b;
                    v[o] = (a < b) == up ? b : a;
                }
            }
        }
        for (uint32_t j = min(k >> 1, 512u); j >= 64; j >>= 1) {
            if (on)
#pragma unroll
                for (int m = 0; m < M; m++) x[t + 1024 * m] = v[m];
            __syncthreads();
            if (on)
#pragma unroll
                for (int m = 0; m < M; m++) {
                    const unsigned long long o = x[(t + 1024 * m) ^ j];
                    const bool up = ((t + 1024u * m) & k) == 0;
                    v[m] = ((t & j) == 0) == up ? (o < v[m] ? o : v[m]) : (o < v[m] ? v[m] : o);
                }
            __syncthreads();
        }
        if (on)
#pragma unroll
            for (int m = 0; m < M; m++) lane_merge<32>(v[m], ((t + 1024u * m) & k) == 0);
    }
}

// Sort (key, val) pairs [0, c) ascending by key in one workgroup, in place: the
// same network over the next power of two, padded with ~0 keys (the arrays
// hold at least that many entries: the staging capacity is a power of two).
__device__ void block_sort_pairs(unsigned long long *key, uint32_t *val, uint32_t c) {
    uint32_t P = 1;
    while (P < c) P <<= 1;
    for (uint32_t t = threadIdx.x; t < P; t += blockDim.x) {
        if (t < c)
            val[t] = t;
        else
            key[t] = ~0ull;
    }
    __syncthreads();
    for (uint32_t k = 2; k <= P; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            for (uint32_t t = threadIdx.x; t < P; t += blockDim.x) {
                uint32_t o = t ^ j;
                if (o > t) {
                    unsigned long long a = key[t], b = key[o];
                    bool up = (t & k) == 0;
                    if ((a > b) == up) {
                        key[t] = b;
                        key[o] = a;
                        uint32_t x = val[t];
                        val[t] = val[o];
                        val[o] = x;
                    }
                }
            }
            __syncthreads();
        }
    }
}

// The staged entry k (key kk) of rank r: given its id and, unless it was
// staged as CELL_DEAD (it takes an id but is not stored), the next slot.
// Every thread of the workgroup calls it; `stored` counts the slots taken.
__device__ __forceinline__ void commit_entry(const CommitArgs &a, int N, bool in, uint32_t r,
                                             uint32_t k, unsigned long long kk, uint32_t base,
                                             uint32_t nid, uint32_t &stored) {
    PState p{};
    float w = 1.0f;
    bool live = false;
    if (in) {
        const uint32_t cc = a.sv.cell[k];
        p = PState{cell_jx(cc), cell_jy(cc), a.sv.ox[k], a.sv.oy[k],
                   a.sv.vx[k],  a.sv.vy[k],  a.sv.vz[k]};
        if (a.sv.w) w = a.sv.w[k];
        live = cc != cell_pack(CELL_DEAD, CELL_DEAD);
    }
    uint32_t tot;
    const uint32_t slot = base + stored + block_excl_scan_1024(live ? 1u : 0u, &tot);
    stored += tot;
    if (!live || slot >= a.cap_dst) return;
    // reflected and backscattered particles (sources 4, 5) keep their id
    const uint32_t src = (uint32_t)(kk >> 32);
    store_state(a.dst, slot, p, (src == 4u || src == 5u) ? (uint32_t)kk : nid + r);
    if (a.dst.w) a.dst.w[slot] = w;
    if (a.deposit && deposit_ok(p, N, a.mode))
        dep_global(a.q, N, p.jx, p.jy, fx_weights_w(p.ox, p.oy, w));
    // the store's histogram for a pending sort pass counts it too
    if (a.hist)
        atomicAdd(&a.hist[(size_t)(bin_key(p.jx, p.jy, a.tilesX) >> a.keyshift) * BIN_STRIDE], 1u);
}

// c <= 1024 M staged entries: sorted by (key, place in the stage) packed in
// one word (sources stay below 2^8, so a key has at most 40 bits, a place 12)
template <int M>
__device__ __forceinline__ uint32_t commit_regs(const CommitArgs &a, int N, uint32_t c,
                                                uint32_t loaded, unsigned long long first,
                                                uint32_t base, uint32_t nid,
                                                unsigned long long *x) {
    const uint32_t t = threadIdx.x;
    uint32_t P = M == 1 ? 64u : 1024u * M;
    while (P < c) P <<= 1;
    unsigned long long v[M];
#pragma unroll
    for (int m = 0; m < M; m++) {
        const uint32_t e = t + 1024u * m;
        v[m] = e < c ? (m == 0 && e < loaded ? first : a.sv.key[e]) << 12 | e : ~0ull;
    }
    block_sort_regs<M>(v, P, x);
    uint32_t stored = 0;
#pragma unroll
    for (int m = 0; m < M; m++) {
        const uint32_t r = t + 1024u * m;
        if (1024u * m < c)  // uniform
            commit_entry(a, N, r < c, r, (uint32_t)v[m] & 4095u, v[m] >> 12, base, nid, stored);
    }
    return stored;
}

// Commit the staged particles of one species: sort by (key, index) in one
// workgroup, then append in key order to dst with consecutive new ids,
// optionally depositing their charge.  Sorting makes the result independent
// of the order in which the staging atomics fired.
//
// Re-injection (pl.on; physical mode, steady walls): the ion pass queued each
// ion lost through a wall (key = id, with its weight) in the wall queue, which
// these walls do not otherwise use; here every queued ion stages the
// electron-ion pair drawn from its own stream (mcc::plop_pair), keyed
// (1 << 32 | id), with its weight, each species' workgroup its own half.  The
// pair sampler (three Philox blocks, six logs and cosines) then stays out of
// the pass and its registers.  The second workgroup to have read the queue's
// count empties it.
//
// Bound by latency: a chain of loads, the sort and the append.  Up to 4096
// entries the sort keeps them in registers, with a barrier only for the steps
// that cross a wavefront (12 of 55 at 1024 entries); the first keys load beside
// the counts.  Argon at 257^2 and 1025^2, mean of a step's two commits: 9.5 and
// 14.3 us with the re-injection, against 10.6 and 19.3 for a sort in LDS plus
// 6.9 and 7.8 for a launch of the re-injection's own.
__device__ __forceinline__ void commit_body(const CommitArgs &a, int N, const PlopArgs &pl,
                                            bool electrons) {
    __shared__ uint32_t s_raw, s_base, s_nid, s_lost;
    __shared__ unsigned long long x[4096];
    const uint32_t t = threadIdx.x;
    if (t == 0) {
        s_raw = a.scnt->stage_count;
        s_base = *a.n_dst;
        s_nid = a.dcnt->next_id;
        uint32_t lost = 0;
        if (pl.on) {
            lost = (uint32_t)__builtin_amdgcn_readfirstlane((int)pl.cw->wall_count);
            asm volatile("" : "+s"(lost) : : "memory");  // read before the ticket is taken
            if (atomicAdd(&pl.cw->wall_ticket, 1u) == 1u) pl.cw->wall_count = pl.cw->wall_ticket = 0;
        }
        s_lost = lost;
    }
    const unsigned long long first = t < a.sv.cap ? a.sv.key[t] : 0ull;  // while the counts load
    __syncthreads();
    const uint32_t raw = s_raw, base = s_base, nid = s_nid, lost = min(s_lost, pl.wq.cap);
    if (raw + lost == 0) return;
    for (uint32_t e = t; e < lost; e += blockDim.x) {
        const uint32_t pid = (uint32_t)pl.wq.key[e], k = raw + e;
        PState pe, pi;
        mcc::plop_pair(pl.mc, pid, pl.step, N, pl.se_sigma, pl.si_sigma, 0, pe, pi);
        if (k >= a.sv.cap) continue;
        a.sv.cell[k] = cell_pack(pe.jx, pe.jy);
        a.sv.ox[k] = pe.ox;
        a.sv.oy[k] = pe.oy;
        a.sv.vx[k] = electrons ? pe.vx : pi.vx;
        a.sv.vy[k] = electrons ? pe.vy : pi.vy;
        a.sv.vz[k] = electrons ? pe.vz : pi.vz;
        a.sv.key[k] = (1ull << 32) | pid;
        // the re-injected pair replaces the lost ion: it carries its weight
        if (a.sv.w) a.sv.w[k] = pl.wq.w ? pl.wq.w[e] : 1.0f;
    }
    if (lost) __syncthreads();
    const uint32_t c = min(raw + lost, a.sv.cap), loaded = min(raw, a.sv.cap);
    uint32_t stored = 0;
    if (c <= 1024) {
        stored = commit_regs<1>(a, N, c, loaded, first, base, nid, x);
    } else if (c <= 2048) {
        stored = commit_regs<2>(a, N, c, loaded, first, base, nid, x);
    } else if (c <= 4096) {
        stored = commit_regs<4>(a, N, c, loaded, first, base, nid, x);
    } else {
        block_sort_pairs(a.sv.key, a.sv.idx, c);
        for (uint32_t r0 = 0; r0 < c; r0 += blockDim.x) {
            const uint32_t r = r0 + t;
            const bool in = r < c;
            commit_entry(a, N, in, r, in ? a.sv.idx[r] : 0u, in ? a.sv.key[r] : 0ull, base, nid,
                         stored);
        }
    }
    if (t == 0) {
        const uint32_t room = base < a.cap_dst ? a.cap_dst - base : 0u;
        const uint32_t written = stored < room ? stored : room;
        *a.n_dst = base + written;
        a.dcnt->next_id = nid + c;
        // a pair that found the stage full counts like one that stage_put refused
        const uint32_t full = raw + lost - max(raw, c);
        const uint32_t dropped = (stored - written) + (raw + lost - c) + full;
        if (dropped) a.dcnt->overflow += dropped;
        a.scnt->stage_count = 0;
    }
}

__global__ void __launch_bounds__(1024) k_commit(CommitArgs a, int N) {
    commit_body(a, N, PlopArgs{}, false);
}

// two independent commits (the ions', then the electrons': disjoint staging,
// stores, counters and charge), workgroup b takes the b-th
__global__ void __launch_bounds__(1024)
    k_commit_pair(CommitArgs a, CommitArgs b, PlopArgs pl, int N) {
    const bool electrons = blockIdx.x != 0;
    commit_body(electrons ? b : a, N, pl, electrons);
}

// ---------------------------------------------- reference steady-state walls
// steady_e_boundary (boundary.cpp:890-1097) pairs, per side, the m-th
// electron outside with the m-th ion outside and re-injects each pair; the
// x sides first (left x < 0, right (int)(x/dx) >= N, boundary.cpp:906-912),
// then the y sides among the particles the x pass left outside.  Order
// within a side = particle id (the reference's vector order depends on its
// removal history, which this store does not keep).
//
// Each axis is one pass over both species with any number of candidates:
// a histogram of (side, id range) buckets, an exclusive scan of the buckets,
// a scatter into bucket order, a sort of each bucket by id (one workgroup per
// bucket) and the pairing, one thread per pair.  A particle the x pass
// re-injects lands inside, so collecting the y candidates from the store
// after the x pass leaves out exactly the particles the x pass paired.

// side of a particle on an axis: 0 low (x < 0 / y < 0), 1 high (cell >= N),
// -1 inside or an empty slot
__device__ __forceinline__ int steady_side(uint32_t c, int N, int axis) {
    const int jx = cell_jx(c);
    if (jx == CELL_HOLE || jx == CELL_DEAD) return -1;
    const int j = axis == 0 ? jx : cell_jy(c);
    return j < 0 ? 0 : (j >= N ? 1 : -1);
}

// bucket of (side, id): side-major, then nb equal ranges of [0, idmax)
__device__ __forceinline__ uint32_t steady_bucket(int side, uint32_t id, uint32_t idmax,
                                                  uint32_t nb) {
    uint32_t r = (uint32_t)(((unsigned long long)id * nb) / idmax);
    return (uint32_t)side * nb + (r < nb ? r : nb - 1);
}

__device__ __forceinline__ uint32_t steady_idmax(const SpCounters *c) {
    const uint32_t m = c->next_id;
    return m ? m : 1u;
}

__global__ void __launch_bounds__(256) k_steady_hist(SteadyArgs a, int N, int axis) {
    const int s = blockIdx.y;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= *a.n[s]) return;
    const int side = steady_side(a.sp[s].cell[i], N, axis);
    if (side < 0) return;
    const SteadyBufs &b = a.b[s];
    atomicAdd(&b.hist[steady_bucket(side, a.sp[s].id[i], steady_idmax(a.cnt[s]), b.nb)], 1u);
}

// exclusive scan of a species' 2 nb bucket counts into start[0..2 nb].  A thread
// takes eight buckets in a row (2 nb is a power of two, at least 32), so two
// species of 262 144 particles (8192 buckets each) are one round: 4.0 us,
// against 12.4 with a bucket a thread and eight rounds.
__global__ void __launch_bounds__(1024) k_steady_scan(SteadyArgs a) {
    const SteadyBufs &b = a.b[blockIdx.x];
    const uint32_t nt = 2 * b.nb;
    uint32_t carry = 0;
    for (uint32_t r0 = 0; r0 < nt; r0 += blockDim.x * 8) {
        const uint32_t r = r0 + threadIdx.x * 8;
        const bool in = r < nt;
        uint4 u{0, 0, 0, 0}, v = u;
        if (in) {
            const uint4 *h = reinterpret_cast<const uint4 *>(b.hist + r);
            u = h[0];
            v = h[1];
        }
        uint32_t tot;
        const uint32_t ex = carry + block_excl_scan_1024(u.x + u.y + u.z + u.w + v.x + v.y + v.z +
                                                             v.w,
                                                         &tot);
        if (in) {
            uint4 *o = reinterpret_cast<uint4 *>(b.start + r);
            const uint4 p{ex, ex + u.x, ex + u.x + u.y, ex + u.x + u.y + u.z};
            const uint32_t e = p.w + u.w;
            o[0] = p;
            o[1] = uint4{e, e + v.x, e + v.x + v.y, e + v.x + v.y + v.z};
        }
        carry += tot;
    }
    if (threadIdx.x == 0) b.start[nt] = carry;
}

// each bucket's count runs back to zero as its entries take their places
__global__ void __launch_bounds__(256) k_steady_scatter(SteadyArgs a, int N, int axis) {
    const int s = blockIdx.y;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= *a.n[s]) return;
    const int side = steady_side(a.sp[s].cell[i], N, axis);
    if (side < 0) return;
    const SteadyBufs &b = a.b[s];
    const uint32_t id = a.sp[s].id[i];
    const uint32_t k = steady_bucket(side, id, steady_idmax(a.cnt[s]), b.nb);
    const uint32_t pos = b.start[k] + atomicSub(&b.hist[k], 1u) - 1u;
    b.id_in[pos] = id;
    b.idx_in[pos] = i;
}

// The entries [lo, lo + k) of a bucket in id order (ids are unique within a
// species), one workgroup: up to STEADY_LDS entries by a bitonic network in
// LDS, larger buckets by counting each entry's rank
#define STEADY_LDS 2048
__device__ __forceinline__ void steady_sort_block(const SteadyBufs &b, uint32_t lo, uint32_t k,
                                                  uint32_t *sk, uint32_t *sv) {
    if (k > STEADY_LDS) {
        for (uint32_t j = threadIdx.x; j < k; j += blockDim.x) {
            const uint32_t v = b.id_in[lo + j];
            uint32_t r = 0;
            for (uint32_t t = 0; t < k; t++) r += b.id_in[lo + t] < v ? 1u : 0u;
            b.id_out[lo + r] = v;
            b.idx_out[lo + r] = b.idx_in[lo + j];
        }
        return;
    }
    uint32_t P = 1;
    while (P < k) P <<= 1;
    for (uint32_t t = threadIdx.x; t < P; t += blockDim.x) {
        sk[t] = t < k ? b.id_in[lo + t] : ~0u;
        sv[t] = t < k ? b.idx_in[lo + t] : 0u;
    }
    __syncthreads();
    for (uint32_t m = 2; m <= P; m <<= 1) {
        for (uint32_t j = m >> 1; j > 0; j >>= 1) {
            for (uint32_t t = threadIdx.x; t < P; t += blockDim.x) {
                const uint32_t o = t ^ j;
                if (o > t) {
                    const uint32_t x = sk[t], y = sk[o];
                    if ((x > y) == ((t & m) == 0)) {
                        sk[t] = y;
                        sk[o] = x;
                        const uint32_t w = sv[t];
                        sv[t] = sv[o];
                        sv[o] = w;
                    }
                }
            }
            __syncthreads();
        }
    }
    for (uint32_t t = threadIdx.x; t < k; t += blockDim.x) {
        b.id_out[lo + t] = sk[t];
        b.idx_out[lo + t] = sv[t];
    }
    __syncthreads();  // read before the next bucket fills them
}

// up to 64 entries [lo, lo + k) in id order, one wavefront: each lane counts
// the smaller ids
__device__ __forceinline__ void steady_sort_wave(const SteadyBufs &b, uint32_t lo, uint32_t k) {
    const uint32_t lane = threadIdx.x & 63;
    const bool on = lane < k;
    const uint32_t v = on ? b.id_in[lo + lane] : ~0u, x = on ? b.idx_in[lo + lane] : 0u;
    uint32_t r = 0;
    for (uint32_t t = 0; t < k; t++)
        r += (uint32_t)__builtin_amdgcn_readlane((int)v, (int)t) < v ? 1u : 0u;
    if (on) {
        b.id_out[lo + r] = v;
        b.idx_out[lo + r] = x;
    }
}

// The buckets' entries in id order.  The buckets are sized for a store that
// has all left, and few particles leave in a step, so most are empty: a
// wavefront takes STEADY_BPW buckets of one side.  All their entries together
// when they are at most 64 (a later bucket of a side holds greater ids),
// otherwise one bucket after the other, and those above 64 entries by the
// whole workgroup.  2 x 262 144 particles: 5.0 us, a workgroup per bucket
// took 6.6.
#define STEADY_BPW 8
__global__ void __launch_bounds__(256) k_steady_sort(SteadyArgs a) {
    const SteadyBufs &b = a.b[blockIdx.y];
    __shared__ uint32_t sk[STEADY_LDS], sv[STEADY_LDS];
    __shared__ uint32_t big[4 * STEADY_BPW], nbig;
    if (threadIdx.x == 0) nbig = 0u;
    __syncthreads();
    const uint32_t per_side = (b.nb + STEADY_BPW - 1) / STEADY_BPW;  // waves of a side
    const uint32_t wave = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (wave < 2 * per_side) {
        const uint32_t side = wave / per_side;
        const uint32_t f = side * b.nb + (wave - side * per_side) * STEADY_BPW;
        const uint32_t m = min((uint32_t)STEADY_BPW, (side + 1) * b.nb - f);
        const uint32_t s0 = b.start[f + min(lane, m)];  // lane m and up: the end
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)s0, 0);
        const uint32_t k = (uint32_t)__builtin_amdgcn_readlane((int)s0, 63) - lo;
        if (k <= 64) {
            if (k) steady_sort_wave(b, lo, k);
        } else {
            const uint32_t kl = __shfl_down(s0, 1, 64) - s0;
            uint64_t todo = __ballot(lane < m && kl > 0);
            while (todo) {
                const int t = __ffsll((unsigned long long)todo) - 1;
                todo &= todo - 1;
                const uint32_t l = (uint32_t)__builtin_amdgcn_readlane((int)s0, t);
                const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)kl, t);
                if (c <= 64)
                    steady_sort_wave(b, l, c);
                else if (lane == 0)
                    big[atomicAdd(&nbig, 1u)] = f + (uint32_t)t;
            }
        }
    }
    __syncthreads();
    const uint32_t nl = nbig;
    for (uint32_t t = 0; t < nl; t++) {
        const uint32_t f = big[t], l = b.start[f];
        steady_sort_block(b, l, b.start[f + 1] - l, sk, sv);
    }
}

// move the pair (e[ie], ion[ii]) to one point with fresh velocities and
// deposit both (boundary.cpp:854-878); the ion's id keys the draws
__device__ __forceinline__ void plop_store(SpView e, SpView ion, uint32_t ie, uint32_t ii,
                                           const mcc::MccConst &mc, uint32_t step, int N,
                                           float se, float si, unsigned long long *qe,
                                           unsigned long long *qi, int mode) {
    PState pe, pi;
    mcc::plop_pair(mc, ion.id[ii], step, N, se, si, 1, pe, pi);
    e.cell[ie] = cell_pack(pe.jx, pe.jy);
    e.ox[ie] = pe.ox;
    e.oy[ie] = pe.oy;
    e.vx[ie] = pe.vx;
    e.vy[ie] = pe.vy;
    e.vz[ie] = pe.vz;
    ion.cell[ii] = cell_pack(pi.jx, pi.jy);
    ion.ox[ii] = pi.ox;
    ion.oy[ii] = pi.oy;
    ion.vx[ii] = pi.vx;
    ion.vy[ii] = pi.vy;
    ion.vz[ii] = pi.vz;
    // each particle keeps its own weight factor
    if (deposit_ok(pe, N, mode))
        dep_global(qe, N, pe.jx, pe.jy, fx_weights_w(pe.ox, pe.oy, load_w(e, ie)));
    if (deposit_ok(pi, N, mode))
        dep_global(qi, N, pi.jx, pi.jy, fx_weights_w(pi.ox, pi.oy, load_w(ion, ii)));
}

// the pairs of both sides of an axis: thread k < m0 pairs rank k of the low
// side, m0 <= k < m0 + m1 rank k - m0 of the high side
__global__ void __launch_bounds__(256)
    k_steady_pair(SteadyArgs a, mcc::MccConst mc, uint32_t step, int N, float se, float si,
                  unsigned long long *__restrict__ qe, unsigned long long *__restrict__ qi,
                  int mode) {
    const SteadyBufs &be = a.b[0], &bi = a.b[1];
    const uint32_t nb = be.nb;
    const uint32_t e0 = be.start[nb] - be.start[0], e1 = be.start[2 * nb] - be.start[nb];
    const uint32_t i0 = bi.start[nb] - bi.start[0], i1 = bi.start[2 * nb] - bi.start[nb];
    const uint32_t m0 = e0 < i0 ? e0 : i0, m1 = e1 < i1 ? e1 : i1;
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= m0 + m1) return;
    const int side = k < m0 ? 0 : 1;
    const uint32_t r = side == 0 ? k : k - m0;
    const uint32_t ie = be.idx_out[be.start[side * nb] + r];
    const uint32_t ii = bi.idx_out[bi.start[side * nb] + r];
    plop_store(a.sp[0], a.sp[1], ie, ii, mc, step, N, se, si, qe, qi, mode);
}

// ------------------------------------------------------------ loader
// Uniform positions in (0,L)^2 and a 3-V Maxwellian, from Philox4x32-10 keyed
// by the seed with counter (id, species, call, 0).
__global__ void __launch_bounds__(256)
    k_load_random(SpView sp, uint32_t n, uint32_t key0, uint32_t key1, uint32_t species, int N,
                  double sigma) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t r[4], g[4], z[4];
    philox4x32_10(i, species, 0u, 0u, key0, key1, r);
    philox4x32_10(i, species, 1u, 0u, key0, key1, g);
    philox4x32_10(i, species, 2u, 0u, key0, key1, z);
    double cells = (double)(N - 1);
    double tx = u01d(r[0], r[1]) * cells, ty = u01d(r[2], r[3]) * cells;
    int jx = (int)floor(tx), jy = (int)floor(ty);
    float ox = (float)(tx - (double)jx), oy = (float)(ty - (double)jy);
    if (ox >= 1.0f) { ox = 0.0f; jx += 1; }
    if (oy >= 1.0f) { oy = 0.0f; jy += 1; }
    double u1 = u01d(g[0], g[1]), u2 = u01d(g[2], g[3]);
    double rad = sqrt(-2.0 * log(u1));
    double u3 = u01d(z[0], z[1]), u4 = u01d(z[2], z[3]);
    double two_pi = 6.283185307179586;
    sp.cell[i] = cell_pack(jx, jy);
    sp.ox[i] = ox;
    sp.oy[i] = oy;
    sp.vx[i] = (float)(sigma * rad * cos(two_pi * u2));
    sp.vy[i] = (float)(sigma * rad * sin(two_pi * u2));
    sp.vz[i] = (float)(sigma * sqrt(-2.0 * log(u3)) * cos(two_pi * u4));
    sp.id[i] = i;
}

// ------------------------------------------------------------ particle source
// inject_more_particles (particle.cpp:491-510): n particles a step, uniform in
// [dx, L-dx]^2, each velocity component vt cos(2 pi R2) sqrt|ln R1|
// (particle.cpp:452-464).  Draws: Philox counter (k, step, species*16 +
// RS_INJECT + 256 d, 0x4D434331), d = 0 position, 1..3 vx, vy, vz.  In the
// reference the source runs after the electron collisions and before the
// gather (pic.cpp:1071-1082): injected electrons are pushed and wall-tested
// here (no collision this step) and staged at their new position; injected
// ions are staged unmoved and join the ion pass.  Staging key 2 << 32 | k.
__device__ __forceinline__ void inject_pos(double x, double dx, int &j, float &o) {
    const double t = x / dx;
    const double k = floor(t);
    float f = (float)(t - k);
    int jj = (int)k;
    if (f >= 1.0f) {
        f = 0.0f;
        jj += 1;
    }
    j = jj;
    o = f;
}

__device__ __forceinline__ float inject_vel(const uint32_t r[4], double vt) {
    const double R1 = u01d(r[0], r[1]), R2 = u01d(r[2], r[3]);
    return (float)(vt * cos(6.283185307179586 * R2) * sqrt(fabs(log(R1))));
}

// one launch for a step's source of both species (blockIdx.y)
__global__ void __launch_bounds__(64)
    k_inject(InjectArgs a0, InjectArgs a1, const float2 *__restrict__ E, uint32_t step,
             uint32_t n_inj, float w, double dx, double L) {
    const InjectArgs &A = blockIdx.y ? a1 : a0;
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n_inj) return;
    const uint32_t s0 = A.species * 16u + RS_INJECT, key0 = A.key0, key1 = A.key1;
    uint32_t a[4], b[4], c[4], d[4];
    philox4x32_10(k, step, s0, RNG_DOMAIN_MCC, key0, key1, a);
    philox4x32_10(k, step, s0 + 256u, RNG_DOMAIN_MCC, key0, key1, b);
    philox4x32_10(k, step, s0 + 512u, RNG_DOMAIN_MCC, key0, key1, c);
    philox4x32_10(k, step, s0 + 768u, RNG_DOMAIN_MCC, key0, key1, d);
    const double span = L - 2.0 * dx;
    PState s;
    inject_pos(fma(u01d(a[0], a[1]), span, dx), dx, s.jx, s.ox);
    inject_pos(fma(u01d(a[2], a[3]), span, dx), dx, s.jy, s.oy);
    s.vx = inject_vel(b, A.vt);
    s.vy = inject_vel(c, A.vt);
    s.vz = inject_vel(d, A.vt);
    int st = ST_KEPT;
    if (A.push) {
        push_one(s, E, A.pc);
        st = classify(s, A.pc.N, A.pc.mode);
    }
    if (st == ST_KEPT)
        stage_put(A.sv, &A.cnt->stage_count, &A.cnt->overflow, s, (2ull << 32) | k, w);
    else
        atomicAdd(&A.cnt->lost[cnt_slot()][st - 1], 1u);
}

// ------------------------------------------------------------ launchers
static inline unsigned blocks_for(int64_t n, int t) {
    int64_t b = (n + t - 1) / t;
    return (unsigned)(b > 0 ? b : 1);
}

void launch_inject(hipStream_t st, const InjectArgs *a, int ns, const float2 *E, uint32_t step,
                   uint32_t n_inj, float w, double dx, double L) {
    if (n_inj == 0) return;
    hipLaunchKernelGGL(k_inject, dim3(blocks_for(n_inj, 64), (unsigned)ns), dim3(64), 0, st, a[0],
                       a[ns - 1], E, step, n_inj, w, dx, L);
}

// the variant whose pinned options match the pass's (PV_GENERIC otherwise)
static int pass_variant(const SpView &sp, const PushConst &pc, const mcc::MccConst &mc,
                        const Spawn *spn) {
    if (pc.mode != PIC_DEV_MODE_PHYS || pc.bfield != 0 || (spn && spn->plop)) return PV_GENERIC;
    const int w = sp.w != nullptr ? PV_W : 0;
    if (!mc.on) return ((spn && (spn->lost_ids || spn->wall)) ? PV_SPAWN : PV_PLAIN) | w;
    if (mc.mode != PIC_DEV_MODE_PHYS) return PV_GENERIC;
    return (mc.electron ? PV_COLL_E : PV_COLL_I) | w;
}

void launch_key_count(hipStream_t st, const SpView &sp, const uint32_t *n, int64_t cap,
                      const PushConst &pc, uint32_t *binCount, int do_push) {
    hipLaunchKernelGGL(k_key_count, dim3(blocks_for(cap, 256 * IPP)), dim3(256), 0, st, sp, n, pc,
                       binCount, do_push);
}

void launch_push_scatter(hipStream_t st, const SpView &src, const SpView &dst, const uint32_t *n,
                         int64_t cap, const float2 *E, const PushConst &pc, const mcc::MccConst &mc,
                         uint32_t step, uint32_t *binCount, const uint32_t *binStart,
                         unsigned long long *q, int do_push, int deposit, const Spawn &spn,
                         unsigned long long *events, uint32_t *lost6, uint32_t *holes) {
    int v = pass_variant(src, pc, mc, &spn);
    if (v != PV_GENERIC && !do_push) v = src.w ? PV_GENERIC : PV_COMPACT;
    const dim3 grid(blocks_for(cap, 256 * IPP)), blk(256);
#define SCATTER(V)                                                                              \
    hipLaunchKernelGGL(k_push_scatter<V>, grid, blk, 0, st, src, dst, n, (uint32_t)cap, E, pc, mc, \
                       step, binCount, binStart, q, do_push, deposit, spn, events, lost6, holes)
    switch (v) {
    case PV_PLAIN: SCATTER(PV_PLAIN); break;
    case PV_SPAWN: SCATTER(PV_SPAWN); break;
    case PV_COLL_E: SCATTER(PV_COLL_E); break;
    case PV_COLL_I: SCATTER(PV_COLL_I); break;
    case PV_PLAIN | PV_W: SCATTER(PV_PLAIN | PV_W); break;
    case PV_SPAWN | PV_W: SCATTER(PV_SPAWN | PV_W); break;
    case PV_COLL_E | PV_W: SCATTER(PV_COLL_E | PV_W); break;
    case PV_COLL_I | PV_W: SCATTER(PV_COLL_I | PV_W); break;
    case PV_COMPACT: SCATTER(PV_COMPACT); break;
    default: SCATTER(PV_GENERIC); break;
    }
#undef SCATTER
}

static int inplace_ipp(int64_t cap) { return cap <= INPL_SMALL_MAX ? IPP_SMALL : IPP; }

void launch_push_inplace(hipStream_t st, const SpView &sp, const uint32_t *n, int64_t cap,
                         const float2 *E, const PushConst &pc, const mcc::MccConst &mc,
                         uint32_t step, unsigned long long *q, int deposit, const Spawn &spn,
                         unsigned long long *events, uint32_t *lost6, uint32_t *holes,
                         uint32_t *hist) {
    const int p = inplace_ipp(cap);
    const dim3 grid(blocks_for(cap, 256 * p)), blk(256);
#define INPLACE(V)                                                                              \
    if (p == IPP)                                                                               \
        hipLaunchKernelGGL((k_push_inplace<V, IPP>), grid, blk, 0, st, sp, n, E, pc, mc, step,  \
                           q, deposit, spn, events, lost6, holes, hist);                        \
    else                                                                                        \
        hipLaunchKernelGGL((k_push_inplace<V, IPP_SMALL>), grid, blk, 0, st, sp, n, E, pc, mc,  \
                           step, q, deposit, spn, events, lost6, holes, hist)
    switch (pass_variant(sp, pc, mc, &spn)) {
    case PV_PLAIN: INPLACE(PV_PLAIN); break;
    case PV_SPAWN: INPLACE(PV_SPAWN); break;
    case PV_COLL_E: INPLACE(PV_COLL_E); break;
    case PV_COLL_I: INPLACE(PV_COLL_I); break;
    case PV_PLAIN | PV_W: INPLACE(PV_PLAIN | PV_W); break;
    case PV_SPAWN | PV_W: INPLACE(PV_SPAWN | PV_W); break;
    case PV_COLL_E | PV_W: INPLACE(PV_COLL_E | PV_W); break;
    case PV_COLL_I | PV_W: INPLACE(PV_COLL_I | PV_W); break;
    default: INPLACE(PV_GENERIC); break;
    }
#undef INPLACE
}

bool inplace_pair_ok(const InplaceArgs &a, const InplaceArgs &b) {
    return pass_variant(a.sp, a.pc, a.mc, &a.spn) == PV_PLAIN &&
           pass_variant(b.sp, b.pc, b.mc, &b.spn) == PV_PLAIN;
}

void launch_push_inplace_pair(hipStream_t st, const InplaceArgs &a, const InplaceArgs &b,
                              const float2 *E, uint32_t step, int deposit) {
    const int p = inplace_ipp(std::max(a.cap, b.cap));
    const uint32_t nba = (uint32_t)blocks_for(a.cap, 256 * p);
    const uint32_t nb = nba + (uint32_t)blocks_for(b.cap, 256 * p);
    if (p == IPP)
        hipLaunchKernelGGL(k_push_inplace_pair<IPP>, dim3(nb), dim3(256), 0, st, a, b, nba, E, step,
                           deposit);
    else
        hipLaunchKernelGGL(k_push_inplace_pair<IPP_SMALL>, dim3(nb), dim3(256), 0, st, a, b, nba, E,
                           step, deposit);
}

void launch_mcc(hipStream_t st, const SpView &sp, const uint32_t *n, int64_t cap,
                const PushConst &pc, const mcc::MccConst &mc, uint32_t step, const Spawn &spn,
                unsigned long long *events) {
    hipLaunchKernelGGL(k_mcc, dim3(blocks_for(cap, 256)), dim3(256), 0, st, sp, n, pc, mc, step,
                       spn, events);
}

void launch_commit_pair(hipStream_t st, const CommitArgs &a, const CommitArgs &b,
                        const PlopArgs &pl, int N) {
    hipLaunchKernelGGL(k_commit_pair, dim3(2), dim3(1024), 0, st, a, b, pl, N);
}

void launch_commit(hipStream_t st, const CommitArgs &a, int N) {
    hipLaunchKernelGGL(k_commit, dim3(1), dim3(1024), 0, st, a, N);
}

void launch_gather(hipStream_t st, const SpView &sp, const uint32_t *n, int64_t cap,
                   const float2 *E, const PushConst &pc, float *exp_, float *eyp) {
    hipLaunchKernelGGL(k_gather, dim3(blocks_for(cap, 256)), dim3(256), 0, st, sp, n, E, pc, exp_,
                       eyp);
}

void launch_move(hipStream_t st, const SpView &sp, const uint32_t *n, int64_t cap,
                 const float *exp_, const float *eyp, const PushConst &pc) {
    hipLaunchKernelGGL(k_move, dim3(blocks_for(cap, 256)), dim3(256), 0, st, sp, n, exp_, eyp, pc);
}

void launch_deposit(hipStream_t st, const SpView &sp, const uint32_t *n, int64_t cap, int N,
                    int mode, unsigned long long *q) {
    hipLaunchKernelGGL(k_deposit, dim3(blocks_for(cap, 256)), dim3(256), 0, st, sp, n, N, mode, q);
}

uint32_t absorb_blocks_pad(int64_t cap) {
    return scan_pad((uint32_t)blocks_for(cap, 256 * ABS_IPP));
}

void launch_absorb(hipStream_t st, const SpView &src, const SpView &dst, const uint32_t *n,
                   uint32_t *nout, int64_t cap, int N, int mode, uint32_t *lost6,
                   const mcc::MccConst &mc, uint32_t step, const Spawn &spn, uint32_t *bcount,
                   uint32_t *bstart, uint32_t *partial) {
    const uint32_t nb = absorb_blocks_pad(cap);
    hipLaunchKernelGGL(k_absorb_count, dim3(nb), dim3(256), 0, st, src, n, N, mode, bcount);
    launch_scan_s<1>(st, bcount, bstart, nb, partial, nout);
    hipLaunchKernelGGL(k_absorb, dim3(blocks_for(cap, 256 * ABS_IPP)), dim3(256), 0, st, src, dst,
                       n, (const uint32_t *)bstart, N, mode, lost6, mc, step, spn);
}

void launch_steady(hipStream_t st, const SteadyArgs &a, const mcc::MccConst &mc, uint32_t step,
                   int N, float se, float si, unsigned long long *qe, unsigned long long *qi,
                   int mode) {
    const int64_t cap = std::max(a.cap[0], a.cap[1]);
    const uint32_t pairs = (uint32_t)std::min(a.cap[0], a.cap[1]);
    for (int axis = 0; axis < 2; axis++) {
        hipLaunchKernelGGL(k_steady_hist, dim3(blocks_for(cap, 256), 2), dim3(256), 0, st, a, N,
                           axis);
        hipLaunchKernelGGL(k_steady_scan, dim3(2), dim3(1024), 0, st, a);
        hipLaunchKernelGGL(k_steady_scatter, dim3(blocks_for(cap, 256), 2), dim3(256), 0, st, a, N,
                           axis);
        const uint32_t waves = 2 * ((a.b[0].nb + STEADY_BPW - 1) / STEADY_BPW);
        hipLaunchKernelGGL(k_steady_sort, dim3((waves + 3) / 4, 2), dim3(256), 0, st, a);
        hipLaunchKernelGGL(k_steady_pair, dim3(blocks_for(pairs, 256)), dim3(256), 0, st, a, mc,
                           step, N, se, si, qe, qi, mode);
    }
}

void launch_load_random(hipStream_t st, const SpView &sp, uint32_t n, uint64_t seed,
                        uint32_t species, int N, double sigma) {
    if (n == 0) return;
    hipLaunchKernelGGL(k_load_random, dim3(blocks_for(n, 256)), dim3(256), 0, st, sp, n,
                       (uint32_t)seed, (uint32_t)(seed >> 32), species, N, sigma);
}

}  // namespace pic
