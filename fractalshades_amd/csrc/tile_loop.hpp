// tile_loop.hpp -- the persistent, work-stealing tile kernel, generic over a
// pixel model (State / init / step / finish).  A wave takes 64 pixels at a
// time, one per lane, from its own first slots, then from pixel cursors that
// the launch's waves share.
#pragma once
#include "bla_key.hpp"
#include "fsg_internal.hpp"
#include "slot_rule.hpp"

namespace fsg {

// a lane's counts (a lane's plain steps stay far below 2^32: 2000 s of them).
// looks: runs of BLA lookups, each of which ends with one that does not jump.
// A pixel's plain steps and the iterations its jumps cover are added when it
// stops, from its n and its sum of jump lengths (State::jl).
struct Counters { unsigned plain, bla, reb, looks; unsigned long long bla_it; };

// Stop reason of a pixel whose binary32 result may differ from the binary64
// loop's (a decision taken within the pixel's error bound): set by the
// FSG_PREC_FP32X kernels, replaced by a second, binary64 pass over exactly
// those pixels (KArgs::redo).  Never left in a finished result.
constexpr int REASON_UNSURE = 3;


// --------------------------------------------------------------------------
// Pixel order over a grid of rows of w pixels (n = h w + a short last row).
// Slot s of the cursor maps to one pixel, a bijection of [0, n): first the
// 8x8 blocks of the top (h & ~7) rows and left (w & ~7) columns, block after
// block along the rows, each block row-major; then the right strip of those
// rows, row-major; then the remaining bottom rows.  A wave that refills 64
// consecutive slots then holds a square of neighbouring pixels, whose
// iteration counts and BLA paths are closer to each other than those of 64
// pixels of one row (2048x2048 frames: 3-7% less kernel time).
template <class T>
__host__ __device__ __forceinline__ T grid_slot_t(T s, T n, T w) {
    const T h8 = (n / w) & ~(T)7, w8 = w & ~(T)7;
    const T a = h8 * w8;
    if (s < a) {
        const T blk = s >> 6, r = s & 63, per_row = w8 >> 3;
        const T by = blk / per_row, bx = blk - by * per_row;
        return ((by << 3) + (r >> 3)) * w + (bx << 3) + (r & 7);
    }
    s -= a;
    const T rem = w - w8, strip = h8 * rem;
    if (s < strip) {
        const T row = s / rem;
        return row * w + w8 + (s - row * rem);
    }
    return h8 * w + (s - strip);
}

__device__ __forceinline__ int64_t grid_slot(int64_t s, int64_t n, int64_t w) {
    if (n <= 0xffffffffll)
        return (int64_t)grid_slot_t<uint32_t>((uint32_t)s, (uint32_t)n, (uint32_t)w);
    return (int64_t)grid_slot_t<uint64_t>((uint64_t)s, (uint64_t)n, (uint64_t)w);
}

// v as it is, for the compiler a new value: it neither rewrites what follows
// in terms of what v was made from nor turns a branch around it into selects
__device__ __forceinline__ void pin(int32_t &v) { asm("" : "+v"(v)); }
// the same, not before x and y are known: a load at index v then takes the
// registers that x and y were made from instead of copying into them later
template <class T> __device__ __forceinline__ void pin_after(T &v, double x, double y) { asm("" : "+v"(v) : "v"(x), "v"(y)); }

// --------------------------------------------------------------------------
// BLA stage selection (ref_BLA_get, perturbation.py:2116-2170).  The tree
// keeps the stage s >= 3 jump starting at iteration w (a multiple of 2^s) at
// index 2 (w >> 3) + 2^(s-3) - 1.  The reference scans the stages from the
// highest one down and takes the first with 2^s < first_invalid - w and
// |z| < r.  Both conditions hold on a prefix of the stages: the first because
// 2^s grows with s, the second because a merged entry's radius is the
// minimum of its first half's radius and the new bound (combine_BLA,
// perturbation.py:2020-2023), so r never grows with the stage for a fixed
// start.  The highest valid stage is therefore found by bisection, with
// about log2(stages) dependent loads instead of one per stage.
// Returns the stage less 3 and the entry's index, -1 if no stage is valid; the
// jump covers 8 << stage iterations.
// zk: the key of |z| (bla_key.hpp), compared with the radii's keys.
// A run of lookups is written do { if (stage >= 0) jump; pin(stage); } while
// (stage >= 0): the jump then updates the pixel's state in place, where a loop
// left from its middle copies it at every lookup (14 instructions).
// A lookup takes 13 vector instructions besides the key where the lowest stage
// fails, 6 more and 8 per bisection step where it does not; with the bounds
// computed before the first test and closed intervals it took 18 and 13 a step.
__device__ __forceinline__ int32_t bla_find(const Tables &t, int64_t zk, int32_t w, int32_t &idx) {
    const int32_t invalid_step = t.first_invalid - w;
    int32_t stage = -1;
    if (invalid_step > 8 && t.stages_bla > 3) {
        const int64_t *rk = t.rk + (w >> 2);        // rk[2^s - 1]: stage s + 3
        // the lowest stage first: invalid there, invalid at every stage (the
        // prefix property), which settles 40 % of the lookups of the 1e-300
        // frame in one read instead of about four (C2 -2.8 %)
        if (zk < rk[0]) {
            // stages that start at w (w a multiple of 2^stage; every one at
            // w = 0), that the table has, and whose jump stays valid
            // (2^stage < invalid_step)
            const int32_t starts = __builtin_ctz((uint32_t)w | 0x80000000u);
            const int32_t fits = 31 - __builtin_clz((uint32_t)(invalid_step - 1));
            int32_t hi = min(min(starts, t.stages_bla - 1), fits) - 2;         // stage valid, hi not
            stage = 0;
            while (hi - stage > 1) {
                const int32_t mid = (stage + hi) >> 1;
                if (zk < rk[(1 << mid) - 1]) stage = mid;
                else hi = mid;
            }
        }
    }
    pin(stage);            // one value for the caller's test, not an exit for each test above
    idx = (w >> 2) + (1 << stage) - 1;
    return stage;
}

// --------------------------------------------------------------------------
// The persistent tile kernel
__device__ __forceinline__ unsigned long long wave_sum(unsigned long long v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// Models whose mantissas drift between renormalisations (LAZY) have them
// renormalised every RENORM_TRIPS trips of the wave (one plain step of a lane
// each, at most): a uniform branch, so the cost is the renormalisation's
// divided by RENORM_TRIPS.
constexpr unsigned RENORM_TRIPS = 8;
template <class M, class = void> struct is_lazy { static constexpr bool value = false; };
template <class M> struct is_lazy<M, decltype((void)M::LAZY)> { static constexpr bool value = M::LAZY; };

// added to a cursor, moves it past every slot of a launch
constexpr unsigned long long CURSOR_DRAIN = 1ull << 44;
constexpr int NC = WORK_NC;
static_assert(NC <= 16, "the cursors' bits are rotated within a 32-bit word");
constexpr unsigned ALL_CURSORS = (1u << NC) - 1u;
constexpr unsigned HAND_STARTED = 1u << 31, HAND_DONE = HAND_STARTED | (ALL_CURSORS << 8);

// The kernel's arguments (its one KArgs), read anew at each use: the compiler
// cannot keep what is read through this reference in scalar registers from
// one use to the next.
__device__ __forceinline__ const KArgs &cold_args() {
    uint64_t p = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const KArgs *)(const __attribute__((address_space(4))) KArgs *)p;
}

// Index of slot base + lane, base a multiple of 64 (uniform over the wave): in
// the blocks' part of a grid the 64 slots are one 8x8 block, found with one
// division; elsewhere each lane maps its own slot.
__device__ __forceinline__ int64_t batch_slot(int64_t base, int64_t n, int64_t w) {
    const unsigned lane = __lane_id();
    if (w <= 0) return base + lane;
    if (n <= 0xffffffffll) {
        const uint32_t w32 = (uint32_t)w, per_row = w32 >> 3, h8 = ((uint32_t)n / w32) & ~7u;
        const uint32_t blk = (uint32_t)(base >> 6);
        if ((uint64_t)blk * 64u < (uint64_t)h8 * (w32 & ~7u)) {
            const uint32_t by = blk / per_row, bx = blk - by * per_row;
            return (int64_t)(((by << 3) + (lane >> 3)) * w32 + (bx << 3) + (lane & 7u));
        }
    }
    const int64_t s = base + lane;
    return s < n ? grid_slot(s, n, w) : s;
}

// One wave takes 64 pixels at a time, iterates them until the last of them has
// stopped, writes their results and takes the next 64.  Switching a lane to a
// new pixel as soon as its own stops would cost the wave the write, two
// dependent memory round trips and the set-up on every trip on which any lane
// switches; the 64 pixels of an 8x8 block stop at about the same trip, and
// waiting for 60 idle lanes instead of all 64 measured within 1 %, on the
// interior-dominated frame too.  The loop over a pixel's trips then is an
// ordinary divergent loop, without a test for idle lanes.
template <class Model>
__device__ __forceinline__ void tile_loop(const KArgs &a) {
    typename Model::State s;
    Counters k = {0, 0, 0, 0, 0};
    unsigned unsure = 0;
    // Slots.  Each wave has its first 64 slots (first_slot), without an atomic;
    // a launch with no more slots than lanes needs no other.  The slots past
    // those of all waves are handed out, 64 at a draw, by NC pixel cursors,
    // each in its own 128-byte line: an atomic takes 12-15 ns on its address
    // whichever wave it comes from, so one cursor serves a draw per 12 ns and
    // 16 one per 1 ns.
    // The slots form groups of 2^gsh (at most 16384 -- 256 8x8 blocks -- and at
    // least 64); cursor x hands out the groups g with g % NC == x, in order.
    // A wave draws from its block's cursor (the blocks of one cursor are on
    // one XCD: they go to the 8 XCDs round robin), then, once that one is
    // drained, from the next one in turn that is not (work stealing), so that
    // every slot is taken exactly once whatever the block-to-XCD placement.
    // The first wave that finds a cursor drained marks it in a global word;
    // every one takes the marks of that word and passes them to its block in
    // LDS: no wave tries the cursors in turn (a read of a cursor's line costs
    // as much as a draw).  Before (eight cursors; every wave drew its first slots too,
    // and at the end from each cursor in turn): 512x512 pixels of one
    // iteration 67 us, now 14; 2048x2048 198, now 105.
    // Group sizes measured against one cursor: 64 slots -5 %, 4096 -7 %, 16384
    // -7 % on the 2048x2048 frame at 1e-300, -15 % on z^3 + c at 1e-800; the
    // interior-dominated frame lost 9 %, 3.5 % and 0.8 %.
    //
    // hand: the wave's cursor (low 8 bits), the cursors it knows drained
    // (ALL_CURSORS << 8) and whether it has taken its first slots (STARTED),
    // uniform over the wave.  Everything else it needs between two batches it
    // takes from the kernel's arguments again (cold_args): held in scalar
    // registers over the loop, that spilled scalar registers the step uses.
    __shared__ unsigned block_seen;                 // cursors known drained to the block
    const unsigned wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    unsigned hand = blockIdx.x % NC;
    if (threadIdx.x == 0) block_seen = 0u;
    __syncthreads();
    // an escape radius past 2^30 lets one step multiply a mantissa further:
    // renormalised on every trip there
    const unsigned renorm_mask = a.M2 > 0x1p60 ? 0u : RENORM_TRIPS - 1u;
    // the binary64 pass: slots of the last batch drawn that are still to take
    unsigned long long rest = 0;
    int64_t rest_idx = 0;
    for (;;) {
        const KArgs &g = cold_args();
        int64_t idx = 0;
        unsigned filled = 0;              // lanes [0, filled) have a pixel
        // The binary64 pass: a wave draws batches until it holds its share of
        // the unsure pixels, and iterates all of the batches drawn, up to 64.
        // Against waves that stopped at their share: 480x270 around the
        // critical orbit, 27050 unsure pixels of 100000 steps, 363 -> 163 ms;
        // 200x200 at 1e-12 and 1e-300 91 -> 72 and 151 -> 94 us.
        unsigned want = 64u;
        if (g.redo) want = redo_share(g.work[6], gridDim.x * (blockDim.x >> 6));
        while (filled < want) {
            if (rest == 0ull) {
                // the next 64 slots, base .. base + 63
                const unsigned waves = blockDim.x >> 6;
                const int64_t held = 64 * (int64_t)(gridDim.x * waves);      // the waves' first slots
                const int64_t left = g.npts - held;                          // the cursors' slots
                int64_t base = -1;
                if ((hand & HAND_STARTED) == 0u) {
                    base = first_slot(blockIdx.x, wave, gridDim.x);
                    hand |= left > 0 ? HAND_STARTED : HAND_DONE;
                } else {
                    unsigned long long *const cursors = g.work + WORK_CURSORS + (g.redo ? 16 * NC : 0);
                    unsigned *const drained = reinterpret_cast<unsigned *>(g.work + WORK_DRAINED + (g.redo ? 16 : 0));
                    // The interrupt flag is host memory, a read across PCIe:
                    // reads from every wave at every refill were served one
                    // after the other, 94 ns each (544 us for a 200x200 tile
                    // whose pixels take 35 us).  So one wave of every eighth
                    // block reads it, when it has finished a batch (the caller
                    // has just looked at the flag itself); when it is set,
                    // that wave drains every cursor, and no wave takes a new
                    // pixel.  The host call of the 200x200 tile: 973 -> 506 us.
                    if (g.stop != nullptr && (blockIdx.x & 7u) == 0u && wave == 0u && __lane_id() < NC &&
                        __hip_atomic_load(g.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != 0u) {
                        atomicAdd(cursors + 16 * __lane_id(), CURSOR_DRAIN);
                        atomicOr(drained, ALL_CURSORS);
                    }
                    const int gsh = min(14, max(6, 63 - __clzll((unsigned long long)(left / NC | 1))));
                    const int64_t low = (1ll << gsh) - 1;
                    unsigned seen = (hand >> 8) & ALL_CURSORS, cur = hand & 0xffu;
                    while (seen != ALL_CURSORS) {
                        seen |= (unsigned)__builtin_amdgcn_readfirstlane((int)__hip_atomic_load(
                            &block_seen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
                        if (seen == ALL_CURSORS) break;
                        // the first cursor from the wave's on that is not known drained
                        const unsigned open = ~seen & ALL_CURSORS;
                        cur = (cur + (unsigned)__builtin_ctz(open >> cur | open << (NC - cur))) % NC;
                        unsigned long long v = 0;
                        if (__lane_id() == 0) v = atomicAdd(cursors + 16 * cur, 64ull);
                        const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
                        const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
                        const int64_t loc = (int64_t)(((unsigned long long)hi << 32) | lo);
                        // the cursor's positions: its whole groups, and the last, short one
                        const int64_t ng = left >> gsh;
                        const int64_t end = (((ng + NC - 1 - (int64_t)cur) / NC) << gsh) +
                                            (ng % NC == (int64_t)cur ? left & low : 0);
                        if (loc < end) {
                            base = held + ((((loc >> gsh) * NC + (int64_t)cur) << gsh) | (loc & low));
                            break;
                        }
                        // the first draw past the cursor's end marks it; every
                        // one takes the marks (a read: an atomic of each wave
                        // on this one word would queue them)
                        unsigned known = 0;
                        if (__lane_id() == 0) {
                            known = loc - end < 64 ? atomicOr(drained, 1u << cur)
                                                   : __hip_atomic_load(drained, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        }
                        seen |= (unsigned)__builtin_amdgcn_readfirstlane((int)known) | (1u << cur);
                        if (__lane_id() == 0) atomicOr(&block_seen, seen);
                    }
                    hand = cur | (seen << 8) | HAND_STARTED;
                }
                if (base < 0) break;
                rest_idx = batch_slot(base, g.npts, g.grid_w);
                bool take = base + (int64_t)__lane_id() < g.npts;
                // the binary64 pass takes only the pixels the binary32 one left unsure
                if (g.redo) take = take && g.stop_reason[take ? rest_idx : 0] == REASON_UNSURE;
                rest = __builtin_amdgcn_ballot_w64(take);
                if (!g.redo) {
                    idx = rest_idx;
                    filled = (unsigned)__popcll(rest);        // the first lanes
                    rest = 0ull;
                    break;
                }
            } else {
                // the batch's unsure slots go to the free lanes, in order
                // (without it a wave iterated only its 44 to 88 % of lanes
                // that drew one); the other lanes complete the permutation
                const auto below = [](unsigned long long m) {
                    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
                };
                const bool goes = ((rest >> __lane_id()) & 1ull) != 0ull && slot_goes(filled, below(rest));
                const unsigned long long sent = __builtin_amdgcn_ballot_w64(goes);
                const unsigned rank = below(sent), end = filled + (unsigned)__popcll(sent);
                const int to = (int)(4u * ((goes ? filled + rank : end + __lane_id() - rank) & 63u));
                const int lo = __builtin_amdgcn_ds_permute(to, (int)(uint32_t)rest_idx);
                const int hi = __builtin_amdgcn_ds_permute(to, (int)(uint32_t)((uint64_t)rest_idx >> 32));
                if (__lane_id() >= filled && __lane_id() < end) idx = (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
                rest &= ~sent;
                filled = end;
            }
        }
        if (filled == 0u) break;
        if (__lane_id() < filled) {
            Model::init(s, g, g.pix[2 * idx], g.pix[2 * idx + 1]);
            int reason;
            // trips: uniform over the lanes still iterating, in a scalar register
            for (unsigned trips = 0;; trips++) {
                if constexpr (is_lazy<Model>::value) {
                    if ((trips & renorm_mask) == renorm_mask) Model::renorm(s, a, (int32_t)trips);
                }
                if (Model::step(s, a, k, reason, (int32_t)trips)) break;
            }
            k.plain += (unsigned)(s.n - s.jl);
            k.bla_it += (unsigned)s.jl;
            Model::finish(s, a, cold_args(), idx, reason);
            unsure += (reason == REASON_UNSURE);
        }
    }
    // All lanes have left the loop.  The block's waves add up their counters
    // in LDS and six lanes add the block's sums to the workspace: one atomic
    // per counter per block.  One per counter per wave queued 4096 waves on
    // six addresses across the dies as they finished (about 0.15 ms of a
    // 1.4 ms launch).  The waves of a persistent launch have nothing left to
    // do once they leave the loop, so waiting at the barrier costs nothing.
    __shared__ unsigned long long part[16][6];
    static_assert(sizeof(part) <= TILE_STATIC_LDS, "static LDS of the tile loop");
    const unsigned long long c[6] = {wave_sum(k.plain), wave_sum(k.bla), wave_sum(k.bla_it),
                                     wave_sum(k.reb), wave_sum((unsigned long long)k.looks + k.bla), wave_sum(unsure)};
    const int wv = (int)(threadIdx.x >> 6);
    if (__lane_id() == 0) {
#pragma unroll
        for (int q = 0; q < 6; q++) part[wv][q] = c[q];
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        unsigned long long sum = 0;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) sum += part[w][threadIdx.x];
        if (sum) atomicAdd(a.work + 1 + threadIdx.x, sum);
    }
}


template <class Model>
__global__ void __launch_bounds__(256) k_tile(const KArgs a) {
    tile_loop<Model>(a);
}

// The same loop with the reference tables staged in LDS: the loop is bound
// by the latency of its table reads (orbit point, derivative paths, BLA
// radius and coefficients at the lane's own iteration index), and an LDS
// read answers in a fraction of an L2 hit's time.  One block of up to 1024
// lanes (tile_block) per CU, or more when they fit, copies the tables once, then runs the loop.
// SHAPE: LDS_FULL: each table pointer is either null or an LDS address, and the
// compiler reads the tables with LDS instructions instead of generic (flat)
// ones.  LDS_ORBIT: the orbit, its codes and the radii are, the derivative paths
// are global addresses; only the BLA coefficients, staged or not, are generic.
// A flat load takes a 64-bit address and waits on both counters; LDS_ORBIT
// instead of LDS_PART: 2048x2048 at 1e-2000 735 -> 702 us, burning ship
// 1920x1080 at 1e-800 795 -> 752 us, at 1e-60 (1001x667) 187 -> 175 us.
template <bool FULL, class T>
__device__ __forceinline__ const T *stage(unsigned char *lds, int32_t off, const T *src, int64_t n) {
    if constexpr (FULL) {
        if (src == nullptr || off < 0) return nullptr;   // off < 0: a table the launch never reads
    } else {
        if (off < 0 || src == nullptr) return src;
    }
    T *dst = reinterpret_cast<T *>(lds + off);
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) dst[i] = src[i];
    return dst;
}

template <class Model, int SHAPE, int BLOCK = 1024>
__global__ void __launch_bounds__(BLOCK) k_tile_lds(const KArgs a) {
    extern __shared__ __align__(16) unsigned char lds[];
    constexpr bool FULL = SHAPE == LDS_FULL, ORBIT = SHAPE != LDS_PART;
    const LdsPlan &p = a.lds;
    KArgs al = a;
    Tables &t = al.t;
    const int64_t K = p.K, KB = p.KB;
    t.Zn = stage<ORBIT>(lds, p.zn, a.t.Zn, K);
    t.zn_k = stage<ORBIT>(lds, p.zn_k, a.t.zn_k, K * a.t.zn_k_w);
    t.rk = stage<ORBIT>(lds, p.r, a.t.rk, KB);
    t.M = stage<FULL>(lds, p.M, a.t.M, KB * p.bla_dim);
    if constexpr (SHAPE != LDS_ORBIT) {
        t.dc = stage<FULL>(lds, p.dc, a.t.dc, K);
        t.dc_e = stage<FULL>(lds, p.dc_e, a.t.dc_e, K);
        if ((FULL || p.dz >= 0) && a.t.dz) {
            cplx *dz = reinterpret_cast<cplx *>(lds + p.dz);
            for (int64_t i = threadIdx.x; i < K; i += blockDim.x) dz[i] = a.t.dz[i];
            if (threadIdx.x == 0) dz[K] = a.t.dz[a.t.L];
            t.dz = dz;
        } else if constexpr (FULL) {
            t.dz = nullptr;
        }
        if ((FULL || p.dz_e >= 0) && a.t.dz_e) {
            int32_t *dze = reinterpret_cast<int32_t *>(lds + p.dz_e);
            for (int64_t i = threadIdx.x; i < K; i += blockDim.x) dze[i] = a.t.dz_e[i];
            if (threadIdx.x == 0) dze[K] = a.t.dz_e[a.t.L];
            t.dz_e = dze;
        } else if constexpr (FULL) {
            t.dz_e = nullptr;
        }
        for (int q = 0; q < 4; q++) {
            t.bs[q] = stage<FULL>(lds, p.bs[q], a.t.bs[q], K);
            t.bs_e[q] = stage<FULL>(lds, p.bs_e[q], a.t.bs_e[q], K);
        }
        if ((FULL || p.dz >= 0) && a.t.dz) t.L = (int32_t)K;   // the wrapped dZndz value is staged at [K]
    }
    __syncthreads();
    tile_loop<Model>(al);
}

}  // namespace fsg
