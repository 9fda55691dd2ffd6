// gasp_window.h -- one replica per workgroup, a window of attempt pairs per round.
//
// For replica counts that leave the split-word kernel (gasp_kernels.h) too few
// waves: a workgroup of W waves serves one replica, and every lane holds one
// attempt pair (2q, 2q + 1), the unit of a Philox block.  A round evaluates the
// pairs of all lanes (a window of 128 W attempts) against the lattice as it was
// at the start of the round.  Attempt j commits iff no earlier attempt of the
// window has its site in j's five-site stencil; otherwise it is deferred, keeps
// its lane and is evaluated again next round.  A committed attempt has read what
// the sequential chain would have shown it (the earlier attempts it depends on
// committed in earlier rounds; no other attempt of the window that commits
// touches its stencil), and the window's earliest attempt always commits, so the
// trajectory is the sequential one and every round makes progress.  Lanes whose
// two attempts have committed take the next pairs from a counter in LDS; which
// lane gets which pair does not matter.
//
// Marks.  An attempt writes a key to its site's entry with an atomic minimum,
// and after a barrier reads the entries of its stencil: an entry below its own
// key belongs to an earlier attempt of the window.  A key is
//   (rounds left) << kWinIdxBits | (attempt index relative to a common base),
// so the keys of later rounds are smaller than every key of earlier ones and
// entries are never cleared (once per 2^18 rounds, when the rounds run out).  The
// base trails the counter by kWinSpan pairs; lanes stop taking pairs while a
// deferred pair is about to fall behind it.
//
// MODE 0 (packed): a dword per site holds the key and, in bit 0, the spin, so
// the five entries an attempt reads give its neighbours and its dependences at
// once: a round's cost per pair is two centre reads (the atomic minimum must keep
// the spin bit), two minima and ten reads, against twenty reads and two minima
// with the spins kept apart.  4 N bytes of LDS per replica.
// MODE 1 (bits and table): lattices beyond that keep one bit per site and a
// table of keys with a power of two of entries (tbl_mask + 1; sites that share
// one only add deferrals).
//
// What bounds it (L = 64, 16384 replicas, two waves each): LDS instructions (23
// per wave and round, seven cycles of the pipe for a read at random sites) and
// instruction issue (119 vector and 62 scalar instructions per 128 attempts); a
// round defers 13% of its attempts.  With few workgroups per CU the rounds are
// latency chains: Philox, the centre read, the mark, a barrier, the entries, the
// threshold, a barrier.  Either way waves wait for each other at the barriers, so
// a wave's priority rises with how soon others need it: 0 while the words are
// drawn (which the others' waits can hide), 2 up to the marks, 1 after the first
// barrier and 3 from the flips to the second.
// Measured (20 sweeps of 8192 replicas at L = 64 1.76 ms, 1.98 without the
// priorities; 10 of 3001 at L = 75 0.48, 0.58; 100 of 256 at L = 32 on two waves
// 0.62 ms, against 4.54 on eighth words; 20 of 256 at L = 256, method 0, table,
// eight waves 1.75, against 2.45 on sweep_hbm_waves; other shapes at window_shape).
//
// IO 0: the engine's bit lattice (layout 1, uint32 [R][stride]); IO 1: the
// caller's int32 +-1 grids [R][N], read and written in place.
#pragma once

#include "gasp_kernels.h"

namespace gasp {

constexpr int kWinThr = 0;     // 32 thresholds of 4 bytes, indexed by the five spins
constexpr int kWinCtl = 128;   // pair counter and deferral count (one 64-bit word), up spins
constexpr int kWinLat = 144;   // entries (MODE 0), or bits then keys (MODE 1)
constexpr uint32_t kWinHold = 1u << 20;  // added to the deferral count: above any round's deferrals
constexpr int kWinIdxBits = 13;
constexpr uint32_t kWinSpan = 1u << (kWinIdxBits - 1);  // pairs a key can reach back
enum { WIN_PACKED = 0, WIN_TABLE = 1 };
enum { WIN_BITS = 0, WIN_INT32 = 1 };

__device__ __forceinline__ void lds_min32(unsigned addr, unsigned v) {
    __hip_atomic_fetch_min(lds_ptr32(addr), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ uint32_t min5(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t e) {
    return min(min(min(a, b), c), min(d, e));
}
// the five entries' spins (bit 0 of each) as an offset into the threshold
// table: c in bit 2, then up, dn, lt, rt
__device__ __forceinline__ uint32_t spins_offset(uint32_t c, uint32_t up, uint32_t dn, uint32_t lt, uint32_t rt) {
    uint32_t x = c << 31;
    x = __builtin_amdgcn_alignbit(up, x, 1);
    x = __builtin_amdgcn_alignbit(dn, x, 1);
    x = __builtin_amdgcn_alignbit(lt, x, 1);
    x = __builtin_amdgcn_alignbit(rt, x, 1);
    return x >> 25;
}

template <int RNG, int W, bool POW2, int MODE, int IO>
__global__ void __launch_bounds__(64 * W) sweep_window(SweepArgs a) {
    static_assert(W >= 1 && W <= 16 && (W & (W - 1)) == 0, "1 to 16 waves per replica");
    static_assert(3 * 64 * W < (int)kWinSpan, "two rounds of new pairs within the span");
    constexpr uint32_t S = 64 * W;
    constexpr int U = MODE == WIN_PACKED ? 4 : 1;  // positions: byte offsets of entries, or sites
    constexpr uint32_t kRounds = (MODE == WIN_PACKED ? 1u << (31 - kWinIdxBits) : 1u << (32 - kWinIdxBits)) - 1u;
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int N = a.N, r = blockIdx.x;  // grid = R workgroups
    if (lds_origin(smem) != 0u || (a.rng_dev && !rng_header_ok(a.rng_dev, a.R))) {  // as in sweep_kernel
        if (tid == 0) a.mag[r] = __builtin_nanf("");
        return;
    }
    const bool active = !(a.freeze && uniform32((uint32_t)a.fate[r]) != 0xffffffffu);  // uniform over the workgroup

    // attempt coordinates as in sweep_kernel: launch-local attempt l is x = l + b,
    // so that pair q = x >> 1 is the global Philox pair P0 + q
    const uint64_t a_begin = a.rng_dev ? uniform64(a.rng_dev->attempts) : a.a_begin;
    const uint64_t seed = a.rng_dev ? uniform64(a.rng_dev->seed) : a.seed;
    const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
    const uint32_t b = (uint32_t)(a_begin & 1ull);
    const uint64_t P0 = a_begin >> 1;
    const bool work = active && a.n_attempts != 0;
    const uint32_t e = (uint32_t)a.n_attempts + b;
    const uint32_t NP = (e + 1u) >> 1;  // pairs

    const uint32_t nbw = ((uint32_t)N + 31u) >> 5;
    unsigned *bits = (unsigned *)a.lattice + (size_t)r * a.stride;
    int *ints = (int *)a.lattice + (size_t)r * N;
    // the word at kWinCtl, in a vector register: an address the compiler takes for
    // uniform would get a lane reduction around its atomics
    unsigned ctl = kWinCtl;
    asm volatile("" : "+v"(ctl));
    if (!work) {
        // frozen, or a measurement only: the spins stay where they are
        uint32_t c = 0u;
        if constexpr (IO == WIN_BITS) {
            for (uint32_t i = (uint32_t)tid; i < nbw; i += S) c += (uint32_t)__popc(bits[i]);
        } else {
            for (int x = tid; x < N; x += (int)S) c += ints[x] == 1 ? 1u : 0u;
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) c += __shfl_xor(c, off, 64);
        if (tid == 0) *lds_ptr32(kWinCtl + 8) = 0u;
        __syncthreads();
        if (lane == 0) __hip_atomic_fetch_add(lds_ptr32(ctl + 8u), c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __syncthreads();
        if (wave == 0) finish_replica(a, tid == 0, r, lds_load32(kWinCtl + 8));
        return;
    }

    // ---------------------------------------------------------- prologue
    // A draw u accepts iff u < T, that is u <= T - 1; the classes with T = 0
    // (never) are kept apart as a mask over the table's index.
    uint32_t never = 0u;
#pragma unroll
    for (int j = 0; j < 10; ++j)
        if (a.thr[j] == 0ull) never |= 1u << j;
    if (tid < 32) {
        const int j = 5 * (tid & 1) + __popc((unsigned)tid >> 1);
        uint64_t T = 0ull;
#pragma unroll
        for (int i = 0; i < 10; ++i)
            if (i == j) T = a.thr[i];
        *lds_ptr32(kWinThr + 4u * (unsigned)tid) = T ? (uint32_t)(T - 1ull) : 0u;
    }
    if (tid == 0) {
        *(lds_u64 *)(uintptr_t)kWinCtl = (uint64_t)min(S, NP);  // next pair to hand out; no deferrals yet
        *lds_ptr32(kWinCtl + 8) = 0u;                           // up spins
    }
    const uint32_t tb = kWinLat + (MODE == WIN_TABLE ? ((nbw + 3u) >> 2) << 4 : 0u);  // the keys
    const uint32_t hm = a.tbl_mask;
    if constexpr (MODE == WIN_PACKED) {
        for (int x = tid; x < N; x += (int)S) {
            unsigned s;
            if constexpr (IO == WIN_BITS) s = (bits[x >> 5] >> (x & 31)) & 1u;
            else s = ints[x] == 1 ? 1u : 0u;
            *lds_ptr32(kWinLat + 4u * (unsigned)x) = ~1u | s;
        }
    } else {
        if constexpr (IO == WIN_BITS) {
            for (uint32_t i = (uint32_t)tid; i < nbw; i += S) *lds_ptr32(kWinLat + 4u * i) = bits[i];
        } else {
            for (int base = wave * 64; base < N; base += (int)S) {
                const int x = base + lane;
                const uint64_t m = wave_mask(x < N && ints[x < N ? x : 0] == 1);
                const uint32_t i = 2u * (uint32_t)(base >> 6) + (uint32_t)lane;
                if (lane < 2 && i < nbw) *lds_ptr32(kWinLat + 4u * i) = lane ? (uint32_t)(m >> 32) : (uint32_t)m;
            }
        }
        for (uint32_t i = (uint32_t)tid; i <= hm; i += S) *lds_ptr32(tb + 4u * i) = ~0u;
    }
    __syncthreads();

    const Geometry<POW2, U> geo{a.L, N, a.lg};
    const uint32_t *drw = nullptr;
    if constexpr (RNG == RNG_DRAWS) drw = a.draws + (size_t)r * (3 * a.n_attempts);

    // ---------------------------------------------------------- rounds
    // Wave masks: attempts A and B still to commit, lanes with a new pair.
    // x = 2 q (A) and 2 q + 1 (B) lie in [b, e): only the launch's first pair can start below b.
    const uint32_t eB = e >> 1;  // 2 q + 1 < e
    uint32_t q = (uint32_t)tid;
    uint64_t mA = wave_mask(q < NP) & wave_mask(2u * q >= b), mB = wave_mask(q < eB);
    uint64_t fresh = mA | mB;
    Stencil sA{}, sB{};
    uint32_t uaA = 0u, uaB = 0u;
    uint32_t nxt = min(S, NP), ndef = 0u, left = kRounds;
    bool hold = false;
    uint32_t ahead = 0u;
    // Wave priorities: lowest while the words are drawn, which can be done at any
    // time, and highest before the barriers that other waves wait at.
    for (;;) {
        __builtin_amdgcn_s_setprio(0);
        if (__builtin_amdgcn_inverse_ballot_w64(fresh)) {
            if constexpr (RNG == RNG_PHILOX) {
                const uint64_t pair = P0 + q;
                uint32_t c0 = (uint32_t)pair, c1 = (uint32_t)(pair >> 32), c2 = (uint32_t)r, c3 = kPhiloxDomain;
                philox4x32_10(c0, c1, c2, c3, k0, k1);
                sA = geo.philox(c0);
                uaA = c1;
                sB = geo.philox(c2);
                uaB = c3;
            } else {
                uint32_t u0 = 0, u1 = 0, v0 = 0, v1 = 0;
                if (2u * q >= b) {
                    const uint32_t *d = drw + 3 * (size_t)(2u * q - b);
                    u0 = d[0]; u1 = d[1]; uaA = d[2];
                }
                if (q < eB) {
                    const uint32_t *d = drw + 3 * (size_t)(2u * q + 1u - b);
                    v0 = d[0]; v1 = d[1]; uaB = d[2];
                }
                sA = geo.mt(u0, u1);
                sB = geo.mt(v0, v1);
            }
        }
        if constexpr (RNG == RNG_DRAWS) {
            // The draws of a pair are 24 bytes that no earlier round has loaded:
            // touch those of the pairs after next round's (a load every 64
            // bytes), so that a round finds its own in the cache.  100 sweeps of
            // 256 replicas at L = 32: 0.97 -> 0.70 ms.
            asm volatile("" ::"v"(ahead));
            const uint64_t at = 6ull * (nxt + S) + 16ull * (uint32_t)tid;
            if (at < 6ull * (nxt + 2u * S) && at < 3ull * a.n_attempts) ahead = drw[at];
        }
        __builtin_amdgcn_s_setprio(2);
        // the pair's keys (B's is one more); MODE 0 keeps the spin below them
        const uint32_t base = (left << kWinIdxBits) - 2u * (nxt - kWinSpan);
        const uint32_t kA = MODE == WIN_PACKED ? 4u * q + 2u * base : 2u * q + base;
        const uint32_t kB = kA + (MODE == WIN_PACKED ? 2u : 1u);
        uint32_t oA = 0u, oB = 0u;  // threshold offsets
        if constexpr (MODE == WIN_PACKED) {
            const uint32_t cA = lds_load32(kWinLat + (unsigned)sA.c), cB = lds_load32(kWinLat + (unsigned)sB.c);
            if (__builtin_amdgcn_inverse_ballot_w64(mA)) lds_min32(kWinLat + (unsigned)sA.c, kA | (cA & 1u));
            if (__builtin_amdgcn_inverse_ballot_w64(mB)) lds_min32(kWinLat + (unsigned)sB.c, kB | (cB & 1u));
        } else {
            if (__builtin_amdgcn_inverse_ballot_w64(mA)) lds_min32(tb + 4u * ((unsigned)sA.c & hm), kA);
            if (__builtin_amdgcn_inverse_ballot_w64(mB)) lds_min32(tb + 4u * ((unsigned)sB.c & hm), kB);
            // no spin changes before the barrier
            auto spin = [&](int x) {
                return lds_load32(kWinLat + (((unsigned)x >> 3) & ~3u)) >> ((unsigned)x & 31u);
            };
            oA = spins_offset(spin(sA.c), spin(sA.up), spin(sA.dn), spin(sA.lt), spin(sA.rt));
            oB = spins_offset(spin(sB.c), spin(sB.up), spin(sB.dn), spin(sB.lt), spin(sB.rt));
        }
        __syncthreads();
        __builtin_amdgcn_s_setprio(1);
        uint64_t dA, dB;  // lanes with an earlier attempt in the stencil
        if constexpr (MODE == WIN_PACKED) {
            auto entry = [&](int x) { return lds_load32(kWinLat + (unsigned)x); };
            const uint32_t a0 = entry(sA.c), a1 = entry(sA.up), a2 = entry(sA.dn), a3 = entry(sA.lt), a4 = entry(sA.rt);
            const uint32_t b0 = entry(sB.c), b1 = entry(sB.up), b2 = entry(sB.dn), b3 = entry(sB.lt), b4 = entry(sB.rt);
            dA = wave_mask(min5(a0, a1, a2, a3, a4) < kA);
            dB = wave_mask(min5(b0, b1, b2, b3, b4) < kB);
            // A spin that another wave flips meanwhile belongs to an attempt of
            // the window in this stencil: an earlier one (this attempt is
            // deferred) or none, as a later one would itself be deferred.
            oA = spins_offset(a0, a1, a2, a3, a4);
            oB = spins_offset(b0, b1, b2, b3, b4);
        } else {
            auto key = [&](int x) { return lds_load32(tb + 4u * ((unsigned)x & hm)); };
            dA = wave_mask(min5(key(sA.c), key(sA.up), key(sA.dn), key(sA.lt), key(sA.rt)) < kA);
            dB = wave_mask(min5(key(sB.c), key(sB.up), key(sB.dn), key(sB.lt), key(sB.rt)) < kB);
        }
        uint64_t fA = mA & ~dA & wave_mask(uaA <= lds_load32(kWinThr + oA));
        uint64_t fB = mB & ~dB & wave_mask(uaB <= lds_load32(kWinThr + oB));
        if (never) {  // uniform: some class never flips at this (beta, h)
            auto may = [&](uint32_t o) {
                const uint32_t i = o >> 2;
                return ((never >> (5u * (i & 1u) + (uint32_t)__popc(i >> 1))) & 1u) == 0u;
            };
            fA &= wave_mask(may(oA));
            fB &= wave_mask(may(oB));
        }
        __builtin_amdgcn_s_setprio(3);
        if (__builtin_amdgcn_inverse_ballot_w64(fA)) {
            if constexpr (MODE == WIN_PACKED) lds_xor32(kWinLat + (unsigned)sA.c, 1u);
            else lds_xor32(kWinLat + (((unsigned)sA.c >> 3) & ~3u), 1u << ((unsigned)sA.c & 31u));
        }
        if (__builtin_amdgcn_inverse_ballot_w64(fB)) {
            if constexpr (MODE == WIN_PACKED) lds_xor32(kWinLat + (unsigned)sB.c, 1u);
            else lds_xor32(kWinLat + (((unsigned)sB.c >> 3) & ~3u), 1u << ((unsigned)sB.c & 31u));
        }
        mA &= dA;
        mB &= dB;
        // Lanes with nothing left take the next pairs.  One atomic per wave
        // hands them out (low half) and adds up the deferrals (high half, which
        // counts over the whole launch).
        const uint64_t busy = mA | mB, idle = ~busy;
        const bool take = nxt < NP && !hold;  // uniform over the workgroup
        uint32_t more = (uint32_t)__popcll(busy);
        // a deferred pair that two more rounds of new pairs would put out of the keys' reach
        if ((busy & wave_mask((int)q < (int)(nxt - kWinSpan + 3u * S))) != 0ull) more += kWinHold;
        uint64_t got = 0ull;
        if (lane == 0)
            got = __hip_atomic_fetch_add((lds_u64 *)(uintptr_t)ctl,
                                         ((uint64_t)more << 32) | (take ? (uint32_t)__popcll(idle) : 0u),
                                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        fresh = 0ull;
        if (take) {
            const uint32_t first = uniform32((uint32_t)got);
            const uint32_t mine = __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)idle, first));
            if (__builtin_amdgcn_inverse_ballot_w64(idle)) q = mine;
            fresh = idle & wave_mask(mine < NP);  // never the launch's first pair
            mA |= fresh;
            mB |= idle & wave_mask(mine < eB);
        }
        __syncthreads();
        const uint64_t word = uniform64(lds_load64(kWinCtl));
        const uint32_t nxt1 = (uint32_t)word, ndef1 = (uint32_t)(word >> 32);
        const uint32_t deferred = ndef1 - ndef;
        if (deferred == 0u && nxt >= NP) break;  // every pair handed out has committed
        hold = deferred >= kWinHold;
        ndef = ndef1;
        nxt = nxt1;
        if (--left == 0u) {
            if constexpr (MODE == WIN_PACKED) {
                for (uint32_t x = (uint32_t)tid; x < (uint32_t)N; x += S) *lds_ptr32(kWinLat + 4u * x) |= ~1u;
            } else {
                for (uint32_t i = (uint32_t)tid; i <= hm; i += S) *lds_ptr32(tb + 4u * i) = ~0u;
            }
            left = kRounds;
            __syncthreads();
        }
    }

    // ---------------------------------------------------------- epilogue
    uint32_t up = 0u;  // uniform over the wave
    for (int x0 = wave * 64; x0 < N; x0 += (int)S) {
        const int x = x0 + lane;
        uint64_t m;
        if constexpr (MODE == WIN_PACKED) {
            m = wave_mask(x < N && (lds_load32(kWinLat + 4u * (unsigned)(x < N ? x : 0)) & 1u) != 0u);
        } else {
            const uint32_t i = 2u * (uint32_t)(x0 >> 6);
            const uint32_t lo = lds_load32(kWinLat + 4u * i);
            const uint32_t hi = i + 1u < nbw ? lds_load32(kWinLat + 4u * (i + 1u)) : 0u;
            m = ((uint64_t)hi << 32) | lo;  // no bit beyond N is set
        }
        up += (uint32_t)__popcll(m);
        if constexpr (IO == WIN_BITS) {
            const uint32_t i = 2u * (uint32_t)(x0 >> 6) + (uint32_t)lane;
            if (lane < 2 && i < nbw) bits[i] = lane ? (uint32_t)(m >> 32) : (uint32_t)m;
        } else {
            if (x < N) ints[x] = (m >> lane) & 1ull ? 1 : -1;
        }
    }
    if (lane == 0) __hip_atomic_fetch_add(lds_ptr32(ctl + 8u), up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __syncthreads();
    if (wave == 0) finish_replica(a, tid == 0, r, lds_load32(kWinCtl + 8));
}

// Caller grids as a sweep would leave them where none runs: any value but 1 is a
// down spin.  (sweep_window writes no spins then; a branch for it there costs every
// call: one sweep of 64 replicas at L = 32 15.82 us, 15.48 without.)
__global__ void __launch_bounds__(256) only_spins(int *__restrict__ g, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        if (g[i] != 1 && g[i] != -1) g[i] = -1;
}

}  // namespace gasp
