// team.hip -- the CG loop in one launch of up to one workgroup per CU.
//
// As launches, an iteration of a middle-sized system is a chain of 10 to 60
// kernels (up to several hundred in natural order) of 3.6-3.9 us: half of it the kernel boundary, the rest three
// memory round trips of an empty chip.  Inside one launch the same chain
// costs what it takes a value to travel:
//   * sweeps: a row waits for the values it gathers, not for a barrier.  m
//     and z hold a marker (one NaN) in every row that is not done; a gather
//     that finds it is made again.  A step of the chain is then one store
//     becoming visible and one load (0.3-0.5 us from one workgroup to another),
//     and the arithmetic of a row: 1.3-2.5 us in all;
//   * the two dot products end in a barrier each: an atomic add and a poll,
//     0.8 us for 8 workgroups, 1.0 for 32, 1.3 for 64, 2.2 for 256 (two
//     levels; one counter takes 3.8);
//   * loads and stores of values that other workgroups write or read are
//     relaxed atomics of agent scope, which the L2s keep coherent; nothing is
//     invalidated or written back, so the matrix stays in the L2s, and each
//     XCD keeps the same piece of the mesh in every phase.
// The marker is put back a phase ahead: m while the product is formed, z in
// the forward sweep that follows its last use (z alternates between two
// buffers), with a barrier between that and the rows that wait on it.
//
// Each row's arithmetic, the partial sums and the order they are added in are
// those of the launches of an iteration (kernels.hip), so both give the same
// bits, and a solve may take either, or both in turn.
//
// Every wait ends: after kPatience ticks a wavefront gives up, the launch
// ends and the host falls back on the launches.
//
// us per iteration, launches -> here (MI355X): natural-order SSOR on 129^2
// 51 -> 26, on 101^2 numbered along its axes (395 launches) 1094 -> 370;
// Rainbow on 10,609 rows and 12 colours (2D P3) 96 -> 56, 35,937 rows and 10
// colours 82 -> 51, 35,937 rows and 17 colours (3D P2) 203 -> 141, H(curl)
// 102,024 rows 64 -> 43 (FP32 69 -> 37), 274,625 rows 100 -> 88.
#include "team.hpp"

#include <atomic>

#include "device_common.hpp"
#include "launch.hpp"

namespace sfa {
namespace {

using namespace dev;

constexpr int kTeamThreads = kTeamWaves * kWave;
constexpr int kCounter = 0, kAborted = 64, kXcdCounters = 128;  // words of TeamArgs::sync
constexpr int kOneLevel = 64;                    // most workgroups on one counter
constexpr long long kPatience = 5000000;         // 50 ms of the 100 MHz clock

// The marker: a NaN told by its upper word (FP64) that no row stores.
// not_marker is 0 for it alone.
__device__ inline unsigned not_marker(double v)
{
    return (unsigned)(__builtin_bit_cast(unsigned long long, v) >> 32) ^ 0x7ffadeadu;
}
__device__ inline unsigned not_marker(float v) { return __builtin_bit_cast(unsigned, v) ^ 0x7fcadeadu; }
template <typename T>
__device__ inline T marker()
{
    if constexpr (sizeof(T) == 8) return __builtin_bit_cast(double, 0x7ffadead00000000ull);
    else return __builtin_bit_cast(float, 0x7fcadeadu);
}
// A computed value that happens to be the marker becomes another NaN.
template <typename T>
__device__ inline T unmarked(T v)
{
    return not_marker(v) == 0u ? (T)__builtin_nan("") : v;
}

template <typename V>
__device__ inline V get(const V* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename V>
__device__ inline void put(V* p, V v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The element at a byte offset: a 32-bit offset from a uniform base takes one
// register where an address takes two.
template <typename V>
__device__ inline V get_at(const V* base, unsigned offset)
{
    return get(reinterpret_cast<const V*>(reinterpret_cast<const char*>(base) + offset));
}

// wave_fold (device_common.hpp) over values other workgroups stored.
__device__ inline double team_fold(const double* v, int count)
{
    const int lane = threadIdx.x % kWave;
    constexpr int B = 16;
    double a = 0.;
    for (int i0 = lane; i0 < count; i0 += B * kWave) {
        double t[B];
#pragma unroll
        for (int u = 0; u < B; u++) {
            const int i = i0 + u * kWave;
            t[u] = i < count ? get(v + i) : 0.;
        }
#pragma unroll
        for (int u = 0; u < B; u++)
            if (i0 + u * kWave < count) a += t[u];
    }
    return wave_sum(a);
}

// The hardware workgroup whose logical block (xcd_block) is b of n.
__device__ inline int xcd_workgroup(int b, int n)
{
    const int per = n / kXcds, rem = n % kXcds;
    const int big = rem * (per + 1);  // blocks of the XCDs with one more
    const int x = b < big ? b / (per + 1) : rem + (b - big) / (per > 0 ? per : 1);
    const int k = b - (x * per + (x < rem ? x : rem));
    return k * kXcds + x;
}

template <typename T>
struct Team {
    const TeamArgs<T> a;
    int tid, lane, wave, lwg, blocks;
    unsigned epoch = 0;
    bool lost = false;  // this wavefront has given up
    double* sums;       // LDS [kTeamMaxGroups]
    TeamGroup* groups;  // LDS: the sweeps' groups
    int* flag;          // LDS

    __device__ Team(const TeamArgs<T>& a_, double* sums_, TeamGroup* groups_, int* flag_)
        : a(a_), sums(sums_), groups(groups_), flag(flag_)
    {
        tid = threadIdx.x;
        lane = tid % kWave;
        wave = __builtin_amdgcn_readfirstlane(tid / kWave);
        blocks = gridDim.x;
        lwg = xcd_block(blockIdx.x, blocks);
    }

    // First of the items [0, count) that falls to piece i of `pieces`, a power
    // of two at most kTeamMaxBlocks (count is below 2^20).
    static __device__ int share(int i, int pieces, int count)
    {
        return (int)((unsigned)i * (unsigned)count >> __builtin_ctz((unsigned)pieces));
    }

    // Whether a wait of `spins` turns since t0 is to be given up.
    __device__ bool too_long(unsigned spins, long long& t0) const
    {
        if (spins % 256 != 0) return false;
        if (spins == 256) t0 = wall_clock64();
        return get(a.sync + kAborted) != 0u || wall_clock64() - t0 > kPatience;
    }

    __device__ void give_up(unsigned spins, long long& t0)
    {
        if (__builtin_amdgcn_readfirstlane(too_long(spins, t0) ? 1 : 0)) lost = true;
    }

    // All workgroups have come here, and what they stored before is visible.
    // False: the launch is given up.
    __device__ bool barrier()
    {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const bool gone = __syncthreads_or(lost) != 0;
        epoch++;
        if (tid == 0) {
            bool bad = gone;
            if (!bad) {
                unsigned goal = epoch * (unsigned)blocks;
                if (blocks <= kOneLevel) {
                    __hip_atomic_fetch_add(a.sync + kCounter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                } else {
                    const unsigned per = (unsigned)(blocks / kXcds);
                    unsigned* mine = a.sync + kXcdCounters + 64 * (blockIdx.x % kXcds);
                    goal = epoch * kXcds;
                    if (__hip_atomic_fetch_add(mine, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u ==
                        epoch * per)
                        __hip_atomic_fetch_add(a.sync + kCounter, 1u, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
                }
                long long t0 = 0;
                for (unsigned spins = 1; (int)(get(a.sync + kCounter) - goal) < 0; spins++)
                    if (too_long(spins, t0)) {
                        bad = true;
                        break;
                    }
            }
            if (bad) {
                put(a.sync + kAborted, 1u);
                put(&a.st->team_lost, 1);
            }
            *flag = bad ? 1 : 0;
        }
        __syncthreads();
        return *flag == 0;
    }

    // vec at the byte offsets c_u, waited for.  ALL: every value is loaded again
    // until none is the marker; otherwise only those that are missing, lane by
    // lane.  The first is less work for a row of up to eight entries (26 us
    // per iteration of the 129^2 system instead of 36); on wider rows the
    // loads of all waiting wavefronts keep the memory system so busy that the
    // values do not come (2 ms per iteration, 35,937 rows and 10 colours,
    // instead of 55 us).
    template <int U, bool ALL>
    __device__ void gather(const T* vec, const unsigned (&c)[U], T (&g)[U])
    {
#pragma unroll
        for (int u = 0; u < U; u++) g[u] = get_at(vec, c[u]);
        long long t0 = 0;
        for (unsigned spins = 1;; spins++) {
            unsigned least = ~0u;
#pragma unroll
            for (int u = 0; u < U; u++) least = min(least, not_marker(g[u]));
            if (__ballot(least == 0u) == 0ull || lost) return;
            __builtin_amdgcn_s_sleep(2);
#pragma unroll
            for (int u = 0; u < U; u++)
                if (ALL || not_marker(g[u]) == 0u) g[u] = get_at(vec, c[u]);
            give_up(spins, t0);
        }
    }
    // *p, waited for.
    __device__ T await(const T* p)
    {
        unsigned c[1] = {0u};
        T g[1];
        gather<1, true>(p, c, g);
        return g[0];
    }

    // Entries k0 .. k0+U-1 of a row of w (the slice's entries begin at o0);
    // past its end (0, the zero slot), so that the arithmetic needs no tests.
    template <int U>
    struct Entries {
        unsigned c[U];  // byte offsets of the columns
        T v[U];
    };
    template <int U>
    __device__ void load(const SellViewT<T>& A, int o0, int k0, int w, Entries<U>& E) const
    {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const unsigned e = (unsigned)(o0 + min(k0 + u, w - 1) * kWave + lane);
            E.c[u] = (unsigned)A.cols[e] * (unsigned)sizeof(T);
            E.v[u] = A.vals[e];
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (k0 + u >= w) E.c[u] = (unsigned)a.n * (unsigned)sizeof(T), E.v[u] = T(0);
    }
    // Offset of slice j of a group and its entries per lane.
    __device__ int slice_at(const SellViewT<T>& A, const SweepGroup& G, int j, int& w) const
    {
        if (G.gw >= 0) {
            w = G.gw;
            return G.gbase + j * (G.gw * kWave);
        }
        const int o0 = __builtin_amdgcn_readfirstlane(A.off[G.slice0 + j]);
        w = (__builtin_amdgcn_readfirstlane(A.off[G.slice0 + j + 1]) - o0) / kWave;
        return o0;
    }

    // first() - sum_k v_k * vec[c_k] over a row, entries in order, each value
    // waited for; first(), which loads more, is called once the row's first
    // entries are on their way, and the next entries are loaded before the
    // wait for these.  Eight at a time: sixteen take 256 registers and spill
    // (48.6 us per iteration on an H(curl) system of 102,024 rows
    // instead of 42.8).
    template <int U, bool ALL, class First>
    __device__ T subtract(const SellViewT<T>& A, int o0, int w, const T* vec, First&& first)
    {
        Entries<U> E, F;
        load<U>(A, o0, 0, w, E);
        T acc = first();
        for (int k0 = 0;;) {
            T g[U];
            if (k0 + U < w) load<U>(A, o0, k0 + U, w, F);
            gather<U, ALL>(vec, E.c, g);
#pragma unroll
            for (int u = 0; u < U; u++) acc -= E.v[u] * g[u];
            k0 += U;
            if (k0 >= w) return acc;
            E = F;
        }
    }
    template <class First>
    __device__ T subtract_row(const SellViewT<T>& A, const SweepGroup& G, int j, const T* vec, First&& first)
    {
        int w;
        const int o0 = slice_at(A, G, j, w);
        if (w == 0) return first();
        if (w <= 4) return subtract<4, true>(A, o0, w, vec, first);
        if (w <= 8) return subtract<8, true>(A, o0, w, vec, first);
        return subtract<8, false>(A, o0, w, vec, first);
    }

    __device__ SweepGroup group(int g) const
    {
        const SweepGroup* p = &groups[g].g;
        SweepGroup G;
        G.slice0 = __builtin_amdgcn_readfirstlane(p->slice0);
        G.nslices = __builtin_amdgcn_readfirstlane(p->nslices);
        G.row0 = __builtin_amdgcn_readfirstlane(p->row0);
        G.nrows = __builtin_amdgcn_readfirstlane(p->nrows);
        G.gbase = __builtin_amdgcn_readfirstlane(p->gbase);
        G.gw = __builtin_amdgcn_readfirstlane(p->gw);
        return G;
    }

    // fn(j) for the slices of group g that fall to this wavefront; the
    // workgroup's are consecutive, so that a piece of the mesh stays on one XCD.
    template <class Fn>
    __device__ void my_slices(int g, int count, Fn&& fn)
    {
        const int j0 = share(lwg, blocks, count), j1 = share(lwg + 1, blocks, count);
        const int turn = __builtin_amdgcn_readfirstlane(groups[g].turn);
        for (int j = j0 + ((wave - turn) & (kTeamWaves - 1)); j < j1; j += kTeamWaves) fn(j);
    }

    // Sums the wavefronts' values, in LDS slots of four, into out[index(b)],
    // b in [b0, b1): the partial of a block of four wavefronts.
    template <class Index>
    __device__ void store_partials(int b0, int b1, double* out, Index&& index)
    {
        __syncthreads();
        for (int b = b0 + tid; b < b1; b += kTeamThreads) {
            double t = 0.;
            for (int k = 0; k < 4; k++) t += sums[4 * (b - b0) + k];
            put(out + index(b), t);
        }
    }

    // A row of A (z + beta d).
    template <int U>
    __device__ T multiply(int o0, int w, const T* src, const T* dold, bool fold, T beta) const
    {
        T acc = T(0);
        for (int k0 = 0; k0 < w; k0 += U) {
            Entries<U> E;
            load<U>(a.full, o0, k0, w, E);
            T s[U], g[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                s[u] = get_at(src, E.c[u]);
                g[u] = get_at(dold, E.c[u]);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const T dn = fold && E.c[u] < (unsigned)a.n_active * (unsigned)sizeof(T) ? s[u] + beta * g[u] : g[u];
                acc += E.v[u] * dn;
            }
        }
        return acc;
    }

    // k_spmv_dir: dn = z + beta d, q = A dn, d.Ad partials; m's marker.
    __device__ void product(const T* src, const T* dold, T* dnew, bool fold, T beta)
    {
        const int nb = (a.full_slices + 3) / 4;
        const int b0 = share(lwg, blocks, nb), b1 = share(lwg + 1, blocks, nb);
        for (int k = wave; k < 4 * (b1 - b0); k += kTeamWaves) {
            const int slice = 4 * b0 + k;
            double part = 0.;
            if (slice < a.full_slices) {
                const int row = group_row(a.full, slice, slice, lane, a.full_row0, a.n_active);
                const int ri = row >= 0 ? row : a.n;
                const int o0 = __builtin_amdgcn_readfirstlane(a.full.off[slice]);
                const int w = (__builtin_amdgcn_readfirstlane(a.full.off[slice + 1]) - o0) / kWave;
                const T s_own = get(src + ri), d_own = get(dold + ri);
                const T acc = multiply<8>(o0, w, src, dold, fold, beta);
                if (row >= 0) {
                    const T dr = fold && row < a.n_active ? s_own + beta * d_own : d_own;
                    put(dnew + row, dr);
                    put(a.q + row, acc);
                    part = (double)(dr * acc);
                    put(a.m + row, marker<T>());
                    if (!a.same_wave) put(a.rs + row, marker<T>());
                }
            }
            part = wave_sum(part);
            if (lane == 0) sums[k] = part;
        }
        store_partials(b0, b1, a.ps, [&](int b) { return xcd_workgroup(b, nb); });
    }

    // k_forward and k_backward of every group; zn: this iteration's z, zo: the
    // other buffer, which gets its marker back.
    __device__ void sweeps(const T* dnew, T* zn, T* zo, T alpha)
    {
        for (int g = 0; g < a.gl; g++) {
            const SweepGroup G = group(g);
            const bool fuse = a.fuse && g == a.gl - 1;
            my_slices(g, G.nslices, [&](int j) {
                const int row = group_row(a.lower, G.slice0 + j, j, lane, G.row0, G.nrows);
                const int ri = row >= 0 ? row : a.n;
                T rr, dd, xx, dg;
                const T acc = subtract_row(a.lower, G, j, a.m, [&] {
                    const T ro = get(a.r + ri), qq = get(a.q + ri);
                    dd = get(dnew + ri);
                    xx = a.x[ri];
                    dg = a.diag[ri];
                    rr = ro - alpha * qq;
                    return rr;
                });
                const T mm = unmarked(acc * a.omega / dg);
                double part = 0.;
                if (row >= 0) {
                    put(a.m + row, mm);
                    put(a.r + row, rr);
                    if (!a.same_wave) put(a.rs + row, unmarked(rr));
                    put(zo + row, marker<T>());
                    a.x[row] = xx + alpha * dd;
                }
                if (fuse) {
                    if (row >= 0) {
                        T t = mm;
                        t *= dg;
                        t *= a.c2;
                        const T zz = unmarked(t * a.omega / dg);
                        put(zn + row, zz);
                        part = (double)(zz * rr);
                    }
                    part = wave_sum(part);
                    if (lane == 0) put(a.pb + group(a.gl).slice0 + j, part);
                }
            });
        }
        for (int g = a.fuse; g < a.gu; g++) {
            const SweepGroup G = group(a.gl + g);
            my_slices(a.gl + g, G.nslices, [&](int j) {
                const int row = group_row(a.upper, G.slice0 + j, j, lane, G.row0, G.nrows);
                const int ri = row >= 0 ? row : a.n;
                T dg;
                const T acc = subtract_row(a.upper, G, j, zn, [&] {
                    dg = a.diag[ri];
                    T t = await(a.m + ri);
                    t *= dg;
                    t *= a.c2;
                    return t;
                });
                const T zz = unmarked(acc * a.omega / dg);
                double part = 0.;
                if (row >= 0) put(zn + row, zz);
                const T rr = a.same_wave ? get(a.r + ri) : await(a.rs + ri);
                if (row >= 0) part = (double)(zz * rr);
                part = wave_sum(part);
                if (lane == 0) put(a.pb + G.slice0 + j, part);
            });
        }
    }

    // The value wavefront 0 forms, in every thread.
    template <class Fn>
    __device__ double shared(Fn&& fn)
    {
        if (wave == 0) {
            const double t = fn();
            if (lane == 0) sums[0] = t;
        }
        __syncthreads();
        const double t = sums[0];
        __syncthreads();
        return t;
    }

    // z.r of the iterate, from the partials of its sweeps.
    __device__ double residual_dot()
    {
        for (int g = wave; g < a.gu; g += kTeamWaves) {
            const SweepGroup G = group(a.gl + g);
            const double t = team_fold(a.pb + G.slice0, G.nslices);
            if (lane == 0) sums[g] = t;
        }
        __syncthreads();
        double t = 0.;
        for (int g = 0; g < a.gu; g++) t += sums[g];
        __syncthreads();
        return t;
    }

    __device__ void run()
    {
        SolveState* st = a.st;
        const bool scribe = blockIdx.x == 0 && tid == 0;
        int K = __builtin_amdgcn_readfirstlane(st->Kp[0]);
        bool fold = __builtin_amdgcn_readfirstlane(st->fold[0]) != 0;
        const int maxK = __builtin_amdgcn_readfirstlane(st->maxK);
        const int small_breaks = __builtin_amdgcn_readfirstlane(st->small_breaks);
        double zr = st->zrp[0];
        const double tol2 = st->tol2;
        const int nb = (a.full_slices + 3) / 4;
        for (int it = 0; it < a.max_iters; it++) {
            const int p = it & 1;
            T* const dold = p ? a.d1 : a.d;
            T* const dnew = p ? a.d : a.d1;
            T* const zn = p ? a.z : a.z0;
            T* const zo = p ? a.z0 : a.z;
            // open_step (kernels.hip)
            double beta = 0.;
            if (fold) {
                const double zr_new = residual_dot();
                beta = zr_new / zr;
                K++;
                const bool cap = K >= maxK, small = ref_absolute(zr_new) < tol2;
                if (scribe) {
                    st->hist[K] = zr_new;
                    st->beta = beta;
                    st->zrp[p] = zr;
                    st->zr = zr_new;
                    st->K = K;
                    if (cap || small) {
                        st->exit_reason = cap ? SFA_EXIT_CAP : SFA_EXIT_CONVERGED;
                        st->done = 1;
                    }
                }
                zr = zr_new;
                if (cap || small) return;
            }
            product(zo, dold, dnew, fold, (T)beta);
            if (!barrier()) return;
            fold = true;
            // dad_step
            const double dAd = shared([&] { return team_fold(a.ps, nb); });
            const bool bad = !isfinite(zr) || zr < 0. || !isfinite(dAd) || dAd < 0.;
            const bool tiny = sqrt(ref_absolute(dAd)) < kMachineEpsilon && small_breaks;
            const double alpha = zr / dAd;
            if (scribe) {
                st->dAd = dAd;
                if (bad || tiny) {
                    st->exit_reason = bad ? SFA_EXIT_BREAKDOWN : SFA_EXIT_SMALL;
                    st->done = 1;
                } else {
                    st->alpha = alpha;
                }
            }
            if (bad || tiny) return;
            sweeps(dnew, zn, zo, (T)alpha);
            if (!barrier()) return;
        }
        // what the launches of an iteration of parity 0 read
        if (blockIdx.x == 0)
            for (int g = wave; g < a.gu; g += kTeamWaves) {
                const SweepGroup G = group(a.gl + g);
                const double t = team_fold(a.pb + G.slice0, G.nslices);
                if (lane == 0) a.grp[g] = t;
            }
        if (scribe) {
            st->Kp[0] = K;
            st->fold[0] = fold ? 1 : 0;
            st->zrp[0] = zr;
            st->K = K;
        }
    }
};

template <typename T>
__global__ void __launch_bounds__(kTeamThreads) k_team(TeamArgs<T> a)
{
    __shared__ double sums[kTeamMaxGroups];
    __shared__ TeamGroup groups[2 * kTeamMaxGroups];
    __shared__ int flag;
    if (a.st->done) return;  // nothing in this launch sets it before every workgroup has read it
    for (int i = threadIdx.x; i < a.gl + a.gu; i += kTeamThreads) groups[i] = a.groups[i];
    Team<T> team(a, sums, groups, &flag);
    if (!team.barrier()) return;
    team.run();
}

// z0 gets the marker in the active rows, the barriers their zeros.
template <typename T>
__global__ void __launch_bounds__(kVecBlock) k_team_start(TeamArgs<T> a)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < a.n_active) a.z0[i] = marker<T>();
    if (i < kTeamSyncWords) a.sync[i] = 0u;
    if (i == 0) a.st->team_lost = 0;
}

std::atomic<int> g_team_cus[64], g_solves[64];

}  // namespace

bool team_acquire(int device, int blocks)
{
    std::atomic<int>& used = g_team_cus[device & 63];
    int u = used.load();
    while (u + blocks <= kTeamMaxBlocks)
        if (used.compare_exchange_weak(u, u + blocks)) return true;
    return false;
}

void team_release(int device, int blocks) { g_team_cus[device & 63] -= blocks; }

SolveGuard::SolveGuard(int device) : device_(device & 63) { g_solves[device_]++; }
SolveGuard::~SolveGuard() { g_solves[device_]--; }
bool SolveGuard::alone(int device) { return g_solves[device & 63].load() <= 1; }

template <typename T>
hipError_t launch_team(hipStream_t s, const TeamArgs<T>& a, int blocks)
{
    const int n = a.n_active > kTeamSyncWords ? a.n_active : kTeamSyncWords;
    launch(k_team_start<T>, dim3((n + kVecBlock - 1) / kVecBlock), dim3(kVecBlock), s, a);
    launch(k_team<T>, dim3(blocks), dim3(kTeamThreads), s, a);
    return hipGetLastError();
}

template hipError_t launch_team<double>(hipStream_t, const TeamArgs<double>&, int);
template hipError_t launch_team<float>(hipStream_t, const TeamArgs<float>&, int);

}  // namespace sfa
