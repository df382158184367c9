// block_solve.hpp -- the CG loop of a small system inside one workgroup.
//
// A launch per colour costs 3.6-3.9 us whatever its size (half of it the
// kernel boundary), so a system of a few thousand rows spends all its time
// on launches: 53 us per iteration for a 33^2 P1 mesh whose data one CU
// reads in 2 us.  Here one workgroup runs the loop, a workgroup
// barrier between colours.  What bounds it then is the chain of a colour --
// gather, sum, division, barrier, about 0.2 us -- and every instruction
// beside it, so the layout takes work off that chain:
//   * the vectors that rows gather from live in LDS: the direction d, and one
//     vector w that is q = A d, then the residual r, then, row by row as the
//     sweeps pass, m and z (a row reads its own r or m, and others' m or z);
//   * x and r are updated once per iteration, in passes over the rows a
//     thread owns; r lives in LDS as well where there is room;
//   * the matrix is kept a second time, in chunks of four entries per lane
//     (vector loads, no test per entry), its columns as 16-bit LDS offsets,
//     row ids and diagonals stored slice by slice beside it;
//   * each wavefront walks a list of its 64-row slices made on the host, the
//     entries of the next two slices in flight across phases and barriers.
//     The loop is unrolled by those two, with loads that no branch guards: a
//     buffer chosen or filled under a branch is copied, and the copy waits
//     for the loads.  The lists therefore hold an even number of items for
//     the sweeps and for the product, and items without a slice load one.
// Every row is formed with the arithmetic, and in the entry order, of the
// one-launch-per-group kernels.
#pragma once

#include "device_common.hpp"

namespace sfa {
namespace dev {

// Wavefronts of the workgroup.  Every wavefront runs the scalar steps and walks
// its list at 4 cycles an instruction, so more of them cost more where there
// are few slices to share, and the registers of 16 do not hold two FP64 slices
// in flight: 4 / 8 / 16 wavefronts take 6.1 / 4.5 / 4.3 ms for the 48 FP64
// solves of twelve 2D systems of 36 to 4,096 rows, 8 / 16 take 0.55 / 0.75 ms
// for one SSOR solve of a 33^2 mesh, and in FP32 5.5 / 4.8 ms and 7.2 / 5.8 ms
// for those twelve systems and an H(curl) system of 5,859 rows.
template <typename T>
constexpr int block_waves = sizeof(T) == 8 ? 8 : 16;
template <typename T>
constexpr int block_threads = block_waves<T> * kWave;
constexpr int kBlockMaxWaves = 16;
constexpr int kBlockChunk = 4;       // entries per lane and chunk

// A wavefront's slice of a phase, as its list holds it: .x the slice's first
// chunk, .y = chunks (bits 0-9) | slice (bits 10-25) | flags.
constexpr unsigned kItemHas = 1u << 26;      // there is a slice (else nothing, or a phase's end)
constexpr unsigned kItemLast = 1u << 27;     // ends the wavefront's part of the phase
constexpr unsigned kItemBackward = 1u << 28;
constexpr unsigned kItemProduct = 1u << 29;
constexpr unsigned kItemFused = 1u << 30;    // forward rows whose backward step needs only their m
constexpr unsigned kItemSwept = 1u << 31;    // the last phase of the sweeps
constexpr int kItemMaxChunks = 1 << 10, kItemMaxSlices = 1 << 16;

// What a workgroup needs of a system (device pointers; see block_matrix in
// host_common.hpp).
template <typename T>
struct BlockMatrix {
    const uint2* cols;           // [chunk][lane]: 4 LDS offsets of columns
    const T* vals;               // FP64 [chunk][2][lane][2], FP32 [chunk][lane][4]
    const unsigned* rows;        // [slice][lane]: LDS offset of the row's entry
    const T* diag;               // [slice][lane]
    const uint2* list;           // the wavefronts' items
    const int* heads;            // wavefront w's from heads[w] to heads[w + 1], the
                                 // product's from heads[kBlockWaves + 1 + w]
    int list_size, r_in_lds;
    const T* precon;             // device order; CG without sweeps: z = precon r, or null: z = r
    int sweeps;                  // 1: z comes from the sweeps
    int n, n_active;
    T omega, c2;
};

// Entries of an LDS vector: n, the zero slot that padding entries read, and a
// slot that padding lanes read and write.
__host__ __device__ constexpr int block_vector(int n) { return n + 2; }

// The scalars of the recurrence.
struct BlockScalars {
    double zr, tol2, rel2;
    double alpha, beta, dAd;
    double zr_prev;  // z.r of the iterate that formed the direction
    double zr_cont;  // > 0: a restart continues the direction d formed at this z.r ...
    double zr_end;   // ... unless its z.r exceeds 1.25 times this one
    int k_cont;      // iterations of the solve that left that direction
    int K, maxK;
    int small_breaks;
    int reason, ended;
    double* hist;    // or null
};

// A value that every lane of the wavefront holds alike, in scalar registers.
__device__ inline double uniform(double v)
{
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
    return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}
__device__ inline float uniform(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(unsigned, v)));
}

// A pointer that every lane of the wavefront holds alike, to global memory:
// into scalar registers, and known not to be LDS (a pointer read from memory
// otherwise takes flat accesses, which wait for LDS as well).
template <typename P>
__device__ inline P* block_global(P* p)
{
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    using G = __attribute__((address_space(1))) P;
    return (P*)(G*)((unsigned long long)hi << 32 | lo);
}

// v of the lane CTRL names (a DPP control), +0 where there is none.
template <int CTRL, int ROWS>
__device__ inline double dpp_or_zero(double v)
{
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, ROWS, 0xf, false);
    const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), CTRL, ROWS, 0xf, false);
    return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}

// Sums over rows of 16 lanes, in each row's lane 15: a quarter of the time
// of the shuffles that go through LDS (210 ns for 64 lanes).
__device__ inline double dpp_row_sum(double v)
{
    v += dpp_or_zero<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8
    v += dpp_or_zero<0x112, 0xf>(v);
    v += dpp_or_zero<0x114, 0xf>(v);
    v += dpp_or_zero<0x118, 0xf>(v);
    return v;
}

// The wavefront's sum, in lane 63.
__device__ inline double dpp_wave_sum(double v)
{
    v = dpp_row_sum(v);
    v += dpp_or_zero<0x142, 0xa>(v);  // row_bcast 15, 31
    v += dpp_or_zero<0x143, 0xc>(v);
    return v;
}

template <typename T>
struct BlockSolver {
    static constexpr int kBlockWaves = block_waves<T>, kBlockThreads = block_threads<T>;
    static constexpr unsigned NC = 2;  // chunks of an item held in registers
    struct Item {
        unsigned at, what;  // its list entry
        uint2 c[NC];
        T v[NC][kBlockChunk];
        unsigned row;       // LDS offset
        T dg;
    };

    const BlockMatrix<T> M;
    char* w;         // LDS: block_vector(n) entries, entry n 0
    char* dl;        // LDS: the direction, likewise
    T* rl;           // LDS: r, or null
    double (*red)[kBlockMaxWaves];  // LDS [2]
    uint2* items;    // LDS: every wavefront's list
    T *x, *r;        // element i at v[i * ls]
    int ls;
    int tid, lane, wave, turn = 0;
    int cur, first, end, product;  // the next list entry to read, and the list's range
    uint2 next;                    // the list entry of the next item

    // LDS needed beside red[] for n rows and `entries` list entries.
    static constexpr size_t lds_bytes(int n, int entries, bool with_r)
    {
        return lists_at(n) + (size_t)entries * sizeof(uint2) + (with_r ? (size_t)n * sizeof(T) : 0);
    }
    static __host__ __device__ constexpr size_t lists_at(int n)
    {
        return ((size_t)2 * block_vector(n) * sizeof(T) + 15) / 16 * 16;
    }

    __device__ BlockSolver(const BlockMatrix<T>& M_, char* lds, double (*red_)[kBlockMaxWaves], T* x_,
                           T* r_, int ls_)
        : M(M_), red(red_), x(x_), r(r_), ls(ls_)
    {
        tid = threadIdx.x;
        lane = tid & (kWave - 1);
        wave = __builtin_amdgcn_readfirstlane(tid / kWave);
        w = lds;
        dl = lds + block_vector(M.n) * sizeof(T);
        items = reinterpret_cast<uint2*>(lds + lists_at(M.n));
        rl = M.r_in_lds ? reinterpret_cast<T*>(items + M.list_size) : nullptr;
        first = cur = __builtin_amdgcn_readfirstlane(M.heads[wave]);
        end = __builtin_amdgcn_readfirstlane(M.heads[wave + 1]);
        product = __builtin_amdgcn_readfirstlane(M.heads[kBlockWaves + 1 + wave]);
    }

    static __device__ T& lds_at(char* v, unsigned offset) { return *reinterpret_cast<T*>(v + offset); }
    __device__ T& wi(int i) const { return reinterpret_cast<T*>(w)[i]; }
    __device__ T& di(int i) const { return reinterpret_cast<T*>(dl)[i]; }
    __device__ T& at(T* v, int i) const { return v[(size_t)i * ls]; }

    // Lists to LDS; the caller synchronises.
    __device__ void load_lists()
    {
        for (int i = tid; i < M.list_size; i += kBlockThreads) items[i] = M.list[i];
    }

    // fn(i, v_i) for the rows this thread owns, four of a vector's loads in
    // flight; STORE: fn's result is stored back.  v has stride `stride`.
    template <bool STORE, class Fn>
    __device__ void own_rows(T* v, int stride, Fn&& fn) const
    {
        constexpr int U = 4;
        for (int i0 = tid; i0 < M.n_active; i0 += U * kBlockThreads) {
            T t[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = i0 + u * kBlockThreads;
                t[u] = v[(size_t)(i < M.n_active ? i : i0) * stride];
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = i0 + u * kBlockThreads;
                if (i < M.n_active) {
                    if constexpr (STORE) v[(size_t)i * stride] = fn(i, t[u]);
                    else fn(i, t[u]);
                }
            }
        }
    }
    // The same over r, wherever it lives.
    template <bool STORE, class Fn>
    __device__ void own_r(Fn&& fn) const
    {
        if (rl) own_rows<STORE>(rl, 1, fn);
        else own_rows<STORE>(r, ls, fn);
    }

    // Sum over the workgroup in a fixed order; every thread gets the same
    // bits.  One barrier; the two buffers alternate.
    __device__ double sum(double part)
    {
        const double s = dpp_wave_sum(part);
        if (lane == kWave - 1) red[turn][wave] = s;
        __syncthreads();
        const double mine = (lane & 15) < kBlockWaves ? red[turn][lane & 15] : 0.;
        const unsigned long long t = __builtin_bit_cast(unsigned long long, dpp_row_sum(mine));
        turn ^= 1;
        const unsigned lo = __builtin_amdgcn_readlane((unsigned)t, 15);
        const unsigned hi = __builtin_amdgcn_readlane((unsigned)(t >> 32), 15);
        return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
    }

    // Chunk k of the values of an item.
    __device__ void load_values(unsigned chunk, T* v) const
    {
        if constexpr (sizeof(T) == 8) {
            typedef double D2 __attribute__((ext_vector_type(2)));
            const D2* p = reinterpret_cast<const D2*>(M.vals) + (chunk * 2u * kWave + (unsigned)lane);
            const D2 a = p[0], b = p[kWave];
            v[0] = a[0], v[1] = a[1], v[2] = b[0], v[3] = b[1];
        } else {
            typedef float F4 __attribute__((ext_vector_type(4)));
            const F4 a = reinterpret_cast<const F4*>(M.vals)[chunk * (unsigned)kWave + (unsigned)lane];
            v[0] = a[0], v[1] = a[1], v[2] = a[2], v[3] = a[3];
        }
    }

    // Starts the walk at list entry i.
    __device__ void seek(int i)
    {
        cur = i;
        next = items[cur];
    }

    // Loads the wavefront's next item.
    __device__ void fetch(Item& I)
    {
        I.at = __builtin_amdgcn_readfirstlane(next.x);
        I.what = __builtin_amdgcn_readfirstlane(next.y);
        cur = cur + 1 == end ? first : cur + 1;
        next = items[cur];
        if (!(I.what & kItemHas)) return;
        const unsigned nc = I.what & (kItemMaxChunks - 1);
        const unsigned slot = ((I.what >> 10) & (kItemMaxSlices - 1)) * kWave + (unsigned)lane;
        I.row = M.rows[slot];
        I.dg = M.diag[slot];
#pragma unroll
        for (unsigned k = 0; k < NC; k++) {
            if (k < nc) {
                I.c[k] = M.cols[(I.at + k) * kWave + (unsigned)lane];
                load_values(I.at + k, I.v[k]);
            }
        }
    }

    // acc - sum of one chunk, and of two: the gathers of both go out together.
    static __device__ T apply_chunk(T acc, uint2 c, const T* v, char* vec)
    {
        const T g0 = lds_at(vec, c.x & 0xffffu), g1 = lds_at(vec, c.x >> 16);
        const T g2 = lds_at(vec, c.y & 0xffffu), g3 = lds_at(vec, c.y >> 16);
        acc -= v[0] * g0;
        acc -= v[1] * g1;
        acc -= v[2] * g2;
        acc -= v[3] * g3;
        return acc;
    }
    static __device__ T apply_chunks(T acc, uint2 c, const T* v, uint2 e, const T* u, char* vec)
    {
        const T g0 = lds_at(vec, c.x & 0xffffu), g1 = lds_at(vec, c.x >> 16);
        const T g2 = lds_at(vec, c.y & 0xffffu), g3 = lds_at(vec, c.y >> 16);
        const T h0 = lds_at(vec, e.x & 0xffffu), h1 = lds_at(vec, e.x >> 16);
        const T h2 = lds_at(vec, e.y & 0xffffu), h3 = lds_at(vec, e.y >> 16);
        acc -= v[0] * g0;
        acc -= v[1] * g1;
        acc -= v[2] * g2;
        acc -= v[3] * g3;
        acc -= u[0] * h0;
        acc -= u[1] * h1;
        acc -= u[2] * h2;
        acc -= u[3] * h3;
        return acc;
    }

    // Two chunks of a row, chunk k and the one after it (or again the last).
    struct Pair {
        uint2 c[2];
        T v[2][kBlockChunk];
    };
    __device__ void load_pair(Pair& p, unsigned at, unsigned k, unsigned nc) const
    {
#pragma unroll
        for (unsigned j = 0; j < 2; j++) {
            const unsigned chunk = at + min(k + j, nc - 1);
            p.c[j] = M.cols[chunk * kWave + (unsigned)lane];
            load_values(chunk, p.v[j]);
        }
    }
    static __device__ T apply_pair(T acc, const Pair& p, unsigned k, unsigned nc, char* vec)
    {
        return k + 1 < nc ? apply_chunks(acc, p.c[0], p.v[0], p.c[1], p.v[1], vec)
                          : apply_chunk(acc, p.c[0], p.v[0], vec);
    }

    // acc - sum_k v_k * vec[c_k] over the row of an item, entries in order.
    // Chunks past the two in registers are loaded two pairs at a time into
    // others, one pair ahead of its use (refilling the item's own registers
    // in a loop would wait for the next item's loads as well).
    __device__ T finish(const Item& I, char* vec, T acc) const
    {
        const unsigned nc = __builtin_amdgcn_readfirstlane(I.what) & (kItemMaxChunks - 1);
        const unsigned at = __builtin_amdgcn_readfirstlane(I.at);
        Pair A, B;
        if (nc > NC) load_pair(A, at, NC, nc);
#pragma unroll
        for (unsigned k = 0; k < NC; k += 2) {
            if (k + 1 < nc) acc = apply_chunks(acc, I.c[k], I.v[k], I.c[k + 1], I.v[k + 1], vec);
            else if (k < nc) acc = apply_chunk(acc, I.c[k], I.v[k], vec);
        }
        if (nc <= NC) return acc;
        for (unsigned k = NC;;) {
            load_pair(B, at, k + 2, nc);
            acc = apply_pair(acc, A, k, nc, vec);
            if ((k += 2) >= nc) return acc;
            load_pair(A, at, k + 2, nc);
            acc = apply_pair(acc, B, k, nc, vec);
            if ((k += 2) >= nc) return acc;
        }
    }

    // One slice of a sweep: forward m = (r - L m) w / diag (:1245-1261),
    // backward z = (m diag c2 - U z) w / diag (:1263-1303), both in w.
    __device__ void sweep(const Item& I)
    {
        const unsigned what = __builtin_amdgcn_readfirstlane(I.what);
        if (!(what & kItemHas)) return;
        T acc = lds_at(w, I.row);
        if (what & kItemBackward) {
            acc *= I.dg;
            acc *= M.c2;
        }
        acc = finish(I, w, acc) * M.omega / I.dg;
        if (what & kItemFused) {
            acc *= I.dg;
            acc *= M.c2;
            acc = acc * M.omega / I.dg;
        }
        lds_at(w, I.row) = acc;
    }

    // One slice of q = A d, into w (:1197-1212, summed with the other sign,
    // which rounds alike); returns the lane's share of d.Ad.
    __device__ double multiply(const Item& I)
    {
        if (!(__builtin_amdgcn_readfirstlane(I.what) & kItemHas)) return 0.;
        const T acc = -finish(I, dl, T(0));
        lds_at(w, I.row) = acc;
        return (double)(lds_at(dl, I.row) * acc);
    }

    // w = r = b - A x (:1061-1075).
    __device__ void residual(const T* b)
    {
        for (int i = tid; i < block_vector(M.n); i += kBlockThreads) wi(i) = i < M.n ? at(x, i) : T(0);
        __syncthreads();
        seek(product);
        for (int k = product; k < end; k++) {
            Item I;
            fetch(I);
            if ((I.what & kItemHas) && I.row / sizeof(T) < (unsigned)M.n) {
                const size_t i = (size_t)(I.row / sizeof(T)) * ls;
                r[i] = finish(I, w, b[i]);
            }
        }
        __syncthreads();
        for (int i = tid; i < block_vector(M.n); i += kBlockThreads)
            wi(i) = i < M.n_active ? at(r, i) : T(0);
    }

    // The restart (when asked for) and iterations until the loop has ended or
    // max_iters of them have run.  Reads and writes x, r and d (dl); between
    // calls nothing else is kept.  s is in LDS: read at the start, written by
    // thread 0.
    __device__ void run(const T* b, bool restart, int max_iters, BlockScalars& s)
    {
        // every loop and branch below is uniform, and must be seen to be
        restart = __builtin_amdgcn_readfirstlane(restart) != 0;
        max_iters = __builtin_amdgcn_readfirstlane(max_iters);
        double zr = uniform(s.zr), tol2 = uniform(s.tol2);
        int K = __builtin_amdgcn_readfirstlane(s.K), maxK = __builtin_amdgcn_readfirstlane(s.maxK);
        double* const hist = block_global(s.hist);
        const bool small_breaks = __builtin_amdgcn_readfirstlane(s.small_breaks) != 0;
        T alpha = T(0);
        if (restart) {
            residual(b);
        } else {
            for (int i = tid; i < block_vector(M.n); i += kBlockThreads) wi(i) = T(0);
        }
        if (rl)
            own_rows<false>(r, ls, [&](int i, T ri) { rl[i] = ri; });
        __syncthreads();

        auto residual_dot = [&]() -> double {
            double t = 0.;
            own_r<false>([&](int i, T ri) { t += (double)(wi(i) * ri); });
            return sum(t);
        };
        // The end of the restart's sweeps, at z.r: the first loop-head test
        // (:1156-1190) and the direction, d = z or the one that is continued.
        auto restarted = [&]() -> bool {
            const double t = residual_dot();
            const double rel2 = uniform(s.rel2), zr_cont = uniform(s.zr_cont), zr_end = uniform(s.zr_end);
            if (rel2 > 0.) tol2 = uniform(rel2 * ref_absolute(t));
            zr = t;
            K = 0;
            const bool ended = ref_absolute(t) < tol2;
            const bool cont = zr_cont > 0. && !ended && t <= 1.25 * zr_end;
            const double beta = cont ? t / zr_cont : 0.;
            if (cont) maxK = min(M.n, max(100, 3 * __builtin_amdgcn_readfirstlane(s.k_cont)));
            for (int i = tid; i < M.n_active; i += kBlockThreads)
                di(i) = cont ? wi(i) + (T)beta * di(i) : wi(i);
            __syncthreads();
            if (tid == 0) {
                if (hist) hist[0] = t;
                s.zr_cont = 0.;
                s.beta = beta;
                if (ended) {
                    s.reason = SFA_EXIT_CONVERGED;
                    s.ended = 1;
                }
            }
            return !ended;
        };
        // The end of the product, at d.Ad: breakdown tests, alpha (:1215-1231)
        // and r.
        auto multiplied = [&](double dAd) -> bool {
            const bool num_bad = !isfinite(zr) || zr < 0.;
            const bool den_bad = !isfinite(dAd) || dAd < 0.;
            const bool small = ref_absolute(dAd) < kMachineEpsilon * kMachineEpsilon &&
                               sqrt(ref_absolute(dAd)) < kMachineEpsilon;
            const bool stop = num_bad || den_bad || (small && small_breaks);
            const double a = zr / dAd;
            if (tid == 0) {
                s.dAd = dAd;
                if (stop) {
                    s.reason = num_bad || den_bad ? SFA_EXIT_BREAKDOWN : SFA_EXIT_SMALL;
                    s.ended = 1;
                } else {
                    s.alpha = a;
                }
            }
            if (stop) return false;
            alpha = uniform((T)a);
            own_r<true>([&](int i, T ri) {
                const T rr = ri - alpha * wi(i);
                wi(i) = rr;
                return rr;
            });
            __syncthreads();
            return true;
        };
        // The end of the sweeps: z.r, beta, K, the exit tests (:1299-1307), x
        // and d.
        auto swept = [&]() -> bool {
            const double t = residual_dot();
            const double beta = t / zr;
            const double before = zr;
            zr = t;
            K++;
            max_iters--;
            const bool cap = K >= maxK;
            const bool ended = cap || ref_absolute(t) < tol2;
            own_rows<true>(x, ls, [&](int i, T xx) {
                const T dd = di(i);
                if (!ended) di(i) = wi(i) + (T)beta * dd;
                return xx + alpha * dd;
            });
            __syncthreads();
            if (tid == 0) {
                if (hist) hist[K] = t;
                s.beta = beta;
                s.zr_prev = before;
                if (ended) {
                    s.reason = cap ? SFA_EXIT_CAP : SFA_EXIT_CONVERGED;
                    s.ended = 1;
                }
            }
            return !ended && max_iters > 0;
        };

        if (restart || max_iters > 0) {
            Item P, Q;
            bool starting = restart;
            seek(restart ? first : product);  // without sweeps the two are one
            fetch(P);
            fetch(Q);
            for (bool skip = !restart;; skip = false) {
                if (!skip) {
                    if (!M.sweeps)
                        own_r<false>([&](int i, T ri) { wi(i) = M.precon ? M.precon[i] * ri : ri; });
                    while (M.sweeps) {  // a barrier between phases
                        sweep(P);
                        const unsigned p = __builtin_amdgcn_readfirstlane(P.what);
                        fetch(P);
                        if (p & kItemLast) __syncthreads();
                        sweep(Q);
                        const unsigned q = __builtin_amdgcn_readfirstlane(Q.what);
                        fetch(Q);
                        if (q & kItemLast) __syncthreads();
                        if ((q & (kItemLast | kItemSwept)) == (kItemLast | kItemSwept)) break;
                    }
                    if (!(starting ? restarted() && max_iters > 0 : swept())) break;
                    starting = false;
                }
                double part = 0.;
                for (;;) {
                    part += multiply(P);
                    fetch(P);
                    part += multiply(Q);
                    const unsigned q = __builtin_amdgcn_readfirstlane(Q.what);
                    fetch(Q);
                    if (q & kItemLast) break;
                }
                if (!multiplied(sum(part))) break;
            }
        }
        if (rl)
            for (int i = tid; i < M.n_active; i += kBlockThreads) at(r, i) = rl[i];
        if (tid == 0) {
            s.zr = zr;
            s.tol2 = tol2;
            s.K = K;
            s.maxK = maxK;
        }
        __syncthreads();
    }
};

// One slice of a SELL part into the workgroup's layout.
struct BlockSlice {
    int part;    // 0 lower, 1 upper, 2 full
    int slice;   // of that part
    int chunk0, chunks;
};

template <typename T>
__global__ void __launch_bounds__(kWave) k_block_pack(const BlockSlice* slices, SellViewT<T> lower,
                                                      SellViewT<T> upper, SellViewT<T> full, int n,
                                                      const T* diag, uint2* cols, T* vals,
                                                      unsigned* rows, T* pdiag)
{
    const int s = blockIdx.x;
    const int lane = threadIdx.x;
    const BlockSlice S = slices[s];
    const SellViewT<T> A = S.part == 0 ? lower : S.part == 1 ? upper : full;
    const int row = A.rows[S.slice * kWave + lane];
    rows[s * kWave + lane] = (unsigned)((row >= 0 ? row : n + 1) * (int)sizeof(T));
    pdiag[s * kWave + lane] = row >= 0 ? diag[row] : T(1);
    const int o0 = A.off[S.slice], w = (A.off[S.slice + 1] - o0) / kWave;
    for (int k = 0; k < S.chunks; k++) {
        unsigned c[kBlockChunk];
        T v[kBlockChunk];
        for (int u = 0; u < kBlockChunk; u++) {
            const int e = k * kBlockChunk + u;
            const bool has = row >= 0 && e < w;
            c[u] = (unsigned)(has ? A.cols[o0 + e * kWave + lane] : n) * (unsigned)sizeof(T);
            v[u] = has ? A.vals[o0 + e * kWave + lane] : T(0);
        }
        const size_t chunk = (size_t)S.chunk0 + k;
        cols[chunk * kWave + lane] = make_uint2(c[0] | c[1] << 16, c[2] | c[3] << 16);
        for (int u = 0; u < kBlockChunk; u++) {
            if (sizeof(T) == 8)
                vals[((chunk * 2 + u / 2) * kWave + lane) * 2 + u % 2] = v[u];
            else
                vals[(chunk * kWave + lane) * kBlockChunk + u] = v[u];
        }
    }
}

}  // namespace dev
}  // namespace sfa
