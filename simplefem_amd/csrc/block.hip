// block.hip -- solves of a System whose loop fits one workgroup.
#include "block_solve.hpp"
#include "kernels.hpp"
#include "launch.hpp"

namespace sfa {
namespace {

using namespace dev;

// The restart (when asked for) and up to max_iters iterations of a solve, one
// workgroup; the state, x, r and the direction are left as the launches of
// an iteration leave them (the direction in slot K % 2, d for 0 and d1 for
// 1).  A restart takes zr_cont, zr_end and k_cont as BlockScalars describes
// them, dprev being the direction to continue.
template <typename T>
__global__ void __launch_bounds__(block_threads<T>) k_block_solve(BlockMatrix<T> M, SolveState* st,
                                                               T* x, T* r, const T* b, T* d,
                                                               T* d1, int restart, int max_iters,
                                                               double zr_cont, double zr_end,
                                                               int k_cont, const T* dprev)
{
    constexpr int kBlockThreads = block_threads<T>;
    extern __shared__ __align__(16) char lds[];
    __shared__ double red[2][kBlockMaxWaves];
    __shared__ BlockScalars c;
    const int tid = threadIdx.x;
    if (st->done) return;
    BlockSolver<T> B(M, lds, red, x, r, 1);
    B.load_lists();
    const bool cont = restart && zr_cont > 0.;
    const T* const from = restart ? dprev : (st->K & 1) ? d1 : d;
    // rows the variant skips keep the direction the scratch vectors start with
    const T skipped = M.sweeps ? T(0) : (T)NAN;
    for (int i = tid; i < block_vector(M.n); i += kBlockThreads)
        B.di(i) = i >= M.n ? T(0) : i >= M.n_active ? skipped : restart && !cont ? T(0) : from[i];
    if (tid == 0) {
        c = BlockScalars{};
        c.zr = st->zr;
        c.tol2 = st->tol2;
        c.rel2 = st->rel2;
        c.zr_cont = cont ? zr_cont : 0.;
        c.zr_end = zr_end;
        c.k_cont = k_cont;
        c.K = st->K;
        c.maxK = st->maxK;
        c.small_breaks = st->small_breaks;
        c.reason = st->exit_reason;
        c.hist = st->hist;
        c.zr_prev = st->zrp[st->K & 1];
        c.alpha = st->alpha;
        c.beta = st->beta;
        c.dAd = st->dAd;
    }
    __syncthreads();
    B.run(b, restart != 0, max_iters, c);
    T* const to = (c.K & 1) ? d1 : d;
    for (int i = tid; i < M.n_active; i += kBlockThreads) to[i] = B.di(i);
    if (tid == 0) {
        st->continued = cont && c.beta > 0. ? 1 : 0;
        st->zr = c.zr;
        st->tol2 = c.tol2;
        if (c.rel2 > 0.) st->tol = sqrt(c.tol2);
        st->K = c.K;
        st->maxK = c.maxK;
        st->zrp[c.K & 1] = c.zr_prev;
        st->alpha = c.alpha;
        st->beta = c.beta;
        st->dAd = c.dAd;
        st->exit_reason = c.reason;
        st->done = c.ended;
    }
}

}  // namespace

template <typename T>
hipError_t launch_block_solve(hipStream_t s, const dev::BlockMatrix<T>& M, size_t lds,
                              SolveState* st, T* x, T* r, const T* b, T* d, T* d1, int restart,
                              int max_iters, double zr_cont, double zr_end, int k_cont,
                              const T* dprev)
{
    return launch_lds(k_block_solve<T>, dim3(1), dim3(dev::block_threads<T>), lds, s, M, st, x, r, b, d,
                      d1, restart, max_iters, zr_cont, zr_end, k_cont, dprev);
}

#define SFA_INSTANTIATE_BLOCK(T)                                                               \
    template hipError_t launch_block_solve<T>(hipStream_t, const dev::BlockMatrix<T>&, size_t, \
                                              SolveState*, T*, T*, const T*, T*, T*, int, int, \
                                              double, double, int, const T*);
SFA_INSTANTIATE_BLOCK(double)
SFA_INSTANTIATE_BLOCK(float)

}  // namespace sfa
