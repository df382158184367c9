// block_host.hpp -- the one-workgroup layout of a system (block_solve.hpp),
// made from its plan and its SELL parts on the device.
#pragma once

#include <vector>

#include "block_solve.hpp"
#include "host_common.hpp"
#include "launch.hpp"
#include "plan.hpp"

namespace sfa {

constexpr size_t kBlockMaxLds = 150 * 1024;  // of a CU's 160 KiB

// The loop of a solve in one workgroup (block.hip): the restart, when asked
// for, and at most max_iters iterations; zr_cont > 0: the restart continues
// the direction dprev (see BlockScalars).
template <typename T>
hipError_t launch_block_solve(hipStream_t s, const dev::BlockMatrix<T>& M, size_t lds,
                              SolveState* st, T* x, T* r, const T* b, T* d, T* d1, int restart,
                              int max_iters, double zr_cont, double zr_end, int k_cont,
                              const T* dprev);

// A system in the layout of one workgroup; lds 0: it does not fit.
template <typename T>
struct BlockLayout {
    dev::BlockMatrix<T> M{};
    size_t lds = 0;
    long long bytes = 0;
    void *cols = nullptr, *vals = nullptr, *rows = nullptr, *diag = nullptr, *list = nullptr, *heads = nullptr;

    void release()
    {
        for (void* p : {cols, vals, rows, diag, list, heads}) dev_free(p);
        cols = vals = rows = diag = list = heads = nullptr;
        lds = 0;
        bytes = 0;
    }

    // Lays the parts out when the two vectors and the lists fit the LDS and
    // the offsets their 16 bits.  Size is the whole rule: up to the largest
    // systems that fit, one workgroup per solve beats a launch per colour and
    // the lockstep engine alike.  Batches, us per iteration, lockstep engine
    // -> here, 4 / 64 / 1,024 solves at once (MI355X, FP64):
    //   7,921 rows, 5 colours, 7 entries a row     201 / 242 / 565 -> 30 / 38 / 409
    //   7,744 rows, 12 colours, 17 entries a row   549 / 630 / 1087 -> 64 / 72 / 628
    //   6,859 rows, 29 colours, 44 entries a row   2102 / 2436 / 3316 -> 201 / 209 / 1347
    // The packing is queued on stream s, which
    // the caller waits for.
    void create(const Plan& plan, const DevPartT<T>& full, const DevPartT<T>& lower,
                const DevPartT<T>& upper, const T* device_diag, hipStream_t s)
    {
        using namespace dev;
        constexpr int kBlockWaves = block_waves<T>;
        release();
        const int n = plan.n;
        if ((size_t)block_vector(n) * sizeof(T) > 65536) return;
        const bool fuse = first_backward_is_last_forward(lower, upper);
        std::vector<BlockSlice> slices;
        std::vector<std::vector<uint2>> lists(kBlockWaves);
        std::vector<int> start(2 * kBlockWaves + 1, 0);
        int chunks = 0;
        bool fits = true;
        auto phase = [&](const SellPart& p, int part, int g, unsigned flags) {
            const int first = (int)slices.size(), count = p.group_slice[g + 1] - p.group_slice[g];
            std::vector<uint2> item(count);
            for (int j = 0; j < count; j++) {
                const int sl = p.group_slice[g] + j;
                const int w = (p.slice_off[sl + 1] - p.slice_off[sl]) / kSliceRows;
                const int nc = (w + kBlockChunk - 1) / kBlockChunk;
                fits = fits && nc < kItemMaxChunks && first + j < kItemMaxSlices;
                slices.push_back({part, sl, chunks, nc});
                item[j] = make_uint2(nc > 0 ? (unsigned)chunks : 0u, (unsigned)nc | (unsigned)(first + j) << 10 |
                                                           kItemHas | flags);
                chunks += nc;
            }
            for (int w = 0; w < kBlockWaves; w++) {
                for (int j = w; j < count; j += kBlockWaves) lists[w].push_back(item[j]);
                if (w >= count) lists[w].push_back(make_uint2(0u, flags));
                lists[w].back().y |= kItemLast;
            }
        };
        // an even number of items up to here, an idle one in front if need be
        auto even = [&](int w, size_t from) {
            if ((lists[w].size() - from) % 2) lists[w].insert(lists[w].begin() + from, make_uint2(0u, 0u));
        };
        const int gl = std::max(0, plan.lower.ngroups()), gu = std::max(0, plan.upper.ngroups());
        const int back = gu - (fuse ? 1 : 0);  // CG and Jacobi: no groups
        for (int g = 0; g < gl; g++)
            phase(plan.lower, 0, g, (fuse && g == gl - 1 ? kItemFused : 0u) |
                                        (g == gl - 1 && back == 0 ? kItemSwept : 0u));
        for (int g = fuse ? 1 : 0; g < gu; g++)
            phase(plan.upper, 1, g, kItemBackward | (g == gu - 1 ? kItemSwept : 0u));
        for (int w = 0; w < kBlockWaves; w++) {
            even(w, 0);
            start[kBlockWaves + 1 + w] = (int)lists[w].size();
        }
        phase(plan.full, 2, 0, kItemProduct);
        for (int w = 0; w < kBlockWaves; w++) even(w, start[kBlockWaves + 1 + w]);
        std::vector<uint2> all;
        for (int w = 0; w < kBlockWaves; w++) {
            start[w] = (int)all.size();
            start[kBlockWaves + 1 + w] += start[w];
            all.insert(all.end(), lists[w].begin(), lists[w].end());
        }
        start[kBlockWaves] = M.list_size = (int)all.size();
        M.r_in_lds = BlockSolver<T>::lds_bytes(n, (int)all.size(), true) <= kBlockMaxLds ? 1 : 0;
        const size_t need = BlockSolver<T>::lds_bytes(n, (int)all.size(), M.r_in_lds != 0);
        if (!fits || need > kBlockMaxLds) return;
        const size_t ns = slices.size(), lanes = std::max<size_t>(ns, 1) * kSliceRows,
                     entries = std::max<size_t>(chunks, 1) * kSliceRows;
        M.sweeps = gl + back > 0 ? 1 : 0;
        M.precon = plan.method == SFA_METHOD_DIAGONAL ? device_diag : nullptr;
        M.n = n;
        M.n_active = plan.n_active;
        M.omega = T(plan.omega);
        M.c2 = T((2. - plan.omega) / plan.omega);
        BlockSlice* table = nullptr;
        try {
            cols = dev_alloc<uint2>(entries);
            vals = dev_alloc<T>(entries * kBlockChunk);
            rows = dev_alloc<unsigned>(lanes);
            diag = dev_alloc<T>(lanes);
            list = dev_alloc<uint2>(all.size());
            heads = dev_alloc<int>(start.size());
            table = dev_alloc<BlockSlice>(ns);
            SFA_HIP(hipMemcpyAsync(list, all.data(), all.size() * sizeof(uint2), hipMemcpyHostToDevice, s));
            SFA_HIP(hipMemcpyAsync(heads, start.data(), start.size() * sizeof(int), hipMemcpyHostToDevice, s));
            // items without entries, or without a slice, load the first chunk and row
            if (chunks == 0) {
                SFA_HIP(hipMemsetAsync(cols, 0, entries * sizeof(uint2), s));
                SFA_HIP(hipMemsetAsync(vals, 0, entries * kBlockChunk * sizeof(T), s));
            }
            if (ns > 0) {
                SFA_HIP(hipMemcpyAsync(table, slices.data(), ns * sizeof(BlockSlice), hipMemcpyHostToDevice, s));
                launch(k_block_pack<T>, dim3((unsigned)ns), dim3(kWave), s, (const BlockSlice*)table,
                       lower.view(), upper.view(), full.view(), n, device_diag, (uint2*)cols, (T*)vals,
                       (unsigned*)rows, (T*)diag);
                SFA_HIP(hipGetLastError());
            }
            SFA_HIP(hipStreamSynchronize(s));  // the table and the host vectors go out of use
        } catch (...) {
            (void)hipStreamSynchronize(s);
            dev_free(table);
            release();
            throw;
        }
        dev_free(table);
        M.cols = (const uint2*)cols;
        M.vals = (const T*)vals;
        M.rows = (const unsigned*)rows;
        M.diag = (const T*)diag;
        M.list = (const uint2*)list;
        M.heads = (const int*)heads;
        lds = need;
        bytes = (long long)(entries * (sizeof(uint2) + kBlockChunk * sizeof(T)) +
                            lanes * (sizeof(unsigned) + sizeof(T)) + all.size() * sizeof(uint2));
    }
};

}  // namespace sfa
