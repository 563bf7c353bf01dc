// vx_edits.hip -- edit lists to Batch buffers on the device.
//
// Input: per tree a contiguous range of edits (x, y, z, value) in submission order.  The
// last write to a voxel wins and is recorded in a zeroed dense Batch exactly as
// Batch::just_set does (core/batch.rs:145-175): a non-default value sets the slot's set bit,
// the default value sets its clear bit, the value is stored either way.
//
// Two launches over arrays of the edited trees' voxels: k_edit_mark takes the maximum of the
// submission indices of each voxel, k_edit_build makes an edited brick's masks and values from
// its eight winners, leaves their array zero again, and clears the masks of the call before.  (A stable radix sort by (tree, Morton
// path), whose run ends were scattered and later cleared, took 23 launches and 640 us on 4.4 M
// sphere edits over 700 trees of 32^3 against 93 us here; 18 launches against 2 on 3000 edits.)
// The winners take four bytes per voxel, so a call of very many voxels goes in windows of
// consecutive trees, two launches each, that share one array of them (kEditWindow).
#include <hip/hip_runtime.h>

#include <cstring>

#include "vx_device.h"

namespace vx {

// States of a cell of 8^3 voxels: its masks are zero; edited by this call; built by it, so that
// the next call clears the masks unless it edits the cell again.
constexpr uint8_t kCellClear = 0, kCellEdited = 1, kCellBuilt = 2;

__device__ inline uint32_t spread3(uint32_t v) {
    v &= 0x3FFu;
    v = (v | (v << 16)) & 0x30000FFu;
    v = (v | (v << 8)) & 0x300F00Fu;
    v = (v | (v << 4)) & 0x30C30C3u;
    v = (v | (v << 2)) & 0x9249249u;
    return v;
}

// The last of trees [lo, hi) whose first edit is at or before e.
__device__ inline uint32_t tree_of_edit(const EditTree* trees, uint32_t lo, uint32_t hi, uint64_t e) {
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (trees[mid].first <= e) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Per edit e of [first, n): win[voxel - v0] = the largest submission index (counted from first)
// + 1, and the voxel's cell of 8^3 is marked.  A coordinate outside its tree (a panic in the
// reference's Vec indexing) fails the tree.  A block's run of edits (per * 256) mostly lies in one tree, found once.
// Bound by the rate of the atomics.  Lanes also reset the status and count of every tree of
// the call, edited or not (a tree without edits is not applied: status 0).
__global__ __launch_bounds__(256) void k_edit_mark(uint64_t first, uint64_t n, uint32_t per, EditTree* trees, uint32_t ntrees,
                                                   const int32_t* xyz, uint64_t v0, uint32_t* win, uint8_t* dirty, uint32_t nall,
                                                   int32_t* status, uint32_t* per_tree) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nall; i += gridDim.x * blockDim.x) {
        status[i] = 0;
        if (per_tree) per_tree[i] = 0;
    }
    __shared__ uint32_t s_t[2];
    const uint64_t run = (uint64_t)per * 256;
    for (uint64_t e0 = first + (uint64_t)blockIdx.x * run; e0 < n; e0 += (uint64_t)gridDim.x * run) {
        const uint64_t e1 = min(e0 + run, n);
        if (threadIdx.x < 2) s_t[threadIdx.x] = tree_of_edit(trees, 0, ntrees, threadIdx.x ? e1 - 1 : e0);
        __syncthreads();
        const uint32_t t0 = s_t[0], t1 = s_t[1];
        __syncthreads();
        for (uint64_t e = e0 + threadIdx.x; e < e1; e += 256) {
            const uint32_t t = t0 == t1 ? t0 : tree_of_edit(trees, t0, t1 + 1, e);
            const EditTree tr = trees[t];
            if (tr.vbase == ~0ull) continue;  // rejected on the host
            const uint32_t x = (uint32_t)xyz[3 * e], y = (uint32_t)xyz[3 * e + 1], z = (uint32_t)xyz[3 * e + 2];
            const uint32_t lim = 1u << tr.depth;
            if (x >= lim || y >= lim || z >= lim) {  // (negative coordinates too)
                trees[t].status = -4;
                continue;
            }
            const uint64_t v = tr.vbase + (spread3(x) | (spread3(y) << 1) | (spread3(z) << 2));
            atomicMax(&win[v - v0], (uint32_t)(e - first) + 1u);
            dirty[v >> 9] = kCellEdited;
        }
    }
}

// A wavefront takes `per` cells of 8^3 voxels (64 bricks) in turn, a lane per brick: masks for
// the bricks of a cell edited by this call, and values for those that have an edit.  A cell
// that only an earlier call edited gets its masks cleared, any other is left: its masks are
// zero.  (300 trees of 128^3 with 20 edits each have 1.2 M cells, 6000 of them edited: the call
// takes 947 us, 1005 with the masks of every cell written.)
template <typename T>
__global__ __launch_bounds__(256) void k_edit_build(uint64_t ncells, uint32_t per, const T* edit_values, uint32_t* win,
                                                    uint8_t* dirty, uint16_t* masks, T* values) {
    struct __align__(sizeof(T) * 8 < 16 ? sizeof(T) * 8 : 16) Vox8 {
        T v[8];
    };
    const uint32_t lane = threadIdx.x & 63u;
    for (uint64_t c0 = ((uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * per; c0 < ncells; c0 += (uint64_t)gridDim.x * 4 * per) {
        // (per is 64 at most)
        const uint8_t state = lane < per && c0 + lane < ncells ? dirty[c0 + lane] : (uint8_t)kCellClear;
        for (uint64_t todo = __ballot(state != kCellClear); todo; todo &= todo - 1) {  // uniform over the wavefront
            const int k = __ffsll((unsigned long long)todo) - 1;
            const uint64_t b = (c0 + k) * 64 + lane;
            uint32_t m = 0;
            if (__builtin_amdgcn_readlane((int)state, k) == (int)kCellEdited) {
                uint4* w4 = (uint4*)(win + 8 * b);
                const uint4 lo = w4[0], hi = w4[1];
                const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                if ((lo.x | lo.y | lo.z | lo.w | hi.x | hi.y | hi.z | hi.w) != 0) {
                    Vox8 q;
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        q.v[i] = (T)0;
                        if (w[i]) q.v[i] = edit_values[w[i] - 1];
                    }
#pragma unroll
                    for (int i = 0; i < 8; i++)
                        if (w[i]) m |= 1u << (q.v[i] != 0 ? i : i + 8);
                    w4[0] = w4[1] = make_uint4(0u, 0u, 0u, 0u);
                    *(Vox8*)(values + 8 * b) = q;
                }
            }
            masks[b] = (uint16_t)m;  // set mask, clear mask
        }
        if (state != kCellClear) dirty[c0 + lane] = state == kCellEdited ? kCellBuilt : kCellClear;
    }
}

}  // namespace vx
