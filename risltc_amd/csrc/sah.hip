// sah.hip -- binned-SAH BVH builder on the device.
//
// The reference traces shadow rays against a hardware acceleration structure
// (src/scene.c:142-406) whose build the driver performs. This builder gives
// the project's traversal a tree of comparable quality: top-down, every node
// split by the surface area heuristic over 16 centroid bins per axis, down
// to one triangle per leaf. On the 1M-triangle city it visits 3.5x fewer
// nodes per shadow ray than the Morton-code LBVH (lbvh.hip), which stays
// available as the alternative builder.
//
// Every decision is a deterministic function of the triangle boxes:
//   * node box and centroid bounds are min/max reductions (exact, and done
//     on an order-preserving integer image of the floats, so -0 < +0 like
//     the CPU restatement);
//   * a centroid's bin is min(15, int((c - lo) * (16 / extent))) in IEEE
//     float;
//   * bins hold counts and box unions (exact); the cost of split s on axis a
//     is n_l * area(l) + n_r * area(r), area = dx dy + dy dz + dz dx,
//     evaluated in a fixed order, the first minimum over (axis, bin) wins;
//     with no axis of non-zero extent the node is halved in index order;
//   * the partition is stable.
// The CPU oracle restates the same steps (orc_bvh_build_sah) and obtains the
// identical tree; the node numbering differs, the pre-order layout does not.
//
// How it is spread over the chip. Nodes above kSahSmall triangles are split
// level by level, in chunks of kSahChunk triangles, one work-group each: bins
// (LDS histogram, then one atomic per bin), the split (one wave per node, one
// lane per axis and bin), the scatter (a chunk's place follows from the bin
// counts of the chunks before it). With one work-group per node and the split
// on one lane, the root alone took 22 ms of one CU. Smaller subtrees are built
// by one wave each from LDS: first its nodes above 16 triangles with all 64
// lanes, then the rest breadth-first, four nodes at a time on 16 lanes each;
// a lane evaluates one split by walking the node's triangles, so there are
// no histograms. 1M triangles: 77 ms before, 3.0 ms now (levels 1.7, small
// subtrees 1.3); 230k: 40 and 1.2; 322: 10.8 and 0.2.
#include <hip/hip_runtime.h>

#include "devmath.hpp"
#include "kernels.hpp"

namespace rl {

constexpr int kSahBins = 16;
constexpr uint32_t kSahSmall = 256;
constexpr uint32_t kSahChunk = 2048;
constexpr int kBinWords = 7;  // count, box low xyz, box high xyz
constexpr int kNodeBinWords = 3 * kSahBins * kBinWords;

// order-preserving image of a float in a signed int (finite values)
__device__ __forceinline__ int fkey(float f) {
    int b = __float_as_int(f);
    return b >= 0 ? b : (b ^ 0x7FFFFFFF);
}
__device__ __forceinline__ float kfloat(int k) { return __int_as_float(k >= 0 ? k : (k ^ 0x7FFFFFFF)); }
constexpr int kKeyPosInf = 0x7F800000;            // +inf
constexpr int kKeyNegInf = (int)(0xFF800000u ^ 0x7FFFFFFFu);  // -inf

__device__ __forceinline__ int bin_of(float c, float lo, float scale) {
    int b = (int)((c - lo) * scale);
    return b < kSahBins - 1 ? b : kSahBins - 1;
}

__device__ __forceinline__ float box_area(const int (&b)[6]) {
    float dx = kfloat(b[3]) - kfloat(b[0]), dy = kfloat(b[4]) - kfloat(b[1]), dz = kfloat(b[5]) - kfloat(b[2]);
    return dx * dy + dy * dz + dz * dx;
}

// low corner and bins per unit of an axis (scale 0: not used for splitting)
__device__ __forceinline__ void axis_scale(int klo, int khi, float& lo, float& scale) {
    lo = kfloat(klo);
    const float ext = kfloat(khi) - lo;
    scale = ext > 0.0f ? (float)kSahBins / ext : 0.0f;
}

__device__ __forceinline__ void empty_box(int (&b)[6]) {
#pragma unroll
    for (int c = 0; c < 6; ++c) b[c] = c < 3 ? kKeyPosInf : kKeyNegInf;
}

// min (c < 3) or max over aligned groups of W lanes
template <int W>
__device__ __forceinline__ int group_min(int v) {
#pragma unroll
    for (int o = W / 2; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o));
    return v;
}
template <int W>
__device__ __forceinline__ int group_max(int v) {
#pragma unroll
    for (int o = W / 2; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o));
    return v;
}

__device__ __forceinline__ void sah_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// the cheapest split over aligned groups of W lanes: the lowest cost, then the
// lowest key (axis * 16 + bin, the order in which the first minimum wins).
// Costs that are not below infinity never win (key -1).
template <int W>
__device__ __forceinline__ void group_best(float& cost, int& key) {
#pragma unroll
    for (int o = W / 2; o > 0; o >>= 1) {
        const float c = __shfl_xor(cost, o);
        const int k = __shfl_xor(key, o);
        if (k >= 0 && (key < 0 || c < cost || (c == cost && k < key))) {
            cost = c;
            key = k;
        }
    }
}

// ---- large nodes --------------------------------------------------------------------
struct SahSlot {
    int node;
    uint32_t first, count, chunk0;
    int cb[6];            // centroid bounds (keys)
    int axis, bin;        // the split (axis -1: halved in index order)
    uint32_t nl;
    int child[2];         // next level's slot of each child, or -1
};

// the state of one level; levels alternate between two of them
struct SahLevel {
    SahSlot* slots;
    int* bins;              // kNodeBinWords per slot
    uint32_t* chunk_slot;
    uint32_t* idx;          // triangle order of the level
};

struct SahWork {
    SahLevel level[2];
    uint32_t* chunk_counts;  // 3 * 16 per chunk
    uint32_t* counters;      // ring of 4 levels: nodes at 2 (level & 3), chunks beside; 8: small subtrees
    uint32_t* small;         // node | level parity of its triangle order << 31
};

__device__ __forceinline__ void slot_init(SahSlot& s, int* bins, int node, uint32_t first, uint32_t count,
                                          uint32_t chunk0, uint32_t lane, uint32_t lanes) {
    if (lane == 0u) {
        s.node = node;
        s.first = first;
        s.count = count;
        s.chunk0 = chunk0;
#pragma unroll
        for (int c = 0; c < 6; ++c) s.cb[c] = c < 3 ? kKeyPosInf : kKeyNegInf;
    }
    for (uint32_t k = lane; k < (uint32_t)kNodeBinWords; k += lanes) {
        const uint32_t w = k % kBinWords;
        bins[k] = w == 0u ? 0 : (w < 4u ? kKeyPosInf : kKeyNegInf);
    }
}

// the root: one slot above kSahSmall triangles, else one small subtree
__global__ void __launch_bounds__(256) sah_init_kernel(SahTree T, SahWork W, uint32_t n) {
    const uint32_t t = threadIdx.x;
    const bool large = n > kSahSmall;
    const uint32_t chunks = (n + kSahChunk - 1u) / kSahChunk;
    if (t < 8u) W.counters[t] = large && t < 2u ? (t == 0u ? 1u : chunks) : 0u;
    if (t == 8u) W.counters[8] = large ? 0u : 1u;
    if (t == 0u) {
        *T.node_counter = 1u;
        T.first[0] = 0;
        T.count[0] = (int)n;
        T.parent[0] = -1;
        W.small[0] = 0u;
    }
    if (!large) return;
    slot_init(W.level[0].slots[0], W.level[0].bins, 0, 0u, n, 0u, t, 256u);
    for (uint32_t k = t; k < chunks; k += 256u) W.level[0].chunk_slot[k] = 0u;
}

// reduces centroid keys over the work-group (256 lanes) and adds them to the
// bounds of a slot (null: none)
__device__ __forceinline__ void bounds_atomic(const int (&lo)[3], const int (&hi)[3], int* cb, int (*part)[6]) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int l = group_min<64>(lo[a]), h = group_max<64>(hi[a]);
        if (lane == 0u) {
            part[wave][a] = l;
            part[wave][3 + a] = h;
        }
    }
    __syncthreads();
    const uint32_t t = threadIdx.x;
    if (cb && t < 6u) {
        int v = part[0][t];
        for (int w = 1; w < 4; ++w) v = t < 3u ? min(v, part[w][t]) : max(v, part[w][t]);
        if (t < 3u) atomicMin(&cb[t], v);
        else atomicMax(&cb[t], v);
    }
    __syncthreads();
}

// triangle boxes (keys) and centroids, and the root's centroid bounds
__global__ void __launch_bounds__(256) sah_prep_kernel(const float* tris, uint32_t n, int* tbox, float* cent,
                                                       uint32_t* idx, SahSlot* root) {
    __shared__ int part[4][6];
    int clo[3] = {kKeyPosInf, kKeyPosInf, kKeyPosInf}, chi[3] = {kKeyNegInf, kKeyNegInf, kKeyNegInf};
    for (uint32_t t = blockIdx.x * 256u + threadIdx.x; t < n; t += gridDim.x * 256u) {
        const float* v = tris + 9 * (size_t)t;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            // key order, as the reductions: -0 counts below +0
            const int lo = min(min(fkey(v[a]), fkey(v[3 + a])), fkey(v[6 + a]));
            const int hi = max(max(fkey(v[a]), fkey(v[3 + a])), fkey(v[6 + a]));
            tbox[6 * (size_t)t + a] = lo;
            tbox[6 * (size_t)t + 3 + a] = hi;
            const float c = 0.5f * (kfloat(lo) + kfloat(hi));
            cent[3 * (size_t)t + a] = c;
            clo[a] = min(clo[a], fkey(c));
            chi[a] = max(chi[a], fkey(c));
        }
        idx[t] = t;
    }
    bounds_atomic(clo, chi, n > kSahSmall ? root->cb : nullptr, part);
}

// bins of one chunk; every axis is binned (one without extent into bin 0), so
// that the union over an axis' bins is the node's box
__global__ void __launch_bounds__(256) sah_bin_kernel(SahTree T, SahWork W, uint32_t level) {
    __shared__ int hist[kNodeBinWords];
    const uint32_t* cnt = W.counters + 2u * (level & 3u);
    uint32_t* clear = W.counters + 2u * ((level + 2u) & 3u);
    if (blockIdx.x == 0u && threadIdx.x < 2u) clear[threadIdx.x] = 0u;
    const SahLevel& S = W.level[level & 1u];
    for (uint32_t chunk = blockIdx.x; chunk < cnt[1]; chunk += gridDim.x) {
        const uint32_t slot = S.chunk_slot[chunk];
        const SahSlot& s = S.slots[slot];
        float lo[3], scale[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) axis_scale(s.cb[a], s.cb[3 + a], lo[a], scale[a]);
        for (uint32_t k = threadIdx.x; k < (uint32_t)kNodeBinWords; k += 256u) {
            const uint32_t w = k % kBinWords;
            hist[k] = w == 0u ? 0 : (w < 4u ? kKeyPosInf : kKeyNegInf);
        }
        __syncthreads();
        const uint32_t p0 = (chunk - s.chunk0) * kSahChunk;
        const uint32_t p1 = min(p0 + kSahChunk, s.count);
        for (uint32_t p = p0 + threadIdx.x; p < p1; p += 256u) {
            const size_t t = S.idx[s.first + p];
            int b[6];
#pragma unroll
            for (int c = 0; c < 6; ++c) b[c] = reinterpret_cast<const int*>(T.tbox)[6 * t + c];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                int* h = hist + (a * kSahBins + bin_of(T.cent[3 * t + a], lo[a], scale[a])) * kBinWords;
                atomicAdd(&h[0], 1);
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    atomicMin(&h[1 + c], b[c]);
                    atomicMax(&h[4 + c], b[3 + c]);
                }
            }
        }
        __syncthreads();
        if (threadIdx.x < 3u * kSahBins) W.chunk_counts[chunk * 3u * kSahBins + threadIdx.x] = (uint32_t)hist[threadIdx.x * kBinWords];
        int* bins = S.bins + (size_t)slot * kNodeBinWords;
        for (uint32_t k = threadIdx.x; k < (uint32_t)kNodeBinWords; k += 256u) {
            const uint32_t w = k % kBinWords;
            if (hist[k - w] == 0) continue;
            if (w == 0u) atomicAdd(&bins[k], hist[k]);
            else if (w < 4u) atomicMin(&bins[k], hist[k]);
            else atomicMax(&bins[k], hist[k]);
        }
        __syncthreads();
    }
}

// the split of each of the level's nodes (one wave per node), its children and
// their places in the next level or among the small subtrees
__global__ void __launch_bounds__(64) sah_split_kernel(SahTree T, SahWork W, uint32_t level) {
    __shared__ int bins[kNodeBinWords];
    const uint32_t nodes = W.counters[2u * (level & 3u)];
    uint32_t* next = W.counters + 2u * ((level + 1u) & 3u);
    const SahLevel& S = W.level[level & 1u];
    const SahLevel& N = W.level[(level + 1u) & 1u];
    const uint32_t lane = threadIdx.x;
    for (uint32_t slot = blockIdx.x; slot < nodes; slot += gridDim.x) {
        SahSlot& s = S.slots[slot];
        for (uint32_t k = lane; k < (uint32_t)kNodeBinWords; k += 64u) bins[k] = S.bins[(size_t)slot * kNodeBinWords + k];
        __syncthreads();
        float cost = __builtin_inff();
        int key = -1;
        if (lane < 45u) {
            const int a = (int)lane / 15, split = (int)lane % 15 + 1;
            float lo, scale;
            axis_scale(s.cb[a], s.cb[3 + a], lo, scale);
            int l[6], r[6], lc = 0, rc = 0;
            empty_box(l);
            empty_box(r);
            for (int b = 0; b < kSahBins; ++b) {
                const int* h = bins + (a * kSahBins + b) * kBinWords;
                const bool left = b < split;
                lc += left ? h[0] : 0;
                rc += left ? 0 : h[0];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    l[c] = left ? min(l[c], h[1 + c]) : l[c];
                    l[3 + c] = left ? max(l[3 + c], h[4 + c]) : l[3 + c];
                    r[c] = left ? r[c] : min(r[c], h[1 + c]);
                    r[3 + c] = left ? r[3 + c] : max(r[3 + c], h[4 + c]);
                }
            }
            if (scale != 0.0f && lc != 0 && rc != 0) {
                cost = (float)lc * box_area(l) + (float)rc * box_area(r);
                if (cost < __builtin_inff()) key = a * kSahBins + split;
            }
        }
        group_best<64>(cost, key);
        const int axis = key >= 0 ? key / kSahBins : -1, bin = key >= 0 ? key % kSahBins : -1;
        // the left count, and the node's box from axis 0's bins
        const uint32_t first = s.first, count = s.count;
        int nl = 0;
        if (axis >= 0) {
            nl = (int)lane < bin ? bins[(axis * kSahBins + (int)lane) * kBinWords] : 0;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) nl += __shfl_xor(nl, o);
        } else {
            nl = (int)(count / 2u);
        }
        if (lane < 6u) {
            int v = bins[1 + lane];
            for (int b = 1; b < kSahBins; ++b) {
                const int h = bins[b * kBinWords + 1 + (int)lane];
                v = lane < 3u ? min(v, h) : max(v, h);
            }
            T.box[6 * (size_t)s.node + lane] = kfloat(v);
        }
        int base = 0;
        if (lane == 0u) base = (int)atomicAdd(T.node_counter, 2u);
        base = __builtin_amdgcn_readfirstlane(base);
        if (lane == 0u) {
            s.axis = axis;
            s.bin = bin;
            s.nl = (uint32_t)nl;
            T.left[s.node] = base;
            T.right[s.node] = base + 1;
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const uint32_t cf = c == 0 ? first : first + (uint32_t)nl, cc = c == 0 ? (uint32_t)nl : count - (uint32_t)nl;
            if (lane == 0u) {
                T.parent[base + c] = s.node;
                T.first[base + c] = (int)cf;
                T.count[base + c] = (int)cc;
            }
            if (cc > kSahSmall) {
                const uint32_t chunks = (cc + kSahChunk - 1u) / kSahChunk;
                uint32_t p = 0, c0 = 0;
                if (lane == 0u) {
                    p = atomicAdd(&next[0], 1u);
                    c0 = atomicAdd(&next[1], chunks);
                }
                p = (uint32_t)__builtin_amdgcn_readfirstlane((int)p);
                c0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)c0);
                slot_init(N.slots[p], N.bins + (size_t)p * kNodeBinWords, base + c, cf, cc, c0, lane, 64u);
                for (uint32_t k = lane; k < chunks; k += 64u) N.chunk_slot[c0 + k] = p;
                if (lane == 0u) s.child[c] = (int)p;
            } else if (lane == 0u) {
                s.child[c] = -1;
                W.small[atomicAdd(&W.counters[8], 1u)] = (uint32_t)(base + c) | (((level + 1u) & 1u) << 31);
            }
        }
        __syncthreads();
    }
}

// stable partition of one chunk into the next level's order, and the
// children's centroid bounds
__global__ void __launch_bounds__(256) sah_scatter_kernel(SahTree T, SahWork W, uint32_t level) {
    __shared__ int part[4][6];
    __shared__ uint32_t wave_left[4];
    const uint32_t chunks = W.counters[2u * (level & 3u) + 1u];
    const SahLevel& S = W.level[level & 1u];
    const SahLevel& N = W.level[(level + 1u) & 1u];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint64_t below = (1ull << lane) - 1ull;
    for (uint32_t chunk = blockIdx.x; chunk < chunks; chunk += gridDim.x) {
        const SahSlot& s = S.slots[S.chunk_slot[chunk]];
        const int axis = s.axis, bin = s.bin;
        const uint32_t nl = s.nl, own = chunk - s.chunk0, p0 = own * kSahChunk, p1 = min(p0 + kSahChunk, s.count);
        float lo = 0.0f, scale = 0.0f;
        if (axis >= 0) axis_scale(s.cb[axis], s.cb[3 + axis], lo, scale);
        // triangles of the node's earlier chunks that go left
        uint32_t before = 0;
        if (axis >= 0) {
            for (uint32_t k = threadIdx.x; k < own * kSahBins; k += 256u)
                if ((int)(k % kSahBins) < bin)
                    before += W.chunk_counts[(s.chunk0 + k / kSahBins) * 3u * kSahBins + (uint32_t)axis * kSahBins + k % kSahBins];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) before += (uint32_t)__shfl_xor((int)before, o);
            if (lane == 0u) wave_left[wave] = before;
            __syncthreads();
            before = wave_left[0] + wave_left[1] + wave_left[2] + wave_left[3];
            __syncthreads();
        } else {
            before = min(nl, p0);
        }
        uint32_t left_at = s.first + before, right_at = s.first + nl + (p0 - before);
        int clo[2][3], chi[2][3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            clo[0][a] = clo[1][a] = kKeyPosInf;
            chi[0][a] = chi[1][a] = kKeyNegInf;
        }
        for (uint32_t q = p0; q < p1; q += 256u) {
            const uint32_t p = q + threadIdx.x;
            const bool valid = p < p1;
            const uint32_t t = valid ? S.idx[s.first + p] : 0u;
            float c[3] = {0.0f, 0.0f, 0.0f};
            bool left = false;
            if (valid) {
#pragma unroll
                for (int a = 0; a < 3; ++a) c[a] = T.cent[3 * (size_t)t + a];
                const float ca = axis == 0 ? c[0] : (axis == 1 ? c[1] : c[2]);
                left = axis >= 0 ? bin_of(ca, lo, scale) < bin : p < nl;
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    const int k = fkey(c[a]);
                    clo[0][a] = left ? min(clo[0][a], k) : clo[0][a];
                    chi[0][a] = left ? max(chi[0][a], k) : chi[0][a];
                    clo[1][a] = left ? clo[1][a] : min(clo[1][a], k);
                    chi[1][a] = left ? chi[1][a] : max(chi[1][a], k);
                }
            }
            const uint64_t m = __ballot(left), mv = __ballot(valid);
            if (lane == 0u) wave_left[wave] = (uint32_t)__popcll(m);
            __syncthreads();
            uint32_t lb = 0, lt = 0;
#pragma unroll
            for (uint32_t w = 0; w < 4u; ++w) {
                lb += w < wave ? wave_left[w] : 0u;
                lt += wave_left[w];
            }
            const uint32_t lrank = lb + (uint32_t)__popcll(m & below);
            const uint32_t vrank = wave * 64u + (uint32_t)__popcll(mv & below);
            if (valid) N.idx[left ? left_at + lrank : right_at + (vrank - lrank)] = t;
            left_at += lt;
            right_at += min(256u, p1 - q) - lt;
            __syncthreads();
        }
#pragma unroll
        for (int c = 0; c < 2; ++c)
            bounds_atomic(clo[c], chi[c], s.child[c] >= 0 ? N.slots[s.child[c]].cb : nullptr, part);
    }
}

// ---- small subtrees ------------------------------------------------------------------
struct SahItem {
    int4 lo;  // low corner (keys), bins of the three axes (4 bits each)
    int4 hi;  // high corner (keys), triangle
};

struct SahLds {
    SahItem item[kSahSmall];
    float cent[3][kSahSmall];
    uint8_t order[kSahSmall];
    uint32_t stack[kSahSmall], stack_node[kSahSmall];  // nodes above 16 triangles: first | count << 16, node
    uint32_t list[kSahSmall], list_node[kSahSmall];    // nodes of 2 to 16 triangles
    uint32_t list_count, next_node;
};

// adds item j of a node to the sides of split `split` of an axis
__device__ __forceinline__ void add_item(const SahItem& it, int shift, int split, int (&l)[6], int (&r)[6], int& lc,
                                         int& rc) {
    const int b[6] = {it.lo.x, it.lo.y, it.lo.z, it.hi.x, it.hi.y, it.hi.z};
    const bool left = ((it.lo.w >> shift) & 15) < split;
    lc += left ? 1 : 0;
    rc += left ? 0 : 1;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        l[c] = min(l[c], left ? b[c] : kKeyPosInf);
        r[c] = min(r[c], left ? kKeyPosInf : b[c]);
        l[3 + c] = max(l[3 + c], left ? b[3 + c] : kKeyNegInf);
        r[3 + c] = max(r[3 + c], left ? kKeyNegInf : b[3 + c]);
    }
}

// The children of `node`: lane c (0, 1) of the node's lanes writes child c.
// Returns the child's entry when it has to be split further, else 0.
__device__ __forceinline__ uint32_t put_child(const SahTree& T, const SahLds& sh, uint32_t c, uint32_t node,
                                              uint32_t base, uint32_t first, uint32_t count, uint32_t nl) {
    const uint32_t cf = c == 0u ? first : first + nl, cc = c == 0u ? nl : count - nl, id = base + c;
    T.parent[id] = (int)node;
    T.count[id] = (int)cc;
    if (c == 0u) {
        T.left[node] = (int)base;
        T.right[node] = (int)base + 1;
    }
    if (cc > 1u) return cf | (cc << 16);
    T.left[id] = -1;
    T.right[id] = -1;
    T.prim[id] = (uint32_t)sh.item[sh.order[cf]].hi.w;
    return 0u;
}

__global__ void __launch_bounds__(64) sah_small_kernel(SahTree T, SahWork W) {
    __shared__ SahLds sh;
    const uint32_t lane = threadIdx.x;
    const uint64_t below = (1ull << lane) - 1ull;
    const uint32_t task = W.small[blockIdx.x];
    const uint32_t root = task & 0x7FFFFFFFu;
    const uint32_t* idx = W.level[task >> 31].idx + T.first[root];
    const uint32_t n = (uint32_t)T.count[root];
    if (n == 1u) {
        if (lane == 0u) {
            T.left[root] = -1;
            T.right[root] = -1;
            T.prim[root] = idx[0];
        }
        return;
    }
    uint32_t base = 0;
    if (lane == 0u) base = atomicAdd(T.node_counter, 2u * (n - 1u));
    for (uint32_t k = lane; k < n; k += 64u) {
        const size_t t = idx[k];
        const int* b = reinterpret_cast<const int*>(T.tbox) + 6 * t;
        sh.item[k].lo = make_int4(b[0], b[1], b[2], 0);
        sh.item[k].hi = make_int4(b[3], b[4], b[5], (int)t);
#pragma unroll
        for (int a = 0; a < 3; ++a) sh.cent[a][k] = T.cent[3 * t + a];
        sh.order[k] = (uint8_t)k;
    }
    uint32_t depth = 0;  // stack entries (the same in every lane)
    if (lane == 0u) {
        sh.next_node = base;
        sh.list_count = n > 16u ? 0u : 1u;
        sh.stack[0] = sh.list[0] = n << 16;
        sh.stack_node[0] = sh.list_node[0] = root;
    }
    if (n > 16u) depth = 1u;
    sah_wave_sync();
    // nodes above 16 triangles, depth-first
    while (depth > 0u) {
        --depth;
        const uint32_t e = sh.stack[depth], node = sh.stack_node[depth];
        const uint32_t first = e & 0xFFFFu, cnt = e >> 16;
        int box[6], cb[6];
        empty_box(box);
        empty_box(cb);
        uint32_t own[kSahSmall / 64u];
#pragma unroll
        for (uint32_t k = 0; k < kSahSmall / 64u; ++k) {
            const uint32_t p = lane + 64u * k;
            own[k] = 0u;
            if (p < cnt) {
                own[k] = sh.order[first + p];
                const SahItem& it = sh.item[own[k]];
                const int b[6] = {it.lo.x, it.lo.y, it.lo.z, it.hi.x, it.hi.y, it.hi.z};
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const int ck = fkey(sh.cent[c][own[k]]);
                    box[c] = min(box[c], b[c]);
                    box[3 + c] = max(box[3 + c], b[3 + c]);
                    cb[c] = min(cb[c], ck);
                    cb[3 + c] = max(cb[3 + c], ck);
                }
            }
        }
        float lo[3], scale[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            box[c] = group_min<64>(box[c]);
            box[3 + c] = group_max<64>(box[3 + c]);
            axis_scale(group_min<64>(cb[c]), group_max<64>(cb[3 + c]), lo[c], scale[c]);
        }
#pragma unroll
        for (uint32_t k = 0; k < kSahSmall / 64u; ++k)
            if (lane + 64u * k < cnt) {
                int bins = 0;
#pragma unroll
                for (int a = 0; a < 3; ++a) bins |= bin_of(sh.cent[a][own[k]], lo[a], scale[a]) << (4 * a);
                sh.item[own[k]].lo.w = bins;
            }
        sah_wave_sync();
        float cost = __builtin_inff();
        int key = -1;
        if (lane < 45u) {
            const int a = (int)lane / 15, split = (int)lane % 15 + 1;
            int l[6], r[6], lc = 0, rc = 0;
            empty_box(l);
            empty_box(r);
            for (uint32_t j = 0; j < cnt; ++j) add_item(sh.item[sh.order[first + j]], 4 * a, split, l, r, lc, rc);
            const float sa = a == 0 ? scale[0] : (a == 1 ? scale[1] : scale[2]);
            if (sa != 0.0f && lc != 0 && rc != 0) {
                cost = (float)lc * box_area(l) + (float)rc * box_area(r);
                if (cost < __builtin_inff()) key = a * kSahBins + split;
            }
        }
        group_best<64>(cost, key);
        // stable partition
        bool left[kSahSmall / 64u];
        uint32_t nl = 0;
#pragma unroll
        for (uint32_t k = 0; k < kSahSmall / 64u; ++k) {
            const uint32_t p = lane + 64u * k;
            left[k] = p < cnt && (key >= 0 ? ((sh.item[own[k]].lo.w >> (4 * (key / kSahBins))) & 15) < key % kSahBins
                                           : p < cnt / 2u);
            nl += (uint32_t)__popcll(__ballot(left[k]));
        }
        sah_wave_sync();
        uint32_t la = first, ra = first + nl;
#pragma unroll
        for (uint32_t k = 0; k < kSahSmall / 64u; ++k) {
            const uint64_t m = __ballot(left[k]), mv = __ballot(lane + 64u * k < cnt);
            const uint32_t lr = (uint32_t)__popcll(m & below), vr = (uint32_t)__popcll(mv & below);
            if (lane + 64u * k < cnt) sh.order[left[k] ? la + lr : ra + (vr - lr)] = (uint8_t)own[k];
            la += (uint32_t)__popcll(m);
            ra += (uint32_t)__popcll(mv) - (uint32_t)__popcll(m);
        }
        sah_wave_sync();
        if (lane < 6u) {
            const int v = lane == 0u ? box[0] : lane == 1u ? box[1] : lane == 2u ? box[2] : lane == 3u ? box[3] : lane == 4u ? box[4] : box[5];
            T.box[6 * (size_t)node + lane] = kfloat(v);
        }
        const uint32_t id = sh.next_node;
        uint32_t child = 0u;
        if (lane < 2u) child = put_child(T, sh, lane, node, id, first, cnt, nl);
        const uint64_t deep = __ballot((child >> 16) > 16u), flat = __ballot(child != 0u && (child >> 16) <= 16u);
        const uint32_t at = sh.list_count;
        sah_wave_sync();
        if ((deep >> lane) & 1ull) {
            const uint32_t p = depth + (uint32_t)__popcll(deep & below);
            sh.stack[p] = child;
            sh.stack_node[p] = id + lane;
        }
        if ((flat >> lane) & 1ull) {
            const uint32_t p = at + (uint32_t)__popcll(flat & below);
            sh.list[p] = child;
            sh.list_node[p] = id + lane;
        }
        if (lane == 0u) {
            sh.next_node = id + 2u;
            sh.list_count = at + (uint32_t)__popcll(flat);
        }
        depth += (uint32_t)__popcll(deep);
        sah_wave_sync();
    }
    // the rest breadth-first: four nodes at a time, 16 lanes each
    const uint32_t group = lane >> 4, gl = lane & 15u;
    for (uint32_t head = 0;;) {
        const uint32_t count = sh.list_count;
        if (head >= count) break;
        const bool has = head + group < count;
        const uint32_t e = has ? sh.list[head + group] : 0u, node = has ? sh.list_node[head + group] : 0u;
        const uint32_t first = e & 0xFFFFu, cnt = e >> 16;
        const bool mine = gl < cnt;
        const uint32_t own = mine ? sh.order[first + gl] : 0u;
        int box[6], cb[6];
        empty_box(box);
        empty_box(cb);
        float c[3] = {0.0f, 0.0f, 0.0f};
        if (mine) {
            const SahItem& it = sh.item[own];
            box[0] = it.lo.x, box[1] = it.lo.y, box[2] = it.lo.z, box[3] = it.hi.x, box[4] = it.hi.y, box[5] = it.hi.z;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                c[a] = sh.cent[a][own];
                cb[a] = cb[3 + a] = fkey(c[a]);
            }
        }
        int bins = 0;
        float scale[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            box[a] = group_min<16>(box[a]);
            box[3 + a] = group_max<16>(box[3 + a]);
            float lo;
            axis_scale(group_min<16>(cb[a]), group_max<16>(cb[3 + a]), lo, scale[a]);
            bins |= bin_of(c[a], lo, scale[a]) << (4 * a);
        }
        if (mine) sh.item[own].lo.w = bins;
        sah_wave_sync();
        float cost = __builtin_inff();
        int key = -1;
#pragma unroll 1
        for (int a = 0; a < 3; ++a) {
            int l[6], r[6], lc = 0, rc = 0;
            empty_box(l);
            empty_box(r);
            for (uint32_t j = 0; j < cnt; ++j) add_item(sh.item[sh.order[first + j]], 4 * a, (int)gl + 1, l, r, lc, rc);
            const float sa = a == 0 ? scale[0] : (a == 1 ? scale[1] : scale[2]);
            if (gl < 15u && sa != 0.0f && lc != 0 && rc != 0) {
                const float v = (float)lc * box_area(l) + (float)rc * box_area(r);
                if (v < cost) {
                    cost = v;
                    key = a * kSahBins + (int)gl + 1;
                }
            }
        }
        group_best<16>(cost, key);
        const bool left = mine && (key >= 0 ? ((bins >> (4 * (key / kSahBins))) & 15) < key % kSahBins : gl < cnt / 2u);
        const uint32_t gm = (uint32_t)(__ballot(left) >> (16u * group)) & 0xFFFFu;
        const uint32_t nl = (uint32_t)__popc(gm), lr = (uint32_t)__popc(gm & ((1u << gl) - 1u));
        sah_wave_sync();
        if (mine) sh.order[first + (left ? lr : nl + (gl - lr))] = (uint8_t)own;
        sah_wave_sync();
        if (has && gl < 6u) {
            const int v = gl == 0u ? box[0] : gl == 1u ? box[1] : gl == 2u ? box[2] : gl == 3u ? box[3] : gl == 4u ? box[4] : box[5];
            T.box[6 * (size_t)node + gl] = kfloat(v);
        }
        const uint32_t id = sh.next_node;
        uint32_t child = 0u;
        if (has && gl < 2u) child = put_child(T, sh, gl, node, id + 2u * group, first, cnt, nl);
        const uint64_t more = __ballot(child != 0u);
        const uint32_t live = min(4u, count - head);
        sah_wave_sync();
        if (child != 0u) {
            const uint32_t p = count + (uint32_t)__popcll(more & below);
            sh.list[p] = child;
            sh.list_node[p] = id + 2u * group + gl;
        }
        if (lane == 0u) {
            sh.next_node = id + 2u * live;
            sh.list_count = count + (uint32_t)__popcll(more);
        }
        head += live;
        sah_wave_sync();
    }
}

namespace {
size_t sah_align(size_t x) { return (x + 255u) & ~(size_t)255u; }
}  // namespace

// the builder's scratch beside the tree's arrays
static size_t sah_carve(char* base, uint32_t n, const SahTree& T, SahWork* W) {
    const size_t nodes = (size_t)n / (kSahSmall + 1u) + 2u, chunks = (size_t)n / kSahChunk + nodes + 1u;
    size_t off = 0;
    auto take = [&](size_t bytes) {
        char* p = base ? base + off : nullptr;
        off += sah_align(bytes);
        return p;
    };
    for (int k = 0; k < 2; ++k) {
        W->level[k].slots = reinterpret_cast<SahSlot*>(take(nodes * sizeof(SahSlot)));
        W->level[k].bins = reinterpret_cast<int*>(take(nodes * kNodeBinWords * sizeof(int)));
        W->level[k].chunk_slot = reinterpret_cast<uint32_t*>(take(chunks * sizeof(uint32_t)));
    }
    W->level[0].idx = T.idx;
    W->level[1].idx = T.tmp;
    W->chunk_counts = reinterpret_cast<uint32_t*>(take(chunks * 3u * kSahBins * sizeof(uint32_t)));
    W->counters = reinterpret_cast<uint32_t*>(take(16u * sizeof(uint32_t)));
    // (a large node's split gives at most two small subtrees, of one triangle
    // or more)
    W->small = reinterpret_cast<uint32_t*>(take(((size_t)n + 2u) * sizeof(uint32_t)));
    return off;
}

size_t sah_scratch_bytes(uint32_t n) {
    SahWork W;
    return sah_carve(nullptr, n, SahTree{}, &W);
}

// Builds the tree over n >= 1 triangles (9 floats each) into T (2n - 1
// nodes; node 0 is the root). scratch: sah_scratch_bytes(n).
hipError_t build_sah_tree(const float* tris, uint32_t n, SahTree& T, void* scratch, hipStream_t s) {
    SahWork W;
    sah_carve(static_cast<char*>(scratch), n, T, &W);
    const uint32_t chunks = n / kSahChunk + 1u;
    const uint32_t grid = chunks < 1024u ? chunks : 1024u;
    hipError_t e;
    hipLaunchKernelGGL(sah_init_kernel, dim3(1), dim3(256), 0, s, T, W, n);
    hipLaunchKernelGGL(sah_prep_kernel, dim3((n + 255u) / 256u < 1024u ? (n + 255u) / 256u : 1024u), dim3(256), 0, s, tris,
                       n, reinterpret_cast<int*>(T.tbox), T.cent, T.idx, W.level[0].slots);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    uint32_t host[9] = {};
    // every split leaves both children smaller than the node, so a node is
    // large for fewer than n levels; the host looks after every run of levels
    // (a level without nodes costs three empty launches)
    for (uint32_t level = 0; level < n;) {
        const uint32_t run = n > kSahSmall ? (level == 0u ? 16u : 8u) : 0u;
        for (uint32_t k = 0; k < run; ++k, ++level) {
            hipLaunchKernelGGL(sah_bin_kernel, dim3(grid), dim3(256), 0, s, T, W, level);
            hipLaunchKernelGGL(sah_split_kernel, dim3(512), dim3(64), 0, s, T, W, level);
            hipLaunchKernelGGL(sah_scatter_kernel, dim3(grid), dim3(256), 0, s, T, W, level);
        }
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if ((e = hipMemcpyAsync(host, W.counters, sizeof(host), hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
        if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
        if (run == 0u || host[2u * (level & 3u)] == 0u) break;
    }
    if (host[8] > n) return hipErrorUnknown;
    if (host[8] > 0u) hipLaunchKernelGGL(sah_small_kernel, dim3(host[8]), dim3(64), 0, s, T, W);
    return hipGetLastError();
}

}  // namespace rl
