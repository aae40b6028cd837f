// lbvh.hip -- linear BVH over the scene triangles and its stackless traversal.
//
// The reference traces shadow rays with VK_KHR_ray_query against a hardware
// acceleration structure (src/shaders/shading_pass.frag.glsl:112-129,
// src/scene.c:142-406). gfx950 has no ray-query hardware, so the project
// builds its own hierarchy:
//   1. triangles dequantised exactly as the shader decodes positions
//      (decode_position_64_bit, mesh_quantization.glsl:38-45);
//   2. 30-bit Morton codes of the centroids in the centroid bounds (the
//      bit interleave of tools/io_export_vulkan_blender28.py:49-77), keys
//      (code << 32 | triangle id) radix-sorted -- unique keys, so the order
//      is deterministic;
//   3. Karras (2012) hierarchy: internal node i splits the sorted range at
//      the highest differing key bit; leaves are node ids n-1 .. 2n-2;
//   4. bottom-up boxes with one atomic arrival counter per internal node;
//   5. the nodes written in depth-first pre-order (left child first) with
//      escape links, for stackless traversal: a box hit continues at the
//      next record in memory, so a descent reads consecutive cache lines.
// The CPU oracle builds the same tree from the same keys; traversal uses the
// same box and Moeller-Trumbore tests in the same operation order, so hit and
// miss flags agree bit for bit.
#include <algorithm>
#include <cmath>

#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include "devmath.hpp"
#include "kernels.hpp"

namespace rl {

// reference to the triangle record at `unit`, or to the pair there and at
// unit + 3 (negative; non-negative references are wide nodes)
__device__ __forceinline__ int wide_leaf(uint32_t unit, uint32_t pair) { return ~(int)(unit * 2u + pair); }

__device__ __forceinline__ uint32_t part_1_by_2(uint32_t x) {
    x &= 0x000003ffu;
    x = (x ^ (x << 16)) & 0xff0000ffu;
    x = (x ^ (x << 8)) & 0x0300f00fu;
    x = (x ^ (x << 4)) & 0x030c30c3u;
    x = (x ^ (x << 2)) & 0x09249249u;
    return x;
}

__global__ void dequant_kernel(const uint2* pos, uint64_t n, float3 f, float3 s, float* tris, float* cent) {
    uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    float v[9];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        uint2 q = pos[t * 3 + k];
        uint32_t qx = q.x & 0x1FFFFFu;
        uint32_t qy = ((q.x & 0xFFE00000u) >> 21) | ((q.y & 0x3FFu) << 11);
        uint32_t qz = (q.y & 0x7FFFFC00u) >> 10;
        v[3 * k + 0] = fma_((float)qx, f.x, s.x);
        v[3 * k + 1] = fma_((float)qy, f.y, s.y);
        v[3 * k + 2] = fma_((float)qz, f.z, s.z);
    }
#pragma unroll
    for (int k = 0; k < 9; ++k) tris[t * 9 + k] = v[k];
#pragma unroll
    for (int a = 0; a < 3; ++a) cent[t * 3 + a] = ((v[a] + v[3 + a]) + v[6 + a]) / 3.0f;
}

// min/max of the centroids: block partials, then one block over partials.
// min and max are exact, so any reduction order gives the same bounds.
__global__ void bounds_kernel(const float* cent, uint64_t n, float* partial) {
    __shared__ float sh[6][256];
    float lo[3] = {__builtin_inff(), __builtin_inff(), __builtin_inff()};
    float hi[3] = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (uint64_t)gridDim.x * blockDim.x) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            float c = cent[t * 3 + a];
            lo[a] = fmin_(lo[a], c);
            hi[a] = fmax_(hi[a], c);
        }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        sh[a][threadIdx.x] = lo[a];
        sh[3 + a][threadIdx.x] = hi[a];
    }
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                sh[a][threadIdx.x] = fmin_(sh[a][threadIdx.x], sh[a][threadIdx.x + w]);
                sh[3 + a][threadIdx.x] = fmax_(sh[3 + a][threadIdx.x], sh[3 + a][threadIdx.x + w]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0)
#pragma unroll
        for (int a = 0; a < 6; ++a) partial[blockIdx.x * 6 + a] = sh[a][0];
}

__global__ void bounds_final_kernel(const float* partial, uint32_t blocks, float* out) {
    if (threadIdx.x != 0) return;
    float r[6] = {__builtin_inff(), __builtin_inff(), __builtin_inff(), -__builtin_inff(), -__builtin_inff(),
                  -__builtin_inff()};
    for (uint32_t b = 0; b < blocks; ++b)
        for (int a = 0; a < 3; ++a) {
            r[a] = fmin_(r[a], partial[b * 6 + a]);
            r[3 + a] = fmax_(r[3 + a], partial[b * 6 + 3 + a]);
        }
    for (int a = 0; a < 6; ++a) out[a] = r[a];
}

__global__ void morton_kernel(const float* cent, uint64_t n, const float* bounds, uint64_t* keys) {
    uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    uint32_t code = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float ext = bounds[3 + a] - bounds[a];
        float factor = (ext > 0.0f) ? 1024.0f / ext : 0.0f;
        float summand = -bounds[a] * factor;
        float q = cent[t * 3 + a] * factor + summand;
        q = fmin_(fmax_(q, 0.0f), 1023.0f);
        code |= part_1_by_2((uint32_t)q) << a;
    }
    keys[t] = ((uint64_t)code << 32) | (uint64_t)t;
}

__device__ __forceinline__ int kdelta(const uint64_t* keys, int n, int i, int j) {
    if (j < 0 || j > n - 1) return -1;
    return __clzll((long long)(keys[i] ^ keys[j]));
}

__global__ void karras_kernel(const uint64_t* keys, int n, int* left, int* right, int* parent, int* count) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    int d = (kdelta(keys, n, i, i + 1) - kdelta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    int dmin = kdelta(keys, n, i, i - d);
    int lmax = 2;
    while (kdelta(keys, n, i, i + lmax * d) > dmin) lmax *= 2;
    int l = 0;
    for (int t = lmax / 2; t >= 1; t /= 2)
        if (kdelta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    int j = i + l * d;
    int dnode = kdelta(keys, n, i, j);
    int s = 0;
    for (int div = 2;; div *= 2) {
        int t = (l + div - 1) / div;
        if (kdelta(keys, n, i, i + (s + t) * d) > dnode) s += t;
        if (t == 1) break;
    }
    int gamma = i + s * d + (d < 0 ? d : 0);
    int lo = i < j ? i : j, hi = i < j ? j : i;
    int lc = (lo == gamma) ? (n - 1 + gamma) : gamma;
    int rc = (hi == gamma + 1) ? (n - 1 + gamma + 1) : gamma + 1;
    left[i] = lc;
    right[i] = rc;
    parent[lc] = i;
    parent[rc] = i;
    count[i] = hi - lo + 1;
}

__global__ void leaf_kernel(const uint64_t* keys, const float* tris, int n, float* box, int* left, int* right,
                            int* count, uint32_t* prim) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    uint32_t t = (uint32_t)(keys[k] & 0xFFFFFFFFull);
    const float* v = tris + (size_t)t * 9;
    const int x = n - 1 + k;
    float* b = box + (size_t)x * 6;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        b[a] = fmin_(fmin_(v[a], v[3 + a]), v[6 + a]);
        b[3 + a] = fmax_(fmax_(v[a], v[3 + a]), v[6 + a]);
    }
    left[x] = -1;
    right[x] = -1;
    count[x] = 1;
    prim[x] = t;
}

__global__ void refit_kernel(int n, const int* left, const int* right, const int* parent, float* box,
                             uint32_t* arrivals) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int node = n - 1 + k;
    int p = parent[node];
    volatile float* vb = box;
    // a well-formed tree has depth < n; the cap keeps a malformed one finite
    for (int depth = 0; p >= 0 && depth < n; ++depth) {
        __threadfence();
        uint32_t old = atomicAdd(&arrivals[p], 1u);
        if (old == 0u) return;  // the sibling subtree is not done yet
        int l = left[p], r = right[p];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            float lo = fmin_(vb[(size_t)l * 6 + a], vb[(size_t)r * 6 + a]);
            float hi = fmax_(vb[(size_t)l * 6 + 3 + a], vb[(size_t)r * 6 + 3 + a]);
            vb[(size_t)p * 6 + a] = lo;
            vb[(size_t)p * 6 + 3 + a] = hi;
        }
        node = p;
        p = parent[node];
    }
}

// Writes node x of a binary tree at its pre-order unit (left child first).
// Before x in pre-order come its ancestors (2 units each) and, for every
// ancestor whose right subtree holds x, that ancestor's whole left subtree
// (a subtree of m leaves spans 5 m - 2 units). The escape unit of x is the
// first unit past its own subtree.
__global__ void layout_kernel(int nodes, const int* left, const int* right, const int* parent, const int* count,
                              const uint32_t* prim, const float* box, const float* tris, const uint2* pos,
                              float4* rec, int* unit) {
    int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= nodes) return;
    int depth = 0, skipped = 0;
    int y = x;
    for (int steps = 0; steps < nodes; ++steps) {
        int p = parent[y];
        if (p < 0) break;
        ++depth;
        if (right[p] == y) skipped += 5 * count[left[p]] - 2;
        y = p;
    }
    const int u = 2 * depth + skipped;
    unit[x] = u;
    if (left[x] >= 0) {
        int esc = u + 5 * count[x] - 2;
        const float* b = box + (size_t)x * 6;
        rec[u] = make_float4(b[0], b[1], b[2], __int_as_float(esc));
        rec[u + 1] = make_float4(b[3], b[4], b[5], 0.0f);
    } else {
        uint32_t t = prim[x];
        const float* v = tris + (size_t)t * 9;
        uint32_t light = pos[(size_t)t * 3].y & 0x80000000u;
        rec[u] = make_float4(v[0], v[1], v[2], __int_as_float(-1));
        rec[u + 1] = make_float4(v[3], v[4], v[5], __uint_as_float(t));
        rec[u + 2] = make_float4(v[6], v[7], v[8], __uint_as_float(light));
    }
}

// ---- four-way nodes for the shadow walk --------------------------------------------
// A wide node stands for a binary node with some of its descendants opened:
// starting from its two children, the openable slot of the largest surface
// area is replaced by its children until four slots are filled. A slot ends
// the opening where it is a triangle or a node over two triangles (its
// record pair is contiguous in pre-order: unit + 2 and unit + 5).
// Level L of the tree is a run of consecutive wide nodes; counts[L] is its
// length, and a level allocates its children behind itself.
__device__ __forceinline__ float node_area(const float* box, int x) {
    const float* b = box + (size_t)x * 6;
    const float dx = b[3] - b[0], dy = b[4] - b[1], dz = b[5] - b[2];
    return dx * dy + dy * dz + dz * dx;
}

__global__ void __launch_bounds__(256) wide_level_kernel(uint32_t level, uint32_t* counts, const int* left,
                                                         const int* right, const int* count, const float* box,
                                                         int* src, int4* slots, int4* refs, const int* unit) {
    // the level's first node: the sum of the levels above (at most 64), one
    // per lane
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t begin = lane < level ? counts[lane] : 0u;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) begin += (uint32_t)__shfl_xor((int)begin, o);
    const uint32_t end = begin + counts[level];
    for (uint32_t i = begin + blockIdx.x * blockDim.x + threadIdx.x; i < end; i += gridDim.x * blockDim.x) {
        const int x = src[i];
        int s[4] = {left[x], right[x], -1, -1};
        float a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < 2; ++k) a[k] = count[s[k]] > 2 ? node_area(box, s[k]) : -1.0f;
        int used = 2;
#pragma unroll
        for (int round = 2; round < 4; ++round) {
            int best = -1;
            float ba = -1.0f;
#pragma unroll
            for (int k = 0; k < 3; ++k)
                if (k < used && a[k] > ba) {
                    ba = a[k];
                    best = k;
                }
            if (best < 0) break;
            int y = s[0];
#pragma unroll
            for (int k = 1; k < 3; ++k)
                if (best == k) y = s[k];
            const int l = left[y], r = right[y];
            const float la = count[l] > 2 ? node_area(box, l) : -1.0f;
            const float ra = count[r] > 2 ? node_area(box, r) : -1.0f;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (k == best) {
                    s[k] = l;
                    a[k] = la;
                } else if (k == used) {
                    s[k] = r;
                    a[k] = ra;
                }
            }
            ++used;
        }
        // small boxes first, then large ones, triangles, and empty slots
        // last: slot 0 is never empty (wide_fill_kernel counts on it)
        float key[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            key[k] = s[k] < 0 ? __builtin_inff() : (count[s[k]] > 2 ? fmin_(node_area(box, s[k]), 1.0e38f) : 2.0e38f);
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const int i0 = k < 3 ? k : (k < 5 ? k - 3 : 0);
            if (key[i0] > key[i0 + 1]) {
                const float t = key[i0];
                key[i0] = key[i0 + 1];
                key[i0 + 1] = t;
                const int u = s[i0];
                s[i0] = s[i0 + 1];
                s[i0 + 1] = u;
            }
        }
        int inner = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) inner += (s[k] >= 0 && count[s[k]] > 2) ? 1 : 0;
        uint32_t next = inner > 0 ? end + atomicAdd(&counts[level + 1u], (uint32_t)inner) : 0u;
        int f[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            f[k] = 0;
            if (s[k] < 0) continue;
            const int c = count[s[k]];
            if (c > 2) {
                src[next] = s[k];
                f[k] = (int)next;
                ++next;
            } else {
                f[k] = c == 2 ? wide_leaf((uint32_t)unit[s[k]] + 2u, 1u) : wide_leaf((uint32_t)unit[s[k]], 0u);
            }
        }
        slots[i] = make_int4(s[0], s[1], s[2], s[3]);
        refs[i] = make_int4(f[0], f[1], f[2], f[3]);
    }
}

// Writes the wide nodes (layout at BvhView). A triangle's slot has the box of
// its binary parent (the box that guards it in the binary walk). The planes
// are bytes on a grid of the node's own bounds, rounded outwards by at least
// a quarter of a step; a step is at least 2^-20 of the coordinates, so that
// the grid's rounding in float stays far below that quarter. A node of fewer
// than four slots has triangles only; its empty slots have inverted planes
// and, should an ill-conditioned ray meet one, the first slot's reference.
// In front of the nodes, downwards, lie their binary nodes' units.
__global__ void __launch_bounds__(256) wide_fill_kernel(uint32_t n, const int4* slots, const int4* refs,
                                                        const int* parent, const int* count, const float* box,
                                                        const int* src, const int* unit, float4* wide) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int4 sl = slots[i], rf = refs[i];
    const int s[4] = {sl.x, sl.y, sl.z, sl.w};
    float lo[3][4], hi[3][4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int x = s[k] < 0 ? -1 : (count[s[k]] == 1 ? parent[s[k]] : s[k]);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            lo[a][k] = x < 0 ? __builtin_inff() : box[(size_t)x * 6 + a];
            hi[a][k] = x < 0 ? -__builtin_inff() : box[(size_t)x * 6 + 3 + a];
        }
    }
    float org[3], step[3];
    uint32_t qlo[3] = {0u, 0u, 0u}, qhi[3] = {0u, 0u, 0u};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float l = fmin_(fmin_(lo[a][0], lo[a][1]), fmin_(lo[a][2], lo[a][3]));
        const float h = fmax_(fmax_(hi[a][0], hi[a][1]), fmax_(hi[a][2], hi[a][3]));
        step[a] = fmax_(fmax_((h - l) * (1.0f / 240.0f), fmax_(fabs_(l), fabs_(h)) * 0x1p-20f), 1.0e-30f);
        org[a] = l - 4.0f * step[a];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            uint32_t ql = 255u, qh = 0u;
            if (s[k] >= 0) {
                ql = (uint32_t)fmin_(fmax_(__builtin_floorf((lo[a][k] - org[a]) / step[a] - 0.25f), 0.0f), 255.0f);
                qh = (uint32_t)fmin_(fmax_(__builtin_ceilf((hi[a][k] - org[a]) / step[a] + 0.25f), 0.0f), 255.0f);
            }
            qlo[a] |= ql << (8 * k);
            qhi[a] |= qh << (8 * k);
        }
    }
    reinterpret_cast<int*>(wide)[-1 - (ptrdiff_t)i] = unit[src[i]];
    uint4* o = reinterpret_cast<uint4*>(wide) + (size_t)i * kWideFloat4;
    o[0] = make_uint4(__float_as_uint(org[0]), __float_as_uint(org[1]), __float_as_uint(org[2]),
                      __float_as_uint(step[0]));
    o[1] = make_uint4(__float_as_uint(step[1]), __float_as_uint(step[2]), qlo[0], qhi[0]);
    o[2] = make_uint4(qlo[1], qhi[1], qlo[2], qhi[2]);
    const int f0 = rf.x;
    o[3] = make_uint4((uint32_t)f0, (uint32_t)(s[1] < 0 ? f0 : rf.y), (uint32_t)(s[2] < 0 ? f0 : rf.z),
                      (uint32_t)(s[3] < 0 ? f0 : rf.w));
}

__global__ void fill_u32(uint32_t* p, uint64_t n, uint32_t v) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

namespace {
// The device memory of one build: one allocation, released on every path
// (twenty cost a millisecond). Carved twice: without memory to measure it,
// then for the pointers.
struct BuildScratch {
    char* base = nullptr;
    size_t used = 0;
    template <class T>
    void get(T** out, size_t bytes) {
        *out = base ? reinterpret_cast<T*>(base + used) : nullptr;
        used += (bytes + 255u) & ~(size_t)255u;
    }
    ~BuildScratch() {
        if (base) hipFree(base);
    }
};
}  // namespace

#define BVH_TRY(x)                         \
    do {                                   \
        hipError_t e_ = (x);               \
        if (e_ != hipSuccess) return e_;   \
    } while (0)

// The wide nodes of the binary tree (node 0 the root, n >= 2 triangles), or
// null for a tree of more than kWideLevels levels: such a tree would overflow
// the walk's stack, and its rays take the binary walk.
// scratch: wide_scratch_bytes(n).
// A node of fewer than four slots holds no wide child, so every wide node
// with children stands for three binary nodes; n / 2 + 1 holds them all. This
// takes areas that compare: a NaN is never opened, and with NaN throughout a
// tree of halves has up to 2 n / 3 wide nodes. So the boxes have to be
// wide_range().
static size_t wide_scratch_bytes(uint32_t n) {
    return (size_t)(n / 2u + 1u) * (2u * sizeof(int4) + sizeof(int)) + (kWideLevels + 2u) * sizeof(uint32_t);
}

// Whether the mesh's coordinates (21-bit values, dequantised with what the
// caller gave) are at most 1e18: no area overflows then, and neither do the
// walk's plane distances. Any other mesh keeps the binary walk.
static bool wide_range(const float f[3], const float s[3]) {
    bool ok = true;
    for (int a = 0; a < 3; ++a) ok = ok && std::fabs(f[a]) * 2097151.0f + std::fabs(s[a]) <= 1.0e18f;
    return ok;
}

static hipError_t build_wide(void* scratch, uint32_t n, const int* left, const int* right, const int* parent,
                             const int* count, const float* box, const int* unit, BvhBuild* out, hipStream_t s) {
    const uint32_t cap = n / 2u + 1u;
    int4* slots = static_cast<int4*>(scratch);
    int4* refs = slots + cap;
    int* src = reinterpret_cast<int*>(refs + cap);
    uint32_t* counts = reinterpret_cast<uint32_t*>(src + cap);
    // level 0: the binary root, node 0
    hipLaunchKernelGGL(fill_u32, dim3(1), dim3(256), 0, s, counts, kWideLevels + 2u, 0u);
    hipLaunchKernelGGL(fill_u32, dim3(1), dim3(64), 0, s, counts, 1, 1u);
    hipLaunchKernelGGL(fill_u32, dim3(1), dim3(64), 0, s, reinterpret_cast<uint32_t*>(src), 1, 0u);
    uint32_t host[kWideLevels + 2u] = {};
    uint32_t total = 0;
    for (uint32_t level = 0; level <= kWideLevels;) {
        // (most trees end within the first run of launches)
        const uint32_t stop = level + 16u < kWideLevels ? level + 16u : kWideLevels + 1u;
        for (; level < stop; ++level)
            hipLaunchKernelGGL(wide_level_kernel, dim3(512), dim3(256), 0, s, level, counts, left, right, count, box,
                               src, slots, refs, unit);
        BVH_TRY(hipGetLastError());
        BVH_TRY(hipMemcpyAsync(host, counts, sizeof(host), hipMemcpyDeviceToHost, s));
        BVH_TRY(hipStreamSynchronize(s));
        if (host[level] == 0u) break;
    }
    if (host[kWideLevels + 1u] != 0u) return hipSuccess;
    for (uint32_t l = 0; l <= kWideLevels; ++l) total += host[l];
    if (total > cap) return hipErrorUnknown;
    const size_t units = ((size_t)total * sizeof(int) + 127u) / 128u * 128u;
    BVH_TRY(hipMalloc(&out->wide_memory, units + (size_t)total * kWideFloat4 * sizeof(float4)));
    out->wide = reinterpret_cast<float4*>(static_cast<char*>(out->wide_memory) + units);
    hipLaunchKernelGGL(wide_fill_kernel, dim3((total + 255u) / 256u), dim3(256), 0, s, total, slots, refs, parent,
                       count, box, src, unit, out->wide);
    return hipGetLastError();
}

hipError_t build_bvh(const uint2* d_pos, uint64_t tri_count, const float deq_factor[3], const float deq_summand[3],
                     uint32_t builder, BvhBuild* out, hipStream_t s) {
    if (tri_count == 0 || tri_count > kMaxBvhTriangles) return hipErrorInvalidValue;
    if (builder != RISLTC_BVH_SAH && builder != RISLTC_BVH_LBVH) return hipErrorInvalidValue;
    const int n = (int)tri_count;
    const uint64_t nodes = 2 * tri_count - 1;
    const uint32_t tb = 256;
    const uint32_t tri_blocks = (uint32_t)((tri_count + tb - 1) / tb);
    const uint32_t node_blocks = (uint32_t)((nodes + tb - 1) / tb);
    const uint32_t red_blocks = 1024;
    const bool sah = builder == RISLTC_BVH_SAH;
    float *tris, *cent, *box, *partial, *bounds;
    int *left, *right, *parent, *count;
    uint32_t *prim, *arrivals;
    uint64_t *keys, *keys_sorted;
    void *temp, *sah_scratch;
    size_t temp_bytes = 0;
    SahTree T;
    if (!sah)
        BVH_TRY(hipcub::DeviceRadixSort::SortKeys(nullptr, temp_bytes, (uint64_t*)nullptr, (uint64_t*)nullptr, n, 0, 64, s));
    auto carve = [&](BuildScratch& w) {
        // (the layout keeps its units in the centroids' space, and the wide
        // nodes' scratch follows in the triangles' space)
        w.get(&tris, std::max(sizeof(float) * 9 * tri_count, wide_scratch_bytes((uint32_t)n)));
        w.get(&cent, sizeof(float) * 3 * tri_count);
        w.get(&box, sizeof(float) * 6 * nodes);
        w.get(&left, sizeof(int) * nodes);
        w.get(&right, sizeof(int) * nodes);
        w.get(&parent, sizeof(int) * nodes);
        w.get(&count, sizeof(int) * nodes);
        w.get(&prim, sizeof(uint32_t) * nodes);
        if (sah) {
            w.get(&T.tbox, sizeof(float) * 6 * tri_count);
            w.get(&T.idx, sizeof(uint32_t) * tri_count);
            w.get(&T.tmp, sizeof(uint32_t) * tri_count);
            w.get(&T.first, sizeof(int) * nodes);
            w.get(&T.node_counter, sizeof(uint32_t));
            w.get(&sah_scratch, sah_scratch_bytes((uint32_t)n));
        } else {
            w.get(&partial, sizeof(float) * 6 * red_blocks);
            w.get(&bounds, sizeof(float) * 6);
            w.get(&keys, sizeof(uint64_t) * tri_count);
            w.get(&keys_sorted, sizeof(uint64_t) * tri_count);
            w.get(&arrivals, sizeof(uint32_t) * tri_count);
            w.get(&temp, temp_bytes);
        }
    };
    BuildScratch w;
    carve(w);
    BVH_TRY(hipMalloc(&w.base, w.used));
    w.used = 0;
    carve(w);
    int* unit = reinterpret_cast<int*>(cent);
    hipLaunchKernelGGL(dequant_kernel, dim3(tri_blocks), dim3(tb), 0, s, d_pos, tri_count,
                       make_float3(deq_factor[0], deq_factor[1], deq_factor[2]),
                       make_float3(deq_summand[0], deq_summand[1], deq_summand[2]), tris, cent);
    BVH_TRY(hipGetLastError());
    if (sah) {
        T.cent = cent;
        T.left = left;
        T.right = right;
        T.parent = parent;
        T.count = count;
        T.prim = prim;
        T.box = box;
        BVH_TRY(build_sah_tree(tris, (uint32_t)n, T, sah_scratch, s));
    } else {
        // (the root keeps no parent)
        hipLaunchKernelGGL(fill_u32, dim3(node_blocks), dim3(tb), 0, s, reinterpret_cast<uint32_t*>(parent), nodes,
                           0xFFFFFFFFu);
        hipLaunchKernelGGL(bounds_kernel, dim3(red_blocks), dim3(256), 0, s, cent, tri_count, partial);
        hipLaunchKernelGGL(bounds_final_kernel, dim3(1), dim3(64), 0, s, partial, red_blocks, bounds);
        hipLaunchKernelGGL(morton_kernel, dim3(tri_blocks), dim3(tb), 0, s, cent, tri_count, bounds, keys);
        BVH_TRY(hipGetLastError());
        BVH_TRY(hipcub::DeviceRadixSort::SortKeys(temp, temp_bytes, keys, keys_sorted, n, 0, 64, s));
        hipLaunchKernelGGL(fill_u32, dim3(tri_blocks), dim3(tb), 0, s, arrivals, tri_count, 0u);
        if (n > 1)
            hipLaunchKernelGGL(karras_kernel, dim3(tri_blocks), dim3(tb), 0, s, keys_sorted, n, left, right, parent,
                               count);
        hipLaunchKernelGGL(leaf_kernel, dim3(tri_blocks), dim3(tb), 0, s, keys_sorted, tris, n, box, left, right,
                           count, prim);
        if (n > 1)
            hipLaunchKernelGGL(refit_kernel, dim3(tri_blocks), dim3(tb), 0, s, n, left, right, parent, box, arrivals);
        BVH_TRY(hipGetLastError());
    }
    const uint64_t units = 5 * tri_count - 2;
    float4* rec = nullptr;
    BVH_TRY(hipMalloc(&rec, sizeof(float4) * (units + 2)));
    // the two padding units after the last record read as zeros
    hipLaunchKernelGGL(fill_u32, dim3(1), dim3(64), 0, s, reinterpret_cast<uint32_t*>(rec + units), 8, 0u);
    hipLaunchKernelGGL(layout_kernel, dim3(node_blocks), dim3(tb), 0, s, (int)nodes, left, right, parent, count, prim,
                       box, tris, d_pos, rec, unit);
    BvhBuild made;
    made.rec = rec;
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && n > 1 && units < kMaxWideUnits && wide_range(deq_factor, deq_summand))
        e = build_wide(tris, (uint32_t)n, left, right, parent, count, box, unit, &made, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) {
        free_bvh(&made);
        return e;
    }
    made.units = (uint32_t)units;
    made.leaf_count = (uint32_t)n;
    *out = made;
    return hipSuccess;
}
#undef BVH_TRY

void free_bvh(BvhBuild* b) {
    if (b->rec) hipFree(b->rec);
    if (b->wide_memory) hipFree(b->wide_memory);
    *b = BvhBuild();
}

// ---- traversal -------------------------------------------------------------------
// four floats in global memory, for loads the compiler must emit as global
// (not flat) instructions
typedef float F4g __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) F4g GlobalF4;
typedef uint32_t U4g __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) U4g GlobalU4;
typedef const __attribute__((address_space(1))) int GlobalInt;
__device__ __forceinline__ float4 global_f4(const GlobalF4* p, int i) {
    const F4g v = p[i];
    return make_float4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ bool ray_box(float3 o, float3 inv, float4 bmin, float4 bmax, float tmin, float tmax) {
    float t0 = (bmin.x - o.x) * inv.x, t1 = (bmax.x - o.x) * inv.x;
    tmin = fmax_(tmin, fmin_(t0, t1));
    tmax = fmin_(tmax, fmax_(t0, t1) * 1.0000004f);
    t0 = (bmin.y - o.y) * inv.y;
    t1 = (bmax.y - o.y) * inv.y;
    tmin = fmax_(tmin, fmin_(t0, t1));
    tmax = fmin_(tmax, fmax_(t0, t1) * 1.0000004f);
    t0 = (bmin.z - o.z) * inv.z;
    t1 = (bmax.z - o.z) * inv.z;
    tmin = fmax_(tmin, fmin_(t0, t1));
    tmax = fmin_(tmax, fmax_(t0, t1) * 1.0000004f);
    return tmin <= tmax;
}

__device__ __forceinline__ bool ray_tri(float3 o, float3 d, float4 a, float4 b, float4 c, float tmin, float tmax,
                                        float& t_out) {
    float e1x = b.x - a.x, e1y = b.y - a.y, e1z = b.z - a.z;
    float e2x = c.x - a.x, e2y = c.y - a.y, e2z = c.z - a.z;
    float px = d.y * e2z - d.z * e2y, py = d.z * e2x - d.x * e2z, pz = d.x * e2y - d.y * e2x;
    float det = fma_(e1z, pz, fma_(e1y, py, e1x * px));
    if (det == 0.0f) return false;
    float inv = 1.0f / det;
    float sx = o.x - a.x, sy = o.y - a.y, sz = o.z - a.z;
    float u = fma_(sz, pz, fma_(sy, py, sx * px)) * inv;
    if (u < 0.0f || u > 1.0f) return false;
    float qx = sy * e1z - sz * e1y, qy = sz * e1x - sx * e1z, qz = sx * e1y - sy * e1x;
    float w = fma_(d.z, qz, fma_(d.y, qy, d.x * qx)) * inv;
    if (w < 0.0f || u + w > 1.0f) return false;
    float t = fma_(e2z, qz, fma_(e2y, qy, e2x * qx)) * inv;
    if (!(t >= tmin && t <= tmax)) return false;
    t_out = t;
    return true;
}

// Every step moves forward in pre-order (by 2, by 3 or to an escape unit
// past the node's subtree), so `units` steps bound the walk; reads of a
// record at unit x < units touch x .. x + 2, inside the padded array.
__device__ __forceinline__ uint32_t closest_hit(const BvhView& B, float3 o, float3 d, float tmin, float tmax) {
    float3 inv = make_float3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    const int end = (int)B.units;
    int x = 0;
    uint32_t best = 0xFFFFFFFFu;
    for (int steps = 0; x < end && steps < end; ++steps) {
        float4 a = B.rec[x], b = B.rec[x + 1], c = B.rec[x + 2];
        int w = __float_as_int(a.w);
        if (w < 0) {
            float t;
            if (ray_tri(o, d, a, b, c, tmin, tmax, t)) {
                tmax = t;
                best = __float_as_uint(b.w) | __float_as_uint(c.w);
            }
            x += 3;
        } else {
            x = ray_box(o, inv, a, b, tmin, tmax) ? x + 2 : w;
        }
    }
    return best;
}

// ---- the shadow walk ---------------------------------------------------------------
// Any hit over the wide nodes, one ray per lane. A step tests the four boxes
// of a node or one triangle. The wave takes one kind of step at a time,
// triangles once a quarter of its walking lanes wait at one: in one step with
// the boxes, the triangle code (about 60 instructions, needed by one lane in
// ten) took more issue slots than they did. (With a fixed count of 16 lanes, a
// triangle in a wave that had fewer walks left waited for all of them: a
// thousand random rays through 5000 triangles 112 us instead of 78.)
//
// What bounds it: the binary walk read 48 bytes per box, 66 boxes per ray of
// the 1080p city, and was limited by the vector cache (0.9 tag lookups per
// clock and CU); four-way nodes of float planes (112 bytes) had the same limit
// (2.2 ms against 1.65). With byte planes a node is four 16-byte loads, and
// issue and lookups are about level: 1.13 ms for 10.8M rays, 13.9 nodes and 2.2
// triangles each (83% occluded; without the chord order 17.4 and 2.6), 35 of
// 64 lanes active at a node. 16,384 lights, 34.6M rays: 7.7 -> 4.8 ms. A step
// is about 140 VALU instructions where a binary step is 30, so waves whose
// rays are nearly the same, and whose binary records stay in their L1, are
// slower than with the binary walk alone (a million rays in bundles of 64
// within 0.004 in a city: 140 us against 105), and so are rays through
// triangles piled on each other.
//
// The flag is the binary walk's, bit for bit: a ray is occluded when some
// triangle passes ray_tri and every binary node above it passes ray_box.
//   * No such triangle is missed: the boxes on the way to it hold boxes of its
//     binary ancestors, and the test below passes wherever ray_box does.
//   * None is added: a triangle that passes ray_tri counts when the ray also
//     passes ray_box on the triangle's own bounds. Every ancestor's box
//     contains them, and ray_box is monotone in the box (each operation is
//     correctly rounded, and 1 / d is finite, so that none is a NaN), so the
//     ancestors pass. Otherwise (a ray within rounding of the bounds' edge)
//     the lane decides the ray by the binary walk: about one ray in a million.
// The binary walk also takes the rays that this and the error bound below do
// not cover (negative tmin, components beyond 1e18 or NaN, a component of the
// direction below 1e-20, 0 among them, a direction so close to an axis that
// the bound exceeds 1% of tmax), hierarchies without wide
// nodes, and the subtree of a node for which a nearly full stack has no room.
// (Clouds of triangles fill it: of a million, for every seventh ray. With such
// rays walked again from the root, a 1080p frame over them took 863 us; 570
// now, 765 with the binary walk for all.)
//
// The test: with i = 1 / d, a plane's distance is
// fma(q, step i, fma(origin, i, -o i)) where ray_box takes (b - o) i. The
// two differ by at most 2^-21 |o i| plus 2^-21 of the distance; the grid's
// own rounding is inside the planes' quarter step. err is 2^-20 times the
// largest |o i|, and the interval test
//   max(near, tmin) <= min(far (1 + 2e-6) + 2 err, tmax (1 + 1e-6))
// (both sides shifted by err; the factor also covers ray_box's 1.0000004)
// passes wherever ray_box's does.
constexpr int kWalkStack = 20;       // entries per lane: 20 KB of LDS per work-group
constexpr uint32_t kShareLanes = 16; // idle lanes that make a wave without further rays share its walks
constexpr uint32_t kNodesPerLeaf = 3;  // lanes at a node for one at a triangle: fewer, and the wave tests triangles
enum WalkMode : uint32_t { kWalkDone = 0, kWalkWide = 1, kWalkBinary = 2 };

// makes one lane's LDS writes visible to the other lanes of its wave
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct Walk {
    float3 o, d;
    float tmin, tmax;
    float3 in, c;        // 1 / d; a plane's distance: fma(b, in, c)
    float lo, hi, slack;  // tmin, tmax and twice the error bound, shifted (wide_boxes)
    const GlobalF4* rec;
    const GlobalF4* wide;
    int end;       // binary: the unit that ends the walk
    int ref;       // wide: the reference to visit; binary: the unit
    int sp;        // stack end
    int bot;       // stack begin (entries below it were given away)
    uint32_t mode;
    bool hit;
};

__device__ __forceinline__ void walk_start(Walk& w, const BvhView& B, float3 o, float3 d, float tmin, float tmax) {
    w.o = o;
    w.d = d;
    w.tmin = tmin;
    w.tmax = tmax;
    w.rec = (const GlobalF4*)B.rec;
    w.wide = (const GlobalF4*)B.wide;
    w.end = (int)B.units;
    w.hit = false;
    w.in = make_float3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    w.c = make_float3(-(o.x * w.in.x), -(o.y * w.in.y), -(o.z * w.in.z));
    const float err = 0x1p-20f * fmax_(fmax_(fabs_(w.c.x), fabs_(w.c.y)), fabs_(w.c.z));
    w.lo = tmin + err;
    w.hi = tmax * (1.0f + 1.0e-6f) + err;
    w.slack = 2.0f * err;
    w.ref = 0;
    w.sp = 0;
    w.bot = 0;
    // (written so that a NaN anywhere, tmax among them, takes the binary walk)
    const float size = fmax_(fmax_(fmax_(fabs_(o.x), fabs_(o.y)), fabs_(o.z)),
                             fmax_(fmax_(fabs_(d.x), fabs_(d.y)), fabs_(d.z)));
    const float steep = fmax_(fmax_(fabs_(w.in.x), fabs_(w.in.y)), fabs_(w.in.z));
    const bool plain = size <= 1.0e18f && steep <= 1.0e20f && tmin >= 0.0f && err <= 0.01f * tmax &&
                       !__builtin_isnan(o.x + o.y + o.z + d.x + d.y + d.z);
    w.mode = plain && B.wide != nullptr ? kWalkWide : kWalkBinary;
}

// The four boxes of one wide node; the slot with the longest part of the ray
// is visited next (the likeliest to hold an occluder: 20% fewer nodes per ray
// than a fixed order), the others are pushed. stack: the lane's column (entry k at stack[256 k])
__device__ __forceinline__ void walk_node(Walk& w, int* stack) {
    if (w.sp > kWalkStack - 4) {
        // no room for three more: the node's subtree in the binary walk, then
        // on with the stack
        w.ref = ((const GlobalInt*)w.wide)[-1 - (ptrdiff_t)w.ref];
        w.end = __float_as_int(global_f4(w.rec, w.ref).w);
        w.mode = kWalkBinary;
        return;
    }
    const GlobalU4* n = (const GlobalU4*)w.wide + (size_t)(uint32_t)w.ref * kWideFloat4;
    const U4g n0 = n[0], n1 = n[1], n2 = n[2], rf = n[3];
    const bool sx = sign_bit(w.in.x), sy = sign_bit(w.in.y), sz = sign_bit(w.in.z);
    const uint32_t nx = sx ? n1[3] : n1[2], fx = sx ? n1[2] : n1[3];
    const uint32_t ny = sy ? n2[1] : n2[0], fy = sy ? n2[0] : n2[1];
    const uint32_t nz = sz ? n2[3] : n2[2], fz = sz ? n2[2] : n2[3];
    const float ox = __uint_as_float(n0[0]), oy = __uint_as_float(n0[1]), oz = __uint_as_float(n0[2]);
    const float ux = __uint_as_float(n0[3]), uy = __uint_as_float(n1[0]), uz = __uint_as_float(n1[1]);
    const float ax = ux * w.in.x, ay = uy * w.in.y, az = uz * w.in.z;
    const float bx = fma_(ox, w.in.x, w.c.x), by = fma_(oy, w.in.y, w.c.y), bz = fma_(oz, w.in.z, w.c.z);
    int sp = w.sp;
    float bl = -1.0f;
    int br = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int sh = 8 * k;
        const float a = fmax_(fmax_(fmax_(fma_((float)((nx >> sh) & 255u), ax, bx), fma_((float)((ny >> sh) & 255u), ay, by)),
                                    fma_((float)((nz >> sh) & 255u), az, bz)),
                              w.lo);
        const float f = fmin_(fmin_(fma_((float)((fx >> sh) & 255u), ax, bx), fma_((float)((fy >> sh) & 255u), ay, by)),
                              fma_((float)((fz >> sh) & 255u), az, bz));
        const float b = fmin_(fma_(f, 1.0f + 2.0e-6f, w.slack), w.hi);
        // the slot with the longest part of the ray is visited next, the
        // others are pushed
        const float len = b - a;
        const bool first = len > bl;
        const int v = first ? br : (int)rf[k];
        stack[sp * 256] = v;
        sp += (len >= 0.0f && bl >= 0.0f) ? 1 : 0;
        br = first ? (int)rf[k] : br;
        bl = fmax_(bl, len);
    }
    const bool met = bl >= 0.0f, more = met || sp > w.bot;
    const int top = sp > w.bot ? sp - 1 : w.bot;
    const int popped = stack[top * 256];
    w.ref = met ? br : popped;
    w.sp = met ? sp : top;
    w.mode = more ? w.mode : kWalkDone;
}

__device__ __forceinline__ bool walk_triangle(const Walk& w, float4 a, float4 b, float4 c, bool& sure) {
    float t;
    if (!ray_tri(w.o, w.d, a, b, c, w.tmin, w.tmax, t)) return false;
    const float4 lo = make_float4(fmin_(fmin_(a.x, b.x), c.x), fmin_(fmin_(a.y, b.y), c.y),
                                  fmin_(fmin_(a.z, b.z), c.z), 0.0f);
    const float4 hi = make_float4(fmax_(fmax_(a.x, b.x), c.x), fmax_(fmax_(a.y, b.y), c.y),
                                  fmax_(fmax_(a.z, b.z), c.z), 0.0f);
    sure = ray_box(w.o, w.in, lo, hi, w.tmin, w.tmax);
    return true;
}

// the triangle at the lane's leaf reference; the first of a pair leaves the
// second as the next reference
__device__ __forceinline__ void walk_leaf(Walk& w, const int* stack) {
    const uint32_t r = (uint32_t)~w.ref;
    const GlobalF4* g = w.rec + (r >> 1);
    const float4 a = global_f4(g, 0), b = global_f4(g, 1), c = global_f4(g, 2);
    bool sure = false;
    const bool met = walk_triangle(w, a, b, c, sure);
    const bool pair = (r & 1u) != 0u, more = pair || w.sp > w.bot;
    const int top = w.sp > w.bot ? w.sp - 1 : w.bot;
    const int popped = stack[top * 256];
    w.hit = met && sure;
    // (the root's escape unit is the hierarchy's end)
    if (met && !sure) w.end = __float_as_int(global_f4(w.rec, 0).w);
    w.ref = met ? 0 : (pair ? wide_leaf((r >> 1) + 3u, 0u) : popped);
    w.sp = met ? 0 : (pair ? w.sp : top);
    w.mode = met ? (sure ? kWalkDone : kWalkBinary) : (more ? kWalkWide : kWalkDone);
}

// Up to `steps` steps of the binary walk. Every step moves forward in pre-order
// (by 2, by 3 or to an escape unit past the node's subtree), so it ends; reads
// of a record at unit x < end touch x .. x + 2, inside the padded array. After a
// subtree without a hit the walk goes on with the stack.
__device__ __forceinline__ void walk_binary(Walk& w, const int* stack, int steps) {
    int x = w.ref;
    bool met = false;
    do {
        const float4 a = global_f4(w.rec, x), b = global_f4(w.rec, x + 1), c = global_f4(w.rec, x + 2);
        const int esc = __float_as_int(a.w);
        if (esc < 0) {
            float t;
            met = ray_tri(w.o, w.d, a, b, c, w.tmin, w.tmax, t);
            x += 3;
        } else {
            x = ray_box(w.o, w.in, a, b, w.tmin, w.tmax) ? x + 2 : esc;
        }
    } while (--steps > 0 && !met && x < w.end);
    const bool over = met || x >= w.end, more = over && !met && w.sp > w.bot;
    w.hit = met;
    w.ref = x;
    if (more) w.ref = stack[--w.sp * 256];
    w.mode = more ? kWalkWide : (over ? kWalkDone : kWalkBinary);
}

// one step of every walking lane of the wave
__device__ __forceinline__ void walk_step(Walk& w, int* stack) {
    const bool at_leaf = w.mode == kWalkWide && w.ref < 0, at_node = w.mode == kWalkWide && w.ref >= 0;
    const uint32_t leaves = (uint32_t)__popcll(__ballot(at_leaf)), nodes = (uint32_t)__popcll(__ballot(at_node));
    if (kNodesPerLeaf * leaves >= nodes) {
        if (at_leaf) walk_leaf(w, stack);
    } else if (at_node) {
        walk_node(w, stack);
    }
    // (a wave whose walks are all binary stays with them for a while)
    if (__ballot(w.mode == kWalkBinary) != 0ull) {
        const int steps = leaves + nodes == 0u ? 16 : 1;
        if (w.mode == kWalkBinary) walk_binary(w, stack, steps);
    }
}

// The end of a launch waits for its longest walks, one step per load latency.
// A wave that has no more rays to fetch spreads the walks it still has over
// its idle lanes: every walking lane gives its oldest stack entry (the
// largest subtree) and a copy of its ray to one of them. pairs: 64 words of
// LDS of the wave. Returns whether the lane's ray is now (or was) shared.
__device__ __forceinline__ bool walk_share(Walk& w, uint32_t& slot, bool shared, uint64_t idle, uint32_t lane,
                                           int* column0, int* pairs, uint32_t* hits) {
    const uint64_t below = (1ull << lane) - 1ull;
    const bool gives = w.mode == kWalkWide && w.sp > w.bot;
    const uint64_t givers = __ballot(gives);
    const uint32_t n_idle = (uint32_t)__popcll(idle), n_give = (uint32_t)__popcll(givers);
    const uint32_t n = n_idle < n_give ? n_idle : n_give;
    const uint32_t give_rank = (uint32_t)__popcll(givers & below), idle_rank = (uint32_t)__popcll(idle & below);
    const bool giver = gives && give_rank < n, taker = w.mode == kWalkDone && idle_rank < n;
    if (giver) pairs[give_rank] = (int)lane;
    wave_sync();
    const int from = taker ? pairs[idle_rank] : (int)lane;
    wave_sync();
    // a ray that is shared for the first time: not hit, unless one of its
    // walks says otherwise
    if (giver && !shared) hits[slot] = 0u;
    const int bot = __shfl(w.bot, from);
    const int entry = column0[bot * 256 + from];
    auto copy = [&](float v) { return __shfl(v, from); };
    w.o = make_float3(copy(w.o.x), copy(w.o.y), copy(w.o.z));
    w.d = make_float3(copy(w.d.x), copy(w.d.y), copy(w.d.z));
    w.in = make_float3(copy(w.in.x), copy(w.in.y), copy(w.in.z));
    w.c = make_float3(copy(w.c.x), copy(w.c.y), copy(w.c.z));
    w.tmin = copy(w.tmin);
    w.tmax = copy(w.tmax);
    w.lo = copy(w.lo);
    w.hi = copy(w.hi);
    w.slack = copy(w.slack);
    w.rec = (const GlobalF4*)(uintptr_t)__shfl((unsigned long long)(uintptr_t)w.rec, from);
    w.wide = (const GlobalF4*)(uintptr_t)__shfl((unsigned long long)(uintptr_t)w.wide, from);
    slot = (uint32_t)__shfl((int)slot, from);
    const bool last = w.bot + 1 == w.sp;
    w.ref = taker ? entry : w.ref;
    w.sp = taker || (giver && last) ? 0 : w.sp;
    w.bot = taker || (giver && last) ? 0 : (giver ? w.bot + 1 : w.bot);
    w.mode = taker ? kWalkWide : w.mode;
    w.hit = taker ? false : w.hit;
    return taker || giver || (shared && w.mode != kWalkDone);
}

// Persistent walk of the shadow-ray list. A lane whose ray is done takes a
// new one as soon as `refill` lanes of its wave are idle (16 by default, 4%
// faster than 32 on the 1080p city: a step of the wide walk is worth four of
// the binary walk, whose best threshold was 24 to 32), so long rays do not
// hold a wave's other 63 lanes idle. Rays come
// in runs: the first from the wave's place in its slice, later ones from
// the slice's counter. (With one atomic per refill, waves without rays queued
// at eight counters: 0.1 of the 0.125 ms of a 63k-ray list.)
// Seven waves per SIMD: 70 VGPRs, no spills (eight spill: 1.8 ms against 1.2).
// Every wave leaves the loop: a wide walk only goes down, visiting a node at
// most once and a triangle at most once per slot that names it, and a binary
// walk moves forward in pre-order; each refill takes rays or moves to the next
// slice, and after kTraceQueues slices there is nothing left to fetch.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(7))) trace_kernel(TraceArgs A) {
    __shared__ int stacks[kWalkStack * 256];
    __shared__ int pair_lanes[256];
    int* stack = stacks + threadIdx.x;
    uint32_t count = *A.ray_count;
    if (count > A.max_rays) count = A.max_rays;
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t below = (1ull << lane) - 1ull;
    // the wave's own run of rays: its share of the first rays of its slice
    // without an atomic, later runs of `run` rays from the slices' counters
    const uint32_t waves = gridDim.x * 4u / kTraceQueues;  // per slice
    uint32_t q = blockIdx.x % kTraceQueues;
    const uint32_t wave = (blockIdx.x / kTraceQueues) * 4u + (threadIdx.x >> 6);
    uint32_t q0 = (uint32_t)(((uint64_t)count * q) / kTraceQueues);
    uint32_t len = (uint32_t)(((uint64_t)count * (q + 1u)) / kTraceQueues) - q0;
    const uint32_t most = (count + kTraceQueues - 1u) / kTraceQueues;  // the longest slice
    // A run is 32 rays while three waves per SIMD hold them all, then grows to
    // 128 with the ray count (a wave of few rays drains: its lanes idle while
    // its last walks end), and beyond what all waves hold, to an eighth of a
    // wave's share. 0.64M rays: 0.19 ms at 64 rays per run, 0.15 at 128; 63k
    // rays: 0.026 ms at 32, 0.046 at 128.
    const uint32_t three = waves * 3u / 7u + 1u, share = most / (waves * 8u);
    const uint32_t fill = most / three < 32u ? 32u : (most / three > 128u ? 128u : most / three);
    const uint32_t run = share <= fill ? fill : (share > 512u ? 512u : share);
    const uint32_t fixed = waves * run;
    uint32_t next = wave * run < len ? q0 + wave * run : q0;
    uint32_t left = wave * run < len ? (len - wave * run < run ? len - wave * run : run) : 0u;
    uint32_t tried = most <= fixed ? kTraceQueues : 0u;  // nothing beyond the first runs
    Walk w = {};
    uint32_t slot = 0;
    bool shared = false;  // the ray is walked by several lanes
    for (;;) {
        uint64_t idle = __ballot(w.mode == kWalkDone);
        uint32_t n_idle = (uint32_t)__popcll(idle);
        if (n_idle >= A.refill || n_idle == 64u) {
            while (left == 0u && tried < kTraceQueues) {
                uint32_t base = 0;
                if (lane == 0u) base = atomicAdd(&A.queues[q * kQueueStride], run);
                base = fixed + (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
                if (base < len) {
                    next = q0 + base;
                    left = len - base < run ? len - base : run;
                } else {
                    ++tried;
                    q = (q + 1u) % kTraceQueues;
                    q0 = (uint32_t)(((uint64_t)count * q) / kTraceQueues);
                    len = (uint32_t)(((uint64_t)count * (q + 1u)) / kTraceQueues) - q0;
                }
            }
            if (left > 0u) {
                const uint32_t j = (uint32_t)__popcll(idle & below);
                if (w.mode == kWalkDone && j < left) {
                    const uint32_t i = next + j;
                    ShadowRay r = A.rays[i];
                    slot = A.ray_slots[i];
                    shared = false;
                    walk_start(w, A.bvhs[__float_as_uint(r.org.w)], make_float3(r.org.x, r.org.y, r.org.z),
                               make_float3(r.dir.x, r.dir.y, r.dir.z), kShadowTMin, r.dir.w);
                }
                const uint32_t taken = n_idle < left ? n_idle : left;
                next += taken;
                left -= taken;
            }
        }
        idle = __ballot(w.mode == kWalkDone);
        if (idle == ~0ull) {
            if (left == 0u && tried >= kTraceQueues) break;
            continue;
        }
        if (left == 0u && tried >= kTraceQueues && (uint32_t)__popcll(idle) >= kShareLanes)
            shared = walk_share(w, slot, shared, idle, lane, stacks + (threadIdx.x & ~63u),
                                pair_lanes + (threadIdx.x & ~63u), A.hits);
#pragma unroll 1
        for (int it = 0; it < 4; ++it) {
            const bool walking = w.mode != kWalkDone;
            walk_step(w, stack);
            const bool ends = walking && w.mode == kWalkDone;
            if (ends && (w.hit || !shared)) A.hits[slot] = w.hit ? 1u : 0u;
            // the other walks of a shared ray that was hit end too
            uint64_t over = __ballot(ends && w.hit && shared);
            while (over != 0ull) {
                const int l = __ffsll((unsigned long long)over) - 1;
                over &= over - 1ull;
                const uint32_t s = (uint32_t)__builtin_amdgcn_readlane((int)slot, l);
                if (shared && slot == s) w.mode = kWalkDone;
            }
        }
    }
}

// the same walk over a caller's rays, 64 to a wave
__global__ void __launch_bounds__(256) trace_rays_kernel(BvhView B, const float* rays, uint32_t n, uint32_t* hits) {
    __shared__ int stacks[kWalkStack * 256];
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    Walk w = {};
    if (i < n) {
        const float4* r = reinterpret_cast<const float4*>(rays) + 2 * (size_t)i;
        float4 a = r[0], b = r[1];
        walk_start(w, B, make_float3(a.x, a.y, a.z), make_float3(b.x, b.y, b.z), a.w, b.w);
    }
    while (__ballot(w.mode != kWalkDone) != 0ull) walk_step(w, stacks + threadIdx.x);
    if (i < n) hits[i] = w.hit ? 1u : 0u;
}

__global__ void __launch_bounds__(256) primary_kernel(BvhView B, risltc_frame_constants_t c, uint32_t* out) {
    uint32_t W = c.viewport_size[0], H = c.viewport_size[1];
    uint32_t tiles_x = (W + 15u) / 16u;
    uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t x = (blockIdx.x % tiles_x) * 16u + (lane & 15u);
    uint32_t y = (blockIdx.x / tiles_x) * 16u + wave * 4u + (lane >> 4);
    if (x >= W || y >= H) return;
    const float(*P)[4] = c.pixel_to_ray_direction_world_space;
    float fx = (float)x, fy = (float)y;
    float3 d = make_float3(fma_(P[0][2], 1.0f, fma_(P[0][1], fy, P[0][0] * fx)),
                           fma_(P[1][2], 1.0f, fma_(P[1][1], fy, P[1][0] * fx)),
                           fma_(P[2][2], 1.0f, fma_(P[2][1], fy, P[2][0] * fx)));
    float3 o = make_float3(c.camera_position_world_space[0], c.camera_position_world_space[1],
                           c.camera_position_world_space[2]);
    out[y * W + x] = closest_hit(B, o, d, 0.0f, __builtin_inff());
}

// One resident grid: as many 256-lane work-groups as fit on the device at
// once, a multiple of the XCD count.
hipError_t trace_blocks(uint32_t* blocks) {
    int dev = 0, cus = 0, per_cu = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, trace_kernel, 256, 0);
    if (e != hipSuccess) return e;
    uint32_t b = (uint32_t)(cus > 0 ? cus : 1) * (uint32_t)(per_cu > 0 ? per_cu : 1);
    *blocks = (b + kTraceQueues - 1u) / kTraceQueues * kTraceQueues;
    return hipSuccess;
}

hipError_t launch_trace(const TraceArgs& a, hipStream_t s, uint32_t blocks) {
    if (blocks == 0 || blocks % kTraceQueues) return hipErrorInvalidValue;
    hipLaunchKernelGGL(trace_kernel, dim3(blocks), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_trace(const TraceArgs& a, hipStream_t s) {
    uint32_t blocks = 0;
    hipError_t e = trace_blocks(&blocks);
    if (e != hipSuccess) return e;
    return launch_trace(a, s, blocks);
}

hipError_t launch_trace_rays(const BvhView& bvh, const float* rays8, uint32_t n, uint32_t* hits, hipStream_t s) {
    hipLaunchKernelGGL(trace_rays_kernel, dim3((n + 255u) / 256u), dim3(256), 0, s, bvh, rays8, n, hits);
    return hipGetLastError();
}

hipError_t launch_primary(const BvhView& bvh, const uint2* positions, const risltc_frame_constants_t& c, uint32_t* out,
                          hipStream_t s) {
    (void)positions;
    uint32_t W = c.viewport_size[0], H = c.viewport_size[1];
    dim3 grid(((W + 15u) / 16u) * ((H + 15u) / 16u));
    hipLaunchKernelGGL(primary_kernel, grid, dim3(256), 0, s, bvh, c, out);
    return hipGetLastError();
}

}  // namespace rl
