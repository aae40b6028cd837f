// mlp.hip -- the learned RIS proposal: feature encoder, MLP inference and
// training on BF16 MFMA with FP32 accumulation.
//
// No reference code: the reference draws RIS candidates uniformly
// (shading_pass.frag.glsl:730-733). The proposal adds a per-pixel
// distribution over light clusters from a 96 -> 64 -> 64 -> 64 -> 256 MLP
// (softmax of its logits); the shade kernel mixes it half and half with the
// uniform source, so every light keeps probability >= 0.5 / N and the RIS
// estimator stays unbiased. It is trained online, by softmax cross-entropy,
// on the clusters of the lights that the pass's own RIS selects.
//
// Matrix products use v_mfma_f32_16x16x32_bf16. Lane l of a wave holds
// A[l % 16][8 (l / 16) .. + 7], B[8 (l / 16) .. + 7][l % 16] and returns
// C[4 (l / 16) + i][l % 16], i = 0..3 (checked on the device against a CPU
// product). Every product is written "NT": both operands K-contiguous, so
// each fragment is one 16-byte load.
//
// Features (96, per shading point): position p in the scene box mapped to
// [-1, 1]^3 (3); sin and cos of pi 2^f p for f = 0..6 (42); shading normal n
// (3); direction to the camera o (3); reflected direction r (3); GGX alpha,
// n.o, luminance of the diffuse albedo and of F0 (4); sin and cos of pi 2^f n
// and of pi 2^f r for f = 0, 1 (24); sin and cos of pi o (6); a constant 1;
// 7 zeros.
#include <hip/hip_runtime.h>

#include "devmath.hpp"
#include "gbuffer.hpp"
#include "kernels.hpp"

namespace rl {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// round to nearest even (finite values)
__device__ __forceinline__ uint16_t bf16_bits(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf16_float(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// two values rounded to nearest even by v_cvt_pk_bf16_f32: a in the low half
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t bf16_pack2(float a, float b) {
    f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

__device__ __forceinline__ bf16x8 frag(const uint16_t* p) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p));
}

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// makes one lane's LDS writes visible to the other lanes of its wave (the
// waves of a work-group run different trip counts, so no block barrier)
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---- feature encoder ----------------------------------------------------------------
// Writes the 96 features of the pixel's shading point; returns false (and
// zeros) for background, light and out-of-mesh pixels.
__device__ bool encode_features(const FeatureView& F, uint32_t pixel, float* f) {
#pragma unroll
    for (int k = 0; k < kMlpIn; ++k) f[k] = 0.0f;
    const SceneView& S = F.scene;
    const risltc_frame_constants_t& c = F.c;
    uint32_t prim = F.visibility[pixel];
    if (prim == 0xFFFFFFFFu || (prim >> 31) != 0u || (uint64_t)prim >= S.triangle_count) return false;
    const uint32_t W = c.viewport_size[0];
    float fx = (float)(pixel % W), fy = (float)(pixel / W);
    const float(*P)[4] = c.pixel_to_ray_direction_world_space;
    f3 ray = mk3(fma_(P[0][2], 1.0f, fma_(P[0][1], fy, P[0][0] * fx)),
                 fma_(P[1][2], 1.0f, fma_(P[1][1], fy, P[1][0] * fx)),
                 fma_(P[2][2], 1.0f, fma_(P[2][1], fy, P[2][0] * fx)));
    f3 p[3], nrm[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        size_t vi = (size_t)prim * 3 + i;
        p[i] = decode_position(S.positions[vi], c.mesh_dequantization_factor, c.mesh_dequantization_summand);
        ushort4 nt = S.normals_uv[vi];
        nrm[i] = decode_normal(nt.x, nt.y);
    }
    f3 org = mk3(c.camera_position_world_space[0], c.camera_position_world_space[1], c.camera_position_world_space[2]);
    f3 e0 = sub3(p[1], p[0]), e1 = sub3(p[2], p[0]);
    f3 rce1 = cross3(ray, e1);
    float rcp_det = 1.0f / dot3(e0, rce1);
    f3 r0 = sub3(org, p[0]);
    float by = rcp_det * dot3(r0, rce1);
    float bz = -rcp_det * dot3(ray, cross3(e0, r0));
    float bx = 1.0f - (by + bz);
    f3 pos = add3(add3(scl3(p[0], bx), scl3(p[1], by)), scl3(p[2], bz));
    f3 n = normalize3<false>(add3(add3(scl3(nrm[0], bx), scl3(nrm[1], by)), scl3(nrm[2], bz)));
    f3 o = normalize3<false>(sub3(org, pos));
    float ndo = dot3(n, o);
    if (ndo < 0.0f) {
        n = scl3(n, -1.0f);
        ndo = -ndo;
    }
    f3 r = sub3(scl3(n, 2.0f * ndo), o);
    uint32_t mi = S.material_idx[prim];
    if (mi >= S.material_count) mi = S.material_count - 1u;
    const float* m = S.materials + 6 * mi;
    float metal = m[5];
    float alum = (0.2126f * m[0] + 0.7152f * m[1] + 0.0722f * m[2]) * (1.0f - metal);
    float f0l = 0.02f * (1.0f - metal) + (0.2126f * m[0] + 0.7152f * m[1] + 0.0722f * m[2]) * metal;
    float alpha = clamp_(m[4] * m[4] * c.roughness_factor, 0.0064f, 1.0f);
    float q[3] = {(pos.x - F.center[0]) * F.inv_half[0], (pos.y - F.center[1]) * F.inv_half[1],
                  (pos.z - F.center[2]) * F.inv_half[2]};
    int k = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) f[k++] = q[a];
    // __builtin_amdgcn_sinf(x) = sin(2 pi x): sin(pi 2^j t) = sin(2 pi 2^(j-1) t)
    float scale = 0.5f;
#pragma unroll
    for (int j = 0; j < 7; ++j, scale *= 2.0f)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            f[k++] = __builtin_amdgcn_sinf(q[a] * scale);
            f[k++] = __builtin_amdgcn_cosf(q[a] * scale);
        }
    const float nv[3] = {n.x, n.y, n.z}, ov[3] = {o.x, o.y, o.z}, rv[3] = {r.x, r.y, r.z};
#pragma unroll
    for (int a = 0; a < 3; ++a) f[k++] = nv[a];
#pragma unroll
    for (int a = 0; a < 3; ++a) f[k++] = ov[a];
#pragma unroll
    for (int a = 0; a < 3; ++a) f[k++] = rv[a];
    f[k++] = alpha;
    f[k++] = ndo;
    f[k++] = alum;
    f[k++] = f0l;
    scale = 0.5f;
#pragma unroll
    for (int j = 0; j < 2; ++j, scale *= 2.0f)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            f[k++] = __builtin_amdgcn_sinf(nv[a] * scale);
            f[k++] = __builtin_amdgcn_cosf(nv[a] * scale);
            f[k++] = __builtin_amdgcn_sinf(rv[a] * scale);
            f[k++] = __builtin_amdgcn_cosf(rv[a] * scale);
        }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        f[k++] = __builtin_amdgcn_sinf(ov[a] * 0.5f);
        f[k++] = __builtin_amdgcn_cosf(ov[a] * 0.5f);
    }
    f[k++] = 1.0f;
    return true;
}

// ---- fused inference: features -> MLP -> per-pixel top-16 table -------------------
constexpr int kLdW1 = kMlpIn + 8;  // bf16 row strides (16-byte multiples)
template <int HID>
constexpr int ld_h() { return HID + 8; }

// What bounds it: VALU work on the logits, beside their matrix products. At
// 1080p, with four cycles to an instruction, VALU takes 58% of the cycles with
// 64 wide and 256 outputs and 72% with 128 wide and 1024, MFMA 10% and 22%,
// and waves wait for a third and a quarter of theirs. So the logits' own
// work is kept small: an insertion into a best-4 in 15 instructions, and for
// 256 outputs only where a group of four can matter. The weights are not in LDS
// (135 KB of it for the narrow network, and one wave per SIMD for the wide
// ones; a view of 62 thousand pixels spent a quarter of its time filling it):
// they are loaded from L2 as MFMA fragments, each once for a wave's 64 pixels.
// LDS holds a region per wave, two waves per SIMD for every network: in turn the
// 64 pixels' features, their hidden activations (a layer reads all its inputs
// into registers, then writes over them) and, with 256 outputs, the logits of
// 16 pixels. At 1920x1080, before and after: 128 wide with 1024 outputs 2810
// and 1332 us, with 256 outputs 1460 and 767, 64 wide with 1024 1369 and 1080,
// with 256 614 and 466; 333x187 with the last 43 and 28 us. Two waves per SIMD
// have 256 VGPRs: 256 outputs spill 46 (128 wide) and 30 of them, 1024 outputs
// 8 or 28 (128 wide, with logits) and none. Three waves per SIMD spill in the
// inner loops (64 wide, 256 outputs: 651 us); chunks of 16 tiles instead of 8 take
// 447 us there but 34 at 333x187, and chunks of 8 instead of 4 with 128 wide
// 980 us.
constexpr int kPropWaves = 4;
constexpr int kLdX = kMlpIn;  // bf16 row stride of the features, read only once
template <int HID, int OUT>
struct PropShared {
    static constexpr int kChunk = 512 / HID;      // output tiles at a time (256 outputs)
    static constexpr int kLdZ = 16 * kChunk + 4;  // floats per pixel of their logits
    static constexpr int kLdPair = 2 * 16 + 4;    // floats per pixel of two tiles (1024 outputs)
    static constexpr int kActBytes = 2 * 64 * (kLdX > ld_h<HID>() ? kLdX : ld_h<HID>());
    static constexpr int kLogitBytes = OUT > 256 ? 0 : 4 * 16 * kLdZ;
    float bias[3 * HID + OUT];
    uint32_t live[OUT];  // all ones, or 0 for an empty cluster
    uint4 region[kPropWaves][(kActBytes > kLogitBytes ? kActBytes : kLogitBytes) / 16];
    static_assert(kActBytes >= 4 * 64 * kLdPair, "two tiles of 64 pixels");
};
static_assert(sizeof(PropShared<64, 256>) <= 80 * 1024 && sizeof(PropShared<128, 256>) <= 80 * 1024 &&
                  sizeof(PropShared<64, 1024>) <= 80 * 1024 && sizeof(PropShared<128, 1024>) <= 80 * 1024,
              "two work-groups per CU");

// inserts value v of id into the sorted best-4 (ties keep the earlier one, a
// NaN is not taken): a sorted list's new entry q is the middle one of v, its
// old entry and the one before
__device__ __forceinline__ void insert4(float v, int id, float (&bv)[4], int (&bi)[4]) {
    const float v0 = bv[0], v1 = bv[1], v2 = bv[2], v3 = bv[3];
    const int i0 = bi[0], i1 = bi[1], i2 = bi[2], i3 = bi[3];
    const int n0 = v > v0 ? id : i0, n1 = v > v1 ? id : i1, n2 = v > v2 ? id : i2, n3 = v > v3 ? id : i3;
    bv[0] = fmax_(v, v0);
    bv[1] = __builtin_amdgcn_fmed3f(v, v0, v1);
    bv[2] = __builtin_amdgcn_fmed3f(v, v1, v2);
    bv[3] = __builtin_amdgcn_fmed3f(v, v2, v3);
    bi[0] = n0;
    bi[1] = v > v0 ? i0 : n1;
    bi[2] = v > v1 ? i1 : n2;
    bi[3] = v > v2 ? i2 : n3;
}

// the logit where `live` is all ones, -inf where it is 0 (one v_bfi)
__device__ __forceinline__ float live_logit(float z, uint32_t live) {
    return __uint_as_float((__float_as_uint(z) & live) | (0xff800000u & ~live));
}
// Four floats or eight halfwords at an address that need only be a multiple of
// four: the callers' logits and features.
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(4)));

// log sum exp of a quad's logits (-inf: not live); NaN when none is live,
// which insert4 never takes
__device__ __forceinline__ float quad_value(const float (&z)[4]) {
    const float m = fmax_(fmax_(z[0], z[1]), fmax_(z[2], z[3]));
    float sum = __expf(z[0] - m);
#pragma unroll
    for (int i = 1; i < 4; ++i) sum += __expf(z[i] - m);
    return m + __logf(sum);
}

// the larger four of two descending lists, descending (values only)
__device__ __forceinline__ void keep4(float (&a)[4], const float (&b)[4]) {
    float t[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) t[i] = fmax_(a[i], b[3 - i]);
    const float p = fmax_(t[0], t[2]), q = fmin_(t[0], t[2]), r = fmax_(t[1], t[3]), s = fmin_(t[1], t[3]);
    a[0] = fmax_(p, r);
    a[1] = fmin_(p, r);
    a[2] = fmax_(q, s);
    a[3] = fmin_(q, s);
}
__device__ __forceinline__ void sort4(float (&a)[4]) {
    const float p = fmax_(a[0], a[1]), q = fmin_(a[0], a[1]), r = fmax_(a[2], a[3]), s = fmin_(a[2], a[3]);
    const float u = fmin_(p, r), v = fmax_(q, s);
    a[0] = fmax_(p, r);
    a[1] = fmax_(u, v);
    a[2] = fmin_(u, v);
    a[3] = fmin_(q, s);
}

// a layer's weight fragments of output tile t: rows 16 t + r of [out][K]
template <int K>
__device__ __forceinline__ void weight_frags(const uint16_t* W, int t, int lane, bf16x8 (&w)[K / 32]) {
    const uint16_t* p = W + (size_t)(16 * t + (lane & 15)) * K + 8 * (lane >> 4);
#pragma unroll
    for (int k = 0; k < K / 32; ++k) w[k] = frag(p + 32 * k);
}

// the wave's 64 pixels' activations as B fragments: sub-tile s in b[s]
template <int K, int LD>
__device__ __forceinline__ void act_frags(const uint16_t* act, int lane, bf16x8 (&b)[4][K / 32]) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int k = 0; k < K / 32; ++k) b[s][k] = frag(act + (16 * s + (lane & 15)) * LD + 32 * k + 8 * (lane >> 4));
}

// hidden layer on the wave's 64 pixels, in place:
// act[pixel][o] = relu(W[o] . act[pixel] + bias[o])
template <int HID, int K, int LD>
__device__ __forceinline__ void hidden_layer(const uint16_t* W, const float* bias, uint16_t* act, int lane) {
    const int g = lane >> 4, r = lane & 15;
    bf16x8 b[4][K / 32], w[K / 32];
    weight_frags<K>(W, 0, lane, w);
    act_frags<K, LD>(act, lane, b);
    wave_sync();
#pragma unroll 2
    for (int t = 0; t < HID / 16; ++t) {
        bf16x8 next[K / 32];
        weight_frags<K>(W, t + 1 < HID / 16 ? t + 1 : t, lane, next);
        const float4 c = *reinterpret_cast<const float4*>(bias + 16 * t + 4 * g);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k = 0; k < K / 32; ++k) acc = mfma(w[k], b[s][k], acc);
            const float v[4] = {fmax_(acc[0] + c.x, 0.0f), fmax_(acc[1] + c.y, 0.0f), fmax_(acc[2] + c.z, 0.0f),
                                fmax_(acc[3] + c.w, 0.0f)};
            *reinterpret_cast<uint2*>(act + (16 * s + r) * ld_h<HID>() + 16 * t + 4 * g) =
                make_uint2(bf16_pack2(v[0], v[1]), bf16_pack2(v[2], v[3]));
        }
#pragma unroll
        for (int k = 0; k < K / 32; ++k) w[k] = next[k];
        __builtin_amdgcn_sched_barrier(0);
    }
    wave_sync();
}

// the four table slots of lane group g of a pixel: ids and weights
// round(255 exp(value - the pixel's largest value))
__device__ __forceinline__ void put_slots(uint8_t* table, int g, bool in, bool shaded, const float (&bv)[4],
                                          const int (&bi)[4]) {
    // the pixel's maximum over its four lanes (lanes r, r+16, r+32, r+48)
    float zmax = bv[0];
    zmax = fmax_(zmax, __shfl_xor(zmax, 16));
    zmax = fmax_(zmax, __shfl_xor(zmax, 32));
    uint32_t ws = 0, ids = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float e = __expf(bv[q] - zmax) * 255.0f + 0.5f;
        const uint32_t we = e >= 255.0f ? 255u : (uint32_t)fmax_(e, 0.0f);
        const uint32_t w = shaded && bv[q] > -__builtin_inff() ? we : 0u;
        ids |= (w == 0u ? 0u : (uint32_t)bi[q]) << (8 * q);
        ws |= w << (8 * q);
    }
    if (in) {
        // slot 4 g + q: id at byte 4 g + q, weight at 16 + 4 g + q
        uint32_t* o = reinterpret_cast<uint32_t*>(table);
        o[g] = ids;
        o[4 + g] = ws;
    }
}

// LOGITS: whether the caller's logits are written. 1024 of them a pixel are
// bound by those stores. A lane has four of a tile, so a tile's store is 64
// bytes at a time, 4 KB apart, and half lines leave L2; and a wait for the next
// weights waits for the stores before it too. Two tiles therefore go through
// LDS and out as 128 contiguous bytes a pixel: 1300x777, 128 wide, 2080 -> 1230
// us (with one tile's ranking between its stores and the next products alone:
// 2060), 64 wide 1580 -> 1050. Without the logits the kernel is its own
// instantiation. With 256 outputs the weights of several tiles are loaded at
// once, the stores cost 80 of 490 us, and one instantiation serves both.
template <int HID, int OUT, bool LOGITS>
__global__ void __launch_bounds__(64 * kPropWaves) __attribute__((amdgpu_waves_per_eu(2)))
proposal_kernel(ProposalArgs A) {
    constexpr MlpLayout L = mlp_layout(HID, OUT);
    constexpr int KH = HID / 32;
    using Sh = PropShared<HID, OUT>;
    __shared__ Sh sh;
    const int tid = (int)threadIdx.x, wave = tid >> 6;
    for (int e = tid; e < HID; e += blockDim.x) {
        sh.bias[e] = A.params[L.pb1 + e];
        sh.bias[HID + e] = A.params[L.pb2 + e];
        sh.bias[2 * HID + e] = A.params[L.pb3 + e];
    }
    for (int e = tid; e < OUT; e += blockDim.x) {
        sh.bias[3 * HID + e] = A.params[L.pb4 + e];
        sh.live[e] = (uint32_t)e < A.cluster_count && A.cluster_offsets[e + 1] != A.cluster_offsets[e] ? ~0u : 0u;
    }
    __syncthreads();
    uint16_t* act = reinterpret_cast<uint16_t*>(sh.region[wave]);
    const uint32_t groups = (A.pixel_count + 63u) / 64u;
    for (uint32_t grp = blockIdx.x * kPropWaves + wave; grp < groups; grp += gridDim.x * kPropWaves) {
        // keeps the weights' loads and the lane's addresses inside this loop:
        // hoisted out of it they would need more registers than there are
        uint32_t none = 0;
        int lane = tid & 63;
        asm volatile("" : "+s"(none), "+v"(lane));
        const int g = lane >> 4, r = lane & 15;
        const uint16_t *wf = A.wf + none, *w4 = wf + L.pw4;
        const float* bias4 = sh.bias + 3 * HID + 4 * g;
        const uint32_t* live4 = sh.live + 4 * g;
        const uint32_t my_pixel = grp * 64u + (uint32_t)lane;
        const bool my_in = my_pixel < A.pixel_count;
        bool my_shaded;
        {
            float f[kMlpIn];
            my_shaded = my_in && encode_features(A.f, my_pixel, f);
            if (!my_in) {
#pragma unroll
                for (int k = 0; k < kMlpIn; ++k) f[k] = 0.0f;
            }
#pragma unroll
            for (int k = 0; k < kMlpIn; k += 8) {
                const uint4 p = make_uint4(bf16_pack2(f[k], f[k + 1]), bf16_pack2(f[k + 2], f[k + 3]),
                                           bf16_pack2(f[k + 4], f[k + 5]), bf16_pack2(f[k + 6], f[k + 7]));
                *reinterpret_cast<uint4*>(act + lane * kLdX + k) = p;
                if (A.features && my_in)
                    *reinterpret_cast<u32x4_any*>(A.features + (size_t)my_pixel * kMlpIn + k) =
                        u32x4_any{p.x, p.y, p.z, p.w};
            }
        }
        wave_sync();
        hidden_layer<HID, kMlpIn, kLdX>(wf + L.pw1, sh.bias, act, lane);
        hidden_layer<HID, HID, ld_h<HID>()>(wf + L.pw2, sh.bias + HID, act, lane);
        hidden_layer<HID, HID, ld_h<HID>()>(wf + L.pw3, sh.bias + 2 * HID, act, lane);
        bf16x8 hb[4][KH];
        act_frags<HID, ld_h<HID>()>(act, lane, hb);
        wave_sync();
        if constexpr (OUT > 256) {
            // quads: for sub-tile s this lane ranks quad 4 t + g of pixel
            // 16 s + r, one value per tile
            float bv[4][4];
            int bi[4][4];
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    bv[s][i] = -__builtin_inff();
                    bi[s][i] = 0;
                }
            bf16x8 w[KH];
            weight_frags<HID>(w4, 0, lane, w);
#pragma unroll 2
            for (int t = 0; t < OUT / 16; ++t) {
                bf16x8 next[KH];
                weight_frags<HID>(w4, t + 1 < OUT / 16 ? t + 1 : t, lane, next);
                const float4 c = *reinterpret_cast<const float4*>(bias4 + 16 * t);
                const uint4 d = *reinterpret_cast<const uint4*>(live4 + 16 * t);
                f32x4 z[4];
#pragma unroll
                for (int s = 0; s < 4; ++s) z[s] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int k = 0; k < KH; ++k)
#pragma unroll
                    for (int s = 0; s < 4; ++s) z[s] = mfma(w[k], hb[s][k], z[s]);
#pragma unroll
                for (int s = 0; s < 4; ++s) z[s] = f32x4{z[s][0] + c.x, z[s][1] + c.y, z[s][2] + c.z, z[s][3] + c.w};
                if constexpr (LOGITS) {
                    float* zs = reinterpret_cast<float*>(act);
#pragma unroll
                    for (int s = 0; s < 4; ++s)
                        *reinterpret_cast<f32x4*>(zs + (16 * s + r) * Sh::kLdPair + 16 * (t & 1) + 4 * g) = z[s];
                    if ((t & 1) != 0) {
                        wave_sync();
                        const uint32_t p0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(grp * 64u));
                        float* out = A.logits + (size_t)p0 * OUT + 16 * (t - 1);
                        const uint32_t row = (uint32_t)lane >> 3, col = 4u * ((uint32_t)lane & 7u);
                        auto put = [&](uint32_t j) {
                            *reinterpret_cast<f32x4_any*>(out + ((row + j) * (uint32_t)OUT + col)) =
                                *reinterpret_cast<const f32x4*>(zs + (row + j) * Sh::kLdPair + col);
                        };
                        // (without the test the eight reads are in flight together)
                        if (A.pixel_count - p0 >= 64u) {
#pragma unroll
                            for (uint32_t j = 0; j < 64u; j += 8u) put(j);
                        } else {
#pragma unroll 1
                            for (uint32_t j = 0; j < 64u; j += 8u)
                                if (row + j < A.pixel_count - p0) put(j);
                        }
                        wave_sync();
                    }
                } else {
                    // (a tile's products mixed with its ranking: 1401 us at
                    // 1920x1080, 128 wide, instead of 1332)
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const float zl[4] = {live_logit(z[s][0], d.x), live_logit(z[s][1], d.y), live_logit(z[s][2], d.z),
                                         live_logit(z[s][3], d.w)};
                    insert4(quad_value(zl), 4 * t + g, bv[s], bi[s]);
                }
#pragma unroll
                for (int k = 0; k < KH; ++k) w[k] = next[k];
            }
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const uint32_t pixel = grp * 64u + (uint32_t)(16 * s + r);
                const bool shaded = __shfl(my_shaded ? 1 : 0, 16 * s + r) != 0;
                put_slots(A.out + (size_t)pixel * kPropBytes, g, pixel < A.pixel_count, shaded, bv[s], bi[s]);
            }
        } else {
            // kChunk tiles' weights stay in registers for the four sub-tiles.
            // Of each the logits go to LDS and the maxima of the lane's
            // groups of four (one a tile) stay in registers. The best four
            // logits lie in groups whose maximum is at least the fourth
            // largest maximum (four others are as large), so only those are
            // inserted one by one: 4 groups instead of 16, unless maxima tie.
            constexpr int CT = Sh::kChunk;
            float* zs = reinterpret_cast<float*>(act);
            float bv[4][4];
            int bi[4][4];
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    bv[s][i] = -__builtin_inff();
                    bi[s][i] = 0;
                }
#pragma unroll 1
            for (int t0 = 0; t0 < OUT / 16; t0 += CT) {
                bf16x8 w[CT][KH];
#pragma unroll
                for (int t = 0; t < CT; ++t) weight_frags<HID>(w4, t0 + t, lane, w[t]);
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const uint32_t pixel = grp * 64u + (uint32_t)(16 * s + r);
                    const bool in = pixel < A.pixel_count;
                    float top[CT];
                    uint32_t none4 = 0;  // as above, for the biases
                    asm volatile("" : "+s"(none4));
                    const float* bias4s = bias4 + none4;
                    const uint32_t* live4s = live4 + none4;
#pragma unroll
                    for (int t4 = 0; t4 < CT; t4 += 4) {
                        f32x4 z[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) z[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int k = 0; k < KH; ++k)
#pragma unroll
                            for (int i = 0; i < 4; ++i) z[i] = mfma(w[t4 + i][k], hb[s][k], z[i]);
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float4 c = *reinterpret_cast<const float4*>(bias4s + 16 * (t0 + t4 + i));
                            z[i] = f32x4{z[i][0] + c.x, z[i][1] + c.y, z[i][2] + c.z, z[i][3] + c.w};
                        }
                        if (A.logits) {
                            if (in) {
#pragma unroll
                                for (int i = 0; i < 4; ++i)
                                    *reinterpret_cast<f32x4_any*>(A.logits + (size_t)pixel * OUT + 16 * (t0 + t4 + i) + 4 * g) =
                                        z[i];
                            }
                        }
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int t = t4 + i;
                            const uint4 d = *reinterpret_cast<const uint4*>(live4s + 16 * (t0 + t));
                            const float4 zl = make_float4(live_logit(z[i][0], d.x), live_logit(z[i][1], d.y),
                                                          live_logit(z[i][2], d.z), live_logit(z[i][3], d.w));
                            *reinterpret_cast<float4*>(zs + r * Sh::kLdZ + 16 * t + 4 * g) = zl;
                            // -inf for four NaN
                            top[t] = fmax_(fmax_(zl.x, fmax_(zl.z, zl.w)), fmax_(zl.y, -__builtin_inff()));
                        }
                    }
                    float best[4] = {top[0], top[1], top[2], top[3]};
                    sort4(best);
#pragma unroll
                    for (int q = 4; q < CT; q += 4) {
                        float more[4] = {top[q], top[q + 1], top[q + 2], top[q + 3]};
                        sort4(more);
                        keep4(best, more);
                    }
                    uint32_t groups_of = 0;
#pragma unroll
                    for (int t = 0; t < CT; ++t)
                        groups_of |= (top[t] >= best[3] && top[t] > bv[s][3]) ? 1u << t : 0u;
                    wave_sync();
                    while (groups_of != 0u) {
                        const int t = __builtin_ctz(groups_of);
                        groups_of &= groups_of - 1u;
                        const int c0 = 16 * (t0 + t) + 4 * g;
                        const float4 z = *reinterpret_cast<const float4*>(zs + r * Sh::kLdZ + 16 * t + 4 * g);
                        insert4(z.x, c0, bv[s], bi[s]);
                        insert4(z.y, c0 + 1, bv[s], bi[s]);
                        insert4(z.z, c0 + 2, bv[s], bi[s]);
                        insert4(z.w, c0 + 3, bv[s], bi[s]);
                    }
                    wave_sync();
                }
            }
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const uint32_t pixel = grp * 64u + (uint32_t)(16 * s + r);
                // every lane of the pixel's column learns whether it is shaded
                const bool shaded = __shfl(my_shaded ? 1 : 0, 16 * s + r) != 0;
                put_slots(A.out + (size_t)pixel * kPropBytes, g, pixel < A.pixel_count, shaded, bv[s], bi[s]);
            }
        }
    }
}

hipError_t launch_proposal(const ProposalArgs& a, hipStream_t s) {
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    const bool wide = a.L.hid == kMlpHidWide, many = a.L.out == kMlpOutWide;
    if ((!wide && a.L.hid != kMlpHid) || (!many && a.L.out != kMlpOut)) return hipErrorInvalidValue;
    const uint32_t groups = (a.pixel_count + 63u) / 64u;
    uint32_t blocks = (groups + kPropWaves - 1u) / kPropWaves;
    // the waves take 64 pixels at a time; more than fit at once would only
    // read the biases again
    const uint32_t cap = 2u * (uint32_t)(cus > 0 ? cus : 1);
    if (blocks > cap) blocks = cap;
    dim3 grid(blocks), block(64 * kPropWaves);
    if (many && a.logits) {
        if (wide) hipLaunchKernelGGL((proposal_kernel<kMlpHidWide, kMlpOutWide, true>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((proposal_kernel<kMlpHid, kMlpOutWide, true>), grid, block, 0, s, a);
    } else if (many) {
        if (wide) hipLaunchKernelGGL((proposal_kernel<kMlpHidWide, kMlpOutWide, false>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((proposal_kernel<kMlpHid, kMlpOutWide, false>), grid, block, 0, s, a);
    } else {
        if (wide) hipLaunchKernelGGL((proposal_kernel<kMlpHidWide, kMlpOut, true>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((proposal_kernel<kMlpHid, kMlpOut, true>), grid, block, 0, s, a);
    }
    return hipGetLastError();
}

// ---- training --------------------------------------------------------------------
// A step is four kernels: the batch's features (train_gather_kernel), the
// forward and backward pass of the batch's rows (train_rows_kernel), the
// weight gradients as split-K products (weight_grad_kernel) and their
// reduction with the Adam update (train_finish_kernel). The rows are
// independent until the weight gradients, so a work-group keeps its rows'
// activations and logits in LDS; what leaves it are the transposed
// activations and gradients, whose rows the weight gradients read K-contiguous.
// What bounds it: 12 GFLOP on 65,536 rows are 10 us of matrix cores; the 24
// small launches that this replaces took 730 us (of them 440 in sums by one
// work-group with one load in flight).
__device__ __forceinline__ uint32_t hash32(uint32_t x) {
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}

// batch item b: a pseudo-random pixel-sample; features (both layouts), the
// cluster of its selected light and a weight (1, or 0 without a selection);
// count: the items of weight 1
__global__ void __launch_bounds__(256) train_gather_kernel(TrainArgs A, uint16_t* X, uint16_t* Xt, uint32_t* target,
                                                           float* y, uint32_t* count) {
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t item = hash32(A.seed * 0x9E3779B9u + b) % A.sample_count;
    const uint32_t pixel = item / A.spp;
    float f[kMlpIn];
    bool ok = encode_features(A.f, pixel, f);
    uint32_t c = A.rec_cluster[item];
    float w = 1.0f;
    if (!ok || c >= (uint32_t)A.L.out) {
        c = 0u;
        w = 0.0f;
    }
    target[b] = c;
    y[b] = w;
    const uint32_t used = (uint32_t)__popcll(__ballot(w != 0.0f));
    if ((threadIdx.x & 63u) == 0u && used != 0u) atomicAdd(count, used);
    uint32_t p[kMlpIn / 2];
#pragma unroll
    for (int k = 0; k < kMlpIn / 2; ++k) p[k] = bf16_pack2(f[2 * k], f[2 * k + 1]);
    uint4* row = reinterpret_cast<uint4*>(X + (size_t)b * kMlpIn);
#pragma unroll
    for (int k = 0; k < kMlpIn / 8; ++k) row[k] = make_uint4(p[4 * k], p[4 * k + 1], p[4 * k + 2], p[4 * k + 3]);
#pragma unroll
    for (int k = 0; k < kMlpIn; ++k) Xt[(size_t)k * A.B + b] = (uint16_t)(p[k / 2] >> (16 * (k & 1)));
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax_(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// rows per work-group: their logits fill 32 to 64 KB of LDS; 8 waves (with 4,
// the default network's 65,536 rows take 85 us instead of 66)
constexpr int kRowWaves = 8;
template <int OUT>
constexpr int train_rows() { return OUT > 256 ? 16 : 32; }

template <int HID, int OUT>
struct RowsShared {
    static constexpr int kRows = train_rows<OUT>();
    static constexpr int kLdZ = OUT + 4;      // floats per row of logits
    static constexpr int kLdG = 2 * kLdZ;     // the same row's gradient as bf16, in place
    uint16_t x[kRows * kLdW1];
    uint16_t h[3][kRows * ld_h<HID>()];
    uint16_t g[2][kRows * ld_h<HID>()];
    float z[kRows * kLdZ];
};
static_assert(sizeof(RowsShared<64, 256>) <= 80 * 1024, "two work-groups per CU");
static_assert(sizeof(RowsShared<128, 1024>) <= 160 * 1024, "LDS");

// C[m][n] = A[m][K] . Wt[n][K]^T of the work-group's rows, A in LDS, Wt in
// global memory (it stays in L2): put(m, n, four values of rows m..m + 3)
template <int ROWS, int N, int K, int LDA, class F>
__device__ __forceinline__ void rows_product(const uint16_t* A, const uint16_t* Wt, F put) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, gq = lane >> 4, r = lane & 15;
    // (a wave keeps its rows, so that narrow layers occupy every wave)
    constexpr int MT = ROWS / 16, WN = kRowWaves / MT;
    const int m = wave / WN;
    for (int t = wave % WN; t < N / 16; t += WN) {
        bf16x8 b[K / 32];
#pragma unroll
        for (int k = 0; k < K / 32; ++k) b[k] = frag(Wt + (size_t)(16 * t + r) * K + 32 * k + 8 * gq);
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < K / 32; ++k) acc = mfma(frag(A + (16 * m + r) * LDA + 32 * k + 8 * gq), b[k], acc);
        put(16 * m + 4 * gq, 16 * t + r, acc);
    }
}

// dst[n][b0 ..] = column n of the work-group's rows (LDS, LD values a row)
template <int ROWS, int N, int LD>
__device__ __forceinline__ void put_transposed(const uint16_t* src, uint16_t* dst, uint32_t B, uint32_t b0) {
    for (int e = threadIdx.x; e < N * (ROWS / 8); e += 64 * kRowWaves) {
        const int n = e % N, q = 8 * (e / N);
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            w[j] = (uint32_t)src[(q + 2 * j) * LD + n] | ((uint32_t)src[(q + 2 * j + 1) * LD + n] << 16);
        *reinterpret_cast<uint4*>(dst + (size_t)n * B + b0 + q) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

struct RowsArgs {
    MlpLayout L;
    const uint16_t *wf, *wb;
    const float* params;
    const uint16_t* X;
    const uint32_t* target;
    const float* y;
    const uint32_t* count;
    uint32_t B;
    uint16_t *Ht[3], *Gt[4];  // Gt[l]: gradient at the output of layer l + 1
    float* row_loss;
};

template <int HID, int OUT>
__global__ void __launch_bounds__(64 * kRowWaves) train_rows_kernel(RowsArgs A) {
    constexpr int ROWS = train_rows<OUT>(), LDH = ld_h<HID>(), PER = OUT / 64;
    using Sh = RowsShared<HID, OUT>;
    constexpr MlpLayout L = mlp_layout(HID, OUT);
    __shared__ Sh sh;
    const uint32_t b0 = blockIdx.x * ROWS;  // B is a multiple of ROWS
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int e = threadIdx.x; e < ROWS * (kMlpIn / 8); e += 64 * kRowWaves) {
        const int row = e / (kMlpIn / 8), q = e % (kMlpIn / 8);
        *reinterpret_cast<uint4*>(sh.x + row * kLdW1 + 8 * q) =
            *reinterpret_cast<const uint4*>(A.X + (size_t)(b0 + row) * kMlpIn + 8 * q);
    }
    __syncthreads();
    // forward
    auto hidden = [&](int layer, int bias) {
        return [&A, layer, bias](int m, int n, f32x4 v) {
            const float c = A.params[bias + n];
#pragma unroll
            for (int i = 0; i < 4; ++i) sh.h[layer][(m + i) * LDH + n] = bf16_bits(fmax_(v[i] + c, 0.0f));
        };
    };
    rows_product<ROWS, HID, kMlpIn, kLdW1>(sh.x, A.wf + L.pw1, hidden(0, L.pb1));
    __syncthreads();
    rows_product<ROWS, HID, HID, LDH>(sh.h[0], A.wf + L.pw2, hidden(1, L.pb2));
    __syncthreads();
    rows_product<ROWS, HID, HID, LDH>(sh.h[1], A.wf + L.pw3, hidden(2, L.pb3));
    __syncthreads();
    rows_product<ROWS, OUT, HID, LDH>(sh.h[2], A.wf + L.pw4, [&](int m, int n, f32x4 v) {
        const float c = A.params[L.pb4 + n];
#pragma unroll
        for (int i = 0; i < 4; ++i) sh.z[(m + i) * Sh::kLdZ + n] = v[i] + c;
    });
#pragma unroll
    for (int l = 0; l < 3; ++l) put_transposed<ROWS, HID, LDH>(sh.h[l], A.Ht[l], A.B, b0);
    __syncthreads();
    // dL/dz = (y_b / Y) (softmax(z_b) - onehot(c_b)), one wave per row at a
    // time, each lane OUT / 64 of the logits; the row's loss term
    uint16_t* g4 = reinterpret_cast<uint16_t*>(sh.z);
    const float Y = (float)*A.count;
    for (int rr = 0; rr < ROWS / kRowWaves; ++rr) {
        const int r = wave * (ROWS / kRowWaves) + rr;
        const uint32_t b = b0 + r;
        float v[PER];
#pragma unroll
        for (int k = 0; k < PER; ++k) v[k] = sh.z[r * Sh::kLdZ + lane + 64 * k];
        float m = v[0];
#pragma unroll
        for (int k = 1; k < PER; ++k) m = fmax_(m, v[k]);
        const float zm = wave_max(m);
        float e[PER], part = 0.0f;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            e[k] = __expf(v[k] - zm);
            part += e[k];
        }
        const float s = wave_sum(part);
        const float wb = Y > 0.0f ? A.y[b] / Y : 0.0f;
        const uint32_t c = A.target[b];
        wave_sync();
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const uint32_t n = (uint32_t)lane + 64u * k;
            g4[r * Sh::kLdG + n] = bf16_bits(wb * (e[k] / s - (n == c ? 1.0f : 0.0f)));
        }
        // z[c] from the lane that holds it (c is the same for the whole wave)
        float vc = v[0];
#pragma unroll
        for (int k = 1; k < PER; ++k)
            if ((c >> 6) == (uint32_t)k) vc = v[k];
        const float zc = __shfl(vc, (int)(c & 63u));
        if (lane == 0) A.row_loss[b] = wb > 0.0f ? -wb * (zc - zm - __logf(s)) : 0.0f;
    }
    __syncthreads();
    // backward: dA[b][i] = sum_o G[b][o] W[o][i], masked by the activation
    // (wb holds the weights as [in][out])
    auto back = [&](int to, int layer) {
        return [to, layer](int m, int n, f32x4 v) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                sh.g[to][(m + i) * LDH + n] =
                    bf16_float(sh.h[layer][(m + i) * LDH + n]) > 0.0f ? bf16_bits(v[i]) : (uint16_t)0;
        };
    };
    rows_product<ROWS, HID, OUT, Sh::kLdG>(g4, A.wb + L.pw4, back(0, 2));
    put_transposed<ROWS, OUT, Sh::kLdG>(g4, A.Gt[3], A.B, b0);
    __syncthreads();
    rows_product<ROWS, HID, HID, LDH>(sh.g[0], A.wb + L.pw3, back(1, 1));
    put_transposed<ROWS, HID, LDH>(sh.g[0], A.Gt[2], A.B, b0);
    __syncthreads();
    rows_product<ROWS, HID, HID, LDH>(sh.g[1], A.wb + L.pw2, back(0, 0));
    put_transposed<ROWS, HID, LDH>(sh.g[1], A.Gt[1], A.B, b0);
    __syncthreads();
    put_transposed<ROWS, HID, LDH>(sh.g[0], A.Gt[0], A.B, b0);
}

// Weight gradients of the four layers: partial[slice][o][i] = sum over the
// slice's batch items of Gt[o][b] At[i][b]. One wave computes a 16 x 32 block
// of one slice; the loads of four steps are in flight together.
constexpr uint32_t kTrainSlice = 2048;  // batch items per slice
struct GradArgs {
    const uint16_t *Gt[4], *At[4];
    uint32_t nout[4], nin[4];
    uint32_t block0[5];   // 16 x 32 blocks of the layers, prefix sums
    size_t partial0[4];   // of each layer's partial sums
    uint32_t B, slices;
    float* partial;
};

__global__ void __launch_bounds__(256) weight_grad_kernel(GradArgs g) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, gq = lane >> 4, r = lane & 15;
    const uint32_t blk = blockIdx.x * 4u + (uint32_t)wave, slice = blockIdx.y;
    if (blk >= g.block0[4]) return;
    int l = 0;
    while (l < 3 && blk >= g.block0[l + 1]) ++l;
    const uint32_t nblk = g.nin[l] / 32u, e = blk - g.block0[l];
    const uint32_t m0 = (e / nblk) * 16u, n0 = (e % nblk) * 32u;
    const uint32_t k0 = slice * kTrainSlice, k1 = min(g.B, k0 + kTrainSlice);
    const uint16_t* pa = g.Gt[l] + (size_t)(m0 + r) * g.B + 8 * gq;
    const uint16_t* pb = g.At[l] + (size_t)(n0 + r) * g.B + 8 * gq;
    const uint16_t* pc = pb + (size_t)16 * g.B;
    f32x4 acc0 = {0.0f, 0.0f, 0.0f, 0.0f}, acc1 = acc0;
    // (B is a multiple of 256, so a slice is a multiple of 128)
    for (uint32_t k = k0; k < k1; k += 128u) {
        bf16x8 a[4], b[4], c[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            a[u] = frag(pa + k + 32 * u);
            b[u] = frag(pb + k + 32 * u);
            c[u] = frag(pc + k + 32 * u);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            acc0 = mfma(a[u], b[u], acc0);
            acc1 = mfma(a[u], c[u], acc1);
        }
    }
    float* o = g.partial + g.partial0[l] + (size_t)slice * g.nout[l] * g.nin[l];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        o[(size_t)(m0 + 4u * gq + i) * g.nin[l] + n0 + r] = acc0[i];
        o[(size_t)(m0 + 4u * gq + i) * g.nin[l] + n0 + 16u + r] = acc1[i];
    }
}

// bf16 copies of layer weights: wf = master layout [out][in], wb = [in][out]
__device__ __forceinline__ void layer_of(const MlpLayout& L, int e, int& off, int& nout, int& nin) {
    if (e < L.pb1) {
        off = L.pw1, nout = L.hid, nin = kMlpIn;
    } else if (e >= L.pw2 && e < L.pb2) {
        off = L.pw2, nout = L.hid, nin = L.hid;
    } else if (e >= L.pw3 && e < L.pb3) {
        off = L.pw3, nout = L.hid, nin = L.hid;
    } else if (e >= L.pw4 && e < L.pb4) {
        off = L.pw4, nout = L.out, nin = L.hid;
    } else {
        off = -1, nout = nin = 0;
    }
}

__device__ __forceinline__ void write_copies(const MlpLayout& L, int e, float v, uint16_t* wf, uint16_t* wb) {
    uint16_t h = bf16_bits(v);
    wf[e] = h;
    int off, nout, nin;
    layer_of(L, e, off, nout, nin);
    if (off >= 0) {
        int o = (e - off) / nin, i = (e - off) % nin;
        wb[off + i * nout + o] = h;
    } else {
        wb[e] = h;
    }
}

// one Adam step of parameter e with gradient gr
__device__ __forceinline__ void adam(const TrainArgs& A, int e, float gr) {
    A.grad[e] = gr;
    const float m = A.beta1 * A.m[e] + (1.0f - A.beta1) * gr;
    const float v = A.beta2 * A.v[e] + (1.0f - A.beta2) * gr * gr;
    A.m[e] = m;
    A.v[e] = v;
    const float bc1 = 1.0f - __powf(A.beta1, (float)A.step);
    const float bc2 = 1.0f - __powf(A.beta2, (float)A.step);
    const float p = A.params[e] - A.lr * (m / bc1) / (__builtin_sqrtf(v / bc2) + A.eps);
    A.params[e] = p;
    write_copies(A.L, e, p, A.wf, A.wb);
}

// thread t's values t, t + 256, .. of a row of n (a multiple of 256) summed in
// that order, 16 loads in flight, then a fixed tree over the work-group
template <class F>
__device__ __forceinline__ float row_sum(uint32_t n, F at) {
    __shared__ float part[256];
    const uint32_t t = threadIdx.x;
    float s = 0.0f;
    uint32_t i = t;
    for (; i + 15u * 256u < n; i += 16u * 256u) {
        float v[16];
#pragma unroll
        for (uint32_t u = 0; u < 16u; ++u) v[u] = at(i + 256u * u);
#pragma unroll
        for (uint32_t u = 0; u < 16u; ++u) s += v[u];
    }
    for (; i < n; i += 256u) s += at(i);
    part[t] = s;
    __syncthreads();
    for (uint32_t w = 128u; w > 0u; w >>= 1) {
        if (t < w) part[t] += part[t + w];
        __syncthreads();
    }
    return part[0];
}

// The end of a step, by work-group: 256 weights (their slices' sum in slice
// order), or one bias (the sum of its row of Gt), each with its Adam update,
// or the loss.
struct FinishArgs {
    TrainArgs t;
    const uint16_t* Gt[4];
    uint32_t weights[4], biases[4];  // counts
    int w0[4], b0[4];                // parameter offsets
    uint32_t block0[5];              // weight work-groups of the layers, prefix sums
    size_t partial0[4];
    uint32_t slices;
    const float* partial;
    const float* row_loss;
};

__global__ void __launch_bounds__(256) train_finish_kernel(FinishArgs F) {
    uint32_t blk = blockIdx.x;
    if (blk < F.block0[4]) {
        int l = 0;
        while (l < 3 && blk >= F.block0[l + 1]) ++l;
        const uint32_t i = (blk - F.block0[l]) * 256u + threadIdx.x;
        if (i >= F.weights[l]) return;
        const float* p = F.partial + F.partial0[l] + i;
        const size_t step = F.weights[l];
        float s = 0.0f;
        uint32_t k = 0;
        for (; k + 8u <= F.slices; k += 8u) {
            float v[8];
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u) v[u] = p[(k + u) * step];
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u) s += v[u];
        }
        for (; k < F.slices; ++k) s += p[k * step];
        adam(F.t, F.w0[l] + (int)i, s);
        return;
    }
    blk -= F.block0[4];
    for (int l = 0; l < 4; ++l) {
        if (blk < F.biases[l]) {
            const uint16_t* g = F.Gt[l] + (size_t)blk * F.t.B;
            const float s = row_sum(F.t.B, [&](uint32_t i) { return bf16_float(g[i]); });
            if (threadIdx.x == 0) adam(F.t, F.b0[l] + (int)blk, s);
            return;
        }
        blk -= F.biases[l];
    }
    const float s = row_sum(F.t.B, [&](uint32_t i) { return F.row_loss[i]; });
    if (threadIdx.x == 0) *F.t.loss = s;
}

__global__ void sync_kernel(MlpLayout L, const float* params, uint16_t* wf, uint16_t* wb) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= L.params) return;
    write_copies(L, e, params[e], wf, wb);
}

hipError_t launch_mlp_sync(const MlpLayout& L, const float* params, uint16_t* wf, uint16_t* wb, hipStream_t s) {
    hipLaunchKernelGGL(sync_kernel, dim3((L.params + 255) / 256), dim3(256), 0, s, L, params, wf, wb);
    return hipGetLastError();
}

namespace {
struct TrainScratch {
    uint16_t *X, *Xt, *Ht[3], *Gt[4];
    float *y, *row_loss, *partial;
    uint32_t *target, *count;
    size_t partial0[4];  // of each layer's partial weight gradients
};
size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }
TrainScratch carve(void* base, uint32_t B, int hid, int out, size_t* total) {
    TrainScratch t;
    size_t off = 0;
    char* p = static_cast<char*>(base);
    auto take = [&](size_t bytes) -> void* {
        void* q = p ? p + off : nullptr;
        off += align256(bytes);
        return q;
    };
    t.X = (uint16_t*)take(2ull * B * kMlpIn);
    t.Xt = (uint16_t*)take(2ull * B * kMlpIn);
    for (int l = 0; l < 3; ++l) t.Ht[l] = (uint16_t*)take(2ull * B * hid);
    for (int l = 0; l < 4; ++l) t.Gt[l] = (uint16_t*)take(2ull * B * (l == 3 ? out : hid));
    t.y = (float*)take(4ull * B);
    t.row_loss = (float*)take(4ull * B);
    const size_t slices = (B + kTrainSlice - 1) / kTrainSlice;
    size_t sums = 0;
    const size_t weights[4] = {(size_t)hid * kMlpIn, (size_t)hid * hid, (size_t)hid * hid, (size_t)out * hid};
    for (int l = 0; l < 4; ++l) {
        t.partial0[l] = sums;
        sums += slices * weights[l];
    }
    t.partial = (float*)take(4ull * sums);
    t.target = (uint32_t*)take(4ull * B);
    t.count = (uint32_t*)take(4);
    if (total) *total = off;
    return t;
}
}  // namespace

size_t train_scratch_bytes(uint32_t B, int hid, int out) {
    size_t total = 0;
    carve(nullptr, B, hid, out, &total);
    return total;
}

hipError_t launch_train_step(const TrainArgs& a, hipStream_t s) {
    if (a.B == 0 || a.B % 256u != 0u || a.sample_count == 0) return hipErrorInvalidValue;
    const MlpLayout& L = a.L;
    const uint32_t H = (uint32_t)L.hid, O = (uint32_t)L.out, B = a.B, slices = (B + kTrainSlice - 1) / kTrainSlice;
    if ((H != (uint32_t)kMlpHid && H != (uint32_t)kMlpHidWide) || (O != (uint32_t)kMlpOut && O != (uint32_t)kMlpOutWide))
        return hipErrorInvalidValue;
    const TrainScratch t = carve(a.scratch, B, L.hid, L.out, nullptr);
    hipError_t e = launch_zero_u32(t.count, 1u, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(train_gather_kernel, dim3(B / 256u), dim3(256), 0, s, a, t.X, t.Xt, t.target, t.y, t.count);
    RowsArgs r{L, a.wf, a.wb, a.params, t.X, t.target, t.y, t.count, B, {}, {}, t.row_loss};
    for (int l = 0; l < 3; ++l) r.Ht[l] = t.Ht[l];
    for (int l = 0; l < 4; ++l) r.Gt[l] = t.Gt[l];
    const bool wide = H == (uint32_t)kMlpHidWide, many = O == (uint32_t)kMlpOutWide;
    if (wide && many)
        hipLaunchKernelGGL((train_rows_kernel<kMlpHidWide, kMlpOutWide>), dim3(B / 16u), dim3(64 * kRowWaves), 0, s, r);
    else if (wide)
        hipLaunchKernelGGL((train_rows_kernel<kMlpHidWide, kMlpOut>), dim3(B / 32u), dim3(64 * kRowWaves), 0, s, r);
    else if (many)
        hipLaunchKernelGGL((train_rows_kernel<kMlpHid, kMlpOutWide>), dim3(B / 16u), dim3(64 * kRowWaves), 0, s, r);
    else
        hipLaunchKernelGGL((train_rows_kernel<kMlpHid, kMlpOut>), dim3(B / 32u), dim3(64 * kRowWaves), 0, s, r);
    GradArgs g{};
    FinishArgs f{};
    f.t = a;
    const uint16_t* At[4] = {t.Xt, t.Ht[0], t.Ht[1], t.Ht[2]};
    const int w0[4] = {L.pw1, L.pw2, L.pw3, L.pw4}, b0[4] = {L.pb1, L.pb2, L.pb3, L.pb4};
    uint32_t biases = 0;
    for (int l = 0; l < 4; ++l) {
        g.Gt[l] = f.Gt[l] = t.Gt[l];
        g.At[l] = At[l];
        g.nout[l] = f.biases[l] = l == 3 ? O : H;
        g.nin[l] = l == 0 ? (uint32_t)kMlpIn : H;
        f.weights[l] = g.nout[l] * g.nin[l];
        g.block0[l + 1] = g.block0[l] + f.weights[l] / (16u * 32u);
        f.block0[l + 1] = f.block0[l] + (f.weights[l] + 255u) / 256u;
        g.partial0[l] = f.partial0[l] = t.partial0[l];
        f.w0[l] = w0[l];
        f.b0[l] = b0[l];
        biases += f.biases[l];
    }
    g.B = B;
    g.slices = f.slices = slices;
    g.partial = t.partial;
    f.partial = t.partial;
    f.row_loss = t.row_loss;
    hipLaunchKernelGGL(weight_grad_kernel, dim3((g.block0[4] + 3u) / 4u, slices), dim3(256), 0, s, g);
    hipLaunchKernelGGL(train_finish_kernel, dim3(f.block0[4] + biases + 1u), dim3(256), 0, s, f);
    return hipGetLastError();
}

}  // namespace rl
