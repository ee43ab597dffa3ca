// fields.hpp -- structure-of-arrays layout of the link and E fields in HBM.
//
// A field is stored in 16-byte words: every plane holds one word of every site
// x, word after word, so that a wavefront over 64 consecutive sites reads
// 1 KiB in one fully coalesced request with 16 bytes per lane.
//   links, f64: per direction 9 planes, entry k = row * 3 + col as (re, im);
//   links, f32: per direction 4 planes of entry pairs (0, 1), (3, 4), (2, 5),
//               (6, 7) as (re, im, re, im), then a plane of 8-byte words with
//               entry 8;
//   E, f64:     per direction 4 planes of components (2w, 2w + 1);
//   E, f32:     per direction 2 planes of components (4w .. 4w + 3).
// Planes have g.npad words.  The words are 16 bytes because the vector L1
// looks up four lanes at a time: a load of 4 or 8 bytes per lane takes it as
// long as one of 16 (about 16 accesses per wavefront either way), and the f32
// MD kernel, with 352 such accesses of 4 and 8 bytes per wavefront, kept it busy
// 79 % of the time.  With 16-byte words it issues 160: a 32^4 f32 trajectory of
// 40 steps went from 11.54 to 10.30 ms, 64 batched chains from 24.2 to 21.5 ms.
//
// Accesses are raw buffer loads / stores: the resource covers the planes of
// one direction (uniform, so it lives in scalar registers), the site enters
// as a 32-bit byte offset and the element plane as the scalar offset.  No
// per-lane 64-bit address arithmetic is left, and an access outside the
// direction's planes reads zero instead of faulting.  The planes of one
// direction must therefore span less than 4 GiB (kMaxPlaneBytes).
#pragma once
#include "geometry.hpp"
#include "su3_device.hpp"

namespace lqcd {

// descriptor word 3 of a raw buffer resource on the gfx9 family
constexpr int kBufferFlags = 0x00020000;

// cache-policy operand of a buffer access on gfx950: 0 is the default; bit 1
// (nt) marks the line non-temporal, so the L2 evicts it first.  Fields that a
// kernel reads or writes exactly once (E, the new links) use kCacheStream and
// leave the L2 to the neighbour links that other sites read again.
constexpr int kCacheDefault = 0;
constexpr int kCacheStream = 2;

template <typename S>
struct vec2;
template <>
struct vec2<float> {
    using type = float2;
};
template <>
struct vec2<double> {
    using type = double2;
};
template <typename S>
using vec2_t = typename vec2<S>::type;

// resource over `planes` planes of npad elements of type E starting at p
template <typename E>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t planes_rsrc(const E* p, int64_t npad, int planes)
{
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)((uint64_t)planes * npad * sizeof(E)),
                                             kBufferFlags);
}

template <typename E, int CP = kCacheDefault>
__device__ __forceinline__ E buf_load(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff)
{
    if constexpr (sizeof(E) == 4) {
        return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, (int)soff, CP));
    } else if constexpr (sizeof(E) == 8) {
        return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, (int)soff, CP));
    } else {
        static_assert(sizeof(E) == 16, "element of 4, 8 or 16 bytes");
        return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, (int)soff, CP));
    }
}

template <typename E, int CP = kCacheDefault>
__device__ __forceinline__ void buf_store(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff, E v)
{
    if constexpr (sizeof(E) == 4) {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, (int)off, (int)soff, CP);
    } else if constexpr (sizeof(E) == 8) {
        using V = __attribute__((ext_vector_type(2))) uint32_t;
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(V, v), r, (int)off, (int)soff, CP);
    } else {
        static_assert(sizeof(E) == 16, "element of 4, 8 or 16 bytes");
        using V = __attribute__((ext_vector_type(4))) uint32_t;
        // soffset 0, the plane offset in the VGPR offset: the compiler inserts
        // the wait state that a VALU write of the data VGPRs right after a
        // store of more than 64 bits needs only when soffset is not a
        // register, and without it such writes reach memory in place of the
        // stored data
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(V, v), r, (int)(off + soff), 0, CP);
    }
}

// The f32 pairs are chosen so that the parts of a link that kernels read or write
// alone are whole words: rows 0 and 1 (the two-row reads and stores) are pairs
// 0-2, columns 0 and 1 (the normalisation) pairs 0, 1 and 3.  With pairs of
// consecutive entries the normalisation read four words for three: us, 2048^2
// 231 -> 198, 128^3 171 -> 148, 32^4 89 -> 77; the per-site kernels with additive
// drift on small D = 3 lattices gained too (25x17x31 17.8 -> 12.5).

// Byte offset of f64 entry k, f32 pair k / 2 or the last f32 entry (k = 8) of
// site `s` within a direction's planes, as a per-lane part and a uniform part.
template <typename S>
__device__ __forceinline__ uint32_t link_off(int64_t s, int k)
{
    return (uint32_t)s * (sizeof(S) == 4 && k < 8 ? 16u : 2u * (uint32_t)sizeof(S));
}
template <typename S>
__device__ __forceinline__ uint32_t link_plane(int64_t npad, int k)
{
    return (uint32_t)k * (uint32_t)npad * 2u * (uint32_t)sizeof(S);
}

// Calls f(pair, entry, entry) for the f32 pairs of entries [K0, K1): all, rows 0
// and 1 (K0 = 0, K1 = 6) or row 2's first two (K0 = 6).  Both parts of a link that a
// kernel reads or writes alone are whole pairs: rows 0 and 1 (the two-row
// reads and stores) pairs 0-2, columns 0 and 1 (the normalisation) pairs 0, 1 and 3.
// With pairs of consecutive entries the normalisation read a third more than it
// needs: XXNORM.
// entries [K0, K1) of the link at byte offset `base` (per lane) of resource r
template <int K0, int K1, typename T, typename S, int CP>
__device__ __forceinline__ void load_entries(__amdgpu_buffer_rsrc_t r, uint32_t base, int64_t npad, int64_t s,
                                             mat3<T>& m)
{
    if constexpr (sizeof(S) == 4) {
        static_assert((K0 == 0 || K0 == 6) && (K1 == 6 || K1 == 9), "f32 links are read in whole pairs");
        const uint32_t off = base + link_off<S>(s, 0);
        if constexpr (K0 == 0) {
            const float4 p = buf_load<float4, CP>(r, off, link_plane<S>(npad, 0));
            const float4 q = buf_load<float4, CP>(r, off, link_plane<S>(npad, 2));
            const float4 t = buf_load<float4, CP>(r, off, link_plane<S>(npad, 4));
            m.e[0] = {T(p.x), T(p.y)};
            m.e[1] = {T(p.z), T(p.w)};
            m.e[2] = {T(t.x), T(t.y)};
            m.e[3] = {T(q.x), T(q.y)};
            m.e[4] = {T(q.z), T(q.w)};
            m.e[5] = {T(t.z), T(t.w)};
        }
        if constexpr (K1 == 9) {
            const float4 p = buf_load<float4, CP>(r, off, link_plane<S>(npad, 6));
            const float2 q = buf_load<float2, CP>(r, base + link_off<S>(s, 8), link_plane<S>(npad, 8));
            m.e[6] = {T(p.x), T(p.y)};
            m.e[7] = {T(p.z), T(p.w)};
            m.e[8] = {T(q.x), T(q.y)};
        }
    } else {
#pragma unroll
        for (int k = K0; k < K1; ++k) {
            const double2 v = buf_load<double2, CP>(r, base + link_off<S>(s, k), link_plane<S>(npad, k));
            m.e[k] = {T(v.x), T(v.y)};
        }
    }
}

// entries [K0, K1) of U_mu(x) from m
template <int K0, int K1, typename T, typename S, int CP>
__device__ __forceinline__ void store_entries(vec2_t<S>* __restrict__ U, int64_t npad, int mu, int64_t s,
                                              const mat3<T>& m)
{
    const __amdgpu_buffer_rsrc_t r = planes_rsrc(U + (int64_t)mu * 9 * npad, npad, 9);
    if constexpr (sizeof(S) == 4) {
        static_assert((K0 == 0 || K0 == 6) && (K1 == 6 || K1 == 9), "f32 links are written in whole pairs");
        const uint32_t off = link_off<S>(s, 0);
        auto word = [&](int i, int j) __attribute__((always_inline)) {
            return make_float4(S(m.e[i].re), S(m.e[i].im), S(m.e[j].re), S(m.e[j].im));
        };
        if constexpr (K0 == 0) {
            buf_store<float4, CP>(r, off, link_plane<S>(npad, 0), word(0, 1));
            buf_store<float4, CP>(r, off, link_plane<S>(npad, 2), word(3, 4));
            float4 v = word(2, 5);
            // opaque here: from the two halves of entries that are not neighbours
            // the compiler makes overlapping vector reads of m, and m then
            // stays in memory (k_drift 6.8 -> 20 us)
            asm("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w));
            buf_store<float4, CP>(r, off, link_plane<S>(npad, 4), v);
        }
        if constexpr (K1 == 9) {
            buf_store<float4, CP>(r, off, link_plane<S>(npad, 6), word(6, 7));
            buf_store<float2, CP>(r, link_off<S>(s, 8), link_plane<S>(npad, 8),
                                  make_float2(S(m.e[8].re), S(m.e[8].im)));
        }
    } else {
#pragma unroll
        for (int k = K0; k < K1; ++k)
            buf_store<double2, CP>(r, link_off<S>(s, k), link_plane<S>(npad, k),
                                   make_double2(S(m.e[k].re), S(m.e[k].im)));
    }
}

template <typename T, typename S, int CP = kCacheDefault>
__device__ __forceinline__ mat3<T> load_link(const vec2_t<S>* __restrict__ U, int64_t npad, int mu,
                                             int64_t s)
{
    mat3<T> m;
    load_entries<0, 9, T, S, CP>(planes_rsrc(U + (int64_t)mu * 9 * npad, npad, 9), 0, npad, s, m);
    return m;
}

// The first two rows of U_mu(x) (entries 0-5); row 2 is not written.
template <typename T, typename S>
__device__ __forceinline__ mat3<T> load_link_rows01(const vec2_t<S>* __restrict__ U, int64_t npad, int mu,
                                                    int64_t s)
{
    mat3<T> m;
    load_entries<0, 6, T, S, kCacheDefault>(planes_rsrc(U + (int64_t)mu * 9 * npad, npad, 9), 0, npad, s, m);
    return m;
}

// U_mu(x) from its first two rows: for a matrix of SU(3) the third row is
// the complex conjugate of the cross product of the first two,
//   u_2c = conj(u_0,c+1 u_1,c+2 - u_0,c+2 u_1,c+1),
// so six of the nine planes are read.  Exact for SU(3); callers use it only on
// links checked to be in SU(3) to rounding.
template <typename T, typename S>
__device__ __forceinline__ mat3<T> load_link_r12(const vec2_t<S>* __restrict__ U, int64_t npad, int mu,
                                                 int64_t s)
{
    mat3<T> m = load_link_rows01<T, S>(U, npad, mu, s);
    complete_su3(m);
    return m;
}

// load_link, or load_link_r12 when R12
template <bool R12, typename T, typename S>
__device__ __forceinline__ mat3<T> load_link_sel(const vec2_t<S>* __restrict__ U, int64_t npad, int mu, int64_t s)
{
    if constexpr (R12)
        return load_link_r12<T, S>(U, npad, mu, s);
    else
        return load_link<T, S>(U, npad, mu, s);
}

template <typename T, typename S, int CP = kCacheDefault>
__device__ __forceinline__ void store_link(vec2_t<S>* __restrict__ U, int64_t npad, int mu, int64_t s,
                                           const mat3<T>& m)
{
    store_entries<0, 9, T, S, CP>(U, npad, mu, s, m);
}

// Rows 0 and 1 of U_mu(x) only (entries 0-5): for links in SU(3) whose
// readers rebuild row 2 (load_link_r12) or which get it back from
// complete_row2_link before any other reader.
template <typename T, typename S, int CP = kCacheDefault>
__device__ __forceinline__ void store_link_rows01(vec2_t<S>* __restrict__ U, int64_t npad, int mu, int64_t s,
                                                  const mat3<T>& m)
{
    store_entries<0, 6, T, S, CP>(U, npad, mu, s, m);
}

// Row 2 of U_mu(x) only (entries 6-8).
template <typename T, typename S, int CP = kCacheDefault>
__device__ __forceinline__ void store_link_row2(vec2_t<S>* __restrict__ U, int64_t npad, int mu, int64_t s,
                                                const mat3<T>& m)
{
    store_entries<6, 9, T, S, CP>(U, npad, mu, s, m);
}

template <typename T, typename S, int CP = kCacheDefault>
__device__ __forceinline__ void load_e(const S* __restrict__ E, int64_t npad, int mu, int64_t s, T* e)
{
    const __amdgpu_buffer_rsrc_t r = planes_rsrc(E + (int64_t)mu * 8 * npad, npad, 8);
    const uint32_t off = (uint32_t)s * 16u, plane = (uint32_t)npad * 16u;
    if constexpr (sizeof(S) == 4) {
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const float4 v = buf_load<float4, CP>(r, off, (uint32_t)w * plane);
            e[4 * w] = T(v.x);
            e[4 * w + 1] = T(v.y);
            e[4 * w + 2] = T(v.z);
            e[4 * w + 3] = T(v.w);
        }
    } else {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const double2 v = buf_load<double2, CP>(r, off, (uint32_t)w * plane);
            e[2 * w] = T(v.x);
            e[2 * w + 1] = T(v.y);
        }
    }
}

template <typename T, typename S, int CP = kCacheDefault>
__device__ __forceinline__ void store_e(S* __restrict__ E, int64_t npad, int mu, int64_t s, const T* e)
{
    const __amdgpu_buffer_rsrc_t r = planes_rsrc(E + (int64_t)mu * 8 * npad, npad, 8);
    const uint32_t off = (uint32_t)s * 16u, plane = (uint32_t)npad * 16u;
    if constexpr (sizeof(S) == 4) {
#pragma unroll
        for (int w = 0; w < 2; ++w)
            buf_store<float4, CP>(r, off, (uint32_t)w * plane,
                                  make_float4(S(e[4 * w]), S(e[4 * w + 1]), S(e[4 * w + 2]), S(e[4 * w + 3])));
    } else {
#pragma unroll
        for (int w = 0; w < 4; ++w)
            buf_store<double2, CP>(r, off, (uint32_t)w * plane, make_double2(S(e[2 * w]), S(e[2 * w + 1])));
    }
}

} // namespace lqcd
