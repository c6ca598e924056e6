// rr_interleaved_dev.hpp -- engine wrappers of the interleaved generators (MRG32k3a,
// MRG31k3p, XORWOW, LFSR113), shared by the per-call kernels (rr_interleaved.hip) and
// the batched kernels (rr_batched.hip).  State layout: structure-of-arrays, word j of
// engine e at states[j*S + e].
#pragma once

#include "rr_launch.hpp"

namespace rr
{
namespace inter_dev
{

// Engines of the DEFAULT grid; the per-call kernels take the call's engine count (the
// DYNAMIC grid may differ), the batched kernels use this one.
constexpr uint32_t S = INTERLEAVED_ENGINES;

template<inter_kind K>
struct ieng;

// One radix-table entry (both components) applied to the state.
template<uint32_t K, uint32_t C1, uint32_t C2>
__device__ __forceinline__ void mrg_entry_apply(const uint32_t* entry, mrg_state& s)
{
    const uint4* p = reinterpret_cast<const uint4*>(entry);
    uint32_t     w[MRG_RADIX_WORDS];
#pragma unroll
    for(int i = 0; i < MRG_RADIX_WORDS / 4; i++)
    {
        const uint4 q = p[i];
        w[4 * i + 0]  = q.x;
        w[4 * i + 1]  = q.y;
        w[4 * i + 2]  = q.z;
        w[4 * i + 3]  = q.w;
    }
    mat3_vec_fold<K, C1>(w, s.g1);
    mat3_vec_fold<K, C2>(w + 9, s.g2);
}

// Jump to subsequence e mod 2^17 with the radix tables: X^(e mod 512), then
// X^(512 ((e / 512) mod 256)); the powers commute.  Same state as the binary expansion
// over the A^(2^(sub + i)) table of the reference's skipahead_subsequence.  (Engines at
// or beyond 2^17, which only a larger DYNAMIC grid has, add their high part by that
// binary expansion: see ieng::sub.)
template<uint32_t K, uint32_t C1, uint32_t C2>
__device__ __forceinline__ void mrg_sub_jump(const uint32_t* tab, uint32_t e, mrg_state& s)
{
    const uint32_t lo = e & (uint32_t)(MRG_RADIX_LO - 1);
    const uint32_t hi = (e >> MRG_RADIX_LO_BITS) & (uint32_t)(MRG_RADIX_HI - 1);
    if(lo != 0u)
        mrg_entry_apply<K, C1, C2>(tab + lo * MRG_RADIX_WORDS, s);
    if(hi != 0u)
        mrg_entry_apply<K, C1, C2>(tab + (MRG_RADIX_LO + hi) * MRG_RADIX_WORDS, s);
}

template<>
struct ieng<inter_kind::mrg32k3a>
{
    static constexpr word_family F = word_family::mrg32;
    mrg_state                    s;
    __device__ void load(const uint32_t* st, uint32_t e, uint32_t ns = S)
    {
#pragma unroll
        for(int j = 0; j < 3; j++)
        {
            s.g1[j] = st[j * ns + e];
            s.g2[j] = st[(3 + j) * ns + e];
        }
    }
    __device__ void store(uint32_t* st, uint32_t e, uint32_t ns = S) const
    {
#pragma unroll
        for(int j = 0; j < 3; j++)
        {
            st[j * ns + e]       = s.g1[j];
            st[(3 + j) * ns + e] = s.g2[j];
        }
    }
    __host__ __device__ void set(const uint32_t* w)
    {
        for(int j = 0; j < 3; j++)
        {
            s.g1[j] = w[j];
            s.g2[j] = w[3 + j];
        }
    }
    __device__ uint32_t next() { return mrg32k3a_next(s); }
    // Apply X^(sum of set bits) from a table of X^(2^i) (rocrand_mrg32k3a.h:204-263).
    __device__ void jump(const uint32_t* tab, uint64_t v)
    {
        for(int i = 0; v > 0; v >>= 1, i++)
            if(v & 1)
            {
                mat3_vec_fold<32, 209>(tab + (i * 2 + 0) * 9, s.g1);
                mat3_vec_fold<32, 22853>(tab + (i * 2 + 1) * 9, s.g2);
            }
    }
    // X^j for j < 512: one radix-table entry
    __device__ void sub_entry(const device_tables& t, uint32_t j)
    {
        mrg_entry_apply<32, 209, 22853>(t.mrg32_subr + j * MRG_RADIX_WORDS, s);
    }
    __device__ void sub(const device_tables& t, uint32_t e)
    {
        mrg_sub_jump<32, 209, 22853>(t.mrg32_subr, e, s);
        if(e >> 17) // A^(2^(76+17+i)) rows of the subsequence table
            jump(t.mrg32_sub + 17 * 2 * 9, e >> 17);
    }
    // k steps ahead (rocrand_mrg32k3a.h:246-263)
    __device__ void advance(const device_tables& t, uint64_t k) { jump(t.mrg32_step, k); }
    __device__ void init(const device_tables& t, uint32_t e, uint64_t off)
    {
        sub(t, e);
        jump(t.mrg32_step, off);
    }
};

template<>
struct ieng<inter_kind::mrg31k3p> : ieng<inter_kind::mrg32k3a>
{
    static constexpr word_family F = word_family::mrg31;
    __device__ uint32_t next() { return mrg31k3p_next(s); }
    __device__ void jump(const uint32_t* tab, uint64_t v)
    {
        for(int i = 0; v > 0; v >>= 1, i++)
            if(v & 1)
            {
                mat3_vec_fold<31, 1>(tab + (i * 2 + 0) * 9, s.g1);
                mat3_vec_fold<31, 21069>(tab + (i * 2 + 1) * 9, s.g2);
            }
    }
    __device__ void sub_entry(const device_tables& t, uint32_t j)
    {
        mrg_entry_apply<31, 1, 21069>(t.mrg31_subr + j * MRG_RADIX_WORDS, s);
    }
    __device__ void sub(const device_tables& t, uint32_t e)
    {
        mrg_sub_jump<31, 1, 21069>(t.mrg31_subr, e, s);
        if(e >> 17) // A^(2^(72+17+i)) rows of the subsequence table
            jump(t.mrg31_sub + 17 * 2 * 9, e >> 17);
    }
    __device__ void advance(const device_tables& t, uint64_t k) { jump(t.mrg31_step, k); }
    __device__ void init(const device_tables& t, uint32_t e, uint64_t off)
    {
        sub(t, e);
        jump(t.mrg31_step, off);
    }
};

// acc ^ (a & b) in one instruction (v_bitop3_b32)
__device__ __forceinline__ uint32_t xor_and(uint32_t acc, uint32_t a, uint32_t b)
{
    return __builtin_amdgcn_bitop3_b32(acc, a, b, 0x78);
}

// GF(2) matrix (row per input bit, N words per row; 16-byte aligned, the same for every
// lane, normally in LDS) times each lane's vector, four rows per N 16-byte broadcast reads.
template<int N>
__device__ __forceinline__ void gf2_mat_vec_shared(const uint32_t* m, uint32_t* v)
{
    const uint4* q    = reinterpret_cast<const uint4*>(m);
    uint32_t     r[N] = {};
#pragma unroll
    for(int i = 0; i < N; i++)
    {
        const uint32_t vi = v[i];
#pragma unroll 2
        for(int j = 0; j < 32; j += 4, q += N)
        {
            uint32_t w[4 * N];
#pragma unroll
            for(int k = 0; k < N; k++)
            {
                const uint4 t = q[k];
                w[4 * k] = t.x, w[4 * k + 1] = t.y, w[4 * k + 2] = t.z, w[4 * k + 3] = t.w;
            }
#pragma unroll
            for(int l = 0; l < 4; l++)
            {
                const uint32_t b = 0u - ((vi >> (j + l)) & 1u);
#pragma unroll
                for(int k = 0; k < N; k++)
                    r[k] = xor_and(r[k], w[l * N + k], b);
            }
        }
    }
#pragma unroll
    for(int k = 0; k < N; k++)
        v[k] = r[k];
}

// v = m v for a whole block with one matrix, staged in LDS (`lds`: 32 N^2 words, 16-byte
// aligned).  Every thread of the block must call it.
template<int N>
__device__ __forceinline__ void gf2_apply_block(uint32_t* v, const uint32_t* m, uint32_t times, uint32_t* lds)
{
    __syncthreads(); // the previous matrix is no longer read
    for(int w = threadIdx.x; w < 32 * N * N; w += blockDim.x)
        lds[w] = m[w];
    __syncthreads();
    for(uint32_t i = 0; i < times; i++)
        gf2_mat_vec_shared<N>(lds, v);
}

// Base-4 digit expansion with matrix k = M^(c * 4^k) applied digit times
// (rocrand_xorwow.h:186-200, rocrand_lfsr113.h jump()), for a whole block whose lanes
// share `n` (block-uniform): each 4^k power is staged once in LDS and read from there by
// every lane.  Every thread of the block must call it.
template<int N>
__device__ void gf2_jump_block(uint32_t* v, const uint32_t* mats, uint64_t n, uint32_t* lds)
{
    for(int k = 0; n > 0; n >>= 2, k++)
        if((n & 3u) != 0)
            gf2_apply_block<N>(v, mats + (size_t)k * 32 * N * N, (uint32_t)(n & 3u), lds);
}

template<>
struct ieng<inter_kind::xorwow>
{
    static constexpr word_family F = word_family::w32;
    xorwow_state                 s;
    __device__ void load(const uint32_t* st, uint32_t e, uint32_t ns = S)
    {
        s.d = st[e];
#pragma unroll
        for(int j = 0; j < 5; j++)
            s.x[j] = st[(1 + j) * ns + e];
    }
    __device__ void store(uint32_t* st, uint32_t e, uint32_t ns = S) const
    {
        st[e] = s.d;
#pragma unroll
        for(int j = 0; j < 5; j++)
            st[(1 + j) * ns + e] = s.x[j];
    }
    __host__ __device__ void set(const uint32_t* w)
    {
        s.d = w[0];
        for(int j = 0; j < 5; j++)
            s.x[j] = w[1 + j];
    }
    __device__ uint32_t next() { return xorwow_next(s); }
    static constexpr int N = 5;
    // the part that jumps as a GF(2) vector, and the Weyl counter's part of k steps
    // (rocrand_xorwow.h:134-145; a subsequence of 2^67 steps leaves the counter)
    __host__ __device__ uint32_t* bits() { return s.x; }
    __host__ __device__ void      count(uint64_t k) { s.d += (uint32_t)k * 362437u; }
    static uint64_t               steps(uint64_t k) { return k; }
    static constexpr int LDS_WORDS = 32 * 5 * 5;
    // the same for a block sharing k (every thread calls it)
    __device__ void advance_block(const device_tables& t, uint64_t k, uint32_t* lds)
    {
        gf2_jump_block<5>(s.x, t.xorwow_jump, k, lds);
        count(k);
    }
};

template<>
struct ieng<inter_kind::lfsr113>
{
    static constexpr word_family F = word_family::w32;
    lfsr113_state                s;
    __device__ void load(const uint32_t* st, uint32_t e, uint32_t ns = S)
    {
#pragma unroll
        for(int j = 0; j < 4; j++)
            s.z[j] = st[j * ns + e];
    }
    __device__ void store(uint32_t* st, uint32_t e, uint32_t ns = S) const
    {
#pragma unroll
        for(int j = 0; j < 4; j++)
            st[j * ns + e] = s.z[j];
    }
    __host__ __device__ void set(const uint32_t* w)
    {
        for(int j = 0; j < 4; j++)
            s.z[j] = w[j];
    }
    __device__ uint32_t next() { return lfsr113_next(s); }
    static constexpr int N = 4;
    __host__ __device__ uint32_t* bits() { return s.z; }
    __host__ __device__ void      count(uint64_t) {}
    // lfsr113.hpp:45-62: the step count travels as an unsigned int
    static uint64_t steps(uint64_t k) { return (uint32_t)k; }
    static constexpr int LDS_WORDS = 32 * 4 * 4;
    __device__ void advance_block(const device_tables& t, uint64_t k, uint32_t* lds)
    {
        gf2_jump_block<4>(s.z, t.lfsr_jump, k, lds);
    }
};


// Non-temporal store of BYTES at base + off through a raw buffer resource built from a
// wavefront-uniform base: the address arithmetic stays in scalar registers (a global
// store with a per-lane 64-bit pointer costs two VALU additions a step).  `limit` bounds
// the byte offsets (the hardware drops a store at or beyond it).
template<int BYTES>
__device__ __forceinline__ void store_uniform_base(char* base, uint32_t off, uint32_t limit, const void* src)
{
    // dword 3 of a gfx9 buffer resource: 32-bit data format, raw (stride 0) addressing
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(base, 0, (int)limit, 0x00020000);
    constexpr int NT = 2; // cache-policy bit 1: nt on gfx950
    using v2 = unsigned int __attribute__((ext_vector_type(2)));
    using v4 = unsigned int __attribute__((ext_vector_type(4)));
    if constexpr(BYTES == 4)
        __builtin_amdgcn_raw_buffer_store_b32(*reinterpret_cast<const uint32_t*>(src), r, (int)off, 0, NT);
    else if constexpr(BYTES == 8)
        __builtin_amdgcn_raw_buffer_store_b64(*reinterpret_cast<const v2*>(src), r, (int)off, 0, NT);
    else
        __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const v4*>(src), r, (int)off, 0, NT);
}

} // namespace inter_dev
} // namespace rr
