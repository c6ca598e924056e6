// rr_mt19937.hip -- MT19937 (8192 generators, 2^1000 words apart) on gfx950.
//
// Streams (library/src/rng/mt19937.hpp, mt19937_octo_engine.hpp):
//   * generator g starts from init_genrand((seed >> 32) ^ seed) jumped by g * 2^1000 words,
//     as two radix-256 digits, with the polynomials x^(i*2^1000) and x^(256*i*2^1000)
//     mod phi (jump kernel :86-274);
//   * before each round every generator twists its 624 words (gen_next_n :259-405); input
//     number q of a round (q < 65536 * (78 / in_w)) comes from thread t = q mod 65536
//     (generator t / 8, lane t mod 8), local words (q / 65536) * in_w + i, where lane l's
//     local word 0 is element {0,113,170,283,340,397,510,567}[l] and local word 1 + 7a + b
//     is element {1,57,114,171,227,284,341,398,454,511,568}[a] + 7l + b (:84-166);
//   * a call consumes vec_n inputs (+1 when there is a head or a tail) from the running
//     position; the extra input fills the head (data[o] = out[o]) and, in reverse, the
//     tail (data[n - 1 - k] = out[out_w - tail + k]) (:355-431, :604-629).
//
// Kernels (own schedule; only the map above is fixed):
//   * jump: the 8192 polynomial products as one Hankel-matrix product over GF(2) with a
//     three-way split (mt_node_kernel), in two stages: 32 high-digit jumps of the seeded
//     state, then 256 low-digit jumps of each.
//   * generate: one block per 8 generators keeps their 8 x 624 words in LDS (element-major)
//     for the whole call, in two buffers: a round twists the current words into the other
//     buffer, each thread following chains of words 227 apart (a word's new value needs
//     the new value 227 words before it, kept in a register), one barrier per round;
//     each wavefront then writes 64 consecutive inputs (8 generators x 8 lanes) per local
//     word while the next round's twist may already write the first buffer.
#include "rr_generator.hpp"

#include <rocrand.h>

#include <algorithm>
#include <mutex>
#include <vector>

extern "C" const unsigned char rr_mt19937_jumps_begin[];
extern "C" const unsigned char rr_mt19937_jumps_end[];

namespace rr
{
namespace
{

constexpr unsigned MT_N      = 624;
constexpr unsigned MT_M      = 397;
constexpr unsigned MT_GENS   = 8192; // config_defaults.hpp:76-80: 256 x 256 threads / 8
constexpr unsigned MT_STRIDE = 65536;
constexpr unsigned MT_LOCAL  = MT_N / 8; // 78 words per lane
constexpr unsigned GPB       = 8;        // generators per generate block

__device__ __forceinline__ uint32_t mt_comp(uint32_t a, uint32_t b, uint32_t m)
{
    const uint32_t y = (a & 0x80000000u) | (b & 0x7fffffffu);
    return m ^ (y >> 1) ^ ((0u - (y & 1u)) & 0x9908b0dfu);
}

__device__ __forceinline__ uint32_t mt_temper(uint32_t y)
{
    y ^= y >> 11;
    y ^= (y << 7) & 0x9d2c5680u;
    y ^= (y << 15) & 0xefc60000u;
    y ^= y >> 18;
    return y;
}

// ---------------------------------------------------------------- jump
// Generator g's words are T[i] = XOR_{j: p_j = 1} S[i + j], i < 624, for a jump polynomial
// p (19937 coefficients) and the sequence S that continues its source state: a Hankel
// matrix times a bit vector.  8192 of these products, each of 19937 x 624 word operations
// done directly, are 102 G operations (2.6 ms of the card's vector ALUs), so the matrix is
// cut into JKB blocks of JB x JB and each block is multiplied by the three-product split of
// a Hankel matrix [[H0, H1], [H1, H2]] (p0, p1):
//     P0 = (H0 + H1) p0,  P1 = H1 (p0 + p1),  P2 = (H1 + H2) p1,  T = (P0 + P1, P1 + P2),
// seven levels deep (640 = 128 * 5): 2187 products of 5 x 5 instead of 16384, with the
// sums over S shared by every polynomial, those over p made once per device
// (mt_poly_kernel) and those over T once after all blocks.  "+" is XOR throughout, so the
// words are those of the direct sum.  A level less (10 x 10) has a fifth more operations; a
// level more would save little over its bit extractions (one per five word operations here)
// and its accumulators would not fit the registers.
constexpr unsigned JB   = 640;           // words and coefficients of a block
constexpr unsigned JKB  = 32;            // blocks of coefficients (20480 >= 19937)
constexpr unsigned JSEQ = JB * JKB + JB; // words of S that the products read (21119 of them)
constexpr unsigned JNODE = 81;           // nodes after four levels, JW output words each
constexpr unsigned JW   = 40;
constexpr unsigned LO = 256, HI = MT_GENS / 256; // generator = 256 * hi + lo
constexpr unsigned HI_LANES = 64;                // HI rounded up to a wavefront
constexpr unsigned JSRC = 9;     // source states per pass of the second stage (see launch_jump)
constexpr unsigned JPARTS = 8;   // parts of the coefficients in the first stage

// Digit l (0 = top level) of a node: which of the three products it is at that level.
__host__ __device__ constexpr unsigned node_digit(unsigned node, unsigned l)
{
    return l == 0 ? node / 27 : l == 1 ? node / 9 % 3 : l == 2 ? node / 3 % 3 : node % 3;
}

// Word k of a product's S: L levels of half sizes h, h/2, ... with digits d[], from the
// block's words.  Digit 0 takes s[k] ^ s[k + h], 1 takes s[k + h], 2 s[k + h] ^ s[k + 2h].
template<unsigned L>
__device__ __forceinline__ uint32_t node_word(const uint32_t* s, unsigned h, const unsigned (&d)[L])
{
    // base offset and the levels that add a second term
    unsigned base = 0, two = 0;
#pragma unroll
    for(unsigned l = 0; l < L; l++)
    {
        base += d[l] != 0 ? h >> l : 0u;
        two |= d[l] != 1 ? 1u << l : 0u;
    }
    // every term is read (none lies outside the block's words) and the ones that do not
    // count are masked: no branch keeps the loads from being in flight together
    uint32_t r = 0;
#pragma unroll
    for(unsigned m = 0; m < 1u << L; m++)
    {
        unsigned o = base;
#pragma unroll
        for(unsigned l = 0; l < L; l++)
            o += (m >> l & 1u) != 0 ? h >> l : 0u;
        r ^= s[o] & (0u - (uint32_t)((m & ~two) == 0u));
    }
    return r;
}

// The coefficients of every polynomial on every node: pt[(node * JKB + kb) * POLYS + poly],
// 40 bits each.  Polynomial 0 is 1 (no jump); `raw` holds polynomials 1, 2, ... (COUNT - 1
// of them), 624 words each, of whose last only bit 0 counts (x^19936).
template<unsigned POLYS, unsigned COUNT>
__global__ __launch_bounds__(POLYS) void mt_poly_kernel(const uint32_t* raw, uint64_t* pt)
{
    const unsigned node = blockIdx.x, kb = blockIdx.y, poly = threadIdx.x;
    uint64_t       r    = 0;
    if(poly < COUNT)
        for(unsigned seg = 0; seg < 16; seg++)
        {
            bool in = true;
            for(unsigned l = 0; l < 4; l++)
            {
                const unsigned d = node_digit(node, l), half = seg >> (3 - l) & 1u;
                in = in && (d == 1 || d == 2 * half);
            }
            if(!in)
                continue;
            // 40 coefficients from bit 40 seg of the block: whole bytes, so two words hold them
            const unsigned bit = 40 * seg, w = kb * (JB / 32) + bit / 32;
            auto           word = [&](unsigned i) -> uint64_t {
                if(poly == 0)
                    return i == 0 ? 1u : 0u;
                if(i >= MT_N)
                    return 0;
                const uint32_t v = raw[(size_t)(poly - 1) * MT_N + i];
                return i == MT_N - 1 ? v & 1u : v;
            };
            r ^= (word(w) | word(w + 1) << 32) >> (bit % 32);
        }
    pt[((size_t)node * JKB + kb) * POLYS + poly] = r & ((1ull << JW) - 1);
}

struct mt_words
{
    uint32_t w[MT_N];
};

// S of one source state per block: JSEQ words, one twist per round through LDS (chains of
// words 227 apart, as twist_block below).
__device__ __forceinline__ void extend(uint32_t (*buf)[MT_N], uint32_t* seq, unsigned t)
{
    for(unsigned r = 1; r * MT_N < JSEQ; r++)
    {
        const uint32_t* src = buf[(r - 1) & 1u];
        uint32_t*       dst = buf[r & 1u];
        auto            put = [&](unsigned k, uint32_t v) {
            dst[k] = v;
            if(r * MT_N + k < JSEQ)
                seq[r * MT_N + k] = v;
        };
        if(t < 227)
        {
            const uint32_t a = mt_comp(src[t], src[t + 1], src[t + MT_M]);
            const uint32_t b = mt_comp(src[t + 227], src[t + 228], a);
            put(t, a);
            put(t + 227, b);
            if(t + 454 < MT_N)
            {
                const uint32_t nx = t + 455 < MT_N ? src[t + 455] : mt_comp(src[0], src[1], src[MT_M]);
                put(t + 454, mt_comp(src[t + 454], nx, b));
            }
        }
        __syncthreads();
    }
}
__global__ __launch_bounds__(256) void mt_seed_seq_kernel(mt_words seed, uint32_t* seq)
{
    __shared__ uint32_t buf[2][MT_N];
    for(unsigned i = threadIdx.x; i < MT_N; i += 256)
        seq[i] = buf[0][i] = seed.w[i];
    __syncthreads();
    extend(buf, seq, threadIdx.x);
}
__global__ __launch_bounds__(256) void mt_seq_kernel(const uint32_t* states, uint32_t* seq)
{
    __shared__ uint32_t buf[2][MT_N];
    seq += (size_t)blockIdx.x * JSEQ;
    for(unsigned i = threadIdx.x; i < MT_N; i += 256)
        seq[i] = buf[0][i] = states[(size_t)blockIdx.x * MT_N + i];
    __syncthreads();
    extend(buf, seq, threadIdx.x);
}

// One level of sums over T: N nodes' three products of W words each, to N nodes of 2 W.
template<unsigned N, unsigned W>
__device__ __forceinline__ void fold_level(const uint32_t (&p)[3 * N][W], uint32_t (&t)[N][2 * W])
{
#pragma unroll
    for(unsigned n = 0; n < N; n++)
#pragma unroll
        for(unsigned i = 0; i < W; i++)
        {
            t[n][i]     = p[3 * n][i] ^ p[3 * n + 1][i];
            t[n][W + i] = p[3 * n + 1][i] ^ p[3 * n + 2][i];
        }
}

// One node (its last three levels: 27 products of 5 x 5) of KB blocks for one source and
// POLYS polynomials, one polynomial per lane: 135 accumulators a lane, and per coefficient
// one bit extraction and five v_bitop3 (acc ^ (word & bit)) on words that the whole
// wavefront shares, read from LDS as broadcasts (3 LDS reads per 30 VALU instructions).
// VALU-bound (164 us per pass of 729 blocks).  tt[((src * parts + part) * JNODE + node) * 10 + i / 4][poly][i % 4] is word
// i of the node's 40.
template<unsigned KB, unsigned POLYS>
__global__ __launch_bounds__(POLYS) __attribute__((amdgpu_waves_per_eu(3))) void mt_node_kernel(const uint32_t* seq,
                                                                                                const uint64_t* pt,
                                                                                                uint4*          tt)
{
    constexpr unsigned  NW = 2 * JW - 1; // words of a node's S
    constexpr unsigned  F = 27, W = 5, LW = 2 * W - 1, LS = 12; // products, their size, words of S, padded row
    __shared__ uint32_t nw[KB * NW];
    __shared__ uint4    leaf4[KB * F * LS / 4];
    uint32_t* const     leaf = reinterpret_cast<uint32_t*>(leaf4);
    const unsigned      t = threadIdx.x, node = blockIdx.x, part = blockIdx.z;
    const uint32_t*     S = seq + (size_t)blockIdx.y * JSEQ + part * KB * JB;
    const unsigned      d[4]
        = {node_digit(node, 0), node_digit(node, 1), node_digit(node, 2), node_digit(node, 3)};
    for(unsigned i = t; i < KB * NW; i += POLYS)
        nw[i] = node_word<4>(S + i / NW * JB + i % NW, JB / 2, d);
    __syncthreads();
    for(unsigned i = t; i < KB * F * LW; i += POLYS)
    {
        const unsigned row = i / LW, k = i % LW, kb = row / F, f = row % F;
        const unsigned e[3] = {f / 9, f / 3 % 3, f % 3};
        leaf[row * LS + k]  = node_word<3>(nw + kb * NW + k, 4 * W, e);
    }
    __syncthreads();

    uint32_t acc[F][W];
#pragma unroll
    for(unsigned f = 0; f < F; f++)
#pragma unroll
        for(unsigned i = 0; i < W; i++)
            acc[f][i] = 0;
    const uint64_t* p = pt + ((size_t)node * JKB + part * KB) * POLYS + t;
#pragma unroll 1
    for(unsigned kb = 0; kb < KB; kb++, p += POLYS)
    {
        const uint64_t bits = *p;
        const uint32_t x0 = (uint32_t)bits, x2 = (uint32_t)(bits >> 20);
        const uint32_t x[3] = {x0, x0 ^ x2, x2};
#pragma unroll
        for(unsigned f = 0; f < F; f++)
        {
            // the product's five coefficients, from bit `at`: the halves of a level are 10,
            // then 5 bits apart, digit 1 takes their sum
            const unsigned d5 = f / 3 % 3, d6 = f % 3;
            const uint32_t y  = d5 == 1 ? x[f / 9] ^ x[f / 9] >> 10 : x[f / 9];
            const uint32_t c  = d6 == 1 ? y ^ y >> 5 : y;
            const unsigned at = (d5 == 2 ? 10 : 0) + (d6 == 2 ? 5 : 0);
            uint32_t       w[LS];
#pragma unroll
            for(unsigned q = 0; q < LS / 4; q++)
            {
                const uint4 v = leaf4[(kb * F + f) * (LS / 4) + q];
                w[4 * q] = v.x, w[4 * q + 1] = v.y, w[4 * q + 2] = v.z, w[4 * q + 3] = v.w;
            }
#pragma unroll
            for(unsigned j = 0; j < W; j++)
            {
                const uint32_t m = (uint32_t)__builtin_amdgcn_sbfe((int)c, at + j, 1);
#pragma unroll
                for(unsigned i = 0; i < W; i++)
                    acc[f][i] = __builtin_amdgcn_bitop3_b32(acc[f][i], w[i + j], m, 0x78); // a ^ (b & c)
            }
        }
    }
    uint32_t t10[F / 3][2 * W], t20[F / 9][4 * W], o[1][8 * W];
    fold_level<F / 3, W>(acc, t10);
    fold_level<F / 9, 2 * W>(t10, t20);
    fold_level<1, 4 * W>(t20, o);
    uint4* dst = tt + (((size_t)blockIdx.y * gridDim.z + part) * JNODE + node) * (JW / 4) * POLYS + t;
#pragma unroll
    for(unsigned q = 0; q < JW / 4; q++)
        dst[q * POLYS] = make_uint4(o[0][4 * q], o[0][4 * q + 1], o[0][4 * q + 2], o[0][4 * q + 3]);
}

// The first four levels' sums over T: thread (poly, c) of block (q, src) gathers word
// 4 q + c of every node into the 16 words of T that it is part of (40 apart), and writes
// them to the state of generator src * COUNT + poly.  With PARTS > 1 the threads of a part
// gather that part, and the parts' words are summed through LDS (one thread after all
// parts, 648 loads in a row, took 41 us).
template<unsigned PARTS, unsigned POLYS, unsigned COUNT>
__global__ __launch_bounds__(64 * (PARTS > 4 ? PARTS : 4)) void mt_fold_kernel(const uint32_t* tt, uint32_t* states)
{
    constexpr unsigned IDS = PARTS > 1 ? 64 : 256; // (poly, c) pairs of a block
    const unsigned     part = threadIdx.x / IDS, local = threadIdx.x % IDS;
    const unsigned     id = blockIdx.z * IDS + local, poly = id / 4, q = blockIdx.x, src = blockIdx.y;
    uint32_t           r[16] = {};
    const uint32_t*    p = tt + ((((size_t)src * PARTS + part) * JNODE) * (JW / 4) + q) * POLYS * 4 + id;
#pragma unroll
    for(unsigned node = 0; node < JNODE; node++)
    {
        const uint32_t v = p[(size_t)node * JW * POLYS];
#pragma unroll
        for(unsigned seg = 0; seg < 16; seg++)
        {
            bool in = true; // digit 0 is in the first half of its level, 2 in the second, 1 in both
            for(unsigned l = 0; l < 4; l++)
            {
                const unsigned d = node_digit(node, l), half = seg >> (3 - l) & 1u;
                in = in && (d == 1 || d == 2 * half);
            }
            if(in)
                r[seg] ^= v;
        }
    }
    if constexpr(PARTS > 1)
    {
        __shared__ uint32_t sum[PARTS][16][IDS];
#pragma unroll
        for(unsigned seg = 0; seg < 16; seg++)
            sum[part][seg][local] = r[seg];
        __syncthreads();
        if(part != 0)
            return;
        for(unsigned o = 1; o < PARTS; o++)
#pragma unroll
            for(unsigned seg = 0; seg < 16; seg++)
                r[seg] ^= sum[o][seg][local];
    }
    if(poly >= COUNT)
        return;
    uint32_t* out = states + ((size_t)src * COUNT + poly) * MT_N;
#pragma unroll
    for(unsigned seg = 0; seg < 16; seg++)
    {
        const unsigned i = seg * JW + 4 * q + id % 4;
        if(i < MT_N)
            out[i] = r[seg];
    }
}

struct mt_call
{
    uint32_t*   states; // [MT_GENS][MT_N], words of the current round
    void*       data;
    size_t      n, mis, vec_n;
    uint32_t    head, tail, extra;
    uint32_t    start; // running input position within the current round (0: used up)
    dist_params params;
};

// State element read by lane `lane` as its local word `local` (mt19937_octo_engine.hpp:84-166).
__constant__ unsigned mt_special[8]  = {0, 113, 170, 283, 340, 397, 510, 567};
__constant__ unsigned mt_offsets[11] = {1, 57, 114, 171, 227, 284, 341, 398, 454, 511, 568};

// `local` is wavefront-uniform in the generate kernel (scalar division and table load);
// `special` = mt_special[lane], loaded once per thread.
__device__ __forceinline__ unsigned mt_element(unsigned lane, unsigned special, unsigned local)
{
    if(local == 0)
        return special;
    const unsigned a = (local - 1) / 7, b = (local - 1) - 7 * a;
    return mt_offsets[a] + 7 * lane + b;
}

// LDS layout of the block's generators: element-major, word k of generator g at
// st[k * GPB + g].  A wavefront's output reads (8 generators x 8 lanes, lanes 7 words
// apart) then fall on 64 distinct banks, and the twist's reads are consecutive.
__device__ __forceinline__ unsigned lds_at(unsigned k, unsigned g) { return k * GPB + g; }

// One round of the recurrence on GPB generators: the round's words in `src`, the next
// round's written to `dst` (both element-major, so item it = 8k + g is word k of
// generator g).  Word k of the new round is x'[k] = f(x[k], x[k + 1], m) with
// m = x[k + 397] for k < 227 and m = x'[k - 227] above, and x[624] read as x'[0].
// A thread takes whole chains k0, k0 + 227, k0 + 454 (k0 < 227) of one generator: each
// link's m is the previous link's result, kept in a register, and every other operand
// is an old word, so no thread waits for another's writes; the one exception, x'[0] for
// k = 623, the thread of chain 169 computes itself from old words.  Nothing in `src`
// is written, so a single barrier -- the new words visible to the output reads -- ends
// the round; `src` is next written by the following round's twist, after every thread
// has passed this barrier and so finished its reads of it.
__device__ __forceinline__ void twist_block(const uint32_t* src, uint32_t* dst, unsigned t)
{
    constexpr unsigned W = GPB * MT_N, D = GPB * 227, J = GPB * MT_M;
    for(unsigned it = t; it < D; it += 256)
    {
        const uint32_t a = mt_comp(src[it], src[it + GPB], src[it + J]);
        dst[it]          = a;
        const uint32_t b = mt_comp(src[it + D], src[it + D + GPB], a);
        dst[it + D]      = b;
        const unsigned k3 = it + 2 * D;
        if(k3 < W)
        {
            uint32_t nx;
            if(k3 + GPB < W)
                nx = src[k3 + GPB];
            else
            {
                const unsigned g0 = k3 + GPB - W; // word 0 of this generator
                nx                = mt_comp(src[g0], src[g0 + GPB], src[g0 + J]);
            }
            dst[k3] = mt_comp(src[k3], nx, b);
        }
    }
    __syncthreads();
}

// 4 blocks per CU (the LDS of 2 x 8 generators each fills it): at most 128 VGPRs
template<class D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void mt_generate_kernel(mt_call c)
{
    using out_t          = typename D::out_t;
    constexpr int IN     = D::in_w;
    constexpr int OUT    = D::out_w;
    constexpr int BYTES  = OUT * (int)sizeof(out_t);
    constexpr unsigned IPS  = MT_LOCAL / IN;
    constexpr uint64_t FULL = (uint64_t)MT_STRIDE * IPS;
    static_assert(BYTES == 4 || BYTES == 8 || BYTES == 16, "vec size");

    // the round's words and the next round's (twist_block), 2 x 39 KiB: 4 blocks per CU
    __shared__ uint32_t buf[2][GPB * MT_N];
    const unsigned t = threadIdx.x, blk = blockIdx.x;
    uint32_t*      gstate = c.states + (size_t)blk * GPB * MT_N;
    uint32_t*      st     = buf[0];
    uint32_t*      nx     = buf[1];
    for(unsigned i = t; i < GPB * MT_N; i += 256)
        st[lds_at(i % MT_N, i / MT_N)] = gstate[i];
    __syncthreads();

    // the wavefront index as a scalar: the local word j, its element offsets and the
    // wavefront's input range below are then uniform (scalar loads and branches)
    const unsigned p = t & 63u, quarter = __builtin_amdgcn_readfirstlane(t >> 6);
    const unsigned gl = p >> 3, lane = p & 7u;
    const uint64_t total = c.vec_n + c.extra;
    const uint64_t qend  = (uint64_t)c.start + total;
    out_t* const   data  = static_cast<out_t*>(c.data);
    out_t* const   vec_data = data + c.mis;
    const unsigned special = mt_special[lane];
    alignas(16) out_t o[OUT];
    uint32_t     in[IN];
    // the transforms' tables stay in constant memory: copies in LDS would leave room for
    // three blocks per CU
    const kernel_params kp{c.params, {}};

    // LDS indices of this thread's inputs, the same every round: local word
    // j = quarter + 4m (m < MW) reads eoff[m][i] for input i (held in registers: every
    // loop over m below is unrolled)
    constexpr unsigned MW = (IPS + 3) / 4;
    unsigned           eoff[MW][IN];
#pragma unroll
    for(unsigned m = 0; m < MW; m++)
#pragma unroll
        for(int i = 0; i < IN; i++)
        {
            const unsigned j = quarter + 4 * m;
            eoff[m][i]       = j < IPS ? lds_at(mt_element(lane, special, j * IN + i), gl) : 0;
        }

    for(uint64_t R = 0; R * FULL < qend; R++)
    {
        if(R > 0 || c.start == 0)
        {
            twist_block(st, nx, t);
            uint32_t* const w = st;
            st                = nx;
            nx                = w;
        }
        const uint64_t R0 = R * FULL;
        if(R0 >= c.start && R0 + FULL <= c.start + c.vec_n)
        {
            // every input of the round is a whole vec: no range checks.  Lane p is the
            // reference's thread blk * 64 + p; its local word j is input
            // R0 + j * 65536 + blk * 64 + p.
            // Up to 8-byte vecs all of the thread's words are read first (an invalid last j
            // reads word 0 and is not stored), so the LDS reads overlap one another; the
            // double-pair transforms need those registers themselves.
            constexpr bool BATCH = BYTES <= 8;
            out_t* const   rbase = vec_data + (R0 - c.start + blk * 64u + p) * OUT;
            uint32_t       w[BATCH ? MW : 1][IN];
            if constexpr(BATCH)
            {
#pragma unroll
                for(unsigned m = 0; m < MW; m++)
#pragma unroll
                    for(int i = 0; i < IN; i++)
                        w[m][i] = st[eoff[m][i]];
            }
#pragma unroll
            for(unsigned m = 0; m < MW; m++)
            {
                const unsigned j = quarter + 4 * m;
                if(j < IPS)
                {
#pragma unroll
                    for(int i = 0; i < IN; i++)
                        in[i] = mt_temper(BATCH ? w[BATCH ? m : 0][i] : st[eoff[m][i]]);
                    D::apply(in, o, kp);
                    out_t* dst = rbase + (size_t)j * MT_STRIDE * OUT;
                    if constexpr(BYTES == 4)
                        *reinterpret_cast<uint32_t*>(dst) = *reinterpret_cast<const uint32_t*>(o);
                    else if constexpr(BYTES == 8)
                        *reinterpret_cast<uint2*>(dst) = *reinterpret_cast<const uint2*>(o);
                    else
                        *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(o);
                }
            }
            continue;
        }
        for(unsigned j = quarter; j < IPS; j += 4)
        {
            const uint64_t Q = R0 + (uint64_t)j * MT_STRIDE + blk * 64u + p;
            if(Q < c.start || Q >= qend)
                continue;
            const uint64_t v = Q - c.start;
#pragma unroll
            for(int i = 0; i < IN; i++)
                in[i] = mt_temper(st[lds_at(mt_element(lane, special, j * IN + i), gl)]);
            D::apply(in, o, kp);
            if(v < c.vec_n)
            {
                out_t* dst = vec_data + v * OUT;
                if constexpr(BYTES == 4)
                    *reinterpret_cast<uint32_t*>(dst) = *reinterpret_cast<const uint32_t*>(o);
                else if constexpr(BYTES == 8)
                    *reinterpret_cast<uint2*>(dst) = *reinterpret_cast<const uint2*>(o);
                else
                    *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(o);
            }
            else
            {
                for(uint32_t k = 0; k < (uint32_t)OUT; k++)
                {
                    if(k < c.head)
                        data[k] = o[k];
                    if(k + c.tail >= (uint32_t)OUT)
                        data[c.n + (OUT - c.tail - 1) - k] = o[k];
                }
            }
        }
        // no barrier: the next round twists into the buffer these reads do not touch
    }
    for(unsigned i = t; i < GPB * MT_N; i += 256)
        gstate[i] = st[lds_at(i % MT_N, i / MT_N)];
}

template<class D>
hipError_t launch_gen(const mt_call& c, hipStream_t s)
{
    hipLaunchKernelGGL((mt_generate_kernel<D>), dim3(MT_GENS / GPB), dim3(256), 0, s, c);
    return hipGetLastError();
}

hipError_t dispatch(out_kind o, const mt_call& c, hipStream_t s)
{
    constexpr word_family F = word_family::w32;
    switch(o)
    {
        case out_kind::u8: return launch_gen<dist<F, out_kind::u8>>(c, s);
        case out_kind::u16: return launch_gen<dist<F, out_kind::u16>>(c, s);
        case out_kind::u32: return launch_gen<dist<F, out_kind::u32>>(c, s);
        case out_kind::uniform_f32: return launch_gen<dist<F, out_kind::uniform_f32>>(c, s);
        case out_kind::uniform_f64: return launch_gen<dist<F, out_kind::uniform_f64>>(c, s);
        case out_kind::uniform_f16: return launch_gen<dist<F, out_kind::uniform_f16>>(c, s);
        case out_kind::normal_f32: return launch_gen<dist<F, out_kind::normal_f32>>(c, s);
        case out_kind::normal_f64: return launch_gen<dist<F, out_kind::normal_f64>>(c, s);
        case out_kind::normal_f16: return launch_gen<dist<F, out_kind::normal_f16>>(c, s);
        case out_kind::lognormal_f32: return launch_gen<dist<F, out_kind::lognormal_f32>>(c, s);
        case out_kind::lognormal_f64: return launch_gen<dist<F, out_kind::lognormal_f64>>(c, s);
        case out_kind::lognormal_f16: return launch_gen<dist<F, out_kind::lognormal_f16>>(c, s);
        case out_kind::poisson: return launch_gen<dist<F, out_kind::poisson>>(c, s);
        case out_kind::u64: return hipErrorInvalidValue;
    }
    return hipErrorInvalidValue;
}

// The jump polynomials of the current device on every node, made once.
struct jump_polys
{
    const uint64_t* lo; // x^(i 2^1000), i < LO
    const uint64_t* hi; // x^(256 i 2^1000), i < HI
};
hipError_t device_jumps(jump_polys& out)
{
    static std::mutex                             mtx;
    static std::vector<std::pair<int, jump_polys>> copies;
    int                                           dev = 0;
    hipError_t                                    e   = hipGetDevice(&dev);
    if(e != hipSuccess)
        return e;
    std::lock_guard<std::mutex> lock(mtx);
    for(const auto& c : copies)
        if(c.first == dev)
        {
            out = c.second;
            return hipSuccess;
        }
    // the file holds x^(i 2^1000) and x^(256 i 2^1000) for i = 1 .. 255
    const size_t bytes = (size_t)(rr_mt19937_jumps_end - rr_mt19937_jumps_begin);
    if(bytes != (size_t)510 * MT_N * 4)
        return hipErrorInvalidImage;
    copies.reserve(copies.size() + 1);
    constexpr size_t lo_words = (size_t)JNODE * JKB * LO, hi_words = (size_t)JNODE * JKB * HI_LANES;
    uint64_t*        pt  = nullptr;
    uint32_t*        raw = nullptr;
    if((e = hipMalloc(&pt, (lo_words + hi_words) * sizeof(uint64_t))) != hipSuccess)
        return e;
    if((e = hipMalloc(&raw, bytes)) == hipSuccess
       && (e = hipMemcpy(raw, rr_mt19937_jumps_begin, bytes, hipMemcpyHostToDevice)) == hipSuccess)
    {
        hipLaunchKernelGGL((mt_poly_kernel<LO, LO>), dim3(JNODE, JKB), dim3(LO), 0, 0, raw, pt);
        hipLaunchKernelGGL((mt_poly_kernel<HI_LANES, HI>), dim3(JNODE, JKB), dim3(HI_LANES), 0, 0,
                           raw + (size_t)255 * MT_N, pt + lo_words);
        if((e = hipGetLastError()) == hipSuccess)
            e = hipStreamSynchronize(0);
    }
    (void)hipFree(raw);
    if(e != hipSuccess)
    {
        (void)hipFree(pt);
        return e;
    }
    out = jump_polys{pt, pt + lo_words};
    copies.emplace_back(dev, out);
    return hipSuccess;
}

// A generator's scratch for its jump: the sequences of the seed and of the HI source
// states, those states, and one pass's node products (the first stage's fit in there).
constexpr size_t JSCRATCH_SEQ  = (size_t)HI * JSEQ;
constexpr size_t JSCRATCH_SRC  = (size_t)HI * MT_N;
constexpr size_t JSCRATCH_NODE = (size_t)JSRC * JNODE * JW * LO;
static_assert((size_t)JPARTS * JNODE * JW * HI_LANES <= JSCRATCH_NODE, "first stage's products");
static_assert(JKB % JPARTS == 0, "whole blocks per part");

// States of all generators under the seed: HI source states (the high digit's jumps of the
// seeded state), then LO jumps of each.  The second stage goes over the sources in passes
// of JSRC: 81 * 9 = 729 equal blocks are 2.85 per CU, near a whole number, and bound the
// scratch (30 MB of products).  0.68 ms a seed (both sequences 27 us, the first stage 26,
// a pass's products 164 at 0.8 of the vector ALUs' rate, its sums 10), against 15.2 ms of
// one block per generator that applied each polynomial by Horner's rule, 32 coefficients a
// step; with 10 x 10 products 0.77 ms.
hipError_t launch_jump(uint32_t* states, uint32_t* scratch, uint32_t seed, const jump_polys& polys, hipStream_t s)
{
    mt_words init;
    init.w[0] = seed;
    for(unsigned i = 1; i < MT_N; i++)
        init.w[i] = 1812433253u * (init.w[i - 1] ^ (init.w[i - 1] >> 30)) + i;
    uint32_t* const seq   = scratch;
    uint32_t* const src   = seq + JSCRATCH_SEQ;
    uint4* const    nodes = reinterpret_cast<uint4*>(src + JSCRATCH_SRC);
    hipLaunchKernelGGL(mt_seed_seq_kernel, dim3(1), dim3(256), 0, s, init, seq);
    hipLaunchKernelGGL((mt_node_kernel<JKB / JPARTS, HI_LANES>), dim3(JNODE, 1, JPARTS), dim3(HI_LANES), 0, s, seq,
                       polys.hi, nodes);
    hipLaunchKernelGGL((mt_fold_kernel<JPARTS, HI_LANES, HI>), dim3(JW / 4, 1, HI_LANES * 4 / 64),
                       dim3(64 * JPARTS), 0, s, reinterpret_cast<const uint32_t*>(nodes), src);
    hipLaunchKernelGGL(mt_seq_kernel, dim3(HI), dim3(256), 0, s, src, seq);
    for(unsigned h = 0; h < HI; h += JSRC)
    {
        const unsigned count = std::min(JSRC, HI - h);
        hipLaunchKernelGGL((mt_node_kernel<JKB, LO>), dim3(JNODE, count, 1), dim3(LO), 0, s, seq + (size_t)h * JSEQ,
                           polys.lo, nodes);
        hipLaunchKernelGGL((mt_fold_kernel<1, LO, LO>), dim3(JW / 4, count, LO * 4 / 256), dim3(256), 0, s,
                           reinterpret_cast<const uint32_t*>(nodes), states + (size_t)h * LO * MT_N);
    }
    return hipGetLastError();
}

template<word_family F, out_kind K>
constexpr dist_shape mt_shape()
{
    return dist_shape{dist<F, K>::in_w, dist<F, K>::out_w, (int)sizeof(typename dist<F, K>::out_t)};
}

// mt19937.hpp:665-1122
class mt19937_generator final : public rocrand_generator_base_type
{
public:
    mt19937_generator() : rocrand_generator_base_type(ROCRAND_RNG_PSEUDO_MT19937) {}
    ~mt19937_generator() override
    {
        if(m_states)
            (void)hipFree(m_states);
    }

    void set_seed(unsigned long long seed) override
    {
        m_seed = seed;
        reset();
    }

    rocrand_status set_offset(unsigned long long) override { return ROCRAND_STATUS_TYPE_ERROR; }

    rocrand_status set_order(rocrand_ordering o) override
    {
        // mt19937.hpp:765-779: DEFAULT, BEST and LEGACY only
        if(o != ROCRAND_ORDERING_PSEUDO_DEFAULT && o != ROCRAND_ORDERING_PSEUDO_BEST
           && o != ROCRAND_ORDERING_PSEUDO_LEGACY)
            return ROCRAND_STATUS_OUT_OF_RANGE;
        order = o;
        reset();
        return ROCRAND_STATUS_SUCCESS;
    }

    rocrand_status init() override
    {
        if(m_initialized)
            return ROCRAND_STATUS_SUCCESS;
        // states, then the jump's scratch: both stay for the next seed (a call under stream
        // capture allocates nothing)
        constexpr size_t state_words = (size_t)MT_GENS * MT_N;
        constexpr size_t all_words   = state_words + JSCRATCH_SEQ + JSCRATCH_SRC + JSCRATCH_NODE;
        if(!m_states && hipMalloc(&m_states, sizeof(uint32_t) * all_words) != hipSuccess)
        {
            m_states = nullptr;
            return ROCRAND_STATUS_ALLOCATION_FAILED;
        }
        jump_polys polys;
        if(device_jumps(polys) != hipSuccess)
            return ROCRAND_STATUS_ALLOCATION_FAILED;
        uint32_t* const states = static_cast<uint32_t*>(m_states);
        if(launch_jump(states, states + state_words, (uint32_t)((m_seed >> 32) ^ m_seed), polys, stream) != hipSuccess)
            return ROCRAND_STATUS_LAUNCH_FAILURE;
        m_start       = 0;
        m_prev_in_w   = 0;
        m_initialized = true;
        return ROCRAND_STATUS_SUCCESS;
    }

    rocrand_status shape(out_kind k, dist_shape& s) const override
    {
        constexpr word_family F = word_family::w32;
        switch(k)
        {
            case out_kind::u8: s = mt_shape<F, out_kind::u8>(); break;
            case out_kind::u16: s = mt_shape<F, out_kind::u16>(); break;
            case out_kind::u32: s = mt_shape<F, out_kind::u32>(); break;
            case out_kind::uniform_f32: s = mt_shape<F, out_kind::uniform_f32>(); break;
            case out_kind::uniform_f64: s = mt_shape<F, out_kind::uniform_f64>(); break;
            case out_kind::uniform_f16: s = mt_shape<F, out_kind::uniform_f16>(); break;
            case out_kind::normal_f32: s = mt_shape<F, out_kind::normal_f32>(); break;
            case out_kind::normal_f64: s = mt_shape<F, out_kind::normal_f64>(); break;
            case out_kind::normal_f16: s = mt_shape<F, out_kind::normal_f16>(); break;
            case out_kind::lognormal_f32: s = mt_shape<F, out_kind::lognormal_f32>(); break;
            case out_kind::lognormal_f64: s = mt_shape<F, out_kind::lognormal_f64>(); break;
            case out_kind::lognormal_f16: s = mt_shape<F, out_kind::lognormal_f16>(); break;
            case out_kind::poisson: s = mt_shape<F, out_kind::poisson>(); break;
            default: return ROCRAND_STATUS_TYPE_ERROR;
        }
        return ROCRAND_STATUS_SUCCESS;
    }

protected:
    void reset() override { m_initialized = false; }

    rocrand_status generate_device(out_kind k, void* data, size_t n, const gen_args& args) override
    {
        dist_shape     s;
        rocrand_status st = shape(k, s);
        if(st != ROCRAND_STATUS_SUCCESS)
            return st;
        mt_call c{};
        if((st = make_params(k, args, c.params)) != ROCRAND_STATUS_SUCCESS)
            return st;
        if((st = init()) != ROCRAND_STATUS_SUCCESS)
            return st;
        if(data == nullptr)
            return ROCRAND_STATUS_SUCCESS;
        const unsigned in_w = (unsigned)s.in_w, out_w = (unsigned)s.out_w;
        const unsigned full = MT_STRIDE * (MT_LOCAL / in_w);
        const uintptr_t addr = reinterpret_cast<uintptr_t>(data);
        c.mis   = (out_w - (addr / s.esz) % out_w) % out_w;
        c.head  = (uint32_t)std::min<size_t>(n, c.mis);
        c.tail  = (uint32_t)((n - c.head) % out_w);
        c.vec_n = (n - c.head) / out_w;
        c.extra = (c.head > 0 || c.tail > 0) ? 1u : 0u;
        // mt19937.hpp:951-964: a new input width starts at the next whole unused input
        if(m_prev_in_w != in_w && m_start > 0)
        {
            const unsigned used = (m_start + MT_STRIDE - 1) / MT_STRIDE * m_prev_in_w;
            m_start             = (used + in_w - 1) / in_w * MT_STRIDE;
            if(m_start >= full)
                m_start = 0;
        }
        c.states = static_cast<uint32_t*>(m_states);
        c.data   = data;
        c.n      = n;
        c.start  = m_start;
        if(dispatch(k, c, stream) != hipSuccess)
            return ROCRAND_STATUS_LAUNCH_FAILURE;
        m_start     = (uint32_t)(((uint64_t)m_start + c.vec_n + c.extra) % full);
        m_prev_in_w = in_w;
        return ROCRAND_STATUS_SUCCESS;
    }

private:
    unsigned long long m_seed        = 0;
    bool               m_initialized = false;
    void*              m_states      = nullptr;
    uint32_t           m_start       = 0;
    uint32_t           m_prev_in_w   = 0;
};

} // namespace

rocrand_generator make_mt19937_generator() { return new mt19937_generator(); }

} // namespace rr
