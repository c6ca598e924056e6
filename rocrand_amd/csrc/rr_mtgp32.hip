// rr_mtgp32.hip -- MTGP32 (Mersenne exponent 11213, 512 parameter sets) on gfx950.
//
// Output map (library/src/rng/mtgp32.hpp:232-305): generator b (one 256-thread block)
// advances its 351-word recurrence 256 words per block-step; thread t's word of a
// step feeds vec index b*256 + t + j*(512*256) on the block's j-th use, taking
// in_w consecutive steps per vec.  The head and tail of a misaligned or ragged
// call come from one extra use, by the threads whose index equals vec_n_up and
// vec_n_up + 1.  State per generator (rocrand_mtgp32.h:130-145, 272-317): a 1024-word
// ring, the recurrence parameters and the tempering table of its parameter set;
// every generator masks with the first set's mask (rocrand_mtgp32.h:381).
//
// The ring lives in LDS for the whole call, turned so that the call starts at word 0, and four
// block-steps go once around it.  The main loop runs them unrolled, so that every LDS address
// is a register that never changes plus an immediate.  A step reads words w = off + t + {0, 1,
// pos - 1, pos} unmasked (w <= 768 + 255 + 95): words 0 to 94 have a second copy behind the
// ring, written by the one step of four that wraps.  One barrier per block-step suffices: a
// step reads ring[off .. off+350] and writes ring[off+351 .. off+606] (indices mod 1024), so
// reads and writes of one step never alias, and the next step's reads see this step's writes
// after the barrier.
//
// The recurrence table of every parameter set is GF(2)-linear in its 4-bit index
// (tbl[i ^ j] = tbl[i] ^ tbl[j], tbl[0] = 0: MTGP is an F2-linear generator; the host
// checks it for all 512 sets when it builds the states), so its lookup, which sits on
// the step's critical path (ring reads -> new word -> ring write -> barrier), is the XOR
// of the entries at 1, 2, 4 and 8 selected by the index bits: eight VALU operations
// on block-uniform operands instead of a dependent LDS round trip.  The tempering
// table's lookup only feeds the output; it stays an LDS read, issued as soon as the
// ring reads return so that its latency overlaps the recurrence (behind the barrier instead:
// u32 3.00 -> 2.91 TB/s, Poisson 2.31 -> 2.13).
//
// 512 generators are two blocks a CU, and a block-step is as wide as the recurrence allows
// (351 - 95 words), so two wavefronts a SIMD have to hide a step's LDS reads, write and
// barrier.  Integers and uniforms are bound by that chain (170 ns a step), the transforms by
// VALU issue on top of it.  With an 18-instruction step (28 with wrap-around masks and a copy
// of every word): 2^26 values, normal f32 147.6 -> 118.6 us, u32 2.74 -> 3.00 TB/s, uniform
// f64 2.97 -> 3.41, Poisson 1.90 -> 2.31.
#include "rr_generator.hpp"

#include <rocrand.h>

#include <algorithm>
#include <mutex>

extern "C" const unsigned char rr_mtgp32_params_begin[];
extern "C" const unsigned char rr_mtgp32_params_end[];

namespace rr
{
namespace
{

constexpr unsigned MTGP_GENS  = 512; // config_defaults.hpp:45-50: 512 blocks
constexpr unsigned MTGP_BLOCK = 256;
constexpr unsigned MTGP_N     = 351; // 11213 / 32 + 1
constexpr unsigned MTGP_RING  = 1024;
constexpr unsigned MTGP_MASKI = MTGP_RING - 1;
constexpr unsigned MTGP_STEPS = MTGP_RING / MTGP_BLOCK; // block-steps once around the ring
constexpr unsigned MTGP_COPY  = MTGP_N - MTGP_BLOCK;    // words that have a second copy

// One generator's device state: ring, ring offset, parameters.
struct mtgp_state
{
    uint32_t status[MTGP_RING];
    uint32_t offset;
    uint32_t pos, sh1, sh2, mask;
    uint32_t tbl[16], tmp[16];
};

struct mtgp_param
{
    uint32_t pos, sh1, sh2, tbl[16], tmp[16], mask;
};

const mtgp_param* params()
{
    static_assert(sizeof(mtgp_param) == 36 * 4, "layout of mtgp32_11213.bin");
    return reinterpret_cast<const mtgp_param*>(rr_mtgp32_params_begin);
}

// The parameter sets on the device (uploaded once per device).
__device__ mtgp_param d_params[MTGP_GENS];

// rocrand_make_state_mtgp32 (rocrand_mtgp32.h:362-390) and rocrand_mtgp32_init_state
// (:130-145), one wavefront per generator: the seeding recurrence is a chain of 350 uniform
// steps (scalar instructions), of which lane l keeps words l, l + 64, ...  Bound by that
// chain (13 us a seed; 512 x 351 words made on the host, copied and waited for, took 380).
__global__ __launch_bounds__(64) void mtgp_seed_kernel(mtgp_state* states, const mtgp_param* params, uint32_t seed)
{
    const uint32_t    b = blockIdx.x, lane = threadIdx.x;
    const mtgp_param& p = params[b];
    mtgp_state&       g = states[b];
    const uint32_t    hidden = p.tbl[4] ^ (p.tbl[8] << 16);
    uint32_t          tmp    = hidden;
    tmp += tmp >> 16;
    tmp += tmp >> 8;
    const uint32_t fill = (tmp & 0xffu) * 0x01010101u;
    uint32_t       x    = __builtin_amdgcn_readfirstlane(seed + b + 1);
    uint32_t       mine = x; // word 0
    for(uint32_t k = 1; k < MTGP_N; k++)
    {
        x = (k == 1 ? hidden : fill) ^ (1812433253u * (x ^ (x >> 30)) + k);
        if(k % 64 == 0)
            g.status[k - 64 + lane] = mine;
        mine = k % 64 == lane ? x : mine;
    }
    constexpr uint32_t last = MTGP_N / 64 * 64;
    for(uint32_t i = last + lane; i < MTGP_RING; i += 64)
        g.status[i] = i < MTGP_N ? mine : 0u;
    if(lane == 0)
    {
        g.offset = 0;
        g.pos    = p.pos;
        g.sh1    = p.sh1;
        g.sh2    = p.sh2;
        g.mask   = params[0].mask;
    }
    if(lane < 16)
    {
        g.tbl[lane] = p.tbl[lane];
        g.tmp[lane] = p.tmp[lane];
    }
}

// d_params of the current device, checked and uploaded on the first call there: the kernel
// evaluates the recurrence table from its entries at 1, 2, 4 and 8 (the tempering table is
// linear too and checked with it), and its unmasked ring reads reach word 768 + 255 + pos,
// which the 95 words copied behind the ring hold for pos <= 95.
rocrand_status device_params(const mtgp_param*& out);

struct mtgp_call
{
    mtgp_state* states;
    void*       data;
    size_t      n, mis, vec_n;
    uint32_t    head, tail;
    dist_params params;
};

// acc ^ tbl[k & 15] of a GF(2)-linear 16-entry table from its entries at 1, 2, 4 and 8: a
// sign-extending bit extraction and a v_bitop3 (a ^ (b & c)) each
__device__ __forceinline__ uint32_t mtgp_lin16(uint32_t acc, uint32_t k, const uint32_t (&e)[4])
{
#pragma unroll
    for(uint32_t i = 0; i < 4; i++)
        acc = __builtin_amdgcn_bitop3_b32(acc, e[i], __builtin_amdgcn_sbfe(k, i, 1), 0x78);
    return acc;
}

uint32_t host_lin16(uint32_t k, const uint32_t* tbl)
{
    return (k & 1 ? tbl[1] : 0) ^ (k & 2 ? tbl[2] : 0) ^ (k & 4 ? tbl[4] : 0) ^ (k & 8 ? tbl[8] : 0);
}

template<class D>
__global__ __launch_bounds__(MTGP_BLOCK) void mtgp_kernel(mtgp_call c)
{
    using out_t         = typename D::out_t;
    constexpr int IN    = D::in_w;
    constexpr int OUT   = D::out_w;
    constexpr int BYTES = OUT * (int)sizeof(out_t);
    static_assert(BYTES == 2 || BYTES == 4 || BYTES == 8 || BYTES == 16, "vec size");

    __shared__ uint32_t ring[MTGP_RING + MTGP_COPY];
    __shared__ uint32_t ttbl[16];

    const uint32_t b = blockIdx.x, t = threadIdx.x;
    mtgp_state*    g = c.states + b;
    const uint32_t off0 = g->offset;
    for(uint32_t i = t; i < MTGP_RING; i += MTGP_BLOCK)
        ring[i] = g->status[(i + off0) & MTGP_MASKI];
    const uint32_t pos = g->pos, sh1 = g->sh1, sh2 = g->sh2, mask = g->mask;
    if(t < 16)
        ttbl[t] = g->tmp[t];
    kernel_params kp{c.params, {}};
    // Poisson: the block samples from its copy of the packed alias table in dynamic LDS
    // (a per-lane load from global memory would wait for the block's earlier stores)
    if constexpr(dist_kind<D>::value == out_kind::poisson)
    {
        extern __shared__ uint64_t lds_packed[];
        const uint32_t             size = c.params.huge ? 0u : c.params.pt.size;
        for(uint32_t i = t; i < size; i += MTGP_BLOCK)
            lds_packed[i] = c.params.pt.packed[i];
        kp.pt.packed = lds_packed;
    }
    const uint32_t lin[4] = {g->tbl[1], g->tbl[2], g->tbl[4], g->tbl[8]};
    stage_tables<D>(kp.tab);
    __syncthreads();

    // one block-step, the `ph`-th of its turn: this thread's tempered word
    const uint32_t* const rx   = ring + t;
    const uint32_t* const ry   = ring + t + pos;
    uint32_t* const       wrap = ring + (t < MTGP_RING - MTGP_N - 2 * MTGP_BLOCK ? t + 2 * MTGP_BLOCK + MTGP_N
                                                                                : t + 2 * MTGP_BLOCK + MTGP_N - MTGP_RING);
    auto step = [&](uint32_t ph) -> uint32_t {
        const uint32_t at = ph * MTGP_BLOCK;
        uint32_t       X  = (rx[at] & mask) ^ rx[at + 1];
        uint32_t       Y  = ry[at];
        uint32_t       T  = ry[(int)at - 1];
        X                 = __builtin_amdgcn_bitop3_b32(X, X << sh1, Y >> sh2, 0x96);
        T ^= T >> 16;
        T ^= T >> 8;
        const uint32_t tt = ttbl[T & 0x0f];
        const uint32_t r  = mtgp_lin16(X, X, lin);
        if(ph == MTGP_STEPS - 1)
            ring[t + at + MTGP_N - MTGP_RING] = r;
        else
            ring[t + at + MTGP_N] = r;
        if(ph == MTGP_STEPS - 2)
            *wrap = r; // the words just written behind the ring, at its start (others: the same word)
        __syncthreads();
        return r ^ tt;
    };

    out_t* const data     = static_cast<out_t*>(c.data);
    out_t* const vec_data = data + c.mis;
    const size_t stride   = (size_t)MTGP_GENS * MTGP_BLOCK;
    const size_t rem      = c.vec_n % MTGP_BLOCK;
    const size_t down     = c.vec_n - rem;
    const size_t up       = rem == 0 ? down : down + MTGP_BLOCK;
    alignas(16) out_t o[OUT];
    uint32_t     in[IN];
    // the block's vec index before this thread's, block-uniform (a scalar loop counter and
    // store base): every thread takes part in every step
    const size_t   base0 = (size_t)b * MTGP_BLOCK;
    const uint32_t steps = base0 < down ? (uint32_t)((down - base0 + stride - 1) / stride) : 0u;
    out_t*         bptr  = vec_data + base0 * OUT;
    auto store = [&]() {
        out_t* const dst = bptr + t * OUT;
        if constexpr(BYTES == 2)
            *reinterpret_cast<uint16_t*>(dst) = *reinterpret_cast<const uint16_t*>(o);
        else if constexpr(BYTES == 4)
            *reinterpret_cast<uint32_t*>(dst) = *reinterpret_cast<const uint32_t*>(o);
        else if constexpr(BYTES == 8)
            *reinterpret_cast<uint2*>(dst) = *reinterpret_cast<const uint2*>(o);
        else
            *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(o);
        bptr += stride * OUT;
    };
    static_assert(MTGP_STEPS % IN == 0, "whole vecs a turn");
    constexpr uint32_t PER = MTGP_STEPS / IN; // vecs a turn
    uint32_t           k = 0, ph = 0;
    for(; k + PER <= steps; k += PER)
#pragma unroll
        for(uint32_t v = 0; v < PER; v++)
        {
#pragma unroll
            for(int i = 0; i < IN; i++)
                in[i] = step(v * IN + i);
            D::apply(in, o, kp);
            store();
        }
    // fewer than a turn is left, and the two extra uses
    auto next_vec = [&]() {
        for(int i = 0; i < IN; i++, ph = (ph + 1) % MTGP_STEPS)
            in[i] = step(ph);
        D::apply(in, o, kp);
    };
    for(; k < steps; k++)
    {
        next_vec();
        store();
    }
    size_t index = base0 + (size_t)steps * stride + t;
    if(index - t < up)
    {
        next_vec();
        if(index < c.vec_n)
            for(int j = 0; j < OUT; j++)
                vec_data[index * OUT + j] = o[j];
        index += stride;
    }
    if(OUT > 1 && (c.head > 0 || c.tail > 0))
    {
        next_vec();
        if(index == up)
            for(uint32_t j = 0; j < (uint32_t)OUT; j++)
                if(j < c.head)
                    data[j] = o[j];
        if(index == up + 1)
            for(uint32_t j = 0; j < (uint32_t)OUT; j++)
                if(j < c.tail)
                    data[c.n - c.tail + j] = o[j];
    }

    for(uint32_t i = t; i < MTGP_RING; i += MTGP_BLOCK)
        g->status[(i + off0) & MTGP_MASKI] = ring[i];
    if(t == 0)
        g->offset = (off0 + ph * MTGP_BLOCK) & MTGP_MASKI;
}

template<class D>
hipError_t launch_gen(const mtgp_call& c, hipStream_t s)
{
    const size_t lds = dist_kind<D>::value == out_kind::poisson && !c.params.huge
                           ? c.params.pt.size * sizeof(uint64_t)
                           : 0;
    hipLaunchKernelGGL((mtgp_kernel<D>), dim3(MTGP_GENS), dim3(MTGP_BLOCK), lds, s, c);
    return hipGetLastError();
}

hipError_t dispatch(out_kind o, const mtgp_call& c, hipStream_t s)
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

rocrand_status device_params(const mtgp_param*& out)
{
    static std::mutex  mtx;
    static mtgp_param* ready[64] = {};
    int                dev = 0;
    if(hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64)
        return ROCRAND_STATUS_INTERNAL_ERROR;
    std::lock_guard<std::mutex> lock(mtx);
    if(ready[dev] == nullptr)
    {
        const mtgp_param* p = params();
        for(unsigned i = 0; i < MTGP_GENS; i++)
        {
            if(p[i].pos == 0 || p[i].pos + MTGP_BLOCK > MTGP_N)
                return ROCRAND_STATUS_INTERNAL_ERROR;
            for(uint32_t k = 0; k < 16; k++)
                if(p[i].tbl[k] != host_lin16(k, p[i].tbl) || p[i].tmp[k] != host_lin16(k, p[i].tmp))
                    return ROCRAND_STATUS_INTERNAL_ERROR;
        }
        void* d = nullptr;
        if(hipGetSymbolAddress(&d, HIP_SYMBOL(d_params)) != hipSuccess
           || hipMemcpy(d, p, sizeof(mtgp_param) * MTGP_GENS, hipMemcpyHostToDevice) != hipSuccess)
            return ROCRAND_STATUS_ALLOCATION_FAILED;
        ready[dev] = static_cast<mtgp_param*>(d);
    }
    out = ready[dev];
    return ROCRAND_STATUS_SUCCESS;
}

// mtgp32.hpp:308-617
class mtgp32_generator final : public rocrand_generator_base_type
{
public:
    mtgp32_generator() : rocrand_generator_base_type(ROCRAND_RNG_PSEUDO_MTGP32) {}
    ~mtgp32_generator() override
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

    rocrand_status init() override
    {
        if(m_initialized)
            return ROCRAND_STATUS_SUCCESS;
        if(!m_states && hipMalloc(&m_states, sizeof(mtgp_state) * MTGP_GENS) != hipSuccess)
        {
            m_states = nullptr;
            return ROCRAND_STATUS_ALLOCATION_FAILED;
        }
        const mtgp_param* params = nullptr;
        rocrand_status    st     = device_params(params);
        if(st != ROCRAND_STATUS_SUCCESS)
            return st;
        hipLaunchKernelGGL(mtgp_seed_kernel, dim3(MTGP_GENS), dim3(64), 0, stream, static_cast<mtgp_state*>(m_states),
                           params, (uint32_t)(m_seed ^ (m_seed >> 32)));
        if(hipGetLastError() != hipSuccess)
            return ROCRAND_STATUS_LAUNCH_FAILURE;
        m_initialized = true;
        m_seeding     = true;
        return ROCRAND_STATUS_SUCCESS;
    }

    // An explicit set-up returns with the states made, whatever stream the generate calls then
    // run on (set-up had copied them and waited).  A capturing stream cannot be waited for.
    rocrand_status settle() override
    {
        hipStreamCaptureStatus c = hipStreamCaptureStatusNone;
        if(!m_seeding
           || (stream != nullptr && hipStreamIsCapturing(stream, &c) == hipSuccess && c != hipStreamCaptureStatusNone))
            return ROCRAND_STATUS_SUCCESS;
        if(hipStreamSynchronize(stream) != hipSuccess)
            return ROCRAND_STATUS_LAUNCH_FAILURE;
        m_seeding = false;
        return ROCRAND_STATUS_SUCCESS;
    }

    rocrand_status shape(out_kind k, dist_shape& s) const override
    {
        switch(k)
        {
#define RR_SHAPE(K)                                                                                    \
    case K:                                                                                            \
        s = dist_shape{dist<word_family::w32, K>::in_w, dist<word_family::w32, K>::out_w,              \
                       (int)sizeof(typename dist<word_family::w32, K>::out_t)};                        \
        return ROCRAND_STATUS_SUCCESS;
            RR_SHAPE(out_kind::u8)
            RR_SHAPE(out_kind::u16)
            RR_SHAPE(out_kind::u32)
            RR_SHAPE(out_kind::uniform_f32)
            RR_SHAPE(out_kind::uniform_f64)
            RR_SHAPE(out_kind::uniform_f16)
            RR_SHAPE(out_kind::normal_f32)
            RR_SHAPE(out_kind::normal_f64)
            RR_SHAPE(out_kind::normal_f16)
            RR_SHAPE(out_kind::lognormal_f32)
            RR_SHAPE(out_kind::lognormal_f64)
            RR_SHAPE(out_kind::lognormal_f16)
            RR_SHAPE(out_kind::poisson)
#undef RR_SHAPE
            default: return ROCRAND_STATUS_TYPE_ERROR;
        }
    }

protected:
    void reset() override { m_initialized = false; }

    rocrand_status generate_device(out_kind k, void* data, size_t n, const gen_args& args) override
    {
        dist_shape     s;
        rocrand_status st = shape(k, s);
        if(st != ROCRAND_STATUS_SUCCESS)
            return st;
        mtgp_call c{};
        if((st = make_params(k, args, c.params)) != ROCRAND_STATUS_SUCCESS)
            return st;
        if((st = init()) != ROCRAND_STATUS_SUCCESS)
            return st;
        if(data == nullptr)
            return settle();
        const uintptr_t addr = reinterpret_cast<uintptr_t>(data);
        c.mis    = (s.out_w - (addr / s.esz) % s.out_w) % s.out_w;
        c.head   = (uint32_t)std::min<size_t>(n, c.mis);
        c.tail   = (uint32_t)((n - c.head) % s.out_w);
        c.vec_n  = (n - c.head) / s.out_w;
        c.states = static_cast<mtgp_state*>(m_states);
        c.data   = data;
        c.n      = n;
        m_seeding = false; // the call's own work follows the seeding on its stream
        if(dispatch(k, c, stream) != hipSuccess)
            return ROCRAND_STATUS_LAUNCH_FAILURE;
        return ROCRAND_STATUS_SUCCESS;
    }

private:
    unsigned long long m_seed        = 0;
    bool               m_initialized = false;
    bool               m_seeding     = false; // seeded since the last wait or generate call
    void*              m_states      = nullptr;
};

} // namespace

rocrand_generator make_mtgp32_generator() { return new mtgp32_generator(); }

} // namespace rr
