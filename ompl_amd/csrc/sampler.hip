// Batched uniform state sampling: RealVectorStateSampler::sampleUniform
// (base/spaces/src/RealVectorStateSpace.cpp:45-52) over ompl::RNG::uniformReal
// (util/RandomNumbers.h:72-76): std::mt19937 seeded with the RNG's local seed
// (util/src/RandomNumbers.cpp:224-228), uniform_real_distribution<>(0,1) as
// libstdc++'s generate_canonical<double,53> (two 32-bit draws w1, w2:
// (w1 + w2*2^32) / 2^64, values rounding to 1 replaced by the largest double
// below 1), then (hi - lo) * u + lo per dimension in order.
//
// One workgroup per generator; the 624-word state lives in LDS and is twisted
// by the block (mt_device.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "grid_device.hpp"
#include "mt_device.hpp"
#include "runtime.hpp"

namespace ompl_amd {

constexpr int kDim7 = OMPL_AMD_ARM_DOF;

// A call's bounds, by value (they are host arrays of at most 16 entries).
struct Bounds {
    double lo[16], span[16];
};

static Bounds bounds_of(const double *lo, const double *hi, int dim)
{
    Bounds b{};
    for (int d = 0; d < dim; ++d) {
        b.lo[d] = lo[d];
        b.span[d] = hi[d] - lo[d];
    }
    return b;
}

struct MtState {
    uint32_t mt[kMtN];
    int32_t idx; // next word; kMtN = twist before the next draw
    int32_t pad[3];
};

__global__ void mt_seed_kernel(const uint32_t *__restrict__ seeds, int n, MtState *__restrict__ st)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    uint32_t v = seeds[s];
    st[s].mt[0] = v;
    for (int i = 1; i < kMtN; ++i) {
        v = 1812433253u * (v ^ (v >> 30)) + (uint32_t)i;
        st[s].mt[i] = v;
    }
    st[s].idx = kMtN;
}

// The block's generator into LDS: seeded (seeds: a device or host-mapped
// array) or resumed.  Ends with a barrier.
__device__ __forceinline__ int load_generator(uint32_t *mt, const uint32_t *seeds, const MtState *gen)
{
    int idx = kMtN;
    if (seeds) {
        if (threadIdx.x == 0) mt_seed_serial(mt, seeds[blockIdx.x]);
    } else {
        for (int i = threadIdx.x; i < kMtN; i += blockDim.x) mt[i] = gen[blockIdx.x].mt[i];
        idx = gen[blockIdx.x].idx;
    }
    __syncthreads();
    return idx;
}

__device__ __forceinline__ void store_generator(const uint32_t *mt, int idx, MtState *gen)
{
    for (int i = threadIdx.x; i < kMtN; i += blockDim.x) gen[blockIdx.x].mt[i] = mt[i];
    if (threadIdx.x == 0) gen[blockIdx.x].idx = idx;
}

// The next `total` canonical draws of the block's generator, draw z handed to
// use(z, value) by one thread.
template <class Use>
__device__ __forceinline__ void draw_block(uint32_t *mt, int &idx, int64_t total, Use use)
{
    for (int64_t z = 0; z < total;) {
        if (idx >= kMtN) {
            mt_twist_block(mt);
            idx = 0;
        }
        const int cnt = (int)min((int64_t)((kMtN - idx) / 2), total - z);
        for (int p = threadIdx.x; p < cnt; p += blockDim.x)
            use(z + p, canonical53(mt_temper(mt[idx + 2 * p]), mt_temper(mt[idx + 2 * p + 1])));
        idx += 2 * cnt;
        z += cnt;
        __syncthreads(); // the words are read before the next twist writes them
    }
}

// n_per_stream states of `dim` doubles per generator ([stream][n][dim]) and,
// when out_f32 is given, their FP32 copy ([dim][n_streams * n]).  Bound by the
// twists (one per 312 coordinates, a chain): 256 generators x 782 states of 7
// take 36 us; with 64 threads and eight barriers a twist they took 58.
__global__ void __launch_bounds__(256) sample_uniform_kernel(const uint32_t *__restrict__ seeds,
                                                             MtState *__restrict__ gen, int64_t n_per_stream, int dim,
                                                             Bounds B, double *__restrict__ out,
                                                             float *__restrict__ out_f32)
{
    __shared__ uint32_t mt[kMtN];
    __shared__ double lo[16], span[16];
    if (threadIdx.x < 16) {
        lo[threadIdx.x] = B.lo[threadIdx.x];
        span[threadIdx.x] = B.span[threadIdx.x];
    }
    int idx = load_generator(mt, seeds, gen);
    const int64_t n_all = (int64_t)gridDim.x * n_per_stream;
    double *o = out + (int64_t)blockIdx.x * n_per_stream * dim;
    const bool small = n_per_stream * dim <= (int64_t)UINT32_MAX;
    draw_block(mt, idx, n_per_stream * dim, [&](int64_t z, double u) {
        const int64_t st = small ? (int64_t)((uint32_t)z / (uint32_t)dim) : z / dim;
        const int d = (int)(z - st * dim);
        const double v = span[d] * u + lo[d];
        o[z] = v;
        if (out_f32) out_f32[(int64_t)d * n_all + (int64_t)blockIdx.x * n_per_stream + st] = (float)v;
    });
    if (gen && !seeds) store_generator(mt, idx, gen);
}

// ---------------------------------------------------------------------------
// UniformValidStateSampler::sample (base/samplers/src/UniformValidStateSampler.cpp:
// 46-57), batched over streams: each stream is one sampler making successive
// sample() calls; a call draws uniform states until one is valid or `attempts`
// draws were made.  One workgroup per stream runs all its calls: it draws a
// batch, one state per thread, checks the batch over the cell grid, and finds
// where calls end.  Draw j ends a call when it is valid or when the draws since
// the last valid one (or since the call under way began) are a multiple of
// `attempts`, so every thread decides its own draw from the batch's valid bits.
// A batch may draw past the last call's end; the generator is then put back to
// the batch's start and advanced by the draws that were used.
//
// 256 samplers x 64 calls, one draw in eighty valid: 198 us, bound by the
// batches' chain (a twist per 44 draws, then the check); in rounds of one launch
// per step it took 3.9 ms (a host round trip, a serial hand-out of 867 us and a
// rewind pass per round).
constexpr int kValidThreads = 512;
// Batches of one launch: a call whose calls could take more (many attempts in a
// scene with nothing valid) goes on in another, from its cursors.
constexpr int kValidBatches = 4096;

struct ValidCursor {
    int64_t call, drawn; // calls made; draws seen by them
    uint32_t carry;      // draws of the call under way
    uint32_t pad;
};

struct ValidArgs {
    GridView g;
    const uint32_t *seeds; // or null: resume gen
    MtState *gen;          // or null: the generators are not kept
    int64_t n_calls;
    int attempts;
    Bounds b;
    double *out;
    uint8_t *found;
    int32_t *draws;
    ValidCursor *cursor; // or null: one launch is enough
    int32_t *open;       // with cursor: streams that are not done
};

__global__ void __launch_bounds__(kValidThreads) sample_valid_kernel(ValidArgs A)
{
    constexpr int kWaves = kValidThreads / 64;
    __shared__ uint32_t mt[kMtN], mt0[kMtN];
    // the batch's draws, until each thread has its state; then the exact tests
    __shared__ union {
        double u[kValidThreads * kDim7];
        WaveTests tests[kWaves];
    } w;
    __shared__ uint64_t valid_bits[kWaves], end_bits[kWaves];
    __shared__ int used;
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    int idx = load_generator(mt, A.seeds, A.gen);
    int64_t call = 0, calls_drawn = 0;
    uint32_t carry = 0; // draws of the call under way (fewer than attempts)
    if (A.cursor) {
        call = A.cursor[blockIdx.x].call;
        calls_drawn = A.cursor[blockIdx.x].drawn;
        carry = A.cursor[blockIdx.x].carry;
        if (call >= A.n_calls) return;
    }
    for (int batch = 0; call < A.n_calls && !(A.cursor && batch == kValidBatches); ++batch) {
        // a batch that should finish the calls, by the draws a call took so far
        const int64_t left = A.n_calls - call;
        const double want = call > 0 ? 1.125 * (double)left * (double)calls_drawn / (double)call
                                     : (calls_drawn ? (double)kValidThreads : 1.25 * (double)left) + 16.0;
        const int m = (int)fmin((double)kValidThreads, fmax(64.0, want));
        for (int i = t; i < kMtN; i += kValidThreads) mt0[i] = mt[i];
        const int idx0 = idx;
        __syncthreads();
        draw_block(mt, idx, (int64_t)m * kDim7, [&](int64_t z, double u) { w.u[z] = u; });
        double v[kDim7];
        float q[kDof];
#pragma unroll
        for (int d = 0; d < kDim7; ++d) {
            v[d] = A.b.span[d] * (t < m ? w.u[t * kDim7 + d] : 0.0) + A.b.lo[d];
            q[d] = (float)v[d];
        }
        __syncthreads(); // the draws are read: their room is free
        const bool live = t < m;
        // every lane of the wave goes in (the exact tests are shared among all 64)
        const bool hit = state_hit1(A.g, q, live, w.tests[wave]);
        const bool valid = live && !hit;
        const uint64_t vb = __ballot(valid);
        if (lane == 0) valid_bits[wave] = vb;
        __syncthreads();
        int last = -1; // the last valid draw before this one
        for (int i = 0; i < wave; ++i)
            if (valid_bits[i]) last = i * 64 + 63 - __builtin_clzll(valid_bits[i]);
        const uint64_t below = vb & (((uint64_t)1 << lane) - 1);
        if (below) last = wave * 64 + 63 - __builtin_clzll(below);
        const uint32_t since = last >= 0 ? (uint32_t)(t - last) : (uint32_t)t + 1u + carry;
        const bool end = live && (valid || since % (uint32_t)A.attempts == 0);
        const uint64_t eb = __ballot(end);
        if (lane == 0) end_bits[wave] = eb;
        if (t == 0) used = m;
        __syncthreads();
        int before = 0, all = 0, last_end = -1;
        for (int i = 0; i < kWaves; ++i) {
            const uint64_t e = end_bits[i];
            if (i < wave) before += __popcll(e);
            all += __popcll(e);
            if (e) last_end = i * 64 + 63 - __builtin_clzll(e);
        }
        const int64_t c = call + before + __popcll(eb & (((uint64_t)1 << lane) - 1));
        if (end && c < A.n_calls) {
            const int64_t o = (int64_t)blockIdx.x * A.n_calls + c;
#pragma unroll
            for (int d = 0; d < kDim7; ++d) A.out[o * kDim7 + d] = v[d];
            A.found[o] = valid ? 1 : 0;
            if (A.draws) A.draws[o] = (int32_t)((since - 1) % (uint32_t)A.attempts) + 1;
            if (c == A.n_calls - 1) used = t + 1;
        }
        __syncthreads();
        carry = last_end >= 0 ? (uint32_t)(m - 1 - last_end) : carry + (uint32_t)m;
        calls_drawn += m;
        call = min(call + all, A.n_calls);
        if (call == A.n_calls && A.gen) {
            // back to the batch's start, then past the draws that were used
            const int take = used;
            for (int i = t; i < kMtN; i += kValidThreads) mt[i] = mt0[i];
            __syncthreads();
            idx = idx0;
            for (int skip = take * 2 * kDim7; skip > 0;) {
                if (idx >= kMtN) {
                    mt_twist_block(mt);
                    idx = 0;
                }
                const int n = min(kMtN - idx, skip);
                idx += n;
                skip -= n;
            }
        }
        __syncthreads(); // `used` and the bits are read before the next batch writes them
    }
    if (A.gen) store_generator(mt, idx, A.gen);
    if (A.cursor && t == 0) {
        A.cursor[blockIdx.x] = ValidCursor{call, calls_drawn, carry, 0};
        if (call < A.n_calls) atomicAdd(A.open, 1);
    }
}

// SE3StateSampler::sampleUniform (a compound sampler: the R^3 component's
// RealVectorStateSampler, then SO3StateSampler::sampleUniform = RNG::quaternion,
// util/src/RandomNumbers.cpp:266-279, Shoemake) from six canonical draws per
// state u[0..5]: x_k = (hi_k - lo_k) u_k + lo_k; x0 = u3, t1 = 2 pi u4,
// t2 = 2 pi u5, q = (sin t1 sqrt(1-x0), cos t1 sqrt(1-x0), sin t2 sqrt(x0),
// cos t2 sqrt(x0)) in FP64 (the device's sin/cos are within an ulp or two of
// the host's).  Output rows (x, y, z, qx, qy, qz, qw) as FP64 and FP32.
__global__ void se3_from_uniform_kernel(const double *__restrict__ u, int64_t n, Bounds B, double *__restrict__ out,
                                        float *__restrict__ out_f32)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double *v = u + i * 6;
    double r[7];
#pragma unroll
    for (int k = 0; k < 3; ++k) r[k] = B.span[k] * v[k] + B.lo[k];
    const double pi = 3.141592653589793238462643383279502884;
    const double x0 = v[3];
    const double r1 = sqrt(1.0 - x0), r2 = sqrt(x0);
    const double t1 = 2.0 * pi * v[4], t2 = 2.0 * pi * v[5];
    r[3] = sin(t1) * r1;
    r[4] = cos(t1) * r1;
    r[5] = sin(t2) * r2;
    r[6] = cos(t2) * r2;
#pragma unroll
    for (int k = 0; k < 7; ++k) {
        out[i * 7 + k] = r[k];
        if (out_f32) out_f32[i * 7 + k] = (float)r[k];
    }
}

// The seeds of a call in the thread's host-mapped staging, which the kernel
// reads; the call waits for the stream before it returns.
static const uint32_t *stage_seeds(const uint32_t *seeds, int n)
{
    ThreadResources &r = thread_resources();
    stage_reserve(r, (size_t)n * sizeof(uint32_t));
    std::copy(seeds, seeds + n, reinterpret_cast<uint32_t *>(r.stage));
    return reinterpret_cast<const uint32_t *>(r.stage_dev);
}

static void sample_uniform(const uint32_t *seeds, MtState *gen, int n_streams, int64_t n_per_stream, int dim,
                           const double *lo, const double *hi, double *out, float *out_f32, hipStream_t s)
{
    ProfScope ps("sample_uniform", s);
    hipLaunchKernelGGL(sample_uniform_kernel, dim3(n_streams), dim3(256), 0, s, seeds, gen, n_per_stream, dim,
                       bounds_of(lo, hi, dim), out, out_f32);
    OA_HIP(hipGetLastError());
}

static void sample_valid(ompl_amd_env env, const uint32_t *seeds, MtState *gen, int n_streams, int64_t n_calls,
                         int attempts, const double *lo, const double *hi, double *out_dev, uint8_t *found_dev,
                         int32_t *draws_dev, hipStream_t s)
{
    ValidArgs A{env->env.grid, seeds,     gen,       n_calls, attempts, bounds_of(lo, hi, kDim7), out_dev,
                found_dev,     draws_dev, nullptr, nullptr};
    auto launch = [&] {
        ProfScope ps("sample_valid", s);
        hipLaunchKernelGGL(sample_valid_kernel, dim3(n_streams), dim3(kValidThreads), 0, s, A);
        OA_HIP(hipGetLastError());
    };
    // no batch holds fewer than 64 draws
    if ((double)n_calls * attempts <= 64.0 * (kValidBatches - 1)) {
        launch();
        OA_HIP(hipStreamSynchronize(s));
        return;
    }
    struct Scratch { // generators of a seeded call, cursors and the count
        hipStream_t s;
        char *p = nullptr;
        ~Scratch()
        {
            if (p) (void)hipFreeAsync(p, s);
            (void)hipStreamSynchronize(s);
        }
    } room{s};
    const size_t cursors = (size_t)n_streams * sizeof(ValidCursor), gens = seeds ? (size_t)n_streams * sizeof(MtState) : 0;
    OA_HIP(device_malloc_async(&room.p, cursors + gens + 256, s));
    A.cursor = (ValidCursor *)room.p;
    A.open = (int32_t *)(room.p + cursors + gens);
    OA_HIP(hipMemsetAsync(A.cursor, 0, cursors, s));
    if (seeds) {
        A.gen = (MtState *)(room.p + cursors);
        A.seeds = nullptr;
        hipLaunchKernelGGL(mt_seed_kernel, dim3((n_streams + 63) / 64), dim3(64), 0, s, seeds, n_streams, A.gen);
    }
    for (int32_t open = 1; open > 0;) {
        OA_HIP(hipMemsetAsync(A.open, 0, sizeof(int32_t), s));
        launch();
        OA_HIP(hipMemcpyAsync(&open, A.open, sizeof(open), hipMemcpyDeviceToHost, s));
        OA_HIP(hipStreamSynchronize(s));
    }
}

} // namespace ompl_amd

using namespace ompl_amd;

extern "C" int ompl_amd_sample_uniform_dev(const uint32_t *seeds, int n_streams, int64_t n_per_stream, int dim,
                                           const double *lo, const double *hi, double *out_dev, float *out_f32,
                                           void *stream)
{
    return guarded([&] {
        OA_REQUIRE(n_streams >= 0 && n_per_stream >= 0, OMPL_AMD_ERR_ARG, "negative sizes");
        OA_REQUIRE(dim >= 1 && dim <= 16, OMPL_AMD_ERR_ARG, "dim must be in [1, 16]");
        if (n_streams == 0 || n_per_stream == 0) return;
        OA_REQUIRE(seeds && lo && hi && out_dev, OMPL_AMD_ERR_ARG, "null pointer");
        hipStream_t s = resolve_stream(stream);
        sample_uniform(stage_seeds(seeds, n_streams), nullptr, n_streams, n_per_stream, dim, lo, hi, out_dev, out_f32,
                       s);
        OA_HIP(hipStreamSynchronize(s)); // the seeds are read from host memory
    });
}

// Generators kept on the device between calls: the exact continuation of a
// long-lived sampler's RNG.
struct ompl_amd_rng_s {
    MtState *gen = nullptr;
    int n = 0;
    ~ompl_amd_rng_s()
    {
        if (gen) hipFree(gen);
    }
};

static MtState *seed_generators(const uint32_t *seeds, int n, hipStream_t s)
{
    MtState *gen = nullptr;
    uint32_t *dseeds = nullptr;
    OA_HIP(device_malloc_async(&gen, (size_t)n * sizeof(MtState), s));
    OA_HIP(device_malloc_async(&dseeds, (size_t)n * sizeof(uint32_t), s));
    OA_HIP(hipMemcpyAsync(dseeds, seeds, (size_t)n * sizeof(uint32_t), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(mt_seed_kernel, dim3((n + 63) / 64), dim3(64), 0, s, dseeds, n, gen);
    OA_HIP(hipGetLastError());
    OA_HIP(hipFreeAsync(dseeds, s));
    OA_HIP(hipStreamSynchronize(s)); // the seeds are a host array
    return gen;
}

extern "C" {

int ompl_amd_sample_valid_dev(ompl_amd_env env, const uint32_t *seeds, int n_streams, int64_t n_calls, int attempts,
                              const double *lo, const double *hi, double *out_dev, uint8_t *found_dev,
                              int32_t *draws_dev, void *stream)
{
    return guarded([&] {
        OA_REQUIRE(env, OMPL_AMD_ERR_ARG, "null environment");
        OA_REQUIRE(n_streams >= 0 && n_calls >= 0 && attempts >= 1, OMPL_AMD_ERR_ARG, "bad sizes");
        if (n_streams == 0 || n_calls == 0) return;
        OA_REQUIRE(seeds && lo && hi && out_dev && found_dev, OMPL_AMD_ERR_ARG, "null pointer");
        hipStream_t s = resolve_stream(stream);
        sample_valid(env, stage_seeds(seeds, n_streams), nullptr, n_streams, n_calls, attempts, lo, hi, out_dev,
                     found_dev, draws_dev, s);
    });
}

int ompl_amd_rng_create(const uint32_t *seeds, int n_streams, ompl_amd_rng *out)
{
    return guarded([&] {
        OA_REQUIRE(out && seeds && n_streams >= 1, OMPL_AMD_ERR_ARG, "bad arguments");
        ensure_init();
        auto *r = new ompl_amd_rng_s();
        try {
            r->gen = seed_generators(seeds, n_streams, default_stream());
        } catch (...) {
            delete r;
            throw;
        }
        r->n = n_streams;
        *out = r;
    });
}

int ompl_amd_rng_destroy(ompl_amd_rng rng)
{
    return guarded([&] {
        if (rng) OA_HIP(hipDeviceSynchronize());
        delete rng;
    });
}

int ompl_amd_rng_sample_uniform_dev(ompl_amd_rng rng, int64_t n_per_stream, int dim, const double *lo,
                                    const double *hi, double *out_dev, float *out_f32_soa_dev, void *stream)
{
    return guarded([&] {
        OA_REQUIRE(rng, OMPL_AMD_ERR_ARG, "null generator");
        OA_REQUIRE(n_per_stream >= 0 && dim >= 1 && dim <= 16, OMPL_AMD_ERR_ARG, "bad sizes");
        if (n_per_stream == 0) return;
        OA_REQUIRE(lo && hi && out_dev, OMPL_AMD_ERR_ARG, "null pointer");
        hipStream_t s = resolve_stream(stream);
        sample_uniform(nullptr, rng->gen, rng->n, n_per_stream, dim, lo, hi, out_dev, out_f32_soa_dev, s);
        OA_HIP(hipStreamSynchronize(s));
    });
}

int ompl_amd_rng_sample_se3_dev(ompl_amd_rng rng, int64_t n_per_stream, const double *lo, const double *hi,
                                double *out_dev, float *out_f32_dev, void *stream)
{
    return guarded([&] {
        OA_REQUIRE(rng, OMPL_AMD_ERR_ARG, "null generator");
        OA_REQUIRE(n_per_stream >= 0, OMPL_AMD_ERR_ARG, "bad sizes");
        if (n_per_stream == 0) return;
        OA_REQUIRE(lo && hi && out_dev, OMPL_AMD_ERR_ARG, "null pointer");
        hipStream_t s = resolve_stream(stream);
        const double zero[6] = {0, 0, 0, 0, 0, 0}, one[6] = {1, 1, 1, 1, 1, 1};
        const int64_t n = (int64_t)rng->n * n_per_stream;
        double *u = nullptr;
        OA_HIP(device_malloc_async(&u, (size_t)n * 6 * sizeof(double), s));
        {
            ProfScope ps("sample_se3", s);
            sample_uniform(nullptr, rng->gen, rng->n, n_per_stream, 6, zero, one, u, nullptr, s);
            hipLaunchKernelGGL(se3_from_uniform_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, u, n,
                               bounds_of(lo, hi, 3), out_dev, out_f32_dev);
            OA_HIP(hipGetLastError());
        }
        OA_HIP(hipFreeAsync(u, s));
        OA_HIP(hipStreamSynchronize(s));
    });
}

int ompl_amd_rng_sample_valid_dev(ompl_amd_rng rng, ompl_amd_env env, int64_t n_calls, int attempts,
                                  const double *lo, const double *hi, double *out_dev, uint8_t *found_dev,
                                  int32_t *draws_dev, void *stream)
{
    return guarded([&] {
        OA_REQUIRE(rng && env, OMPL_AMD_ERR_ARG, "null generator or environment");
        OA_REQUIRE(n_calls >= 0 && attempts >= 1, OMPL_AMD_ERR_ARG, "bad sizes");
        if (n_calls == 0) return;
        OA_REQUIRE(lo && hi && out_dev && found_dev, OMPL_AMD_ERR_ARG, "null pointer");
        sample_valid(env, nullptr, rng->gen, rng->n, n_calls, attempts, lo, hi, out_dev, found_dev, draws_dev,
                     resolve_stream(stream));
    });
}

} // extern "C"
