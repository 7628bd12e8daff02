// fill.hip -- seeded synthetic GEMM inputs generated on the device, so a bench or
// a test can create 4096^3-sized operands without a host round trip. Element i is
// a pure function of (seed, i); the CPU oracle computes the same values, which is
// how the tests pin these kernels bit for bit.

#include "ridge_gemm.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));

constexpr int kThreads = 256;

// Both fills are one pass of stores with the element's value computed in registers.
// A thread makes VEC consecutive elements: 8, one 16-byte store, where dst is 16-byte
// aligned, else 1. A workgroup takes chunks of kThreads * VEC elements, a grid apart.
// Before -> after, one 2-byte store per element -> these: uniform 2^26 elements 58 ->
// 49 us (2.7 TB/s; the integer products bound it), 2^24 24.6 -> 16.8; LCG, which
// squared its map up to 27 times per element, 2^26 356 -> 24 us (5.5 TB/s), 2^22
// 24.3 -> 6.2.
template <int VEC, typename Gen>
__device__ __forceinline__ void fillChunks(_Float16* dst, size_t n, Gen gen) {
    constexpr size_t kChunk = (size_t)kThreads * VEC;
    const size_t stride = gridDim.x * kChunk;
    gen.start(blockIdx.x * kChunk, threadIdx.x * VEC);
    for (size_t i = blockIdx.x * kChunk + threadIdx.x * VEC; i < n; i += stride, gen.advance()) {
        _Float16 v[VEC];
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[j] = gen.next();
        if (VEC == 8 && i + VEC <= n) {
            *reinterpret_cast<half8_t*>(dst + i) = half8_t{v[0], v[1 % VEC], v[2 % VEC], v[3 % VEC],
                                                           v[4 % VEC], v[5 % VEC], v[6 % VEC], v[7 % VEC]};
        } else {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                if (i + j < n) dst[i + j] = v[j];
        }
    }
}

// splitmix64 (Steele, Lea and Flood, 2014): output i of the stream seeded with s
// is the finaliser applied to s + (i + 1) * 0x9e3779b97f4a7c15. Only its top 24 bits
// are used, which the finaliser's last step (z ^ z >> 31) leaves alone. Multiplying
// by 0xbf58476d1ce4e5b9 and 0x94d049bb133111eb takes six 32-bit products, which bound
// the fill.
constexpr uint64_t kGamma = 0x9e3779b97f4a7c15ull;

struct UniformGen {
    uint64_t base;   // state before the thread's next element
    uint64_t skip;   // what a grid stride adds to the state, less the elements made
    __device__ __forceinline__ void start(size_t chunk, unsigned offset) { base += (chunk + offset) * kGamma; }
    __device__ __forceinline__ void advance() { base += skip; }
    __device__ __forceinline__ _Float16 next() {
        base += kGamma;
        // In 32-bit halves: 64-bit shifts and the conversion of a 64-bit integer
        // to float are several instructions each.
        uint32_t lo = (uint32_t)base, hi = (uint32_t)(base >> 32);
        xorShift<30>(lo, hi);
        const uint64_t z = (uint64_t)lo * 0x1ce4e5b9u;
        hi = (uint32_t)(z >> 32) + lo * 0xbf58476du + hi * 0x1ce4e5b9u;
        lo = (uint32_t)z;
        xorShift<27>(lo, hi);
        hi = __umulhi(lo, 0x133111ebu) + lo * 0x94d049bbu + hi * 0x133111ebu;
        // top24 * 2^-23 is exact in float and so is the subtraction of 1, which
        // leaves the conversion to half as the only rounding (nearest even).
        return (_Float16)((float)(hi >> 8) * (1.0f / 8388608.0f) - 1.0f);
    }
    // (hi:lo) ^= (hi:lo) >> S
    template <int S>
    static __device__ __forceinline__ void xorShift(uint32_t& lo, uint32_t& hi) {
        lo ^= __builtin_amdgcn_alignbit(hi, lo, S);
        hi ^= hi >> S;
    }
};

// The reference fill (bench/check-gemm.cu:139-145) advances a 32-bit LCG once per
// element: element i needs state T^{i+1}(seed) with T(s) = a s + c mod 2^32. The
// powers of T commute and T^{2^32} is the identity, so the state after `steps` steps
// is the composition of the T^{2^b} of the set bits of steps mod 2^32.
struct LcgPowers {
    uint32_t mul[32], add[32];
    constexpr LcgPowers() : mul{}, add{} {
        uint32_t m = 1664525u, a = 1013904223u;
        for (int b = 0; b < 32; ++b) {
            mul[b] = m;
            add[b] = a;
            a = m * a + a;
            m = m * m;
        }
    }
};
constexpr LcgPowers kLcg{};

__host__ __device__ inline uint32_t lcgSteps(uint32_t s, uint32_t steps) {
    constexpr LcgPowers p{};
#pragma unroll
    for (int b = 0; b < 32; ++b)
        if (steps >> b & 1u) s = p.mul[b] * s + p.add[b];
    return s;
}

struct LcgGen {
    uint32_t s;                  // state of the thread's previous element
    uint32_t skipMul, skipAdd;   // the map of a grid stride, less the elements made
    // The chunk's bits are uniform over the workgroup and cost scalar work; a
    // thread's own offset is below 2^11.
    __device__ __forceinline__ void start(size_t chunk, unsigned offset) {
        s = lcgSteps(s, (uint32_t)chunk);
#pragma unroll
        for (int b = 0; b < 11; ++b) s = offset >> b & 1u ? kLcg.mul[b] * s + kLcg.add[b] : s;
    }
    __device__ __forceinline__ void advance() { s = skipMul * s + skipAdd; }
    __device__ __forceinline__ _Float16 next() {
#pragma clang fp contract(off)
        s = kLcg.mul[0] * s + kLcg.add[0];
        // x / 32767 - 0.5 in float, rounded to half. The product with the rounded
        // reciprocal differs from the quotient in its last bit for some x, but
        // after the subtraction and the rounding to half all 32768 values of x
        // agree (tests/test_oracle.py compares them). A fused multiply-add would
        // not: it moves x = 32747.
        const float q = (float)((s >> 16) & 0x7fffu) * (1.0f / 32767.0f);
        return (_Float16)(q - 0.5f);
    }
};

template <int VEC>
__global__ __launch_bounds__(kThreads) void fillUniformKernel(_Float16* dst, size_t n, UniformGen gen) {
    fillChunks<VEC>(dst, n, gen);
}

template <int VEC>
__global__ __launch_bounds__(kThreads) void fillLcgKernel(_Float16* dst, size_t n, LcgGen gen) {
    fillChunks<VEC>(dst, n, gen);
}

// Workgroups: eight per CU of 256, so that a thread's start is shared by its chunks.
constexpr size_t kMostBlocks = 2048;

unsigned gridFor(size_t n, int vec) {
    const size_t chunk = (size_t)kThreads * vec;
    const size_t blocks = (n + chunk - 1) / chunk;
    return (unsigned)(blocks < kMostBlocks ? blocks : kMostBlocks);
}

int vectorOf(const void* dst) { return ((uintptr_t)dst & 15u) == 0 ? 8 : 1; }

template <int VEC>
void fillUniform(_Float16* dst, size_t n, uint64_t seed, hipStream_t stream) {
    const unsigned grid = gridFor(n, VEC);
    const UniformGen gen{seed, ((uint64_t)grid * kThreads * VEC - VEC) * kGamma};
    hipLaunchKernelGGL((fillUniformKernel<VEC>), dim3(grid), dim3(kThreads), 0, stream, dst, n, gen);
}

template <int VEC>
void fillLcg(_Float16* dst, size_t n, uint32_t seed, hipStream_t stream) {
    const unsigned grid = gridFor(n, VEC);
    // The map of k steps takes 0 to its addend and 1 to multiplier + addend.
    const uint32_t steps = grid * kThreads * VEC - VEC;
    const uint32_t add = lcgSteps(0u, steps);
    const LcgGen gen{seed, lcgSteps(1u, steps) - add, add};
    hipLaunchKernelGGL((fillLcgKernel<VEC>), dim3(grid), dim3(kThreads), 0, stream, dst, n, gen);
}

}  // namespace

extern "C" int ridge_fill_uniform_f16(void* dst, size_t n, uint64_t seed, void* stream) {
    if (n == 0) return 0;
    if (dst == nullptr) return (int)hipErrorInvalidValue;
    auto* p = static_cast<_Float16*>(dst);
    if (vectorOf(dst) == 8) {
        fillUniform<8>(p, n, seed, static_cast<hipStream_t>(stream));
    } else {
        fillUniform<1>(p, n, seed, static_cast<hipStream_t>(stream));
    }
    return (int)hipGetLastError();
}

extern "C" int ridge_fill_lcg_f16(void* dst, size_t n, uint32_t seed, void* stream) {
    if (n == 0) return 0;
    if (dst == nullptr) return (int)hipErrorInvalidValue;
    auto* p = static_cast<_Float16*>(dst);
    if (vectorOf(dst) == 8) {
        fillLcg<8>(p, n, seed, static_cast<hipStream_t>(stream));
    } else {
        fillLcg<1>(p, n, seed, static_cast<hipStream_t>(stream));
    }
    return (int)hipGetLastError();
}
