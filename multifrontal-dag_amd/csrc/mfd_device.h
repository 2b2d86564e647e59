// Device helpers shared by the kernels (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace mfd {

namespace {

constexpr int kThreads = 256;

// ------------------------------------------------------------ MFMA traits
typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

// D(16x16) += A(16x4) B(4x16); lane l supplies A[l%16][l/16] and
// B[l/16][l%16].  The accumulator layouts differ (measured on gfx950):
//   f64: element v of lane l is D[l/16 + 4v][l%16]
//   f32: element v of lane l is D[4(l/16) + v][l%16]
template <typename T> struct Mfma;
template <> struct Mfma<double> {
    typedef d4 acc_t;
    static __device__ acc_t mma(double a, double b, acc_t c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
    static __device__ int row(int lane, int v) { return (lane >> 4) + 4 * v; }
};
template <> struct Mfma<float> {
    typedef f4 acc_t;
    static __device__ acc_t mma(float a, float b, acc_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    static __device__ int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

// 1 / sqrt(d): the hardware estimate r (v_rsq, good to about 2^-23) refined
// with e = 1 - d r^2: in double one third-order step r + r e (1/2 + 3/8 e),
// whose chain is two operations shorter than two Newton-Raphson steps, in
// float one Newton-Raphson step: within a few ulp of the exact value, where a
// correctly rounded sqrt and division take about twenty dependent steps.
__device__ __forceinline__ double rsqrt_nr(double d)
{
    const double r = __builtin_amdgcn_rsq(d), e = fma(-(d * r), r, 1.0);
    return fma(r * e, fma(0.375, e, 0.5), r);
}
__device__ __forceinline__ float rsqrt_nr(float d)
{
    const float r = __builtin_amdgcn_rsqf(d);
    const float e = fmaf(-(d * r), r, 1.0f);
    return fmaf(0.5f * r, e, r);
}
// Computes v here: left to itself the compiler puts the updates of a chain
// off until each value is needed and keeps every operand in registers till then.
template <typename T> __device__ __forceinline__ void pin(T& v) { asm volatile("" : "+v"(v)); }

// a / b given rb ~ 1 / b (within a few ulp): q = a rb, then one correction
// with the exact residual a - q b (Markstein), which returns a / b exactly
// whenever it is representable and is within an ulp of it otherwise.  Its
// chain is a multiply and two fmas after rb and b, against the ten
// dependent steps of a correctly rounded division.
template <typename T> __device__ __forceinline__ T quot(T a, T b, T rb)
{
    const T q = a * rb;
    return fma(fma(-q, b, a), rb, q);
}

// p[i] for a uniform base p and a 32-bit unsigned index: the address is
// base + zero-extended byte offset, which keeps one VGPR per address when
// many loads are in flight.
template <typename T> __device__ __forceinline__ T ld_off(const T* p, unsigned i)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + (size_t)(i * (unsigned)sizeof(T)));
}

// Value of v in lane src (uniform src; only its low 6 bits select the lane).
__device__ __forceinline__ double bcast(double v, int src)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, src);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), src);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ float bcast(float v, int src)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}

// Orders one wave's LDS accesses (they complete in issue order within a
// wave) against compiler reordering; no workgroup barrier is involved.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// sqrt(d) from r ~ 1/sqrt(d) (within a few ulp): s = d r and one Newton
// step s + (d - s^2) r / 2 with the exact residual (fma); exact whenever
// sqrt(d) is representable, within an ulp otherwise, in three dependent
// operations after r.
template <typename T> __device__ __forceinline__ T sqrt_from_rs(T d, T r)
{
    const T s = d * r;
    return fma(fma(-s, s, d), T(0.5) * r, s);
}

// ------------------------------- values passed between running workgroups
// Relaxed agent-scope accesses meet in memory common to the eight XCDs; a
// workgroup that raises a counter first waits for its stores (stores_done,
// then a barrier).
template <typename V> __device__ __forceinline__ V ld_agent(const V* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename V> __device__ __forceinline__ void st_agent(V* p, V v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int add_agent(int* p, int v)
{
    return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// One thread: polls counter p until it reaches target.  After as many polls as
// the word after stop says (kWaitPolls: about 6 s), or once another workgroup
// has done so, gives up: raises stop and *err (host memory), so that every
// wait of the launch ends.  SLOW: polls every 0.4 us at most.
template <bool SLOW = false> __device__ __forceinline__ void poll(const int* p, int target, int* stop, int* err)
{
    for (int spins = 0; ld_agent(p) < target;) {
        if (SLOW)
            __builtin_amdgcn_s_sleep(12);
        else
            __builtin_amdgcn_s_sleep(1);
        if ((++spins & 255) == 0 && (ld_agent(stop) != 0 || spins >= ld_agent(stop + 1))) {
            st_agent(stop, 1);
            __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            break;
        }
    }
}

// *p by scalar loads (uniform address, memory that no launch writes while
// this one runs).
template <typename S> __device__ __forceinline__ S ld_scalar(const S* p)
{
    typedef const __attribute__((address_space(4))) int* words;
    static_assert(sizeof(S) % 4 == 0, "copied in words");
    S v;
    words w = (words)(const void*)p;
#pragma unroll
    for (unsigned i = 0; i < sizeof(S) / 4; ++i) reinterpret_cast<int*>(&v)[i] = w[i];
    return v;
}

}  // namespace

}  // namespace mfd
