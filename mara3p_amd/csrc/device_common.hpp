// Device helpers shared by every kernel.  CDNA4 (gfx950), wave64.
//
// All HIP code is compiled with -ffp-contract=off: no FMA is formed unless it
// is written explicitly, so the FP64 kernels round exactly as the reference's
// x86-64 build and every face flux is bit-identical wherever it is computed
// (which keeps fluxes shared by two tiles conservative).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

namespace m3p {

constexpr int kWave = 64;

// std::max(a, b) == (a < b) ? b : a ; std::min(a, b) == (b < a) ? b : a
template<typename R> __device__ __forceinline__ R smax(R a, R b) { return (a < b) ? b : a; }
template<typename R> __device__ __forceinline__ R smin(R a, R b) { return (b < a) ? b : a; }

template<typename R> struct is_fp64 : std::is_same<R, double> {};

// Generalised-minmod PLM slope, src/scheme_plm_gradient.hpp:59-67 with
// coordinates (0, 1, 2).  The divisions by 1.0 and 2.0 there are exact, so
// they are written as the identical-valued forms below.
//
// The reference's 0.25 |sa + sb| (sa + sc) min(|a|, |b|, |c|) (s = sign) is
// sign(a) min|.| when a, b, c share a sign (the factors are 0.25 * 2 * 2,
// exact) and zero otherwise: the value of the median of (min(a, b, c),
// max(a, b, c), 0), which FP64 takes as max(min, min(max, 0)) -- the same
// number in every case (a zero may differ only in its sign, which no sum
// or product that follows can tell apart from the other zero's, since the
// face state adds it to a nonzero primitive or the product is zero anyway).
template<typename R>
__device__ __forceinline__ R plm(R yl, R y0, R yr, R theta)
{
    R a = (y0 - yl) * theta;
    R b = (yr - yl) * R(0.5);
    R c = (yr - y0) * theta;
    if constexpr (is_fp64<R>::value) {
        R mn = fmin(fmin(a, b), c), mx = fmax(fmax(a, b), c);
        return fmax(mn, fmin(mx, R(0)));
    } else {
        // Same value: non-zero only when a, b, c share a sign; then sign(a) * min|.|.
        R m = fminf(fminf(fabsf(a), fabsf(b)), fabsf(c));
        bool same = (signbit(a) == signbit(b)) && (signbit(a) == signbit(c));
        return same ? copysignf(m, a) : R(0);
    }
}

// Half the PLM slope, 0.5 * plm(...), used for the face states p -/+ 0.5 g:
// the factor one half goes into the three differences (exact), as the least
// of the halves is half the least.
template<typename R>
__device__ __forceinline__ R plm_half(R yl, R y0, R yr, R theta)
{
    R ht = R(0.5) * theta;
    R a = (y0 - yl) * ht;
    R b = (yr - yl) * R(0.25);
    R c = (yr - y0) * ht;
    if constexpr (is_fp64<R>::value) {
        R mn = fmin(fmin(a, b), c), mx = fmax(fmax(a, b), c);
        return fmax(mn, fmin(mx, R(0)));
    } else {
        // median of (min, max, 0): min if all are positive, max if all are
        // negative, 0 when the signs differ
        return __builtin_amdgcn_fmed3f(fminf(fminf(a, b), c), fmaxf(fmaxf(a, b), c), R(0));
    }
}

// Division / square root: IEEE for FP64 (parity), fast for FP32 (mixed).
template<typename R> __device__ __forceinline__ R fdiv(R a, R b)
{
    if constexpr (is_fp64<R>::value) return a / b;
    else return a * __builtin_amdgcn_rcpf(b);
}
template<typename R> __device__ __forceinline__ R frcp(R b)
{
    if constexpr (is_fp64<R>::value) return R(1) / b;
    else return __builtin_amdgcn_rcpf(b);
}
template<typename R> __device__ __forceinline__ R fsqrt(R a)
{
    if constexpr (is_fp64<R>::value) return sqrt(a);
    else return __builtin_amdgcn_sqrtf(a);
}

// FP64 reciprocal, reciprocal square root and square root from the
// hardware estimates (v_rcp_f64, v_rsq_f64) refined by two Newton steps each
// (quadratic convergence from the estimate's ~2^-22 to the last bit or two):
// a few ulp instead of IEEE rounding, at a third of the instructions of the
// IEEE division and square root sequences.  As they are, for the FP64 kernels
// whose bar against the reference is 1e-12 relative (minidisk, MHD); the kernels
// that equal it bit for bit take quotients and roots that correct the estimate
// by a remainder (Divisor, sqrt_ieee).
__device__ __forceinline__ double rcp_nr(double b)
{
    double r = __builtin_amdgcn_rcp(b);
    r = fma(r, fma(-b, r, 1.0), r);
    return fma(r, fma(-b, r, 1.0), r);
}
__device__ __forceinline__ double rsqrt_nr(double x)
{
    double y = __builtin_amdgcn_rsq(x);
    const double h = 0.5 * x;
    y = y * fma(-h * y, y, 1.5);
    return y * fma(-h * y, y, 1.5);
}
// sqrt(x) = x rsqrt(x) for finite x > 0; +-0, +inf and NaN as they are,
// NaN for x < 0 (the IEEE results; a select, since a branch here split the
// schedule of every wave speed)
__device__ __forceinline__ double sqrt_nr(double x)
{
    const double r = x * rsqrt_nr(x);
    return __builtin_amdgcn_class(x, 0x260) ? x : r;     // +-0 and +inf
}

// Quotients by one denominator: FP64 the IEEE quotient a / b, bit for bit.
// The steps are those of a correctly rounded division (reciprocal estimate,
// two Newton steps, quotient, one correction by its remainder; Markstein,
// IBM J. Res. Dev. 34, 1990), which the compiler's a / b repeats in full for
// every numerator with the scaling of extreme operands around them (11
// instructions and the wait before the last of them); here the reciprocal is
// taken once and a further quotient costs 5.  The remainder is formed 2^64
// larger, so it is exact for numerators down to 2^-1033 (and zero), and
// div_fixup gives zero, infinite and NaN operands their IEEE results.  The
// denominator must be a normal number below 2^958 in magnitude, zero,
// infinite or NaN, the numerator below 2^958 or infinite; a quotient that
// overflows comes out NaN, not infinite, and one by a subnormal denominator is
// not to be had from it.  FP64 Kelvin-Helmholtz step at 4096^2 (HLLC): 1.16
// to 1.10 ms; 256^2 in 32^2 blocks (HLLE): 23.7 to 21.6 us.
template<typename R> struct Divisor {
    R r;
    __device__ __forceinline__ explicit Divisor(R b) : r(frcp(b)) {}
    __device__ __forceinline__ R operator()(R a) const { return a * r; }
};
template<> struct Divisor<double> {
    double b, r, bs, rs;
    __device__ __forceinline__ explicit Divisor(double d) : b(d), r(rcp_nr(d))
    {
        bs = __builtin_ldexp(b, 64);
        rs = __builtin_ldexp(r, -64);
    }
    __device__ __forceinline__ double operator()(double a) const
    {
        const double q = a * r;
        const double rem = fma(-bs, q, __builtin_ldexp(a, 64));
        return __builtin_amdgcn_div_fixup(fma(rem, rs, q), b, a);
    }
};

// The same for every operand: IEEE's a / b outside the range above (operands of
// extreme size, quotients that overflow or come out subnormal).  For functions
// of arrays that hold anything; a stage kernel's recovery with it would pay a
// test and a branch per quotient.
struct WideDivisor {
    Divisor<double> by;
    bool usual;
    __device__ __forceinline__ explicit WideDivisor(double d) : by(d), usual(fabs(d) >= 0x1p-1022 && fabs(d) < 0x1p958) {}
    __device__ __forceinline__ double operator()(double a) const
    {
        const double q = by(a), m = fabs(a);
        const bool in = usual && m < 0x1p958 && (a == 0.0 || (m >= 0x1p-1033 && fabs(q) >= 0x1p-1022 && fabs(q) < __builtin_inf()));
        return in ? q : a / by.b;
    }
};

// The IEEE square root: the coupled iteration for g -> sqrt(x) and
// h -> 1 / (2 sqrt(x)) from one estimate of the reciprocal root, closed by two
// corrections of g by its remainder x - g g, the last of which rounds correctly
// (Markstein, IBM J. Res. Dev. 34, 1990).  Nothing is scaled, so the remainders
// must be normal numbers: the root is IEEE's bit for bit for x >= 2^-960; +-0,
// +inf, NaN and negative x as IEEE.  sqrt() scales every argument for the sake
// of those below 2^-767, five instructions on the chain from the sound speed
// to the flux (FP64 Kelvin-Helmholtz 4096^2, with the shared reciprocals: 1.16
// to 1.09 ms a step).
__device__ __forceinline__ double sqrt_ieee(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = y * 0.5;
    const double e = fma(-h, g, 0.5);
    h = fma(h, e, h);
    g = fma(g, e, g);
    g = fma(fma(-g, g, x), h, g);
    g = fma(fma(-g, g, x), h, g);
    return __builtin_amdgcn_class(x, 0x260) ? x : g;     // +-0 and +inf
}

// Error slot: err[0] = status code (first writer wins), err[1] = block, err[2] = zone.
__device__ __forceinline__ void report_error(int* err, int code, int block, int zone)
{
    if (err && atomicCAS(&err[0], 0, code) == 0) {
        err[1] = block;
        err[2] = zone;
    }
}

// Max of a non-negative double over a workgroup of NT threads (whole waves), then one atomic max into one of kRateSlots
// slots picked by the workgroup index (non-negative doubles order like their
// bit patterns; spreading the atomics keeps thousands of workgroups that end
// together from serialising on one address).  The atomic is skipped when the
// slot already holds at least the workgroup's maximum: slots only grow, so a
// stale read can only cost an atomic, never lose one, and a launch of tens
// of thousands of small workgroups does few atomics after its first ones.
// Every thread of the workgroup must call it.
constexpr int kRateSlots = 64;

__device__ __forceinline__ void slot_atomic_max(unsigned long long* slot, double m)
{
    const unsigned long long mb = (unsigned long long)__double_as_longlong(m);
    if (mb > __atomic_load_n(slot, __ATOMIC_RELAXED)) atomicMax(slot, mb);
}

template<int NT>
__device__ __forceinline__ void workgroup_atomic_max(double v, unsigned long long* slots)
{
    static_assert(NT % 64 == 0, "whole waves");
    unsigned long long* slot = slots + (blockIdx.x & (kRateSlots - 1));
    __shared__ double part[NT / 64];
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = part[0];
        for (int w = 1; w < NT / 64; ++w) m = fmax(m, part[w]);
        slot_atomic_max(slot, m);
    }
}

// Fill n words with v (clears reduction slots; a kernel, not a memset, so a
// captured graph replays it correctly).
static __global__ void fill_u64_kernel(unsigned long long* p, int n, unsigned long long v)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Wave64 reductions through DPP/permute shuffles.
__device__ __forceinline__ double wave_max(double v)
{
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, kWave));
    return v;
}
__device__ __forceinline__ double wave_sum(double v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

// The value of the lane before / after in the wave; the first / last lane
// takes `edge`.  Every lane must be active.
__device__ __forceinline__ float lane_before(float x, float edge)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(edge), __float_as_int(x), 0x138 /* wave_shr:1 */,
                                                      0xf, 0xf, false));
}
__device__ __forceinline__ float lane_after(float x, float edge)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(edge), __float_as_int(x), 0x130 /* wave_shl:1 */,
                                                      0xf, 0xf, false));
}
__device__ __forceinline__ double lane_before(double x, double edge)
{
    return __hiloint2double(__builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(x), 0x138, 0xf, 0xf, false),
                            __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(x), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ double lane_after(double x, double edge)
{
    return __hiloint2double(__builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(x), 0x130, 0xf, 0xf, false),
                            __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(x), 0x130, 0xf, 0xf, false));
}

// The same where the first / last lane's value is of no use (it is 0): the
// compiler can make the shift part of the instruction that takes the value
// (fused 1D step: 20 of 50 shifts, 3 to 4 % of the step).
__device__ __forceinline__ float lane_before(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ int lane_after(int x) { return __builtin_amdgcn_update_dpp(0, x, 0x130, 0xf, 0xf, true); }
__device__ __forceinline__ float lane_after(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ double lane_before(double x)
{
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x138, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ double lane_after(double x)
{
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x130, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x130, 0xf, 0xf, true));
}

// XCD-aware workgroup remap.  Workgroups are dispatched round-robin over the
// 8 XCDs (each with its own L2); give each XCD a contiguous range of logical
// tiles so that tiles sharing halo rows share an L2.
__device__ __forceinline__ int xcd_remap(int w, int total)
{
    constexpr int nxcd = 8;
    if (total % nxcd != 0) return w;
    return (w % nxcd) * (total / nxcd) + (w / nxcd);
}

// The same within each run of `chunk` workgroups (a multiple of 8; the
// workgroups after the last whole run stay): the XCDs advance through the
// runs together, each on its own contiguous part of the run.
__device__ __forceinline__ int xcd_remap_chunk(int w, int total, int chunk)
{
    const int first = w - w % chunk;
    return first + chunk <= total ? first + xcd_remap(w - first, chunk) : w;
}

} // namespace m3p
