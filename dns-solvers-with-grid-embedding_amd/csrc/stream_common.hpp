// stream_common.hpp -- device helpers shared by the collide-stream kernels
// (k_stream.hip) and the two-substep band kernel (k_band2.hip): the compute type
// of each storage type, the collision dispatch, row-wise access through buffer
// resources and the fused-reduction sums.
#pragma once
#include "internal.hpp"
#include "lattice.hpp"

namespace dnsg {

template <class S>
struct ComputeOf {
    using T = float;
};
template <>
struct ComputeOf<double> {
    using T = double;
};

__device__ __forceinline__ PreSums<double> collide_any(double *f, double G, double om) { return collide64(f, G, om); }
__device__ __forceinline__ PreSums<float> collide_any(float *f, float G, float om) { return collide32(f, G, om); }

// Row-wise access through buffer resources: the base of a layer and the row and
// direction offset are scalars, so a lane holds one 32-bit offset for all 19 directions
// (as 64-bit addresses, 19 loads or stores in flight take 38 VGPRs), and a lane that
// must not store takes the offset DROP, which lies past every resource and is dropped
// by the resource's bounds check, so that stores need no branches.  A resource, a row or
// a layer, must be below 2 GiB.
constexpr unsigned DROP = 0x80000000u;
typedef __amdgpu_buffer_rsrc_t Rsrc;
typedef unsigned u2v __attribute__((ext_vector_type(2)));
// p and bytes must be the same over the wave (they are made scalars: without that, where
// the compiler cannot prove it, each access becomes a loop over the wave's values)
__device__ __forceinline__ Rsrc buf_rsrc(const void *p, unsigned bytes) {
    const unsigned long long a = reinterpret_cast<unsigned long long>(p);
    const unsigned lo = __builtin_amdgcn_readfirstlane((int)(unsigned)a), hi = __builtin_amdgcn_readfirstlane((int)(a >> 32));
    void *u = reinterpret_cast<void *>((unsigned long long)hi << 32 | lo);
    return __builtin_amdgcn_make_buffer_rsrc(u, 0, __builtin_amdgcn_readfirstlane((int)bytes), 0x00027000);
}
// loads: v the lane's byte offset, s the scalar one; the pointer names the storage type
__device__ __forceinline__ double buf_load(Rsrc R, unsigned v, unsigned s, const double *) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(R, v, s, 0));
}
__device__ __forceinline__ float buf_load(Rsrc R, unsigned v, unsigned s, const float *) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(R, v, s, 0));
}
__device__ __forceinline__ float buf_load(Rsrc R, unsigned v, unsigned s, const __half *) {
    const unsigned short a = __builtin_amdgcn_raw_buffer_load_b16(R, v, s, 0);
    return __half2float(__builtin_bit_cast(__half, a));
}
__device__ __forceinline__ void buf_load_pair(Rsrc R, unsigned v, unsigned s, const float *, float &a, float &b) {
    const u2v d = __builtin_amdgcn_raw_buffer_load_b64(R, v, s, 0);
    a = __uint_as_float(d.x);
    b = __uint_as_float(d.y);
}
__device__ __forceinline__ void buf_load_pair(Rsrc R, unsigned v, unsigned s, const __half *, float &a, float &b) {
    const __half2 d = __builtin_bit_cast(__half2, __builtin_amdgcn_raw_buffer_load_b32(R, v, s, 0));
    a = __low2float(d);
    b = __high2float(d);
}
// stores; AUX 2: non-temporal.  At most 8 bytes a lane: 16-byte buffer stores of FP64
// pairs wrote sporadically wrong values here (the data registers can be rewritten before
// a store of more than 8 bytes has read them, which the compiler does not guard where
// the scalar offset is a register).
template <int AUX>
__device__ __forceinline__ void buf_store(Rsrc R, unsigned v, unsigned s, const double *, double a) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2v, a), R, v, s, AUX);
}
template <int AUX>
__device__ __forceinline__ void buf_store(Rsrc R, unsigned v, unsigned s, const float *, float a) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(a), R, v, s, AUX);
}
template <int AUX>
__device__ __forceinline__ void buf_store(Rsrc R, unsigned v, unsigned s, const __half *, float a) {
    __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, __float2half(a)), R, v, s, AUX);
}
template <int AUX>
__device__ __forceinline__ void buf_store_pair(Rsrc R, unsigned v, unsigned s, const float *, float a, float b) {
    asm("" : "+v"(a));  // else the compiler reads the pair as 8 bytes of the array holding a, which keeps it in memory
    u2v d;
    d.x = __float_as_uint(a);
    d.y = __float_as_uint(b);
    __builtin_amdgcn_raw_buffer_store_b64(d, R, v, s, AUX);
}
template <int AUX>
__device__ __forceinline__ void buf_store_pair(Rsrc R, unsigned v, unsigned s, const __half *, float a, float b) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, __halves2half2(__float2half(a), __float2half(b))), R, v, s, AUX);
}

__device__ __forceinline__ double wave_sum64(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

// Workgroups are dispatched round-robin over the 8 XCDs; remap the linear block
// id so that each XCD gets one contiguous range of (row, chunk) pairs.  The
// neighbouring chunks of a row, whose e_x-shifted writes share cache lines,
// then meet in the same L2.
__device__ __forceinline__ int xcd_remap(int b, int nb) {
    const int per = nb >> 3;
    return (b < (per << 3)) ? (b & 7) * per + (b >> 3) : b;
}

// density and u_x of a node from its collision's moments, in FP64 in every tier
__device__ __forceinline__ double pre_rho(const PreSums<double> &p) { return p.zeroth; }
__device__ __forceinline__ double pre_rho(const PreSums<float> &p) { return 1. + (double)p.zeroth; }
__device__ __forceinline__ double pre_u(const PreSums<double> &p) { return p.u0; }
__device__ __forceinline__ double pre_u(const PreSums<float> &p) { return (double)p.mx / pre_rho(p); }

// fused-reduction sums of one thread's nodes: pre-collision moments (rho, mom, u)
// and the destination-weighted sums of what it writes (dm, dd)
struct RowSums {
    double rho = 0., mom = 0., u = 0., dm = 0., dd = 0.;
    template <class S, class T>
    __device__ __forceinline__ void add(const PreSums<T> &p) {
        rho += pre_rho(p);
        mom += (double)p.mx;
        u += pre_u(p);
    }
};

// encalc2 weight of a destination layer (LatArgs::dsum)
__device__ __forceinline__ double dest_w(const LatArgs &L, int zt) {
    return (zt < L.klo || zt > L.khi) ? 0. : (zt == L.khalf ? 0.5 * L.kscale : L.kscale);
}
// a layer's part of those sums; nothing from a layer of weight 0, also where its sum is
// not finite (0 x NaN would reach the force)
__device__ __forceinline__ double weighted(double w, double sum) { return w != 0. ? w * sum : 0.; }

}  // namespace dnsg
