// cc1d_device.hpp -- device helpers shared by the gfx950 causal conv1d kernels.
//
// Storage types are tag structs around the raw bits so that every conversion
// is explicit: bf16/fp16 widen exactly to fp32 and narrow with one
// round-to-nearest-even conversion (v_cvt_pk_bf16_f32 / v_cvt_f16_f32 on
// gfx950). Rows move through HBM as 16-byte vectors (global_load_dwordx4).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cc1d_fastdiv.hpp"

namespace cc1d {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct f16 { uint16_t bits; };
struct bf16 { uint16_t bits; };

template <typename T> struct elems16 { static constexpr int value = 16 / (int)sizeof(T); };

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16 v) { return __uint_as_float((uint32_t)v.bits << 16); }
__device__ __forceinline__ float to_f32(f16 v) { return (float)__builtin_bit_cast(_Float16, v.bits); }

template <typename T> __device__ __forceinline__ T from_f32(float v);
template <> __device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16 from_f32<bf16>(float v) {
    return bf16{__builtin_bit_cast(uint16_t, (__bf16)v)};
}
template <> __device__ __forceinline__ f16 from_f32<f16>(float v) {
    return f16{__builtin_bit_cast(uint16_t, (_Float16)v)};
}

// Two fp32 values narrowed into one dword, a in the low half: one
// v_cvt_pk_bf16_f32 / v_cvt_pk_f16_f32 (RNE, the same rounding as from_f32).
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
template <typename T> __device__ __forceinline__ uint32_t pack2(float a, float b);
template <> __device__ __forceinline__ uint32_t pack2<bf16>(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
template <> __device__ __forceinline__ uint32_t pack2<f16>(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
}

// Round-trip through the storage dtype (what a store followed by a load gives).
template <typename T> __device__ __forceinline__ float round_to(float v) { return to_f32(from_f32<T>(v)); }

// Element e (compile-time after unrolling) of a 16-byte vector, widened to fp32.
template <typename T> __device__ __forceinline__ float vget(const u32x4& v, int e);
template <> __device__ __forceinline__ float vget<float>(const u32x4& v, int e) { return __uint_as_float(v[e]); }
template <> __device__ __forceinline__ float vget<bf16>(const u32x4& v, int e) {
    const uint32_t d = v[e >> 1];
    return (e & 1) ? __uint_as_float(d & 0xffff0000u) : __uint_as_float(d << 16);
}
template <> __device__ __forceinline__ float vget<f16>(const u32x4& v, int e) {
    const uint32_t d = v[e >> 1];
    const uint16_t h = (e & 1) ? (uint16_t)(d >> 16) : (uint16_t)(d & 0xffffu);
    return (float)__builtin_bit_cast(_Float16, h);
}

// Pack EPV fp32 values into one 16-byte vector of T (one RNE rounding each).
template <typename T> __device__ __forceinline__ u32x4 vpack(const float* f);
template <> __device__ __forceinline__ u32x4 vpack<float>(const float* f) {
    u32x4 r;
    r[0] = __float_as_uint(f[0]); r[1] = __float_as_uint(f[1]);
    r[2] = __float_as_uint(f[2]); r[3] = __float_as_uint(f[3]);
    return r;
}
template <> __device__ __forceinline__ u32x4 vpack<bf16>(const float* f) {
    u32x4 r;
#pragma unroll
    for (int d = 0; d < 4; ++d) r[d] = pack2<bf16>(f[2 * d], f[2 * d + 1]);
    return r;
}
template <> __device__ __forceinline__ u32x4 vpack<f16>(const float* f) {
    u32x4 r;
#pragma unroll
    for (int d = 0; d < 4; ++d) r[d] = pack2<f16>(f[2 * d], f[2 * d + 1]);
    return r;
}

__device__ __forceinline__ u32x4 vzero() { u32x4 z = {0u, 0u, 0u, 0u}; return z; }

template <typename T> __device__ __forceinline__ u32x4 vload(const T* p) {
    return *reinterpret_cast<const u32x4*>(p);
}
template <typename T> __device__ __forceinline__ void vstore(T* p, const u32x4& v) {
    *reinterpret_cast<u32x4*>(p) = v;
}

// Streaming (non-temporal) 16-byte accesses for data touched exactly once:
// global_load/store_dwordx4 ... nt, so the stream does not displace reused
// lines (weights, seq_idx, halos) from L2 / the Infinity Cache.
template <typename T> __device__ __forceinline__ u32x4 vload_nt(const T* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}
template <typename T> __device__ __forceinline__ void vstore_nt(T* p, const u32x4& v) {
    __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(p));
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// The same 16-byte accesses at any element boundary. The hardware takes a
// dwordx4 at any 2-byte address (the HSA ABI turns unaligned access on), in
// one instruction: copying 20480 rows of 4 KB takes 27.6 us from and to
// aligned addresses, 29.4 with the loads one bf16 off, 30.0 with the stores,
// 31.3 with both, and 30.1 with rows of 2041 elements (every offset occurs).
template <int BYTES> struct AnyAddr;  // dword types at element boundaries
template <> struct AnyAddr<2> {
    typedef u32x4 __attribute__((aligned(2))) v4;
    typedef u32x2 __attribute__((aligned(2))) v2;
    typedef uint32_t __attribute__((aligned(2))) v1;
};
template <> struct AnyAddr<4> {
    typedef u32x4 __attribute__((aligned(4))) v4;
    typedef u32x2 __attribute__((aligned(4))) v2;
    typedef uint32_t v1;
};
template <typename T> __device__ __forceinline__ u32x4 vload_any(const T* p) {
    return *reinterpret_cast<const typename AnyAddr<sizeof(T)>::v4*>(p);
}
template <typename T> __device__ __forceinline__ u32x4 vload_any_nt(const T* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const typename AnyAddr<sizeof(T)>::v4*>(p));
}
template <typename T> __device__ __forceinline__ void vstore_any_nt(T* p, const u32x4& v) {
    __builtin_nontemporal_store(v, reinterpret_cast<typename AnyAddr<sizeof(T)>::v4*>(p));
}

// The first rem (1 .. EPV - 1, the same for every lane) elements of a 16-byte
// vector at p: a row's last ones, where reading the whole vector would leave
// the row. Read as at most one access each of 8, 4 and 2 bytes; load() only
// issues them, vec() waits and puts them in place (zero from rem on), so a
// kernel can issue its other loads in between.
template <typename T> struct RowTail {
    u32x2 a;
    uint32_t b, c;
    __device__ __forceinline__ void load(const T* p, int rem) {
        typedef typename AnyAddr<sizeof(T)>::v2 any2;
        typedef typename AnyAddr<sizeof(T)>::v1 any1;
        constexpr int PER = 4 / (int)sizeof(T);  // elements per dword
        a = u32x2{0u, 0u};
        b = c = 0u;
        if (rem & (2 * PER)) a = *reinterpret_cast<const any2*>(p);
        if (rem & PER) b = *reinterpret_cast<const any1*>(p + (rem & (2 * PER)));
        if constexpr (PER == 2) {
            if (rem & 1) c = *reinterpret_cast<const uint16_t*>(p + (rem & 6));
        }
    }
    __device__ __forceinline__ u32x4 vec(int rem) const {
        constexpr int PER = 4 / (int)sizeof(T);
        const bool two = (rem & (2 * PER)) != 0, one = (rem & PER) != 0;
        u32x4 r;
        r[0] = two ? a[0] : (one ? b : c);
        r[1] = two ? a[1] : (one ? c : 0u);
        r[2] = two ? (one ? b : c) : 0u;
        r[3] = two && one ? c : 0u;
        return r;
    }
    // the first rem elements of v to p
    static __device__ __forceinline__ void store(T* p, const u32x4& v, int rem) {
        typedef typename AnyAddr<sizeof(T)>::v2 any2;
        typedef typename AnyAddr<sizeof(T)>::v1 any1;
        constexpr int PER = 4 / (int)sizeof(T);
        const bool two = (rem & (2 * PER)) != 0, one = (rem & PER) != 0;
        if (two) *reinterpret_cast<any2*>(p) = u32x2{v[0], v[1]};
        if (one) *reinterpret_cast<any1*>(p + (rem & (2 * PER))) = two ? v[2] : v[0];
        if constexpr (PER == 2) {
            if (rem & 1) *reinterpret_cast<uint16_t*>(p + (rem & 6)) = (uint16_t)(two ? (one ? v[3] : v[2]) : (one ? v[1] : v[0]));
        }
    }
};

// The elements of T in one dword (2 of 16 bits, 1 fp32): a lane's adjacent
// channels in the channel-last kernels, accessed at any element boundary
// (rows of an odd number of 16-bit channels start at odd ones). Element
// indices are compile-time after unrolling.
template <typename T> struct Lanes {
    static constexpr int N = 4 / (int)sizeof(T);
    typedef typename AnyAddr<sizeof(T)>::v1 dword;
    uint32_t d;

    __device__ __forceinline__ void zero() { d = 0u; }
    template <bool NT> __device__ __forceinline__ void load(const T* p) {
        d = NT ? __builtin_nontemporal_load(reinterpret_cast<const dword*>(p)) : *reinterpret_cast<const dword*>(p);
    }
    template <bool NT> __device__ __forceinline__ void store(T* p) const {
        if (NT) __builtin_nontemporal_store(d, reinterpret_cast<dword*>(p));
        else *reinterpret_cast<dword*>(p) = d;
    }
    __device__ __forceinline__ float get(int e) const {
        if constexpr (sizeof(T) == 4) return __uint_as_float(d);
        else if constexpr (__is_same(T, bf16)) return (e & 1) ? __uint_as_float(d & 0xffff0000u) : __uint_as_float(d << 16);
        else return (float)__builtin_bit_cast(_Float16, (e & 1) ? (uint16_t)(d >> 16) : (uint16_t)(d & 0xffffu));
    }
    __device__ __forceinline__ void set(const float* f) {
        if constexpr (sizeof(T) == 4) d = __float_as_uint(f[0]);
        else d = pack2<T>(f[0], f[1]);
    }
};

template <typename T> __device__ __forceinline__ float ld(const T* p, int64_t i) { return to_f32(p[i]); }

// Reads of wave-uniform addresses through the scalar data cache (constant
// address space): for data that no wavefront writes during the kernel, such
// as weights, bias and halo vectors of read-only inputs. Their completion is
// tracked by lgkmcnt, so waiting for them never waits for the wavefront's
// outstanding vector-memory reads.
typedef const __attribute__((address_space(4))) uint32_t* const_u32_ptr;
typedef const __attribute__((address_space(4))) u32x4* const_u32x4_ptr;

// Element at p (wave-uniform), widened to fp32: reads the aligned dword holding it.
template <typename T> __device__ __forceinline__ float ld_uniform(const T* p) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(p);
    const uint32_t d = *(const_u32_ptr)(a & ~(uintptr_t)3);
    if constexpr (sizeof(T) == 4) {
        return __uint_as_float(d);
    } else {
        const uint16_t h = (a & 2) ? (uint16_t)(d >> 16) : (uint16_t)(d & 0xffffu);
        return to_f32(T{h});
    }
}
__device__ __forceinline__ int32_t ld_uniform(const int32_t* p) {
    return (int32_t)*(const_u32_ptr)reinterpret_cast<uintptr_t>(p);
}
// 16-byte vector at the wave-uniform, 16-byte aligned address p.
template <typename T> __device__ __forceinline__ u32x4 vload_uniform(const T* p) {
    return *(const_u32x4_ptr)reinterpret_cast<uintptr_t>(p);
}
template <typename T> __device__ __forceinline__ void st(T* p, int64_t i, float v) { p[i] = from_f32<T>(v); }

// Dword d of a 16-byte vector of T: the bits of its elements e < n (all of
// them for n >= EPV, none for n <= 0).
template <typename T> __device__ __forceinline__ uint32_t lead_mask(int d, int32_t n) {
    if constexpr (sizeof(T) == 4) return d < n ? ~0u : 0u;
    else return 2 * d + 1 < n ? ~0u : (2 * d < n ? 0xffffu : 0u);
}
// Store element e of the packed vector v at p (its raw bits: no rounding).
template <typename T> __device__ __forceinline__ void st_elem(T* p, const u32x4& v, int e) {
    if constexpr (sizeof(T) == 4) *reinterpret_cast<uint32_t*>(p) = v[e];
    else *reinterpret_cast<uint16_t*>(p) = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
}
// Elements m .. EPV - 1 (m > 0, the same for every lane) of v to p + m ..
template <typename T> __device__ __forceinline__ void store_from(T* p, const u32x4& v, int m) {
#pragma unroll
    for (int e = 1; e < elems16<T>::value; ++e) {
        if (e >= m) st_elem<T>(p + e, v, e);
    }
}
// Storage bits of an fp32 value that T represents exactly.
template <typename T> __device__ __forceinline__ uint32_t tbits(float v) {
    if constexpr (sizeof(T) == 4) return __float_as_uint(v);
    else return from_f32<T>(v).bits;
}

// a[k] for a runtime k (0 outside [0, N)), as a chain of selects: a register
// array indexed at run time would be placed in scratch memory
template <int N> __device__ __forceinline__ float pick(const float* a, int k) {
    float r = 0.0f;
#pragma unroll
    for (int i = 0; i < N; ++i) r = (i == k) ? a[i] : r;
    return r;
}

// How a wavefront of the row kernels takes rows whose time stride is one.
//   kRowsAligned  one row, on 16-byte boundaries, whole vectors long
//   kRowsAlike    one row of any start and length that lies alike in every
//                 tensor modulo 16 bytes: vectors count from the boundary at
//                 or before the row's first element, so every access is
//                 aligned (a vector that holds one of the row's elements is in
//                 the same memory page, so reading it whole is safe)
//   kRowsAny      one row of any start and length, wherever it lies in each
//                 tensor: unaligned vectors from its first element on
//   kRowsShort    several rows of at most 32 vectors, read as in kRowsAny, one
//                 vector per lane: the row and all that belongs to it differ
//                 from lane to lane
enum RowsMode { kRowsAligned = 0, kRowsAlike = 1, kRowsAny = 2, kRowsShort = 3 };
constexpr int64_t kShortVecs = 32;  // vectors of the longest row of kRowsShort

// Wavefront-uniform value (lets the compiler keep it in an SGPR).
__device__ __forceinline__ uint32_t uniform32(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float uniform_f32(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ __forceinline__ int64_t uniform(int64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)(uint64_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}
// A per-lane value the compiler can neither see through nor move: address
// arithmetic of a rarely taken branch that uses it stays inside the branch
// instead of being hoisted out of the loop around it (where it would hold
// registers for the whole loop).
__device__ __forceinline__ int32_t opaque(int32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}

// The ids of the N (4 or 8) row positions from p on, at any 4-byte address.
template <int N> __device__ __forceinline__ void ids_any(const int32_t* p, int32_t* id) {
#pragma unroll
    for (int q = 0; q < N / 4; ++q) {
        const u32x4 s = *reinterpret_cast<const AnyAddr<4>::v4*>(p + 4 * q);
#pragma unroll
        for (int r = 0; r < 4; ++r) id[4 * q + r] = (int32_t)s[r];
    }
}
// ids from .. to - 1 (the same range for every lane) of the N from p on,
// element by element; the others keep what id holds.
template <int N> __device__ __forceinline__ void ids_some(const int32_t* p, int from, int to, int32_t* id) {
#pragma unroll
    for (int e = 0; e < N; ++e)
        if (e >= from && e < to) id[e] = p[e];
}

// SiLU = x * sigmoid(x), as x * rcp(1 + exp(-x)) in fp32.
__device__ __forceinline__ float silu(float x) {
    return x * __builtin_amdgcn_rcpf(1.0f + __expf(-x));
}

// d silu / d x = s * (1 + x * (1 - s)), s = sigmoid(x).
__device__ __forceinline__ float silu_grad(float x) {
    const float s = __builtin_amdgcn_rcpf(1.0f + __expf(-x));
    return s * (1.0f + x * (1.0f - s));
}

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// g * silu'(p) given q = -log2(e) * p (so exp(-p) = exp2(q)):
//   s = 1 / (1 + exp2(q));  g * s * (1 + p * (1 - s)) = gs + (gs * q) * (-ln2 * (1 - s))
// Five VALU operations plus exp2 and rcp.
__device__ __forceinline__ float silu_bwd_q(float g, float q) {
    const float s = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(q));
    const float gs = g * s;
    return __builtin_fmaf(gs * q, __builtin_fmaf(s, kLn2, -kLn2), gs);
}

// Causal taps: bias + sum_k w[k] * win[k], fp32 fma in k order. The forward
// and the decode update both use this, so a decode loop reproduces the full
// forward bit for bit.
template <int W>
__device__ __forceinline__ float conv_taps(float bias, const float* w, const float* win) {
    float acc = bias;
#pragma unroll
    for (int k = 0; k < W; ++k) acc = __builtin_fmaf(w[k], win[k], acc);
    return acc;
}

// As conv_taps, keeping tap k only when ids[k] equals the current id ids[W-1].
template <int W>
__device__ __forceinline__ float conv_taps_gated(float bias, const float* w, const float* win,
                                                 const int32_t* ids) {
    float acc = bias;
    const int32_t cur = ids[W - 1];
#pragma unroll
    for (int k = 0; k < W; ++k)
        if (ids[k] == cur) acc = __builtin_fmaf(w[k], win[k], acc);
    return acc;
}

// Value of `v` held by lane `src` of this wavefront (ds_bpermute_b32).
__device__ __forceinline__ uint32_t lane_get(uint32_t v, int src) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute(src << 2, (int)v);
}
__device__ __forceinline__ float lane_get(float v, int src) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(src << 2, __float_as_int(v)));
}
__device__ __forceinline__ int32_t lane_get(int32_t v, int src) {
    return __builtin_amdgcn_ds_bpermute(src << 2, v);
}

// Between LDS writes and reads of one wavefront's lanes: what any lane wrote
// before is what every lane reads after. A wavefront's LDS accesses complete in
// order, so the fences cost no instruction; they keep the compiler, to which the
// lanes are separate threads, from moving or forwarding an access across (a wave
// barrier alone orders no memory).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// DPP controls (GFX9 encoding) for the wavefront reduction below.
constexpr int kDppQuadSwap1 = 0xb1;   // quad_perm [1, 0, 3, 2]
constexpr int kDppQuadSwap2 = 0x4e;   // quad_perm [2, 3, 0, 1]
constexpr int kDppRowRor4 = 0x124;    // row_ror:4 (rotate within 16 lanes)
constexpr int kDppRowRor8 = 0x128;    // row_ror:8
constexpr int kDppRowBcast15 = 0x142; // row_bcast:15 (lane 15 of a row into the next row)
constexpr int kDppRowBcast31 = 0x143; // row_bcast:31 (lane 31 into rows 2 and 3)

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_f32(float v) {
    // rows outside ROW_MASK receive 0 (the `old` operand), so `v + dpp` leaves them unchanged
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xf, false));
}

// Sum over the 64 lanes of a wavefront, returned wave-uniform (every lane
// receives it). Cross-lane moves are DPP modifiers on VALU adds -- no LDS
// round trips: sums within quads, then rows of 16, then rows 0+1 and 2+3 into
// rows 1 and 3, then rows 0+1 into rows 2 and 3; lane 63 holds the total.
// All 64 lanes must be active.
__device__ __forceinline__ float wave_sum(float v) {
    v += dpp_f32<kDppQuadSwap1, 0xf>(v);
    v += dpp_f32<kDppQuadSwap2, 0xf>(v);
    v += dpp_f32<kDppRowRor4, 0xf>(v);
    v += dpp_f32<kDppRowRor8, 0xf>(v);
    v += dpp_f32<kDppRowBcast15, 0xa>(v);
    v += dpp_f32<kDppRowBcast31, 0xc>(v);
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

}  // namespace cc1d
