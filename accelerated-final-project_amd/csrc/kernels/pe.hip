// Positional-encoding pre-pass (gfx950): out[row] = PE(in[row]) with position
// row % seq_len, over one tensor (atn_pe_apply_ex) or two at once (Q and K of
// the "separate" pipelines).
//
// Pure copy traffic, so bytes in flight and idle lanes decide.  k_pe_rows
// numbers the 4-dim groups of all rows through and gives every thread U of
// them, 256 apart, with the loads of all U issued before any arithmetic:
// every lane works whatever head_d is (a workgroup per row, as k_pe_apply
// below, uses 32 of 256 lanes at head_d 128).  fp32 (4,32,512,128) with the
// caller's duplicated caches, Q and K (67 MB in, 67 MB out): two launches of
// 41.7 us -> one of 30.9 us (1.6 -> 4.35 TB/s; a large copy reaches 4.7), and
// the "separate" RoPE call at that shape 152 -> 102 us.
#include <algorithm>

#include "common.hpp"
#include "launch.hpp"
#include "split16.hpp"

namespace atn {

namespace {

// x / d and x % d for x < 2^16 + d by a host-made multiplier (d < 2^15), or,
// for d >= 2^15, by one compare (there x < 2 d)
struct SmallDiv {
    unsigned d, mul;  // mul = ceil(2^32 / d), 0: the compare form
    __device__ __forceinline__ unsigned div(unsigned x) const {
        return mul ? __umulhi(x, mul) : (x >= d ? 1u : 0u);
    }
};
SmallDiv small_div(long d) {
    SmallDiv s;
    s.d = (unsigned)d;
    // ceil(2^32 / d) times x, >> 32, is x / d while x d < 2^32; d = 1 has no
    // 32-bit multiplier and is taken apart by the kernel
    s.mul = d < (1 << 15) ? (unsigned)((((uint64_t)1 << 32) + d - 1) / d) : 0u;
    return s;
}

struct PeSeg {
    const void* in;
    void* out;
    long units;    // groups in all rows
    int seq_len;
    SmallDiv pos;  // by seq_len
    PeSide pe;
};

struct PeRowsArgs {
    PeSeg seg[2];
    unsigned blocks0;  // workgroups of seg[0]
    int D;
    int upr;           // units per row
    SmallDiv row;      // by upr
};

// A unit: 4 dims of a row (8 for rotate-half: a group below half the rotary
// width and its partner group, so that the two are read once and an in-place
// call reads both before it writes either).  Rotate-half rows hold rotary / 8
// pair units, then (D - rotary) / 4 plain ones.
template <typename T, typename TO, int PEK, bool DUP, int U>
__global__ __launch_bounds__(256) void k_pe_rows(PeRowsArgs a) {
    const bool second = blockIdx.x >= a.blocks0;
    const PeSeg& g = a.seg[second ? 1 : 0];
    const long base = (long)(blockIdx.x - (second ? a.blocks0 : 0)) * (256 * U);
    const long row0 = base / a.upr;
    const unsigned c0 = (unsigned)(base - row0 * a.upr), p0 = (unsigned)(row0 % g.seq_len);
    const T* in = static_cast<const T*>(g.in);
    TO* out = static_cast<TO*>(g.out);
    const int D = a.D, rot = g.pe.rotary, h = rot >> 1, ld = g.pe.ld;
    constexpr bool kHalf = PEK == kPeRopeHalf;

    float4 x[U], y[U], c[U], s[U];
    const T* src[U];
    int d[U];
    bool on[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const unsigned i = threadIdx.x + 256u * u;
        on[u] = base + i < g.units;
        const unsigned k = on[u] ? c0 + i : c0;
        const unsigned dr = a.upr == 1 ? k : a.row.div(k);
        const unsigned unit = k - dr * (unsigned)a.upr;
        const unsigned p = p0 + dr;
        const int pos = g.seq_len == 1 ? 0 : (int)(p - g.pos.div(p) * g.pos.d);
        src[u] = in + (size_t)(row0 + dr) * D;
        bool enc = true;
        if constexpr (kHalf) {
            enc = (int)unit < (rot >> 3);
            d[u] = enc ? (int)unit * 4 : rot + ((int)unit - (rot >> 3)) * 4;
            x[u] = Elem<T>::ld4(src[u], d[u]);
            y[u] = Elem<T>::ld4(src[u], enc ? d[u] + h : d[u]);
        } else {
            d[u] = (int)unit * 4;
            enc = PEK == kPeSinusoidal || d[u] < rot;
            x[u] = Elem<T>::ld4(src[u], d[u]);
        }
        // the angles (groups past the rotary width read a valid, unused one)
        const int e = enc ? d[u] : 0;
        if constexpr (PEK == kPeSinusoidal) {
            if constexpr (DUP) {
                const float4 sn = *reinterpret_cast<const float4*>(g.pe.a + (size_t)pos * ld + e);
                const float4 cs = *reinterpret_cast<const float4*>(g.pe.b + (size_t)pos * ld + e);
                c[u] = make_float4(sn.x, cs.y, sn.z, cs.w);
            } else {
                const size_t t = (size_t)pos * ld + (e >> 1);
                const float2 sn = *reinterpret_cast<const float2*>(g.pe.a + t);
                const float2 cs = *reinterpret_cast<const float2*>(g.pe.b + t);
                c[u] = make_float4(sn.x, cs.x, sn.y, cs.y);
            }
        } else if constexpr (kHalf) {
            if constexpr (DUP) {
                const float* pc = g.pe.a + (size_t)pos * ld + 2 * e;
                const float* ps = g.pe.b + (size_t)pos * ld + 2 * e;
                const float4 ca = *reinterpret_cast<const float4*>(pc);
                const float4 cb = *reinterpret_cast<const float4*>(pc + 4);
                const float4 sa = *reinterpret_cast<const float4*>(ps);
                const float4 sb = *reinterpret_cast<const float4*>(ps + 4);
                c[u] = make_float4(ca.x, ca.z, cb.x, cb.z);
                s[u] = make_float4(sa.x, sa.z, sb.x, sb.z);
            } else {
                c[u] = *reinterpret_cast<const float4*>(g.pe.a + (size_t)pos * ld + e);
                s[u] = *reinterpret_cast<const float4*>(g.pe.b + (size_t)pos * ld + e);
            }
        } else {
            if constexpr (DUP) {
                const float4 cs = *reinterpret_cast<const float4*>(g.pe.a + (size_t)pos * ld + e);
                const float4 sn = *reinterpret_cast<const float4*>(g.pe.b + (size_t)pos * ld + e);
                c[u] = make_float4(cs.x, sn.x, cs.z, sn.z);
            } else {
                const size_t t = (size_t)pos * ld + (e >> 1);
                const float2 cs = *reinterpret_cast<const float2*>(g.pe.a + t);
                const float2 sn = *reinterpret_cast<const float2*>(g.pe.b + t);
                c[u] = make_float4(cs.x, sn.x, cs.y, sn.y);
            }
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (!on[u]) continue;
        TO* dst = out + (src[u] - in);
        const float4 v = x[u];
        if (!g.pe.on) {  // widened or copied only
            Elem<TO>::st4(dst, d[u], v);
            if (kHalf && d[u] < h) Elem<TO>::st4(dst, d[u] + h, y[u]);
        } else if constexpr (PEK == kPeSinusoidal) {
            Elem<TO>::st4(dst, d[u], make_float4(v.x + c[u].x, v.y + c[u].y, v.z + c[u].z,
                                                v.w + c[u].w));
        } else if constexpr (kHalf) {
            if (d[u] < h) {
                const float4 w = y[u];
                Elem<TO>::st4(dst, d[u],
                             make_float4(rot_first(v.x, w.x, c[u].x, s[u].x),
                                         rot_first(v.y, w.y, c[u].y, s[u].y),
                                         rot_first(v.z, w.z, c[u].z, s[u].z),
                                         rot_first(v.w, w.w, c[u].w, s[u].w)));
                Elem<TO>::st4(dst, d[u] + h,
                             make_float4(rot_second(v.x, w.x, c[u].x, s[u].x),
                                         rot_second(v.y, w.y, c[u].y, s[u].y),
                                         rot_second(v.z, w.z, c[u].z, s[u].z),
                                         rot_second(v.w, w.w, c[u].w, s[u].w)));
            } else {
                Elem<TO>::st4(dst, d[u], v);
            }
        } else {
            Elem<TO>::st4(dst, d[u],
                         d[u] < rot ? make_float4(rot_first(v.x, v.y, c[u].x, c[u].y),
                                                  rot_second(v.x, v.y, c[u].x, c[u].y),
                                                  rot_first(v.z, v.w, c[u].z, c[u].w),
                                                  rot_second(v.z, v.w, c[u].z, c[u].w))
                                    : v);
        }
    }
}

// Any head_d, rotary width, alignment and table: a workgroup per row.
template <typename T, typename TO, int PEK>
__global__ __launch_bounds__(256) void k_pe_apply(const T* __restrict__ in, TO* __restrict__ out,
                                                   long n_rows, int seq_len, int D, PeSide pe,
                                                   int vec_ok) {
    const bool vec = vec_ok != 0;
    for (long row = blockIdx.x; row < n_rows; row += gridDim.x) {
        const int pos = (int)(row % seq_len);
        const T* xr = in + (size_t)row * D;
        TO* yr = out + (size_t)row * D;
        for (int d = threadIdx.x * 4; d < D; d += 256 * 4) {
            const float4 v = load_row4_pe<T, PEK>(xr, pos, d, D, pe, vec);
            if (vec && d + 3 < D) {
                Elem<TO>::st4(yr, d, v);
            } else {
                const float vv[4] = {v.x, v.y, v.z, v.w};
                for (int c = 0; c < 4 && d + c < D; ++c) Elem<TO>::st(yr, d + c, vv[c]);
            }
        }
    }
}

// Whether k_pe_rows takes this call: whole 4-dim groups whose angles are
// whole vectors of the tables (16-byte aligned tables and rows where the
// caller brings them), and unit counts that a grid holds.
bool rows_ok(int pek, int D, const PeSide& pe, int vec_ok) {
    if (!vec_ok || D % 4 != 0 || D >= (1 << 30)) return false;
    const bool a16 = ((uintptr_t)pe.a % 16) == 0 && ((uintptr_t)pe.b % 16) == 0;
    if (!a16) return false;
    if (pek == kPeRopeInterleaved) return pe.rotary % 4 == 0 && pe.ld % (pe.dup ? 4 : 2) == 0;
    if (pek == kPeRopeHalf) return pe.rotary % 8 == 0 && pe.ld % 4 == 0;
    return pe.ld % (pe.dup ? 4 : 2) == 0;
}

template <typename T, typename TO, int PEK, bool DUP>
void run_rows(const PeRowsArgs& a, unsigned blocks, hipStream_t st) {
    hipLaunchKernelGGL((k_pe_rows<T, TO, PEK, DUP, PEK == kPeRopeHalf ? 2 : 4>), dim3(blocks),
                       dim3(256), 0, st, a);
}

template <typename T, typename TO>
hipError_t pe_rows_t(int pek, const PeTensor* t, int n, int D, hipStream_t st) {
    const int U = pek == kPeRopeHalf ? 2 : 4;
    PeRowsArgs a{};
    a.D = D;
    a.upr = pek == kPeRopeHalf ? t[0].pe.rotary / 8 + (D - t[0].pe.rotary) / 4 : D / 4;
    a.row = small_div(a.upr);
    long blocks[2] = {0, 0};
    for (int i = 0; i < n; ++i) {
        PeSeg& g = a.seg[i];
        g.in = t[i].in;
        g.out = t[i].out;
        g.units = t[i].n_rows * a.upr;
        g.seq_len = t[i].seq_len;
        g.pos = small_div(t[i].seq_len);
        g.pe = t[i].pe;
        blocks[i] = (g.units + 256 * U - 1) / (256 * U);
    }
    if (blocks[0] + blocks[1] > INT32_MAX / 2) return hipErrorInvalidConfiguration;
    a.blocks0 = (unsigned)blocks[0];
    const unsigned grid = (unsigned)(blocks[0] + blocks[1]);
    const bool dup = t[0].pe.dup != 0;
    switch (pek) {
        case kPeRopeInterleaved:
            dup ? run_rows<T, TO, kPeRopeInterleaved, true>(a, grid, st)
                : run_rows<T, TO, kPeRopeInterleaved, false>(a, grid, st);
            break;
        case kPeRopeHalf:
            dup ? run_rows<T, TO, kPeRopeHalf, true>(a, grid, st)
                : run_rows<T, TO, kPeRopeHalf, false>(a, grid, st);
            break;
        case kPeSinusoidal:
            dup ? run_rows<T, TO, kPeSinusoidal, true>(a, grid, st)
                : run_rows<T, TO, kPeSinusoidal, false>(a, grid, st);
            break;
        default:
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <typename T, typename TO>
hipError_t pe_apply_t(int pek, const PeTensor& t, int D, int vec_ok, hipStream_t st) {
    const dim3 grid((unsigned)std::min<long>(t.n_rows, 65536)), block(256);
    const T* x = static_cast<const T*>(t.in);
    TO* y = static_cast<TO*>(t.out);
    switch (pek) {
        case kPeRopeInterleaved:
            hipLaunchKernelGGL((k_pe_apply<T, TO, kPeRopeInterleaved>), grid, block, 0, st, x, y,
                               t.n_rows, t.seq_len, D, t.pe, vec_ok);
            break;
        case kPeRopeHalf:
            hipLaunchKernelGGL((k_pe_apply<T, TO, kPeRopeHalf>), grid, block, 0, st, x, y, t.n_rows,
                               t.seq_len, D, t.pe, vec_ok);
            break;
        case kPeSinusoidal:
            hipLaunchKernelGGL((k_pe_apply<T, TO, kPeSinusoidal>), grid, block, 0, st, x, y, t.n_rows,
                               t.seq_len, D, t.pe, vec_ok);
            break;
        default:
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <typename T, typename TO>
hipError_t pe_any(int pek, const PeTensor* t, int n, int D, int vec_ok, hipStream_t st) {
    bool rows = true;
    for (int i = 0; i < n; ++i)
        rows = rows && rows_ok(pek, D, t[i].pe, vec_ok) &&
               t[i].n_rows <= ((long)1 << 40) / std::max(1, D / 4);
    if (rows) return pe_rows_t<T, TO>(pek, t, n, D, st);
    for (int i = 0; i < n; ++i) {
        const hipError_t e = pe_apply_t<T, TO>(pek, t[i], D, vec_ok, st);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

hipError_t launch_pe_apply(int dtype, int out_dtype, int pek, const PeTensor* t, int n, int D,
                           int vec_ok, hipStream_t st) {
    if (dtype == kDtypeF32) return pe_any<float, float>(pek, t, n, D, vec_ok, st);
    return out_dtype == kDtypeF32 ? pe_any<uint16_t, float>(pek, t, n, D, vec_ok, st)
                                  : pe_any<uint16_t, uint16_t>(pek, t, n, D, vec_ok, st);
}

// K~ of the flash kernel, bf16 to fp16: one workgroup per tile of 64 keys
// (the flash kernel's), NG groups of 4 dims per thread, all loads first.  The
// tile's largest finite magnitude is known before anything is written, so
// the values and units are those of the flash kernel's own staging.  Bound by
// the latency of those loads (bits, partners, two tables) on few workgroups a
// CU: 512 threads with half the groups each keep twice the waves in flight as
// 256: (4,8,1107,1107,128) rotate-half 11.5 -> 10.7 us, the calls
// (4,16,300,1500,128) 57.4 -> 55.3, (2,32,900,900,96) 52.1 -> 50.5.
namespace {
constexpr int kKeyTileThreads = 512;
template <int PEK, int NG>
__global__ __launch_bounds__(kKeyTileThreads) void k_encode_key_tiles(
    const uint16_t* __restrict__ K, uint16_t* __restrict__ out, float* __restrict__ unit, int tiles,
    int Lk, int D, PeSide pe) {
    constexpr int NT = kKeyTileThreads;
    __shared__ float slot[NT / 64];
    const int tid = threadIdx.x, vpr = D >> 2;
    const int bh = blockIdx.x / tiles, k0 = (blockIdx.x % tiles) * 64;
    const int groups = min(64, Lk - k0) * vpr;  // the tile's rows are consecutive
    const uint16_t* src = K + ((size_t)bh * Lk + k0) * D;
    uint16_t* dst = out + ((size_t)bh * Lk + k0) * D;
    float4 x[NG];
    int d[NG], pos[NG];
    const uint16_t* row[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const int g = min(tid + NT * i, groups - 1), r = g / vpr;
        d[i] = (g - r * vpr) * 4;
        pos[i] = k0 + r;
        row[i] = src + (size_t)r * D;
        x[i] = Elem<uint16_t>::ld4(row[i], d[i]);
    }
    if (pe.on) {
        if (pe4_batch_ok(PEK, pe)) {
            pe4_batch<uint16_t, PEK, NG>(x, d, row, pos, D, pe);
        } else {
#pragma unroll
            for (int i = 0; i < NG; ++i)
                x[i] = apply_pe4<uint16_t, PEK>(x[i], row[i], pos[i], d[i], D, pe, true);
        }
    }
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < NG; ++i) m = max_finite4(m, x[i]);
    m = wave_max(m);
    if ((tid & 63) == 0) slot[tid >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) m = fmaxf(m, slot[w]);
    const bool plain = m >= 0.125f && m < kF16Range;
    const float s = plain ? 1.f : pow2_scale(m);
    if (tid == 0) unit[blockIdx.x] = plain ? 1.f : pow2_unit(m);
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const f16x2 a = {(_Float16)(x[i].x * s), (_Float16)(x[i].y * s)};
        const f16x2 b = {(_Float16)(x[i].z * s), (_Float16)(x[i].w * s)};
        if (tid + NT * i < groups)
            *reinterpret_cast<uint2*>(dst + 4 * (size_t)(tid + NT * i)) =
                make_uint2(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b));
    }
}

template <int PEK>
void run_key_tiles(const uint16_t* K, uint16_t* out, float* unit, int BH, int Lk, int D,
                   const PeSide& pe, hipStream_t st) {
    const int tiles = (Lk + 63) / 64;
    const dim3 grid((unsigned)(BH * tiles)), block(kKeyTileThreads);
    if (D <= 64)
        hipLaunchKernelGGL((k_encode_key_tiles<PEK, 2>), grid, block, 0, st, K, out, unit, tiles, Lk,
                           D, pe);
    else
        hipLaunchKernelGGL((k_encode_key_tiles<PEK, 4>), grid, block, 0, st, K, out, unit, tiles, Lk,
                           D, pe);
}
}  // namespace

hipError_t launch_encode_key_tiles(int pek, const uint16_t* K, uint16_t* out, float* unit, int BH,
                                   int Lk, int D, const PeSide& pe, hipStream_t st) {
    if (D > kFlashMaxDEncoded || D % 4 != 0) return hipErrorInvalidValue;
    switch (pek) {
        case kPeRopeInterleaved:
            run_key_tiles<kPeRopeInterleaved>(K, out, unit, BH, Lk, D, pe, st);
            break;
        case kPeRopeHalf: run_key_tiles<kPeRopeHalf>(K, out, unit, BH, Lk, D, pe, st); break;
        case kPeSinusoidal: run_key_tiles<kPeSinusoidal>(K, out, unit, BH, Lk, D, pe, st); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// Rows of D bf16 into rows of Dp (a multiple of 8), zeros past D: up to three
// tensors, 8 elements of a row per thread: 16 bytes at whatever alignment the
// source row has (the device runs in unaligned-access mode).  Pure traffic:
// (2,8,400,400,1500), Q, K and V (58 MB in, 58 out), 36 us with two-byte
// loads, 19 so.
namespace {
struct PadArgs {
    const uint16_t* in[3];
    uint16_t* out[3];
    long units[3];
    unsigned first[3];  // the tensor's first workgroup
    int D, Dp;
};
__global__ __launch_bounds__(256) void k_pad_rows(PadArgs a) {
    const int s = blockIdx.x >= a.first[2] ? 2 : (blockIdx.x >= a.first[1] ? 1 : 0);
    const unsigned per = (unsigned)a.Dp >> 3;
    const long u0 = (long)(blockIdx.x - a.first[s]) * 256, row0 = u0 / per;
    if (u0 + threadIdx.x >= a.units[s]) return;
    const unsigned k = (unsigned)(u0 - row0 * per) + threadIdx.x, dr = k / per;
    const long row = row0 + dr;
    const int d = (int)(k - dr * per) * 8;
    const uint16_t* x = a.in[s] + (size_t)row * a.D + d;
    uint32_t w[4];
    if (d + 8 <= a.D) {
        __builtin_memcpy(w, x, 16);
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t lo = d + 2 * c < a.D ? x[2 * c] : 0u;
            const uint32_t hi = d + 2 * c + 1 < a.D ? x[2 * c + 1] : 0u;
            w[c] = lo | (hi << 16);
        }
    }
    *reinterpret_cast<uint4*>(a.out[s] + (size_t)row * a.Dp + d) = make_uint4(w[0], w[1], w[2], w[3]);
}
}  // namespace

hipError_t launch_pad_rows(const PadTensor* t, int n, int D, int Dp, hipStream_t st) {
    PadArgs a{};
    a.D = D;
    a.Dp = Dp;
    long blocks = 0;
    for (int i = 0; i < 3; ++i) {
        a.first[i] = (unsigned)blocks;
        if (i >= n) continue;
        a.in[i] = static_cast<const uint16_t*>(t[i].in);
        a.out[i] = static_cast<uint16_t*>(t[i].out);
        a.units[i] = t[i].n_rows * (Dp / 8);
        blocks += (a.units[i] + 255) / 256;
        if (blocks > INT32_MAX / 2) return hipErrorInvalidConfiguration;
    }
    for (int i = n; i < 3; ++i) a.first[i] = ~0u;
    hipLaunchKernelGGL(k_pad_rows, dim3((unsigned)blocks), dim3(256), 0, st, a);
    return hipGetLastError();
}

}  // namespace atn
