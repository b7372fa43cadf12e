// The split-D pipeline on pipelined 16-bit MFMA tiles (gfx950): k_qk_tile
// (partial scores over a D-chunk), k_softmax_split (exact row softmax, P as
// 16-bit parts) and k_pv_tile (O = P V).
//
// Operands (KIND): fp32 as hi + lo fp16 parts (split16.hpp, three exact
// products per product), fp32 as three bf16 parts (X: all 24 bits at any
// magnitude, six products) or two (B2: 16 bits, three products), or raw bf16
// (one exact product).  P leaves the softmax already split, so the PV kernel
// converts V alone.
//
// X serves fp32 rows at any alignment (head_d % 4 != 0, misaligned bases), which
// ran on fp32 MFMA before and keep its accuracy at any magnitude.  Two fp16
// parts keep 22 bits, an absolute 2^-25 below 2^-3: V of 2^-20 loses half of
// them, and one large element takes them from its whole stage.  Six products
// and 11 instead of 4 instructions to split a value pair make the tiles 1.25 to
// 1.5 times as long, still half of what fp32 MFMA takes, and the error against
// 64 bits halves, for the parts lose nothing: (2,2,422,422,2361) 189 us on
// fp32 MFMA, 67 on two parts, 94 on three (5.7e-7, 4.3e-7, 2.2e-7 normwise);
// (1,4,1453,1453,1025) 797, 199, 305 us.  An infinity's later parts are NaN,
// and its product with a part that is zero: a tile that holds one (or a value
// that rounds to one) is computed again on fp32 MFMA.
//
// What bounds these kernels is VALU issue (the fp16 split: 4 instructions per
// value pair) beside the MFMAs where the grid fills the chip, and the latency
// of a stage where it leaves a CU one workgroup.  So a stage's 16-byte loads
// go out one stage (128 x 128 tiles) or two (64 x 64: two register sets)
// before their LDS writes, LDS is double-buffered with one barrier per stage,
// and two stages run through one MFMA chain before their sum is added to the
// sum (half the additions of a sum per stage; the rounding against exact
// 64-bit results stays below that of a sum per stage and of one chain: 4.3e-7
// normwise at (1,4,512,512,2048), 6.7e-7 with one chain).  Register use stays
// clear of spills: a spill's reload waits (vmcnt) for the loads in flight.  A
// value beyond fp16's range is found in passing (one v_max3 per pair); its
// workgroup then computes the tile again, every stage scaled by powers of two
// from its largest finite magnitudes, the next stage's loads in flight.  Where
// the first stage already holds one, the pass before is left out: K of 2^20
// at (1,4,512,512,2048) 92 -> 75 us, with V of 2^20 115 -> 82 (a look at every
// pair of stages instead made ordinary calls 6-8 % longer).
//
// Tiles of 128 x 128 or 64 x 64 (4 waves) on 32 x 32 x 16 MFMA.  A grid of at
// most one 128 x 128 workgroup a CU runs it as 8 waves of 64 x 32, two to a
// SIMD: half the sums per wave leave registers for loads two stages ahead,
// and one wave's fp16 split runs beside the other's MFMAs.  (1,4,512,512,2048)
// Q K^T 22.8 -> 20.9 us, P V 22.4 -> 20.3; (2,4,1024,1024,512) P V 45.7 ->
// 36.7.  With two workgroups on a CU 4 waves of 64 x 64 are the better: they
// read a third fewer fragments per product ((2,2,504,1387,4424) Q K^T 124.7
// us against 136.9).  LDS rows of 32 elements (64 bytes) per part, their
// 16-byte chunks permuted by tile_swz(row) so that fragment reads hit
// distinct banks unpadded (SQ_LDS_BANK_CONFLICT 0): 64 KiB for both stages of
// a 128 x 128 tile, two workgroups per CU (X: 96 KiB, one, always of 8 waves).
// Rows of S and P are padded to
// whole vectors, so ragged key counts store and load 16 bytes as well; rows
// of O whose D is odd are stored 4 elements at a time at any alignment
// ((2,8,400,400,1501) P V of bf16 56 -> 33 us).
//
// fp32 calls, before (stream16.hip's kernels) -> these: (1,4,512,512,2048)
// 57.9 -> 45.9 us, (2,2,422,422,2360) 81 -> 49, (2,2,128,1415,1520) 98 -> 40,
// (1,2,517,517,1272) 58 -> 31; at (1,4,1453,1453,1024) Q K^T runs at 215
// TFLOP/s of fp32 work (650 of fp16 products).  bf16: (1,2,273,757,3081)
// 184 -> 35 us (before: fp32 MFMA on two-byte loads), and the GEMM path's
// small grids ((1,2,68,68,624) 37.3 -> 10.6 us, see the host's rule).
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"
#include "split16.hpp"

namespace atn {

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));

constexpr int kKindF32 = kTileF32, kKindBF16 = kTileBF16, kKindX = kTileF32Exact, kKindB2 = kTileF32Bf16x2;

// Depth of a QK stage: 128 bytes of a row either way (fp32: 32 elements as
// PARTS parts; bf16: 64 elements, the two 32-deep halves in the parts' places).
template <int KIND>
struct Tile {
    using T = typename std::conditional<KIND == kKindBF16, uint16_t, float>::type;
    static constexpr int ES = KIND == kKindBF16 ? 2 : 4;
    static constexpr int DEPTH = 128 / ES;
    static constexpr int PER16 = 16 / ES;  // elements per 16-byte load
    static constexpr int PARTS = KIND == kKindX ? 3 : 2;
};

__device__ __forceinline__ int tile_swz(int row) { return ((row >> 1) & 3) ^ ((row >> 3) & 1); }
// 16-bit element offset of chunk c (8 elements) of a 32-element LDS row
__device__ __forceinline__ int tile_at(int row, int c) { return row * 32 + ((c ^ tile_swz(row)) << 3); }

template <int KIND>
__device__ __forceinline__ v16f mfma32(const uint4& a, const uint4& b, const v16f& c) {
    if constexpr (KIND == kKindF32)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                      __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a),
                                                       __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}

__device__ __forceinline__ uint4 ld_buf_u4(__amdgpu_buffer_rsrc_t r, unsigned off) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
    return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ float4 as_f4(const uint4& u) {
    return make_float4(__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z),
                       __uint_as_float(u.w));
}

// 4 values times s as hi and lo fp16 parts
__device__ __forceinline__ void split4(const uint4& u, float one, uint2& hi, uint2& lo) {
    const float4 v = as_f4(u);
    split2_f16_one(v.x, v.y, one, hi.x, lo.x);
    split2_f16_one(v.z, v.w, one, hi.y, lo.y);
}
__device__ __forceinline__ void split4_scaled(const uint4& u, float s, uint2& hi, uint2& lo) {
    const float4 v = as_f4(u);
    split2_f16(v.x * s, v.y * s, hi.x, lo.x);
    split2_f16(v.z * s, v.w * s, hi.y, lo.y);
}

// two values as bf16, rounded to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
    const v2f v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, v2bf));
}
// a and b as N bf16 parts each, every part the nearest to what the ones before
// it leave; three hold an fp32 value exactly (8 + 8 + 8 bits)
template <int N>
__device__ __forceinline__ void split_bf16(float a, float b, uint32_t (&w)[N]) {
#pragma unroll
    for (int p = 0; p < N; ++p) {
        w[p] = pk_bf16(a, b);
        a -= __uint_as_float(w[p] << 16);
        b -= __uint_as_float(w[p] & 0xffff0000u);
    }
}
// Magnitudes from here on round to an infinite first part.
constexpr float kBf16Range = 0x1.ffp127f;

// The parts of 4 values (16 bytes) of kind F32 (one = 1), X or B2
template <int KIND>
__device__ __forceinline__ void split_parts(const uint4& u, float one, uint2 (&p)[Tile<KIND>::PARTS]) {
    if constexpr (KIND == kKindF32) {
        split4(u, one, p[0], p[1]);
    } else {
        constexpr int N = Tile<KIND>::PARTS;
        const float4 v = as_f4(u);
        uint32_t a[N], b[N];
        split_bf16(v.x, v.y, a);
        split_bf16(v.z, v.w, b);
#pragma unroll
        for (int k = 0; k < N; ++k) p[k] = make_uint2(a[k], b[k]);
    }
}

// One 32 x 32 x 16 product of split operands added to c: the parts' products
// down to 2^-22 (two fp16 parts), 2^-25 (three bf16 parts) or 2^-17 (two) of the
// leading one, the smallest first.
template <int KIND, int N>
__device__ __forceinline__ v16f mfma_parts(const uint4 (&a)[N], const uint4 (&b)[N], v16f c) {
    if constexpr (KIND == kKindX) {
        c = mfma32<KIND>(a[2], b[0], c);
        c = mfma32<KIND>(a[0], b[2], c);
        c = mfma32<KIND>(a[1], b[1], c);
    }
    c = mfma32<KIND>(a[1], b[0], c);
    c = mfma32<KIND>(a[0], b[1], c);
    return mfma32<KIND>(a[0], b[0], c);
}
__device__ __forceinline__ v16f mfma_f32(float a, float b, const v16f& c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Consecutive tiles on one XCD: workgroup ids are dealt to the 8 XCDs in
// turn, each XCD takes a contiguous share of the n tiles.
__device__ __forceinline__ unsigned xcd_tile(unsigned id, unsigned n) {
    const unsigned x = id & 7, i = id >> 3, per = n >> 3, rem = n & 7;
    return x * per + min(x, rem) + i;
}

// Workgroup maximum of two per-thread values; every thread must call it.
template <int NW>
__device__ __forceinline__ void wg_max2(float& a, float& b, float* sh) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    a = wave_max(a);
    b = wave_max(b);
    if (lane == 0) {
        sh[wave] = a;
        sh[NW + wave] = b;
    }
    __syncthreads();
    a = sh[0];
    b = sh[NW];
#pragma unroll
    for (int w = 1; w < NW; ++w) {
        a = fmaxf(a, sh[w]);
        b = fmaxf(b, sh[NW + w]);
    }
}

__device__ __forceinline__ float max4abs(float m, const uint4& u) {
    const float4 v = as_f4(u);
    return vmax3abs(vmax3abs(m, v.x, v.y), v.z, v.w);
}

// Whether any thread of the workgroup saw a magnitude of `range` or more:
// told before a barrier, asked behind it (of words that nothing overwrites)
__device__ __forceinline__ void tell_over(float big, float range, int* flag) {
    const bool over = __ballot(!(big < range)) != 0;
    if ((threadIdx.x & 63) == 0) flag[threadIdx.x >> 6] = over;
}
template <int NW>
__device__ __forceinline__ bool any_over(const int* flag) {
    int any = flag[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) any |= flag[w];
    return __builtin_amdgcn_readfirstlane(any) != 0;
}

// 4 consecutive elements to an address of element alignment only: one store
// (the device runs in unaligned-access mode)
__device__ __forceinline__ void st4_any(float* p, float4 v) { __builtin_memcpy(p, &v, 16); }
__device__ __forceinline__ void st4_any(uint16_t* p, float4 v) {
    uint2 w;
    w.x = (uint32_t)f32_to_bf16_bits(v.x) | ((uint32_t)f32_to_bf16_bits(v.y) << 16);
    w.y = (uint32_t)f32_to_bf16_bits(v.z) | ((uint32_t)f32_to_bf16_bits(v.w) << 16);
    __builtin_memcpy(p, &w, 8);
}

// Partial scores S_split[bh][i][j] = sum over the chunk's dims of q_id k_jd
// for one TL x TL tile.  Wave w computes S^T for its TL/2 keys x TL/2
// queries: a lane holds 4 consecutive keys of one query per 16-byte store
// (rows of S are ldS, a multiple of 4, apart).  RAG: head_d is no multiple of
// 4 (fp32; rows then start at 4-byte boundaries and the last group of a row
// is read element by element).  COMP: compensated sums.  Encoded rows make long
// sums of one sign (sinusoidal), whose additions' roundings grow with the
// D-chunk, and chunks are longer here than on the kernels without copies:
// (4,4,567,279,904) sinusoidal 6.8e-7 there, 7.6e-7 with plain sums, 5.6e-7 with
// compensated ones (at 2048 dims 8.0, 8.5, 6.9), for 4 % of the call; sums
// without an encoding are no further off than there as they are.
template <int KIND, int TL, int NW, bool RAG, bool COMP>
__global__ __launch_bounds__(64 * NW, NW == 8 ? 1 : 2) void k_qk_tile(QkTileArgs a) {
    using G = Tile<KIND>;
    constexpr int LROWS = 8 * NW, ROUNDS = TL / LROWS;  // loader: rows per round, rounds
    constexpr int WK = NW / 2;                          // waves along the keys (2 along the queries)
    constexpr int NK = TL / WK / 32, NQ = TL / 64;      // 32 x 32 MFMA tiles per wave
    constexpr int PART = TL * 32;       // elements of one part of one operand
    constexpr int AHEAD = TL == 64 || NW == 8 ? 2 : 1;  // stages a load is issued before its LDS write
    constexpr int NP = G::PARTS;
    __shared__ __align__(16) uint16_t sq[2][NP * PART];  // [stage][part][row][32]
    __shared__ __align__(16) uint16_t sk[2][NP * PART];
    __shared__ float slot[2 * NW];
    __shared__ int flag[2][NW];
    constexpr bool kRanged = KIND != kKindBF16;
    constexpr float kRange = KIND == kKindF32 ? kF16Range : kBf16Range;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    unsigned t = xcd_tile(blockIdx.x, gridDim.x);
    const int tk = (int)(t % a.tiles_k);
    t /= a.tiles_k;
    const int tq = (int)(t % a.tiles_q);
    t /= a.tiles_q;
    const int split = (int)(t % a.nsplit), bh = (int)(t / a.nsplit);
    const int q0 = tq * TL, k0 = tk * TL;
    const int dbeg = split * a.dchunk, dend = min(a.D, dbeg + a.dchunk);

    const char* Qh = static_cast<const char*>(a.Q) + (size_t)bh * a.Lq * a.D * G::ES;
    const char* Kh = static_cast<const char*>(a.K) + (size_t)bh * a.Lk * a.D * G::ES;
    const int qbytes = a.Lq * a.D * G::ES, kbytes = a.Lk * a.D * G::ES;
    // loader: row lrow + 32 i, the 16 bytes lc of the stage's 128
    const int lrow = tid >> 3, lc = tid & 7;
    unsigned qoff[ROUNDS], koff[ROUNDS];  // (a row outside the tensor stays past its end)
#pragma unroll
    for (int i = 0; i < ROUNDS; ++i) {
        const int qi = q0 + lrow + LROWS * i, kj = k0 + lrow + LROWS * i;
        qoff[i] = qi < a.Lq ? (unsigned)(qi * a.D * G::ES + lc * 16) : (unsigned)kBufOob;
        koff[i] = kj < a.Lk ? (unsigned)(kj * a.D * G::ES + lc * 16) : (unsigned)kBufOob;
    }
    struct Regs {
        uint4 q[ROUNDS], k[ROUNDS];
    };
    auto issue = [&](Regs& r, int d0) {
        // the stage's depth goes into the (scalar) buffer base
        const int d = d0 + lc * G::PER16, sh = min(d0, a.D) * G::ES;
        const bool in = d < dend;
        const __amdgpu_buffer_rsrc_t rq = buf_rsrc(Qh + sh, qbytes - sh);
        const __amdgpu_buffer_rsrc_t rk = buf_rsrc(Kh + sh, kbytes - sh);
        if (RAG && d0 + G::DEPTH > a.D) {
            // the row's last stage, element by element
#pragma unroll
            for (int i = 0; i < ROUNDS; ++i) {
                uint32_t w[8];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const bool ok = d + c < dend;
                    w[c] = __builtin_amdgcn_raw_buffer_load_b32(
                        rq, ok ? (int)qoff[i] + 4 * c : kBufOob, 0, 0);
                    w[4 + c] = __builtin_amdgcn_raw_buffer_load_b32(
                        rk, ok ? (int)koff[i] + 4 * c : kBufOob, 0, 0);
                }
                r.q[i] = make_uint4(w[0], w[1], w[2], w[3]);
                r.k[i] = make_uint4(w[4], w[5], w[6], w[7]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < ROUNDS; ++i) {
                r.q[i] = ld_buf_u4(rq, in ? qoff[i] : (unsigned)kBufOob);
                r.k[i] = ld_buf_u4(rk, in ? koff[i] : (unsigned)kBufOob);
            }
        }
    };
    float big = 0.f;
    const float one = unit_opaque();
    // LDS place of this thread's 16 bytes: fp32 half a chunk of every part,
    // bf16 a chunk of one part
    auto place = [&](int i) {
        const int row = lrow + LROWS * i;
        return KIND != kKindBF16 ? tile_at(row, lc >> 1) + 4 * (lc & 1)
                                : (lc >> 2) * PART + tile_at(row, lc & 3);
    };
    auto store = [&](const Regs& r, uint16_t* q, uint16_t* k) {
#pragma unroll
        for (int i = 0; i < ROUNDS; ++i) {
            const int o = place(i);
            if constexpr (KIND != kKindBF16) {
                uint2 w[NP];
                split_parts<KIND>(r.q[i], one, w);
#pragma unroll
                for (int p = 0; p < NP; ++p) *reinterpret_cast<uint2*>(q + p * PART + o) = w[p];
                split_parts<KIND>(r.k[i], one, w);
#pragma unroll
                for (int p = 0; p < NP; ++p) *reinterpret_cast<uint2*>(k + p * PART + o) = w[p];
                big = max4abs(max4abs(big, r.q[i]), r.k[i]);
            } else {
                *reinterpret_cast<uint4*>(q + o) = r.q[i];
                *reinterpret_cast<uint4*>(k + o) = r.k[i];
            }
        }
    };

    const int wq = (wave & 1) * (TL / 2), wk = (wave >> 1) * (TL / WK);  // wave's queries, keys
    const int fr = lane & 31, fc = lane >> 5;
    v16f acc[NK][NQ], sum[NK][NQ];  // [key tile][query tile]
    auto each = [&](auto f) {
#pragma unroll
        for (int i = 0; i < NK; ++i)
#pragma unroll
            for (int j = 0; j < NQ; ++j) f(acc[i][j], sum[i][j]);
    };
    auto zero = [&]() { each([](v16f& x, v16f& y) { x = y = v16f{}; }); };
    // the pair of stages just summed, into the tile's sum; COMP: what the
    // addition rounds off starts the next chain
    auto flush = [&]() {
        each([](v16f& x, v16f& y) {
            if constexpr (COMP) {
                const v16f t = y + x;
                x -= t - y;
                y = t;
            } else {
                y += x;
            }
        });
    };
    auto compute = [&](const uint16_t* q, const uint16_t* k, auto fresh) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            uint4 ka[NK][NP], qa[NQ][NP];
#pragma unroll
            for (int p = 0; p < NP; ++p) {
#pragma unroll
                for (int i = 0; i < NK; ++i)
                    ka[i][p] = *reinterpret_cast<const uint4*>(
                        k + p * PART + tile_at(wk + 32 * i + fr, 2 * ks + fc));
#pragma unroll
                for (int j = 0; j < NQ; ++j)
                    qa[j][p] = *reinterpret_cast<const uint4*>(
                        q + p * PART + tile_at(wq + 32 * j + fr, 2 * ks + fc));
            }
#pragma unroll
            for (int i = 0; i < NK; ++i)
#pragma unroll
                for (int j = 0; j < NQ; ++j) {
                    v16f c = decltype(fresh)::value && ks == 0 && !COMP ? v16f{} : acc[i][j];
                    if constexpr (KIND != kKindBF16) {
                        c = mfma_parts<KIND>(ka[i], qa[j], c);
                    } else {
                        c = mfma32<KIND>(ka[i][0], qa[j][0], c);
                        c = mfma32<KIND>(ka[i][1], qa[j][1], c);
                    }
                    acc[i][j] = c;
                }
        }
    };

    Regs r0, r1;
    Regs& rb = AHEAD == 2 ? r1 : r0;
    issue(r0, dbeg);
    if (AHEAD == 2) issue(r1, dbeg + G::DEPTH);
    zero();
    store(r0, sq[0], sk[0]);
    if (kRanged) tell_over(big, kRange, flag[0]);
    issue(r0, dbeg + AHEAD * G::DEPTH);
    __syncthreads();
    // a tensor far from 1 shows in the first stage: no pass in vain then
    bool redo = kRanged && any_over<NW>(flag[0]);
    if (!redo) {
        const int stages = (dend - dbeg + G::DEPTH - 1) / G::DEPTH;
        for (int n = 0, d0 = dbeg; n < stages >> 1; ++n, d0 += 2 * G::DEPTH) {
            compute(sq[0], sk[0], std::true_type{});
            store(rb, sq[1], sk[1]);
            issue(rb, d0 + G::DEPTH * (AHEAD + 1));
            __syncthreads();
            compute(sq[1], sk[1], std::false_type{});
            flush();
            store(r0, sq[0], sk[0]);
            issue(r0, d0 + G::DEPTH * (AHEAD + 2));
            __syncthreads();
        }
        if (stages & 1) compute(sq[0], sk[0], std::true_type{});
        if (COMP || (stages & 1)) flush();
        if (kRanged) {
            tell_over(big, kRange, flag[1]);
            __syncthreads();
            redo = any_over<NW>(flag[1]);
            if (redo) zero();
        }
    }
    if constexpr (KIND == kKindF32) {
        if (redo) {  // every stage scaled by its largest magnitudes
            // (4 waves of 128 x 128 without loads ahead: with them the
            // compiler's schedule of the ordinary loop above is 3 % longer)
            constexpr bool kLoadAhead = TL == 64 || NW == 8 || COMP;
            if (kLoadAhead) issue(r0, dbeg);
            for (int d0 = dbeg; d0 < dend; d0 += G::DEPTH) {
                if (!kLoadAhead) issue(r0, d0);
                float mq = 0.f, mk = 0.f;
#pragma unroll
                for (int i = 0; i < ROUNDS; ++i) {
                    mq = max_finite4(mq, as_f4(r0.q[i]));
                    mk = max_finite4(mk, as_f4(r0.k[i]));
                }
                __syncthreads();  // the last stage's reads (and the slots') are done
                wg_max2<NW>(mq, mk, slot);
                const float s1 = pow2_scale(mq), s2 = pow2_scale(mk);
#pragma unroll
                for (int i = 0; i < ROUNDS; ++i) {
                    const int o = place(i);
                    uint2 hi, lo;
                    split4_scaled(r0.q[i], s1, hi, lo);
                    *reinterpret_cast<uint2*>(sq[0] + o) = hi;
                    *reinterpret_cast<uint2*>(sq[0] + PART + o) = lo;
                    split4_scaled(r0.k[i], s2, hi, lo);
                    *reinterpret_cast<uint2*>(sk[0] + o) = hi;
                    *reinterpret_cast<uint2*>(sk[0] + PART + o) = lo;
                }
                if (kLoadAhead) issue(r0, d0 + G::DEPTH);
                __syncthreads();
                const float u = pow2_unit(mq) * pow2_unit(mk);
                each([](v16f& x, v16f&) { x = v16f{}; });
                compute(sq[0], sk[0], std::true_type{});
                each([u](v16f& x, v16f& y) { y += x * u; });
            }
        }
    }

    if constexpr (KIND == kKindX || KIND == kKindB2) {
        if (redo) {
            // on fp32 MFMA, from rows of fp32 (33 apart) in the parts' places
            constexpr int R = 33;
            float* fq = reinterpret_cast<float*>(sq);
            float* fk = reinterpret_cast<float*>(sk);
            for (int d0 = dbeg; d0 < dend; d0 += G::DEPTH) {
                issue(r0, d0);
                __syncthreads();  // the last stage's reads are done
#pragma unroll
                for (int i = 0; i < ROUNDS; ++i) {
                    const int o = (lrow + LROWS * i) * R + 4 * lc;
                    st4_any(fq + o, as_f4(r0.q[i]));
                    st4_any(fk + o, as_f4(r0.k[i]));
                }
                __syncthreads();
                for (int d = fc; d < G::DEPTH; d += 2)
#pragma unroll
                    for (int i = 0; i < NK; ++i)
#pragma unroll
                        for (int j = 0; j < NQ; ++j)
                            sum[i][j] = mfma_f32(fk[(wk + 32 * i + fr) * R + d],
                                                 fq[(wq + 32 * j + fr) * R + d], sum[i][j]);
            }
        }
    }

    // register r of a tile: key 8 (r / 4) + 4 (lane / 32) + r % 4 of query lane % 32
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
        const int qi = q0 + wq + 32 * j + fr;
        if (qi >= a.Lq) continue;
        float* srow = a.S + (((size_t)split * a.BH + bh) * a.Lq + qi) * a.ldS;
#pragma unroll
        for (int i = 0; i < NK; ++i)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int kj = k0 + wk + 32 * i + 8 * b + 4 * fc;
                const float4 v = make_float4(sum[i][j][4 * b], sum[i][j][4 * b + 1],
                                             sum[i][j][4 * b + 2], sum[i][j][4 * b + 3]);
                if (kj < a.ldS) *reinterpret_cast<float4*>(srow + kj) = v;
            }
    }
}

// P as its 16-bit parts, 4 values at column c of its row: two fp16 parts of
// 2^15 p (so that small probabilities keep their bits), or NP bf16 parts of p
// (fp32's exponents: nothing to scale, and no V whose products then overflow).
struct PParts {
    uint16_t* p[3];
};
template <int KIND, int NP>
__device__ __forceinline__ void store_p4(const PParts& out, size_t at, float4 v) {
    uint2 w[3];
    if constexpr (KIND == kKindF32) {
        split2_f16(v.x, v.y, w[0].x, w[1].x);
        split2_f16(v.z, v.w, w[0].y, w[1].y);
    } else {
        uint32_t a[NP], b[NP];
        split_bf16(v.x, v.y, a);
        split_bf16(v.z, v.w, b);
#pragma unroll
        for (int k = 0; k < NP; ++k) w[k] = make_uint2(a[k], b[k]);
    }
#pragma unroll
    for (int k = 0; k < NP; ++k) *reinterpret_cast<uint2*>(out.p[k] + at) = w[k];
}
template <int KIND>
constexpr float kPScale = KIND == kKindF32 ? 32768.0f : 1.0f;

// Row softmax of the summed partial scores, exact (max, exp, sum, divide),
// written as 16-bit parts (rows ldP apart, zeros from Lk on).
// TPR threads per row hold it in registers (thread t the 4 keys from
// 4 (t + TPR u) on), so S is read once; every partial's load is independent.
template <int KIND, int NP, int TPR, int NV>
__global__ __launch_bounds__(256) void k_softmax_split(const float* __restrict__ S, PParts out,
                                                       long rows, int Lk, int ldS, int ldP, int nsplit,
                                                       size_t split_stride, float scale) {
    __shared__ float red[8];
    const int tid = threadIdx.x, t = tid % TPR;
    const long row = (long)blockIdx.x * (256 / TPR) + tid / TPR;
    if (TPR == 64 && row >= rows) return;
    const float* s = S + (size_t)row * ldS;
    float4 v[NV];
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int c = 4 * (t + TPR * u);
        v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (c < Lk) v[u] = *reinterpret_cast<const float4*>(s + c);
    }
#pragma unroll 4
    for (int sp = 1; sp < nsplit; ++sp) {
        const float* q = s + (size_t)sp * split_stride;
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int c = 4 * (t + TPR * u);
            if (c < Lk) {
                const float4 w = *reinterpret_cast<const float4*>(q + c);
                v[u].x += w.x;
                v[u].y += w.y;
                v[u].z += w.z;
                v[u].w += w.w;
            }
        }
    }
    float m = -INFINITY;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int c = 4 * (t + TPR * u);
        v[u].x = c < Lk ? v[u].x * scale : -INFINITY;
        v[u].y = c + 1 < Lk ? v[u].y * scale : -INFINITY;
        v[u].z = c + 2 < Lk ? v[u].z * scale : -INFINITY;
        v[u].w = c + 3 < Lk ? v[u].w * scale : -INFINITY;
        m = fmaxf(m, fmaxf(fmaxf(v[u].x, v[u].y), fmaxf(v[u].z, v[u].w)));
    }
    m = wave_max(m);
    if constexpr (TPR == 256) {
        if ((tid & 63) == 0) red[tid >> 6] = m;
        __syncthreads();
        m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    }
    float l = 0.f;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int c = 4 * (t + TPR * u);
        v[u].x = c < Lk ? expf(v[u].x - m) : 0.f;
        v[u].y = c + 1 < Lk ? expf(v[u].y - m) : 0.f;
        v[u].z = c + 2 < Lk ? expf(v[u].z - m) : 0.f;
        v[u].w = c + 3 < Lk ? expf(v[u].w - m) : 0.f;
        l += (v[u].x + v[u].y) + (v[u].z + v[u].w);
    }
    l = wave_sum(l);
    if constexpr (TPR == 256) {
        if ((tid & 63) == 0) red[4 + (tid >> 6)] = l;
        __syncthreads();
        l = (red[4] + red[5]) + (red[6] + red[7]);
    }
    l *= 1.0f / kPScale<KIND>;  // (exact)
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int c = 4 * (t + TPR * u);
        if (c < ldP) {
            store_p4<KIND, NP>(out, (size_t)row * ldP + c,
                               make_float4(v[u].x / l, v[u].y / l, v[u].z / l, v[u].w / l));
        }
    }
}

// Rows longer than the registers hold: the sums go back to the first
// partial's place, and the row is read three times.
template <int KIND, int NP>
__global__ __launch_bounds__(256) void k_softmax_long(float* S, PParts out, long rows, int Lk,
                                                      int ldS, int ldP, int nsplit,
                                                      size_t split_stride, float scale) {
    __shared__ float red[8];
    const int tid = threadIdx.x;
    for (long row = blockIdx.x; row < rows; row += gridDim.x) {
        float* s = S + (size_t)row * ldS;
        float m = -INFINITY;
        for (int c = tid; c < Lk; c += 256) {
            float x = s[c];
            for (int sp = 1; sp < nsplit; ++sp) x += s[(size_t)sp * split_stride + c];
            x *= scale;
            s[c] = x;
            m = fmaxf(m, x);
        }
        m = wave_max(m);
        if ((tid & 63) == 0) red[tid >> 6] = m;
        __syncthreads();
        m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        float l = 0.f;
        for (int c = tid; c < Lk; c += 256) {
            const float e = expf(s[c] - m);
            s[c] = e;
            l += e;
        }
        l = wave_sum(l);
        if ((tid & 63) == 0) red[4 + (tid >> 6)] = l;
        __syncthreads();
        l = ((red[4] + red[5]) + (red[6] + red[7])) * (1.0f / kPScale<KIND>);
        for (int c = 4 * tid; c < ldP; c += 1024) {
            float p[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) p[k] = c + k < Lk ? s[c + k] / l : 0.f;
            store_p4<KIND, NP>(out, (size_t)row * ldP + c, make_float4(p[0], p[1], p[2], p[3]));
        }
        __syncthreads();  // red reused by the next row
    }
}

// O[bh][i][d] = sum_j P_ij V_jd for one tile of TL queries x TL dims, 32 keys
// a stage.  Wave w computes O^T for its TL/2 dims x TL/2 queries: a lane
// holds 4 consecutive dims of one query.  P rows go to LDS as they are; V
// stays [key][dim] there and reaches the MFMA by the transposing LDS read
// (rows of TL + 32 elements: the four rows of a read on distinct banks).
template <int KIND, int PP, int TL, int NW, bool RAG>
__global__ __launch_bounds__(64 * NW, NW == 8 ? 1 : 2) void k_pv_tile(PvTileArgs a) {
    using G = Tile<KIND>;
    constexpr int PART = TL * 32, WD = NW / 2;          // waves along the dims (2 along the queries)
    constexpr int ND = TL / WD / 32, NQ = TL / 64;      // 32 x 32 MFMA tiles per wave
    constexpr int AHEAD = TL == 64 || NW == 8 ? 2 : 1;
    constexpr int VSTR = TL + 32, VPARTS = KIND == kKindBF16 ? 1 : G::PARTS, VPART = 32 * VSTR;
    constexpr int VL = TL / G::PER16;             // V loader: lanes per row
    constexpr int VROWS = 64 * NW / VL, VROUNDS = 32 / VROWS > 0 ? 32 / VROWS : 1;
    static_assert(KIND == kKindBF16 || PP == VPARTS, "parts of P");
    static_assert(VROWS <= 32, "a round of V rows within a stage");
    __shared__ __align__(16) uint16_t sp[2][PP * PART];
    __shared__ __align__(16) uint16_t sv[2][VPARTS * VPART];
    __shared__ float slot[2 * NW];
    __shared__ int flag[2][NW];
    constexpr bool kRanged = KIND != kKindBF16;
    constexpr float kRange = KIND == kKindF32 ? kF16Range : kBf16Range;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    unsigned t = xcd_tile(blockIdx.x, gridDim.x);
    const int tq = (int)(t % a.tiles_q);
    t /= a.tiles_q;
    const int td = (int)(t % a.tiles_d), bh = (int)(t / a.tiles_d);
    const int q0 = tq * TL, d0 = td * TL;

    const size_t pbase = (size_t)bh * a.Lq * a.ldP;
    const int pbytes = a.Lq * a.ldP * 2, vbytes = a.Lk * a.D * G::ES;
    const char* Vh = static_cast<const char*>(a.V) + (size_t)bh * a.Lk * a.D * G::ES;
    // P loader: row lrow + PROWS i, chunk lc of every part
    constexpr int PROWS = 16 * NW, PR = TL / PROWS;
    const int lrow = tid >> 2, lc = tid & 3;
    unsigned poff[PR];
#pragma unroll
    for (int i = 0; i < PR; ++i) {
        const int row = q0 + lrow + PROWS * i;
        poff[i] = row < a.Lq ? (unsigned)((row * a.ldP + 8 * lc) * 2) : (unsigned)kBufOob;
    }
    const int vrow = tid / VL, vcol = (tid % VL) * G::PER16;
    unsigned voff[VROUNDS];  // (past the head's end from key Lk on)
#pragma unroll
    for (int i = 0; i < VROUNDS; ++i)
        voff[i] = d0 + vcol < a.D
                      ? (unsigned)(((vrow + VROWS * i) * a.D + d0 + vcol) * G::ES)
                      : (unsigned)kBufOob;
    struct Regs {
        uint4 p[PP][PR], v[VROUNDS];
    };
    auto issue = [&](Regs& r, int kk) {
        const int psh = min(kk, a.ldP);
#pragma unroll
        for (int w = 0; w < PP; ++w) {
            const __amdgpu_buffer_rsrc_t rp = buf_rsrc(a.p[w] + pbase + psh, pbytes - 2 * psh);
#pragma unroll
            for (int i = 0; i < PR; ++i)
                r.p[w][i] = ld_buf_u4(rp, kk + 8 * lc < a.ldP ? poff[i] : (unsigned)kBufOob);
        }
        const size_t vsh = (size_t)min(kk, a.Lk) * a.D * G::ES;
        const __amdgpu_buffer_rsrc_t rv = buf_rsrc(Vh + vsh, vbytes - (int)vsh);
#pragma unroll
        for (int i = 0; i < VROUNDS; ++i) {
            if (RAG && KIND != kKindBF16 && d0 + TL > a.D) {
                uint32_t w[4];
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    w[c] = __builtin_amdgcn_raw_buffer_load_b32(
                        rv, d0 + vcol + c < a.D ? (int)voff[i] + 4 * c : kBufOob, 0, 0);
                r.v[i] = make_uint4(w[0], w[1], w[2], w[3]);
            } else {
                r.v[i] = ld_buf_u4(rv, voff[i]);
            }
        }
    };
    float big = 0.f;
    const float one = unit_opaque();
    auto store_p = [&](const Regs& r, uint16_t* p) {
#pragma unroll
        for (int i = 0; i < PR; ++i) {
            const int o = tile_at(lrow + PROWS * i, lc);
#pragma unroll
            for (int w = 0; w < PP; ++w) *reinterpret_cast<uint4*>(p + w * PART + o) = r.p[w][i];
        }
    };
    auto store = [&](const Regs& r, uint16_t* p, uint16_t* v) {
        store_p(r, p);
#pragma unroll
        for (int i = 0; i < VROUNDS; ++i) {
            const int o = (vrow + VROWS * i) * VSTR + vcol;
            if constexpr (KIND != kKindBF16) {
                uint2 w[VPARTS];
                split_parts<KIND>(r.v[i], one, w);
#pragma unroll
                for (int p = 0; p < VPARTS; ++p) *reinterpret_cast<uint2*>(v + p * VPART + o) = w[p];
                big = max4abs(big, r.v[i]);
            } else {
                *reinterpret_cast<uint4*>(v + o) = r.v[i];
            }
        }
    };

    const int wq = (wave & 1) * (TL / 2), wd = (wave >> 1) * (TL / WD);
    const int fr = lane & 31, fc = lane >> 5;
    // V^T fragment: dims 16 (lane / 16 % 2) + lane % 16, keys 8 (lane / 32) + 0..7
    const int va = (8 * fc + ((lane & 15) >> 2)) * VSTR + wd + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    v16f acc[ND][NQ], sum[ND][NQ];  // [dim tile][query tile]
    auto each = [&](auto f) {
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int j = 0; j < NQ; ++j) f(acc[i][j], sum[i][j]);
    };
    auto zero = [&]() { each([](v16f&, v16f& y) { y = v16f{}; }); };
    // the pair of stages just summed, into the tile's sum
    auto flush = [&]() { each([](v16f& x, v16f& y) { y += x; }); };
    auto compute = [&](const uint16_t* p, const uint16_t* v, auto fresh) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            uint4 pa[NQ][PP], vv[ND][VPARTS];
#pragma unroll
            for (int i = 0; i < ND; ++i)
#pragma unroll
                for (int w = 0; w < VPARTS; ++w) {
                    const uint16_t* at = v + w * VPART + va + 16 * ks * VSTR + 32 * i;
                    const uint2 x = lds_tr16(at), y = lds_tr16(at + 4 * VSTR);
                    vv[i][w] = make_uint4(x.x, x.y, y.x, y.y);
                }
#pragma unroll
            for (int j = 0; j < NQ; ++j)
#pragma unroll
                for (int w = 0; w < PP; ++w)
                    pa[j][w] = *reinterpret_cast<const uint4*>(
                        p + w * PART + tile_at(wq + 32 * j + fr, 2 * ks + fc));
#pragma unroll
            for (int i = 0; i < ND; ++i)
#pragma unroll
                for (int j = 0; j < NQ; ++j) {
                    v16f c = decltype(fresh)::value && ks == 0 ? v16f{} : acc[i][j];
                    if constexpr (KIND != kKindBF16) {
                        c = mfma_parts<KIND>(vv[i], pa[j], c);
                    } else {
#pragma unroll
                        for (int w = PP - 1; w >= 0; --w) c = mfma32<KIND>(vv[i][0], pa[j][w], c);
                    }
                    acc[i][j] = c;
                }
        }
    };

    Regs r0, r1;
    Regs& rb = AHEAD == 2 ? r1 : r0;
    issue(r0, 0);
    if (AHEAD == 2) issue(r1, 32);
    zero();
    store(r0, sp[0], sv[0]);
    if (kRanged) tell_over(big, kRange, flag[0]);
    issue(r0, 32 * AHEAD);
    __syncthreads();
    // a tensor far from 1 shows in the first stage: no pass in vain then
    bool redo = kRanged && any_over<NW>(flag[0]);
    if (!redo) {
        const int stages = (a.Lk + 31) / 32;
        for (int n = 0, kk = 0; n < stages >> 1; ++n, kk += 64) {
            compute(sp[0], sv[0], std::true_type{});
            store(rb, sp[1], sv[1]);
            issue(rb, kk + 32 * (AHEAD + 1));
            __syncthreads();
            compute(sp[1], sv[1], std::false_type{});
            flush();
            store(r0, sp[0], sv[0]);
            issue(r0, kk + 32 * (AHEAD + 2));
            __syncthreads();
        }
        if (stages & 1) {
            compute(sp[0], sv[0], std::true_type{});
            flush();
        }
        if (kRanged) {
            tell_over(big, kRange, flag[1]);
            __syncthreads();
            redo = any_over<NW>(flag[1]);
            if (redo) zero();
        }
    }
    if constexpr (KIND == kKindF32) {
        if (redo) {  // V's stages scaled by their largest magnitudes
            issue(r0, 0);
            for (int kk = 0; kk < a.Lk; kk += 32) {
                float mv = 0.f, none = 0.f;
#pragma unroll
                for (int i = 0; i < VROUNDS; ++i) mv = max_finite4(mv, as_f4(r0.v[i]));
                __syncthreads();
                wg_max2<NW>(mv, none, slot);
                const float s1 = pow2_scale(mv), u = pow2_unit(mv);
                store_p(r0, sp[0]);
#pragma unroll
                for (int i = 0; i < VROUNDS; ++i) {
                    const int o = (vrow + VROWS * i) * VSTR + vcol;
                    uint2 hi, lo;
                    split4_scaled(r0.v[i], s1, hi, lo);
                    *reinterpret_cast<uint2*>(sv[0] + o) = hi;
                    *reinterpret_cast<uint2*>(sv[0] + (VPARTS - 1) * VPART + o) = lo;
                }
                issue(r0, kk + 32);
                __syncthreads();
                compute(sp[0], sv[0], std::true_type{});
                each([u](v16f& x, v16f& y) { y += x * u; });
            }
        }
    }

    if constexpr (KIND == kKindX) {
        if (redo) {
            // on fp32 MFMA: P put together again (rows 33 apart), V as it is
            constexpr int R = 33;
            float* fp = reinterpret_cast<float*>(sp);
            float* fv = reinterpret_cast<float*>(sv);
            for (int kk = 0; kk < a.Lk; kk += 32) {
                issue(r0, kk);
                __syncthreads();  // the last stage's reads are done
#pragma unroll
                for (int i = 0; i < PR; ++i) {
                    float* o = fp + (lrow + PROWS * i) * R + 8 * lc;
#pragma unroll
                    for (int c = 0; c < 8; ++c) {
                        float x = 0.f;
#pragma unroll
                        for (int w = 0; w < PP; ++w) {
                            const uint32_t u = (&r0.p[w][i].x)[c >> 1];
                            x += __uint_as_float(c & 1 ? u & 0xffff0000u : u << 16);
                        }
                        o[c] = x;
                    }
                }
#pragma unroll
                for (int i = 0; i < VROUNDS; ++i)
                    *reinterpret_cast<uint4*>(fv + (vrow + VROWS * i) * TL + vcol) = r0.v[i];
                __syncthreads();
                for (int k = fc; k < 32; k += 2)
#pragma unroll
                    for (int i = 0; i < ND; ++i)
#pragma unroll
                        for (int j = 0; j < NQ; ++j)
                            sum[i][j] = mfma_f32(fv[k * TL + wd + 32 * i + fr],
                                                 fp[(wq + 32 * j + fr) * R + k], sum[i][j]);
            }
        }
    }

    constexpr float kPInv = 1.0f / kPScale<KIND>;
    using T = typename G::T;
    T* Oh = static_cast<T*>(a.O) + (size_t)bh * a.Lq * a.ldO;
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
        const int qi = q0 + wq + 32 * j + fr;
        if (qi >= a.Lq) continue;
        T* orow = Oh + (size_t)qi * a.ldO;
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int d = d0 + wd + 32 * i + 8 * b + 4 * fc;
                float v[4];
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    v[c] = sum[i][j][4 * b + c] * kPInv;
                if (d + 3 < a.ldO) {
                    // (rows of any alignment: 8 or 16 bytes at once all the same)
                    if (!RAG)
                        Elem<T>::st4(orow, d, make_float4(v[0], v[1], v[2], v[3]));
                    else
                        st4_any(orow + d, make_float4(v[0], v[1], v[2], v[3]));
                } else if (RAG) {
#pragma unroll
                    for (int c = 0; c < 3; ++c)
                        if (d + c < a.ldO) Elem<T>::st(orow, d + c, v[c]);
                }
            }
    }
}

// 128 x 128 tiles take 8 waves (64 x 32 each) while no CU gets a second
// workgroup: two waves per SIMD then, and loads two stages ahead (fp32
// (1,4,512,512,2048): Q K^T 22.8 -> 20.9 us, P V 22.4 -> 20.3; (2,4,1024,1024,
// 512) P V 45.7 -> 36.7).  Beyond that 4 waves of 64 x 64, two workgroups per
// CU, read a third less from LDS ((2,2,504,1387,4424) Q K^T 124.7 us against
// 136.9).
constexpr unsigned kOnePerCu = 256;

template <int KIND, int TL, int NW>
void run_qk(const QkTileArgs& a, bool rag, unsigned grid, hipStream_t st) {
    // (the other kinds' rows are whole 16-byte vectors)
    if (KIND == kKindX && rag)
        hipLaunchKernelGGL((k_qk_tile<KIND, TL, NW, KIND == kKindX, false>), dim3(grid),
                           dim3(64 * NW), 0, st, a);
    else if (KIND == kKindF32 && a.comp)
        hipLaunchKernelGGL((k_qk_tile<KIND, TL, NW, false, KIND == kKindF32>), dim3(grid),
                           dim3(64 * NW), 0, st, a);
    else
        hipLaunchKernelGGL((k_qk_tile<KIND, TL, NW, false, false>), dim3(grid), dim3(64 * NW), 0, st,
                           a);
}
template <int KIND>
void run_qk_tile(int tile, const QkTileArgs& a, bool rag, unsigned grid, hipStream_t st) {
    if (tile == 64)
        run_qk<KIND, 64, 4>(a, rag, grid, st);
    else if (KIND == kKindX || grid <= kOnePerCu)
        run_qk<KIND, 128, 8>(a, rag, grid, st);
    else if constexpr (KIND != kKindX)
        run_qk<KIND, 128, 4>(a, rag, grid, st);
}

template <int KIND, int PP, int TL, int NW>
void run_pv(const PvTileArgs& a, bool rag, unsigned grid, hipStream_t st) {
    if (KIND != kKindF32 && rag)
        hipLaunchKernelGGL((k_pv_tile<KIND, PP, TL, NW, KIND != kKindF32>), dim3(grid), dim3(64 * NW),
                           0, st, a);
    else
        hipLaunchKernelGGL((k_pv_tile<KIND, PP, TL, NW, false>), dim3(grid), dim3(64 * NW), 0, st, a);
}
template <int KIND, int PP>
void run_pv_tile(int tile, const PvTileArgs& a, bool rag, unsigned grid, hipStream_t st) {
    if (tile == 64)
        run_pv<KIND, PP, 64, 4>(a, rag, grid, st);
    else if (KIND == kKindX || grid <= kOnePerCu)
        run_pv<KIND, PP, 128, 8>(a, rag, grid, st);
    else if constexpr (KIND != kKindX)
        run_pv<KIND, PP, 128, 4>(a, rag, grid, st);
}

template <int KIND, int NP>
hipError_t softmax_k(float* S, const PParts& out, long rows, int Lk, int ldS, int ldP, int nsplit,
                     size_t stride, float scale, hipStream_t st) {
    // a wave per row while that gives every CU several waves; a workgroup
    // per row for few rows and for rows longer than a wave's registers hold
    const bool wave = Lk <= 2048 && (rows >= 4096 || Lk <= 256);
#define ATN_SOFTMAX(TPR, NV)                                                                    \
    hipLaunchKernelGGL((k_softmax_split<KIND, NP, TPR, NV>),                                    \
                       dim3((unsigned)((rows + 256 / TPR - 1) / (256 / TPR))), dim3(256), 0, st, \
                       S, out, rows, Lk, ldS, ldP, nsplit, stride, scale)
    if (Lk > 8192 || rows > INT32_MAX)
        hipLaunchKernelGGL((k_softmax_long<KIND, NP>), dim3((unsigned)std::min<long>(rows, 65536)),
                           dim3(256), 0, st, S, out, rows, Lk, ldS, ldP, nsplit, stride, scale);
    else if (wave && Lk <= 256)
        ATN_SOFTMAX(64, 1);
    else if (wave && Lk <= 512)
        ATN_SOFTMAX(64, 2);
    else if (wave && Lk <= 1024)
        ATN_SOFTMAX(64, 4);
    else if (wave)
        ATN_SOFTMAX(64, 8);
    else if (Lk <= 1024)
        ATN_SOFTMAX(256, 1);
    else if (Lk <= 2048)
        ATN_SOFTMAX(256, 2);
    else if (Lk <= 4096)
        ATN_SOFTMAX(256, 4);
    else
        ATN_SOFTMAX(256, 8);
#undef ATN_SOFTMAX
    return hipGetLastError();
}

}  // namespace

hipError_t launch_qk_tile(int kind, int tile, QkTileArgs a, hipStream_t st) {
    if (a.D % 4 != 0 && kind != kTileF32Exact) return hipErrorInvalidValue;
    a.tiles_q = (a.Lq + tile - 1) / tile;
    a.tiles_k = (a.Lk + tile - 1) / tile;
    const unsigned grid = (unsigned)((long)a.BH * a.tiles_q * a.tiles_k * a.nsplit);
    const bool rag = a.D % 4 != 0;
    if (kind == kTileF32)
        run_qk_tile<kKindF32>(tile, a, rag, grid, st);
    else if (kind == kTileBF16)
        run_qk_tile<kKindBF16>(tile, a, false, grid, st);
    else if (kind == kTileF32Bf16x2)
        run_qk_tile<kKindB2>(tile, a, rag, grid, st);
    else
        run_qk_tile<kKindX>(tile, a, rag, grid, st);
    return hipGetLastError();
}

hipError_t launch_softmax_split(int kind, int pparts, float* S, uint16_t* const p[3], long rows,
                                int Lk, int ldS, int ldP, int nsplit, size_t split_stride,
                                float scale, hipStream_t st) {
    const PParts out{{p[0], p[1], p[2]}};
    if (kind == kTileF32)
        return softmax_k<kKindF32, 2>(S, out, rows, Lk, ldS, ldP, nsplit, split_stride, scale, st);
    return pparts == 2
               ? softmax_k<kKindX, 2>(S, out, rows, Lk, ldS, ldP, nsplit, split_stride, scale, st)
               : softmax_k<kKindX, 3>(S, out, rows, Lk, ldS, ldP, nsplit, split_stride, scale, st);
}

hipError_t launch_pv_tile(int kind, int pparts, int tile, PvTileArgs a, hipStream_t st) {
    a.tiles_q = (a.Lq + tile - 1) / tile;
    a.tiles_d = (a.D + tile - 1) / tile;
    const unsigned grid = (unsigned)((long)a.BH * a.tiles_q * a.tiles_d);
    const bool rag = a.ldO % 4 != 0 || a.o_align == 0;
    if (rag && kind == kTileF32) return hipErrorInvalidValue;
    if (kind == kTileF32)
        run_pv_tile<kKindF32, 2>(tile, a, rag, grid, st);
    else if (kind == kTileF32Exact)
        run_pv_tile<kKindX, 3>(tile, a, rag, grid, st);
    else if (pparts == 2)
        run_pv_tile<kKindBF16, 2>(tile, a, rag, grid, st);
    else
        run_pv_tile<kKindBF16, 3>(tile, a, rag, grid, st);
    return hipGetLastError();
}

}  // namespace atn
