// Causal flash attention forward, fp32 exact mode, for gfx950 (CDNA4).
//
// Replaces flash_attention_forward (FlashAttention.cpp:24-182). The reference
// runs 256x256 tiles with two cblas_sgemm calls per tile and a scalar softmax;
// here a persistent workgroup walks 128-query items (flash_items.h: snake order
// over items sorted by causal cost, so a long query tile is paired with a short
// one) and streams 32-key tiles of K and V through LDS. A launch that fits one
// round folds its units instead (flash_items.h): an item is then the 64-query
// tiles p and n-1-p of one (batch, head), rows 0-63 and 64-127.
//
// Products. Every fp32 operand x is taken times 2^24 and split into three bf16 values x = h + m + l (each the rounding
// of what the ones before it leave: 24 significand bits in three times 8, so the sum is x itself), and a product x y is
// formed on v_mfma_f32_32x32x16_bf16 from the six partial products lh, hl, mm, mh, hm, hh, accumulated in fp32. The
// three left out (ml, lm, ll) come to at most 2^-24 of x y, the size of one fp32 rounding, and to 2^-28 on average. Six
// bf16 MFMAs take 192 cycles for 16 steps of k where v_mfma_f32_32x32x2_f32 takes 512, and the result is nearer to the
// exact one: over random 128-long dot products the relative error (2-norm) is 6.1e-8 with the small partial products
// summed first, against 2.0e-7 for the fp32 instruction, which rounds after every second k instead of after every
// sixteenth.
//
// The factor 2^24 (for Q: scale log2 e times a power of two) keeps every part of every fp32 number, the smallest too, above
// bf16's denormals, whatever lies beside it in its row. It is exact, and taken out again where a score enters exp2 and
// at an item's end. What is left out of the split's range is 2^103 and above, infinities and NaN: they give a result that
// is not finite (a scaled operand or sum that overflows to infinity, inf * 0 = NaN), an empty softmax where there are keys,
// or a score of -inf. A wave that finds one of these repeats its keys with the fp32 instruction, straight from memory
// (slow_keys), and keeps that result.
//
// Work split: 8 waves in two groups of 4. Both groups hold the same 128 queries
// (32 per wave) and split the key tiles: group g takes tiles g, g+2, g+4, ... At
// the end the two partials (m, l, O) are merged through LDS with the same rescale
// the reference applies between tiles (FlashAttention.cpp:134-156), each group
// finalising half of the dims. Each wave computes S^T = K Q^T for its 32 queries,
// so that in the accumulator layout one lane holds one query (lane % 32) and 16
// keys; the row max / row sum of the online softmax are then a per-lane reduction
// plus one exchange with lane ^ 32. The probabilities stay in registers, are split
// there and feed the PV product O^T += V^T P^T as the B operand (the MFMA's k
// index is only a summation label, so V rows are read in the accumulator's key
// order, by the transposing ds_read_b64_tr_b16).
//
// K and V tiles pass through registers on their way to LDS: a wave loads a quarter of its group's tile (four floats
// per lane and row pair), one half step ahead, splits it and writes the three bf16 planes, V's under the MFMAs of the
// S product and the next K's under those of the PV product, so the split has no phase of its own: two barriers per
// step, K planes free and V planes ready at one, the other way round at the other. Group 1 runs half a step behind
// group 0, and a wave in its S product and softmax has the higher issue priority, so that one group's softmax issues
// under the other's PV product. Plane rows are padded (K's 272 bytes, V's 320) so that the row-wise K reads and the
// transposing V reads fall in different banks and every LDS address is one register plus a constant.
//
// What bounds it: the matrix pipe is busy 6144 of the ~9600 cycles of a step (two waves per SIMD, 96 MFMAs each); the
// rest is the split (without it 95 us where the kernel takes 118, B = 2, T = 1500, H = 16) and the softmax's first
// half. Before, on v_mfma_f32_32x32x2_f32: 201 us there, and at B = 1, T = 64, 16.5 us against 12.1. Fragments
// prefetched in finer steps, and the tiles staged as fp32 in LDS by DMA instead of through registers, took 128 and 120.
//
// Numerics follow the reference: S = scale * Q K^T (FlashAttention.cpp:83-91),
// keys with k_pos > q_pos masked (:102), m = row max of the scaled scores,
// l = sum exp(s - m) (:159-163), output O / l, and a row with l == 0 written as
// zeros (:165-174). The softmax runs in the log2 domain on Q scale log2(e), with
// a reference point that moves only when a score exceeds it by 2^8; m is the true
// row maximum and l is rescaled to it at the end.

#include "flash_items.h"

#include <type_traits>
#include <utility>

namespace dt {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef short shortx8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) shortx4 lds_shortx4;

constexpr int kD = 128;                      // head_dim (model_config.h:3)
constexpr int kBM = kItemRows;               // queries per item
constexpr int kBN = 32;                      // keys per tile
constexpr int kThreads = 512;                // 8 waves
constexpr int kRowK = kD * 2 + 16;           // a row of one of K's planes
constexpr int kRowV = kD * 2 + 64;           // a row of one of V's planes
constexpr int kPlaneK = kBN * kRowK;
constexpr int kPlaneV = kBN * kRowV;
constexpr int kGroupBytes = 3 * (kPlaneK + kPlaneV);  // 55.5 KB
constexpr int kObufRow = kD * 4 + 16;        // a row of the output staging tile
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegInf = -__builtin_huge_valf();
constexpr float kInf = __builtin_huge_valf();
constexpr uint32_t kRescaleExp = 3;  // the reference point moves when a score exceeds it by 2^3 in the log2 domain
constexpr float kUp = 0x1p24f;  // the operands' factor
constexpr int kBufferDword3 = 0x00020000;  // raw buffer, 32-bit data format (gfx9 family)

// LDS: the groups' planes [group](K h, m, l, V h, m, l) in the loop; at an item's end the exchange between the groups
// (xo, xs) and the output tile
constexpr int kXoBytes = 2 * 4 * 8 * 64 * 16;   // 64 KB
constexpr int kXsBytes = 2 * 4 * 3 * 64 * 4;    // 6 KB
constexpr int kLdsBytes = kXoBytes + kXsBytes + kBM * kObufRow;
static_assert(2 * kGroupBytes <= kLdsBytes && kLdsBytes <= 160 * 1024, "LDS of one CU");

template <typename F, int... Is>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
// calls f(std::integral_constant<int, I>{}) for I = 0 .. N-1 (compile-time unrolled)
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}
// keeps each group of MFMAs with the LDS accesses issued beside it: the scheduler may not move work across
#define DT_BUNDLE_END __builtin_amdgcn_sched_barrier(0)

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
    bf16x2 r = __builtin_convertvector((floatx2){lo, hi}, bf16x2);
    return __builtin_bit_cast(uint32_t, r);
}
// the bf16 planes of a pair of floats: x = h + m + l exactly for 0 and |x| in 2^-102 .. 2^127 (fp32 numbers times 2^24)
struct Split2 {
    uint32_t h, m, l;
};
__device__ __forceinline__ Split2 split2(float x0, float x1) {
    Split2 s;
    s.h = pack_bf16x2(x0, x1);
    const float r0 = x0 - __uint_as_float(s.h << 16), r1 = x1 - __uint_as_float(s.h & 0xffff0000u);
    s.m = pack_bf16x2(r0, r1);
    s.l = pack_bf16x2(r0 - __uint_as_float(s.m << 16), r1 - __uint_as_float(s.m & 0xffff0000u));
    return s;
}
// an operand's three planes
struct Frag3 {
    bf16x8 h, m, l;
};
__device__ __forceinline__ floatx16 mfma(bf16x8 a, bf16x8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ floatx16 mfma_f32(float a, float b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Row reductions over the two lane halves (lane l and lane l ^ 32 hold the same query): v_permlane32_swap with x as
// both operands leaves the lower half's value and the upper half's in every lane (the same order in both halves).
__device__ __forceinline__ float max_halves(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_halves(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Buffer descriptor over [base, base + bytes): loads at or past the end return zeros.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, kBufferDword3);
}

__device__ __forceinline__ float4 load16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

__device__ __forceinline__ float load4(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}

// LDS accesses only: vector memory requests in flight (the next tiles, output stores) are not waited for
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The lane, formed anew: what is computed from it belongs to the place of the call and is not kept in registers across the
// item loop, which needs all of them (kept, some forty of them were spilled to scratch memory).
__device__ __forceinline__ int lane_here() {
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}

// likewise the scale
__device__ __forceinline__ float scale_here(float s) {
    asm volatile("" : "+s"(s));
    return s;
}

// Per-wave state of one item: O^T: o[db][i] = O[qrow][32*db + 8*(i/4) + 4*hh + i%4] (unnormalised, relative to m_s). In the
// split products' loop o is 2^48 times that and m_t and m_s are 1 / down times what they say.
struct Acc {
    floatx16 o[4];
    float m_t, m_s, l;  // this lane half's maximum, the reference point (the same in both halves), this half's sum
};

// The wave's keys with v_mfma_f32_32x32x2_f32, operands straight from memory (rk, rv: the sequence's rows, zeros past it):
// tiles kt0, kt0 + 2, ... of the queries' visible ones. Taken when the split products gave a result that is not finite;
// scores that are -inf, +inf or NaN in fp32 arithmetic come out as such here. Inlined, with every index a constant: a call,
// or an element of A picked at run time, would put registers in scratch memory, which the runtime has to allocate.
__device__ __forceinline__ void slow_keys(Acc& A, const float* q, __amdgpu_buffer_rsrc_t rk, __amdgpu_buffer_rsrc_t rv, int ldk,
                                          int ldv, int kt0, int n_tiles, int qw0, int lim, int causal, float c) {
    const int lane = lane_here(), ln = lane & 31, hh = lane >> 5;
    float m_run = kNegInf, l_run = 0.0f;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) A.o[db][i] = 0.0f;
    float4 qx[16];  // k step s of lane half hh is dim 64*hh + s
#pragma unroll
    for (int j = 0; j < 16; ++j) qx[j] = *reinterpret_cast<const float4*>(q + 64 * hh + 4 * j);
#pragma unroll 1
    for (int kt = kt0; kt < n_tiles; kt += 2) {
        const int k0 = kt * kBN;
        if (causal && k0 > qw0 + 31) break;
        floatx16 st;
#pragma unroll
        for (int i = 0; i < 16; ++i) st[i] = 0.0f;
        const uint32_t krow = (uint32_t)((k0 + ln) * ldk + 64 * hh) * 4u;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float4 kx = load16(rk, krow + 16 * j);
            st = mfma_f32(kx.x, qx[j].x, st);
            st = mfma_f32(kx.y, qx[j].y, st);
            st = mfma_f32(kx.z, qx[j].z, st);
            st = mfma_f32(kx.w, qx[j].w, st);
        }
        float tmax = kNegInf;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            if (k0 + 8 * (i / 4) + 4 * hh + (i % 4) > lim) st[i] = kNegInf;
            tmax = fmaxf(tmax, st[i]);
        }
        const float m_new = fmaxf(m_run, max_halves(tmax) * c);
        const float m_use = (m_new == kNegInf) ? 0.0f : m_new;
        const float alpha = exp2f(m_run - m_use);  // 0 when m_run == -inf
        float psum = 0.0f;
        {
#pragma clang fp contract(off)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                st[i] = __builtin_amdgcn_exp2f(st[i] * c - m_use);
                psum += st[i];
            }
        }
        l_run = l_run * alpha + psum;  // this half's keys
        m_run = m_new;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) A.o[db][i] *= alpha;
        const uint32_t vrow = (uint32_t)((k0 + 4 * hh) * ldv + ln) * 4u;
#pragma unroll
        for (int i = 0; i < 16; ++i)
#pragma unroll
            for (int db = 0; db < 4; ++db)
                A.o[db] = mfma_f32(load4(rv, vrow + (uint32_t)((8 * (i / 4) + (i % 4)) * ldv + 32 * db) * 4u), st[i], A.o[db]);
    }
    A.m_t = A.m_s = m_run;
    A.l = l_run;
}

__global__ __launch_bounds__(kThreads, 1) void flash_fwd_f32_kernel(FlashArgs a, Schedule sc) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kLdsBytes];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2;  // key-tile group
    // 32-query block within the item, also this wave's quarter of the group's tiles. Group 1's waves take the blocks
    // in the other half, so each SIMD (waves w and w + 4) holds one wave of each 64 queries: an item whose second
    // 64 rows lie past the sequence's end, or see more keys than its first, still keeps all four SIMDs busy.
    const int wq = (wave & 3) ^ (2 * grp);
    const int ln = lane & 31;   // query within the wave's 32 (MFMA n index)
    const int hh = lane >> 5;   // lane half

    // K fragment chunk cc of row ln: dims 16*cc + 8*hh .. +8
    const uint8_t* const kfrag = lds + grp * kGroupBytes + ln * kRowK + 16 * hh;
    // V transposing reads: lane i of 16-lane group G reads row 4*hh + i/4 (+8 for the second read) of a 16-key chunk,
    // dims 32*db + 16*(G&1) + 4*(i&3) .. +3
    const int i16 = lane & 15;
    const uint8_t* const vfrag =
        lds + grp * kGroupBytes + 3 * kPlaneK + (4 * hh + (i16 >> 2)) * kRowV + 32 * ((lane >> 4) & 1) + 8 * (i16 & 3);
    // this wave's quarter of a tile: unit n is rows 8*n + 2*wq and 8*n + 2*wq + 1, four floats per lane
    const int r0 = 2 * wq + hh;
    uint8_t* const kput = lds + grp * kGroupBytes + r0 * kRowK + 8 * ln;
    uint8_t* const vput = lds + grp * kGroupBytes + 3 * kPlaneK + r0 * kRowV + 8 * ln;
    const uint32_t koff = (uint32_t)((r0 * a.ldk + 4 * ln) * 4);
    const uint32_t voff = (uint32_t)((r0 * a.ldv + 4 * ln) * 4);

    const int T = a.T;
    const int G = gridDim.x;
    // Q's factor: c = scale log2 e times the power of two 2^24 / 2^e, 2^e <= scale < 2^(e+1); and what takes it and K's out of
    // a score again, 2^(e-48), which would be denormal for the smallest scales: such calls take the fp32 instruction
    const uint32_t sb = __float_as_uint(a.scale), se = sb >> 23;  // se = e + 127
    const bool scale_fits = se > 56;
    const float cu = __uint_as_float((sb & 0x7fffffu) | (127u + 24u) << 23) * kLog2e;
    const float down = __uint_as_float((scale_fits ? se - 48 : 127u) << 23);
    const float grow_by = __uint_as_float((scale_fits ? 127u + kRescaleExp + (48 + 127) - se : 127u) << 23);  // 2^kRescaleExp / down

    for (int round = 0;; ++round) {
        const int k_unit = snake_item(round, G, (int)blockIdx.x);
        if (k_unit >= sc.n_units) break;
        const Unit u = decode_unit(k_unit, sc, a.H, sc.cum);  // a whole item: this kernel's schedules split nothing
        const int lane = lane_here(), ln = lane & 31, hh = lane >> 5;
        const int b = u.b, h = u.h;
        const int L = u.L;  // valid keys / rows of this sequence
        const int q0 = u.qa;
        const int qw0 = (wq < 2 ? u.qa : u.qb - 64) + wq * 32;  // first query of this wave
        const int qrow = qw0 + ln;

        const float* Qg = static_cast<const float*>(a.q) + (int64_t)b * T * a.ldq + (int64_t)h * kD;
        const float* Kg = static_cast<const float*>(a.k) + (int64_t)b * T * a.ldk + (int64_t)h * kD;
        const float* Vg = static_cast<const float*>(a.v) + (int64_t)b * T * a.ldv + (int64_t)h * kD;
        float* Og = static_cast<float*>(a.o) + (int64_t)b * T * a.ldo + (int64_t)h * kD;
        const int64_t stat_base = ((int64_t)b * T) * a.H + h;  // m/l index of row t: stat_base + t*H

        if (q0 >= L) {  // every row of this tile is padding: the reference's empty row (l == 0)
            if (grp == 0 && qrow < T) {
                const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
                for (int j = 0; j < 16; ++j) *reinterpret_cast<float4*>(&Og[(int64_t)qrow * a.ldo + 64 * hh + 4 * j]) = z;
                if (hh == 0) {
                    if (a.m) a.m[stat_base + (int64_t)qrow * a.H] = kNegInf;
                    if (a.l) a.l[stat_base + (int64_t)qrow * a.H] = 0.0f;
                }
            }
            continue;  // no LDS was touched: no barrier needed
        }

        const int k_end = a.causal ? min(u.qb + 64, L) : L;
        const int n_tiles = (k_end + kBN - 1) / kBN;
        const int n_steps = (n_tiles + 1) / 2;
        const int lim = a.causal ? min(qrow, L - 1) : L - 1;  // keys > lim are masked

        // unit n of this wave's quarter of the group's tile kt of K (kv = 0) or V (kv = 1), on its way from HBM (zeros
        // past the sequence; nothing is fetched past the last tile)
        const __amdgpu_buffer_rsrc_t rk = make_rsrc(Kg, (uint32_t)L * (uint32_t)a.ldk * 4u);
        const __amdgpu_buffer_rsrc_t rv = make_rsrc(Vg, (uint32_t)L * (uint32_t)a.ldv * 4u);
        auto load = [&](int kv, int kt, int n) {
            const uint32_t ld4 = (uint32_t)(kv ? a.ldv : a.ldk) * 4u;
            const uint32_t row = kt < n_tiles ? (uint32_t)(kt * kBN + 8 * n) * ld4 : 0x80000000u;
            return load16(kv ? rv : rk, (kv ? voff : koff) + row);
        };
        // that unit -> the planes
        auto put = [&](int kv, int n, float4 x) {
            const Split2 s0 = split2(x.x * kUp, x.y * kUp), s1 = split2(x.z * kUp, x.w * kUp);
            uint8_t* p = kv ? vput + n * 8 * kRowV : kput + n * 8 * kRowK;
            const int plane = kv ? kPlaneV : kPlaneK;
            *reinterpret_cast<uint2*>(p) = make_uint2(s0.h, s1.h);
            *reinterpret_cast<uint2*>(p + plane) = make_uint2(s0.m, s1.m);
            *reinterpret_cast<uint2*>(p + 2 * plane) = make_uint2(s0.l, s1.l);
        };
        float4 x[4];  // the units between HBM and the planes: K's and V's in turn
        float4 xk[4];
#pragma unroll
        for (int n = 0; n < 4; ++n) xk[n] = load(0, grp, n);

        // Q fragment, times cu, split: qf[cc] = Q[qrow][16*cc + 8*hh .. +8] * cu
        Frag3 qf[8];
        {
            const float* qp = Qg + (int64_t)min(qrow, T - 1) * a.ldq + 8 * hh;  // (rows past T: any values)
            float4 xq[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) xq[j] = *reinterpret_cast<const float4*>(qp + 16 * (j >> 1) + 4 * (j & 1));
#pragma unroll
            for (int n = 0; n < 4; ++n) x[n] = load(1, grp, n);
#pragma unroll
            for (int n = 0; n < 4; ++n) put(0, n, xk[n]);  // the group's first K tile
#pragma unroll
            for (int cc = 0; cc < 8; ++cc) {
                const float4 x0 = xq[2 * cc], x1 = xq[2 * cc + 1];
                const Split2 s0 = split2(x0.x * cu, x0.y * cu), s1 = split2(x0.z * cu, x0.w * cu);
                const Split2 s2 = split2(x1.x * cu, x1.y * cu), s3 = split2(x1.z * cu, x1.w * cu);
                qf[cc].h = __builtin_bit_cast(bf16x8, make_uint4(s0.h, s1.h, s2.h, s3.h));
                qf[cc].m = __builtin_bit_cast(bf16x8, make_uint4(s0.m, s1.m, s2.m, s3.m));
                qf[cc].l = __builtin_bit_cast(bf16x8, make_uint4(s0.l, s1.l, s2.l, s3.l));
            }
        }
        Acc A;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) A.o[db][i] = 0.0f;
        A.m_t = kNegInf;
        A.m_s = kNegInf;
        A.l = 0.0f;
        uint64_t low = 0;  // the lanes that had a score of -inf

        lds_barrier();

        // group 1 runs half a step behind group 0: one group's softmax issues under the other's PV product
        const bool skew = n_steps >= 4;
        if (grp && skew) lds_barrier();
        for (int it = 0; it < n_steps; ++it) {
            const int kt = 2 * it + grp;
            const int k0 = kt * kBN;
            const bool visible = kt < n_tiles && qw0 < L && !(a.causal && k0 > qw0 + 31);
            floatx16 st;
            uint32_t pw[3][8];  // P's planes, packed pairs
            auto split_p = [&](int j) {
                const Split2 s = split2(st[2 * j] * kUp, st[2 * j + 1] * kUp);
                pw[0][j] = s.h;
                pw[1][j] = s.m;
                pw[2][j] = s.l;
            };
            if (visible) {
                // S^T, with V's planes written under it: st[i] = t[qrow][key] / down, key = k0 + 8*(i/4) + 4*hh + i%4; the five
                // small partial products of every chunk first, then the large one (K's h plane is read again for it).
                // Fragments are read one chunk ahead of their MFMAs.
                auto read_k = [&](int cc, int p) {
                    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(kfrag + 32 * cc + p * kPlaneK));
                };
                auto read_k3 = [&](int cc) { return Frag3{read_k(cc, 0), read_k(cc, 1), read_k(cc, 2)}; };
#pragma unroll
                for (int i = 0; i < 16; ++i) st[i] = 0.0f;
                __builtin_amdgcn_s_setprio(2);
                Frag3 kr[2];
                bf16x8 kh[4];
                kr[0] = read_k3(0);
                static_for<8>([&](auto CC) {
                    constexpr int cc = decltype(CC)::value;
                    if constexpr (cc + 1 < 8) kr[(cc + 1) & 1] = read_k3(cc + 1);
                    else kh[0] = read_k(0, 0), kh[1] = read_k(1, 0);
                    const Frag3 k = kr[cc & 1];
                    st = mfma(k.l, qf[cc].h, st);
                    st = mfma(k.h, qf[cc].l, st);
                    st = mfma(k.m, qf[cc].m, st);
                    st = mfma(k.m, qf[cc].h, st);
                    st = mfma(k.h, qf[cc].m, st);
                    if constexpr (cc & 1) {
                        put(1, cc / 2, x[cc / 2]);
                        x[cc / 2] = load(0, kt + 2, cc / 2);
                    }
                    DT_BUNDLE_END;
                });
                static_for<4>([&](auto C2) {
                    constexpr int c2 = decltype(C2)::value;
                    if constexpr (c2 < 3) kh[2 * ((c2 + 1) & 1)] = read_k(2 * c2 + 2, 0), kh[2 * ((c2 + 1) & 1) + 1] = read_k(2 * c2 + 3, 0);
                    st = mfma(kh[2 * (c2 & 1)], qf[2 * c2].h, st);
                    st = mfma(kh[2 * (c2 & 1) + 1], qf[2 * c2 + 1].h, st);
                    DT_BUNDLE_END;
                });

                {  // (as bit patterns: below 0 a lower score is a larger one, -inf 0xff800000)
                    uint32_t u0 = __float_as_uint(st[0]), u1 = __float_as_uint(st[1]);
#pragma unroll
                    for (int i = 2; i < 16; i += 2) {
                        u0 = max(u0, __float_as_uint(st[i]));
                        u1 = max(u1, __float_as_uint(st[i + 1]));
                    }
                    low |= __builtin_amdgcn_ballot_w64(max(u0, u1) >= 0xff800000u);
                }
                if (k0 + kBN > L || (a.causal && k0 + kBN - 1 > qw0)) {  // diagonal / ragged tail only
                    asm volatile("");  // keeps this block a branch
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (k0 + 8 * (i / 4) + 4 * hh + (i % 4) > lim) st[i] = kNegInf;
                }
                float t0 = st[0], t1 = st[1];
#pragma unroll
                for (int i = 2; i < 16; i += 2) {
                    t0 = fmaxf(t0, st[i]);
                    t1 = fmaxf(t1, st[i + 1]);
                }
                const float tmax = fmaxf(t0, t1);
                A.m_t = fmaxf(A.m_t, tmax);
                const bool grow = (A.m_s == kNegInf) ? (tmax > kNegInf) : (tmax > A.m_s + grow_by);
                if (__builtin_amdgcn_ballot_w64(grow) != 0) {  // wave-uniform, rare after the first tile
                    asm volatile("");  // keeps this block a branch
                    const float m_new = max_halves(A.m_t);
                    const float alpha = (A.m_s == kNegInf) ? 0.0f : exp2f((A.m_s - m_new) * down);
                    A.m_s = m_new;
                    A.l *= alpha;
#pragma unroll
                    for (int db = 0; db < 4; ++db)
#pragma unroll
                        for (int i = 0; i < 16; ++i) A.o[db][i] *= alpha;
                }
                const float ref = (A.m_s == kNegInf) ? 0.0f : A.m_s * down;
                float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
                for (int i = 0; i < 16; i += 2) {
                    st[i] = __builtin_amdgcn_exp2f(fmaf(st[i], down, -ref));
                    st[i + 1] = __builtin_amdgcn_exp2f(fmaf(st[i + 1], down, -ref));
                    s0 += st[i];
                    s1 += st[i + 1];
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) split_p(j);  // (the second 16 keys' under the PV product)
                A.l += s0 + s1;
                __builtin_amdgcn_s_setprio(0);
            } else {
#pragma unroll
                for (int n = 0; n < 4; ++n) {
                    put(1, n, x[n]);
                    x[n] = load(0, kt + 2, n);
                }
            }
            lds_barrier();  // V's planes are written, K's are free

            if (visible) {
                // O^T += V^T P^T with the next K tile's planes written under it. Chunk ch = 4*u + db: 16 keys u, 32 dims
                // db; k index 8*hh + e <-> key 16*u + 8*(e/4) + 4*hh + e%4. Two chunks' accumulators alternate.
                auto read_v = [&](int ch, int p) {
                    const uint8_t* at = vfrag + p * kPlaneV + (ch >> 2) * 16 * kRowV + 64 * (ch & 3);
                    const shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)at);
                    const shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)(at + 8 * kRowV));
                    return __builtin_bit_cast(bf16x8, (shortx8){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
                };
                auto frag_p = [&](int p, int u) {
                    return __builtin_bit_cast(bf16x8, make_uint4(pw[p][4 * u], pw[p][4 * u + 1], pw[p][4 * u + 2], pw[p][4 * u + 3]));
                };
                // fragment f = 3 * ch + (0: l, 1: m, 2: h), read 2 ahead
                bf16x8 vr[3];
#pragma unroll
                for (int f = 0; f < 2; ++f) vr[f] = read_v(f / 3, 2 - f % 3);
                static_for<24>([&](auto F) {
                    constexpr int f = decltype(F)::value, u = f / 12, db = (f / 3) & 3;
                    if constexpr (f + 2 < 24) vr[(f + 2) % 3] = read_v((f + 2) / 3, 2 - (f + 2) % 3);
                    const bf16x8 v = vr[f % 3];
                    if constexpr (f % 3 == 2) A.o[db] = mfma(v, frag_p(2, u), A.o[db]);
                    if constexpr (f % 3 >= 1) A.o[db] = mfma(v, frag_p(1, u), A.o[db]);
                    A.o[db] = mfma(v, frag_p(0, u), A.o[db]);
                    if constexpr (f >= 4 && f < 8) split_p(f);
                    if constexpr (f % 6 == 5) {
                        put(0, f / 6, x[f / 6]);
                        x[f / 6] = load(1, kt + 2, f / 6);
                    }
                    DT_BUNDLE_END;
                });
            } else {
#pragma unroll
                for (int n = 0; n < 4; ++n) {
                    put(0, n, x[n]);
                    x[n] = load(1, kt + 2, n);
                }
            }
            lds_barrier();  // the next K's planes are written, V's are free
        }
        if (!grp && skew) lds_barrier();

        float f = 1.0f / (kUp * kUp), fm = down;  // take the operands' factors out
        {
            // a result that is not finite, an empty softmax over visible keys, or a score of -inf: the wave's keys again,
            // in fp32
            float z = A.l * 0.0f;
#pragma unroll
            for (int db = 0; db < 4; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i) z = fmaf(A.o[db][i], 0.0f, z);
            const bool keys = qrow < L && grp * kBN <= lim;
            const bool bad = keys && (!(z == 0.0f) || !(sum_halves(A.l) > 0.0f) || !scale_fits);
            if ((__builtin_amdgcn_ballot_w64(bad) | (low & __builtin_amdgcn_ballot_w64(keys))) != 0) {
                slow_keys(A, Qg + (int64_t)min(qrow, T - 1) * a.ldq, rk, rv, a.ldk, a.ldv, grp, n_tiles, qw0, lim, a.causal,
                          scale_here(a.scale) * kLog2e);
                f = fm = 1.0f;
            }
        }

        {
            // Merge: group g finalises dims 64g .. 64g+63 of its block's rows and hands the other half of its partial O to the
            // other group (float4 k of lane `lane` at xo(g)[k*64 + lane]), with its (m_s, m_t, l) at xs(g). The loop's last
            // barrier has freed the planes.
            A.m_t = max_halves(A.m_t) * fm;
            A.m_s *= fm;
            A.l = sum_halves(A.l);
            const int lane = lane_here(), ln = lane & 31, hh = lane >> 5, qrow = qw0 + ln;
            auto xo = [&](int g) { return reinterpret_cast<float4*>(lds) + (g * 4 + wq) * (8 * 64); };
            auto xs = [&](int g) { return reinterpret_cast<float*>(lds + kXoBytes) + (g * 4 + wq) * (3 * 64); };
            uint8_t* obuf = lds + kXoBytes + kXsBytes;  // the output tile on its way to HBM
            {
                float4* out = xo(grp);
                auto hand = [&](auto DB) {
                    constexpr int db = decltype(DB)::value;
#pragma unroll
                    for (int I = 0; I < 4; ++I)
                        out[(4 * (db & 1) + I) * 64 + lane] =
                            make_float4(A.o[db][4 * I] * f, A.o[db][4 * I + 1] * f, A.o[db][4 * I + 2] * f, A.o[db][4 * I + 3] * f);
                };
                if (grp == 0) {
                    hand(std::integral_constant<int, 2>{});
                    hand(std::integral_constant<int, 3>{});
                } else {
                    hand(std::integral_constant<int, 0>{});
                    hand(std::integral_constant<int, 1>{});
                }
                float* s = xs(grp);
                s[lane] = A.m_s;
                s[64 + lane] = A.m_t;
                s[128 + lane] = A.l;
            }
            lds_barrier();
            {
                // both groups form the same statistics, group 0's terms first (FlashAttention.cpp:159-175)
                const float* so = xs(1 - grp);
                const float os = so[lane], ot = so[64 + lane], ol = so[128 + lane];
                const float m0s = grp ? os : A.m_s, m1s = grp ? A.m_s : os;
                const float m0t = grp ? ot : A.m_t, m1t = grp ? A.m_t : ot;
                const float l0 = grp ? ol : A.l, l1 = grp ? A.l : ol;
                const float ms = fmaxf(m0s, m1s);
                const float a0 = (m0s == kNegInf) ? 0.0f : exp2f(m0s - ms);
                const float a1 = (m1s == kNegInf) ? 0.0f : exp2f(m1s - ms);
                const float l = l0 * a0 + l1 * a1;
                const float mt = fmaxf(m0t, m1t);
                const bool valid = qrow < L && l > 0.0f;
                const float inv = valid ? 1.0f / l : 0.0f;
                const float4* in = xo(1 - grp);
                uint8_t* orow = obuf + (32 * wq + ln) * kObufRow + 16 * hh;
                auto fin = [&](auto DB) {
                    constexpr int db = decltype(DB)::value;
#pragma unroll
                    for (int I = 0; I < 4; ++I) {
                        const float4 y = in[(4 * (db & 1) + I) * 64 + lane];
                        const float yv[4] = {y.x, y.y, y.z, y.w};
                        float v[4];
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const float own = A.o[db][4 * I + r] * f;
                            const float x = (db < 2) ? own * a0 + yv[r] * a1 : yv[r] * a0 + own * a1;
                            const float q = x * inv;  // x / l (l >= 1), with one correction step
                            const float e = fmaf(fmaf(-q, l, x), inv, q);
                            v[r] = valid ? (fabsf(q) < kInf ? e : q) : 0.0f;
                        }
                        *reinterpret_cast<float4*>(orow + 32 * (4 * db + I)) = make_float4(v[0], v[1], v[2], v[3]);
                    }
                };
                if (grp == 0) {
                    fin(std::integral_constant<int, 0>{});
                    fin(std::integral_constant<int, 1>{});
                    if (qrow < T && hh == 0) {
                        if (a.m) a.m[stat_base + (int64_t)qrow * a.H] = valid ? mt * (a.scale / (scale_here(a.scale) * kLog2e)) : kNegInf;
                        if (a.l) a.l[stat_base + (int64_t)qrow * a.H] = valid ? l * exp2f(ms - mt) : 0.0f;
                    }
                } else {
                    fin(std::integral_constant<int, 2>{});
                    fin(std::integral_constant<int, 3>{});
                }
            }
            lds_barrier();
            // the item's 128 output rows: 32 lanes per 512-byte row, 2 rows per store instruction
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int ch = j * kThreads + 64 * wave + lane;  // 16-byte chunk ch % 32 of row ch / 32
                const int r = ch >> 5, cq = ch & 31;
                const int qr = (j < 4 ? u.qa : u.qb - 64) + r;  // rows 0-63 in j < 4
                const float4 w = *reinterpret_cast<const float4*>(obuf + r * kObufRow + 16 * cq);
                if (qr < T) *reinterpret_cast<float4*>(&Og[(int64_t)qr * a.ldo + 4 * cq]) = w;
            }
        }
        // every wave has read the output tile before the next item's planes may overwrite it; the output stores need not
        // have completed
        lds_barrier();
    }
}

}  // namespace

int launch_flash_fwd_f32(const FlashArgs& a, const SeqLens* lens, hipStream_t stream) {
    SeqLens sl;
    if (a.ragged) sl = *lens;
    else sl.len[0] = a.T;
    const int64_t ld = a.ldk > a.ldv ? a.ldk : a.ldv;
    if ((int64_t)a.T * ld * 4 >= ((int64_t)1 << 31))
        return set_error(DT_ERR_UNSUPPORTED, "K/V extent of one sequence exceeds 2 GiB");
    int grid = 0;
    DT_TRY(persistent_grid((int64_t)((a.T + kBM - 1) / kBM) * a.B * a.H, &grid));
    Schedule sc;
    build_schedule(a, sl, grid, false, &sc, true);
    hipLaunchKernelGGL(flash_fwd_f32_kernel, dim3(grid), dim3(kThreads), 0, stream, a, sc);
    DT_HIP_TRY(hipGetLastError());
    return DT_OK;
}

}  // namespace dt
