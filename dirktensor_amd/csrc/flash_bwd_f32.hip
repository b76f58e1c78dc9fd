// Causal flash attention backward, fp32 exact mode, for gfx950 (CDNA4).
//
// Replaces flash_attention_backward (FlashAttention.cpp:185-359) with fp32 tensors. As in the forward
// (flash_fwd_f32.hip), every fp32 product runs on v_mfma_f32_32x32x16_bf16: an operand x is the exact sum of three
// bf16 values h + m + l, and x y is formed from six of their partial products (the other three come to 2^-24 of x y at most),
// small ones first, accumulated in fp32. That is 192 matrix-pipe cycles per 16 steps of k against 512 on
// v_mfma_f32_32x32x2_f32, with less rounding (it rounds every second k). Every operand, P and dS too, is split times 2^24,
// so that no part of any fp32 number is lost under bf16's denormals; that is taken out again where a score enters exp2, in
// dP, and at a block's end. What a split does not hold (2^103 and above, infinities, NaN) shows in a result that is not
// finite or in a score of -inf, and the wave then repeats its block with the fp32 instruction, straight from memory
// (slow_dkdv, slow_dq).
//
// Decomposition, as in the bf16 mode: flash_bwd_dkdv owns a block of keys of one (batch, head), 32 per wave with the
// planes of their K and V rows in registers, and streams 32-query tiles of Q and dO; flash_bwd_dq owns queries (Q and
// dO planes in registers) and streams 32-key tiles of K and V. Each gradient row has a single owner, so no atomics; S
// and dP are computed in both. Each workgroup owns one block; the grid lists the blocks in decreasing causal cost, so
// the hardware's first-free-CU dispatch runs the longest blocks first. With more than one block per CU and pass the
// dS path replaces the dQ kernel: the dK/dV kernel also stores dS (fp32) and flash_bwd_dq_ds forms dQ = dS K from it
// (5 products per tile pair instead of 7).
//
// A workgroup is 4 waves in G groups; the groups hold the same block and take alternate tiles, each with LDS of its
// own, and add up their partial gradients at the end. G = 1: blocks of 128 rows; G = 2: blocks of 64, twice as many
// of half the length, where 128-row blocks would leave the longest one to set the time (flash_bwd_two_groups).
//
// A streamed tile passes through registers: a thread loads four floats of a row at a time, a phase or two ahead,
// splits them and writes the three planes under the MFMAs of another product. Per tile and wave (dK/dV):
//   S = Q K^T      under it: Q planes of the next tile
//   dP = dO V^T    under it: P = exp2(S c - lse2) and its split
//   dV^T += dO^T P under it: dS = P (dP - delta) and its split      -- then a barrier: dO's planes are free
//   dK^T += Q^T dS under it: dO planes of the next tile             -- then a barrier: the next tile is ready
// so Q has two sets of planes and dO one (72 KB with the row statistics, 145 KB for two groups). dQ is the same with
// K, V in the places of Q, dO, and one product less.
//
// What bounds it: the matrix pipe, 192 MFMAs per tile and wave for dK/dV at one wave per SIMD (K, V, dK and dV of 32 keys
// take 320 of a lane's 512 registers), and with few blocks the longest of them. B = 1, H = 16, us per call against the
// same decomposition on v_mfma_f32_32x32x2_f32: T = 1000 268 -> 109, T = 2048 568 -> 325, T = 4096 1540 -> 998.
//
// LDS planes: 32 rows of 256 bytes, 16-byte chunk c of row r at c ^ swz(r), swz(r) = 4*(r & 3) + ((r >> 2) & 3):
// row-wise fragment reads, transposing reads (ds_read_b64_tr_b16, in the accumulator's row order) and the split's
// 8-byte writes are all free of bank conflicts.
//
// MFMA operand layouts: the A operand is a 32-row fragment, lane l holding row l%32 and k elements 8*(l/32) .. +8; the
// B operand a 32-column fragment, lane l holding column l%32 and the same k elements; accumulator element i of lane l
// is row 8*(i/4) + 4*(l/32) + i%4, column l%32, so an accumulator's 8 elements 8u .. 8u+7 are a B operand over 16 rows
// in that order.

#include "dt_internal.h"

#include <climits>

#include <type_traits>
#include <utility>

namespace dt {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef short shortx8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) shortx4 lds_shortx4;

constexpr int kD = 128;
constexpr int kTile = 32;                        // rows per streamed tile
constexpr int kRow = kD * 2;                     // a row of a bf16 plane
constexpr int kPlane = kTile * kRow;             // 8 KB
constexpr int kPlanes = 3 * kPlane;              // h, m, l
constexpr int kBlk = 128;                        // rows owned by a workgroup of one group
constexpr int kThreads = 256;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kUp = 0x1p24f;      // the operands' factor
constexpr float kDown2 = 0x1p-48f;  // takes it out of a product
constexpr int kBufferDword3 = 0x00020000;  // raw buffer, 32-bit data format (gfx9 family)

__device__ __forceinline__ floatx16 mfma(bf16x8 a, bf16x8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ floatx16 mfma_f32(float a, float b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ floatx16 zero16() {
    floatx16 z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.0f;
    return z;
}

template <typename F, int... Is>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
// calls f(std::integral_constant<int, I>{}) for I = 0 .. N-1 (compile-time unrolled)
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}
// keeps each group of MFMAs with the work issued beside it: the scheduler may not move work across
#define DT_BUNDLE_END __builtin_amdgcn_sched_barrier(0)

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
// LDS accesses complete before any wave passes; loads in flight are not waited for
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

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
// sixteen accumulator elements (two B operands) times 2^24, packed pair by pair
struct Words3 {
    uint32_t w[3][8];  // [h, m, l][pair of elements]
    __device__ __forceinline__ void put(int pair, float x0, float x1) {
        const Split2 s = split2(x0 * kUp, x1 * kUp);
        w[0][pair] = s.h;
        w[1][pair] = s.m;
        w[2][pair] = s.l;
    }
    __device__ __forceinline__ bf16x8 frag(int p, int u) const {
        return __builtin_bit_cast(bf16x8, make_uint4(w[p][4 * u], w[p][4 * u + 1], w[p][4 * u + 2], w[p][4 * u + 3]));
    }
};
__device__ __forceinline__ int swz(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

// Lane addresses inside a plane.
struct LaneAddr {
    uint32_t raddr[8];     // row fragment chunk cc: row ln, dims 16*cc + 8*hh .. +8
    uint32_t taddr[2][4];  // transposing read s of dim block db in a 16-row chunk (chunk u adds 4096)
};
__device__ __forceinline__ LaneAddr lane_addr(int lane) {
    LaneAddr A;
    const int ln = lane & 31, hh = lane >> 5;
    const int g = hh ^ swz(ln);
#pragma unroll
    for (int cc = 0; cc < 8; ++cc) A.raddr[cc] = (uint32_t)(ln * kRow + (((2 * cc) ^ g) << 4));
    // lane i of 16-lane group g2 reads row 4*hh + i/4 (+8 for s = 1), dims 32*db + 16*(g2 & 1) + 4*(i & 3) .. +3
    const int i16 = lane & 15;
    const int g2 = (lane >> 4) & 1;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int r = 4 * hh + (i16 >> 2) + 8 * s;
#pragma unroll
        for (int db = 0; db < 4; ++db) {
            const int chunk = 4 * db + 2 * g2 + ((i16 & 3) >> 1);
            A.taddr[s][db] = (uint32_t)(r * kRow + ((chunk ^ swz(r)) << 4) + 8 * (i16 & 1));
        }
    }
    return A;
}

// The product over the head dimension: rows of a tile (M) times the lane's row f (N), the five small partial products
// of every chunk first, then the large one (whose plane is read again). Fragments are read one chunk ahead; ride(I)
// is issued beside bundle I of 12. kSwap: partial products in the order that the product with the roles exchanged has, so
// that S and dP, and with them dS, have the same bits in the dK/dV pass (tiles of Q and dO) and the dQ pass (of K and V).
template <bool kSwap = false, typename Ride>
__device__ __forceinline__ floatx16 dot_rows(const uint8_t* tile, const LaneAddr& LA, const Frag3 (&f)[8], Ride&& ride) {
    auto rd = [&](int cc, int p) {
        return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(tile + LA.raddr[cc] + p * kPlane));
    };
    auto rd3 = [&](int cc) { return Frag3{rd(cc, 0), rd(cc, 1), rd(cc, 2)}; };
    floatx16 c = zero16();
    Frag3 x[2];
    bf16x8 xh[4];
    x[0] = rd3(0);
    static_for<8>([&](auto CC) {
        constexpr int cc = decltype(CC)::value;
        if constexpr (cc + 1 < 8) x[(cc + 1) & 1] = rd3(cc + 1);
        else xh[0] = rd(0, 0), xh[1] = rd(1, 0);
        const Frag3 k = x[cc & 1];
        if constexpr (!kSwap) {
            c = mfma(k.l, f[cc].h, c);
            c = mfma(k.h, f[cc].l, c);
            c = mfma(k.m, f[cc].m, c);
            c = mfma(k.m, f[cc].h, c);
            c = mfma(k.h, f[cc].m, c);
        } else {
            c = mfma(k.h, f[cc].l, c);
            c = mfma(k.l, f[cc].h, c);
            c = mfma(k.m, f[cc].m, c);
            c = mfma(k.h, f[cc].m, c);
            c = mfma(k.m, f[cc].h, c);
        }
        ride(CC);
        DT_BUNDLE_END;
    });
    static_for<4>([&](auto C2) {
        constexpr int c2 = decltype(C2)::value;
        if constexpr (c2 < 3) xh[2 * ((c2 + 1) & 1)] = rd(2 * c2 + 2, 0), xh[2 * ((c2 + 1) & 1) + 1] = rd(2 * c2 + 3, 0);
        c = mfma(xh[2 * (c2 & 1)], f[2 * c2].h, c);
        c = mfma(xh[2 * (c2 & 1) + 1], f[2 * c2 + 1].h, c);
        ride(std::integral_constant<int, 8 + c2>{});
        DT_BUNDLE_END;
    });
    return c;
}
// acc[db] += the tile's rows (k) transposed times w, over its 32 rows; ride(I) beside chunk I = 4*u + db of 8
template <typename Ride>
__device__ __forceinline__ void acc_cols(floatx16 (&acc)[4], const uint8_t* tile, const LaneAddr& LA, const Words3& w, Ride&& ride) {
    auto rd = [&](int ch, int p) {
        const uint32_t off = (uint32_t)(p * kPlane + (ch >> 2) * 16 * kRow);
        const shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)(tile + LA.taddr[0][ch & 3] + off));
        const shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)(tile + LA.taddr[1][ch & 3] + off));
        return __builtin_bit_cast(bf16x8, (shortx8){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
    };
    auto rd3 = [&](int ch) { return Frag3{rd(ch, 0), rd(ch, 1), rd(ch, 2)}; };
    Frag3 x[2];
    x[0] = rd3(0);
    static_for<8>([&](auto CH) {
        constexpr int ch = decltype(CH)::value, u = ch >> 2, db = ch & 3;
        if constexpr (ch + 1 < 8) x[(ch + 1) & 1] = rd3(ch + 1);
        const Frag3 v = x[ch & 1];
        acc[db] = mfma(v.l, w.frag(0, u), acc[db]);
        acc[db] = mfma(v.h, w.frag(2, u), acc[db]);
        acc[db] = mfma(v.m, w.frag(1, u), acc[db]);
        acc[db] = mfma(v.m, w.frag(0, u), acc[db]);
        acc[db] = mfma(v.h, w.frag(1, u), acc[db]);
        acc[db] = mfma(v.h, w.frag(0, u), acc[db]);
        ride(CH);
        DT_BUNDLE_END;
    });
}

// A group's share of the streaming: unit n (0 .. 4G-1) is the four floats 4*ln .. +3 of row (8/G)*n + 2*w + hh of a
// tile, w the wave within its group.
template <int G>
struct Stream {
    static constexpr int kUnits = 4 * G;
    uint32_t waddr;  // of unit 0 in a plane
    uint32_t off;    // of unit 0 in the tensor's rows, bytes
    uint32_t ld4;    // the tensor's row stride, bytes
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ Stream(const float* base, int T, int ld, int lane, int w)
        : off((uint32_t)((2 * w + (lane >> 5)) * ld + 4 * (lane & 31)) * 4u),
          ld4((uint32_t)ld * 4u),
          r(make_rsrc(base, (uint32_t)T * (uint32_t)ld * 4u)) {
        const int row = 2 * w + (lane >> 5), ln = lane & 31;
        waddr = (uint32_t)(row * kRow + (((ln >> 1) ^ swz(row)) << 4) + 8 * (ln & 1));
    }
    // byte offset of a tile's first row; a tile at or past n_tiles is not fetched (its loads return zeros, as do rows
    // at or past T). Formed once per tile: a condition per load would end a scheduling region each time.
    __device__ __forceinline__ uint32_t at(int tile, int row0, int n_tiles) const {
        return (uint32_t)(row0 + min(tile, n_tiles) * kTile) * ld4 | (tile < n_tiles ? 0u : 0x80000000u);
    }
    __device__ __forceinline__ float4 load(uint32_t tile_at, int n) const {
        return load16(r, off + (tile_at + (uint32_t)((8 / G) * n) * ld4));
    }
    __device__ __forceinline__ void put(uint8_t* planes, int n, float4 x) const {
        const Split2 s0 = split2(x.x * kUp, x.y * kUp), s1 = split2(x.z * kUp, x.w * kUp);
        // swz's upper bits count rows of 8/G: G = 1 flips bit 1 on odd units, G = 2 takes n mod 4
        const uint32_t flip = G == 1 ? (uint32_t)(n & 1) << 5 : (uint32_t)(n & 3) << 4;
        uint8_t* p = planes + ((waddr ^ flip) + (uint32_t)(n * (8 / G) * kRow));
        *reinterpret_cast<uint2*>(p) = make_uint2(s0.h, s1.h);
        *reinterpret_cast<uint2*>(p + kPlane) = make_uint2(s0.m, s1.m);
        *reinterpret_cast<uint2*>(p + 2 * kPlane) = make_uint2(s0.l, s1.l);
    }
};

// the lane's own row, split: f[cc] = X[row][16*cc + 8*hh .. +8] * 2^24 (zeros when row >= T)
__device__ __forceinline__ void load_frags(Frag3 (&f)[8], const float* base, int row, int T, int ld, int hh) {
    const bool in = row < T;
    const float* p = base + (int64_t)(in ? row : 0) * ld + 8 * hh;
    float4 x[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) x[j] = *reinterpret_cast<const float4*>(p + 16 * (j >> 1) + 4 * (j & 1));
    auto up = [&](float v) { return in ? v * kUp : 0.0f; };
#pragma unroll
    for (int cc = 0; cc < 8; ++cc) {
        const float4 a = x[2 * cc], b = x[2 * cc + 1];
        const Split2 s0 = split2(up(a.x), up(a.y)), s1 = split2(up(a.z), up(a.w));
        const Split2 s2 = split2(up(b.x), up(b.y)), s3 = split2(up(b.z), up(b.w));
        f[cc].h = __builtin_bit_cast(bf16x8, make_uint4(s0.h, s1.h, s2.h, s3.h));
        f[cc].m = __builtin_bit_cast(bf16x8, make_uint4(s0.m, s1.m, s2.m, s3.m));
        f[cc].l = __builtin_bit_cast(bf16x8, make_uint4(s0.l, s1.l, s2.l, s3.l));
    }
}
// accumulator X^T (4 blocks of 32 dims x 32 rows, lane = row) * mul -> row `row` of [T][ld] at base
__device__ __forceinline__ void store_rows(float* base, int row, int ld, int hh, const floatx16 (&x)[4], float mul) {
    float* p = base + (int64_t)row * ld;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<float4*>(p + 32 * db + 8 * g + 4 * hh) =
                make_float4(x[db][4 * g] * mul, x[db][4 * g + 1] * mul, x[db][4 * g + 2] * mul, x[db][4 * g + 3] * mul);
}
// 0 for finite accumulators, NaN otherwise
__device__ __forceinline__ float finite_probe(const floatx16 (&x)[4]) {
    float z = 0.0f;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) z = fmaf(x[db][i], 0.0f, z);
    return z;
}

// Keeps a block's finished sums apart from the registers its loop accumulates in (without it the compiler gives the loop's
// accumulators a place that suits the tail, and spills some eighty registers around the loop).
__device__ __forceinline__ void settle(floatx16 (&x)[4]) { asm volatile("" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3])); }
// A score's factor scale log2 e 2^-48 is denormal for the smallest scales: such calls take the fp32 instruction. (scale > 0;
// compared as an integer, in scalar registers.)
__device__ __forceinline__ bool scale_fits(float scale) { return __float_as_int(scale) > (127 - 70) << 23; }

// The lane, formed anew: what is computed from it belongs to the place of the call and is not kept in registers before it.
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
// The fp32 rows of one (batch, head) for the fp32 instruction, straight from memory (rows at or past T: zeros)
struct Rows {
    __amdgpu_buffer_rsrc_t r;
    uint32_t ld4;
    __device__ __forceinline__ Rows(const void* base, int b, int h, int T, int ld)
        : r(make_rsrc(static_cast<const float*>(base) + (int64_t)b * T * ld + (int64_t)h * kD, (uint32_t)T * (uint32_t)ld * 4u)),
          ld4((uint32_t)ld * 4u) {}
    __device__ __forceinline__ float at(int row, int dim) const { return load4(r, (uint32_t)row * ld4 + 4u * dim); }
    // dims 64*hh .. +63 of a row
    __device__ __forceinline__ void half_row(float4 (&x)[16], int row, int hh) const {
#pragma unroll
        for (int j = 0; j < 16; ++j) x[j] = load16(r, (uint32_t)row * ld4 + 256u * hh + 16u * j);
    }
    // this lane's row (M) times the lane's half row f (N)
    __device__ __forceinline__ floatx16 dot(int row, int hh, const float4 (&f)[16]) const {
        floatx16 c = zero16();
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float4 x = load16(r, (uint32_t)row * ld4 + 256u * hh + 16u * j);
            c = mfma_f32(x.x, f[j].x, c);
            c = mfma_f32(x.y, f[j].y, c);
            c = mfma_f32(x.z, f[j].z, c);
            c = mfma_f32(x.w, f[j].w, c);
        }
        return c;
    }
};

// LDS of one group: the first operand's planes twice, the second's once, and for dK/dV the tile rows' lse2 and delta
struct GroupLds {
    uint8_t a[2][kPlanes];
    uint8_t b[kPlanes];
    float stats[2][2][kTile];
};
template <int G>
union BwdLds {
    GroupLds g[G];
    float4 x[4][16][64];  // the groups' exchange (G = 2): 64 KB
};
static_assert(sizeof(BwdLds<2>) <= 160 * 1024, "LDS of one CU");

// The two groups' partial sums: group g keeps own + other of `keep` and hands `give` over (group 0's terms first).
__device__ __forceinline__ void add_groups(floatx16 (&keep)[4], const floatx16 (&give)[4], float f, float4 (&x)[4][16][64], int grp, int wave, int lane) {
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            x[wave][4 * db + g][lane] = make_float4(give[db][4 * g] * f, give[db][4 * g + 1] * f, give[db][4 * g + 2] * f, give[db][4 * g + 3] * f);
    lds_barrier();
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const float4 y = x[wave ^ 2][4 * db + g][lane];
            keep[db][4 * g] = keep[db][4 * g] * f + y.x;
            keep[db][4 * g + 1] = keep[db][4 * g + 1] * f + y.y;
            keep[db][4 * g + 2] = keep[db][4 * g + 2] * f + y.z;
            keep[db][4 * g + 3] = keep[db][4 * g + 3] * f + y.w;
        }
}

// ------------------------------------------------------------------------------------------------ dK, dV
// dS workspace blocks (the dS path): per 128-key block and 64-query tile, 128 key rows of 256 bytes (the 64 queries of
// the tile), chunk c of a row holding queries 4c .. 4c+3 (one dK/dV lane's four consecutive accumulator rows).
constexpr int kDsRowBytes = 256;
constexpr int kDsBlockBytes = 128 * kDsRowBytes;  // 32 KB

struct KvAcc {
    floatx16 dv[4], dk[4];
};
// The wave's dK and dV with v_mfma_f32_32x32x2_f32, operands straight from memory (k step s of lane half hh is dim 64*hh + s,
// or one row per half). This and the two below are inlined, with every index a constant: a call, or an element picked at run
// time, would put registers in scratch memory, which the runtime has to allocate.
__device__ __forceinline__ void slow_dkdv(KvAcc& A, const FlashBwdArgs& a, int bh, int kw, int tile0, int step, int n_tiles, int q_begin,
                                          bool emit) {
    const int lane = lane_here(), ln = lane & 31, hh = lane >> 5;
    const int T = a.T, key = kw + ln, b = bh / a.H, h = bh % a.H;
    const float c = scale_here(a.scale) * kLog2e;
    const Rows Q(a.q, b, h, T, a.ld_qkv), K(a.k, b, h, T, a.ld_qkv), V(a.v, b, h, T, a.ld_qkv), G(a.d_o, b, h, T, a.ld_o);
    const __amdgpu_buffer_rsrc_t rl = make_rsrc(a.lse2 + (int64_t)bh * T, (uint32_t)T * 4u);
    const __amdgpu_buffer_rsrc_t rd = make_rsrc(a.delta + (int64_t)bh * T, (uint32_t)T * 4u);
#pragma unroll
    for (int db = 0; db < 4; ++db) A.dv[db] = A.dk[db] = zero16();
    float4 kx[16], vx[16];
    K.half_row(kx, key, hh);
    V.half_row(vx, key, hh);
#pragma unroll 1
    for (int t = tile0; t < n_tiles; t += step) {
        const int q0 = q_begin + t * kTile;
        if (a.causal && q0 + kTile - 1 < kw) continue;
        floatx16 sc = Q.dot(q0 + ln, hh, kx), dp = G.dot(q0 + ln, hh, vx);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int qr = q0 + 8 * (i / 4) + 4 * hh + (i % 4);  // past T: lse2, delta and the rows read as zeros
            const bool masked = (a.causal && key > qr) || (emit && key >= T);
            const float p = masked ? 0.0f : __builtin_amdgcn_exp2f(sc[i] * c - load4(rl, 4u * qr));
            const float ds = p * (dp[i] - load4(rd, 4u * qr));
            dp[i] = ds;
#pragma unroll
            for (int db = 0; db < 4; ++db) {
                A.dv[db] = mfma_f32(G.at(qr, 32 * db + ln), p, A.dv[db]);
                A.dk[db] = mfma_f32(Q.at(qr, 32 * db + ln), ds, A.dk[db]);
            }
        }
        if (emit) {
            const BwdDsLayout lay(T, a.causal);
            const int kb = kw / 128;
            uint8_t* blk = static_cast<uint8_t*>(a.ds_ws) +
                           (uint64_t)(bh * lay.per_head() + lay.block_offset(kb) + (q0 / 64 - lay.first_tile(kb))) * kDsBlockBytes;
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *reinterpret_cast<float4*>(blk + (kw % 128 + ln) * kDsRowBytes + (q0 & 32) * 4 + 16 * (2 * g + hh)) =
                    make_float4(dp[4 * g], dp[4 * g + 1], dp[4 * g + 2], dp[4 * g + 3]);
        }
    }
}

// dK and dV of block kb_own (128/G keys) of (batch, head) bh; kEmitDs: also dS -> the dS workspace
template <int G, bool kEmitDs>
__device__ __forceinline__ void dkdv_block(const FlashBwdArgs& a, int kb_own, int bh, BwdLds<G>& lds) {
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = G == 1 ? 0 : wave >> 1;
    const int w = G == 1 ? wave : wave & 1;
    const int ln = lane & 31;
    const int hh = lane >> 5;
    const int T = a.T;
    const float c = a.scale * kLog2e;
    const int b = bh / a.H, h = bh % a.H;

    const int64_t qkv = (int64_t)b * T * a.ld_qkv + (int64_t)h * kD;
    const float* Kg = static_cast<const float*>(a.k) + qkv;
    const float* Vg = static_cast<const float*>(a.v) + qkv;
    float* dKg = static_cast<float*>(a.d_k) + (int64_t)b * T * a.ld_grad + (int64_t)h * kD;
    float* dVg = static_cast<float*>(a.d_v) + (int64_t)b * T * a.ld_grad + (int64_t)h * kD;
    const Stream<G> sq(static_cast<const float*>(a.q) + qkv, T, a.ld_qkv, lane, w);
    const Stream<G> sg(static_cast<const float*>(a.d_o) + (int64_t)b * T * a.ld_o + (int64_t)h * kD, T, a.ld_o, lane, w);
    // waves 0 and 1 of a group also bring the rows' lse2 and delta
    const __amdgpu_buffer_rsrc_t rst = make_rsrc((w ? a.delta : a.lse2) + (int64_t)bh * T, (uint32_t)T * 4u);
    const LaneAddr LA = lane_addr(lane);
    GroupLds& my = lds.g[grp];

    const int kw = kb_own * (kBlk / G) + 32 * w;  // the wave's first key
    const int key = kw + ln;                      // this lane's key (the products' N index)
    const int q_begin = a.causal ? kb_own * (kBlk / G) : 0;
    const int n_tiles = (T - q_begin + kTile - 1) / kTile;
    const int n_steps = (n_tiles + G - 1) / G;
    auto tile_stat = [&](int t) { return load4(rst, (uint32_t)(q_begin + t * kTile + ln) * 4u); };

    float4 x[Stream<G>::kUnits];  // units between memory and the planes: Q's and dO's in turn
    float xs = tile_stat(grp);
#pragma unroll
    for (int n = 0; n < Stream<G>::kUnits; ++n) x[n] = sq.load(sq.at(grp, q_begin, n_tiles), n);
    float4 y[Stream<G>::kUnits];
#pragma unroll
    for (int n = 0; n < Stream<G>::kUnits; ++n) y[n] = sg.load(sg.at(grp, q_begin, n_tiles), n);
    Frag3 kf[8], vf[8];
    load_frags(kf, Kg, key, T, a.ld_qkv, hh);
    load_frags(vf, Vg, key, T, a.ld_qkv, hh);
    uint32_t s_low = 0;  // the lowest score, as the largest bit pattern (-inf: 0xff800000; without a sign: any)
    KvAcc A;
#pragma unroll
    for (int db = 0; db < 4; ++db) A.dv[db] = A.dk[db] = zero16();

    auto put_q = [&](int t, int n) {  // unit n of Q's tile t -> its planes, then dO's unit of that tile is requested
        sq.put(my.a[t & 1], n, x[n]);
    };
    auto put_g = [&](int n) { sg.put(my.b, n, x[n]); };
    auto put_stat = [&](int buf) {
        if (w < 2 && lane < 32) my.stats[buf][w][lane] = xs;
    };
#pragma unroll
    for (int n = 0; n < Stream<G>::kUnits; ++n) put_q(0, n);
    put_stat(0);
#pragma unroll
    for (int n = 0; n < Stream<G>::kUnits; ++n) {
        x[n] = y[n];
        put_g(n);
        x[n] = sq.load(sq.at(G + grp, q_begin, n_tiles), n);
    }
    xs = tile_stat(G + grp);
    lds_barrier();

    for (int it = 0; it < n_steps; ++it) {
        const int t = it * G + grp;
        const int q0 = q_begin + t * kTile;
        const int cur = it & 1, nxt = cur ^ 1;
        const uint8_t* qt = my.a[cur];
        const int lane = lane_here(), ln = lane & 31, hh = lane >> 5, key = kw + ln;
        // some query of the tile is at or after some key of the wave
        const bool visible = t < n_tiles && !(a.causal && q0 + kTile - 1 < kw) && kw < T;
        const uint32_t g_at = sg.at(t + G, q_begin, n_tiles), q_at = sq.at(t + 2 * G, q_begin, n_tiles);
        auto move_q = [&](int n) {  // the next tile's Q -> planes; its dO is requested
            put_q(nxt, n);
            x[n] = sg.load(g_at, n);
        };
        auto move_g = [&](int n) {  // the next tile's dO -> planes; the Q after it is requested
            put_g(n);
            x[n] = sq.load(q_at, n);
        };
        floatx16 sc, dp;
        Words3 pw, dw;
        if (visible) {
            sc = dot_rows(qt, LA, kf, [&](auto I) {
                constexpr int i = decltype(I)::value;
                if constexpr (G == 2 && i < 8) move_q(i);
                if constexpr (G == 1 && i < 8 && (i & 1)) move_q(i / 2);
            });
            put_stat(nxt);
            xs = tile_stat(t + 2 * G);
            float L[16], D[16];  // the rows' lse2 and delta: element i is query q0 + 8*(i/4) + 4*hh + i%4
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float4 l4 = *reinterpret_cast<const float4*>(&my.stats[cur][0][8 * g + 4 * hh]);
                const float4 d4 = *reinterpret_cast<const float4*>(&my.stats[cur][1][8 * g + 4 * hh]);
                L[4 * g] = l4.x, L[4 * g + 1] = l4.y, L[4 * g + 2] = l4.z, L[4 * g + 3] = l4.w;
                D[4 * g] = d4.x, D[4 * g + 1] = d4.y, D[4 * g + 2] = d4.z, D[4 * g + 3] = d4.w;
            }
            // element i is masked when dmask > 8*(i/4) + i%4, i.e. when key > query (causal); with dS stored, keys past
            // T are masked too (their dS would otherwise be exp2(-lse2) (-delta))
            const int dmask = (kEmitDs && key >= T) ? INT_MAX : a.causal ? key - (q0 + 4 * hh) : INT_MIN;
            const __amdgpu_buffer_rsrc_t ds_block = [&] {
                if constexpr (kEmitDs) {
                    const BwdDsLayout lay(T, a.causal);
                    const int kb = kw / 128;
                    return make_rsrc(static_cast<const uint8_t*>(a.ds_ws) +
                                         (uint64_t)(bh * lay.per_head() + lay.block_offset(kb) + (q0 / 64 - lay.first_tile(kb))) * kDsBlockBytes,
                                     (uint32_t)kDsBlockBytes);
                } else {
                    return make_rsrc(a.ds_ws, 0u);
                }
            }();
            const uint32_t ds_row = (uint32_t)((kw % 128 + ln) * kDsRowBytes + (q0 & 32) * 4 + 16 * hh);
            dp = dot_rows(my.b, LA, vf, [&](auto I) {  // P = exp2(S c - lse2), in place of S, and its split
                constexpr int i = decltype(I)::value;
                if constexpr (i < 4) {
#pragma unroll
                    for (int e = 4 * i; e < 4 * i + 4; ++e) {
                        s_low = max(s_low, __float_as_uint(sc[e]));
                        const float p = __builtin_amdgcn_exp2f(fmaf(sc[e], c * kDown2, -L[e]));
                        sc[e] = dmask > 8 * (e / 4) + (e % 4) ? 0.0f : p;
                    }
                } else {
                    pw.put(i - 4, sc[2 * (i - 4)], sc[2 * (i - 4) + 1]);
                }
            });
            acc_cols(A.dv, my.b, LA, pw, [&](auto I) {  // dV^T += dO^T P; dS = P (dP - delta), in place of dP, and its split
                constexpr int i = decltype(I)::value;
                if constexpr (i < 4) {
#pragma unroll
                    for (int e = 4 * i; e < 4 * i + 4; ++e) dp[e] = sc[e] * fmaf(dp[e], kDown2, -D[e]);
                } else {
                    constexpr int g = i - 4;
                    dw.put(2 * g, dp[4 * g], dp[4 * g + 1]);
                    dw.put(2 * g + 1, dp[4 * g + 2], dp[4 * g + 3]);
                    if constexpr (kEmitDs)  // chunk 2*g + hh of this query block's half of the lane's key row
                        __builtin_amdgcn_raw_buffer_store_b128(
                            __builtin_bit_cast(u32x4, make_float4(dp[4 * g], dp[4 * g + 1], dp[4 * g + 2], dp[4 * g + 3])), ds_block,
                            ds_row + 32 * g, 0, 0);
                }
            });
        } else {
#pragma unroll
            for (int n = 0; n < Stream<G>::kUnits; ++n) move_q(n);
            put_stat(nxt);
            xs = tile_stat(t + 2 * G);
        }
        lds_barrier();  // dO's planes are free
        if (visible) {
            acc_cols(A.dk, qt, LA, dw, [&](auto I) {  // dK^T += Q^T dS
                constexpr int i = decltype(I)::value;
                if constexpr (G == 2) move_g(i);
                else if constexpr (i & 1) move_g(i / 2);
            });
        } else {
#pragma unroll
            for (int n = 0; n < Stream<G>::kUnits; ++n) move_g(n);
        }
        lds_barrier();  // the next tile's planes are written
    }

    {
        const int lane = lane_here(), hh = lane >> 5, key = kw + (lane & 31);
        const float z = finite_probe(A.dv) + finite_probe(A.dk);
        const bool bad = key < T && (!(z == 0.0f) || s_low >= 0xff800000u || !scale_fits(a.scale));
        float f = kDown2;  // takes the operands' factors out
        if (__builtin_amdgcn_ballot_w64(bad) != 0) {
            KvAcc S;
            slow_dkdv(S, a, bh, kw, grp, G, n_tiles, q_begin, kEmitDs);
            settle(S.dv);
            settle(S.dk);
            A = S;
            f = 1.0f;
        }
        if constexpr (G == 2) {
            if (grp == 0) {
                add_groups(A.dv, A.dk, f, lds.x, 0, wave, lane);
                if (key < T) store_rows(dVg, key, a.ld_grad, hh, A.dv, 1.0f);
            } else {
                add_groups(A.dk, A.dv, f, lds.x, 1, wave, lane);
                if (key < T) store_rows(dKg, key, a.ld_grad, hh, A.dk, a.scale);  // dS carries the reference's scale (:293)
            }
        } else if (key < T) {
            store_rows(dKg, key, a.ld_grad, hh, A.dk, a.scale * f);
            store_rows(dVg, key, a.ld_grad, hh, A.dv, f);
        }
    }
}

// ------------------------------------------------------------------------------------------------ dQ
struct QAcc {
    floatx16 dq[4];
};
__device__ __forceinline__ void slow_dq(QAcc& A, const FlashBwdArgs& a, int bh, int qw, int tile0, int step, int n_tiles) {
    const int lane = lane_here(), ln = lane & 31, hh = lane >> 5;
    const int T = a.T, q = qw + ln, b = bh / a.H, h = bh % a.H;
    const float c = scale_here(a.scale) * kLog2e;
    const Rows Q(a.q, b, h, T, a.ld_qkv), K(a.k, b, h, T, a.ld_qkv), V(a.v, b, h, T, a.ld_qkv), G(a.d_o, b, h, T, a.ld_o);
    const float lse2 = q < T ? a.lse2[(int64_t)bh * T + q] : 0.0f, delta = q < T ? a.delta[(int64_t)bh * T + q] : 0.0f;
    const int lim = a.causal ? min(q, T - 1) : T - 1;
#pragma unroll
    for (int db = 0; db < 4; ++db) A.dq[db] = zero16();
    float4 qx[16], gx[16];
    Q.half_row(qx, q, hh);
    G.half_row(gx, q, hh);
#pragma unroll 1
    for (int t = tile0; t < n_tiles; t += step) {
        const int k0 = t * kTile;
        if (a.causal && k0 > qw + 31) break;
        const floatx16 sc = K.dot(k0 + ln, hh, qx), dp = V.dot(k0 + ln, hh, gx);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int key = k0 + 8 * (i / 4) + 4 * hh + (i % 4);
            const float p = key > lim ? 0.0f : __builtin_amdgcn_exp2f(sc[i] * c - lse2);
            const float ds = p * (dp[i] - delta);
#pragma unroll
            for (int db = 0; db < 4; ++db) A.dq[db] = mfma_f32(K.at(key, 32 * db + ln), ds, A.dq[db]);
        }
    }
}

// dQ of block qb_own (128/G queries) of (batch, head) bh
template <int G>
__device__ __forceinline__ void dq_block(const FlashBwdArgs& a, int qb_own, int bh, BwdLds<G>& lds) {
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = G == 1 ? 0 : wave >> 1;
    const int w = G == 1 ? wave : wave & 1;
    const int ln = lane & 31;
    const int hh = lane >> 5;
    const int T = a.T;
    const float c = a.scale * kLog2e;
    const int b = bh / a.H, h = bh % a.H;

    const int64_t qkv = (int64_t)b * T * a.ld_qkv + (int64_t)h * kD;
    const float* Gg = static_cast<const float*>(a.d_o) + (int64_t)b * T * a.ld_o + (int64_t)h * kD;
    float* dQg = static_cast<float*>(a.d_q) + (int64_t)b * T * a.ld_grad + (int64_t)h * kD;
    const Stream<G> sk(static_cast<const float*>(a.k) + qkv, T, a.ld_qkv, lane, w);
    const Stream<G> sv(static_cast<const float*>(a.v) + qkv, T, a.ld_qkv, lane, w);
    const LaneAddr LA = lane_addr(lane);
    GroupLds& my = lds.g[grp];

    const int qw = qb_own * (kBlk / G) + 32 * w;  // the wave's first query
    const int q = qw + ln;
    const int k_end = a.causal ? min((qb_own + 1) * (kBlk / G), T) : T;
    const int n_tiles = (k_end + kTile - 1) / kTile;
    const int n_steps = (n_tiles + G - 1) / G;

    float4 x[Stream<G>::kUnits], y[Stream<G>::kUnits];
#pragma unroll
    for (int n = 0; n < Stream<G>::kUnits; ++n) x[n] = sk.load(sk.at(grp, 0, n_tiles), n);
#pragma unroll
    for (int n = 0; n < Stream<G>::kUnits; ++n) y[n] = sv.load(sv.at(grp, 0, n_tiles), n);
    Frag3 qf[8], gf[8];
    load_frags(qf, static_cast<const float*>(a.q) + qkv, q, T, a.ld_qkv, hh);
    load_frags(gf, Gg, q, T, a.ld_o, hh);
    uint32_t s_low = 0;  // the lowest score, as the largest bit pattern (-inf: 0xff800000; without a sign: any)
    const float lse2 = q < T ? a.lse2[(int64_t)bh * T + q] : 0.0f;
    const float delta = q < T ? a.delta[(int64_t)bh * T + q] : 0.0f;
    const int lim = a.causal ? min(q, T - 1) : T - 1;  // keys > lim are masked
    QAcc A;
#pragma unroll
    for (int db = 0; db < 4; ++db) A.dq[db] = zero16();
    auto put_k = [&](int buf, int n) { sk.put(my.a[buf], n, x[n]); };
    auto put_v = [&](int n) { sv.put(my.b, n, x[n]); };
#pragma unroll
    for (int n = 0; n < Stream<G>::kUnits; ++n) put_k(0, n);
#pragma unroll
    for (int n = 0; n < Stream<G>::kUnits; ++n) {
        x[n] = y[n];
        put_v(n);
        x[n] = sk.load(sk.at(G + grp, 0, n_tiles), n);
    }
    lds_barrier();

    for (int it = 0; it < n_steps; ++it) {
        const int t = it * G + grp;
        const int k0 = t * kTile;
        const int cur = it & 1, nxt = cur ^ 1;
        const uint8_t* kt = my.a[cur];
        const bool visible = t < n_tiles && !(a.causal && k0 > qw + 31) && qw < T;
        const uint32_t v_at = sv.at(t + G, 0, n_tiles), k_at = sk.at(t + 2 * G, 0, n_tiles);
        auto move_k = [&](int n) {  // the next tile's K -> planes; its V is requested
            put_k(nxt, n);
            x[n] = sv.load(v_at, n);
        };
        auto move_v = [&](int n) {  // the next tile's V -> planes; the K after it is requested
            put_v(n);
            x[n] = sk.load(k_at, n);
        };
        floatx16 sc, dp;
        Words3 dw;
        if (visible) {
            sc = dot_rows<true>(kt, LA, qf, [&](auto I) {  // S^T = K Q^T
                constexpr int i = decltype(I)::value;
                if constexpr (G == 2 && i < 8) move_k(i);
                if constexpr (G == 1 && i < 8 && (i & 1)) move_k(i / 2);
            });
            const int emask = lim - (k0 + 4 * hh);  // element i (key k0 + 8*(i/4) + 4*hh + i%4) is masked past it
            dp = dot_rows<true>(my.b, LA, gf, [&](auto I) {  // dP^T = V dO^T; P^T in place of S^T
                constexpr int i = decltype(I)::value;
                if constexpr (i < 8) {
#pragma unroll
                    for (int e = 2 * i; e < 2 * i + 2; ++e) {
                        s_low = max(s_low, __float_as_uint(sc[e]));
                        const float p = __builtin_amdgcn_exp2f(fmaf(sc[e], c * kDown2, -lse2));
                        sc[e] = 8 * (e / 4) + (e % 4) > emask ? 0.0f : p;
                    }
                }
            });
#pragma unroll
            for (int e = 0; e < 16; ++e) dp[e] = sc[e] * fmaf(dp[e], kDown2, -delta);
#pragma unroll
            for (int e = 0; e < 4; ++e) dw.put(e, dp[2 * e], dp[2 * e + 1]);
        } else {
#pragma unroll
            for (int n = 0; n < Stream<G>::kUnits; ++n) move_k(n);
        }
        lds_barrier();  // V's planes are free
        if (visible) {
            acc_cols(A.dq, kt, LA, dw, [&](auto I) {  // dQ^T += K^T dS^T
                constexpr int i = decltype(I)::value;
                if constexpr (i < 2) {  // the second 16 keys' dS
                    dw.put(4 + 2 * i, dp[8 + 4 * i], dp[9 + 4 * i]);
                    dw.put(5 + 2 * i, dp[10 + 4 * i], dp[11 + 4 * i]);
                }
                if constexpr (G == 2) move_v(i);
                else if constexpr (i & 1) move_v(i / 2);
            });
        } else {
#pragma unroll
            for (int n = 0; n < Stream<G>::kUnits; ++n) move_v(n);
        }
        lds_barrier();  // the next tile's planes are written
    }

    const bool bad = q < T && (!(finite_probe(A.dq) == 0.0f) || s_low >= 0xff800000u || !scale_fits(a.scale));
    float f = kDown2;  // takes the operands' factors out
    if (__builtin_amdgcn_ballot_w64(bad) != 0) {
        QAcc S;
        slow_dq(S, a, bh, qw, grp, G, n_tiles);
        settle(S.dq);
        A = S;
        f = 1.0f;
    }
    if constexpr (G == 2) {  // group g stores dims 64g .. 64g+63
        float4(&ex)[4][16][64] = lds.x;
        auto at = [&](int db, int g) -> float4& { return ex[wave][4 * (db & 1) + g][lane]; };
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const floatx16 v = grp ? A.dq[d] : A.dq[2 + d];
                at(d, g) = make_float4(v[4 * g] * f, v[4 * g + 1] * f, v[4 * g + 2] * f, v[4 * g + 3] * f);
            }
        lds_barrier();
        if (q < T) {
            float* p = dQg + (int64_t)q * a.ld_grad + 64 * grp + 4 * hh;
#pragma unroll
            for (int d = 0; d < 2; ++d)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const floatx16 v = grp ? A.dq[2 + d] : A.dq[d];
                    const float4 o = ex[wave ^ 2][4 * d + g][lane];
                    *reinterpret_cast<float4*>(p + 32 * d + 8 * g) =
                        make_float4((v[4 * g] * f + o.x) * a.scale, (v[4 * g + 1] * f + o.y) * a.scale, (v[4 * g + 2] * f + o.z) * a.scale,
                                    (v[4 * g + 3] * f + o.w) * a.scale);
                }
        }
    } else if (q < T) {
        store_rows(dQg, q, a.ld_grad, hh, A.dq, a.scale * f);
    }
}

// ------------------------------------------------------------------------------------------------ dQ from dS
struct DsLds {
    uint8_t k[2][kPlanes];
};

__device__ __forceinline__ void slow_dq_ds(QAcc& A, const FlashBwdArgs& a, int bh, int qw, int n_use) {
    const int lane = lane_here(), ln = lane & 31, hh = lane >> 5;
    const int T = a.T, b = bh / a.H, h = bh % a.H;
    const Rows K(a.k, b, h, T, a.ld_qkv);
    const BwdDsLayout lay(T, a.causal);
    const uint8_t* head = static_cast<const uint8_t*>(a.ds_ws) + (uint64_t)(bh * lay.per_head()) * kDsBlockBytes;
#pragma unroll
    for (int db = 0; db < 4; ++db) A.dq[db] = zero16();
#pragma unroll 1
    for (int t = 0; t < n_use; ++t) {
        const int k0 = t * kTile, kb = k0 / 128;
        const uint8_t* col = head + (uint64_t)(lay.block_offset(kb) + (qw / 64 - lay.first_tile(kb))) * kDsBlockBytes + 4 * (qw % 64 + ln);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int r = 8 * (i / 4) + 4 * hh + (i % 4);
            const float ds = *reinterpret_cast<const float*>(col + (k0 % 128 + r) * kDsRowBytes);
#pragma unroll
            for (int db = 0; db < 4; ++db) A.dq[db] = mfma_f32(K.at(k0 + r, 32 * db + ln), ds, A.dq[db]);
        }
    }
}

// dQ of query block qb_own (128 queries) of (batch, head) bh from the dS the dK/dV pass stored: per 32-key tile
// dQ^T += K^T dS^T, K's planes from LDS (two stages, one barrier per tile) and dS straight from memory, one tile ahead:
// a lane's element is one key row at its own query, so a load instruction reads two rows of 128 bytes.
__device__ __forceinline__ void dq_ds_block(const FlashBwdArgs& a, int qb_own, int bh, DsLds& lds) {
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 31;
    const int hh = lane >> 5;
    const int T = a.T;
    const int b = bh / a.H, h = bh % a.H;
    float* dQg = static_cast<float*>(a.d_q) + (int64_t)b * T * a.ld_grad + (int64_t)h * kD;
    const Stream<1> sk(static_cast<const float*>(a.k) + (int64_t)b * T * a.ld_qkv + (int64_t)h * kD, T, a.ld_qkv, lane, wave);
    const BwdDsLayout lay(T, a.causal);
    const uint8_t* ds_head = static_cast<const uint8_t*>(a.ds_ws) + (uint64_t)(bh * lay.per_head()) * kDsBlockBytes;
    const LaneAddr LA = lane_addr(lane);

    const int qw = qb_own * kBlk + 32 * wave;  // the wave's first query
    const int q = qw + ln;
    const int k_end = a.causal ? min(qb_own * kBlk + kBlk, T) : T;
    const int n_tiles = (k_end + kTile - 1) / kTile;
    // the tiles whose dS this wave's queries have (under causality the later ones were not stored)
    const int n_use = qw >= T ? 0 : (a.causal ? min(n_tiles, qw / kTile + 1) : n_tiles);

    floatx16 ds;  // element i: dS of key k0 + 8*(i/4) + 4*hh + i%4 and this lane's query
    const uint32_t lane_off = (uint32_t)(4 * hh * kDsRowBytes + 4 * (qw % 64 + ln));
    auto load_ds = [&](int t) {
        const int k0 = t * kTile, kb = k0 / 128;
        const uint8_t* blk = ds_head + (uint64_t)(lay.block_offset(kb) + (qw / 64 - lay.first_tile(kb))) * kDsBlockBytes;
        const __amdgpu_buffer_rsrc_t r = make_rsrc(t < n_use ? blk : ds_head, t < n_use ? (uint32_t)kDsBlockBytes : 0u);
#pragma unroll
        for (int i = 0; i < 16; ++i)
            ds[i] = load4(r, lane_off + (uint32_t)((k0 % 128 + 8 * (i / 4) + (i % 4)) * kDsRowBytes));
    };
    QAcc A;
#pragma unroll
    for (int db = 0; db < 4; ++db) A.dq[db] = zero16();
    float4 x[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) x[n] = sk.load(sk.at(0, 0, n_tiles), n);
    load_ds(0);
    auto move_k = [&](int t, uint32_t next_at, int n) {
        sk.put(lds.k[t & 1], n, x[n]);
        x[n] = sk.load(next_at, n);
    };
#pragma unroll
    for (int n = 0; n < 4; ++n) move_k(0, sk.at(1, 0, n_tiles), n);
    lds_barrier();
    for (int t = 0; t < n_tiles; ++t) {
        const uint32_t k_at = sk.at(t + 2, 0, n_tiles);
        if (t < n_use) {
            Words3 dw;
#pragma unroll
            for (int e = 0; e < 8; ++e) dw.put(e, ds[2 * e], ds[2 * e + 1]);
            load_ds(t + 1);
            acc_cols(A.dq, lds.k[t & 1], LA, dw, [&](auto I) {
                constexpr int i = decltype(I)::value;
                if constexpr (i & 1) move_k(t + 1, k_at, i / 2);
            });
        } else {
#pragma unroll
            for (int n = 0; n < 4; ++n) move_k(t + 1, k_at, n);
        }
        lds_barrier();
    }
    const bool bad = q < T && !(finite_probe(A.dq) == 0.0f);
    float f = a.scale * kDown2;
    if (__builtin_amdgcn_ballot_w64(bad) != 0) {
        slow_dq_ds(A, a, bh, qw, n_use);
        f = a.scale;
    }
    if (q < T) store_rows(dQg, q, a.ld_grad, hh, A.dq, f);
}

// One block per workgroup, listed in decreasing causal cost, so that the hardware, which hands the next workgroup to
// the first CU that frees up, runs a longest-first schedule.
// pass = 0 (dK/dV) or 1 (dQ): one pass per launch; workgroup BH*j + bh takes, for (batch, head) bh,
//   key block j (dK/dV; key block 0 sees every query tile) or query block n-1-j (dQ).
// pass = 2: both passes in one launch; workgroup 2*BH*j + BH*kind + bh takes the dK/dV of key block j
//   (kind 0) or the dQ of query block n-1-j (kind 1), which see the same number of tiles under
//   causality, so the list stays in decreasing cost and the two passes share the CUs.
template <int G>
__global__ __launch_bounds__(kThreads, 1) void flash_bwd_f32_kernel(FlashBwdArgs a, int pass) {
    __shared__ __attribute__((aligned(1024))) BwdLds<G> lds;
    const int BH = a.B * a.H;
    const int n = (a.T + kBlk / G - 1) / (kBlk / G);
    const int j = (int)blockIdx.x / (pass == 2 ? 2 * BH : BH);
    const int kind = pass == 2 ? ((int)blockIdx.x / BH) & 1 : pass;
    const int bh = (int)blockIdx.x % BH;
    if (kind == 0) dkdv_block<G, false>(a, j, bh, lds);
    else dq_block<G>(a, n - 1 - j, bh, lds);
}

// The dS path: the dK/dV pass (workgroup BH*j + bh: key block j) storing dS, then dQ = dS K (workgroup
// BH*j + bh: query block n-1-j), both in decreasing causal cost.
template <int G>
__global__ __launch_bounds__(kThreads, 1) void flash_bwd_dkdv_ds_f32_kernel(FlashBwdArgs a) {
    __shared__ __attribute__((aligned(1024))) BwdLds<G> lds;
    const int BH = a.B * a.H;
    dkdv_block<G, true>(a, (int)blockIdx.x / BH, (int)blockIdx.x % BH, lds);
}
__global__ __launch_bounds__(kThreads, 2) void flash_bwd_dq_ds_f32_kernel(FlashBwdArgs a) {
    __shared__ __attribute__((aligned(1024))) DsLds lds;
    const int BH = a.B * a.H;
    const int n = (a.T + kBlk - 1) / kBlk;
    dq_ds_block(a, n - 1 - (int)blockIdx.x / BH, (int)blockIdx.x % BH, lds);
}

template <int G>
int launch(const FlashBwdArgs& a, int64_t blocks128, int cus, hipStream_t stream) {
    const int64_t blocks = G == 1 ? blocks128 : (int64_t)((a.T + kBlk / G - 1) / (kBlk / G)) * a.B * a.H;
    if (a.ds_ws) {  // dS stored by the dK/dV pass, dQ = dS K
        hipLaunchKernelGGL(flash_bwd_dkdv_ds_f32_kernel<G>, dim3((unsigned)blocks), dim3(kThreads), 0, stream, a);
        DT_HIP_TRY(hipGetLastError());
        hipLaunchKernelGGL(flash_bwd_dq_ds_f32_kernel, dim3((unsigned)blocks128), dim3(kThreads), 0, stream, a);
        DT_HIP_TRY(hipGetLastError());
        return DT_OK;
    }
    if (blocks128 <= cus) {  // the passes share one launch (at most one 128-row block per CU and pass)
        hipLaunchKernelGGL(flash_bwd_f32_kernel<G>, dim3((unsigned)(2 * blocks)), dim3(kThreads), 0, stream, a, 2);
        DT_HIP_TRY(hipGetLastError());
    } else {
        for (int pass = 0; pass < 2; ++pass) {
            hipLaunchKernelGGL(flash_bwd_f32_kernel<G>, dim3((unsigned)blocks), dim3(kThreads), 0, stream, a, pass);
            DT_HIP_TRY(hipGetLastError());
        }
    }
    return DT_OK;
}

}  // namespace

int launch_flash_bwd_f32(const FlashBwdArgs& a, hipStream_t stream) {
    const int64_t ld = a.ld_qkv > a.ld_o ? a.ld_qkv : a.ld_o;
    if ((int64_t)a.T * ld * 4 >= ((int64_t)1 << 31))
        return set_error(DT_ERR_UNSUPPORTED, "Q/K/V/dO extent of one sequence exceeds 2 GiB");
    DT_TRY(launch_flash_bwd_prep(a, 0, stream));
    const int64_t blocks = (int64_t)((a.T + kBlk - 1) / kBlk) * a.B * a.H;  // per pass, one per workgroup
    if (2 * blocks > 0x7fffffff) return set_error(DT_ERR_UNSUPPORTED, "too many workgroups");
    int cus = 0;
    DT_TRY(persistent_grid(0x7fffffff, &cus));
    return flash_bwd_two_groups((int64_t)a.B * a.H, a.T, a.causal, cus, kBwdGroupRowsF32) ? launch<2>(a, blocks, cus, stream)
                                                                                   : launch<1>(a, blocks, cus, stream);
}

}  // namespace dt
