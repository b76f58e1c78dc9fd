// Causal flash attention forward, bf16 MFMA mode, for launches with few queries (gfx950, CDNA4).
//
// The persistent kernel of flash_fwd_bf16.hip works on items of 128 queries whose keys two groups of waves share. Where
// a launch has fewer 64-query tiles than the device has CUs, those items leave half of the CUs without one and the
// longest item's chain of key steps sets the time. Here a workgroup owns 64 queries of one (batch, head), and four
// groups of two waves (32 queries each) share its keys in tiles of 32: group g takes tiles g, g+4, g+8, ... So a
// workgroup's chain has as many steps as there, of half the keys each, on twice as many CUs. What it costs is traffic,
// twice the K and V bytes per query through LDS, which is why launches that fill the chip keep the other kernel.
// What bounds it: the latency of a chain (launch, first tile, steps of ~2 k cycles, merge). B = 1, H = 16, us per call,
// before and now: T = 511 12.7 and 11.4, T = 1000 18.2 and 15.8; H = 8, T = 1500 22.8 and 19.6. With the next tile
// requested in mid-step, as there, T = 1000 took 17.5.
//
// Everything else is as there: S^T = K Q^T on v_mfma_f32_32x32x16_bf16 with one lane per query, the lazily rescaled
// softmax in the log2 domain seeded through the accumulator, P in registers as the B operand of O^T += V^T P^T, K and V by
// LDS DMA into swizzled 256-byte rows, double-buffered. At the end the groups' partial results meet in LDS and group g
// finalises dims 32g .. 32g+31, with the reference's rescale (FlashAttention.cpp:134-156), group 0's term first.
#include "dt_internal.h"

#include <type_traits>
#include <utility>

namespace dt {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef short shortx8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) shortx4 lds_shortx4;
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kD = 128;
constexpr int kRows = 64;      // queries per workgroup
constexpr int kBN = 32;        // keys per tile
constexpr int kGroups = 4;
constexpr int kThreads = 512;  // 8 waves: group wave / 2, query block wave % 2
constexpr int kRowBytes = 256;
constexpr int kTileBytes = kBN * kRowBytes;  // 8 KB per tensor
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegInf = -__builtin_huge_valf();
constexpr float kRescaleLog2 = 8.0f;
constexpr int kBufferDword3 = 0x00020000;  // raw buffer, 32-bit data format (gfx9 family)

union Lds {
    uint8_t kv[2][kGroups][2][kTileBytes];  // [stage][group][K, V]: 128 KB
    struct {
        float4 o[8][4][4][64];  // [wave][dim block][I][lane]
        float s[8][3][64];      // [wave][m_s, m_t, l][lane]
    } end;
};

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
    bf16x2 r = __builtin_convertvector((floatx2){lo, hi}, bf16x2);
    return __builtin_bit_cast(uint32_t, r);
}
// over the two lane halves (lane l and lane l ^ 32 hold the same query): both results, the lower half's first
__device__ __forceinline__ float max_halves(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_halves(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, kBufferDword3);
}
__device__ __forceinline__ float bf16_lo(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }
// chunk c of row r lives at position c ^ swz(r)
__device__ __forceinline__ int swz(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

template <typename F, int... Is>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}
#define DT_BUNDLE_END __builtin_amdgcn_sched_barrier(0)

// LDS DMA through inline assembly, which the compiler does not wait for before it reads the other stage (stage_barrier
// does); s_nop 4 covers the wait states the compiler cannot insert around it.
__device__ __forceinline__ uint32_t lds_addr(const void* p) { return (uint32_t)(uintptr_t)(const lds_void*)p; }
__device__ __forceinline__ void dma16(uint32_t lds, uint32_t voff, __amdgpu_buffer_rsrc_t r) {
    asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(voff), "s"(r), "{m0}"(lds) : "memory");
}
__device__ __forceinline__ void stage_barrier() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// workgroup BH*j + bh: query tile n-1-j of (batch, head) bh (decreasing causal cost)
template <bool kRagged>
__global__ __launch_bounds__(kThreads, 1) void flash_fwd_bf16_few_kernel(FlashArgs a, std::conditional_t<kRagged, SeqLens, int> lens) {
    __shared__ __attribute__((aligned(1024))) Lds lds;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 1, qb = wave & 1;
    const int ln = lane & 31, hh = lane >> 5;
    const int T = a.T, BH = a.B * a.H;
    const int bh = (int)blockIdx.x % BH;
    const int b = bh / a.H, h = bh - b * a.H;
    const int q0 = ((T + kRows - 1) / kRows - 1 - (int)blockIdx.x / BH) * kRows;
    int L = T;
    if constexpr (kRagged) L = lens.len[b];
    const int qw0 = q0 + 32 * qb;  // this wave's first query
    const int qrow = qw0 + ln;
    const float c = a.scale * kLog2e;

    const uint16_t* Qg = static_cast<const uint16_t*>(a.q) + (int64_t)b * T * a.ldq + (int64_t)h * kD;
    const uint16_t* Kg = static_cast<const uint16_t*>(a.k) + (int64_t)b * T * a.ldk + (int64_t)h * kD;
    const uint16_t* Vg = static_cast<const uint16_t*>(a.v) + (int64_t)b * T * a.ldv + (int64_t)h * kD;
    const int k_end = a.causal ? min(q0 + kRows, L) : L;
    const int n_tiles = q0 < L ? (k_end + kBN - 1) / kBN : 0;  // (a tile of padding rows only: none)
    const int n_steps = (n_tiles + kGroups - 1) / kGroups;
    const int lim = a.causal ? min(qrow, L - 1) : L - 1;  // keys > lim are masked

    // DMA: instruction n of wave qb of a group fills rows 8*n + 4*qb + lane/16 of a tile; the lane fetches the chunk the
    // swizzle puts at position lane%16 (swz's upper bits alternate with n)
    uint32_t off[2];
    {
        const int rlo = lane >> 4;
#pragma unroll
        for (int o = 0; o < 2; ++o) off[o] = (uint32_t)(((4 * qb + rlo) * a.ldk + 8 * ((lane & 15) ^ (4 * rlo + 2 * o + qb))) * 2);
    }
    auto dma = [&](int stage, int kv, int kt) {
        const int k0 = kt * kBN;
        const __amdgpu_buffer_rsrc_t r = make_rsrc((kv ? Vg : Kg) + (int64_t)k0 * a.ldk, (uint32_t)(L - k0) * (uint32_t)a.ldk * 2u);
        const uint32_t l0 = __builtin_amdgcn_readfirstlane(lds_addr(&lds.kv[stage][grp][kv][qb * 1024]));
#pragma unroll
        for (int n = 0; n < 4; ++n) dma16(l0 + 2048 * n, off[n & 1] + (uint32_t)(16 * n) * (uint32_t)a.ldk, r);
    };
    if (grp < n_tiles) {
        dma(0, 0, grp);
        dma(0, 1, grp);
    }
    // fragment addresses in a group's stage (stage 1 lies kStage bytes further)
    const uint8_t* const base = &lds.kv[0][grp][0][0];
    constexpr uint32_t kStage = kGroups * 2 * kTileBytes;
    uint32_t kaddr[8], vaddr[2][4];
    {
        const int g = hh ^ swz(ln);
#pragma unroll
        for (int cc = 0; cc < 8; ++cc) kaddr[cc] = (uint32_t)(ln * kRowBytes + (((2 * cc) ^ g) << 4));
        const int i16 = lane & 15, g2 = (lane >> 4) & 1;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int r = 4 * hh + (i16 >> 2) + 8 * s;
#pragma unroll
            for (int db = 0; db < 4; ++db) {
                const int chunk = 4 * db + 2 * g2 + ((i16 & 3) >> 1);
                vaddr[s][db] = (uint32_t)(kTileBytes + r * kRowBytes + ((chunk ^ swz(r)) << 4) + 8 * (i16 & 1));
            }
        }
    }
    // Q fragment, times scale * log2 e: qf[cc] = Q[qrow][16*cc + 8*hh .. +8] * c (rows past T: any values)
    bf16x8 qf[8];
    {
        const uint16_t* qp = Qg + (int64_t)min(qrow, T - 1) * a.ldq + 8 * hh;
        uint4 raw[8];
#pragma unroll
        for (int cc = 0; cc < 8; ++cc) raw[cc] = *reinterpret_cast<const uint4*>(qp + 16 * cc);
#pragma unroll
        for (int cc = 0; cc < 8; ++cc) {
            const uint32_t w[4] = {raw[cc].x, raw[cc].y, raw[cc].z, raw[cc].w};
            uint32_t sw[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) sw[e] = pack_bf16x2(bf16_lo(w[e]) * c, bf16_hi(w[e]) * c);
            qf[cc] = __builtin_bit_cast(bf16x8, make_uint4(sw[0], sw[1], sw[2], sw[3]));
        }
    }
    floatx16 o[4], neg_ms;
#pragma unroll
    for (int i = 0; i < 16; ++i) o[0][i] = o[1][i] = o[2][i] = o[3][i] = neg_ms[i] = 0.0f;
    float m_t = kNegInf, m_s = kNegInf, l = 0.0f;
    stage_barrier();

    for (int it = 0; it < n_steps; ++it) {
        const int kt = kGroups * it + grp;
        const int k0 = kt * kBN;
        const uint32_t so = (it & 1) ? kStage : 0u;
        const bool next = kt + kGroups < n_tiles;
        if (next) {  // the whole step hides the requests' latency (a step is shorter than it)
            dma((it & 1) ^ 1, 0, kt + kGroups);
            dma((it & 1) ^ 1, 1, kt + kGroups);
        }
        if (kt < n_tiles && qw0 < L && !(a.causal && k0 > qw0 + 31)) {
            const uint8_t* st_base = base + so;
            floatx16 st = neg_ms;
            {
                bf16x8 kr[4];
                auto rd = [&](int cc) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(st_base + kaddr[cc])); };
                kr[0] = rd(0);
                kr[1] = rd(1);
                kr[2] = rd(2);
                static_for<8>([&](auto R) {
                    constexpr int r = decltype(R)::value;
                    if constexpr (r + 3 < 8) kr[(r + 3) & 3] = rd(r + 3);
                    st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kr[r & 3], qf[r], st, 0, 0, 0);
                    DT_BUNDLE_END;
                });
            }
            // chunk ch = 4*u + db: keys 16*u .. +16, dims 32*db .. +32
            auto read_v = [&](int ch) {
                const uint8_t* p = st_base + (ch >> 2) * 16 * kRowBytes;
                const shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)(p + vaddr[0][ch & 3]));
                const shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)(p + vaddr[1][ch & 3]));
                return __builtin_bit_cast(bf16x8, (shortx8){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
            };
            bf16x8 vr[4];  // the first V chunks stream in while the softmax runs
            vr[0] = read_v(0);
            vr[1] = read_v(1);
            vr[2] = read_v(2);
            if ((a.causal && k0 + kBN - 1 > qw0) || k0 + kBN > L) {
                asm volatile("");  // keeps this rare block a branch
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
            const float ref = (m_s == kNegInf) ? 0.0f : m_s;  // what the S chain subtracted
            m_t = fmaxf(m_t, tmax + ref);
            const bool grow = (m_s == kNegInf) ? (tmax > kNegInf) : (tmax > kRescaleLog2);
            if (__builtin_amdgcn_ballot_w64(grow) != 0) {  // wave-uniform, rare after the first tile
                asm volatile("");
                const float m_new = max_halves(m_t);
                const float delta = (m_new == kNegInf) ? 0.0f : m_new - ref;
                const float alpha = (m_s == kNegInf) ? 0.0f : exp2f(m_s - m_new);
                m_s = m_new;
                l *= alpha;
#pragma unroll
                for (int db = 0; db < 4; ++db)
#pragma unroll
                    for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
                const float nm = (m_s == kNegInf) ? 0.0f : -m_s;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    st[i] -= delta;
                    neg_ms[i] = nm;
                }
            }
            // p = exp2(t) in bf16; the row sum is over the bf16 values the PV product uses
            const bf16x2 ones = {(__bf16)1.0f, (__bf16)1.0f};
            float psum[2] = {0.0f, 0.0f};
            bf16x8 pb[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                uint32_t w[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    w[e] = pack_bf16x2(__builtin_amdgcn_exp2f(st[8 * u + 2 * e]), __builtin_amdgcn_exp2f(st[8 * u + 2 * e + 1]));
                    psum[u] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w[e]), ones, psum[u], false);
                }
                pb[u] = __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
            }
            l += psum[0] + psum[1];
            static_for<8>([&](auto C) {
                constexpr int ch = decltype(C)::value;
                if constexpr (ch + 3 < 8) vr[(ch + 3) & 3] = read_v(ch + 3);
                o[ch & 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vr[ch & 3], pb[ch >> 2], o[ch & 3], 0, 0, 0);
                DT_BUNDLE_END;
            });
        }
        stage_barrier();
    }

    // merge through LDS: wave (grp, qb) finalises dims 32*grp .. +32 of its 32 queries
    m_t = max_halves(m_t);
    l = sum_halves(l);
    static_for<4>([&](auto DB) {
        constexpr int db = decltype(DB)::value;
#pragma unroll
        for (int I = 0; I < 4; ++I)
            lds.end.o[wave][db][I][lane] = make_float4(o[db][4 * I], o[db][4 * I + 1], o[db][4 * I + 2], o[db][4 * I + 3]);
    });
    lds.end.s[wave][0][lane] = m_s;
    lds.end.s[wave][1][lane] = m_t;
    lds.end.s[wave][2][lane] = l;
    lds_barrier();
    float ms = kNegInf, mt = kNegInf, lsum = 0.0f, f[kGroups];
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
        f[g] = lds.end.s[2 * g + qb][0][lane];
        ms = fmaxf(ms, f[g]);
        mt = fmaxf(mt, lds.end.s[2 * g + qb][1][lane]);
    }
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
        f[g] = (f[g] == kNegInf) ? 0.0f : exp2f(f[g] - ms);
        lsum += lds.end.s[2 * g + qb][2][lane] * f[g];
    }
    const bool valid = qrow < L && lsum > 0.0f;
    const float inv = valid ? 1.0f / lsum : 0.0f;
    if (qrow < T) {
        uint16_t* op = static_cast<uint16_t*>(a.o) + ((int64_t)b * T + qrow) * a.ldo + (int64_t)h * kD + 32 * grp + 4 * hh;
#pragma unroll
        for (int I = 0; I < 4; ++I) {
            float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            static_for<kGroups>([&](auto GG) {  // group 0's term first
                constexpr int g = decltype(GG)::value;
                const float4 x = lds.end.o[2 * g + qb][grp][I][lane];
                const float s = f[g] * inv;
                v[0] += x.x * s;
                v[1] += x.y * s;
                v[2] += x.z * s;
                v[3] += x.w * s;
            });
            uint2 w;
            w.x = valid ? pack_bf16x2(v[0], v[1]) : 0u;
            w.y = valid ? pack_bf16x2(v[2], v[3]) : 0u;
            *reinterpret_cast<uint2*>(op + 8 * I) = w;
        }
        if (grp == 0 && hh == 0) {
            const int64_t st = ((int64_t)b * T + qrow) * a.H + h;
            if (a.m) a.m[st] = valid ? mt * (1.0f / kLog2e) : kNegInf;
            if (a.l) a.l[st] = valid ? lsum * exp2f(ms - mt) : 0.0f;
        }
    }
}

}  // namespace

int launch_flash_fwd_bf16_few(const FlashArgs& a, const SeqLens* lens, hipStream_t stream) {
    const unsigned grid = (unsigned)((a.T + kRows - 1) / kRows) * (unsigned)a.B * (unsigned)a.H;
    if (a.ragged) hipLaunchKernelGGL(flash_fwd_bf16_few_kernel<true>, dim3(grid), dim3(kThreads), 0, stream, a, *lens);
    else hipLaunchKernelGGL(flash_fwd_bf16_few_kernel<false>, dim3(grid), dim3(kThreads), 0, stream, a, 0);
    DT_HIP_TRY(hipGetLastError());
    return DT_OK;
}

}  // namespace dt
