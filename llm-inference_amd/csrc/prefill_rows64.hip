// Causal prefill attention for gfx950 on fp16 MFMA, 64 query rows per wave:
// any grouping of query heads, head_dim 64 or 128, 16-byte aligned rows.
//
// Same semantics as prefill.hip (causal_attention.hip.cpp:271-374: query t of
// head h attends to keys 0..t of KV head h / (Hq/Hkv), fp32 softmax of
// q.k/sqrt(D), fp16 output).
//
// A workgroup is 4 waves, one per SIMD; each wave takes 64 consecutive queries
// of one head as two 32-query blocks A and B and walks keys in 32-key units.
// What bounds the 32-row tiles of prefill.hip is not the matrix cores but the
// LDS and the order of issue: per 32 rows x 64 keys a wave reads 32 KiB of K
// and V operands from LDS for 1024 cycles of MFMAs (four waves then ask for
// all of the LDS's 128 B per cycle), and its softmax and its MFMAs follow each
// other.  Here both blocks use each operand read (half the LDS bytes per
// MFMA), and the wave's instruction stream alternates two phases
//   1: softmax of A, next to the QK MFMAs of B and its PV MFMAs (previous unit)
//   2: softmax of B, next to the QK MFMAs of A (next unit) and its PV MFMAs
// with a few softmax instructions and operand reads placed after every MFMA
// (slot), so the vector ALU works in the MFMAs' shadow: an MFMA occupies the
// matrix core for 32 cycles and the issue port for about 8.
//  * S^T = K . Q^T and O^T = V^T . P^T on v_mfma_f32_32x32x16_f16, P in
//    registers, K and V tiles copied by LDS-DMA into rows whose 16-byte chunks
//    are XOR-swizzled (as in prefill.hip; 64-dim rows are 128 bytes and swizzle
//    by row pair).
//  * No row maximum is taken on the way: P is computed with the maximum as it
//    stands (a block's first unit sets it), and in the rare case that a query's
//    16 weights of a unit sum past kSumLimit the maximum is raised, O and l
//    rescaled and the unit redone.  Each query decides by its own weights, so a
//    row does not depend on the other rows of the wave.
//  * KS waves split a head's keys, their states combined through LDS at the
//    end.  KS = 4: one head per workgroup, each wave with rings of its own for
//    K and V and no barriers: the shortest chains.  KS = 2: two heads of one KV
//    head per workgroup, the copies shared by the two waves of a part.
//  * LO: the fp32 weights go into the PV product as two fp16 values (the
//    rounded weight and what it leaves, 22 bits together), so the outputs are
//    as close to float64 as attention_generic's, whose layouts these instances
//    take over (relative error 2.01e-4 either way at 16/4 heads of 64 and 16/16
//    of 128, the fp16 rounding of the output; 2.5e-4 without).  Far below the
//    row's largest weight two halves run out of exponent, which shows where the
//    large weights meet a V of zero (an attention sink): what is left of weights
//    14.6 nats and more below is multiplied apart (2.1e-4 either way beside sinks
//    of 6 to 20 nats; without it 2.9e-4 at 12 and 0.3-0.5 at 20).  Units with such
//    weights cost 2-3 phases instead of one: 16/16 heads of 128, 1000 tokens 18.7 us
//    where scores have a deviation of 1, 24 of 2, 47 of 3; 16/4 of 64, 1500 tokens
//    18.1, 24, 35 (attention_generic 570 and 650).
// Measured (one MI355X, graphs of 20 calls, us, against attention_generic):
// 16/4 heads of 64: 500 tokens 8.5 (78), 1500 17.1 (643), 4096 64 (4818);
// 16/16 heads of 128: 130 tokens 8.6 (18.4), 1000 17.0 (582), 4096 118 (9267);
// against prefill_skn at 16/4 heads of 128: 800 tokens 12.6 (14.7), 999 14.4
// (17.8), 32/8 heads 1000 tokens 23 (34).  A phase takes
// ~600 cycles for 512 cycles of MFMAs; short prompts are bound by the ~4 us of
// first copies (all of them: the compiler's wait for Q leaves none in flight), code
// fetch and state fold, long ones by the power the MFMAs draw.
#include "attn_internal.hpp"
#include "rows64_copies.hpp"

#include <type_traits>
#include <utility>

namespace attn {

namespace {

constexpr int kRows = 64;  // queries per workgroup
constexpr int kUnit = 32;  // keys per unit
// a lane's 16 fp16 weights of one unit may sum to this before the maximum is
// raised: each stays below the fp16 maximum, and weights that small keys get
// only gain by a maximum that lags
constexpr float kSumLimit = 4096.f;
// LO: weights are 2^kUp times the plain ones (as much as leaves flat scores half of
// the limit), because fp16 ends at 2^-24: the two halves hold 22 bits of a weight
// from 2^-3 on and 14 at kSmall.  What they leave of weights below kSmall (14.6 nats
// under the maximum) is multiplied apart, 2^kUpRest times as large.
constexpr float kUp = 11.f;
constexpr float kSumLimitLo = 65000.f;
constexpr float kSmall = 0x1p-10f;
constexpr uint16_t kSmallBits = 0x1400;  // as fp16
constexpr float kUpRest = 0x1p36f;
// running maximum before the first key: finite, so masked scores (-inf) get
// weight 0 without a special case
constexpr float kNoMax = -1.0e30f;

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

// The score MFMAs of one-wave-per-SIMD kernels, as inline assembly so that the
// scores land in vector registers (the compiler puts every MFMA result of
// such a kernel into accumulation registers and copies the scores back, 16
// moves per unit and block).  Nothing inserts the wait before a vector
// instruction that reads the result: within the loop eight more MFMAs follow
// before the block ends (each only issues once the one before it has left the
// pipe), and the chain before the loop ends with mfma32_last, which carries 32
// wait states, more than the 8 passes of the instruction.
__device__ __forceinline__ void mfma32_first(f32x16& c, f16x8 a, f16x8 b) {
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "a"(b));
}
__device__ __forceinline__ void mfma32_next(f32x16& c, f16x8 a, f16x8 b) {
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "a"(b));
}
__device__ __forceinline__ void mfma32_last(f32x16& c, f16x8 a, f16x8 b) {
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0\n\ts_nop 15\n\ts_nop 15"
                 : "+v"(c)
                 : "v"(a), "a"(b));
}
// four values kept in accumulation registers times f
__device__ __forceinline__ void scale_acc4(float& a, float& b, float& c, float& d, float f) {
    float t0, t1, t2, t3;
    asm volatile(
        "v_accvgpr_read_b32 %4, %0\n\t"
        "v_accvgpr_read_b32 %5, %1\n\t"
        "v_accvgpr_read_b32 %6, %2\n\t"
        "v_accvgpr_read_b32 %7, %3\n\t"
        "v_mul_f32 %4, %4, %8\n\t"
        "v_mul_f32 %5, %5, %8\n\t"
        "v_mul_f32 %6, %6, %8\n\t"
        "v_mul_f32 %7, %7, %8\n\t"
        "v_accvgpr_write_b32 %0, %4\n\t"
        "v_accvgpr_write_b32 %1, %5\n\t"
        "v_accvgpr_write_b32 %2, %6\n\t"
        "v_accvgpr_write_b32 %3, %7"
        : "+a"(a), "+a"(b), "+a"(c), "+a"(d), "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3)
        : "v"(f));
}
// four values kept in accumulation registers plus v times f
__device__ __forceinline__ void add_acc4(float& a, float& b, float& c, float& d, f32x4 v, float f) {
    float t0, t1, t2, t3;
    asm volatile(
        "v_accvgpr_read_b32 %4, %0\n\t"
        "v_accvgpr_read_b32 %5, %1\n\t"
        "v_accvgpr_read_b32 %6, %2\n\t"
        "v_accvgpr_read_b32 %7, %3\n\t"
        "v_fma_f32 %4, %8, %12, %4\n\t"
        "v_fma_f32 %5, %9, %12, %5\n\t"
        "v_fma_f32 %6, %10, %12, %6\n\t"
        "v_fma_f32 %7, %11, %12, %7\n\t"
        "v_accvgpr_write_b32 %0, %4\n\t"
        "v_accvgpr_write_b32 %1, %5\n\t"
        "v_accvgpr_write_b32 %2, %6\n\t"
        "v_accvgpr_write_b32 %3, %7"
        : "+a"(a), "+a"(b), "+a"(c), "+a"(d), "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3)
        : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(f));
}
// LDS reads at a byte address: 16 bytes, and four fp16 of one column
// (ds_read_b64_tr_b16, see prefill.hip)
__device__ __forceinline__ f16x8 lds16_at(uint32_t byte) {
    return *reinterpret_cast<LDS_AS const f16x8*>((uintptr_t)byte);
}
__device__ __forceinline__ f16x4 lds_tr4_at(uint32_t byte) {
    const s16x4 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(uintptr_t)byte);
    return __builtin_bit_cast(f16x4, r);
}
// f(0), ..., f(N - 1) with constant arguments (indexes of register arrays)
template <int N, class F>
__device__ __forceinline__ void each(F&& f) {
    [&]<int... I>(std::integer_sequence<int, I...>) __attribute__((always_inline)) {
        (f(std::integral_constant<int, I>{}), ...);
    }(std::make_integer_sequence<int, N>{});
}
// blockIdx -> (head group, query tile): longest tiles first, head groups
// pinned to XCDs when they divide the 8 of them
__device__ __forceinline__ void map_block(uint32_t bid, uint32_t groups, uint32_t q_tiles,
                                          uint32_t& grp, uint32_t& tile) {
    const uint32_t rank = (uint32_t)__builtin_amdgcn_readfirstlane(bid / groups);
    grp = bid - rank * groups;
    tile = q_tiles - 1u - rank;
}

// one 32-query block's running state
template <int D>
struct Block {
    f32x16 o[D / 32];
    f16x8 q[D / 16];
    f16x8 p[4];  // fp16 weights, then (LO) what they leave of the fp32 ones: B operands
    f32x16 s;
    f16x2 wmin;  // LO: the least of the lane's weights of the unit, as fp16
    float m, l, psum;
};

// One LDS-DMA copy (see dma16) into LDS byte `lds` + OFF.  M0 is left changed:
// a reserved register that nothing else in this kernel uses.
template <int OFF>
__device__ __forceinline__ void copy16(u32x4 r, uint32_t lds, uint32_t voff) {
    asm volatile(
        "s_add_u32 m0, %0, %3\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds),
        "v"(voff), "s"(r), "n"(OFF)
        : "memory", "scc");
}

// the lesser of each half; one instruction (the builtin quiets NaNs of both first)
__device__ __forceinline__ f16x2 min_pair(f16x2 a, f16x2 b) {
    f16x2 r;
    asm("v_pk_min_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// weight pairs w[0..7] (and w[8..15]) as the B operands of their PV steps
template <bool LO>
__device__ __forceinline__ void operands(f16x8 (&p)[4], const f16x2 (&w)[16]) {
    each<LO ? 4 : 2>([&](auto k_tag) __attribute__((always_inline)) {
        constexpr int k = decltype(k_tag)::value, i = 4 * k;
        p[k] = f16x8{w[i][0],     w[i][1],     w[i + 1][0], w[i + 1][1],
                     w[i + 2][0], w[i + 2][1], w[i + 3][0], w[i + 3][1]};
    });
}

// Output dims [d0, d0 + dims) (dims <= 128) of one (query, head) row by one
// wave, as attention_generic.hip computes it: 256 keys at a time, each lane
// scoring four, then each lane summing one or two dims over them in key order.
__device__ __forceinline__ void plain_row(const PrefillArgs& a, uint32_t row, uint32_t head,
                                          uint32_t g, uint32_t d0, uint32_t dims) {
    const uint32_t lane = threadIdx.x & 63u, D = a.head_dim;
    const f16* const q = a.q + (uint64_t)row * a.q_stride + (uint64_t)head * D;
    const f16* const k = a.k + (uint64_t)g * D;
    const f16* const v = a.v + (uint64_t)g * D + d0;
    // this lane's dims; lanes past the last repeat it
    const uint32_t d0l = min(lane, dims - 1u), d1l = min(lane + 64u, dims - 1u);
    float m = -INFINITY, l = 0.f, acc[2] = {0.f, 0.f};
    for (uint32_t j0 = 0; j0 <= row; j0 += 256u) {
        float s[4] = {0.f, 0.f, 0.f, 0.f}, mx = -INFINITY, sum = 0.f, part[2] = {0.f, 0.f};
        const f16* kr[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            kr[i] = k + (uint64_t)min(j0 + 64u * (uint32_t)i + lane, row) * a.kv_stride;
#pragma unroll 4
        for (uint32_t d = 0; d < D; d += 8u) {
            const f16x8 qd = ld16(q + d);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f16x8 kd = ld16(kr[i] + d);
#pragma unroll
                for (int e = 0; e < 8; ++e) s[i] += (float)qd[e] * (float)kd[e];
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s[i] = j0 + 64u * (uint32_t)i + lane <= row ? s[i] * a.scale_log2 : -INFINITY;
            mx = fmaxf(mx, s[i]);
        }
        const float mn = fmaxf(m, wave_max(mx));
        const float alpha = fast_exp2(m - mn);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s[i] = j0 + 64u * (uint32_t)i + lane <= row ? fast_exp2(s[i] - mn) : 0.f;
            sum += s[i];
        }
#pragma unroll 1
        for (int i = 0; i < 4; ++i) {
            const uint32_t first = j0 + 64u * (uint32_t)i;
            const float w = i < 2 ? (i == 0 ? s[0] : s[1]) : (i == 2 ? s[2] : s[3]);
            if (first > row) break;
            const uint32_t keys = row - first + 1u;
            for (uint32_t j1 = 0; j1 < min(64u, keys); j1 += 16u) {
                // sixteen loads at a time, pinned: the compiler moves each into the
                // branch that adds it, one round trip per key (past the row: the row's)
                f16 x[16][2];
#pragma unroll
                for (uint32_t e = 0; e < 16u; ++e) {
                    const f16* const vr = v + (uint64_t)min(first + j1 + e, row) * a.kv_stride;
                    x[e][0] = vr[d0l];
                    x[e][1] = vr[d1l];
                }
#pragma unroll
                for (uint32_t e = 0; e < 16u; ++e) asm volatile("" : "+v"(x[e][0]), "+v"(x[e][1]));
#pragma unroll
                for (uint32_t e = 0; e < 16u; ++e) {
                    if (j1 + e >= keys) break;
                    const float p = __builtin_bit_cast(
                        float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), (int)(j1 + e)));
                    part[0] += p * (float)x[e][0];
                    part[1] += p * (float)x[e][1];
                }
            }
        }
        l = l * alpha + wave_sum(sum);
        acc[0] = acc[0] * alpha + part[0];
        acc[1] = acc[1] * alpha + part[1];
        m = mn;
    }
    f16* const o = a.out + ((uint64_t)row * a.num_heads + head) * D + d0;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the row's first stores
    if (lane < dims) o[lane] = (f16)(acc[0] / l);
    if (lane + 64u < dims) o[lane + 64u] = (f16)(acc[1] / l);
}

template <int D, int KS, bool LO>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(D == 64 ? 2 : 1, D == 64 ? 2 : 1))) void prefill_rows64(
    PrefillArgs a) {
    constexpr int ND = D / 32;   // 32-dim output tiles
    constexpr int NK = D / 16;   // k-steps of the QK product
    constexpr int CH = D / 8;    // 16-byte chunks per row
    constexpr int NI = CH / 2;   // 1 KiB copies per unit of K or V
    constexpr int RI = 64 / CH;  // rows per copy
    constexpr uint32_t kUnitB = kUnit * D * 2;  // bytes of one unit of K or V
    constexpr int NP = LO ? 4 * ND : 2 * ND;    // PV MFMAs per phase
    constexpr int NS = NK + NP;                 // MFMAs (slots) per phase
    constexpr bool kAsm = D == 128;             // O in accumulation registers
    // LDS.  KS 2: four stages of two units, each K then V.  KS 4: per wave a ring
    // of three K units, then one of two V units.  At the end each wave's state
    // (4 units' bytes) and (m, l).
    constexpr uint32_t kStages = 4;
    constexpr uint32_t kStageB = KS * 2u * kUnitB;
    constexpr uint32_t kWaveB = (KS == 4 ? 5u : 4u) * kUnitB;
    __shared__ __attribute__((aligned(16))) char
        lds[4u * kWaveB + (KS == 2 ? 4096u : 0u)];
    static_assert(KS == 4 || kStages * kStageB == 4u * kWaveB);

    const int tid = threadIdx.x;
    const uint32_t lane = (uint32_t)tid & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t n = lane & 31u, hh = lane >> 5;
    const uint32_t part = KS == 2 ? wave >> 1 : wave;  // key part
    uint32_t grp, tile;
    map_block(blockIdx.x, a.num_heads * KS / 4u, a.q_tiles, grp, tile);
    const uint32_t head = KS == 2 ? 2u * grp + (wave & 1u) : grp;
    // the workgroup's heads share one KV head (uniform: keeps the copies' resources in SGPRs)
    const uint32_t g = (uint32_t)__builtin_amdgcn_readfirstlane(head / a.group);
    const uint32_t q0 = tile * kRows;
    const uint32_t N = a.seq_len;
    const uint32_t row_bytes = (uint32_t)(a.kv_stride * 2);
    const uint32_t dA = 2u * tile, dB = dA + 1u;  // the blocks' diagonal units
    // unit i of this wave is key unit KS i + part
    const uint32_t units = KS == 4 ? (part <= dB ? (dB - part) / 4u + 1u : 0u) : tile + 1u;
    auto unit_of = [&](uint32_t i) { return KS * i + part; };

    // ---- copies.  Copy j of a unit fills LDS bytes [1024 j, 1024 j + 1024) of
    // it: rows RI j .. RI j + RI - 1; lane L writes slot L % CH of row L / CH,
    // which holds the row's chunk slot ^ swizzle(row).  A stream's resource
    // starts at the row of its next stage (KS 4: unit) and ends at row N - 1:
    // past it reads return zero without touching memory, so copies past the
    // last stage are issued like the others and cost nothing.
    auto k_swz = [](uint32_t r) { return D == 128 ? (r & 15u) : ((r >> 1) & 7u); };
    auto v_swz = [](uint32_t r) { return D == 128 ? 4u * (r & 3u) : 4u * ((r >> 1) & 1u); };
    constexpr int NC = KS * NI / 4;  // copies per stage, wave and operand
    // KS 2: the 4 waves share a stage's rows, wave w takes copies w + 4 t, whose
    // rows swizzle alike; KS 4: copies t + 4 swizzle like t (D = 64: t + 2)
    constexpr int kKPat = KS == 4 ? (D == 128 ? 4 : 2) : 1;
    constexpr uint32_t kRowStep = KS == 4 ? (uint32_t)RI : 4u * RI;  // rows from copy to copy
    const uint32_t row0 = (KS == 4 ? 0u : (uint32_t)RI * wave) + lane / CH;
    uint32_t k_off[kKPat];
#pragma unroll
    for (int t = 0; t < kKPat; ++t)
        k_off[t] = (row0 + (uint32_t)RI * t) * row_bytes +
                   16u * ((lane % CH) ^ k_swz(row0 + (uint32_t)RI * t));
    const uint32_t v_off = row0 * row_bytes + 16u * ((lane % CH) ^ v_swz(row0));
    constexpr uint32_t kRowsPer = KS * kUnit;  // rows from stage to stage
    const uint64_t step_bytes = (uint64_t)kRowsPer * row_bytes;  // < 2^32: N + 64 rows fit
    // a stream's copy resource: base, bytes left
    struct Stream {
        uint64_t base;
        uint32_t left;
    };
    const uint32_t first_row = KS == 4 ? part * kUnit : 0u;
    auto stream = [&](const f16* p) __attribute__((always_inline)) {
        return Stream{reinterpret_cast<uint64_t>(p + (uint64_t)g * D) +
                          (uint64_t)first_row * row_bytes,
                      N > first_row ? (N - first_row - 1u) * row_bytes + 2u * D : 0u};
    };
    Stream sk = stream(a.k), sv = stream(a.v);
    auto resource = [&](const Stream& st) __attribute__((always_inline)) {
        return rsrc_words(reinterpret_cast<const void*>(st.base), st.left);
    };
    auto advance = [&](Stream& st) __attribute__((always_inline)) {
        st.base += step_bytes;
        st.left = st.left > (uint32_t)step_bytes ? st.left - (uint32_t)step_bytes : 0u;
    };
    const uint32_t lds0 = lds_addr(lds);
    // copy t of a stage (KS 4: unit) of K / V whose LDS starts at `to`
    auto copy_at = [&](auto t_tag, uint32_t off, u32x4 r, uint32_t to)
                       __attribute__((always_inline)) {
        constexpr int t = decltype(t_tag)::value;
        if constexpr (KS == 4) copy16<1024 * t>(r, to, off);
        else copy16<(4 * t / NI) * 2 * (int)kUnitB + 1024 * (4 * t % NI)>(r, to, off);
    };
    auto copy_kt = [&](auto t_tag, u32x4 r, uint32_t to) __attribute__((always_inline)) {
        constexpr int t = decltype(t_tag)::value;
        copy_at(t_tag, k_off[t % kKPat] + (uint32_t)(t - t % kKPat) * kRowStep * row_bytes, r, to);
    };
    auto copy_vt = [&](auto t_tag, u32x4 r, uint32_t to) __attribute__((always_inline)) {
        constexpr int t = decltype(t_tag)::value;
        copy_at(t_tag, v_off + (uint32_t)t * kRowStep * row_bytes, r, to);
    };
    uint32_t st_to = lds0 + (KS == 4 ? 0u : 1024u * wave);  // KS 2: next stage's LDS
    uint32_t k_to = lds0 + wave * kWaveB;                    // KS 4: the rings' next units
    uint32_t v_to = k_to + 3u * kUnitB;
    const uint32_t ring = lds0 + wave * kWaveB;
    auto next_k = [&](uint32_t& p) __attribute__((always_inline)) {
        p = p == ring + 2u * kUnitB ? ring : p + kUnitB;
    };
    auto next_v = [&](uint32_t& p) __attribute__((always_inline)) {
        p = p == ring + 3u * kUnitB ? p + kUnitB : ring + 3u * kUnitB;
    };
    auto next_stage = [&](uint32_t& p, uint32_t first) __attribute__((always_inline)) {
        p = p == first + (kStages - 1u) * kStageB ? first : p + kStageB;
    };
    auto stage = [&]() __attribute__((always_inline)) {  // a whole stage at once
        const u32x4 rk = resource(sk), rv = resource(sv);
        [&]<int... T>(std::integer_sequence<int, T...>) {
            (copy_kt(std::integral_constant<int, T>{}, rk, st_to), ...);
            (copy_vt(std::integral_constant<int, T>{}, rv, st_to + kUnitB), ...);
        }(std::make_integer_sequence<int, NC>{});
        advance(sk);
        advance(sv);
        next_stage(st_to, lds0 + 1024u * wave);
    };
    auto unit_k = [&]() __attribute__((always_inline)) {
        const u32x4 r = resource(sk);
        [&]<int... T>(std::integer_sequence<int, T...>) {
            (copy_kt(std::integral_constant<int, T>{}, r, k_to), ...);
        }(std::make_integer_sequence<int, NC>{});
        advance(sk);
        next_k(k_to);
    };
    auto unit_v = [&]() __attribute__((always_inline)) {
        const u32x4 r = resource(sv);
        [&]<int... T>(std::integer_sequence<int, T...>) {
            (copy_vt(std::integral_constant<int, T>{}, r, v_to), ...);
        }(std::make_integer_sequence<int, NC>{});
        advance(sv);
        next_v(v_to);
    };

    // ---- operand reads.  K: row n, chunk 2 ks + hh.  V: transposing reads of
    // keys 4 hh + 0..3 (+ 8, + 16), 32 dims per tile (see prefill.hip).  Byte
    // offsets into a unit.
    const uint32_t jl = lane & 15u, sub = (lane >> 4) & 1u;
    uint32_t k_rd[NK], v_rd[ND];
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) k_rd[ks] = 2u * n * D + 16u * ((2u * ks + hh) ^ k_swz(n));
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
        v_rd[dt] = 2u * ((4u * hh + (jl >> 2)) * D + 16u * sub + 4u * (jl & 3u) +
                         32u * ((uint32_t)dt ^ (D == 128 ? jl >> 2 : jl >> 3)));
    f16x8 kf[NK], vf[2][ND];
    auto load_k = [&](uint32_t u, int ks) __attribute__((always_inline)) { kf[ks] = lds16_at(u + k_rd[ks]); };
    auto load_v = [&](uint32_t u, int f) __attribute__((always_inline)) {
        const int ks = f / ND, dt = f % ND;
        const f16x4 lo = lds_tr4_at(u + v_rd[dt] + 32 * ks * D);
        const f16x4 hi = lds_tr4_at(u + v_rd[dt] + (32 * ks + 16) * D);
        vf[ks][dt] = f16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };

    Block<D> A, B;
    auto init = [&](Block<D>& x) __attribute__((always_inline)) {
        each<ND>([&](auto t) __attribute__((always_inline)) { x.o[decltype(t)::value] = f32x16{}; });
        x.m = kNoMax;
        x.l = 0.f;
    };
    init(A);
    init(B);

    // k-step ks of the scores of block x with the K operands at hand
    auto score = [&](Block<D>& x, int ks, bool wait = false) __attribute__((always_inline)) {
        if constexpr (kAsm) {
            if (ks == 0) mfma32_first(x.s, kf[ks], x.q[ks]);
            else if (wait && ks == NK - 1) mfma32_last(x.s, kf[ks], x.q[ks]);
            else mfma32_next(x.s, kf[ks], x.q[ks]);
        } else {
            x.s = mfma32(kf[ks], x.q[ks], ks == 0 ? f32x16{} : x.s);
        }
    };
    const float scale = a.scale_log2;
    constexpr float up = LO ? kUp : 0.f;
    constexpr float kLimit = LO ? kSumLimitLo : kSumLimit;
    // P of the unit with the running maximum as it is, and the lane's sum of it
    // (of the weights PV multiplies: the fp16 ones, or with LO the fp32 ones),
    // added in the order of `phase`: a row whose weights are only computed again
    // because others' are keeps its bits
    auto weights = [&](Block<D>& x) __attribute__((always_inline)) {
        f16x2 w[16];
        float psum[2] = {0.f, 0.f};
        each<8>([&](auto j_tag) __attribute__((always_inline)) {
            constexpr int j = decltype(j_tag)::value;
            const float w0 = fast_exp2(__builtin_fmaf(x.s[2 * j], scale, -x.m));
            const float w1 = fast_exp2(__builtin_fmaf(x.s[2 * j + 1], scale, -x.m));
            w[j] = f16x2{(f16)w0, (f16)w1};
            if constexpr (LO)
                w[8 + j] = f16x2{(f16)(w0 - (float)(f16)w0), (f16)(w1 - (float)(f16)w1)};
            if constexpr (LO) psum[j & 1] += w0 + w1;
            else psum[j & 1] = add_pair(psum[j & 1], w[j]);
            if constexpr (LO) x.wmin = j == 0 ? w[0] : min_pair(x.wmin, w[j]);
        });
        operands<LO>(x.p, w);
        x.psum = psum[0] + psum[1];
    };
    // scores of unit u past the diagonal of block y, whose diagonal unit is d <= u
    auto mask = [&](Block<D>& y, uint32_t u, uint32_t d) __attribute__((always_inline)) {
        // keys of the unit up to n are visible; of the lane's, those below top
        const int top = u > d ? 0 : (int)n + 1 - 4 * (int)hh;
        each<16>([&](auto e_tag) __attribute__((always_inline)) {
            constexpr int e = decltype(e_tag)::value;
            y.s[e] = 8 * (e >> 2) + (e & 3) >= top ? -INFINITY : y.s[e];
        });
    };
    auto unit_max = [&](const Block<D>& x) __attribute__((always_inline)) {
        float mx = x.s[0];
        each<15>([&](auto t) __attribute__((always_inline)) {
            mx = fmaxf(mx, x.s[decltype(t)::value + 1]);
        });
        return mx;
    };
    // LO: whether a weight of the lane's unit is below kSmall
    auto small = [&](const Block<D>& x) __attribute__((always_inline)) {
        if constexpr (!LO) return false;
        else {
            // weights are not negative: as integers in their order
            const u16x2 less = __builtin_bit_cast(u16x2, x.wmin) - kSmallBits;
            return (__builtin_bit_cast(uint32_t, less) & 0x80008000u) != 0;
        }
    };
    // ... and the least exponent of the unit's visible keys
    auto unit_min = [&](const Block<D>& x) __attribute__((always_inline)) {
        float mn = INFINITY;
        each<16>([&](auto e_tag) __attribute__((always_inline)) {
            constexpr int e = decltype(e_tag)::value;
            mn = fminf(mn, x.s[e] == -INFINITY ? INFINITY : x.s[e]);
        });
        return __builtin_fmaf(mn, scale, -x.m);
    };
    // In accumulation registers the asm on O neither waits for MFMAs before it nor
    // keeps those after it away: 32 wait states on both sides do
    auto apart = [&](Block<D>& x) __attribute__((always_inline)) {
        if constexpr (kAsm)
            asm volatile("s_nop 15\n\ts_nop 15"
                         : "+a"(x.o[0]), "+a"(x.o[1]), "+a"(x.o[2]), "+a"(x.o[3]));
    };
    // O times f
    auto scale_o = [&](Block<D>& x, float f) __attribute__((always_inline)) {
        apart(x);
        each<4 * ND>([&](auto i_tag) __attribute__((always_inline)) {
            constexpr int dt = decltype(i_tag)::value / 4, e = decltype(i_tag)::value % 4 * 4;
            float v[4] = {x.o[dt][e], x.o[dt][e + 1], x.o[dt][e + 2], x.o[dt][e + 3]};
            if constexpr (kAsm) {
                scale_acc4(v[0], v[1], v[2], v[3], f);
            } else {
                v[0] *= f;
                v[1] *= f;
                v[2] *= f;
                v[3] *= f;
            }
            x.o[dt][e] = v[0];
            x.o[dt][e + 1] = v[1];
            x.o[dt][e + 2] = v[2];
            x.o[dt][e + 3] = v[3];
        });
        apart(x);
    };
    // What both halves leave of the weights of x's unit below kSmall, through a
    // product of its own.  Weights from kSmall on leave nothing here, so that a
    // row does not depend on the others.  The unit's V operands are at hand.
    auto pv_rest = [&](Block<D>& x) __attribute__((always_inline)) {
        f16x8 p[2];
        // read back from the operands' registers; else they stay in others as well
        each<4>([&](auto k_tag) __attribute__((always_inline)) {
            f16x8& own = x.p[decltype(k_tag)::value];
            asm volatile("" : "+v"(own));
        });
        each<8>([&](auto j_tag) __attribute__((always_inline)) {
            constexpr int j = decltype(j_tag)::value, k = j / 4, i = j % 4 * 2;
            f16x2 left;
            each<2>([&](auto h_tag) __attribute__((always_inline)) {
                constexpr int h = decltype(h_tag)::value;
                const float w = fast_exp2(__builtin_fmaf(x.s[2 * j + h], scale, -x.m));
                const f16 hi = x.p[k][i + h];
                const float l = (w - (float)hi) - (float)x.p[2 + k][i + h];
                left[h] = (f16)(hi < (f16)kSmall ? l * kUpRest : 0.f);
            });
            asm volatile("" : "+v"(left));  // one pair at a time: registers are short
            p[k][i] = left[0];
            p[k][i + 1] = left[1];
        });
        apart(x);
        each<ND>([&](auto dt_tag) __attribute__((always_inline)) {
            constexpr int dt = decltype(dt_tag)::value;
            f32x16 t = mfma32(vf[0][dt], p[0], f32x16{});
            t = mfma32(vf[1][dt], p[1], t);
            if constexpr (kAsm) asm volatile("s_nop 15\n\ts_nop 15" : "+v"(t));
            each<4>([&](auto i_tag) __attribute__((always_inline)) {
                constexpr int e = 4 * decltype(i_tag)::value;
                float v[4] = {x.o[dt][e], x.o[dt][e + 1], x.o[dt][e + 2], x.o[dt][e + 3]};
                if constexpr (kAsm) {
                    add_acc4(v[0], v[1], v[2], v[3], f32x4{t[e], t[e + 1], t[e + 2], t[e + 3]},
                             1.f / kUpRest);
                } else {
                    v[0] = __builtin_fmaf(t[e], 1.f / kUpRest, v[0]);
                    v[1] = __builtin_fmaf(t[e + 1], 1.f / kUpRest, v[1]);
                    v[2] = __builtin_fmaf(t[e + 2], 1.f / kUpRest, v[2]);
                    v[3] = __builtin_fmaf(t[e + 3], 1.f / kUpRest, v[3]);
                }
                x.o[dt][e] = v[0];
                x.o[dt][e + 1] = v[1];
                x.o[dt][e + 2] = v[2];
                x.o[dt][e + 3] = v[3];
            });
        });
        apart(x);
    };
    // Between two phases.  x's weights of its unit are complete: raise the
    // maximum of the queries whose weights passed the limit (the two lanes of a
    // query together), rescale O and l and redo the unit.  y's scores of unit u
    // are complete: mask them past the diagonal, y's diagonal unit being d.  One
    // test and one branch for both, rarely taken.  inside: x's unit is before its
    // diagonal; lanes: those whose weights ask for it; get_v: the V operands of x's
    // unit into vf.
    auto settle = [&](Block<D>& x, bool inside, Block<D>& y, uint32_t u, uint32_t d,
                      uint64_t lanes, auto&& get_v) __attribute__((always_inline)) {
        if (__builtin_expect((lanes | (u >= d ? ~0ull : 0ull)) != 0, 0)) {
            const bool over = !(x.psum < kLimit);
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(over) != 0, 0)) {
                const float mx = unit_max(x);
                const bool raise = max_xor<32>(over ? 1.f : 0.f) != 0.f;
                const float m_unit = max_xor<32>(mx) * scale - up;
                const float mn = raise ? fmaxf(x.m, m_unit) : x.m;
                const float al = fast_exp2(x.m - mn);
                x.m = mn;
                weights(x);
                x.l *= al;
                scale_o(x, al);
            }
            if constexpr (LO) {
                // keys past the diagonal have weight 0, which is not small
                const bool low = small(x) && (inside || unit_min(x) < -10.f);
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(low) != 0, 0)) {
                    get_v();
                    pv_rest(x);
                }
            }
            if (u >= d) mask(y, u, d);
        }
        x.l += x.psum;
    };
    // before a block's first weights: the maximum of its first unit
    auto first_max = [&](Block<D>& x) __attribute__((always_inline)) {
        x.m = fmaxf(kNoMax, max_xor<32>(unit_max(x)) * scale - up);
    };
    // PV MFMA f of block y: dim tile f % ND, step f / ND (LO: the weights, then in steps
    // 2 and 3 what they leave)
    auto pv = [&](Block<D>& y, auto f_tag) __attribute__((always_inline)) {
        constexpr int ks = decltype(f_tag)::value / ND, dt = decltype(f_tag)::value % ND;
        y.o[dt] = mfma32(vf[ks & 1][dt], y.p[ks], y.o[dt]);
    };
    // One phase: the softmax of x next to the QK MFMAs of y's next unit and then
    // the PV MFMAs of y's current one, one MFMA per slot, each with its share of
    // the rest; rd 1: K operands of the unit at `u` read once the QK MFMAs have
    // gone, rd 2: V operands read before the PV MFMAs; cp(slot): copies and
    // waits.  A pair of scores moves one step (scale and shift, exponential,
    // conversion, sum) per slot, so no step waits for the one before it.  The
    // empty assembly statements pin every step to its slot (the MFMAs and
    // copies are volatile or bounded by the scheduling barriers).
    auto phase = [&](Block<D>& x, Block<D>& y, auto rd_tag, uint32_t u, auto&& cp)
                     __attribute__((always_inline)) {
        constexpr int kRd = decltype(rd_tag)::value;
        const float mneg = -x.m;
        float psum[2] = {0.f, 0.f};
        float sh[16], ex[16];
        f16x2 w[16], wmin;
        uint64_t lanes = 0;
        [&]<int... SL>(std::integer_sequence<int, SL...>) {
            ([&] {
                constexpr int sl = SL;
                if constexpr (sl < NK) {
                    score(y, sl);
                    if constexpr (kRd == 2 && sl < ND) {
                        load_v(u, 2 * sl);
                        load_v(u, 2 * sl + 1);
                    }
                }
                cp(std::integral_constant<int, sl>{});
                if constexpr (sl >= NK) {
                    constexpr int f = sl - NK;
                    pv(y, std::integral_constant<int, f>{});
                    if constexpr (kRd == 1 && f < NK / 2) {
                        load_k(u, 2 * f);
                        load_k(u, 2 * f + 1);
                    }
                }
                [&]<int... J>(std::integer_sequence<int, J...>) {
                    ([&] {
                        // slot of pair J's first step
                        constexpr int e = 2 * J;
                        constexpr int f = J * (NS - 3) / 8;
                        if constexpr (sl == f + 2) {
                            // LO: in asm, or the compiler converts again for the
                            // operands (s_nop: v_exp_f32's result may be read one
                            // instruction after it, which the compiler sees to for
                            // instructions of its own only)
                            if constexpr (LO)
                                asm("s_nop 0\n\tv_cvt_pk_f16_f32 %0, %1, %2"
                                    : "=v"(w[J])
                                    : "v"(ex[e]), "v"(ex[e + 1]));
                            else w[J] = f16x2{(f16)ex[e], (f16)ex[e + 1]};
                            if constexpr (LO) psum[J & 1] += ex[e] + ex[e + 1];
                            else psum[J & 1] = add_pair(psum[J & 1], w[J]);
                            asm volatile("" ::"v"(w[J]), "v"(psum[J & 1]));
                            if constexpr (LO) {
                                wmin = J == 0 ? w[0] : min_pair(wmin, w[J]);
                                w[8 + J] = f16x2{(f16)(ex[e] - (float)w[J][0]),
                                                 (f16)(ex[e + 1] - (float)w[J][1])};
                                asm volatile("" : "+v"(w[8 + J]) : "v"(wmin));
                            }
                        }
                        if constexpr (sl == f + 1) {
                            ex[e] = fast_exp2(sh[e]);
                            ex[e + 1] = fast_exp2(sh[e + 1]);
                            asm volatile("" ::"v"(ex[e]), "v"(ex[e + 1]));
                        }
                        if constexpr (sl == f) {
                            sh[e] = __builtin_fmaf(x.s[e], scale, mneg);
                            sh[e + 1] = __builtin_fmaf(x.s[e + 1], scale, mneg);
                            asm volatile("" ::"v"(sh[e]), "v"(sh[e + 1]));
                        }
                    }(), ...);
                }(std::make_integer_sequence<int, 8>{});
                // every weight is there: which lanes have something for settle
                if constexpr (sl == NS - 2) {
                    x.psum = psum[0] + psum[1];
                    if constexpr (LO) x.wmin = wmin;
                    lanes = __builtin_amdgcn_ballot_w64(!(x.psum < kLimit)) |
                            __builtin_amdgcn_ballot_w64(small(x));
                }
                __builtin_amdgcn_sched_barrier(0);
            }(), ...);
        }(std::make_integer_sequence<int, NS>{});
        operands<LO>(x.p, w);
        return lanes;
    };

    using rK = std::integral_constant<int, 1>;
    using rV = std::integral_constant<int, 2>;
    auto landed = [](auto n_tag) {  // at most n copies of this wave are in flight
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(decltype(n_tag)::value));
        asm volatile("" ::: "memory");
    };
    auto meet = []() {  // the workgroup's waves; LDS reads stay on their side
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if (units) {
        // Q^T B operands of both blocks, before the first copies; rows past N
        // read as zero
        const uint32_t q_row_bytes = (uint32_t)(a.q_stride * 2);
        const BufRsrc rq = make_rsrc(a.q + (uint64_t)head * D,
                                     __builtin_amdgcn_readfirstlane((N - 1u) * q_row_bytes + 2u * D));
        const uint32_t qoff = (q0 + n) * q_row_bytes + 16u * hh;
#pragma unroll
        for (int s = 0; s < NK; ++s) {
            A.q[s] = buf_ld16(rq, qoff + 32u * s);
            B.q[s] = buf_ld16(rq, qoff + 32u * q_row_bytes + 32u * s);
        }
        // LDS of the unit at hand: K, and V
        uint32_t ku = KS == 4 ? ring : lds0 + part * 2u * kUnitB;
        uint32_t vu = KS == 4 ? ring + 3u * kUnitB : ku + kUnitB;
        if constexpr (KS == 4) {
            each<4>([&](auto t) __attribute__((always_inline)) {
                if constexpr (rows64::kFirst.k[decltype(t)::value]) unit_k();
                else unit_v();
            });
            landed(std::integral_constant<int, rows64::kLeftFirst * NI>{});
        } else {
            stage();
            stage();
            stage();
            landed(std::integral_constant<int, 4 * NC>{});
            meet();
        }
        // Q has landed too: without this, the compiler waits for it at its first
        // uses in the loop, and with it, in every iteration, for every copy.  Its
        // wait here leaves none of the first copies in flight either (it does not
        // count them); nothing below relies on that
#pragma unroll
        for (int s = 0; s < NK; ++s) {
            if constexpr (kAsm) asm volatile("" : "+a"(A.q[s]), "+a"(B.q[s]));
            else asm volatile("" : "+v"(A.q[s]), "+v"(B.q[s]));
        }
#pragma unroll
        for (int ks = 0; ks < NK; ++ks) load_k(ku, ks);
#pragma unroll
        for (int ks = 0; ks < NK; ++ks) score(A, ks);
#pragma unroll
        for (int ks = 0; ks < NK; ++ks) score(B, ks, true);
        // the maxima to start from (phase 1 computes B's scores again)
        if (unit_of(0) >= dA) mask(A, unit_of(0), dA);
        if (unit_of(0) >= dB) mask(B, unit_of(0), dB);
        first_max(A);
        first_max(B);
        // B's weights "before the first unit" are 0, as are the V operands
        each<4>([&](auto k) __attribute__((always_inline)) { B.p[decltype(k)::value] = f16x8{}; });
        each<2 * ND>([&](auto f_tag) __attribute__((always_inline)) {
            constexpr int f = decltype(f_tag)::value;
            vf[f / ND][f % ND] = f16x8{};
        });
        u32x4 rk = resource(sk), rv = resource(sv);
        // Unit i: A's scores and its K operands are there.  Phase 1 reads K of
        // unit i + 1 (past the last unit: whatever is there, for scores nobody
        // reads), phase 2 V of unit i.
        for (uint32_t i = 0; i < units; ++i) {
            if constexpr (KS == 4) next_k(ku);
            else next_stage(ku, lds0 + part * 2u * kUnitB);
            uint64_t lanes =
                phase(A, B, rK{}, ku, [&](auto sl_tag) __attribute__((always_inline)) {
                constexpr int sl = decltype(sl_tag)::value;
                if constexpr (KS == 4) {
                    // K of unit i has been read: its LDS takes unit i + 3's.  K of
                    // unit i + 1 has landed; K i + 2, V i and K i + 3 may be in
                    // flight (rows64_copies.hpp)
                    if constexpr (sl < NC) copy_kt(sl_tag, rk, k_to);
                    if constexpr (sl == NK - 1)
                        landed(std::integral_constant<int, rows64::kLeftK * NI>{});
                    if constexpr (sl == NC) {
                        advance(sk);
                        rk = resource(sk);
                        next_k(k_to);
                    }
                } else {
                    // stage i + 1 has landed for this wave, then for all; every
                    // wave has read stage i - 1, whose LDS takes stage i + 3
                    if constexpr (sl == NK - 2) landed(std::integral_constant<int, 2 * NC>{});
                    if constexpr (sl == NK - 1) meet();
                }
            });
            settle(A, unit_of(i) < dA, B, unit_of(i), dB, lanes,
                   [&]() __attribute__((always_inline)) {
                // phase 1 is done with the V operands of unit i - 1
                if constexpr (KS == 4) landed(std::integral_constant<int, rows64::kLeftV * NI>{});
                each<2 * ND>([&](auto f) __attribute__((always_inline)) {
                    load_v(vu, decltype(f)::value);
                });
            });
            if constexpr (KS == 4)  // V of unit i; K i + 3 may be in flight
                landed(std::integral_constant<int, rows64::kLeftV * NI>{});
            lanes = phase(B, A, rV{}, vu, [&](auto sl_tag) __attribute__((always_inline)) {
                constexpr int sl = decltype(sl_tag)::value;
                constexpr int c = sl - ND;  // the slots without operand reads
                if constexpr (KS == 4) {
                    // V of unit i - 1 has been read: its LDS takes unit i + 1's
                    if constexpr (c >= 0 && c < NC)
                        copy_vt(std::integral_constant<int, c>{}, rv, v_to);
                    if constexpr (c == NC) {
                        advance(sv);
                        rv = resource(sv);
                        next_v(v_to);
                    }
                } else {
                    if constexpr (c >= 0 && c < NC)
                        copy_kt(std::integral_constant<int, c>{}, rk, st_to);
                    if constexpr (c >= NC && c < 2 * NC)
                        copy_vt(std::integral_constant<int, c - NC>{}, rv, st_to + kUnitB);
                    if constexpr (c == 2 * NC) {
                        advance(sk);
                        rk = resource(sk);
                    }
                    if constexpr (c == 2 * NC + 1) {
                        advance(sv);
                        rv = resource(sv);
                        next_stage(st_to, lds0 + 1024u * wave);
                    }
                }
            });
            settle(B, unit_of(i) < dB, A, i + 1 < units ? unit_of(i + 1) : 0u, dA, lanes, []() {});
            if constexpr (KS == 4) next_v(vu);
            else vu = ku + kUnitB;
        }
        [&]<int... F>(std::integer_sequence<int, F...>) {
            (pv(B, std::integral_constant<int, F>{}), ...);
        }(std::make_integer_sequence<int, NP>{});
        // copies past the last stage still write (zeros) to LDS
        landed(std::integral_constant<int, 0>{});
    }

    // ---- epilogue: O = O^T / l, packed [N][Hq][D]; lane (hh, n) holds dims
    // 32 dt + 8 (i / 4) + 4 hh + i % 4 of query n
    float bad = 0.f;  // NaN once a stored value was not finite
    auto store = [&](uint32_t blk, uint32_t dt, const f32x16& o, float inv) {
        const uint32_t query = q0 + 32u * blk + n;
        if (query >= N) return;
        f16* const orow = a.out + ((uint64_t)query * a.num_heads + head) * D + 32u * dt + 4u * hh;
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
            f16x4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v = o[4 * i4 + e] * inv;
                bad = __builtin_fmaf(v, 0.f, bad);
                w[e] = (f16)v;
            }
            *reinterpret_cast<f16x4*>(orow + 8 * i4) = w;
        }
    };
    {
        // every wave leaves its state in LDS ([block][dim tile][4 words] x 64
        // lanes of 16 bytes), then folds its share of the rows and dims over
        // the parts of its head: M = max m, l and O scaled by 2^(m - M)
        if constexpr (KS == 2) __syncthreads();  // every wave's stages are consumed and landed
        auto state = [&](uint32_t w) {
            return reinterpret_cast<f32x4*>(lds + w * kWaveB) + lane;
        };
        auto state_ml = [&](uint32_t w) {
            return reinterpret_cast<f32x2*>(KS == 4 ? lds + w * kWaveB + 4u * kUnitB
                                                    : lds + 4u * kWaveB + w * 1024u) + lane;
        };
        auto put = [&](const Block<D>& x, uint32_t blk) __attribute__((always_inline)) {
            each<4 * ND>([&](auto i_tag) __attribute__((always_inline)) {
                constexpr int i = decltype(i_tag)::value, dt = i / 4, e = i % 4 * 4;
                state(wave)[64u * (blk * ND * 4u + i)] =
                    f32x4{x.o[dt][e], x.o[dt][e + 1], x.o[dt][e + 2], x.o[dt][e + 3]};
            });
            state_ml(wave)[64u * blk] = f32x2{x.m, x.l};
        };
        put(A, 0);
        put(B, 1);
        __syncthreads();
        constexpr int kDt = KS == 2 ? ND : ND / 2;  // dim tiles per wave
        const uint32_t blk = KS == 2 ? part : part >> 1;
        const uint32_t dt0 = KS == 2 ? 0u : (part & 1u) * (uint32_t)kDt;
        auto from = [&](int w) { return KS == 2 ? (wave & 1u) + 2u * (uint32_t)w : (uint32_t)w; };
        f32x2 ml[KS];
        float M = kNoMax;
#pragma unroll
        for (int w = 0; w < KS; ++w) {
            ml[w] = state_ml(from(w))[64u * blk];
            M = fmaxf(M, ml[w][0]);
        }
        float l = 0.f, wt[KS];
#pragma unroll
        for (int w = 0; w < KS; ++w) {
            wt[w] = fast_exp2(ml[w][0] - M);
            l += wt[w] * ml[w][1];
        }
        l = add_xor<32>(l);
        const float inv = 1.f / l;
#pragma unroll
        for (int d = 0; d < kDt; ++d) {
            f32x16 o = f32x16{};
#pragma unroll
            for (int w = 0; w < KS; ++w) {
                const f32x4* src = state(from(w)) + 64u * ((blk * ND + dt0 + d) * 4u);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const f32x4 x = src[64 * q];
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[4 * q + e] += wt[w] * x[e];
                }
            }
            store(blk, dt0 + d, o, inv);
        }
        // Rows with a value that is not finite are done again key by key: an MFMA
        // multiplies the masked keys of a tile (weight 0) too, so an infinity or NaN
        // in V reaches rows before it, and the two halves of a weight (LO) turn an
        // infinity into a NaN.  A sum that is NaN (a score was NaN or +infinity)
        // makes the row NaN either way: with every input NaN, 16/4 heads of 128 at
        // 1000 tokens took 10.6 ms, 16/16 10.8, without this test.
        uint64_t rows = __builtin_amdgcn_ballot_w64(bad != 0.f && l == l);
        rows = (rows | rows >> 32) & 0xffffffffull;
        if constexpr (!LO) {
            // only where one of the tile's keys after the row is at fault
            if (rows != 0) {
                const uint32_t key = q0 + lane;
                bool fault = false;
#pragma unroll 1
                for (uint32_t c = 0; key < N && c < 4u * (uint32_t)kDt; ++c) {
                    const f16x8 x = ld16(a.v + (uint64_t)key * a.kv_stride + (uint64_t)g * D +
                                         32u * dt0 + 8u * c);
#pragma unroll
                    for (int e = 0; e < 8; ++e) fault |= !((float)x[e] * 0.f == 0.f);
                }
                const uint64_t keys = __builtin_amdgcn_ballot_w64(fault) >> (32u * blk);
                const uint32_t past = keys == 0 ? 0u : 63u - (uint32_t)__builtin_clzll(keys);
                if (past < 32u) rows &= (1ull << past) - 1u;  // rows 0 .. past - 1 of the block
            }
        }
        for (; rows != 0; rows &= rows - 1)
            plain_row(a, q0 + 32u * blk + (uint32_t)__builtin_ctzll(rows), head, g,
                      32u * dt0, 32u * (uint32_t)kDt);
    }
}

}  // namespace

// Which calls take this kernel: key parts per head (2 or 4), 0 when another
// kernel takes the call.  `mfma`: prefill.hip takes the layout too.
int rows64_parts(const PrefillArgs& a, bool mfma, int device) {
    if (get_option(kOptPrefillForceGeneric)) return 0;
    if (a.head_dim != 64 && a.head_dim != 128) return 0;
    if (a.group == 0 || a.q_stride % 8 != 0 || a.kv_stride % 8 != 0) return 0;
    if (!aligned16(a.q) || !aligned16(a.k) || !aligned16(a.v) || !aligned16(a.out)) return 0;
    // every row offset must fit the 32-bit buffer ranges, 128 rows a 32-bit step
    const uint64_t stride = a.q_stride > a.kv_stride ? a.q_stride : a.kv_stride;
    if ((uint64_t)(a.seq_len + kRows) * stride * 2 + a.head_dim * 2u > 0xffffffffull) return 0;
    if (stride * 2 > 0x1000000u) return 0;
    const uint64_t cus = (uint64_t)device_cu_count(device);
    const uint64_t wgs = (uint64_t)((a.seq_len + kRows - 1) / kRows) * a.num_heads;
    if (mfma) {
        // Part of the streaming split-keys form's range (the same units, split
        // over the waves the same way), unless an option asks for a form of
        // prefill.hip; the key-halves tile keeps its range from 1025 tokens (where
        // this kernel is ahead by 5-13 % up to 2048).
        if (a.seq_len <= 256u || a.seq_len > 1024u || get_option(kOptPrefillSplitKeys) ||
            get_option(kOptPrefillWaves) || get_option(kOptPrefillStageAll) ||
            get_option(kOptPrefillKeyHalves) == 2)
            return 0;
        // From 11/16 of a workgroup per CU to two: fewer leave the shorter chains
        // of prefill_skn's 32-query workgroups ahead, more (160 KiB of LDS: one
        // per CU at a time) a third round.  us against prefill_skn: 16 heads 600
        // tokens (160 workgroups) 11.6 against 11.1, 800 (208) 12.6 / 14.7, 999
        // (256) 14.4 / 17.8; 32 heads 350 (192) 10.5 / 10.7, 500 (256) 11.4 /
        // 14.2, 1000 (512) 23 / 34; 8 heads 1000 (128) 14.1 / 12.7.  A second
        // round pays from 417 tokens, or where prefill_skn's workgroups pass 9/4
        // per CU: 64 heads 280 (576 of those) 14.6 / 13.9, 289 (640) 14.7 / 15.6, 48
        // heads 340 (528) 14.6 / 13.4, 40 heads 400 (520) 14.5 / 13.5, 448 (560) 14.8 /
        // 16.2.  Up to 256 tokens prefill_d128's all-tiles form: 64 heads 150 tokens
        // 9.1 / 7.6, 192 10.0 / 8.6, 128 heads 150 14.6 / 11.7.
        const uint64_t wgs32 = (uint64_t)((a.seq_len + 31) / 32) * a.num_heads;
        if (16u * wgs <= 11u * cus || wgs > 2u * cus) return 0;
        return wgs <= cus || a.seq_len > 416u || 4u * wgs32 > 9u * cus ? 4 : 0;
    }
    // The other layouts ran attention_generic, whose time grows with the heads, up to
    // ~140 tokens this kernel's does not.  us, attention_generic / this: 64-dim heads, 64
    // tokens 1 head 5.56 / 5.64, 2 5.69 / 5.83, 16 6.50 / 5.90; 68 tokens 1 5.78 / 5.71.
    // 128-dim heads: 64 tokens 20 heads 8.44 / 7.81; 74 12 7.59 / 7.83, 16 8.15 / 7.77;
    // 80 10 8.04 / 7.81, 12 7.78 / 7.85; 88 12 8.39 / 7.87; 104 4 8.08 / 8.20, 8 8.88 /
    // 8.19; 112 2 8.13 / 8.42, 4 8.61 / 8.42; 136 1 8.81 / 8.83, 2 9.03 / 8.82
    const uint32_t h = a.num_heads;
    const uint32_t least = a.head_dim == 64 ? (h >= 8 ? 64u : 66u)
                           : h >= 20        ? 64u
                           : h >= 16        ? 74u
                           : h >= 10        ? 84u
                           : h >= 8         ? 104u
                           : h >= 4         ? 112u
                                            : 136u;
    if (a.seq_len < least) return 0;
    // Four parts until the workgroups are two rounds of what the CUs hold (one
    // workgroup of 128-dim heads per CU, two of 64-dim heads), then two parts
    // and shared copies where pairs of heads share a KV head: 16/8 heads of 128
    // at 1200 tokens (304 workgroups) 21 against 28 us, 4096 (1024) 116 / 110;
    // 16/4 of 64 at 4096 (1024) 64 / 72, 8192 (2048) 234 / 222.
    return wgs <= (a.head_dim == 64 ? 4u : 2u) * cus || a.group % 2 != 0 ? 4 : 2;
}

hipError_t launch_prefill_rows64(const PrefillArgs& a0, int parts, bool mfma,
                                 hipStream_t stream) {
    PrefillArgs a = a0;
    a.q_tiles = (a.seq_len + kRows - 1) / kRows;
    const uint64_t blocks = (uint64_t)a.q_tiles * a.num_heads * (uint32_t)parts / 4u;
    if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
    const dim3 grid((uint32_t)blocks), block(256);
    const auto launch = [&](auto d_tag, auto lo_tag) {
        constexpr int D = decltype(d_tag)::value;
        constexpr bool LO = decltype(lo_tag)::value;
        if (parts == 2)
            hipLaunchKernelGGL((prefill_rows64<D, 2, LO>), grid, block, 0, stream, a);
        else
            hipLaunchKernelGGL((prefill_rows64<D, 4, LO>), grid, block, 0, stream, a);
    };
    using d64 = std::integral_constant<int, 64>;
    using d128 = std::integral_constant<int, 128>;
    if (parts != 2 && parts != 4) return hipErrorInvalidValue;
    if (a.head_dim == 64) launch(d64{}, std::true_type{});
    else if (!mfma) launch(d128{}, std::true_type{});
    else if (parts == 4) hipLaunchKernelGGL((prefill_rows64<128, 4, false>), grid, block, 0, stream, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace attn
