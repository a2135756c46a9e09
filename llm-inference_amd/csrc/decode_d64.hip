// Split decode attention for 64-dim heads on gfx950: single query token,
// grouped-query heads, fp16 KV cache, fp32 scores, weights and partial states.
//
// Same semantics as flash_decode.hip (causal_attention.hip.cpp:493-838; all
// kv_len keys visible).  These heads ran attention_generic, one workgroup per
// query head and a serial chain of 256-key tiles: 215 us at 3000 keys and 16/4
// heads, the whole cache read by 16 CUs.  Here the keys of each KV head are cut
// into chunks of at least 64, a workgroup of 4 waves per chunk and KV head (up
// to 8 of its query heads: larger groups take further workgroups), then a merge
// kernel folds the partial states.
//  * Bound by latency up to ~16 K keys (two dependent kernels, one or two
//    rounds of loads per wave), by the K/V bytes above.
//  * Eight lanes hold a key (16 bytes of K and of V each), a wave 32 keys per
//    round with all loads issued first; a score is 8 products per lane and three
//    DPP adds.  Each eight lanes keep a running softmax of their own; the eight
//    of a wave meet over lane exchanges, the four waves over LDS.
//  * Everything past the fp16 inputs is fp32, as in attention_generic: vector
//    ALU products (the matrix cores would take fp16 weights), fp32 states in the
//    caller's workspace.  The arithmetic (4 query heads: ~130 instructions per
//    wave and 8 keys) is a small part of the time.
// Measured (one MI355X): a decode token over 12 layers at 3000 keys, 16/4
// heads, projections included, 2849 -> 215 us.
#include "attn_internal.hpp"

#include <algorithm>

namespace attn {

namespace {

constexpr uint32_t kD = 64;
constexpr int kU = 4;               // keys per eight lanes and round
constexpr uint32_t kMaxStates = 256;
constexpr uint32_t kMinChunk = 64;  // keys
constexpr float kNoMax = -1.0e30f;  // finite: masked scores (-inf) get weight 0
constexpr int kDppHalfMirror = 0x141;  // lane i <-> 7 - i within eight lanes

// the sum of eight lanes' x in each of them
__device__ __forceinline__ float sum8(float x) {
    x += dpp_f<kDppXor1>(x);
    x += dpp_f<kDppXor2>(x);
    return x + dpp_f<kDppHalfMirror>(x);
}
// max / sum over the eight lane octets of a wave (equal within an octet for max)
__device__ __forceinline__ float max_octets(float x) {
    x = fmaxf(x, dpp_f<kDppRor8>(x));
    return max_xor<32>(max_xor<16>(x));
}
__device__ __forceinline__ float sum_octets(float x) {
    x += dpp_f<kDppRor8>(x);
    return add_xor<32>(add_xor<16>(x));
}

// GP: query heads per workgroup (1, 2, 4 or 8; lanes of heads past the group
// repeat its last head and are not stored)
template <int GP>
__global__ __launch_bounds__(256) void decode_d64_split(DecodeD64Args a) {
    __shared__ float s_acc[4][GP][kD];
    __shared__ float s_m[4][GP], s_l[4][GP];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t oct = lane >> 3, c8 = 8u * (lane & 7u);
    const uint32_t parts = (a.group + GP - 1u) / GP;  // workgroups per KV head
    const uint32_t g = blockIdx.x / parts;
    const uint32_t h0 = (blockIdx.x - g * parts) * GP;        // first head within the group
    const uint32_t heads = min((uint32_t)GP, a.group - h0);
    const uint32_t c = blockIdx.y;
    const uint32_t row_bytes = (uint32_t)(a.kv_stride * 2);
    // this wave's keys: a quarter of the chunk
    const uint32_t share = a.chunk / 4u;
    const uint32_t k0 = c * a.chunk + wave * share;
    const uint32_t nk = a.kv_len > k0 ? min(share, a.kv_len - k0) : 0u;
    const uint32_t span = nk ? (nk - 1u) * row_bytes + kD * 2u : 0u;
    // rows past the wave's share read as zero
    const BufRsrc rk = make_rsrc(a.k + (uint64_t)k0 * a.kv_stride + (uint64_t)g * kD, span);
    const BufRsrc rv = make_rsrc(a.v + (uint64_t)k0 * a.kv_stride + (uint64_t)g * kD, span);

    f16x8 q[GP];
#pragma unroll
    for (int h = 0; h < GP; ++h)
        q[h] = ld16(a.q + (uint64_t)(g * a.group + h0 + min((uint32_t)h, heads - 1u)) * kD + c8);
    float m[GP], l[GP], acc[GP][8];
#pragma unroll
    for (int h = 0; h < GP; ++h) {
        m[h] = kNoMax;
        l[h] = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[h][e] = 0.f;
    }
    for (uint32_t b = 0; b < nk; b += 8u * kU) {
        f16x8 k[kU], v[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u)
            k[u] = buf_ld16_nt(rk, (b + 8u * (uint32_t)u + oct) * row_bytes + 2u * c8);
#pragma unroll
        for (int u = 0; u < kU; ++u)
            v[u] = buf_ld16_nt(rv, (b + 8u * (uint32_t)u + oct) * row_bytes + 2u * c8);
#pragma unroll
        for (int h = 0; h < GP; ++h) {
            float s[kU], mx = m[h];
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                float d = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) d = __builtin_fmaf((float)q[h][e], (float)k[u][e], d);
                d = sum8(d) * a.scale_log2;
                s[u] = b + 8u * (uint32_t)u + oct < nk ? d : -INFINITY;
                mx = fmaxf(mx, s[u]);
            }
            const float alpha = fast_exp2(m[h] - mx);
            m[h] = mx;
            l[h] *= alpha;
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[h][e] *= alpha;
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const float p = fast_exp2(s[u] - mx);
                l[h] += p;
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    acc[h][e] = __builtin_fmaf(p, (float)v[u][e], acc[h][e]);
            }
        }
    }
    // the octets of the wave, then the waves of the workgroup
#pragma unroll
    for (int h = 0; h < GP; ++h) {
        const float M = max_octets(m[h]);
        const float w = fast_exp2(m[h] - M);  // an octet without keys: 0, or l = 0
        const float lw = sum_octets(l[h] * w);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float x = sum_octets(acc[h][e] * w);
            if (oct == 0) s_acc[wave][h][c8 + e] = x;
        }
        if (lane == 0) {
            s_m[wave][h] = M;
            s_l[wave][h] = lw;
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < heads * kD; i += 256u) {
        const uint32_t h = i / kD, d = i - h * kD;
        float M = s_m[0][h];
#pragma unroll
        for (int w = 1; w < 4; ++w) M = fmaxf(M, s_m[w][h]);
        float x = 0.f, lw = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float wt = fast_exp2(s_m[w][h] - M);
            x += wt * s_acc[w][h][d];
            lw += wt * s_l[w][h];
        }
        const uint64_t st = (uint64_t)(g * a.group + h0 + h) * a.nsplit + c;
        a.part_out[st * kD + d] = x;
        if (d == 0) {
            a.part_max[st] = M;
            a.part_sum[st] = lw;
        }
    }
}

// One workgroup per query head: thread t weighs state t, then wave w sums the
// states w, w + 4, ... with a dim per lane.
__global__ __launch_bounds__(256) void decode_d64_merge(DecodeD64Args a) {
    __shared__ float s_w[kMaxStates];
    __shared__ float s_x[4][kD], s_red[4], s_den[4];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, t = threadIdx.x;
    const uint32_t S = a.nsplit;  // <= kMaxStates
    const uint64_t s0 = (uint64_t)blockIdx.x * S;
    const float* const po = a.part_out + s0 * kD + lane;
    // the first states of each wave, alongside the maxima
    constexpr int kFirst = 8;
    float x0[kFirst];
#pragma unroll
    for (int i = 0; i < kFirst; ++i) {
        const uint32_t c = wave + 4u * (uint32_t)i;
        x0[i] = c < S ? po[(uint64_t)c * kD] : 0.f;
    }
    const float m = t < S ? a.part_max[s0 + t] : -INFINITY;
    const float l = t < S ? a.part_sum[s0 + t] : 0.f;
    const float wm = wave_max(m);
    if (lane == 0) s_red[wave] = wm;
    __syncthreads();
    const float M = fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
    const float w = fast_exp2(m - M);
    s_w[t] = w;  // past S: 0
    const float den = wave_sum(w * l);
    if (lane == 0) s_den[wave] = den;
    __syncthreads();
    float x = 0.f;
#pragma unroll
    for (int i = 0; i < kFirst; ++i) x = __builtin_fmaf(s_w[wave + 4u * (uint32_t)i], x0[i], x);
#pragma unroll 4
    for (uint32_t c = wave + 4u * kFirst; c < S; c += 4u)
        x = __builtin_fmaf(s_w[c], po[(uint64_t)c * kD], x);
    s_x[wave][lane] = x;
    __syncthreads();
    if (t < kD) {
        const float num = (s_x[0][t] + s_x[1][t]) + (s_x[2][t] + s_x[3][t]);
        const float d = (s_den[0] + s_den[1]) + (s_den[2] + s_den[3]);
        a.out[(uint64_t)blockIdx.x * kD + t] = (f16)(num / d);
    }
}

uint32_t heads_per_workgroup(uint32_t group) {
    return group >= 8 ? 8u : group > 2 ? 4u : group;
}

const void* split_symbol(uint32_t group) {
    switch (heads_per_workgroup(group)) {
        case 1: return reinterpret_cast<const void*>(&decode_d64_split<1>);
        case 2: return reinterpret_cast<const void*>(&decode_d64_split<2>);
        case 4: return reinterpret_cast<const void*>(&decode_d64_split<4>);
        default: return reinterpret_cast<const void*>(&decode_d64_split<8>);
    }
}

}  // namespace

// The plan for a.kv_len: a workgroup per CU, chunks of at least kMinChunk keys,
// no more states than the workspace of the call holds (a.capacity per head).
bool plan_decode_d64(DecodeD64Args& a, int device) {
    if (a.group == 0 || a.kv_len == 0 || a.kv_len > 0x7fffffffu) return false;
    if (a.kv_stride % 8 != 0 || a.kv_stride > 0x800000u) return false;
    if (!aligned16(a.q) || !aligned16(a.k) || !aligned16(a.v)) return false;
    if (!a.part_out || !a.part_max || !a.part_sum) return false;
    const uint32_t hpw = heads_per_workgroup(a.group);
    const uint64_t groups = (uint64_t)a.num_kv_heads * ((a.group + hpw - 1) / hpw);
    const uint64_t cus = (uint64_t)std::max(1, device_cu_count(device));
    const uint64_t want = std::max<uint64_t>(1, cus / groups);
    const uint64_t n = std::min<uint64_t>(
        {want, kMaxStates, a.capacity, (a.kv_len + (uint64_t)kMinChunk - 1) / kMinChunk});
    if (n == 0 || groups > 0x7fffffffu) return false;
    // waves take a quarter each, in whole rounds of eight keys
    const uint64_t chunk = ((a.kv_len + n - 1) / n + 31u) / 32u * 32u;
    // a wave's rows fit one 32-bit buffer range
    if (chunk / 4u * a.kv_stride * 2u > 0x7fffffffull) return false;
    a.chunk = (uint32_t)chunk;
    a.nsplit = (uint32_t)((a.kv_len + chunk - 1) / chunk);
    return true;
}

// Whether two kernels take less than attention_generic's one.  That takes 3 us and
// 0.035 per key; these 4.7-5.2 us up to 256 keys with 1 or 2 heads per workgroup,
// 6.6-6.8 with 4, 9.4-9.6 with 8 (a merge that waits for the split, and the split's
// code, which grows with the heads).  us at 16/4 heads, two kernels / one: 32 keys
// 6.7 / 4.1, 100 6.65 / 6.57, 128 6.8 / 7.6; 8/8: 32 4.9 / 4.1, 64 4.9 / 5.3; 16/2:
// 100 9.5 / 6.5, 200 9.5 / 10.0.
bool decode_d64_pays(uint32_t kv_len, uint32_t group) {
    const uint32_t hpw = heads_per_workgroup(group);
    return kv_len >= (hpw <= 2 ? 64u : hpw == 4 ? 104u : 192u);
}

const void* decode_d64_split_symbol(const DecodeD64Args& a) { return split_symbol(a.group); }
const void* decode_d64_merge_symbol() { return reinterpret_cast<const void*>(&decode_d64_merge); }
bool is_decode_d64_split(const void* fn) {
    return fn == split_symbol(1) || fn == split_symbol(2) || fn == split_symbol(4) ||
           fn == split_symbol(8);
}
dim3 decode_d64_grid(const DecodeD64Args& a) {
    const uint32_t hpw = heads_per_workgroup(a.group);
    return dim3(a.num_kv_heads * ((a.group + hpw - 1) / hpw), a.nsplit);
}

hipError_t launch_decode_d64_split(const DecodeD64Args& a, hipStream_t stream) {
    void* args[1] = {const_cast<DecodeD64Args*>(&a)};
    return hipLaunchKernel(decode_d64_split_symbol(a), decode_d64_grid(a), dim3(256), args, 0,
                           stream);
}

hipError_t launch_decode_d64_merge(const DecodeD64Args& a, hipStream_t stream) {
    void* args[1] = {const_cast<DecodeD64Args*>(&a)};
    return hipLaunchKernel(decode_d64_merge_symbol(), dim3(a.num_heads), dim3(256), args, 0,
                           stream);
}

}  // namespace attn
