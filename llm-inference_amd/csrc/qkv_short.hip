// QKV projection of short prompts (up to 256 tokens, K >= 1024) for gfx950 on
// fp16 MFMA, optionally with the RoPE + KV-cache append folded into its
// epilogue.  Semantics, layouts and the fused epilogue's bytes are those of
// qkv_prefill.hip.
//
// What bounds it: the copies into LDS.  A CU takes 8-10 ns per KiB when the
// lines are in its XCD's L2 and 16-18 ns when they are not (whatever the depth
// of the copies: three and six stages in flight run alike), so a workgroup's
// time is its tile's bytes, (BM + BN) rows of K values, and the 64 x 128 tiles
// of qkv_prefill.hip give a short prompt 24-96 workgroups of 192 rows each.
// Here:
//  * tiles from 16 x 16 to 64 x 64 (tokens x features), chosen so that the
//    rounds of workgroups times the rows of a tile are least
//    (qkv_short_tile): 128 instead of 192 rows per workgroup at 254 tokens, 48
//    at 24.  A tile's features are BN/2 columns of a head and the same columns
//    + D / 2, so both halves of every rotation pair are in the workgroup (not
//    fused: as for D = 128).
//  * the waves split K: wave w takes the 64-value units w, w + W, ... with a
//    ring of copies (buffer_load ... lds) of its own, computes the whole tile
//    for them, and the W fp32 tiles are added through LDS at the end, in wave
//    order (so the last bit of a token's projection depends on W, that is on the
//    tile and with it on how many tokens share the call; one order for 4 and 8
//    waves costs the 64 x 64 tile 3 %).  No barrier stands between the first copy and the sum, so the waves
//    do not wait for each other's copies.
//  * LDS rows are the 128 bytes of a unit (whole cache lines: with 64-byte
//    units the two halves of a line are fetched twice, 15.3 us at 254 tokens),
//    the 16-byte chunk c of row r at position c ^ ((r >> 1) & 7): the operand
//    reads (16 rows x 16 B per pass) hit 16 distinct bank groups; the copies'
//    source lanes produce that order.
//    Rows past M or N and units past K read as zero (buffer range check).
// Measured (one MI355X, us, K = 2048, N = 3072, weights streamed from HBM; the
// 64 x 128 tiles before): 16 tokens 16.3 -> 6.6, 24 16.5 -> 7.1, 64 17.5 -> 8.4,
// 128 17.0 -> 10.3, 192 17.3 -> 12.2, 254 17.0 -> 12.1.  Level or worse: the
// non-temporal hint on W (7.1 -> 6.9 at 24 from HBM, 5.8 -> 6.8 when the weights
// are in the memory-side cache), starting the workgroups that share rows at
// different units (254 tokens: 12.1 -> 11.0 and 9.8 -> 10.8).
#include "attn_internal.hpp"

#include <type_traits>

namespace attn {

namespace {

// BM x BN tile, W waves, S units of each wave in its ring; P pairs of features
// per thread in the epilogue
template <int BM, int BN, int W, int S, int P, bool FUSED>
__global__ __launch_bounds__(64 * W, 1) void qkv_gemm_short(QkvGemmArgs a) {
    constexpr int kA = BM / 16, kB = BN / 16;
    constexpr int kDma = (BM + BN) / 8;              // 1 KiB copies per unit
    constexpr uint32_t kUnit = 1024u * kDma;                   // bytes of a unit's rows
    constexpr uint32_t kHalf = BN / 2;
    constexpr int kPad = BN + 4;  // floats per row of a partial tile (conflict-free stores)
    static_assert((S - 1) * kDma < 64, "vmcnt range");
    constexpr uint32_t kRing = S * kUnit;
    constexpr uint32_t kLds = W * kRing > W * BM * kPad * 4u ? W * kRing : W * BM * kPad * 4u;
    static_assert(kLds <= 160 * 1024, "LDS");
    __shared__ __attribute__((aligned(16))) char lds[kLds];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // Workgroups go round-robin over the 8 XCDs: with the feature tiles a
    // multiple of 8, every token tile of a feature tile is on one XCD (W is
    // read from memory once)
    uint32_t mt0, nt0;
    if ((a.n_tiles & 7u) == 0) {
        const uint32_t per = a.n_tiles >> 3, j = blockIdx.x >> 3;
        mt0 = j / per;
        nt0 = (blockIdx.x & 7u) + 8u * (j - mt0 * per);
    } else {
        mt0 = blockIdx.x / a.n_tiles;
        nt0 = blockIdx.x - mt0 * a.n_tiles;
    }
    mt0 = __builtin_amdgcn_readfirstlane(mt0);
    nt0 = __builtin_amdgcn_readfirstlane(nt0);
    const uint32_t pair = FUSED ? a.head_dim >> 1 : 64u;  // distance of a pair's columns
    const uint32_t per_head = pair / kHalf;
    const uint32_t head = nt0 / per_head, c0 = (nt0 - head * per_head) * kHalf;
    const uint32_t m0 = mt0 * BM, n0 = head * 2u * pair;
    const uint32_t K = a.K, row_bytes = K * 2u;
    const char* xb = reinterpret_cast<const char*>(a.x + (uint64_t)m0 * K);
    const char* wb = reinterpret_cast<const char*>(a.w + (uint64_t)n0 * K);
    const uint32_t x_bytes = min(a.M - m0, (uint32_t)BM) * row_bytes;
    const uint32_t w_bytes = min(a.N - n0, 2u * pair) * row_bytes;

    // copy t: tile rows 8 t .. 8 t + 7 (X rows first, then W rows), lane L
    // writes position L % 8 of row L / 8
    uint32_t voff[kDma];
    const uint32_t lr = (uint32_t)lane >> 3;
#pragma unroll
    for (int t = 0; t < kDma; ++t) {
        uint32_t row;
        if (t < BM / 8) {
            row = 8u * t + lr;
        } else {
            const uint32_t f = 8u * (t - BM / 8) + lr;
            row = c0 + (f < kHalf ? f : pair + f - kHalf);
        }
        voff[t] = row * row_bytes +
                  16u * (((uint32_t)lane & 7u) ^ ((4u * (t & 1) + (lr >> 1)) & 7u));
    }
    // this thread's epilogue item: P feature pairs of one token (a BM x BN tile
    // has at most one item per thread); its table entries are on their way
    // before the copies
    static_assert(BM * kHalf / P <= 64 * W, "one epilogue item per thread");
    typedef f16 hv __attribute__((ext_vector_type(P)));
    const uint32_t Hq = a.num_heads, Hkv = a.num_kv_heads;
    const bool is_q = head < Hq, is_k = !is_q && head < Hq + Hkv;
    const bool rot = FUSED && a.apply != 0 && (is_q || is_k);
    const uint32_t erow = (uint32_t)tid / (kHalf / P), ec = ((uint32_t)tid % (kHalf / P)) * P;
    const uint32_t m = m0 + erow, col = c0 + ec;  // and col + pair
    const bool mine = erow < (uint32_t)BM && m < a.M;
    const uint64_t pos = (uint64_t)a.start_pos + m;
    hv cs = {}, sn = {};
    if (rot && mine) {
        cs = *reinterpret_cast<const hv*>(a.cos_t + pos * pair + col);
        sn = *reinterpret_cast<const hv*>(a.sin_t + pos * pair + col);
    }

    const uint32_t units = K / 64u;
    const uint32_t ring = lds_addr(lds) + wave * kRing;
    auto issue = [&](uint32_t i, uint32_t slot) __attribute__((always_inline)) {
        const uint32_t u = i * W + wave;
        const uint32_t off = u < units ? 128u * u : 0u;
        const u32x4 rx = rsrc_words(xb + off, u < units ? x_bytes - off : 0u);
        const u32x4 rw = rsrc_words(wb + off, u < units ? w_bytes - off : 0u);
        const uint32_t dst = ring + slot * kUnit;
#pragma unroll
        for (int t = 0; t < kDma; ++t) dma16(t < BM / 8 ? rx : rw, dst + 1024u * t, voff[t]);
    };

    const uint32_t rows = (uint32_t)lane & 15u, q = (uint32_t)lane >> 4;
    // operand chunks 4 ks + q of rows 16 i + lane % 16
    const uint32_t op0 = rows * 128u + 16u * (q ^ (rows >> 1)) + wave * kRing;
    const uint32_t op1 = rows * 128u + 16u * ((4u + q) ^ (rows >> 1)) + wave * kRing;
    f16x8 av[2][2][kA], bv[2][2][kB];
    f32x4 acc[kA][kB];
#pragma unroll
    for (int i = 0; i < kA; ++i)
#pragma unroll
        for (int j = 0; j < kB; ++j) acc[i][j] = f32x4{};
    auto fetch = [&](uint32_t slot, auto buf_tag) __attribute__((always_inline)) {
        constexpr int buf = decltype(buf_tag)::value;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const char* p = lds + (ks ? op1 : op0) + slot * kUnit;
#pragma unroll
            for (int i = 0; i < kA; ++i)
                av[buf][ks][i] = *reinterpret_cast<const f16x8*>(p + 2048 * i);
#pragma unroll
            for (int j = 0; j < kB; ++j)
                bv[buf][ks][j] = *reinterpret_cast<const f16x8*>(p + 2048 * (kA + j));
        }
    };
    // unit i: its operands are in registers (or on their way), so its slot takes
    // unit i + S, and unit i + 1's operands are read under its MFMAs
    uint32_t slot = 0;
    auto step = [&](uint32_t i, auto buf_tag) __attribute__((always_inline)) {
        constexpr int buf = decltype(buf_tag)::value;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue(i + S, slot);
        slot = slot + 1 == S ? 0 : slot + 1;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((S - 1) * kDma));
        asm volatile("" ::: "memory");
        fetch(slot, std::integral_constant<int, buf ^ 1>{});
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i4 = 0; i4 < kA; ++i4)
#pragma unroll
                for (int j = 0; j < kB; ++j)
                    acc[i4][j] = mfma16(av[buf][ks][i4], bv[buf][ks][j], acc[i4][j]);
    };
    const uint32_t n = ((units + W - 1) / W + 1u) & ~1u;  // even: units past K are zero
#pragma unroll
    for (uint32_t i = 0; i < S; ++i) issue(i, i);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(vmcnt_imm((S - 1) * kDma));
    asm volatile("" ::: "memory");
    fetch(0, std::integral_constant<int, 0>{});
    for (uint32_t i = 0; i < n; i += 2) {
        step(i, std::integral_constant<int, 0>{});
        step(i + 1, std::integral_constant<int, 1>{});
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __syncthreads();  // every wave is done with its ring

    // acc[i][j][e] is token 16 i + 4 q + e, tile feature 16 j + lane % 16
    float* part = reinterpret_cast<float*>(lds) + wave * (BM * kPad);
#pragma unroll
    for (int i = 0; i < kA; ++i)
#pragma unroll
        for (int j = 0; j < kB; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                part[(16u * i + 4u * q + e) * kPad + 16u * j + rows] = acc[i][j][e];
    __syncthreads();
    if (!mine) return;
    const float* sum = reinterpret_cast<const float*>(lds) + erow * kPad + ec;
    float l[P], h[P];
#pragma unroll
    for (int e = 0; e < P; ++e) l[e] = h[e] = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w)
#pragma unroll
        for (int e = 0; e < P; ++e) {
            l[e] += sum[w * BM * kPad + e];
            h[e] += sum[w * BM * kPad + kHalf + e];
        }
    hv lo, hi;
#pragma unroll
    for (int e = 0; e < P; ++e) {
        lo[e] = (f16)l[e];
        hi[e] = (f16)h[e];
    }
    f16* yr = a.y + (uint64_t)m * a.N + n0 + col;
    if (!FUSED) {
        if (a.vec_out) {  // N % 8 == 0: P features are wholly inside or outside
            if (n0 + col < a.N) *reinterpret_cast<hv*>(yr) = lo;
            if (n0 + 64u + col < a.N) *reinterpret_cast<hv*>(yr + 64) = hi;
        } else {
#pragma unroll
            for (int e = 0; e < P; ++e) {
                if (n0 + col + e < a.N) yr[e] = lo[e];
                if (n0 + 64u + col + e < a.N) yr[64 + e] = hi[e];
            }
        }
        return;
    }
    hv r0 = lo, r1 = hi;
    if (rot) {
#pragma unroll
        for (int e = 0; e < P; ++e) {
            f16 o0, o1;
            rope_pair(lo[e], hi[e], cs[e], sn[e], o0, o1);
            r0[e] = o0;
            r1[e] = o1;
        }
    }
    if (is_q) {
        *reinterpret_cast<hv*>(yr) = r0;
        *reinterpret_cast<hv*>(yr + pair) = r1;
    } else {
        *reinterpret_cast<hv*>(yr) = lo;
        *reinterpret_cast<hv*>(yr + pair) = hi;
        f16* cr = (is_k ? a.kc + (uint64_t)(head - Hq) * a.head_dim
                        : a.vc + (uint64_t)(head - Hq - Hkv) * a.head_dim) +
                  pos * ((uint64_t)Hkv * a.head_dim) + col;
        *reinterpret_cast<hv*>(cr) = r0;
        *reinterpret_cast<hv*>(cr + pair) = r1;
    }
}

template <int BM, int BN, int W, int S, int P>
hipError_t launch(const QkvGemmArgs& a, bool fused, hipStream_t stream) {
    QkvGemmArgs b = a;
    b.m_tiles = (a.M + BM - 1u) / BM;
    const uint32_t span = fused ? a.head_dim : 128u;  // features whose tiles pair up
    b.n_tiles = (a.N + span - 1u) / span * (span / BN);
    b.vec_out = (a.N % 8u == 0 && ((uintptr_t)a.y & 15u) == 0) ? 1u : 0u;
    const uint64_t blocks = (uint64_t)b.m_tiles * b.n_tiles;
    if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
    if (fused)
        hipLaunchKernelGGL((qkv_gemm_short<BM, BN, W, S, P, true>), dim3((uint32_t)blocks),
                           dim3(64 * W), 0, stream, b);
    else
        hipLaunchKernelGGL((qkv_gemm_short<BM, BN, W, S, P, false>), dim3((uint32_t)blocks),
                           dim3(64 * W), 0, stream, b);
    return hipGetLastError();
}

struct Tile {
    uint32_t bm, bn;
};
constexpr Tile kTiles[] = {{64, 64}, {64, 32}, {32, 32}, {32, 16}, {16, 16}};

}  // namespace

// The tile with the least rounds of workgroups times rows of a tile, which is
// what the copies of a CU take (-1: the tiles of qkv_prefill.hip), and their cost
// on the scale of qkv_prefill.hip's tiles: 8.1 us for a round of 128 rows at K =
// 2048.  At 64 tokens 32 x 32 (192 workgroups of 64 rows) takes 8.4 us, 64 x 32 (96
// of 96 rows) 9.9.  Up to 256 tokens: beyond, the tiles of qkv_prefill.hip alone
// give every length one order of the k-values.  Below K = 1024 a wave has two units or less, nothing for a
// ring.
int qkv_short_tile(const QkvGemmArgs& a, int device, uint64_t& cost) {
    if (a.M > 256u || a.K < 1024u || get_option(kOptQkvGemmTokensPerWave) ||
        get_option(kOptQkvGemmWide) == 2)
        return -1;
    const uint64_t cus = (uint64_t)device_cu_count(device);
    int best = -1;
    uint64_t least = 0;
    for (int i = 0; i < (int)(sizeof(kTiles) / sizeof(kTiles[0])); ++i) {
        const uint64_t wgs = (uint64_t)((a.M + kTiles[i].bm - 1) / kTiles[i].bm) *
                             ((a.N + 127u) / 128u * (128u / kTiles[i].bn));
        const uint64_t rows = (wgs + cus - 1) / cus * (kTiles[i].bm + kTiles[i].bn);
        if (best < 0 || rows < least) {
            best = i;
            least = rows;
        }
    }
    cost = least * 81u / 128u;
    return best;
}

hipError_t launch_qkv_gemm_short(const QkvGemmArgs& a, int tile, bool fused, hipStream_t stream) {
    switch (tile) {
        case 0: return launch<64, 64, 4, 2, 8>(a, fused, stream);
        case 1: return launch<64, 32, 4, 3, 4>(a, fused, stream);
        case 2: return launch<32, 32, 8, 2, 4>(a, fused, stream);
        case 3: return launch<32, 16, 8, 3, 4>(a, fused, stream);
        default: return launch<16, 16, 8, 4, 4>(a, fused, stream);
    }
}

}  // namespace attn
