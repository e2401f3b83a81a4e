// dq_gemm_direct.hip - the prefill GEMM for few tokens (up to 128):
// Y[t][r] = sum_k W[r][k] X[t][k], the semantics and operands of dq_gemm.hip
// (fp16(q_x * dx * s) against fp16(a * q_w), the Q4_K min term as one more
// MFMA slice per super-block, fp32 accumulation, 1/s on the output).
//
// With few tokens the product is bound by reading the weights once, and the
// 128-token tiles of dq_gemm.hip leave most of the GPU idle (64 workgroups on
// 256 CUs for 4096 rows). Here a workgroup owns 16 RT weight rows for 16 MT
// tokens over the whole K range: its waves split K by super-blocks and add
// their partials through LDS in wave order, so there are no partial sums in
// memory, and the order of a token's sum does not depend on how many tokens
// the call has. Nothing is staged and the waves meet only once:
//  * weights go straight from memory to registers. Lane (n, g) = (l % 16,
//    l / 16) of v_mfma_f32_16x16x32_f16 holds item g (64 weights) of row n's
//    super-block, so each load reads 16 rows x 64 contiguous bytes, and the
//    MFMA's K slice c (0..7) takes the c-th 8 weights of each of the four
//    items; the sum over K does not depend on how K is dealt to the slices;
//  * the activations are written by the quantizer in the order of these
//    slices, [super-block][slice][item][token][8 halfs] (tokens padded to
//    16), so a fragment load is 4 runs of 256 bytes. Every workgroup reads
//    them from L2.
// A super-block's weights are loaded one super-block ahead, its activation
// fragments are replaced by the next ones as each slice is consumed, in the
// order they will be waited for, so no wait is for a younger load.
#include "dq_common.h"
#include "dq_f16.h"
#include "dq_gemm_direct.h"

namespace {

typedef float f4v __attribute__((ext_vector_type(4)));

template <int FMT>
constexpr int planes() { return FMT == DQ_FMT_Q8_0 ? 4 : FMT == DQ_FMT_Q6_K ? 3 : 2; }

// One matrix of a launch. Row groups of all of them are concatenated into
// grid x; wg_end is the first row group past this matrix.
struct DirectJob {
    const uint8_t* w;    // packed rows, or tiles
    size_t p_stride;     // between quant sub-planes
    size_t x_off, d_off;
    uint32_t q_sb, x_sb, d_sb;     // bytes per super-block: quants, Q4_K header / Q6_K scales, fp16 scales
    uint32_t q_row, x_row, d_row;  // packed rows: row strides
    int fmt, tiled, n_stages, N, wg_end;
    const _Float16* A;
    const _Float16* minp;
    const float* inv;
    float* y;
};
struct DirectArgs {
    DirectJob job[DQ_GEMM_DIRECT_JOBS];
    int n, M, mp, mb, nsb;
};

// This lane's byte offsets of super-block 0 of row r, item g.
struct LaneOff {
    uint32_t q, x, d;
};
// Row r of the tile copy: slice r / 64 holds n_stages runs (see
// gemm_tiles_pack_kernel in dq_gemm.hip); a super-block is one run of 4 items
// (Q4_K, Q4_0) or two runs of 2.
template <int FMT>
__device__ __forceinline__ LaneOff lane_off(const DirectJob& a, int r, int g) {
    LaneOff o;
    if (a.tiled) {
        constexpr bool TWO = FMT == DQ_FMT_Q6_K || FMT == DQ_FMT_Q8_0;
        constexpr int SB = TWO ? 2 : 4;
        constexpr uint32_t PL = 64 * SB * 16;
        constexpr uint32_t AUX = planes<FMT>() * PL;
        constexpr uint32_t SLICE = AUX + (FMT == DQ_FMT_Q4_K ? 1024 : FMT == DQ_FMT_Q6_K ? 768 : SB * 256);
        const int nl = r & 63, it = TWO ? (g & 1) : g;
        const int sw = TWO ? ((nl >> 2) ^ (nl >> 3)) & 1 : (nl >> 2) & 3;
        const uint32_t b = (uint32_t)(r >> 6) * (uint32_t)a.n_stages * SLICE + (TWO ? (uint32_t)(g >> 1) * SLICE : 0u);
        o.q = b + nl * (SB * 16) + 16 * (it ^ sw);
        o.x = b + AUX + (FMT == DQ_FMT_Q4_K ? nl * 16 : it * 256 + nl * 4);
        o.d = b + AUX + (FMT == DQ_FMT_Q6_K ? 512 + nl * 4 : it * 256 + nl * 4);
    } else {
        o.q = (uint32_t)r * a.q_row + 16 * g;
        o.x = (uint32_t)r * a.x_row + (FMT == DQ_FMT_Q6_K ? 4 * g : 0);
        o.d = (uint32_t)r * a.d_row + (FMT == DQ_FMT_Q6_K ? 0 : 4 * g);
    }
    return o;
}

// A lane's item of one super-block: the 16-byte pieces of its sub-planes and
// its scales (Q4_K: the 16-byte header; Q6_K: 4 int8 scales in x and d;
// Q8_0, Q4_0: the two fp16 block scales in d).
template <int FMT>
struct Item {
    dq_u32x4 p[planes<FMT>()];
    dq_u32x4 hd;
    uint32_t x, d;
};
template <int FMT>
__device__ __forceinline__ void load_item(const DirectJob& a, const LaneOff& o, int sb, Item<FMT>& it) {
    const uint8_t* q = a.w + (size_t)sb * a.q_sb;
#pragma unroll
    for (int k = 0; k < planes<FMT>(); ++k) it.p[k] = dq_ld16(q + k * a.p_stride + o.q);
    if constexpr (FMT == DQ_FMT_Q4_K) it.hd = dq_ld16(a.w + a.x_off + (size_t)sb * a.x_sb + o.x);
    if constexpr (FMT == DQ_FMT_Q6_K)
        it.x = *reinterpret_cast<const uint32_t*>(a.w + a.x_off + (size_t)sb * a.x_sb + o.x);
    if constexpr (FMT == DQ_FMT_Q6_K)
        it.d = *reinterpret_cast<const uint16_t*>(a.w + a.d_off + (size_t)sb * a.d_sb + o.d);
    if constexpr (FMT == DQ_FMT_Q8_0 || FMT == DQ_FMT_Q4_0)
        it.d = *reinterpret_cast<const uint32_t*>(a.w + a.d_off + (size_t)sb * a.d_sb + o.d);
}

// The item's scales as fp16 pairs, rounded as b_scales_j of dq_gemm.hip
// rounds them: Q4_K a of sub-blocks 2g, 2g + 1 and -64 a of each; Q6_K a of
// its four 16-blocks; Q8_0, Q4_0 d of its two blocks.
struct Scales {
    h2 s[4];
};
template <int FMT>
__device__ __forceinline__ Scales item_scales(const Item<FMT>& it, int g) {
    Scales S;
    if constexpr (FMT == DQ_FMT_Q4_K) {
        uint32_t lo, hi;
        q4k_sc_bytes(it.hd, lo, hi);
        const uint32_t w = ((g & 2) ? hi : lo) >> (16 * (g & 1));
        const float d = dq_h2f((uint16_t)(it.hd.x & 0xFFFF));
        const _Float16 a0 = (_Float16)(d * (float)(w & 0xFF));
        const _Float16 a1 = (_Float16)(d * (float)((w >> 8) & 0xFF));
        S.s[0] = h2{a0, a0};
        S.s[1] = h2{a1, a1};
        const h2 m64 = {(_Float16)-64.0f, (_Float16)-64.0f};
        S.s[2] = S.s[0] * m64;  // exact while |a| < 1024
        S.s[3] = S.s[1] * m64;
    } else if constexpr (FMT == DQ_FMT_Q6_K) {
        const float d = dq_h2f((uint16_t)it.d);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const _Float16 v = (_Float16)(d * (float)(int8_t)((it.x >> (8 * k)) & 0xFF));
            S.s[k] = h2{v, v};
        }
    } else {
        const _Float16 d0 = __builtin_bit_cast(_Float16, (uint16_t)(it.d & 0xFFFF));
        const _Float16 d1 = __builtin_bit_cast(_Float16, (uint16_t)(it.d >> 16));
        S.s[0] = S.s[1] = h2{d0, d0};
        S.s[2] = S.s[3] = h2{d1, d1};
    }
    return S;
}

// The 8 weights of slice C of the item, in the activation's column order
// (dq_quantize_act_f16): columns 8C .. 8C+7 of the item. The conversions are
// those of b_frag_j in dq_gemm.hip (one rounding per weight).
template <int FMT, int C>
__device__ __forceinline__ h8 slice(const Item<FMT>& it, const Scales& S) {
    constexpr int KK = C / 2, H = C % 2;
    uint32_t t[4];
    if constexpr (FMT == DQ_FMT_Q4_K) {
        const uint32_t w = it.p[H][KK];
        const uint32_t magic = 0x54005400u;
        const uint32_t e[4] = {((w << 4) & 0x00F000F0u) | magic, (w & 0x00F000F0u) | magic,
                               ((w >> 4) & 0x00F000F0u) | magic, ((w >> 8) & 0x00F000F0u) | magic};
#pragma unroll
        for (int k = 0; k < 4; ++k)
            t[k] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(h2, e[k]), S.s[k & 1],
                                                                          S.s[2 + (k & 1)]));
    } else if constexpr (FMT == DQ_FMT_Q8_0) {
        const h2 bias = {(_Float16)1152.0f, (_Float16)1152.0f};
        bytes_to_h2(it.p[KK][2 * H] ^ 0x80808080u, bias, S.s[KK], &t[0]);
        bytes_to_h2(it.p[KK][2 * H + 1] ^ 0x80808080u, bias, S.s[KK], &t[2]);
    } else if constexpr (FMT == DQ_FMT_Q4_0) {
        const h2 bias = {(_Float16)1032.0f, (_Float16)1032.0f};
        constexpr int sh = (KK & 1) ? 4 : 0;
        bytes_to_h2((it.p[KK / 2][2 * H] >> sh) & 0x0F0F0F0Fu, bias, S.s[KK], &t[0]);
        bytes_to_h2((it.p[KK / 2][2 * H + 1] >> sh) & 0x0F0F0F0Fu, bias, S.s[KK], &t[2]);
    } else {
        const h2 bias = {(_Float16)1056.0f, (_Float16)1056.0f};
#pragma unroll
        for (int wd = 0; wd < 2; ++wd) {
            const uint32_t lo = it.p[KK & 1][2 * H + wd];
            const uint32_t l4 = KK < 2 ? (lo & 0x0F0F0F0Fu) : ((lo >> 4) & 0x0F0F0F0Fu);
            const uint32_t v6 = l4 | (((it.p[2][2 * H + wd] >> (2 * KK)) & 0x03030303u) << 4);
            bytes_to_h2(v6, bias, S.s[KK], &t[2 * wd]);
        }
    }
    return __builtin_bit_cast(h8, dq_u32x4{t[0], t[1], t[2], t[3]});
}

constexpr int MAX_WAVES = 8;

// The 16 RT rows from n0 of one matrix for the token tiles tile0 .. tile0 +
// MT - 1. Wave w takes the super-blocks w, w + W, ... (the
// waves of a workgroup read neighbouring pieces of a row at the same time). AR
// activation slices are held ahead (8 = a whole super-block).
template <int FMT, int RT, int MT>
__device__ __forceinline__ void direct_rows(const DirectArgs& A, const DirectJob& a, int n0, int tile0,
                                            float (&red)[MAX_WAVES][RT * MT * 4][64]) {
    constexpr int AR = MT <= 2 ? 8 : 4;
    constexpr bool MINT = FMT == DQ_FMT_Q4_K;
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int l16 = lane & 15, g = lane >> 4;
    const int tiles = A.mp / 16;
    const int s0 = wave, s1 = A.nsb, ds = nw;

    f4v acc[RT][MT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = f4v{0.0f, 0.0f, 0.0f, 0.0f};

    if (s0 < s1) {  // wave-uniform
        LaneOff off[RT];
#pragma unroll
        for (int i = 0; i < RT; ++i) off[i] = lane_off<FMT>(a, min(n0 + 16 * i + l16, a.N - 1), g);
        uint32_t aoff[MT], moff[MT];
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int t = 16 * min(tile0 + j, tiles - 1) + l16;
            aoff[j] = (uint32_t)(g * A.mp + t) * 16;
            moff[j] = (uint32_t)min(t, A.M - 1) * 16;
        }
        const uint32_t a_slice = (uint32_t)A.mp * 64;  // bytes of one slice: 4 items x mp tokens x 16
        auto load_a = [&](int sb, int c, h8 (&f)[MT]) {
            const uint8_t* p = (const uint8_t*)a.A + (size_t)(sb * 8 + c) * a_slice;
#pragma unroll
            for (int j = 0; j < MT; ++j) f[j] = *reinterpret_cast<const h8*>(p + aoff[j]);
        };
        auto load_m = [&](int sb, h8 (&f)[MT]) {
            const uint8_t* p = (const uint8_t*)a.minp + (size_t)sb * A.M * 16;
#pragma unroll
            for (int j = 0; j < MT; ++j) f[j] = *reinterpret_cast<const h8*>(p + moff[j]);
        };
        Item<FMT> w[RT], wn[RT];
        h8 af[AR][MT], am[MT], amn[MT];
#pragma unroll
        for (int i = 0; i < RT; ++i) load_item<FMT>(a, off[i], s0, w[i]);
        if constexpr (MINT) load_m(s0, am);
#pragma unroll
        for (int c = 0; c < AR; ++c) load_a(s0, c, af[c]);
        // one super-block; MORE: the next one's loads go out beside it
        auto body = [&](int sb, auto more) {
            constexpr bool MORE = decltype(more)::value;
            Scales S[RT];
            h8 bm[RT];
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                S[i] = item_scales<FMT>(w[i], g);
                if constexpr (MINT) {
                    const h8 v = q4k_neg_mins(w[i].hd, true), zero = {};
                    bm[i] = g == 0 ? v : zero;  // the 8 sub-blocks sit in item 0's K values
                }
            }
            if constexpr (MORE) {
#pragma unroll
                for (int i = 0; i < RT; ++i) load_item<FMT>(a, off[i], sb + ds, wn[i]);
                if constexpr (MINT) load_m(sb + ds, amn);
            }
            __builtin_amdgcn_sched_barrier(0);
            auto step = [&](auto cc) {
                constexpr int C = decltype(cc)::value;
                h8 bf[RT];
#pragma unroll
                for (int i = 0; i < RT; ++i) bf[i] = slice<FMT, C>(w[i], S[i]);
#pragma unroll
                for (int i = 0; i < RT; ++i)
#pragma unroll
                    for (int j = 0; j < MT; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[C % AR][j], bf[i], acc[i][j], 0, 0, 0);
                if constexpr (C + AR < 8) load_a(sb, C + AR, af[C % AR]);
                else if constexpr (MORE) load_a(sb + ds, C + AR - 8, af[C % AR]);
                __builtin_amdgcn_sched_barrier(0);
            };
            step(std::integral_constant<int, 0>{});
            step(std::integral_constant<int, 1>{});
            step(std::integral_constant<int, 2>{});
            step(std::integral_constant<int, 3>{});
            step(std::integral_constant<int, 4>{});
            step(std::integral_constant<int, 5>{});
            step(std::integral_constant<int, 6>{});
            step(std::integral_constant<int, 7>{});
            if constexpr (MINT) {
#pragma unroll
                for (int i = 0; i < RT; ++i)
#pragma unroll
                    for (int j = 0; j < MT; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(am[j], bm[i], acc[i][j], 0, 0, 0);
            }
            if constexpr (MORE) {
#pragma unroll
                for (int i = 0; i < RT; ++i) w[i] = wn[i];
                if constexpr (MINT) {
#pragma unroll
                    for (int j = 0; j < MT; ++j) am[j] = amn[j];
                }
            }
        };
        int sb = s0;
        for (; sb + ds < s1; sb += ds) body(sb, std::true_type{});
        body(sb, std::false_type{});
    }

#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][(i * MT + j) * 4 + r][lane] = acc[i][j][r];
    __syncthreads();
    // D of 16x16x32: lane l, register r -> row n = l % 16, token 4 (l / 16) + r
    for (int u = threadIdx.x; u < RT * MT * 256; u += blockDim.x) {
        const int k = u >> 6, l = u & 63;
        float v = red[0][k][l];
        for (int q = 1; q < nw; ++q) v += red[q][k][l];
        const int r = k & 3, j = (k >> 2) % MT, i = (k >> 2) / MT;
        const int n = n0 + 16 * i + (l & 15), m = 16 * (tile0 + j) + 4 * (l >> 4) + r;
        if (n < a.N && m < A.M) a.y[(size_t)m * a.N + n] = v * a.inv[m];  // a power of two: exact
    }
}

// Grid: the row groups of 16 RT of the matrices times the token blocks of 16
// MT. Workgroup ids go to the 8 XCDs round-robin: the token blocks of one row
// group follow each other on one XCD, so its weights come from HBM once.
// F2 >= 0: the launch mixes matrices of two formats (a workgroup has one).
template <int F1, int F2, int RT, int MT>
__global__ __launch_bounds__(64 * MAX_WAVES) void gemm_direct_kernel(DirectArgs A) {
    __shared__ float red[MAX_WAVES][RT * MT * 4][64];
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int rg = slot / A.mb * 8 + xcd, tile0 = slot % A.mb * MT;
    if (rg >= A.job[A.n - 1].wg_end) return;
    int k = 0;
    while (k + 1 < A.n && rg >= A.job[k].wg_end) ++k;
    const DirectJob& a = A.job[k];
    const int n0 = (rg - (k ? A.job[k - 1].wg_end : 0)) * (16 * RT);
    if constexpr (F2 >= 0) {
        if (a.fmt == F2) {
            direct_rows<F2, RT, MT>(A, a, n0, tile0, red);
            return;
        }
    }
    direct_rows<F1, RT, MT>(A, a, n0, tile0, red);
}

// Waves per workgroup (K ranges): a function of the columns alone, so a
// token's sum depends neither on the token count nor on which matrices share
// a launch.
int k_waves(int nsb) { return nsb >= 32 ? 8 : nsb >= 4 ? 4 : nsb; }

template <int F1, int F2>
int launch(DirectArgs& a, hipStream_t s) {
    // Tokens in blocks of up to 64 (16 MT), two row tiles per wave (half the
    // activation reads per weight byte) where that leaves 8 waves per CU.
    // M = 4 tokens, 14336 x 4096 Q4_K: 20.1 us with two, 22.0 with one;
    // 4096 x 14336 Q6_K: 33.3 with two (4 waves per CU), 24.2 with one.
    int row_tiles = 0;
    for (int k = 0; k < a.n; ++k) row_tiles += (a.job[k].N + 15) / 16;
    const int waves = k_waves(a.nsb);
    const int tiles = a.mp / 16;
    const int mt = tiles >= 3 ? 4 : tiles;
    a.mb = (tiles + mt - 1) / mt;
    const int rt = (long)row_tiles / 2 * a.mb * waves >= 7L * dq_gemm_cus() ? 2 : 1;
    int end = 0;
    for (int k = 0; k < a.n; ++k) a.job[k].wg_end = end += (a.job[k].N + 16 * rt - 1) / (16 * rt);
    const unsigned grid = (unsigned)((end + 7) / 8 * 8 * a.mb);
    auto go = [&](auto kern) { kern<<<grid, 64 * waves, 0, s>>>(a); };
    if (rt == 2) {
        if (mt == 1) go(gemm_direct_kernel<F1, F2, 2, 1>);
        else if (mt == 2) go(gemm_direct_kernel<F1, F2, 2, 2>);
        else go(gemm_direct_kernel<F1, F2, 2, 4>);
    } else {
        if (mt == 1) go(gemm_direct_kernel<F1, F2, 1, 1>);
        else if (mt == 2) go(gemm_direct_kernel<F1, F2, 1, 2>);
        else go(gemm_direct_kernel<F1, F2, 1, 4>);
    }
    return dq_launch_status();
}

bool fill_job(const DqDirectJob& j, size_t cols, DirectJob& a) {
    DqLayout L;
    if (!dq_layout(j.fmt, j.rows, cols, &L)) return false;
    a.w = (const uint8_t*)j.w;
    a.fmt = j.fmt;
    a.N = (int)j.rows;
    a.A = j.act.a;
    a.minp = j.act.minp;
    a.inv = j.act.inv;
    a.y = j.y;
    a.tiled = j.tiled;
    if (j.tiled) {
        const bool two = j.fmt == DQ_FMT_Q6_K || j.fmt == DQ_FMT_Q8_0;
        const uint32_t sb = two ? 2 : 4, pl = 64 * sb * 16;
        const uint32_t slice = L.np * pl + (j.fmt == DQ_FMT_Q4_K ? 1024 : j.fmt == DQ_FMT_Q6_K ? 768 : sb * 256);
        a.n_stages = (int)(cols / 64 / sb);
        a.p_stride = pl;
        a.q_sb = a.x_sb = a.d_sb = slice * (two ? 2 : 1);
    } else {
        a.p_stride = L.p_stride;
        a.q_sb = 64;
        a.x_sb = 16;
        a.d_sb = j.fmt == DQ_FMT_Q6_K ? 2 : 16;
        a.x_off = L.s_off;
        a.d_off = L.d_off;
        a.q_row = (uint32_t)L.q_row;
        a.x_row = (uint32_t)L.s_row;
        a.d_row = (uint32_t)L.d_row;
    }
    return true;
}

}  // namespace

bool dq_gemm_direct_ok(int fmt, size_t rows, size_t cols, size_t n_tok) {
    DqLayout L;
    if (n_tok == 0 || n_tok > (rows > 8192 ? DQ_GEMM_DIRECT_TOK / 2 : DQ_GEMM_DIRECT_TOK) || cols % 256 || cols == 0 || rows == 0) return false;
    if (rows > (1u << 30) || cols > (1u << 20) || !dq_layout(fmt, rows, cols, &L)) return false;
    // lane offsets are 32 bits; the tile copy pads rows to 256
    return (rows + 255) / 256 * 256 * dq_gguf_row_bytes(fmt, cols) + L.total < (1ull << 31);
}

int dq_gemm_direct(const DqDirectJob* jobs, int n, size_t cols, size_t n_tok, hipStream_t s) {
    if (n < 1 || n > DQ_GEMM_DIRECT_JOBS) return DQ_ERR_INVALID_ARG;
    bool done[DQ_GEMM_DIRECT_JOBS] = {};
    auto kq = [](int f) { return f == DQ_FMT_Q4_K || f == DQ_FMT_Q6_K; };
    for (int i = 0; i < n; ++i) {
        if (done[i]) continue;
        // the matrices that share this one's launch: its format, or both K-quants
        DirectArgs a{};
        a.M = (int)n_tok;
        a.mp = (int)((n_tok + 15) / 16 * 16);
        a.nsb = (int)(cols / 256);
        bool mixed = false;
        for (int j = i; j < n; ++j) {
            if (done[j] || !(jobs[j].fmt == jobs[i].fmt || (kq(jobs[j].fmt) && kq(jobs[i].fmt)))) continue;
            if (!fill_job(jobs[j], cols, a.job[a.n++])) return DQ_ERR_NOT_SUPPORTED;
            mixed |= jobs[j].fmt != jobs[i].fmt;
            done[j] = true;
        }
        int rc;
        if (mixed) rc = launch<DQ_FMT_Q4_K, DQ_FMT_Q6_K>(a, s);
        else if (jobs[i].fmt == DQ_FMT_Q4_K) rc = launch<DQ_FMT_Q4_K, -1>(a, s);
        else if (jobs[i].fmt == DQ_FMT_Q6_K) rc = launch<DQ_FMT_Q6_K, -1>(a, s);
        else if (jobs[i].fmt == DQ_FMT_Q8_0) rc = launch<DQ_FMT_Q8_0, -1>(a, s);
        else if (jobs[i].fmt == DQ_FMT_Q4_0) rc = launch<DQ_FMT_Q4_0, -1>(a, s);
        else rc = DQ_ERR_NOT_SUPPORTED;
        if (rc != DQ_OK) return rc;
    }
    return DQ_OK;
}
