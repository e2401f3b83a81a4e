// dq_moe_few.hip - the expert FFN for few tokens per expert, on int8 MFMA.
//
// Semantics as dq_moe.hip: activations quantized per 256 (core/matmul.cpp
// :1660-1778), matmul_q4_k, h = silu(gate) * up quantized the same way. Exact
// as the reference's integer sums are: per 32-block I_j = sum q_w q_x, then
// sum_j sc_j I_j and sum_j m_j sum q_x (the latter on the matrix cores too,
// against the min byte repeated) in integers over the super-block, and one
// float combination per super-block, dx * (d * isum - dmin * msum)
// (:1940-1993).
//
// With a few tokens per expert the call is bound by streaming the routed
// experts' weights once: they go from memory to registers, 16 rows to a wave
// and a super-block ahead; the waves of a workgroup split K and add up through
// LDS (no partials in memory). Gate and up rows are paired in a workgroup,
// which writes silu(gate) * up.
#include <type_traits>

#include "dq_common.h"
#include "dq_f16.h"
#include "dq_moe_tiles.h"

namespace {

// ------------------------------------------------------------ activations --
// Layout of the quantized activation of n rows (pairs) of K values, K % 256
// == 0: q as [K/256][4 items t][4 lane groups g][n][16 bytes], the 16 bytes
// being positions 8g .. 8g+7 of sub-blocks 2t and 2t + 1 (a 16-row fragment
// of the expert GEMM is 4 runs of 256 bytes), and the scales as [K/256][n + 4]
// floats (a lane loads four at once).
struct ActOut {
    uint8_t* q;
    float* d;
    int n;
};
// 256-block b of row p, values v[4] of positions 4 lane .. +3: the reference's
// per-256 quantizer d = amax / 127, id = 127 / amax, q = rint(v * id)
// (core/matmul.cpp:1681-1700). One wave.
__device__ __forceinline__ void quant_256_block(const float4& f, int lane, int b, int p, const ActOut& o) {
    const float v[4] = {f.x, f.y, f.z, f.w};
    const float amax = dq_wave_max_uniform(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
    const float d = amax > 0.0f ? amax / 127.0f : 0.0f;
    const float id = d > 0.0f ? 127.0f / amax : 0.0f;
    uint32_t w = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        int q = (int)rintf(v[i] * id);
        q = q > 127 ? 127 : (q < -127 ? -127 : q);
        w |= (uint32_t)(q & 0xFF) << (8 * i);
    }
    const int t = lane >> 4, sub = (lane >> 3) & 1, g = (lane >> 1) & 3;
    *reinterpret_cast<uint32_t*>(o.q + (((size_t)(b * 4 + t) * 4 + g) * o.n + p) * 16 + sub * 8 + (lane & 1) * 4) = w;
    if (lane == 0) o.d[(size_t)b * (o.n + 4) + p] = d;
}

// One wave per (row, 256-block): row p from x[pairs[p] / k] (pairs given) or
// x[p].
__global__ __launch_bounds__(256) void moe_quant_kernel(const float* __restrict__ x, const int32_t* __restrict__ pairs,
                                                        int k, int K, long n_units, ActOut o) {
    const int lane = threadIdx.x & 63;
    const long u = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (u >= n_units) return;  // uniform per wave
    const int nblk = K / 256, p = (int)(u / nblk), b = (int)(u % nblk);
    const size_t row = pairs ? (size_t)(pairs[p] / k) : (size_t)p;
    quant_256_block(*reinterpret_cast<const float4*>(x + row * K + 256 * b + 4 * lane), lane, b, p, o);
}

// ------------------------------------------------------------ expert GEMM --
typedef int i4v __attribute__((ext_vector_type(4)));

struct MoeGemm {
    const uint8_t* w[2];  // stacked matrices ([n_exp * rows][K]): packed rows, or expert tiles
    DqLayout L;
    float* y;             // [n][rows]
    const uint8_t* q;     // quantized activation (ActOut)
    const float* d;
    const int32_t* offsets;
    int rows, nsb, n, n_tiles;  // n_tiles: 16-row tiles of an expert
};

// Weights of one super-block: this lane's 8 bytes of each item (qd[2t],
// qd[2t+1]) and its row's header.
struct WRaw {
    uint32_t qd[8];
    dq_u32x4 hd;
};
__device__ __forceinline__ long pack64(uint32_t a, uint32_t b) { return (long)(((uint64_t)b << 32) | a); }

constexpr int MAX_WAVES = 8;

// The 16 rows of tile `tile` (NM matrices) for MT tiles of 16 of the expert's
// rows from p0: the workgroup's waves take super-blocks w, w + W, ... A
// super-block's weights are loaded one ahead, its activation fragments
// replaced by the next ones as each item is consumed. D of 16x16x32: lane l,
// register r -> weight row l % 16, activation row 4 (l / 16) + r.
template <int NM, int MT, bool TILED>
__device__ __forceinline__ void expert_rows(const MoeGemm& G, int e, int tile, int p0, int p_end,
                                            float (&red)[MAX_WAVES][NM * MT * 4][64]) {
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int n16 = lane & 15, g = lane >> 4;
    float acc[NM][MT][4];
#pragma unroll
    for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0f;
    if (wave < G.nsb) {  // wave-uniform
        uint32_t off, hoff;
        const uint8_t* base[NM];
        if constexpr (TILED) {
            const size_t c0 = ((size_t)e * ((G.rows + WROWS - 1) / WROWS) + tile / 8) * G.nsb * WT_BYTES;
#pragma unroll
            for (int i = 0; i < NM; ++i) base[i] = G.w[i] + c0 + (tile % 8) * WG_BYTES;
            off = lane * 16;
            hoff = n16 * 16;
        }
        const uint8_t* hbase[NM];
        if constexpr (!TILED) {
            const size_t row0 = (size_t)e * G.rows + 16 * (size_t)tile;
            const int r = min(n16, G.rows - 1 - 16 * tile);
#pragma unroll
            for (int i = 0; i < NM; ++i) {
                hbase[i] = G.w[i] + G.L.s_off + row0 * G.L.s_row;
                base[i] = G.w[i] + G.L.q_off + row0 * G.L.q_row + (g >> 1) * G.L.p_stride;
            }
            off = (uint32_t)(r * G.L.q_row) + 8 * (g & 1);
            hoff = (uint32_t)(r * G.L.s_row);
        }
        auto load = [&](int i, int sb, WRaw& r) {
            if constexpr (TILED) {
                const uint8_t* c = base[i] + (size_t)sb * WT_BYTES;
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const dq_u32x4 v = dq_ld16_stream(c + 1024 * k + off);
                    r.qd[4 * k] = v.x, r.qd[4 * k + 1] = v.y, r.qd[4 * k + 2] = v.z, r.qd[4 * k + 3] = v.w;
                }
                r.hd = dq_ld16_stream(c + 2048 + hoff);
            } else {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const dq_u32x2 v = *reinterpret_cast<const dq_u32x2*>(base[i] + (size_t)sb * 64 + 16 * t + off);
                    r.qd[2 * t] = v.x, r.qd[2 * t + 1] = v.y;
                }
                r.hd = dq_ld16(hbase[i] + (size_t)sb * 16 + hoff);
            }
        };
        uint32_t ao[MT], po[MT];
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            ao[j] = (uint32_t)(g * G.n + min(p0 + 16 * j + n16, p_end - 1)) * 16;
            po[j] = (uint32_t)min(p0 + 16 * j + 4 * g, G.n - 1) * 4;  // 4 scales: the plane has 4 spare
        }
        auto load_a = [&](int sb, int t, int j) {
            return dq_ld16(G.q + (size_t)(sb * 4 + t) * 64 * G.n + ao[j]);
        };
        auto load_d = [&](int sb, int j) {
            const float* s = reinterpret_cast<const float*>(reinterpret_cast<const uint8_t*>(G.d + (size_t)sb * (G.n + 4)) + po[j]);
            return float4{s[0], s[1], s[2], s[3]};
        };
        WRaw w[NM], wn[NM];
        dq_u32x4 af[4][MT];
        float4 dx[MT];
#pragma unroll
        for (int i = 0; i < NM; ++i) load(i, wave, w[i]);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int j = 0; j < MT; ++j) af[t][j] = load_a(wave, t, j);
        auto body = [&](int sb, auto more) {
            constexpr bool MORE = decltype(more)::value;
            // loads in the order they are waited for: this super-block's scales
            // before the next one's weights
#pragma unroll
            for (int j = 0; j < MT; ++j) dx[j] = load_d(sb, j);
            if constexpr (MORE) {
#pragma unroll
                for (int i = 0; i < NM; ++i) load(i, sb + nw, wn[i]);
            }
            uint32_t sc[NM][2], mn[NM][2];
            int is[NM][MT][4];
            i4v ms[NM][MT];
#pragma unroll
            for (int i = 0; i < NM; ++i) {
                q4k_sc_bytes(w[i].hd, sc[i][0], sc[i][1]);
                q4k_m_bytes(w[i].hd, mn[i][0], mn[i][1]);
#pragma unroll
                for (int j = 0; j < MT; ++j) {
                    ms[i][j] = i4v{0, 0, 0, 0};
#pragma unroll
                    for (int r = 0; r < 4; ++r) is[i][j][r] = 0;
                }
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
#pragma unroll
                for (int i = 0; i < NM; ++i) {
                    const uint32_t u = w[i].qd[2 * t], v = w[i].qd[2 * t + 1];
                    const long lo = pack64(u & 0x0F0F0F0Fu, v & 0x0F0F0F0Fu);
                    const long hi = pack64((u >> 4) & 0x0F0F0F0Fu, (v >> 4) & 0x0F0F0F0Fu);
                    const int sh = 16 * (t & 1);
                    const int s0 = (sc[i][t >> 1] >> sh) & 0xFF, s1 = (sc[i][t >> 1] >> (sh + 8)) & 0xFF;
                    const uint32_t sel = (t & 1) ? 0x02020202u : 0x00000000u;
                    const uint32_t m0 = __builtin_amdgcn_perm(0u, mn[i][t >> 1], sel);
                    const uint32_t m1 = __builtin_amdgcn_perm(0u, mn[i][t >> 1], sel + 0x01010101u);
#pragma unroll
                    for (int j = 0; j < MT; ++j) {
                        const long a0 = pack64(af[t][j].x, af[t][j].y), a1 = pack64(af[t][j].z, af[t][j].w);
                        const i4v z = {0, 0, 0, 0};
                        const i4v i0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a0, lo, z, 0, 0, 0);
                        const i4v i1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a1, hi, z, 0, 0, 0);
                        ms[i][j] = __builtin_amdgcn_mfma_i32_16x16x32_i8(a0, pack64(m0, m0), ms[i][j], 0, 0, 0);
                        ms[i][j] = __builtin_amdgcn_mfma_i32_16x16x32_i8(a1, pack64(m1, m1), ms[i][j], 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            is[i][j][r] += __mul24(i0[r], s0) + __mul24(i1[r], s1);
                    }
                }
                if constexpr (MORE) {
#pragma unroll
                    for (int j = 0; j < MT; ++j) af[t][j] = load_a(sb + nw, t, j);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int i = 0; i < NM; ++i) {
                const float d = dq_h2f((uint16_t)(w[i].hd.x & 0xFFFF)), dmin = dq_h2f((uint16_t)(w[i].hd.x >> 16));
#pragma unroll
                for (int j = 0; j < MT; ++j) {
                    const float x[4] = {dx[j].x, dx[j].y, dx[j].z, dx[j].w};
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        acc[i][j][r] += x[r] * (d * (float)is[i][j][r] - dmin * (float)ms[i][j][r]);
                }
            }
            if constexpr (MORE) {
#pragma unroll
                for (int i = 0; i < NM; ++i) w[i] = wn[i];
            }
        };
        int sb = wave;
        for (; sb + nw < G.nsb; sb += nw) body(sb, std::true_type{});
        body(sb, std::false_type{});
    }
#pragma unroll
    for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][(i * MT + j) * 4 + r][lane] = acc[i][j][r];
    __syncthreads();
    for (int u = threadIdx.x; u < MT * 256; u += blockDim.x) {
        const int k = u >> 6, l = u & 63;  // k = 4 j + r
        float v[NM];
#pragma unroll
        for (int i = 0; i < NM; ++i) {
            v[i] = red[0][i * MT * 4 + k][l];
            for (int q = 1; q < nw; ++q) v[i] += red[q][i * MT * 4 + k][l];
        }
        const int row = 16 * tile + (l & 15), p = p0 + 16 * (k >> 2) + 4 * (l >> 4) + (k & 3);
        float o = v[0];
        if constexpr (NM == 2) o = dq_ffn_act<DQ_ACT_SILU>(v[0]) * v[1];
        if (row < G.rows && p < p_end) G.y[(size_t)p * G.rows + row] = o;
    }
}

// Workgroup id -> expert, then 16-row tile: an expert's workgroups spread over
// all XCDs (one token uses two experts; an expert per XCD would leave six
// XCDs idle). An expert with more than 16 entries takes further passes.
template <int NM, bool TILED>
__global__ __launch_bounds__(64 * MAX_WAVES) __attribute__((amdgpu_waves_per_eu(NM == 2 ? 3 : 4, 8)))
void moe_few_gemm_kernel(MoeGemm G) {
    __shared__ float red[MAX_WAVES][NM * 4][64];
    const int e = blockIdx.x / G.n_tiles, tile = blockIdx.x % G.n_tiles;
    const int p_end = G.offsets[e + 1];
    for (int p = G.offsets[e]; p < p_end; p += 16) {  // uniform
        expert_rows<NM, 1, TILED>(G, e, tile, p, p_end, red);
        __syncthreads();  // red is reused
    }
}

// y [n][rows] of every expert's rows: NM = 2 pairs gate (w0) and up (w1).
template <int NM>
int launch_gemm(bool tiled, const uint8_t* w0, const uint8_t* w1, int n_exp, int rows, int K, const uint8_t* q,
                const float* d, const int32_t* offsets, int n, float* y, hipStream_t s) {
    MoeGemm G{};
    G.w[0] = w0;
    G.w[1] = w1;
    if (!dq_layout(DQ_FMT_Q4_K, (size_t)n_exp * rows, K, &G.L)) return DQ_ERR_NOT_SUPPORTED;
    G.y = y;
    G.q = q;
    G.d = d;
    G.offsets = offsets;
    G.rows = rows;
    G.nsb = K / 256;
    G.n = n;
    G.n_tiles = (rows + 15) / 16;
    const long wgs = (long)G.n_tiles * n_exp;
    if (wgs > 0x7FFFFFFF) return DQ_ERR_NOT_SUPPORTED;
    const int waves = G.nsb >= 32 ? 8 : G.nsb >= 4 ? 4 : G.nsb;
    if (tiled) moe_few_gemm_kernel<NM, true><<<(unsigned)wgs, 64 * waves, 0, s>>>(G);
    else moe_few_gemm_kernel<NM, false><<<(unsigned)wgs, 64 * waves, 0, s>>>(G);
    return dq_launch_status();
}

int quant_rows(const float* x, const int32_t* pairs, int k, int n, int K, uint8_t* q, float* d, hipStream_t s) {
    const long units = (long)n * (K / 256);
    moe_quant_kernel<<<(unsigned)((units + 3) / 4), 256, 0, s>>>(x, pairs, k, K, units, ActOut{q, d, n});
    return dq_launch_status();
}

struct FewWs {
    uint8_t *q_in, *q_h;
    float *d_in, *d_h, *h, *down;
    size_t total;
};
FewWs few_carve(const dq_moe_t* m, size_t n, uint8_t* base) {
    const size_t E = m->n_embd, F = m->n_ff;
    FewWs w{};
    size_t off = 0;
    auto take = [&](size_t bytes) {
        uint8_t* p = base ? base + off : nullptr;
        off += dq_align256(bytes);
        return p;
    };
    w.q_in = take(n * E);
    w.d_in = (float*)take((n + 4) * (E / 256) * 4);
    w.q_h = take(n * F);
    w.d_h = (float*)take((n + 4) * (F / 256) * 4);
    w.h = (float*)take(n * F * 4);
    w.down = (float*)take(n * E * 4);
    w.total = off;
    return w;
}

}  // namespace

size_t dq_moe_few_bytes(const dq_moe_t* m, size_t n_ent) { return few_carve(m, n_ent, nullptr).total; }

int dq_moe_few_ffn(const dq_moe_t* m, const float* d_x, const int32_t* d_pairs, const int32_t* d_offsets,
                   size_t n_ent, float** d_down, uint8_t* work, hipStream_t s) {
    const FewWs w = few_carve(m, n_ent, work);
    const bool tiled = m->fmt == DQ_FMT_Q4_K_TILES;
    const int n = (int)n_ent, k = (int)m->n_expert_used, X = (int)m->n_expert;
    const int E = (int)m->n_embd, F = (int)m->n_ff;
    int rc = quant_rows(d_x, d_pairs, k, n, E, w.q_in, w.d_in, s);
    if (rc == DQ_OK)
        rc = launch_gemm<2>(tiled, (const uint8_t*)m->wgate, (const uint8_t*)m->wup, X, F, E, w.q_in, w.d_in, d_offsets,
                            n, w.h, s);
    if (rc == DQ_OK) rc = quant_rows(w.h, nullptr, 1, n, F, w.q_h, w.d_h, s);
    if (rc == DQ_OK)
        rc = launch_gemm<1>(tiled, (const uint8_t*)m->wdown, nullptr, X, E, F, w.q_h, w.d_h, d_offsets, n, w.down, s);
    *d_down = w.down;
    return rc;
}
