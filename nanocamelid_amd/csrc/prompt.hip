// Prompt (prefill) path on gfx950: the batch matmuls for many tokens at once on the matrix cores,
// and the elementwise steps that the verify GEMMs fuse into their epilogues (RoPE and the
// KV-cache scatter, the residual add, SwiGLU + Q8_0), as separate kernels over the matmul's f32
// output.
//
// Q4_0 and Q8_0: each output is the reference's f32 chain over the row's blocks in order
// (matmul_q4_0_batch, inference.rs:1385-1418, and the swizzled form :1525-1574; matmul_q8_0_batch
// :1343-1383):
//   sum = 0; for b: sum += (w_scale[b] * x_scale[b]) * (float)dot_b
// so any number of tokens gives the bits of the 1-token loop.  Per 16 x 16 tile and block the chain
// leaves eight f32 VALU operations per lane (a product and an add for each of its four outputs);
// everything else comes from the matrix cores, whose results arrive as f32:
//   dot_b: v_mfma_f32_16x16x32_f16 on the weights and activations as f16.  Both are integers (weights
//     -8..7 or -128..127, activations -128..127), every partial sum is below 2^20, so the f32 result is
//     the exact integer: no conversion, and no correction for the unsigned nibble;
//   w_scale * x_scale: v_mfma_f32_16x16x1_4b_f32, an outer product of one term per block, four blocks
//     at once.  With one term and a zero addend it rounds like the multiply, subnormals included.
// Operands: A lane (g, r) = row r's elements 4g..4g+3 and 16+4g..+3 of the block, B lane (g, c) = token
// c's (both in the order 0, 2, 16, 18, 1, 3, 17, 19 + 4g that unpacking a nibble dword gives), D lane
// (g, c) = token c, rows 4g..4g+3.
#include "nc_internal.h"
#include "nc_device.h"
#include "nc_offsets.h"

namespace nc {

typedef float p_v4f __attribute__((ext_vector_type(4)));
typedef float p_v16f __attribute__((ext_vector_type(16)));
typedef _Float16 p_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 p_h8 __attribute__((ext_vector_type(8)));

struct PromptGemm {
    const uint8_t* w = nullptr;
    int groups = 0;   // chunks per tile row (R16, Q8_0: 32 blocks each, R64: 8)
    int tiles16 = 0;  // 16-row tiles present in storage
    int M = 0, nb = 0, N = 0, ld_out = 0;
    // the activations in operand order (prompt_repack_kernel), blocks padded to quads: xh [N/16][4 nq]
    // units of [64 lanes] 8 f16, xsm [N/16][nq][64 lanes] x_scale of (block lane / 16, token lane % 16)
    const uint8_t* xh = nullptr;
    const float* xsm = nullptr;
    float* out = nullptr;  // out[n * ld_out + row]
};

// 8 f16 weights of a lane's nibble dword: 0x6400 | n is 1024 + n, so one packed add gives n - 8.
// one (a constant in a VGPR) lets the mask and the or be one v_and_or_b32.
__device__ __forceinline__ p_h8 unpack_q40(uint32_t w, uint32_t one) {
    uint32_t u[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int sh = i == 0 ? 0 : i == 1 ? 4 : i == 2 ? 8 : 12;  // bytes 0,2 low, high; bytes 1,3 low, high
        const p_h2 v = __builtin_bit_cast(p_h2, ((w >> sh) & 0x000F000Fu) | one);
        u[i] = __builtin_bit_cast(uint32_t, v - (p_h2){(_Float16)1032.0f, (_Float16)1032.0f});
    }
    return __builtin_bit_cast(p_h8, make_uint4(u[0], u[1], u[2], u[3]));
}
// the same of a Q8_0 lane's two dwords of signed bytes
__device__ __forceinline__ p_h8 unpack_q80(uint32_t w0, uint32_t w1, uint32_t one) {
    const uint32_t a = w0 ^ 0x80808080u, b = w1 ^ 0x80808080u;
    uint32_t u[4] = {(a & 0x00FF00FFu) | one, (b & 0x00FF00FFu) | one, ((a >> 8) & 0x00FF00FFu) | one,
                     ((b >> 8) & 0x00FF00FFu) | one};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const p_h2 v = __builtin_bit_cast(p_h2, u[i]);
        u[i] = __builtin_bit_cast(uint32_t, v - (p_h2){(_Float16)1152.0f, (_Float16)1152.0f});
    }
    return __builtin_bit_cast(p_h8, make_uint4(u[0], u[1], u[2], u[3]));
}

// Workgroup = 4 waves x (16 rows x 16 KT tokens): the waves take consecutive row tiles of the same
// tokens, whose activation units go through LDS (double-buffered stages of one quad of blocks, loaded
// SD stages ahead into registers), so each is fetched once per workgroup; weights come straight from
// memory, WD - 1 stages ahead.  Token tiles and stages past the last one load the last one's (nc_offsets.h) and
// are never stored or added.  blockIdx.x = token group + row group * token groups.
template <int LAYOUT, int KT, int WD, int SD>
__global__ __launch_bounds__(256, 4) void gemm_b32_prompt_kernel(PromptGemm p, int tgroups) {
    constexpr bool Q8 = LAYOUT == LAYOUT_Q80;
    constexpr int NW = Q8 ? 2 : 1;
    static_assert(WD % 2 == 0 && WD % SD == 0, "ring slots and LDS buffers follow the unrolled stage");
    __shared__ __align__(16) uint4 bs[2][4][KT][64];
    // wave index through readfirstlane: the buffer offsets below are then scalar
    const int lane = threadIdx.x & 63, wv = wave_id_uniform();
    const int g = lane >> 4, r = lane & 15;
    const int t16 = blockIdx.x / tgroups * 4 + wv, tt = blockIdx.x % tgroups * KT;  // row tile, first token tile
    const int nq = (p.nb + 3) / 4, n16 = (p.N + 15) / 16;
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc((void*)p.xh, 0, n16 * nq * 4096, 0x00020000);
    const __amdgpu_buffer_rsrc_t sres = __builtin_amdgcn_make_buffer_rsrc((void*)p.xsm, 0, n16 * nq * 256, 0x00020000);
    // the row tile's storage (clamped into the padded rows) and this lane's offsets in a quad
    const int tile_bytes = LAYOUT == LAYOUT_R64 ? p.groups * kQ40ChunkBytes : p.groups * 8 * r16_quad_bytes(Q8);
    const int ts = min(t16, p.tiles16 - 1), sub = ts & 3;
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(p.w + (size_t)(LAYOUT == LAYOUT_R64 ? ts >> 2 : ts) * tile_bytes), 0, tile_bytes, 0x00020000);
    int nvo, svo;
    if constexpr (LAYOUT == LAYOUT_R64) {
        nvo = (16 * sub + r) * 16 + 4 * g;        // + 1024 * (block % 8)
        svo = 8192 + (16 * sub + r) * 8 + 2 * g;  // scales [row][block % 4], + 512 per half-chunk
    } else {
        nvo = r * 16 + 4 * g;                                       // + 256 j within the quad
        svo = NW * 1024 + 2 * (16 * (r >> 2) + 4 * g + (r & 3));  // scales [row / 4][block][row % 4]
    }
    // this wave's share of a stage's units: token tile wv % KT, blocks wv / KT, + 4 / KT, ...
    const int uk = wv % KT, uj = wv / KT;
    uint32_t wd[WD][4][NW], sw[WD];
    float xsr[WD][KT];
    uint4 st[SD][KT];
#define NC_PB_UNITS(S, SLOT)                                                                                       \
    {                                                                                                              \
        const int uo_ = prompt_unit(tt + uk, (S), n16, nq) * 4096 + uj * 1024;                                     \
        _Pragma("unroll") for (int u = 0; u < KT; u++) st[SLOT][u] = __builtin_bit_cast(                           \
            uint4, __builtin_amdgcn_raw_buffer_load_b128(xres, lane * 16 + u * (4 / KT) * 1024, uo_, 0));          \
    }
#define NC_PB_WEIGHTS(S, SLOT)                                                                                     \
    {                                                                                                              \
        const int h_ = LAYOUT == LAYOUT_R64 ? prompt_r64_half((S), nq) : 0;                                        \
        const int qo_ = LAYOUT == LAYOUT_R64 ? prompt_r64_chunk((S), nq, kQ40ChunkBytes)                           \
                                             : prompt_r16_quad((S), nq, r16_quad_bytes(Q8));                       \
        _Pragma("unroll") for (int j = 0; j < 4; j++) _Pragma("unroll") for (int x = 0; x < NW; x++)               \
            wd[SLOT][j][x] = __builtin_amdgcn_raw_buffer_load_b32(                                                 \
                wres, nvo + (LAYOUT == LAYOUT_R64 ? 1024 : 256) * j + 1024 * x, qo_ + 4096 * h_, 0);               \
        sw[SLOT] = __builtin_amdgcn_raw_buffer_load_b16(wres, svo, qo_ + 512 * h_, 0);                             \
        _Pragma("unroll") for (int k = 0; k < KT; k++) xsr[SLOT][k] = __builtin_bit_cast(                          \
            float, __builtin_amdgcn_raw_buffer_load_b32(sres, lane * 4, prompt_unit(tt + k, (S), n16, nq) * 256, 0)); \
    }
    uint32_t one = 0x64006400u;  // two f16 1024
    asm("" : "+v"(one));
    p_v4f acc[KT];
#pragma unroll
    for (int k = 0; k < KT; k++) acc[k] = p_v4f{0.0f, 0.0f, 0.0f, 0.0f};
    const p_v16f zero16 = {};
    const p_v4f zero4 = {};
#pragma unroll
    for (int b = 0; b < WD; b++) {
        if (b < SD) NC_PB_UNITS(b, b)
        if (b < WD - 1) NC_PB_WEIGHTS(b, b)
    }
#pragma unroll
    for (int u = 0; u < KT; u++) bs[0][u * (4 / KT) + uj][uk][lane] = st[0][u];
    __syncthreads();
    for (int s0 = 0; s0 < nq; s0 += WD) {
#pragma unroll
        for (int b = 0; b < WD; b++) {
            const int s = s0 + b;
            if (s >= nq) break;  // uniform over the workgroup
            NC_PB_UNITS(s + SD, b % SD)  // that slot's stage is in LDS
            NC_PB_WEIGHTS(s + WD - 1, (b + WD - 1) % WD)
            const float ws = f16_to_f32((uint16_t)sw[b]);
            p_h8 a[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if constexpr (Q8) a[j] = unpack_q80(wd[b][j][0], wd[b][j][NW - 1], one);
                else a[j] = unpack_q40(wd[b][j][0], one);
            }
#pragma unroll
            for (int k = 0; k < KT; k++) {
                // the quad's matrix instructions of one token tile back to back, then its chains: the
                // first results are there when the last one has issued, so neither waits
                p_v4f d[4];
                const p_v16f sc = __builtin_amdgcn_mfma_f32_16x16x1f32(ws, xsr[b][k], zero16, 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 4; j++)
                    d[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j], __builtin_bit_cast(p_h8, bs[b & 1][j][k][lane]),
                                                                  zero4, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int v = 0; v < 4; v++) acc[k][v] = acc[k][v] + sc[4 * j + v] * d[j][v];
                __builtin_amdgcn_sched_barrier(0);
            }
            // the other buffer was last read a stage ago, before the barrier that ended that stage
#pragma unroll
            for (int u = 0; u < KT; u++) bs[(b + 1) & 1][u * (4 / KT) + uj][uk][lane] = st[(b + 1) % SD][u];
            __syncthreads();
        }
    }
#undef NC_PB_UNITS
#undef NC_PB_WEIGHTS
#pragma unroll
    for (int k = 0; k < KT; k++) {
        const int n = (tt + k) * 16 + r, row = t16 * 16 + 4 * g;
        if (n >= p.N) continue;
        float* o = p.out + (size_t)n * p.ld_out + row;
        if (row + 3 < p.M && (p.ld_out & 3) == 0) {
            *(float4*)o = make_float4(acc[k][0], acc[k][1], acc[k][2], acc[k][3]);
        } else {
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (row + v < p.M) o[v] = acc[k][v];
        }
    }
}

template <int LAYOUT>
static void launch_b32_prompt(const PromptGemm& p, hipStream_t st) {
    const int64_t rt = (p.M + 15) / 16, n16 = (p.N + 15) / 16;
    auto go = [&]<int KT, int WD, int SD>() {
        const int tg = (int)((n16 + KT - 1) / KT);
        const dim3 grid((unsigned)((rt + 3) / 4 * tg));
        NC_LAUNCH((gemm_b32_prompt_kernel<LAYOUT, KT, WD, SD>), grid, dim3(256), 0, st, p, tg);
    };
    // Token tiles per wave: a wave unpacks its weights once for all of them, but needs company: one wave
    // issues a VALU instruction every 8 cycles at most, four share a SIMD's rate.  Measured (us, Q4_0, K = 4096,
    // 4 / 2 / 1 token tiles): 28672 rows x 256 tokens 144 / 180 / 259, x 64 (448 workgroups) 57 / 63 / 80;
    // 6144 x 256 (384) 55 / 48 / 67; 6144 x 128 (384 with 2) 46 / 38 / 40; 4096 x 128 (256) 46 / 32 / 28.
    const int64_t g4 = (rt + 3) / 4;
    if (n16 > 2 && g4 * ((n16 + 3) / 4) >= 448) go.template operator()<4, 2, 1>();
    else if (n16 > 1 && g4 * ((n16 + 1) / 2) >= 384) go.template operator()<2, 2, 1>();
    else go.template operator()<1, 2, 2>();
}

int launch_gemm_prompt(const QMatDev& w, float* out, int ld_out, int N, hipStream_t st, const void* xh,
                       const float* xsm) {
    const bool q40 = w.type == NC_TYPE_Q4_0 && (w.layout == LAYOUT_R16 || w.layout == LAYOUT_R64);
    if (!q40 && !(w.type == NC_TYPE_Q8_0 && w.layout == LAYOUT_Q80))
        return fail(NC_EINVAL, "prompt matmul: Q4_0 and Q8_0 matrices only");
    if (!xh || !xsm) return fail(NC_EINVAL, "prompt matmul: repacked activations required");
    if (N < 1 || (int64_t)N * w.cols >= (int64_t)1 << 30 || w.dev_bytes >= (int64_t)1 << 31)
        return fail(NC_ERANGE, "prompt matmul: operands exceed 2 GiB");
    PromptGemm p;
    p.w = w.dev;
    p.groups = (int)w.groups;
    p.tiles16 = (int)(w.layout == LAYOUT_R64 ? 4 * w.tiles : w.tiles);
    p.M = (int)w.rows;
    p.nb = (int)(w.cols / 32);
    p.N = N;
    p.ld_out = ld_out;
    p.xh = (const uint8_t*)xh;
    p.xsm = xsm;
    p.out = out;
    if (w.layout == LAYOUT_Q80) launch_b32_prompt<LAYOUT_Q80>(p, st);
    else if (w.layout == LAYOUT_R16) launch_b32_prompt<LAYOUT_R16>(p, st);
    else launch_b32_prompt<LAYOUT_R64>(p, st);
    NC_HIP(hipGetLastError());
    return NC_OK;
}

// ---------------------------------------------------------------- Q4_K and Q5_K prompt matmul
// matmul_q4_k_batch (inference.rs:2006-2132, x86 path :2083-2130) for many tokens: per row and
// token, super-blocks in order, each the f32 sum from 0.0 over its eight 32-value sub-blocks j of
//   xs_j * (sc_j * (float)W_j - mn_j * (float)A_j),   sc_j = d * s_j, mn_j = dmin * m_j
// (q8.rs:1339-1376 dot_q8_scaled_preloaded, scales by q4_k_scale_min q8.rs:2009-2018; Q5_K likewise,
// q8.rs:1551-1594), with W_j = sum q * x (unsigned values) and A_j = sum x of the sub-block; that
// super-block sum is added to the row's sum.  W_j arrives as an exact f32 from f16 MFMA, mn_j * A_j from a
// one-term f32 MFMA, as in the kernel above; four VALU operations per output and sub-block remain.
// The values q are unsigned and below 2^10, so their bits alone are the f16 subnormal q * 2^-24, which the matrix
// core multiplies exactly: unpacking is a shift and a mask, W_j comes times 2^-24 and sc_j carries the 2^24 (both
// exact, so the product rounds as before).  With an or and a packed subtraction a pair, as the signed Q4_0 values
// need, 4096 x 4096 at 96 tokens took 31.4 us against 27.8, 5120 x 3072 at 64 25.5 against 22.5, 8192 x 3072 at 250
// 51.2 against 47.8 (two calls in turn).
// Sub-block 2p is the low nibbles of bytes 32p..32p+31, 2p + 1 the high nibbles.  Lane (g, r)
// decodes its row's scales and mins of sub-blocks 2g and 2g + 1 into a per-wave LDS table.  Same tiles,
// stages (half a super-block) and activation staging as gemm_b32_prompt_kernel; weights stay in the verify
// layouts (R16K: 16-row tiles, chunks of 4 super-blocks; R64: 64-row tiles, one super-block per
// chunk), each chunk 9 (Q5_K 11) slots of [64 lanes x 16 B]: header (d, dmin, 12 scale bytes), Q5_K's two
// slots of high-bit bytes, nibbles.
// Q4_K, 250 / 256 tokens, against int8 MFMA with conversions and 32 x 32 wave tiles: 8192 x 3072 58 -> 56 us,
// 3072 x 8192 92 -> 73, 16384 x 3072 108 -> 97 (before the subnormals).  Q5_K 14336 x 4096 took 16-token slices (16 x 62 us), now 137.
constexpr float kSubnormal = 16777216.0f;  // 2^24: an f16 subnormal's bits over its value
struct PromptGemmK {
    const uint8_t* w = nullptr;
    int nsb = 0, groups = 0, tiles16 = 0;  // super-blocks per row; R16K chunks per tile; 16-row tiles stored
    int M = 0, N = 0, ld_out = 0;
    const uint8_t* xh = nullptr;  // as PromptGemm
    const float* xsm = nullptr;   // [N/16][nq][16 tokens] float4: a quad's x_scales
    const float* xam = nullptr;   // [N/16][nq][64 lanes]: (float) sum of block lane / 16's values, token lane % 16
    float* out = nullptr;         // out[n * ld_out + row]
};

__device__ __forceinline__ void q4k_scale_min_dev(int j, uint32_t s0, uint32_t s1, uint32_t s2, uint32_t* s, uint32_t* m) {
    // 12 scale bytes in three dwords; byte k = (dw[k / 4] >> 8 (k % 4)) & 255 (q8.rs:2009-2018)
    auto byte = [&](int k) -> uint32_t {
        const uint32_t d = k < 4 ? s0 : k < 8 ? s1 : s2;
        return (d >> (8 * (k & 3))) & 0xffu;
    };
    if (j < 4) {
        *s = byte(j) & 63;
        *m = byte(j + 4) & 63;
    } else {
        *s = (byte(j + 4) & 0x0f) | ((byte(j - 4) >> 6) << 4);
        *m = (byte(j + 4) >> 4) | ((byte(j) >> 6) << 4);
    }
}

template <int LAYOUT, bool Q5, int KT, int SD>
__global__ __launch_bounds__(256, KT == 4 ? 3 : 4) void gemm_k_prompt_kernel(PromptGemmK p, int tgroups) {
    constexpr int NSLOT = Q5 ? 11 : 9, QS = Q5 ? 3 : 1, CHUNK = 1024 * NSLOT, WD = 2;
    __shared__ __align__(16) uint4 bs[2][4][KT][64];
    __shared__ __align__(16) float xss[2][KT][64];
    __shared__ __align__(16) float tab[4][8][2][16];  // per wave: [sub-block][sc, mn][row]
    const int lane = threadIdx.x & 63, wv = wave_id_uniform();
    const int g = lane >> 4, r = lane & 15;
    const int t16 = blockIdx.x / tgroups * 4 + wv, tt = blockIdx.x % tgroups * KT;  // row tile, first token tile
    const int nq = 2 * p.nsb, n16 = (p.N + 15) / 16;
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc((void*)p.xh, 0, n16 * nq * 4096, 0x00020000);
    const __amdgpu_buffer_rsrc_t sres = __builtin_amdgcn_make_buffer_rsrc((void*)p.xsm, 0, n16 * nq * 256, 0x00020000);
    const __amdgpu_buffer_rsrc_t ares = __builtin_amdgcn_make_buffer_rsrc((void*)p.xam, 0, n16 * nq * 256, 0x00020000);
    // the row tile's storage (clamped into the padded rows)
    const int ts = min(t16, p.tiles16 - 1);
    const int tile_bytes = (LAYOUT == LAYOUT_R16K ? p.groups : p.nsb) * CHUNK;
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(p.w + (size_t)(LAYOUT == LAYOUT_R16K ? ts : ts >> 2) * tile_bytes), 0, tile_bytes, 0x00020000);
    const int hvo = LAYOUT == LAYOUT_R16K ? r * 16 : (16 * (ts & 3) + r) * 16, nvo = hvo + 4 * g;
    const int uk = wv % KT, uj = wv / KT;  // this wave's share of a stage's units
    uint32_t wd[WD][2][2], hdn[6];
    float xar[WD][KT], xst[SD];
    uint4 st[SD][KT];
#define NC_PK_UNITS(S, SLOT)                                                                                       \
    {                                                                                                              \
        const int un_ = prompt_unit(tt + uk, (S), n16, nq);                                                        \
        _Pragma("unroll") for (int u = 0; u < KT; u++) st[SLOT][u] = __builtin_bit_cast(                           \
            uint4, __builtin_amdgcn_raw_buffer_load_b128(xres, lane * 16 + u * (4 / KT) * 1024, un_ * 4096 + uj * 1024, 0)); \
        xst[SLOT] = __builtin_bit_cast(                                                                            \
            float, __builtin_amdgcn_raw_buffer_load_b32(sres, lane * 4, un_ * 256, 0));                            \
    }
#define NC_PK_WEIGHTS(S, SLOT, HEAD)                                                                               \
    {                                                                                                              \
        const int co_ = prompt_k_chunk(LAYOUT == LAYOUT_R16K, (S), nq, CHUNK);                                     \
        _Pragma("unroll") for (int pp = 0; pp < 2; pp++) _Pragma("unroll") for (int x = 0; x < 2; x++)             \
            wd[SLOT][pp][x] = __builtin_amdgcn_raw_buffer_load_b32(                                                \
                wres, nvo + 1024 * (2 * pp + x), co_ + (QS + 4 * prompt_k_half((S), nq)) * 1024, 0);                            \
        if (HEAD) {                                                                                                \
            const uint4 h_ = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(wres, hvo, co_, 0));  \
            hdn[0] = h_.x, hdn[1] = h_.y, hdn[2] = h_.z, hdn[3] = h_.w;                                            \
            if (Q5) {                                                                                              \
                hdn[4] = __builtin_amdgcn_raw_buffer_load_b32(wres, nvo + 1024, co_, 0);                           \
                hdn[5] = __builtin_amdgcn_raw_buffer_load_b32(wres, nvo + 2048, co_, 0);                           \
            }                                                                                                      \
        }                                                                                                          \
        _Pragma("unroll") for (int k = 0; k < KT; k++) xar[SLOT][k] = __builtin_bit_cast(                          \
            float, __builtin_amdgcn_raw_buffer_load_b32(ares, lane * 4, prompt_unit(tt + k, (S), n16, nq) * 256, 0)); \
    }
    p_v4f acc[KT], part[KT];
#pragma unroll
    for (int k = 0; k < KT; k++) acc[k] = p_v4f{0.0f, 0.0f, 0.0f, 0.0f};
    const p_v16f zero16 = {};
    const p_v4f zero4 = {};
#pragma unroll
    for (int b = 0; b < SD; b++) NC_PK_UNITS(b, b)
    NC_PK_WEIGHTS(0, 0, true)
#pragma unroll
    for (int u = 0; u < KT; u++) bs[0][u * (4 / KT) + uj][uk][lane] = st[0][u];
    xss[0][uk][lane] = xst[0];
    __syncthreads();
    uint32_t h0 = 0, h1 = 0;
    for (int s0 = 0; s0 < nq; s0 += 2) {  // nq is even: a super-block per turn
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const int s = s0 + b;
            if (b == 0) {
                // this lane's row r, sub-blocks 2g and 2g + 1: scales and mins into the table
                const float d = f16_to_f32((uint16_t)(hdn[0] & 0xffff)), dmin = f16_to_f32((uint16_t)(hdn[0] >> 16));
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    uint32_t sv, mv;
                    q4k_scale_min_dev(2 * g + e, hdn[1], hdn[2], hdn[3], &sv, &mv);
                    tab[wv][2 * g + e][0][r] = (d * (float)sv) * kSubnormal;
                    tab[wv][2 * g + e][1][r] = dmin * (float)mv;
                }
                if (Q5) h0 = hdn[4], h1 = hdn[5];
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
                for (int k = 0; k < KT; k++) part[k] = p_v4f{0.0f, 0.0f, 0.0f, 0.0f};
            }
            NC_PK_UNITS(s + SD, b % SD)  // that slot's stage is in LDS
            NC_PK_WEIGHTS(s + 1, (b + 1) & 1, b == 1)
            p_h8 a[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t w0 = wd[b][j >> 1][0], w1 = wd[b][j >> 1][1];
                const int sh = j & 1 ? 4 : 0;
                uint32_t u[4] = {w0 >> sh, w1 >> sh, w0 >> (8 + sh), w1 >> (8 + sh)};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    u[i] = u[i] & 0x000F000Fu;
                    if constexpr (Q5) {  // bit 4 b + j of a byte of h0 / h1 is the value's bit 4
                        const uint32_t h = (i & 1 ? h1 : h0) >> (8 * (i >> 1));
                        const int bit = 4 * b + j;
                        u[i] |= (bit < 4 ? h << (4 - bit) : h >> (bit - 4)) & 0x00100010u;
                    }
                }
                a[j] = __builtin_bit_cast(p_h8, make_uint4(u[0], u[1], u[2], u[3]));
            }
            const float mnv = tab[wv][4 * b + g][1][r];  // A operand of the outer product: (sub-block, row)
            p_v4f sc[4];
#pragma unroll
            for (int j = 0; j < 4; j++) sc[j] = *(const p_v4f*)&tab[wv][4 * b + j][0][4 * g];
#pragma unroll
            for (int k = 0; k < KT; k++) {
                p_v4f d[4];
                const p_v16f bo = __builtin_amdgcn_mfma_f32_16x16x1f32(mnv, xar[b][k], zero16, 0, 0, 0);
                const p_v4f xs4 = *(const p_v4f*)&xss[b][k][4 * r];
#pragma unroll
                for (int j = 0; j < 4; j++)
                    d[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j], __builtin_bit_cast(p_h8, bs[b][j][k][lane]), zero4,
                                                                  0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        part[k][v] = part[k][v] + xs4[j] * (sc[j][v] * d[j][v] - bo[4 * j + v]);
                // the next token tile's products start after these sums (all would be live at once otherwise)
                if (k + 1 < KT) asm volatile("" : "+v"(part[k]), "+v"(xar[b][k + 1]));
            }
            if (b == 1) {
#pragma unroll
                for (int k = 0; k < KT; k++)
#pragma unroll
                    for (int v = 0; v < 4; v++) acc[k][v] = acc[k][v] + part[k][v];
            }
            // the other buffer was last read a stage ago, before the barrier that ended that stage; the
            // wave's own table is rewritten after it too
#pragma unroll
            for (int u = 0; u < KT; u++) bs[(b + 1) & 1][u * (4 / KT) + uj][uk][lane] = st[(b + 1) % SD][u];
            xss[(b + 1) & 1][uk][lane] = xst[(b + 1) % SD];
            __syncthreads();
        }
    }
#undef NC_PK_UNITS
#undef NC_PK_WEIGHTS
#pragma unroll
    for (int k = 0; k < KT; k++) {
        const int n = (tt + k) * 16 + r, row = t16 * 16 + 4 * g;
        if (n >= p.N) continue;
        float* o = p.out + (size_t)n * p.ld_out + row;
        if (row + 3 < p.M && (p.ld_out & 3) == 0) {
            *(float4*)o = make_float4(acc[k][0], acc[k][1], acc[k][2], acc[k][3]);
        } else {
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (row + v < p.M) o[v] = acc[k][v];
        }
    }
}

template <int LAYOUT, bool Q5>
static void launch_k_prompt(const PromptGemmK& p, hipStream_t st) {
    const int64_t g4 = (p.M + 63) / 64, n16 = (p.N + 15) / 16;
    auto go = [&]<int KT, int SD>() {
        const int tg = (int)((n16 + KT - 1) / KT);
        NC_LAUNCH((gemm_k_prompt_kernel<LAYOUT, Q5, KT, SD>), dim3((unsigned)(g4 * tg)), dim3(256), 0, st, p, tg);
    };
    // As launch_b32_prompt, with more work per output to spread over waves.  Measured (us, Q4_K, 4 / 2 / 1 token
    // tiles): 16384 x 3072 x 256 tokens (1024 workgroups with 4) 97 / 101 / 135, 8192 x 3072 x 250 (512 with 4) 58 /
    // 56 / 74, x 128 (512 with 2) 47 / 39 / 43, x 64 (256) 45 / 32 / 28; 3072 x 8192 x 256 (384 with 2) 108 / 83 / 73.
    if (n16 > 2 && g4 * ((n16 + 3) / 4) >= 1024) go.template operator()<4, 1>();
    else if (n16 > 1 && g4 * ((n16 + 1) / 2) >= 512) go.template operator()<2, 1>();
    else go.template operator()<1, 2>();
}

int launch_gemm_prompt_k(const QMatDev& w, float* out, int ld_out, int N, hipStream_t st, const void* xh,
                         const float* xsm, const float* xam) {
    if ((w.type != NC_TYPE_Q4_K && w.type != NC_TYPE_Q5_K) || (w.layout != LAYOUT_R16K && w.layout != LAYOUT_R64))
        return fail(NC_EINVAL, "K-quant prompt matmul: Q4_K and Q5_K matrices only");
    if (!xh || !xsm || !xam) return fail(NC_EINVAL, "K-quant prompt matmul: repacked activations required");
    if (N < 1 || (int64_t)N * w.cols >= (int64_t)1 << 30 || w.dev_bytes >= (int64_t)1 << 31)
        return fail(NC_ERANGE, "K-quant prompt matmul: operands exceed 2 GiB");
    PromptGemmK p;
    p.w = w.dev;
    p.nsb = (int)(w.cols / 256);
    p.groups = (int)w.groups;
    p.tiles16 = (int)(w.layout == LAYOUT_R16K ? w.tiles : 4 * w.tiles);
    p.M = (int)w.rows;
    p.N = N;
    p.ld_out = ld_out;
    p.xh = (const uint8_t*)xh;
    p.xsm = xsm;
    p.xam = xam;
    p.out = out;
    if (w.type == NC_TYPE_Q5_K) {
        if (w.layout == LAYOUT_R16K) launch_k_prompt<LAYOUT_R16K, true>(p, st);
        else launch_k_prompt<LAYOUT_R64, true>(p, st);
    } else {
        if (w.layout == LAYOUT_R16K) launch_k_prompt<LAYOUT_R16K, false>(p, st);
        else launch_k_prompt<LAYOUT_R64, false>(p, st);
    }
    NC_HIP(hipGetLastError());
    return NC_OK;
}

// Activations in operand order as f16: xh unit (tile t, block b of 4 nq, lane (g, c)) = token 16t +
// c's elements 0, 2, 16, 18, 1, 3, 17, 19 + 4g of the block, zero past N and past the row's blocks.  xam null:
// xsm (t, quad, lane (j, c)) = its scale of block 4 quad + j; else (K-quants) xsm (t, quad, c, j) and xam (t,
// quad, lane (j, c)) = the float sum of the block's values (exact).  One thread per unit lane, then per scale.
__global__ void prompt_repack_kernel(const int8_t* x, const float* xs, int N, int nb, uint4* xh, float* xsm,
                                     float* xam) {
    const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int n16 = (N + 15) / 16, nbp = (nb + 3) / 4 * 4, K = 32 * nb;
    const int64_t nx = (int64_t)n16 * nbp * 64;
    if (id < nx) {
        const int lane = (int)(id & 63), g = lane >> 4, c = lane & 15;
        const int64_t tb = id >> 6;
        const int b = (int)(tb % nbp), n = (int)(tb / nbp) * 16 + c;
        p_h8 v = {};
        if (n < N && b < nb) {
            const int8_t* e = x + (size_t)n * K + 32 * b + 4 * g;
            const char4 lo = *(const char4*)e, hi = *(const char4*)(e + 16);
            v = p_h8{(_Float16)lo.x, (_Float16)lo.z, (_Float16)hi.x, (_Float16)hi.z,
                     (_Float16)lo.y, (_Float16)lo.w, (_Float16)hi.y, (_Float16)hi.w};
        }
        xh[id] = __builtin_bit_cast(uint4, v);
        return;
    }
    const int64_t id2 = id - nx;
    if (id2 >= (int64_t)n16 * nbp * 16) return;
    const int c = (int)(id2 & 15), j = (int)(id2 >> 4) & 3;
    const int64_t tq = id2 >> 6;
    const int b = (int)(tq % (nbp / 4)) * 4 + j, n = (int)(tq / (nbp / 4)) * 16 + c;
    const bool live = n < N && b < nb;
    xsm[xam ? tq * 64 + 4 * c + j : id2] = live ? xs[(size_t)n * nb + b] : 0.0f;
    if (xam) {
        int sum = 0;
        if (live) {
            const int* e = (const int*)(x + (size_t)n * K + 32 * b);
#pragma unroll
            for (int d = 0; d < 8; d++) sum = __builtin_amdgcn_sdot4(e[d], 0x01010101, sum, false);
        }
        xam[id2] = (float)sum;
    }
}

int launch_prompt_repack(const int8_t* x, const float* xs, int N, int K, void* xh, float* xsm, hipStream_t st,
                         float* xam) {
    const int nb = K / 32;
    const int64_t total = (int64_t)((N + 15) / 16) * ((nb + 3) / 4 * 4) * 80;
    NC_LAUNCH(prompt_repack_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, x, xs, N, nb, (uint4*)xh,
              xsm, xam);
    NC_HIP(hipGetLastError());
    return NC_OK;
}

// ---------------------------------------------------------------- elementwise steps
// inference.rs:3894-3924: RoPE (NORM pairs 2i, 2i+1 of each head) on the q and k rows of the
// fused q|k|v output, then q to q_out and k, v into the KV cache at positions start + n.
// The same arithmetic as the verify GEMMs' EPI_QKV_ROPE epilogue.
__global__ void prompt_qkv_rope_kernel(const float* y, int ld, int start, int aw, int kw, int hd, int rope_half,
                                       const float* rope_tab, float* q_out, float* kcache, float* vcache,
                                       int max_ctx) {
    const int n = blockIdx.y;
    const int row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= aw + 2 * kw) return;
    const float* yr = y + (size_t)n * ld;
    float v = yr[row];
    const int pos = start + n;
    const bool is_q = row < aw, is_k = !is_q && row < aw + kw;
    const int rr = is_q ? row : (is_k ? row - aw : row - aw - kw);
    if (is_q || is_k) {
        const int i = (rr % hd) >> 1;
        if (i < rope_half) {
            const float* sc = rope_tab + ((size_t)pos * rope_half + i) * 2;
            const float sn = sc[0], cs = sc[1];
            const float x0 = yr[row & ~1], x1 = yr[row | 1];
            v = (row & 1) ? (x0 * sn + x1 * cs) : (x0 * cs - x1 * sn);
        }
    }
    if (is_q) {
        q_out[(size_t)n * aw + rr] = v;
    } else {
        const int kvh = rr / hd, d = rr % hd;
        if (is_k) kcache[(((size_t)kvh * (hd / 4) + d / 4) * max_ctx + pos) * 4 + (d & 3)] = v;
        else vcache[(((size_t)kvh * (max_ctx / 4) + pos / 4) * hd + d) * 4 + (pos & 3)] = v;
    }
}

int launch_prompt_qkv_rope(const float* y, int N, int start, int aw, int kw, int hd, int rope_half,
                           const float* rope_tab, float* q_out, float* kcache, float* vcache, int max_ctx,
                           hipStream_t st) {
    if ((aw | kw) & 1) return fail(NC_EINVAL, "prompt RoPE: widths must be even");
    const int rows = aw + 2 * kw;
    NC_LAUNCH(prompt_qkv_rope_kernel, dim3((rows + 255) / 256, N), dim3(256), 0, st, y, rows, start, aw, kw,
                       hd, rope_half, rope_tab, q_out, kcache, vcache, max_ctx);
    NC_HIP(hipGetLastError());
    return NC_OK;
}

// hidden += matmul output (inference.rs:3985, 4073; add_residual_batch :4122), as the
// EPI_RESIDUAL epilogue: h = y + h.
__global__ void prompt_residual_kernel(const float* y, float* hidden, int64_t total) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < total) hidden[i] = y[i] + hidden[i];
}

int launch_prompt_residual(const float* y, float* hidden, int N, int d, hipStream_t st) {
    const int64_t total = (int64_t)N * d;
    NC_LAUNCH(prompt_residual_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, y, hidden, total);
    NC_HIP(hipGetLastError());
    return NC_OK;
}

// fused_silu_mul (inference.rs:3367-3390) on the interleaved gate|up output (64-row group t:
// gate rows 32t..32t+31 in rows 64t..64t+31, the matching up rows in 64t+32..64t+63) or, with
// split, on gate rows 0..F-1 followed by up rows F..2F-1; then quantize_f32_to_q8_0 of each
// 32-wide block (inference.rs:4034-4041), as the EPI_SWIGLU_Q8 epilogue.  One half-wave per
// (token, block).
__global__ void prompt_swiglu_q8_kernel(const float* y, int F, int total_blocks, int8_t* xq, float* xs,
                                        int32_t* xs8, int split) {
    const int hb = (blockIdx.x * blockDim.x + threadIdx.x) >> 5;  // (token, block) index
    if (hb >= total_blocks) return;                                 // whole half-waves exit together
    const int l = threadIdx.x & 31;
    const int nbf = F / 32, n = hb / nbf, t = hb % nbf;
    const float* yr = y + (size_t)n * 2 * F + (split ? 32 * t : 64 * t);
    const float g = yr[l], up = yr[(split ? F : 32) + l];
    const float sig = 1.0f / (1.0f + expf_glibc(-g));
    const float v = g * sig * up;
    const float amax = halfwave_amax(v);
    float scale;
    const int q = quantize_lane_q8(v, amax, &scale);
    const int qs = halfwave_isum(q);
    xq[(size_t)n * F + 32 * t + l] = (int8_t)q;
    if (l == 0) {
        xs[hb] = scale;
        xs8[hb] = -8 * qs;
    }
}

int launch_prompt_swiglu_q8(const float* y, int N, int F, int8_t* xq, float* xs, int32_t* xs8, hipStream_t st,
                            bool split) {
    if (F % 32) return fail(NC_EINVAL, "prompt SwiGLU: width must be a multiple of 32");
    const int total = N * (F / 32);
    NC_LAUNCH(prompt_swiglu_q8_kernel, dim3((total * 32 + 255) / 256), dim3(256), 0, st, y, F, total, xq, xs,
                       xs8, split ? 1 : 0);
    NC_HIP(hipGetLastError());
    return NC_OK;
}

}  // namespace nc
