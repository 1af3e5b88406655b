// Attention for passes with many (row, head) units (prompt passes, wide verify passes at long
// contexts), in the reference's order (apply_attention_head, inference.rs:4142-4292): scores, softmax
// and the weighted V sum as three kernels over tiles of 16 queries that share a KV head.  The scores kernel
// also serves every smaller pass whose rows outgrow the one-kernel attention: from one row on it is at
// least as fast as a lane per position with the keys staged in LDS was (64 heads x 9 rows at 8180 positions
// 55 -> 33 us, 32 x 16 at 8000 69 -> 26, 32 x 4 at 4000 14.6 -> 7.2, 64 x 1 at 2500 8.0 -> 5.9, head dim 64
// 32 x 1 at 4000 5.2 -> 5.0).
//
//   scores: s_p = (((-0 + q_0 k_0) + q_1 k_1) + ...) * scale, dims in order (dot :3542-3558);
//   softmax: max, e_p = expf(s_p - max), sum = e_0 + e_1 + ... left to right (:3522-3540);
//   output:  o_d = (prob_0 v_0d + prob_1 v_1d) + ..., prob_p = e_p * (1 / sum), in order (:3603-3623).
//
// Every chain step is a rounded product and a rounded add, so no fused or reordered sum will do.  The
// per-unit kernels (layer.hip) run both on the VALU, one lane per position or dim, re-reading the keys and
// values for every unit.  Here v_mfma_f32_16x16x1_4b_f32 forms the products: an outer product with one term
// and a zero addend rounds like the multiply (subnormals included; a -0 product arrives as +0, which no
// later step can tell).  One instruction gives 16 queries x 16 positions (or dims) x 4 chain steps, leaving 16
// adds per lane: half the VALU instructions, and a wave issues one of those per 8 cycles at most.  Each
// operand is one 16-byte load per lane for 16 chain steps, shared by 16 queries or 16 columns.
// Bound: issue (MFMA 33 + adds 37 cycles per 1024 steps on a SIMD; they do not overlap on this chip).
// Measured, 8B layer, pass of 256 rows over 2048 positions in all (mean of 8 passes): scores 48, softmax 25, V
// sum 53 us at the last ones; the attention of the whole prompt 6.8 -> 2.3 ms a layer pair.
#include "nc_internal.h"
#include "nc_device.h"
#include "nc_offsets.h"

namespace nc {

typedef float t_v4f __attribute__((ext_vector_type(4)));
typedef float t_v16f __attribute__((ext_vector_type(16)));

// Queries of KV head kvh: qi = g * N + n (head kvh * G + g, row n), tiles of 16; past the last one the
// index is clamped and nothing is stored.
struct TileQuery {
    int n, h;
    bool live;
};
__device__ __forceinline__ TileQuery tile_query(const AttnParams& a, int kvh, int qi) {
    const int G = a.H / a.Hkv, GN = G * a.N;
    const int q = min(qi, GN - 1);
    return {q % a.N, kvh * G + q / a.N, qi < GN};
}

// acc[v] += the 16 steps 4j + e (j, e in order) of MFMA results d[e][4j + v]: lane (g, c) holds queries
// 4g + v of column c.
__device__ __forceinline__ void tile_add16(t_v4f& acc, const t_v16f (&d)[4]) {
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int v = 0; v < 4; v++) acc[v] = acc[v] + d[e][4 * j + v];
}

// Scores.  Workgroup = one query tile x 64 * PT positions; wave w takes the 16-position tiles w, w + 4, ...
// MFMA operands of dims 16 I + 4 j + e: A lane (j, r) = query r, B lane (j, c) = position c (key dim quads
// [hd/4][ctx][4]), so register e of one 16-byte load each.  The wave's queries stay in registers.  A tile that holds
// a position of the pass lies inside the cache (max_ctx is a multiple of 16), so no load is out of range.
template <int HD, int PT>
__global__ __launch_bounds__(256, 3) void attn_tile_scores_kernel(AttnParams a) {
    constexpr int NI = HD / 16;
    const int lane = threadIdx.x & 63, w = wave_id_uniform();
    const int j = lane >> 4, r = lane & 15;
    const int kvh = blockIdx.x % a.Hkv, tile = blockIdx.x / a.Hkv;
    const int pos0 = a.d_pos[0], p0 = blockIdx.y * 64 * PT;
    // the longest row of the tile: row N - 1 when the tile spans two heads' rows, else its last query's
    const TileQuery qa = tile_query(a, kvh, 16 * tile), qz = tile_query(a, kvh, 16 * tile + 15);
    const int last = pos0 + (qa.h == qz.h ? qz.n : a.N - 1);
    if (p0 > last) return;
    const TileQuery q = tile_query(a, kvh, 16 * tile + r);
    t_v4f qv[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) qv[i] = *(const t_v4f*)(a.q + ((size_t)q.n * a.H + q.h) * HD + 16 * i + 4 * j);
    // this lane's stores: queries 4j + v
    float* out[4];
    int lim[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const TileQuery s = tile_query(a, kvh, 16 * tile + 4 * j + v);
        out[v] = a.scores + ((size_t)s.n * a.H + s.h) * a.max_ctx;
        lim[v] = s.live ? pos0 + s.n : -1;
    }
    const __amdgpu_buffer_rsrc_t kres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.kcache + (size_t)kvh * a.max_ctx * HD), 0, a.max_ctx * HD * 4, 0x00020000);
    const int qstride = a.max_ctx * 16;  // bytes between dim quads
    const t_v16f zero = {};
    for (int t = 0; t < PT; t++) {
        const int pt = p0 + 16 * (w + 4 * t);
        if (pt > last) break;
        const int kvo = (pt + r) * 16 + j * qstride;
        t_v4f acc = {-0.0f, -0.0f, -0.0f, -0.0f};
        t_v4f kv[NI];
#pragma unroll
        for (int i = 0; i < NI; i++)
            kv[i] = __builtin_bit_cast(t_v4f, __builtin_amdgcn_raw_buffer_load_b128(kres, kvo, 4 * i * qstride, 0));
#pragma unroll
        for (int i = 0; i < NI; i++) {
            t_v16f d[4];
#pragma unroll
            for (int e = 0; e < 4; e++) d[e] = __builtin_amdgcn_mfma_f32_16x16x1f32(qv[i][e], kv[i][e], zero, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            tile_add16(acc, d);
            // the next products start after these adds (all NI would be live at once otherwise)
            if (i + 1 < NI) asm volatile("" : "+v"(acc), "+v"(kv[i + 1]));
        }
        const int p = pt + r;
#pragma unroll
        for (int v = 0; v < 4; v++)
            if (p <= lim[v]) out[v][p] = acc[v] * a.scale;
    }
}

// Softmax numerators and sums of a tile's 16 rows.  Waves 0-7 take two rows each: the row's max, then
// e = expf(s - max) 256 positions at a time, written over the scores and into LDS; wave 8 adds the
// previous 256 of every row in order (lane = row), so each sum is the literal left-to-right chain: with 16
// rows per workgroup and many workgroups its latency is hidden, which a parallel exact evaluation
// per row is not worth here.  inv[n * H + h] = 1 / sum.
constexpr int kTileSpan = 256, kTileWaves = 8;
__global__ __launch_bounds__(64 * (kTileWaves + 1)) void attn_tile_softmax_kernel(AttnParams a, float* inv) {
    __shared__ __align__(16) float et[2][16][kTileSpan + 4];
    const int lane = threadIdx.x & 63, w = wave_id_uniform();
    const int kvh = blockIdx.x % a.Hkv, tile = blockIdx.x / a.Hkv;
    const int pos0 = a.d_pos[0];
    const TileQuery qa = tile_query(a, kvh, 16 * tile), qz = tile_query(a, kvh, 16 * tile + 15);
    const int longest = pos0 + (qa.h == qz.h ? qz.n : a.N - 1) + 1;
    constexpr int RW = 16 / kTileWaves;  // rows per wave
    float* row[RW];
    int len[RW];
    float mx[RW];
    if (w < kTileWaves) {
#pragma unroll
        for (int i = 0; i < RW; i++) {
            const TileQuery q = tile_query(a, kvh, 16 * tile + RW * w + i);
            row[i] = a.scores + ((size_t)q.n * a.H + q.h) * a.max_ctx;
            len[i] = q.live ? pos0 + q.n + 1 : 0;  // 0: a clamped query writes nothing
            float m = -__builtin_inff();
            for (int p = 4 * lane; p < len[i]; p += kTileSpan) {  // rows are padded to whole quads
                const t_v4f s = *(const t_v4f*)(row[i] + p);
#pragma unroll
                for (int e = 0; e < 4; e++) m = p + e < len[i] && s[e] > m ? s[e] : m;
            }
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) {
                const float o = __shfl_xor(m, off, 64);
                m = o > m ? o : m;
            }
            mx[i] = m;
        }
    }
    float sum = 0.0f;
    const int nspan = (longest + kTileSpan - 1) / kTileSpan;
    for (int b = 0; b <= nspan; b++) {
        if (w < kTileWaves) {
            if (b < nspan) {
                const int p = b * kTileSpan + 4 * lane;
#pragma unroll
                for (int i = 0; i < RW; i++) {
                    t_v4f e = {0.0f, 0.0f, 0.0f, 0.0f};
                    if (p < len[i]) {
                        const t_v4f s = *(const t_v4f*)(row[i] + p);
#pragma unroll
                        for (int k = 0; k < 4; k++) e[k] = p + k < len[i] ? expf_glibc(s[k] - mx[i]) : 0.0f;
                        *(t_v4f*)(row[i] + p) = e;
                    }
                    *(t_v4f*)&et[b & 1][RW * w + i][4 * lane] = e;
                }
            }
        } else if (b > 0 && lane < 16) {
            const float* src = et[(b - 1) & 1][lane];
#pragma unroll 4
            for (int k = 0; k < kTileSpan; k += 4) {
                const t_v4f e = *(const t_v4f*)(src + k);
                sum = sum + e.x;
                sum = sum + e.y;
                sum = sum + e.z;
                sum = sum + e.w;
            }
        }
        __syncthreads();
    }
    if (w == kTileWaves && lane < 16) {
        const TileQuery q = tile_query(a, kvh, 16 * tile + lane);
        if (q.live) inv[q.n * a.H + q.h] = 1.0f / sum;
    }
}

// Weighted V sum and the Q8_0 quantisation of the output.  Workgroup = one query tile, wave w = output
// dims 16w..16w+15.  MFMA operands of positions 16 P + 4 j + e: A lane (j, r) = prob of query r, B lane (j, c) =
// value dim c (value position quads [ctx/4][hd][4]).  A ring of 4 steps of loads is in flight; a step past the cache
// loads its last one (max_ctx is a multiple of 16) and is not added.
template <int HD>
__global__ __launch_bounds__(4 * HD, 4) void attn_tile_pv_kernel(AttnParams a, const float* inv) {
    __shared__ __align__(16) float out[16][HD + 4];
    const int lane = threadIdx.x & 63, w = wave_id_uniform();
    const int j = lane >> 4, r = lane & 15;
    const int kvh = blockIdx.x % a.Hkv, tile = blockIdx.x / a.Hkv;
    const int pos0 = a.d_pos[0];
    const TileQuery qa = tile_query(a, kvh, 16 * tile), qz = tile_query(a, kvh, 16 * tile + 15);
    const bool one_head = qa.h == qz.h;
    const int shortest = pos0 + (one_head ? qa.n : 0) + 1, longest = pos0 + (one_head ? qz.n : a.N - 1) + 1;
    const TileQuery q = tile_query(a, kvh, 16 * tile + r);
    const int row = q.n * a.H + q.h;
    const float iv = inv[row];
    int len[4];  // row lengths of the lane's results, queries 4j + v
#pragma unroll
    for (int v = 0; v < 4; v++) len[v] = pos0 + tile_query(a, kvh, 16 * tile + 4 * j + v).n + 1;
    const float* prow = a.scores + (size_t)row * a.max_ctx + 4 * j;
    const __amdgpu_buffer_rsrc_t vres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.vcache + (size_t)kvh * a.max_ctx * HD), 0, a.max_ctx * HD * 4, 0x00020000);
    const int vvo = (j * HD + 16 * w + r) * 16;
    const int steps = (longest + 15) / 16;
    constexpr int D = 4;
    t_v4f rp[D], rv[D];
#define NC_TILE_LOAD(S, SLOT)                                                                                  \
    {                                                                                                          \
        const int s_ = kv_step((S), a.max_ctx);                                                                \
        rp[SLOT] = *(const t_v4f*)(prow + 16 * s_);                                                            \
        rv[SLOT] = __builtin_bit_cast(t_v4f, __builtin_amdgcn_raw_buffer_load_b128(vres, vvo, s_ * HD * 64, 0)); \
    }
#pragma unroll
    for (int k = 0; k < D - 1; k++) NC_TILE_LOAD(k, k)
    t_v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const t_v16f zero = {};
    for (int s0 = 0; s0 < steps; s0 += D) {
#pragma unroll
        for (int k = 0; k < D; k++) {
            const int s = s0 + k;
            if (s >= steps) break;  // uniform
            NC_TILE_LOAD(s + D - 1, (k + D - 1) % D)
            const t_v4f p = rp[k] * iv;
            t_v16f d[4];
#pragma unroll
            for (int e = 0; e < 4; e++) d[e] = __builtin_amdgcn_mfma_f32_16x16x1f32(p[e], rv[k][e], zero, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (16 * s + 16 <= shortest) {
                tile_add16(acc, d);
            } else {
                // positions past a row leave its sum unchanged (a select: later cache rows hold any bits)
#pragma unroll
                for (int jj = 0; jj < 4; jj++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
#pragma unroll
                        for (int v = 0; v < 4; v++) {
                            const float n = acc[v] + d[e][4 * jj + v];
                            acc[v] = 16 * s + 4 * jj + e < len[v] ? n : acc[v];
                        }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#undef NC_TILE_LOAD
#pragma unroll
    for (int v = 0; v < 4; v++) out[4 * j + v][16 * w + r] = acc[v];
    __syncthreads();
    // quantize_f32_to_q8_0 (inference.rs:1012-1029): 8 lanes per 32-block, 4 values per lane, one item each
    const int qr = threadIdx.x / (HD / 4), c4 = threadIdx.x % (HD / 4) * 4;
    const TileQuery o = tile_query(a, kvh, 16 * tile + qr);
    const t_v4f y = *(const t_v4f*)&out[qr][c4];
    float amax = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; e++) amax = __builtin_fabsf(y[e]) > amax ? __builtin_fabsf(y[e]) : amax;
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) {
        const float m = __shfl_xor(amax, off, 8);
        amax = m > amax ? m : amax;
    }
    float scale = 0.0f;
    int qs = 0;
    uint32_t packed = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int v = quantize_lane_q8(y[e], amax, &scale);
        qs += v;
        packed |= (uint32_t)(v & 0xff) << (8 * e);
    }
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) qs += __shfl_xor(qs, off, 8);
    if (o.live) {
        const size_t at = (size_t)o.n * a.H * HD + (size_t)o.h * HD + c4;
        *(uint32_t*)(a.xq + at) = packed;
        if ((threadIdx.x & 7) == 0) {
            a.xs[at / 32] = scale;
            a.xs8[at / 32] = -8 * qs;
        }
    }
}

template <int PT>
static void launch_scores(const AttnParams& a, hipStream_t st) {
    const int tiles = (a.H / a.Hkv * a.N + 15) / 16;
    // position groups rounded up to 512 positions, so that one grid serves a captured pass at 512
    // consecutive positions (a workgroup past the rows ends at once)
    const dim3 grid(a.Hkv * tiles, (a.max_pos + 512) / 512 * (512 / (64 * PT)));
    if (a.hd == 128) NC_LAUNCH((attn_tile_scores_kernel<128, PT>), grid, dim3(256), 0, st, a);
    else NC_LAUNCH((attn_tile_scores_kernel<64, PT>), grid, dim3(256), 0, st, a);
}

// 64 PT positions a workgroup: more of them spread the loads of the queries and leave a tile's waves in
// step, as long as the launch fills the chip.  8 KV heads, head dim 128, us at PT 1 / 2 / 4: 1280 groups at
// PT 4 (72 queries a KV head, 8180 positions) 41.9 / 35.8 / 32.7; 512 groups at PT 2 (16 queries) 13.4 / 11.7;
// 160 groups at PT 2 (8 queries, 2500 positions) 5.9 / 8.2.
int launch_attention_scores(const AttnParams& a, hipStream_t st) {
    if (a.max_ctx % 16 || a.max_pos >= a.max_ctx)
        return fail(NC_EINVAL, "attention: cache rows must be whole 16-position tiles that hold the pass");
    const int64_t g1 = (int64_t)a.Hkv * ((a.H / a.Hkv * a.N + 15) / 16) * ((a.max_pos + 512) / 512 * 8);
    if (g1 >= 4 * 1024) launch_scores<4>(a, st);
    else if (g1 >= 2 * 512) launch_scores<2>(a, st);
    else launch_scores<1>(a, st);
    NC_HIP(hipGetLastError());
    return NC_OK;
}

int launch_attention_tiles(const AttnParams& a, hipStream_t st) {
    const dim3 grid(a.Hkv * ((a.H / a.Hkv * a.N + 15) / 16));
    if (int rc = launch_attention_scores(a, st)) return rc;
    NC_LAUNCH(attn_tile_softmax_kernel, grid, dim3(64 * (kTileWaves + 1)), 0, st, a, a.inv);
    if (a.hd == 128) NC_LAUNCH((attn_tile_pv_kernel<128>), grid, dim3(512), 0, st, a, a.inv);
    else NC_LAUNCH((attn_tile_pv_kernel<64>), grid, dim3(256), 0, st, a, a.inv);
    NC_HIP(hipGetLastError());
    return NC_OK;
}

}  // namespace nc
