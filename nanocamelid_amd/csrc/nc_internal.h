// Host-side internals of libnanocamelid_hip (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <cstdint>
#include <cstdio>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/nanocamelid_gpu.h"

namespace nc {

// ---------------------------------------------------------------- errors
void set_error(const std::string& msg);
int fail(int code, const std::string& msg);

#define NC_HIP(call)                                                                   \
    do {                                                                               \
        hipError_t _e = (call);                                                        \
        if (_e != hipSuccess)                                                          \
            return ::nc::fail(NC_EHIP, std::string(#call) + ": " + hipGetErrorString(_e)); \
    } while (0)

// ---------------------------------------------------------------- stage timing
// While t_stage_ev1 is set (a session's stage timing), kernels launched through NC_LAUNCH are
// dispatched with events stamped by the dispatch itself: t_stage_ev0 records the first such
// kernel's start (and is then cleared), t_stage_ev1 every kernel's end, so the pair spans the
// kernels of one stage and nothing between launches.
extern thread_local hipEvent_t t_stage_ev0, t_stage_ev1;
#define NC_LAUNCH(K, G, B, L, S, ...)                                                          \
    do {                                                                                       \
        if (::nc::t_stage_ev1) {                                                               \
            hipExtLaunchKernelGGL(K, G, B, L, S, ::nc::t_stage_ev0, ::nc::t_stage_ev1, 0, __VA_ARGS__); \
            ::nc::t_stage_ev0 = nullptr;                                                       \
        } else {                                                                               \
            hipLaunchKernelGGL(K, G, B, L, S, __VA_ARGS__);                                    \
        }                                                                                      \
    } while (0)

// ---------------------------------------------------------------- weight layouts
// Q4_0 device layout ("tile-group"): rows padded to 64-row tiles; per (tile, group of 8
// blocks) a 9216-byte chunk = 8 x [64 lanes x 16 B nibbles] followed by the f16 scales as
// 2 x [64 lanes x 4 scales] (blocks 0-3, then 4-7).  Lane l of a wave loads row 64*tile + l;
// a round of 4 blocks reads 4 KB of nibbles and 512 contiguous bytes of scales.
constexpr int kTileRows = 64;
constexpr int kQ40GroupBlocks = 8;
constexpr int kQ40ChunkBytes = kQ40GroupBlocks * 1024 + 1024;  // 9216
// Q4_K device layout: per (tile, super-block) 9 x [64 lanes x 16 B]: slot 0 = d, dmin and
// the 12 packed scale bytes, slots 1..8 = the 128 nibble bytes.
constexpr int kQ4KChunkBytes = 9 * 1024;

// Q4_0 "R16" layout (matrices with fewer than 512 64-row tiles, so that a launch still
// spans every CU): rows padded to 16-row tiles; blocks taken in quads (block b = 4*qd + j)
// and groups of 8 quads.  Per (tile16, group) a 9216-byte chunk of 8 quads, each 1152 bytes:
// [64 lanes x 16 B nibbles] with lane = 16*j + r holding block 4*qd + j of row 16*tile + r,
// then the 64 f16 scales of the same blocks in [r / 4][j][r % 4] order.  One wave load covers
// 4 blocks x 16 rows and its scales are one contiguous 128-byte line.
constexpr int kTileRowsR16 = 16;
constexpr int kQ40R16QuadBytes = 1024 + 128;  // 1152; 8 per chunk = kQ40ChunkBytes
// Q8_0 layout: as R16 with 32 signed bytes per block: a quad is 2 x [64 lanes x 16 B] (a block's bytes
// 0-15, then 16-31) and the same 128-byte scale line; 8 quads per chunk.
constexpr int kQ80R16QuadBytes = 2048 + 128;
constexpr int kQ80ChunkBytes = 8 * kQ80R16QuadBytes;  // 32 blocks x 16 rows
__host__ __device__ constexpr int r16_quad_bytes(bool q8) { return q8 ? kQ80R16QuadBytes : kQ40R16QuadBytes; }
// Q6_K layout: 16-row tiles, super-blocks in quads; per (tile, quad) 13 x [64 lanes x 16 B] (lane
// 16*q + r = super-block 4*quad + q of row r: ql 8 slots, qh 4, scales 1), then [64 lanes] f16 d.
constexpr int kQ6KQuadBytes = 13 * 1024 + 128;
enum Layout : int { LAYOUT_R64 = 0, LAYOUT_R16 = 1, LAYOUT_R16K = 2, LAYOUT_Q6K = 3, LAYOUT_Q80 = 4 };  // R16K: Q4_K on 16-row tiles

struct QMatDev {
    int type = NC_TYPE_Q4_0;
    int layout = LAYOUT_R64;
    int64_t rows = 0, cols = 0;
    int64_t tiles = 0;       // padded rows / 64 (R16, R16K, Q8_0, Q6_K: / 16)
    int64_t units = 0;       // Q4_0, Q8_0: blocks per row; Q4_K: super-blocks per row
    int64_t groups = 0;      // Q4_0: ceil(blocks / 8) (R16, Q8_0: ceil(blocks / 32))
    uint8_t* dev = nullptr;  // repacked bytes
    int64_t dev_bytes = 0;
    int64_t algo_bytes = 0;  // rows * cols * 18/32 (Q4_0) or 144/256 (Q4_K)
};

// Repacks row-major GGUF blocks of `rows_src` rows into the device layout, writing tile
// rows [row_off, row_off + rows_src) of `dst` (host staging buffer of the whole matrix).
// interleave_pairs: rows_src rows are the gate half (tile lanes 0..31) or up half
// (lanes 32..63) of an interleaved SwiGLU matrix (half = 0 or 1), else -1.
void repack_q4_0(const uint8_t* src, int64_t rows_src, int64_t cols, uint8_t* dst, int64_t groups,
                 int64_t row_off, int half);
void repack_q4_k(const uint8_t* src, int64_t rows_src, int64_t cols, uint8_t* dst, int64_t row_off, int half,
                 int nslot = 9);
void repack_q4_0_r16(const uint8_t* src, int64_t rows_src, int64_t cols, uint8_t* dst, int64_t groups, int64_t row_off,
                     int half);
int64_t q40_r16_layout_bytes(int64_t rows, int64_t cols);
int64_t q40_layout_bytes(int64_t rows, int64_t cols);
int64_t q4k_layout_bytes(int64_t rows, int64_t cols);
int64_t q4k_r16_layout_bytes(int64_t rows, int64_t cols, int nslot = 9);
// Q4_K on 16-row tiles: per (tile, quad of 4 super-blocks) 9 x [64 lanes x 16 B], lane
// 16*q + r = super-block 4*quad + q of row r.  half >= 0: rows of an interleaved gate (0) or up
// (1) matrix, placed in 64-row groups as the Q4_0 repacks do.
int64_t q80_layout_bytes(int64_t rows, int64_t cols);
void repack_q8_0(const uint8_t* src, int64_t rows_src, int64_t cols, uint8_t* dst, int64_t groups, int64_t row_off,
                 int half);
void repack_q4_k_r16(const uint8_t* src, int64_t rows_src, int64_t cols, uint8_t* dst, int64_t groups,
                     int64_t row_off, int half = -1, int nslot = 9);

// ---------------------------------------------------------------- GEMM launch
enum Epi : int {
    EPI_STORE = 0,      // out[n*ld + row] = acc
    EPI_RESIDUAL = 1,   // out[n*ld + row] = acc + out[n*ld + row]
    EPI_QKV_ROPE = 2,   // RoPE on q/k rows, q -> q_out, k/v -> KV cache
    EPI_SWIGLU_Q8 = 3,  // silu(gate)*up then Q8_0 quantisation -> activations
    EPI_HEAD = 4,       // logits + per-tile argmax partials
};

struct GemmParams {
    const uint8_t* w = nullptr;
    int ntiles = 0, units = 0, groups = 0, M = 0, K = 0, N = 0;
    const int8_t* x = nullptr;     // [N][K]
    const float* xs = nullptr;     // [N][K/32]
    const int32_t* xs8 = nullptr;  // [N][K/32] -8 * (sum of the 32 int8 values of each block), or null
                                   // (only where the kernel reads no sums or makes its own)
    int epi = EPI_STORE;
    float* out = nullptr;
    int ld_out = 0;
    // EPI_QKV_ROPE
    float* q_out = nullptr;
    int aw = 0, kw = 0, hd = 0, rope_half = 0, max_ctx = 0, kv_heads = 0;
    const float* rope_tab = nullptr;  // [max_ctx][rope_half][2] = (sin, cos)
    float* kcache = nullptr;          // layer base of [kv_heads][hd/4][max_ctx][4] (dim quads)
    float* vcache = nullptr;          // layer base of [kv_heads][max_ctx/4][hd][4] (position quads)
    const int32_t* d_pos = nullptr;   // start position of row 0
    // EPI_SWIGLU_Q8
    int8_t* xq_out = nullptr;
    float* xs_out = nullptr;
    int32_t* xs8_out = nullptr;
    int F = 0;
    // EPI_HEAD
    float* part_val = nullptr;  // [N][ntiles]
    int32_t* part_idx = nullptr;
    int kernel = NC_GEMM_KERNEL_AUTO;  // dot-product path for 16-row tiles (nc_ctx_set_gemm_kernel)
};

// ev0/ev1: optional events stamped at the kernel's own start and end (timing).
int launch_gemm(const QMatDev& w, const GemmParams& p, hipStream_t stream, hipEvent_t ev0 = nullptr,
                hipEvent_t ev1 = nullptr);
// Waves of the 16-row K-quant kernel: 4, or 8 for rows of at least 8 quads of super-blocks in a launch of at most one
// workgroup a CU (more of them hold 12 waves a CU as four, 8 as eight: 16000 x 8192 at 1 / 5 tokens 20.3 / 34.8 us with
// eight, 15.5 / 24.5 with four).  Rows of one or two quads take one or two, as the others would only wait, from
// two workgroups a CU on, whose waves the idle ones keep out (5 tokens, four / these: 14000 x 1024 13.6 / 7.4 us,
// 16000 x 2048 15.3 / 9.9; with fewer workgroups the shorter chains and sums of four count: 8000 x 2048 at 16 tokens
// 14.9 / 15.7).
inline int q4k_r16_waves(const QMatDev& w) {
    return w.groups >= 8 && w.tiles <= 256 ? 8 : w.groups > 2 || w.tiles <= 512 ? 4 : (int)w.groups;
}
// Its LDS: two rounds of terms, and the activations' block sums when it makes its own.
inline size_t q4k_r16_lds_bytes(const QMatDev& w, int n, bool own_sums) {
    const size_t nmax = n <= 9 ? n : 16, S = q4k_r16_waves(w);
    return 2 * 4 * S * nmax * 16 * sizeof(float) + (own_sums ? (size_t)n * w.units * 8 * sizeof(float) : 0);
}
bool needs_block_sums(const nc_ctx* ctx, const QMatDev& q, int n);  // of an operator call of n <= 16 tokens
int launch_blockdots(const QMatDev& w, const int8_t* x, int32_t* dots, int N, hipStream_t stream);
// Q6_K matmul of up to q6k_launch_tokens tokens (plain outputs or the head's logits + argmax partials)
int launch_gemm_q6k(const QMatDev& w, const GemmParams& p, hipStream_t stream);
int64_t q6k_layout_bytes(int64_t rows, int64_t cols);

// ---------------------------------------------------------------- layer kernels
int launch_rmsnorm_q8(const float* hidden, const float* weight, int N, int d, float eps, int8_t* xq, float* xs,
                      int32_t* xs8, hipStream_t stream);
// Activation side buffers: xs = per-block f32 scale, xs8 = -8 * per-block int8 sum.
int launch_quantize_q8(const float* x, int N, int dim, int8_t* xq, float* xs, int32_t* xs8, hipStream_t stream);
int launch_expf_range(uint32_t first, int64_t count, float* out, hipStream_t stream);
int launch_block_sums(const int8_t* x, int N, int dim, int32_t* xs8, hipStream_t stream);
struct TokenArgs {
    uint32_t t[16];
};
// Writes d_pos[0] = pos and, when toks != NULL, d_toks[0..n) = toks (n <= 16).
int launch_set_pass_state(int32_t* d_pos, int32_t pos, uint32_t* d_toks, const uint32_t* toks, int n, hipStream_t st);
int launch_embed(const float* table, const uint32_t* toks, int N, int d, float* hidden, hipStream_t stream);
struct AttnParams {
    const float* q = nullptr;  // [N][H*hd]
    const float* kcache = nullptr;  // layer base [Hkv][hd/4][max_ctx][4]: 4 dims of a position per 16 B
    const float* vcache = nullptr;  // layer base [Hkv][max_ctx/4][hd][4]: 4 positions of a dim per 16 B
    float* scores = nullptr;  // [N][H][max_ctx]
    int8_t* xq = nullptr;     // [N][H*hd] quantised attention output
    float* xs = nullptr;
    int32_t* xs8 = nullptr;
    const int32_t* d_pos = nullptr;
    int N = 0, H = 0, Hkv = 0, hd = 0, max_ctx = 0, max_pos = 0;
    float scale = 0.f;
    float* inv = nullptr;     // [N][H] 1 / softmax sum (launch_attention_tiles; null: per-unit kernels only)
    // split-position order (NC_ATTN_SPLIT): per (row, head, 64-position chunk) partials
    bool split = false;
    float* part_o = nullptr;   // [N][H][nchunks][hd]
    float* part_ml = nullptr;  // [N][H][nchunks][2] chunk max, chunk sum of exp
    int nchunks = 0;
};
int launch_attention(const AttnParams& a, hipStream_t stream);
// The same outputs by tiles of 16 queries (attn_tile.hip), for passes with many (row, head) units.
int launch_attention_tiles(const AttnParams& a, hipStream_t stream);
int launch_attention_scores(const AttnParams& a, hipStream_t stream);  // a pass's scores, any number of units
// Launch variant of launch_attention: passes with equal values launch the same kernels with the
// same grids and blocks (the kernels read the rows' positions from d_pos, not from max_pos), so
// a captured pass replays correctly at every start position of its variant.
int64_t attention_variant(const AttnParams& a);

// ---------------------------------------------------------------- prompt (prefill) path
// Batch matmuls for any number of tokens on the matrix cores: out[n * ld_out + row] over the activations
// as f16 in operand order (launch_prompt_repack; xh: 16 * ceil(N/16) * prompt_cols(K) * 2 bytes, xsm and, for
// the K-quants only, xam: 16 * ceil(N/16) * prompt_cols(K) / 32 floats).
int launch_gemm_prompt(const QMatDev& w, float* out, int ld_out, int N, hipStream_t stream, const void* xh,
                       const float* xsm);  // Q4_0 (R16, R64), Q8_0
int launch_gemm_prompt_k(const QMatDev& w, float* out, int ld_out, int N, hipStream_t stream, const void* xh,
                         const float* xsm, const float* xam);  // Q4_K, Q5_K (R16K, R64)
int launch_prompt_repack(const int8_t* x, const float* xs, int N, int K, void* xh, float* xsm, hipStream_t stream,
                         float* xam = nullptr);
inline int64_t prompt_cols(int64_t cols) { return (cols + 127) / 128 * 128; }  // whole quads of blocks
// The verify GEMMs' epilogues as separate kernels over a prompt matmul's f32 output y.
int launch_prompt_qkv_rope(const float* y, int N, int start, int aw, int kw, int hd, int rope_half,
                           const float* rope_tab, float* q_out, float* kcache, float* vcache, int max_ctx,
                           hipStream_t stream);
int launch_prompt_residual(const float* y, float* hidden, int N, int d, hipStream_t stream);
int launch_prompt_swiglu_q8(const float* y, int N, int F, int8_t* xq, float* xs, int32_t* xs8, hipStream_t stream,
                            bool split = false);
constexpr int kPromptRows = 256;   // tokens per prompt pass
constexpr int kPromptMin = 32;     // shorter prompts run as verify-sized passes
int launch_argmax_final(const float* part_val, const int32_t* part_idx, int N, int ntiles, uint32_t* preds,
                        hipStream_t stream);
int launch_accept_greedy(const uint32_t* toks, const uint32_t* preds, int n, int32_t* d_pos, int32_t* result,
                         uint32_t* next_tok_slot, hipStream_t stream);

// ---------------------------------------------------------------- stochastic acceptance
// probs[r][j] = expf((l_j - max)/temp) * (1 / sum), the sum exact left to right (rows x V).
// Temperature probabilities of `rows` rows; scratch: temperature_scratch_floats(rows) floats of
// device memory owned by the caller (stream-ordered reuse), 256-byte aligned; the samplers below
// use its first part, so a sample may follow the probabilities it reads on the same stream.
size_t temperature_scratch_floats(int rows);
// sample_logits (inference.rs:4834-4873) of `rows` rows (<= kSampleMaxRows): temp > 0 draws row r
// with the uniform u[r] (the reference's inverse-CDF walk, bit-exact); temp <= 0 takes the first
// maximum.  probs: rows x ld_p floats of work (the rows' e_j), scratch as above; out: device ids.
constexpr int kSampleMaxRows = 17;
struct SampleUniforms {
    float u[kSampleMaxRows];
};
int launch_sample_logits(const float* logits, int64_t ld_in, int rows, int V, float temp, const float* u, float* probs,
                         int64_t ld_p, float* scratch, uint32_t* out, hipStream_t stream);
int launch_temperature_probs(const float* logits, int64_t ld_in, float* probs, int64_t ld_out, int rows, int V,
                             float temp, float* scratch, hipStream_t st);
// fast[r] (host) = which evaluation gave row r's sum in the last temperature pass on scratch.
int temperature_row_paths(const float* scratch, int rows, int32_t* fast, hipStream_t st);
// p [k+1][ld] target probs, q [k][ld] draft probs, drafts[k] (device); result = {n_accepted,
// next_token, start_pos + n_accepted + 1}; d_pos (nullable) receives the new position.
int launch_accept_stochastic(const float* p, const float* q, int64_t ld, const uint32_t* drafts, int k, int V,
                             uint64_t seed, int64_t start_pos, int32_t* result, int32_t* d_pos, float* scratch,
                             hipStream_t st);
// One fixed-point inverse-CDF sample of probs[V] with the Philox uniform (seed, pos, purpose).
int launch_sample_probs(const float* probs, int V, uint64_t seed, int64_t pos, uint32_t purpose, uint32_t* out0,
                        uint32_t* out1, float* scratch, hipStream_t st);

// Address of the allocation-free entry point's scratch array on the current device
// (hipGetSymbolAddress of a file-scope __device__ array; each device has its own copy).
int static_scratch_address(int32_t** out);
// Capacity of that array in int32 entries: per-block sums of up to 16 rows x 65536 columns.
constexpr size_t kStaticScratchInts = 16 * 65536 / 32;

}  // namespace nc

// ---------------------------------------------------------------- C ABI handles (opaque in the header)
struct nc_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    // Scratch of the operator-level entry points, allocated by nc_ctx_create for up to 16
    // rows of 65536 columns (every Llama projection); a larger call grows it once.
    int32_t* xsum = nullptr;  // -8 * per-block int8 sums of the activations
    size_t xsum_cap = 0;
    float* tp_scratch = nullptr;  // temperature softmax partials
    size_t tp_cap = 0;
    // activations of the prompt matmul (more than 16 tokens) repacked in MFMA operand order
    // with their scales and block sums, for kPromptRows tokens of 65536 columns per slice;
    // allocated by nc_ctx_create
    int8_t* pxm = nullptr;
    float* pxsm = nullptr;
    float* pxam = nullptr;
    // the same for Q8_0, whose calls need nothing of another call's: only those on the stream that asked
    // first use them, one launch sequence at a time (q8_mu); other streams take 16-token slices, which use none
    int8_t* q8_xm = nullptr;
    float* q8_xsm = nullptr;
    std::mutex q8_mu;
    hipStream_t q8_stream = nullptr;
    // device address of the static scratch array on this context's device (never freed)
    int32_t* static_scratch = nullptr;
    int gemm_kernel = NC_GEMM_KERNEL_AUTO;  // dot-product path of the quantized matmuls
    int attn_order = NC_ATTN_SEQUENTIAL;     // summation order of the verify passes' attention
    int pass_launch = NC_PASS_DIRECT;         // NC_PASS_GRAPH: session passes replayed from HIP graphs
};

struct nc_qmat {
    nc_ctx* ctx = nullptr;
    nc::QMatDev m;
};
