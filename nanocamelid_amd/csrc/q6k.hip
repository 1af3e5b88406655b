// Q6_K x Q8_0 batch matmul on gfx950, for the Q6_K output projection that llama.cpp writes
// into most quantised files (its Q4_0 and Q4_K_M mixes among them).
//
// The reference's portable path (matmul_q6_k_batch, inference.rs:1882-2000, with
// Q6KBlock::dot_q8_scaled, q8.rs:2093-2150) sums every element's term in f32, in a fixed
// order, per 256-value super-block, then adds the super-block sums along the row:
//   ws[i] = d * sc[i];  c = ws[group] * x_scale[32-block]
//   block: s = 0; for half, for l in 0..32, for k in 0..4: s += (c * (float)q) * (float)x
//   row:   sum = 0; for b: sum += s_b
// So an (element, token) costs three f32 operations whatever the launch shape, and the super-block
// sums are independent: the kernel spreads those over lanes and waves and keeps everything else
// off the element loop.
//
// Bound: VALU issue.  At 128256 x 4096 and 5 tokens the 41 M (wave, element, token) steps take
// two full-rate operations and one DPP one (11.2 cycles for the three in a loop of nothing else, at
// any occupancy), 0.19 ms on 1024 SIMDs at 2.4 GHz, and unpacking the elements 0.03 ms, against 0.09 ms
// for the 0.43 GB of weights.  Lane (q, r) of a wave holds super-block
// 4 * quad + q of row r (a 16-row tile), so weights load as 1 KB per wave instruction, a
// 16-lane DPP row shares one super-block's activations, and v_mul_f32_dpp row_newbcast reads
// each value from the lane that converted it: no per-lane activation loads or conversions.
// Measured, 128256 x 4096 at 5 tokens: 254 us, where one lane per super-block with its own activation
// loads and conversions, on code for 8 tokens with a branch per token, took 1767 us.
//
// Device layout (repack_q6_k): rows padded to 16-row tiles, super-blocks to quads; per (tile, quad)
// 13 slots of [64 lanes x 16 B] (ql 8, qh 4, scales 1), then [64 lanes] f16 d.
#include "nc_internal.h"
#include "nc_device.h"
#include "nc_offsets.h"

namespace nc {

template <int J>
__device__ __forceinline__ float q6_bcast(float v) {  // lane J of each 16-lane row
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + J, 0xf, 0xf, true));
}

__device__ __forceinline__ float q6_byte(uint32_t v, int j) { return (float)(int8_t)(v >> (8 * j)); }

// Workgroup = one 16-row tile x NMAX tokens (blockIdx.x = tile * groups + token group, so the
// groups of a tile run close together and share its weights in cache); wave w takes quads w, w + W, ...
// A token past N repeats the last one and is not stored.
template <int NMAX, int W>
__global__ __launch_bounds__(64 * W) void gemm_q6_k_kernel(GemmParams p, int nb, int nquads, int groups) {
    extern __shared__ float sblk[];  // [4 * nquads][NMAX][16] super-block sums
    const int lane = threadIdx.x & 63, wave = wave_id_uniform();
    const int q = lane >> 4, r = lane & 15;
    const int tile = blockIdx.x / groups, n0 = (blockIdx.x % groups) * NMAX;
    const int N = p.N, K = p.K, nx = K / 32;
    const uint8_t* wt = p.w + (size_t)tile * nquads * kQ6KQuadBytes;
    for (int quad = wave; quad < nquads; quad += W) {
        const uint8_t* c0 = wt + (size_t)quad * kQ6KQuadBytes + lane * 16;
        const int b = min(4 * quad + q, nb - 1);  // a padded super-block's sum is not read
        const uint4 scv = *(const uint4*)(c0 + 12 * 1024);
        const float d = f16_to_f32(*(const uint16_t*)(c0 + 13 * 1024 - lane * 14));
        float s[NMAX];
#pragma unroll
        for (int t = 0; t < NMAX; t++) s[t] = 0.0f;
#pragma unroll 1
        for (int half = 0; half < 2; half++) {
            // lane r's eight activations 8r..8r+7 of the half (k = r / 4, l = 8 (r % 4) + e) and the
            // four x_scales, per token
            float xf[NMAX][8], xs4[NMAX][4];
#pragma unroll
            for (int t = 0; t < NMAX; t++) {
                const int n = min(n0 + t, N - 1);
                const uint2 xv = *(const uint2*)(p.x + (size_t)n * K + 256 * b + 128 * half + 8 * r);
                const float4 sv = *(const float4*)(p.xs + (size_t)n * nx + 8 * b + 4 * half);
                xs4[t][0] = sv.x; xs4[t][1] = sv.y; xs4[t][2] = sv.z; xs4[t][3] = sv.w;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    xf[t][e] = q6_byte(xv.x, e);
                    xf[t][4 + e] = q6_byte(xv.y, e);
                }
            }
            float ws[8];
            {
                const uint32_t s0 = half ? scv.z : scv.x, s1 = half ? scv.w : scv.y;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    ws[i] = d * q6_byte(s0, i);
                    ws[4 + i] = d * q6_byte(s1, i);
                }
            }
            uint32_t ql[16], qh[8];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint4 v = *(const uint4*)(c0 + (4 * half + i) * 1024);
                ql[4 * i] = v.x; ql[4 * i + 1] = v.y; ql[4 * i + 2] = v.z; ql[4 * i + 3] = v.w;
            }
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint4 v = *(const uint4*)(c0 + (8 + 2 * half + i) * 1024);
                qh[4 * i] = v.x; qh[4 * i + 1] = v.y; qh[4 * i + 2] = v.z; qh[4 * i + 3] = v.w;
            }
            // the half's 32 steps of l, eight at a time (l = 8 M + e): the activation of (k, l) sits in
            // lane 4k + M, register e
            auto eight = [&]<int M>(const float (&c)[NMAX][4]) {
#pragma unroll
                for (int e4 = 0; e4 < 2; e4++) {
                    const uint32_t lo = ql[2 * M + e4], l32 = ql[8 + 2 * M + e4], hb = qh[2 * M + e4];
                    // four elements' 6-bit values per dword, then - 32 per byte (no borrow between bytes)
                    uint32_t v[4] = {(lo & 0x0f0f0f0fu) | ((hb << 4) & 0x30303030u),
                                     (l32 & 0x0f0f0f0fu) | ((hb << 2) & 0x30303030u),
                                     ((lo >> 4) & 0x0f0f0f0fu) | (hb & 0x30303030u),
                                     ((l32 >> 4) & 0x0f0f0f0fu) | ((hb >> 2) & 0x30303030u)};
#pragma unroll
                    for (int k = 0; k < 4; k++) v[k] = ((v[k] | 0x80808080u) - 0x20202020u) ^ 0x80808080u;
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const int e = 4 * e4 + j;
                        const float qf[4] = {q6_byte(v[0], j), q6_byte(v[1], j), q6_byte(v[2], j), q6_byte(v[3], j)};
                        // two k at a time: products, then the DPP products, then the adds.  All four at
                        // once hold 20 more registers and took 216 -> 254 us at 4 tokens; left to the
                        // scheduler, which mixes the three, 5 tokens took 250 -> 297 us.
#pragma unroll
                        for (int k = 0; k < 4; k += 2) {
                            float pa[NMAX], pb[NMAX];
#pragma unroll
                            for (int t = 0; t < NMAX; t++) {
                                pa[t] = c[t][k] * qf[k];
                                pb[t] = c[t][k + 1] * qf[k + 1];
                            }
                            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                            for (int t = 0; t < NMAX; t++) {
                                pa[t] = (k ? q6_bcast<8 + M>(xf[t][e]) : q6_bcast<M>(xf[t][e])) * pa[t];
                                pb[t] = (k ? q6_bcast<12 + M>(xf[t][e]) : q6_bcast<4 + M>(xf[t][e])) * pb[t];
                            }
                            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                            for (int t = 0; t < NMAX; t++) s[t] = (s[t] + pa[t]) + pb[t];
                        }
                    }
                }
            };
            float c[NMAX][4];
#pragma unroll
            for (int t = 0; t < NMAX; t++)
#pragma unroll
                for (int k = 0; k < 4; k++) c[t][k] = ws[2 * k] * xs4[t][k];
            eight.template operator()<0>(c);
            eight.template operator()<1>(c);
#pragma unroll
            for (int t = 0; t < NMAX; t++)
#pragma unroll
                for (int k = 0; k < 4; k++) c[t][k] = ws[2 * k + 1] * xs4[t][k];
            eight.template operator()<2>(c);
            eight.template operator()<3>(c);
        }
#pragma unroll
        for (int t = 0; t < NMAX; t++) sblk[((4 * quad + q) * NMAX + t) * 16 + r] = s[t];
    }
    __syncthreads();
    // the rows' chains over their super-blocks: thread (token, row)
    for (int c = threadIdx.x; c < 16 * NMAX; c += 64 * W) {  // whole 16-lane groups
        const int t = c >> 4, rr = c & 15, n = n0 + t, row = tile * 16 + rr;
        float acc = 0.0f;
#pragma unroll 8
        for (int bb = 0; bb < nb; bb++) acc = acc + sblk[(bb * NMAX + t) * 16 + rr];
        if (n >= N) continue;  // uniform over the 16 lanes of a token
        if (row < p.M) p.out[(size_t)n * p.ld_out + row] = acc;
        if (p.epi == EPI_HEAD) {
            // the first maximum of the tile's rows (inference.rs:4836-4846): value, lower index on ties
            float bv;
            int bi;
            head_entry(acc, row, p.M, &bv, &bi);
#pragma unroll
            for (int off = 8; off >= 1; off >>= 1) {
                const float ov = __shfl_xor(bv, off, 64);
                const int oi = __shfl_xor(bi, off, 64);
                if (ov > bv || (ov == bv && oi < bi)) {
                    bv = ov;
                    bi = oi;
                }
            }
            if (rr == 0) {
                p.part_val[(size_t)n * p.ntiles + tile] = bv;
                p.part_idx[(size_t)n * p.ntiles + tile] = bi;
            }
        }
    }
}

int64_t q6k_layout_bytes(int64_t rows, int64_t cols) {
    return (rows + 15) / 16 * ((cols / 256 + 3) / 4) * kQ6KQuadBytes;
}

// Up to q6k_launch_tokens tokens: groups of at most 8 (the registers of one wave), as even as they come.
int launch_gemm_q6k(const QMatDev& w, const GemmParams& p0, hipStream_t st) {
    GemmParams p = p0;
    const int nb = (int)(w.cols / 256), nquads = (nb + 3) / 4;
    if (w.cols % 256 || nb < 1 || nb > 64) return fail(NC_EINVAL, "Q6_K matmul: cols must be 256..16384, multiple of 256");
    if (p.epi != EPI_STORE && p.epi != EPI_HEAD) return fail(NC_EINVAL, "Q6_K matmul: plain or head outputs only");
    if (p.N < 1) return fail(NC_EINVAL, "Q6_K matmul: batch must be >= 1");
    p.w = w.dev;
    p.M = (int)w.rows;
    p.K = (int)w.cols;
    p.ntiles = (int)w.tiles;
    const int groups = (p.N + kQ6KTokens - 1) / kQ6KTokens, per = (p.N + groups - 1) / groups;
    if (p.N > q6k_launch_tokens(w.tiles)) return fail(NC_ERANGE, "Q6_K matmul: rows x batch too large for one launch");
    // waves per workgroup: a power of two up to the quads of a row; four, so that a wave is a small part
    // of a SIMD's work and the last ones end together (128256 x 4096, one wave a group -> four: 119 ->
    // 98 us at 1 token, 32768 x 4096 at 5 tokens 82 -> 79 us), eight where the launch is short of four
    // waves per SIMD
    int W = 1;
    while (W < 8 && W < nquads && (W < 4 || w.tiles * groups * W < 4096)) W *= 2;
    const dim3 grid((unsigned)(w.tiles * groups));
    const size_t lds = (size_t)4 * nquads * per * 16 * sizeof(float);
#define NC_Q6K(NM)                                                                                                 \
    case NM:                                                                                                      \
        if (W == 1) NC_LAUNCH((gemm_q6_k_kernel<NM, 1>), grid, dim3(64), lds, st, p, nb, nquads, groups);          \
        else if (W == 2) NC_LAUNCH((gemm_q6_k_kernel<NM, 2>), grid, dim3(128), lds, st, p, nb, nquads, groups);    \
        else if (W == 4) NC_LAUNCH((gemm_q6_k_kernel<NM, 4>), grid, dim3(256), lds, st, p, nb, nquads, groups);    \
        else NC_LAUNCH((gemm_q6_k_kernel<NM, 8>), grid, dim3(512), lds, st, p, nb, nquads, groups);                \
        break
    switch (per) {
        NC_Q6K(1);
        NC_Q6K(2);
        NC_Q6K(3);
        NC_Q6K(4);
        NC_Q6K(5);
        NC_Q6K(6);
        NC_Q6K(7);
        NC_Q6K(8);
    }
#undef NC_Q6K
    NC_HIP(hipGetLastError());
    return NC_OK;
}

}  // namespace nc
