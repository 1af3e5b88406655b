// Offsets and launch limits that the kernels, their launches and a host check of their ranges share.
//
// Scalar (wave-uniform) parts of buffer-load offsets that run ahead of what is used.
// The range check of a raw buffer load is documented for the per-lane offset; the scalar one is not part of
// it on every reading of the rule, so no load here relies on it: a prefetched stage or step past the last
// one, or a token tile past the last one, takes the last one's place.  What it brings is never used.
#pragma once

#ifdef __HIP__
#define NC_HD __host__ __device__ __forceinline__
#else
#define NC_HD inline
#endif

namespace nc {

NC_HD constexpr int clamp_last(int i, int count) { return i < count ? i : count - 1; }

// Prompt matmuls: the (token tile, quad of blocks) index in the activations' [n16][nq] units and scales.
NC_HD constexpr int prompt_unit(int tile, int quad, int n16, int nq) {
    return clamp_last(tile, n16) * nq + clamp_last(quad, nq);
}
// Byte offset of a quad of blocks in a row tile's weights: chunks of 8 quads end to end (R16, Q8_0), or of
// two half-chunks whose nibbles lie 4096 bytes apart (R64; the scales' 512: prompt_r64_half).
NC_HD constexpr int prompt_r16_quad(int quad, int nq, int quad_bytes) { return clamp_last(quad, nq) * quad_bytes; }
NC_HD constexpr int prompt_r64_chunk(int quad, int nq, int chunk_bytes) { return (clamp_last(quad, nq) >> 1) * chunk_bytes; }
NC_HD constexpr int prompt_r64_half(int quad, int nq) { return clamp_last(quad, nq) & 1; }
// K-quants, half a super-block a stage: R16K chunks hold 4 super-blocks of a row tile, R64 chunks one.
NC_HD constexpr int prompt_k_chunk(bool r16k, int stage, int nq, int chunk_bytes) {
    const int sb = clamp_last(stage, nq) >> 1;
    return r16k ? (sb >> 2) * chunk_bytes + 256 * (sb & 3) : sb * chunk_bytes;
}
NC_HD constexpr int prompt_k_half(int stage, int nq) { return clamp_last(stage, nq) & 1; }

// Positions of a session's KV cache and score rows: whole 16-position tiles, so that a tile of positions
// or a 16-position step of values that begins inside the cache also ends inside it.
NC_HD constexpr long long kv_positions(long long max_ctx) { return (max_ctx + 15) / 16 * 16; }
// The 16-position step of a value or probability load, of ctx = kv_positions(...) positions.
NC_HD constexpr int kv_step(int step, int ctx) { return clamp_last(step, ctx / 16); }

// The Q6_K kernel's launches: a workgroup per 16-row tile and group of at most 8 tokens, of at most 512
// threads, where a grid holds fewer than 2^32 threads along x.  The most tokens of one launch; a batch
// beyond them (2^29 outputs at least) takes several.
constexpr int kQ6KTokens = 8, kQ6KThreads = 512;
NC_HD constexpr long long q6k_launch_tokens(long long tiles) {
    const long long groups = 0xffffffffLL / (kQ6KThreads * tiles);
    return kQ6KTokens * (groups < 1 ? 1 : groups);
}

}  // namespace nc
