"""Every buffer load of the prompt matmuls and the tiled attention lies inside its buffer, whatever the
range check of a raw buffer load covers: the offsets (nc_offsets.h, the functions the kernels use) are
walked on the host in the kernels' loop order, prefetched stages and token tiles past the last ones
included, and compared with the bytes the host allocates.  The slices of a large Q6_K batch fit a grid.
"""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

WALK = r"""
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
#include "nc_offsets.h"
using namespace nc;

static void inside(const char* what, long long offset, long long bytes, long long end, int a, int b) {
    if (offset >= 0 && offset + bytes <= end) return;
    std::printf("%s: %lld + %lld past %lld (%d, %d)\n", what, offset, bytes, end, a, b);
    std::exit(1);
}

// activations of n tokens and nb blocks a row: units and scales, and the row tile's weights
static void prompt(int n, int nb, int KT, int WD, int SD, bool k_quant) {
    const int n16 = (n + 15) / 16, nq = (nb + 3) / 4, tg = (n16 + KT - 1) / KT;
    const long long units = (long long)n16 * nq * 4096, scales = (long long)n16 * nq * 256;
    for (int tt = 0; tt < tg * KT; tt += KT)
        for (int s = 0; s < nq + (WD > SD ? WD : SD) + WD; s++)  // no prologue or turn of the ring asks for more
            for (int k = 0; k < KT; k++) {
                const int u = prompt_unit(tt + k, s, n16, nq);
                inside("units", (long long)u * 4096, 4096, units, n, nb);
                inside("scales", (long long)u * 256, 256, scales, n, nb);
            }
    for (int s = 0; s < nq + 2 * WD; s++) {
        if (!k_quant) {
            for (int quad : {1152, 2176})  // Q4_0 and Q8_0 16-row tiles: chunks of 8 quads
                inside("r16 weights", prompt_r16_quad(s, nq, quad), quad, (nb + 31) / 32 * 8LL * quad, n, nb);
            const long long tile = (nb + 7) / 8 * 9216LL, chunk = prompt_r64_chunk(s, nq, 9216);
            inside("r64 nibbles", chunk + 4096 * prompt_r64_half(s, nq), 4096, tile, n, nb);
            inside("r64 scales", chunk + 8192 + 512 * prompt_r64_half(s, nq), 512, tile, n, nb);
        } else {
            for (int slots : {9, 11}) {
                const int chunk = 1024 * slots, qs = slots - 8, nsb = nb / 8;
                for (bool r16k : {false, true}) {
                    const long long tile = r16k ? (nsb + 3) / 4 * (long long)chunk : nsb * (long long)chunk;
                    const long long at = prompt_k_chunk(r16k, s, nq, chunk);
                    // a lane's bytes: 16 rows (R16K) or one of four row quarters of 64 rows (R64) of 16 bytes
                    const int lanes = r16k ? 256 : 1024;
                    inside("K header", at, lanes, tile, n, nb);
                    inside("K nibbles", at + (qs + 4 * prompt_k_half(s, nq) + 3) * 1024, lanes, tile, n, nb);
                }
            }
        }
    }
}

static void attention(int max_ctx, int hd) {
    const int ctx = (int)kv_positions(max_ctx);
    const long long end = (long long)ctx * hd * 4;  // of a KV head, and ctx floats of a score row
    if (ctx < max_ctx) inside("positions", ctx, 1, max_ctx, max_ctx, hd);
    for (int last = 0; last < max_ctx; last++)  // the last position of a pass
        if (last < 64 || last > max_ctx - 64) {
            const int pt = last / 16 * 16;  // the last 16-position tile of keys, the last dim quads
            const int quad = ctx * 16;      // bytes between dim quads
            inside("keys", (long long)(pt + 15) * 16 + 3LL * quad + 4LL * (hd / 16 - 1) * quad, 16, end, last, ctx);
            for (int s = last / 16; s < last / 16 + 1 + 2 * 4; s++) {  // a ring of 4 steps
                inside("values", (long long)kv_step(s, ctx) * hd * 64, hd * 64, end, last, ctx);
                inside("probabilities", 64LL * kv_step(s, ctx), 64, 4LL * ctx, last, ctx);
            }
        }
}

// rows x tokens in launches of q6k_launch_tokens: every grid below 2^32 threads, no more launches than needed
static void q6k(long long rows, long long tokens) {
    const long long tiles = (rows + 15) / 16, most = q6k_launch_tokens(tiles);
    const long long n = tokens < most ? tokens : most;
    inside("Q6_K grid", 0, tiles * ((n + 7) / 8) * 512, 0xffffffffLL, (int)rows, (int)tokens);
    inside("outputs of the smallest first launch", 0, 1LL << 29, 16 * tiles * most, (int)rows, (int)tokens);
}

int main() {
    for (long long rows : {1, 17, 4096, 32000, 128256, 256000})
        for (long long tokens : {1, 16, 255, 8368, 16400, 1 << 20, 1 << 28}) q6k(rows, tokens);
    for (int n : {1, 2, 15, 16, 17, 31, 33, 48, 49, 64, 65, 113, 250, 256})
        for (int nb = 1; nb <= 200; nb += nb < 40 ? 1 : 7) {
            for (int KT : {1, 2, 4}) prompt(n, nb, KT, 2, KT == 1 ? 2 : 1, false);
            if (nb % 8 == 0)
                for (int KT : {1, 2, 4}) prompt(n, nb, KT, 2, KT == 1 ? 2 : 1, true);
        }
    for (int max_ctx = 1; max_ctx <= 400; max_ctx++)
        for (int hd : {64, 128}) attention(max_ctx, hd);
    for (int max_ctx : {2047, 2048, 2049, 8191, 8256, 16383, 16384})
        for (int hd : {64, 128}) attention(max_ctx, hd);
    return 0;
}
"""


def test_prefetched_loads_stay_inside_their_buffers(tmp_path):
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(WALK)
    subprocess.run(["g++", "-std=c++20", "-O1", "-I", os.path.join(ROOT, "nanocamelid_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
