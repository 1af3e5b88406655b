"""Quantised matmuls at the edges of their tiles: ragged rows, columns that cut the super-block
quads and block groups, every token-group size and prompt slices, bit-exact against the oracle (which
evaluates the reference's per-row chains left to right)."""
import numpy as np
import pytest

import nanocamelid_amd as nc
from oracle import oracle as O
from tests import gguf_writer as GW
from tests.gpu_util import q8_activations, random_q4_0, random_q4_k, random_q5_k, random_q8_0

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return nc.Context(0)


def check(ctx, qtype, w, ref, M, K, batches, seed):
    import torch
    qm = nc.QMat(ctx, qtype, M, K, w)
    for N in batches:
        _, xq, xs = q8_activations(N, K, seed + N)
        xq.reshape(-1)[:5] = [-128, 127, 0, -1, 1]  # the operator takes any int8
        out = torch.full((N, M), float("nan"), device="cuda")
        nc.matmul_quantized_batch(ctx, qm, torch.from_numpy(xq).cuda(), torch.from_numpy(xs).cuda(), out=out)
        got = out.cpu().numpy()
        want = ref(xq, xs, w, N, M, K, nthreads=8)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (M, K, N)
    qm.close()


# K: one super-block, a cut quad (2, 5), a whole one and more quads than waves; N: every token-group
# size 1..8, two and three uneven groups, prompt slices
@pytest.mark.parametrize("M,K", [(1, 256), (17, 512), (100, 1280), (64, 1024), (33, 9472), (16, 16384)])
def test_q6_k_tile_edges(ctx, M, K):
    w = GW.q6_k_weights(M * K // 256, seed=M + K).reshape(M, K // 256, 210)
    check(ctx, nc._ffi.NC_TYPE_Q6_K, w, O.matmul_q6_k, M, K, [1, 2, 3, 4, 5, 6, 7, 8, 9, 16, 17, 50], 3)


# more workgroups than one grid of 256-thread workgroups holds: the batch takes several launches, and its first
# and last rows and those around their boundary are what the same rows give in a small batch
def test_q6_k_batch_past_one_grid(ctx):
    import torch
    M, K, N = 131072, 2304, 16400
    if torch.cuda.mem_get_info()[0] < 24 << 30:
        pytest.skip("needs 24 GB of free device memory")
    w = np.tile(GW.q6_k_weights(1024 * K // 256, seed=11).reshape(1024, K // 256, 210), (M // 1024, 1, 1))
    qm = nc.QMat(ctx, nc._ffi.NC_TYPE_Q6_K, M, K, w)
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randint(-127, 128, (N, K), dtype=torch.int8, device="cuda", generator=g)
    s = torch.rand(N, K // 32, device="cuda", generator=g)
    out = nc.matmul_quantized_batch(ctx, qm, x, s)
    for lo in (0, 8176, 8184, 8192, N // 2, N - 9):
        some = nc.matmul_quantized_batch(ctx, qm, x[lo:lo + 9], s[lo:lo + 9])
        assert torch.equal(out[lo:lo + 9].view(torch.int32), some.view(torch.int32)), lo
    qm.close()


# K: one block, a cut quad, a whole one, a cut chunk of 8 quads, 12 term waves (>= 64 quads); N: every width
# the kernel is built for, both widths with their chains on term waves (9, 16) and a cut 16-token slice
@pytest.mark.parametrize("M,K", [(1, 32), (17, 96), (100, 1024), (64, 1120), (33, 8224), (1040, 64)])
def test_q8_0_tile_edges(ctx, M, K):
    w = random_q8_0(M, K, seed=M + K)
    check(ctx, nc.NC_TYPE_Q8_0, w, O.matmul_q8_0, M, K, [1, 2, 3, 4, 5, 6, 7, 8, 9, 16, 17, 50], 4)


# the prompt matmuls' workgroups: 64 rows x 16, 32 or 64 tokens (one, two or four token tiles a wave), by how many a
# launch has.  K: one unit, cut quads, an odd number of quads; ragged rows and tokens.  K-quants: one tile up to 200 rows
# and at 40 and 4 (of 260) tokens of 16000, two at 66 to 260 tokens of 16000 and more, on 64-row tiles from 16321
# rows four at 200 and 256 tokens and, for the 257th token alone, one.  (Four on 16-row tiles needs an
# interleaved gate,up: test_prompt_pass_of_a_wide_q4_k_gateup.)
@pytest.mark.parametrize("qtype", ["q4_k", "q5_k"])
@pytest.mark.parametrize("M,K,batches", [(17, 256, [17, 33, 64]), (200, 1280, [40, 130, 300]),
                                         (16401, 512, [129, 66, 200, 257]), (16000, 256, [260, 40])])
def test_prompt_k_quant_matmul_wave_tiles(ctx, qtype, M, K, batches):
    if qtype == "q4_k":
        check(ctx, nc.NC_TYPE_Q4_K, random_q4_k(M, K, seed=M), O.matmul_q4_k, M, K, batches, 9)
    else:
        check(ctx, nc.NC_TYPE_Q5_K, random_q5_k(M, K, seed=M), O.matmul_q5_k, M, K, batches, 10)


# Q4_0 and Q8_0: one token tile up to 200 rows, two at 20 tokens of 32785, four at 66 tokens and more of 16401; Q4_0 on
# 64-row tiles from 65473 rows: two at 20 tokens, four at 65 and 256, one for the 257th token alone
@pytest.mark.parametrize("qtype", ["q4_0", "q8_0"])
@pytest.mark.parametrize("M,K,batches", [(17, 32, [17, 33, 64]), (200, 416, [40, 130, 300]), (16401, 96, [129, 66]),
                                         (32785, 288, [130, 20]), (65553, 96, [20, 65, 257]), (20, 8224, [31, 49])])
def test_prompt_block_matmul_wave_tiles(ctx, qtype, M, K, batches):
    if qtype == "q4_0":
        check(ctx, nc.NC_TYPE_Q4_0, random_q4_0(M, K, seed=M), O.matmul_q4_0, M, K, batches, 5)
    else:
        check(ctx, nc.NC_TYPE_Q8_0, random_q8_0(M, K, seed=M), O.matmul_q8_0, M, K, batches, 6)


# K-quant matrices on 16-row tiles (and from 16321 rows on 64-row ones): one super-block, cut quads, every wave count
# (4; 8 from 29 super-blocks at up to 4096 rows; 1 and 2 for one and two quads at more than 8192), operator calls whose
# kernel sums the activations itself and, at 16 tokens of a long row, ones that take a separate launch
@pytest.mark.parametrize("qtype", ["q4_k", "q5_k"])
@pytest.mark.parametrize("M,K", [(1, 256), (17, 1280), (100, 768), (40, 7680), (33, 8192), (4113, 7424), (8209, 768),
                                 (8209, 1280), (16400, 256)])
def test_k_quant_tile_edges(ctx, qtype, M, K):
    batches = [1, 2, 3, 4, 5, 6, 7, 8, 9, 16, 18]
    if qtype == "q4_k":
        check(ctx, nc.NC_TYPE_Q4_K, random_q4_k(M, K, seed=M + K), O.matmul_q4_k, M, K, batches, 7)
    else:
        check(ctx, nc.NC_TYPE_Q5_K, random_q5_k(M, K, seed=M + K), O.matmul_q5_k, M, K, batches, 8)


# the K-quant prompt matmul's values are f16 subnormals and its scales carry the 2^24: super-block scales at the ends
# of f16's range, subnormal, zero and negative
@pytest.mark.parametrize("qtype", ["q4_k", "q5_k"])
def test_prompt_k_quant_extreme_scales(ctx, qtype):
    M, K = 80, 768
    w = random_q4_k(M, K, seed=31) if qtype == "q4_k" else random_q5_k(M, K, seed=31)
    bits = np.array([0x0001, 0x03ff, 0x0400, 0x7bff, 0x8001, 0x83ff, 0xfbff, 0x0000, 0x8000, 0x3c00], np.uint16)
    pick = np.random.default_rng(32).integers(0, len(bits), (M, K // 256, 2))
    w[:, :, 0:4] = np.ascontiguousarray(bits[pick]).view(np.uint8).reshape(M, K // 256, 4)
    t, ref = (nc.NC_TYPE_Q4_K, O.matmul_q4_k) if qtype == "q4_k" else (nc.NC_TYPE_Q5_K, O.matmul_q5_k)
    check(ctx, t, w, ref, M, K, [18, 40], 33)


# Q8_0 calls of more than 16 tokens share no scratch with any other call: on two streams at once, beside Q4_0 ones
# on a third, and replayed from a graph, every output is the one that the same call gives alone
def test_q8_0_prompt_matmul_on_several_streams():
    import torch
    M, K, N, reps = 4096, 2048, 100, 12
    ctx = nc.Context(0)
    q8 = nc.QMat(ctx, nc.NC_TYPE_Q8_0, M, K, random_q8_0(M, K, seed=12))
    q4 = nc.QMat(ctx, nc.NC_TYPE_Q4_0, M, K, random_q4_0(M, K, seed=13))
    calls = [(w, *[torch.from_numpy(a).cuda() for a in q8_activations(N, K, 20 + i)[1:]]) for i, w in enumerate((q8, q8, q4, q8))]
    streams = [torch.cuda.Stream() for _ in calls]
    torch.cuda.synchronize()
    with torch.cuda.stream(streams[0]):  # the first stream: the one with the buffers
        want = [nc.matmul_quantized_batch(ctx, w, x, s) for w, x, s in calls]
    got = [[torch.zeros_like(want[0]) for _ in range(reps)] for _ in calls]
    captured = torch.zeros_like(want[0])
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=streams[3]):
        nc.matmul_quantized_batch(ctx, *calls[3], out=captured)
    for j in range(reps):
        for i in range(3):
            with torch.cuda.stream(streams[i]):
                nc.matmul_quantized_batch(ctx, *calls[i], out=got[i][j])
        with torch.cuda.stream(streams[3]):
            captured.zero_()
            graph.replay()
            got[3][j].copy_(captured)
    torch.cuda.synchronize()
    for i in range(4):
        for j in range(reps):
            assert torch.equal(got[i][j].view(torch.int32), want[i].view(torch.int32)), (i, j)
    q8.close()
    q4.close()
