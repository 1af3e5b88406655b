"""The allocation-free matmul entry point (nc_matmul_quantized_batch_noalloc) against the
allocating one, through the C ABI: two calls in a row, the second smaller, bit-identical."""
import ctypes as C

import numpy as np
import pytest

from tests import gguf_writer as GW
from tests.gpu_util import q8_activations, random_q4_0, random_q4_k, random_q5_k, random_q8_0

torch = pytest.importorskip("torch")


@pytest.mark.gpu
def test_noalloc_matmul_matches_allocating_entry():
    import nanocamelid_amd as nc
    from nanocamelid_amd._ffi import NC_ERANGE, NcError, check, lib
    ctx = nc.Context(0)
    for M, K, N in ((4096, 14336, 9), (1024, 4096, 3)):  # the second call is smaller
        print(f"noalloc matmul {M}x{K} N={N}", flush=True)
        w = nc.QMat(ctx, nc.NC_TYPE_Q4_0, M, K, random_q4_0(M, K, seed=M + N))
        _, q, s = q8_activations(N, K, seed=N)
        xq = torch.from_numpy(q).cuda()
        xs = torch.from_numpy(s).cuda()
        ref = nc.matmul_quantized_batch(ctx, w, xq, xs)
        out = torch.full((N, M), float("nan"), dtype=torch.float32, device="cuda")
        stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        check(lib().nc_matmul_quantized_batch_noalloc(ctx.h, w.h, xq.data_ptr(), xs.data_ptr(), out.data_ptr(), N, M,
                                                       K, stream))
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy().view(np.uint32), ref.cpu().numpy().view(np.uint32)), (M, K, N)
    # beyond the static scratch: refused before any launch
    big = nc.QMat(ctx, nc.NC_TYPE_Q4_0, 16, 131072, random_q4_0(16, 131072, seed=1))
    xq = torch.zeros((16, 131072), dtype=torch.int8, device="cuda")
    xs = torch.zeros((16, 4096), dtype=torch.float32, device="cuda")
    out = torch.empty((16, 16), dtype=torch.float32, device="cuda")
    rc = lib().nc_matmul_quantized_batch_noalloc(ctx.h, big.h, xq.data_ptr(), xs.data_ptr(), out.data_ptr(), 16, 16,
                                                 131072, None)
    assert rc == NC_ERANGE


# every type, with and without block sums: K-quants on 16-row tiles sum for themselves unless the row is long
# (16 tokens of 65536 columns), those on 64-row tiles (16400 rows) and Q4_0 on the MFMA path read the scratch array
@pytest.mark.gpu
@pytest.mark.parametrize("qtype,M,K,N,mfma", [("q4_0", 40, 1024, 5, True), ("q8_0", 40, 1024, 16, False),
                                              ("q6_k", 40, 1024, 16, False), ("q4_k", 40, 1024, 7, False),
                                              ("q5_k", 40, 1024, 16, False), ("q4_k", 16, 65536, 16, False),
                                              ("q4_k", 16400, 512, 3, False), ("q5_k", 16400, 512, 3, False)])
def test_noalloc_matmul_of_every_type(qtype, M, K, N, mfma):
    import nanocamelid_amd as nc
    from nanocamelid_amd._ffi import NC_GEMM_KERNEL_MFMA, NC_TYPE_Q6_K, check, lib
    ctx = nc.Context(0)
    t, blocks = {"q4_0": (nc.NC_TYPE_Q4_0, random_q4_0), "q8_0": (nc.NC_TYPE_Q8_0, random_q8_0),
                 "q4_k": (nc.NC_TYPE_Q4_K, random_q4_k), "q5_k": (nc.NC_TYPE_Q5_K, random_q5_k),
                 "q6_k": (NC_TYPE_Q6_K, lambda m, k, seed: GW.q6_k_weights(m * k // 256, seed))}[qtype]
    w = nc.QMat(ctx, t, M, K, blocks(M, K, seed=M + N))
    _, q, s = q8_activations(N, K, seed=N)
    xq, xs = torch.from_numpy(q).cuda(), torch.from_numpy(s).cuda()
    ref = nc.matmul_quantized_batch(ctx, w, xq, xs)
    if mfma:
        ctx.set_gemm_kernel(NC_GEMM_KERNEL_MFMA)
    out = torch.full((N, M), float("nan"), dtype=torch.float32, device="cuda")
    check(lib().nc_matmul_quantized_batch_noalloc(ctx.h, w.h, xq.data_ptr(), xs.data_ptr(), out.data_ptr(), N, M, K,
                                                  None))
    check(lib().nc_ctx_synchronize(ctx.h))
    assert torch.equal(out.view(torch.int32), ref.view(torch.int32))
