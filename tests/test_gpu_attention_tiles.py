"""The tiled attention of passes with many (row, head) units, at the edges of its 16-query tiles and
16- and 256-position steps: bit-exact against the oracle's sequential attention."""
import numpy as np
import pytest

import nanocamelid_amd as nc
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# heads, KV heads, head dim and the chunk lengths of one prompt, each a pass of at least 1536 (head dim 128) or 2048
# (64) units, where the tiles begin: rows that cut a tile (49, 51, 101), tiles across two heads' rows, eight and one
# heads per KV head, starts off the 16- and 256-position steps
@pytest.mark.parametrize("H,Hkv,hd,chunks", [(32, 4, 128, [49, 70, 256, 51]), (32, 32, 128, [101, 48]),
                                             (32, 8, 64, [70, 190, 67, 256]), (64, 8, 64, [35, 33, 200])])
def test_tiled_attention_vs_oracle(H, Hkv, hd, chunks):
    ctx = nc.Context(0)
    spec = dict(layers=2, embedding_length=H * hd, head_count=H, head_count_kv=Hkv, feed_forward_length=256,
                vocab_size=300, context_length=1024, tied=1, norm_mode=1)
    img = nc.synth_gguf(**spec, seed=H + Hkv + hd)
    gs = nc.Session(nc.Model(ctx, data=img), sum(chunks) + 16, 16)
    os_ = O.Session(O.Model(data=img.tobytes(), nthreads=8), sum(chunks) + 16, 16)
    pos = 0
    for n in chunks:
        toks = nc.uniform_prompt(pos + n, n, 300)
        gs.prefill_pass_batch(toks, pos, want_logits=False)
        for i in range(0, n, 16):
            os_.prefill_pass_batch(toks[i:i + 16], pos + i)
        pos += n
    # layer 0's tiles feed layer 1's keys and values, which these logits read
    batch = nc.uniform_prompt(7, 5, 300)
    _, _, _, preds = gs.verify_greedy(batch, pos)
    opreds, _, ologits = os_.verify_greedy(batch, pos, want_logits=True)
    assert np.array_equal(preds, opreds)
    for i in range(5):
        assert np.array_equal(gs.logits(i).view(np.uint32), ologits[i].view(np.uint32)), i


def filled(H, Hkv, hd, start, end):
    """A two-layer model's session and the oracle's, both with the same keys and values before start."""
    ctx = nc.Context(0)
    img = nc.synth_gguf(layers=2, embedding_length=H * hd, head_count=H, head_count_kv=Hkv, feed_forward_length=256,
                        vocab_size=300, context_length=16384, tied=1, norm_mode=1, seed=H + Hkv + hd + start)
    gs = nc.Session(nc.Model(ctx, data=img), end, 16)
    os_ = O.Session(O.Model(data=img.tobytes(), nthreads=8), end, 16)
    gs.fill_kv(start, 9)
    os_.fill_kv(start, 9)
    return gs, os_


def verify_both(gs, os_, pos, rows):
    toks = nc.uniform_prompt(pos + rows, rows, 300)
    _, _, _, preds = gs.verify_greedy(toks, pos)
    opreds, _, ologits = os_.verify_greedy(toks, pos, want_logits=True)
    assert np.array_equal(preds, opreds)
    for i in range(rows):
        assert np.array_equal(gs.logits(i).view(np.uint32), ologits[i].view(np.uint32)), (pos, i)


# the same at long positions, over a filled cache: a pass of 49 or 67 rows (1568, 2144 units) that ends past 2048, 4096
# and 8192 positions and at the last position a pass can have before the verify rows (16384 in all)
@pytest.mark.parametrize("H,Hkv,hd,start,rows", [(32, 4, 128, 2030, 49), (32, 32, 128, 4090, 49), (32, 4, 128, 8190, 49),
                                                 (32, 4, 128, 16384 - 54, 49), (32, 8, 64, 4090, 67), (32, 4, 64, 8150, 67)])
def test_tiled_attention_at_long_positions_vs_oracle(H, Hkv, hd, start, rows):
    gs, os_ = filled(H, Hkv, hd, start, start + rows + 5)
    toks = nc.uniform_prompt(start, rows, 300)
    gs.prefill_pass_batch(toks, start, want_logits=False)
    for i in range(0, rows, 16):
        os_.prefill_pass_batch(toks[i:i + 16], start + i)
    verify_both(gs, os_, start + rows, 5)  # reads layer 1's keys and values, made from layer 0's tiles


# wide verify passes (more units than CUs, too few for the tiles) on the 256-thread softmax and V kernels, at the last
# and the first row length of each: up to 2048, 4096 and 8192 positions, and the one extra position a thread past 8192
@pytest.mark.parametrize("H,Hkv,hd,rows", [(32, 4, 128, 9), (64, 8, 64, 5)])
@pytest.mark.parametrize("longest", [2048, 2049, 4096, 4097, 8192, 8199])
def test_wide_verify_at_long_positions_vs_oracle(H, Hkv, hd, rows, longest):
    gs, os_ = filled(H, Hkv, hd, longest - rows, longest)
    verify_both(gs, os_, longest - rows, rows)


# rows just past the one-kernel attention (512, 1024 or 1536 positions by head dim and units) and the scores'
# grid steps of 64, 128 and 256 positions a workgroup: one and eight heads per KV head, tiles of one, of 15 and of
# 16 queries, the last prefill row a pass of 49 rows
@pytest.mark.parametrize("H,Hkv,hd,start,rows", [(8, 1, 128, 1023, [1, 2, 3]), (8, 8, 128, 1021, [5, 16]),
                                                 (8, 4, 64, 1533, [3, 8]), (32, 4, 128, 505, [9, 8, 1]),
                                                 (32, 32, 64, 1535, [1, 2]), (32, 32, 64, 1537, [49, 3])])
def test_tile_scores_vs_oracle(H, Hkv, hd, start, rows):
    ctx = nc.Context(0)
    img = nc.synth_gguf(layers=2, embedding_length=H * hd, head_count=H, head_count_kv=Hkv, feed_forward_length=256,
                        vocab_size=300, context_length=2048, tied=1, norm_mode=1, seed=H + Hkv + hd + start)
    end = start + sum(rows)
    gs = nc.Session(nc.Model(ctx, data=img), end + 16, 16)
    os_ = O.Session(O.Model(data=img.tobytes(), nthreads=8), end + 16, 16)
    gs.fill_kv(end, 9)
    os_.fill_kv(end, 9)
    pos = start
    for n in rows:
        toks = nc.uniform_prompt(pos + n, n, 300)
        if n > 16:
            gs.prefill_pass_batch(toks, pos, want_logits=False)
            for i in range(0, n, 16):
                os_.prefill_pass_batch(toks[i:i + 16], pos + i)
        else:
            _, _, _, preds = gs.verify_greedy(toks, pos)
            opreds, _, ologits = os_.verify_greedy(toks, pos, want_logits=True)
            assert np.array_equal(preds, opreds)
            for i in range(n):
                assert np.array_equal(gs.logits(i).view(np.uint32), ologits[i].view(np.uint32)), (pos, i)
        pos += n
