"""attend_tile_kernel (decode and chunked prefill over tiled records of any shape) against the
fp32 oracle and the portable kernel, at the edges of its tiles."""
import numpy as np
import pytest

from test_prefill import _oracle, _run, _say


def _batch(H, kv, rope, page, dtype, seed):
    from cpp_inference_train_engine_amd.ops import latent_word, rope_word
    from cpp_inference_train_engine_amd.workloads import DecodeBatch, to_bits
    # one key, tile and page edges, several units per wave; decode rows and chunks
    q = np.array([1, 1, 1, 1, 1, 1, 2, 5, 17, 33], np.int32)
    k = np.array([1, 15, 16, page + 1, 129, 700, 2, 70, 17, 300], np.int32)
    need = (k + page - 1) // page + 1
    P, rows, rng = int(need.sum()), int(q.sum()), np.random.default_rng(seed)
    draw = lambda *s: to_bits(rng.standard_normal(s, dtype=np.float32), dtype)
    batch = DecodeBatch(
        ctx_len=k - q, q_len=q, cu_pages=np.concatenate([[0], np.cumsum(need)]).astype(np.int32),
        page_ids=rng.permutation(P).astype(np.int32), num_pages=P, max_pages=int(need.max()),
        pages=draw(1, P, page * (kv + rope)), q_latent=draw(rows, H, kv),
        q_rope=draw(rows, H, rope), page_size=page, kv_rank=kv, rope_dim=rope, n_heads=H,
        dtype=dtype)
    for b, n in enumerate(k):  # NaN past every session's end
        lst = batch.page_ids[batch.cu_pages[b]:batch.cu_pages[b + 1]]
        for t in range(int(n), len(lst) * page):
            rec = batch.pages[0, lst[t // page]]
            rec[latent_word(t % page, np.arange(kv), page, kv, rope)] = 0x7FC0
            rec[rope_word(t % page, np.arange(rope), page, kv, rope)] = 0x7FC0
    return batch


@pytest.mark.gpu
@pytest.mark.parametrize("H,kv,rope,page,dtype", [
    (4, 32, 8, 16, 0), (1, 64, 16, 64, 1), (16, 96, 24, 48, 0), (17, 128, 16, 64, 1),
    (20, 128, 64, 32, 0), (33, 64, 40, 16, 1), (8, 128, 32, 64, 0), (32, 256, 32, 32, 1),
    (12, 224, 8, 64, 0), (16, 288, 64, 16, 1), (8, 64, 0, 32, 0), (16, 512, 64, 64, 0), (40, 512, 56, 64, 1)])
def test_tile_kernel_edges(gpu, orc, H, kv, rope, page, dtype):
    """Probabilities keep fp32 precision, so the bound is fp32's: scores of magnitude <= 16 in
    log2 units carry 16 * 2^-24 = 1e-6 into each weight, the sums about as much again."""
    batch = _batch(H, kv, rope, page, dtype, seed=kv + rope)
    scale = 1.0 / np.sqrt(kv + rope)
    _say(f"tile kernel H={H} kv={kv} rope={rope} page={page} dtype={dtype}")
    want, want_lse = _oracle(orc, batch, scale=scale)
    for flags in (0, 1):
        got, lse = _run(gpu, batch, flags=flags, scale=scale)
        np.testing.assert_allclose(got, want, rtol=1e-5, atol=1e-5, err_msg=f"flags={flags}")
        np.testing.assert_allclose(lse, want_lse, rtol=1e-5, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("H,kv,rope,page,dtype", [
    (4, 32, 8, 16, 0), (17, 128, 16, 64, 1), (32, 256, 32, 32, 1), (16, 512, 64, 64, 0)])
def test_nonfinite_latents_reach_only_the_rows_that_weigh_them(gpu, H, kv, rope, page, dtype):
    """Infinite and NaN latents of a chunk's token leave the queries before it alone, and make
    those from it on NaN; a decode row whose score of such a key is -inf does not see it.  As in the
    portable kernel, and equal to it up to the bound of test_tile_kernel_edges."""
    from cpp_inference_train_engine_amd.ops import latent_word
    _say(f"tile kernel, non-finite latents H={H} kv={kv} page={page} dtype={dtype}")
    batch, scale = _batch(H, kv, rope, page, dtype, seed=7), 1.0 / np.sqrt(kv + rope)
    one, inf, nan = (0x3C00, 0x7C00, 0x7FC0) if dtype == 0 else (0x3F80, 0x7F80, 0x7FC0)
    q0 = np.concatenate([[0], np.cumsum(batch.q_len)])

    def put(b, t, c, bits):
        p = batch.page_ids[batch.cu_pages[b] + t // page]
        batch.pages[0, p, latent_word(t % page, c, page, kv, rope)] = bits

    batch.q_latent[q0[9]:, :, 3] = one    # a score of inf, and NaN its softmax
    batch.q_latent[q0[5], :, 5] = one     # decode: a score of -inf
    clean, _ = _run(gpu, batch, scale=scale)
    put(9, 267 + 23, 3, inf)              # seen by queries 23.. of 33
    put(9, 267 + 30, kv - 1, nan)
    put(8, 9, 0, nan)                     # the session's own tokens only: queries 9.. of 17
    put(5, 300, 5, 0x8000 | inf)
    got, lse = _run(gpu, batch, scale=scale)
    want, want_lse = _run(gpu, batch, flags=1, scale=scale)
    for first, n, seen in ((q0[9], 33, 23), (q0[8], 17, 9)):
        assert np.isnan(got[first + seen:first + n]).all()
        np.testing.assert_allclose(got[first:first + seen], clean[first:first + seen],
                                   rtol=1e-5, atol=1e-5)
    assert np.isfinite(got[q0[5]]).all()
    np.testing.assert_allclose(got, want, rtol=1e-5, atol=1e-5)
    np.testing.assert_allclose(lse, want_lse, rtol=1e-5, atol=1e-5)
