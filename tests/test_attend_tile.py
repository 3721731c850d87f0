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
    (4, 32, 8, 16, 0), (16, 64, 16, 64, 1), (20, 128, 32, 32, 0), (32, 256, 32, 32, 1),
    (16, 512, 64, 64, 0)])
def test_scores_that_rise_and_fall_along_the_keys(gpu, orc, H, kv, rope, page, dtype):
    """Scores between 0 and 40 log2 units, rising and falling along the keys: the reference maximum
    of a wave is raised again, and its sums and accumulators rescaled, when a later unit passes the
    first one's maximum by more than 8 units.  Bound: a score of 40 units (27.7 nats), summed in
    fp32 from up to 576 products, carries about 27.7 * 2^-24 * sqrt(576) = 4e-5 into its weight, in
    the oracle as well."""
    from cpp_inference_train_engine_amd.ops import latent_word
    from cpp_inference_train_engine_amd.workloads import to_bits
    batch, scale = _batch(H, kv, rope, page, dtype, seed=11), 1.0 / np.sqrt(kv + rope)
    rng = np.random.default_rng(12)
    u = rng.standard_normal(kv, dtype=np.float32)
    near = 0.02 * rng.standard_normal(batch.q_latent.shape, dtype=np.float32)
    batch.q_latent[:] = to_bits(u + near, dtype)
    batch.q_rope[:] = to_bits(0.1 * rng.standard_normal(batch.q_rope.shape, dtype=np.float32), dtype)
    raised = 0
    for b, n in enumerate(batch.k_len):
        t = np.arange(int(n))
        f = 40 * np.abs((t / 350 + b % 2) % 2 - 1)  # log2 units, peaks 700 keys apart
        row = f[:, None] / (1.4427 * scale * (u @ u)) * u
        bits = to_bits((row + 0.05 * rng.standard_normal((len(t), kv))).astype(np.float32), dtype)
        pg = batch.page_ids[batch.cu_pages[b] + t // page]
        batch.pages[0, pg[:, None],
                    latent_word(t[:, None] % page, np.arange(kv)[None], page, kv, rope)] = bits
        # split_pages = 4 pages an item for decode rows; wave w takes every 4th unit of 32 keys
        span = 4 * page if batch.q_len[b] == 1 else int(n)
        for first in range(0, int(n), span):
            units = [f[i:min(i + 32, first + span)].max() for i in range(first, min(int(n), first + span), 32)]
            raised += sum(max(units[w + 4::4], default=0) > units[w] + 9 for w in range(min(4, len(units))))
    assert raised > 0
    _say(f"tile kernel, rising scores H={H} kv={kv} dtype={dtype}: {raised} waves rescale")
    want, want_lse = _oracle(orc, batch, scale=scale)
    for flags in (0, 1):
        got, lse = _run(gpu, batch, flags=flags, scale=scale)
        np.testing.assert_allclose(got, want, rtol=1e-4, atol=1e-4, err_msg=f"flags={flags}")
        np.testing.assert_allclose(lse, want_lse, rtol=1e-5, atol=1e-4)


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
