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
    (12, 224, 8, 64, 0), (16, 288, 64, 16, 1), (16, 512, 64, 64, 0), (40, 512, 56, 64, 1)])
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
