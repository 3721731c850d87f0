"""Logits of many rows or of a large vocabulary (g7_rows_kernel) against the smaller kernel: the
embedding repeats a 500-row one, so every column of every row has to repeat the logits of the
500-token model bit for bit, and the greedy winner is the lowest of its equals."""
import numpy as np
import pytest

from conftest import MLA36M
from test_model_step import _dev, _say

BASE = 500


def _step(gpu, cfg, params, n, page=16):
    import torch
    rng = np.random.default_rng(n)
    kv, rope = cfg["kv_lora_rank"], cfg["head_dim_rope"]
    pages = [_dev(rng.standard_normal((n, page * (kv + rope)), dtype=np.float32)
                  .astype(np.float16).view(np.int16)).view(torch.float16)]
    ctx, cu = np.full(n, page - 3, np.int32), np.arange(n + 1, dtype=np.int32)
    model = gpu.HipModel(gpu.ModelConfig.from_dict(cfg), params, max_batch=n, page_size=page)
    rb = gpu.build_metadata(_dev(ctx), _dev(np.ones(n, np.int32)), _dev(cu), _dev(cu[:-1].copy()),
                            page, 1, n, split_pages=4)
    ws = gpu.decode_workspace(rb.max_work, n, cfg["n_heads"], kv)
    logits, nxt = model.step(rb, _dev(rng.integers(0, BASE, n).astype(np.int32)), _dev(ctx),
                             pages, ws)
    out = logits.cpu().numpy(), nxt.cpu().numpy()
    model.close()
    return out


# 64-column groups: 516 of 33000, 250 of 16000, 1024 of 65535.  d_model: the 8 K groups hold one
# k-step (200: the last group none), two, three (520: most groups two; 768) and four.
@pytest.mark.gpu
@pytest.mark.parametrize("vocab,d,n", [(33000, 200, 1), (33000, 200, 65), (16000, 512, 129),
                                       (16000, 512, 200), (16000, 520, 193), (16000, 768, 130),
                                       (16000, 1024, 192), (65535, 512, 3), (33000, 104, 64)])
def test_columns_repeat(gpu, vocab, d, n):
    from cpp_inference_train_engine_amd.workloads import model_params
    cfg = dict(MLA36M, n_layers=1, vocab_size=BASE, d_model=d, max_sequence_length=64)
    params = np.asarray(model_params(cfg, seed=5))
    embed = params[:BASE * d].reshape(BASE, d)
    large = np.concatenate([embed[np.arange(vocab) % BASE].ravel(), params[BASE * d:]])
    _say(f"logits routes vocab={vocab} d={d} rows={n}")
    want, want_next = _step(gpu, cfg, params, n)
    got, got_next = _step(gpu, dict(cfg, vocab_size=vocab), large, n)
    assert np.isfinite(want).all() and (np.abs(want).max(axis=1) > 0).all()
    np.testing.assert_array_equal(got, want[:, np.arange(vocab) % BASE])
    np.testing.assert_array_equal(got_next, want_next)
    np.testing.assert_array_equal(want_next, want.argmax(axis=1))
