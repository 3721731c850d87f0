"""Page pools that do not start at 16 bytes: the model step and forward then take the portable
attention kernels, whatever the shape, and give the results of an aligned pool."""
import ctypes

import numpy as np
import pytest

from conftest import MLA36M
from test_model_step import CACHE_ATOL, CACHE_RTOL, LOGIT_ATOL, _dev, _say

SMALL = dict(MLA36M, n_layers=2, vocab_size=1000, max_sequence_length=512)


@pytest.mark.gpu
@pytest.mark.parametrize("cfg", [SMALL, dict(SMALL, kv_lora_rank=64)], ids=["page", "tile"])
@pytest.mark.parametrize("q", [[1, 1, 1], [1, 40, 3]], ids=["step", "forward"])
@pytest.mark.parametrize("words", [1, 4])
def test_unaligned_pools(gpu, cfg, q, words):
    import torch
    from cpp_inference_train_engine_amd.workloads import model_params
    _say(f"pools at {2 * words} bytes, kv {cfg['kv_lora_rank']}, new rows {q}")
    rng, p = np.random.default_rng(words), gpu.ptr
    L, kv, rope = cfg["n_layers"], cfg["kv_lora_rank"], cfg["head_dim_rope"]
    q, ctx = np.array(q, np.int32), np.array([200, 7, 64], np.int32)
    need = (ctx + q + 63) // 64
    cu = np.concatenate([[0], np.cumsum(need)]).astype(np.int32)
    P, rec, rows = int(cu[-1]), 64 * (kv + rope), int(q.sum())
    cache = _dev(rng.standard_normal((L, P * rec), dtype=np.float32).astype(np.float16))
    tokens = _dev(rng.integers(0, cfg["vocab_size"], rows).astype(np.int32))
    positions = _dev(np.concatenate([c + np.arange(n) for c, n in zip(ctx, q)]).astype(np.int32))
    model = gpu.HipModel(gpu.ModelConfig.from_dict(cfg), model_params(cfg, seed=9), max_batch=rows)
    rb = gpu.build_metadata(_dev(ctx), _dev(q), _dev(cu), _dev(rng.permutation(P).astype(np.int32)),
                            64, int(need.max()), P, split_pages=4, max_rows=rows)
    out = []
    for off in (0, words):
        pools = [torch.zeros(P * rec + 8, dtype=torch.float16, device="cuda")[off:off + P * rec]
                 for _ in range(L)]
        for l in range(L):
            pools[l].copy_(cache[l])
        assert pools[0].data_ptr() % 16 == 2 * off % 16
        ws = gpu.decode_workspace(rb.max_work, 3, cfg["n_heads"], kv)
        logits = torch.zeros((3, cfg["vocab_size"]), device="cuda")
        nxt = torch.zeros(3, dtype=torch.int32, device="cuda")
        ptrs = (ctypes.c_void_p * L)(*[x.data_ptr() for x in pools])
        gpu.check(gpu.lib().mla_model_forward(
            model._h, gpu.stream_handle(), rows, p(tokens), p(positions), 3, int(q.max()),
            p(rb.cu_seqlens_q), p(rb.cu_seqlens_k), p(rb.page_table), rb.max_pages,
            rb.num_pool_pages, p(rb.slot_mapping), p(rb.num_splits), p(rb.cu_splits),
            p(rb.work_desc), p(rb.work_pages), p(rb.info), rb.max_work, ptrs, p(ws), ws.numel(),
            p(logits), p(nxt), 0))
        rb.read_info()
        out.append((logits.cpu().numpy(), torch.stack(pools).float().cpu().numpy()))
    model.close()
    (want, pages), (got, got_pages) = out
    assert np.isfinite(want).all() and np.abs(want).max() > 0
    assert np.abs(got - want).max() <= LOGIT_ATOL
    np.testing.assert_allclose(got_pages, pages, atol=CACHE_ATOL, rtol=CACHE_RTOL)
