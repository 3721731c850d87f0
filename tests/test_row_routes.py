"""The projection kernels that a row goes through depend on the batch's row count; a session's
results must not: the same sessions alone and inside a larger batch give the same bits."""
import numpy as np
import pytest

from conftest import MLA36M, TINY
from test_model_step import _dev, _say

ODD = dict(vocab_size=500, max_sequence_length=300, n_layers=2, d_model=520, n_heads=5,
           head_dim_nope=22, head_dim_rope=10, head_dim_value=24, q_lora_rank=40,
           kv_lora_rank=24, d_ff=1000, norm_epsilon=1e-5, rope_theta=10000.0)
WIDE = dict(ODD, d_model=1024, n_heads=16, q_lora_rank=256, kv_lora_rank=128, d_ff=2048,
            head_dim_nope=48, head_dim_rope=16)


def _steps(gpu, cfg, counts, page=16):
    """One decode step of the first n of max(counts) sessions, for each n; logits and pages."""
    import torch
    from cpp_inference_train_engine_amd.workloads import model_params
    rng = np.random.default_rng(len(counts) + cfg["d_model"])
    N, L, kv, rope = max(counts), cfg["n_layers"], cfg["kv_lora_rank"], cfg["head_dim_rope"]
    ctx = rng.integers(1, 40, N).astype(np.int32)
    need = ctx // page + 1
    cu = np.concatenate([[0], np.cumsum(need)]).astype(np.int32)
    P = int(cu[-1])
    ids = rng.permutation(P).astype(np.int32)
    tokens = rng.integers(0, cfg["vocab_size"], N).astype(np.int32)
    cache = rng.standard_normal((L, P, page * (kv + rope)), dtype=np.float32).astype(np.float16)
    model = gpu.HipModel(gpu.ModelConfig.from_dict(cfg), model_params(cfg, seed=3), max_batch=N,
                         page_size=page)
    out = []
    for n in counts:
        pages = [_dev(cache[l].view(np.int16)).view(torch.float16) for l in range(L)]
        rb = gpu.build_metadata(_dev(ctx[:n]), _dev(np.ones(n, np.int32)), _dev(cu[:n + 1]),
                                _dev(ids[:cu[n]]), page, int(need.max()), P, split_pages=4)
        ws = gpu.decode_workspace(rb.max_work, n, cfg["n_heads"], kv)
        logits, _ = model.step(rb, _dev(tokens[:n]), _dev(ctx[:n]), pages, ws)
        rb.read_info()
        mine = torch.stack(pages)[:, torch.from_numpy(ids[:cu[min(counts)]].astype(np.int64))]
        out.append((logits[:min(counts)].cpu().numpy(), mine.cpu().numpy().view(np.uint16)))
    model.close()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("cfg", [dict(MLA36M, n_layers=2), TINY, ODD, WIDE],
                         ids=["mla36m", "tiny", "odd", "wide"])
@pytest.mark.parametrize("counts", [(3, 16, 17, 70), (13, 191, 192, 260)])
def test_row_count_does_not_change_a_bit(gpu, cfg, counts):
    _say(f"row routes d={cfg['d_model']} {counts}")
    got = _steps(gpu, cfg, counts)
    assert np.isfinite(got[0][0]).all() and np.abs(got[0][0]).max() > 0
    for n, (logits, pages) in zip(counts[1:], got[1:]):
        np.testing.assert_array_equal(logits, got[0][0], err_msg=f"logits, {n} rows")
        np.testing.assert_array_equal(pages, got[0][1], err_msg=f"pages, {n} rows")
