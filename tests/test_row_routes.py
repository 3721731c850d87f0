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


def _params(cfg):
    """Random parameters with norm gains around 1 (a gain of 1 makes its product exact, and hides
    how often a route rounds it)."""
    from cpp_inference_train_engine_amd.workloads import model_params, parameter_shapes
    flat, at, rng = model_params(cfg, seed=3), 0, np.random.default_rng(4)
    for i, (r, c) in enumerate(parameter_shapes(cfg)):
        if i == 1 or (i > 1 and (i - 2) % 13 in (0, 2, 5, 9)):
            flat[at:at + r * c] += 0.1 * rng.standard_normal(r * c, dtype=np.float32)
        at += r * c
    return flat


def _steps(gpu, cfg, ranges, page=16):
    """One decode step of the sessions [lo, hi) for each range, every step on its own copy of the
    cache; logits [hi - lo x vocab] and the sessions' pages."""
    import torch
    N = max(hi for _, hi in ranges)
    rng = np.random.default_rng(N + cfg["d_model"])
    L, kv, rope = cfg["n_layers"], cfg["kv_lora_rank"], cfg["head_dim_rope"]
    ctx = rng.integers(1, 40, N).astype(np.int32)
    need = ctx // page + 1
    cu = np.concatenate([[0], np.cumsum(need)]).astype(np.int32)
    P = int(cu[-1])
    ids = rng.permutation(P).astype(np.int32)
    tokens = rng.integers(0, cfg["vocab_size"], N).astype(np.int32)
    cache = rng.standard_normal((L, P, page * (kv + rope)), dtype=np.float32).astype(np.float16)
    cache = _dev(cache.view(np.int16)).view(torch.float16)
    model = gpu.HipModel(gpu.ModelConfig.from_dict(cfg), _params(cfg), max_batch=N, page_size=page)
    out = []
    for lo, hi in ranges:
        pages, n = cache.clone(), hi - lo
        mine = ids[cu[lo]:cu[hi]]
        rb = gpu.build_metadata(_dev(ctx[lo:hi]), _dev(np.ones(n, np.int32)),
                                _dev(cu[lo:hi + 1] - cu[lo]), _dev(mine), page, int(need.max()), P,
                                split_pages=4)
        ws = gpu.decode_workspace(rb.max_work, n, cfg["n_heads"], kv)
        logits, _ = model.step(rb, _dev(tokens[lo:hi]), _dev(ctx[lo:hi]), list(pages), ws)
        rb.read_info()
        out.append((logits.cpu().numpy(),
                    pages[:, torch.from_numpy(mine.astype(np.int64))].cpu().numpy().view(np.uint16)))
    model.close()
    return out


# Largest batch of one projection launch: 16 rows times 32 / ceil((heads + 1) / 8).
@pytest.mark.gpu
@pytest.mark.parametrize("cfg, line", [(dict(MLA36M, n_layers=2), 256), (TINY, 512), (ODD, 512),
                                       (WIDE, 160)], ids=["mla36m", "tiny", "odd", "wide"])
def test_row_count_does_not_change_a_bit(gpu, cfg, line):
    """Every row of batches on both sides of the lines (the logits', at parts x row blocks of 64 >
    512, among them for the larger vocabulary) against the row in a batch of at most 16."""
    _say(f"row routes d={cfg['d_model']} line {line}")
    N = line + 17
    small = [(lo, min(lo + 16, N)) for lo in range(0, N, 16)]
    large = [(0, 17), (0, 70), (3, line), (0, line), (0, line + 1), (0, N)]
    got = _steps(gpu, cfg, small + large)
    logits = np.concatenate([x for x, _ in got[:len(small)]])
    pages = np.concatenate([p for _, p in got[:len(small)]], axis=1)
    assert np.isfinite(logits).all() and np.abs(logits).max() > 0
    for (lo, hi), (l, p) in zip(large, got[len(small):]):
        np.testing.assert_array_equal(l, logits[lo:hi], err_msg=f"logits, rows {lo} to {hi}")
        if lo == 0:
            np.testing.assert_array_equal(p, pages[:, :p.shape[1]], err_msg=f"pages, {hi} rows")
