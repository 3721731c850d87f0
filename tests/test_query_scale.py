"""W_uq and W_uk reach the step as they are stored: moving a power of two between them and q_norm
changes no bit of a step.  (Their product rounded to fp16 as one weight would: at the smaller scale
it lies among fp16's subnormals.)"""
import numpy as np
import pytest

from conftest import MLA36M
from test_model_step import _dev, _say

CFG = dict(MLA36M, n_layers=2, max_sequence_length=512)
ODD = dict(CFG, n_heads=4, head_dim_nope=23, head_dim_rope=10, kv_lora_rank=40, q_lora_rank=72)


def _params(cfg, q_norm, uq, uk):
    """Parameters with q_norm gains 2^q_norm and W_uq's nope columns and W_uk of magnitude
    2^uq and 2^uk (the rope columns undo the gain).  Magnitudes are 7-bit numbers in [1/2, 1) of
    that, so that every one of them is exact and normal in fp16 at every scale."""
    from cpp_inference_train_engine_amd.workloads import model_params, parameter_shapes
    flat, at = model_params(cfg, seed=5), 0
    flat = flat.astype(np.float16).astype(np.float32)
    rng = np.random.default_rng(6)
    qk, nope = cfg["head_dim_nope"] + cfg["head_dim_rope"], cfg["head_dim_nope"]
    for i, (r, c) in enumerate(parameter_shapes(cfg)):
        slot, w = -1 if i < 2 else (i - 2) % 13, flat[at:at + r * c].reshape(r, c)
        at += r * c
        if slot == 2:
            w *= 2.0 ** q_norm
        if slot in (3, 6):  # w_uq, w_uk
            v = (rng.integers(64, 128, (r, c)) * rng.choice([-1, 1], (r, c))).astype(np.float32)
            w[:] = v / 128 * 2.0 ** (uk if slot == 6 else uq)
            if slot == 3:
                w.reshape(r, -1, qk)[:, :, nope:] *= 2.0 ** (-q_norm - uq - 1)
    return flat


@pytest.mark.gpu
@pytest.mark.parametrize("cfg", [CFG, ODD], ids=["mla36m", "odd"])
@pytest.mark.parametrize("sessions", [5, 35])
def test_small_query_weights_keep_their_precision(gpu, cfg, sessions):
    import torch
    _say(f"query weight scales, {sessions} sessions, {cfg['n_heads']} heads")
    rng = np.random.default_rng(sessions)
    L, kv, rope = cfg["n_layers"], cfg["kv_lora_rank"], cfg["head_dim_rope"]
    ctx = rng.integers(1, 200, sessions).astype(np.int32)
    need = ctx // 64 + 1
    cu = np.concatenate([[0], np.cumsum(need)]).astype(np.int32)
    P = int(cu[-1])
    tokens = _dev(rng.integers(0, cfg["vocab_size"], sessions).astype(np.int32))
    cache = rng.standard_normal((L, P, 64 * (kv + rope)), dtype=np.float32).astype(np.float16)
    rb = gpu.build_metadata(_dev(ctx), _dev(np.ones(sessions, np.int32)), _dev(cu),
                            _dev(np.arange(P, dtype=np.int32)), 64, int(need.max()), P,
                            split_pages=4)
    ws = gpu.decode_workspace(rb.max_work, sessions, cfg["n_heads"], kv)
    out = []
    for scales in ((6, -5, -5), (12, -8, -8)):  # q_norm . W_uq . W_uk at one scale
        model = gpu.HipModel(gpu.ModelConfig.from_dict(cfg), _params(cfg, *scales),
                             max_batch=sessions)
        pages = [_dev(cache[l].view(np.int16)).view(torch.float16) for l in range(L)]
        logits, _ = model.step(rb, tokens, _dev(ctx), pages, ws)
        out.append((logits.cpu().numpy(), torch.stack(pages).cpu().numpy().view(np.uint16)))
        rb.read_info()
        model.close()
    assert np.isfinite(out[0][0]).all() and np.abs(out[0][0]).max() > 0
    np.testing.assert_array_equal(out[1][0], out[0][0])
    np.testing.assert_array_equal(out[1][1], out[0][1])
