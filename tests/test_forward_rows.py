"""mla_engine_forward's rows come back in pieces moved by several threads: every row in its place
for one piece and many, whole sequences and chunks, and with a non-finite logit."""
import numpy as np
import pytest

from conftest import MLA36M
from test_model_step import LOGIT_ATOL, _say

CFG = dict(MLA36M, n_layers=1)


def _engine(gpu, params, max_rows):
    return gpu.HipEngine(gpu.ModelConfig.from_dict(CFG), params, max_sessions=4,
                         max_rows=max_rows, num_pages=32)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,sequence,max_rows", [(1, 1, 8), (1, 33, 64), (3, 40, 50),
                                                     (2, 100, 64), (4, 64, 256)])
def test_rows_in_place(gpu, batch, sequence, max_rows):
    from cpp_inference_train_engine_amd.workloads import model_params
    rng = np.random.default_rng(batch * sequence)
    ids = rng.integers(0, CFG["vocab_size"], (batch, sequence)).astype(np.uint16)
    eng = _engine(gpu, model_params(CFG, seed=1), max_rows)
    _say(f"forward rows {batch}x{sequence} max_rows={max_rows}")
    got = eng.forward(ids, batch, sequence).reshape(batch, sequence, -1)
    ex = eng.session()
    for b in range(batch):
        for n in sorted({1, sequence // 2 + 1, sequence}):
            np.testing.assert_allclose(got[b, n - 1], ex.prefill(ids[b, :n]), rtol=0, atol=1e-5)
    eng.close()


def _rows(gpu, eng, ids, batch):
    """mla_engine_forward into a buffer of sentinels: its status and the rows."""
    out = np.full((ids.size, CFG["vocab_size"]), 12345.0, np.float32)
    st = gpu.lib().mla_engine_forward(eng._h, batch, ids.size // batch, ids.ctypes.data,
                                      out.ctypes.data)
    return st, out


@pytest.mark.gpu
def test_nonfinite_row_is_an_error_and_rows_are_out(gpu):
    from cpp_inference_train_engine_amd.workloads import model_params
    params = model_params(CFG, seed=1)
    eng = _engine(gpu, params, 128)
    ids = np.arange(100, 200, dtype=np.uint16)
    st, want = _rows(gpu, eng, ids, 1)
    assert st == 0
    eng.close()
    d = CFG["d_model"]
    params[77 * d:78 * d] = np.inf  # token 77's embedding: its column of every row, and its rows
    eng = _engine(gpu, params, 128)
    with pytest.raises(gpu.MlaError) as e:
        eng.forward(ids, 1, 100)
    assert e.value.code == "numerical_error" and eng.info()["active_sessions"] == 0
    st, got = _rows(gpu, eng, ids, 1)
    assert st == 6 and not np.isfinite(got[:, 77]).any()  # MLA_ERR_NUMERICAL
    others = np.delete(np.arange(CFG["vocab_size"]), 77)
    np.testing.assert_array_equal(got[:, others], want[:, others])
    eng.close()


@pytest.mark.gpu
def test_last_row_of_the_last_piece_not_finite(gpu):
    """Token 77's embedding is finite, but overflows fp16 under the first norm's gain: only the
    row of its position, the very last one, is not finite.  (97 tokens: the page kernel works in
    units of 32 keys, so the last key has its unit to itself.)"""
    from cpp_inference_train_engine_amd.workloads import model_params
    params = model_params(CFG, seed=1)
    d, V = CFG["d_model"], CFG["vocab_size"]
    params[77 * d:78 * d] = 60000.0
    params[V * d + d:V * d + 2 * d] = 2.0  # attn_norm of layer 0 (after the embedding, final_norm)
    eng = _engine(gpu, params, 128)
    ids = np.arange(100, 197, dtype=np.uint16)
    st, want = _rows(gpu, eng, ids, 1)
    assert st == 0 and np.isfinite(want).all()
    ids[-1] = 77
    st, got = _rows(gpu, eng, ids, 1)
    assert st == 6 and not np.isfinite(got[96]).all()
    np.testing.assert_array_equal(got[:96], want[:96])
    st, got = _rows(gpu, eng, np.roll(ids, 1)[:50].copy(), 1)  # first: every row attends to it
    assert st == 6 and not (got == 12345.0).any()
    eng.close()


@pytest.mark.gpu
@pytest.mark.parametrize("forced", [0, 1])
def test_one_wait_for_each_model_forward(gpu, forced):
    """Rows, and a single host wait for each model forward, with the fused merge's check passing
    and (forced) failing, which reruns the step before any row is moved on."""
    from cpp_inference_train_engine_amd.workloads import model_params
    eng = _engine(gpu, model_params(CFG, seed=1), 8)
    ids = np.array([5, 9, 300], np.uint16)
    want = eng.forward(np.repeat(ids, 2), 3, 2).reshape(3, 2, -1)[:, 0]  # 3 prompts of 2
    s0 = eng.stats()
    gpu.check(gpu.lib().mla_testing_fail_decode_status(forced))
    try:
        st, got = _rows(gpu, eng, ids, 3)  # 3 sequences of one token: decode rows, placed
    finally:
        gpu.check(gpu.lib().mla_testing_fail_decode_status(0))
    s1 = eng.stats()
    assert st == 0 and s1["fused_reruns"] - s0["fused_reruns"] == forced
    np.testing.assert_allclose(got, want, rtol=0, atol=LOGIT_ATOL)
    assert s1["graph_submissions"] - s0["graph_submissions"] == 1
    assert s1["host_waits"] - s0["host_waits"] == 1 + forced
    eng.close()
