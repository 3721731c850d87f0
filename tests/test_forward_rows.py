"""mla_engine_forward's rows come back in pieces moved by several threads: every row in its place
for one piece and many, whole sequences and chunks, and with a non-finite logit."""
import numpy as np
import pytest

from conftest import MLA36M
from test_model_step import _say

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


@pytest.mark.gpu
def test_nonfinite_row_is_an_error_and_rows_are_out(gpu):
    from cpp_inference_train_engine_amd.workloads import model_params
    params = model_params(CFG, seed=1)
    d = CFG["d_model"]
    params[77 * d:78 * d] = np.inf  # token 77's embedding: its column of every row, and its rows
    eng = _engine(gpu, params, 128)
    ids = np.arange(100, 200, dtype=np.uint16)
    with pytest.raises(gpu.MlaError) as e:
        eng.forward(ids, 1, 100)
    assert e.value.code == "numerical_error" and eng.info()["active_sessions"] == 0
    eng.close()
