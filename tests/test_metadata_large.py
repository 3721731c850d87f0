"""Metadata builds of two launches (page table past 8192 entries): their error paths, and the
smallest and raggedest tables (the bit-exact cases are in test_gpu_kernels.py and
test_placement.py)."""
import numpy as np
import pytest

from test_gpu_kernels import _gpu_metadata, _say
from test_metadata_oracle import py_metadata, random_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", ["neg_q", "short_pages", "bad_id", "bad_last_id",
                                  "too_many_pages", "max_work", "max_rows", "first_of_two"])
def test_errors_match_oracle(gpu, orc, case):
    rng = np.random.default_rng(11)
    B = 300
    ctx, q, cu_pages, ids, P, max_pages = random_batch(rng, B, decode=False, spare=0)
    assert B * max_pages > 8192
    ctx, q, ids = ctx.copy(), q.copy(), ids.copy()
    max_work, max_rows = 65535, 1 << 20
    if case == "neg_q":
        q[171] = -1
    elif case == "short_pages":
        ctx[5] += 64 * 3
    elif case == "bad_id":
        ids[cu_pages[90]] = P
    elif case == "bad_last_id":
        ids[-1] = -1
    elif case == "too_many_pages":
        max_pages = int(np.diff(cu_pages).max()) - 1
    elif case == "max_work":
        max_work = 100
    elif case == "max_rows":
        max_rows = 40
    else:
        q[200], ids[cu_pages[123]] = -5, P + 7
    assert B * max_pages > 8192
    want = py_metadata(list(ctx), list(q), list(cu_pages), list(ids), 64, max_pages, P, 1, 512,
                       max_work, max_rows)
    _say(f"large metadata error {case}: session {want[1]}")
    rb = _gpu_metadata(gpu, ctx, q, cu_pages, ids, 64, max_pages, P, 1, 512, max_work, max_rows)
    with pytest.raises(gpu.MlaError):
        rb.read_info()
    assert rb.info.cpu().numpy().tolist() == [-1, want[1], 0, 0, 0, 0, 0, 0]
    assert np.all(rb.work_desc.cpu().numpy().reshape(-1, 8)[:, 0] == -1)  # no work issued


@pytest.mark.parametrize("B,longest", [(1, 9000), (3, 3000), (1500, 7)])
def test_table_shapes(gpu, orc, B, longest):
    """One very long session; a few; many short ones with empty sessions among them."""
    rng = np.random.default_rng(B)
    need = rng.integers(0, longest + 1, B)
    need[0] = longest
    ctx, q = np.maximum(need * 16 - 3, 0), (need > 0).astype(np.int64)
    cu_pages = np.concatenate([[0], np.cumsum(need)])
    P = int(cu_pages[-1]) + 1
    ids = rng.permutation(P)[:-1]
    want = orc.build_metadata(ctx, q, cu_pages, ids, 16, longest, P, 5, 512, 65535)
    _say(f"large metadata B={B} longest={longest}")
    rb = _gpu_metadata(gpu, ctx, q, cu_pages, ids, 16, longest, P, 5, 512, 65535, B)
    assert rb.read_info() == want["info"].tolist()
    W = int(want["info"][0])
    np.testing.assert_array_equal(rb.page_table[:B * longest].cpu().numpy(),
                                  want["page_table"].reshape(-1))
    np.testing.assert_array_equal(rb.work_desc.cpu().numpy().reshape(-1, 8)[:W],
                                  want["work_desc"][:W])
    np.testing.assert_array_equal(rb.slot_mapping[:int(want["info"][2])].cpu().numpy(),
                                  want["slot_mapping"][:int(want["info"][2])])


def _long(need, q, ps=16):
    """Sessions of `need` pages each, the last `q` tokens of each new."""
    need, q = np.asarray(need), np.asarray(q)
    cu_pages = np.concatenate([[0], np.cumsum(need)])
    P = int(cu_pages[-1]) + 3
    ids = np.random.default_rng(len(need)).permutation(P)[:cu_pages[-1]]
    return need * ps - 5 - q, q, cu_pages, ids, P, int(need.max())


@pytest.mark.parametrize("placed", [False, True])
@pytest.mark.parametrize("need,q", [([8193], [1]), ([9000], [5000]), ([2800, 1, 2731], [1024, 1, 1023]),
                                    ([700, 1100, 1, 2100], [1, 1, 0, 1]), ([70] * 127, [1] * 127)])
def test_long_sessions(gpu, orc, need, q, placed):
    """A session's row of the table and its slots are written by several workgroups when sessions
    are few: every output against the oracle."""
    import torch
    from test_placement import _placed
    ctx, q, cu_pages, ids, P, max_pages = _long(need, q)
    B, n = len(q), gpu.xcd_count() if placed else 0
    assert B * max_pages > 8192
    max_work = 65535
    want = orc.build_metadata(ctx, q, cu_pages, ids, 16, max_pages, P, 3, 512, max_work,
                              placement_xcds=n) if placed else \
        orc.build_metadata(ctx, q, cu_pages, ids, 16, max_pages, P, 3, 512, max_work)
    _say(f"long sessions B={B} max_pages={max_pages} rows={q.sum()} placed={placed}")
    rb = _placed(gpu, ctx, q, cu_pages, ids, 16, max_pages, P, 3, max_work, placement=placed)
    torch.cuda.synchronize()
    assert rb.read_info() == want["info"].tolist()
    W, T = int(want["info"][0]), int(want["info"][2])
    occ = want["occupied"] if placed else np.arange(max_work) < W
    desc = rb.work_desc.cpu().numpy().reshape(-1, 8)[:max_work]
    np.testing.assert_array_equal(desc[:, 0] >= 0, occ)
    sel = (lambda x: x[occ]) if placed else (lambda x: x[:W])
    np.testing.assert_array_equal(desc[occ], sel(want["work_desc"]))
    np.testing.assert_array_equal(rb.work_pages.cpu().numpy().reshape(-1, 8)[:max_work][occ],
                                  sel(want["work_pages"]))
    np.testing.assert_array_equal(rb.page_table[:B * max_pages].cpu().numpy(),
                                  want["page_table"].reshape(-1))
    np.testing.assert_array_equal(rb.slot_mapping[:T].cpu().numpy(), want["slot_mapping"][:T])


@pytest.mark.parametrize("where", [0, 1023, 1024, 16383, 16384, 20000, -1])
@pytest.mark.parametrize("need", [[25001], [9000, 16001], [5000, 1, 20000]])
def test_bad_id_of_a_long_session(gpu, where, need):
    ctx, q, cu_pages, ids, P, max_pages = _long(need, [1] * len(need))
    ids = ids.copy()
    ids[where] = P if where % 2 else -1
    session = int(np.searchsorted(cu_pages, where % len(ids), side="right")) - 1
    _say(f"bad id {where} of sessions of {need} pages")
    rb = _gpu_metadata(gpu, ctx, q, cu_pages, ids, 16, max_pages, P, 4, 512, 65535, len(need))
    assert rb.info.cpu().numpy().tolist() == [-1, session, 0, 0, 0, 0, 0, 0]
    assert np.all(rb.work_desc.cpu().numpy().reshape(-1, 8)[:, 0] == -1)
