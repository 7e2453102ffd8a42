"""GPU parity of the device-side batch builder against the oracle's restatement of batch_builder.build:
tokens, positions and the block-diagonal causal mask bit for bit."""
import ctypes as C

import numpy as np
import pytest
import torch

from tests.helpers import to_np_u32

pytestmark = pytest.mark.gpu


def _requests(seed, lens):
    rng = np.random.default_rng(seed)
    toks = [rng.integers(0, 50000, n).astype(np.uint32) for n in lens]
    base = [int(rng.integers(0, 4000)) if n == 1 else int(rng.integers(0, 100)) for n in lens]
    return toks, base


def test_batch_build_reference_cases(dmoe, ws, golden):
    """The literal cases of the reference's batch builder tests (src/tests/batch_builder_tests.zig:61-316)."""
    for case in golden["batch_builder"]["cases"]:
        lens = [len(r["tokens"]) for r in case["requests"]]
        flat = [t for r in case["requests"] for t in r["tokens"]]
        d_tok, d_pos, d_mask, d_req = dmoe.batch_build(flat, lens, [r["base"] for r in case["requests"]], ws)
        assert d_tok.numel() == case.get("total_tokens", sum(lens)) and int(d_req.max()) + 1 == case["num_requests"]
        if case["tokens"] is not None:
            np.testing.assert_array_equal(to_np_u32(d_tok), case["tokens"], err_msg=case["name"])
        if case["positions"] is not None:
            np.testing.assert_array_equal(d_pos.cpu().numpy(), case["positions"], err_msg=case["name"])
        m = d_mask.cpu().numpy()
        assert m.shape == (len(flat), len(flat))
        for r, c, att in case["attending"]:
            assert (m[r, c] == 0.0) == bool(att), (case["name"], r, c)


@pytest.mark.parametrize("lens", [[5, 3, 1, 1], [512, 512, 1, 1, 1, 7], [1], [3, 0, 4], [129, 2]])
def test_batch_build_matches_oracle(dmoe, orc, ws, lens):
    toks, base = _requests(3, lens)
    want_tok, want_pos, offs = orc.batch_concat(toks, base)
    want_mask = orc.batch_mask(lens)
    flat = np.concatenate(toks) if sum(lens) else np.zeros(0, np.uint32)
    d_tok, d_pos, d_mask, d_req = dmoe.batch_build(flat.tolist(), lens, base, ws)
    np.testing.assert_array_equal(to_np_u32(d_tok), want_tok)
    np.testing.assert_array_equal(d_pos.cpu().numpy(), want_pos)
    np.testing.assert_array_equal(d_mask.cpu().numpy().view(np.uint32), want_mask.view(np.uint32))
    want_req = np.repeat(np.arange(len(lens)), lens)
    np.testing.assert_array_equal(d_req.cpu().numpy(), want_req)
    # mask properties of the reference's tests: 0 on and below the diagonal inside a request, -inf elsewhere
    m = d_mask.cpu().numpy()
    assert np.isneginf(m[np.triu_indices(m.shape[0], 1)]).all() and (np.diag(m) == 0).all()


def test_batch_build_baseline_config_4_shape(dmoe, orc, ws):
    """4 x 512 prefill rows then 32 decode rows (the mixed batch of configuration 4), without the mask too."""
    lens = [512] * 4 + [1] * 32
    toks, base = _requests(4, lens)
    flat = np.concatenate(toks)
    _, d_pos, d_mask, d_req = dmoe.batch_build(flat.tolist(), lens, base, ws, want_mask=False)
    assert d_mask is None
    _, want_pos, _ = orc.batch_concat(toks, base)
    np.testing.assert_array_equal(d_pos.cpu().numpy(), want_pos)
    assert int(d_req[-1]) == len(lens) - 1


def test_batch_build_rejects_inconsistent_requests(dmoe, ws):
    with pytest.raises(dmoe.DmoeError, match="sum"):
        dmoe.batch_build([1, 2, 3], [2, 2], [0, 0], ws)
    with pytest.raises(dmoe.DmoeError, match="negative"):
        dmoe.batch_build([1, 2, 3], [4, -1], [0, 0], ws)


def test_batch_build_base_positions_shorter_and_longer_than_the_requests(dmoe, ws):
    """A missing base position is 0; one too many is refused."""
    _, pos, _, _ = dmoe.batch_build([1, 2, 3], [2, 1], [5], ws)
    assert pos.tolist() == [5, 6, 0]
    with pytest.raises(IndexError):
        dmoe.batch_build([1, 2, 3], [2, 1], [5, 0, 7], ws)


@pytest.mark.parametrize("lens", [[1] * 255, [256], [257], [1] * 600, [0, 255, 0, 0, 1, 0, 256, 0], [513, 0, 1, 510], [2047, 1, 1, 1], [3]])
def test_batch_build_block_edges(dmoe, orc, ws, lens):
    """Requests that start, end and fall empty at the edges of the 256-token blocks, and masks whose rows start on every
    residue of the 16-byte stores."""
    toks, base = _requests(sum(lens), lens)
    want_tok, want_pos, _ = orc.batch_concat(toks, base)
    d_tok, d_pos, d_mask, d_req = dmoe.batch_build(np.concatenate(toks).tolist(), lens, base, ws)
    np.testing.assert_array_equal(to_np_u32(d_tok), want_tok)
    np.testing.assert_array_equal(d_pos.cpu().numpy(), want_pos)
    np.testing.assert_array_equal(d_mask.cpu().numpy().view(np.uint32), orc.batch_mask(lens).view(np.uint32))
    np.testing.assert_array_equal(d_req.cpu().numpy(), np.repeat(np.arange(len(lens)), lens))


def test_batch_build_calls_in_flight_do_not_share_lists(dmoe, orc, ws):
    """Calls of equal, growing and shrinking size enqueued behind some tens of milliseconds of other work: each reads its own
    lists, although none of their kernels has run when the later calls are made."""
    cases, got = [], []
    busy = torch.ones((8192, 8192), dtype=torch.bfloat16, device="cuda")
    dmoe.batch_build([1], [1], [0], ws)
    for _ in range(40):
        busy @ busy
    for i, n in enumerate((700, 700, 700, 700, 40, 3000, 3000, 9, 9000, 300)):
        lens = [n // 2, 0, n - n // 2 - 1, 1]
        cases.append((lens, *_requests(100 + i, lens)))
    for lens, toks, base in cases:
        got.append(dmoe.batch_build(np.concatenate(toks).tolist(), lens, base, ws, want_mask=False))
    for (lens, toks, base), (d_tok, d_pos, _, d_req) in zip(cases, got):
        want_tok, want_pos, _ = orc.batch_concat(toks, base)
        np.testing.assert_array_equal(to_np_u32(d_tok), want_tok)
        np.testing.assert_array_equal(d_pos.cpu().numpy(), want_pos)
        np.testing.assert_array_equal(d_req.cpu().numpy(), np.repeat(np.arange(len(lens)), lens))


def test_batch_build_under_capture_is_refused(dmoe, ws):
    """The host lists are read from staging memory that later calls refill: a replay would read another batch's."""
    x = torch.zeros(4, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x.add_(1)
        with pytest.raises(dmoe.DmoeError, match="captured graph"):
            dmoe.batch_build([1, 2, 3], [2, 1], [0, 0], ws)
    tok, pos, _, _ = dmoe.batch_build([1, 2, 3], [2, 1], [0, 7], ws)
    assert tok.tolist() == [1, 2, 3] and pos.tolist() == [0, 1, 7]


def test_batch_build_on_a_new_workspace_beside_a_capture(dmoe, ws):
    """The first calls on a workspace allocate nothing, its two slots are made with it. Seen while another stream is being
    captured: an allocation would be refused there and would invalidate the capture."""
    T, x, side = 8192, torch.zeros(4, device="cuda"), torch.cuda.Stream()
    outs = [(torch.empty(T, dtype=torch.int32, device="cuda"), torch.empty(T, dtype=torch.int32, device="cuda")) for _ in range(2)]
    lists = [((C.c_uint32 * T)(*range(i, T + i)), (C.c_int32 * 2)(T - 1, 1), (C.c_int32 * 2)(i, 7)) for i in range(2)]
    new = dmoe.Workspace(1 << 20)
    torch.cuda.synchronize()
    graph, rc = torch.cuda.CUDAGraph(), []
    with torch.cuda.graph(graph):
        x.add_(1)
        for (tok, pos), (h_tok, h_len, h_base) in zip(outs, lists):
            rc.append(dmoe.lib().dmoe_batch_build(dmoe._ptr(tok), dmoe._ptr(pos), None, None, h_tok, h_len, h_base, 2, T, new.h,
                                                  dmoe._Handle(side.cuda_stream)))
        x.add_(1)
    assert rc == [0, 0]
    graph.replay()
    torch.cuda.synchronize()
    assert x.tolist() == [2.0] * 4
    for i, (tok, pos) in enumerate(outs):
        assert torch.equal(tok.cpu(), torch.arange(i, T + i, dtype=torch.int32))
        assert torch.equal(pos.cpu(), torch.cat([torch.arange(i, T - 1 + i), torch.tensor([7])]).int())
    new.close()
