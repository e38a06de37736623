"""GPU test of the explicit-context kernel's tile sizes: row counts at the
edges where the rule changes from 32- to 64-, 96- and 128-row tiles and a
partial last tile of each, all three MLP cores, logits and CDF tables."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

N_CU = 256


@pytest.fixture(scope="module", params=["per_tensor", "per_channel", "plain"])
def codec(request, int_models):
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a HIP device")
    from sigcomp_amd.model_io import random_int_model
    from sigcomp_amd.quant_mlp_export import QuantMLPCompression
    mp = pytest.MonkeyPatch()
    if request.param == "plain":
        mp.setenv("SC_HIP_PLAIN_CORE", "1")
    m = random_int_model(seed=4) if request.param == "per_channel" else int_models["lossless"]
    c = QuantMLPCompression(chunk_len=64, gpu=0, model=m)
    mp.undo()
    assert c.hip.core == {"per_tensor": 2, "per_channel": 1, "plain": 0}[request.param]
    return m, c


@pytest.mark.parametrize("rows", [1, 33, 4096, 4097, 32 * N_CU, 32 * N_CU + 1, 64 * N_CU + 7, 96 * N_CU + 95])
def test_tile_sizes(codec, oracle_mod, rows):
    m, c = codec
    rng = np.random.default_rng(rows)
    ctx = rng.integers(0, 257, (rows, 64)).astype(np.int64)
    dev = torch.from_numpy(ctx).cuda()
    logits = c.hip.forward_windows(dev, "logits").cpu().numpy()
    cdf = c.hip.forward_windows(dev, "cdf").cpu().numpy()
    # ends of tiles and of the call, and some rows in between
    pick = np.unique(np.concatenate([[0, rows - 1], rng.integers(0, rows, 60), np.arange(max(0, rows - 100), rows, 7)]))
    ref = oracle_mod.mlp_forward(oracle_mod.OracleModel(m), ctx[pick])
    assert np.array_equal(logits[pick], ref)
    assert np.array_equal(cdf[pick].astype(np.int64), oracle_mod.logits_to_cdf(ref, m.exp_lut))
    # every row, through calls of another tile size (the same one up to 5,000 rows)
    again = np.concatenate([c.hip.forward_windows(dev[i:i + 5000], "logits").cpu().numpy() for i in range(0, rows, 5000)])
    assert np.array_equal(again, logits)


def test_no_rows_and_bad_token(codec):
    _, c = codec
    empty = torch.zeros((0, 64), dtype=torch.int64, device="cuda")
    assert c.hip.forward_windows(empty, "logits").shape == (0, 256)
    assert c.hip.forward_windows(empty, "cdf").shape == (0, 257)
    for bad in (-1, 257):
        ctx = torch.zeros((70, 64), dtype=torch.int64, device="cuda")
        ctx[69, 63] = bad
        with pytest.raises(ValueError):
            c.hip.forward_windows(ctx, "logits")


@pytest.mark.parametrize("rows", [1, 33, 4096])
def test_workspace_that_is_not_used(codec, rows):
    """Without workspace, with too little and with one that is not 16-byte
    aligned: one launch, the workspace untouched, the same results."""
    from sigcomp_amd import _hip
    m, c = codec
    ctx = torch.from_numpy(np.random.default_rng(rows).integers(0, 257, (rows, 64)).astype(np.int64)).cuda()
    want = {k: c.hip.forward_windows(ctx, k) for k in ("logits", "cdf")}
    need = _hip.lib().sc_mlp_forward_workspace_bytes(rows)
    ws = torch.full((need + 16,), 0xAB, dtype=torch.uint8, device="cuda")
    assert need > 0 and ws.data_ptr() % 16 == 0
    for ptr, nbytes in ((None, 0), (ws.data_ptr(), need - 1), (ws.data_ptr() + 1, need), (ws.data_ptr() + 8, need)):
        for out in ("logits", "cdf"):
            got, status = torch.zeros_like(want[out]), torch.zeros(1, dtype=torch.int32, device="cuda")
            to = (got.data_ptr(), None) if out == "logits" else (None, got.data_ptr())
            _hip.check(_hip.lib().sc_mlp_forward_ws(c.hip.handle, ctx.data_ptr(), rows, *to, status.data_ptr(), ptr, nbytes,
                                                    _hip.stream_ptr()))
            torch.cuda.synchronize()
            assert torch.equal(got, want[out]) and not status.item()
        assert (ws == 0xAB).all()
