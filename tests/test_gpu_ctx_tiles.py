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
    # every row, through calls of another tile size
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
