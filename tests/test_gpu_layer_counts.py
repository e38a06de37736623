"""GPU tests of the bundled architecture with other numbers of layers (the
checkpoint's --num-dec-layers): the two-launch windows, compress, and the
fed, split and unsplit decodes, which treat the first, the last hidden and
the output layer apart, against the oracle."""

import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n_hidden", [1, 2, 3, 4, 15])
def test_layer_counts(oracle_mod, monkeypatch, capfd, n_hidden):
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a HIP device")
    from sigcomp_amd.model_io import random_int_model
    from sigcomp_amd.quant_mlp_export import QuantMLPCompression
    m = random_int_model(seed=40 + n_hidden, n_hidden=n_hidden, per_channel=False)
    codec, om = QuantMLPCompression(chunk_len=2048, gpu=0, model=m), oracle_mod.OracleModel(m)
    assert codec.hip.core == 2
    rng = np.random.default_rng(n_hidden)
    ctx = rng.integers(0, 257, (150, 64)).astype(np.int64)
    ref = oracle_mod.mlp_forward(om, ctx)
    many = np.tile(ctx, (30, 1))   # 4,500 rows: one launch; 150: two
    assert np.array_equal(codec.hip.forward_windows(torch.from_numpy(ctx).cuda(), "logits").cpu().numpy(), ref)
    assert np.array_equal(codec.hip.forward_windows(torch.from_numpy(many).cuda(), "logits").cpu().numpy(),
                          np.tile(ref, (30, 1)))
    assert np.array_equal(codec.hip.forward_windows(torch.from_numpy(ctx).cuda(), "cdf").cpu().numpy().astype(np.int64),
                          oracle_mod.logits_to_cdf(ref, m.exp_lut))
    lengths = [1, 2, 63, 64, 65, 0, 130] + list(rng.integers(1, 70, 63))
    chunks = [rng.integers(0, 60, n).astype(np.uint8) for n in lengths]
    enc = codec.compress_chunks(chunks)
    assert enc == oracle_mod.compress_chunks(om, chunks)
    monkeypatch.setenv("SC_HIP_DEC_LOG", "1")
    fed = "fed launch" if n_hidden >= 3 else "split launch p8"   # four layers at least
    for env, what in (({}, fed), ({"SC_HIP_DEC_FED": "2"}, fed), ({"SC_HIP_DEC_SPLIT": "8"}, "split launch p8"),
                      ({"SC_HIP_DEC_SPLIT": "4"}, "split launch p4"), ({"SC_HIP_DEC_SPLIT": "0"}, "launch")):
        with monkeypatch.context() as mp:
            for k, v in env.items():
                mp.setenv(k, v)
            capfd.readouterr()
            back = codec.decompress_chunks(enc, lengths)
            assert re.search(rf"leftover 70 {what} steps", capfd.readouterr().err), env
        assert all(np.array_equal(a, b) for a, b in zip(chunks, back)), env
