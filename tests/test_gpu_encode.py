"""GPU tests of the range encoder over coded pairs: its scalar form (up to
4,096 chunks per call) and its vector form, ragged lengths around its batches
of 16 steps, words that a carry changes after they were written, and
capacity."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def codec(int_models):
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a HIP device")
    from sigcomp_amd.quant_mlp_export import QuantMLPCompression
    return QuantMLPCompression(chunk_len=2048, gpu=0, model=int_models["lossless"])


@pytest.mark.parametrize("n", [1, 4096, 4097, 9000])
def test_encoder_forms_match_oracle(codec, int_models, oracle_mod, n):
    """Uniform random tokens take about eleven bits each here, so a chunk
    writes a word every three steps and one in some hundred of them is later
    changed by a carry."""
    rng = np.random.default_rng(n)
    lengths = rng.choice([0, 1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 64, 65], n).astype(np.int32)
    lengths[0] = 500
    tokens = rng.integers(0, 256, int(lengths.sum())).astype(np.uint8)
    words, off, cnt = codec.compress_flat(tokens, lengths)
    starts = np.concatenate([[0], np.cumsum(lengths[:-1])])
    pick = np.unique(np.concatenate([[0], rng.integers(0, n, min(n, 400))]))
    ref = oracle_mod.compress_chunks(oracle_mod.OracleModel(int_models["lossless"]),
                                     [tokens[starts[c]:starts[c] + lengths[c]] for c in pick])
    for c, want in zip(pick, ref):
        assert words[off[c]:off[c] + cnt[c]].astype("<u4").tobytes() == want, c
    # the same chunks through the other form
    half = n // 2
    if n > 4096 and half <= 4096:
        w2, o2, c2 = codec.compress_flat(tokens[:int(lengths[:half].sum())], lengths[:half])
        assert np.array_equal(c2, cnt[:half]) and np.array_equal(w2, words[:int(cnt[:half].sum())])
