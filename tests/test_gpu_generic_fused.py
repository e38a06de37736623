"""GPU tests of the fused generic kernel: architectures at the edges of what
it takes (embedding widths that are multiples of 16, windows that are no
power of two, widths that are no multiple of 32, one and many layers) and
just beyond it, against the oracle; and which calls run in it instead of in
separate launches."""

import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# window, embedding width, hidden width, hidden layers: an odd k-tile count
# with a half tile of padding; more n-tiles than two per wave; a deep, narrow
# one; a window of 65; just too wide for the LDS (separate launches)
ARCHS = {"half_tile": (3, 16, 80, 2), "wide": (16, 32, 608, 1), "deep": (7, 48, 32, 12), "window65": (65, 16, 96, 2),
         "one_layer": (33, 64, 0, 0), "beyond": (4, 32, 2080, 1)}


@pytest.fixture(scope="module", params=sorted(ARCHS))
def arch(request):
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a HIP device")
    from sigcomp_amd.model_io import random_int_model
    from sigcomp_amd.quant_mlp_export import QuantMLPCompression
    w, e, h, nh = ARCHS[request.param]
    m = random_int_model(seed=3 + nh, window=w, emb_dim=e, hidden=max(h, 1), n_hidden=nh, per_channel=True)
    return m, QuantMLPCompression(chunk_len=300, gpu=0, model=m)


@pytest.mark.parametrize("rows", [1, 31, 33, 100])
def test_forward(arch, oracle_mod, rows):
    m, codec = arch
    ctx = np.random.default_rng(rows).integers(0, 257, (rows, m.window)).astype(np.int64)
    ref = oracle_mod.mlp_forward(oracle_mod.OracleModel(m), ctx)
    dev = torch.from_numpy(ctx).cuda()
    assert np.array_equal(codec.hip.forward_windows(dev, "logits").cpu().numpy(), ref)
    cdf = codec.hip.forward_windows(dev, "cdf").cpu().numpy().astype(np.int64)
    assert np.array_equal(cdf, oracle_mod.logits_to_cdf(ref, m.exp_lut))


def test_round_trip_and_corrupt_chunk(arch, oracle_mod):
    m, codec = arch
    rng = np.random.default_rng(8)
    lengths = [1, 2, 31, 63, 64, 65, 127, 129, 0, 200] + list(rng.integers(1, 70, 30))
    chunks = [rng.integers(0, 60, n).astype(np.uint8) for n in lengths]
    enc = codec.compress_chunks(chunks)
    assert enc == oracle_mod.compress_chunks(oracle_mod.OracleModel(m), chunks)
    assert all(np.array_equal(a, b) for a, b in zip(chunks, codec.decompress_chunks(enc, lengths)))
    enc[4] = b"\xff" * 8
    with pytest.raises(ValueError, match="chunk 4"):
        codec.decompress_chunks(enc, lengths)


@pytest.mark.parametrize("fused", ["0", "1"])
def test_requantisation_beyond_32_bit_products(oracle_mod, monkeypatch, fused):
    """Layers whose constants need the whole 64-bit product (a shift below 32,
    or a multiplier of 2**31 that becomes 2**30 with a shift of 31) beside
    ones that do not; one output of such a layer takes the whole layer there."""
    import dataclasses
    from sigcomp_amd.model_io import make_layer, random_int_model
    from sigcomp_amd.quant_mlp_export import QuantMLPCompression
    monkeypatch.setenv("SC_HIP_GEN_FUSED", fused)
    rng = np.random.default_rng(31)
    m = random_int_model(seed=31, window=7, emb_dim=32, hidden=96, n_hidden=4, per_channel=True)
    layers = list(m.layers)

    def change(i, outputs, m0, shift):
        L = layers[i]
        new_m0, new_shift = np.array(L.m0, np.int64), np.array(L.shift, np.int32)
        new_m0[outputs], new_shift[outputs] = m0(new_m0[outputs], new_shift[outputs]), shift
        layers[i] = make_layer(L.weight, L.bias, new_m0, new_shift, L.relu)

    scaled = lambda to: lambda m0, sh: np.maximum(m0 >> (sh - to), 1)   # the same factor at another shift
    change(0, slice(None), scaled(31), 31)
    change(1, slice(5, 6), scaled(24), 24)
    change(2, slice(0, 96, 7), lambda m0, sh: 1 << 31, 32)
    change(2, slice(1, 96, 7), lambda m0, sh: 1 << 31, 40)
    change(4, slice(3, 200), scaled(30), 30)
    m = dataclasses.replace(m, layers=layers)
    codec = QuantMLPCompression(chunk_len=300, gpu=0, model=m)
    om = oracle_mod.OracleModel(m)
    ctx = rng.integers(0, 257, (100, m.window)).astype(np.int64)
    ref = oracle_mod.mlp_forward(om, ctx)
    assert len(np.unique(ref)) > 30   # (not saturated throughout)
    assert np.array_equal(codec.hip.forward_windows(torch.from_numpy(ctx).cuda(), "logits").cpu().numpy(), ref)
    lengths = [1, 64, 129]
    chunks = [rng.integers(0, 60, n).astype(np.uint8) for n in lengths]
    enc = codec.compress_chunks(chunks)
    assert enc == oracle_mod.compress_chunks(om, chunks)
    assert all(np.array_equal(a, b) for a, b in zip(chunks, codec.decompress_chunks(enc, lengths)))


def test_more_tiles_than_cus(oracle_mod, monkeypatch):
    """A workgroup that takes several 32-row tiles: forward of more than 32
    rows per CU, compress of more 32-step tiles than CUs (some of them past
    their chunk's end)."""
    from sigcomp_amd.model_io import random_int_model
    from sigcomp_amd.quant_mlp_export import QuantMLPCompression
    monkeypatch.setenv("SC_HIP_GEN_FUSED", "1")
    n_cu = torch.cuda.get_device_properties(0).multi_processor_count
    m = random_int_model(seed=4, window=9, emb_dim=16, hidden=48, n_hidden=2, per_channel=True)
    codec, om = QuantMLPCompression(chunk_len=300, gpu=0, model=m), oracle_mod.OracleModel(m)
    rng = np.random.default_rng(6)
    ctx = rng.integers(0, 257, (2 * 32 * n_cu + 70, m.window)).astype(np.int64)
    ref = oracle_mod.mlp_forward(om, ctx)
    dev = torch.from_numpy(ctx).cuda()
    assert np.array_equal(codec.hip.forward_windows(dev, "logits").cpu().numpy(), ref)
    assert np.array_equal(codec.hip.forward_windows(dev, "cdf").cpu().numpy().astype(np.int64),
                          oracle_mod.logits_to_cdf(ref, m.exp_lut))
    lengths = rng.choice([0, 1, 31, 32, 33, 64, 100, 128, 129, 300], 2 * n_cu + 11)
    chunks = [rng.integers(0, 60, n).astype(np.uint8) for n in lengths]
    enc = codec.compress_chunks(chunks)
    assert enc == oracle_mod.compress_chunks(om, chunks)
    assert all(np.array_equal(a, b) for a, b in zip(chunks, codec.decompress_chunks(enc, list(lengths))))


def _wide():
    from sigcomp_amd.model_io import random_int_model
    from sigcomp_amd.quant_mlp_export import QuantMLPCompression
    m = random_int_model(seed=5, window=64, emb_dim=16, hidden=1400, n_hidden=4, per_channel=False)
    return m, QuantMLPCompression(chunk_len=300, gpu=0, model=m)


@pytest.mark.parametrize("fused", ["0", "1", None])
def test_wide_model_in_both_forms(oracle_mod, monkeypatch, fused):
    """A model with wide layers, whose small calls run in separate launches
    and whose large ones run fused."""
    if fused is not None:
        monkeypatch.setenv("SC_HIP_GEN_FUSED", fused)
    m, codec = _wide()
    rng = np.random.default_rng(2)
    om = oracle_mod.OracleModel(m)
    ctx = rng.integers(0, 257, (2100, m.window)).astype(np.int64)
    ref = oracle_mod.mlp_forward(om, ctx)
    for rows in (1, 40, 2100):
        got = codec.hip.forward_windows(torch.from_numpy(ctx[:rows]).cuda(), "logits").cpu().numpy()
        assert np.array_equal(got, ref[:rows]), rows
    lengths = [1, 31, 63, 64, 65, 100]
    chunks = [rng.integers(0, 60, n).astype(np.uint8) for n in lengths]
    enc = codec.compress_chunks(chunks)
    assert enc == oracle_mod.compress_chunks(om, chunks)
    assert all(np.array_equal(a, b) for a, b in zip(chunks, codec.decompress_chunks(enc, lengths)))


def test_few_rows_of_a_wide_model_take_the_faster_form(monkeypatch):
    """Sixteen chunks: 61 us a step in separate launches, 132 fused."""
    _, codec = _wide()
    tokens, lengths = np.random.default_rng(1).integers(0, 60, 16 * 96).astype(np.uint8), np.full(16, 96, np.int32)
    words, off, cnt = (np.array(a) for a in codec.compress_flat(tokens, lengths))
    best = {}
    for form in ("0", "1", None):
        monkeypatch.delenv("SC_HIP_GEN_FUSED", raising=False)
        if form is not None:
            monkeypatch.setenv("SC_HIP_GEN_FUSED", form)
        for _ in range(4):
            torch.cuda.synchronize()
            start = time.perf_counter()
            assert np.array_equal(codec.decompress_flat(words, off, cnt, lengths)[0], tokens)
            best[form] = min(best.get(form, 1e9), time.perf_counter() - start)
    assert best["1"] > 1.4 * best["0"] and best[None] < 1.2 * best["0"], best
