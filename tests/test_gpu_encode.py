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


def _compress_with_caps(codec, tokens, lengths, cap):
    """sc_compress_chunks with a word capacity per chunk -> (word slots, slot
    offsets, counts, status)."""
    from sigcomp_amd import _hip
    n, p = len(lengths), _hip.ptr
    toff = np.concatenate([[0], np.cumsum(lengths[:-1], dtype=np.int64)]).astype(np.int64)
    woff = np.concatenate([[0], np.cumsum(np.maximum(cap[:-1], 0), dtype=np.int64)]).astype(np.int64)
    words, cnt, status, ws = codec._compress_buffers(n, len(tokens), int(np.maximum(cap, 0).sum()))
    words.fill_(-1)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda()
           for a in (tokens, toff, lengths.astype(np.int32), woff, cap.astype(np.int32))]
    _hip.check(_hip.lib().sc_compress_chunks(
        codec.hip.handle, p(dev[0]), p(dev[1]), p(dev[2]), n, len(tokens), p(words), p(dev[3]), p(dev[4]), p(cnt),
        p(status), p(ws), ws.numel(), _hip.stream_ptr()))
    torch.cuda.synchronize()
    return words.cpu().numpy().view(np.uint32), woff, cnt.cpu().numpy(), status.cpu().numpy()


def _committed(cum, freq, cap):
    """(words, overflow) of a chunk at a capacity, by the coder that holds
    words back until no carry can change them (cpu_entropy_coding.py:121-227);
    a step or seal whose words do not fit leaves none of them."""
    M64, words, lower, rng, held = (1 << 64) - 1, [], 0, (1 << 64) - 1, []
    for c, f in zip(cum, freq):
        new, scale = [], rng >> 24
        lo, ra = lower + scale * c, scale * f
        if held and ((lo & M64) + ra) <= M64:
            new, held = _carried(held, lo > M64), []
        lo &= M64
        if ra < 1 << 32:
            word, lo, ra = lo >> 32, (lo << 32) & M64, ra << 32
            if held or lo + ra > M64:
                held = held + [word if not held else 0xFFFFFFFF]
            else:
                new = new + [word]
        if len(words) + len(new) > cap:
            return words, True
        words, lower, rng = words + new, lo, ra
    if not len(cum):
        return words, False
    point = lower + 0xFFFFFFFF
    new = _carried(held, point > M64)
    point = (point & M64) >> 32
    new = new + [point] + ([0] if ((lower + rng) & M64) >> 32 == point else [])
    return (words, True) if len(words) + len(new) > cap else (words + new, False)


def _carried(held, carry):
    return [(held[0] + 1) & 0xFFFFFFFF] + [0] * (len(held) - 1) if held and carry else held


# (token seeds with a chunk that overflows while a word is held back)
@pytest.mark.parametrize("seed,copies", [(23, 1), (26, 11), (29, 11), (30, 1)])
def test_overflowing_chunks_leave_the_committed_words(codec, int_models, oracle_mod, seed, copies):
    """Every capacity from 0 (and a negative one) to more words than a chunk
    needs, in the encoder's scalar and vector form: status, count and words
    are those of the coder that holds words back."""
    rng = np.random.default_rng(seed)
    kinds, caps = [0, 1, 16, 33, 64, 70, 95], np.arange(-1, 57)
    base = [rng.integers(0, 256, k).astype(np.uint8) for k in kinds]
    model, refs = oracle_mod.OracleModel(int_models["lossless"]), []
    for tok in base:
        ctx = np.array([np.concatenate([np.full(64, 256), tok[:t]])[-64:] for t in range(len(tok))], np.int64).reshape(-1, 64)
        cdf = oracle_mod.logits_to_cdf(oracle_mod.mlp_forward(model, ctx), int_models["lossless"].exp_lut) if len(tok) else []
        pairs = [(int(r[k]), int(r[k + 1] - r[k])) for r, k in zip(cdf, tok.tolist())]
        refs += [_committed([c for c, _ in pairs], [f for _, f in pairs], int(cap)) for cap in caps]
    chunks = [tok for tok in base for _ in caps] * copies
    refs = refs * copies
    n = len(chunks)
    assert (n > 4096) == (copies > 1)
    words, woff, cnt, status = _compress_with_caps(codec, np.concatenate(chunks),
                                                   np.array([len(c) for c in chunks], np.int32), np.tile(caps, n // len(caps)))
    want = np.array([over for _, over in refs])
    assert want.any() and not want.all() and np.array_equal(status, want.astype(np.int32))
    assert np.array_equal(cnt, [len(w) for w, _ in refs])
    for c, (w, _) in enumerate(refs):
        assert words[woff[c]:woff[c] + cnt[c]].tolist() == w, c
    assert any(over and 0 <= cap != len(w) for (w, over), cap in zip(refs, np.tile(caps, len(base))))
    # the reference above is the oracle's where all words fit
    ref = oracle_mod.compress_chunks(model, base)
    assert [np.array(refs[len(caps) * (k + 1) - 1][0], "<u4").tobytes() for k in range(len(base))] == ref


def test_overflowing_long_chunk(codec):
    """A million tokens into four words: the encoder stops at the overflow."""
    tokens = np.random.default_rng(3).integers(0, 256, 1 << 20).astype(np.uint8)
    _, _, cnt, status = _compress_with_caps(codec, tokens, np.array([len(tokens)], np.int32), np.array([4], np.int64))
    assert status[0] == 1 and 0 <= cnt[0] <= 4
