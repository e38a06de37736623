"""GPU tests of the fed decode (heads and feeder sets): batch sizes at the
edges of its tiles, sets and limits, ragged lengths, and two concurrent
calls, against the input and the unsplit decode."""

import re
import threading

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


def _chunks(codec, lengths, seed):
    rng = np.random.default_rng(seed)
    lengths = np.asarray(lengths, np.int32)
    tokens = rng.integers(0, 60, int(lengths.sum())).astype(np.uint8)
    words, off, cnt = (np.array(a) for a in codec.compress_flat(tokens, lengths))
    return tokens, lengths, words, off, cnt


def _decode(codec, monkeypatch, capfd, words, off, cnt, lengths):
    monkeypatch.setenv("SC_HIP_DEC_LOG", "1")
    capfd.readouterr()
    back = np.array(codec.decompress_flat(words, off, cnt, lengths)[0])
    m = re.search(r"fed (\d+)\+(\d+)x16", capfd.readouterr().err)
    return back, (int(m.group(1)), int(m.group(2)))


# heads x sets expected on 256 CUs: one partial tile; a tile and one row; the
# second set; 65 tiles; 64-row heads with a partial last one, and at their limit
@pytest.mark.parametrize("n,heads,sets", [(1, 1, 1), (32, 1, 1), (33, 2, 1), (193, 7, 2), (2049, 65, 11), (4171, 66, 11),
                                          (8191, 128, 8)])
def test_fed_decode_sizes(codec, monkeypatch, capfd, n, heads, sets):
    rng = np.random.default_rng(n)
    lengths = rng.integers(1, 200 if n < 1000 else 90, n)
    lengths[rng.integers(0, n)] = 201   # one row alone past the others' end
    tokens, lengths, words, off, cnt = _chunks(codec, lengths, n)
    back, shape = _decode(codec, monkeypatch, capfd, words, off, cnt, lengths)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert shape == (heads, sets)
    assert np.array_equal(back, tokens)
    monkeypatch.setenv("SC_HIP_DEC_SPLIT", "0")
    plain, shape = _decode(codec, monkeypatch, capfd, words, off, cnt, lengths)
    assert shape == (0, 0) and np.array_equal(plain, tokens)


@pytest.mark.parametrize("rt", ["1", "2"])
@pytest.mark.parametrize("longest", [1, 2, 3, 63, 64, 65, 129])
def test_fed_decode_step_edges(codec, monkeypatch, capfd, longest, rt):
    """Few steps (a feeder waits for tokens from the third on) and the
    64-step flush and refill; empty chunks and whole tiles that end early."""
    lengths = np.concatenate([np.full(32, longest), np.zeros(33, int), np.full(40, min(longest, 2)), [longest, 0, 1]])
    tokens, lengths, words, off, cnt = _chunks(codec, lengths, longest)
    monkeypatch.setenv("SC_HIP_DEC_FED", rt)
    back, shape = _decode(codec, monkeypatch, capfd, words, off, cnt, lengths)
    assert shape[0] > 0 and np.array_equal(back, tokens)


def test_fed_decodes_of_two_threads(codec, int_models):
    """Two host threads, each with its own stream and batch, one model."""
    jobs, out, errs = [], {}, []
    for k in range(2):
        jobs.append(_chunks(codec, np.full(600, 120 + k), 10 + k))

    def work(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                tokens, lengths, words, off, cnt = jobs[k]
                for _ in range(3):
                    out[k] = np.array(codec.decompress_flat(words, off, cnt, lengths)[0])
        except Exception as e:  # reported by the main thread
            errs.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errs, errs
    assert all(np.array_equal(out[k], jobs[k][0]) for k in range(2))


def test_smaller_workspace_runs_split(codec, monkeypatch, capfd):
    """A workspace of the split decode's size (32 KiB + 32 bytes of exchange
    per 32 chunks) is taken and decodes split, one byte less is refused."""
    from sigcomp_amd import _hip
    tokens, lengths, words, off, cnt = _chunks(codec, np.full(70, 130), 3)
    n, groups = len(lengths), 3
    need = (n * 40 + 255) // 256 * 256 + 256 + groups * 32768 + 256
    assert need < _hip.lib().sc_decompress_workspace_bytes(n)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    toff = np.arange(n, dtype=np.int64) * 130
    t = [d(words.view(np.int32)), d(off), d(cnt), d(lengths)]
    out = torch.zeros(len(tokens), dtype=torch.uint8, device="cuda")
    t_toff, status = d(toff), torch.full((n,), -1, dtype=torch.int32, device="cuda")
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")

    def call(nbytes):
        return _hip.lib().sc_decompress_chunks(
            codec.hip.handle, *[x.data_ptr() for x in t], n, out.data_ptr(), t_toff.data_ptr(), status.data_ptr(),
            lengths.ctypes.data, ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)

    monkeypatch.setenv("SC_HIP_DEC_LOG", "1")
    capfd.readouterr()
    assert call(need - 1) == _hip.SC_ERR_ARG
    _hip.check(call(need))
    torch.cuda.synchronize()
    log = capfd.readouterr().err
    assert "split launch p8" in log and "fed 0+0" in log
    assert not status.any().item() and np.array_equal(out.cpu().numpy(), tokens)


@pytest.mark.parametrize("n,rt", [(2049, "1"), (4171, "2")])
def test_large_fed_decode_never_reports_a_timeout(codec, monkeypatch, n, rt):
    """Batches of more than 64 tiles never waited between workgroups before
    they ran fed: where a wait expires (here each at once, SC_HIP_DEC_SPIN=0)
    the call decodes the tiles again without waiting, so that its tokens are
    right, every status is written and a corrupt chunk, and only it, is
    reported as such."""
    from sigcomp_amd import _hip
    rng = np.random.default_rng(n)
    tokens, lengths, words, off, cnt = _chunks(codec, rng.integers(0, 70, n), n)
    bad = int(np.argmax(lengths))
    words = np.concatenate([words, np.full(2, 0xFFFFFFFF, np.uint32)])
    off[bad], cnt[bad] = len(words) - 2, 2
    toff = np.concatenate([[0], np.cumsum(lengths[:-1], dtype=np.int64)]).astype(np.int64)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    dev = [d(words.view(np.int32)), d(off), d(cnt), d(lengths), d(toff)]
    out = torch.zeros(len(tokens), dtype=torch.uint8, device="cuda")
    status = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    ws = codec._decompress_workspace(n)
    monkeypatch.setenv("SC_HIP_DEC_FED", rt)
    want = np.zeros(n, np.int32)
    want[bad] = _hip.SC_STATUS_INVALID_STREAM
    keep = np.ones(len(tokens), bool)
    keep[toff[bad]:toff[bad] + lengths[bad]] = False
    for spin in ("0", None):
        if spin is None:
            monkeypatch.delenv("SC_HIP_DEC_SPIN")
        else:
            monkeypatch.setenv("SC_HIP_DEC_SPIN", spin)
        out.zero_()
        status.fill_(-1)
        _hip.check(_hip.lib().sc_decompress_chunks(
            codec.hip.handle, *[x.data_ptr() for x in dev[:4]], n, out.data_ptr(), dev[4].data_ptr(), status.data_ptr(),
            lengths.ctypes.data, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert np.array_equal(status.cpu().numpy(), want), spin
        assert np.array_equal(out.cpu().numpy()[keep], tokens[keep]), spin


@pytest.mark.parametrize("n,longest,what", [(700, 1, "split launch p8"), (700, 8, "fed launch"), (1100, 1, "split launch p4"),
                                            (8191, 2, "launch"), (8191, 30, "fed launch"), (4000, 1, "launch"),
                                            (4000, 3, "fed launch")])
def test_few_steps_run_without_feeders(codec, monkeypatch, capfd, n, longest, what):
    """A fed launch starts 30 to 60 us later than others (its feeders load
    layer 0): decodes of a step or two take the split or unsplit launch,
    whichever the costs say (8,191 chunks of 1 token: 133 us fed, 88
    unsplit)."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the chunk counts are for 256 CUs")
    lengths = np.full(n, longest)
    lengths[n // 2:] = max(longest - 1, 1)
    tokens, lengths, words, off, cnt = _chunks(codec, lengths, n)
    monkeypatch.setenv("SC_HIP_DEC_LOG", "1")
    capfd.readouterr()
    back = np.array(codec.decompress_flat(words, off, cnt, lengths)[0])
    log = capfd.readouterr().err
    assert f"leftover {n} {what} steps {longest} " in log, log
    assert np.array_equal(back, tokens)
