"""GPU tests of the decode's rotating launches (chunk counts between whole
waves of workgroups): every workgroup size, sorted and unsorted chunks, empty
and corrupt ones, a workspace that holds another call's state, and graph
capture, against the input and the plan of full waves."""

import re

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


class _Call:
    """One sc_decompress_chunks call with its device buffers."""

    def __init__(self, codec, words, woff, wcnt, lengths):
        from sigcomp_amd import _hip
        self.hip, self.codec, self.n = _hip, codec, len(lengths)
        toff = np.concatenate([[0], np.cumsum(lengths[:-1], dtype=np.int64)]).astype(np.int64)
        self.host = np.ascontiguousarray(lengths, np.int32)
        self.dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda()
                    for a in (words.view(np.int32), woff.astype(np.int64), wcnt.astype(np.int32), self.host, toff)]
        self.tokens = torch.zeros(int(lengths.sum()), dtype=torch.uint8, device="cuda")
        self.status = torch.full((self.n,), -1, dtype=torch.int32, device="cuda")
        self.ws = torch.full((_hip.lib().sc_decompress_workspace_bytes(self.n),), 1, dtype=torch.uint8, device="cuda")

    def enqueue(self):
        p = self.hip.ptr
        w, wo, wc, ln, to = self.dev
        self.hip.check(self.hip.lib().sc_decompress_chunks(
            self.codec.hip.handle, p(w), p(wo), p(wc), p(ln), self.n, p(self.tokens), p(to), p(self.status),
            self.host.ctypes.data, p(self.ws), self.ws.numel(), self.hip.stream_ptr()))

    def results(self):
        torch.cuda.synchronize()
        return self.tokens.cpu().numpy(), self.status.cpu().numpy()


def _inputs(codec, n, longest, seed):
    """Chunks of `longest` tokens and a tenth of them shorter (empty ones and
    segment edges among them); some are given a corrupt stream."""
    rng = np.random.default_rng(seed)
    lengths = np.full(n, longest, np.int32)
    short = rng.choice(n, n // 10, replace=False)
    lengths[short] = rng.integers(0, longest, len(short))
    edges = [e for e in (0, 1, 63, 64, 65, 127, 128, 129, 255, 256, 257) if e <= longest]
    lengths[short[:len(edges)]] = edges
    tokens = rng.integers(0, 60, int(lengths.sum())).astype(np.uint8)
    words, woff, wcnt = (np.array(a) for a in codec.compress_flat(tokens, lengths))
    words = np.concatenate([words, np.full(2, 0xFFFFFFFF, np.uint32)])
    bad = np.concatenate([rng.choice(np.flatnonzero(lengths == longest), 3, replace=False), [n - 1]])
    lengths_ok = lengths[bad] > 0
    bad = bad[lengths_ok]
    woff[bad], wcnt[bad] = len(words) - 2, 2
    return tokens, lengths, words, woff, wcnt, bad


# waves of 32-chunk workgroups on all CUs, the longest chunk, the workgroup
# size (row tiles) that the step costs choose for sorted chunks
@pytest.mark.parametrize("order", ["sorted", "as given"])
@pytest.mark.parametrize("waves,longest,rt", [(1.1, 512, 1), (1.5, 300, 2), (2.5, 512, 2), (3.5, 512, 3), (6.3, 257, None)])
def test_rotating_decode(codec, monkeypatch, capfd, waves, longest, rt, order):
    n = int(waves * 32 * torch.cuda.get_device_properties(0).multi_processor_count) + 5
    tokens, lengths, words, woff, wcnt, bad = _inputs(codec, n, longest, n)
    start = np.concatenate([[0], np.cumsum(lengths[:-1], dtype=np.int64)])
    o = np.argsort(-lengths, kind="stable") if order == "sorted" else np.arange(n)
    call = _Call(codec, words, woff[o], wcnt[o], lengths[o])
    monkeypatch.setenv("SC_HIP_DEC_LOG", "1")
    capfd.readouterr()
    call.enqueue()
    got, status = call.results()
    m = re.search(r"rotating launches: rt (\d)", capfd.readouterr().err)
    if order == "sorted" and rt and torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert m and int(m.group(1)) == rt
    want_status = np.zeros(n, np.int32)
    want_status[np.isin(o, bad)] = 2   # SC_STATUS_INVALID_STREAM
    assert np.array_equal(status, want_status)
    off = np.concatenate([[0], np.cumsum(lengths[o][:-1], dtype=np.int64)])
    keep = np.ones(len(got), bool)
    for i in np.flatnonzero(want_status):
        keep[off[i]:off[i] + lengths[o[i]]] = False
    want = np.concatenate([tokens[start[c]:start[c] + lengths[c]] for c in o])
    assert np.array_equal(got[keep], want[keep])
    # the plan of full waves: the same status and tokens
    monkeypatch.setenv("SC_HIP_DEC_SPLIT", "0")
    call.tokens.zero_()
    call.status.fill_(-1)
    call.enqueue()
    plain, plain_status = call.results()
    assert "rotating" not in capfd.readouterr().err
    assert np.array_equal(plain_status, status) and np.array_equal(plain[keep], got[keep])


def test_rotating_decode_under_graph_capture(codec, monkeypatch, capfd):
    """Captured once, replayed three times with eager work between."""
    n = int(1.5 * 32 * torch.cuda.get_device_properties(0).multi_processor_count)
    rng = np.random.default_rng(12)
    lengths = np.sort(rng.integers(200, 301, n).astype(np.int32))[::-1].copy()
    tokens = rng.integers(0, 60, int(lengths.sum())).astype(np.uint8)
    words, woff, wcnt = (np.array(a) for a in codec.compress_flat(tokens, lengths))
    call = _Call(codec, words, woff, wcnt, lengths)
    monkeypatch.setenv("SC_HIP_DEC_LOG", "1")
    capfd.readouterr()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        call.enqueue()
    assert "rotating" in capfd.readouterr().err
    for rep in range(3):
        call.tokens.fill_(0xAB)
        call.status.fill_(-1)
        call.ws.fill_(rep)
        torch.cuda.synchronize()
        graph.replay()
        got, status = call.results()
        assert not status.any() and np.array_equal(got, tokens), rep


@pytest.mark.parametrize("n,rotates", [(20480, False), (25000, True)])
def test_batches_of_mostly_short_chunks(codec, monkeypatch, capfd, n, rotates):
    """Full waves whose workgroups end early take less than their longest
    chunks' steps, so that rotating launches have to promise more: 65.7 ms as
    full waves and 67.7 rotating for the first of these, 87.8 and 74.8 for
    the second."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the chunk counts are for 256 CUs")
    rng = np.random.default_rng(n)
    lengths = -np.sort(-np.minimum(rng.geometric(1 / 200, n), 1024)).astype(np.int32)
    lengths[0] = 1024
    tokens = rng.integers(0, 60, int(lengths.sum())).astype(np.uint8)
    words, woff, wcnt = (np.array(a) for a in codec.compress_flat(tokens, lengths))
    monkeypatch.setenv("SC_HIP_DEC_LOG", "1")
    capfd.readouterr()
    back, _ = codec.decompress_flat(words, woff, wcnt, lengths)
    assert ("rotating" in capfd.readouterr().err) == rotates
    assert np.array_equal(back, tokens)
