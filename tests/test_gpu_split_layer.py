"""Layers with tensors on both sides of k = 1024 through
hh_hctt_decode_lz4_batch, which decodes the two kinds beside each other on
two streams: the records, the tile bytes and the weights of the
one-stream route (a chosen LZ4 decoder), bit for bit, over orders of the
tensors, output types, blocks that hold bytes of both kinds, failed blocks,
tensors that share memory, other streams, several threads and a captured
call."""
import threading

import numpy as np
import pytest

import gpu_util as G

pytestmark = pytest.mark.gpu

DENSE, DENSE2, SPARSE, SPARSE2 = (4096, 6144, 0.30), (512, 4096, 0.45), (1024, 2048, 0.10), (640, 1024, 0.20)
DTYPES = {"f32": 4, "f16": 2, "bf16": 2}


def layer(specs, seed, cut=None, gap=0, most=1 << 30):
    """The tensors' tile bytes one after another (`gap` bytes between them),
    in blocks of whole tiles (`most` of them at most) or, with `cut`, of that
    many bytes across the tensors.  A tensor repeats 64 encoded tiles."""
    import haagenti_amd as H
    rng = np.random.default_rng(seed)
    comp = H.Lz4Compressor()
    raw, tensors, ends = [], [], []
    for rows, cols, rho in specs:
        k = H.hctt_retain_count(rho)
        base = H.hctt_encode(rng.normal(0, 0.02, (512, 512)).astype(np.float32), k).reshape(64, -1)
        tiles = base[rng.integers(0, 64, rows * cols // 4096)].reshape(-1)
        soff = sum(r.size for r in raw)
        tensors.append(dict(rows=rows, cols=cols, k=k, soff=soff, n=tiles.size))
        raw += [tiles, np.zeros(gap, np.uint8)]
    raw = np.concatenate(raw)
    if cut:
        starts = [(a, min(a + cut, raw.size)) for a in range(0, raw.size, cut)]
    else:
        starts = []
        for t in tensors:
            t["per"] = min(most, 16352 // H.hctt_tile_bytes(t["k"]))
            per = t["per"] * H.hctt_tile_bytes(t["k"])
            starts += [(a, min(a + per, t["soff"] + t["n"])) for a in range(t["soff"], t["soff"] + t["n"], per)]
    seen, blobs = {}, []
    for a, b in starts:
        chunk = raw[a:b].tobytes()
        if chunk not in seen:
            seen[chunk] = comp.compress(chunk)
        blobs.append(seen[chunk])
    lens = np.array([len(b) for b in blobs], np.uint32)
    return dict(tensors=tensors, raw=raw, blob=np.frombuffer(b"".join(blobs), np.uint8).copy(), in_len=lens,
                in_off=np.concatenate([[0], np.cumsum(lens.astype(np.uint64))[:-1]]).astype(np.uint64),
                out_off=np.array([a for a, _ in starts], np.uint64),
                out_cap=np.array([b - a for a, b in starts], np.uint32))


class Call:
    """One layer on the device and its buffers; run() decodes it."""

    def __init__(self, L, dtype="bf16", ctx=None):
        T = G.torch()
        import haagenti_amd as H
        self.L, self.ctx = L, ctx or G.ctx()
        self.dt = {"f32": H.F32, "f16": H.F16, "bf16": H.BF16}[dtype]
        self.args = [G.dev(L[x]) for x in ("blob", "in_off", "in_len", "out_off", "out_cap")]
        self.n = L["in_len"].size
        self.st = T.empty(self.n * 32, dtype=T.uint8, device="cuda")
        self.scratch = T.empty(L["raw"].size, dtype=T.uint8, device="cuda")
        sizes = [t["rows"] * t["cols"] * DTYPES[dtype] for t in L["tensors"]]
        self.out = T.empty(sum(sizes), dtype=T.uint8, device="cuda")
        self.tst = T.empty(sum(sizes) // DTYPES[dtype] // 4096, dtype=T.int32, device="cuda")
        self.tensors, o, ts = [], 0, 0
        for t, size in zip(L["tensors"], sizes):
            self.tensors.append((self.scratch.data_ptr() + t["soff"], t["n"], t["rows"], t["cols"], t["k"],
                                 self.out.data_ptr() + o, self.tst.data_ptr() + 4 * ts))
            o += size
            ts += t["rows"] * t["cols"] // 4096
        T.cuda.synchronize()

    def run(self, stream=None):
        blob, io, il, oo, oc = self.args
        self.ctx.hctt_decode_lz4_batch(blob, blob.numel(), io, il, self.scratch, oo, oc, self.n, self.st,
                                       self.tensors, dtype=self.dt, stream=G.stream() if stream is None else stream)

    def clear(self):
        for x in (self.st, self.scratch, self.out, self.tst):
            x.fill_(77)

    def results(self):
        G.sync()
        return [x.clone() for x in (self.st, self.scratch, self.out, self.tst)]


def general(call):
    """The one-stream route's results."""
    call.clear()
    call.ctx.set_lz4_decoder("seq")
    try:
        call.run()
    finally:
        call.ctx.set_lz4_decoder("auto")
    return call.results()


def same(a, b):
    T = G.torch()
    return all(T.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("dtype", sorted(DTYPES))
@pytest.mark.parametrize("order", [(0, 1, 2, 3), (2, 0, 3, 1), (3, 2, 1, 0)])
def test_against_one_stream(dtype, order):
    specs = [(DENSE, DENSE2, SPARSE, SPARSE2)[i] for i in order]
    c = Call(layer(specs, 1, gap=4 * order[0]), dtype)
    want = general(c)
    assert (want[0].view(G.torch().int32)[0::8] == 0).all() and (want[3] == 0).all()
    for _ in range(3):
        c.clear()
        c.run()
        assert same(c.results(), want)


def test_blocks_of_both_kinds_and_failed_blocks():
    L = layer([SPARSE, DENSE, SPARSE2, DENSE2], 2, cut=10007)
    c = Call(L)
    want = general(c)
    c.clear()
    c.run()
    assert same(c.results(), want)
    L = layer([DENSE, SPARSE, SPARSE2], 3)
    n = L["in_len"].size
    L["in_len"][[5, n - 200, n - 3]] = [0, 3, 1]            # cut short
    L["in_off"][[9, n - 7]] = 1 << 40                       # outside the input
    L["out_cap"][[11, n - 9]] -= 100                        # too small a capacity
    c = Call(L)
    want = general(c)
    assert (want[0].view(G.torch().int32)[0::8] != 0).sum() >= 5
    c.clear()
    c.run()
    assert same(c.results(), want)


def test_outputs_over_the_compressed_input():
    # legal with one stream (the tiles run after every block): kept so
    T = G.torch()
    c = Call(layer([DENSE, SPARSE], 4))
    want = general(c)
    blob, at = c.args[0].clone(), c.out.numel() - c.args[0].numel() & ~255
    c.out[at:at + blob.numel()] = blob
    c.args[0] = c.out[at:at + blob.numel()]
    T.cuda.synchronize()
    c.run()
    assert same(c.results(), want)


def test_streams_threads_and_capture():
    T = G.torch()
    ctx = G.ctx()
    calls = [Call(layer([DENSE, SPARSE, SPARSE2], 5 + i), ctx=ctx) for i in range(3)]
    want = [general(c) for c in calls]
    for c in calls:
        c.clear()
    T.cuda.synchronize()
    streams = [T.cuda.Stream() for _ in calls]

    def work(c, s):
        for _ in range(8):
            c.run(s.cuda_stream)

    threads = [threading.Thread(target=work, args=a) for a in zip(calls, streams)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    T.cuda.synchronize()
    for c, w in zip(calls, want):
        assert same(c.results(), w)
    # captured: one stream; an eager call of the same context meanwhile
    g = T.cuda.CUDAGraph()
    with T.cuda.graph(g):
        calls[0].run()
        calls[1].run(streams[1].cuda_stream)
    T.cuda.synchronize()
    assert same(calls[1].results(), want[1])
    for _ in range(3):
        calls[0].clear()
        g.replay()
        assert same(calls[0].results(), want[0])
        calls[2].run()
        assert same(calls[2].results(), want[2])


def test_calls_on_other_streams_do_not_wait():
    # neither for what a caller has put on the context's stream, nor for an
    # earlier call on a stream that is still busy
    T = G.torch()
    ctx = G.ctx()
    calls = [Call(layer([DENSE, SPARSE, SPARSE2], 5 + i), ctx=ctx) for i in range(2)]
    want = [general(c) for c in calls]
    m = T.randn(8192, 8192, device="cuda")

    def busy(stream):
        # about 100 ms: long after the layer's call has returned and run
        with T.cuda.stream(stream):
            for _ in range(12):
                m @ m
            return stream.record_event()

    def beside(*others):
        # a stream that shares no hardware queue with those
        for _ in range(16):
            x, free = T.cuda.Stream(), True
            for o in others:
                done = busy(o)
                with T.cuda.stream(x):
                    T.zeros(1, device="cuda")
                x.synchronize()
                free = free and not done.query()
                T.cuda.synchronize()
            if free:
                return x
        pytest.skip("every stream shares a hardware queue with one of those")

    own = T.cuda.ExternalStream(ctx.stream)
    s = beside(own)
    calls[0].clear()
    T.cuda.synchronize()
    for _ in range(8):          # each after the halves of the one before
        calls[0].run(s.cuda_stream)
    assert same(calls[0].results(), want[0])
    calls[0].clear()
    T.cuda.synchronize()
    done = busy(own)
    calls[0].run(s.cuda_stream)
    s.synchronize()
    assert not done.query()
    assert same(calls[0].results(), want[0])
    t = beside(s, own)
    for c in calls:
        c.clear()
    T.cuda.synchronize()
    done = busy(s)
    calls[0].run(s.cuda_stream)
    calls[1].run(t.cuda_stream)
    t.synchronize()
    assert not done.query()
    for c, w in zip(calls, want):
        assert same(c.results(), w)
