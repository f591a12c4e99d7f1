"""Blocks of many short LZ4 sequences on the sequence-batched decoder
(csrc/lz4_seq.hpp), against the oracle: the edges of what its token walk
takes (literal lengths without, with one and with two extension bytes, match
lengths without and with one), more sequences than its list and a batch
hold, tokens on every position of the 64-byte windows and of the stage's
end, matches that chain through one batch, repeat their own bytes or reach
back past the ring; and tiles of very low retention through both layer
routes."""
import numpy as np
import pytest

import gpu_util as G
import oracle_lib as O
from test_gpu_lz4 import _seq, check_against_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True, params=["seq", "seq8"])
def decoder(request):
    G.ctx().set_lz4_decoder(request.param)
    yield request.param
    G.ctx().set_lz4_decoder("auto")


def stream(rng, nseq, lits, mls, offs):
    """nseq sequences with lengths and offsets drawn from the given lists
    (an offset is kept within the output), ending with literals."""
    out, size = bytearray(_seq(bytes(rng.integers(0, 256, 40, dtype=np.uint8)), 7, 5)), 45
    for _ in range(nseq):
        n, m = int(rng.choice(lits)), int(rng.choice(mls))
        off = min(int(rng.choice(offs)), size + n)
        out += _seq(bytes(rng.integers(0, 256, n, dtype=np.uint8)), off, m)
        size += n + m
    tail = bytes(rng.integers(0, 256, 9, dtype=np.uint8))
    return bytes(out + _seq(tail)), size + 9


CASES = {
    "shortest": ([0], [4], [1, 2, 3, 4, 5, 60, 300]),
    "no_extension": (range(0, 15), range(4, 19), range(1, 400)),
    "one_literal_byte": ([0, 3, 14, 15, 16, 100, 268, 269], [4, 5, 18], range(1, 3000)),
    "two_literal_bytes": ([5, 269, 270, 271, 524, 525], [4, 9], range(1, 3000)),
    "match_extension": ([0, 1, 7], [4, 18, 19, 20, 270, 273, 274], [1, 2, 5, 17, 400]),
    "chained": ([0, 1, 2], [4, 5, 8], [4, 5, 6, 7, 8]),
    "far": ([2, 6, 9], [4, 5, 8, 9, 10, 18], [3900, 4000, 4032, 4064, 4096, 8100, 8192, 12000]),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_short_sequences(case):
    lits, mls, offs = (list(x) for x in CASES[case])
    rng = np.random.default_rng(sorted(CASES).index(case))
    items = [stream(rng, n, lits, mls, offs) for n in (1, 3, 62, 63, 64, 65, 127, 200, 255, 256, 257, 1500)]
    # every start within a window, and lengths that move the stage's ends
    items += [stream(rng, 700 + i, lits, mls, offs) for i in range(24)]
    streams, caps = [s for s, _ in items], [c for _, c in items]
    for in_align, out_align in ((0, 0), (5, 11)):
        check_against_oracle(streams, caps, in_align=in_align, out_align=out_align, in_pad=in_align, out_pad=3)
    # a capacity that ends inside a batch, and damaged bytes: the same records
    check_against_oracle(streams, [c * 2 // 3 for c in caps], out_pad=3)
    broken = []
    for s in streams:
        b = bytearray(s)
        b[int(rng.integers(len(b) // 3, len(b)))] ^= int(rng.integers(1, 256))
        broken.append(bytes(b))
    check_against_oracle(broken, caps, out_pad=3)


def after_long_run(rng, ring, first, mlen, off, tail=5):
    """`first` literals and a match of `mlen` bytes from ring - 128 back
    (copied as long runs, a batch that ends there), then a match of 4 from
    `off` back and the last literals: a batch of 4 + `tail` bytes, whose
    source lies where the long run's last chunk of 16 bytes ends."""
    out = _seq(bytes(rng.integers(0, 256, first, dtype=np.uint8)), ring - 128, mlen)
    out += _seq(b"", off, 4) + _seq(bytes(rng.integers(0, 256, tail, dtype=np.uint8)))
    return out, first + mlen + 4 + tail


@pytest.mark.parametrize("tail", [5, 7, 11, 13])
def test_short_batch_after_a_long_run(decoder, tail):
    # every alignment of the long run's end, sources around the ring's end
    ring = 8192 if decoder == "seq8" else 4096
    rng = np.random.default_rng(ring + tail)
    items = [after_long_run(rng, ring, 2 * ring + 1900 + a, 61 + b, ring - o, tail)
             for a in range(16) for b in (0, 1) for o in range(-2, 42)]
    for out_align in (0, 9):
        check_against_oracle([s for s, _ in items], [c for _, c in items], out_align=out_align, out_pad=3)


@pytest.mark.parametrize("seed", range(4))
def test_long_runs_between_short_sequences(decoder, seed):
    # batches of long runs and of a few short sequences by turns
    ring = 8192 if decoder == "seq8" else 4096
    rng = np.random.default_rng(100 * seed + ring)
    items = []
    for _ in range(96):
        out, size = bytearray(), 0
        for _ in range(6):
            n, m = int(rng.integers(300, 3000)), int(rng.integers(40, 80))
            size += n
            out += _seq(bytes(rng.integers(0, 256, n, dtype=np.uint8)), min(size, ring - 128 - int(rng.integers(3))), m)
            size += m
            for _ in range(int(rng.integers(1, 4))):
                m, n = int(rng.integers(4, 7)), int(rng.integers(0, 3))
                size += n
                out += _seq(bytes(rng.integers(0, 256, n, dtype=np.uint8)), min(size, ring - int(rng.integers(-4, 64))), m)
                size += m
        out += _seq(bytes(rng.integers(0, 256, 5, dtype=np.uint8)))
        items.append((bytes(out), size + 5))
    check_against_oracle([s for s, _ in items], [c for _, c in items], out_align=seed * 5, out_pad=3)


def test_length_extensions_across_stages(decoder):
    # lengths whose extension bytes end before, at and past one and two input
    # stages (4 KiB, or 2 KiB with the 8 KiB ring), from several positions in
    # a stage, whole, cut short, and with too small a capacity
    stage = 2048 if decoder == "seq8" else 4096
    rng = np.random.default_rng(stage)
    streams, caps = [], []
    for n in (stage - 8, stage + 1, 2 * stage + 9):
        for at in (0, 1, 100, stage - 70):
            head = bytes(rng.integers(0, 256, at + 1, dtype=np.uint8))
            lit = bytes(rng.integers(0, 256, 4096, dtype=np.uint8)) * (n * 255 // 4096 + 1)
            lit = lit[:15 + 255 * n + at % 255]
            for s, c in ((_seq(head, 1, 9) + _seq(lit, 60000, 30) + _seq(b"tail5"), at + len(lit) + 45),
                         (_seq(head, at // 2 + 1, 19 + 255 * n + at) + _seq(b"tail5"), at + 25 + 255 * n + at),
                         (_seq(head, 1, 9) + _seq(b"", at // 2 + 1, 19 + 255 * n) + _seq(b"tail5"),
                          at + 34 + 255 * n)):
                streams += [s, s[:at + 10 + n // 2], s]
                caps += [c, c, c - 7]
    check_against_oracle(streams, caps, in_pad=3, out_pad=3)


@pytest.mark.parametrize("mls", [[4, 5, 18], [4, 19], [200, 640]])
@pytest.mark.parametrize("mean", [128, 250, 330, 640, 660, 1300])
def test_long_literals(mean, mls):
    # literals around the averages from which runs are copied one per pass,
    # with matches that are all short, partly or none
    rng = np.random.default_rng(mean + len(mls))
    items = [stream(rng, 60 + i, list(range(mean - 100, mean + 100)), mls, [1, 3, 17, 800, 3000, 4090, 8000])
             for i in range(16)]
    check_against_oracle([s for s, _ in items], [c for _, c in items], out_align=7, out_pad=3)


@pytest.mark.parametrize("rho", [0.05, 0.10, 0.15, 0.20])
def test_sparse_tiles_on_both_routes(rho):
    import haagenti_amd as H
    from layer_util import encode_layer
    T = G.torch()
    k = H.hctt_retain_count(rho)
    shapes = [("a", 256, 1024), ("b", 640, 512)]
    L = encode_layer(H, shapes, [k, H.hctt_retain_count(0.3)], 11, 16352)
    d_in, n = G.dev(L["blob"]), L["in_off"].size
    st = T.zeros(n * 32, dtype=T.uint8, device="cuda")
    scratch = T.zeros(L["scratch_bytes"], dtype=T.uint8, device="cuda")
    two = [T.empty(t["rows"] * t["cols"], dtype=T.float32, device="cuda") for t in L["tensors"]]
    one = [T.empty_like(o) for o in two]
    G.ctx().hctt_decode_lz4_batch(
        d_in, d_in.numel(), G.dev(L["in_off"]), G.dev(L["in_len"]), scratch, G.dev(L["out_off"]), G.dev(L["out_cap"]),
        n, st, [(scratch.data_ptr() + t["soff"], t["tiles"].size, t["rows"], t["cols"], t["k"], o)
                for t, o in zip(L["tensors"], two)], stream=G.stream())
    G.sync()
    want = np.concatenate([t["tiles"].ravel() for t in L["tensors"]])
    assert np.array_equal(G.host_u8(scratch), want)
    rc = G.ctx().hctt_decode_lz4_fused(
        d_in, d_in.numel(), G.dev(L["in_off"]), G.dev(L["in_len"]), n, st,
        [(t["rows"], t["cols"], t["k"], o) for t, o in zip(L["tensors"], one)],
        [16352 // H.hctt_tile_bytes(t["k"]) for t in L["tensors"]], stream=G.stream())
    assert rc == H.OK
    G.sync()
    assert (G.host_u8(st).view(np.int32)[0::8] == 0).all()
    for a, b in zip(two, one):
        assert T.equal(a, b)
