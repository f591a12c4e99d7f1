"""Uploads through pinned staging: chunk edges of a file's upload, spectral
tensors whose container lies in the staging buffer (copied piece by piece),
is put together there (gaps, many fragments, a frame larger than the buffer)
or in ordinary memory, one after the other on one context; and that nothing
reaches the output before every check has passed.

Bound: both sides of the comparison are the two-pass f32 transforms of the
same coefficients, each within 5.2e-7 of f64 (test_gpu_dct_lines.py); twice
that, rounded up."""
import struct

import numpy as np
import pytest

import gpu_util as G
from test_gpu_hct3 import H

pytestmark = pytest.mark.gpu
REL = 1.1e-6


@pytest.mark.parametrize("n", [1, (1 << 20) - 1, 1 << 20, (1 << 20) + 1, 8 << 20, (8 << 20) + 1, (19 << 20) + 3])
def test_upload_is_whole(n):
    data = np.random.default_rng(n).integers(0, 256, n, np.uint8).tobytes()
    assert H()._upload(data).cpu().numpy().tobytes() == data


def tensor(rows, cols, keep, frags, f32, drop, seed=3):
    """([(index, bytes)], dense coefficients) with fragment `drop` left out."""
    rng = np.random.default_rng(seed)
    mask = rng.random(rows * cols, np.float32) < keep
    n, csz = int(mask.sum()), 4 if f32 else 2
    vals = rng.standard_normal(n, np.float32).astype(np.float32 if f32 else np.float16)
    ess = n if frags == 1 else max(1, n // 5)
    per = 0 if frags == 1 else -(-(n - ess) // (frags - 1))
    v = vals.tobytes()
    out = [(0, struct.pack("<6I", 0x48435432 if f32 else 0x48435433, cols, rows, n, ess, per)
            + np.packbits(mask, bitorder="little").tobytes() + v[:csz * ess])]
    for f in range(1, frags):
        a, b = min(n, ess + (f - 1) * per), min(n, ess + f * per)
        if f == drop:
            vals[a:b] = 0
            continue
        out.append((f, struct.pack("<HHI", f, frags, b - a) + v[csz * a:csz * b]))
    dense = np.zeros(rows * cols, np.float32)
    dense[mask] = vals
    return out, dense


def turbo(frags, rows, cols):
    from haagenti_amd import turbo as T
    w = T.TurboWriter()
    w.add_tensor("t", frags, [rows, cols])
    return w.to_bytes()


@pytest.mark.parametrize("rows,cols,keep,frags,f32,drop",
                         [(64, 48, 0.3, 1, False, 0), (600, 1000, 0.3, 4, False, 0), (601, 999, 0.3, 4, False, 2),
                          (601, 999, 0.3, 4, False, 3), (300, 500, 0.4, 20, False, 0), (1200, 1100, 0.3, 3, True, 0),
                          (4096, 5120, 0.8, 3, False, 0), (4096, 5120, 0.8, 3, False, 1)])
def test_turbo_through_staging(rows, cols, keep, frags, f32, drop):
    from haagenti_amd import turbo as T
    t, c = G.torch(), G.ctx()
    fr, dense = tensor(rows, cols, keep, frags, f32, drop)
    want = t.empty(rows * cols, device="cuda")
    c.idct_2d(t.from_numpy(dense).cuda(), rows, cols, want, stream=G.stream())
    for verify in (True, False):
        got = T.TurboReader(turbo(fr, rows, cols)).decode_gpu("t", c, verify=verify, stream=G.stream()).reshape(-1)
        assert float((got - want).norm() / want.norm()) <= REL


def test_checks_come_before_the_output():
    from haagenti_amd import turbo as T
    t, c, m = G.torch(), G.ctx(), H()
    rows, cols = 200, 300
    fr, dense = tensor(rows, cols, 0.3, 4, False, 0)
    out = t.full((rows * cols,), 7.0, device="cuda")
    raw = m.hct3_container(fr)
    at = raw.index(fr[1][1]) + 100

    def decode(data):
        w, h, st = m._u32(0), m._u32(0), m.BlockStatus()
        rc = m._lib.hh_turbo_tensor_decode(c.handle, data, len(data), 1, m.F32, out.data_ptr(), out.numel(),
                                           m.C.byref(w), m.C.byref(h), m.C.byref(st), G.stream())
        return rc, st.position, (w.value, h.value)
    for wrap in (bytes, T.zstd_frame_raw):
        flip = raw[:at] + bytes([raw[at] ^ 1]) + raw[at + 1:]
        assert decode(wrap(flip))[:2] == (m.CHECKSUM_MISMATCH, 1)
        assert decode(wrap(flip[:-1]))[:2] == (m.CHECKSUM_MISMATCH, 1)     # before the truncated one
        assert decode(wrap(raw[:-1]))[0] == m.CORRUPTED_DATA
        G.sync()
        assert bool((out == 7).all())
        assert decode(wrap(raw))[0] == m.OK
        want = t.empty(rows * cols, device="cuda")
        c.idct_2d(t.from_numpy(dense).cuda(), rows, cols, want, stream=G.stream())
        assert float((out - want).norm() / want.norm()) <= REL
        out.fill_(7.0)
