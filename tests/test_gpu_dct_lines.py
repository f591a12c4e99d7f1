"""The two-pass whole-matrix transforms (csrc/dct_lines.hip) at the lengths
where they can go wrong: one line, odd numbers of lines and lengths, every
radix and the direct sums of the other primes, padded and unpadded LDS
layouts, the longest lines, columns that go to the result by way of panels
(more than 8192 rows) with ragged tiles, panels that several workgroups share,
outputs that are not aligned; and HCT3 fragments whose rows start inside a
bitmap byte.

Bound: a length-N f32 FFT has a relative 2-norm error of about
0.6 eps sqrt(log2 N) per pass (eps = 2^-24 roundings of the sums, as much
again from the rounded twiddles), at most 1.4e-7 for N <= 2^14; a direct sum
over p <= 127 terms adds about eps sqrt(p) / 2 = 3.4e-7.  Two passes in
quadrature: below 5.2e-7, tested at 1e-6."""
import numpy as np
import pytest

import gpu_util as G
import oracle_lib as O
from test_gpu_hct3 import H, dec, rel_err, route
from test_oracle_hct3 import container, random_fragment

pytestmark = pytest.mark.gpu
REL = 1e-6


def basis64(n):
    T = G.torch()
    k = T.arange(n, device="cuda")[:, None]
    i = T.arange(n, device="cuda")[None, :]
    m = T.cos((k * (2 * i + 1) % (4 * n)).double() * (np.pi / (2 * n))) * np.sqrt(2.0 / n)
    m[0] = np.sqrt(1.0 / n)
    return m


@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 77), (2, 3), (16, 17), (37, 53), (127, 126), (143, 11), (48, 80),
                                       (320, 448), (576, 576), (640, 1376), (2752, 96), (255, 1000), (16384, 34),
                                       (33, 16384), (11008, 64), (64, 14336), (4096, 66), (8505, 5), (8232, 64),
                                       (9000, 67), (16384, 129), (12288, 1025), (301, 9000)])
def test_transforms_vs_f64(rows, cols):
    T, h, c = G.torch(), H(), G.ctx()
    x = T.randn(rows, cols, device="cuda", generator=T.Generator(device="cuda").manual_seed(rows + cols))
    br, bc, xd = basis64(rows), basis64(cols), x.double()
    fwd = T.empty(rows * cols, device="cuda")
    inv = T.empty(rows * cols, device="cuda")
    c.dct_2d(x, rows, cols, fwd, stream=G.stream())
    c.idct_2d(x, rows, cols, inv, stream=G.stream())
    for got, ref in ((fwd, br @ xd @ bc.t()), (inv, br.t() @ xd @ bc)):
        e = float((got.view(rows, cols).double() - ref).norm() / ref.norm())
        assert e <= REL, e
    # 16-bit outputs are the rounding of the f32 result, at any element address
    for dt, td in ((h.BF16, T.bfloat16), (h.F16, T.float16)):
        for off in (0, 1):
            out = T.full((rows * cols + 2,), 7.0, dtype=td, device="cuda")
            c.idct_2d(x, rows, cols, out.data_ptr() + 2 * off, dtype=dt, stream=G.stream())
            G.sync()
            assert T.equal(out[off:off + rows * cols], inv.to(td))
            assert bool((out[off + rows * cols:] == 7).all()) and (off == 0 or float(out[0]) == 7)


@pytest.mark.parametrize("rows,cols", [(2058, 16384), (4116, 8192)])
def test_rows_32_kib_apart(rows, cols):
    # f32 results of such rows come from panels of one row workgroup each,
    # 16-bit ones from panels that two share
    T, h, c = G.torch(), H(), G.ctx()
    x = T.randn(rows, cols, device="cuda", generator=T.Generator(device="cuda").manual_seed(rows + cols))
    inv = T.empty(rows * cols, device="cuda")
    half = T.empty(rows * cols, dtype=T.bfloat16, device="cuda")
    for _ in range(2):  # the second with the other's intermediate in place
        c.idct_2d(x, rows, cols, inv, stream=G.stream())
        c.idct_2d(x, rows, cols, half, dtype=h.BF16, stream=G.stream())
        G.sync()
        assert T.equal(half, inv.to(T.bfloat16))
    ref = basis64(rows).t() @ x.double() @ basis64(cols)
    e = float((inv.view(rows, cols).double() - ref).norm() / ref.norm())
    assert e <= REL, e


@pytest.mark.parametrize("rows,cols", [(2048, 4096), (2047, 4096), (2057, 4095), (1025, 8190), (513, 16384), (8192, 1025),
                                       (5504, 1533)])
def test_forward_panels_apart(rows, cols):
    # from 2^23 elements on (8192 rows at most) there are two points between
    # the panels of the rows; ragged last panels, prime passes
    T, c = G.torch(), G.ctx()
    x = T.randn(rows, cols, device="cuda", generator=T.Generator(device="cuda").manual_seed(rows + cols))
    out = T.empty(rows * cols, device="cuda")
    c.dct_2d(x, rows, cols, out, stream=G.stream())
    ref = basis64(rows) @ x.double() @ basis64(cols).t()
    e = float((out.view(rows, cols).double() - ref).norm() / ref.norm())
    assert e <= REL, e


@pytest.mark.parametrize("rows,cols", [(1, 31), (127, 1), (11, 13), (127, 127), (8001, 3), (2, 8001), (8128, 3),
                                       (1651, 140), (140, 2431), (961, 600), (1016, 300), (3, 16002)])
def test_prime_passes(rows, cols):
    # one to 63 butterflies to a workgroup (a thread per output pair; 3,969
    # pairs, four to a thread, at 63 x 127) and 64 (one more: wave tasks), both
    # in one length (127 x 13, 11 x 13 x 17), and passes after others
    T, c = G.torch(), G.ctx()
    x = T.randn(rows, cols, device="cuda", generator=T.Generator(device="cuda").manual_seed(rows + cols))
    br, bc, xd = basis64(rows), basis64(cols), x.double()
    out = T.empty(rows * cols, device="cuda")
    for f, ref in ((c.dct_2d, br @ xd @ bc.t()), (c.idct_2d, br.t() @ xd @ bc)):
        f(x, rows, cols, out, stream=G.stream())
        e = float((out.view(rows, cols).double() - ref).norm() / ref.norm())
        assert e <= REL, e


@pytest.mark.parametrize("shape", [(97, 131), (64, 1000), (1000, 77), (1, 3000), (130, 2048)])
def test_fragments_whose_rows_start_inside_a_byte(shape):
    rng = np.random.default_rng(shape[0])
    total = shape[0] * shape[1]
    bm, v, _ = random_fragment(rng, total, 0.05)
    data = container([random_fragment(rng, total, 0.3), (bm, v[:v.size // 2], None),
                      random_fragment(rng, total, 0.01)])
    rc, ref = O.hct3_decode(data, shape)
    assert rc == O.OK
    got = dec().decompress_to_gpu(data, shape).cpu().numpy()
    assert rel_err(got, ref) <= 1e-5
    with route("dense"):
        dense = dec().decompress_to_gpu(data, shape).cpu().numpy()
    assert rel_err(got, dense) <= 2e-5


@pytest.mark.parametrize("nfrag", [1, 3, 16])
@pytest.mark.parametrize("rows,cols", [(3, 16), (64, 64), (1024, 256), (1024, 512), (1027, 300), (300, 700), (2048, 520),
                                       (1300, 1024), (4100, 64), (9000, 33), (16384, 34), (2310, 1152), (600, 5120)])
def test_fragments_by_workgroup_size(rows, cols, nfrag):
    # one to sixteen waves to a workgroup, one to four to a line, with idle
    # lanes (short lines), ragged last workgroups and several of them to a CU
    T, c = G.torch(), G.ctx()
    rng = np.random.default_rng(rows + cols + nfrag)
    total = rows * cols
    data = container([random_fragment(rng, total, 0.6 / (f + 2)) for f in range(nfrag)])
    x = dec().reconstruct_coefficients_gpu(data, total).view(rows, cols).double()
    ref = basis64(rows).t() @ x @ basis64(cols)
    got = dec().decompress_to_gpu(data, (rows, cols))
    e = float((got.view(rows, cols).double() - ref).norm() / ref.norm())
    assert e <= REL, e


@pytest.mark.parametrize("rows,cols", [(2, 64), (16, 80), (64, 1024), (1024, 192), (512, 1000), (260, 5120), (5120, 64),
                                       (1030, 514), (4096, 72), (9000, 65), (1376, 513)])
def test_small_passes_of_many_waves(rows, cols):
    # more waves than radix-16 butterflies need, with every lane or only some
    # at work, one to a few workgroups to a CU, a prime pass, panels of columns
    T, c = G.torch(), G.ctx()
    x = T.randn(rows, cols, device="cuda", generator=T.Generator(device="cuda").manual_seed(rows + cols))
    br, bc, xd = basis64(rows), basis64(cols), x.double()
    out = T.empty(rows * cols, device="cuda")
    for f, ref in ((c.dct_2d, br @ xd @ bc.t()), (c.idct_2d, br.t() @ xd @ bc)):
        f(x, rows, cols, out, stream=G.stream())
        e = float((out.view(rows, cols).double() - ref).norm() / ref.norm())
        assert e <= REL, e


@pytest.mark.parametrize("rows,cols", [(4096, 1280), (4100, 1280), (5324, 1287), (1280, 4200), (2560, 2562)])
def test_workgroups_past_one_round(rows, cols):
    # 256 workgroups and a few more, up to three tenths more
    T, c = G.torch(), G.ctx()
    x = T.randn(rows, cols, device="cuda", generator=T.Generator(device="cuda").manual_seed(rows + cols))
    br, bc, xd = basis64(rows), basis64(cols), x.double()
    out = T.empty(rows * cols, device="cuda")
    for f, ref in ((c.dct_2d, br @ xd @ bc.t()), (c.idct_2d, br.t() @ xd @ bc)):
        f(x, rows, cols, out, stream=G.stream())
        e = float((out.view(rows, cols).double() - ref).norm() / ref.norm())
        assert e <= REL, e
