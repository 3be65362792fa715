"""The two-pass form of the iteration (pk_fold_dev.hpp) against the oracle and
against the three-pass form, which pk_tune_set pins.

Sizes cover its branches: one and two dim-2 steps in the row pass, one to
three steps along the row, none and one dim-2 step in the column pass, one to
three along dim 3, 4-, 8- and 16-column tiles, tiles whose last columns are padding,
one and two row groups per block.  No other test uses these sizes: a pinned
size stays pinned for the process's later plans."""
import threading
import time

import numpy as np
import pytest

import petakit5d_amd as pk
from petakit5d_amd import synth

pytestmark = pytest.mark.gpu

SIZES = [
    (64, 32, 50),    # two row groups per block, one dim-2 step between the rows
    (54, 120, 36),   # rows of 27 pairs, two dim-2 steps
    (60, 48, 30),
    (96, 135, 20),   # odd dim 2
    (128, 36, 45),
    (250, 40, 27),   # three steps of 5 along the row
    (640, 16, 18),   # the smallest dim-2 step
    (30, 540, 16),   # one step along the row, one along dim 3
    (90, 16, 243),   # dim 2 whole in the row pass, three steps along dim 3
    (50, 64, 32),
    (72, 64, 16),
    (54, 1024, 100),  # the largest dim-2 steps, 8-column tiles
    (10, 324, 288),  # 4-column tiles
]


def _volume(shape, seed):
    g = np.random.default_rng(seed)
    psf = synth.gaussian_psf(tuple(min(n, 9) for n in shape), 1.2, 2.0, 10.0)
    img = synth._fft_convolve_circular(synth.point_emitters(shape, 60, (500, 3000), g), psf) + 100
    return synth.poisson_u16(img, g), psf, np.ascontiguousarray(psf[::-1, ::-1, ::-1])


def _rel(a, b):
    a, b = a.astype(np.float64), b.astype(np.float64)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _three_pass(shape, ctx=None):
    """A context (a new one) whose plan of this size is pinned to the three-pass kernels."""
    ctx = ctx or pk.Context(0)
    L = shape[0] // 2
    divisors = [1, 2, 3, 4, 5, 6, 8, 9, 10, 12, 15, 16, 18, 20, 24, 25, 27, 30, 32]

    def cover(n, tile):
        """Values per thread of an all-register plan of n points whose tile fits a 256-thread block."""
        for e in divisors:
            if n % e == 0 and n // e * tile <= 256 and all(e % p == 0 for p in (2, 3, 5) if n % p == 0):
                return e
        return None

    def axis(n):
        for tile in (16, 8, 4, 2, 1):
            if cover(n, tile):
                return cover(n, tile), 256, tile
        raise AssertionError(n)

    ctx.tune_set(shape, (cover(L, 1),) + axis(shape[1]) + axis(shape[2]) + (3,))
    return ctx


@pytest.mark.parametrize("shape", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_two_pass_form_matches_oracle_and_three_pass(oracle, shape):
    I, psf, psf_b = _volume(shape, sum(shape))
    two = pk.Context(0)  # before the pin: plans made later in the process take it
    J2 = pk.decon_lucy_omw_function(I, psf, psf_b, 2, Background=100, save16bit=False, ctx=two)[0]
    R2 = pk.decon_lucy_function(I.astype(np.float32), psf, 4, Background=100, save16bit=False, ctx=two)[0]
    O2 = oracle.decon_lucy_omw_function(I, psf, psf_b, 2, Background=100, save16bit=False)[0]
    OR = oracle.decon_lucy_function(I, psf, 4, Background=100, save16bit=False)[0]
    # 32-bit sums over the transforms: the three-pass form is 2e-7 to 1.4e-6 from 64 bits on such volumes; a wrong
    # index, twiddle or element is off by 1e-3 or more
    assert _rel(J2, O2) <= 1e-5
    assert _rel(R2, OR) <= 1e-5
    three = _three_pass(shape)
    J3 = pk.decon_lucy_omw_function(I, psf, psf_b, 2, Background=100, save16bit=False, ctx=three)[0]
    R3 = pk.decon_lucy_function(I.astype(np.float32), psf, 4, Background=100, save16bit=False, ctx=three)[0]
    assert _rel(J2, J3) <= 1e-5
    assert _rel(R2, R3) <= 1e-5


# Either side of the rule that keeps the three passes: rows of 1024 with 8-column tiles; the same with a dim-3 transform
# of one stage, with 16-column tiles, with rows of 1000; four columns with short dim-2 and dim-3 transforms; and with a
# dim-3 transform of 30 values a thread
@pytest.mark.parametrize("shape, form", [
    ((1024, 128, 64), "three"), ((1024, 128, 32), "two"), ((1024, 64, 64), "two"), ((1000, 128, 64), "two"),
    ((64, 625, 108), "three"), ((64, 625, 180), "two"),
], ids=str)
def test_default_form_of_a_size(shape, form):
    I, psf, psf_b = _volume(shape, sum(shape))
    ctx = pk.Context(0)
    ctx.profile(True)
    out = pk.decon_lucy_omw_function(I, psf, psf_b, 1, Background=100, save16bit=False, ctx=ctx)[0]
    passes = ctx.profile_read()
    assert ("yz_conv" in passes, "z_conv" in passes) == (form == "two", form == "three"), passes
    other = pk.Context(0)
    if form == "two":
        _three_pass(shape, other)
        assert _rel(out, pk.decon_lucy_omw_function(I, psf, psf_b, 1, Background=100, save16bit=False, ctx=other)[0]) <= 1e-5
    other.close()
    ctx.close()


def test_two_pass_batch_and_options_equal_single_calls():
    """Chunks of several sizes (padded ones among them: 59 x 59 x 29 runs as 60 x 60 x 30 in two passes, 53 x 40 x 27 as
    54 x 40 x 27 in three) in one call give the single calls' bits; so do the options that ride in the last update."""
    shapes = [(60, 60, 30), (80, 64, 45), (53, 40, 27), (96, 64, 32), (45, 40, 27), (59, 59, 29)]
    ctx = pk.Context(0)
    ctx.profile(True)
    for shape, name in (((59, 59, 29), "b_yz_conv"), ((53, 40, 27), "b_z_conv")):
        v, psf, psf_b = _volume(shape, 3)
        pk.decon_batch([v], psf, psf_b, 1, method="omw", Background=100, ctx=ctx)
        passes = ctx.profile_read()
        assert name in passes and (name == "b_z_conv" or "b_z_conv" not in passes), passes
    ctx.close()
    vols = [_volume(s, 7 + k)[0] for k, s in enumerate(shapes)]
    _, psf, psf_b = _volume((32, 32, 24), 1)
    for method, it in (("omw", 2), ("rl", 4)):
        for kw in ({}, {"dampFactor": 2, "scaleFactor": 0.5, "deconOffset": 3}, {"save16bit": False}):
            outs = pk.decon_batch(vols, psf, psf_b, it, method=method, Background=100, **kw)
            for v, o in zip(vols, outs):
                args = (psf, psf_b, it) if method == "omw" else (psf, it)
                fn = pk.decon_lucy_omw_function if method == "omw" else pk.decon_lucy_function
                J = fn(v, *args, Background=100, pad=True, **kw)[0]
                assert np.array_equal(o, J), (method, kw, v.shape)


def test_tune_set_takes_the_lines_of_the_tune_file(tmp_path, monkeypatch):
    """Either sign of the first shape pins the three passes; zero is refused."""
    shape = (100, 64, 36)
    I, psf, psf_b = _volume(shape, 9)
    monkeypatch.setenv("PK_TUNE_FILE", str(tmp_path / "tune.txt"))
    ctx = pk.Context(0)
    ctx.autotune(shape)
    line = [int(x) for x in (tmp_path / "tune.txt").read_text().split()]
    assert tuple(line[:3]) == shape and len(line) == 11
    out = []
    for sign in (1, -1):
        shapes = [sign * abs(line[3])] + line[4:]
        ctx.tune_set(shape, shapes)
        ctx.profile(True)
        out.append(pk.decon_lucy_omw_function(I, psf, psf_b, 2, Background=100, save16bit=False, ctx=ctx)[0])
        passes = ctx.profile_read()
        assert "z_conv" in passes or "y_conv" in passes, passes
        assert "yz_conv" not in passes
    np.testing.assert_array_equal(out[0], out[1])
    for first in (0, -2 ** 31):
        with pytest.raises(pk.PkDeconError):
            ctx.tune_set(shape, [first] + line[4:])
    ctx.close()


@pytest.mark.parametrize("shapes, method", [([(60, 80, 36), (54, 80, 36), (80, 80, 36)], "omw"),
                                            ([(48, 80, 36), (72, 80, 36), (96, 80, 36)], "rl")], ids=["omw", "rl"])
def test_request_in_flight_keeps_its_form_when_its_size_is_pinned(shapes, method):
    """The size of a request goes to the three passes between two of its steps: the request goes on in the two-pass
    form, whose spectrum order, OTFs and partial sums it was admitted with, and the next one takes the new form."""
    n = 3000  # iterations: about 0.1 s
    fn = pk.decon_lucy_omw_function if method == "omw" else pk.decon_lucy_function
    kw = dict(Background=100, save16bit=False)
    ctx = pk.Context(0)
    srv = pk.Server(ctx)
    for shape in shapes:  # a size a try, should the pin come after the last step
        I, psf, psf_b = _volume(shape, sum(shape))

        def alone(iters):
            return fn(I, psf, *((psf_b,) if method == "omw" else ()), iters, ctx=ctx, **kw)[0]

        def served(iters):
            return srv.submit(I, psf, psf_b, iters, method=method, **kw)

        two, two_short = alone(n), alone(3)
        req = served(n)
        while req.info()["iterations_done"] < 2:
            time.sleep(1e-4)
        # the scheduler gives the context up between two steps only for a moment, longer while it waits for the queue's lock
        stop = threading.Event()
        ask = [threading.Thread(target=lambda: [req.info() for _ in iter(stop.is_set, True)]) for _ in range(3)]
        for t in ask:
            t.start()
        _three_pass(shape, ctx)
        done = req.info()["iterations_done"]
        stop.set()
        for t in ask:
            t.join()
        print(f"[fold] {method} {shape}: pinned after {done} of {n} iterations", flush=True)
        np.testing.assert_array_equal(req.result(timeout_s=60), two)
        after = served(3).result(timeout_s=60)
        np.testing.assert_array_equal(after, alone(3))  # three passes, served and alone
        assert not np.array_equal(after, two_short) and _rel(after, two_short) <= 1e-5
        if done < n:
            break
    srv.stop()
    ctx.close()
    if done == n:
        pytest.skip("no request was still running when its size was pinned")


def test_call_keeps_its_form_when_its_iteration_hook_pins_the_size(monkeypatch, tmp_path):
    from petakit5d_amd import decon
    shape = (120, 80, 36)
    I, psf, psf_b = _volume(shape, 5)
    ctx = pk.Context(0)

    def call(pin):
        monkeypatch.setattr(decon, "_debug_hook", lambda *a: decon._HOOK_T(
            lambda _user, k, _data, _dims: (pin and k == 2 and _three_pass(shape, ctx)) and None))
        return pk.decon_lucy_omw_function(I, psf, psf_b, 5, Background=100, save16bit=False, debug=True, saveStep=1,
                                          debug_folder=str(tmp_path), ctx=ctx)[0]

    two = call(False)
    np.testing.assert_array_equal(call(True), two)
    three = call(False)
    assert not np.array_equal(three, two) and _rel(three, two) <= 1e-5
    ctx.close()


@pytest.mark.parametrize("shape", [(160, 96, 48), (512, 64, 32), (300, 100, 60)], ids=lambda s: "x".join(map(str, s)))
def test_two_pass_form_is_no_further_from_64_bits_than_three_passes(oracle, shape):
    """A back projector that sharpens brings the transforms' rounding out.  With twiddles that are powers of one table
    value the two passes were up to 1.4 times as far from 64 bits as the three; 1.1: the spread of four volumes."""
    psf = synth.gaussian_psf((15, 15, 21), 1.2, 2.5, 20.0)
    h = np.fft.fftn(np.fft.ifftshift(psf.astype(np.float64)))
    wiener = np.conj(h) / (np.abs(h) ** 2 + 0.005) * np.clip(np.log10(np.maximum(np.abs(h), 1e-12)) / 2 + 1, 0, 1)
    psf_b = np.asfortranarray(np.fft.fftshift(np.fft.ifftn(wiener).real), dtype=np.float32)
    vols = []
    for k in range(4):
        g = np.random.default_rng(50 + k)
        obj = synth.point_emitters(shape, int(np.prod(shape)) // 3000, (20000, 90000), g)
        vols.append(synth.poisson_u16(synth._fft_convolve_circular(obj, psf) + 105, g))
    two = pk.Context(0)
    ref = [oracle.decon_lucy_omw_function(v, psf, psf_b, 2, Background=100, save16bit=False, precision="f64")[0]
           for v in vols]

    def error(ctx):
        out = [pk.decon_lucy_omw_function(v, psf, psf_b, 2, Background=100, save16bit=False, ctx=ctx)[0] for v in vols]
        return float(np.sqrt(np.mean([_rel(o, r) ** 2 for o, r in zip(out, ref)])))

    e2 = error(two)
    e3 = error(_three_pass(shape, two))
    print(f"[fold] {shape}: error against 64 bits, two passes {e2:.3e}, three {e3:.3e}", flush=True)
    assert e2 <= 1.1 * e3
