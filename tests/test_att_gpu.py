"""GPU parity of the attenuated SIR (alpha > 0; src/attenuation.cc:72-140)
against the oracle.  The GPU sums every point's contributions in the
frequency domain and transforms once; the oracle transforms each
contribution (as the reference does), so the two agree to rounding: the bar
is 1e-10 of the largest sample (FP64 output).  Error codes as without
attenuation."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CP = 1500.0


def _close(H, ref, tol=1e-10):
    return np.max(np.abs(H - ref)) <= tol * np.abs(ref).max()


@pytest.mark.parametrize("nt", [128, 129])
def test_dreamrect_attenuated(gpu, oracle, nt):
    from dream_amd.dreamrect import dreamrect
    rng = np.random.default_rng(31)
    No = 12
    Ro = np.c_[rng.uniform(-2, 2, No), rng.uniform(-2, 2, No), rng.uniform(8, 15, No)]
    d = Ro[:, 2] * 1000.0 / CP - 1.0
    H = dreamrect(Ro, [1.0, 2.0], [0.1, 0.1, 0.05, nt], d, [1.0, CP, 5.0], "ignore")
    ref, _, _ = oracle.dreamrect(Ro, 1.0, 2.0, 0.1, 0.1, 0.05, nt, d, 1.0, CP,
                                 err_level="ignore", nthreads=2, alpha=5.0)
    assert _close(H, ref)


def test_dream_arr_rect_attenuated_focused_apodized(gpu, oracle):
    from dream_amd.dream_arr_rect import dream_arr_rect
    rng = np.random.default_rng(32)
    L, No = 4, 8
    G = np.c_[np.linspace(-1.5, 1.5, L), np.zeros(L), np.zeros(L)]
    Ro = np.c_[rng.uniform(-3, 3, No), rng.uniform(-1, 1, No), rng.uniform(10, 20, No)]
    d = Ro[:, 2] * 1000.0 / CP - 2.0
    H = dream_arr_rect(Ro, [0.5, 1.5], G, [0.1, 0.1, 0.04, 200], d, [1.0, CP, 2.5], "xy", 15.0,
                       "x", [5.0, 0.0], "hann", None, 0.0, "ignore")
    ref, _, _ = oracle.dream_arr_rect(Ro, 0.5, 1.5, 0.1, 0.1, 0.04, 200, d, 1.0, CP, G,
                                      foc_met="xy", focal=15.0, steer_met="x", theta=5.0,
                                      apod_met="hann", err_level="ignore", nthreads=2,
                                      alpha=2.5)
    assert _close(H, ref)


def test_disc_cylinder_and_annulus_attenuated(gpu, oracle):
    from dream_amd.dream_arr_annu import dream_arr_annu
    from dream_amd.dreamcirc import dreamcirc
    from dream_amd.dreamcylind import dreamcylind
    Ro = np.array([[0.0, 0.0, 10.0], [0.5, 0.2, 12.0], [-1.0, 0.3, 9.0]])
    H = dreamcirc(Ro, [0.6], [0.1, 0.1, 0.05, 128], 5.0, [1.0, CP, 5.0], "ignore")
    ref, _, _ = oracle.dreamcirc(Ro, 0.6, 0.1, 0.1, 0.05, 128, 5.0, 1.0, CP,
                                 err_level="ignore", nthreads=2, alpha=5.0)
    assert _close(H, ref)
    H = dreamcylind(Ro, [0.5, 1.2, -6.0], [0.1, 0.1, 0.05, 128], 5.0, [1.0, CP, 5.0], "ignore")
    ref, _, _ = oracle.dreamcylind(Ro, 0.5, 1.2, -6.0, 0.1, 0.1, 0.05, 128, 5.0, 1.0, CP,
                                   err_level="ignore", nthreads=2, alpha=5.0)
    assert _close(H, ref)
    gr = [0.4, 0.5, 0.8, 0.9, 1.1]
    H = dream_arr_annu(Ro, np.array(gr).reshape(-1, 1), [0.1, 0.1, 0.05, 128], 5.0,
                       [1.0, CP, 5.0], "x", 12.0, "off", None, 0.0, "ignore")
    ref, _, _ = oracle.dream_arr_annu(Ro, gr, 0.1, 0.1, 0.05, 128, 5.0, 1.0, CP, foc_met="x",
                                      focal=12.0, err_level="ignore", nthreads=2, alpha=5.0)
    assert _close(H, ref)


def test_attenuated_single_point_many_chunks_and_codes(gpu, oracle):
    """One point: its contributions are split over many work-groups whose
    spectra add atomically; out-of-range samples give the usual codes."""
    from dream_amd.dreamrect import dreamrect
    Ro = np.array([[0.2, 0.1, 10.0]])
    H = dreamrect(Ro, [2.0, 4.0], [0.05, 0.05, 0.05, 160], 5.5, [1.0, CP, 4.0], "ignore")
    ref, _, _ = oracle.dreamrect(Ro, 2.0, 4.0, 0.05, 0.05, 0.05, 160, 5.5, 1.0, CP,
                                 err_level="ignore", nthreads=1, alpha=4.0)
    assert _close(H, ref)
    Ro2 = np.array([[0.0, 0.0, 10.0], [2.0, 0.0, 10.0]])
    with pytest.raises(RuntimeError):
        dreamrect(Ro2, [2.0, 4.0], [0.05, 0.05, 0.05, 28], 5.5, [1.0, CP, 4.0], "stop")
    H = dreamrect(Ro2, [2.0, 4.0], [0.05, 0.05, 0.05, 28], 5.5, [1.0, CP, 4.0], "ignore")
    ref, e, _ = oracle.dreamrect(Ro2, 2.0, 4.0, 0.05, 0.05, 0.05, 28, 5.5, 1.0, CP,
                                 err_level="ignore", nthreads=2, alpha=4.0)
    assert e == 1 and _close(H, ref)


@pytest.mark.parametrize("nt", [9000, 9001])
def test_long_responses_split_their_spectra(gpu, oracle, nt):
    """nt above one work-group's share of LDS (3584 bins): each point's
    spectrum is accumulated in bin blocks by several work-groups."""
    from dream_amd.dreamrect import dreamrect
    Ro = np.array([[0.0, 0.0, 10.0], [0.4, 0.1, 12.0], [-0.7, 0.0, 11.0]])
    d = Ro[:, 2] * 1000.0 / CP - 1.0
    H = dreamrect(Ro, [0.3, 0.3], [0.1, 0.1, 0.05, nt], d, [1.0, CP, 3.0], "ignore")
    ref, _, _ = oracle.dreamrect(Ro, 0.3, 0.3, 0.1, 0.1, 0.05, nt, d, 1.0, CP,
                                 err_level="ignore", nthreads=2, alpha=3.0)
    assert _close(H, ref)


def test_device_entry_point_with_attenuation(gpu, oracle):
    """dream_hip_sir_att_dev on device tensors (arrays of rectangles and of
    discs, 'ud' delays, FP64 and FP32 output) against the oracle."""
    import torch
    from dream_amd.torch_ops import sir_attenuated
    rng = np.random.default_rng(35)
    L, No, nt = 3, 6, 300
    G = np.c_[np.linspace(-1.0, 1.0, L), np.zeros(L), np.zeros(L)]
    Ro = np.c_[rng.uniform(-2, 2, No), rng.uniform(-1, 1, No), rng.uniform(8, 14, No)]
    d = Ro[:, 2] * 1000.0 / CP - 1.5
    focal = rng.uniform(0.0, 0.3, L)
    Rt = torch.tensor(Ro.T.copy(), device="cuda")
    dt_ = torch.tensor(d, device="cuda")
    base = dict(Ro=Rt, dx=0.1, dy=0.1, dt=0.05, nt=nt, delay=dt_, v=1.0, cp=CP, G=G,
                foc_met="ud", focal=focal, apod_met="hann", err_level="ignore")
    ref, e, oob = oracle.dream_arr_rect(Ro, 0.4, 0.8, 0.1, 0.1, 0.05, nt, d, 1.0, CP, G,
                                        foc_met="ud", focal=focal, apod_met="hann",
                                        err_level="ignore", nthreads=2, alpha=4.0)
    for out_dtype, tol in ((torch.float64, 1e-10), (torch.float32, 1e-6)):
        H, code, n_oob = sir_attenuated(dict(base, a=0.4, b=0.8), 4.0, out_dtype)
        assert _close(H.double().cpu().numpy().T, ref, tol)
        assert code == e and n_oob == oob
    ref, e, oob = oracle.dream_arr_circ(Ro, 0.5, 0.1, 0.1, 0.05, nt, d, 1.0, CP, G, foc_met="ud",
                                        focal=focal, apod_met="hann", err_level="ignore",
                                        nthreads=2, alpha=4.0)
    H, code, n_oob = sir_attenuated(dict(base, shape="circ", R=0.5), 4.0)
    assert _close(H.cpu().numpy().T, ref) and code == e and n_oob == oob


@pytest.mark.parametrize("alpha,delay,nt", [
    (0.5, None, 160),       # 8 moments, the per-sample table
    (20.0, None, 161),      # 12 moments
    (60.0, None, 160),      # two sub-cells per sample, no table
    (900.0, None, 160),     # many sub-cells, everything but near samples gone
    (40.0, -45.0, 1200),    # a far negative delay: factors evaluated per cell
    (5.0, 2.0, 700),        # an element over more than one window of 256 samples
])
def test_attenuated_moments(gpu, oracle, alpha, delay, nt):
    """The moment expansion's terms, sub-cells, windows and table rule."""
    from dream_amd.dreamrect import dreamrect
    wide = nt == 700
    No = 3 if wide else 40
    rng = np.random.default_rng(37)
    Ro = np.c_[rng.uniform(-2, 2, No), rng.uniform(-1, 1, No), rng.uniform(4, 7, No)]
    dt = 0.02 if wide else 0.05
    geom, step = ([16.0, 4.0], 0.4) if wide else ([0.8, 1.2], 0.1)
    d = Ro[:, 2] * 1000.0 / CP - 1.0 if delay is None else delay
    H = dreamrect(Ro, geom, [step, step, dt, nt], d, [1.0, CP, alpha], "ignore")
    ref, _, _ = oracle.dreamrect(Ro, *geom, step, step, dt, nt, d, 1.0, CP, err_level="ignore",
                                 nthreads=4, alpha=alpha)
    assert _close(H, ref)


def _att_batch(n, nt, dts, points):
    """n one-element problems with their own intervals in one call."""
    import ctypes

    import torch
    from dream_amd import _lib
    Ro = torch.tensor(np.c_[np.linspace(-1, 1, points), np.zeros(points),
                            np.linspace(3, 5, points)].T.copy(), device="cuda")
    d = torch.zeros(1, dtype=torch.float64, device="cuda")
    H = torch.empty((n, points, nt), dtype=torch.float64, device="cuda")
    G, one = np.zeros((1, 3)), np.ones(1)
    q = (_lib.DreamSirProblem * n)()
    for i in range(n):
        p = q[i]
        p.Ro, p.No, p.a, p.b, p.dx, p.dy = Ro.data_ptr(), points, 0.2, 0.2, 0.1, 0.1
        p.dt, p.nt, p.delay_type, p.delay, p.v, p.cp = dts[i], nt, 0, d.data_ptr(), 1.0, CP
        p.num_elements, p.G, p.focal, p.apod = 1, G.ctypes.data, one.ctypes.data, one.ctypes.data
        p.foc_met, p.steer_met = _lib.FOC_MET["off"], _lib.STEER_MET["off"]
        p.err_level = _lib.ERR_LEVEL["ignore"]
        p.h = H.data_ptr() + i * points * nt * 8

    def run(lo, hi):
        _lib.check(_lib.lib().dream_hip_sir_att_dev(
            ctypes.cast(ctypes.byref(q, lo * ctypes.sizeof(_lib.DreamSirProblem)),
                        ctypes.POINTER(_lib.DreamSirProblem)),
            hi - lo, 5.0, _lib.F64, None, None, torch.cuda.current_stream().cuda_stream))
        return H[lo:hi].cpu().numpy()
    return run


@pytest.mark.parametrize("n,nt,points,pick", [
    (66000, 4, 1, [0, 32767, 32768, 65535, 65536, 65999]),    # more than one launch's grids
    (12, 2000, 130, [0, 7, 8, 11]),                           # more than the tables' 256 MiB
])
def test_many_intervals_in_one_call(gpu, n, nt, points, pick):
    """Problems that share no frequency grid: as many as a caller has, each
    equal to its own call, whether its factors came from a table or not (the two
    evaluate the same exponentials, apart by a few ulp of phases of 2 pi nt)."""
    dts = np.linspace(0.8, 1.2, n) * 4.0 / CP * 1000.0 / nt * 2.0
    run = _att_batch(n, nt, dts, points)
    every = run(0, n)
    for i in pick:
        alone = run(i, i + 1)[0]
        assert np.abs(alone).max() > 0
        assert np.max(np.abs(every[i] - alone)) <= 1e-11 * np.abs(alone).max()


@pytest.mark.parametrize("alpha", [1.0, 5.0])
def test_negative_speed_as_the_oracle(gpu, oracle, alpha):
    """A negative speed turns delays and samples round; no value is refused.
    The element's distances span some fifty samples."""
    from dream_amd.dreamrect import dreamrect
    Ro = np.array([[0.0, 0.0, 5.0], [0.4, 0.2, 6.0]])
    d = -Ro[:, 2] * 1000.0 / CP - 1.6
    H = dreamrect(Ro, [1.0, 6.0], [0.1, 0.1, 0.01, 200], d, [1.0, -CP, alpha], "ignore")
    ref, _, _ = oracle.dreamrect(Ro, 1.0, 6.0, 0.1, 0.1, 0.01, 200, d, 1.0, -CP,
                                 err_level="ignore", nthreads=2, alpha=alpha)
    assert np.abs(ref).max() > 0
    assert _close(H, ref)
