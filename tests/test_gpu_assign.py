"""GPU assignment through the C ABI vs the sequential-FP32 oracle: bit-exact labels."""
import numpy as np
import pytest

from oracle import native as on
from pyemma_amd import _native

pytestmark = pytest.mark.gpu

MODES = [_native.EMMA_ASSIGN_FP32_PLAIN, _native.EMMA_ASSIGN_BF16X3_RECHECK]


def _run(X, C, mode):
    t = _native.torch()
    Xt = _native.as_device_f32(X)
    Ct = _native.as_device_f32(C)
    nre = t.zeros(1, dtype=t.int64, device=Xt.device)
    lab = _native.assign(Xt, Ct, mode=mode, n_rechecked=nre)
    t.cuda.synchronize()
    return lab.cpu().numpy(), int(nre.item())


def _data(n, d, k, seed, offset=0.0, scale=1.0):
    rng = np.random.default_rng(seed)
    X = (rng.standard_normal((n, d)) * scale + offset).astype(np.float32)
    C = X[rng.choice(n, k, replace=n < k)] + (rng.standard_normal((k, d)) * 0.3 * scale).astype(np.float32)
    return X, C.astype(np.float32)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n,d,k", [(1000, 30, 100), (2049, 300, 257), (777, 3, 1), (1500, 1, 5),
                                   (3000, 128, 512), (1024, 512, 64), (513, 17, 33), (300, 64, 1000)])
def test_labels_bit_exact(mode, n, d, k):
    X, C = _data(n, d, k, seed=n + d + k)
    ref = on.assign(X, C, nthreads=4)
    lab, nre = _run(X, C, mode)
    np.testing.assert_array_equal(lab, ref)
    if mode == _native.EMMA_ASSIGN_FP32_PLAIN:
        assert nre == 0


@pytest.mark.parametrize("mode", MODES)
def test_far_from_origin_and_large_spread(mode):
    """Shifted data (mean 1e3) and mixed scales: the shift and the bound must hold."""
    X, C = _data(4000, 40, 80, seed=5, offset=1000.0, scale=0.5)
    np.testing.assert_array_equal(_run(X, C, mode)[0], on.assign(X, C, nthreads=4))


@pytest.mark.parametrize("mode", MODES)
def test_exact_ties_first_index_wins(mode):
    rng = np.random.default_rng(1)
    C = rng.standard_normal((10, 8)).astype(np.float32)
    C = np.concatenate([C, C[::-1]], axis=0)  # every center twice
    X = np.concatenate([C, rng.standard_normal((500, 8)).astype(np.float32)], axis=0)
    ref = on.assign(X, C)
    lab, nre = _run(X, C, mode)
    np.testing.assert_array_equal(lab, ref)
    if mode == _native.EMMA_ASSIGN_BF16X3_RECHECK:
        assert nre >= 20  # duplicated centers always tie


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("bad_center", [None, 0, 3])
def test_non_finite_rows_and_centers(mode, bad_center):
    """NaN and inf in frames (and NaN in one center): the reference loop starts
    from center 0 and replaces it only on a smaller distance, so a NaN
    distance never wins and a NaN distance to center 0 keeps label 0."""
    X, C = _data(700, 20, 40, seed=11)
    X[5, 3] = np.nan
    X[17, :] = np.inf
    X[18, 0] = -np.inf
    X[40:44, 7] = 3e19  # squares overflow to inf for every center
    if bad_center is not None:
        C[bad_center, 2] = np.nan
    ref = on.assign(X, C)
    np.testing.assert_array_equal(_run(X, C, mode)[0], ref)


@pytest.mark.parametrize("mode", MODES)
def test_listed_candidate_after_a_tie(mode):
    """Exact ties where the later center of a tied pair is also the nearer in
    the MFMA pass's rounding: the first minimum in index order must win."""
    rng = np.random.default_rng(2)
    base = rng.standard_normal((16, 64)).astype(np.float32)
    C = np.concatenate([base, base], axis=0)  # center j and j + 16 identical
    X = (base[rng.integers(0, 16, 3000)] + rng.standard_normal((3000, 64)).astype(np.float32) * 0.05).astype(np.float32)
    ref = on.assign(X, C)
    lab, nre = _run(X, C, mode)
    np.testing.assert_array_equal(lab, ref)
    assert np.all(lab < 16)


def test_golden_hmm_labels(golden_hmm):
    g = golden_hmm
    for mode in MODES:
        np.testing.assert_array_equal(_run(g["X"], g["lloyd_centers"], mode)[0], g["labels"])


def test_recheck_rate_is_small_on_separated_data():
    from pyemma_amd.synthetic import hmm_trajectory
    X = hmm_trajectory(20000, 30, seed=3)
    C = X[::200][:100].copy()
    lab, nre = _run(X, C, _native.EMMA_ASSIGN_BF16X3_RECHECK)
    np.testing.assert_array_equal(lab, on.assign(X, C, nthreads=4))
    assert nre < 0.2 * len(X)


def test_mfma_dimension_limit_and_plain_beyond():
    X, C = _data(300, 600, 7, seed=2)
    with pytest.raises(ValueError):
        _run(X, C, _native.EMMA_ASSIGN_BF16X3_RECHECK)
    np.testing.assert_array_equal(_run(X, C, _native.EMMA_ASSIGN_FP32_PLAIN)[0], on.assign(X, C))


def test_deterministic_repeat():
    X, C = _data(5000, 300, 300, seed=9)
    a, na = _run(X, C, _native.EMMA_ASSIGN_BF16X3_RECHECK)
    b, nb = _run(X, C, _native.EMMA_ASSIGN_BF16X3_RECHECK)
    np.testing.assert_array_equal(a, b)
    assert na == nb


@pytest.mark.parametrize("d,k", [(20, 70), (64, 256), (128, 200), (128, 300), (200, 100), (300, 1000), (512, 64)])
def test_every_tile_variant_bit_exact(d, k):
    """Each tile variant (waves per workgroup, workgroups per CU, frame blocks per wave) gives the
    oracle's labels, including a ragged last workgroup."""
    L = _native.lib()
    n = 4 * 1024 + 77
    X, C = _data(n, d, k, seed=d * 7 + k)
    ref = on.assign(X, C, nthreads=4)
    try:
        for v in range(L.emma_assign_variants(d)):
            _native.check(L.emma_assign_select(d, k, v), "emma_assign_select")
            lab, _ = _run(X, C, _native.EMMA_ASSIGN_BF16X3_RECHECK)
            np.testing.assert_array_equal(lab, ref, err_msg="variant %d" % v)
    finally:
        _native.check(L.emma_assign_select(d, k, 0), "emma_assign_select")


@pytest.mark.parametrize("d", [64, 128, 300, 301, 510, 512])
@pytest.mark.parametrize("aligned", [True, False])
def test_frame_load_forms(d, aligned):
    """Both frame-load forms of the MFMA passes give the oracle's labels in every tile
    variant: 16-byte loads (d % 4 == 0 and 16-byte aligned frames; in groups of
    K-steps beyond 8 K-steps) and the dword loads otherwise (d % 4 != 0, or frames
    starting 4 bytes past a 16-byte boundary)."""
    t = _native.torch()
    L = _native.lib()
    n, k = 3 * 1024 + 45, 160
    X, C = _data(n, d, k, seed=d + (0 if aligned else 1))
    ref = on.assign(X, C, nthreads=4)
    if aligned:
        Xt = _native.as_device_f32(X)
    else:
        buf = t.empty(n * d + 1, dtype=t.float32, device=_native.device())
        Xt = buf[1:].view(n, d)
        Xt.copy_(t.from_numpy(X))
        assert Xt.data_ptr() % 16 == 4
    Ct = _native.as_device_f32(C)
    try:
        for v in range(L.emma_assign_variants(d)):
            _native.check(L.emma_assign_select(d, k, v), "emma_assign_select")
            lab = _native.assign(Xt, Ct, mode=_native.EMMA_ASSIGN_BF16X3_RECHECK)
            t.cuda.synchronize()
            np.testing.assert_array_equal(lab.cpu().numpy(), ref, err_msg="variant %d" % v)
    finally:
        _native.check(L.emma_assign_select(d, k, 0), "emma_assign_select")


@pytest.mark.parametrize("reps", [2, 8, 9, 12])
def test_recheck_candidate_paths(reps):
    """Every center repeated `reps` times: each frame ties between `reps`
    centers (every frame is listed).  Up to 8 candidates the tie is settled by
    the reference loop over the recorded candidates, above 8 by the full loop
    over every center.  The first minimum wins in both."""
    rng = np.random.default_rng(reps)
    base = rng.standard_normal((6, 24)).astype(np.float32)
    C = np.repeat(base, reps, axis=0)
    X = (base[rng.integers(0, 6, 3000)] + 0.3 * rng.standard_normal((3000, 24))).astype(np.float32)
    ref = on.assign(X, C, nthreads=4)
    lab, nre = _run(X, C, _native.EMMA_ASSIGN_BF16X3_RECHECK)
    np.testing.assert_array_equal(lab, ref)
    assert nre == 3000
    assert np.all(ref % reps == 0)


def _every_variant(X, C):
    """Labels of X under every variant (both first-pass pipelines, every tile shape)."""
    L = _native.lib()
    d, k = X.shape[1], C.shape[0]
    out = []
    try:
        for v in range(L.emma_assign_variants(d)):
            _native.check(L.emma_assign_select(d, k, v), "emma_assign_select")
            out.append(_run(X, C, _native.EMMA_ASSIGN_BF16X3_RECHECK)[0])
    finally:
        _native.check(L.emma_assign_select(d, k, -1), "emma_assign_select")
    return out


@pytest.mark.parametrize("d", [64, 300])
@pytest.mark.parametrize("case", ["outliers", "tiny", "huge", "mixed_scale"])
def test_coarse_pass_edge_cases(d, case):
    """The coarse pass scales frames and centers by 2^t (max |b| near 2^9) into
    fp16.  Outlier frames beyond 64 max|b| overflow fp16 and must reach the fine
    pass; tiny (1e-30) and huge (1e30) data clamp the exponent t to +-60; frames
    with some dimensions 1e-6 of the others underflow fp16 there.  Every
    variant gives the oracle's labels."""
    rng = np.random.default_rng({"outliers": 1, "tiny": 2, "huge": 3, "mixed_scale": 4}[case] + d)
    X, C = _data(3000, d, 40, seed=d + 1)
    if case == "outliers":
        X[::7] *= 5000.0
    elif case == "tiny":
        X, C = X * np.float32(1e-30), C * np.float32(1e-30)
    elif case == "huge":
        X, C = X * np.float32(1e30), C * np.float32(1e30)
    else:
        scale = np.where(rng.random(d) < 0.3, 1e-6, 1.0).astype(np.float32)
        X, C = X * scale, C * scale
    X, C = np.ascontiguousarray(X, np.float32), np.ascontiguousarray(C, np.float32)
    ref = on.assign(X, C, nthreads=4)
    for v, lab in enumerate(_every_variant(X, C)):
        np.testing.assert_array_equal(lab, ref, err_msg="variant %d" % v)


@pytest.mark.parametrize("n", [1, 31, 33, 129, 16383, 16385, 32767, 32769])
@pytest.mark.parametrize("d,k", [(1, 31), (3, 65), (4, 1), (5, 32), (33, 33), (63, 129), (129, 64), (191, 97), (257, 63),
                                 (303, 130), (305, 34), (383, 66), (385, 255), (511, 65)])
def test_tile_edges(n, d, k):
    """Labels at the edges of the tile kernel: one frame more or less than a row block and than
    the frame counts where the small and the large workgroup shape take over, dimensions
    around the K-step sizes (d < 4, d % 4 != 0, one past a size), center counts around one
    and two tiles per wave.  Every variant gives the plain loop's labels."""
    t = _native.torch()
    g = t.Generator(device="cuda").manual_seed(1000 * d + k + n)
    means = 2.0 * t.randn((7, d), generator=g, device="cuda")
    X = (means[t.randint(0, 7, (n,), generator=g, device="cuda")] + t.randn((n, d), generator=g, device="cuda")).contiguous()
    C = (X[t.randint(0, n, (k,), generator=g, device="cuda")] + 0.3 * t.randn((k, d), generator=g, device="cuda")).contiguous()
    ref = _native.assign(X, C, mode=_native.EMMA_ASSIGN_FP32_PLAIN)
    L = _native.lib()
    try:
        for v in range(L.emma_assign_variants(d)):
            _native.check(L.emma_assign_select(d, k, v), "emma_assign_select")
            lab = _native.assign(X, C, mode=_native.EMMA_ASSIGN_BF16X3_RECHECK)
            assert t.equal(lab, ref), "variant %d: %d labels differ" % (v, int((lab != ref).sum()))
    finally:
        _native.check(L.emma_assign_select(d, k, -1), "emma_assign_select")


@pytest.mark.parametrize("n,d,k", [(5, 1, 2), (300, 1, 2), (300, 31, 40), (3000, 300, 33), (40000, 32, 40)])
@pytest.mark.parametrize("big", [3e38, 1e25, 1e19])
def test_overflowing_frames_in_short_lists(n, d, k, big):
    """Frames and a center whose squares or products overflow, in a workspace that holds
    negative leftovers: rows past the end of a list record no candidates, and the labels
    are those of the loop."""
    t = _native.torch()
    rng = np.random.default_rng(n + d)
    X = rng.standard_normal((n, d)).astype(np.float32)
    X[n // 2] = big
    X[n - 1, d - 1] = -big
    C = rng.standard_normal((k, d)).astype(np.float32)
    for center in (None, big):
        if center is not None:
            C[k - 1] = np.float32(0.9) * np.float32(center)
        Xt, Ct = _native.as_device_f32(X), _native.as_device_f32(C)
        size = _native.lib().emma_assign_workspace_size(n, d, k, _native.EMMA_ASSIGN_BF16X3_RECHECK)
        _native.workspace(size, "assign").fill_(0xC5)
        lab = _native.assign(Xt, Ct, mode=_native.EMMA_ASSIGN_BF16X3_RECHECK)
        ref = _native.assign(Xt, Ct, mode=_native.EMMA_ASSIGN_FP32_PLAIN)
        assert bool(t.equal(lab, ref))


@pytest.mark.parametrize("n", [40, 20_000, 40_000])
@pytest.mark.parametrize("d", [2, 70])
@pytest.mark.parametrize("k", [28, 32, 60, 64, 96])
@pytest.mark.parametrize("big", [1.5e19, 5e19, 2e25])
def test_finite_outlier_center(n, d, k, big):
    """A finite center so far out that its squared norm overflows, as the last one that a
    lane takes and as any other: its distance becomes +inf or no number in the matrix
    pass, and no frame may be decided from that."""
    rng = np.random.default_rng(n + k)
    X = rng.standard_normal((n, d)).astype(np.float32)
    C0 = rng.standard_normal((k, d)).astype(np.float32)
    X[n // 3] = np.float32(0.9 * big)
    Xt = _native.as_device_f32(X)
    for j in (k - 1, k - 5, 27, 0):
        C = C0.copy()
        C[j] = np.float32(big)
        ref = _run(X, C, _native.EMMA_ASSIGN_FP32_PLAIN)[0]
        for v, lab in enumerate(_every_variant(X, C)):
            np.testing.assert_array_equal(lab, ref, err_msg="center %d, variant %d" % (j, v))


def _near_ties(d, k, seed):
    """Frames near the midplane of two of k centers, on a lattice of a few values, so that
    at small scales many distances are equal or a unit apart."""
    rng = np.random.default_rng(seed)
    C = rng.integers(-3, 4, (k, d)).astype(np.float64)
    a, b = rng.integers(0, k, 3000), rng.integers(0, k, 3000)
    X = 0.5 * (C[a] + C[b]) + 0.02 * rng.standard_normal((3000, d))
    return X, C + 1e-3 * rng.standard_normal((k, d))


@pytest.mark.parametrize("d", [1, 2, 8, 64, 300])
@pytest.mark.parametrize("k", [4, 33])
@pytest.mark.parametrize("exponent", [-16, -17, -18, -19, -20, -21, -22, -23])
def test_squares_that_underflow(d, k, exponent):
    """Data whose squared distances or squared residuals are below the smallest normal
    FP32 number: the loop's own distances are then a few units of 2^-149 apart, and the
    matrix passes may decide only what that leaves no doubt about."""
    X, C = _near_ties(d, k, d + k)
    s = 10.0 ** exponent
    X, C = (X * s).astype(np.float32), (C * s).astype(np.float32)
    ref = on.assign(X, C, nthreads=4)
    for v, lab in enumerate(_every_variant(X, C)):
        np.testing.assert_array_equal(lab, ref, err_msg="variant %d" % v)


@pytest.mark.parametrize("mode", MODES)
def test_counts_of_an_empty_call(mode):
    """No frames: the counts say so, whatever they held before."""
    t = _native.torch()
    X = t.empty((0, 7), dtype=t.float32, device="cuda")
    C = t.zeros((3, 7), device="cuda")
    counts = t.full((3,), 99, dtype=t.int64, device="cuda")
    _native.assign(X, C, mode=mode, n_rechecked=counts[:1], n_looped=counts[1:2])
    rc = _native.lib().emma_assign_noalloc(_native.ptr(X), 0, 7, _native.ptr(C), 3, None, mode,
                                           _native.ptr(counts[2:]), _native.stream_ptr())
    assert rc == 0
    assert counts.tolist() == [0, 0, 0]


@pytest.mark.parametrize("n", [32768, 32769, 40961, 65537, (1 << 20) - 1, (1 << 20) + 33])
@pytest.mark.parametrize("ties", ["all", "some", "none"])
def test_list_of_undecided_frames(n, ties):
    """Lists of every length, in chunks of both sizes: all frames undecided (each center
    twice), a quarter of them, almost none."""
    t = _native.torch()
    g = t.Generator(device="cuda").manual_seed(n)
    base = 3.0 * t.randn((40, 5), generator=g, device="cuda")
    C = {"all": t.cat([base, base]), "some": t.cat([base, base[:10]]), "none": base}[ties].contiguous()
    X = (base[t.randint(0, 40, (n,), generator=g, device="cuda")] + 0.05 * t.randn((n, 5), generator=g, device="cuda"))
    ref = _native.assign(X, C, mode=_native.EMMA_ASSIGN_FP32_PLAIN)
    L = _native.lib()
    counts = t.zeros(1, dtype=t.int64, device="cuda")
    try:
        for v in (0, L.emma_assign_variants(5) // 2):
            _native.check(L.emma_assign_select(5, len(C), v), "emma_assign_select")
            lab = _native.assign(X, C, n_rechecked=counts)
            assert t.equal(lab, ref)
            assert {"all": n, "some": n // 8}.get(ties, 0) <= int(counts.item()) <= n
    finally:
        _native.check(L.emma_assign_select(5, len(C), -1), "emma_assign_select")


@pytest.mark.parametrize("n,d,k", [(200, 30, 40), (33_000, 10, 64), (117_187, 256, 100), (117_188, 256, 100),
                                   (50_000, 40, 1562), (50_000, 40, 1600), (3_000, 400, 10), (3_000, 512, 600)])
def test_default_pipeline(n, d, k):
    """Without a selection the sizes choose the first pass, on either side of the line the
    labels are the loop's, and the call in chunks re-evaluates the same frames as the whole."""
    t = _native.torch()
    g = t.Generator(device="cuda").manual_seed(n + d)
    X = t.randn((n, d), generator=g, device="cuda")
    C = X[t.randint(0, n, (k,), generator=g, device="cuda")] + 0.2 * t.randn((k, d), generator=g, device="cuda")
    L = _native.lib()
    _native.check(L.emma_assign_select(d, k, -1), "emma_assign_select")
    ref = _native.assign(X, C, mode=_native.EMMA_ASSIGN_FP32_PLAIN)
    counts = t.zeros(2, dtype=t.int64, device="cuda")
    lab = _native.assign(X, C, n_rechecked=counts[:1])
    assert t.equal(lab, ref)
    lab.fill_(-1)
    rc = L.emma_assign_noalloc(_native.ptr(X), n, d, _native.ptr(C), k, _native.ptr(lab),
                               _native.EMMA_ASSIGN_BF16X3_RECHECK, _native.ptr(counts[1:]), _native.stream_ptr())
    _native.check(rc, "emma_assign_noalloc")
    assert t.equal(lab, ref)
    a, b = counts.tolist()
    assert a == b


@pytest.mark.parametrize("n", [65_535, 65_536, 65_537, 65_599, 131_073])
@pytest.mark.parametrize("d,k", [(1, 5), (2, 32), (3, 1), (4, 33), (7, 1024), (31, 1025), (32, 100), (33, 64), (63, 1023),
                                 (64, 31)])
def test_one_wave_workgroups(n, d, k):
    """The shape of few centers at small d on either side of its lines, with frames that tie,
    overflow or are not finite among the others; both pipelines and the default."""
    t = _native.torch()
    g = t.Generator(device="cuda").manual_seed(n + 7 * d + k)
    X = 2.0 * t.randn((n, d), generator=g, device="cuda")
    C = (X[t.randint(0, n, (k,), generator=g, device="cuda")] + 0.3 * t.randn((k, d), generator=g, device="cuda")).contiguous()
    C[k // 2] = C[0]
    X[n // 5] = 2e19
    X[n - 1, d - 1] = float("nan")
    X[n - 2, 0] = float("inf")
    ref = _native.assign(X, C, mode=_native.EMMA_ASSIGN_FP32_PLAIN)
    L = _native.lib()
    looped = t.zeros(1, dtype=t.int64, device="cuda")
    try:
        for v in (0, L.emma_assign_variants(d) // 2, -1):
            _native.check(L.emma_assign_select(d, k, v), "emma_assign_select")
            lab = _native.assign(X, C, n_looped=looped)
            assert t.equal(lab, ref), "variant %d: %d labels differ" % (v, int((lab != ref).sum()))
            assert int(looped.item()) >= 3
    finally:
        _native.check(L.emma_assign_select(d, k, -1), "emma_assign_select")


@pytest.mark.parametrize("n", [32_767, 32_768, 32_769, 40_031])
@pytest.mark.parametrize("d,k", [(385, 31), (400, 512), (511, 513), (512, 10), (512, 257)])
def test_few_centers_of_large_dimension(n, d, k):
    """The coarse pass's shape for few centers beyond 384 dimensions, on either side of its
    lines, with frames that tie, overflow or are not finite among the others."""
    t = _native.torch()
    g = t.Generator(device="cuda").manual_seed(n + d + k)
    X = t.randn((n, d), generator=g, device="cuda")
    C = (X[t.randint(0, n, (k,), generator=g, device="cuda")] + 0.3 * t.randn((k, d), generator=g, device="cuda")).contiguous()
    C[k // 2] = C[0]
    X[n // 5] = 2e19
    X[n - 1, d - 1] = float("nan")
    ref = _native.assign(X, C, mode=_native.EMMA_ASSIGN_FP32_PLAIN)
    L = _native.lib()
    try:
        for v in (0, -1):
            _native.check(L.emma_assign_select(d, k, v), "emma_assign_select")
            lab = _native.assign(X, C)
            assert t.equal(lab, ref), "variant %d: %d labels differ" % (v, int((lab != ref).sum()))
    finally:
        _native.check(L.emma_assign_select(d, k, -1), "emma_assign_select")


@pytest.mark.parametrize("d", [20, 60, 130, 190, 256, 300, 350, 512])
def test_lists_longer_than_the_grid(d):
    """Every frame undecided, more of them than the resident workgroups of the listed
    passes hold at once, so that each takes several blocks of the list."""
    t = _native.torch()
    g = t.Generator(device="cuda").manual_seed(d)
    n = 100_003
    base = 2.0 * t.randn((20, d), generator=g, device="cuda")
    C = t.cat([base, base]).contiguous()
    X = base[t.randint(0, 20, (n,), generator=g, device="cuda")] + 0.2 * t.randn((n, d), generator=g, device="cuda")
    ref = _native.assign(X, C, mode=_native.EMMA_ASSIGN_FP32_PLAIN)
    L = _native.lib()
    counts = t.zeros(1, dtype=t.int64, device="cuda")
    try:
        for v in (0, L.emma_assign_variants(d) // 2):
            _native.check(L.emma_assign_select(d, 40, v), "emma_assign_select")
            lab = _native.assign(X, C, n_rechecked=counts)
            assert t.equal(lab, ref) and int(counts.item()) == n
    finally:
        _native.check(L.emma_assign_select(d, 40, -1), "emma_assign_select")
