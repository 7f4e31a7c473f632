"""GPU FDTD updates: the reference's FDTD tests (meanas/test/test_fdtd.py) with the time
stepping on the GPU, and the stepped fields against the oracle's."""
import numpy
import pytest
import torch

from oracle import fdfd_ref as ref
import fdtd_checks as fc

pytestmark = pytest.mark.gpu


def gpu_step(e, h, eps, dt, dxes):
    from meanas_amd import fdtd
    fdtd.maxwell_h(dt, dxes)(e, h)
    fdtd.maxwell_e(dt, dxes)(e, h, eps)
    return e, h


@pytest.mark.parametrize('case', fc.cases())
def test_reference_fdtd_checks_on_gpu(case):
    sim = fc.make_sim(case, gpu_step)
    for check in fc.CHECKS:
        check(sim)
    ora = fc.make_sim(case, fc.oracle_step)
    for a, b in zip(sim.es + sim.hs, ora.es + ora.hs):
        numpy.testing.assert_allclose(a, b, rtol=1e-12, atol=1e-13)


def _fields(shape, seed, dtype):
    rng = numpy.random.default_rng(seed)
    e = rng.standard_normal((3, *shape)).astype(dtype)
    h = rng.standard_normal((3, *shape)).astype(dtype)
    eps = (1 + rng.random((3, *shape))).astype(dtype)
    mu = (1 + rng.random((3, *shape))).astype(dtype)
    dxes = [[0.8 + 0.4 * rng.random(n) for n in shape] for _ in range(2)]
    return e, h, eps, mu, dxes


@pytest.mark.parametrize('shape', [(9, 10, 70), (1, 12, 5), (7, 1, 1), (40, 7, 100), (33, 5, 64), (17, 3, 130)])
@pytest.mark.parametrize('steps', [5, 6])
@pytest.mark.parametrize('dtype', [numpy.float64, numpy.float32])
def test_run_matches_steps_and_oracle(shape, steps, dtype):
    """The fused runner (one pass per step over a ping-pong pair; slabs, partial y and z
    tiles, odd step counts) equals the separate H and E updates bit for bit."""
    from meanas_amd import fdtd
    e, h, eps, mu, dxes = _fields(shape, 1, dtype)
    dt = 0.2
    et = torch.from_numpy(e.copy()).cuda()
    ht = torch.from_numpy(h.copy()).cuda()
    fdtd.run(et, ht, eps, dt, dxes, steps=steps, mu=mu)
    e2, h2 = e.copy(), h.copy()
    me, mh = fdtd.maxwell_e(dt, dxes), fdtd.maxwell_h(dt, dxes)
    for _ in range(steps):
        mh(e2, h2, mu)
        me(e2, h2, eps)
    numpy.testing.assert_array_equal(et.cpu().numpy(), e2)   # same expressions, same order
    numpy.testing.assert_array_equal(ht.cpu().numpy(), h2)
    if dtype == numpy.float32:
        return
    e3, h3 = e.copy(), h.copy()
    for _ in range(steps):
        ref.maxwell_h(dt, dxes)(e3, h3, mu)
        ref.maxwell_e(dt, dxes)(e3, h3, eps)
    numpy.testing.assert_allclose(e2, e3, rtol=1e-11, atol=1e-12)
    numpy.testing.assert_allclose(h2, h3, rtol=1e-11, atol=1e-12)


@pytest.mark.parametrize('shape', [(2, 8, 60), (5, 9, 61), (1, 7, 59), (130, 16, 121), (3, 2, 2), (6, 25, 1)])
@pytest.mark.parametrize('eps_kind,mu_kind', [('field', None), ('field', 'field'), ('field', 'scalar'), ('scalar', None),
                                              ('scalar', 'field')])
@pytest.mark.parametrize('dtype', [numpy.float64, numpy.float32])
@pytest.mark.parametrize('steps', [1, 2, 3])
def test_run_passes_at_tile_edges(shape, eps_kind, mu_kind, dtype, steps):
    """Passes of two steps and a last one of one: tiles of 8 (one step: 10) rows and 60 (62)
    cells with remainders 0 and 1, several slabs, and every material form, against the
    separate updates bit for bit."""
    from meanas_amd import fdtd
    e, h, eps, mu, dxes = _fields(shape, 3, dtype)
    eps = eps if eps_kind == 'field' else 2.5
    mu = mu if mu_kind == 'field' else 1.7 if mu_kind == 'scalar' else None
    dt = 0.2
    et, ht = torch.from_numpy(e.copy()).cuda(), torch.from_numpy(h.copy()).cuda()
    fdtd.run(et, ht, eps, dt, dxes, steps=steps, mu=mu)
    me, mh = fdtd.maxwell_e(dt, dxes), fdtd.maxwell_h(dt, dxes)
    e2, h2 = torch.from_numpy(e.copy()).cuda(), torch.from_numpy(h.copy()).cuda()
    for _ in range(steps):
        mh(e2, h2, mu)
        me(e2, h2, eps)
    assert torch.equal(et, e2) and torch.equal(ht, h2)


@pytest.mark.parametrize('shape', [(326, 9, 61), (326, 10, 61), (214, 19, 61)])
@pytest.mark.parametrize('mu_kind', [None, 'field'])
@pytest.mark.parametrize('steps', [1, 4])
def test_float32_runs_in_blocks_of_14_rows(shape, mu_kind, steps):
    """Long thin float32 grids, where blocks of 14 rows (10 stored by a pass of two steps) fit
    the chip better than those of 12: 9, 10 and 19 rows, a last slab shorter than the others,
    against the separate updates bit for bit."""
    from meanas_amd import fdtd
    e, h, eps, mu, dxes = _fields(shape, 4, numpy.float32)
    mu = mu if mu_kind == 'field' else None
    dt = 0.2
    et, ht = torch.from_numpy(e.copy()).cuda(), torch.from_numpy(h.copy()).cuda()
    fdtd.run(et, ht, eps, dt, dxes, steps=steps, mu=mu)
    me, mh = fdtd.maxwell_e(dt, dxes), fdtd.maxwell_h(dt, dxes)
    e2, h2 = torch.from_numpy(e.copy()).cuda(), torch.from_numpy(h.copy()).cuda()
    for _ in range(steps):
        mh(e2, h2, mu)
        me(e2, h2, eps)
    assert torch.equal(et, e2) and torch.equal(ht, h2)


@pytest.mark.parametrize('shape', [(100_003, 1, 1), (30_000, 2, 3), (129, 1, 70), (1, 1, 400)])
@pytest.mark.parametrize('dtype', [torch.float64, torch.float32])
def test_runs_on_long_thin_grids(shape, dtype):
    """Runs equal the separate updates bit for bit on grids of many slabs, or of one plane."""
    from meanas_amd import fdtd
    gen = torch.Generator(device='cuda').manual_seed(2)
    e, h = [torch.randn((3, *shape), dtype=dtype, device='cuda', generator=gen) for _ in range(2)]
    eps = 1 + torch.rand((3, *shape), dtype=dtype, device='cuda', generator=gen)
    dxes = [[0.8 + 0.4 * numpy.random.default_rng(a).random(n) for a, n in enumerate(shape)] for _ in range(2)]
    e1, h1 = e.clone(), h.clone()
    fdtd.run(e1, h1, eps, 0.2, dxes, steps=5)
    me, mh = fdtd.maxwell_e(0.2, dxes), fdtd.maxwell_h(0.2, dxes)
    for _ in range(5):
        mh(e, h)
        me(e, h, eps)
    assert torch.equal(e, e1) and torch.equal(h, h1)


@pytest.mark.parametrize('shape', [(1, 40, 70), (2, 40, 70), (2, 1500, 1600), (3, 23, 130), (4, 40, 64), (5, 40, 64)])
@pytest.mark.parametrize('dtype', [torch.float64, torch.float32])
@pytest.mark.parametrize('with_mu', [False, True])
@pytest.mark.parametrize('steps', [1, 4, 5])
def test_runs_on_few_planes(shape, dtype, with_mu, steps):
    """Runs on one to five x planes (separate updates, passes of one step, of two) equal the
    separate updates bit for bit."""
    from meanas_amd import fdtd
    gen = torch.Generator(device='cuda').manual_seed(2)
    e, h = [torch.randn((3, *shape), dtype=dtype, device='cuda', generator=gen) for _ in range(2)]
    eps, mu = [1 + torch.rand((3, *shape), dtype=dtype, device='cuda', generator=gen) for _ in range(2)]
    mu = mu if with_mu else None
    dxes = [[0.8 + 0.4 * numpy.random.default_rng(a).random(n) for a, n in enumerate(shape)] for _ in range(2)]
    e1, h1 = e.clone(), h.clone()
    fdtd.run(e1, h1, eps, 0.2, dxes, steps=steps, mu=mu)
    me, mh = fdtd.maxwell_e(0.2, dxes), fdtd.maxwell_h(0.2, dxes)
    for _ in range(steps):
        mh(e, h, mu)
        me(e, h, eps)
    assert torch.equal(e, e1) and torch.equal(h, h1)


@pytest.mark.parametrize('with_mu', [False, True])
def test_run_with_components_beyond_4_gib(with_mu):
    """float64 passes with 64-bit offsets (a component of 5.4e8 cells, 4.3 GB; about 100 GB in
    all) equal the separate updates bit for bit."""
    from meanas_amd import fdtd
    shape = (840, 805, 800)
    fields = [torch.empty((3, *shape), dtype=torch.float64, device='cuda').uniform_(-1, 1) for _ in range(2)]
    eps = torch.empty_like(fields[0]).uniform_(1, 2)
    mu = eps if with_mu else None
    e, h = [f.clone() for f in fields]
    fdtd.run(e, h, eps, 0.25, None, steps=3, mu=mu)
    e1, h1 = fields
    me, mh = fdtd.maxwell_e(0.25), fdtd.maxwell_h(0.25)
    for _ in range(3):
        mh(e1, h1, mu)
        me(e1, h1, eps)
    assert torch.equal(e, e1) and torch.equal(h, h1)


@pytest.mark.parametrize('dtype', [numpy.float64, numpy.float32])
def test_updates_keep_infinities_zeros_and_nan(dtype):
    """Infinite fields and materials, zero and NaN values divide as numpy divides them."""
    from meanas_amd import fdtd
    shape = (6, 12, 70)
    e, h, eps, mu, dxes = _fields(shape, 5, dtype)
    e[1, 2, 3, 4] = numpy.inf
    e[2, 4, 9, 65] = numpy.nan
    h[0, 1, 1, 1] = -numpy.inf
    eps[:, 3, 5, 20] = numpy.inf
    eps[0, 5, 11, 30] = 0.0
    mu[2, 1, 10, 40] = numpy.inf
    # float32 numpy updates keep the float64 widths' precision, so they round differently
    tol = 1e-12 if dtype == numpy.float64 else 1e-4
    with numpy.errstate(all='ignore'):
        e1, h1 = e.copy(), h.copy()
        for _ in range(2):
            ref.maxwell_h(0.2, dxes)(e1, h1, mu)
            ref.maxwell_e(0.2, dxes)(e1, h1, eps)
    et, ht = torch.from_numpy(e.copy()).cuda(), torch.from_numpy(h.copy()).cuda()
    fdtd.run(et, ht, eps, 0.2, dxes, steps=2, mu=mu)
    numpy.testing.assert_allclose(et.cpu().numpy(), e1, rtol=tol, atol=tol)
    numpy.testing.assert_allclose(ht.cpu().numpy(), h1, rtol=tol, atol=tol)


def _plain_step(e, h, dt, dxes, eps, mu, which):
    """One update in torch, in the fields' own precision, by the updates' expressions."""
    w = [[torch.as_tensor(d).to(e).reshape([-1 if b == a else 1 for b in range(3)]) for a, d in enumerate(side)]
         for side in dxes]

    def d(f, a):
        if which == 'h':
            return (torch.roll(f, -1, a) - f) / w[0][a]
        return (f - torch.roll(f, 1, a)) / w[1][a]
    f = e if which == 'h' else h
    c = torch.stack([d(f[2], 1) - d(f[1], 2), d(f[0], 2) - d(f[2], 0), d(f[1], 0) - d(f[0], 1)])
    dt = torch.tensor(dt, dtype=e.dtype, device=e.device)
    return (e, h - dt * c / mu) if which == 'h' else (e + dt * c / eps, h)


def _same_values(got, want, tol, what):
    got = got.cpu()
    assert torch.equal(got.isnan(), want.isnan()), what
    assert torch.equal(torch.where(got.isinf(), got, 0), torch.where(want.isinf(), want, 0)), what
    fin = want.isfinite()
    torch.testing.assert_close(got[fin], want[fin], rtol=tol, atol=tol * float(want[fin].abs().median()), msg=what)


@pytest.mark.parametrize('shape', [(6, 12, 70), (9, 23, 61)])
@pytest.mark.parametrize('dtype,big,small_width,tiny,top', [(torch.float32, 1e38, 1e-3, 1e-39, 8e37),
                                                            (torch.float64, 1e307, 1e-5, 1e-309, 1.7e308)])
def test_quotients_that_overflow_and_extreme_divisors(shape, dtype, big, small_width, tiny, top):
    """Finite dividends whose quotient overflows, and the largest divisors: infinities, NaN and
    values where division puts them, in the separate updates, the CPML updates and runs.
    Divisors out of the documented range: subnormal ones count as zero, float32 ones above
    2^126 as infinite."""
    from meanas_amd import fdtd
    gen = torch.Generator().manual_seed(3)
    e, h = [torch.randn((3, *shape), dtype=dtype, generator=gen) for _ in range(2)]
    eps, mu = [1 + torch.rand((3, *shape), dtype=dtype, generator=gen) for _ in range(2)]
    dxes = [[0.8 + 0.4 * numpy.random.default_rng(a).random(n) for a, n in enumerate(shape)] for _ in range(2)]
    for side in dxes:
        side[1][3] = small_width
        side[2][30] = small_width
    e[0, 1, 3, 4] = h[2, 1, 3, 40] = big                 # over the small width: overflow
    e[1, 4, 7, 30] = h[0, 4, 7, 30] = -big
    e[1, 3, 1, 50] = h[0, 3, 1, 50] = big                # and a quotient by the largest divisors
    mu[:, 2:4, 0:3, 48:52] = eps[:, 2:4, 0:3, 48:52] = top
    mu[:, 5, 9, 12] = eps[:, 5, 10, 12] = tiny           # subnormal divisors
    if dtype == torch.float32:
        mu[:, 0, 6, 58] = eps[:, 0, 6, 58] = 3e38
    tol = 1e-5 if dtype == torch.float32 else 1e-13
    dev = [t.cuda() for t in (e, h, eps, mu)]
    for m in (eps, mu):
        m[m < 2 * tiny] = 0.0
        m[m > (2.0 ** 126 if dtype == torch.float32 else torch.inf)] = torch.inf
    want_h = _plain_step(e, h, 0.2, dxes, eps, mu, 'h')[1]
    want_e = _plain_step(e, h, 0.2, dxes, eps, mu, 'e')[0]
    assert want_h.isinf().any() and want_e.isinf().any()
    et, ht = dev[0].clone(), dev[1].clone()
    _same_values(fdtd.maxwell_h(0.2, dxes)(dev[0], ht, dev[3]), want_h, tol, 'maxwell_h')
    _same_values(fdtd.maxwell_e(0.2, dxes)(et, dev[1], dev[2]), want_e, tol, 'maxwell_e')
    if dtype == torch.float64:   # (its float32 form divides in double)
        same = [dxes[1], dxes[1]]
        uE, uH = fdtd.updates_with_cpml([[None, None]] * 3, 0.2, same, dev[2])
        et, ht = dev[0].clone(), dev[1].clone()
        uE(et, dev[1], dev[2])
        uH(dev[0], ht, dev[3])
        # dt / material is formed first there
        for got, f, w, m in ((et, e, 'e', eps), (ht, h, 'h', mu)):
            zero = torch.zeros_like(f)
            c = _plain_step(e if w == 'h' else zero, zero if w == 'h' else h, 1.0, same, 1.0, 1.0, w)[w == 'h']
            _same_values(got, f + (0.2 / m) * c, tol, 'cpml ' + w)   # (c carries the H update's sign)
    for steps in (1, 2, 3):
        e1, h1 = e, h
        for _ in range(steps):
            e1, h1 = _plain_step(e1, h1, 0.2, dxes, eps, mu, 'h')
            e1, h1 = _plain_step(e1, h1, 0.2, dxes, eps, mu, 'e')
        et, ht = dev[0].clone(), dev[1].clone()
        fdtd.run(et, ht, dev[2], 0.2, dxes, steps=steps, mu=dev[3])
        _same_values(et, e1, tol, f'run e {steps}')
        _same_values(ht, h1, tol, f'run h {steps}')


def test_unit_widths_scalar_materials_and_float32():
    from meanas_amd import fdtd
    shape = (8, 6, 66)
    e, h, eps, mu, dxes = _fields(shape, 2, numpy.float64)
    dt = 0.25
    e64, h64 = e.copy(), h.copy()
    fdtd.run(e64, h64, 2.0, dt, None, steps=5, mu=1.5)          # numpy in, updated in place
    e1, h1 = e.copy(), h.copy()                                 # the separate updates, bit for bit
    me, mh = fdtd.maxwell_e(dt), fdtd.maxwell_h(dt)
    for _ in range(5):
        mh(e1, h1, 1.5)
        me(e1, h1, 2.0)
    numpy.testing.assert_array_equal(e64, e1)
    numpy.testing.assert_array_equal(h64, h1)
    eo, ho = e.copy(), h.copy()
    for _ in range(5):
        ref.maxwell_h(dt)(eo, ho, 1.5)
        ref.maxwell_e(dt)(eo, ho, 2.0)
    numpy.testing.assert_allclose(e64, eo, rtol=1e-11, atol=1e-12)
    numpy.testing.assert_allclose(h64, ho, rtol=1e-11, atol=1e-12)
    e32, h32 = e.astype(numpy.float32), h.astype(numpy.float32)
    fdtd.run(e32, h32, 2.0, dt, None, steps=5, mu=1.5)
    assert e32.dtype == numpy.float32
    numpy.testing.assert_allclose(e32, eo, rtol=1e-4, atol=1e-4)
    numpy.testing.assert_allclose(h32, ho, rtol=1e-4, atol=1e-4)


# ---- CPML (meanas/fdtd/pml.py) against the oracle's restatement ---------------------
def _cpml_case(shape, faces, thickness, seed, fdt, with_mu):
    rng = numpy.random.default_rng(seed)
    e = rng.standard_normal((3, *shape)).astype(fdt)
    h = rng.standard_normal((3, *shape)).astype(fdt)
    eps = (1 + rng.random((3, *shape))).astype(fdt)
    mu = (1 + rng.random((3, *shape))).astype(fdt) if with_mu else None
    dxes = [[0.8 + 0.4 * rng.random(n) for n in shape] for _ in range(2)]
    return e, h, eps, mu, dxes


@pytest.mark.parametrize('fdt,pdt,tol', [(numpy.float64, numpy.float64, 1e-11), (numpy.float64, numpy.float32, 1e-5),
                                         (numpy.float32, numpy.float32, 1e-4), (numpy.float32, numpy.float64, 1e-4)])
@pytest.mark.parametrize('shape,faces,thickness', [
    ((14, 12, 9), fc.ALL_FACES, 4),
    ((10, 9, 7), fc.ALL_FACES, 4),                 # z layers overlap (2 * 4 > 7)
    ((16, 1, 11), [(0, 1), (2, -1)], 5),           # two faces, one flat axis
])
@pytest.mark.parametrize('with_mu', [False, True])
def test_cpml_updates_match_oracle(fdt, pdt, tol, shape, faces, thickness, with_mu):
    from meanas_amd import fdtd
    e, h, eps, mu, dxes = _cpml_case(shape, faces, thickness, 5, fdt, with_mu)
    dt = 0.3
    kw = dict(epsilon_eff=2.0, cfs_alpha=0.05)
    uE, uH = ref.updates_with_cpml(fc.cpml_layers(ref.cpml_params, dt, faces, thickness, **kw), dt, dxes, eps,
                                   dtype=pdt)
    gE, gH = fdtd.updates_with_cpml(fc.cpml_layers(fdtd.cpml_params, dt, faces, thickness, **kw), dt, dxes, eps,
                                    dtype=pdt)
    et, ht = torch.from_numpy(e.copy()).cuda(), torch.from_numpy(h.copy()).cuda()
    epst = torch.from_numpy(eps).cuda()
    mut = None if mu is None else torch.from_numpy(mu).cuda()
    for _ in range(6):
        if mu is None:
            uH(e, h)
            gH(et, ht)
        else:
            uH(e, h, mu)
            gH(et, ht, mut)
        uE(e, h, eps)
        gE(et, ht, epst)
    scale = max(numpy.abs(e).max(), numpy.abs(h).max())
    numpy.testing.assert_allclose(et.cpu().numpy(), e, rtol=tol, atol=tol * scale)
    numpy.testing.assert_allclose(ht.cpu().numpy(), h, rtol=tol, atol=tol * scale)


@pytest.mark.parametrize('fdt,pdt,tol', [(numpy.float64, numpy.float64, 1e-11), (numpy.float32, numpy.float32, 1e-4)])
@pytest.mark.parametrize('shape', [(4, 16, 16), (5, 16, 17), (67, 5, 51), (18, 3, 6)])
def test_cpml_columns_and_slabs(fdt, pdt, tol, shape):
    """(y, z) planes of exactly one 256-thread block, one cell more, and less than one; x
    axes of one slab, of whole slabs and of a remainder; layers on every face that fits."""
    from meanas_amd import fdtd
    dt, thick = 0.2, 3
    rng = numpy.random.default_rng(11)
    e = rng.standard_normal((3, *shape)).astype(fdt)
    h = rng.standard_normal((3, *shape)).astype(fdt)
    eps = (1 + rng.random((3, *shape))).astype(fdt)
    dxes = [[0.8 + 0.4 * rng.random(n) for n in shape] for _ in range(2)]
    make = [[mod.cpml_params(a, p, dt, thickness=thick) if shape[a] > thick else None for p in (-1, 1)] for mod in (fdtd, ref)
            for a in range(3)]
    uE, uH = fdtd.updates_with_cpml(make[:3], dt, dxes, eps, dtype=pdt)
    rE, rH = ref.updates_with_cpml(make[3:], dt, dxes, eps, dtype=pdt)
    et, ht = torch.from_numpy(e.copy()).cuda(), torch.from_numpy(h.copy()).cuda()
    for _ in range(4):
        uE(et, ht, eps)
        uH(et, ht)
        rE(e, h, eps)
        rH(e, h)
    numpy.testing.assert_allclose(et.cpu().numpy(), e, rtol=tol, atol=tol)
    numpy.testing.assert_allclose(ht.cpu().numpy(), h, rtol=tol, atol=tol)


def test_cpml_plane_beyond_32_bit_offsets():
    """A float64 (y, z) plane of more than 4 GiB (one x plane; about 30 GB in all): rows at
    both ends and in the middle against the same differences in torch."""
    from meanas_amd import fdtd
    shape = (1, 23200, 23200)
    e = torch.empty((3, *shape), dtype=torch.float64, device='cuda').uniform_(-1, 1)
    h = torch.zeros_like(e)
    n = shape[1]
    dxes = [[numpy.ones(k) for k in shape] for _ in range(2)]
    _, uH = fdtd.updates_with_cpml([[None, None]] * 3, 0.25, dxes, e)
    uH(e, h)
    for j in (0, n // 2, n - 1):
        here, up = e[:, 0, j], e[:, 0, (j + 1) % n]
        dz = [torch.roll(here[c], -1, 0) - here[c] for c in range(3)]
        want = torch.stack([(up[2] - here[2]) - dz[1], dz[0], -(up[0] - here[0])]) * -0.25
        torch.testing.assert_close(h[:, 0, j], want, rtol=1e-14, atol=1e-14)


@pytest.mark.parametrize('axis', [1, 2])
def test_cpml_psi_beyond_32_bit_offsets(axis):
    """float32 fields of less than 4 GiB a plane with float64 psi of more (one x plane, a layer
    of 8 cells over the short axis; about 40 GB in all): two H updates at cells at both ends,
    in the middle and on both sides of the psi's 4 GiB line."""
    from meanas_amd import fdtd
    n, t, dt = 70_000_000, 8, 0.25
    shape = (1, t, n) if axis == 1 else (1, n, t)
    e = torch.empty((3, *shape), dtype=torch.float32, device='cuda').uniform_(-1, 1)
    h = torch.zeros_like(e)
    layer = fdtd.cpml_params(axis=axis, polarity=-1, dt=dt, thickness=t)
    layers = [[None, None] for _ in range(3)]
    layers[axis][0] = layer
    _, uH = fdtd.updates_with_cpml(layers, dt, [[numpy.ones(k) for k in shape] for _ in range(2)], e, dtype=numpy.float64)
    uH(e, h)
    uH(e, h)
    line = 2 ** 29 // t if axis == 2 else 2 ** 29 - (2 ** 29 // n) * n   # where 8-byte offsets pass 2^32
    p0, p1, p2 = [torch.from_numpy(q.ravel()).cuda() for q in layer['param_h']]
    for at in (0, line - 1, line, n // 2, n - 1):
        here, nxt = [e[:, 0, :, k] if axis == 1 else e[:, 0, k] for k in (at, (at + 1) % n)]   # (3, t)
        across = (torch.roll(here, -1, 1) - here).double() * p2   # along the layer's axis
        along = (nxt - here).double()
        dy, dz = (across, along) if axis == 1 else (along, across)
        curl = torch.stack([dy[2] - dz[1], dz[0], -dy[0]])
        psi = p1 * across                                  # after the first update
        both = 2 * psi + p0 * psi                          # and summed over the two
        aux = torch.zeros_like(curl)
        if axis == 1:
            aux[0], aux[2] = both[2], -both[0]
        else:
            aux[0], aux[1] = -both[1], both[0]
        want = -dt * (2 * curl + aux)
        got = h[:, 0, :, at] if axis == 1 else h[:, 0, at]
        # |h| < 4, rounded to float32 once per update: at most 2 x 1.2e-7
        assert float((got.double() - want).abs().max()) < 3e-7, (axis, at)


@pytest.mark.parametrize('axis,comp', [(0, 1), (1, 2), (2, 0)])
def test_cpml_absorbs_a_pulse_on_gpu(axis, comp):
    from meanas_amd import fdtd
    upd = lambda p, dt, dxes, eps: fdtd.updates_with_cpml(p, dt, dxes, eps)
    final, top = fc.pulse_energy(upd, axis, comp, make=fdtd.cpml_params,
                                 to_dev=lambda a: torch.from_numpy(a).cuda(), to_host=lambda t: t.cpu().numpy())
    assert final < 1e-8 and top < 1.05


def test_cpml_numpy_fields_and_defaults():
    """numpy fields are written back in place; mu defaults to (1, 1, 1); no layers and
    equal E/H widths give the plain updates."""
    from meanas_amd import fdtd
    e, h, eps, _, dxes = _cpml_case((6, 5, 4), [], 3, 7, numpy.float64, False)
    dxes = [dxes[1], dxes[1]]
    gE, gH = fdtd.updates_with_cpml([[None, None]] * 3, 0.2, dxes, eps, dtype=numpy.float64)
    e1, h1 = e.copy(), h.copy()
    assert gH(e1, h1) is None and gE(e1, h1, eps) is None
    e2, h2 = e.copy(), h.copy()
    ref.maxwell_h(0.2, dxes)(e2, h2)
    ref.maxwell_e(0.2, dxes)(e2, h2, eps)
    numpy.testing.assert_allclose(e1, e2, rtol=1e-12, atol=1e-12)
    numpy.testing.assert_allclose(h1, h2, rtol=1e-12, atol=1e-12)


def test_cpml_rejects_what_has_no_kernel_form():
    import ctypes
    from meanas_amd import _lib, fdtd
    shape = (8, 8, 8)
    eps = numpy.ones((3, *shape))
    lay = fdtd.cpml_params(0, -1, 0.3, thickness=3)
    bad = dict(lay, region=(slice(2, 5), slice(None), slice(None)))
    with pytest.raises(ValueError):
        fdtd.updates_with_cpml([[bad, None], [None, None], [None, None]], 0.3, None, eps)
    with pytest.raises(ValueError):   # a polarity -1 layer in the +1 slot
        fdtd.updates_with_cpml([[None, lay], [None, None], [None, None]], 0.3, None, eps)
    # the C ABI refuses layers out of (axis, polarity) order
    gE, _ = fdtd.updates_with_cpml([[lay, fdtd.cpml_params(0, 1, 0.3, thickness=3)], [None, None], [None, None]],
                                   0.3, None, eps)
    tab = (_lib.MxCpmlLayer * 2)()
    ptrs = [a.data_ptr() for a in gE.psi_state[:4]]
    tab[0] = _lib.MxCpmlLayer(0, 1, 3, 0, *ptrs)
    tab[1] = _lib.MxCpmlLayer(0, -1, 3, 0, *ptrs)
    e = torch.zeros((3, *shape), dtype=torch.float64, device='cuda')
    grid = _lib.MxFdtdGrid(8, 8, 8, 0, (ctypes.c_void_p * 3)(), (ctypes.c_void_p * 3)())
    rc = _lib.lib().mx_fdtd_cpml_e(ctypes.byref(grid), _lib.MX_REAL64, _lib.MX_REAL32, 0.3, e.data_ptr(), e.data_ptr(),
                                   None, 1.0, tab, 2, None)
    assert rc != 0 and b'order' in _lib.lib().mx_last_error()


# ---- conducting boundary (meanas/fdtd/boundaries.py) ------------------------------
@pytest.mark.parametrize('direction', [0, 1, 2])
@pytest.mark.parametrize('polarity', [-1, 1])
@pytest.mark.parametrize('dtype', [numpy.float64, numpy.float32])
@pytest.mark.parametrize('size', ['minimal', 'regular'])
def test_conducting_boundary_matches_oracle(direction, polarity, dtype, size):
    """Both field updates of one face equal the oracle's bit for bit (copies, zeros and
    negations only); the smallest axis each polarity accepts is included."""
    from meanas_amd import fdtd
    shape = [5, 6, 7] if size == 'regular' else [3, 4, 1]
    if size == 'minimal':
        shape[direction] = 2 if polarity < 0 else 3
    rng = numpy.random.default_rng(10 + direction + 3 * polarity)
    for kind in (0, 1):
        f = rng.standard_normal((3, *shape)).astype(dtype)
        want = ref.conducting_boundary(direction, polarity)[kind](f.copy())
        t = torch.from_numpy(f.copy()).cuda()
        got = fdtd.conducting_boundary(direction, polarity)[kind](t)
        assert got is t
        numpy.testing.assert_array_equal(t.cpu().numpy(), want)


@pytest.mark.parametrize('direction', [0, 1, 2])
@pytest.mark.parametrize('dtype,tol', [(numpy.float64, 1e-13), (numpy.float32, 1e-5)])
def test_conducting_boundary_is_a_mirror_on_gpu(direction, dtype, tol):
    """GPU updates with the GPU boundaries on both faces equal a plain periodic GPU run on
    the doubled mirror-symmetric domain."""
    from meanas_amd import fdtd
    mh, me = fdtd.maxwell_h(0.3), fdtd.maxwell_e(0.3)

    def step(e, h, eps, after_h, after_e):
        mh(e, h)
        after_h()
        me(e, h, eps)
        after_e()
    worst = fc.mirror_mismatch(direction, 7, step, fdtd.conducting_boundary, dtype=dtype, seed=direction,
                               to_dev=lambda a: torch.from_numpy(a).cuda(), to_host=lambda t: t.cpu().numpy())
    assert worst <= tol


def test_conducting_boundary_numpy_and_errors():
    from meanas_amd import fdtd
    en, hn = fdtd.conducting_boundary(0, -5)        # any negative polarity is the low face
    f = numpy.random.default_rng(0).standard_normal((3, 4, 3, 2))
    want = ref.conducting_boundary(0, -1)[1](f.copy())
    assert hn(f) is f                                # numpy written back in place
    numpy.testing.assert_array_equal(f, want)
    ep, _ = fdtd.conducting_boundary(2, 1)
    with pytest.raises(IndexError):                  # +1 needs three cells along the axis
        ep(torch.zeros((3, 4, 4, 2), dtype=torch.float64, device='cuda'))
    with pytest.raises(TypeError):
        en(torch.zeros((3, 4, 4, 2), dtype=torch.complex128, device='cuda'))
    with pytest.raises(Exception, match='Invalid direction'):
        fdtd.conducting_boundary(3, 1)
    with pytest.raises(Exception, match='Bad polarity'):
        fdtd.conducting_boundary(1, 0)


# ---- energy and Poynting functions (meanas/fdtd/energy.py) -------------------------
def _gpu_energy():
    from types import SimpleNamespace
    from meanas_amd import fdtd
    return SimpleNamespace(energy_hstep=fdtd.energy_hstep, energy_estep=fdtd.energy_estep,
                           delta_energy_j=fdtd.delta_energy_j, poynting_divergence=fdtd.poynting_divergence,
                           poynting=fdtd.poynting)


@pytest.mark.parametrize('case', fc.cases())
def test_reference_fdtd_checks_with_gpu_energy(case):
    """The reference's FDTD checks (initial energy, energy conservation, Poynting
    divergence and planes) on GPU-stepped fields, with the GPU's energy and Poynting
    functions as the checker."""
    sim = fc.make_sim(case, gpu_step)
    sim.en = _gpu_energy()
    for check in fc.CHECKS:
        check(sim)


@pytest.mark.parametrize('dtype,tol', [(numpy.float64, 1e-14), (numpy.float32, 1e-6)])
@pytest.mark.parametrize('shape', [(5, 6, 7), (1, 4, 9), (8, 1, 3)])
@pytest.mark.parametrize('widths', [True, False])
@pytest.mark.parametrize('mats', ['field', 'scalar', None])
def test_energy_functions_match_oracle(dtype, tol, shape, widths, mats):
    """Every function of energy.py against the oracle's, which follows the reference's
    expression order (products and component sums in the field precision, widths in
    float64, one axis at a time)."""
    from meanas_amd import fdtd
    rng = numpy.random.default_rng(len(shape) * 7 + shape[0])
    f = [rng.standard_normal((3, *shape)).astype(dtype) for _ in range(4)]
    dxes = [[0.5 + rng.random(n) for n in shape] for _ in range(2)] if widths else None
    eps = {'field': (1 + rng.random((3, *shape))).astype(dtype), 'scalar': 2.5, None: None}[mats]
    mu = {'field': (1 + rng.random((3, *shape))).astype(dtype), 'scalar': 1.5, None: None}[mats]
    dt = 0.37
    kw = dict(epsilon=eps, mu=mu, dxes=dxes)
    dxes_given = dxes if dxes is not None else [[numpy.ones(n) for n in shape]] * 2
    pairs = {
        'hstep': (fdtd.energy_hstep(f[0], f[1], f[2], **kw), ref.energy_hstep(f[0], f[1], f[2], **kw)),
        'estep': (fdtd.energy_estep(f[0], f[1], f[2], **kw), ref.energy_estep(f[0], f[1], f[2], **kw)),
        'h2e': (fdtd.delta_energy_h2e(dt, *f, **kw), ref.delta_energy_h2e(dt, *f, **kw)),
        'e2h': (fdtd.delta_energy_e2h(dt, *f, **kw), ref.delta_energy_e2h(dt, *f, **kw)),
        'j': (fdtd.delta_energy_j(f[0], f[1], dxes=dxes), ref.delta_energy_j(f[0], f[1], dxes=dxes)),
        'dxmul': (fdtd.dxmul(f[0], f[1], **kw), ref.dxmul(f[0], f[1], **kw)),
        'poynting': (fdtd.poynting(f[0], f[1], dxes), ref.fdtd_poynting(f[0], f[1], dxes)),
        'div_s': (fdtd.poynting_divergence(f[2]), ref.poynting_divergence(f[2])),
        'div_eh': (fdtd.poynting_divergence(e=f[0], h=f[1], dxes=dxes_given),
                   ref.poynting_divergence(e=f[0], h=f[1], dxes=dxes_given)),
    }
    for name, (got, want) in pairs.items():
        assert isinstance(got, numpy.ndarray) and got.dtype == want.dtype and got.shape == want.shape, name
        scale = numpy.abs(want).max()
        numpy.testing.assert_allclose(got, want, rtol=tol, atol=tol * scale, err_msg=name)


def test_energy_functions_on_device_tensors():
    """CUDA tensors in, CUDA tensors out, equal to the numpy path; mixed dtypes refused."""
    from meanas_amd import fdtd
    rng = numpy.random.default_rng(3)
    e, h, e2 = (rng.standard_normal((3, 6, 5, 4)) for _ in range(3))
    dev = [torch.from_numpy(a).cuda() for a in (e, h, e2)]
    u = fdtd.energy_hstep(*dev, epsilon=2.0)
    assert isinstance(u, torch.Tensor) and u.is_cuda and u.dtype == torch.float64
    numpy.testing.assert_array_equal(u.cpu().numpy(), fdtd.energy_hstep(e, h, e2, epsilon=2.0))
    s = fdtd.poynting(dev[0], dev[1])
    assert isinstance(s, torch.Tensor) and s.shape == (3, 6, 5, 4)
    numpy.testing.assert_array_equal(s.cpu().numpy(), fdtd.poynting(e, h))
    dxes = [[0.5 + rng.random(n) for n in (6, 5, 4)] for _ in range(2)]
    first = fdtd.energy_estep(e, h, e2, dxes=dxes)
    numpy.testing.assert_allclose(first, ref.energy_estep(e, h, e2, dxes=dxes), rtol=1e-14)
    dxes[0][1] *= 1.5                        # changed in place: the device widths follow
    numpy.testing.assert_allclose(fdtd.energy_estep(e, h, e2, dxes=dxes), ref.energy_estep(e, h, e2, dxes=dxes),
                                  rtol=1e-14)
    with pytest.raises(ValueError):
        fdtd.energy_estep(e, h.astype(numpy.float32), e2)
    with pytest.raises(AssertionError):     # as the reference: e, h and dxes, or s
        fdtd.poynting_divergence(e=e, h=h)


@pytest.mark.parametrize('dtype', [numpy.float64, numpy.float32])
@pytest.mark.parametrize('shape', [(4, 16, 16), (5, 16, 17), (13, 5, 60), (1, 1, 300)])
def test_column_kernels_at_block_and_slab_edges(dtype, shape):
    """Updates, energy, Poynting vector and divergence on (y, z) planes of one 256-thread
    block, one cell more, less, and several, with whole and partial slabs."""
    from meanas_amd import fdtd
    e, h, eps, mu, dxes = _fields(shape, 17, dtype)
    tol = 1e-13 if dtype == numpy.float64 else 2e-5
    kw = dict(rtol=tol, atol=tol)
    e2, h2 = numpy.roll(e, 1, axis=2), numpy.roll(h, 1, axis=3)
    numpy.testing.assert_allclose(fdtd.energy_hstep(e, h, e2, eps, mu, dxes), ref.energy_hstep(e, h, e2, eps, mu, dxes), **kw)
    numpy.testing.assert_allclose(fdtd.delta_energy_e2h(0.2, h, e, h2, e2, eps, mu, dxes),
                                  ref.delta_energy_e2h(0.2, h, e, h2, e2, eps, mu, dxes), rtol=tol, atol=20 * tol)
    s = ref.fdtd_poynting(e, h, dxes)
    numpy.testing.assert_allclose(fdtd.poynting(e, h, dxes), s, **kw)
    numpy.testing.assert_allclose(fdtd.poynting_divergence(s.astype(dtype)), ref.poynting_divergence(s.astype(dtype)), **kw)
    e1, h1 = e.copy(), h.copy()
    ref.maxwell_h(0.2, dxes)(h=h1, e=e1, mu=mu)
    ref.maxwell_e(0.2, dxes)(e1, h1, eps)
    fdtd.maxwell_h(0.2, dxes)(e, h, mu)
    fdtd.maxwell_e(0.2, dxes)(e, h, eps)
    numpy.testing.assert_allclose(h, h1, **kw)
    numpy.testing.assert_allclose(e, e1, **kw)


@pytest.mark.parametrize('dtype', [numpy.float64, numpy.float32])
@pytest.mark.parametrize('shape', [(3000, 1, 1), (600, 1, 3), (9, 7, 73), (9, 8, 64), (7, 19, 27), (1, 3, 256), (13, 30, 26)])
def test_cells_and_columns_by_plane_size(dtype, shape):
    """The same on thin planes (a thread per cell), of 511 cells and of 512, 513 and more
    (columns), and the CPML updates."""
    test_column_kernels_at_block_and_slab_edges(dtype, shape)
    test_cpml_columns_and_slabs(dtype, dtype, 1e-11 if dtype == numpy.float64 else 1e-4, shape)


@pytest.mark.parametrize('fdt,pdt,tol', [(numpy.float64, numpy.float32, 1e-5), (numpy.float32, numpy.float64, 1e-4)])
@pytest.mark.parametrize('shape', [(10, 90, 7), (10, 7, 90), (10, 9, 7)])
def test_cpml_overlapping_layers_by_plane_size(fdt, pdt, tol, shape):
    """Layers that overlap on a short axis, in columns and with a thread per cell."""
    test_cpml_updates_match_oracle(fdt, pdt, tol, shape, fc.ALL_FACES, 4, True)


@pytest.mark.parametrize('dtype,shape', [(torch.float64, (140, 163, 163)), (torch.float64, (141, 163, 166)),
                                         (torch.float32, (195, 196, 196)), (torch.float64, (177, 177, 178)),
                                         (torch.float64, (178, 177, 178))])
def test_large_grids_on_both_sides_of_the_cache(dtype, shape):
    """Grids just below and above the sizes where the work goes by blocks instead of by XCD, and
    where float64 updates with a material take a thread per cell, against the same in torch."""
    from meanas_amd import fdtd
    gen = torch.Generator(device='cuda').manual_seed(1)
    e, h, e2 = [torch.randn((3, *shape), dtype=dtype, device='cuda', generator=gen) for _ in range(3)]
    eps = 1 + torch.rand((3, *shape), dtype=dtype, device='cuda', generator=gen)
    dxes = [[0.8 + 0.4 * numpy.random.default_rng(a).random(n) for a, n in enumerate(shape)] for _ in range(2)]
    tol = dict(rtol=1e-13, atol=1e-12) if dtype == torch.float64 else dict(rtol=1e-5, atol=1e-4)
    torch.testing.assert_close(fdtd.energy_hstep(e, h, e2, epsilon=eps),
                               ((e * e2 * eps).double().sum(0) + (h * h).double().sum(0)), **tol)
    nx, ny, nz = [torch.roll(e, -1, a) for a in (1, 2, 3)]
    torch.testing.assert_close(fdtd.poynting(e, h), torch.stack([nx[1] * h[2] - nx[2] * h[1], ny[2] * h[0] - ny[0] * h[2],
                                                                 nz[0] * h[1] - nz[1] * h[0]]), **tol)
    w = [[torch.as_tensor(d).cuda().reshape([-1 if b == a else 1 for b in range(3)]) for a, d in enumerate(side)] for side in dxes]
    hw = [h[a].double() * w[1][a] for a in range(3)]
    flux = [nx[1] * w[0][1] * hw[2] - nx[2] * w[0][2] * hw[1], ny[2] * w[0][2] * hw[0] - ny[0] * w[0][0] * hw[2],
            nz[0] * w[0][0] * hw[1] - nz[1] * w[0][1] * hw[0]]
    torch.testing.assert_close(fdtd.poynting(e, h, dxes), torch.stack(flux).to(dtype), **tol)
    want_h = _plain_step(e, h, 0.2, dxes, None, eps, 'h')[1]
    want_e = _plain_step(e, h, 0.2, dxes, eps, None, 'e')[0]
    torch.testing.assert_close(fdtd.maxwell_h(0.2, dxes)(e, h.clone(), eps), want_h, **tol)
    torch.testing.assert_close(fdtd.maxwell_e(0.2, dxes)(e.clone(), h, eps), want_e, **tol)


def test_updates_on_a_line_of_1e8_cells():
    """A grid of one cell across and 1.1e8 cells along x: as many blocks as a launch may have."""
    from meanas_amd import fdtd
    n = 110_000_000
    f = torch.empty((3, n, 1, 1), dtype=torch.float32, device='cuda').uniform_(-1, 1)
    e, h = torch.zeros_like(f), torch.zeros_like(f)
    fdtd.maxwell_h(0.5)(f, h)
    fdtd.maxwell_e(0.5)(e, f, 1.0)
    x = f[:, :, 0, 0]
    for got, sign, d in ((h, -0.5, torch.roll(x, -1, 1) - x), (e, 0.5, x - torch.roll(x, 1, 1))):
        assert not got[0].any()
        assert torch.equal(got[1, :, 0, 0], -sign * d[2]) and torch.equal(got[2, :, 0, 0], sign * d[1])


@pytest.mark.parametrize('name', ['update', 'energy', 'poynting'])
def test_planes_beyond_32_bit_offsets(name):
    """One float64 x plane of more than 4 GiB: rows at both ends and in the middle."""
    from meanas_amd import fdtd
    n = 23200
    e = torch.empty((3, 1, n, n), dtype=torch.float64, device='cuda').uniform_(-1, 1)
    rows = (0, n // 2, n - 1)
    if name == 'energy':
        got = fdtd.dxmul(e, e)
        for j in rows:
            torch.testing.assert_close(got[0, j], 2 * e[:, 0, j].sum(0), rtol=1e-13, atol=1e-13)
        return
    if name == 'poynting':
        got = fdtd.poynting(e, e)
        for j in rows:
            x, y = e[:, 0, j], e[:, 0, (j + 1) % n]
            z = torch.roll(x, -1, 1)
            want = torch.stack([x[1] * x[2] - x[2] * x[1], y[2] * x[0] - y[0] * x[2], z[0] * x[1] - z[1] * x[0]])
            torch.testing.assert_close(got[:, 0, j], want, rtol=1e-13, atol=1e-13)
        return
    out = torch.zeros_like(e)
    fdtd.maxwell_e(0.25)(out, e, 2.0)
    for j in rows:
        x, y = e[:, 0, j], e[:, 0, j - 1]
        z = torch.roll(x, 1, 1)
        want = torch.stack([(x[2] - y[2]) - (x[1] - z[1]), x[0] - z[0], -(x[0] - y[0])]) * 0.125
        torch.testing.assert_close(out[:, 0, j], want, rtol=1e-13, atol=1e-13)


def test_calls_go_to_the_current_stream():
    """The stream handle of a call is the current stream's: the default one, a side stream, and
    the default one again; an explicit stream is taken as it is."""
    import torch
    from meanas_amd.fdfd.device import torch_stream_handle
    side = torch.cuda.Stream()
    default = torch.cuda.current_stream().cuda_stream

    def handle(*args):
        return torch_stream_handle(*args).value or 0
    assert handle() == default
    with torch.cuda.stream(side):
        assert handle() == side.cuda_stream
        assert handle(torch.cuda.default_stream()) == torch.cuda.default_stream().cuda_stream
    assert handle() == default
    assert handle(side) == side.cuda_stream
