"""ShapeFunction and ScatterGatherImpl through the C ABI (csrst_sg_*,
csrst_sf_*) against the CPU oracle, and the caller-geometry entries of the
two-grid step (csrst_set_mask, csrst_set_boundary_cells, csrst_set_stream).

The stateless kernels keep the reference's per-particle summation order, so
every result is compared bit for bit.  The charge-density difference is
checked against the discrete continuity equation with the GPU's own
currents (dt div J = -(rho(R) - rho(oldR)) to round-off).
"""
import ctypes as C
import threading
import time

import numpy as np
import pytest

from csrst_amd import Commands, TwoGridStep, gaussian_bunch, shapefn as SF
from csrst_amd._lib import CsrstError, check
from csrst_amd.mw import MovingWindowStep
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def same(a, b):
    return np.array_equal(np.asarray(a).view(np.uint64), np.asarray(b).view(np.uint64))


@pytest.mark.parametrize("order", [0, 1, 2])
@pytest.mark.parametrize("kind", ["Ex", "Ey", "cell"])
@pytest.mark.parametrize("s2bug", [False, True])
def test_gather_bitwise(gpu, order, kind, s2bug):
    rng = np.random.default_rng(order * 7 + len(kind))
    field = rng.normal(size=(30, 40))
    org, dx = (0.013, -0.021), (0.7, 1.3)
    R = np.stack([rng.uniform(org[0] + 4 * dx[0], org[0] + 34 * dx[0], 500),
                  rng.uniform(org[1] + 4 * dx[1], org[1] + 24 * dx[1], 500)], 1)
    got = SF.gather(order, kind, field, org, dx, R, s2bug=s2bug)
    if kind == "cell":
        ref = O.gather_cell(order, field, org, dx, R, s2bug)
    else:
        ref = O.gather_edge(order, 0 if kind == "Ex" else 1, field, org, dx, R, s2bug)
    assert same(got, ref)


@pytest.mark.parametrize("order", [0, 1, 2])
@pytest.mark.parametrize("kind", ["Ex", "Ey", "cell"])
def test_scatter_bitwise(gpu, order, kind):
    rng = np.random.default_rng(order * 5 + len(kind))
    org, dx = (0.0, 0.0), (1.0, 1.0)
    R = rng.uniform(5, 15, (2000, 2))          # many particles per node: the order of the sums matters
    val = rng.normal(size=2000)
    got = SF.scatter(order, kind, (24, 24), org, dx, R, val)
    if kind == "cell":
        ref = O.scatter_cell(order, (24, 24), org, dx, R, val)
    else:
        ref = O.scatter_edge(order, 0 if kind == "Ex" else 1, (24, 24), org, dx, R, val)
    assert same(got, ref)


def trajectories(n, seed, scale=(0.7, 1.3)):
    rng = np.random.default_rng(seed)
    oldR = rng.uniform(8, 20, (n, 2)) * np.array(scale)
    R = oldR + rng.uniform(-0.99, 0.99, (n, 2)) * np.array(scale)
    return oldR, R, rng.uniform(-1, 1, n)


@pytest.mark.parametrize("order", [0, 1, 2])
def test_current_and_charge_bitwise(gpu, order):
    dx, dt = (0.7, 1.3), 0.37
    box, org = (-6, -6, 40, 40), (0.0, 0.0)
    oldR, R, q = trajectories(3000, order + 3)
    for comp in (0, 1):
        got = SF.getCurrentDensity(order, comp, box, org, dx, dt, oldR, R, q)
        ref = O.deposit(order, comp, box, org, dx, dt, oldR, R, q)
        assert same(got, ref), "comp %d" % comp
    assert same(SF.getChargeDensity(order, box, org, dx, R, q), O.charge_density(order, box, org, dx, R, q))


@pytest.mark.parametrize("order", [0, 1, 2])
def test_charge_diff_continuity(gpu, order):
    dx, dt = (0.7, 1.3), 0.37
    box, org = (-6, -6, 40, 40), (0.0, 0.0)
    oldR, R, q = trajectories(3000, order + 17)
    diff = SF.getChargeDensity(order, box, org, dx, R, q, oldR=oldR)
    r1 = O.charge_density(order, box, org, dx, R, q)
    r0 = O.charge_density(order, box, org, dx, oldR, q)
    scale = np.abs(r1).max()
    assert np.abs(diff - (r1 - r0)).max() < 1e-13 * scale
    Jx = SF.getCurrentDensity(order, 0, box, org, dx, dt, oldR, R, q)
    Jy = SF.getCurrentDensity(order, 1, box, org, dx, dt, oldR, R, q)
    div = np.zeros_like(diff)
    div[:, 1:] += (Jx[:, 1:] - Jx[:, :-1]) / dx[0]
    div[1:, :] += (Jy[1:, :] - Jy[:-1, :]) / dx[1]
    assert np.abs(diff + dt * div).max() < 1e-12 * scale


@pytest.mark.parametrize("order", [0, 1, 2])
@pytest.mark.parametrize("n", [1, 63, 65, 20312, 20313, 60000])
def test_small_and_sorted_deposits_bitwise(gpu, order, n):
    """Particle counts around a wavefront and above, and runs of hundreds of
    contributions per node; the repeated call takes the first one's workspace."""
    dx, dt = (0.7, 1.3), 0.37
    box, org = (-6, -6, 40, 40), (0.0, 0.0)
    oldR, R, q = trajectories(n, order + n)
    for comp in (0, 1):
        ref = O.deposit(order, comp, box, org, dx, dt, oldR, R, q)
        for _ in range(2):
            assert same(SF.getCurrentDensity(order, comp, box, org, dx, dt, oldR, R, q), ref), "comp %d" % comp
    assert same(SF.getChargeDensity(order, box, org, dx, R, q), O.charge_density(order, box, org, dx, R, q))


@pytest.mark.parametrize("order", [0, 1, 2])
@pytest.mark.parametrize("n,nx,ny", [(8192, 40, 40), (8193, 40, 40), (1, 300, 298), (1, 300, 300)])
def test_deposits_at_the_node_scans_limits_bitwise(gpu, order, n, nx, ny):
    """Both sides of the lines between the node scan and the sorted deposit:
    32768 items (4 a trajectory), and the cost of the nodes themselves."""
    dx, dt = (0.7, 1.3), 0.37
    box, org = (-6, -6, nx, ny), (0.0, 0.0)
    oldR, R, q = trajectories(n, order + n)
    for comp in (0, 1):
        assert same(SF.getCurrentDensity(order, comp, box, org, dx, dt, oldR, R, q),
                    O.deposit(order, comp, box, org, dx, dt, oldR, R, q)), "comp %d" % comp


def test_few_particles_on_a_large_patch(gpu):
    """The time of one particle's charge on 4096 x 4096 nodes is that of the
    cleared patch, as a thousand particles' is (a wave per node took 40 times as
    long)."""
    n, side = 1024, 4096
    f = SF.DeviceArray(shape=(side * side,))
    R, Q = SF.DeviceArray(host=np.random.default_rng(3).uniform(8, 4000, (n, 2))), SF.DeviceArray(host=np.ones(n))

    def median(k):
        t = []
        for _ in range(15):
            t0 = time.perf_counter()
            check(gpu.csrst_sf_charge_density(C.c_int(1), f.ptr, C.c_int(0), C.c_int(0), C.c_int(side), C.c_int(side),
                                              SF._v2((0, 0)), SF._v2((1, 1)), R.ptr, Q.ptr, C.c_int(k), None))
            t.append(time.perf_counter() - t0)
        return sorted(t)[7]

    many = median(n)
    assert median(1) <= 2 * many


def test_patch_overflow_is_reported(gpu):
    oldR, R, q = trajectories(50, 1)
    with pytest.raises(CsrstError) as e:
        SF.getCurrentDensity(2, 0, (10, 10, 5, 5), (0.0, 0.0), (0.7, 1.3), 0.37, oldR, R, q)
    assert e.value.code == -4


GEOM = dict(lenBefore=0.05, lenAfter=0.01, width=0.0128, phiDeg=10.0, ekinMeV=50.59, bz=0.1704)


def stepper():
    cmd = Commands(numgridpx=1100, numgridpy=120, lengthbefore=GEOM["lenBefore"], length=GEOM["lenAfter"],
                   width=GEOM["width"], phi=GEOM["phiDeg"], Ekin=GEOM["ekinMeV"], Bz=GEOM["bz"], order=1,
                   statmodulus=1)
    return TwoGridStep(cmd)


def test_caller_geometry_and_stream(gpu):
    """The Bend's own mask and cells handed back through csrst_set_mask and
    csrst_set_boundary_cells, and the work moved to a caller stream, leave
    the steps bit-identical to the oracle; a changed cell list changes them."""
    from tests.test_twogrid_parity import compare
    R, P, Q = gaussian_bunch(1500, (0.046, 0.0064), 1e-3, 0.5e-3, 100.0, 1.0, seed=5)
    g = stepper()
    mask, ij, data = g.boundary_cells()
    g.set_mask(mask)
    g.set_boundary_cells(ij, data)
    stream = SF.Stream()
    g.set_stream(stream.handle)
    g.init_bunch(R, P, Q)
    o = O.Sim(1100, 120, order=1, statModulus=1, **GEOM)
    o.init(R, P, Q)
    for k in range(30):
        g.step(1)
        o.step(1)
    compare(g, o, "caller geometry, step 30")
    g.set_stream(None)
    g.step(1)
    o.step(1)
    compare(g, o, "own stream again")
    # cut cells given half their area: the fields at the walls change
    g2 = stepper()
    data2 = data.copy()
    data2[:, 2] *= 0.5
    g2.set_boundary_cells(ij, data2)
    g2.init_bunch(R, P, Q)
    g2.step(31)
    assert not same(g2.field("H"), g.field("H"))
    with pytest.raises(CsrstError):
        g2.set_mask(mask)                     # the geometry is fixed once the bunch is in
    g3 = stepper()
    bad = ij.copy()
    bad[0] = bad[1]
    with pytest.raises(CsrstError):
        g3.set_boundary_cells(bad, data)      # a cell listed twice
    stream.close()


def test_empty_bunch_and_one_node_patch(gpu):
    """No particles: the deposits and the charge density are zero on the
    patch, a scatter leaves the field as it was, a gather returns nothing.
    The smallest patch that holds an S0 (CIC) charge, the 2 x 2 vertices of
    its cell, gets the oracle's values."""
    org, dx, dt = (0.0, 0.0), (0.7, 1.3), 0.37
    none = np.zeros((0, 2))
    for order in (0, 1, 2):
        for comp in (0, 1):
            J = SF.getCurrentDensity(order, comp, (0, 0, 7, 5), org, dx, dt, none, none, np.zeros(0))
            assert J.shape == (5, 7) and not J.any()
        assert not SF.getChargeDensity(order, (0, 0, 7, 5), org, dx, none, np.zeros(0)).any()
        field = np.arange(35.0).reshape(5, 7)
        assert same(SF.scatter(order, "cell", (5, 7), org, dx, none, np.zeros(0), field=field), field)
        assert SF.gather(order, "Ex", field, org, dx, none).shape == (0,)
    R, q = np.array([[3.2 * dx[0], 2.1 * dx[1]]]), np.array([2.0])
    rho = SF.getChargeDensity(0, (3, 2, 2, 2), org, dx, R, q)
    assert rho.shape == (2, 2) and same(rho, O.charge_density(0, (3, 2, 2, 2), org, dx, R, q))
    with pytest.raises(CsrstError):
        SF.getChargeDensity(0, (3, 2, 1, 1), org, dx, R, q)      # the stencil leaves a 1 x 1 patch


def device_bytes(nbytes, fill):
    """A device block of `nbytes` bytes of value `fill` (no host copy)."""
    a = SF.DeviceArray(shape=(-(-nbytes // 8),))
    assert SF.hip().hipMemset(a.ptr, C.c_int(fill), C.c_size_t(nbytes)) == 0
    assert SF.hip().hipDeviceSynchronize() == 0
    return a


@pytest.mark.parametrize("order", [0, 2])
def test_gather_beyond_2_30_particles(gpu, order):
    """The coordinates of particle 2^30 and later lie past 2^31 doubles.  All
    particles sit at the origin but the last three, one cell further."""
    n = 2 ** 30 + 3
    R, out = device_bytes(16 * n, 0), device_bytes(8 * n, 0xff)
    last, head, tail = np.ones(6), np.empty(4), np.empty(8)
    field = SF.DeviceArray(host=np.arange(64.0))
    assert SF.hip().hipMemcpy(C.c_void_p(R.ptr.value + 16 * (n - 3)), last.ctypes.data_as(C.c_void_p), C.c_size_t(48), 1) == 0
    rc = gpu.csrst_sg_gather(C.c_int(order), C.c_int(0), C.c_int(2), field.ptr, C.c_int(8), C.c_int(8), SF._v2((-4.25, -4.25)),
                             SF._v2((1.0, 1.0)), R.ptr, C.c_int(n), out.ptr, None)
    check(rc)
    for a, at in ((head, 0), (tail, n - 8)):
        assert SF.hip().hipMemcpy(a.ctypes.data_as(C.c_void_p), C.c_void_p(out.ptr.value + 8 * at), C.c_size_t(a.nbytes), 2) == 0
    # splines reproduce a linear field: node (i, j) at (i + 1/2, j + 1/2) holds i + 8 j
    want = np.where(np.arange(12) < 9, 3.75 * 9, 4.75 * 9)
    assert np.abs(np.concatenate([head, tail]) - want).max() < 1e-13 * want.max()


def test_charge_on_a_patch_wider_than_2_28(gpu):
    """Columns past 2^28 = 268 435 456 of a patch of 3e8 x 2 nodes: the charge
    lands on its own nodes, and one past the last column is reported."""
    nx, ny, i0 = 300_000_000, 2, -1000
    f = device_bytes(8 * nx * ny, 0xff)
    R = SF.DeviceArray(host=np.array([[2.9e8 + 0.25 + i0, 0.5], [2.0e8 + 0.25 + i0, 0.5]]))
    Q = SF.DeviceArray(host=np.array([1.0, 2.0]))

    def node(i, j):
        v = np.empty(1)
        assert SF.hip().hipMemcpy(v.ctypes.data_as(C.c_void_p), C.c_void_p(f.ptr.value + 8 * (j * nx + i)), C.c_size_t(8), 2) == 0
        return v[0]

    def run():
        return gpu.csrst_sf_charge_density(C.c_int(0), f.ptr, C.c_int(i0), C.c_int(0), C.c_int(nx), C.c_int(ny), SF._v2((0, 0)),
                                           SF._v2((1, 1)), R.ptr, Q.ptr, C.c_int(2), None)

    check(run())
    for i, q in ((290_000_000, 1.0), (200_000_000, 2.0)):
        assert [node(i + a, j) for j in (0, 1) for a in (0, 1)] == [0.375 * q, 0.125 * q] * 2
    assert all(node(2 ** 28 + a, j) == 0 for j in (0, 1) for a in (-1, 0, 1))
    # the second node of the stencil is past the patch: dropped and reported
    R = SF.DeviceArray(host=np.array([[nx - 1 + 0.25 + i0, 0.5], [3.2e8, 0.5]]))
    assert run() == -4
    assert [node(nx - 1, j) for j in (0, 1)] == [0.375, 0.375] and node(0, 1) == 0 and node(2 ** 28, 0) == 0


def test_deposits_from_several_threads(gpu):
    """Four threads, each on a stream of its own, with counts on both sides of
    the sort: the shared workspaces never mix, bit for bit."""
    dx, dt = (0.7, 1.3), 0.37
    box, org = (-6, -6, 40, 40), (0.0, 0.0)
    jobs = [(order, trajectories(n, order + n)) for order in (0, 1, 2) for n in (300, 9000, 30000)]
    want = [O.deposit(order, 0, box, org, dx, dt, *t) for order, t in jobs]
    bad = []

    def work(first):
        st = SF.Stream()
        for r in range(3):
            for k in range(len(jobs)):
                k = (k * (first + 1) + r) % len(jobs)
                order, t = jobs[k]
                J, o, e, q = SF.DeviceArray(shape=box[2:]), *(SF.DeviceArray(host=a) for a in t)
                rc = gpu.csrst_sf_current_density(C.c_int(order), C.c_int(0), J.ptr, *(C.c_int(v) for v in box), SF._v2(org),
                                                  SF._v2(dx), C.c_double(dt), o.ptr, e.ptr, q.ptr, C.c_int(len(t[2])), st.h)
                if rc != 0 or not same(J.get(), want[k]):
                    bad.append((first, r, k))
        st.close()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert SF.hip().hipDeviceSynchronize() == 0
    assert SF.hip().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def sorted_deposit(n, comp=None):
    """A charge (comp None) or current deposit of n S2 particles on a patch
    large enough that it is sorted: 24 bytes of workspace a contribution, and
    the sort's own."""
    oldR = np.random.default_rng(n).uniform(6, 150, (n, 2))
    if comp is None:
        SF.getChargeDensity(2, (0, 0, 160, 160), (0.0, 0.0), (1.0, 1.0), oldR, np.ones(n))
    else:
        SF.getCurrentDensity(2, comp, (0, 0, 160, 160), (0.0, 0.0), (1.0, 1.0), 1.0, oldR, oldR + 0.25, np.ones(n))


def test_kept_workspaces(gpu):
    """Device memory that the deposits keep between calls: a request does not
    take a block many times its size (the particle counts of a current deposit
    would take the sort's, and the sort a second one), and a workspace beyond
    the bound of 512 MiB is freed without the blocks that are idle."""
    MiB = 2 ** 20
    for _ in range(70):                         # blocks of other calls age out
        sorted_deposit(30_000)
    before = free_bytes()
    sorted_deposit(600_000)                     # 230 MB and the sort's own
    one = free_bytes()
    assert 200 * MiB < before - one < 512 * MiB
    sorted_deposit(400_000, comp=0)             # 1.5 segments of 12 contributions each: 170 MB and the sort's own
    assert one - free_bytes() < 30 * MiB
    sorted_deposit(2_000_000)                   # 770 MB and the sort's own
    assert abs(one - free_bytes()) < 30 * MiB


def test_kept_workspaces_make_room(gpu):
    """On a card with 1 GiB left besides a kept workspace of some 450 MB, a
    window whose fields take 1.25 GiB still fits: the workspace is given back.
    A window that does not fit at all is refused, and the next call works."""
    sorted_deposit(800_000)
    hold = []
    try:
        while free_bytes() > 2 ** 30 + 2 ** 26 and len(hold) < 8:      # memory freed late shows up here
            hold.append(SF.DeviceArray(shape=((free_bytes() - 2 ** 30) // 8,)))
        assert 2 ** 30 - 2 ** 26 < free_bytes() < 2 ** 30 + 2 ** 26
        geom = dict(lenBefore=0.05, lenAfter=0.01, width=0.0128, phiDeg=10.0, ekinMeV=50.59, bz=0.1704)
        MovingWindowStep(4096, 3150, 1e-5, 1e-5, order=1, fp32=False, **geom).close()
        with pytest.raises(CsrstError) as e:
            MovingWindowStep(16384, 8192, 1e-5, 1e-5, order=1, fp32=False, **geom)
        assert e.value.code == -2
        sorted_deposit(30_000)
    finally:
        for h in hold:
            h.free()
