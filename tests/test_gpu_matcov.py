"""GPU parity of the matcov generator against the oracle (oracle/matcov_oracle.c, which is
bit-identical to the hand-built reference on these fixtures).

Tolerance: the device pow/exp/sqrt may differ from the host libm in the last ulp; the 4-point
second differences of the structure function amplify that by |D|/|cov| (<= ~1e4 here), so
elements must agree to 1e-12 of the matrix's largest entry and the relative Frobenius error
must be <= 3e-13 (measured: 1.0e-13 on the nx456 2-layer Ctm).
"""
import numpy as np
import pytest

from conftest import FIXTURES, fixture_system
from moao_amd import matcov as gm
from moao_amd.tomo import Tomo
from oracle import matcov as om
from oracle.tomo import Tomo as OTomo

pytestmark = pytest.mark.gpu


def _pair(name):
    s, a = fixture_system(name)
    print(f"[matcov] system {name}", flush=True)
    return Tomo(s, a), OTomo.from_files(s, a)


def _close(g, o, rtol_el=1e-12, rtol_fro=3e-13):
    scale = np.max(np.abs(o))
    el = np.max(np.abs(g - o)) / scale
    fro = np.linalg.norm(g - o) / np.linalg.norm(o)
    assert el <= rtol_el, f"elementwise {el:.3e}"
    assert fro <= rtol_fro, f"frobenius {fro:.3e}"


@pytest.mark.parametrize("name", FIXTURES)
def test_cmm_ctm_ctt_match_oracle(name):
    t, o = _pair(name)
    n, m = t.nmeas(), t.nmeasts()
    # Cmm: lower triangle generated, strictly-upper part left as the caller had it
    sentinel = 7.25
    g = np.full((n, n), sentinel, order="F")
    gm.matcov_tile(g, n, n, 0, 0, n, t, gm.CMM)
    ref = np.full((n, n), sentinel, order="F")
    om.matcov_tile(ref, n, n, 0, 0, n, o, 1)
    assert np.all(g[np.triu_indices(n, 1)] == sentinel)
    _close(np.tril(g), np.tril(ref))
    t.set_target(0)
    o.set_target(0)
    _close(gm.ctm(t), om.ctm(o))
    _close(gm.ctt(t), om.ctt(o))


def test_offset_tiles_and_lda():
    t, o = _pair(FIXTURES[1])
    for (nr, nc, xo, yo, lda, typ) in [(100, 70, 37, 11, 128, 1), (64, 64, 300, 300, 64, 1),
                                       (33, 91, 5, 700, 40, 3), (152, 152, 0, 0, 152, 4),
                                       (17, 19, 100, 3, 17, 4)]:
        if typ == 3:
            t.set_target(0)
            o.set_target(0)
        buf = np.full(lda * nc, -1.0)
        gm.matcov_tile(buf, nr, nc, xo, yo, lda, t, typ)
        ref = np.full(lda * nc, -1.0)
        om.matcov_tile(ref, nr, nc, xo, yo, lda, o, typ)
        scale = np.max(np.abs(ref))
        assert np.max(np.abs(buf - ref)) <= 1e-12 * scale, (nr, nc, xo, yo, lda, typ)
        # entries outside the tile rows (lda padding) are untouched
        pad = buf.reshape(nc, lda)[:, nr:]
        assert np.all(pad == -1.0)


def test_bad_type_is_an_error():
    from moao_amd.lib import MoaoError
    t, _ = _pair(FIXTURES[0])
    buf = np.zeros((4, 4), order="F")
    with pytest.raises(MoaoError):
        gm.matcov_tile(buf, 4, 4, 0, 0, 4, t, 5)


def test_cmm_is_spd_and_symmetric_blocks():
    t, _ = _pair(FIXTURES[0])
    c = gm.cmm(t)
    full = np.tril(c) + np.tril(c, -1).T
    w = np.linalg.eigvalsh(full)
    assert w.min() > 0


def test_elt_workload_tiles(tmp_path):
    """The n = 18,688 system (40x40 subapertures, 6 LGS + 2 NGS, 10 layers: elongated LGS next to
    NGS, layers some WFS do not see): 256 x 256 tiles of Cmm (on and off the diagonal, the
    last rows and columns), Ctm and Ctt against the oracle.  As for the whole fixture matrices,
    elements must agree to 1e-12 of the matrix's largest entry (its diagonal: Cmm's own for Cmm,
    the truth sensor's Ctt for Ctm and Ctt).  A per-tile relative norm is not a meaningful bar
    away from the diagonal: the ulp-level device/libm differences of the structure function
    stay at ~1e-14 of the diagonal scale everywhere (measured), while far-apart WFS pairs have
    covariances 1e2-1e5 times smaller than that scale."""
    from moao_amd import systems
    s, a = systems.make_system(str(tmp_path), "elt")
    t, o = Tomo(s, a[0]), OTomo.from_files(s, a[0])
    n, m = t.nmeas(), t.nmeasts()
    print(f"[matcov] elt workload n={n} m={m}", flush=True)
    t.set_target(0)
    o.set_target(0)
    T = 256

    def tile(typ, xo, yo):
        buf = np.full((T, T), -1.0, order="F")
        gm.matcov_tile(buf, T, T, xo, yo, T, t, typ)
        ref = np.full((T, T), -1.0, order="F")
        om.matcov_tile(ref, T, T, xo, yo, T, o, typ)
        if typ == 1:  # only the lower part (row >= col) is generated
            keep = (np.arange(T)[:, None] + xo) >= (np.arange(T)[None, :] + yo)
            assert np.all(buf[~keep] == -1.0)
            buf, ref = np.where(keep, buf, 0.0), np.where(keep, ref, 0.0)
        return buf, ref

    scale = {1: np.max(np.abs(tile(1, 0, 0)[1]))}
    scale[3] = scale[4] = np.max(np.abs(tile(4, 0, 0)[1]))
    tiles = [(1, 0, 0), (1, 9000, 4000), (1, n - T, n - T), (1, 12000, 11900), (1, n - T, 0),
             (1, 3000, 2000), (3, 1000, 15000), (3, m - T, n - T), (4, 0, 0), (4, 2000, 1000)]
    for typ, xo, yo in tiles:
        g, r = tile(typ, xo, yo)
        err = np.max(np.abs(g - r)) / scale[typ]
        print(f"    type {typ} tile at ({xo}, {yo}): {err:.2e} of the diagonal scale", flush=True)
        assert err <= 1e-12


def test_whole_matrix_pair_kernel_is_bit_identical_to_element_tiles(tmp_path):
    """A whole Cmm or Ctm runs the pair kernel (one lane per subaperture pair, shared structure
    functions); any other tile runs the element kernel.  Both must give the same bits: the
    fixtures (LGS only, equal subaperture sizes per layer) and the n = 18,688 system (LGS and
    NGS: unequal sizes on the layers the LGS cone shrinks), column blocks of the whole matrix
    against the same columns generated as tiles at a column offset."""
    from moao_amd import systems
    s, a = systems.make_system(str(tmp_path), "elt")
    cases = [Tomo(*fixture_system(FIXTURES[0])), Tomo(*fixture_system(FIXTURES[1])), Tomo(s, a[0])]
    for t in cases:
        n, m = t.nmeas(), t.nmeasts()
        t.set_target(0)
        print(f"[matcov-pairs] n={n} m={m}", flush=True)
        C = gm.cmm(t)
        B = gm.ctm(t)
        W = 300
        for c0 in sorted({0, n // 3, n - W}):
            blk = np.full((n, W), -1.0, order="F")
            gm.matcov_tile(blk, n, W, 0, c0, n, t, gm.CMM)
            lower = np.arange(n)[:, None] >= np.arange(c0, c0 + W)[None, :]
            assert np.array_equal(blk[lower], C[:, c0:c0 + W][lower]), (n, "Cmm", c0)
            bb = np.empty((m, W), order="F")
            gm.matcov_tile(bb, m, W, 0, c0, m, t, gm.CTM)
            assert np.array_equal(bb, B[:, c0:c0 + W]), (n, "Ctm", c0)


@pytest.mark.parametrize("L0", [0.3, 2.0, 10.66, 25.0, 400.0, 1e5])
def test_structure_function_range(tmp_path, L0):
    """Outer scales that take the structure function's arguments q = 2 pi r / L0 through the whole
    range of its table and past both ends (q < 1/32, q > 45), and near the border of its two
    branches (r = 3/4 L0: 8 m for L0 = 10.66): Cmm, Ctm and Ctt within 1e-12 of the largest entry
    of the oracle's, as for the fixtures (second differences amplify the last-ulp differences)."""
    from moao_amd import systems
    spec = systems.SystemSpec(diam=8.0, nssp=9, nlgs=2, nngs=1, nlayer=3, L0=L0, seed=77)
    s, a = systems.make_system(str(tmp_path), spec)
    t, o = Tomo(s, a[0]), OTomo.from_files(s, a[0])
    t.set_target(0)
    o.set_target(0)
    for g, r in ((np.tril(gm.cmm(t)), np.tril(om.cmm(o))), (gm.ctm(t), om.ctm(o)),
                 (gm.ctt(t), om.ctt(o))):
        err = np.max(np.abs(g - r)) / np.max(np.abs(r))
        print(f"[matcov-range] L0={L0} {g.shape}: {err:.2e}", flush=True)
        assert err <= 1e-12


def _edit(path, field, values):
    """Replace the values line that follows the field's name in a parameter file."""
    lines = open(path).read().split("\n")
    k = lines.index(field)
    lines[k + 1] = " ".join(repr(v) for v in values)
    open(path, "w").write("\n".join(lines))


@pytest.mark.parametrize("field,value", [(None, 0.0), ("thetaML", 7.0), ("XPup", 0.37),
                                         ("thetaCam", 5.0)])
def test_grids_and_free_sensors(tmp_path, field, value):
    """Sensors on one regular grid read their covariances from tables of the grid's differences,
    others (here one LGS rotated or shifted in the pupil; LGS against NGS on the layers the cone
    shrinks) are evaluated pair by pair: Cmm, Ctm and Cmaa against the oracle, and tiles of every
    size, small ones evaluated without a table, against the whole matrices bit for bit."""
    from moao_amd import systems
    spec = systems.SystemSpec(diam=8.0, nssp=12, nlgs=3, nngs=2, nlayer=4, seed=19)
    s, a = systems.make_system(str(tmp_path), spec)
    if field:
        _edit(s, field, [0.0, value, 0.0, 0.0, 0.0, 0.0])
    t, o = Tomo(s, a[0]), OTomo.from_files(s, a[0])
    t.set_target(0)
    o.set_target(0)
    n, m = t.nmeas(), t.nmeasts()
    print(f"[matcov-grids] {field} n={n} m={m}", flush=True)
    C, B = gm.cmm(t), gm.ctm(t)
    _close(np.tril(C), np.tril(om.cmm(o)))
    assert np.max(np.abs(B - om.ctm(o))) <= 1e-12 * np.max(np.abs(om.ctt(o)))
    for nr, nc, xo, yo in [(n, 7, 0, 0), (9, 11, n - 9, 3), (40, 40, n // 2, n // 3),
                           (130, 70, n - 130, n // 2), (1, 1, n - 1, 0), (250, 333, 411, 290)]:
        buf = np.full((nr, nc), -1.0, order="F")
        gm.matcov_tile(buf, nr, nc, xo, yo, nr, t, gm.CMM)
        low = np.arange(xo, xo + nr)[:, None] >= np.arange(yo, yo + nc)[None, :]
        assert np.array_equal(buf[low], C[xo:xo + nr, yo:yo + nc][low]), (nr, nc, xo, yo)
        assert np.all(buf[~low] == -1.0)
        nr = min(nr, m)
        xo = min(xo, m - nr)
        buf = np.empty((nr, nc), order="F")
        gm.matcov_tile(buf, nr, nc, xo, yo, nr, t, gm.CTM)
        assert np.array_equal(buf, B[xo:xo + nr, yo:yo + nc]), ("Ctm", nr, nc, xo, yo)
    g, r = np.empty((n, m), order="F"), np.empty((n, m), order="F")
    gm.matcov_tile(g, n, m, 0, 0, n, t, gm.CMAA)
    om.matcov_tile(r, n, m, 0, 0, n, o, 2)
    assert np.max(np.abs(g - r)) <= 1e-12 * np.max(np.abs(om.ctt(o)))


@pytest.mark.parametrize("xo,yo", [(0, 90), (10, 90), (49, 89), (50, 89), (51, 89)])
def test_cmm_tiles_at_and_above_the_diagonal(tmp_path, xo, yo):
    """A 40 x 30 tile of Cmm wholly above the diagonal writes nothing; one that touches it with its
    last row writes what lies on or below it."""
    from moao_amd import systems
    s, a = systems.make_system(str(tmp_path), systems.SystemSpec(diam=8.0, nssp=8, nlgs=2, nngs=1,
                                                                 nlayer=2, seed=5))
    t = Tomo(s, a[0])
    t.set_target(0)
    C = gm.cmm(t)
    buf = np.full((40, 30), -1.0, order="F")
    gm.matcov_tile(buf, 40, 30, xo, yo, 40, t, gm.CMM)
    low = np.arange(xo, xo + 40)[:, None] >= np.arange(yo, yo + 30)[None, :]
    assert np.array_equal(buf[low], C[xo:xo + 40, yo:yo + 30][low])
    assert np.all(buf[~low] == -1.0)


def _poke(t, field, index, value):
    """Overwrites one value of the library's model (the view points into it)."""
    getattr(t.view(), field)[index] = value


@pytest.mark.parametrize("field,value", [("u", np.inf), ("v", -np.inf), ("u", np.nan), ("u", 1e200),
                                         ("L0", 0.0), ("L0", 1e-160)])
def test_separations_out_of_range(tmp_path, field, value):
    """Infinite positions, positions whose square overflows and an outer scale of zero give NaN where
    the reference's formulas do, an outer scale whose inverse square overflows gives their values: Cmm,
    Ctm and a small tile (evaluated without covariance tables).  Finite elements within 1e-12 of
    Ctt's largest, as above (Ctt of the unchanged system)."""
    from moao_amd import systems
    s, a = systems.make_system(str(tmp_path), systems.SystemSpec(diam=8.0, nssp=8, nlgs=2, nngs=1,
                                                                 nlayer=2, seed=8))
    t, o = Tomo(s, a[0]), OTomo.from_files(s, a[0])
    t.set_target(0)
    o.set_target(0)
    scale = np.max(np.abs(om.ctt(o)))
    k = 0 if field == "L0" else 5
    _poke(t, field, k, value)
    (o.L0diff if field == "L0" else getattr(o, field).reshape(-1))[k] = value
    print(f"[matcov-inf] {field} = {value}", flush=True)
    for g, r in ((np.tril(gm.cmm(t)), np.tril(om.cmm(o))), (gm.ctm(t), om.ctm(o))):
        bad = ~np.isfinite(r)
        assert bad.any() == (value != 1e-160)
        assert np.array_equal(np.isnan(g), np.isnan(r))
        assert np.max(np.abs(g - r)[~bad], initial=0.0) <= 1e-12 * scale
    tile, whole = np.zeros((9, 7), order="F"), gm.ctm(t)
    gm.matcov_tile(tile, 9, 7, 0, 0, 9, t, gm.CTM)
    assert np.array_equal(tile, whole[:9, :7], equal_nan=True)
