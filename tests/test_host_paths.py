"""Host code of the library without a GPU: tests/cpp/host_paths.cpp stands in for the HIP runtime
and reports which kernels a call launches and what it allocates."""
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT

LIBDIR = os.path.join(ROOT, "moao_amd", "_lib")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host") / "host_paths")
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
           f"-I{ROOT}/include", f"-I{ROOT}/moao_amd/csrc",
           os.path.join(ROOT, "tests", "cpp", "host_paths.cpp"), "-o", exe, "-rdynamic",
           f"-L{LIBDIR}", "-lmoao_hip", f"-Wl,-rpath,{LIBDIR}", "-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def run(*args, **env):
        r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=300,
                           env={**os.environ, **{k: str(v) for k, v in env.items()}})
        assert r.returncode == 0, r.stdout + r.stderr
        return [line.split() for line in r.stdout.splitlines()]
    return run


def kernels(lines):
    """Kernels launched, each as (name, template arguments)."""
    names = [" ".join(w[1:-3]) for w in lines if w[0] == "launch"]
    return [(n.split("<")[0], n[n.index("<") + 1:-1].replace(" ", "").split(",") if "<" in n else [])
            for n in names]


# Largest leading dimensions whose lane offsets (up to 3 ld + 31 rows of A, 3 ld + 127 of op(B) =
# B^T) stay within 32 bits in bytes.
A_FIT = {"f64": (2 ** 32 // 8 - 1 - 31) // 3, "f32": (2 ** 32 // 4 - 1 - 31) // 3}
B_FIT = {"f64": (2 ** 32 // 8 - 1 - 127) // 3, "f32": (2 ** 32 // 4 - 1 - 127) // 3}


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("transb", [0, 1])
def test_direct_kernel_keeps_to_its_32_bit_offsets(host, prec, transb):
    """A small product runs on the direct kernel up to the leading dimensions that its 32-bit lane
    offsets reach, and on the slice kernel (64-bit column bases) past them."""
    def kernel(lda, ldb):
        return [k for k, _ in kernels(host("gemm", prec, transb, 20, 20, 5, lda, ldb))]
    assert kernel(20, 20) == ["gemm_direct_kernel"]
    assert kernel(A_FIT[prec], 20) == ["gemm_direct_kernel"]
    assert kernel(A_FIT[prec] + 1, 20) == ["gemm_dl_kernel"]
    assert kernel(2 ** 40, 20) == ["gemm_dl_kernel"]
    if transb == 1:
        assert kernel(20, B_FIT[prec]) == ["gemm_direct_kernel"]
        assert kernel(20, B_FIT[prec] + 1) == ["gemm_dl_kernel"]


def test_symmetric_operand_without_room_for_all_of_it(host):
    """The symmetric operand is written out in full where that scratch is to be had; else its diagonal
    blocks serve, and only without those does the product take the register-staged kernel."""
    K, full, blocks = 2000, 8 * 2000 * 2000, 8 * 128 * 2048
    for lim, want in ((full, ["expand_sym_kernel", "gemm_dl_kernel"]),
                      (full - 1, ["symdiag_kernel", "gemm_dl_kernel"]),
                      (blocks, ["symdiag_kernel", "gemm_dl_kernel"]),
                      (blocks - 1, ["gemm_kernel"])):
        out = host("gemm", "f64", 2, 3000, K, K, 3000, K, ASYNC_LIMIT=lim)
        got = kernels(out)
        assert [k for k, _ in got] == want, (lim, out)
        if lim < full and lim >= blocks:
            assert got[-1][1][:2] == ["double", "2"]
        assert out[-1] == ["rc", "0"]


def _words(lines, first):
    return [{w[k]: int(w[k + 1]) for k in range(len(w) % 2, len(w) - 1, 2)}
            for w in lines if w[0] == first]


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("n,m", [(700, 300), (1500, 448), (2000, 900)])
def test_mixed_solve_allocates_nothing_but_its_workspace(host, mode, n, m):
    """The workspace that mixed_workspace_bytes names is all that a mixed solve takes: its residuals
    run with the symmetric operand's diagonal blocks there, and with all of it in the larger
    workspace; the entry that makes its own asks for the larger one, then for the least."""
    out = host("mixed", n, m, mode)
    least, spare = (_words([out[0]], out[0][0])[0][k] for k in ("least", "spare"))
    assert spare == (max(0, 8 * n * n - 8 * 128 * -(-n // 128) * 128) if m >= 448 else 0)
    parts = [k for k, w in enumerate(out) if w[0] == "workspace"]
    asked = [w for w in out if w[0] == "async"]
    assert asked == [["async", str(least + spare), "given"]]
    assert out.index(asked[0]) > parts[1]
    names = [[k for k, _ in kernels(out[a:b])] for a, b in
             ((parts[0], parts[1]), (parts[1], out.index(asked[0])), (out.index(asked[0]), None))]
    full = "expand_sym_kernel" if spare else "symdiag_kernel"
    assert "symdiag_kernel" in names[0] and "gemm_kernel" not in names[0]
    assert full in names[1] and full in names[2]
    if spare:
        out = host("mixed", n, m, mode, ASYNC_LIMIT=least)
        assert [w[2] for w in out if w[0] == "async"] == ["refused", "given"]
        assert out[-1] == ["rc", "0"]
        out = host("mixed", n, m, mode, ASYNC_LIMIT=least - 1)
        assert out[-1] == ["rc", "-3"]


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_served_requests_hold_what_they_say(host, tmp_path, mode):
    """All device memory that the requests take from the pool is in their footprints and so in the
    budget; a mixed solve's spare bytes are given with a wide budget and not at the cost of another
    request's place, and a budget of one plain request still serves it."""
    from moao_amd import systems
    s, a = systems.make_system(str(tmp_path), systems.SystemSpec(diam=8.0, nssp=24, nlgs=2, nngs=1,
                                                                 nlayer=2, seed=3))
    def serve(slots, budget, requests):
        out = host("serve", s, a[0], mode, slots, budget, requests)
        assert all(w[:3] == ["request", "status", "0"] for w in out if w[0] == "request"), out
        return (_words(out, "request"), _words(out, "peak")[0],
                {w[1].split("<")[0] for w in out if w[0] == "launched"})
    req, mem, names = serve(1, 0, 1)
    assert req[0]["m"] >= 448  # rows from which the residuals use the whole operand
    assert mem["taken"] <= mem["peak"] == req[0]["footprint"]
    assert ("expand_sym_kernel" in names) == (mode != 0)
    wide = req[0]["footprint"]
    n = req[0]["n"]
    plain = wide - (8 * n * n - 8 * 128 * -(-n // 128) * 128 if mode else 0)
    for slots, budget in ((1, plain), (1, max(plain, wide - 1)), (2, 2 * plain),
                          (4, wide + 3 * plain - (1 if mode else 0))):
        req, mem, names = serve(slots, budget, 6)
        assert mem["taken"] <= mem["peak"] <= budget
        assert all(r["footprint"] in (plain, wide) for r in req)
        if slots < 4:
            assert all(r["footprint"] == plain for r in req)


def test_covariance_tables_of_a_request_are_in_its_block(host, tmp_path):
    """A slot keeps the upload of a request's system (subapertures' positions, noise and places: some
    120 bytes each here, and the structure function's table of 64 KB), not the covariance
    tables of its sensor pairs, which lie in the request's own block."""
    from moao_amd import systems
    s, a = systems.make_system(str(tmp_path), systems.SystemSpec(diam=8.0, nssp=24, nlgs=8, nngs=0,
                                                                 nlayer=2, seed=4))
    out = host("serve", s, a[0], 0, 1, 0, 2)
    req, mem = _words(out, "request"), _words(out, "peak")[0]
    tables = 36 * 3 * 8 * (2 * 24 - 1) ** 2  # 8 sensors' pairs, xx, yy and xy, 47 x 47 differences
    assert ["launched", "lattice_table"] in out and ["launched", "lattice_fill"] in out
    assert mem["kept"] <= 120 * req[0]["n"] // 2 * 9 // 8 + 70_000 + 16_384 < tables
    assert mem["taken"] <= mem["peak"] == req[0]["footprint"]


@pytest.mark.parametrize("field", ["X", "Y"])
@pytest.mark.parametrize("index", [0, 7])
def test_sensor_with_a_nan_position_is_no_grid(host, tmp_path, field, index):
    """A NaN among a sensor's positions takes the sensor out of the covariance tables, also where no
    layer's positions can show it (a sensor that sees no layer): its place on a grid would be an
    index without bounds."""
    from moao_amd import systems
    s, a = systems.make_system(str(tmp_path), systems.SystemSpec(diam=8.0, nssp=16, nlgs=3, nngs=0,
                                                                 nlayer=2, seed=3))
    unseen = ["sspSizeL", 0, 0.0, "sspSizeL", 1, 0.0]
    names = [k for k, _ in kernels(host("matcov", s, a[0], 1, *unseen))]
    assert names == ["lattice_table", "lattice_fill", "pair_kernel"]  # sensor 0 is a grid of its own
    tables = _grids(host("matcov", s, a[0], 1, *unseen))
    assert tables == 1 + 3  # sensor 0 with itself, sensors 1 and 2 with each other
    assert _grids(host("matcov", s, a[0], 1, *unseen, field, index, "nan")) == 3


def _grids(lines):
    """Sensor pairs with a covariance table."""
    return [int(w[-2]) for w in lines if w[:2] == ["launch", "lattice_table"]][0]


def test_plan_of_an_irregular_index_takes_little_more_than_its_lists(host):
    """A PSF plan of an index in random order lists its entries (4 bytes each); no list of
    single-entry runs (16 bytes each and more while it grows) is built on the way.  An index in order
    takes a run per row of actuators."""
    pairs = 30 ** 4
    out = host("plan", 30, 512, 1)
    assert out[-1] == ["rc", "0"]
    heap = _words(out, "plan")[0]["heap"]
    assert 4 * pairs <= heap <= 8 * pairs + 8 * 4 * 59 ** 2
    assert _words(host("plan", 30, 512, 0), "plan")[0]["heap"] <= 2 * pairs


def test_gpu_gemm_shapes_reach_their_kernels(host):
    """The shapes that tests/test_gpu_gemm.py gives to the 128-row tiles, to the direct kernel and to the
    slice kernels go there."""
    from test_gpu_gemm import RAGGED, RAGGED_ROWS, TILES_128
    for dtype, transb, M, N, K in TILES_128:
        p, t = ("f64", "double") if dtype == np.float64 else ("f32", "float")
        (name, args), = kernels(host("gemm", p, transb, M, N, K, M, N if transb else K))
        assert name == "gemm_dl_kernel" and args[:2] == [t, str(transb)] and args[3] == "128", \
            (dtype, transb, M, N, K, name, args)
    N, K = RAGGED
    for p in ("f64", "f32"):
        for transb in (0, 1):
            got = [kernels(host("gemm", p, transb, r, N, K, 66000, 200))[0] for r in RAGGED_ROWS]
            assert {k for k, _ in got[:-1]} == {"gemm_direct_kernel"}
            assert {a[2] for _, a in got[:-1]} == {"1", "2"}  # 16- and 32-row workgroups
            assert got[-1][0] == "gemm_dl_kernel"


def test_footprint_of_a_mixed_request_piece_by_piece(host, tmp_path):
    """Cmm, Ctm, the FP32 factor and right-hand sides with U^T, the leaves' inverses, residual and saved
    Ctm, the Woodbury terms, norms, range ids, status and ranges, and the symmetric operand's
    diagonal blocks: nothing for sums that find room in what is idle."""
    from moao_amd import systems
    s, a = systems.make_system(str(tmp_path), systems.SystemSpec(diam=8.0, nssp=12, nlgs=4, nngs=0,
                                                                 nlayer=2, seed=3))
    req = _words(host("serve", s, a[0], 1, 1, 0, 1), "request")[0]
    n, m, p = req["n"], req["m"], 8
    assert m < 448  # no larger workspace
    leaves = -(-n // 128)
    pieces = [8 * n * n, 8 * m * n, 4 * n * n, 4 * (m + p) * n, 4 * leaves * 128 * 128, 8 * m * n,
              8 * m * n, 8 * p * n, 8 * m * p, 8 * m * p, 8 * p * p, 8 * p * p, 8 * 1024, 4 * n, 16,
              4 * 2 * p, 8 * 128 * 128 * leaves]
    assert req["footprint"] == sum(-(-b // 256) * 256 for b in pieces)
