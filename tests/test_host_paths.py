"""Host code of the library without a GPU: tests/cpp/host_paths.cpp stands in for the HIP runtime
and reports which kernels a call launches and what it allocates."""
import os
import subprocess

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
