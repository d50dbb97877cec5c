"""Cofactors by minors (csrc/qmc_minors.h), compiled for the host.

The header has no device dependence, so the expansion the kernels inline is
checked on the CPU: cofactors of the first row against determinants of the
matrices with that row replaced by unit vectors, for every size it is used at,
on random matrices and on near-singular ones.
"""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qmctorch_amd", "csrc")
SRC = """
#define QMC_MINORS_FN inline
#include "qmc_minors.h"
template <int N, bool ACC>
static void go(const double* m, double* c, long n) {
    for (long i = 0; i < n; ++i, m += (N - 1) * N, c += N) {
        double R[N > 1 ? N - 1 : 1][N], o[N];
        for (int r = 0; r + 1 < N; ++r)
            for (int k = 0; k < N; ++k) R[r][k] = m[r * N + k];
        qmc::first_row_cofactors<N, ACC>(R, o);
        for (int k = 0; k < N; ++k) c[k] = o[k];
    }
}
#define CASE(N) case N: acc ? go<N, true>(m, c, n) : go<N, false>(m, c, n); break;
extern "C" void cofactors(int size, int acc, const double* m, double* c, long n) {
    switch (size) { CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("minors")
    (d / "m.cpp").write_text(SRC)
    subprocess.run([cxx, "-std=c++17", "-O1", "-fPIC", "-shared", "-I", CSRC, str(d / "m.cpp"), "-o", str(d / "m.so")],
                   check=True)
    return ctypes.CDLL(str(d / "m.so"))


@pytest.mark.parametrize("n", range(1, 8))
@pytest.mark.parametrize("acc", [0, 1])
def test_first_row_cofactors(lib, n, acc):
    rng = np.random.default_rng(n)
    mats = rng.standard_normal((200, n, n))
    if n > 2:  # two almost equal rows: cofactors far below the products they come from
        mats[100:, 2] = mats[100:, 1] * (1.0 + 1e-6 * rng.standard_normal((100, n)))
    low = np.ascontiguousarray(mats[:, 1:])
    out = np.empty((200, n))
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    lib.cofactors(n, acc, p(low), p(out), ctypes.c_long(200))
    for k in range(n):
        m = mats.copy()
        m[:, 0] = np.eye(n)[k]
        ref = np.linalg.det(m)
        # n! products of magnitude below the rows' norms, each rounded a few times
        bound = 50 * 2.3e-16 * np.prod(np.linalg.norm(mats[:, 1:], axis=2), axis=1)
        assert np.all(np.abs(out[:, k] - ref) <= bound)
