"""The series behind the 64-bin angle basis (csrc/moment_series.hpp, compiled for the host here) against the Gaussian itself
in 64 bits: the nodes of inference may not be further off than the nodes of training, neither at most nor on average."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SHIM = r"""
#include "moment_series.hpp"
using namespace cfh;
template <typename T> static void node(double u, T ws, double* c, double* eps) {
    const double step = (double)LEAN_NUM / LEAN_DEN, n = std::nearbyint(u / step);
    const double at = std::min(std::max(n, 0.0), LEAN_NODES - 1.0) * step;
    for (int m = 0; m < 64; m++) {
        T out[NORD];
        node_coefficients((T)(m - at) / ws, (T)(0.5 * step) / ws, out);
        for (int o = 0; o < NORD; o++) c[m * NORD + o] = out[o];
    }
    *eps = (u - at) / (0.5 * step);
}
extern "C" {
// coefficients (bin, o) of the training series around the bin nearest to u / of the inference series, and u's eps
void training(double u, double ws, double* c, double* eps) {
    const double node = std::min(std::max(std::nearbyint(u), 0.0), 63.0);
    for (int m = 0; m < 64; m++)
        for (int o = 0; o < NORD; o++) c[m * NORD + o] = moment_matrix<double>(o, m - node, ws);
    *eps = 2.0 * (u - node);
}
void inference(double u, double ws, double* c, double* eps) { node<double>(u, ws, c, eps); }
void inference32(double u, double ws, double* c, double* eps) { node<float>(u, (float)ws, c, eps); }
int terms() { return NORD; }
int words() { return 64 + 3 * NORD * LEAN_NODES; }
}
"""


@pytest.fixture(scope="module")
def series(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("series")
    (d / "shim.cpp").write_text("#include <algorithm>\n#include <cmath>\n" + SHIM)
    subprocess.run([cxx, "-O1", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "crystalframer_amd", "csrc"), "-o",
                    str(d / "shim.so"), str(d / "shim.cpp")], check=True)
    return ctypes.CDLL(str(d / "shim.so"))


def _errors(series, name, ws, points):
    f, n = getattr(series, name), series.terms()
    f.argtypes = [ctypes.c_double, ctypes.c_double, ctypes.c_void_p, ctypes.c_void_p]
    c, eps, m = np.zeros((64, n)), np.zeros(1), np.arange(64)
    diff = np.empty((len(points), 64))
    for i, u in enumerate(points):
        f(u, ws, c.ctypes.data, eps.ctypes.data)
        assert abs(eps[0]) <= 1.0 + 1e-12
        diff[i] = c @ eps[0] ** np.arange(n) - np.exp(-0.5 * ((m - u) / ws) ** 2)
    return np.abs(diff).max(), np.sqrt((diff ** 2).mean())


@pytest.mark.parametrize("ws", [3.0, 4.0, 6.0, 8.0])      # (the core takes the series from 3 bins on)
def test_inference_nodes_are_as_good_as_a_node_per_bin(series, ws):
    points = (np.arange(63 * 96) + 0.5) / 96
    # (the ends, and where two nodes meet)
    ends = np.concatenate([[0.0, 63.0]] + [t + s for t in (np.arange(63) + 0.5, 1.5 * np.arange(42) + 0.75) for s in (-1e-9, 1e-9)])
    top, rms = _errors(series, "training", ws, points)
    top = max(top, _errors(series, "training", ws, ends)[0])
    top_i, rms_i = _errors(series, "inference", ws, points)
    top_i = max(top_i, _errors(series, "inference", ws, ends)[0])
    assert top_i <= top and rms_i <= rms, (top_i / top, rms_i / rms)
    if ws == 4.0:       # the figures stated beside the series
        assert abs(top - 1.43e-6) < 1e-8 and abs(rms - 1.35e-7) < 1e-9
        assert abs(top_i - 1.22e-6) < 1e-8 and abs(rms_i - 1.31e-7) < 1e-9
    # the coefficients in 32 bits: each a sum of a few products below 1, a rounding of 6e-8 each
    top_f, rms_f = _errors(series, "inference32", ws, points)
    assert top_f <= top_i + 5e-7 and rms_f <= rms_i + 1e-7
    # the cosines that every frame has, 1, 0 and -1 (with |cos| 0 and 1): nodes, exact but for the rounding of a coefficient
    for u in (63.0, 31.5, 0.0):
        assert _errors(series, "inference", ws, [u])[0] < 1e-9 and _errors(series, "inference32", ws, [u])[0] < 2e-7
    assert series.words() <= 720
