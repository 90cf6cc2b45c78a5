"""The host's choice of a march (csrc/march_choice.h), compiled by itself: the share of rays that
hit against the oracle's intersections of the same rays, and a choice that never goes back and
forth with the quarters hit or the windows needed (a graph captures the ends of both)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle
from spimagine_amd.utils import mat4_ortho, mat4_perspective, mat4_rotation, mat4_translate
from spimagine_amd.volumerender.volumerender import render_matrices

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "spimagine_amd", "csrc")
PROGRAM = r"""
#include "march_choice.h"
extern "C" float share(const float* p, const float* m, const float* box) { return spr::hit_share(p, m, box); }
extern "C" int pays(int nearest, int batch, float need, int nmax, float step, float hits) {
    return spr::windows_pay(nearest != 0, batch != 0, need, nmax, step, hits);
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    at = tmp_path_factory.mktemp("choice")
    (at / "choice.cpp").write_text(PROGRAM)
    so = str(at / "choice.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, "-o", so,
                           str(at / "choice.cpp")])
    f = ctypes.CDLL(so)
    f.share.restype = ctypes.c_float
    f.pays.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_float, ctypes.c_int, ctypes.c_float, ctypes.c_float]
    return f


BOXES = [(-1, 1, -1, 1, -1, 1), (-1, .2, -.5, 1, -1, 1), (.3, .4, -1, 1, -1, 1), (-3, 2, -1, 1, -1, 4)]
PROJECTIONS = [mat4_perspective(45, 1.7, .1, 10), mat4_perspective(110, .4, .1, 10),
               mat4_ortho(-2, 2, -1, 1, -10, 10)]


@pytest.mark.parametrize("box", BOXES)
@pytest.mark.parametrize("proj", range(len(PROJECTIONS)))
def test_share_is_that_of_the_reference_rays(lib, box, proj):
    # pixels 1, 3 ... 15 of a 16x16 frame are the 8x8 rays; one may graze the box
    vol = np.ones((4, 6, 5), np.float32)
    rng = np.random.default_rng(proj)
    seen = []
    for k in range(40):
        M = np.dot(mat4_translate(*rng.uniform(-.8, .8, 2), -rng.uniform(0., 6.)),
                   mat4_rotation(rng.uniform(0, 6.28), *rng.normal(size=3)))
        iP, iM = render_matrices(M, PROJECTIONS[proj], (5, 6, 4), (1., 1., rng.uniform(.5, 3.)))
        _, alpha = oracle.max_project(vol, iP, iM, box=box, max_steps=16, width=16, height=16)
        want = (alpha[1::2, 1::2] != -1.).sum()
        a = [np.ascontiguousarray(v, np.float32) for v in (iP, iM, box)]
        got = 64. * lib.share(*[ctypes.c_void_p(v.ctypes.data) for v in a])
        assert abs(got - want) <= 1., (k, got, want)
        seen.append(want)
    assert len(set(seen)) > 3


@pytest.mark.parametrize("nearest", [0, 1])
@pytest.mark.parametrize("batch", [0, 1])
def test_choice_goes_one_way(lib, nearest, batch):
    needs = [0., .1, .22, .24, .26, .28, .34, .36, .41, .45, .52, .56, .61, .69, .71, .89, .91, 1.]
    hits = [0., 499., 501., 699., 701., 999., 1001., 1499., 1501., 2999., 3001., 3999., 4001., 5999., 6001.,
            7999., 8001., 11999., 12001., 19999., 20001., 1e9]
    chosen = []
    for nmax in (1, 111, 159, 160, 189, 190, 223, 224, 319, 320, 2048):
        for step in (.1, .99, 1., 1.49, 1.5, 1.99, 2., 9.):
            at = np.array([[lib.pays(nearest, batch, n, nmax, step, h) for h in hits] for n in needs])
            assert (np.diff(at, axis=0) <= 0).all() and (np.diff(at, axis=1) <= 0).all(), (nmax, step)
            chosen.append(at.mean())
    assert 0 < np.mean(chosen) < 1
