"""Transfers of several engines at once, in threads of their own: the pinned
rings that they hand on are never shared, and engines made one after the other
get their particles whole."""
from __future__ import annotations

import threading

import numpy as np
import pytest

from sphcode_amd import ics

pytestmark = pytest.mark.gpu


def _round_trips(n, rounds, errors):
    from sphcode_amd import GPUEngine
    try:
        p, _ = ics.rollout(4)
        rng = np.random.default_rng(n)
        with GPUEngine(p) as g:
            for _ in range(rounds):
                f = dict(pos=rng.random((n, 3)), vel=rng.random((n, 3)), mass=rng.random(n), ene=rng.random(n))
                g.upload(f)
                g.make_tree()
                out = g.download(tuple(f))
                for k in f:
                    np.testing.assert_array_equal(out[k], f[k], err_msg=k)
    except BaseException as e:  # noqa: BLE001 (to the test's own thread)
        errors.append(e)


def test_engines_in_threads(gpu):
    errors: list = []
    threads = [threading.Thread(target=_round_trips, args=(n, 3, errors)) for n in (1000, 50_003, 200_000, 300_007)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


def test_engines_one_after_the_other(gpu):
    errors: list = []
    for n in (5, 120_000, 700, 400_001, 64):
        _round_trips(n, 2, errors)
    assert not errors, errors
