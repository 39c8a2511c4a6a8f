"""The tuning options are process-wide: the fixture in conftest.py gives every one its
default again after each test, also after one that fails before its own reset."""
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CAPI = os.path.join(ROOT, "holographic-projector-simulations_amd", "csrc", "holo_capi.hip")
DEFAULTS = {}


def options():
    text = open(CAPI).read()
    body = text[text.index("long holo_get_option("):]
    return re.findall(r'n == "(\w+)"', body[:body.index("return -1;\n}")])


@pytest.mark.parametrize("value", [2, 1, 0])
def test_set_every_option(pkg, value):
    """(leaves them changed)"""
    names = options()
    assert {"grid_pairs", "splits", "mc_passes"} <= set(names)
    for n in names:
        now = pkg.get_option(n)
        assert DEFAULTS.setdefault(n, now) == now, n
        try:
            pkg.set_option(n, value)
        except pkg.HoloError:
            pass


def test_defaults_are_back(pkg):
    assert {n: pkg.get_option(n) for n in DEFAULTS} == DEFAULTS
