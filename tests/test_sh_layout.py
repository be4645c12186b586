"""The layout of an SH simulation's radial lines by gauge and method."""
import pytest

from ionization_amd import engine


@pytest.mark.parametrize("n, layout", [(1000, (128, 8)), (1024, (128, 8)), (2000, (256, 8)), (4000, (256, 16)), (250, (64, 4))])
def test_length_gauge_takes_short_chains_on_short_lines(n, layout):
    assert engine.choose_sh_layout(n, "length", "sio") == layout


def test_everything_else_keeps_the_rule():
    for n in range(3, 8193, 7):
        rule = engine.choose_layout(n, "sh")
        assert engine.choose_sh_layout(n, "velocity", "sio") == rule
        assert engine.choose_sh_layout(n, "length", "adi") == rule
        P, m = engine.choose_sh_layout(n, "length", "sio")
        assert P * m == rule[0] * rule[1] and P <= 512  # the same padding
    assert engine.choose_sh_layout(1000, "length", "sio", rows=16) == (64, 16)  # forced rows win
    engine.set_sh_layout_table({1024: (64, 16)})
    try:
        assert engine.choose_sh_layout(1000, "length", "sio") == (64, 16)  # and so does a measured table
    finally:
        engine.set_sh_layout_table({})
