"""The operation counts agree with the tables that explain them."""
import re

from sedcol import flops


def test_linearly_implicit_attempt():
    table = flops.__doc__.split("Linearly implicit ROS2 attempt")[1]
    rows = [int(m) for m in re.findall(r"^  \S.*?\s{2,}(\d+)\b", table, re.M)]
    assert rows[-1] == sum(rows[:-1]) == flops.ROS2_ATTEMPT_PER_CELL
    # one Jacobian for both stages, one transport factor per class of species
    assert flops.KIN_JAC in rows and flops.CLASS_FACTORS in rows
