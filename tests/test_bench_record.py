"""The benchmark's record and log name only settings that the library has: the row cost and row tile are
options accepted without effect, so they are neither applied nor reported."""
import ast
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_no_setting_without_effect_is_reported():
    with open(os.path.join(ROOT, "bench.py")) as f:
        tree = ast.parse(f.read())
    called = {n.attr for n in ast.walk(tree) if isinstance(n, ast.Attribute)}
    strings = {n.value for n in ast.walk(tree) if isinstance(n, ast.Constant) and isinstance(n.value, str)}
    keys = {k.value for n in ast.walk(tree) if isinstance(n, ast.Dict) for k in n.keys if isinstance(k, ast.Constant)}
    assert not called & {"set_row_cost", "set_row_tile", "autotune_rows", "row_cost", "row_tile"}
    assert not keys & {"row_cost", "row_tile"}
    assert not [s for s in strings if "row cost" in s or "row tile" in s]
    assert {"--row-cost", "--row-tile"} <= strings  # still accepted
