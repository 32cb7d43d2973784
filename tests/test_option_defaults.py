"""The options that the shared engine is brought back to between tests are
those of a new engine, as the public header states them."""
import os
import re

from conftest import ROOT, option_defaults, restore_options


class _Recorder:
    def __init__(self):
        self.options = {}

    def set_option(self, name, value):
        self.options[name] = value
        return self


def test_defaults_are_the_documented_ones():
    with open(os.path.join(ROOT, "include", "ma", "ma.h")) as f:
        header = f.read()
    stated = {name.lower(): int(v) for name, v in
              re.findall(r"MA_OPT_(\w+) = \d+,?\s*/\*[^*]*default (\d+)\)", header)}
    defaults = option_defaults()
    got = {"local_rings": defaults["local_rings"], "walk_budget": defaults["walk_budget"],
           "amg_omega": defaults["amg_omega_permille"], "amg_corr": defaults["amg_corr_permille"],
           "amg_sweeps": defaults["amg_sweeps"]}
    assert stated == got
    assert defaults["graphs"] == 1 and defaults["far_cells"] == 1
    assert defaults["force_general"] == 0


def test_every_option_is_restored():
    with open(os.path.join(ROOT, "mongeampere_amd", "api.py")) as f:
        names = re.search(r"key = \{(.*?)\}\[name\]", f.read(), re.S).group(1)
    e = _Recorder()
    restore_options(e)
    assert set(re.findall(r'"(\w+)"', names)) == set(e.options)
