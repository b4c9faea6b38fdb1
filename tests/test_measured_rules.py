"""The rules that choose between the framework's products and the library, replayed over the measurements they rest on (profiles/): the tables'
picks are what the rules return, and no shape measured is slower than its alternative by more than the rules' docstrings say."""
import json
import math
import os

from chronos.ops import gemm as G

PROFILES = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "profiles")


def _table(name):
    with open(os.path.join(PROFILES, name)) as f:
        return json.load(f)


def _mean(ratios):
    return math.exp(sum(map(math.log, ratios)) / len(ratios))


def _slower(ratios):
    return sum(r < 1 / 1.03 for r in ratios)


def test_few_rows():
    table = _table("few_rows_gemm.json")
    for key, count, mean, slower, worst in (("rows", 885, 1.45, 2, 0.93), ("off the grid", 143, 1.23, 6, 0.87)):
        ratios = []
        for m, n, k, library, gemv, best, best_us, picked, us in table[key]:
            plan = G.few_rows_plan(m, n, k)
            assert (None if plan is None else "%d/%d" % plan) == picked, (m, n, k)
            if us is not None:
                ratios.append(min(library, gemv or library) / us)
        assert len(ratios) == count and _mean(ratios) >= mean and _slower(ratios) <= slower and min(ratios) >= worst


def test_few_rows_with_more_behind():
    table = _table("few_rows_gemm.json")["more behind"]
    taken = {"rows": [], "act": [], "glu": []}
    for kind, m, n, k, nf, plain, two, picked, *us in table["rows"]:
        rows = -(-(n + nf) // 32) * 32
        assert G._few_more(m, rows, k, {"rows": 0, "act": 1, "glu": 2}[kind]) == picked, (kind, m, n, k)
        if picked:
            taken[kind].append(two / us[picked - 12])
    for kind, count, mean in (("rows", 91, 1.53), ("act", 45, 1.39), ("glu", 24, 1.20)):
        assert len(taken[kind]) == count and _mean(taken[kind]) >= mean and min(taken[kind]) >= 0.94, kind
