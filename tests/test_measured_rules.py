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
    for kind, count, mean in (("rows", 91, 1.53), ("act", 45, 1.39), ("glu", 29, 1.20)):
        assert len(taken[kind]) == count and _mean(taken[kind]) >= mean and min(taken[kind]) >= 0.90, kind


def test_mid_rows():
    table = _table("mid_rows_gemm.json")
    for least, most, count, mean, slower, worst in ((33, 64, 105, 1.21, 0, 0.97), (65, 128, 460, 1.28, 11, 0.91), (129, 256, 123, 1.21, 9, 0.91),
                                              (257, 512, 86, 1.10, 15, 0.91)):
        ratios = []
        for row in table["rows"]:
            m, n, k, library = row[:4]
            if least <= m <= most:
                plan = G.mid_rows_plan(m, n, k)
                assert "%d/%d" % plan == row[-1], (m, n, k)
                ratios.append(library / row[table["columns"].index(row[-1])])
        assert len(ratios) == count and _mean(ratios) >= mean and _slower(ratios) <= slower and min(ratios) >= worst
    assert all("%d/%d" % G.mid_rows_plan(*row[:3]) == row[-1] for row in table["beyond"])
    ratios = [row[3] / row[table["columns"].index(row[-1])] for row in table["beyond"]]
    assert len(ratios) == 58 and _mean(ratios) >= 1.28 and _slower(ratios) <= 5 and min(ratios) >= 0.92
    for m, n, k in ((32, 16384, 1024), (64, 153616, 1024), (100, 153616, 1024), (100, 1024, 32832), (256, 1024, 28736), (100, 151936, 4288), (129, 4112, 1024), (257, 2064, 1024), (512, 2048, 8256), (513, 1024, 1024), (100, 496, 1024), (100, 1024, 448), (64, 8192, 1024), (100, 1032, 1024), (100, 1024, 1056), (100, 6144, 4096)):
        assert G.mid_rows_plan(m, n, k) is None   # (the last: a shape that the measured plan lists)


def test_slab_rows():
    table = _table("slab_rows_gemm.json")
    ratios = []
    for row in table["rows"]:
        m, n, k, library, before, picked = *row[:4], *row[-2:]
        name = lambda p: None if p is None else "%d/%d" % p  # noqa: E731
        assert name(G.many_rows_plan(m, n, k)) == before and name(G.slab_rows_plan(m, n, k)) == picked, (m, n, k)
        if before != picked:
            of = lambda c: library if c is None else row[table["columns"].index(c)]  # noqa: E731
            ratios.append(of(before) / of(picked))
    assert len(ratios) == 122 and _mean(ratios) >= 1.18 and _slower(ratios) <= 1 and min(ratios) >= 0.89
    for m, n, k in ((256, 4096, 8192), (4128, 4096, 11008), (1100, 1008, 8192), (1100, 8208, 4096), (1100, 5120, 14336)):
        assert G.slab_rows_plan(m, n, k) == G.many_rows_plan(m, n, k)


def _rows(table):
    for row in table["rows"]:
        yield dict(zip(table["columns"], row))


def test_many_rows():
    table = _table("many_rows_gemm.json")
    for key, count, mean, slower, worst in (("unsplit", 302, 1.14, 25, 0.86), ("off the grid", 166, 1.16, 16, 0.86), ("split", 51, 1.23, 1, 0.91)):
        ratios = []
        for r in _rows(table[key]):
            plan = G.many_rows_plan(r["m"], r["n"], r["k"]) if r["m"] >= G.MANY_MIN else None
            if plan is None or (key == "split") != (plan[1] > 1) and key != "off the grid":
                continue
            us = r.get("%d,%d" % plan) if key != "off the grid" or plan[1] == 1 else r["88,split"] if r["split"] == plan[1] else None
            if us is not None:
                ratios.append(r["lib"] / us)
        assert len(ratios) == count and _mean(ratios) >= mean and _slower(ratios) <= slower and min(ratios) >= worst, key


def test_many_rows_with_an_activation():
    taken = {True: [], False: []}
    for r in _rows(_table("many_rows_gemm.json")["unsplit"]):
        m, n, k = r["m"], r["n"], r["k"]
        for glu, own, apart in ((True, "glu", "sepglu"), (False, "act", "sepact")):
            if m >= G.MANY_MIN and r[own] and G._many_act_pays(-(-m // 128) * 128, n, k, glu):
                plan = G.many_rows_plan(m, n, k)
                product = min(r["lib"], r["%d,1" % plan[0]] if plan and plan[1] == 1 else r["lib"])
                taken[glu].append((product + r[apart]) / r[own])
    for glu, count, mean, worst in ((True, 188, 1.11, 0.91), (False, 196, 1.14, 0.89)):
        assert len(taken[glu]) == count and _mean(taken[glu]) >= mean and min(taken[glu]) >= worst


def test_vocabulary_rows():
    tables = _table("vocabulary_rows_steps.json")
    for key, first in (("decode", 1), ("other contexts", 2)):
        for row in tables[key]["rows"]:
            us = dict(zip(tables[key]["columns"][first:], row[first:]))
            cfg, split = G.pp_plan(row[0], 128256, 4096, G.PP_PLAIN)
            assert split == 1 and us[str(cfg)] <= 1.015 * min(v for v in us.values() if v), row   # (captures of one config differ by 0.7 %)


def _linear(m, n, k):
    """The plan that linear() takes a plain product by."""
    return (G.few_rows_plan(m, n, k) if m <= 64 else G.slab_rows_plan(m, n, k) if m >= G.MANY_MIN else None) or (G.mid_rows_plan(m, n, k) if 32 < m <= 512 else None)


def test_the_tables_measured_again():
    for name, key, count, mean, slower, worst in (("few_rows_gemm.json", "weights read once", 1072, 1.43, 8, 0.89), ("many_rows_gemm.json", "by rows", 781, 1.15, 100, 0.81)):
        ratios, behind = [], []
        for r in _rows(_table(name)[key]):
            plan = _linear(r["m"], r["n"], r["k"])
            assert (None if plan is None else "%d/%d" % plan) == r["picked"], r
            if plan is not None:
                ratios.append(min(r.get("library", r.get("lib")), r.get("gemv") or math.inf) / r["us"])
                behind.append(r["us"] / r.get("best_us", r["us"]))
        assert len(ratios) == count and _mean(ratios) >= mean and _slower(ratios) <= slower and min(ratios) >= worst and _mean(behind) <= 1.021, name


def test_tiles_of_experts():
    import torch

    from chronos.ops import hybrid as hops

    hops.load()
    behind, before = [], []
    for r in _rows(_table("moe_tiles.json")):
        items, up = r["T"] * r["top"], r["F"] * (2 if r["form"] == "glu" else 1)
        tile = torch.ops.chronos.hy_moe_tile(items, r["E"], r["d"], r["F"], up)
        us = r[str(min(tile, 128))]   # (256 rows are another rule's, over 128)
        behind.append(min(r["32"], r["64"], r["128"]) / us)
        before.append(r["32" if items <= 16 * r["E"] else "128"] / us)
    assert len(behind) == 1428 and _mean(behind) >= 1 / 1.026 and min(behind) >= 1 / 1.42
    assert _mean(before) >= 1.08 and _slower(before) <= 27 and min(before) >= 1 / 1.23


def test_splits_of_windowed_decode_rows():
    """A key tile per split or two: the pick is no slower than the other by more than 3 %, and than ten splits with some workgroups on two tiles."""
    import torch

    from chronos.ops import hybrid as hops

    hops.load()
    picks = set()
    for H, G, window, keep, B, ctx, two, ten, one in _table("window_decode_splits.json")["rows"]:
        tiles = min(ctx, window + 1) // 64 + 1 + (keep > 0) if window else ctx // 64 + 1
        splits = torch.ops.chronos.hy_window_nsplit(B, 1, H, G, 128, 128, window, keep, ctx)
        wgs = B * G
        assert splits == max(1, min(-(-512 // wgs), 16, tiles if 4 <= tiles <= 16 else tiles // 2))
        picks.add((tiles, splits))
        us = one if 4 <= tiles <= 16 else two
        # (17 to 21 tiles: one that is left over costs two per split a round; sixteen splits gain there and lose from 17 on)
        assert us <= 1.035 * min(two, ten, one) or 16 < tiles <= 21, (H, G, window, B, ctx)
    assert len(picks) >= 12
    steps = _table("window_decode_splits.json")["steps"]["rows"]
    assert all((one < two) == (tokens > 60) for width, B, tokens, two, one in steps if width == "1k")


def _lines(key, pick, least):
    """Every measured pair of forms: what the rule picks is not slower than the other form by more than `least`."""
    for r in _rows(_table("decode_forms.json")[key]):
        a, b = list(r)[-2:]
        first = r[a] if pick(r) else r[b]
        assert first <= least * min(r[a], r[b]) or first - min(r[a], r[b]) <= 0.25, (key, r)   # (launches of 5 us scatter by a quarter)


def test_rows_of_decays_in_one_launch():
    from chronos.ops import hybrid as hops

    _lines("rows", lambda r: not hops.rows_step_pays(r["B"], r["H"], r["D"], r["Dv"], r["R"]), 1.18)


def test_router_in_one_launch():
    import torch

    from chronos.ops import hybrid as hops

    hops.load()
    _lines("router", lambda r: not torch.ops.chronos.hy_moe_route_one(r["T"], r["N"], r["d"]), 1.04)


def test_products_per_head():
    import torch

    from chronos.ops import hybrid as hops

    hops.load()
    _lines("head", lambda r: torch.ops.chronos.hy_head_few_rows(r["T"], r["N"], r["H"], r["K"]) == 0, 1.06)


def test_splits_of_latent_attention():
    import torch

    from chronos.ops import hybrid as hops

    hops.load()
    _lines("latent", lambda r: torch.ops.chronos.hy_latent_nsplit(r["B"] * -(-r["H"] // 64), 200, False, r["rank"]) == 1, 1.05)
