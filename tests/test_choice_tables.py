"""The attention launches' choices against measured times of every candidate
(profiles/*.csv): what the estimates cost over the fastest build, on average
and at worst.  Host arithmetic over stored figures: no GPU."""
import csv
import ctypes
from pathlib import Path

import pytest

from smooth_attn import _lib

PROFILES = Path(__file__).resolve().parents[1] / "profiles"


def _table(name):
    """[(B, Hq, Hkv, T, D, window), {candidate: us}] of one file."""
    with open(PROFILES / name) as f:
        rows = list(csv.DictReader(line for line in f if not line.startswith("#")))
    sizes = ("B", "Hq", "Hkv", "T", "D", "window")
    return [([int(r[c]) for c in sizes], {c: float(v) for c, v in r.items() if c not in sizes and v}) for r in rows]


def _over_fastest(costs):
    """Mean and worst of chosen / fastest."""
    return sum(costs) / len(costs), max(costs)


def _class(D):
    return 128 if D > 64 else 64 if D > 32 else 32


@pytest.mark.parametrize("cls,mean,worst,over_one", [(128, 1.006, 1.17, 1.1), (64, 1.006, 1.17, 1.18), (32, 1.011, 1.26, 1.1)])
def test_forward_key_split(cls, mean, worst, over_one):
    lib, cost, one = _lib.load(), [], []
    for shape, us in _table("attention_fwd_key_split_us.csv"):
        if _class(shape[4]) != cls:
            continue
        ks = lib.sa_flash_fwd_key_split(*shape, 0, 2 * shape[4])
        cost.append(us[f"ks{ks}"] / min(us.values()))
        one.append(us[f"ks{ks}"] / us["ks1"])
    assert len(cost) > 100
    got = _over_fastest(cost)
    assert got[0] <= mean and got[1] <= worst
    assert sum(one) / len(one) <= 0.85 and max(one) <= over_one  # against no split at all


@pytest.mark.parametrize("kind,cls,mean,worst", [
    ("kv", 128, 1.004, 1.06), ("kv", 64, 1.003, 1.05), ("dq", 128, 1.003, 1.06), ("dq", 64, 1.002, 1.02),
    ("exact", 128, 1.004, 1.04), ("exact", 64, 1.005, 1.08), ("exact", 32, 1.013, 1.11)])
def test_backward_plan(kind, cls, mean, worst):
    lib, cost, plan = _lib.load(), [], (ctypes.c_int * 3)()
    for shape, us in _table("attention_bwd_plan_us.csv"):
        exact = kind == "exact"
        us = {n: t for n, t in us.items() if n == "dq2" or n.startswith("x_") == exact}
        if _class(shape[4]) != cls or ("x_s1" if exact else "g1_s1") not in us:
            continue
        ws = lib.sa_flash_bwd_workspace_size(*shape, _lib.SA_BF16)
        assert lib.sa_flash_bwd_plan(*shape, exact, ws, plan) == 0
        dq2 = us.pop("dq2", None)
        if kind == "dq":
            if dq2 is not None:
                pair = (us["g1_s1"], dq2)
                cost.append(pair[plan[0] - 1] / min(pair))
            continue
        cost.append(us[f"x_s{plan[2]}" if exact else f"g{plan[1]}_s{plan[2]}"] / min(us.values()))
    assert len(cost) >= 15
    got = _over_fastest(cost)
    assert got[0] <= mean and got[1] <= worst
