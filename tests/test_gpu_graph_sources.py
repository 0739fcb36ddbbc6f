"""Replayed launch sequences (HIP graph) of plans with soft and hard data, of
Float64 images on either route and of slabs in global scratch, against runs
launched kernel by kernel."""
import numpy as np
import pytest

import iqhip
from test_gpu_graph import _res, _same
from test_gpu_simulate import _smooth

pytestmark = pytest.mark.gpu


def _args(case):
    rng = np.random.default_rng(91)
    if case in ("gather", "matrix"):
        T, aux_ti, aux = (_smooth(rng, n, 5, np.float32) for n in ((40, 38), (40, 38), (52, 50)))
        hard = {tuple(int(rng.integers(n)) for n in (52, 50)): float(rng.standard_normal()) for _ in range(8)}
        hard.update({(20 + i, 21 + j): 0.5 for i in range(6) for j in range(6)})  # tiles of few points and of many
        return T, (10, 9), (52, 50), dict(overlap=(0.25, 0.25), soft=[(aux, aux_ti)], hard=hard, nreal=2)
    if case in ("offset", "rounded"):
        T = _smooth(rng, (45, 44), 5, np.float64) + (1e4 if case == "offset" else 0.0)
        return T, (10, 11), (50, 55), dict(overlap=(0.25, 0.25), nreal=2, path="random")
    return _smooth(rng, (58, 55, 27), 5, np.float32), (40, 40, 20), (70, 72, 36), dict(overlap=(0.2, 0.1, 0.15))


@pytest.mark.parametrize("case", ["gather", "matrix", "offset", "rounded", "slabs"])
def test_replays_equal_host_launches(monkeypatch, case):
    T, tile, sim, kw = _args(case)
    if case in ("gather", "matrix"):
        monkeypatch.setenv("IQHIP_MAPS", case)
    print("graph replay", case, flush=True)
    plans = []
    for graph in ("0", "1"):
        monkeypatch.setenv("IQHIP_GRAPH", graph)
        plans.append(iqhip.make_plan(T, tile, sim, rng=np.random.default_rng(1), **kw)[0])
    eager, graph = plans
    us = [np.random.default_rng(k).random((kw.get("nreal", 1), eager.npath)) for k in range(2)]
    ref = []
    for u in us:
        eager.run(u)
        ref.append(_res(eager))
    for k in [0, 1, 0, 1]:  # capture, then replays, other work between them
        graph.run(us[k])
        _same(_res(graph), ref[k])
        eager.run(us[1 - k])
        _same(_res(eager), ref[1 - k])
    for p in plans:
        p.close()
