"""A captured graph whose steps read the map of repeated x planes, replayed after the potential table was
rewritten: the map has to describe the table that the replay finds."""

import pytest
import torch

from wavefunctionsimpython_amd import _abi

pytestmark = pytest.mark.gpu

DX, DT = (0.4, 0.35, 0.3), 0.01
STEPS = 3
# the slab scheme, square complex64 planes, planes of unequal sides, complex128 planes
GRIDS = [((32, 128, 128), _abi.WFS_C64, "yz_slab"), ((16, 96, 96), _abi.WFS_C64, "yz_split"),
         ((32, 64, 96), _abi.WFS_C64, "yz_split"), ((16, 64, 64), _abi.WFS_C128, "yz_split")]


def _potentials(shape, dev):
    """One plane repeated along x, and two potentials without equal planes."""
    g = torch.Generator(device=dev).manual_seed(shape[0] + shape[2])
    V = [torch.rand(shape, device=dev, generator=g) - 0.5 - 0.05j * torch.rand(shape, device=dev, generator=g)
         for _ in range(3)]
    V[0][:] = V[0][:1].clone()
    return [v.to(torch.complex64).contiguous() for v in V]


def _plan(shape, precision):
    return _abi.Plan(shape, DX, DT, 1.0, precision, _abi.WFS_METHOD_FOURIER)


def _rewrite(p, kind, route, other, V):
    """Makes V the plan's potential by the given route; graphs made on the way are returned."""
    box = [((0, 0, 0), p.n)]
    if route == "step":
        p.step(other, V, 2)
    elif route == "step_observe":
        p.step_observe(other, V, 2, 2, box)
    elif route == "set":
        p.set_potential(V)
    elif route == "sharing off":
        p.set_variant("pv_planes", 0)
        p.set_potential(V)
    elif route == "sharing off, reordered":
        on = p.variants()[kind]
        p.set_variant("pv_planes", 0)
        p.set_variant(kind, 0)
        p.set_potential(V)
        p.set_variant(kind, on)
        p.step(other, None, 1)
    else:
        s = torch.cuda.Stream()
        torch.cuda.synchronize()
        with _abi.Graph(s) as g:
            p.step(other, V, 2, stream=s)
        g.launch()
        s.synchronize()
        if route == "set after a captured one":
            p.set_potential(V)
        return [g]
    return []


ROUTES = ["step", "step_observe", "set", "sharing off", "sharing off, reordered", "captured",
          "set after a captured one"]


@pytest.mark.parametrize("route", ROUTES)
@pytest.mark.parametrize("shape,precision,kind", GRIDS)
def test_replay_reads_the_current_tables_map(dev, shape, precision, kind, route):
    V = _potentials(shape, dev)
    g = torch.Generator(device=dev).manual_seed(1)
    start = torch.randn(shape, dtype=torch.complex128, device=dev, generator=g)
    start = start.to(torch.complex64 if precision == _abi.WFS_C64 else torch.complex128)
    p = _plan(shape, precision)
    assert p.variants()[kind] and p.variants()["pv_planes"] == 1
    p.set_potential(V[0])
    psi, other = start.clone(), start.clone()
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with _abi.Graph(s) as graph:
        p.step(psi, None, STEPS, stream=s)
    own = _plan(shape, precision)                      # every plane's own copy, never a map
    own.set_variant("pv_planes", 0)
    keep, held = [], V[0]
    for replay, nxt in enumerate((V[0], V[1], V[2], V[0])):
        if replay:
            torch.cuda.synchronize()
            # the graph replayed inside the captured routes brings its own potential
            keep += _rewrite(p, kind, route if nxt is not V[0] else "set", other, nxt)
            held = nxt
            torch.cuda.synchronize()
        psi.copy_(start)
        torch.cuda.synchronize()
        graph.launch()
        s.synchronize()
        own.set_potential(held)
        own.set_step_index(0)                          # a replay uses the table copies of its capture
        want = start.clone()
        own.step(want, None, STEPS)
        torch.cuda.synchronize()
        assert torch.equal(psi, want), f"replay {replay}"
        p.step(other, None, 1)                         # eager work between the replays
    # eager calls after the replays read the last potential
    p.set_step_index(0)
    eager = start.clone()
    p.step(eager, None, STEPS)
    torch.cuda.synchronize()
    assert torch.equal(eager, want)
