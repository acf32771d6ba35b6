"""Stage calls and transforms replayed from HIP graphs: what a plan knows of its
grid must follow the replays, which run without the plan being called. (A graph
belongs to the points it was captured with; the points change only between.)

Type 2 forms only the rows its points read, so a replay leaves the grid partly
formed, and later calls must find that out. Every replay is compared with the
eager calls on a plan that forms every row.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_grid_state import BOUND, SHAPES, Inputs, rel
from test_gpu_stages import d2h

pytestmark = pytest.mark.gpu

NP = np.complex64


def _captured(stream, call):
    """A graph of call() on the plan's stream, after an eager run of it."""
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        call()
    return g


def _replay(g, stream):
    with torch.cuda.stream(stream):
        g.replay()
    torch.cuda.synchronize()


def _plan(v):
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        return stream, v.plan(v.dx, stream=stream)


def _cells(p):
    return int(np.prod(p.info()["grid"]))


@pytest.mark.parametrize("modes", SHAPES)
@pytest.mark.parametrize("asked", ["before", "after"])
def test_captured_type_2_and_the_grid(modes, asked):
    """Once a plan has been asked for its grid, type 2 forms every row, also in
    graphs captured before."""
    v = Inputs(modes)
    stream, p = _plan(v)
    out, buf = v.out(), v.df.clone()
    p.transform_type_2(buf, None, out)
    if asked == "before":
        ptr = p.fine_grid_ptr()
    g = _captured(stream, lambda: p.transform_type_2(buf, None, out))
    if asked == "after":
        ptr = p.fine_grid_ptr()
    for k in range(3):
        buf.copy_(v.df * (k + 1) if k != 1 else v.df2)
        torch.cuda.synchronize()
        _replay(g, stream)
        whole = v.whole_grid(buf)
        assert rel(d2h(ptr, _cells(p), NP), whole) < 1e-6, k
        # eager calls between the replays
        p.transform_type_2(v.df2, None, v.out())
        torch.cuda.synchronize()
        assert rel(d2h(ptr, _cells(p), NP), v.whole_grid(v.df2)) < 1e-6, k


@pytest.mark.parametrize("modes", SHAPES)
def test_replayed_type_2_then_other_points(modes):
    """interp() after a replay of type 2 that followed an eager spread()."""
    v = Inputs(modes)
    stream, p = _plan(v)
    out, buf = v.out(), v.df.clone()
    v.stale(p)
    p.transform_type_2(buf, None, out)
    g = _captured(stream, lambda: p.transform_type_2(buf, None, out))
    for f, df in ((v.f2, v.df2), (v.f, v.df)):
        p.set_points(v.m, v.dx)
        p.spread(v.dc)
        buf.copy_(df)
        torch.cuda.synchronize()
        _replay(g, stream)
        p.set_points(v.m, v.dy)
        other = v.out()
        p.interp(other)
        torch.cuda.synchronize()
        assert rel(other.cpu().numpy(), v.at_y(f)) < BOUND


@pytest.mark.parametrize("modes", SHAPES)
def test_captured_interp(modes):
    """A captured interp() reads the grid of the last call before each replay:
    an eager spread(), or an eager type 2 that left rows out."""
    v = Inputs(modes)
    stream, p = _plan(v)
    out = v.out()
    p.transform_type_2(v.df, None, out)
    p.set_points(v.m, v.dy)  # rows of these points are missing while capturing
    g = _captured(stream, lambda: p.interp(out))
    ref = v.plan(v.dy)
    want = v.out()
    ref.spread(v.dc)
    ref.interp(want)
    for _ in range(2):
        p.spread(v.dc)
        torch.cuda.synchronize()
        _replay(g, stream)
        assert rel(out.cpu().numpy(), want.cpu().numpy()) < 1e-6
        p.set_points(v.m, v.dx)
        p.transform_type_2(v.df2, None, v.out())
        p.set_points(v.m, v.dy)
        torch.cuda.synchronize()
        _replay(g, stream)
        assert rel(out.cpu().numpy(), v.at_y(v.f2)) < BOUND


@pytest.mark.parametrize("modes", SHAPES)
def test_captured_spread(modes):
    """A captured spread() overwrites, and a captured accumulating one adds to,
    whatever the grid holds at the replay."""
    v = Inputs(modes)
    stream, p = _plan(v)
    p.transform_type_2(v.df, None, v.out())
    over = _captured(stream, lambda: p.spread(v.dc))
    add = _captured(stream, lambda: p.spread(v.dc, accumulate=True))
    ref = v.plan(v.dx)
    ref.spread(v.dc)
    sums = d2h(ref.fine_grid_ptr(), _cells(ref), NP).astype(np.complex128)
    ref.spread(v.dc)
    at_y, want = v.out(), v.out()
    for _ in range(2):
        # type 2 leaves rows out, the replay overwrites the whole grid
        p.set_points(v.m, v.dx)
        p.transform_type_2(v.df2, None, v.out())
        torch.cuda.synchronize()
        _replay(over, stream)
        p.set_points(v.m, v.dy)
        p.interp(at_y)
        ref.set_points(v.m, v.dy)
        ref.interp(want)
        torch.cuda.synchronize()
        scale = np.linalg.norm(sums) / np.sqrt(sums.size) * np.sqrt(v.m)
        assert np.linalg.norm((at_y - want).cpu().numpy()) < 1e-6 * scale
        # type 2 leaves rows out, two replays add to all of them
        p.set_points(v.m, v.dx)
        p.transform_type_2(v.df2, None, v.out())
        torch.cuda.synchronize()
        _replay(add, stream)
        _replay(add, stream)
        p.set_points(v.m, v.dy)
        p.interp(at_y)
        torch.cuda.synchronize()
        grid = v.whole_grid(v.df2).astype(np.complex128) + 2 * sums
        got = d2h(p.fine_grid_ptr(), _cells(p), NP)
        assert rel(got, grid) < 1e-6
