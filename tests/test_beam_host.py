"""Host-side beam bookkeeping on CPU tensors: a layer whose rows are not what
the move reads never reaches the library; the drain's periodic joining
keeps the order of the layers pushed (beam3d/beam_io.py:50-73, whose drain
appends every layer to its buffer as it arrives), and buffers rounded to a power of
two are ordinary contiguous tensors of the asked shape."""
import pytest

torch = pytest.importorskip('torch')

from lcodepy_amd.beam3d.beam_io import BeamDrain  # noqa: E402
from lcodepy_amd.beam3d.data import BeamParticles, empty_rounded  # noqa: E402


def _layer(first, n):
    f = torch.arange(first, first + n, dtype=torch.float64).repeat(9, 1)
    f[1] *= -1
    i = torch.arange(first, first + n, dtype=torch.int64).repeat(2, 1)
    return BeamParticles(f=f, i=i)


def test_drain_joins_in_push_order():
    drain = BeamDrain(None)
    sizes = [3, 0, 5, 1, 7] * 20          # 100 layers, empty ones among them
    first = 0
    for n in sizes:
        drain.push_beam_layer(_layer(first, n))
        first += n
        assert len(drain._layers) <= BeamDrain.JOIN_EVERY + 1
    out = drain.beam_slice()
    assert out.size == first == sum(sizes)
    assert torch.equal(out.id, torch.arange(first))
    assert torch.equal(out.x, -torch.arange(first, dtype=torch.float64))
    assert out.f.is_contiguous() and out.i.is_contiguous()


@pytest.mark.parametrize('shape', [(3, 0), (3, 1), (9, 5), (3, 9, 1000), (2, 7)])
def test_rounded_buffers(shape):
    t = empty_rounded(shape, torch.float64, 'cpu')
    n = 1
    for s in shape:
        n *= s
    assert tuple(t.shape) == shape and t.is_contiguous()
    cap = t.untyped_storage().nbytes() // 8
    assert cap >= n and (cap & (cap - 1)) == 0


def test_append_into_rounded_buffer_keeps_values():
    a = _layer(0, 6)
    a = BeamParticles(f=a.f[:, 1:4], i=a.i[:, 1:4])    # a strided column slice
    b = _layer(10, 2)
    a.append(b)
    assert a.size == 5
    assert torch.equal(a.id, torch.tensor([1, 2, 3, 10, 11]))
    assert a.f.is_contiguous()


class _Refuses:
    """A library whose entry points must not be called."""

    def __getattr__(self, name):
        def call(*args):
            raise AssertionError(f'{name} was called')
        return call


@pytest.mark.parametrize('float_rows,int_rows,ids,dtype,error', [
    (8, 2, 5, torch.float64, IndexError), (6, 2, 5, torch.float64, IndexError),
    (9, 1, 5, torch.float64, IndexError), (9, 2, 4, torch.float64, ValueError),
    (9, 2, 6, torch.float64, ValueError), (9, 2, 5, torch.float32, TypeError)])
@pytest.mark.parametrize('part', ['layer', 'fell'])
def test_advance_refuses_rows_it_would_read_past(monkeypatch, part, float_rows, int_rows, ids,
                                                 dtype, error):
    """A layer without all its rows (or with fewer or more ids than columns)
    raises what indexing the missing row raises, before any kernel gets its
    address (beam_calculator.py:97-143)."""
    from types import SimpleNamespace

    from lcodepy_amd import runtime
    from lcodepy_amd.beam3d import beam_calculator, move
    monkeypatch.setattr(torch.Tensor, 'is_cuda', property(lambda t: True))
    monkeypatch.setattr(runtime, 'device', lambda: torch.device('cpu'))
    monkeypatch.setattr(beam_calculator, 'stream_ptr', lambda: 0)
    ctx = SimpleNamespace(lib=_Refuses(), handle=None, check=None)
    monkeypatch.setattr(runtime, 'context', lambda config: ctx)
    calc = beam_calculator.BeamCalculator.__new__(beam_calculator.BeamCalculator)
    calc.ctx, calc.substep_energy, calc.time_step = ctx, 2.0, 1.0
    calc.move_particles = move.get_move_beam_particles(None)
    fields = SimpleNamespace(**{k: torch.zeros(3, 3, dtype=torch.float64)
                                for k in ('Ex', 'Ey', 'Ez', 'Bx', 'By', 'Bz')})
    wrong = BeamParticles(f=torch.zeros(float_rows, 5, dtype=dtype),
                          i=torch.zeros(int_rows, ids, dtype=torch.int64))
    none = BeamParticles(f=torch.zeros(9, 0, dtype=torch.float64),
                         i=torch.zeros(2, 0, dtype=torch.int64))
    layer, fell = (wrong, none) if part == 'layer' else (none, wrong)
    with pytest.raises(error):
        calc.advance_layer_async(layer, fell, 4, fields, fields)


def test_array_module_of_a_beam_can_be_set():
    """``xp`` is torch until something else is put there, as a class of a
    caller's may (beam3d/data.py:21-40)."""
    class Own(BeamParticles):
        def __init__(self, xp):
            super().__init__(f=torch.zeros(9, 2), i=torch.zeros(2, 2, dtype=torch.int64))
            self.xp = xp

    assert BeamParticles(f=torch.zeros(9, 1), i=torch.zeros(2, 1)).xp is torch
    marker = object()
    assert Own(marker).xp is marker
