"""desc(): one filled layout per shape, strides and types, the address of the
tensor at hand; what it refuses it refuses every time."""
import pytest
import torch

from chatterbox_amdvulkan_amd import cbxops as C


def fields(d):
    return d.data, d.type, tuple(d.ne), tuple(d.nb)


@pytest.mark.parametrize("make", [
    lambda: torch.zeros(3, 5), lambda: torch.zeros(2, 3, 4, 5), lambda: torch.zeros(7), lambda: torch.zeros(6, 8).t(),
    lambda: torch.zeros(4, 8)[:, :3], lambda: torch.zeros(4, 1, 8).expand(4, 3, 8), lambda: torch.zeros(0, 4),
    lambda: torch.zeros(5, 4)[None], lambda: torch.zeros((), dtype=torch.float32), lambda: torch.zeros(3, 4).half(),
    lambda: torch.zeros(9, dtype=torch.int32)])
def test_layouts(make):
    a, b = make(), make()
    C._layouts.clear()
    first, again, other = fields(C.desc(a)), fields(C.desc(a)), fields(C.desc(b))
    assert first == again and first[1:] == other[1:]
    assert first[0] == (a.data_ptr() or None) and other[0] == (b.data_ptr() or None)
    d, e = C.desc(a), C.desc(b)
    e.ne[0] = 77                       # a caller's descriptor is its own
    assert fields(d) == first and fields(C.desc(b)) == other


def test_types_and_views_differ():
    x = torch.zeros(4, 68, dtype=torch.uint8)
    q = C.desc(x, C.Q8_0)
    assert q.type == C.Q8_0 and q.ne[0] == 64
    for _ in range(2):
        with pytest.raises(C.CbxError):
            C.desc(x)
        with pytest.raises(C.CbxError):
            C.desc(torch.zeros(4, 33, dtype=torch.uint8), C.Q8_0)
        with pytest.raises(C.CbxError):
            C.desc(torch.zeros(1, 1, 1, 1, 1))
    y = torch.zeros(8, 8)
    assert tuple(C.desc(y).nb) != tuple(C.desc(y[:, ::2]).nb)


def test_the_record_is_bounded():
    C._layouts.clear()
    for n in range(1, C._LAYOUTS_MAX + 10):
        C._layouts[n] = b""
        if len(C._layouts) >= C._LAYOUTS_MAX:
            break
    C.desc(torch.zeros(2, 2))
    assert len(C._layouts) <= C._LAYOUTS_MAX
    C._layouts.clear()
