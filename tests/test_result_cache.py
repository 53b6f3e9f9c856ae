"""``QuantizeResultCache`` is the dataclass of four optional tensors that the reference's callers construct
(quantized_grouped_linear.py:121-129, 467-470), also while it points into the stacked codes of all weights."""
import copy
import dataclasses
import pickle

import pytest
import torch

from atorch_amd.quantization import QuantizeResultCache, WeightCodeStack

NAMES = ["data", "scale", "data_t", "scale_t"]


def _stacked(n=3):
    caches = [QuantizeResultCache() for _ in range(n)]
    codes = tuple(torch.arange(n * 4, dtype=torch.float32).view(n, 4) + 10 * k for k in range(4))
    return caches, codes, WeightCodeStack(codes, caches)


def test_fields_defaults_and_repr():
    c = QuantizeResultCache()
    assert dataclasses.is_dataclass(c) and [f.name for f in dataclasses.fields(c)] == NAMES
    assert all(getattr(c, n) is None and f.default is None for n, f in zip(NAMES, dataclasses.fields(c)))
    assert repr(c) == "QuantizeResultCache(data=None, scale=None, data_t=None, scale_t=None)"
    t = [torch.full((2,), float(k)) for k in range(4)]
    c = QuantizeResultCache(t[0], t[1], scale_t=t[3])
    assert c.data is t[0] and c.scale is t[1] and c.data_t is None and c.scale_t is t[3]
    c.note = "kept"  # (an ordinary object)
    with pytest.raises(TypeError):
        hash(c)


def test_equality_and_replace():
    t = [torch.full((2,), float(k)) for k in range(4)]
    a = QuantizeResultCache(*t)
    assert a == QuantizeResultCache(*t) and a != QuantizeResultCache(*t[:3]) and QuantizeResultCache() == QuantizeResultCache()
    b = dataclasses.replace(a, data_t=None)
    assert b.data is t[0] and b.data_t is None and a.data_t is t[2]
    assert dataclasses.asdict(QuantizeResultCache()) == dict.fromkeys(NAMES)


def test_places_in_a_stack_read_write_and_copy_as_fields():
    caches, codes, stack = _stacked()
    assert stack.serves(caches)
    c = caches[1]
    assert all(torch.equal(getattr(c, n), codes[k][1]) for k, n in enumerate(NAMES))
    assert "data=tensor" in repr(c)
    other = dataclasses.replace(c, scale=None)
    assert other.scale is None and torch.equal(other.data, codes[0][1]) and stack.serves(caches)
    twins = copy.deepcopy(caches)
    assert twins[0].stack is twins[1].stack is not stack and twins[0].stack.serves(twins) and torch.equal(twins[2].data_t, c.stack.codes[2][2])
    back = pickle.loads(pickle.dumps(c))
    assert torch.equal(back.scale_t, c.scale_t)
    c.scale = torch.zeros(4)
    assert not stack.serves(caches) and c.stack is None and torch.equal(c.data, codes[0][1]) and torch.equal(c.scale, torch.zeros(4))


def test_codes_of_one_weight_from_a_stack_that_holds_one_orientation():
    """Dense, equally spaced and, for all weights together, one copy: what the operator interface runs in one launch."""
    from atorch_amd.quantization import _base_of_stack

    caches = [QuantizeResultCache() for _ in range(3)]
    data, scale = torch.arange(3 * 4 * 6).view(3, 4, 6), torch.arange(3 * 2 * 3.0).view(3, 2, 3)
    stack = WeightCodeStack((data, scale, data.transpose(1, 2), scale.transpose(1, 2)), caches)
    assert caches[0].holds("data_t") and stack.dense == [None] * 4  # (asking whether does not make it)
    for name, want in (("data", data), ("scale", scale), ("data_t", data.transpose(1, 2)), ("scale_t", scale.transpose(1, 2))):
        got = [getattr(c, name) for c in caches]
        assert all(torch.equal(g, w) and g.is_contiguous() for g, w in zip(got, want))
        assert _base_of_stack(got) == (got[0].data_ptr(), want[0].numel())
        assert len({g.untyped_storage().data_ptr() for g in got}) == 1
    assert stack.serves(caches) and caches[1].data.data_ptr() == data[1].data_ptr()  # the stored orientation is not copied


def test_replacing_fields_one_by_one_copies_nothing():
    caches = [QuantizeResultCache() for _ in range(2)]
    data = torch.arange(2 * 4 * 6).view(2, 4, 6)
    stack = WeightCodeStack((data, data[:, :1], data.transpose(1, 2), None), caches)
    for c in caches:
        c.data = c.scale = torch.zeros(1)
    assert not stack.serves(caches) and stack.dense == [None] * 4 and caches[0].scale_t is None
    assert torch.equal(caches[1].data_t, data[1].t())
    c = copy.deepcopy(caches[0])
    assert torch.equal(c.data_t, data[0].t()) and torch.equal(pickle.loads(pickle.dumps(caches[0])).data_t, data[0].t())
    c.data_t = c.scale_t = None
    assert c.data_t is None and not c.holds("scale_t") and not c.holds("data_t") and c.holds("data")
