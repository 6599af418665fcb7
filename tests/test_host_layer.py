"""The packed-descriptor path of the int8 wrappers against make_desc and the library's shape rules
(no GPU): the same bytes and output shape for what it takes, and nothing it should refuse."""
import ctypes as C
import itertools

import pytest

import my_own_cnn_amd as M
from my_own_cnn_amd import conv


class Shaped:
    def __init__(self, *shape):
        self.shape = shape


def test_same_descriptor_and_shape_or_refused():
    taken = refused = 0
    for stride, padding, dilation, groups, k, hw in itertools.product((1, (2, 1), 0, -1), (0, 1, (0, 3), -2),
                                                                     (1, (1, 2), 0, -1), (1, 2, 3, 0, -1), (4, 6, 0),
                                                                     ((5, 7), (2, 2), (0, 3))):
        x, w = Shaped(2, *hw, 6), Shaped(k, 3, 2, 6)
        kw = dict(stride=stride, padding=padding, dilation=dilation, groups=groups, relu=True, in_scale=0.02,
                  out_scale=0.5, algo="igemm")
        desc = conv.make_desc(x.shape, w.shape, **kw)
        got = conv._plain_layer(x, w, stride, padding, dilation, groups, True, 0.02, 0.5, "igemm")
        try:
            ho, wo = M.infer_conv_shape(2, *hw, 6, 3, 2, k, desc.conv)
        except M.MiqError:
            assert got is None
            refused += 1
            continue
        assert got == (bytes(desc), (2, ho, wo, k))
        taken += 1
    assert taken > 100 and refused > 100


def test_values_a_descriptor_cannot_pack_take_the_other_path():
    x, w = Shaped(1, 8, 8, 4), Shaped(4, 3, 3, 4)
    assert conv._plain_layer(x, w, 1, 0, 1, 1, False, 1e39, 1.0, "auto") is None
    assert conv._plain_layer(x, w, 1, 2 ** 40, 1, 1, False, 1.0, 1.0, "auto") is None
    assert conv._plain_layer(x, w, 1, 0, 1, 1, False, "1", 1.0, "auto") is None
    with pytest.raises(KeyError):
        conv._plain_layer(x, w, 1, 0, 1, 1, False, 1.0, 1.0, "none")
    with pytest.raises(ValueError):
        conv._plain_layer(Shaped(1, 8, 8), w, 1, 0, 1, 1, False, 1.0, 1.0, "auto")
    assert C.sizeof(M.QConvDesc) == conv._DESC.size
