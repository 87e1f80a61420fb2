"""A prompt finds its pages in the prefix tree whatever sequence its token ids come in."""
import numpy as np
import pytest
import torch

from ullm_amd.cache.prefix_tree import PrefixTree

FORMS = dict(list=list, tuple=tuple, numpy=lambda t: np.asarray(t, dtype=np.int64), tensor=lambda t: torch.tensor(t, dtype=torch.int64),
             numpy_ints=lambda t: [np.int32(x) for x in t], mixed=lambda t: [np.int64(x) if i % 37 == 36 else x for i, x in enumerate(t)])


@pytest.mark.parametrize("n", [0, 3, 4, 63, 64, 65, 130])
@pytest.mark.parametrize("stored", sorted(FORMS))
def test_keys_do_not_depend_on_the_kind_of_sequence(n, stored):
    tokens = [(7 * i + 3) % 1000 for i in range(n)]
    tree = PrefixTree(4, [])
    assert tree.insert(FORMS[stored](tokens), n, []) == n // 4
    want = [tuple(tokens[i:i + 4]) for i in range(0, n // 4 * 4, 4)]
    for asked in FORMS.values():
        assert list(tree._keys(asked(tokens), n)) == want
        assert len(tree.match(asked(tokens), n)) == n // 4
        assert tree.insert(asked(tokens), n, []) == 0
        assert all(type(x) is int for key in tree._keys(asked(tokens), n) for x in key)
    if n >= 4:
        assert len(tree.match([1] + tokens[1:], n)) == 0
