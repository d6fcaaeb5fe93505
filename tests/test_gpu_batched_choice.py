"""The variant that a rule picks for a list of pairs is kept with the sizes and the
iteration count: lists that differ in one of them do not take each other's, and long lists
(of which the rule looks at some pairs) give every pair its solve."""
import numpy as np
import pytest
import torch

from hindemith_amd import batched
from hindemith_amd._lib import lib

pytestmark = pytest.mark.gpu


def _list(shapes, iters, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    f = lambda: [torch.randn(*s, generator=g, device="cuda") for s in shapes]  # noqa: E731
    return batched.BatchedHS(f(), f(), [0.5 + 0.25 * (i % 5) for i in range(len(shapes))],
                             iters=iters)


def test_choices_are_kept_by_sizes_and_iterations():
    rng = np.random.default_rng(4)
    tiny = [(int(h), int(w)) for h, w in rng.integers(1, 40, (300, 2))]
    other = [(w, h) for h, w in tiny]
    few = [(200, 300), (90, 40), (1, 64)]
    lists = [_list(s, it, i) for i, (s, it) in enumerate(
        [(tiny, 20), (tiny, 3), (tiny, 1), (other, 20), (few, 20), (few, 200), (few, 2)])]
    refs = [[(u.clone(), v.clone()) for u, v in b.solve_each(variant=0, k=1)] for b in lists]
    for rep in range(2):
        for b, ref in zip(lists, refs):
            for (u, v), (ru, rv) in zip(b.run(graph=rep == 1), ref):
                assert torch.equal(u, ru) and torch.equal(v, rv), (b.iters, tuple(u.shape))
        lib().hmx_hs_batched_release()
