"""The quad form's Sigma, replayed on the CPU: each of a half's four lanes rotates by one amount, two quad
permutations (lane i reads lane NEXT[i], then AFTER[i]) add the other rotations, and every lane ends on the sum
the two-lane form computes in one lane (tests/test_sha_lanes_math.py replays the rest, which both forms share)."""
import random
import re
from pathlib import Path

import pytest

from tests.test_sha_lanes_math import MASK, Lane, rotr

SOURCE = (Path(__file__).resolve().parent.parent / "kvsnap_amd" / "csrc" / "kernels.hip").read_text()


def permutations():
    """The permutations as the assembly spells them, in the order a slot applies them."""
    macro = SOURCE[SOURCE.index("#define SHA_QUAD("):]
    found = re.findall(r"quad_perm:\[(\d),(\d),(\d),(\d)\]", macro[:macro.index("#define SHA_SLOT(")])
    return [tuple(map(int, p)) for p in found]


def sigma(x, rotations, next_, after):
    y = [rotr(x, r) for r in rotations]
    p = [y[next_[i]] ^ y[i] for i in range(4)]
    return [y[after[i]] ^ p[i] for i in range(4)]


@pytest.mark.parametrize("a_lane", [False, True])
def test_every_lane_of_a_quad_ends_on_sigma(a_lane):
    next_, after = permutations()
    r1, r2, r3 = Lane(a_lane).r
    for seed in range(50):
        x = random.Random(seed).randrange(MASK + 1)
        assert sigma(x, (r1, r2, r3, r1), next_, after) == [Lane(a_lane).sigma(x)] * 4


def test_the_builtin_permutations_are_the_assembly_s():
    names = {}
    for name in ("kDppQuadNext", "kDppQuadAfter"):
        terms = re.search(rf"{name} = ([^;]+);", SOURCE).group(1)
        names[name] = eval(terms, {"__builtins__": {}})          # shifts and ors of literals
    assert [tuple((names[n] >> 2 * i) & 3 for i in range(4)) for n in ("kDppQuadNext", "kDppQuadAfter")] == \
        permutations()
