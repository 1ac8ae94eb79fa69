"""Seeded programs keep their texts: draws, token steps, prompts and replies against values recorded earlier
(seeded_cases.py says from what)."""
import json

import pytest

import seeded_cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["draws", "edge_draws", "steps", "prompts", "replies"])
def test_seeded_values_stay(name):
    with open(seeded_cases.GOLDEN) as f:
        want = json.load(f)[name]
    print(f"seeded {name}", flush=True)
    got = getattr(seeded_cases, name)()
    changed = [k for k in want if got[k] != want[k]]
    assert not changed, f"{len(changed)} of {len(want)} {name} differ: {changed[:20]}"
