"""Which kernel scope bench.py quotes its roofline for (CPU only)."""
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


def test_the_roofline_names_a_scope_of_the_critical_path():
    prof = {"contact_group": {"ms": 0.96, "launches": 8}, "hash_query": {"ms": 0.9, "launches": 0},
            "narrow_set": {"ms": 0.8, "launches": 10}, "contact_pk": {"ms": 0.5, "launches": 8}}
    ranked = sorted(prof.items(), key=lambda kv: -kv[1]["ms"])
    assert bench.dominant_scope(ranked)[0] == "narrow_set"
    assert bench.dominant_scope([kv for kv in ranked if kv[0] in bench.SIDE_SCOPES]) is None
