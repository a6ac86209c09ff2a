"""bench.py's loaders by the plan flags they stand for (no GPU)."""
import os
import sys
from types import SimpleNamespace

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402
import onegraph_amd as og  # noqa: E402


def test_plan_flags():
    args = SimpleNamespace(loader="zerocopy", no_pack=False, no_overlap=False, no_fuse=False)
    assert bench.plan_flags(args, "ascetic") == og.PLAN_ZERO_COPY
    # the comparison runs Subway as gather and copy, whatever the headline's loader
    assert bench.plan_flags(args, "subway", "copy") == og.PLAN_NO_FUSE
    assert bench.plan_flags(args, "usm", "copy") == 0
    args.loader, args.no_overlap = "copy", True
    assert bench.plan_flags(args, "ascetic") == og.PLAN_NO_FUSE | og.PLAN_NO_OVERLAP
