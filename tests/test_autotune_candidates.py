"""The autotuner tries the shapes that a context starts with, so that it can end
at what was measured best, and begins each search with the present shape, so
that a stage keeps it unless another is faster.  Read from the source: which
shape wins on a GPU is a matter of its timings."""
import re
from pathlib import Path

import pytest

SOURCE = (Path(__file__).resolve().parent.parent / "binarymeshfitting_amd" / "csrc" / "bmf_capi.hip").read_text()


def _tuner():
    at = SOURCE.index("int bmf_autotune(")
    return SOURCE[at:SOURCE.index("// confirmation", at)]


@pytest.mark.parametrize("field", ["sample_blocks", "row_blocks", "smooth_blocks"])
def test_candidates_hold_the_start(field):
    start = int(re.search(r"c->tune\.%s = c->cu_count \* (\d+);" % field, SOURCE).group(1))
    tried = re.search(r"search\(&bmf_tuning::%s,\s*\{([^}]*)\}" % field, _tuner()).group(1)
    assert f"{start} * cu" in [t.strip() for t in tried.split(",")]


def test_search_begins_with_the_present_shape():
    body = _tuner()
    first = body.index("attempt(cur.*shape)")
    assert first < body.index("for (int b : others)")
