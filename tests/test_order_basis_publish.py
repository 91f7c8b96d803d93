"""The M_Basis kernel hands panels and bookings from wave to wave through LDS: words
first, then a count that another wave polls.  LDS does one wave's accesses in order,
but only a compiler fence keeps the count's store behind the words' stores (they are
different arrays), so every count goes through publish(), which has one."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "linbox_amd", "csrc")


def test_counts_are_published_behind_their_words():
    text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, "order_basis.hip")).read())
    body = re.search(r"void publish\(.*?\n}", text, re.S).group(0)
    assert re.search(r"__atomic_signal_fence\(__ATOMIC_SEQ_CST\);\s*__hip_atomic_store\(", body)
    for word in ("s_pub", "s_book"):
        assert re.search(r"\bpublish\(&%s\b" % word, text), word
        # other stores only clear it (before a barrier)
        assert not [v for v in re.findall(r"\b%s\s*=\s*([^=;][^;]*);" % word, text) if v != "0"], word
        assert not re.search(r"atomic_store\(&%s\b" % word, text), word
