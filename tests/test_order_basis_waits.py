"""The waits of the order-basis kernels end after a number of polls, and one that
gives up must say so: the host then fails the call instead of returning a basis made
of unfinished data.  A wait can only run out on a device that lost a wave, so what is
checked is the source: each use of the poll limit raises the failure flag."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "linbox_amd", "csrc")


def test_every_wait_that_gives_up_reports():
    text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, "order_basis.hip")).read())
    text = text.replace("constexpr unsigned kMcSpinLimit", "")
    uses = len(re.findall(r"\bkMcSpinLimit\b", text))
    assert uses == 3  # the grid barrier, the panels, their booking
    assert len(re.findall(r"if \(\+\+polls == kMcSpinLimit\) \{\s*report_wait\(bar\);", text)) == uses
    assert re.search(r"void report_wait\(unsigned \*bar\)\s*\{\s*__hip_atomic_store\(bar \+ 1, 1u,", text)
    assert "&failed, R.mb.bar + 1" in text and re.search(r"&& failed\) st = LBX_ERR_HIP", text)  # the host reads it
