"""Device memory is filled and copied in the order of the context's stream, which
does not wait for the null stream: no asynchronous fill goes anywhere else."""
import os
import re

from exadglm_amd.build import CSRC, HIP_SRCS


def _calls(src, name):
    """The argument text of every call of a function."""
    for m in re.finditer(r"\b%s\(" % name, src):
        depth, i = 1, m.end()
        while depth:
            depth += {"(": 1, ")": -1}.get(src[i], 0)
            i += 1
        yield src[m.end():i - 1]


def test_fills_and_async_copies_go_to_the_context_stream():
    seen = 0
    for f in HIP_SRCS:
        src = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, f)).read())
        # (a fill of device memory may return before it is done, on the null stream)
        assert not list(_calls(src, "hipMemset")), f
        for name in ("hipMemsetAsync", "hipMemcpyAsync"):
            for args in _calls(src, name):
                assert re.search(r",\s*c->stream$", args.strip()), (f, name, args)
                seen += 1
    assert seen > 10
