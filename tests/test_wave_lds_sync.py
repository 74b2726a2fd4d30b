"""The kernels that transpose a tile through wave-private LDS (one lane stores
words that other lanes of its wave load) state the order of the stores and the
loads: the compiler may otherwise move one past the other wherever it can tell
that a lane's own addresses differ.  Read from the sources, the generated
kernel's among them, so that the check needs no GPU."""

import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "mojogp_amd" / "csrc"


@pytest.mark.parametrize("name", ["direct.hip", "tree_jit.hip"])
def test_transposition_is_ordered(name):
    text = (CSRC / name).read_text()
    spots = list(re.finditer(r"float\* sc = tsc\[wave\]\[r & 1\];", text))
    assert len(spots) == 1
    body = text[spots[0].end():]
    store = re.search(r"\(sc \+ lm \* VS \+ 4 \* lq\) =", body).start()
    load = re.search(r"sc\[\(4 \* lq \+ s\) \* VS \+ lm\]", body).start()
    assert store < load
    assert "wave_lds_sync();" in body[store:load]


@pytest.mark.parametrize("name", ["sym_common.h", "tree_jit.hip"])
def test_sync_is_a_fence_and_a_wave_barrier(name):
    text = (CSRC / name).read_text()
    body = re.search(r"void wave_lds_sync\(\) \{(.*?)\}", text, re.S).group(1)
    at = [body.index(x) for x in ("__ATOMIC_RELEASE, \"wavefront\"", "__builtin_amdgcn_wave_barrier()",
                                  "__ATOMIC_ACQUIRE, \"wavefront\"")]
    assert at == sorted(at)
