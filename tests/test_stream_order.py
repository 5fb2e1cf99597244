"""CPU check of the host code's order on the device: the contexts' streams do
not wait for the null stream, so a clear on it (hipMemset returns before it is
done) or a copy on it from pageable memory (which may return once the bytes are
staged) is waited for before a launch can meet it."""
from __future__ import annotations

import re
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "bobcat_amd" / "csrc"


def unwaited(pattern: str) -> list[str]:
    """Calls that no synchronisation follows within their function."""
    found = []
    for path in sorted(CSRC.glob("*.hip")):
        text = path.read_text()
        for m in re.finditer(pattern, text):
            rest = text[m.end():].split("\n}\n", 1)[0]
            if not re.search(r"hipStreamSynchronize\(|hipDeviceSynchronize\(", rest):
                found.append(f"{path.name}: {m.group(0)}")
    return found


def test_null_stream_clears_are_waited_for():
    assert unwaited(r"hipMemset\(") == []


def test_null_stream_copies_to_the_device_are_waited_for():
    assert unwaited(r"hipMemcpy\([^;]*hipMemcpyHostToDevice") == []
