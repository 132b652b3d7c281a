"""The native sources keep off the default stream: the device serves four hardware queues per
process, a default stream that has been used holds one of them, and a batch spread over four
streams then runs some of its classes one behind another (no GPU)."""
import pathlib
import re

import pis_amd

CSRC = pathlib.Path(pis_amd.__file__).parent / "csrc"
# synchronous forms run on the default stream; so do asynchronous ones and launches given stream 0
DEFAULT_STREAM = re.compile(r"\bhip(?:Memcpy|Memset|Memcpy2D|Memset2D|MemsetD32|MemcpyDtoH|MemcpyHtoD)\s*\("
                            r"|\bhipStreamDefault\b|<<<"
                            r"|\bhip(?:Memcpy|Memset)Async\([^;]*,\s*(?:0|nullptr)\)")


def test_native_sources_use_no_default_stream():
    files = sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.cpp"))
    assert files
    found = [f"{f.name}:{i}: {line.strip()}" for f in files
             for i, line in enumerate(f.read_text().splitlines(), 1)
             if DEFAULT_STREAM.search(line) and not line.lstrip().startswith("//")]
    assert not found, "\n".join(found)
