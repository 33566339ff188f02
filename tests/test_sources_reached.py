"""Every launcher and device helper of the library's sources is called (CPU test)."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "brig-join_amd", "csrc")
FILES = sorted(glob.glob(CSRC + "/*.h") + glob.glob(CSRC + "/*.hip") + glob.glob(CSRC + "/*.cpp"))
TEXT = "\n".join(re.sub(r"//[^\n]*", "", open(f).read()) for f in FILES)


def named(pattern):
    return sorted(set(re.findall(pattern, TEXT)))


@pytest.mark.parametrize("name", named(r"\bhipError_t (launch_\w+)\("))
def test_launcher_is_called(name):
    assert len(re.findall(rf"(?<!hipError_t )\b{name}\(", TEXT)) > 0


@pytest.mark.parametrize("name", named(r"__device__ (?:__forceinline__ )?[\w:<> ]+?\b(\w+)\(")
                         + named(r"__global__[^;{]*?\b(kb?_\w+)\("))
def test_device_function_is_called(name):
    # its definition, and at least one use (a call, a launch or a template instance)
    assert len(re.findall(rf"\b{name}\b", TEXT)) > len(re.findall(rf"[\w>] {name}\([^;{{]*\)\s*(?:const\s*)?\{{", TEXT))
