"""Kernel tables are made from traces by the kernels' names: every kernel of a prompt or decode step belongs to an entry point."""
import pathlib
import re

import minivllm_amd.csrc.build as build
from minivllm_amd.engine import roofline

SOURCES = pathlib.Path(build.__file__).parent
# launched on their own, outside the steps that tables are made of
ELSEWHERE = {"empty_kernel", "rope_table_kernel"}


def test_every_kernel_belongs_to_an_entry():
    names = set()
    for path in list(SOURCES.glob("*.hip")) + list(SOURCES.glob("*.h")):
        text = re.sub(r"//.*", "", path.read_text())
        for part in text.split("__global__")[1:]:
            head = part[:part.index("{")]
            names.add(re.findall(r"(\w+_kernel)\s*\(", head)[0])
    assert len(names) > 60
    unknown = sorted(n for n in names - ELSEWHERE if not roofline._OURS.search(n))
    assert not unknown, unknown
