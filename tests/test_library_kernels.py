"""The stage kernels the built library holds, by their symbol names: every
stage that a launch can ask for in each storage type, and none besides."""
import re

from volumefluxes import _capi as C


def test_stage_instantiations():
    names = open(C.lib_path(), "rb").read()
    for family in (b"k_march", b"k_block"):
        found = {(s.decode(), int(n)) for s, n in re.findall(family + rb"I([df])Li(\d)ELi", names)}
        assert found == {("d", 1), ("d", 2), ("d", 3), ("d", 4), ("f", 1), ("f", 2), ("f", 3)}, family
