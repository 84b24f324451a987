"""The attention kernel's measured HBM traffic is quoted for the code it was measured on."""
import hashlib
import json
import os
import re

from blockgtq_amd import _capi, build

TABLE = os.path.join(os.path.dirname(build.CSRC), "measured_traffic.json")


def _code(name):
    text = open(os.path.join(build.CSRC, name)).read()
    return re.sub(r"\s+", "", re.sub(r"/\*.*?\*/|//[^\n]*", "", text, flags=re.S))


def test_traffic_figures_belong_to_the_kernel_as_it_is():
    table = json.load(open(TABLE))
    have = hashlib.sha256("".join(_code(f) for f in ("bgtq_decode_seg.hip", "bgtq_lds.h")).encode()).hexdigest()[:16]
    assert table["decode_kernel_source"] == have, (
        "the attention kernel changed: raise bgtq_decode_kernel_revision(), so that the old figures are not quoted, measure "
        f"again as the profile says and put the new revision and the fingerprint {have} into measured_traffic.json")
    assert {e["decode_kernel_revision"] for e in table["entries"].values()} == {_capi.lib().bgtq_decode_kernel_revision()}
    root = os.path.dirname(os.path.dirname(build.CSRC))
    for entry in table["entries"].values():
        assert f"decode kernel revision {entry['decode_kernel_revision']}" in open(os.path.join(root, entry["profile"])).read()
