"""The bench line's counter figures come from summaries of the clip kernel as it
is in the tree; a summary of another kernel is left out."""
import hashlib
import json
import os

import bench


def _tree(tmp_path, kernel):
    for d in ("profiles", "proteusgpu_amd/csrc"):
        os.makedirs(tmp_path / d)
    (tmp_path / "proteusgpu_amd/csrc/voronoi_kernel.h").write_bytes(kernel)
    return str(tmp_path)


def test_counts_of_another_kernel_are_left_out(tmp_path):
    root = _tree(tmp_path, b"kernel")
    assert bench.clip_profile("s.json", root) is None
    for summary, kept in (({}, False), ({"voronoi_kernel_h_sha1": hashlib.sha1(b"older").hexdigest()}, False),
                          ({"voronoi_kernel_h_sha1": hashlib.sha1(b"kernel").hexdigest()}, True)):
        (tmp_path / "profiles/s.json").write_text(json.dumps(summary))
        assert (bench.clip_profile("s.json", root) is not None) == kept


def test_issue_share_of_the_committed_counts():
    """At the first pass's time of 8.5 ms in four launches."""
    v = bench.clip_valu(4, 2.125)
    assert v is None or 0.5 < v["issue_share"] < 1.0
