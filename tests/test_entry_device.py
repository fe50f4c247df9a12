"""Every C entry that launches kernels or allocates device memory selects the handle's device first: the caller's
current device may be another one, and each host thread starts on device 0.  One GPU cannot show a missing
call, so the entries are read from the source."""
from __future__ import annotations

import re

from vkscanlinepr_amd import build

REACHES = r"spr::launch_|\brun_frame\(|\brun_learned_frame\(|\brun_records_frame\(|\brender_nosync\(|\bread_image\(|" \
          r"\bload_arrays\(|\.ensure\(|\.upload\(|mlp_train\(|mlp_gradients\("


def test_entries_select_the_device():
    src = (build.CSRC / "spr_api.cpp").read_text()
    entries = re.findall(r"^int (spr_\w+)\((.*?)^}", src, re.S | re.M)
    assert len(entries) > 20
    seen, missing = set(), []
    for name, body in entries:
        m = re.search(REACHES, body)
        # loads select it where they all end (load_arrays); the allocation-free scan takes no handle
        if not m or name == "spr_scan_i32_noalloc" or m.group() == "load_arrays(":
            continue
        seen.add(name)
        if "hipSetDevice(" not in body[:m.start()]:
            missing.append(name)
    assert {"spr_render_frame", "spr_batch_image", "spr_scan_i32"} <= seen
    assert not missing
