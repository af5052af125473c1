"""The measured HBM traffic that bench.py reports beside the headline holds for the
tile kernel it was measured on only, so the record carries that source's digest: a
change to the kernel needs a new measurement."""
import hashlib
import json
import os

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_traffic_record_is_of_this_kernel():
    with open(os.path.join(REPO, "profiles", "tile_kernel_traffic_4d_gauss2e6.txt")) as f:
        rec = json.load(f)
    with open(os.path.join(REPO, "dendro-kt_amd", "csrc", "tile_kernel.h"), "rb") as f:
        assert rec["tile_kernel_sha256"] == hashlib.sha256(f.read()).hexdigest()
    assert rec["hbm_bytes_per_launch_f64"] > rec["hbm_bytes_per_launch_f32"] > 0
