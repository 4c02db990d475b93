"""bench.py attaches counters only to the kernel they were collected for."""
import json
import os

import bench
import veckern_amd as vk

RECORDS = os.path.join(bench.ROOT, "profiles", "traffic.json")


def test_counters_belong_to_the_kernel_that_ran():
    with open(RECORDS) as f:
        records = json.load(f)
    for name, record in records.items():
        config, _, v9 = name.partition("/")
        assert bench.load_traffic(config, v9 == "v9", record["kernel"]) == record
        assert bench.load_traffic(config, v9 == "v9", "fused_wave_kernel_t<another>") is None
        assert os.path.exists(os.path.join(bench.ROOT, record["source"]))


def test_headline_record_is_of_the_abandoning_scan():
    kernel = vk.ScanKernel(4, 1, 4, 16, 1, 1024, False, False, True, True)
    assert kernel.symbol == "fused_wave_kernel_t<4, 1, 4, 16, 1, 1024, false, false, false, true, true>"
    assert bench.load_traffic("B", False, kernel.symbol)["bound"] == "valu"
