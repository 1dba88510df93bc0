"""The tuner's cache: what another generation of the panels measured is not
applied to these."""
import json
import types

import torch


def test_cache_of_another_generation_is_not_used(nla, tmp_path, monkeypatch):
    from nextla_amd import tune
    path = tmp_path / "tune.json"
    monkeypatch.setenv("NEXTLA_AMD_TUNE_CACHE", str(path))
    props = types.SimpleNamespace(name="AMD Instinct", gcnArchName="gfx950", multi_processor_count=256)
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda dev: props)
    measured = []
    monkeypatch.setattr(tune, "tune_panels", lambda dt: measured.append(dt) or {"rows": 512, "strip": 16, "ms": {}})
    monkeypatch.setattr(tune, "tune_batch", lambda dt: {"mask": 0x1F, "ms": {}})
    # a file without a generation in its key, as earlier versions wrote it
    old = {"panel": {"f64": {"rows": 256, "strip": 32}}, "batch_classes": 0x8}
    path.write_text(json.dumps({"AMD Instinct|gfx950|256": old}))
    cfg = tune.tune(device="cuda", apply_result=False)
    assert measured == ["f32", "f64"] and cfg["panel"]["f64"]["rows"] == 512
    assert tune.tune(device="cuda", apply_result=False) == cfg and len(measured) == 2
    assert json.loads(path.read_text())["AMD Instinct|gfx950|256"] == old
