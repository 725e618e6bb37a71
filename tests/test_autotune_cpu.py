"""waves and chunk have no effect on the kernels: the tuner does not time them."""
import json

from hcgrid_amd import autotune


def test_launch_shape_is_not_timed(tmp_path, monkeypatch):
    def no_batch(*a, **k):
        raise AssertionError("a batch was built")

    monkeypatch.setattr(autotune._batch, "Batch", no_batch)
    t = autotune.Autotuner(str(tmp_path / "tune.json"))
    assert t.launch_for([dict()], "mix") == (4, 256)
    t.save()
    assert json.loads((tmp_path / "tune.json").read_text())["launch"] == {"mix": [4, 256]}


def test_stored_launch_shape_is_kept(tmp_path):
    p = tmp_path / "tune.json"
    p.write_text(json.dumps({"tiles": {"c1": 32}, "launch": {"mix": [2, 128]}}))
    t = autotune.Autotuner(str(p))
    assert t.launch_for([], "mix") == (2, 128) and t.tiles == {"c1": 32}
