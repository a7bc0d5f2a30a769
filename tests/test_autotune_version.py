"""File entries of the autotuner carry a version: one measured when the option
values stood for other kernels is not applied."""
import os
import types

import pytest

from ocelot_amd import autotune


@pytest.mark.parametrize("version,source", [(None, "measured"), (autotune.FILE_VERSION, "file")])
def test_entries_of_another_version_are_measured_again(version, source, tmp_path, monkeypatch):
    torch = pytest.importorskip("torch")
    from ocelot_amd import _lib, sc as scmod
    monkeypatch.setenv("OCSC_AUTOTUNE_CACHE", os.path.join(tmp_path, "autotune.json"))
    monkeypatch.setattr(autotune, "_cache", {})
    monkeypatch.setattr(autotune, "_arch", lambda dev: "gfx950")
    set_to = {}
    monkeypatch.setattr(_lib, "set_option", lambda dev, k, v: set_to.__setitem__(k, v))
    monkeypatch.setattr(_lib, "get_option", lambda dev, k: 0)
    monkeypatch.setattr(autotune, "search", lambda space, measure, start: (dict(start), {"overlap": {0: 1.0}}, {}))
    monkeypatch.setattr(scmod, "_nmesh_of", lambda sc: (31, 31, 31))
    monkeypatch.setattr(scmod, "_prec_of", lambda sc: _lib.OCSC_FP64)

    class Rows(torch.Tensor):
        is_cuda = True
        device = types.SimpleNamespace(index=0)
        shape = (6, 1000)

    p = types.SimpleNamespace(rparticles=torch.empty(0).as_subclass(Rows))
    entry = {"options": {"overlap": 1}}
    if version is not None:
        entry["version"] = version
    autotune.store_file(autotune.file_key("gfx950", (31, 31, 31), _lib.OCSC_FP64, 1000), entry)
    res = autotune.tune_tracking(p, types.SimpleNamespace(), 0.1, 0.1, space={"overlap": (0, 1)}, check_bits=False)
    assert res["source"] == source
    assert set_to["overlap"] == (1 if source == "file" else 0)
    assert autotune.load_file()[autotune.file_key("gfx950", (31, 31, 31), _lib.OCSC_FP64, 1000)]["version"] == \
        autotune.FILE_VERSION
