"""The NN autotuner's saved choices: an index is saved under the names of the
candidates it was chosen from, so that a switch that changes the list
(AFHIP_NN_X3, AFHIP_NN_GATHER) neither reads nor replaces the other list's."""
import json

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_choice_belongs_to_its_list(af, rng, tmp_path, monkeypatch):
    path = tmp_path / "tune.json"
    monkeypatch.setenv("AFHIP_AUTOTUNE_CACHE", str(path))
    X = af.Array(rng.standard_normal((11, 9, 40, 2)).astype(np.float32))
    W = af.Array(rng.standard_normal((3, 3, 40, 24)).astype(np.float32))
    for name, value in ((None, None), ("AFHIP_NN_X3", "0"), ("AFHIP_NN_GATHER", "1")):
        if name:
            monkeypatch.setenv(name, value)
        af.convolve2NN(X, W, (1, 1), (1, 1), (1, 1))
        af.sync()
        if name:
            monkeypatch.delenv(name)
    saved = {k: v for k, v in json.load(open(path)).items() if "x11,9,40,2" in k}
    lists = {tuple(k.split(":of ")[1].split(",")): v for k, v in saved.items()}
    assert len(lists) == 3  # patch, x3 and gemm; patch and gemm; gemm
    for names, choice in lists.items():
        assert len(set(names)) == len(names) and 0 <= choice < len(names)
    assert sum(any("x3" in n for n in names) for names in lists) == 1
    assert sum(any("patch" in n for n in names) for names in lists) == 2
