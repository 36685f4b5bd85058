"""The NN autotuner's saved choices: an index is saved under the names of the
candidates it was chosen from, so that a switch that changes the list
(AFHIP_NN_X3, AFHIP_NN_GATHER) neither reads nor replaces the other list's.
Layers that fill the chip, strided data gradients that do so phase by phase and
all filter gradients are not timed at all: the same bits with the autotuner on
and off."""
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


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("x,w,st", [((64, 64, 32, 32), (3, 3, 32, 48), 1), ((75, 75, 16, 32), (3, 3, 16, 32), 1),
                                    ((67, 40, 48, 24), (1, 1, 48, 64), 1), ((112, 112, 24, 32), (3, 3, 24, 64), 2)],
                         ids=["rows of vectors", "odd rows", "1x1", "stride 2"])
def test_layers_that_fill_the_chip_are_not_timed(af, rng, dt, x, w, st, tmp_path, monkeypatch):
    t = {"f32": af.f32, "bf16": af.bf16}[dt]
    geo = ((st, st), (w[0] // 2,) * 2, (1, 1))
    X = af.Array(rng.standard_normal(x).astype(np.float32)).astype(t)
    W = af.Array((rng.standard_normal(w) * 0.1).astype(np.float32)).astype(t)
    y = af.convolve2NN(X, W, *geo)
    DY = af.Array(rng.standard_normal(y.dims).astype(np.float32)).astype(t)

    def step():
        out = [af.convolve2NN(X, W, *geo)]
        out += [af.convolve2GradientNN(DY, X, W, y, *geo, k)
                for k in (af.AF_CONV_GRADIENT_DATA, af.AF_CONV_GRADIENT_FILTER)]
        return [o.to_numpy() for o in out]

    path = tmp_path / "tune.json"
    monkeypatch.setenv("AFHIP_AUTOTUNE_CACHE", str(path))
    timed = step()
    monkeypatch.setenv("AFHIP_NN_AUTOTUNE", "0")
    for a, b in zip(timed, step()):
        np.testing.assert_array_equal(a, b)
    keys = [k for k in json.load(open(path)) if f"x{x[0]},{x[1]},{x[2]},{x[3]}:" in k] if path.exists() else []
    assert not keys
