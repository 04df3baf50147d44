"""The tuning cache names the forms of the kernels a choice was timed with:
entries of other forms are not taken over, entries of these are."""
import re

import pytest

from plegma_amd import capi

import gpu_util as G

pytestmark = pytest.mark.gpu

MASK = capi.G_NUCL | capi.G_DELTAPP_ALL


@pytest.mark.parametrize("mode", ["f64", "mixed"])
@pytest.mark.parametrize("kind", ["twopt", "mesmes"])
def test_choices_of_other_forms_are_timed_again(kind, mode, tmp_path, monkeypatch):
    torch = G.torch_cuda()
    cache = tmp_path / "tune"
    monkeypatch.setenv("PLG_TUNE_CACHE", str(cache))
    L, src, totalT = [4, 4, 4, 4], [0, 1, 2, 1], 3
    print(f"\n[gpu] plg_init {L}", flush=True)
    capi.init(L, 0)
    try:
        keep = [G.make_prop(L, 3, 1 + i, src[3], 0.5) for i in range(2)]
        m = capi.MODE_F64
        views = [v for _, v in keep]
        if mode == "mixed":
            m = capi.MODE_MIXED
            keep += [G.cast_f32(t, v) for t, v in keep]
            views = [v for _, v in keep[2:]]
        moms = capi.momlist(1)
        code, mask = (capi.TWOPT, MASK) if kind == "twopt" else (capi.MESON_MESON, 0)
        jobs = [(src, totalT, 0, 0) + ((1,) if kind == "mesmes" else ())]

        def tuned():
            b = capi.Batch(code, mask, views, jobs, moms, m, flags=capi.BATCH_TUNE)
            b.close()
            return cache.read_text().splitlines()

        first = tuned()
        assert first and all(re.search(r" kernels=[^,]+,", line) for line in first)
        assert tuned() == first
        other = [re.sub(r" kernels=[^,]+,", "", line) for line in first]
        cache.write_text("\n".join(other) + "\n")
        again = tuned()
        assert again[:len(other)] == other and len(again) == len(other) + len(first)
    finally:
        capi.finalize()
