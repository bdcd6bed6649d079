"""Films of a batch: one launch over the concatenated pixels of all entries.
Entries of one pixel, below, at and above a 256-pixel workgroup, and with
samples on pixel borders, in one batch: each film is its own render's."""
import numpy as np
import pytest

import gyunity_amd as g


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[(1, 1)], [(1, 1), (3, 85), (16, 16), (257, 1), (9, 64)], [(64, 64), (1, 255), (2, 1)]])
@pytest.mark.parametrize("use_graph", [True, False])
def test_films_of_ragged_entries(gpu_ctx, sizes, use_graph):
    sa, _, _ = g.generate_scene(g.GY_SCENE_CORNELL, 0, 64)
    with g.Scene(gpu_ctx, sa) as sc, g.Batch(gpu_ctx, use_graph=use_graph) as b:
        views = [(g.camera((0.5, 0.5, 2.35), (0.5, 0.5, 0.0), (0, 1, 0), 40.0, w, h),
                  g.render_params(5 + 27 * i, 3, mode=g.GY_RENDER_WAVEFRONT, samples_per_pass=5 + 27 * i))
                 for i, (w, h) in enumerate(sizes)]
        refs = [sc.render(cam, prm) for cam, prm in views]
        ids = [b.add(sc, cam, prm) for cam, prm in views]
        for _ in range(3):
            b.render()
            for e, (color, weight) in zip(ids, refs):
                got = b.film(e)
                assert np.array_equal(got[1], weight) and np.array_equal(got[0], color)
            sc.render(*views[0])
        assert all(c.sum() > 0 for c, _ in refs)
        # samples on pixel borders count in more than one pixel
        assert len(sizes) == 1 or any((w > 5 + 27 * i).any() for i, (_, w) in enumerate(refs))
