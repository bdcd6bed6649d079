"""The wavefront's packed path state (sample cursor, depth, flags, footprint in
one word) at its ends: the longest path a render may ask for, every vertex
drawing all its samples, gives the megakernel's film, and a longer one is
refused."""
import numpy as np
import pytest

import gyunity_amd as g
from tests.scene_util import furnace_scene


@pytest.mark.gpu
@pytest.mark.parametrize("depth", [99, 100])
@pytest.mark.parametrize("sampler", [g.GY_SAMPLER_SOBOL, g.GY_SAMPLER_HALTON])
def test_longest_paths_render_alike(gpu_ctx, depth, sampler):
    sa = furnace_scene(albedo=0.98)
    sa.light_le[1:] = 0.0  # most walls dark: no path ends early, light comes from deep vertices
    cam = g.camera((0.5, 0.5, 0.5), (0.5, 0.5, 0.0), (0, 1, 0), 60.0, 21, 19)
    with g.Scene(gpu_ctx, sa) as sc:
        films = []
        for mode in (g.GY_RENDER_MEGAKERNEL, g.GY_RENDER_WAVEFRONT):
            films.append(sc.render(cam, g.render_params(3, depth, 1000, mode, sampler=sampler)))
            assert gpu_ctx.stats().rays > 0.9 * 21 * 19 * 3 * depth
        shallow = sc.render(cam, g.render_params(3, depth - 1, 1000, g.GY_RENDER_WAVEFRONT, sampler=sampler))
        with pytest.raises(g.GyError):
            sc.render(cam, g.render_params(3, 101, 1000, g.GY_RENDER_WAVEFRONT, sampler=sampler))
    assert np.array_equal(films[0][0], films[1][0]) and np.array_equal(films[0][1], films[1][1])
    # the last vertex counts with Sobol samples (Halton's dimensions past 255 read 0)
    assert sampler == g.GY_SAMPLER_HALTON or not np.array_equal(shallow[0], films[1][0])
