"""Frames uploaded while their link is busy: chains of frames per link, arenas from one frame's room up
(where nothing is uploaded ahead) to room for all, give the estimates of the links' own handles,
bitwise (the same kernels run in the same order per link), and every frame finishes.
"""
import numpy as np
import pytest

from test_gpu_serve import cfg_of, frames_of, make_server, plain_run, trace

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_links,n_frames,rooms", [(1, 6, 1.0), (1, 6, 4.0), (1, 9, 9.0), (2, 12, 5.0), (3, 16, 40.0), (4, 24, 400.0)])
def test_chains_of_frames(require_gpu, n_links, n_frames, rooms):
    fr, links = trace(n_links, n_frames, rate_hz=1e6, seed=31 + n_frames)
    largest = max(8 * (f["N"] * (f["samples"] + f["pilots"]) + f["samples"] + f["pilots"]) for f in fr)
    srv = make_server(links, cfg_of, arena=int(largest * rooms) + 4096)
    frames = frames_of(fr)
    for _ in range(2):  # a second replay on the learnt state starts from a clean arena
        res = srv.replay(frames)
        assert len(res) == len(frames) and all(r["status"] == 0 for r in res)
    print(f"{n_links} links, {n_frames} frames, arena of {rooms} frames", flush=True)
    for link in range(n_links):
        mine = [k for k, f in enumerate(fr) if f["link"] == link]
        ref = plain_run(links[link], [fr[k] for k in mine] * 2)[len(mine):]
        for k, p in zip(mine, ref):
            np.testing.assert_array_equal(frames[k].est[0], p, err_msg=f"link {link} frame {k}")
