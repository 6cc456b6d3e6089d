"""The renderer's marches take 16, 8 or 4 lanes per pixel by the frame's size.  A
pixel's arithmetic does not depend on that choice, so a frame of either larger
size equals, bit for bit in its image and exactly in its per-pixel counts, the
same pixels rendered through small windows (16 lanes per pixel, the form that
the oracle tests cover).  A window's principal point is the frame's less its
offset, which is exact in float for these values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,win", [
    (131, 127, 96),   # 8 lanes per pixel, ragged tiles
    (363, 367, 121),  # 4 lanes per pixel, ragged tiles
])
@pytest.mark.parametrize("f32", [False, True])
def test_frame_equals_its_windows(H, W, win, f32):
    from plenvdb_amd import scenes, vdbio
    from plenvdb_amd.renderer import MGRenderer

    ms = scenes.merged_scene("c2", H=H, W=W, focal=1111.0 * W / 800, n_poses=10)
    den = ms["den"].astype(np.float32)
    if f32:  # values that fp16 does not hold
        den[1:] += np.float32(1e-4)
    topo, slot_idx = vdbio.index_grid_arrays(ms["idx"])
    p = ms["mlp"]

    def frame(h, w, oy, ox):
        r = MGRenderer(12, 27, 128, 3)
        r.load_params(p["w0"], p["b0"], p["w1"], p["b1"], p["w2"], p["b2"])
        r.load_data_grid(den, ms["col"].astype(np.float32).reshape(-1), topo, slot_idx, len(den))
        assert r.payload_f32 == f32
        K = ms["K"].copy()
        K[0, 2] -= ox
        K[1, 2] -= oy
        r.setScene(ms["reso"], K, ms["xyz_min"], ms["xyz_max"])
        r.setKwargs(ms["near"], ms["far"], ms["stepdist"], ms["act_shift"], ms["interval"],
                    ms["fast_color_thres"], ms["bg"], False, h, w)
        r.set_t_stop(1e-4)
        r.input_a_c2w(ms["poses"][3])
        r.render_an_image()
        count, written = r.pixel_counts()
        return (r.output_an_image().reshape(h, w, 3), count.reshape(h, w), written.reshape(h, w),
                r.sample_counts())

    img, count, written, (gathers, kept) = frame(H, W, 0, 0)
    assert count.sum() > 1000
    g = k = 0
    for oy in range(0, H, win):
        for ox in range(0, W, win):
            h, w = min(win, H - oy), min(win, W - ox)
            wi, wc, ww, (wg, wk) = frame(h, w, oy, ox)
            np.testing.assert_array_equal(count[oy:oy + h, ox:ox + w], wc)
            np.testing.assert_array_equal(written[oy:oy + h, ox:ox + w], ww)
            np.testing.assert_array_equal(img[oy:oy + h, ox:ox + w], wi)
            g += wg
            k += wk
    assert (g, k) == (gathers, kept)
