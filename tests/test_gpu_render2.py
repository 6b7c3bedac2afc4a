"""render2 (fut/voxel_renderer.fut:257-305), the reference's ray-march
renderer, on the GPU (fsx_render2) against the oracle's literal
restatement: bit-exact frames."""
import numpy as np
import pytest

from futspace_amd import View, scene
from oracle import fs_oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

VIEWS = [
    View(x=20.37, y=41.61, height=180.0, angle=0.7, horizon=10.0, distance=300.0, fov=1.2,
         h=48, w=64),
    View(x=100.5, y=3.25, height=260.0, angle=3.9, horizon=-12.0, distance=800.0, fov=1.2,
         h=61, w=77),                                        # rays wrap around the map
    View(x=64.0, y=64.0, height=120.0, angle=0.0, horizon=25.0, distance=160.0, fov=1.2,
         h=40, w=30),                                        # integral camera position
    View(x=12.9, y=80.1, height=-3.0, angle=5.5, horizon=0.0, distance=50.0, fov=1.2,
         h=16, w=20),                                        # camera inside the terrain
]


def _maps(kind):
    if kind == "p2":
        col, hts = scene.scene_maps(23, 128)
    elif kind == "np2":
        col, hts = scene.scene_maps(24, 128)
        col, hts = np.ascontiguousarray(col[:100, :90]), np.ascontiguousarray(hts[:100, :90])
    else:                                                    # colour-0 texels
        col, hts = scene.scene_maps(25, 64)
        col = col.copy()
        col[::4, :] = 0
    return col, hts


@pytest.mark.parametrize("kind", ["p2", "np2", "zero"])
@pytest.mark.parametrize("vi", range(len(VIEWS)))
def test_render2_matches_oracle(ctx, kind, vi):
    col, hts = _maps(kind)
    v = VIEWS[vi]
    m = ctx.map(col, hts)
    got = ctx.render2(m, v)
    want = O.render2(v, col, np.asarray(hts, dtype=np.int32) & 255)
    bad = int(np.count_nonzero(got != want))
    assert bad == 0, f"{bad} of {got.size} pixels differ"


def test_render2_sixteen_bit_heights_and_pitch(ctx):
    hts = scene.heightmap(26, 128, 0.6, 900)
    col = scene.colormap(26, hts, 900)
    m = ctx.map(col, hts, height_bits=16)
    v = View(x=40.2, y=77.9, height=1000.0, angle=2.2, horizon=15.0, distance=600.0, fov=1.2,
             h=37, w=53)
    out = torch.zeros((v.h, 64), dtype=torch.int32, device="cuda")
    ctx.render2(m, v, out)
    ctx.sync()
    want = O.render2(v, col, np.asarray(hts, dtype=np.int32) & 0xFFFF)
    got = out.cpu().numpy().view(np.uint32)
    assert np.array_equal(got[:, :v.w], want)
    assert np.all(got[:, v.w:] == 0)


def test_render2_rejects_unbounded_march(ctx):
    col, hts = _maps("p2")
    m = ctx.map(col, hts)
    v = View(x=1.0, y=1.0, height=100.0, angle=0.0, horizon=0.0, distance=1e8, fov=1.2, h=4, w=4)
    with pytest.raises(RuntimeError):
        ctx.render2(m, v)


@pytest.mark.parametrize("distance,h,w,horizon,bits", [
    (-8.0, 5, 7, 3.0, 8),                                    # no step at all
    (3.0, 33, 65, 8.0, 8),                                   # one step
    (60.0, 32, 64, 30.0, 8), (64.0, 31, 63, 30.0, 16),       # one group of steps, and one more
    (1020.0, 65, 129, 2.0, 8), (1024.0, 40, 66, 1.0, 8),     # one chunk of steps, and one more
    (2100.0, 34, 70, -0.5, 16),                              # looking up and down
    (400.0, 33, 65, float("inf"), 8), (400.0, 20, 30, float("-inf"), 8),
])
def test_render2_steps_and_tiles(ctx, distance, h, w, horizon, bits):
    """Marches and frames at the edges of the kernel's groups, chunks and
    workgroups, over a map that misses in places."""
    hts = scene.heightmap(27, 128, 0.6, 255 if bits == 8 else 900)
    hts = np.ascontiguousarray(hts[:, :96])
    col = scene.colormap(27, hts, 255 if bits == 8 else 900)
    m = ctx.map(col, hts, height_bits=bits)
    for x, height in ((40.2, 1.2 * hts.max()), (90.7, 0.5 * hts.max())):
        v = View(x=x, y=77.9, height=float(height), angle=2.2, horizon=horizon,
                 distance=distance, h=h, w=w)
        want = O.render2(v, col, np.asarray(hts, np.int32) & (255 if bits == 8 else 0xFFFF))
        got = ctx.render2(m, v)
        bad = int(np.count_nonzero(got != want))
        assert bad == 0, f"{bad} of {got.size} pixels differ"


@pytest.mark.parametrize("h,w,distance,bits,cols", [
    (40, 70, 252.0, 8, 128), (40, 70, 256.0, 16, 96), (33, 65, 700.0, 8, 96),   # a workgroup per CU
    (35, 16640, 20.0, 8, 96), (3, 16640, 280.0, 16, 128),                       # two per CU
    (3, 49200, 260.0, 8, 128), (129, 24640, 24.0, 16, 96),                      # 128 rows
])
def test_render2_of_low_cameras(ctx, h, w, distance, bits, cols):
    """Cameras in, on and little above the ground, level and steep, whose hits
    lie before, in and after the short first chunk, in each of the kernel's
    shapes."""
    top = 255 if bits == 8 else 900
    hts = scene.heightmap(33, 128, 0.6, top)
    col = scene.colormap(33, hts, top)[:, :cols].copy()
    hts = np.ascontiguousarray(hts[:, :cols])
    m = ctx.map(col, hts, height_bits=bits)
    alt = np.asarray(hts, np.int32) & (255 if bits == 8 else 0xFFFF)
    cases = [(-5.0, 3.0), (0.5, 60.0), (9.0, 20.0), (30.0, 4.0)]
    for above, horizon in cases if h * w < 1 << 20 else cases[1:2]:
        v = View(x=40.2, y=77.9, height=float(hts[77, 40] + above), angle=2.2, horizon=horizon,
                 distance=distance, h=h, w=w)
        want = O.render2(v, col, alt)
        got = ctx.render2(m, v)
        bad = int(np.count_nonzero(got != want))
        assert bad == 0, f"{above} {horizon}: {bad} of {got.size} pixels differ"
