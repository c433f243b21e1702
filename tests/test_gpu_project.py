"""The tiled projection (partition by image tile, LDS sums) against the fixed-point definition
computed with numpy integers: bitwise, at the edges of its groups, tiles and chunks."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import announce, assert_bitwise

pytestmark = pytest.mark.gpu


def _reference(pos, mass, extent, bins):
    """Image of the fixed-point definition: masses scaled by 2^s (largest below 2^34), rounded
    half to even, summed as integers, unscaled once."""
    f32 = np.float32
    lo_a, hi_a, lo_b, hi_b = extent
    with np.errstate(invalid="ignore", over="ignore"):
        fa = np.floor((pos[:, 0] - f32(lo_a)) / f32((hi_a - lo_a) / bins))
        fb = np.floor((pos[:, 1] - f32(lo_b)) / f32((hi_b - lo_b) / bins))
        top = mass[mass > 0]
        shift = 33 - int(np.floor(np.log2(top.max()))) if top.size else 0
        q = np.ldexp(mass.astype(np.float64), shift)
        ok = (fa >= 0) & (fa < bins) & (fb >= 0) & (fb < bins) & (q > 0) & (q < 1.8e16)
    img = np.zeros(bins * bins, np.int64)
    np.add.at(img, fa[ok].astype(np.int64) * bins + fb[ok].astype(np.int64),
              np.rint(q[ok]).astype(np.int64))
    return np.ldexp(img.astype(np.float64), -shift).astype(f32).reshape(bins, bins)


@pytest.mark.parametrize("n,bins,order", [
    (384 * 64, 64, "random"),        # the rule's first tiled size, one tile
    (384 * 65 + 1, 65, "random"),    # a second tile row of one bin, a last group of few
    (384 * 16, 16, "hot"),           # bins below a tile, every particle in one bin
    (4096 * 97 + 5, 1000, "random"),
    (4096 * 100, 1024, "sorted"),    # large images: the direct path below 544 a bin of side
    (8192 * 30, 300, "hot"),         # every chunk adds to one bin
    ((1 << 24) + 4097, 200, "random"),  # more records than the workspace holds at once
])
def test_tiled_projection_matches_integers(device, n, bins, order):
    announce(f"tiled projection n={n} bins={bins} {order}")
    from galaxy_collision_amd.data import ParticleState
    from galaxy_collision_amd.project import scatter_density

    rng = np.random.default_rng(n + bins)
    side = 40.0
    pos = rng.normal(20.0, 6.0, (n, 3)).astype(np.float32)  # some fall outside
    if order == "hot":
        pos[:] = (13.37, 21.5, 5.0)
    elif order == "sorted":
        pos = pos[np.lexsort((pos[:, 1], np.floor(pos[:, 0])))]
    mass = rng.uniform(0.1, 3.0, n).astype(np.float32)
    # dropped or ignored: non-finite and exactly-outside positions, masses that add nothing
    pos[0, 0], pos[1, 1], pos[2, 0] = np.nan, np.inf, side
    mass[3], mass[4], mass[5] = 0.0, -1.0, np.nan
    parts = ParticleState(n)
    parts.load(pos, None, mass)
    img = torch.full((bins, bins), 7.0, device=device)
    scatter_density(parts, img, (0.0, side, 0.0, side))
    assert_bitwise(img.cpu().numpy(), _reference(pos, mass, (0.0, side, 0.0, side), bins), "image")


@pytest.mark.parametrize("n,bins", [(2048, 1), (8192, 4), (10240, 16), (10240, 26), (384 * 27, 27),
                                    (544 * 513, 513), (4096 * 137 + 5, 1000), (544 * 1024, 1024)])
def test_tiled_projection_from_its_first_size(device, n, bins):
    """The first tiled sizes of small and of large images and the last direct ones: the image of
    integers."""
    test_tiled_projection_matches_integers(device, n, bins, "random")
    test_tiled_projection_matches_integers(device, n - 1, bins, "sorted")


def test_tiled_projection_with_the_most_tiles(device):
    test_tiled_projection_matches_integers(device, 4096 * 140, 1024, "sorted")


def test_tiled_projection_rule(device):
    """Images of few bins, and of more than 512, are tiled only from the particles on that pay for
    the extra launches and passes."""
    import ctypes

    from galaxy_collision_amd import _native as nat

    size = ctypes.c_int64()
    for n, bins in ((400, 1), (2047, 1), (3000, 4), (8191, 4), (6144, 16), (10239, 16),
                    (10239, 26), (384 * 27 - 1, 27), (544 * 513 - 1, 513), (345_600, 900),
                    (544 * 1024 - 1, 1024)):
        nat.call("pm_project_work_bytes", n, bins, ctypes.byref(size))
        assert size.value == (bins * bins + 1) * 8, (n, bins)
        nat.call("pm_project_work_bytes", 2 * n + 10240, bins, ctypes.byref(size))
        assert size.value > (bins * bins + 1) * 8, (n, bins)


def test_tiled_projection_workspace_rule(device):
    """The workspace the tiled path asks for stays bounded by its slab of records."""
    import ctypes

    from galaxy_collision_amd import _native as nat

    size = ctypes.c_int64()
    for n, bins, direct in ((1000, 512, True), (384 * 512 - 1, 512, True), (1 << 28, 1025, True),
                            (384 * 512, 512, False), (1 << 28, 1024, False)):
        nat.call("pm_project_work_bytes", n, bins, ctypes.byref(size))
        small = (bins * bins + 1) * 8
        assert (size.value == small) == direct
        # 2^24 records of 8 bytes, 256 tile counts and a maximum per group, the tile totals
        assert size.value <= small + (1 << 27) + 257 * 4 * ((n + 4095) // 4096) + 4096


def test_projection_without_memory_for_records(device):
    """A set whose records do not fit is projected by global atomics, to the same image."""
    from galaxy_collision_amd.data import ParticleState
    from galaxy_collision_amd.project import scatter_density

    n, bins, side = 1 << 21, 64, 40.0
    announce(f"projection, records refused n={n} bins={bins}")
    g = torch.Generator(device=device)
    g.manual_seed(4)
    parts = ParticleState(n)
    parts.load_tensors(torch.rand((n, 3), generator=g, device=device) * side, None,
                       torch.rand(n, generator=g, device=device))
    img = [torch.full((bins, bins), 7.0, device=device) for _ in range(2)]
    scatter_density(parts, img[0], (0.0, side, 0.0, side))
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    # room for the image's sums (32 KB, from a 2 MiB block) and not for 16 MiB of records
    held = torch.cuda.memory_reserved() + (4 << 20)
    torch.cuda.set_per_process_memory_fraction(held / torch.cuda.mem_get_info()[1])
    try:
        scatter_density(parts, img[1], (0.0, side, 0.0, side))
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(img[0], img[1])


def test_tiled_projection_of_a_small_image_in_one_bin(device):
    """Fewer bins than a tile holds, every particle in one of them."""
    test_tiled_projection_matches_integers(device, 10240, 16, "hot")
